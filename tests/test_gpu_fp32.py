"""The fp32 products (csrc/gemm_f32.hip: three bf16 parts per value, six partial products) against fp64, at the sizes
where their tiles, stages and runs end: rows around the 128-column tile, widths around the 32-value stage and not a
multiple of it, vocabularies around the 256-row tile and not a multiple of 4, grad_h's contraction in one run and in
several, rows through the map with a device count, the soft-cap, values of very different size.

Every sum is of exact partial products down to 2^-23 of each product, added in fp32: its error is at most
2^-23 + 2^-24 (terms / 32 + 6) times the sum of the products' sizes in the worst case, and about 2^-23 of their norm in
practice, which the bounds below take eight times."""

import pytest
import torch

from octopus_amd import head_op
from octopus_amd.head_op import Post, fused_head

pytestmark = pytest.mark.gpu
DEV = "cuda"
EPS = 8 * 2.0 ** -23


def _case(N, d, V, post, spread, seed):
    g = torch.Generator().manual_seed(seed)
    h = torch.randn(N, d, generator=g)
    W = torch.randn(V, d, generator=g) * d ** -0.5
    if spread:  # columns of very different size, the other operand's inversely: every product counts
        e = torch.randint(-spread, spread + 1, (d,), generator=g).float()
        h, W = h * 2.0 ** e, W * 2.0 ** -e
    y = torch.randint(0, V, (N,), generator=g)
    scored = torch.rand(N, generator=g) < 0.7
    scored[0] = True
    return h, W, y, scored, torch.randn(N, generator=g)


@pytest.mark.parametrize("N,d,V,post,spread", [
    (1, 4, 5, None, 0), (127, 36, 255, None, 0), (129, 32, 257, None, 0), (190, 1000, 3001, None, 0),
    (300, 128, 20480, None, 0), (500, 260, 8190, (0.2, 5.0), 0), (200, 256, 4099, None, 40),
], ids=str)
def test_fp32_head_against_64_bits(N, d, V, post, spread):
    h, W, y, scored, g = _case(N, d, V, post, spread, seed=N + V)
    T = 0.8
    hd, Wd = h.to(DEV).requires_grad_(True), W.to(DEV).requires_grad_(True)
    idx, count = head_op.compact_rows(scored.to(DEV))
    out = fused_head(hd, Wd, y.to(DEV), T, Post(post[0], post[1], True) if post else Post(), idx=idx, count=count,
                     labels_via_idx=True, scatter=True)
    (out[:, 0] * g.to(DEV)).sum().backward()
    torch.cuda.synchronize()
    at = scored.nonzero()[:, 0]
    a, w = h[at].double().requires_grad_(True), W.double().requires_grad_(True)
    z = a @ w.T
    if post:
        z = post[1] * torch.tanh(post[0] * z)
    lp = torch.log_softmax(z / T, 1)
    col = lp.gather(1, y[at][:, None])[:, 0]
    (col * g[at].double()).sum().backward()
    ent = -(lp.exp() * lp).sum(1)
    size = (h[at].double().norm(dim=1) * W.double().norm(dim=1).max()).max().item() / T if spread == 0 else \
        (h[at].double().abs() @ W.double().abs().T).max().item() / T * 0.2
    o = out.detach().cpu().double()
    assert (o[at, 0] - col.detach()).abs().max() <= EPS * (size + 20)
    assert (o[at, 1] - ent.detach()).abs().max() <= EPS * (size + 20)
    assert (o[~scored] == 0).all() and (hd.grad[~scored.to(DEV)] == 0).all()

    def rel(x, ref, scale):  # columns of very different size: each on its own scale
        return ((x.double() - ref) * scale).norm() / (ref * scale).norm()

    sh = 1 / a.grad.norm(dim=0).clamp(min=1e-300) if spread else torch.ones(d, dtype=torch.float64)
    sw = 1 / w.grad.norm(dim=0).clamp(min=1e-300) if spread else torch.ones(d, dtype=torch.float64)
    # dz carries the logits' error (EPS x size, relative) and the gradients' own sums theirs
    assert rel(hd.grad.cpu()[at], a.grad, sh) <= EPS * (size + 20)
    assert rel(Wd.grad.cpu(), w.grad, sw) <= EPS * (size + 20)


def test_fp32_operands_split_exactly():
    """Powers of two, values with all 24 bits set and values next to them: a product with the identity returns W's
    own entries as logits, bit for bit, so every part of every value arrived."""
    d = 64
    g = torch.Generator().manual_seed(9)
    W = torch.randn(300, d, generator=g) * 2.0 ** torch.randint(-30, 30, (300, d), generator=g).float()
    W.view(torch.int32)[:100] |= 0x00000fff
    W[100:110] = 2.0 ** torch.arange(10.0)[:, None]
    h = torch.eye(d)
    # a row's logprob and entropy at V = 1 are 0 and its row state is the logit in base 2
    for v in (0, 5, 57, 101, 299):
        _, lse = head_op.head_fwd(h.to(DEV), W[v:v + 1].to(DEV), None, torch.zeros(d, dtype=torch.int64, device=DEV), None,
                                  None, 1.0, 1.0, 1.0, False, False, False)
        assert torch.equal(lse[:, 0].cpu(), W[v] * torch.tensor(1.4426950408889634))
