"""fused_head with its logits kept for the backward (octo_head_fwd_logits, octo_head_bwd_logits): gradients against 64
bits and against the recomputing route, at the edges of what takes this route."""
import pytest
import torch

from octopus_amd import head_op

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _case(n, d, V, scored, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    W = (torch.randn(V, d, generator=g, device=DEV) * 0.05).bfloat16()
    h = torch.randn(n, d, generator=g, device=DEV).bfloat16()
    y = torch.randint(0, V, (n,), generator=g, device=DEV)
    coef = torch.randn(n, generator=g, device=DEV)
    mask = torch.rand(n, generator=g, device=DEV) < scored
    mask[0] = True
    return h, W, y, coef, mask


def _run(case, T, post, need, monkeypatch, staged, times=1):
    h, W, y, coef, mask = case
    monkeypatch.setattr(head_op, "_STAGE_WORK", 0 if staged else 1 << 62)
    hd, Wd = h.clone().requires_grad_(need[0]), W.clone().requires_grad_(need[1])
    kw = {}
    if not bool(mask.all()):
        idx, count = head_op.compact_rows(mask)
        kw = dict(idx=idx, count=count, labels_via_idx=True, scatter=True)
    out = head_op.fused_head(hd, Wd, y, T, post, **kw)
    loss = (coef * out[:, 0]).sum()
    for k in range(times):
        hd.grad = Wd.grad = None
        loss.backward(retain_graph=k + 1 < times)
    return out.detach(), hd.grad, Wd.grad


def _exact(case, T, post):
    h, W, y, coef, mask = case
    hd, Wd = h.double().requires_grad_(True), W.double().requires_grad_(True)
    z = hd @ Wd.T
    z = (post.post * torch.tanh(post.pre * z) if post.tanh else post.post * post.pre * z) / T
    lp = torch.log_softmax(z, 1)
    col = lp.gather(1, y[:, None])[:, 0] * mask
    (coef * col).sum().backward()
    return col.detach(), hd.grad, Wd.grad


def _rel(a, b):
    return ((a.double() - b).norm() / b.norm().clamp(min=1e-30)).item()


# one row; a ragged row count; whole tiles; widths and vocabularies that grad_h reads through W^T (d % 256, V % 64); a
# temperature at which most rows' exponentials are rescaled; the softcap; one gradient alone
@pytest.mark.parametrize("n,d,V,scored,T,cap,need", [
    (1, 256, 640, 1.0, 1.0, False, (True, True)),
    (300, 512, 5003, 0.7, 0.7, False, (True, True)),
    (257, 136, 1000, 0.5, 1.0, False, (True, True)),
    (700, 512, 2048, 0.8, 0.012, False, (True, True)),
    (512, 256, 2048, 0.8, 1.0, False, (True, True)),
    (333, 256, 1500, 0.9, 1.0, True, (True, True)),
    (300, 512, 3000, 0.7, 1.0, False, (True, False)),
    (300, 512, 3000, 0.7, 1.0, False, (False, True)),
])
def test_staged_gradients(n, d, V, scored, T, cap, need, monkeypatch):
    post = head_op.Post(1 / 30.0, 30.0, True) if cap else head_op.Post()
    case = _case(n, d, V, scored, n + V)
    got = _run(case, T, post, need, monkeypatch, True)
    old = _run(case, T, post, need, monkeypatch, False)
    want = _exact(case, T, post)
    assert (got[0] - old[0]).abs().max() <= 1e-5 * old[0].abs().max()  # fp32 sums of one order or another
    assert (got[0][:, 0].double() - want[0]).abs().max() <= 2e-5 * max(1.0, want[0].abs().max().item())
    for a, b, w, on in zip(got[1:], old[1:], want[1:], need):
        assert (a is not None) == on
        if on:
            # dz and the result rounded to bf16 (2^-9 each, 2^-9 sqrt(2) / sqrt(3) rms), no worse than recomputed
            assert _rel(a, w) <= 5e-3 and _rel(a, w) <= 1.1 * _rel(b, w) + 1e-4


def test_staged_backward_repeats_and_lets_go(monkeypatch):
    """A retained graph gives the same gradients again; after the last backward nothing holds the buffer."""
    case = _case(300, 512, 5003, 0.7, 3)
    once = _run(case, 0.1, head_op.Post(), (True, True), monkeypatch, True)
    again = _run(case, 0.1, head_op.Post(), (True, True), monkeypatch, True, times=3)
    assert torch.equal(once[1], again[1]) and torch.equal(once[2], again[2])
    h, W, y, coef, _ = case
    hd, Wd = h.clone().requires_grad_(True), W.clone().requires_grad_(True)
    before = torch.cuda.memory_allocated()
    out = head_op.fused_head(hd, Wd, y, 1.0)
    held = torch.cuda.memory_allocated() - before
    assert held >= 512 * 5120 * 2
    (coef * out[:, 0]).sum().backward()
    hd.grad = Wd.grad = None
    assert torch.cuda.memory_allocated() - before < 512 * 5120  # out alone is still here
