"""fp32 operands outside the range the three bf16 parts hold: infinite weights, and finite ones above bf16's largest.
What 64-bit sums of the same products give, infinities and NaN in the same places."""
import pytest
import torch

from octopus_amd import head_op

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _inputs(n, d, V, what):
    g = torch.Generator(device=DEV).manual_seed(n + V)
    h = torch.randn(n, d, generator=g, device=DEV)
    W = torch.randn(V, d, generator=g, device=DEV) * 0.05
    y = torch.randint(0, V - 1, (n,), generator=g, device=DEV)
    if what == "inf":  # logits of -inf for some rows (a finite logprob), +inf for others (NaN)
        W[V - 1, 3], W[V - 1, d - 1] = float("inf"), float("-inf")
        h[:, d - 1] = h[:, d - 1].abs()
    elif what == "-inf":  # -inf for every row
        W[V - 1, 3] = float("-inf")
        h[:, 3] = h[:, 3].abs()
    else:  # products of ordinary size, of a weight that bf16 rounds to infinity
        W[V - 1, 3] = 3.4e38
        h[:, 3] = torch.sign(h[:, 3]) * torch.empty(n, device=DEV).uniform_(0.5, 1.5, generator=g) * 2e-37
    return h, W, y


def _exact(h, W, y, g):
    h, W = h.double().cpu(), W.double().cpu()
    y, g = y.cpu(), g.double().cpu()
    z = h @ W.T
    lp = z - torch.logsumexp(z, 1, keepdim=True)
    p = lp.exp()
    dz = -p * g[:, None]
    dz.scatter_add_(1, y[:, None], g[:, None])
    return lp.gather(1, y[:, None])[:, 0], dz @ W, dz.T @ h


def _like(a, want, tol):
    a, want = a.double().cpu(), want.float().double()
    assert torch.equal(torch.isnan(a), torch.isnan(want)) and torch.equal(torch.isinf(a), torch.isinf(want))
    ok = torch.isfinite(want)
    assert ok.any() and ((a - want)[ok].norm() / want[ok].norm()).item() <= tol


# one tile and several, d and V off the tiles; 1.5e-5: 32-bit sums, as the in-range ones
@pytest.mark.parametrize("n,d,V", [(70, 64, 640), (300, 132, 1003)])
@pytest.mark.parametrize("what", ["inf", "-inf", "large"])
def test_operands_out_of_bf16_range(n, d, V, what):
    h, W, y = _inputs(n, d, V, what)
    coef = torch.randn(n, generator=torch.Generator(device=DEV).manual_seed(1), device=DEV)
    want = _exact(h, W, y, coef)
    hd, Wd = h.clone().requires_grad_(True), W.clone().requires_grad_(True)
    out = head_op.fused_head(hd, Wd, y, 1.0)
    _like(out[:, 0].detach(), want[0], 1.5e-5)
    if what == "inf":
        return  # NaN rows: every gradient of W is NaN
    (coef * out[:, 0]).sum().backward()
    _like(hd.grad, want[1], 1.5e-5)
    _like(Wd.grad, want[2], 1.5e-5)
