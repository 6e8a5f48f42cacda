"""octo_columns_fwd / octo_columns_bwd over the forms their 16-byte loads distinguish: rows that start on a 16-byte
boundary or off it (odd V, a view into a wider or shifted buffer), vocabularies shorter than a chunk, around one
workgroup's sweep and past it, the gradient's rows aligned as the logits' or not, few rows (1,024 threads each) and
many (256); and the values an online softmax can get wrong: -inf logits ahead of the first finite one, a maximum that
only the last value raises, logits far from zero.

Against fp64 (oracle/head.py columns): logprob and entropy within 2^-22 of the logits' spread (their sums are fp32,
V of them grouped by thread), the gradient within half its type's spacing (2^-8 and 2^-11 of the value) or, in fp32, 1e-6."""

import ctypes

import pytest
import torch

from octopus_amd import _lib, head_op
from oracle import head as ohead

pytestmark = pytest.mark.gpu
DEV = "cuda"
CODE = {torch.bfloat16: _lib.BF16, torch.float16: _lib.F16, torch.float32: _lib.F32}
P = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731


def _reference(x, y, T):
    z = x.double() / T
    lp = z - torch.logsumexp(z, 1, keepdim=True)
    p = lp.exp()
    ent = -(p * lp).sum(1)
    return lp.gather(1, y[:, None])[:, 0], ent, p


@pytest.mark.parametrize("dtype", list(CODE), ids=["bf16", "f16", "f32"])
@pytest.mark.parametrize("n,V,shift,gap,dshift", [
    (3, 1, 0, 0, 0), (2, 5, 3, 2, 0), (3, 8, 0, 0, 0), (5, 2047, 0, 0, 0), (4, 8193, 1, 0, 1), (3, 8192, 0, 8, 0),
    (2, 50257, 0, 0, 0), (600, 3001, 0, 7, 4), (513, 4096, 8, 8, 8),
], ids=str)
def test_columns_at_every_alignment(n, V, shift, gap, dshift, dtype):
    """shift, gap: the logits' first element and row stride past V in their buffer; dshift: the gradient's."""
    gen = torch.Generator().manual_seed(V + shift)
    T, ld = 0.7, V + gap
    buf = torch.randn(shift + n * ld, generator=gen) * 4
    buf[shift + V - 1::ld] += 30  # the last value of each row raises the maximum
    buf = buf.to(dtype).to(DEV)
    x = buf[shift:].view(n, ld)[:, :V]
    y = torch.randint(0, V, (n,), generator=gen)
    g = torch.randn(n, generator=gen)
    yd, gd = y.to(DEV), g.to(DEV)
    out, lse = torch.full((n, 2), float("nan"), device=DEV), torch.empty(n, 2, device=DEV)
    dbuf = torch.full((dshift + n * ld,), 7.0, dtype=dtype, device=DEV)
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    _lib.call("octo_columns_fwd", P(x), ld, CODE[dtype], P(yd), n, V, 1 / T, P(out), P(lse), st)
    dx = dbuf[dshift:].view(n, ld)
    _lib.call("octo_columns_bwd", P(x), ld, CODE[dtype], P(yd), n, V, 1 / T, P(lse), P(gd), P(dx), ld, st)
    torch.cuda.synchronize()
    lp, ent, p = _reference(x.cpu(), y, T)
    spread = 2.0 ** -22 * (x.float().abs().max().item() / T + 20)
    assert (out[:, 0].cpu().double() - lp).abs().max() <= spread
    assert (out[:, 1].cpu().double() - ent).abs().max() <= spread
    ref = -p * g.double()[:, None] / T
    ref.scatter_add_(1, y[:, None], g.double()[:, None] / T)
    d = dx[:, :V].cpu().double()
    # half a spacing, relative to the value: at most 2^-8 with bf16's 8 significand bits, 2^-11 with f16's 11
    half = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 0.0}[dtype]
    tiny = 2.0 ** -25 if dtype == torch.float16 else 0.0  # f16's subnormals
    assert ((d - ref).abs() <= (half + 1e-5) * ref.abs() + 1e-6 * g.double().abs()[:, None] / T + tiny).all()
    assert (dx[:, V:] == 7.0).all() and (dbuf[:dshift] == 7.0).all()  # nothing outside the rows


@pytest.mark.parametrize("dtype", list(CODE), ids=["bf16", "f16", "f32"])
def test_columns_of_masked_and_far_logits(dtype):
    """Logits of -inf (masked entries) at the head of the row, over a whole thread's share, and at the label: finite
    logprobs elsewhere, -inf at a masked label, an entropy of NaN (0 x -inf, as the composite gives); a row of -inf
    alone is NaN; a row far from zero keeps its differences."""
    n, V = 4, 20011
    x = torch.randn(n, V, generator=torch.Generator().manual_seed(5))
    x[0, :20000] = -float("inf")
    x[1, 7] = -float("inf")
    x[2] = -float("inf")
    x[3] -= 1000.0
    x = x.to(dtype)
    y = torch.tensor([20005, 7, 3, 11])
    out = head_op.head_columns(x.to(DEV), 1.0, y.to(DEV)).cpu().double()
    lp, ent, _ = _reference(x, y, 1.0)
    assert abs(out[0, 0] - lp[0]) <= 1e-5 and out[1, 0] == -float("inf") and torch.isnan(out[2]).all()
    assert torch.isnan(out[:2, 1]).all() and torch.isnan(ent[:2]).all()
    assert abs(out[3, 0] - lp[3]) <= 2e-3 and abs(out[3, 1] - ent[3]) <= 2e-3  # 1,000 x 2^-24 x a few
    lp2, ent2 = ohead.columns(x[3:], 1.0, y[3:])[:2]
    assert torch.allclose(lp2, lp[3:]) and torch.allclose(ent2, ent[3:])
