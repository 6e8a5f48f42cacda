"""grad_h's split K (csrc/tile_order.h k_splits): with few tiles, each tile's vocabulary is cut into runs whose fp32
partial tiles a kernel sums. A workspace one byte short of the queried size has no room for the partial tiles and runs
the unsplit product, so the two must agree to fp32 summation order: both sum V products per element in fp32, in
another order, within 2^-24 sqrt(V) < 1e-4 of the sum's terms, and in fp32 outputs nothing else differs. Row counts at
the edges of 1 to 3 M-tiles, through the row map with a device count below the row bound; widths with a ragged last
tile; V read K-major as stored and through W^T; both routes (the backward, and the step with and without grad_W)."""

import ctypes

import pytest
import torch

from octopus_amd import _lib, head_op
from oracle import head as ohead

pytestmark = pytest.mark.gpu
DEV = "cuda"
CODE = {torch.bfloat16: _lib.BF16, torch.float16: _lib.F16}
P = lambda t: None if t is None else ctypes.c_void_p(t.data_ptr())  # noqa: E731


def _rel(a, b):
    return ((a.double() - b.double()).norm() / b.double().norm()).item()


@pytest.mark.parametrize("route", ["bwd", "step", "step_grad_h"])
@pytest.mark.parametrize("n,d,V,dtype", [
    (1, 64, 8192, torch.bfloat16), (255, 264, 5120, torch.bfloat16), (257, 256, 6400, torch.float16),
    (513, 520, 5001, torch.bfloat16), (300, 512, 12800, torch.bfloat16),
    (2945, 2560, 2048, torch.bfloat16),  # 120 tiles: two runs beside grad_W too
], ids=str)
def test_runs_sum_to_the_unsplit_product(route, n, d, V, dtype):
    gen = torch.Generator().manual_seed(n + V)
    N = n + n // 2 + 3  # packed rows, n of them scored
    h = torch.randn(N, d, generator=gen).to(dtype)
    W = (torch.randn(V, d, generator=gen) * 0.05).to(dtype)
    y = torch.randint(0, V, (N,), generator=gen)
    scored = torch.zeros(N, dtype=torch.bool)
    scored[torch.randperm(N, generator=gen)[:n]] = True
    at = scored.nonzero()[:, 0]
    hd, Wd, yd, T = h.to(DEV), W.to(DEV), y.to(DEV), 0.9
    idx, count = head_op.compact_rows(scored.to(DEV))
    adv, mask = torch.randn(N, generator=gen).to(DEV), scored.float().to(DEV)
    code, st = CODE[dtype], ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    flags = _lib.ROWS_VIA_IDX | _lib.LSE_PAIR
    ws_flags = {"bwd": _lib.WS_BACKWARD, "step": _lib.WS_STEP, "step_grad_h": _lib.WS_STEP | _lib.WS_NO_GRADW}[route]
    room = _lib.workspace_bytes(N, d, V, code, ws_flags)
    runs = []
    for wsb in (room, room - 1):
        ws = torch.full((wsb,), 0xFF, dtype=torch.uint8, device=DEV)  # NaN: a partial tile not written shows
        gh = torch.full((N, d + 3), 7.0, device=DEV)
        gw = None if route == "step_grad_h" else torch.empty(V, d, device=DEV)
        lse, g, loss = torch.zeros(N, 2, device=DEV), torch.zeros(N, device=DEV), torch.zeros((), device=DEV)
        common = (P(hd), N, d, code, P(Wd), d, code, None, P(yd), P(idx), P(count), N, d, V, flags, 1.0 / T, 1.0, 1.0,
                  0)
        tail = _lib.GrpoTail(None, None, P(adv), P(mask), N, 0.2, 0.28, 5.0, P(g), P(loss))
        if route == "bwd":
            fws = torch.empty(_lib.workspace_bytes(N, d, V, code, 0), dtype=torch.uint8, device=DEV)
            _lib.call("octo_head_fwd_grpo", *common, None, None, P(lse), None, 2, ctypes.byref(tail), P(fws),
                      fws.numel(), st)
            _lib.call("octo_head_bwd", *common, P(lse), P(g), P(gh), d + 3, _lib.F32, P(gw), _lib.F32, P(ws), wsb, st)
        else:
            _lib.call("octo_head_step_grpo", *common, None, None, P(lse), None, 2, ctypes.byref(tail), P(gh), d + 3,
                      _lib.F32, P(gw), _lib.F32, P(ws), wsb, st)
        torch.cuda.synchronize()
        assert (gh[n:] == 7.0).all() and (gh[:, d:] == 7.0).all()  # rows past the count and the stride's gap untouched
        runs.append((gh[:n, :d].cpu(), g[:n].cpu()))
    (split, g_ref), (whole, _) = runs
    assert _rel(split, whole) <= 1e-4
    ref, _ = ohead.head_backward(h[at], W, y[at], T, g_ref, want_w=False)
    assert _rel(split, ref) <= 1e-2

