"""The gradient GEMMs' stores: whole-width 16-bit tiles go through the LDS in 512-byte rows, everything else value by
value (a ragged last tile of d, an output whose rows or base do not sit on 16 bytes, an accumulating output). The same
sums rounded once, so every form must give the same bits; and nothing is written outside the rows and columns."""

import ctypes

import pytest
import torch

from octopus_amd import _lib, head_op

pytestmark = pytest.mark.gpu
DEV = "cuda"
CODE = {torch.bfloat16: _lib.BF16, torch.float16: _lib.F16}
P = lambda t: None if t is None else ctypes.c_void_p(t.data_ptr())  # noqa: E731


@pytest.mark.parametrize("dtype", list(CODE), ids=["bf16", "f16"])
@pytest.mark.parametrize("n,d,V", [(1, 256, 256), (255, 512, 300), (257, 264, 1024), (300, 776, 1000)], ids=str)
def test_stores_of_every_alignment_agree(n, d, V, dtype):
    gen = torch.Generator().manual_seed(n + d)
    h = torch.randn(n, d, generator=gen).to(dtype).to(DEV)
    W = (torch.randn(V, d, generator=gen) * 0.05).to(dtype).to(DEV)
    y = torch.randint(0, V, (n,), generator=gen).to(DEV)
    g = torch.randn(n, generator=gen).to(DEV)
    code, st = CODE[dtype], ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    _, lse = head_op.head_fwd(h, W, None, y, None, None, 1.0, 1.0, 1.0, False, False, False)
    ws = torch.empty(_lib.workspace_bytes(n, d, V, code, _lib.WS_BACKWARD), dtype=torch.uint8, device=DEV)

    def run(ld, shift, accumulate):
        """grad_h in rows of ld values from `shift` values into its buffer, grad_W [V, d] from shift on."""
        gh = torch.full((shift + n * ld + 64,), 3.0, dtype=dtype, device=DEV)
        gw = torch.full((shift + V * d + 64,), 0.0 if accumulate else 3.0, dtype=dtype, device=DEV)
        flags = _lib.LSE_PAIR | (_lib.GRADW_ACCUMULATE if accumulate else 0)
        _lib.call("octo_head_bwd", P(h), n, d, code, P(W), d, code, None, P(y), None, None, n, d, V, flags, 1.0, 1.0,
                  1.0, 0, P(lse), P(g), P(gh[shift:]), ld, code, P(gw[shift:]), code, P(ws), ws.numel(), st)
        torch.cuda.synchronize()
        rows = gh[shift:shift + n * ld].view(n, ld)
        assert (rows[:, d:] == 3.0).all() and (gh[:shift] == 3.0).all() and (gh[shift + n * ld:] == 3.0).all()
        end = gw[shift + V * d:]
        assert (end == end[0]).all() and (gw[:shift] == end[0]).all()
        return rows[:, :d].clone(), gw[shift:shift + V * d].view(V, d).clone()

    gh, gw = run(d, 0, False)
    assert torch.isfinite(gh).all() and torch.isfinite(gw).all() and gh.abs().sum() > 0
    for form in ((d + 3, 0, False), (d + 8, 1, False), (d, 4, True)):
        a, b = run(*form)
        assert torch.equal(a, gh) and torch.equal(b, gw), form
