"""Which calls keep a buffer between forward and backward, and its size (host planning only)."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.fx.experimental.symbolic_shapes import DimDynamic, ShapeEnv, StatelessSymbolicContext
from torch.utils.checkpoint import checkpoint

from octopus_amd import _lib, head_op


@pytest.mark.parametrize("n,d,V,rows", [
    (1, 256, 640, 256), (300, 136, 1000, 256), (300, 512, 5003, 512),
    (5119, 2560, 151936, 2560),  # as many as the width
    (8192, 4096, 128256, 4096), (8192, 4096, 151936, 3328),  # 2 GiB
    (8192, 4096, 3 << 20, 0),  # not one tile of rows
])
def test_rows_whose_logits_are_kept(n, d, V, rows):
    assert head_op._kept_rows(n, d, V) == rows
    assert rows * head_op._pad256(V) * 4 <= head_op._KEEP_BYTES


def test_what_is_left_for_later():
    assert _lib.later_bytes(300, 512, 5003, _lib.FP8E4M3, True) == _lib.later_bytes(300, 512, 5003, _lib.F32, True) == 0
    assert _lib.later_bytes(0, 512, 5003, _lib.BF16, True) == 0
    assert _lib.later_bytes(32768, 2560, 151936, _lib.BF16, True) == 0  # several passes
    for n in (1, 257, 1536):
        P = -(-n // 256) * 256
        plain = _lib.later_bytes(n, 2560, 151936, _lib.BF16, False)
        assert plain >= P * (-(-151936 // 256) * 256) * 2 + 2560 * P * 2  # dz and h^T
        assert 0 <= _lib.later_bytes(n, 2560, 151936, _lib.BF16, True) - plain <= 256 * 256 * 256 * 4  # one round of runs


def _operands(n=512, d=1024, V=33024, weight_grad=True):
    """Operands without storage, of a size that keeps logits (under FakeTensorMode)."""
    return (torch.empty(n, d, dtype=torch.bfloat16, device="cuda", requires_grad=True),
            torch.empty(V, d, dtype=torch.bfloat16, device="cuda", requires_grad=weight_grad),
            torch.zeros(n, dtype=torch.int64, device="cuda"))


def _kept(out):
    return "head_fwd_logits" in type(out.grad_fn).__name__


def test_a_frozen_weight_keeps_no_logits():
    with FakeTensorMode():
        assert _kept(head_op.fused_head(*_operands(), 1.0))
        assert not _kept(head_op.fused_head(*_operands(weight_grad=False), 1.0))


def test_checkpointed_and_offloaded_calls_keep_no_logits():
    """What such a caller's hooks do not reach would stay on the device, once per checkpointed chunk."""
    with FakeTensorMode():
        rows, weight, y = _operands()
        routes = []

        def head(h):
            out = head_op.fused_head(h, weight, y, 1.0)
            routes.append(_kept(out))
            return out

        checkpoint(head, rows, use_reentrant=False)
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t):
            head(rows)
        head(rows)
        assert routes == [False, False, True]


def test_live_logits_of_a_device_share_one_bound(monkeypatch):
    with FakeTensorMode():
        rows, weight, y = _operands()
        monkeypatch.setattr(head_op, "_KEEP_BYTES", 512 * 33024 * 4)
        first, second = (head_op.fused_head(rows, weight, y, 1.0) for _ in range(2))
        assert _kept(first) and not _kept(second)
        del first
        again = head_op.fused_head(rows, weight, y, 1.0)
        assert _kept(again)
        del again
        assert head_op._Room._taken[rows.device] == 0


def test_out_of_memory_recomputes(monkeypatch):
    def full(*_):
        raise torch.OutOfMemoryError("full")

    with FakeTensorMode():
        operands = _operands()
        with monkeypatch.context() as m:
            m.setattr(head_op, "head_fwd_logits", full)
            assert not _kept(head_op.fused_head(*operands, 1.0))
        assert head_op._Room._taken[operands[0].device] == 0
        assert _kept(head_op.fused_head(*operands, 1.0))


@pytest.mark.parametrize("n,d,V,least", [
    (64, 4096, 50257, 1), (300, 4096, 50257, 1), (1536, 1024, 50257, 1), (1351, 2304, 64000, 1),
    (225, 2560, 151936, 1), (1536, 2560, 151936, 1),
    (57, 1024, 65536, 768), (768, 1024, 65536, 768), (768, 1024, 32768, 1536),  # short calls, which the host paces
])
def test_a_step_keeps_no_more_than_the_gradient_it_would_hold(n, d, V, least):
    """dz and h^T alone, whatever else the step works in (W^T where V % 64 or d % 256)."""
    P, Vp = -(-n // 256) * 256, -(-V // 256) * 256
    with FakeTensorMode():
        rows, weight, _ = _operands(n, d, V)
        kept = head_op._later_bytes(rows, weight, None, True, True)
    assert kept <= V * d * 2
    assert kept == (P * Vp * 2 + d * P * 2 if P * (Vp + d) <= V * d and n >= least else 0)


def test_symbolic_sizes_take_the_routes_that_serve_any():
    """A call traced with symbols for its sizes (make_fx, export) neither fixes them nor picks a route by them."""
    env = ShapeEnv()
    mode = FakeTensorMode(shape_env=env)
    dynamic = StatelessSymbolicContext(dynamic_sizes=[DimDynamic.DYNAMIC, DimDynamic.STATIC])
    with FakeTensorMode() as plain:
        rows, weight, y = _operands(V=151936)
    assert head_op._keeps(rows, weight, None) and head_op._later_bytes(rows, weight, None, True, True)
    rows, weight = (mode.from_tensor(torch.empty(t.shape, dtype=t.dtype, device="meta"), symbolic_context=dynamic)
                    for t in (rows, weight))
    with mode:
        rows, weight = (torch.empty(t.shape, dtype=t.dtype, device="cuda", requires_grad=True) for t in (rows, weight))
        assert not isinstance(rows.shape[0], int)
        assert head_op._keeps(rows, weight, None) == head_op._later_bytes(rows, weight, None, True, True) == 0
    assert not env.guards
