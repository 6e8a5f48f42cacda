"""grad_W's fp32 partials over several row passes, with and without a device row count, and head_columns' logprobs close to 0."""
import math

import pytest
import torch

from octopus_amd import _lib, head_op

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _passes_workspace(n, d, V):
    """A workspace in which the step runs three passes or more."""
    full = _lib.workspace_bytes(n, d, V, _lib.BF16, _lib.WS_STEP)
    for b in range(full, 0, -(full // 64)):
        try:
            passes = _lib.bwd_plan(n, d, V, _lib.BF16, _lib.WS_STEP, b)[1]
        except ValueError:
            break
        if passes >= 3:
            return b
    raise AssertionError("no plan of three passes")


# whole tiles (blocked partials) and widths past them (row-major ones); row counts that end inside a tile
@pytest.mark.parametrize("n,d,V", [(1030, 256, 5003), (2048, 512, 1024), (1500, 328, 2050), (1900, 136, 1000)])
@pytest.mark.parametrize("counted", [False, True])
def test_gradients_over_several_passes(n, d, V, counted, monkeypatch):
    g = torch.Generator(device=DEV).manual_seed(n)
    h = torch.randn(n, d, generator=g, device=DEV).bfloat16()
    W = (torch.randn(V, d, generator=g, device=DEV) * 0.05).bfloat16()
    y = torch.randint(0, V, (n,), generator=g, device=DEV)
    adv = torch.randn(n, generator=g, device=DEV)
    mask = torch.ones(n, device=DEV)
    kw = {}
    if counted:
        idx, count = head_op.compact_rows(mask.bool())
        kw = dict(idx=idx, count=count, labels_via_idx=True, scatter=True)
    got = {}
    for name in ("one", "several"):
        ws = _passes_workspace(n, d, V) if name == "several" else None
        monkeypatch.setattr(head_op, "STEP_WORKSPACE_BYTES", ws)
        hd, Wd = h.clone().requires_grad_(True), W.clone().requires_grad_(True)
        loss, _ = head_op.fused_grpo_head(hd, Wd, y, 1.0, adv, mask, **kw)
        loss.backward()
        got[name] = (hd.grad, Wd.grad)
    for a, b in zip(got["one"], got["several"]):
        # the same dz, its products summed in fp32 in another order, rounded to bf16: a value in 2^8 or so falls to its
        # other neighbour, 2^-8 away
        assert ((a.float() - b.float()).norm() / a.float().norm()).item() <= 2.0 ** -8 / 4


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_columns_close_to_zero(dtype):
    """head_columns of logits of 14 .. 18 over 32,000 others: logprobs of -5e-2 .. -8e-4."""
    n, V = 64, 32000
    g = torch.Generator(device=DEV).manual_seed(1)
    y = torch.randint(0, V, (n,), generator=g, device=DEV)
    zl = torch.randn(n, V, generator=g, device=DEV).scatter_(1, y[:, None], torch.linspace(14, 18, n, device=DEV)[:, None]).to(dtype)
    want = zl.double().gather(1, y[:, None])[:, 0] - torch.logsumexp(zl.double(), 1)
    got = head_op.head_columns(zl, 1.0, y)[:, 0].double()
    # the label's own logit among the sums: what is left is the sum's rounding, 1.05 in 24 merges (wave and workgroup)
    # of at most 2^-24 each, and the label's thread, whose 125 terms are each rounded against 1
    assert (got - want).abs().max() <= (24 + math.sqrt(125)) * 2.0 ** -24
