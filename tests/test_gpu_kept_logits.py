"""fused_head with logits kept for the backward (octo_head_fwd_logits, octo_head_bwd_logits): to the bit what the
recomputing backward gives, over what both take."""
import threading

import pytest
import torch

from octopus_amd import _lib, head_op
from tests.test_gpu_poisoned import _bwd_ws, poisoned

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _both(n, d, V, scored, T, cap, monkeypatch, need=(True, True), rows=None, ws=None, bad_labels=False):
    """(columns, grad_rows, grad_weight) with logits kept (of `rows` rows at most) and without; ws: the backward's
    workspace."""
    g = torch.Generator(device=DEV).manual_seed(n + V)
    W = (torch.randn(V, d, generator=g, device=DEV) * 0.05).bfloat16()
    h = torch.randn(n, d, generator=g, device=DEV).bfloat16()
    y = torch.randint(0, V, (n,), generator=g, device=DEV)
    if bad_labels:
        y[::3] = -100
        y[1::7] = V
    coef = torch.randn(n, generator=g, device=DEV)
    mask = torch.rand(n, generator=g, device=DEV) < scored
    kw = {}
    if scored < 1:
        idx, count = head_op.compact_rows(mask)
        kw = dict(idx=idx, count=count, labels_via_idx=True, scatter=True)
    post = head_op.Post(1 / 30.0, 30.0, True) if cap else head_op.Post()
    if rows is not None:
        monkeypatch.setattr(head_op, "_KEEP_BYTES", rows * head_op._pad256(V) * 4)
    got = []
    for least in (0, 1 << 62):
        monkeypatch.setattr(head_op, "_STAGE_WORK", least)
        hd, Wd = h.clone().requires_grad_(need[0]), W.clone().requires_grad_(need[1])
        assert bool(head_op._keeps(hd, Wd, kw.get("idx"))) == (least == 0 and n <= 2 * d and need[1])
        out = head_op.fused_head(hd, Wd, y, T, post, **kw)
        with monkeypatch.context() as m:
            if ws is not None:
                m.setattr(head_op, "BWD_WORKSPACE_BYTES", ws)
            (coef * out[:, 0])[~torch.isnan(out[:, 0])].sum().backward()
        got.append((out.detach(), hd.grad, Wd.grad))
    return got


# one row; ragged rows; widths and vocabularies read through W^T (d % 256, V % 64); no scored row; the softcap; a
# temperature at which most probabilities are far below 2^-25 of the row's largest; labels outside the vocabulary
@pytest.mark.parametrize("n,d,V,scored,T,cap,bad", [
    (1, 256, 640, 1.0, 1.0, False, False),
    (300, 512, 5003, 0.7, 0.7, False, True),
    (257, 136, 1000, 0.5, 1.0, False, False),
    (300, 512, 3000, 0.0, 1.0, False, False),
    (333, 256, 1500, 0.9, 1.0, True, True),
    (700, 512, 2048, 0.8, 0.012, False, False),
])
def test_as_recomputed(n, d, V, scored, T, cap, bad, monkeypatch):
    a, b = _both(n, d, V, scored, T, cap, monkeypatch, bad_labels=bad)
    assert all(torch.equal(torch.nan_to_num(x), torch.nan_to_num(y)) for x, y in zip(a, b))


# fewer rows kept than there are, the count below and above them; vocabulary chunks and several row passes
@pytest.mark.parametrize("n,scored,rows,ws", [
    (900, 0.9, 256, None), (900, 0.2, 256, None), (900, 1.0, 512, 8 << 20), (700, 1.0, 256, 3 << 20),
])
@pytest.mark.parametrize("cap", [False, True])
def test_some_rows_kept(n, scored, rows, ws, cap, monkeypatch):
    a, b = _both(n, 512, 2500, scored, 0.7, cap, monkeypatch, rows=rows, ws=ws)
    assert all(torch.equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("scored", [1.0, 0.6, 0.1])
def test_several_passes_of_one_chunk(scored, monkeypatch):
    """Both gradients in one launch per pass, grad_W's sum over the passes in fp32, the last one the count decides; the
    kept rows end within the second pass."""
    ws = _bwd_ws(4000, 2048, 192, _lib.BF16, 0, lambda plan: plan[1] == 2 and plan[3] == 1)
    a, b = _both(4000, 2048, 192, scored, 0.7, False, monkeypatch, rows=2560, ws=ws)
    assert all(torch.equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("need", [(True, False), (False, True)])
def test_one_gradient(need, monkeypatch):
    a, b = _both(300, 512, 3000, 0.7, 1.0, False, monkeypatch, need=need)
    assert all((x is None and y is None) or torch.equal(x, y) for x, y in zip(a, b))


def test_out_of_memory_in_the_backward(monkeypatch):
    """The backward lets the logits go and recomputes."""
    want = _both(300, 512, 3000, 0.7, 1.0, False, monkeypatch)[1]
    bwd = head_op.head_bwd

    def full(*args):
        if len(args) == 16 and args[15] is not None:
            raise torch.OutOfMemoryError("full")
        return bwd(*args)

    monkeypatch.setattr(head_op, "head_bwd", full)
    got = _both(300, 512, 3000, 0.7, 1.0, False, monkeypatch)[0]
    assert all(torch.equal(x, y) for x, y in zip(got, want))


def test_a_weight_changed_in_place(monkeypatch):
    """The backward reads the weight as it is then, as the recomputing one does."""
    g = torch.Generator(device=DEV).manual_seed(5)
    W = (torch.randn(3000, 512, generator=g, device=DEV) * 0.05).bfloat16()
    h = torch.randn(300, 512, generator=g, device=DEV).bfloat16()
    y = torch.randint(0, 3000, (300,), generator=g, device=DEV)
    got = []
    for least in (0, 1 << 62):
        monkeypatch.setattr(head_op, "_STAGE_WORK", least)
        hd, Wd = h.clone().requires_grad_(True), W.clone().requires_grad_(True)
        out = head_op.fused_head(hd, Wd, y, 1.0)
        with torch.no_grad():
            Wd.mul_(0.875)
        out[:, 0].sum().backward()
        got.append((hd.grad, Wd.grad))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


@pytest.mark.parametrize("n,d,V,scored,rows", [(300, 512, 5003, 0.7, None), (900, 512, 2500, 0.9, 256),
                                               (900, 512, 2500, 0.2, 256), (300, 136, 1000, 0.0, None)])
def test_reads_only_what_it_wrote(n, d, V, scored, rows, monkeypatch):
    want = _both(n, d, V, scored, 0.7, False, monkeypatch, rows=rows)[1]
    with poisoned():
        got = _both(n, d, V, scored, 0.7, False, monkeypatch, rows=rows)[0]
    assert all(torch.equal(x, y) for x, y in zip(got, want))


def _inputs(seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    W = (torch.randn(5003, 512, generator=g, device=DEV) * 0.05).bfloat16().requires_grad_(True)
    h = torch.randn(300, 512, generator=g, device=DEV).bfloat16().requires_grad_(True)
    y = torch.randint(0, 5003, (300,), generator=g, device=DEV)
    gout = torch.randn(300, 2, generator=g, device=DEV)
    return h, W, y, gout


def _step(h, W, y, gout):
    return torch.autograd.grad(head_op.fused_head(h, W, y, 0.7), (h, W), gout)


def test_captured(monkeypatch):
    """Forward and backward in one graph, replayed on new values between the program's own calls."""
    monkeypatch.setattr(head_op, "_STAGE_WORK", 0)
    static = _inputs(0)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _step(*static)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = _step(*static)
    for seed in (1, 2, 3):
        new = _inputs(seed)
        with torch.no_grad():
            for a, b in zip(static, new):
                a.copy_(b)
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, _step(*new)))


def test_threads_and_streams(monkeypatch):
    """Threads with a stream of their own, more of them than the bound on live logits serves."""
    monkeypatch.setattr(head_op, "_STAGE_WORK", 0)
    monkeypatch.setattr(head_op, "_KEEP_BYTES", 2 * 512 * 5120 * 4)
    inputs = [_inputs(k) for k in range(4)]
    want = [_step(*x) for x in inputs]
    torch.cuda.synchronize()
    wrong = []

    def work(k):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(20):
                got = _step(*inputs[k])
                torch.cuda.current_stream().synchronize()
                if not all(torch.equal(a, b) for a, b in zip(got, want[k])):
                    wrong.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong and head_op._Room._taken[inputs[0][0].device] == 0
