"""The fused GRPO step whose weight gradient the backward makes (octo_head_step_later) against the step that makes it in
the forward, over what both take."""
import pytest
import torch

from octopus_amd import head_op
from octopus_amd.rl.prefix_tree import TreeMeta
from tests.test_gpu_poisoned import poisoned

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _both(run, monkeypatch):
    got, routes = [], []
    later_bytes = head_op._later_bytes
    monkeypatch.setattr(head_op, "_LATER_SHARE", 1 << 20)
    monkeypatch.setattr(head_op, "_LATER_WORK", 1 << 62)
    monkeypatch.setattr(head_op, "_later_bytes", lambda *a: routes.append(later_bytes(*a)) or routes[-1])
    for least in (0, 1 << 62):
        monkeypatch.setattr(head_op, "_LATER_WEIGHTS", least)
        got.append(run())
    assert len(routes) == 2 and routes[0] > 0 and routes[1] == 0
    return got


def _close(a, b, dtype):
    """Same operands and products, sums in fp32: what differs is the rounding to 16 bits, once (the product with the
    loss's gradient included) against twice. Three roundings, each at most half a unit in the last place (2^-7 of bf16's
    8 bits, 2^-10 of f16's 11) and evenly spread: 3^(1/2) x half a unit / 3^(1/2)."""
    ulp = 2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -10
    assert ((a.float() - b.float()).norm() / b.float().norm().clamp(min=1e-30)).item() <= ulp / 2


# one row; ragged rows, widths and vocabularies; as many rows as are taken; f16; the softcap; a scaled loss
@pytest.mark.parametrize("n,d,V,scored,dtype,cap,c,need_rows", [
    (1, 256, 640, 1.0, torch.bfloat16, False, 1.0, True),
    (300, 512, 5003, 0.7, torch.bfloat16, False, 1 / 3, True),
    (512, 256, 1024, 1.0, torch.bfloat16, False, 1.0, True),
    (257, 136, 1000, 0.5, torch.float16, False, -2.0, True),
    (333, 256, 1500, 0.9, torch.float16, True, 1.0, True),
    (300, 512, 3000, 0.0, torch.bfloat16, False, 1.0, True),
    (300, 512, 3000, 0.7, torch.bfloat16, True, 1.0, False),
])
def test_later_weight_gradient(n, d, V, scored, dtype, cap, c, need_rows, monkeypatch):
    g = torch.Generator(device=DEV).manual_seed(n + V)
    W = (torch.randn(V, d, generator=g, device=DEV) * 0.05).to(dtype)
    h = torch.randn(n, d, generator=g, device=DEV).to(dtype)
    y = torch.randint(0, V, (n,), generator=g, device=DEV)
    adv = torch.randn(n, generator=g, device=DEV)
    mask = (torch.rand(n, generator=g, device=DEV) < scored).float()
    old = torch.full((n,), -7.0, device=DEV)
    kw = {}
    if scored < 1:
        idx, count = head_op.compact_rows(mask.bool())
        kw = dict(idx=idx, count=count, labels_via_idx=True, scatter=True)
    post = head_op.Post(1 / 30.0, 30.0, True) if cap else head_op.Post()

    def run():
        hd, Wd = h.clone().requires_grad_(need_rows), W.clone().requires_grad_(True)
        loss, out = head_op.fused_grpo_head(hd, Wd, y, 0.7, adv, mask, old=old, post=post, **kw)
        hd.data.zero_()  # the gradients are those of the values the forward saw
        Wd.data.zero_()
        (c * loss).backward(retain_graph=True)
        first = Wd.grad
        Wd.grad = hd.grad = None
        (c * loss).backward()
        assert torch.equal(first, Wd.grad)
        return loss.detach(), out, hd.grad, Wd.grad

    a, b = _both(run, monkeypatch)
    assert abs(a[0] - b[0]) <= 1e-6 * max(1.0, abs(b[0])) and torch.equal(a[1], b[1])
    assert (a[2] is not None) == need_rows
    if need_rows:
        _close(a[2], b[2], dtype)
    _close(a[3], b[3], dtype)


def test_later_weight_gradient_of_a_tree(monkeypatch):
    T, d, V = 400, 256, 1000
    g = torch.Generator(device=DEV).manual_seed(2)
    f2t = torch.cat([torch.arange(200), torch.cat([torch.arange(100), torch.arange(200, 300)])]).to(DEV)
    flat = torch.randint(0, V, (300,), generator=g, device=DEV)[f2t]
    cu = torch.tensor([0, 200, 400], device=DEV)
    W = (torch.randn(V, d, generator=g, device=DEV) * 0.05).bfloat16()
    h = torch.randn(1, 300, d, generator=g, device=DEV).bfloat16()
    adv, mask = torch.randn(T, generator=g, device=DEV), torch.ones(T, device=DEV)
    mask[cu[1:] - 1] = 0.0

    def run():
        hd, Wd = h.clone().requires_grad_(True), W.clone().requires_grad_(True)
        meta = TreeMeta.on_device(flat, cu, f2t, 300, torch.ones(T, dtype=torch.bool, device=DEV))
        loss, out = head_op.fused_grpo_tree_head(hd, Wd, meta, 1.0, adv, mask, old=torch.full((T,), -7.0, device=DEV))
        loss.backward()
        return loss.detach(), out, hd.grad, Wd.grad

    a, b = _both(run, monkeypatch)
    assert abs(a[0] - b[0]) <= 1e-6 * max(1.0, abs(b[0])) and torch.equal(a[1], b[1])
    _close(a[2], b[2], torch.bfloat16)
    _close(a[3], b[3], torch.bfloat16)


def test_the_gradients_of_the_gradients(monkeypatch):
    """Differentiated with respect to the loss's factor: what the step that holds its gradients gives."""
    n, d, V = 300, 256, 2048
    g = torch.Generator(device=DEV).manual_seed(4)
    W = (torch.randn(V, d, generator=g, device=DEV) * 0.05).bfloat16().requires_grad_(True)
    h = torch.randn(n, d, generator=g, device=DEV).bfloat16().requires_grad_(True)
    y = torch.randint(0, V, (n,), generator=g, device=DEV)
    adv = torch.randn(n, generator=g, device=DEV)

    def run():
        loss, _ = head_op.fused_grpo_head(h, W, y, 0.7, adv, torch.ones(n, device=DEV))
        s = torch.tensor(1.7, device=DEV, requires_grad=True)
        gh, gw = torch.autograd.grad(s * loss, (h, W), create_graph=True)
        return torch.autograd.grad(gw.float().square().sum() + gh.float().square().sum(), s)[0]

    a, b = _both(run, monkeypatch)
    assert abs(a - b) <= 2.0 ** -8 * abs(b)  # gradients rounded to bf16 once or twice


@pytest.mark.parametrize("d,V,dtype", [(512, 5003, torch.bfloat16), (136, 1000, torch.float16),
                                       (512, 2048, torch.bfloat16)])
def test_reads_only_what_it_wrote(d, V, dtype, monkeypatch):
    n = 300
    g = torch.Generator(device=DEV).manual_seed(V)
    W = (torch.randn(V, d, generator=g, device=DEV) * 0.05).to(dtype)
    h = torch.randn(n, d, generator=g, device=DEV).to(dtype)
    y = torch.randint(0, V, (n,), generator=g, device=DEV)
    adv, mask = torch.randn(n, generator=g, device=DEV), (torch.rand(n, generator=g, device=DEV) < 0.7).float()
    idx, count = head_op.compact_rows(mask.bool())

    def run():
        hd, Wd = h.clone().requires_grad_(True), W.clone().requires_grad_(True)
        loss, out = head_op.fused_grpo_head(hd, Wd, y, 0.7, adv, mask, idx=idx, count=count, labels_via_idx=True,
                                            scatter=True)
        loss.backward()
        return out, hd.grad, Wd.grad

    want = _both(run, monkeypatch)[0]
    with poisoned(), monkeypatch.context() as m:
        m.setattr(head_op, "_LATER_WEIGHTS", 0)
        got = run()
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_captured(monkeypatch):
    """The step and its backward in one graph, replayed on new values between the program's own calls."""
    monkeypatch.setattr(head_op, "_LATER_WEIGHTS", 0)
    monkeypatch.setattr(head_op, "_LATER_SHARE", 1 << 20)

    def inputs(seed):
        g = torch.Generator(device=DEV).manual_seed(seed)
        W = (torch.randn(5003, 512, generator=g, device=DEV) * 0.05).bfloat16().requires_grad_(True)
        h = torch.randn(300, 512, generator=g, device=DEV).bfloat16().requires_grad_(True)
        y = torch.randint(0, 5003, (300,), generator=g, device=DEV)
        return h, W, y, torch.randn(300, generator=g, device=DEV), torch.randn((), generator=g, device=DEV)

    mask = torch.ones(300, device=DEV)

    def step(h, W, y, adv, c):
        loss, out = head_op.fused_grpo_head(h, W, y, 0.7, adv, mask)
        return (out, *torch.autograd.grad(loss, (h, W), c))

    static = inputs(0)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step(*static)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = step(*static)
    for seed in (1, 2, 3):
        new = inputs(seed)
        with torch.no_grad():
            for a, b in zip(static, new):
                a.copy_(b)
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, step(*new)))
