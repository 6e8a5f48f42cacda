"""octohead::scaled, the fused step's backward: c x in fp32 rounded once, against the same arithmetic in torch, bit for
bit, over vector lengths around the kernel's 16-byte chunks and its grid's stride; and a retained graph's second
backward, which finds the held gradients as the first did."""

import pytest
import torch

from octopus_amd import head_op

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "f16", "f32"])
@pytest.mark.parametrize("n", [0, 1, 3, 8, 2047, 2048 * 256 * 8 + 5, 3 * 2048 * 256 * 8 + 8])
def test_scaled_rounds_the_fp32_product_once(n, dtype):
    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn(n, generator=g, device="cuda").to(dtype)
    for c in (1.0, -2.0, 1 / 3):
        c = torch.tensor(c, device="cuda")
        assert torch.equal(head_op.scaled(x, c), (x.float() * c).to(dtype))


def test_a_retained_graph_gives_its_gradients_twice():
    g = torch.Generator().manual_seed(3)
    h = torch.randn(70, 64, generator=g).to(torch.bfloat16).cuda().requires_grad_(True)
    W = (torch.randn(640, 64, generator=g) * 0.1).to(torch.bfloat16).cuda().requires_grad_(True)
    y = torch.randint(0, 640, (70,), generator=g).cuda()
    loss, _ = head_op.fused_grpo_head(h, W, y, 1.0, torch.randn(70, generator=g).cuda(), torch.ones(70).cuda())
    first = [t.clone() for t in torch.autograd.grad(2 * loss, (h, W), retain_graph=True)]
    second = torch.autograd.grad(2 * loss, (h, W), retain_graph=True)
    assert all(torch.equal(a, b) for a, b in zip(first, second))
    third = torch.autograd.grad(loss, (h, W), create_graph=True)
    assert all(torch.equal((b.float() * 2).to(b.dtype), a) for a, b in zip(first, third))
