"""octohead::scaled, the fused step's backward: c x in fp32 rounded once, against the same arithmetic in torch, bit for
bit, over vector lengths around the kernel's 16-byte chunks and its workgroups' 1,024; the in-place form, which walks
the vector; and a retained graph's second backward, which finds the held gradients as the first did."""

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


# the in-place form walks the vector with 2,048 workgroups of 256 threads and 4 loads in flight: lengths around one load
# of every thread, around all four, and past them
_WALK = 2048 * 256


@pytest.mark.parametrize("dtype,per", [(torch.bfloat16, 8), (torch.float16, 8), (torch.float32, 4)])
@pytest.mark.parametrize("chunks,over", [(0, 3), (1, 0), (_WALK, -1), (_WALK, 5), (4 * _WALK, 5), (5 * _WALK, 1)])
def test_scale_add_in_place(chunks, over, dtype, per):
    """y = c y + x, formed in fp32 and rounded once; x left out while skip is set, or not given at all."""
    n = chunks * per + over
    g = torch.Generator(device="cuda").manual_seed(n)
    y, x = (torch.randn(n, generator=g, device="cuda").to(dtype) for _ in range(2))
    on, off = (torch.tensor([k], dtype=torch.int32, device="cuda") for k in (0, 1))
    for c in (1.0, -1.7):
        c = torch.tensor([c], device="cuda")
        for rest, skip in ((None, None), (x, None), (x, on), (x, off)):
            got = head_op._scale_add(y.clone(), rest, c, skip)
            want = c.double() * y.double()
            if rest is not None and skip is not off:
                want += x.double()
            # 64-bit sums rounded to fp32, and then to 16 bits: a sum next to a tie of the two roundings may fall either
            # way
            want = want.float()
            if dtype == torch.float32:
                assert ((got - want).abs() <= want.abs() * 2.0 ** -23).all()
            else:
                assert torch.equal(got, want.to(dtype))


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
