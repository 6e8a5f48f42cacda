"""head_columns over logits whose vocabulary is masked with very low finite values, and with the row count changing."""
import pytest
import torch

from octopus_amd import head_op

pytestmark = pytest.mark.gpu
DEV = "cuda"


# longer than what a workgroup reads at a time (32,768 values of 16 bits, 16,384 of fp32), so that a
# thread's first logits are all at the type's lowest value, at a temperature that keeps x / T log2 e finite
@pytest.mark.parametrize("dtype,n,V,T,low", [
    (torch.bfloat16, 3, 40000, 2.0, None),
    (torch.float32, 3, 20001, 2.0, None),
    (torch.float32, 600, 20003, 1.0, -1e38),
    (torch.float16, 3, 40000, 1.0, None),
])
def test_masked_with_low_finite_values(dtype, n, V, T, low):
    g = torch.Generator(device=DEV).manual_seed(V)
    z = torch.randn(n, V, generator=g, device=DEV).to(dtype)
    z[:, : V * 9 // 10] = torch.finfo(dtype).min if low is None else low
    z[:, -7:] = torch.finfo(dtype).min if low is None else low
    y = torch.randint(V * 9 // 10, V - 7, (n,), generator=g, device=DEV)
    out = head_op.head_columns(z, T, y)
    lp = torch.log_softmax(z.double() / T, 1)
    ent = -torch.where(lp.exp() > 0, lp.exp() * lp, torch.zeros_like(lp)).sum(1)
    assert (out[:, 0].double() - lp.gather(1, y[:, None])[:, 0]).abs().max() <= 2e-5
    assert (out[:, 1].double() - ent).abs().max() <= 2e-5  # 32-bit sums of terms of order 10


@pytest.mark.parametrize("dtype,V", [(torch.bfloat16, 9000), (torch.float32, 5003)])
def test_a_row_does_not_depend_on_the_rows_beside_it(dtype, V):
    g = torch.Generator(device=DEV).manual_seed(V)
    z = (torch.randn(700, V, generator=g, device=DEV) * 4).to(dtype)
    y = torch.randint(0, V, (700,), generator=g, device=DEV)
    assert torch.equal(head_op.head_columns(z, 0.7, y)[:100], head_op.head_columns(z[:100], 0.7, y[:100]))
