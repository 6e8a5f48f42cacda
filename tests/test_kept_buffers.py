"""Which calls keep a buffer between forward and backward, and its size (host planning only)."""
import pytest

from octopus_amd import _lib, head_op


@pytest.mark.parametrize("n,d,V", [(1, 256, 640), (300, 136, 1000), (5119, 2560, 151936), (8192, 4096, 128256)])
def test_stage_size_is_the_one_a_traced_call_expects(n, d, V):
    buf, ws = _lib.stage_bytes(n, d, V, _lib.BF16)
    P, Vp = -(-n // 256) * 256, -(-V // 256) * 256
    assert buf == head_op._stage_numel(n, V) and buf >= P * Vp * 2 + P * 4 + n * (Vp // 256) * 16
    assert ws >= P * Vp * 2 + d * P * 2 + (d * Vp * 2 if V % 64 or d % 256 else 0)


def test_what_is_not_staged():
    for w in (_lib.F16, _lib.F32, _lib.FP8E4M3):
        assert _lib.stage_bytes(256, 256, 1024, w) == (0, 0)
    assert _lib.stage_bytes(0, 256, 1024, _lib.BF16) == (0, 0)
    assert _lib.stage_bytes(32768, 256, 151936, _lib.BF16) == (0, 0)  # past 2 GiB


def test_what_is_left_for_later():
    assert _lib.later_bytes(300, 512, 5003, _lib.FP8E4M3, True) == _lib.later_bytes(300, 512, 5003, _lib.F32, True) == 0
    assert _lib.later_bytes(0, 512, 5003, _lib.BF16, True) == 0
    assert _lib.later_bytes(32768, 2560, 151936, _lib.BF16, True) == 0  # several passes
    for n in (1, 257, 1536):
        P = -(-n // 256) * 256
        plain = _lib.later_bytes(n, 2560, 151936, _lib.BF16, False)
        assert plain >= P * (-(-151936 // 256) * 256) * 2 + 2560 * P * 2  # dz and h^T
        assert 0 <= _lib.later_bytes(n, 2560, 151936, _lib.BF16, True) - plain <= 256 * 256 * 256 * 4  # one round of runs
