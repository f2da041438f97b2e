"""The encoder's eight elements per lane: lanes whose products are all at least 2^-6 take a path of their own, the others and
every scale above 2^100 the general one.  One small, zero, denormal, infinite or NaN element at each place of a lane, around
the saturation and the 2^-6 line, at lengths that end inside a lane, against the CPU oracle, bit for bit."""
import numpy as np
import pytest
import torch

from flame_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("inv_scale", [56.0, -3.0, 2.0 ** 100, 2.0 ** 101, 2.0 ** 126])
@pytest.mark.parametrize("n", [16, 1000, 8 * 4096 + 5])
def test_mixed_lanes(oracle, inv_scale, n):
    from flame_amd import capi
    x = W.normal_f32(7300 + n, 1, n) / np.float32(abs(inv_scale)) * np.float32(100.0)
    odd = np.array([0.0, -0.0, 1e-40, -1e-40, 2.0 ** -6, 2.0 ** -7, 2.0 ** -10, 247.9, 248.0, 1e9, np.inf, -np.inf], np.float32)
    for i in range(min(len(odd) * 8, n // 8)):       # element i % 8 of lane i
        x[8 * i + i % 8] = odd[(i // 8) % len(odd)] / np.float32(abs(inv_scale) if 1e-7 < abs(odd[(i // 8) % len(odd)]) < 1e10 else 1.0)
    bits = W.f32_to_bf16_bits(x)
    bits[n // 2] = 0x7fc0
    got = capi.bf16_to_fp8(torch.from_numpy(bits.view(np.int16)).cuda().view(torch.bfloat16), inv_scale).cpu().numpy()
    assert np.array_equal(got, oracle.bf16_to_fp8(bits, inv_scale))
