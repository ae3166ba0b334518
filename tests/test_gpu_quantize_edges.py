"""The Q4_K weight quantizer against the CPU oracle, bit for bit, where its
work split can go wrong: superblock counts around a wave (8) and a workgroup
(32), and values around its clamps and divisions (levels at exact halves,
constant and zero sub-blocks, scales from subnormal to the top of f32,
infinities and NaN)."""
import numpy as np
import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu


def _input(name, rng):
    x = rng.standard_normal((512, 256)).astype(np.float32)
    if name.startswith("count"):
        return x[:int(name[5:])] * np.float32(0.02)
    if name == "halves":
        return (rng.integers(-8, 24, x.shape) * 0.5).astype(np.float32)
    if name == "constant":
        x.reshape(-1, 32)[::2] = 3.25
        x[:9] = 0.0
        return x
    if name == "scales":
        return np.ldexp(x, rng.integers(-140, 120, (512, 1))).astype(np.float32)
    if name == "scales32":
        return np.ldexp(x.reshape(-1, 32), rng.integers(-30, 30, (512 * 8, 1))).astype(np.float32).reshape(x.shape)
    x[::3, 5] = np.inf
    x[1::3, 9] = -np.inf
    x[2::5, 200] = np.nan
    return x


@pytest.mark.parametrize("name", ["count1", "count7", "count8", "count9", "count31", "count32", "count33", "halves",
                                  "constant", "scales", "scales32", "nonfinite"])
def test_quantize_q4k_bits(name):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import lloom_amd as L

    x = _input(name, np.random.default_rng(1))
    got = L.QTensor.quantize(torch.from_numpy(x).cuda(), O.Q4K).data()
    with np.errstate(all="ignore"):
        assert np.array_equal(got, O.quantize(O.Q4K, x.ravel()))
