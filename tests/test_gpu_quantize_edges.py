"""The dequantizers into outputs aligned to their element alone, and the Q4_K
weight quantizer against the CPU oracle, bit for bit, where its
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


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("dt", [O.Q8_0, O.Q4K, O.Q6K, O.Q8K])
def test_dequantize_unaligned_output(dt, f16):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import lloom_amd as L
    from lloom_amd.lib import check, lib
    from lloom_amd.quantized import _ctx, _stream

    x = torch.from_numpy(_input("count9", np.random.default_rng(2))).cuda()
    q = L.QTensor.quantize(x, dt)
    want = q.dequantize_f16() if f16 else q.dequantize()
    for off in (1, 2, 3):
        y = torch.full((x.numel() + 8,), 7.0, dtype=want.dtype, device="cuda")
        check(lib().lloom_hip_dequantize(_ctx(0), int(dt), q.storage.data_ptr(), x.numel(), y[off:].data_ptr(),
                                         1 if f16 else 0, _stream(y)))
        assert torch.equal(y[off:off + x.numel()], want.reshape(-1))
        assert (y[:off] == 7).all() and (y[off + x.numel():] == 7).all()
