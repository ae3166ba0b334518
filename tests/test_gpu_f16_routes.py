"""F16 activations and outputs on every dense route: y is bit for bit the
round-to-nearest-even of what the same call on x widened to F32 stores
(matmul_t_f16, k_quants.rs:2802-2835), for the plain, SiLU and multiply-into
stores.  Rows cover each route's band, n is even, odd and a multiple of 4."""
import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu

ROWS = {O.Q4K: [1, 3, 5, 16, 17, 130, 330, 700], O.Q6K: [1, 4, 9, 20, 60, 200, 660], O.Q8_0: [1, 4, 6, 40, 150, 400]}


@pytest.mark.parametrize("dt,n,k", [(dt, n, k) for dt in (O.Q4K, O.Q6K, O.Q8_0)
                                    for n, k in ((260, 2048), (129, 512), (70, 4352))] + [(O.Q4K, 14000, 4096)])
def test_f16_is_the_rounded_f32_call(dt, n, k):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import lloom_amd as L

    g = torch.Generator(device="cuda")
    g.manual_seed(n + k)
    w = torch.randn(n, k, generator=g, device="cuda") * 0.02
    mm = L.QMatMul(L.QTensor.quantize(w, dt))
    for m in ROWS[dt] if n < 1000 else [4, 9]:
        x = torch.randn(m, k, generator=g, device="cuda").half()
        gate = torch.randn(m, n, generator=g, device="cuda").half()
        wide, into32, into16 = x.float(), gate.float(), gate.clone()
        assert torch.equal(mm.forward(x), mm.forward(wide).half()), (m, "plain")
        assert torch.equal(mm.forward_silu(x), mm.forward_silu(wide).half()), (m, "silu")
        mm.forward_mul_into(wide, into32)
        mm.forward_mul_into(x, into16)
        assert torch.equal(into16, into32.half()), (m, "mul_into")
