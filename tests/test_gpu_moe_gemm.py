"""The grouped GEMM of the routed experts (Q4_K and Q6_K with several planes
an expert on average) against a float64 product of the dequantized
weights (O.dequantize, the CPU oracle's to_float), through the public calls.

Where it can go wrong: planes of one expert around the 32-plane tile and the
64-plane cut (1, 31, 32, 33, 63, 64, 65, 129 and none), weight rows off the
workgroup's 128 (64 for the SwiGLU), one superblock a row and many, activations
one row a token and one a slot, tiles of 32 planes and of 64, an outlier beside
small elements, more experts than routing workgroups, out-of-range ids, and a
capture whose workspace holds only the routing.  Each case asserts whether the
grouped GEMM is what serves it.

The bound: an element of x loses at most 2^-23 of itself, or 2^-50 of its row's
largest element, to its two halves; Q6_K drops lo * lo, 2^-22 of the product,
and Q4_K's pair of a sub-block's coefficient holds 2^-22; a row is summed in f32
in fewer than K / 8 steps.  So |err| <= (2^-21 + K / 8 * 2^-24) * S + 2^-49 *
max|x| * W, with the sub-blocks' S = sum |x| (|d sc q| + |dmin m|) <= 3 max|w|
sum |x| and W the same for |x| = 1: what an element's own weight is zero for
never enters.
"""
import numpy as np
import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu

COUNTS = [1, 31, 32, 33, 63, 64, 65, 129, 0]
FEW = [1, 4, 31, 32, 33, 9, 0, 8]  # up to 16 an expert on average: tiles of 32


@pytest.fixture(scope="module")
def L():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import lloom_amd

    lloom_amd.lib()
    return lloom_amd


def _case(rng, dt, E, n, k, topk, per_slot, counts):
    w = (rng.standard_normal((2, E, n, k)) * 0.05).astype(np.float32)
    planes = sum(counts)
    batch = -(-planes // topk)
    flat = np.concatenate([np.full(c, e) for e, c in enumerate(counts)] + [np.full(batch * topk - planes, 0)])
    ids = rng.permutation(flat).reshape(batch, topk).astype(np.int32)
    x = rng.standard_normal((batch, topk if per_slot else 1, k)).astype(np.float32)
    x[0, 0, :32] *= 1e4
    x[-1] *= 1e-30
    return w, x, ids


def _want(dt, q, E, n, k, x, ids):
    dense = O.dequantize(dt, q, E * n * k).reshape(E, n, k).astype(np.float64)
    xs = np.broadcast_to(x, (ids.shape[0], ids.shape[1], k)).astype(np.float64)
    want = np.zeros(ids.shape + (n,))
    tol = np.zeros(ids.shape + (n,))
    for e in range(E):
        at = ids == e
        want[at] = xs[at] @ dense[e].T
        top = np.abs(dense[e]).reshape(n, k // 32, 32).max(2)
        xa = np.abs(xs[at])
        tol[at] = 3 * (2.0 ** -21 + k / 8 * 2.0 ** -24) * (xa.reshape(-1, k // 32, 32).sum(2) @ top.T) \
            + 3 * 2.0 ** -49 * xa.max(1, keepdims=True) * (32 * top.sum(1))
    return want, tol


def _on_small_context(q, x, ids, call="one", q2=None, mib=1):
    """The call captured on a context that holds `mib` MiB of workspace: the
    kernels that need no copy of x serve it.  The result of one replay."""
    import ctypes

    from lloom_amd.lib import check, lib
    from lloom_amd.quantized import _ptr, _stream

    (E, n, k), (batch, in_dim1, _), topk = q.shape, x.shape, ids.shape[1]
    y = torch.zeros(batch, topk, n, device="cuda")
    ctx = ctypes.c_void_p()
    check(lib().lloom_hip_ctx_create(0, ctypes.byref(ctx)))
    check(lib().lloom_hip_ctx_reserve(ctx, mib << 20))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        if call == "one":
            check(lib().lloom_hip_moe_matmul(ctx, int(q.dtype), _ptr(q.storage), E, n, k, _ptr(x), batch, in_dim1,
                                             _ptr(ids), topk, _ptr(y), 0, _stream(x)))
        else:
            check(lib().lloom_hip_moe_matmul_glu(ctx, int(q.dtype), _ptr(q.storage), _ptr(q2.storage), E, n, k,
                                                 _ptr(x), batch, in_dim1, _ptr(ids), topk, _ptr(y), 0, _stream(x)))
    for _ in range(2):  # the second replay counts
        y.zero_()
        graph.replay()
    got = y.cpu().numpy()
    del graph
    lib().lloom_hip_ctx_destroy(ctx)
    return got


def _served(dt, E, n, k, x, ids):
    """Whether the grouped GEMM serves the call: its workspace holds x."""
    from lloom_amd.quantized import moe_workspace_bytes

    return moe_workspace_bytes(dt, E, n, k, x.shape[0], x.shape[1], ids.shape[1]) > 4 * x.size


SHAPES = [(200, 768, 4, False), (8, 256, 3, True), (1100, 512, 1, False), (177, 2048, 2, True), (2065, 256, 2, False),
          (600, 2048, 3, True), (601, 768, 2, False)]


@pytest.mark.parametrize("dt", [O.Q4K, O.Q6K])
@pytest.mark.parametrize("counts", [COUNTS, FEW], ids=["many", "few"])
@pytest.mark.parametrize("n,k,topk,per_slot", SHAPES)
def test_moe_gemm_matches_f64(L, dt, n, k, topk, per_slot, counts):
    rng = np.random.default_rng(n + k)
    E = len(counts)
    w, x, ids = _case(rng, dt, E, n, k, topk, per_slot, counts)
    # small Q6_K calls are another kernel's: the same result
    assert _served(dt, E, n, k, x, ids) == (dt == O.Q4K or ids.size * n >= 65536)
    qg, qu = (L.QTensor.quantize(torch.from_numpy(v).cuda(), dt) for v in w)
    xd, idd = torch.from_numpy(x).cuda(), torch.from_numpy(ids).cuda()
    g, u = (q.indexed_moe_forward(xd, idd).cpu().numpy() for q in (qg, qu))
    for got, q in ((g, qg), (u, qu)):
        want, tol = _want(dt, q.data(), E, n, k, x, ids)
        assert (np.abs(got - want) <= tol).all(), (np.abs(got - want) / tol).max()
    # the pair is the two calls bit for bit, the SwiGLU their silu(g) * u
    pg, pu = (v.cpu().numpy() for v in qg.indexed_moe_forward_pair(qu, xd, idd))
    assert np.array_equal(pg.view(np.uint32), g.view(np.uint32)) and np.array_equal(pu.view(np.uint32), u.view(np.uint32))
    glu = qg.indexed_moe_forward_glu_as(qu, xd, idd).cpu().numpy()
    np.testing.assert_allclose(glu, g / (1 + np.exp(-g.astype(np.float64))) * u, rtol=2e-6, atol=1e-30)


@pytest.mark.parametrize("dt", [O.Q4K, O.Q6K])
def test_moe_gemm_bad_id_and_nonfinite(L, dt):
    """A bad id zeroes its plane and is refused; a row with an infinity
    spoils its own planes and no other."""
    rng = np.random.default_rng(3)
    E, n, k = 3, 900, 512
    w = (rng.standard_normal((E, n, k)) * 0.05).astype(np.float32)
    q = L.QTensor.quantize(torch.from_numpy(w).cuda(), dt)
    ids = rng.integers(0, E, (40, 2)).astype(np.int32)
    x = rng.standard_normal((40, 1, k)).astype(np.float32)
    assert _served(dt, E, n, k, x, ids)
    want, tol = _want(dt, q.data(), E, n, k, x, ids)
    bad = ids.copy()
    bad[7, 1] = E
    xd = torch.from_numpy(x).cuda()
    with pytest.raises(L.LloomHipError) as err:
        q.indexed_moe_forward(xd, torch.from_numpy(bad).cuda())
    assert err.value.name == "EEXPERT"
    y = q.indexed_moe_forward(xd, torch.from_numpy(bad).cuda(), strict=False).cpu().numpy()
    assert not y[7, 1].any()
    y[7, 1] = want[7, 1]
    assert (np.abs(y - want) <= tol).all()
    from lloom_amd.lib import lib
    from lloom_amd.quantized import _ctx

    assert lib().lloom_hip_ctx_sync(_ctx(0)) == 4
    x[5, 0, 100] = np.inf
    y = q.indexed_moe_forward(torch.from_numpy(x).cuda(), torch.from_numpy(ids).cuda()).cpu().numpy()
    assert not np.isfinite(y[5]).any()
    keep = np.arange(40) != 5
    assert (np.abs(y - want) <= tol)[keep].all()


def _us(f):
    """The median time of a call among others, in microseconds."""
    f()
    torch.cuda.synchronize()
    times = []
    for _ in range(5):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(10):
            f()
        b.record()
        b.synchronize()
        times.append(a.elapsed_time(b) * 100)
    return sorted(times)[2]


@pytest.mark.parametrize("dt", [O.Q4K, O.Q6K])
def test_moe_gemm_many_bad_ids(L, dt):
    """Half of the ids out of range, in every 64 planes: their outputs are zero
    in each of the three calls, the others as without them, and such planes cost
    no more than good ones."""
    from lloom_amd.lib import lib
    from lloom_amd.quantized import _ctx

    rng = np.random.default_rng(8)
    E, n, k, batch, topk = 5, 129, 512, 731, 4
    w = (rng.standard_normal((2, E, n, k)) * 0.05).astype(np.float32)
    qg, qu = (L.QTensor.quantize(torch.from_numpy(v).cuda(), dt) for v in w)
    ids = torch.from_numpy(rng.integers(0, E, (batch, topk)).astype(np.int32)).cuda()
    x = torch.from_numpy(rng.standard_normal((batch, 1, k)).astype(np.float32)).cuda()
    out = torch.from_numpy(rng.random((batch, topk)) < 0.5).cuda()
    bad = ids.clone()
    bad[out] = torch.from_numpy(rng.choice([E, -1, 1 << 30], int(out.sum())).astype(np.int32)).cuda()
    calls = [lambda i: [qg.indexed_moe_forward(x, i, strict=False)],
             lambda i: qg.indexed_moe_forward_pair(qu, x, i, strict=False),
             lambda i: [qg.indexed_moe_forward_glu_as(qu, x, i, strict=False)]]
    for call in calls:
        torch.full((2 * batch * topk * n,), 7.0, device="cuda")  # the outputs' memory held something else
        for got, good in zip(call(bad), call(ids)):
            assert not got[out].any()
            assert torch.equal(got[~out], good[~out])
    assert lib().lloom_hip_ctx_sync(_ctx(0)) == 4
    q = L.QTensor.quantize(torch.randn(8, 768, 2048, device="cuda"), dt)
    x, ids = torch.randn(4096, 1, 2048, device="cuda"), torch.arange(4096, device="cuda", dtype=torch.int32)[:, None] % 8
    y = torch.empty(4096, 1, 768, device="cuda")
    good, none = (_us(lambda i=i: q.indexed_moe_forward_into(x, i, y)) for i in (ids, ids + 8))
    assert none < 3 * good, (none, good)
    assert lib().lloom_hip_ctx_sync(_ctx(0)) == 4


@pytest.mark.parametrize("dt,E", [(O.Q4K, 255), (O.Q4K, 257), (O.Q4K, 600), (O.Q6K, 1025), (O.Q4K, 4096)])
def test_moe_gemm_many_experts(L, dt, E):
    """More experts than routing workgroups, some of them with no plane."""
    rng = np.random.default_rng(E)
    n, k, planes = 40, 256, 14 * E
    q = L.QTensor.quantize(torch.from_numpy((rng.standard_normal((E, n, k)) * 0.05).astype(np.float32)).cuda(), dt)
    ids = np.minimum((rng.random((planes // 2, 2)) ** 2 * E).astype(np.int32), E - 1)
    ids[ids % 7 == 3] = E - 1
    x = rng.standard_normal((planes // 2, 1, k)).astype(np.float32)
    assert _served(dt, E, n, k, x, ids)
    got = q.indexed_moe_forward(torch.from_numpy(x).cuda(), torch.from_numpy(ids).cuda()).cpu().numpy()
    want, tol = _want(dt, q.data(), E, n, k, x, ids)
    assert (np.abs(got - want) <= tol).all()


def test_moe_gemm_routing_cost(L):
    """128 K planes over 4096 experts cost about what they do over 256."""
    us = []
    for E in (256, 4096):
        q = L.QTensor.quantize(torch.randn(E, 64, 256, device="cuda"), O.Q4K)
        x, y = torch.randn(1 << 17, 1, 256, device="cuda"), torch.empty(1 << 17, 1, 64, device="cuda")
        ids = torch.arange(1 << 17, device="cuda", dtype=torch.int32)[:, None] % E
        us.append(_us(lambda: q.indexed_moe_forward_into(x, ids, y)))
    assert us[1] < 2 * us[0], us


@pytest.mark.parametrize("dt", [O.Q4K, O.Q6K])
@pytest.mark.parametrize("counts", [[40, 33, 64, 130], [12, 13, 9, 30]], ids=["64", "32"])
@pytest.mark.parametrize("bits", [0, 20, 26])
def test_moe_gemm_small_beside_outlier(L, dt, counts, bits):
    """An element 2^bits larger than the rest meets weights that are zero: the
    others keep their precision (f32 dots lose nothing to it either)."""
    rng = np.random.default_rng(bits)
    E, n, k = len(counts), 3100, 768
    w = (rng.standard_normal((E, n, k)) * 0.05).astype(np.float32)
    w[..., 32:64] = w[..., 512:544] = 0
    q = L.QTensor.quantize(torch.from_numpy(w).cuda(), dt)
    ids = np.repeat(np.arange(E), counts).astype(np.int32)[:, None]
    x = rng.standard_normal((len(ids), 1, k)).astype(np.float32)
    assert _served(dt, E, n, k, x, ids)
    x[..., 37] *= 2.0 ** bits
    x[::2, ..., 513] *= -(2.0 ** bits)
    want, tol = _want(dt, q.data(), E, n, k, x, ids)
    got = q.indexed_moe_forward(torch.from_numpy(x).cuda(), torch.from_numpy(ids).cuda()).cpu().numpy()
    assert (np.abs(got - want) <= tol).all(), (np.abs(got - want) / tol).max()


@pytest.mark.parametrize("dt", [O.Q4K, O.Q6K])
def test_moe_gemm_tiny_rows(L, dt):
    """Rows whose power-of-two scale would leave the normal numbers, down to
    subnormal x, on the grouped GEMM and without room for a copy of x (half of
    the last place of a subnormal result comes on top of the bound)."""
    rng = np.random.default_rng(9)
    E, n, k = 4, 320, 2048
    q = L.QTensor.quantize(torch.from_numpy((rng.standard_normal((E, n, k)) * 0.05).astype(np.float32)).cuda(), dt)
    ids = rng.integers(0, E, (240, 1)).astype(np.int32)
    x = np.ldexp(rng.standard_normal((240, 1, k)).astype(np.float32), np.repeat([-100, -114, -119, -133], 60)[:, None, None])
    assert _served(dt, E, n, k, x, ids)
    want, tol = _want(dt, q.data(), E, n, k, x, ids)
    xd, idd = torch.from_numpy(x).cuda(), torch.from_numpy(ids).cuda()
    for got in (q.indexed_moe_forward(xd, idd).cpu().numpy(), _on_small_context(q, xd, idd)):
        assert (np.abs(got - want) <= tol + 2.0 ** -149).all()


@pytest.mark.parametrize("dt,E,n,k,per", [(O.Q4K, 64, 416, 2048, 5), (O.Q4K, 64, 512, 768, 7), (O.Q4K, 16, 320, 2048, 40),
                                          (O.Q6K, 64, 640, 2048, 5), (O.Q6K, 64, 512, 768, 14), (O.Q6K, 16, 320, 2048, 40)])
def test_moe_gemm_no_further_off_than_the_other_kernels(L, dt, E, n, k, per):
    """Against 64 bits (2-norm), the grouped GEMM is no further off than what
    serves the same call without a copy of x (f32 dots below 8 planes an expert
    and for Q6_K)."""
    rng = np.random.default_rng(per)
    q = L.QTensor.quantize(torch.from_numpy((rng.standard_normal((E, n, k)) * 0.02).astype(np.float32)).cuda(), dt)
    ids = rng.integers(0, E, (E * per, 1)).astype(np.int32)
    x = (rng.standard_normal((E * per, 1, k)) * rng.standard_normal((E * per, 1, k))).astype(np.float32)
    xd, idd = torch.from_numpy(x).cuda(), torch.from_numpy(ids).cuda()
    assert _served(dt, E, n, k, x, ids)
    want, _ = _want(dt, q.data(), E, n, k, x, ids)
    off = [np.linalg.norm(y - want) / np.linalg.norm(want)
           for y in (q.indexed_moe_forward(xd, idd).cpu().numpy(), _on_small_context(q, xd, idd))]
    assert off[0] <= off[1], off


@pytest.mark.parametrize("dt", [O.Q4K, O.Q6K])
def test_moe_gemm_captured(L, dt):
    """Replays equal the eager call, on a context that reserved what the size
    query says too."""
    from lloom_amd.quantized import moe_workspace_bytes

    rng = np.random.default_rng(4)
    E, n, k, batch, topk = 4, 400, 2048, 128, 4
    w = (rng.standard_normal((E, n, k)) * 0.05).astype(np.float32)
    q = L.QTensor.quantize(torch.from_numpy(w).cuda(), dt)
    ids = torch.from_numpy(rng.integers(0, E, (batch, topk)).astype(np.int32)).cuda()
    x = torch.from_numpy(rng.standard_normal((batch, topk, k)).astype(np.float32)).cuda()
    eager = q.indexed_moe_forward(x, ids)
    y = torch.empty_like(eager)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        q.indexed_moe_forward_into(x, ids, y)
    for _ in range(3):
        y.zero_()
        graph.replay()
        assert torch.equal(y, eager)
    need = moe_workspace_bytes(dt, E, n, k, batch, topk, topk)
    assert np.array_equal(_on_small_context(q, x, ids, mib=(need + (1 << 20) - 1) >> 20), eager.cpu().numpy())


@pytest.mark.parametrize("dt,E,n,k,topk,planes", [
    (O.Q4K, 4, 400, 2048, 4, 512), (O.Q4K, 8, 200, 768, 4, 1600),  # 8 planes an expert: in-kernel and sorted routing
    (O.Q4K, 160, 132, 512, 7, 1120), (O.Q6K, 4, 400, 2048, 4, 512), (O.Q6K, 64, 200, 512, 4, 1280)])
@pytest.mark.parametrize("call", ["one", "glu"])
def test_moe_captured_without_room_for_x(L, dt, E, n, k, topk, planes, call):
    """A capture on a context whose workspace cannot hold the copy of x is
    served all the same, leaves no error message, and replays right, in-kernel
    routing (up to 1024 planes) and sorted."""
    from lloom_amd.lib import lib

    rng = np.random.default_rng(planes)
    w = (rng.standard_normal((2, E, n, k)) * 0.05).astype(np.float32)
    qg, qu = (L.QTensor.quantize(torch.from_numpy(v).cuda(), dt) for v in w)
    ids = rng.integers(0, E, (planes // topk, topk)).astype(np.int32)
    x = rng.standard_normal((planes // topk, topk, k)).astype(np.float32)
    assert lib().lloom_hip_ctx_create(-1, None) and b"out is null" in lib().lloom_hip_last_error()
    y = _on_small_context(qg, torch.from_numpy(x).cuda(), torch.from_numpy(ids).cuda(), call, qu)
    assert b"out is null" in lib().lloom_hip_last_error()
    g, gtol = _want(dt, qg.data(), E, n, k, x, ids)
    if call == "one":
        assert (np.abs(y - g) <= gtol).all()
        return
    u, utol = _want(dt, qu.data(), E, n, k, x, ids)
    silu = g / (1 + np.exp(-g))
    assert (np.abs(y - silu * u) <= 1.1 * gtol * np.abs(u) + np.abs(silu) * utol + 2 * gtol * utol + 1e-6 * np.abs(silu * u)).all()
