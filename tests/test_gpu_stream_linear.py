"""The streaming decode linear (linear_stream.hip) on the automatic route.

Shapes at the edges of its tiles: K an odd number of 64-k steps, a tail
shorter than its chunks, K splits with a short last one, N not a multiple of
16 and of a workgroup's row tiles, every count of activation tiles; wide
matrices of one and two tiles per wave.  Each result is held to the oracle at
relative L2 1e-4 per row (1e-5 over dense rows), repeats to the same bits, and the no-allocation
entry point to the same bits too.
"""
import numpy as np
import pytest

import oracle
from air_amd import capi, quant
from tests import helpers
from tests.test_gpu_dense import _weights

pytestmark = pytest.mark.gpu

DECODE_TOL = 1e-4
DENSE_TOL = 1e-5          # the gate of the dense kernels

# (format, K, N, widths)
CASES = [
    (capi.TYPE_Q8_0, 2080, 5000, (17, 33, 64)),       # 33 steps, 313 row tiles, K splits
    (capi.TYPE_Q8_0, 4640, 1613, (25, 48)),            # 73 steps, long K, ragged N
    (capi.TYPE_Q8_0, 2048, 16500, (2, 16, 40)),       # wide, eight tiles a workgroup
    (capi.TYPE_Q8_0, 2112, 34000, (3, 64)),           # ten
    (capi.TYPE_Q8_0, 2048, 41000, (9, 33, 49)),       # twenty, two per wave
    (capi.TYPE_Q4_0, 2144, 4200, (17, 64)),
    (capi.TYPE_Q4_0, 5152, 1530, (18, 33)),
    (capi.TYPE_Q4_0, 2048, 41000, (5, 32, 50)),
    (capi.TYPE_Q4_K, 2304, 4200, (20, 48)),
    (capi.TYPE_Q4_K, 8448, 1530, (2, 16, 17, 64)),
    (capi.TYPE_Q4_K, 2048, 41000, (7, 30, 64)),
    (capi.TYPE_Q6_K, 2304, 4200, (3, 17, 33, 64)),    # dense rows: two splits of nine super-blocks
    (capi.TYPE_Q6_K, 8448, 1530, (2, 16, 40)),
    (capi.TYPE_Q6_K, 2048, 41000, (5, 20, 50)),
    (capi.TYPE_F16, 3104, 4200, (17, 33, 64)),        # a row ends on the first block of a step
    (capi.TYPE_F16, 8224, 1530, (18, 48)),
    (capi.TYPE_F16, 2048, 41000, (24, 49)),
    (capi.TYPE_Q8_0, 3616, 5000, (17, 33, 64)),       # 57 steps, 313 row tiles, K splits
    (capi.TYPE_Q8_0, 8224, 2101, (25, 48)),            # 129 steps, long K, ragged N
    (capi.TYPE_Q8_0, 3136, 16500, (2, 16)),
    (capi.TYPE_Q8_0, 2048, 56400, (9, 33, 49)),       # twenty tiles a workgroup
    (capi.TYPE_Q4_0, 3168, 4200, (17, 64)),
    (capi.TYPE_Q4_0, 5152, 2060, (18, 33)),
    (capi.TYPE_Q4_0, 2048, 51300, (5, 32, 50)),
    (capi.TYPE_Q4_K, 2048, 51300, (7, 30, 64)),
    (capi.TYPE_F16, 2048, 51300, (24, 49)),
]

# Shapes of the list above on which other kernels are faster: short K at 257..1024
# row tiles, few row tiles, up to four rows of short K, workgroups that leave a
# round half empty.  They are held to the oracle on the route they take.
OTHER_ROUTE = {
    (capi.TYPE_Q8_0, 2080, 5000): (17, 33, 64),
    (capi.TYPE_Q8_0, 4640, 1613): (25, 48),
    (capi.TYPE_Q8_0, 2048, 16500): (2,),
    (capi.TYPE_Q8_0, 2048, 41000): (9, 33, 49),
    (capi.TYPE_Q4_0, 2144, 4200): (17, 64),
    (capi.TYPE_Q4_0, 5152, 1530): (18, 33),
    (capi.TYPE_Q4_0, 2048, 41000): (5, 32, 50),
    (capi.TYPE_Q4_K, 2048, 41000): (7, 30, 64),
    (capi.TYPE_F16, 2048, 41000): (24,),
}


@pytest.mark.parametrize("type_id,k,n,ms", CASES, ids=[f"{capi.TYPE_NAMES[c[0]]}-{c[2]}x{c[1]}" for c in CASES])
def test_stream_linear(torch_cuda, hip_ctx, type_id, k, n, ms):
    torch = torch_cuda
    dev = torch.device("cuda:0")
    dense = type_id in (capi.TYPE_Q6_K, capi.TYPE_F16)
    canon = (_weights if dense else helpers.weights)(type_id, k, n, seed=k + n)
    mat = capi.Matrix(hip_ctx, type_id, k, n, canon, canon.nbytes, on_device=False)
    tol = DENSE_TOL if dense else DECODE_TOL
    rows = np.unique(np.concatenate([np.arange(0, n, max(1, n // 200)), np.arange(max(0, n - 40), n)])).astype(np.uint64)
    bias = (np.random.default_rng(n).standard_normal(n) * 0.02).astype(np.float32)
    bias_d = torch.from_numpy(bias).to(dev)
    try:
        for m in ms:
            plan = mat.plan(m)
            print(f"stream {capi.TYPE_NAMES[type_id]} {n}x{k} M={m}: {plan}", flush=True)
            assert ("stream_kernel" in plan) == (m not in OTHER_ROUTE.get((type_id, k, n), ())), plan
            x = helpers.activations(m, k, seed=m + k)
            x[:, ::61] *= 40.0
            x[m // 2] *= 1e-5
            xd = torch.from_numpy(x).to(dev)
            outs = []
            for _ in range(2):
                y = torch.full((m, n), float("nan"), dtype=torch.float32, device=dev)
                mat.linear(xd, y, m, bias=bias_d)
                torch.cuda.synchronize()
                outs.append(y.cpu().numpy())
            assert np.isfinite(outs[0]).all(), (m, plan)
            y = torch.full((m, n), float("nan"), dtype=torch.float32, device=dev)
            mat.linear_noalloc(xd, y, m, bias=bias_d)
            torch.cuda.synchronize()
            outs.append(y.cpu().numpy())
            for other in outs[1:]:
                assert np.array_equal(outs[0].view(np.uint32), other.view(np.uint32)), (m, plan)
            want = oracle.linear_row_list(type_id, canon, k, n, x, rows, bias=bias)
            got = outs[0][:, rows.astype(np.int64)]
            for r in range(m):
                assert helpers.rel_l2(got[r], want[r]) <= tol, (m, r, plan)
    finally:
        mat.release()


@pytest.mark.parametrize("k,m", [(3104, 20), (4064, 20), (4064, 40), (4064, 64), (3616, 33)])
def test_stream_f16_half_step(torch_cuda, hip_ctx, k, m):
    """F16 rows of an odd number of 32-blocks, their last step at the start, the
    end and the middle of a trip: an infinite weight in the last block reaches
    its own output as an infinity (not a NaN: the block past the row is left
    out, not multiplied by zeros) and no other."""
    torch = torch_cuda
    n = 4200
    canon = _weights(capi.TYPE_F16, k, n, seed=k)
    w = canon.view(np.float16).reshape(n, k)
    w[70, k - 1] = np.inf
    w[n - 1, k - 9] = -np.inf
    mat = capi.Matrix(hip_ctx, capi.TYPE_F16, k, n, canon, canon.nbytes, on_device=False)
    try:
        assert "stream_kernel" in mat.plan(m), mat.plan(m)
        x = helpers.activations(m, k, seed=m)
        x[:, k - 9] = x[:, k - 1] = 1.2345678      # hi and lo parts both non-zero
        rows = np.unique(np.concatenate([np.arange(0, n, 40), [70, n - 1]])).astype(np.uint64)
        y = torch.empty((m, n), dtype=torch.float32, device="cuda:0")
        mat.linear(torch.from_numpy(x).to("cuda:0"), y, m)
        torch.cuda.synchronize()
        got = y.cpu().numpy()
        assert (got[:, 70] == np.inf).all() and (got[:, n - 1] == -np.inf).all(), mat.plan(m)
        finite = rows[(rows != 70) & (rows != n - 1)]
        want = oracle.linear_row_list(capi.TYPE_F16, canon, k, n, x, finite)
        for r in range(m):
            assert helpers.rel_l2(got[r, finite.astype(np.int64)], want[r]) <= DENSE_TOL, (r, mat.plan(m))
    finally:
        mat.release()


@pytest.mark.parametrize("k,n,m,splits", [(18944, 3584, 64, 9), (18944, 3584, 40, 9), (8448, 11008, 40, 2),
                                          (2304, 6656, 64, 0), (4608, 4096, 40, 0), (3584, 37888, 48, 1)])
def test_stream_q4_k_split_lengths(torch_cuda, hip_ctx, k, n, m, splits):
    """Q4_K at 33..64 rows keeps one running sum a split: whole records round
    down where the GPU has room for one more split, and where a split would be
    over a sixteenth longer than the skinny kernel's that one stays (0)."""
    zeros = torch_cuda.zeros(n * (k // 256) * 144, dtype=torch_cuda.uint8, device="cuda:0")
    mat = capi.Matrix(hip_ctx, capi.TYPE_Q4_K, k, n, zeros, zeros.numel(), on_device=True)
    try:
        plan = mat.plan(m)
        assert ("stream_kernel" in plan) == (splits != 0), plan
        assert not splits or f" splits={splits}" in plan, plan
    finally:
        mat.release()


# (format, K, N, widths): long unsplit K, where a single running sum would show.
SUM_CASES = [
    (capi.TYPE_F16, 16384, 41000, (48, 64)),
    (capi.TYPE_F16, 16384, 51300, (24, 40)),
    (capi.TYPE_F16, 16384, 33000, (64,)),
]


@pytest.mark.parametrize("type_id,k,n,ms", SUM_CASES)
def test_stream_k_sum_in_levels(torch_cuda, hip_ctx, type_id, k, n, ms):
    """Relative L2 against float64 products at K = 16384 unsplit: 3e-7 = the
    split's truncation (1.2e-7) and a K sum in levels (about 1.8e-7), with a third
    to spare; one running sum of its 512 blocks is 4.3e-7."""
    torch = torch_cuda
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(k + n)
    w = torch.empty((n, k), dtype=torch.float16, device="cuda:0").normal_(0.0, 0.02, generator=gen)
    mat = capi.Matrix(hip_ctx, type_id, k, n, w.view(torch.uint8), n * k * 2, on_device=True)
    sample = torch.arange(0, n, n // 500, device="cuda:0")
    ws = w[sample].double().T.contiguous()
    try:
        for m in ms:
            plan = mat.plan(m)
            assert "stream_kernel" in plan and " splits=1 " in plan + " ", plan
            x = torch.randn((m, k), generator=gen, device="cuda:0")
            y = torch.empty((m, n), dtype=torch.float32, device="cuda:0")
            mat.linear(x, y, m)
            want = x.double() @ ws
            error = float((y[:, sample].double() - want).norm() / want.norm())
            print(f"levels {capi.TYPE_NAMES[type_id]} {n}x{k} M={m} {error:.2e}: {plan}", flush=True)
            assert error <= 3e-7, (m, error, plan)
    finally:
        mat.release()


def test_stream_outliers_keep_small_channels(torch_cuda, hip_ctx):
    """A few channels 1e4 times the rest: the error against the small channels'
    own share of the output stays at 1e-3 (f32 rounding of the outputs)."""
    torch = torch_cuda
    k, n, m = 2048, 16500, 24
    canon = helpers.weights(capi.TYPE_Q4_0, k, n, seed=5)
    mat = capi.Matrix(hip_ctx, capi.TYPE_Q4_0, k, n, canon, canon.nbytes, on_device=False)
    try:
        assert "stream_kernel" in mat.plan(m), mat.plan(m)
        x = helpers.activations(m, k, seed=6)
        channels = np.array([3, 700, 1999])
        x[:, channels] *= np.float32(1e4)
        small = x.copy()
        small[:, channels] = 0.0
        rows = np.arange(0, n, 37).astype(np.uint64)
        y = torch.empty((m, n), dtype=torch.float32, device="cuda:0")
        mat.linear(torch.from_numpy(x).to("cuda:0"), y, m)
        torch.cuda.synchronize()
        got = y.cpu().numpy()[:, rows.astype(np.int64)].astype(np.float64)
        want = oracle.linear_row_list(capi.TYPE_Q4_0, canon, k, n, x, rows).astype(np.float64)
        share = oracle.linear_row_list(capi.TYPE_Q4_0, canon, k, n, small, rows).astype(np.float64)
        for r in range(m):
            assert np.linalg.norm(got[r] - want[r]) <= 1e-3 * np.linalg.norm(share[r]), r
    finally:
        mat.release()


# (format, K, N, M): the matrices the streaming kernel takes from kernels that
# scale the activations per step or block -- from the wave-split kernel over f32
# rows, the fused one (256 MiB of codes, up to four rows) and the dense one.
BLOCK_CASES = [
    (capi.TYPE_Q8_0, 2048, 16500, 8),
    (capi.TYPE_Q8_0, 2048, 51300, 7),
    (capi.TYPE_Q8_0, 8224, 2101, 28),
    (capi.TYPE_Q8_0, 4096, 65600, 3),
    (capi.TYPE_Q4_0, 2112, 34000, 5),
    (capi.TYPE_Q4_0, 2048, 17000, 16),
    (capi.TYPE_Q4_K, 2304, 17000, 12),
    (capi.TYPE_Q4_K, 8448, 1530, 8),
    (capi.TYPE_Q6_K, 8448, 1530, 13),
    (capi.TYPE_Q6_K, 2048, 41000, 20),
    (capi.TYPE_Q6_K, 2304, 4200, 40),
    (capi.TYPE_Q6_K, 2304, 4200, 64),
    (capi.TYPE_F16, 2048, 51300, 24),
    (capi.TYPE_F16, 3104, 4200, 33),
    (capi.TYPE_F16, 8224, 1530, 64),
]


@pytest.mark.parametrize("type_id,k,n,m", BLOCK_CASES, ids=[f"{capi.TYPE_NAMES[c[0]]}-{c[2]}x{c[1]}-{c[3]}" for c in BLOCK_CASES])
def test_stream_keeps_blocks_beside_a_large_one(torch_cuda, hip_ctx, type_id, k, n, m):
    """A channel 1e7 times the rest whose weights are zero: the outputs are the
    other channels', and each row is within 6e-7 of the oracle -- the split's
    truncation (below 2^-21 of a value, 1.2e-7 in the mean square) and f32 sums
    (about 1.6e-7) with a factor of two; twice that in Q4_K, whose products are
    of codes 0..15, about twice the weights, before their offset comes off.
    Under one scale per row their low parts would be subnormal and the error
    2e-5."""
    torch = torch_cuda
    dense = type_id in (capi.TYPE_Q6_K, capi.TYPE_F16)
    if dense:
        canon = _weights(type_id, k, n, seed=k + n)
    else:
        canon = quant.synthetic_weights_device(type_id, k, n, k + n, torch.device("cuda:0"), 0.02).cpu().numpy().reshape(-1)
    rows_view = canon.reshape(n, -1)
    if type_id == capi.TYPE_F16:
        rows_view[:, :64] = 0
    elif type_id == capi.TYPE_Q6_K:
        rows_view[:, 208:210] = 0
    else:
        rows_view[:, :4 if type_id == capi.TYPE_Q4_K else 2] = 0
    mat = capi.Matrix(hip_ctx, type_id, k, n, canon, canon.nbytes, on_device=False)
    rows = np.unique(np.concatenate([np.arange(0, n, max(1, n // 200)), np.arange(n - 20, n)])).astype(np.uint64)
    try:
        plan = mat.plan(m)
        print(f"blocks {capi.TYPE_NAMES[type_id]} {n}x{k} M={m}: {plan}", flush=True)
        assert "stream_kernel" in plan, plan
        x = helpers.activations(m, k, seed=m + k)
        x[:, 5] = 1e7 * np.where(np.arange(m) % 2 == 0, 1.0, -1.0)
        y = torch.empty((m, n), dtype=torch.float32, device="cuda:0")
        mat.linear(torch.from_numpy(x).to("cuda:0"), y, m)
        torch.cuda.synchronize()
        got = y.cpu().numpy()[:, rows.astype(np.int64)]
        want = oracle.linear_row_list(type_id, canon, k, n, x, rows)
        errors = [helpers.rel_l2(got[r], want[r]) for r in range(m)]
        print(f"blocks error {max(errors):.2e}", flush=True)
        assert max(errors) <= (1.2e-6 if type_id == capi.TYPE_Q4_K else 6e-7), plan
    finally:
        mat.release()


@pytest.mark.parametrize("k,n,m,path,wsplit", [(2048, 20000, 20, 0, 0), (2048, 640, 24, 2, 0), (2048, 640, 40, 0, 1)],
                         ids=["stream", "skinny", "wsplit"])
def test_q4_k_block_sums_of_large_values(torch_cuda, hip_ctx, k, n, m, path, wsplit):
    """Runs of eight neighbours near 1e38: their sum is past f32's range, the
    scaled one is not, and neither is any output."""
    torch = torch_cuda
    canon = helpers.weights(capi.TYPE_Q4_K, k, n, seed=8)
    mat = capi.Matrix(hip_ctx, capi.TYPE_Q4_K, k, n, canon, canon.nbytes, on_device=False)
    try:
        hip_ctx.set_decode_path(path, 0, 0)
        hip_ctx.set_wsplit(wsplit, 0, 0, 0, 0, 1 if wsplit else 0)
        x = helpers.activations(m, k, seed=9)
        x[1, 64:72] = 1e38
        x[m - 1, 1000:1016] = -9e37
        rows = np.arange(0, n, max(1, n // 200)).astype(np.uint64)
        y = torch.empty((m, n), dtype=torch.float32, device="cuda:0")
        mat.linear(torch.from_numpy(x).to("cuda:0"), y, m)
        torch.cuda.synchronize()
        got = y.cpu().numpy()
        assert np.isfinite(got).all(), mat.plan(m)
        want = oracle.linear_row_list(capi.TYPE_Q4_K, canon, k, n, x, rows)
        for r in range(m):
            assert helpers.rel_l2(got[r, rows.astype(np.int64)], want[r]) <= DECODE_TOL, (r, mat.plan(m))
    finally:
        hip_ctx.set_decode_path(0, 0, 0)
        hip_ctx.set_wsplit(0, 0, 0, 0, 0, 0)
        mat.release()


# (format, K, N of the fused gate|up, widths): one and two tiles per wave,
# eight waves, a last workgroup short of tiles, an odd count of gate tiles;
# the Q8_0 rows at 2000..4096 row tiles and 17..32 rows sum their two K splits
# in one workgroup (33 steps: unequal halves).
SWIGLU_CASES = [
    (capi.TYPE_Q8_0, 2112, 32 * 1001, (17, 32)),
    (capi.TYPE_Q8_0, 2048, 32 * 1301, (2, 16, 20, 31, 64)),
    (capi.TYPE_Q8_0, 2112, 32 * 997, (5, 40)),
    (capi.TYPE_Q8_0, 3616, 32 * 2048, (25, 49)),
    (capi.TYPE_Q4_0, 2048, 32 * 1301, (3, 18, 33, 64)),
    (capi.TYPE_Q4_0, 2112, 32 * 999, (16, 47)),
    (capi.TYPE_Q4_K, 2304, 32 * 1283, (9, 32, 64)),
    (capi.TYPE_Q4_K, 2304, 32 * 1033, (16, 48)),
    (capi.TYPE_Q8_0, 2112, 32 * 1765, (3, 16, 17, 32, 40, 64)),
    (capi.TYPE_Q4_0, 2048, 32 * 1651, (3, 18, 33, 64)),
    (capi.TYPE_Q4_K, 2304, 32 * 1651, (9, 32, 64)),
]


@pytest.mark.parametrize("type_id,k,n,ms", SWIGLU_CASES,
                         ids=[f"{capi.TYPE_NAMES[c[0]]}-{c[2]}x{c[1]}" for c in SWIGLU_CASES])
def test_stream_swiglu_bits(torch_cuda, hip_ctx, type_id, k, n, ms):
    """The SwiGLU in the linear's launch: the bits of the linear followed by
    air_hip_silu_mul, and no write past the output."""
    torch = torch_cuda
    lib = capi.lib()
    h = hip_ctx.handle
    f = n // 2
    canon = helpers.weights(type_id, k, n, seed=k + n)
    mat = capi.Matrix(hip_ctx, type_id, k, n, canon, canon.nbytes, on_device=False)
    bias = torch.from_numpy((np.random.default_rng(n).standard_normal(n) * 0.3).astype(np.float32)).to("cuda:0")
    try:
        for m in ms:
            x = helpers.activations(m, k, seed=m + k)
            x[:, ::61] *= 40.0
            x[m // 2] *= 1e-5
            xd = torch.from_numpy(x).to("cuda:0")
            for b in (None, bias):
                bp = b.data_ptr() if b is not None else None
                lin = torch.empty((m, n), dtype=torch.float32, device="cuda:0")
                want = torch.empty((m, f), dtype=torch.float32, device="cuda:0")
                capi.check(lib.air_hip_linear(h, mat.handle, xd.data_ptr(), lin.data_ptr(), bp, m, capi.LINEAR_DECODE))
                capi.check(lib.air_hip_silu_mul(h, lin.data_ptr(), want.data_ptr(), m, f))
                got = torch.full((m + 1, f), -7.0, dtype=torch.float32, device="cuda:0")
                capi.check(lib.air_hip_linear_epilogue(h, mat.handle, xd.data_ptr(), m, got.data_ptr(), bp,
                                                       capi.EPILOGUE_SWIGLU, None, None, 0.0, capi.LINEAR_DECODE))
                torch.cuda.synchronize()
                case = (m, b is not None, mat.plan(m))
                assert np.array_equal(got[:m].cpu().numpy().view(np.uint32), want.cpu().numpy().view(np.uint32)), case
                assert bool((got[m] == -7.0).all()), case
    finally:
        mat.release()


@pytest.mark.parametrize("type_id,k,n,m", [(capi.TYPE_Q6_K, 8448, 1530, 13), (capi.TYPE_F16, 3104, 4200, 33),
                                           (capi.TYPE_Q8_0, 2048, 16500, 5)])
@pytest.mark.parametrize("reserved", [False, True], ids=["unreserved", "reserved"])
def test_stream_first_call_under_capture(torch_cuda, reserved, type_id, k, n, m):
    """A linear whose first call is recorded into a graph allocates nothing
    there: without a reserve it takes the kernel it had before the streaming
    one (no scratch), after one the streaming kernel, and replays repeat."""
    torch = torch_cuda
    dev = torch.device("cuda:0")
    main = torch.cuda.current_stream(dev)
    dense = type_id in (capi.TYPE_Q6_K, capi.TYPE_F16)
    canon = (_weights if dense else helpers.weights)(type_id, k, n, seed=k + n)
    ctx = capi.Context(0, main.cuda_stream)
    mat = capi.Matrix(ctx, type_id, k, n, canon, canon.nbytes, on_device=False)
    graph = torch.cuda.CUDAGraph()
    try:
        assert "stream_kernel" in mat.plan(m), mat.plan(m)
        x = helpers.activations(m, k, seed=m + k)
        xd = torch.from_numpy(x).to(dev)
        y = torch.full((m, n), float("nan"), dtype=torch.float32, device=dev)
        if reserved:
            ctx.reserve(k, m)
        generation = ctx.stats()["workspace_generation"]
        capture = torch.cuda.Stream(dev)
        ctx.set_stream(capture.cuda_stream)
        with torch.cuda.graph(graph, stream=capture):
            mat.linear(xd, y, m)
        ctx.set_stream(main.cuda_stream)
        assert ctx.stats()["workspace_generation"] == generation
        eager = torch.empty((m, n), dtype=torch.float32, device=dev)
        mat.linear_noalloc(xd, eager, m)          # the streaming kernel's bits
        rows = np.arange(0, n, max(1, n // 200)).astype(np.uint64)
        want = oracle.linear_row_list(type_id, canon, k, n, x, rows)
        first = None
        for _ in range(3):
            y.fill_(float("nan"))
            graph.replay()
            mat.linear(xd, torch.empty((m, n), dtype=torch.float32, device=dev), m)   # eager work between
            torch.cuda.synchronize()
            got = y.cpu().numpy()
            first = got if first is None else first
            assert np.array_equal(got.view(np.uint32), first.view(np.uint32))
            if reserved:
                assert np.array_equal(got.view(np.uint32), eager.cpu().numpy().view(np.uint32))
            assert helpers.rel_l2(got[:, rows.astype(np.int64)], want) <= (DENSE_TOL if dense else DECODE_TOL)
    finally:
        torch.cuda.synchronize()
        graph = None
        mat.release()
        ctx.close()
