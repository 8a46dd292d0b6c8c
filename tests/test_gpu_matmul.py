"""Device matmul with f64 accumulation (la.matmul la/la.v:38-55, gate_matmul
autograd/gates_blas.v:6-23), the unquantized Linear forward and
LinearGate.backward (nn/gates/layers/linear.v:57-79) against the CPU oracle.

Bar: the device sums the same f64 products in another order, so the f64 sums
agree to ~1e-16 relative and the results rounded to f32 agree except where a
sum lies that close to a rounding boundary: at most one unit in the last
place, on a tiny fraction of elements (far inside the 1e-5 relative tolerance
of the f32 outputs of this path).  Integer-valued operands make every order
exact, and there the comparison is bit for bit at full size."""
import numpy as np
import pytest

import oracle
from helpers import CPU_THREADS, dev
from vtl_amd import capi
from vtl_amd.layers import (linear_backward_hip_f32, linear_forward_hip_exact, matmul_gate_backward_hip,
                            matmul_hip_host)
from vtl_amd.tensor import colsum_hip, linear_backward_hip, linear_hip, matmul_hip

pytestmark = pytest.mark.gpu


def ulp_diff(a, b):
    it = np.int32 if a.dtype == np.float32 else np.int64
    return np.abs(a.view(it).astype(np.int64) - b.view(it).astype(np.int64))


def assert_close_to_oracle(got, want, abs_products=None):
    assert got.shape == want.shape and got.dtype == want.dtype
    if got.dtype == np.float32:
        d = ulp_diff(got, want)
        assert d.max() <= 1, f"max ulp distance {d.max()}"
        assert (d > 0).mean() < 1e-3, f"{(d > 0).mean():.2e} of the elements differ"
    else:
        # f64 results: 2^-52 per operation over the K-term sum of |a||b|
        assert np.all(np.abs(got - want) <= 1e-13 * abs_products)


def run_matmul(A, B, ta, tb):
    a, b = dev(A), dev(B)
    c = matmul_hip(a, b, ta, tb)
    out = c.cpu()
    for t in (a, b, c):
        t.release()
    return out


SHAPES = [(1, 1, 1), (2, 3, 4), (2, 2, 2), (17, 33, 65), (64, 256, 784), (128, 128, 16), (130, 70, 250),
          (256, 1024, 96), (1, 512, 300), (300, 1, 77), (513, 255, 1030)]


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
def test_matmul_shapes_and_layouts(hip, dt, ta, tb):
    rng = np.random.default_rng(21)
    for (M, N, K) in SHAPES:
        A = rng.standard_normal((K, M) if ta else (M, K)).astype(dt)
        B = rng.standard_normal((N, K) if tb else (K, N)).astype(dt)
        print("matmul", dt.__name__, ta, tb, M, N, K, flush=True)
        got = run_matmul(A, B, ta, tb)
        want = oracle.matmul(A, B, ta, tb, threads=CPU_THREADS)
        absprod = None
        if dt == np.float64:
            absprod = np.abs(A.T if ta else A) @ np.abs(B.T if tb else B)
        assert_close_to_oracle(got, want, absprod)


@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_split_k_paths(hip, dt, knobs):
    """Few output tiles and a long K slice K over the grid; forced slice counts cover
    ragged K, edge tiles and the unsplit fallback."""
    rng = np.random.default_rng(27)
    cases = [(256, 4096, 11008, False, False, None), (256, 1024, 4096, False, True, None),
             (64, 64, 2048, True, False, None), (100, 70, 1000, False, True, "3"), (128, 192, 4096, True, True, "5"),
             (33, 65, 777, False, False, "16"), (64, 128, 96, False, True, "4")]
    for (M, N, K, ta, tb, force) in cases:
        if force is None:
            knobs.delenv("VTL_HIP_MATMUL_SPLITS", raising=False)
        else:
            knobs.setenv("VTL_HIP_MATMUL_SPLITS", force)
        A = rng.standard_normal((K, M) if ta else (M, K)).astype(dt)
        B = rng.standard_normal((N, K) if tb else (K, N)).astype(dt)
        print("split-K", dt.__name__, M, N, K, ta, tb, force, flush=True)
        got = run_matmul(A, B, ta, tb)
        want = oracle.matmul(A, B, ta, tb, threads=CPU_THREADS)
        absprod = np.abs(A.T if ta else A).astype(np.float64) @ np.abs(B.T if tb else B).astype(np.float64)
        assert_close_to_oracle(got, want, absprod)
        # integer-valued operands: bit for bit whatever the slicing
        Ai, Bi = np.rint(A * 4).astype(dt), np.rint(B * 4).astype(dt)
        exact = (Ai.T if ta else Ai).astype(np.float64) @ (Bi.T if tb else Bi).astype(np.float64)
        assert np.array_equal(run_matmul(Ai, Bi, ta, tb), exact.astype(dt))
    # the Linear form keeps bias and ReLU after the sliced sum
    knobs.delenv("VTL_HIP_MATMUL_SPLITS", raising=False)
    x = rng.standard_normal((128, 4096)).astype(dt)
    w = (rng.standard_normal((256, 4096)) * 0.05).astype(dt)
    b = rng.standard_normal(256).astype(dt)
    xd, wd, bd = dev(x), dev(w), dev(b.reshape(1, -1))
    y = linear_hip(xd, wd, bd, relu=True)
    ref = oracle.matmul(x, w, False, True) + b
    assert_close_to_oracle(y.cpu(), np.where(ref < 0, dt(0), ref).astype(dt),
                           np.abs(x).astype(np.float64) @ np.abs(w.T).astype(np.float64) + np.abs(b))
    for t in (xd, wd, bd, y):
        t.release()


# K cut for the last round's tiles alone (f64 with K along both operands' rows): rounds of 256 tiles before it, none (every
# tile is of the last), steps of K that do not divide and a rest of K, all it may be cut into; all values are whole, so
# every sum is exact
@pytest.mark.parametrize("slices", ["-2", "-5", "-8"])
@pytest.mark.parametrize("mnk", [(130, 8301, 113), (301, 7200, 96), (65, 63, 47), (64, 16385, 160), (4, 16449, 769)])
def test_last_round_cut_by_k(hip, slices, mnk, knobs):
    knobs.setenv("VTL_HIP_MATMUL_TILE", "5")
    knobs.setenv("VTL_HIP_MATMUL_SPLITS", slices)
    M, N, K = mnk
    rng = np.random.default_rng(M + N + K)
    A, B, bias = (rng.integers(-9, 10, shape).astype(np.float64) for shape in ((M, K), (N, K), (N,)))
    exact = A @ B.T
    assert np.array_equal(run_matmul(A, B, False, True), exact)
    x, w, b = dev(A), dev(B), dev(bias)
    y = linear_hip(x, w, b, relu=True)
    assert np.array_equal(y.cpu(), np.maximum(exact + bias, 0))
    for t in (x, w, b, y):
        t.release()


# (the shapes that only f64 with K along both operands' rows has, and the others at the edges of the largest tiles, and
# of long rows)
@pytest.mark.parametrize("shape", ["4", "5", "6"])
@pytest.mark.parametrize("mnk", [(64, 64, 16), (65, 63, 113), (129, 130, 47), (127, 2, 33), (2, 129, 300), (200, 70, 64),
                                 (3, (1 << 22) + 1, 5)])
def test_large_shapes_at_their_edges(hip, shape, mnk, knobs):
    knobs.setenv("VTL_HIP_MATMUL_TILE", shape)
    M, N, K = mnk
    rng = np.random.default_rng(M + N + K)
    bias = rng.integers(-9, 10, N)
    for dt in (np.float32, np.float64):
        for ta, tb in [(False, False), (False, True), (True, False), (True, True)][:2 if N > 1 << 20 else 4]:
            A = rng.integers(-9, 10, (K, M) if ta else (M, K)).astype(dt)
            B = rng.integers(-9, 10, (N, K) if tb else (K, N)).astype(dt)
            exact = (A.T if ta else A).astype(np.float64) @ (B.T if tb else B).astype(np.float64)
            assert np.array_equal(run_matmul(A, B, ta, tb), exact.astype(dt)), (dt, ta, tb)
            if not ta and tb:
                x, w, b = dev(A), dev(B), dev(bias.astype(dt))
                y = linear_hip(x, w, b, relu=True)
                assert np.array_equal(y.cpu(), np.maximum(exact + bias, 0).astype(dt)), dt
                for t in (x, w, b, y):
                    t.release()


# What K has beyond steps of 16 is the first step, which loads elements of the second that it clears: around one step, as
# many as are in flight (2 or 4) and one wave's or eight waves' share of them, with K in one piece and cut.  Whole values, exact
# sums; a row of A meets an infinity in the elements that two steps load, which twice nothing must not turn into a NaN.
@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("shape", ["1", "2", "3", "4", "5", "6"])
def test_k_of_no_whole_steps(hip, shape, dt, knobs):
    knobs.setenv("VTL_HIP_MATMUL_TILE", shape)
    rng = np.random.default_rng(int(shape))
    M, N = 35, 69
    for K in (1, 15, 16, 17, 31, 32, 33, 47, 49, 63, 64, 65, 113, 127, 129, 143, 255, 257, 511, 513, 525):
        for slices in ("0", "2") if K >= 64 else ("0",):
            knobs.setenv("VTL_HIP_MATMUL_SPLITS", slices)
            for ta, tb in [(False, False), (False, True), (True, False), (True, True)]:
                A = rng.integers(-9, 10, (M, K)).astype(dt)
                B = rng.integers(1, 10, (K, N)).astype(dt)
                A[3, :] = 1
                A[3, min(K - 1, K % 16 + 2)] = np.inf
                A[4, 0] = np.inf
                A[4, 1:] = 2
                exact = A.astype(np.float64) @ B.astype(np.float64)
                got = run_matmul(np.ascontiguousarray(A.T) if ta else A, np.ascontiguousarray(B.T) if tb else B, ta, tb)
                assert np.array_equal(got, exact.astype(dt)), (K, slices, ta, tb)


# Either side of where 32-bit offsets end: rows of C (64 to a wave), rows with K along them (64), rows with K across (16).  Many
# rows, and K across many, end nowhere.  Whole values: sums are exact, and so is their rounding.
@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("case", ["many rows", "long K across", "long K along", "long rows of C", "long rows of B"])
def test_products_at_the_end_of_32_bit_offsets(hip, case, dt):
    along, across = ((1 << 32) - 1) // (64 * np.dtype(dt).itemsize), ((1 << 32) - 1) // (16 * np.dtype(dt).itemsize)
    rng = np.random.default_rng(len(case))
    for M, N, K, ta, tb in {"many rows": [((1 << 22) + 1, 3, 5, False, True), ((1 << 22) + 1, 3, 18, False, False)],
                            "long K across": [(3, 5, (1 << 22) + 1, True, False), (34, 2, along + 1, True, False)],
                            "long K along": [(3, 2, along, False, True), (2, 3, along + 1, False, True), (2, 2, along + 1, False, False)],
                            "long rows of C": [(34, along, 2, False, True), (34, along + 1, 2, False, True)],
                            "long rows of B": [(2, across, 3, False, False), (2, across + 1, 3, False, False)]}[case]:
        print(case, M, N, K, ta, tb, flush=True)
        A = rng.integers(-9, 10, (K, M) if ta else (M, K), dtype=np.int8).astype(dt)
        B = rng.integers(-9, 10, (N, K) if tb else (K, N), dtype=np.int8).astype(dt)
        got = run_matmul(A, B, ta, tb)
        exact = (A.T if ta else A).astype(np.float64) @ (B.T if tb else B).astype(np.float64)
        assert np.array_equal(got, exact.astype(dt)), (M, N, K, ta, tb)


@pytest.mark.parametrize("tile", ["64", "128"])
def test_forced_tile_sizes(hip, tile, knobs):
    """VTL_HIP_MATMUL_TILE forces the 64x64 or the 128x128 tile kernel: whole and ragged
    tiles, all four layouts, both give the oracle's result (integers bit for bit)."""
    knobs.setenv("VTL_HIP_MATMUL_TILE", tile)
    rng = np.random.default_rng(int(tile))
    for (M, N, K, ta, tb) in [(256, 384, 128, False, True), (300, 200, 96, True, False), (129, 65, 260, True, True),
                              (1, 1, 1, False, False), (640, 512, 64, False, False)]:
        A = rng.standard_normal((K, M) if ta else (M, K)).astype(np.float32)
        B = rng.standard_normal((N, K) if tb else (K, N)).astype(np.float32)
        got = run_matmul(A, B, ta, tb)
        want = oracle.matmul(A, B, ta, tb, threads=CPU_THREADS)
        absprod = np.abs(A.T if ta else A).astype(np.float64) @ np.abs(B.T if tb else B).astype(np.float64)
        assert_close_to_oracle(got, want, absprod)
        Ai, Bi = np.rint(A * 4).astype(np.float32), np.rint(B * 4).astype(np.float32)
        exact = (Ai.T if ta else Ai).astype(np.float64) @ (Bi.T if tb else Bi).astype(np.float64)
        assert np.array_equal(run_matmul(Ai, Bi, ta, tb), exact.astype(np.float32))


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("shape", ["1", "2", "3", "4", "5"])
def test_direct_shapes_at_their_edges(hip, shape, dt, knobs):
    """Every shape of the kernel that loads operands straight from memory, all four layouts: single
    rows and columns, pairs that end inside and at the edge of a tile, one element of K, part of
    a step, whole steps for some of the waves only, one step more than the loads in flight, K in
    slices with a part of a step left.  Integers bit for bit."""
    knobs.setenv("VTL_HIP_MATMUL_TILE", shape)
    rng = np.random.default_rng(100 + int(shape))
    for (M, N, K, splits) in [(1, 1, 1, None), (1, 33, 15, None), (31, 1, 16, None), (2, 3, 17, None),
                              (32, 64, 64, None), (33, 65, 79, None), (63, 127, 257, None), (65, 129, 145, None),
                              (64, 128, 530, None), (5, 70, 1003, "3"), (130, 31, 1024, "5")]:
        if splits is None:
            knobs.delenv("VTL_HIP_MATMUL_SPLITS", raising=False)
        else:
            knobs.setenv("VTL_HIP_MATMUL_SPLITS", splits)
        for ta, tb in [(False, False), (False, True), (True, False), (True, True)]:
            A = rng.standard_normal((K, M) if ta else (M, K)).astype(dt)
            B = rng.standard_normal((N, K) if tb else (K, N)).astype(dt)
            print("direct", shape, dt.__name__, M, N, K, splits, ta, tb, flush=True)
            absprod = np.abs(A.T if ta else A).astype(np.float64) @ np.abs(B.T if tb else B).astype(np.float64)
            assert_close_to_oracle(run_matmul(A, B, ta, tb), oracle.matmul(A, B, ta, tb, threads=CPU_THREADS), absprod)
            Ai, Bi = np.rint(A * 4).astype(dt), np.rint(B * 4).astype(dt)
            exact = (Ai.T if ta else Ai).astype(np.float64) @ (Bi.T if tb else Bi).astype(np.float64)
            assert np.array_equal(run_matmul(Ai, Bi, ta, tb), exact.astype(dt))


def test_short_products_on_two_streams_do_not_meet(hip):
    """Products with K below 2048 need nothing of the library's: two threads, a non-blocking stream each,
    many products under way at once, every result exact."""
    import ctypes as C
    import threading
    hiprt = C.CDLL("libamdhip64.so")
    shapes = [(64, 256, 784), (16, 256, 1024), (64, 256, 2000)]
    rng = np.random.default_rng(31)
    work = []
    for _ in range(2):
        stream = C.c_void_p()
        assert hiprt.hipStreamCreateWithFlags(C.byref(stream), C.c_uint(1)) == 0
        jobs = []
        for m, n, k in shapes:
            a, b = rng.integers(-8, 9, (m, k)).astype(np.float32), rng.integers(-8, 9, (k, n)).astype(np.float32)
            outs = [dev(np.zeros((m, n), np.float32)) for _ in range(8)]
            jobs.append((m, n, k, dev(a), dev(b), outs, (a.astype(np.float64) @ b).astype(np.float32)))
        work.append((stream, jobs))
    capi.call("vtl_hip_sync")
    failed = []

    def products(stream, jobs):
        try:
            capi.call("vtl_hip_set_device", 0)
            capi.call("vtl_hip_set_stream", stream)
            for i in range(8):
                for m, n, k, a, b, outs, _ in jobs:
                    capi.call("vtl_hip_matmul_f32", a.ptr, b.ptr, outs[i].ptr, m, n, k, 0, 0)
            capi.call("vtl_hip_sync")
        except Exception as e:      # noqa: BLE001 - reported by the test
            failed.append(e)

    threads = [threading.Thread(target=products, args=w) for w in work]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed
    for stream, jobs in work:
        for m, n, k, a, b, outs, want in jobs:
            for o in outs:
                assert np.array_equal(o.cpu(), want), (m, n, k)
            for t in (a, b, *outs):
                t.release()
        assert hiprt.hipStreamDestroy(stream) == 0


def test_reference_literals(hip):
    # la/la_test.v:30-37
    a = np.array([[1.0, 0], [0.0, 1]])
    b = np.array([[4.0, 1], [2.0, 2]])
    assert np.array_equal(matmul_hip_host(a, b), b)
    assert np.array_equal(matmul_hip_host(a.astype(np.float32), b.astype(np.float32)), b.astype(np.float32))
    # la/la_test.v:39-57: rank-3 and vector operands are refused
    with pytest.raises(ValueError):
        matmul_hip_host(np.zeros((2, 2, 4)), np.zeros((2, 4, 2)))
    with pytest.raises(ValueError):
        matmul_hip_host(a, np.array([1.0, 2]))
    with pytest.raises(ValueError, match="Invalid shapes for matrix multiplication"):
        matmul_hip_host(np.zeros((2, 3)), np.zeros((2, 3)))
    # benchmarks/vs_numpy/matmul_bench.v:28-33 at its largest size, against exact integers
    n = 512
    i, j = np.indices((n, n))
    ai, bi = (i + j) % 7, (i * j) % 5
    got = matmul_hip_host(ai * 0.01, bi * 0.02)
    want_int = ai.astype(np.int64) @ bi.astype(np.int64)
    assert np.all(np.abs(got - want_int * 2e-4) <= 1e-12 * np.maximum(want_int, 1))


@pytest.mark.parametrize("M,N,K,ta,tb", [(4096, 4096, 4096, False, True), (4096, 4096, 4096, False, False),
                                         (2048, 4096, 1024, True, False), (1000, 1500, 2100, True, True),
                                         (256, 11008, 4096, False, True)])
def test_integer_valued_operands_exact_at_full_size(hip, M, N, K, ta, tb):
    """Operands in [-8, 8]: every partial sum is an integer below 2^24, so any
    summation order gives the same f32 and f64; numpy's f64 BLAS supplies it."""
    rng = np.random.default_rng(22)
    Ai = rng.integers(-8, 9, (K, M) if ta else (M, K)).astype(np.float64)
    Bi = rng.integers(-8, 9, (N, K) if tb else (K, N)).astype(np.float64)
    want = (Ai.T if ta else Ai) @ (Bi.T if tb else Bi)
    assert np.abs(want).max() < 2 ** 24
    print("exact f32", M, N, K, ta, tb, flush=True)
    got32 = run_matmul(Ai.astype(np.float32), Bi.astype(np.float32), ta, tb)
    assert np.array_equal(got32, want.astype(np.float32))
    if M * N <= 2048 * 4096:
        print("exact f64", M, N, K, ta, tb, flush=True)
        assert np.array_equal(run_matmul(Ai, Bi, ta, tb), want)


def test_full_size_random_against_oracle_rows(hip):
    """4096^3 f32 with normal operands; the oracle restates a band of rows."""
    rng = np.random.default_rng(23)
    M = N = K = 4096
    A = rng.standard_normal((M, K)).astype(np.float32)
    W = rng.standard_normal((N, K)).astype(np.float32)
    got = run_matmul(A, W, False, True)
    rows = np.r_[0:24, 2040:2056, 4072:4096]
    want = oracle.matmul(A[rows], W, False, True, threads=CPU_THREADS)
    assert_close_to_oracle(got[rows], want)
    # linearity in the first operand holds exactly for a power-of-two factor
    got2 = run_matmul(A * np.float32(0.25), W, False, True)
    assert np.array_equal(got2, got * np.float32(0.25))


@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_linear_forward_with_bias_and_relu(hip, dt):
    rng = np.random.default_rng(24)
    for (M, N, K) in [(1, 2, 3), (64, 256, 784), (33, 130, 257), (256, 1024, 512)]:
        x = rng.standard_normal((M, K)).astype(dt)
        w = (rng.standard_normal((N, K)) * 0.05).astype(dt)
        b = rng.standard_normal(N).astype(dt)
        if dt == np.float32:
            want = oracle.linear_f32_via_f64(x, w, b)
        else:
            want = oracle.matmul(x, w, False, True) + b
        absprod = np.abs(x).astype(np.float64) @ np.abs(w.T).astype(np.float64) + np.abs(b)
        assert_close_to_oracle(linear_forward_hip_exact(x, w, b), want, absprod)
        xd, wd, bd = dev(x), dev(w), dev(b.reshape(1, -1))
        y = linear_hip(xd, wd, bd, relu=True)
        assert_close_to_oracle(y.cpu(), np.where(want < 0, dt(0), want).astype(dt), absprod)
        y0 = linear_hip(xd, wd, None)
        want0 = oracle.matmul(x, w, False, True)
        assert_close_to_oracle(y0.cpu(), want0, absprod)
        for t in (xd, wd, bd, y, y0):
            t.release()
    # autograd_cuda/device_session_test.v:34-47 literals, CPU reference within 1e-9
    x = np.array([[1.0, 2.0, 3.0]])
    w = np.array([[0.1, 0.2, 0.3], [0.4, 0.5, 0.6]])
    b = np.array([[0.01, 0.02]])
    assert np.all(np.abs(linear_forward_hip_exact(x, w, b) - [[1.41, 3.22]]) < 1e-9)


@pytest.mark.parametrize("rows,cols", [(0, 5), (1, 1), (7, 3), (256, 4096), (300, 1001), (65536, 256),
                                       (100000, 4), (5000, 130), (64, 11008)])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_column_sums(hip, dt, rows, cols):
    rng = np.random.default_rng(25)
    x = rng.standard_normal((rows, cols)).astype(dt)
    xd = dev(x) if rows else None
    if rows == 0:
        from vtl_amd.tensor import HipTensor
        out = HipTensor.empty([1, cols], dt)
        capi.call("vtl_hip_colsum_f32" if dt == np.float32 else "vtl_hip_colsum_f64", None, 0, cols, out.ptr)
        assert not out.cpu().any()
        out.release()
        return
    s = colsum_hip(xd)
    got = s.cpu().reshape(-1)
    want = oracle.colsum(x)
    assert_close_to_oracle(got, want, np.abs(x).sum(axis=0))
    xd.release()
    s.release()


@pytest.mark.parametrize("cols", [1, 2, 3, 4, 5, 6, 7, 63, 64, 65, 66, 67, 68, 130])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_column_sums_of_few_rows(hip, guard_bands, dt, cols):
    """Where the last columns' loads begin before them: whole numbers, so every sum is exact; a tensor that ends where its memory does."""
    rng = np.random.default_rng(cols)
    for rows in (1, 15, 16, 17, 48, 49, 63, 64, 65, 112, 512):
        x = rng.integers(-1000, 1001, (rows, cols)).astype(dt)
        xd = dev(x)
        s = colsum_hip(xd)
        assert np.array_equal(s.cpu().reshape(-1), x.sum(axis=0)), (rows, cols)
        xd.release()
        s.release()


@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_linear_backward_against_oracle(hip, dt):
    rng = np.random.default_rng(26)
    for (M, N, K) in [(1, 2, 3), (64, 256, 784), (37, 130, 65), (256, 1024, 4096), (512, 4096, 1024)]:
        g = rng.standard_normal((M, N)).astype(dt)
        x = rng.standard_normal((M, K)).astype(dt)
        w = (rng.standard_normal((N, K)) * 0.05).astype(dt)
        print("backward", dt.__name__, M, N, K, flush=True)
        want = oracle.linear_backward(g, x, w, threads=CPU_THREADS)
        gd, xd, wd = dev(g), dev(x), dev(w)
        outs = linear_backward_hip(gd, xd, wd)
        g64, x64, w64 = np.abs(g).astype(np.float64), np.abs(x).astype(np.float64), np.abs(w).astype(np.float64)
        bounds = (g64 @ w64, g64.T @ x64, g64.sum(axis=0))
        for got_t, want_a, bnd in zip(outs, want, bounds):
            assert_close_to_oracle(got_t.cpu().reshape(want_a.shape), want_a, bnd)
        # gradients that are not required are not computed
        only_dw = linear_backward_hip(gd, xd, wd, need_dx=False, need_db=False)
        assert only_dw[0] is None and only_dw[2] is None
        assert np.array_equal(only_dw[1].cpu(), outs[1].cpu())
        for t in (gd, xd, wd, *outs, only_dw[1]):
            t.release()


@pytest.mark.parametrize("m,n,k", [(16, 2625, 3136), (64, 1024, 2688), (128, 1984, 1615), (128, 1646, 3609)])
def test_f64_weight_gradient_of_large_tiles(hip, m, n, k):
    # tiles of 64 x 128 that store pairs of doubles one behind the other: every bit of both has to arrive, each time
    rng = np.random.default_rng(m + n)
    g, x = rng.standard_normal((m, n)), rng.standard_normal((m, k))
    want, bound = g.T @ x, (m + 2) * 2.0 ** -53 * (np.abs(g).T @ np.abs(x))
    gd, xd, wd = dev(g), dev(x), dev(np.zeros((n, k)))
    print("weight gradient", m, n, k, flush=True)
    for _ in range(10):
        dw = linear_backward_hip(gd, xd, wd, need_dx=False, need_db=False)[1]
        assert np.all(np.abs(dw.cpu() - want) <= 2 * bound)
        dw.release()
    for t in (gd, xd, wd):
        t.release()


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("m,n,k", [(1, 2, 2), (1, 3, 17), (15, 33, 31), (16, 64, 32), (17, 65, 97), (33, 63, 130), (64, 4, 1030),
                                   (128, 1000, 70), (40, 2500, 65), (512, 66, 34), (513, 66, 34), (129, 1100, 1450)])
def test_gradients_in_one_launch(hip, knobs, dt, m, n, k):
    """Edges of the tiles, of the column sums' groups of four and 64, of a step of K, and of the rows that one launch
    sums; dX's K in one piece and in slices: as launch by launch, within the order of the sums."""
    rng = np.random.default_rng(m * n + k)
    g, x, w = (rng.standard_normal(s).astype(dt) for s in ((m, n), (m, k), (n, k)))
    gd, xd, wd = dev(g), dev(x), dev(w)
    bounds = (n * (np.abs(g).astype(np.float64) @ np.abs(w)), m * (np.abs(g).T.astype(np.float64) @ np.abs(x)),
              m * np.abs(g).astype(np.float64).sum(axis=0)[None])
    want = [g.astype(np.float64) @ w.astype(np.float64), g.T.astype(np.float64) @ x.astype(np.float64),
            g.astype(np.float64).sum(axis=0)[None]]
    for mode in ("0", "1"):
        knobs.setenv("VTL_HIP_BACKWARD_GROUP", mode)
        for need in ((True, True, True), (True, True, False), (False, True, True), (True, False, True)):
            print("gradients", dt.__name__, m, n, k, mode, need, flush=True)
            outs = linear_backward_hip(gd, xd, wd, *need)
            for o, exact, b in zip(outs, want, bounds):
                if o is not None:
                    # sums of m or n products in f64, numpy's too, and one rounding to the tensor's type
                    got = o.cpu().astype(np.float64)
                    assert np.all(np.abs(got - exact) <= 2.0 ** -52 * b + (np.abs(exact) * 2.0 ** -24 if dt == np.float32 else 0))
                    o.release()
    for t in (gd, xd, wd):
        t.release()


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (1, 2, 3), (17, 33, 65), (64, 64, 64), (40, 700, 64), (16, 256, 256), (64, 300, 300), (64, 256, 512)])
def test_small_gradients_from_the_host(hip, monkeypatch, dt, m, n, k):
    """Small layers, host to host.  (Here beside tests that name streams, so each operand goes up by itself; what goes up together is in
    test_gpu_null_stream.py.)"""
    monkeypatch.setenv("VTL_USE_HIP", "1")
    monkeypatch.setenv("VTL_HIP_BACKWARD", "1")
    rng = np.random.default_rng(m + n + k)
    g, x, w = (rng.integers(-8, 9, s).astype(dt) for s in ((m, n), (m, k), (n, k)))   # (whole numbers: every sum exact)
    for bias in (True, False):
        for _ in range(3):
            print("gradients from the host", dt.__name__, m, n, k, bias, flush=True)
            dx, dw, db = linear_backward_hip_f32(g, x, w, bias)
            assert np.array_equal(dx, g @ w) and np.array_equal(dw, g.T @ x)
            assert np.array_equal(db.reshape(-1), g.sum(axis=0) if bias else np.zeros(n))


@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_weight_gradient_over_the_weights(hip, knobs, dt):
    """dX is complete before dW is written: dW may take the place of W."""
    m, n, k = 64, 192, 160
    rng = np.random.default_rng(7)
    g, x, w = (rng.integers(-8, 9, s).astype(dt) for s in ((m, n), (m, k), (n, k)))   # (whole numbers: every sum exact)
    for mode in ("0", "1"):
        knobs.setenv("VTL_HIP_BACKWARD_GROUP", mode)
        gd, xd, wd, dx, db = dev(g), dev(x), dev(w), dev(np.zeros_like(x)), dev(np.zeros((1, n), dt))
        capi.call("vtl_hip_linear_backward_f32" if dt == np.float32 else "vtl_hip_linear_backward_f64", gd.ptr, xd.ptr, wd.ptr,
                  dx.ptr, wd.ptr, db.ptr, m, n, k)
        assert np.array_equal(dx.cpu(), g @ w) and np.array_equal(wd.cpu(), g.T @ x)
        assert np.array_equal(db.cpu().reshape(-1), g.sum(axis=0))
        for t in (gd, xd, wd, dx, db):
            t.release()


def test_linear_backward_host_entry(hip, monkeypatch):
    # operands of autograd_cuda/device_session_test.v:52-60; gradients worked by hand
    g = np.array([[1.0, 0.5]], np.float32)
    x = np.array([[1.0, 2.0, 3.0]], np.float32)
    w = np.array([[0.1, 0.2, 0.3], [0.4, 0.5, 0.6]], np.float32)
    monkeypatch.delenv("VTL_HIP_BACKWARD", raising=False)
    with pytest.raises(RuntimeError, match="VTL_HIP_BACKWARD"):
        linear_backward_hip_f32(g, x, w, True)
    monkeypatch.setenv("VTL_USE_HIP", "1")
    monkeypatch.setenv("VTL_HIP_BACKWARD", "1")
    d_in, d_w, d_b = linear_backward_hip_f32(g, x, w, True)
    assert d_in.shape == (1, 3) and d_w.shape == (2, 3) and d_b.shape == (1, 2)
    assert np.allclose(d_in, [[0.3, 0.45, 0.6]], rtol=1e-6)
    assert np.array_equal(d_w, [[1, 2, 3], [0.5, 1, 1.5]]) and np.array_equal(d_b, [[1, 0.5]])
    # the reference's CUDA test asks for 1e-6 agreement with the CPU gradients (device_session_test.v:62-80)
    want = oracle.linear_backward(g.astype(np.float64), x.astype(np.float64), w.astype(np.float64))
    got = linear_backward_hip_f32(g.astype(np.float64), x.astype(np.float64), w.astype(np.float64), True)
    for a, b in zip(got, want):
        assert np.all(np.abs(a.reshape(b.shape) - b) < 1e-6)
    _, _, zeros = linear_backward_hip_f32(g, x, w, False)
    assert zeros.shape == (1, 2) and not zeros.any()


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("where", ["dw", "dw and db", "db"])
def test_gradients_into_the_memory_of_w(hip, where, dt):
    """A program that drops its weights with the step lets dW, or db, take their place: dX is of the weights as they were.
    Whole values, so every sum is exact; large enough for results that launches write to the host themselves."""
    from vtl_amd.storage import host_array
    M, N, K = 64, 2048, 64
    rng = np.random.default_rng(31)
    grad, x, w0 = (rng.integers(-9, 10, shape).astype(dt) for shape in ((M, N), (M, K), (N, K)))
    arena, _ = host_array(N * K + N, np.dtype(dt))
    w, behind = arena[:N * K].reshape(N, K), arena[N * K:]
    w[:] = w0
    dx = np.zeros((M, K), dt)
    dw = w if "dw" in where else np.zeros((N, K), dt)
    db = w.reshape(-1)[:N] if where == "db" else behind
    capi.call("vtl_hip_linear_backward_host_f32" if dt == np.float32 else "vtl_hip_linear_backward_host_f64",
              grad.ctypes.data, x.ctypes.data, w.ctypes.data, dx.ctypes.data, dw.ctypes.data, db.ctypes.data, M, N, K)
    assert np.array_equal(dx, grad @ w0) and np.array_equal(dw, grad.T @ x) and np.array_equal(db, grad.sum(0))


def test_argument_errors(hip):
    from helpers import raw_device_buffer
    buf = raw_device_buffer(4096)
    p = buf.ptr
    assert capi.status("vtl_hip_matmul_f32", p, p, p, -1, 2, 2, 0, 0) == capi.ERR_INVALID_ARG
    assert capi.status("vtl_hip_matmul_f32", None, p, p, 2, 2, 2, 0, 0) == capi.ERR_INVALID_ARG
    assert capi.status("vtl_hip_matmul_f64", p, p, None, 2, 2, 2, 0, 0) == capi.ERR_INVALID_ARG
    assert capi.status("vtl_hip_matmul_f32", p, p, p, 0, 5, 3, 0, 0) == capi.OK
    assert capi.status("vtl_hip_colsum_f32", None, 4, 4, p) == capi.ERR_INVALID_ARG
    assert capi.status("vtl_hip_linear_backward_f32", None, p, p, p, p, p, 2, 2, 2) == capi.ERR_INVALID_ARG
    assert capi.status("vtl_hip_linear_backward_f32", p, p, None, p, None, None, 2, 2, 2) == capi.ERR_INVALID_ARG
    # K == 0: zeros (plus the bias for the Linear form)
    capi.call("vtl_hip_memset", p, 0xFF, 4096)
    capi.call("vtl_hip_matmul_f32", None, None, p, 3, 4, 0, 0, 0)
    from helpers import d2h
    assert not d2h(p, 12, np.float32).any()
    buf.release()


def test_matmul_gate_backward(hip, monkeypatch):
    """MatMulGate.backward (autograd/gates_blas.v:43-48): dA = g . B^T, dB = A^T . g."""
    monkeypatch.setenv("VTL_USE_HIP", "1")
    monkeypatch.setenv("VTL_HIP_BACKWARD", "1")
    rng = np.random.default_rng(28)
    for dt in (np.float32, np.float64):
        a = rng.standard_normal((37, 53)).astype(dt)
        b = rng.standard_normal((53, 29)).astype(dt)
        g = rng.standard_normal((37, 29)).astype(dt)
        da, db = matmul_gate_backward_hip(g, a, b)
        want_a = oracle.matmul(g, np.ascontiguousarray(b.T))
        want_b = oracle.matmul(np.ascontiguousarray(a.T), g)
        absa = np.abs(g).astype(np.float64) @ np.abs(b.T).astype(np.float64)
        absb = np.abs(a.T).astype(np.float64) @ np.abs(g).astype(np.float64)
        assert_close_to_oracle(da, want_a, absa)
        assert_close_to_oracle(db, want_b, absb)
    with pytest.raises(ValueError, match="Invalid shapes"):
        matmul_gate_backward_hip(np.zeros((3, 3)), np.zeros((3, 4)), np.zeros((5, 3)))


# Slices of K whose sums meet within their launch: every shape, tiles at the edges, one and many slices, a K on either side of where that begins, more
# tiles than there are counters, and the same launches again (the counters are left at zero).  Whole numbers: every order of the sums is exact.
@pytest.mark.parametrize("mnk", [(33, 65, 800), (1, 70, 1616), (64, 1, 2047), (100, 300, 3001), (17, 33, 799), (130, 129, 848), (1100, 1100, 800), (64, 256, 2000)])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_slices_that_meet_within_their_launch(hip, mnk, dt, knobs):
    m, n, k = mnk
    rng = np.random.default_rng(m * 3 + n * 5 + k)
    a, w = rng.integers(-8, 9, (m, k)).astype(dt), rng.integers(-8, 9, (n, k)).astype(dt)
    bias = rng.integers(-500, 500, n).astype(dt)
    want = (a.astype(np.int64) @ w.astype(np.int64).T).astype(dt)
    A, W, B, Wt = dev(a), dev(w), dev(bias), dev(np.ascontiguousarray(w.T))
    print(mnk, dt.__name__, flush=True)
    for tile in ("0", "1", "2", "3", "4", "5", "6"):
        knobs.setenv("VTL_HIP_MATMUL_TILE", tile)
        for splits in ("-1", "2", "7", "25"):
            knobs.setenv("VTL_HIP_MATMUL_SPLITS", splits)
            for _ in range(2):
                y = matmul_hip(A, Wt)
                assert np.array_equal(y.cpu(), want), (tile, splits)
                y.release()
            y = linear_hip(A, W, B, relu=True)
            assert np.array_equal(y.cpu(), np.maximum(want + bias, 0)), (tile, splits)
            y.release()
            assert np.array_equal(matmul_hip_host(a, np.ascontiguousarray(w.T)), want), (tile, splits)
    for t in (A, W, B, Wt):
        t.release()


# C in the memory of A or of B, K in slices: what the slices are made from has been read before anything is stored
@pytest.mark.parametrize("mnk", [(64, 256, 2000), (64, 64, 4096), (33, 65, 800)])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("over", ["a", "b"])
def test_products_over_their_operands(hip, mnk, dt, over, knobs):
    m, n, k = mnk
    rng = np.random.default_rng(m + n * 3 + k * 5)
    a, w = rng.integers(-8, 9, (m, k)).astype(dt), rng.integers(-8, 9, (n, k)).astype(dt)
    want = (a.astype(np.int64) @ w.astype(np.int64).T).astype(dt)
    name = "vtl_hip_linear_f32" if dt == np.float32 else "vtl_hip_linear_f64"
    print(mnk, dt.__name__, over, flush=True)
    knobs.setenv("VTL_HIP_MATMUL_TILE", "2")
    for splits in ("2", "7", "25"):
        knobs.setenv("VTL_HIP_MATMUL_SPLITS", splits)
        A, W = dev(a), dev(w)
        at = (A if over == "a" else W).ptr + 3 * dt().itemsize
        capi.call(name, A.ptr, W.ptr, None, at, m, n, k, 0)
        got = (A if over == "a" else W).cpu().reshape(-1)[3:3 + m * n].reshape(m, n)
        assert np.array_equal(got, want), splits
        A.release()
        W.release()
