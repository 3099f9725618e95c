"""GPU checks of the MFMA GEMM and the blocked factorizations against numpy (LAPACK)."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def banner(msg):
    print(f"[gpu-dense] {msg}", flush=True)


@pytest.mark.parametrize("ta", [False, True])
@pytest.mark.parametrize("tb", [False, True])
@pytest.mark.parametrize("shape", [(1, 1, 1), (17, 33, 5), (128, 128, 16), (300, 200, 1000), (130, 7, 5000)])
def test_dgemm(hip, ta, tb, shape):
    M, N, K = shape
    banner(f"dgemm {shape} ta={ta} tb={tb}")
    rng = np.random.default_rng(M + N + K)
    A = rng.standard_normal((K, M) if ta else (M, K))
    B = rng.standard_normal((N, K) if tb else (K, N))
    C0 = rng.standard_normal((M, N))
    ref = 0.5 * ((A.T if ta else A) @ (B.T if tb else B)) - 2.0 * C0
    got = hip.gemm(A, B, ta, tb, alpha=0.5, beta=-2.0, C=C0)
    scale = np.sqrt(K) * np.abs(A).max() * np.abs(B).max() + np.abs(C0).max()
    assert np.max(np.abs(got - ref)) <= 1e-14 * scale * 8


def test_sgemm(hip):
    banner("sgemm")
    rng = np.random.default_rng(3)
    A = rng.standard_normal((257, 300)); B = rng.standard_normal((300, 129))
    got = hip.gemm(A, B, f32=True)
    ref = A.astype(np.float32).astype(np.float64) @ B.astype(np.float32).astype(np.float64)
    assert np.max(np.abs(got - ref)) <= 1e-5 * np.sqrt(300) * 4


@pytest.mark.parametrize("n", [1, 5, 128, 129, 700])
def test_potrf(hip, n):
    banner(f"potrf n={n}")
    rng = np.random.default_rng(n)
    X = rng.standard_normal((n, n + 10))
    G = X @ X.T
    L, info = hip.potrf_lower(G)
    assert info == 0
    assert np.allclose(np.triu(L, 1), 0)
    ref = np.linalg.cholesky(G)
    assert np.max(np.abs(L - ref)) <= 1e-12 * np.abs(ref).max()
    # non-positive pivot is reported
    G2 = G.copy(); G2[n // 2, n // 2] = -1.0
    _, info2 = hip.potrf_lower(G2)
    assert info2 > 0


@pytest.mark.parametrize("upper", [False, True])
@pytest.mark.parametrize("unit", [False, True])
@pytest.mark.parametrize("n,nrhs", [(3, 5), (100, 37), (128, 64), (300, 1000), (700, 130), (200, 5000), (64, 4100)])
def test_trsm_left(hip, upper, unit, n, nrhs):
    banner(f"trsm_left n={n} nrhs={nrhs} upper={upper} unit={unit}")
    rng = np.random.default_rng(n * 3 + nrhs)
    T = rng.standard_normal((n, n)) * 0.1 + np.eye(n) * 2
    T = np.triu(T) if upper else np.tril(T)
    Teff = T.copy()
    if unit:
        np.fill_diagonal(Teff, 1.0)
    X = rng.standard_normal((n, nrhs))
    got = hip.trsm_left(T, X, upper, unit)
    ref = np.linalg.solve(Teff, X)
    assert np.max(np.abs(got - ref)) <= 1e-12 * np.abs(ref).max()


@pytest.mark.parametrize("upper", [False, True])
@pytest.mark.parametrize("unit", [False, True])
@pytest.mark.parametrize("n,nrhs", [(100, 16384), (128, 20000), (300, 16400), (1000, 16384)])
def test_trsm_left_wide(hip, upper, unit, n, nrhs):
    """Wide right-hand sides (the leaves' many-wavefront form): the solution matches LAPACK's, and
    on a graded triangle (an R factor of singular values falling over six decades, the triangles
    the Cholesky QR passes solve with) the solve stays backward stable: ||T X - B|| is at rounding
    level relative to ||T|| ||X|| (relative to ||B|| it can reach u cond(T), for LAPACK too)."""
    import scipy.linalg as sl
    banner(f"trsm_left wide n={n} nrhs={nrhs} upper={upper} unit={unit}")
    rng = np.random.default_rng(n + nrhs + 2 * upper + unit)
    T = rng.standard_normal((n, n)) * 0.1 + np.eye(n) * 2
    T = np.triu(T) if upper else np.tril(T)
    X = rng.standard_normal((n, nrhs))
    got = hip.trsm_left(T, X, upper, unit)
    ref = sl.solve_triangular(T, X, lower=not upper, unit_diagonal=unit)
    assert np.max(np.abs(got - ref)) <= 1e-12 * np.abs(ref).max()
    if unit:
        return
    # graded: R factor of a matrix with singular values 1 .. 1e-6
    q1, _ = np.linalg.qr(rng.standard_normal((2 * n, n)))
    q2, _ = np.linalg.qr(rng.standard_normal((n, n)))
    R = np.linalg.qr((q1 * np.geomspace(1.0, 1e-6, n)) @ q2.T, mode="r")
    G = R if upper else np.ascontiguousarray(R.T)
    got = hip.trsm_left(G, X, upper, False)
    # normwise backward error (substitution: 1e-17 and below here; LAPACK's dtrtrs alike)
    back = np.linalg.norm(G @ got - X) / (np.linalg.norm(G) * np.linalg.norm(got))
    assert back <= 1e-15, back


@pytest.mark.parametrize("lower_t", [False, True])
@pytest.mark.parametrize("n,rows", [(3, 5), (128, 64), (300, 1000), (700, 130), (200, 5000), (64, 4100)])
def test_trsm_right(hip, lower_t, n, rows):
    banner(f"trsm_right n={n} rows={rows} lower_t={lower_t}")
    rng = np.random.default_rng(n * 5 + rows)
    T = rng.standard_normal((n, n)) * 0.1 + np.eye(n) * 2
    T = np.tril(T) if lower_t else np.triu(T)
    Op = T.T if lower_t else T
    X = rng.standard_normal((rows, n))
    got = hip.trsm_right(T, X, lower_t)
    ref = np.linalg.solve(Op.T, X.T).T
    assert np.max(np.abs(got - ref)) <= 1e-12 * np.abs(ref).max()


@pytest.mark.parametrize("n", [4, 128, 300, 1000])
def test_lu_sign(hip, n):
    banner(f"lu_sign n={n}")
    rng = np.random.default_rng(n)
    Q, _ = np.linalg.qr(rng.standard_normal((n, n)))
    LU, s = hip.lu_sign(Q)
    L = np.tril(LU, -1) + np.eye(n)
    U = np.triu(LU)
    assert set(np.unique(s)) <= {-1.0, 1.0}
    assert np.max(np.abs(L @ U - (Q - np.diag(s)))) <= 1e-12 * n
    assert np.all(np.abs(np.diag(U)) >= 1.0 - 1e-12), "pivots have magnitude >= 1"


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("ta", [False, True])
@pytest.mark.parametrize("tb", [False, True])
def test_gemm_edges(hip, f32, ta, tb):
    """Sizes around the tiles, the K steps and the 16-byte units, with and without a workspace, on
    matrices inside larger arrays that start one element off and hold NaN around them. The bound is
    the a-priori one of a K-term dot product in any order, |err| <= (K + 2) u |A||B|."""
    dt, u = (np.float32, 2.0 ** -24) if f32 else (np.float64, 2.0 ** -53)
    rng = np.random.default_rng(11)
    for (M, N, K) in ((1, 1, 1), (1, 3, 2), (2, 1, 700), (3, 200, 1000), (64, 64, 16), (65, 129, 17), (130, 1, 300),
                      (127, 255, 31), (128, 128, 64), (257, 66, 1030), (600, 1026, 5)):
        banner(f"gemm {M}x{N}x{K} ta={ta} tb={tb} f32={f32}")
        A, B = rng.standard_normal((M, K)).astype(dt), rng.standard_normal((K, N)).astype(dt)
        C = rng.standard_normal((M, N)).astype(dt)

        def inside(X, pad):
            big = np.full(1 + X.shape[0] * (X.shape[1] + pad), np.nan, dt)
            big[1:].reshape(X.shape[0], -1)[:, :X.shape[1]] = X
            return hip.DeviceArray.from_host(big), X.shape[1] + pad

        want = 0.5 * (A.astype(np.float64) @ B.astype(np.float64)) - 2.0 * C.astype(np.float64)
        bound = (K + 4) * u * (np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64) + 2.0 * np.abs(C) + 1.0)
        dA, lda = inside(A.T if ta else A, 3)
        dB, ldb = inside(B.T if tb else B, 5)
        for work in (False, True):
            dC, ldc = inside(C, 1)
            ws = hip.workspace(hip.lib.exc_gemm_workspace(M, N, K))
            s = np.dtype(dt).itemsize
            hip.call("exc_sgemm" if f32 else "exc_dgemm", int(ta), int(tb), M, N, K, 0.5, dA.ptr + s, lda, dB.ptr + s,
                     ldb, -2.0, dC.ptr + s, ldc, ws.ptr if work else None, ws.nbytes if work else 0, None)
            hip.sync()
            got = dC.to_host()
            assert np.isnan(got[0])
            got = got[1:].reshape(M, ldc)
            assert np.isnan(got[:, N:]).all()
            assert (np.abs(got[:, :N] - want) <= bound).all(), (M, N, K, work)


@pytest.mark.parametrize("f32,M,N,K,longest", [
    (False, 500, 1000, 496, 64), (False, 1000, 1000, 992, 128), (False, 1000, 1000, 2000, 256),
    (False, 200, 600, 96, 16), (False, 843, 1365, 320, 80), (False, 364, 1027, 8000, 1008),
    (True, 584, 584, 5200, 336), (True, 996, 996, 14384, 1200), (True, 1202, 1202, 8000, 1152),
    (True, 2000, 2000, 20000, 2000), (True, 234, 234, 128, 16)])
def test_gemm_sum_length(hip, f32, M, N, K, longest):
    """The rounding error of a product grows with the terms of a running sum, so with a workspace K is split
    at least this far. All factors are one except the first of every row, 2^27 (2^56 in FP64): a running
    sum that starts there loses each later term (up to 7 at a time are less than half a unit of the last
    place), the others are whole numbers and exact, so the result shows the first sum's length."""
    dt, first = (np.float32, 2.0 ** 27) if f32 else (np.float64, 2.0 ** 56)
    banner(f"gemm sum length {M}x{N}x{K} f32={f32}")
    A = np.ones((M, K), dt)
    A[:, 0] = first
    dA, dB = hip.DeviceArray.from_host(A), hip.DeviceArray.from_host(np.ones((N, K), dt))
    dC = hip.DeviceArray((M, N), dt)
    ws = hip.workspace(hip.lib.exc_gemm_workspace(M, N, K))
    hip.call("exc_sgemm" if f32 else "exc_dgemm", 0, 1, M, N, K, 1.0, dA.ptr, K, dB.ptr, K, 0.0, dC.ptr, N, ws.ptr,
             ws.nbytes, None)
    hip.sync()
    # K and the lengths are multiples of the unit of the last place, 16
    assert np.max(K - (dC.to_host().astype(np.float64) - first)) <= longest


class GemmOpts(ctypes.Structure):
    """ExcGemmOpts of csrc/gemm.hpp, the products as the factorizations call them."""
    _fields_ = [("tri", ctypes.c_int), ("lower_only", ctypes.c_int), ("mirror", ctypes.c_int),
                ("work", ctypes.c_void_p), ("work_bytes", ctypes.c_size_t)]


class GemmProblem(ctypes.Structure):
    """ExcGemmProblem of csrc/gemm.hpp."""
    _fields_ = [("A", ctypes.c_void_p), ("lda", ctypes.c_long), ("B", ctypes.c_void_p), ("ldb", ctypes.c_long),
                ("C", ctypes.c_void_p), ("ldc", ctypes.c_long), ("M", ctypes.c_long), ("N", ctypes.c_long),
                ("K", ctypes.c_long), ("tri", ctypes.c_int), ("lower_only", ctypes.c_int), ("mirror", ctypes.c_int),
                ("beta_zero_hint", ctypes.c_int)]


LOWER, UPPER = 1, 2  # EXC_TRI_A_LOWER, EXC_TRI_A_UPPER


def internal(hip, f32, grouped=False):
    """The internal (C++) entry points that the factorizations use."""
    i, l, d, p = ctypes.c_int, ctypes.c_long, ctypes.c_double, ctypes.c_void_p
    if grouped:
        f = getattr(hip.lib, "_Z21exc_gemm_grouped_optsiiiPK14ExcGemmProblemddlPvmP12ihipStream_t")
        f.argtypes = [i, i, i, p, d, d, l, p, ctypes.c_size_t, p]
    else:
        f = getattr(hip.lib, "_Z14exc_sgemm_optsiillldPKflS0_ldPflRK11ExcGemmOptsP12ihipStream_t" if f32 else
                    "_Z13exc_gemm_optsiillldPKdlS0_ldPdlRK11ExcGemmOptsP12ihipStream_t")
        f.argtypes = [i, i, l, l, l, d, p, l, p, l, d, p, l, p, p]
    f.restype = i
    return f


def triangle(rng, m, upper, dt):
    """A triangular factor and the same with NaN in the triangle that is not part of it."""
    A = np.triu(rng.standard_normal((m, m))) if upper else np.tril(rng.standard_normal((m, m)))
    A = A.astype(dt)
    dirty = A.copy()
    dirty[np.tril_indices(m, -1) if upper else np.triu_indices(m, 1)] = np.nan
    return A, dirty


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("ta,tri", [(0, LOWER), (1, LOWER), (1, UPPER)])
@pytest.mark.parametrize("m,N", [(1, 1), (3, 5), (63, 70), (64, 1), (65, 130), (129, 67), (193, 66), (257, 1025),
                                 (321, 321), (500, 500), (1001, 999), (2049, 130), (641, 19097), (1025, 12753)])
def test_triangular_gemm(hip, f32, ta, tri, m, N):
    """op(A) triangular: odd and even numbers of tile rows of both tiles (the large one from about 19,097 columns at
    order 641 and 12,753 at 1025), split and unsplit, odd leading dimensions, NaN in the triangle that is
    not part of A. The bound is the a-priori one of the dot products in any order, here and in numpy."""
    dt, u = (np.float32, 2.0 ** -24) if f32 else (np.float64, 2.0 ** -53)
    s = np.dtype(dt).itemsize
    banner(f"triangular gemm m={m} N={N} ta={ta} tri={tri} f32={f32}")
    rng = np.random.default_rng(m + N + ta + tri)
    A, dirty = triangle(rng, m, tri == UPPER, dt)
    B, C = (rng.standard_normal((m, N)).astype(dt) for _ in range(2))
    cols = np.unique(np.r_[0:min(N, 130), max(0, N - 130):N])
    A64, B64, C64 = A.astype(np.float64), B[:, cols].astype(np.float64), C[:, cols].astype(np.float64)
    want = -1.0 * (A64 @ B64) + C64
    bound = (2 * m + 4) * u * (np.abs(A64) @ np.abs(B64) + np.abs(C64) + 1.0)
    stored = np.full((m, m + 1), np.nan, dt)
    stored[:, :m] = dirty.T if ta else dirty
    dA, dB = hip.DeviceArray.from_host(np.append(dt(np.nan), stored)), hip.DeviceArray.from_host(B)
    for work in (False, True):
        dC = hip.DeviceArray.from_host(C)
        ws = hip.workspace(hip.lib.exc_gemm_workspace(m, N, m)) if work else None
        o = GemmOpts(tri, 0, 0, ws.ptr if work else None, ws.nbytes if work else 0)
        assert internal(hip, f32)(ta, 0, m, N, m, -1.0, dA.ptr + s, m + 1, dB.ptr, N, 1.0, dC.ptr, N, ctypes.byref(o),
                                  None) == 0
        hip.sync()
        got = dC.to_host()
        assert np.isfinite(got).all()
        assert (np.abs(got[:, cols] - want) <= bound).all(), work


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("m,K", [(1, 1), (65, 40), (129, 700), (200, 4099), (600, 3000)])
def test_mirrored_gram(hip, f32, m, K):
    """Symmetric products of which the tiles on and below the diagonal are formed and mirrored."""
    dt, u = (np.float32, 2.0 ** -24) if f32 else (np.float64, 2.0 ** -53)
    banner(f"mirrored gram m={m} K={K} f32={f32}")
    X = np.random.default_rng(m + K).standard_normal((m, K)).astype(dt)
    X64 = X.astype(np.float64)
    dX = hip.DeviceArray.from_host(X)
    for work in (False, True):
        dC = hip.DeviceArray.from_host(np.full((m, m), np.nan, dt))
        ws = hip.workspace(hip.lib.exc_gemm_workspace(m, m, K)) if work else None
        o = GemmOpts(0, 1, 1, ws.ptr if work else None, ws.nbytes if work else 0)
        assert internal(hip, f32)(0, 1, m, m, K, 1.0, dX.ptr, K, dX.ptr, K, 0.0, dC.ptr, m, ctypes.byref(o), None) == 0
        hip.sync()
        got = dC.to_host()
        assert np.array_equal(got, got.T)
        assert (np.abs(got - X64 @ X64.T) <= (2 * K + 4) * u * (np.abs(X64) @ np.abs(X64).T)).all()


def test_triangular_gemm_refuses_what_it_has_no_kernel_for(hip):
    A = hip.DeviceArray.from_host(np.eye(8))
    C = hip.DeviceArray.from_host(np.zeros((8, 8)))
    for tb, lower in ((1, 0), (0, 1)):
        o = GemmOpts(LOWER, lower, 0, None, 0)
        assert internal(hip, False)(0, tb, 8, 8, 8, 1.0, A.ptr, 8, A.ptr, 8, 0.0, C.ptr, 8, ctypes.byref(o), None) == -1
    assert not C.to_host().any()


@pytest.mark.parametrize("kchunk", [0, 64, 100])
def test_grouped_products(hip, kchunk):
    """Grouped products in FP64, whole and in chunks of K: A B with triangular A of odd orders (NaN in the other
    triangle), and mirrored A A^T of blocks with one column and with none (whose product is zero)."""
    banner(f"grouped products kchunk={kchunk}")
    rng, u = np.random.default_rng(5), 2.0 ** -53
    grouped = internal(hip, False, grouped=True)
    size = getattr(hip.lib, "_Z26exc_gemm_grouped_workspaceiiPK14ExcGemmProbleml")
    size.argtypes, size.restype = [ctypes.c_int, ctypes.c_int, ctypes.c_void_p, ctypes.c_long], ctypes.c_size_t

    def run(tb, probs):
        arr = (GemmProblem * len(probs))(*probs)
        ws = hip.workspace(size(8, len(probs), arr, kchunk))
        assert grouped(8, tb, len(probs), arr, 1.0, 0.0, kchunk, ws.ptr, ws.nbytes, None) == 0
        hip.sync()

    keep, probs, want, bounds = [], [], [], []
    for m, N in ((1, 3), (63, 65), (129, 200), (193, 1), (321, 130)):
        A, dirty = triangle(rng, m, False, np.float64)
        B = rng.standard_normal((m, N))
        d = [hip.DeviceArray.from_host(x) for x in (dirty, B, np.full((m, N), np.nan))]
        keep.append(d)
        probs.append(GemmProblem(d[0].ptr, m, d[1].ptr, N, d[2].ptr, N, m, N, m, LOWER, 0, 0, 0))
        want.append(A @ B)
        bounds.append((2 * m + 4) * u * (np.abs(A) @ np.abs(B)))
    run(0, probs)
    for d, w, b in zip(keep, want, bounds):
        assert (np.abs(d[2].to_host() - w) <= b).all()

    keep, probs, want, bounds = [], [], [], []
    for m, K in ((129, 1), (70, 0), (65, 333), (3, 0), (200, 129)):
        X = rng.standard_normal((m, K))
        d = [hip.DeviceArray.from_host(X if K else np.zeros((m, 1))), hip.DeviceArray.from_host(np.full((m, m), np.nan))]
        keep.append(d)
        probs.append(GemmProblem(d[0].ptr, K, d[0].ptr, K, d[1].ptr, m, m, m, K, 0, 1, 1, 0))
        want.append(X @ X.T)
        bounds.append((2 * K + 4) * u * (np.abs(X) @ np.abs(X).T))
    run(1, probs)
    for d, w, b in zip(keep, want, bounds):
        got = d[1].to_host()
        assert np.array_equal(got, got.T) and (np.abs(got - w) <= b).all()
