"""GPU parity of the bidiagonal SVD kernels (C ABI) against the oracle: Sturm counts, bisection
leaves, twist indices, singular values and vectors are bit-identical."""
import numpy as np
import pytest

from conftest import random_bidiagonal

pytestmark = pytest.mark.gpu

KINDS = ["gauss", "positive", "graded"]


def banner(msg):
    print(f"[gpu-bsvd] {msg}", flush=True)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n", [1, 2, 17, 300])
def test_sturm_counts_bit_exact(hip, oracle, kind, n):
    banner(f"sturm n={n} kind={kind}")
    rng = np.random.default_rng(n)
    a, b = random_bidiagonal(rng, n, kind) if n > 1 else (np.array([1.5]), np.zeros(0))
    s = np.linalg.svd(np.diag(a) + (np.diag(b, 1) if n > 1 else 0), compute_uv=False)
    mus = np.concatenate([rng.uniform(0, 2 * s.max(), 500), s, np.nextafter(s, 0), [0.0, 1e-310]])
    got = hip.sturm_count(a, b, mus)
    want = oracle.negative_count_batch(a, b, mus)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("kind", KINDS + ["clustered"])
@pytest.mark.parametrize("n,top_k", [(1, 1), (2, 2), (40, 40), (40, 7), (1000, 1000), (2000, 100)])
def test_bisection_bit_exact(hip, oracle, kind, n, top_k):
    banner(f"bisection n={n} top_k={top_k} kind={kind}")
    rng = np.random.default_rng(1000 + n)
    a, b = random_bidiagonal(rng, n, kind) if n > 1 else (np.array([0.75]), np.zeros(0))
    ub = oracle.sigma_upper_bound(a, b)
    sg, lo, hi = hip.bisection(a, b, 0.0, ub, 1e-20, top_k)
    so, loo, hio = oracle.bisection(a, b, 0.0, ub, 1e-20, top_k)
    assert sg.size == so.size
    assert np.array_equal(sg, so)
    assert np.array_equal(lo, loo) and np.array_equal(hi, hio)


def test_bisection_quirks(hip, oracle):
    banner("bisection quirks")
    # equal singular values: one leaf, one value
    a, b = np.full(6, 2.0), np.zeros(5)
    sg, _, _ = hip.bisection(a, b, 0.0, 36.0, 1e-20, 6)
    so, _, _ = oracle.bisection(a, b, 0.0, 36.0, 1e-20, 6)
    assert np.array_equal(sg, so) and sg.size == 1
    # root already a leaf
    sg, _, _ = hip.bisection(np.zeros(3), np.zeros(2), 0.0, 0.0, 1e-20, 3)
    assert sg.size == 1 and sg[0] == 0.0
    # empty interval: nothing
    sg, _, _ = hip.bisection(np.array([1.0, 2.0]), np.array([0.5]), 5.0, 6.0, 1e-20, 2)
    so, _, _ = oracle.bisection(np.array([1.0, 2.0]), np.array([0.5]), 5.0, 6.0, 1e-20, 2)
    assert sg.size == so.size == 0


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n", [1, 3, 64, 500])
def test_twisted_vectors_bit_exact(hip, oracle, kind, n):
    banner(f"twisted n={n} kind={kind}")
    rng = np.random.default_rng(2000 + n)
    a, b = random_bidiagonal(rng, n, kind) if n > 1 else (np.array([2.0]), np.zeros(0))
    ub = oracle.sigma_upper_bound(a, b)
    sig, _, _ = oracle.bisection(a, b, 0.0, ub, 1e-20, n)
    u, v, tw = hip.twisted_vectors(a, b, sig)
    uo, vo, two = oracle.two_side(a, b, sig)
    assert np.array_equal(tw, two)
    assert np.array_equal(u, uo)
    assert np.array_equal(v, vo)


@pytest.mark.parametrize("kind", KINDS + ["clustered"])
@pytest.mark.parametrize("n,top_k", [(5, 5), (100, 100), (1000, 1000), (1000, 64)])
def test_bidiag_svd_bit_exact(hip, oracle, kind, n, top_k):
    banner(f"bidiag_svd n={n} top_k={top_k} kind={kind}")
    rng = np.random.default_rng(3000 + n)
    a, b = random_bidiagonal(rng, n, kind)
    so, uo, vo, two, rco = oracle.bidiag_svd(a, b, top_k)
    sg, ug, vg, twg, rcg = hip.bidiag_svd(a, b, top_k)
    if rco < 0:
        assert rcg == -5  # EXC_ERR_COUNT where the reference asserts
        return
    assert rcg == 0
    assert np.array_equal(sg, so)
    assert np.array_equal(twg, two)
    assert np.array_equal(ug, uo)
    assert np.array_equal(vg, vo)


def test_bidiag_svd_check_none(hip, oracle):
    banner("bidiag_svd check-none")
    a = np.array([3.0, 2.0, 1.0, 0.5])
    b = np.zeros(3)
    sg, ug, vg, _, rc = hip.bidiag_svd(a, b)
    assert rc == 0 and np.array_equal(sg, a)
    assert np.array_equal(ug, np.eye(4)) and np.array_equal(vg, np.eye(4))


def test_bidiag_svd_golden(hip, oracle):
    import os
    banner("bidiag_svd golden")
    z = np.load(os.path.join(os.path.dirname(__file__), "golden", "bidiag_lapack.npz"))
    for key in [k for k in z.files if k.startswith("alpha_")]:
        tag = key[len("alpha_"):]
        a, b, s = z[key], z["beta_" + tag], z["sigma_" + tag]
        sg, ug, vg, _, rc = hip.bidiag_svd(a, b)
        assert rc == 0
        assert np.max(np.abs(sg - s)) <= 32 * np.finfo(float).eps * s[0] * np.sqrt(a.size)
        so, uo, vo, _, _ = oracle.bidiag_svd(a, b)
        assert np.array_equal(sg, so) and np.array_equal(ug, uo) and np.array_equal(vg, vo)
        if not tag.startswith("graded"):
            # graded inputs trip the reference's absolute |sigma_i - alpha_i| < 1e-15 rewrite
            B = np.diag(a) + np.diag(b, 1)
            assert np.linalg.norm(B @ vg.T - ug * sg) <= 1e-12 * s[0] * a.size


@pytest.mark.parametrize("n", [300, 2000])
def test_bisection_nonmonotone_counts_bit_exact(hip, oracle, n):
    """Graded bidiagonals make the floating-point Sturm count non-monotone near singular values;
    the reference's search then records extra leaves, which the exact replay reproduces."""
    banner(f"bisection graded full n={n}")
    rng = np.random.default_rng(1000 + n)
    a, b = random_bidiagonal(rng, n, "graded")
    ub = oracle.sigma_upper_bound(a, b)
    sg, lo, hi = hip.bisection(a, b, 0.0, ub, 1e-20, n)
    so, loo, hio = oracle.bisection(a, b, 0.0, ub, 1e-20, n)
    assert np.array_equal(sg, so)
    assert np.array_equal(lo, loo) and np.array_equal(hi, hio)


@pytest.mark.parametrize("kind", ["gauss", "graded", "clustered"])
@pytest.mark.parametrize("n,top_k", [(31, 31), (32, 7), (33, 33), (97, 65), (255, 255), (256, 256), (257, 3),
                                     (1026, 1026), (1300, 129)])
def test_bidiag_svd_edges(hip, oracle, kind, n, top_k):
    """Orders around the chunks of 32 rows, the order from which the first levels are shared and the
    values that halve the lanes per value; value counts around the wavefront. Bit for bit."""
    banner(f"bidiag_svd edges n={n} top_k={top_k} kind={kind}")
    a, b = random_bidiagonal(np.random.default_rng(n + top_k), n, kind)
    so, uo, vo, two, rco = oracle.bidiag_svd(a, b, top_k)
    sg, ug, vg, twg, rcg = hip.bidiag_svd(a, b, top_k)
    if rco < 0:
        assert rcg == -5
        return
    assert rcg == 0
    assert np.array_equal(sg, so) and np.array_equal(twg, two)
    assert np.array_equal(ug, uo) and np.array_equal(vg, vo)


@pytest.mark.parametrize("n,top_k", [(1, 1), (2, 1), (2, 2), (3, 2), (32, 32), (100, 60), (256, 3), (300, 5), (300, 20),
                                     (311, 4), (312, 4), (933, 7), (934, 7)])
def test_bidiag_svd_fewer_values_in_the_workspace_of_all(hip, oracle, n, top_k):
    """A workspace of the size for all values serves a call for fewer, where the shared levels' counts
    lie in the search's scratch (few values) or in the sequences, and the bisection alone. Bit for bit."""
    banner(f"bidiag_svd n={n} top_k={top_k} in the workspace of {n}")
    a, b = random_bidiagonal(np.random.default_rng(7 * n + top_k), n, "gauss")
    so, uo, vo, two, rco = oracle.bidiag_svd(a, b, top_k)
    assert rco >= 0
    da = hip.DeviceArray.from_host(a)
    db = hip.DeviceArray.from_host(np.append(b, 0.0))
    du, dv, ds = hip.DeviceArray((n, top_k)), hip.DeviceArray((top_k, n)), hip.DeviceArray((top_k,))
    dt = hip.DeviceArray((2 * top_k,), np.int32)
    ws = hip.workspace(hip.lib.exc_bidiag_svd_workspace(n, n))
    hip.call("exc_bidiag_svd", n, da.ptr, db.ptr, du.ptr, dv.ptr, ds.ptr, top_k, dt.ptr, ws.ptr, ws.nbytes, None)
    hip.sync()
    assert np.array_equal(ds.to_host(), so) and np.array_equal(dt.to_host().reshape(two.shape), two)
    assert np.array_equal(du.to_host(), uo) and np.array_equal(dv.to_host(), vo)
    ub = float(np.sum(a * a) + np.sum(b * b))
    sg, lo, hi = hip.bisection(a, b, 0.0, ub, 1e-20, top_k)
    so, loo, hio = oracle.bisection(a, b, 0.0, ub, 1e-20, top_k)
    assert np.array_equal(sg, so) and np.array_equal(lo, loo) and np.array_equal(hi, hio)
