"""The one-launch Cholesky factorization at the edges of its tiles: orders on either side of the
64-column diagonal blocks and 128x128 tiles, every precision, against LAPACK, and the INFO of a
non-positive pivot in every 16-column group and block position."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EDGES = [1, 2, 15, 17, 63, 64, 65, 127, 128, 129, 191, 193, 255, 257, 385, 641]


@pytest.fixture(scope="module")
def api():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from bd_box_amd import system
    return system


def _matrix(n):
    """SPD with 3 on the diagonal and 1 / (2 + 0.1 d^2) off it, plus a ripple."""
    d = np.arange(n)[:, None] - np.arange(n)[None, :]
    return np.where(d == 0, 3.0, 1.0 / (2.0 + 0.1 * d * d)) + 0.01 * np.cos(d * 1.7)


@pytest.mark.parametrize("n", EDGES)
def test_factor_edges_vs_lapack(api, n):
    """FP64: entries within n eps |a| of LAPACK's, taken 8 times for the two orders of summation.
    FP32 storage: each entry of L is rounded to 2^-24, so |L L^T - A| <= 2 2^-24 a_max, taken 4
    times for the accumulation; split-bf16 products drop terms below 2^-17 |l l'|."""
    A = _matrix(n)
    ref = np.linalg.cholesky(A)
    print(f"factor n={n}", flush=True)
    L, info = api.dpotrf(A, "L", api.FP64)
    assert info == 0
    assert np.abs(np.tril(L) - ref).max() <= 8 * max(n, 16) * 2.0 ** -53 * 3.0
    for prec, tol in ((api.MIXED, 4 * 2 * 2.0 ** -24 * 3.02), (api.MIXED_SPLIT, 4 * 2.0 ** -17 * 3.02)):
        L, info = api.dpotrf(A, "L", prec)
        assert info == 0
        L = np.tril(L)
        assert np.abs(L @ L.T - A).max() <= tol, prec


@pytest.mark.parametrize("n", [2816, 2817, 4225])
def test_factor_shared_cus(api, n):
    """253, 276 and 595 tiles: one workgroup a CU, a few CUs with two, more workgroups than are
    resident.  FP64 and split as above; FP32 adds one rounding of a partial sum per 256 columns."""
    A = _matrix(n)
    print(f"factor n={n}", flush=True)
    for prec, tol in ((api.FP64, 8 * n * 2.0 ** -53 * 3.02), (api.MIXED, (4 + n / 256) * 2 * 2.0 ** -24 * 3.02),
                      (api.MIXED_SPLIT, 4 * 2.0 ** -17 * 3.02)):
        L, info = api.dpotrf(A, "L", prec)
        assert info == 0
        L = np.tril(L)
        assert np.abs(L @ L.T - A).max() <= tol, prec


@pytest.mark.parametrize("row", [0, 1, 15, 16, 47, 63, 64, 79, 127, 128, 191, 192, 299])
def test_factor_reports_first_bad_pivot(api, row):
    """LAPACK's INFO: the 1-based row of the first non-positive pivot."""
    A = _matrix(300)
    A[row, row] = -1.0
    if row + 5 < 300:
        A[row + 5, row + 5] = -2.0
    print(f"bad pivot row={row}", flush=True)
    for prec in (api.FP64, api.MIXED):
        from bd_box_amd import _lib
        import ctypes as C
        M = np.asfortranarray(A).copy(order="F")
        rc = _lib.load().bdh_dpotrf(b"L", M.ctypes.data_as(C.POINTER(C.c_double)), 300, 300, prec)
        assert rc == row + 1, (prec, rc)


@pytest.mark.parametrize("N", [256, 451, 1000])
def test_factor_rounding_of_chains(api, N):
    """FP64 factor of a chain's tensor in extended precision: an entry of A - L L^T collects a rounding
    of what remains of A's entry per 256 columns, and those of a partial sum of 256 columns, which
    are relative to that sum: as 16 of the former.  Random signs, 2^-53 each."""
    from bd_box_amd import workloads as wl
    from oracle import pyoracle as po
    s = wl.chain(N, seed=1)
    A = po.compute_D(s.coord, po.params_from(wl.parse_params(wl.chain_params())))
    A = np.tril(A) + np.tril(A, -1).T
    print(f"factor rounding N={N}", flush=True)
    L, info = api.dpotrf(A, "L", api.FP64)
    assert info == 0
    A, L = A.astype(np.longdouble), np.tril(L).astype(np.longdouble)
    x = np.random.default_rng(N).normal(size=3 * N).astype(np.longdouble)
    y = A @ x
    err = np.sqrt((((y - L @ (L.T @ x)) ** 2).sum() / (y ** 2).sum()))
    assert err <= 2.0 ** -53 * np.sqrt(16 + 3 * N / 256), float(err)


def test_factorizations_beside_each_other(api):
    """Two systems and a batch step from threads of their own, their factorizations in flight together
    on three streams with more tiles than the chip has places each: every one bitwise what it is alone."""
    import threading

    from bd_box_amd import workloads as wl
    sizes = [1500, 1400]
    systems = [wl.chain(N, seed=N) for N in sizes]
    small = wl.chains([300 + k for k in range(40)], seed=77)
    P = wl.parse_params(wl.chain_params())

    def single(k):
        s = api.BDSystem(systems[k], P, precision=(api.FP64, api.MIXED)[k])
        return s, s.coords

    def batch(_):
        b = api.BDBatch(small, P, list(range(40)), precision=api.MIXED)
        return b, b.coords

    def step(make, k, out):
        obj, coords = make(k)
        for _ in range(4):
            obj.compute_hydro(1)
        out[k] = coords()
        obj.close()

    jobs = [(single, 0), (single, 1), (batch, 2)]
    alone, beside = {}, {}
    for make, k in jobs:
        print("alone", k, flush=True)
        step(make, k, alone)
    print("together", flush=True)
    threads = [threading.Thread(target=step, args=(make, k, beside)) for make, k in jobs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k in alone:
        assert np.array_equal(alone[k], beside[k]), k
