"""TEA steps in free space on either side of the pair sums' workgroup widths (8 and 4 wavefronts)
and of their 64-bead tiles: one step's displacement against the oracle, FP64 <= 1e-10 relative (sums
of N terms in another order), mixed <= 1e-5."""
import numpy as np
import pytest

from bd_box_amd import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [2, 63, 64, 65, 1984, 2049])
def test_tea_step_vs_oracle(N):
    from bd_box_amd import system as S
    from oracle import pyoracle as po
    sysm = wl.chain(N, seed=70 + N)
    P = wl.parse_params(wl.chain_params(hydro="geyer"))
    xi = np.random.default_rng(N).normal(size=(1, 3 * N))
    print(f"tea step N={N}", flush=True)
    ref = po.Sim(sysm, po.params_from(P), seed=1)
    ref.run(1, xi)
    d_ref = ref.coords()[:, :3] - sysm.coord[:, :3]
    for prec, tol in ((S.FP64, 1e-10), (S.MIXED, 1e-5)):
        s = S.BDSystem(sysm, P, precision=prec)
        s.compute_hydro(1, xi)
        d = s.coords()[:, :3] - sysm.coord[:, :3]
        assert np.linalg.norm(d - d_ref) <= tol * np.linalg.norm(d_ref), prec


@pytest.mark.parametrize("hydro", ["cholesky", "geyer"])
def test_pair_sums_of_a_lost_bead(hydro):
    """A bead so far away that its squared distance is beyond FP64's range (and its blocks with the
    others zero) moves by its own mobility, and the others as without it: 1e-14, a few roundings."""
    from bd_box_amd import system as S
    N = 70
    sysm = wl.chain(N, seed=3)
    sysm = wl.System(sysm.coord, sysm.Q, sysm.LJ, sysm.bonds[:0], sysm.bond_parms[:0])
    sysm.coord[9, :3] = [1e160, -2e160, 3e160]
    P = wl.parse_params(wl.chain_params(hydro=hydro))
    print("lost bead", hydro, flush=True)
    F = np.random.default_rng(1).normal(size=(N, 3))
    s = S.BDSystem(sysm, P, precision=S.FP64)
    s.set_forces(F)
    Rf = s.compute_Rf().reshape(N, 3)
    rest = np.arange(N) != 9
    less = wl.System(sysm.coord[rest], sysm.Q[rest], sysm.LJ[rest], sysm.bonds[:0], sysm.bond_parms[:0])
    r = S.BDSystem(less, P, precision=S.FP64)
    r.set_forces(F[rest])
    ref = r.compute_Rf().reshape(-1, 3)
    assert np.abs(Rf[rest] - ref).max() <= 1e-14 * np.abs(ref).max()
    one = S.BDSystem(wl.System(sysm.coord[9:10], sysm.Q[:1], sysm.LJ[:1], sysm.bonds[:0], sysm.bond_parms[:0]), P,
                     precision=S.FP64)
    one.set_forces(F[9:10])
    assert np.array_equal(Rf[9], one.compute_Rf())
