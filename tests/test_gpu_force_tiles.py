"""Brute-force forces on either side of the tile-pair kernel's workgroup widths (16, 8 and 4
wavefronts), with a ragged last tile, a bead of six bonds and scaled interactions of partners.

  FP64  : <= 1e-12 of max|F| against the oracle (the order of the sums differs)
  mixed : <= 1e-5 of max|F|
"""
import numpy as np
import pytest

from bd_box_amd import workloads as wl

pytestmark = pytest.mark.gpu


def _system(N, seed):
    """A chain with a branched bead: bonds from bead 3 to its next neighbours as well."""
    sysm = wl.chain(N, seed=seed)
    extra = [(3, k) for k in (5, 6, 7, 8) if k < N]
    if extra:
        d = np.linalg.norm(sysm.coord[[b for _, b in extra], :3] - sysm.coord[3, :3], axis=1)
        sysm.bonds = np.concatenate([sysm.bonds, np.array(extra, sysm.bonds.dtype)])
        sysm.bond_parms = np.concatenate([sysm.bond_parms, [[0.9 * r, 3.0 * r, 5.0] for r in d]])
    return sysm


@pytest.mark.parametrize("N", [2, 64, 65, 257, 1536, 1601, 4097])
@pytest.mark.parametrize("box", [0.0, 400.0])
def test_forces_vs_oracle(N, box):
    from bd_box_amd import system as S
    from oracle import pyoracle as po
    sysm = _system(N, 60 + N)
    kw = dict(hydro="none", bond_lj_scale=0.5, bond_c_scale=0.25)
    if box:
        c = sysm.coord.copy()
        c[:, :3] -= box * np.floor(c[:, :3] / box + 0.5)
        sysm.coord = c
        kw.update(bc="periodic", xbox=box)
    P = wl.parse_params(wl.chain_params(**kw))
    print(f"forces N={N} box={box}", flush=True)
    Fo, Eo, ro = po.forces(sysm, po.params_from(P))
    F, E, rep = S.BDSystem(sysm, P, precision=S.FP64).compute_forces()
    scale = np.abs(Fo).max()
    assert np.abs(F - Fo).max() <= 1e-12 * scale
    np.testing.assert_allclose(E, Eo, rtol=1e-11, atol=1e-12)
    F32, _, _ = S.BDSystem(sysm, P, precision=S.MIXED).compute_forces()
    assert np.abs(F32 - Fo).max() <= 1e-5 * scale


@pytest.mark.parametrize("nb", ["brute", "bucket_list"])
@pytest.mark.parametrize("prec,u", [("FP64", 2.0 ** -53), ("MIXED", 2.0 ** -24)])
def test_pair_force_rounding(nb, prec, u):
    """Screened Coulomb forces of 1000 isolated pairs against extended precision: a dozen roundings
    (root, exponential, five products and sums, two quotients, the components), each uniform in
    +-u of its result: rms u sqrt(12 / 3)."""
    from bd_box_amd import system as S
    M, LD = 1000, np.longdouble
    rng = np.random.default_rng(1)
    r = np.exp(rng.uniform(np.log(3.2), np.log(11.9), M))
    k = np.arange(M)
    v = rng.normal(size=(M, 3))
    c = np.ones((2 * M, 4))
    c[0::2, :3] = (np.stack([k // 100, k // 10 % 10, k % 10], 1) - 5) * 100.0 + rng.uniform(-3, 3, (M, 3))
    c[1::2, :3] = c[0::2, :3] + v / np.linalg.norm(v, axis=1, keepdims=True) * r[:, None]
    Q = rng.choice([-1.0, 1.0], 2 * M)
    sysm = wl.System(c, Q, np.tile([2.0, 0.6], (2 * M, 1)), np.zeros((0, 2), np.int32), np.zeros((0, 3)))
    P = wl.parse_params(wl.chain_params(hydro="none", alpha_lj=0.0, nb_list=nb))
    d = c[1::2, :3].astype(LD) - c[0::2, :3]
    r = np.sqrt((d * d).sum(1))
    kr, qq = LD(P.kappa_c) * r, LD(P.gamma_c / P.epsilon_c) * Q[0::2] * Q[1::2]
    ref = -d * (qq * (1 + kr) * np.exp(-kr) / (r * r * r))[:, None]
    print(f"pair force rounding {nb} {prec}", flush=True)
    F, _, _ = S.BDSystem(sysm, P, precision=getattr(S, prec)).compute_forces()
    err = ((F.reshape(-1, 3)[0::2] - ref) ** 2).sum(1) / (ref ** 2).sum(1)
    assert np.sqrt(err.mean()) <= u * np.sqrt(12 / 3), float(np.sqrt(err.mean()))
