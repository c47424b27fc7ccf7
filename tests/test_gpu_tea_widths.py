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
