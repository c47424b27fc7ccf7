"""The reverse step's inverse and noise product at orders on either side of the 64-blocks, for
even, odd and power-of-two numbers of blocks at every doubling, and past one span (4096 rows) of
the running sums: one step against the oracle adjoint, <= 1e-9 relative (the bound of the other
step tests)."""
import numpy as np
import pytest

from bd_box_amd import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [1, 2, 21, 22, 43, 128, 171, 300, 385, 1400])
def test_step_vjp_sizes(N):
    from bd_box_amd import system as S
    from oracle import adjoint as ad
    from oracle import pyoracle as po
    sysm = wl.chain(max(N, 2), seed=900 + N)
    if N == 1:
        sysm = wl.System(sysm.coord[:1].copy(), sysm.Q[:1].copy(), sysm.LJ[:1].copy(), sysm.bonds[:0],
                         sysm.bond_parms[:0])
    P = wl.parse_params(wl.chain_params())
    rng = np.random.default_rng(N)
    xi, g = rng.normal(size=3 * N), rng.normal(size=3 * N)
    print(f"step vjp N={N}", flush=True)
    s = S.BDSystem(sysm, P, precision=S.FP64, refactor_every=1)
    rbar = s.step_vjp(sysm.coord, xi, g)
    ref = ad.step_vjp(sysm, po.params_from(P), sysm.coord, xi, g)
    assert np.linalg.norm(rbar - ref) < 1e-9 * np.linalg.norm(ref)
