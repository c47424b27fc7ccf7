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


def test_step_vjp_rounding():
    """The noise term's rounding at 300 beads (Gaussians 1e5 times their size, so that it is all that
    counts), against a factor and an inverse in extended precision: two products whose partial sums
    have 32 terms, sqrt(32) 2^-53 each, and as much again for the factor, its inverse and L^T g:
    12 2^-53."""
    from bd_box_amd import system as S
    from oracle import adjoint as ad
    from oracle import pyoracle as po
    N, LD = 300, np.longdouble
    n = 3 * N
    sysm = wl.chain(N, seed=900 + N)
    P = wl.parse_params(wl.chain_params())
    p = po.params_from(P)
    rng = np.random.default_rng(N)
    xi, g = 1e5 * rng.normal(size=n), rng.normal(size=n)
    D = po.compute_D(sysm.coord, p).astype(LD)
    L, M = np.zeros((n, n), LD), np.zeros((n, n), LD)
    for j in range(n):
        v = D[j:, j] - L[j:, :j] @ L[j, :j]
        L[j:, j] = v / np.sqrt(v[0])
    for i in range(n):
        M[i] = -(L[i, :i] @ M[:i]) / L[i, i]
        M[i, i] = 1 / L[i, i]
    Phi = np.tril(np.outer(L.T @ g.astype(LD), xi.astype(LD))) * np.sqrt(2 * LD(P.dt))
    Phi -= np.diag(np.diag(Phi)) / 2
    Z = M.T @ Phi @ M
    F, _, _ = po.forces(sysm, p)
    c = P.dt / (ad.KB * P.T)
    U = (((Z + Z.T) / 2).astype(float) + c * 0.5 * (np.outer(g, F) + np.outer(F, g)))
    ref = g + ad.rpy_contract_grad(sysm.coord, U, p) - c * ad.hessian_vec(sysm, p, sysm.coord, D.astype(float) @ g)
    print(f"step vjp rounding N={N}", flush=True)
    rbar = S.BDSystem(sysm, P, precision=S.FP64, refactor_every=1).step_vjp(sysm.coord, xi, g)
    assert np.linalg.norm(rbar - ref) <= 12 * 2.0 ** -53 * np.linalg.norm(ref)
