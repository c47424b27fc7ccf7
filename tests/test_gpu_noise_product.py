"""L times a cycle's noise vectors: every width the product is built for (1 .. 16 right-hand sides, whole
and in part), on matrices that end within, at and just past its tiles of 128 and 256 rows, against the
steps composed on the host.  Tolerances: 1e-10 (FP64) and 1e-5 (FP32 storage) of the displacement, the
steps' own bounds; a batch's chain bitwise its own system."""
import numpy as np
import pytest

from bd_box_amd import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R", [1, 2, 3, 7, 10, 16])
def test_cycle_of_noise(R):
    from bd_box_amd import system as S
    from compose import compose_steps
    sizes = (1, 43, 85, 86, 171)   # 3, 129, 255, 258, 513 rows
    systems = [wl.chain(N, seed=N) for N in sizes]
    P = wl.parse_params(wl.chain_params())
    xi = [np.random.default_rng(N).normal(size=(R, 3 * N)) for N in sizes]
    for prec, tol in ((S.FP64, 1e-10), (S.MIXED, 1e-5)):
        ends = []
        for sysm, x in zip(systems, xi):
            print(f"R={R} N={sysm.N} prec={prec}", flush=True)
            s = S.BDSystem(sysm, P, precision=prec, refactor_every=R)
            s.compute_hydro(R, x)
            ends.append(s.coords())
            x0, want = sysm.coord[:, :3], compose_steps(sysm, P, x, R)[0][-1][:, :3]
            err = np.linalg.norm(ends[-1][:, :3] - want) / np.linalg.norm(want - x0)
            assert err < tol, (sysm.N, prec, err)
        b = S.BDBatch(systems, P, list(range(1, 1 + len(sizes))), precision=prec, refactor_every=R)
        b.compute_hydro(R, np.concatenate(xi, axis=1))
        for c, end in enumerate(ends):
            assert np.array_equal(b.chain_coords(c), end), (prec, c)
