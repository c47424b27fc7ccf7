"""A system's Gaussian draws on either side of the sizes that take one workgroup, two launches with
two attempts a thread, and eight: values and stream state equal to bdh_gauss's, which the host's
stream pins."""
import numpy as np
import pytest

from bd_box_amd import workloads as wl

pytestmark = pytest.mark.gpu


def _spheres(N):
    from bd_box_amd import system as S
    rng = np.random.default_rng(N)
    coord = np.ones((N, 4))
    L = 6.0 * N ** (1.0 / 3.0)
    coord[:, :3] = rng.uniform(-0.5 * L, 0.5 * L, size=(N, 3))
    sysm = wl.System(coord, np.zeros(N), np.tile([0.5, 0.1], (N, 1)), np.zeros((0, 2), np.int32), np.zeros((0, 3)))
    P = wl.parse_params(wl.chain_params(hydro="none", elec="no", cutoff_lj=2.5, nb_list="bucket_list", rand_seed=77))
    return S.BDSystem(sysm, P, precision=S.FP64)


@pytest.mark.parametrize("N", [1, 2, 533, 683, 933, 934, 1001, 30001])
def test_draws_equal_gauss(N):
    from bd_box_amd import system as S
    s = _spheres(N)
    print(f"draws N={N}", flush=True)
    state = s.rng_state()
    for _ in range(2):
        r = s.compute_r()
        ref, state = S.gauss(state, 3 * N)
        assert s.rng_state() == state
        k = np.flatnonzero(ref)[0]
        assert np.allclose(r, ref * (r[k] / ref[k]), rtol=1e-14, atol=0.0)   # radii are equal


def test_many_steps_in_one_draw():
    """16 steps of 60001 spheres: 2.9 million values, the last step's against the stream's."""
    from bd_box_amd import system as S
    N, m = 60001, 16
    s = _spheres(N)
    state = s.rng_state()
    print(f"draws N={N} steps={m}", flush=True)
    s.compute_hydro(m)
    for _ in range(m):
        ref, state = S.gauss(state, 3 * N)
    assert s.rng_state() == state
    r = s.last_displacement()[1]
    k = np.flatnonzero(ref)[0]
    assert np.allclose(r, ref * (r[k] / ref[k]), rtol=1e-14, atol=0.0)
