"""Batches with fewer and with more factorization tiles (495, 550) than the workgroups the chip holds:
every chain bitwise the trajectory of its own system."""
import numpy as np
import pytest

from bd_box_amd import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chains", [9, 10])
def test_batch_equals_systems(chains):
    from bd_box_amd import system as S
    sizes = [400 + 2 * k for k in range(chains)]   # ten tile rows each
    systems = [wl.chain(N, seed=N) for N in sizes]
    P = wl.parse_params(wl.chain_params())
    seeds = list(range(7, 7 + chains))
    for prec in (S.MIXED, S.FP64, S.MIXED_SPLIT):
        print(f"batch chains={chains} prec={prec}", flush=True)
        b = S.BDBatch(systems, P, seeds, precision=prec)
        b.compute_hydro(2)
        for c in (0, chains - 1):
            p = wl.parse_params(wl.chain_params(rand_seed=seeds[c]))
            s = S.BDSystem(systems[c], p, precision=prec)
            s.compute_hydro(2)
            assert np.array_equal(b.chain_coords(c), s.coords()), (prec, c)


def test_tuner_times_one_schedule():
    """Candidates that are the same launches get one time and the first is kept."""
    from bd_box_amd import system as S
    b = S.BDBatch([wl.chain(N, seed=N) for N in (60, 200, 700)], wl.parse_params(wl.chain_params()), [1, 2, 3],
                  precision=S.MIXED)
    print("tuner", flush=True)
    for tune, first in ((b.autotune, 0), (b.autotune_tiles, (0, 256))):
        best, times = tune(reps=2)
        assert best == first and len(times) > 1
        assert len(set(times.values())) == 1 and times[best] > 0.0
    b.close()
