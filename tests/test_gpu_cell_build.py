"""The cell builds at the edges of their ranges: fewer beads than workgroups, a bead more than one
round of a workgroup's threads (one launch), a count that no vector load divides and the largest
size (every bit of a thread's mask) of the build from precomputed cells, 1 to 48 cells an axis with
and without wrapping.

  neighbour sets : equal to a k-d tree's, itself checked against the oracle's pair finder
  forces (FP64)  : two calls bitwise equal (the lists do not depend on the atomics' order)
"""
import numpy as np
import pytest

from bd_box_amd import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("periodic", [False, True])
@pytest.mark.parametrize("N,box,cutoffs", [(5, 40.0, [3.0, 15.0]), (1025, 60.0, [1.2, 6.0, 14.0, 19.0, 25.0]),
                                           (8195, 120.0, [2.5, 30.5]), (65536, 290.0, [2.5, 6.5])])
def test_cell_build(N, box, cutoffs, periodic):
    from scipy.spatial import cKDTree

    from bd_box_amd import system as S
    rng = np.random.default_rng(N)
    coord = np.ones((N, 4))
    coord[:, :3] = rng.uniform(-0.5 * box, 0.5 * box, size=(N, 3))
    sysm = wl.System(coord, np.zeros(N), np.tile([0.5, 0.1], (N, 1)), np.zeros((0, 2), np.int32), np.zeros((0, 3)))
    kw = dict(bc="periodic", xbox=box) if periodic else {}
    P = wl.parse_params(wl.chain_params(hydro="none", elec="no", cutoff_lj=2.5, nb_list="bucket_list", **kw))
    s = S.BDSystem(sysm, P, precision=S.FP64)
    tree = cKDTree(coord[:, :3] + 0.5 * box, boxsize=box) if periodic else cKDTree(coord[:, :3])
    for cut in cutoffs:
        print(f"N={N} periodic={periodic} cutoff={cut}", flush=True)
        ref = np.array(sorted(tree.query_pairs(cut)), dtype=np.int64).reshape(-1, 2)
        assert np.array_equal(s.neighbour_pairs(cut), ref), cut
    F0, E0, _ = s.compute_forces()
    F1, E1, _ = s.compute_forces()
    assert np.array_equal(F0, F1) and np.array_equal(E0, E1)
