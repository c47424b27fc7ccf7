"""What a system hands back, through its pinned memory and, past its size, without: positions equal
to those set, bit for bit, forces and energies of one call equal to those of another, from another
thread as well."""
import threading

import numpy as np
import pytest

from bd_box_amd import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [1, 7, 4096, 4097, 70001])
def test_round_trip(N):
    from bd_box_amd import system as S
    rng = np.random.default_rng(N)
    L = 6.0 * N ** (1.0 / 3.0)
    coord = np.ones((N, 4))
    coord[:, :3] = rng.uniform(-0.5 * L, 0.5 * L, size=(N, 3))
    sysm = wl.System(coord, np.zeros(N), np.tile([1.5, 0.1], (N, 1)), np.zeros((0, 2), np.int32), np.zeros((0, 3)))
    P = wl.parse_params(wl.chain_params(hydro="none", elec="no", cutoff_lj=4.0, nb_list="bucket_list"))
    print(f"round trip N={N}", flush=True)
    s = S.BDSystem(sysm, P, precision=S.FP64)
    moved = coord.copy()
    moved[:, :3] += rng.normal(scale=0.1, size=(N, 3))
    s.set_coords(moved)
    got = []
    t = threading.Thread(target=lambda: got.append(s.coords()))
    t.start()
    t.join()
    assert np.array_equal(got[0], moved) and np.array_equal(s.coords(), moved)
    F, E, _ = s.compute_forces()
    assert np.array_equal(s.forces(), F) and np.isfinite(E).all()
    assert N == 1 or np.any(F != 0.0)


@pytest.mark.parametrize("N", [40, 3000])
def test_readers_in_threads(N):
    """Positions and forces of one system read by four threads at once, 200 times each: every reader
    gets its own array, whole."""
    from bd_box_amd import system as S
    sysm = wl.chain(N, seed=N)
    s = S.BDSystem(sysm, wl.parse_params(wl.chain_params(hydro="none")), precision=S.FP64)
    s.compute_hydro(1)
    xyz, F = s.coords(), s.forces()
    wrong = []

    def read(get, want):
        for _ in range(200):
            if not np.array_equal(get(), want):
                wrong.append(get)

    print(f"readers in threads N={N}", flush=True)
    threads = [threading.Thread(target=read, args=a) for a in 2 * [(s.coords, xyz), (s.forces, F)]]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


def test_reading_leaves_the_device():
    """A system of one GPU read by a thread whose current device is another: it still is afterwards."""
    import torch

    from bd_box_amd import system as S
    if torch.cuda.device_count() < 2:
        pytest.skip("needs two GPUs")
    s = S.BDSystem(wl.chain(20, seed=1), wl.parse_params(wl.chain_params()), precision=S.FP64, device=0)
    s.compute_hydro(1)
    torch.cuda.set_device(1)
    print("reading leaves the device", flush=True)
    try:
        s.coords(), s.forces()
        assert torch.cuda.current_device() == 1
    finally:
        torch.cuda.set_device(0)
