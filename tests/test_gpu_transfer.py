"""State and velocity arrays between device and host in pinned pieces by several host threads: sizes
below, at and across the pieces of 1 MiB (state: whole doubles; velocities: whole blocks of 256 sites),
against per-population calls, per-plane calls and the values themselves."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# ghosted arrays of 19 x 27 doubles (one piece) up to nine pieces and more; velocities of 24 bytes up to 5 pieces
SHAPES = [(2, 2, 2), (2, 3, 2), (17, 5, 9), (62, 6, 11), (65, 33, 40), (96, 64, 68)]


def lattice(shape, mode, storage):
    from euplectella_hpc_amd.lib import Lattice

    lat = Lattice(*shape, svisc=0.05, u_inflow=0.05, mode=mode, storage=storage, x_open=True)
    if mode == "grey":
        lat.set_grey(np.zeros(shape[::-1]))
    else:
        lat.set_mask(np.zeros(shape[::-1], bool))
    return lat


def exchange(shape, mode, storage, seed):
    l, m, n = shape
    rng = np.random.default_rng(seed)
    pops = rng.uniform(0.01, 0.06, (19, n + 2, m + 2, l + 2))
    with lattice(shape, mode, storage) as lat:
        lat.set_state(pops)
        got = lat.get_state()
        single = np.stack([lat.get_pops(q) for q in range(1, 20)])
        assert np.array_equal(got, single)
        for q in range(1, 20):
            lat.set_pops(q, pops[q - 1])
        assert np.array_equal(lat.get_state(), got)
        inner = np.s_[:, 1:-1, 1:-1, 1:-1]
        if mode == "parity":
            assert np.array_equal(got, pops)
        elif storage == "f64":
            assert np.array_equal(got[inner], pops[inner])
        else:
            # FP32 holds the deviation from the rest state, or the value itself: half a unit in the last place of 0.6
            assert np.abs(got[inner] - pops[inner]).max() <= 2.0 ** -25
        if mode != "parity":
            shell = got.copy()
            shell[inner] = 0.0
            assert not shell.any()
        if mode != "grey":
            volume = lat.vtk_velocity(3).reshape(n, m, l, 3)
            for k in (1, n):
                assert np.array_equal(volume[k - 1].reshape(-1, 3), lat.vtk_velocity(2, k))
            for j in (1, m):
                assert np.array_equal(volume[:, j - 1].reshape(-1, 3), lat.vtk_velocity(1, j))
            for i in (1, l):
                assert np.array_equal(volume[:, :, i - 1].reshape(-1, 3), lat.vtk_velocity(0, i))


@pytest.mark.parametrize("mode,storage", [("parity", "f64"), ("physics", "f64"), ("physics", "f32"), ("grey", "f32")])
@pytest.mark.parametrize("shape", SHAPES)
def test_pieces_hold_the_state(shape, mode, storage):
    print(f"transfer {shape} {mode} {storage}", flush=True)
    exchange(shape, mode, storage, 3)


def test_handles_in_several_threads():
    """One handle per host thread: their transfers share neither pieces nor helpers."""
    failed = []

    def work(seed):
        try:
            exchange((65, 33, 40), "physics", "f64", seed)
        except BaseException as e:  # noqa: BLE001 - reported below
            failed.append(e)

    threads = [threading.Thread(target=work, args=(s,)) for s in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed
