"""Drag, probe and global means at the edges of their single-launch reductions: fewer mixed tiles than
one block takes, a last block with one tile, more tiles than blocks; repeated calls give the same bits."""
import numpy as np
import pytest

from euplectella_hpc_amd import d3q19, geometry

pytestmark = pytest.mark.gpu


def mask_of(kind, l, m, n):
    if kind == "one":
        mask = np.zeros((n, m, l), bool)
        mask[n // 2, m // 2, l // 2] = True
        return mask
    return geometry.scattered(l, m, n, fraction=0.1, seed=3).astype(bool)


@pytest.mark.parametrize("mode,storage", [("parity", "f64"), ("physics", "f64"), ("physics", "f32"), ("physics", "e3m12")])
@pytest.mark.parametrize("shape,kind", [((4, 3, 3), "one"), ((65, 9, 5), "one"), ((70, 33, 5), "dense"), ((130, 97, 40), "dense")])
def test_reductions(shape, kind, mode, storage):
    from euplectella_hpc_amd.lib import Lattice

    print(f"reductions {shape} {kind} {mode} {storage}", flush=True)
    l, m, n = shape
    mask = mask_of(kind, l, m, n)
    with Lattice(l, m, n, svisc=0.05, u_inflow=0.05, mode=mode, storage=storage, x_open=True) as lat:
        lat.set_mask(mask)
        lat.init_equilibrium(0.05, 0.01, -0.02, 1e-2, 3)
        lat.step(3)
        drag, means = lat.drag_mem(), lat.diagno()
        for _ in range(3):  # the other results in between leave nothing behind
            assert np.array_equal(lat.diagno(), means)
            probe = lat.probe(l, m, n)
            assert np.array_equal(lat.drag_mem(), drag)
            assert np.array_equal(lat.probe(l, m, n), probe)
        f = lat.get_state()[:, 1:-1, 1:-1, 1:-1]
    C = np.asarray(d3q19.C)
    force, size = np.zeros(3), 0.0
    for p in range(18):
        cx, cy, cz = (int(c) for c in C[p])
        solid = np.roll(mask, (-cz, -cy, -cx), (0, 1, 2))
        if cx:
            solid[:, :, -1 if cx > 0 else 0] = False
        hit = 2.0 * f[p][~mask & solid]
        force += C[p] * hit.sum()
        size += np.abs(hit).sum()
    # sums of at most a few 10^5 terms, each within 2^-53 of their absolute sum per addition
    assert np.abs(drag - force).max() <= 2.0 ** -53 * 4096 * max(size, 1.0)
    rho = f.sum(0)
    u = np.tensordot(C.T.astype(float), f, 1) / rho
    rho, u = np.where(mask, 1.0, rho), np.where(mask, 0.0, u)
    want = np.array([rho.mean(), *(u[d].mean() for d in range(3)), (u * u).sum(0).mean()])
    assert np.abs(means - want).max() <= 2.0 ** -53 * 4096
