"""The grey-lattice kernels at the edges of their branches: wavefronts of free fluid beside grey ones,
lattices whose rows and totals are no multiple of 64 sites, grey sites in the first and last columns
and on the periodic seams, and checkpoint intervals around the segment lengths, against the FP64 oracle."""
import numpy as np
import pytest

from euplectella_hpc_amd import geometry
from euplectella_hpc_amd.lib import omega_from_svisc

pytestmark = pytest.mark.gpu

SVISC, U = 1.0 / 30.0, 0.05


def fields(l, m, n, where):
    """solid fraction: a few spheres, scattered single sites (ends and seams included), everywhere, none"""
    if where == "spheres":
        return geometry.grey_spheres(l, m, n, n_spheres=3, rmin=1.5, rmax=3.0, sigma=0.7, seed=4)
    if where == "none":
        return np.zeros((n, m, l))
    rng = np.random.default_rng(8)
    s = rng.random((n, m, l))
    if where == "scattered":
        s[rng.random((n, m, l)) > 0.004] = 0.0
        for k, j, i in ((0, 0, 0), (n - 1, m - 1, l - 1), (n // 2, 0, l - 1), (0, m // 2, 0)):
            s[k, j, i] = 0.7
    return s


def dense(pops):
    return np.ascontiguousarray(pops[:, 1:-1, 1:-1, 1:-1])


@pytest.mark.parametrize("x_open", [True, False])
@pytest.mark.parametrize("where", ["spheres", "scattered", "everywhere", "none"])
@pytest.mark.parametrize("shape", [(64, 8, 6), (70, 9, 5), (33, 7, 4), (130, 4, 3)])
def test_steps_force_objective_and_gradient(shape, where, x_open):
    from euplectella_hpc_amd.lib import Lattice
    from oracle import oracle as orc

    print(f"grey paths {shape} {where} x_open={x_open}", flush=True)
    l, m, n = shape
    s = fields(l, m, n, where)
    pops = geometry.initial_state(l, m, n, U, noise=1e-3, seed=6)
    om = omega_from_svisc(SVISC)
    with Lattice(l, m, n, svisc=SVISC, u_inflow=U, mode="grey", storage="f64", x_open=x_open) as lat:
        lat.set_grey(s)
        lat.set_state(pops)
        F = lat.grey_force()
        assert np.allclose(F, orc.grey_force(dense(pops), s, U, x_open=x_open), rtol=0, atol=1e-12 * l * m * n)
        # t1 below, at and past the checkpoint interval
        for t0, t1, every in ((1, 2, 5), (2, 6, 3), (1, 7, 3), (5, 5, 1)):
            Jr, gr = orc.grey_objective(dense(pops), s, om, U, t0, t1, every, 1.0, x_open=x_open)
            J, g = lat.grey_objective(t0, t1, every, 1.0)
            J2, _ = lat.grey_objective(t0, t1, every, 1.0, grad=False)
            assert J == J2
            # sums of at most 10 * l m n terms of size 1 in FP64, in another order than the oracle's
            assert abs(J - Jr) <= 1e-15 * 10 * l * m * n
            assert np.abs(g - gr).max() <= 1e-12 * max(np.abs(gr).max(), 1e-3)
        lat.step(3)
        ref = dense(pops)
        orc.grey_steps(ref, s, om, U, 3, x_open=x_open)
        assert np.array_equal(dense(lat.get_state()), ref)


@pytest.mark.parametrize("storage", ["f32", "f64"])
@pytest.mark.parametrize("x_open", [True, False])
@pytest.mark.parametrize("shape", [(70, 9, 5), (33, 7, 4)])
def test_offsets_of_large_arrays_move_no_bit(shape, x_open, storage, monkeypatch):
    """The kernels of arrays of 4 GiB and more, forced at a small size, against those of smaller ones."""
    from euplectella_hpc_amd.lib import Lattice

    print(f"grey offsets {shape} x_open={x_open} {storage}", flush=True)
    got = []
    for wide in ("0", "1"):
        monkeypatch.setenv("EUP_GREY_64BIT", wide)
        with Lattice(*shape, svisc=SVISC, u_inflow=U, mode="grey", storage=storage, x_open=x_open) as lat:
            lat.set_grey(fields(*shape, "scattered"))
            lat.init_equilibrium(U, 0.01, -0.02, 1e-3, 3)
            lat.step(2)
            F = lat.grey_force()
            out = [F]
            for fused in ("0", "1"):
                monkeypatch.setenv("EUP_ADJ_FUSED", fused)
                out += lat.grey_objective(2, 7, 3, 1.0)
            got.append(out + [lat.get_state()])
    for a, b in zip(*got):
        assert np.array_equal(a, b)
