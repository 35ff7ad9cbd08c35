"""Two steps per launch (FP32 and FP64 physics mode) against one step per launch: the same state, outlet
plane and drag, bit for bit, on lattices at the edges of the two-step kernel's windows (FP32 64 x 13
sites, FP64 32 x 12) and chunks.  The environment switch EUP_PAIR forces either form, so that sizes
for which single steps are the faster choice are covered too."""
import numpy as np
import pytest

from euplectella_hpc_amd import geometry

pytestmark = pytest.mark.gpu

SHAPES = [(2, 2, 2), (33, 2, 4), (34, 30, 3), (63, 13, 5), (64, 12, 7), (65, 14, 9), (70, 45, 36), (130, 27, 6),
          (192, 25, 11)]


def after(shape, storage, x_open, mask, steps, pair, monkeypatch):
    from euplectella_hpc_amd.lib import Lattice

    monkeypatch.setenv("EUP_PAIR", pair)
    with Lattice(*shape, svisc=0.05, u_inflow=0.05, mode="physics", storage=storage, x_open=x_open,
                 fgrad=0.0 if x_open else 1e-5) as lat:
        lat.set_mask(mask)
        lat.init_equilibrium(0.05, 0.01, -0.02, 1e-2, 3)
        lat.step(steps)
        state, drag = lat.get_state(), lat.drag_mem()
        monkeypatch.setenv("EUP_PAIR", "0")
        lat.step(1)  # a further single step reads the outlet plane that the last one left
        return state, drag, lat.get_state()


@pytest.mark.parametrize("storage", ["f32", "f64"])
@pytest.mark.parametrize("x_open", [True, False])
@pytest.mark.parametrize("shape", SHAPES)
def test_two_steps_equal_single_steps(shape, x_open, storage, monkeypatch):
    print(f"two-step {shape} x_open={x_open} {storage}", flush=True)
    # solid sites everywhere, the first and last x planes and the periodic seams included
    mask = geometry.scattered(*shape, fraction=0.08, seed=5)
    for steps in (2, 5):
        one = after(shape, storage, x_open, mask, steps, "0", monkeypatch)
        two = after(shape, storage, x_open, mask, steps, "1", monkeypatch)
        for a, b in zip(one, two):
            assert np.isfinite(a).all()
            assert np.array_equal(a, b)


@pytest.mark.parametrize("storage", ["f32", "f64"])
@pytest.mark.parametrize("chunk", ["-3", "0", "100", ""])
def test_chunk_switch_outside_the_lattice(chunk, storage, monkeypatch):
    """The switch is held to 1 .. n planes."""
    shape = (40, 16, 9)
    print(f"two-step chunk switch {chunk!r} {storage}", flush=True)
    mask = geometry.cylinder(*shape, 3, (12, 8))
    one = after(shape, storage, True, mask, 4, "0", monkeypatch)
    monkeypatch.setenv("EUP_PAIR_ZC", chunk)
    two = after(shape, storage, True, mask, 4, "1", monkeypatch)
    for a, b in zip(one, two):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("storage", ["f32", "f64"])
@pytest.mark.parametrize("x_open", [True, False])
def test_more_workgroups_than_one_deal(x_open, storage, monkeypatch):
    """Workgroups are dealt to the XCDs in whole groups of 256, the rest in order: 720 (FP32) and 1200 (FP64)."""
    shape = (130, 66, 40)
    print(f"two-step deal x_open={x_open} {storage}", flush=True)
    mask = geometry.scattered(*shape, fraction=0.03, seed=5)
    one = after(shape, storage, x_open, mask, 4, "0", monkeypatch)
    monkeypatch.setenv("EUP_PAIR_ZC", "1")
    two = after(shape, storage, x_open, mask, 4, "1", monkeypatch)
    for a, b in zip(one, two):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("storage", ["f32", "f64"])
@pytest.mark.parametrize("chunk", ["1", "3", "7"])
def test_chunks_of_planes(chunk, storage, monkeypatch):
    """Any cut into chunks of planes gives the same state, the last chunk a short one."""
    shape = (100, 20, 17)
    print(f"two-step chunks of {chunk} planes {storage}", flush=True)
    mask = geometry.cylinder(*shape, 5, (25, 10))
    one = after(shape, storage, True, mask, 4, "0", monkeypatch)
    monkeypatch.setenv("EUP_PAIR_ZC", chunk)
    two = after(shape, storage, True, mask, 4, "1", monkeypatch)
    for a, b in zip(one, two):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("storage", ["f32", "f64", "f16", "bf16", "e3m12"])
@pytest.mark.parametrize("x_open", [True, False])
@pytest.mark.parametrize("shape", [(70, 14, 9), (128, 6, 5)])
def test_mask_changed_between_steps(shape, x_open, storage, monkeypatch):
    """A site that a new mask makes solid keeps, from the commit on, the values it had there, whatever
    the number of steps that follow and however they are taken; released again, it flows on from them."""
    from euplectella_hpc_amd.lib import Lattice

    print(f"mask changed {shape} x_open={x_open} {storage}", flush=True)
    masks = [geometry.scattered(*shape, fraction=f, seed=s).astype(bool) for f, s in ((0.05, 5), (0.1, 6), (0.05, 7))]
    masks[1][:, : shape[1] // 2, :64] = True  # whole tiles of solid sites
    for steps in (1, 2, 5):
        runs = []
        for pair in ("0", "1"):
            monkeypatch.setenv("EUP_PAIR", pair)
            with Lattice(*shape, svisc=0.05, u_inflow=0.05, mode="physics", storage=storage, x_open=x_open,
                         fgrad=0.0 if x_open else 1e-5) as lat:
                lat.set_mask(masks[0])
                lat.init_equilibrium(0.05, 0.01, -0.02, 1e-2, 3)
                lat.step(3)
                before = lat.get_state()
                lat.set_mask(masks[1])
                lat.step(steps)
                after = lat.get_state()
                lat.set_mask(masks[2])
                lat.step(2)
                runs.append((after, lat.get_state(), lat.drag_mem()))
            solid = masks[1]
            inner = np.s_[:, 1:-1, 1:-1, 1:-1]
            assert np.array_equal(after[inner][:, solid], before[inner][:, solid])
            assert not np.array_equal(after[inner][:, ~solid], before[inner][:, ~solid])
        for a, b in zip(*runs):
            assert np.isfinite(a).all()
            assert np.array_equal(a, b)


@pytest.mark.parametrize("mode,storage,pairs", [("physics", "f32", 2), ("physics", "f64", 2), ("physics", "f16", 1),
                                                ("physics", "e3m12", 1), ("parity", "f64", 1), ("grey", "f32", 1)])
def test_steps_per_launch_says_which_form_runs(mode, storage, pairs, monkeypatch):
    from euplectella_hpc_amd.lib import EupError, Lattice

    with Lattice(64, 12, 7, svisc=0.05, u_inflow=0.05, mode=mode, storage=storage) as lat:
        monkeypatch.setenv("EUP_PAIR", "1")
        assert [lat.steps_per_launch(n) for n in (1, 2, 3)] == [1, pairs, pairs]
        monkeypatch.setenv("EUP_PAIR", "0")
        assert lat.steps_per_launch(2) == 1
        with pytest.raises(EupError):
            lat.steps_per_launch(0)


@pytest.mark.parametrize("storage", ["f32", "f64"])
def test_mostly_solid_lattices_take_single_steps(storage):
    """A single step skips tiles that are solid throughout, a pair does not: the default follows the mask."""
    from euplectella_hpc_amd.lib import Lattice

    l, m, n = 192, 96, 96
    mask = np.zeros((n, m, l), bool)
    with Lattice(l, m, n, svisc=0.05, u_inflow=0.05, mode="physics", storage=storage) as lat:
        lat.set_mask(mask)
        assert lat.steps_per_launch(2) == 2
        mask[:, : 7 * m // 10] = True
        lat.set_mask(mask)
        assert lat.steps_per_launch(2) == 1
        mask[:, 1:] = False
        lat.set_mask(mask)
        assert lat.steps_per_launch(2) == 2
