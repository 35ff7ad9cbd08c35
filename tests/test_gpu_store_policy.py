"""Cached against non-temporal stores of the step kernels: the store policy moves no bit of the state,
the outlet plane or the drag.  The switch EUP_CACHED_STORES forces either at any size."""
import numpy as np
import pytest

from euplectella_hpc_amd import geometry

pytestmark = pytest.mark.gpu

CASES = [("physics", s, x) for s in ("f64", "f32", "f16", "bf16", "e3m12") for x in (True, False)] + [("parity", "f64", True)]


@pytest.mark.parametrize("mode,storage,x_open", CASES)
@pytest.mark.parametrize("pair", ["0", "1"])
@pytest.mark.parametrize("shape", [(37, 14, 9), (130, 27, 6)])
def test_store_policy_moves_no_bit(shape, pair, mode, storage, x_open, monkeypatch):
    from euplectella_hpc_amd.lib import Lattice

    print(f"store policy {shape} {mode} {storage} x_open={x_open} pair={pair}", flush=True)
    monkeypatch.setenv("EUP_PAIR", pair)
    got = []
    for cached in ("0", "1"):
        monkeypatch.setenv("EUP_CACHED_STORES", cached)
        with Lattice(*shape, svisc=0.05, u_inflow=0.05, mode=mode, storage=storage, x_open=x_open,
                     fgrad=0.0 if x_open else 1e-5) as lat:
            lat.set_mask(geometry.cylinder(*shape, 3, (shape[0] // 3, shape[1] // 2)))
            lat.init_equilibrium(0.05, 0.01, -0.02, 1e-2, 3)
            lat.step(5)
            got.append((lat.get_state(), lat.drag_mem()))
    for a, b in zip(*got):
        assert np.isfinite(a).all()
        assert np.array_equal(a, b)
