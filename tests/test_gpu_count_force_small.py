"""Amounts that the count-mode force reaches without listed tries, and the
first that it lists them for, against the sequential oracle: stops within the
first 1024 tries, past them (few feasible cells) and never, on lattices of
fewer cells than that and larger ones, one call after another."""
import numpy as np
import pytest

from oracle import oracle as orc

pytestmark = pytest.mark.gpu

Q = {0: 4, 1: 6, 2: 7, 3: 7}


@pytest.mark.parametrize("model,direction", [(0, "x"), (1, "y"), (2, "x"), (3, "y")])
@pytest.mark.parametrize("dx,dy,p", [(6, 4, 0.5), (40, 30, 0.3), (300, 200, 0.3), (1001, 302, 0.02), (300, 200, 0.99)])
def test_small_amounts_stop_where_the_sequence_does(model, direction, dx, dy, p):
    from lgca_amd import Lattice
    rng = np.random.default_rng(dx + model)
    state = np.zeros(dx * dy, dtype=np.uint8)
    for d in range(Q[model]):
        state |= (rng.random(dx * dy) < p).astype(np.uint8) << d
    types = rng.choice(np.array([0, 0, 0, 0, 1, 2], np.uint8), dx * dy)
    lat = Lattice(model, dim_x=dx, dim_y=dy, coarse_graining_radius=1, seed=91)
    lat.set_cell_types(types)
    lat.set_state_u8(state)
    for call, forcing in enumerate((0, 1, 3, 17, 63, 64, 65, 2, 200, 64)):
        print(f"[count-force] model={model} {dx}x{dy} p={p} {direction} {forcing}", flush=True)
        want = orc.body_force_count(model, dx, dy, types, state, 91, call, direction, forcing)
        assert lat.apply_body_force_count(direction, forcing) == want
        np.testing.assert_array_equal(lat.get_state_u8(), state)
    lat.close()
