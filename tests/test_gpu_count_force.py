"""The count-mode force against the sequential oracle where its batches can go
wrong: stops inside the first and later batches of 4096 tries and on both
sides of a 1024-try boundary, within the listed tries and past them (amounts
that repeats or few feasible cells push beyond the list), lattices of far
fewer cells than a batch (every try repeats), amounts that are never reached,
and both rules of the FHP y direction."""
import numpy as np
import pytest

from oracle import oracle as orc

pytestmark = pytest.mark.gpu

Q = {0: 4, 1: 6, 2: 7, 3: 7}


@pytest.mark.parametrize("model,direction", [(0, "x"), (0, "y"), (1, "x"), (2, "y"), (3, "x")])
@pytest.mark.parametrize("dx,dy,forcing", [
    (6, 4, 2), (40, 40, 300), (320, 200, 100), (320, 200, 135), (320, 200, 1100), (320, 200, 4000),
    (320, 200, 9000), (1001, 300, 30000), (20, 12, 5), (700, 500, 17000)])
def test_count_force_stops_where_the_sequence_does(model, direction, dx, dy, forcing):
    from lgca_amd import Lattice
    rng = np.random.default_rng(forcing + 5 * model)
    state = rng.integers(0, 1 << Q[model], dx * dy, dtype=np.uint8)
    types = rng.choice(np.array([0, 0, 0, 0, 1, 2], np.uint8), dx * dy)
    print(f"[count-force] model={model} {dx}x{dy} {direction} {forcing}", flush=True)
    lat = Lattice(model, dim_x=dx, dim_y=dy, coarse_graining_radius=1, seed=91)
    lat.set_cell_types(types)
    lat.set_state_u8(state)
    for call in range(2):
        want = orc.body_force_count(model, dx, dy, types, state, 91, call, direction, forcing)
        assert lat.apply_body_force_count(direction, forcing) == want
        np.testing.assert_array_equal(lat.get_state_u8(), state)
    lat.close()


@pytest.mark.parametrize("p", [0.004, 0.97])
def test_count_force_past_the_listed_tries(p):
    """So few cells are feasible that the listed tries do not reach the amount."""
    from lgca_amd import Lattice
    dx, dy, model = 640, 400, 2
    rng = np.random.default_rng(3)
    state = np.zeros(dx * dy, dtype=np.uint8)
    for d in range(7):
        state |= (rng.random(dx * dy) < p).astype(np.uint8) << d
    lat = Lattice(model, dim_x=dx, dim_y=dy, coarse_graining_radius=1, seed=5)
    lat.set_state_u8(state)
    for call, forcing in enumerate((300, 40, 5000)):
        print(f"[count-force] p={p} forcing={forcing}", flush=True)
        want = orc.body_force_count(model, dx, dy, None, state, 5, call, "x", forcing)
        assert lat.apply_body_force_count("x", forcing) == want
        np.testing.assert_array_equal(lat.get_state_u8(), state)
    lat.close()
