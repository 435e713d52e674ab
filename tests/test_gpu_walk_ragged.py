"""Walked passes over rows with a short last word, whose bits past the row's end
are cleared only at the store: last words of one cell, a few and 31 cells,
rows that are one word, one segment, one strip and several strips; plain,
forced and solid tiles; SLIP cells on and off the lattice's rim; every steps
per pass, from steps inside and at the start of a chirality group."""
import numpy as np
import pytest

from oracle import oracle as orc

pytestmark = pytest.mark.gpu

Q = {0: 4, 1: 6, 2: 7, 3: 7}


@pytest.mark.parametrize("dx", [31, 33, 63, 97, 1001, 1985, 2015, 2017, 4001])
@pytest.mark.parametrize("geom", [None, "walls", "slip", "inner_slip"])
@pytest.mark.parametrize("k", [1, 2, 4, 8])
def test_ragged_walks_match_the_oracle(dx, geom, k):
    from lgca_amd import Lattice
    model, dy, th = (dx + k) % 4, 54, 18
    rng = np.random.default_rng(dx * 16 + k)
    types = np.zeros((dy, dx), np.uint8)
    if geom == "walls":
        types[0] = types[-1] = 1
    elif geom:
        types[0], types[-1], types[:, 0], types[:, -1] = 2, 2, 2, 2
        if geom == "inner_slip":
            types[rng.random((dy, dx)) < 0.05] = 2
            types[rng.random((dy, dx)) < 0.05] = 1
    types = types.reshape(-1)
    force = [None, dict(dir="x", p=0.1), dict(dir="y", p=0.1, x0=0, x1=max(dx // 2, 1))][(dx + k // 2) % 3]
    print(f"[walk] model={model} {dx}x{dy} {geom} {force} k={k}", flush=True)
    state = rng.integers(0, 1 << Q[model], dx * dy, dtype=np.uint8)
    for step0 in (0, 3):
        lat = Lattice(model, dim_x=dx, dim_y=dy, coarse_graining_radius=1, seed=99)
        if geom:
            lat.set_cell_types(types)
        lat.set_state_u8(state)
        lat.set_step(step0)
        if force:
            lat.set_forcing(force["dir"], force["p"], force.get("x0", 0), force.get("x1"))
        lat.set_tuning(k, th)
        lat.step(3 * k)
        want = orc.run(model, dx, dy, types, state, 99, step0, 3 * k, force, nthreads=8)
        np.testing.assert_array_equal(lat.get_state_u8(), want)
        lat.close()
