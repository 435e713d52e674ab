"""Calls of a few steps on lattices that run in blocks: the walks that some of
them take (short_walk_rows) give the bits of a fixed shape, in any order with
calls in blocks, with lgca_step and lgca_step_noalloc."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def make(model, dx, dy, solids, force):
    from lgca_amd import Lattice
    lat = Lattice(model, dim_x=dx, dim_y=dy, coarse_graining_radius=1, seed=dx)
    if solids:
        types = np.zeros((dy, dx), dtype=np.uint8)
        types[0], types[-1], types[dy // 2: dy // 2 + 40, dx // 3: dx // 3 + 50] = 1, 1, 1
        types[dy // 4: dy // 4 + 9, 100:180] = 2
        lat.set_cell_types(types.reshape(-1))
    lat.init_random(0.3)
    if force:
        lat.set_forcing(force, 0.01, 5, dx - 700)
    return lat


# the sizes just above the lines of 1, 2 and 4 steps, whole and short last words
@pytest.mark.parametrize("model,dx,dy,solids,force", [
    (2, 4096, 1966, True, "x"), (0, 5990, 2700, True, "y"), (1, 7001, 3460, False, None), (3, 7168, 3450, True, "x"),
    (2, 600, 49200, True, "y"), (0, 7168, 3450, False, "x")])
def test_short_calls_match_a_fixed_shape(model, dx, dy, solids, force):
    from lgca_amd._capi import check, lib
    print(f"[short] model={model} {dx}x{dy} solids={solids} force={force}", flush=True)
    lat, ref = make(model, dx, dy, solids, force), make(model, dx, dy, solids, force)
    ref.set_tuning(4, 16)
    for n in (1, 4, 2, 3, 2, 1, 1, 4, 13, 4):
        lat.step(n)
        ref.step(n)
    np.testing.assert_array_equal(lat.get_state_u8(), ref.get_state_u8())
    for n in (4, 1, 2):
        rc = lib().lgca_step_noalloc(lat.handle, C.c_uint64(n))
        if force and rc:  # (the fixed scratch holds 2^21 words)
            lat.step(n)
        else:
            check(rc, lat.handle)
        ref.step(n)
    np.testing.assert_array_equal(lat.get_state_u8(), ref.get_state_u8())
    lat.close()
    ref.close()
