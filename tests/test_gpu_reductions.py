"""The whole-lattice sums and the coarse fields at the sizes where their
kernels' work splits can go wrong: rows of one word and of more words than a
workgroup has threads, more rows than the grid covers at once, more coarse
cells than one workgroup's 64, radii on both sides of a unit of 16 columns and
of the largest radius the popcounts serve, and the wrapped column."""
import numpy as np
import pytest

from oracle import oracle as orc

pytestmark = pytest.mark.gpu

Q = {0: 4, 1: 6, 2: 7, 3: 7}


def make(model, dx, dy, r, solids):
    from lgca_amd import Lattice
    rng = np.random.default_rng(dx * 7 + dy + model)
    state = rng.integers(0, 1 << Q[model], dx * dy, dtype=np.uint8)
    types = rng.choice(np.array([0, 0, 0, 1, 2], np.uint8), dx * dy) if solids else np.zeros(dx * dy, np.uint8)
    lat = Lattice(model, dim_x=dx, dim_y=dy, coarse_graining_radius=r)
    if solids:
        lat.set_cell_types(types)
    lat.set_state_u8(state)
    lat.copy_data_to_output_buffer()
    return lat, state, types


@pytest.mark.parametrize("model,dx,dy,solids", [
    (0, 2, 3, False), (1, 31, 2, True), (2, 33, 8200, True), (3, 1000, 66, False),
    (2, 32768 + 40, 4, True), (0, 70000, 5, True), (1, 4096, 300, False), (2, 2048, 2050, False)])
def test_particle_count_and_mean_velocity_are_exact(model, dx, dy, solids):
    print(f"[sum] model={model} {dx}x{dy} solids={solids}", flush=True)
    lat, state, types = make(model, dx, dy, 1, solids)
    assert lat.get_n_particles() == orc.count_particles(state)
    b = [((state >> d) & 1).astype(np.int64) for d in range(Q[model])]
    rho = sum(b)
    if model == 0:
        kx, ky, ux, uy = b[0] - b[2], b[1] - b[3], 1.0, 1.0
    else:
        kx, ky = 2 * b[0] + b[1] - b[2] - 2 * b[3] - b[4] + b[5], b[1] + b[2] - b[4] - b[5]
        ux, uy = 0.5, float(np.float32(0.866025388240814208984375))
    fluid = types == 0
    n = float(fluid.sum())
    per = np.where(fluid & (rho > 0), 840 // np.maximum(rho, 1), 0)
    sx, sy = int((kx * per).sum()), int((ky * per).sum())
    # the sums are exact integers, then one double division and one rounding
    want = [float(np.float32(sx * ux / (840.0 * n))), float(np.float32(sy * uy / (840.0 * n)))] if n else [0.0, 0.0]
    assert lat.get_mean_velocity() == want
    lat.close()


@pytest.mark.parametrize("model", [0, 1, 2])
@pytest.mark.parametrize("dx,dy,r", [
    (2, 2, 1), (300, 130, 1), (640, 96, 7), (480, 64, 15), (512, 96, 16), (612, 70, 17), (1000, 130, 31),
    (2112, 132, 32), (132, 200, 33), (64, 100, 32), (130, 260, 65), (2046, 2046, 1023), (2048, 2050, 1024)])
def test_coarse_fields_bit_exact_at_unit_edges(model, dx, dy, r):
    print(f"[coarse] model={model} {dx}x{dy} r={r}", flush=True)
    lat, state, _ = make(model, dx, dy, r, False)
    lat.post_process(cells=False)
    _, _, md, mm = orc.post_process(model, dx, dy, r, state)
    np.testing.assert_array_equal(lat.mean_density().view(np.uint32), md.view(np.uint32))
    np.testing.assert_array_equal(lat.mean_momentum().view(np.uint32), mm.view(np.uint32))
    lat.close()


# a row's columns in one unit of more than a word, in one of all its columns,
# and in two and three units
@pytest.mark.parametrize("model", [0, 1, 3])
@pytest.mark.parametrize("dx,dy,r", [(620, 130, 31), (700, 140, 34), (1050, 144, 35), (72, 146, 36), (720, 150, 37),
                                     (710, 284, 71), (1000, 300, 72), (880, 450, 109)])
def test_coarse_fields_bit_exact_at_long_units(model, dx, dy, r):
    test_coarse_fields_bit_exact_at_unit_edges(model, dx, dy, r)


@pytest.mark.parametrize("dx,dy", [(582, 600), (584, 600)])  # coarse fields just below and above 1 MiB
def test_small_results_in_turn(dx, dy):
    """Counts, velocities, refused inputs and coarse fields one after another:
    each result is its own call's."""
    from lgca_amd import LgcaError
    lat, state, types = make(2, dx, dy, 1, True)
    velocity = lat.get_mean_velocity()
    for _ in range(3):
        assert lat.get_n_particles() == orc.count_particles(state)
        assert lat.get_mean_velocity() == velocity
        with pytest.raises(LgcaError):
            lat.set_cell_types(np.full(dx * dy, 3, np.uint8))
        lat.set_cell_types(types)
        with pytest.raises(LgcaError):
            lat.set_state_u8(np.full(dx * dy, 255, np.uint8))
        lat.set_state_u8(state)
        lat.post_process(cells=False)
        _, _, md, mm = orc.post_process(2, dx, dy, 1, state)
        np.testing.assert_array_equal(lat.mean_density().view(np.uint32), md.view(np.uint32))
        np.testing.assert_array_equal(lat.mean_momentum().view(np.uint32), mm.view(np.uint32))
    lat.close()
