"""lgca_get_pass reports the passes that lgca_step runs: blocks on lattices
that run in them, the trial's or the fixed tiles elsewhere."""
import pytest

pytestmark = pytest.mark.gpu


def shape(lat):
    p = lat.pass_shape()
    return p.blocks, p.steps, p.rows, p.waves


@pytest.mark.parametrize("tune", [False, True])
def test_pass_shape_of_a_lattice_in_blocks(tune):
    from lgca_amd import Lattice
    lat = Lattice("HPP", dim_x=256, dim_y=256, coarse_graining_radius=1, seed=1)
    lat.init_random(0.2)
    assert shape(lat) == (1, 0, 0, 0)
    if tune:
        lat.tune()
    else:
        lat.step(100)
    blocks, steps, rows, waves = shape(lat)
    assert blocks == 1 and 4 < steps <= 28 and 0 < rows <= 256 and rows % 2 == 0 and waves in (4, 8, 12, 16)
    lat.step(50)
    assert shape(lat) == (blocks, steps, rows, waves)
    lat.set_forcing("x", 0.01)
    assert shape(lat) == (1, 0, 0, 0)
    lat.set_tuning(4, 9)
    assert shape(lat) == (0, 4, 10, 1)
    lat.set_tuning(8, 0)
    assert shape(lat) == (0, 0, 0, 1)
    lat.set_tuning(0, 0)
    assert shape(lat) == (0, 1, 0, 1)
    lat.close()
