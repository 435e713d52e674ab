"""The timed trial of launch shapes where it runs: on a lattice that walks by
itself (16384 x 4640, just past those that run in blocks), and at fixed steps
per pass on smaller ones.  It reports nothing until its launches have finished,
then one of its candidates; results are a fixed shape's; new forcing starts
it again; lgca_tune decides at once.  Lattices in blocks report the fixed rule
and make no trial."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

HEIGHTS = {2, 4, 8, 12, 16, 20, 24, 32}


def make(dx, dy, tuning=None):
    from lgca_amd import Lattice
    lat = Lattice(2, dim_x=dx, dim_y=dy, coarse_graining_radius=1, seed=dx)
    types = np.zeros((dy, dx), dtype=np.uint8)
    types[0], types[-1], types[dy // 2: dy // 2 + dy // 8, dx // 3: dx // 3 + 90] = 1, 1, 1
    lat.set_cell_types(types.reshape(-1))
    lat.init_random(0.3)
    lat.set_forcing("x", 0.02, 0, 200)
    if tuning:
        lat.set_tuning(*tuning)
    return lat


def shape(lat):
    i = lat.info()
    return i.steps_per_pass, i.tile_rows


def run_trial(lat, ref, k_open, calls):
    """Steps both through the calls; the trial is still open after the first."""
    assert shape(lat) == (k_open, 0)
    for i, n in enumerate(calls):
        lat.step(n)
        ref.step(n)
        if i == 0:
            assert shape(lat) == (k_open, 0)
    lat.synchronize()
    lat.step(8)
    ref.step(8)
    return shape(lat)


def test_trial_of_a_lattice_that_walks():
    print("[trial] 16384 x 4640", flush=True)
    lat, ref = make(16384, 4640), make(16384, 4640, (4, 16))
    assert lat.pass_shape().blocks == 0
    k, rows = run_trial(lat, ref, -1, (9, 31, 160, 120))
    print(f"[trial] kept {k} steps, {rows} rows", flush=True)
    assert (k == 4 and rows in HEIGHTS) or (k == 8 and rows >= 16 and rows % 2 == 0)
    np.testing.assert_array_equal(lat.get_state_u8(), ref.get_state_u8())
    lat.set_forcing("x", 0.01, 0, 100)
    assert shape(lat) == (-1, 0)
    lat.step(4)
    assert shape(lat) == (-1, 0)
    lat.tune()
    assert shape(lat)[0] in (4, 8) and shape(lat)[1] > 0
    lat.close()
    ref.close()


@pytest.mark.parametrize("dx,dy,k,heights", [(4096, 1024, 4, HEIGHTS), (4096, 1024, 8, HEIGHTS), (2048, 512, 2, HEIGHTS),
                                             (1024, 14, 4, {2, 4, 8, 12})])
def test_trial_of_heights(dx, dy, k, heights):
    """(1024 x 14: heights above the lattice's are left out)"""
    print(f"[trial] {dx} x {dy}, {k} steps per pass", flush=True)
    lat, ref = make(dx, dy, (k, 0)), make(dx, dy, (4, 10))
    got_k, rows = run_trial(lat, ref, k, (k, 3, 64, 17, 120))
    print(f"[trial] kept {rows} rows", flush=True)
    assert got_k == k and rows in heights
    np.testing.assert_array_equal(lat.get_state_u8(), ref.get_state_u8())
    # lgca_tune decides the same question without a step
    lat.set_tuning(k, 0)
    before = lat.get_state_u8()
    lat.tune()
    assert shape(lat)[0] == k and shape(lat)[1] in heights
    np.testing.assert_array_equal(lat.get_state_u8(), before)
    assert lat.steps == ref.steps
    lat.step(21)
    ref.step(21)
    np.testing.assert_array_equal(lat.get_state_u8(), ref.get_state_u8())
    lat.close()
    ref.close()


@pytest.mark.parametrize("dx,dy", [(4096, 1024), (1024, 14), (2048, 512), (4096, 512)])
def test_blocks_report_the_rule(dx, dy):
    lat = make(dx, dy)
    assert lat.pass_shape().blocks == 1 and shape(lat) == (-1, 0)
    lat.step(5)
    assert shape(lat) == (4, 2)  # the rule's: 2 rows on lattices of this size
    lat.tune()
    lat.step(300)
    assert shape(lat) == (4, 2)
    lat.close()
