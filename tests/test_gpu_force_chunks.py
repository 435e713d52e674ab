"""Force decisions of regions whose chunks of 1024 (row, word) pairs fill the
GPU, at sizes around whole chunks, where few words fire (whole chunks) and where
most do (short ones), in single lattices and in batches, against the oracle."""
import numpy as np
import pytest

from oracle import oracle as orc

pytestmark = pytest.mark.gpu


# 64, 64.5 and 81 chunks of pairs in the region, 16 and 17 groups of steps
@pytest.mark.parametrize("words,rows", [(128, 512), (129, 512), (127, 653)])
@pytest.mark.parametrize("p", [1e-4, 5e-3, 0.04, 0.05, 0.6])
def test_large_draws_match_the_oracle(words, rows, p):
    from lgca_amd import Batch, Job, Lattice
    dx, dy = 32 * words + 40, rows + 6 + (rows & 1)
    rng = np.random.default_rng(words * rows)
    state = rng.integers(0, 128, dx * dy, dtype=np.uint8)
    force = dict(dir="x", p=p, x0=5, x1=5 + 32 * words - 10, y0=3, y1=3 + rows)
    print(f"[draw] {words} words x {rows} rows p={p}", flush=True)
    lat = Lattice(2, dim_x=dx, dim_y=dy, coarse_graining_radius=1, seed=17)
    lat.set_state_u8(state)
    lat.set_step(3)
    lat.set_forcing("x", p, force["x0"], force["x1"], force["y0"], force["y1"])
    lat.step(64)
    want = orc.run(2, dx, dy, None, state, 17, 3, 64, force, nthreads=8)
    np.testing.assert_array_equal(lat.get_state_u8(), want)
    lat.close()
    # two jobs of this region: 128 chunks and more for each of 8 groups
    jobs = [Job("FHP_II", dx, dy, 34, seed=17, state=state, force_dir="x", force_p=p,
                force_region=(force["x0"], force["x1"], force["y0"], force["y1"])) for _ in range(2)]
    want = orc.run(2, dx, dy, np.zeros(dx * dy, np.uint8), state, 17, 0, 34, force, nthreads=8)
    with Batch(hbm_budget=10**9) as b:
        ids = [b.submit(j) for j in jobs]
        b.wait(timeout=60)
        for i in ids:
            np.testing.assert_array_equal(b.result(i)[0], want)


@pytest.mark.parametrize("p", [0.049, 0.5])
def test_windows_of_one_pass(p):
    """A region whose windows hold one pass: passes of whole groups of steps
    where most words fire, and any number else, against a fixed shape."""
    from lgca_amd import Lattice
    dx, dy = 8200, 4000
    print(f"[window] {dx}x{dy} p={p}", flush=True)
    lats = [Lattice(2, dim_x=dx, dim_y=dy, coarse_graining_radius=1, seed=5) for _ in range(2)]
    lats[1].set_tuning(4, 16)
    for lat in lats:
        lat.init_random(0.3)
        lat.set_step(2)
        lat.set_forcing("y", p)
        for n in (3, 61, 14):
            lat.step(n)
    np.testing.assert_array_equal(lats[0].get_state_u8(), lats[1].get_state_u8())
    for lat in lats:
        lat.close()
