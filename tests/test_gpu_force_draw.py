"""Force decisions of regions whose (row, word) pairs end around a workgroup's
1024, from windows that start inside a four-step group, at probabilities where
no word, a few and every word fires, in single lattices and in batches, against
the oracle."""
import numpy as np
import pytest

from oracle import oracle as orc

pytestmark = pytest.mark.gpu


# words x rows of the forced region: 1023, 1024, 1025 and 4100 pairs, one row, one word
@pytest.mark.parametrize("words,rows", [(33, 31), (32, 32), (41, 25), (82, 50), (130, 1), (1, 700)])
@pytest.mark.parametrize("p", [1e-7, 1e-3, 0.05, 0.7, 1.0])
def test_draws_match_the_oracle(words, rows, p):
    from lgca_amd import Batch, Job, Lattice
    dx, dy = 32 * words + 40, rows + 6 + (rows & 1)
    rng = np.random.default_rng(words * rows)
    state = rng.integers(0, 128, dx * dy, dtype=np.uint8)
    force = dict(dir="x", p=p, x0=5, x1=5 + 32 * words - 10, y0=3, y1=3 + rows)
    print(f"[draw] {words} words x {rows} rows p={p}", flush=True)
    for step0, calls in ((0, (9,)), (3, (2, 70)), (6, (1, 1, 7))):
        lat = Lattice(2, dim_x=dx, dim_y=dy, coarse_graining_radius=1, seed=17)
        lat.set_state_u8(state)
        lat.set_step(step0)
        lat.set_forcing("x", p, force["x0"], force["x1"], force["y0"], force["y1"])
        for n in calls:
            lat.step(n)
        want = orc.run(2, dx, dy, None, state, 17, step0, sum(calls), force, nthreads=8)
        np.testing.assert_array_equal(lat.get_state_u8(), want)
        lat.close()
    jobs = [Job("FHP_II", dx, dy, n, seed=17, state=state, force_dir="x", force_p=p,
                force_region=(force["x0"], force["x1"], force["y0"], force["y1"])) for n in (3, 45)]
    with Batch(hbm_budget=10**9) as b:
        ids = [b.submit(j) for j in jobs]
        b.wait(timeout=60)
        for i, j in zip(ids, jobs):
            want = orc.run(2, dx, dy, np.zeros(dx * dy, np.uint8), state, 17, 0, j.steps, force, nthreads=8)
            np.testing.assert_array_equal(b.result(i)[0], want)
