"""Passes held in blocks (the automatic launch path of lattices that walks
cannot fill the GPU with) against the oracle, where their blocks can go wrong:
every number of steps a pass may have, from every step offset; rows of one
word, of several segments per wave, of exactly 64 words and of several strips,
with short last words; lattices of fewer rows than a block holds and row
tiles with a short last one; walls, slip, obstacles and forcing on some waves
only; and shapes of 1, 2, 4 and 6 rows per wave (chosen by the lattice's
size)."""
import numpy as np
import pytest

from oracle import oracle as orc

pytestmark = pytest.mark.gpu

Q = {0: 4, 1: 6, 2: 7, 3: 7}


def make_types(rng, dx, dy, kind):
    g = np.zeros((dy, dx), dtype=np.uint8)
    if kind == "pipe":
        g[0] = g[-1] = 1
    elif kind == "slip":
        g[0], g[-1], g[:, 0], g[:, -1] = 2, 2, 2, 2
    elif kind == "mixed":
        g[rng.random((dy, dx)) < 0.05] = 1
        g[rng.random((dy, dx)) < 0.03] = 2
        g[0], g[:, -1] = 2, 2
    elif kind == "cylinder":
        g[0] = g[-1] = 1
        ys, xs = np.mgrid[0:dy, 0:dx]
        g[(xs - dx // 3) ** 2 + (ys - dy // 2) ** 2 < (dy // 4) ** 2] = 1
    return g.reshape(-1)


def check(model, dx, dy, geom, force, calls, step0=0, seed=41, tune=False):
    from lgca_amd import Lattice
    rng = np.random.default_rng(dx * 3 + dy + model)
    types = make_types(rng, dx, dy, geom)
    state = rng.integers(0, 1 << Q[model], dx * dy, dtype=np.uint8)
    print(f"[block] model={model} {dx}x{dy} {geom} {force} calls={calls} step0={step0}", flush=True)
    lat = Lattice(model, dim_x=dx, dim_y=dy, coarse_graining_radius=1, seed=seed)
    if geom:
        lat.set_cell_types(types)
    lat.set_state_u8(state)
    lat.set_step(step0)
    if force:
        lat.set_forcing(force["dir"], force["p"], force.get("x0", 0), force.get("x1"), force.get("y0", 0),
                        force.get("y1"))
    if tune:
        lat.tune()
    for n in calls:
        lat.step(n)
    want = orc.run(model, dx, dy, types, state, seed, step0, sum(calls), force, nthreads=8)
    np.testing.assert_array_equal(lat.get_state_u8(), want)
    lat.close()


CASES = [
    (0, 2, 2, None, None),
    (0, 33, 7, "mixed", dict(dir="y", p=0.3)),                        # odd rows, two short words
    (1, 17, 30, "slip", dict(dir="x", p=0.2)),                        # one word per row
    (2, 96, 300, "mixed", dict(dir="x", p=0.1, y0=50, y1=250)),       # 21 segments, idle lanes
    (3, 700, 90, "cylinder", dict(dir="x", p=0.01, x0=0, x1=64)),     # 2 segments, short word
    (1, 1001, 202, "slip", dict(dir="y", p=0.05, x0=300, x1=500)),
    (0, 1500, 51, "pipe", dict(dir="x", p=0.4, x0=31, x1=33)),        # one strip that wraps
    (2, 2048, 70, "cylinder", dict(dir="x", p=0.05)),                 # rows of exactly 64 words
    (1, 2048, 64, None, None),
    (3, 2017, 40, "mixed", None),                                     # 64 words, the last of one cell
    (2, 4100, 60, "mixed", dict(dir="y", p=0.1, x0=2000, x1=4100)),   # strips, short last word
    (2, 4096, 64, "pipe", dict(dir="x", p=0.02, x0=0, x1=40)),        # force on the wrapped words
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"m{c[0]}_{c[1]}x{c[2]}_{c[3]}")
@pytest.mark.parametrize("step0", [0, 3])
def test_block_passes_match_the_oracle(case, step0):
    check(*case, calls=(1, 2, 5, 9, 61), step0=step0)


@pytest.mark.parametrize("steps", range(1, 31))
def test_every_pass_length(steps):
    check(2, 260, 48, "cylinder", dict(dir="x", p=0.1), calls=(steps,), step0=steps % 4)


# larger lattices take more rows per wave; the last two are the plan's 4 and 6
@pytest.mark.parametrize("model,dx,dy,geom,force,n", [
    (2, 1480, 740, "pipe", dict(dir="x", p=0.01), 37),
    (3, 4400, 2200, "cylinder", dict(dir="x", p=0.02, x0=0, x1=64), 23),
    (0, 6016, 3001, None, None, 31),
    (1, 8000, 2600, "slip", dict(dir="y", p=0.002), 19),
    (2, 8192, 4000, "pipe", dict(dir="x", p=0.005, y0=100, y1=1000), 13)])
def test_block_shapes_of_larger_lattices(model, dx, dy, geom, force, n):
    check(model, dx, dy, geom, force, calls=(n,), step0=6)


@pytest.mark.parametrize("dx,dy,geom", [(256, 256, None), (1001, 300, "mixed"), (2048, 130, "pipe")])
def test_tuned_block_shapes(dx, dy, geom):
    check(2, dx, dy, geom, dict(dir="x", p=0.03), calls=(7, 64, 20), step0=1, tune=True)


def test_batch_blocks_match_the_oracle():
    """A batch small enough to run in blocks: every model, rows of several
    strips and segments, short last words, forcing, given cell types, and steps
    that end in the middle of a round."""
    from lgca_amd import Batch, Job
    rng = np.random.default_rng(8)
    jobs, want = [], []
    for i, (model, dx, dy, geom, force) in enumerate(
            [c for c in CASES if c[1] > 16] + [(2, 2100, 90, "mixed", None), (0, 4160, 33, "slip", None)]):
        types = make_types(rng, dx, dy, geom)
        state = rng.integers(0, 1 << Q[model], dx * dy, dtype=np.uint8)
        f = force or {}
        jobs.append(Job(model, dx, dy, 17 + 5 * i, seed=60 + i, geometry="types", cell_types=types, state=state,
                        force_dir=f.get("dir"), force_p=f.get("p", 0.0),
                        force_region=(f.get("x0", 0), f.get("x1") or dx, f.get("y0", 0), f.get("y1") or dy)))
        want.append(orc.run(model, dx, dy, types, state, 60 + i, 0, jobs[-1].steps, force, nthreads=8))
    print(f"[block batch] {len(jobs)} jobs", flush=True)
    with Batch(hbm_budget=4 * 10**9) as b:
        ids = [b.submit(j) for j in jobs]
        b.wait(timeout=60)
        assert b.stats()["wave_target"] <= 16  # waves per workgroup: the rounds ran in blocks
        for i, w in zip(ids, want):
            np.testing.assert_array_equal(b.result(i)[0], w)


# rows that share waves with the next row tile's: widths whose rows end within,
# at and past a wave's words, short last words with one and two halo words,
# heights whose last tile is short or the only one, every kind of cell and
# force, and lattices large enough for each number of rows per wave
@pytest.mark.parametrize("case", [
    (2, 1100, 130, "slip", dict(dir="y", p=0.05)), (1, 1056, 64, None, None), (0, 1057, 63, "mixed", dict(dir="x", p=0.1)),
    (2, 1969, 200, "pipe", dict(dir="x", p=0.1)), (3, 2050, 46, "mixed", dict(dir="x", p=0.2)),
    (1, 4017, 500, "cylinder", dict(dir="x", p=0.05, x0=0, x1=64)), (2, 4400, 740, "pipe", dict(dir="x", p=0.01)),
    (0, 2700, 1001, "slip", None), (2, 6000, 1500, "cylinder", dict(dir="x", p=0.01)), (1, 4400, 2200, None, None),
    (3, 2177, 2, "pipe", None), (2, 6000, 3000, "pipe", dict(dir="y", p=0.01))], ids=lambda c: f"m{c[0]}_{c[1]}x{c[2]}")
@pytest.mark.parametrize("tune", [False, True])
def test_rows_packed_into_waves(case, tune):
    check(*case, calls=(1, 3, 26), step0=2, tune=tune)
