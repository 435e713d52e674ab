"""Bytes to and from planes, cell types, hash fill and cell fields at the widths
where their kernels' work splits can go wrong: rows shorter than one 16-byte
access, rows that end within, at and one past a half word, a word, a wave's
cells and a workgroup's lanes, rows that start at any byte, and a caller's
device buffer that starts at any byte."""
import numpy as np
import pytest
import torch

from lgca_amd import LgcaError
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

Q = {0: 4, 1: 6, 2: 7, 3: 7}
SEED = 0x0123456789ABCDEF
WIDTHS = [2, 15, 16, 17, 31, 32, 33, 48, 63, 65, 127, 128, 129, 257, 511, 513, 1023, 1025, 2047, 4097, 4130]


def cases():
    return [(n % 4, w, [2, 4, 6, 34][n // 4 % 4]) for n, w in enumerate(WIDTHS)]


def make(model, dx, dy):
    from lgca_amd import Lattice
    return Lattice(model, dim_x=dx, dim_y=dy, coarse_graining_radius=1, seed=SEED)


@pytest.mark.parametrize("model,dx,dy", cases())
def test_state_bytes_round_trip(model, dx, dy):
    from lgca_amd import _capi as capi
    print(f"[state] model={model} {dx}x{dy}", flush=True)
    lat = make(model, dx, dy)
    n = dx * dy
    rng = np.random.default_rng(n)
    state = rng.integers(0, 1 << Q[model], n, dtype=np.uint8)
    lat.set_state_u8(state)
    assert np.array_equal(lat.get_state_u8(), state)
    assert lat.get_n_particles() == orc.count_particles(state)  # nothing past the rows' ends
    for off in (1, 7):
        buf = torch.full((n + 32,), 0xA5, dtype=torch.uint8, device="cuda")
        dev = torch.zeros(n + 32, dtype=torch.uint8, device="cuda")
        dev[off:off + n] = torch.from_numpy(state[::-1].copy()).cuda()
        torch.cuda.synchronize()
        capi.check(capi.lib().lgca_set_state_u8_device(lat.handle, dev.data_ptr() + off), lat.handle)
        capi.check(capi.lib().lgca_get_state_u8_device(lat.handle, buf.data_ptr() + off), lat.handle)
        got = buf.cpu().numpy()
        assert np.array_equal(got[off:off + n], state[::-1])
        assert (got[:off] == 0xA5).all() and (got[off + n:] == 0xA5).all()
    for cell in (0, n // 2, n - 1):
        bad = state.copy()
        bad[cell] |= 1 << Q[model]
        with pytest.raises(LgcaError):
            lat.set_state_u8(bad)
    lat.close()


@pytest.mark.parametrize("model,dx,dy", cases())
def test_types_fill_and_fields(model, dx, dy):
    print(f"[types] model={model} {dx}x{dy}", flush=True)
    lat = make(model, dx, dy)
    n = dx * dy
    rng = np.random.default_rng(n + 1)
    for share in (0.0, 0.01, 0.6):
        types = np.where(rng.random(n) < share, rng.integers(1, 3, n), 0).astype(np.uint8)
        lat.set_cell_types(types)
        assert np.array_equal(lat.get_cell_types(), types)
        for fill in (0.0, 0.3, 1.0):
            lat.set_state_u8(np.zeros(n, np.uint8))
            lat.init_random(fill)
            assert np.array_equal(lat.get_state_u8(), orc.init_random(model, dx, dy, types, SEED, fill))
        # a step sees the solid cells where the rows' ranges say they are
        lat.init_random(0.3)
        want = orc.step(model, dx, dy, types, lat.get_state_u8(), SEED, 0)
        lat.set_step(0)
        lat.step(1)
        assert np.array_equal(lat.get_state_u8(), want)
    for cell, value in ((0, 3), (n // 2, 4), (n - 1, 255)):
        bad = types.copy()
        bad[cell] = value
        with pytest.raises(LgcaError):
            lat.set_cell_types(bad)
    state = rng.integers(0, 1 << Q[model], n, dtype=np.uint8)
    lat.set_state_u8(state)
    lat.copy_data_to_output_buffer()
    lat.post_process()
    density, momentum = orc.cell_post_process(model, dx, dy, state)
    assert np.array_equal(lat.cell_density(), density)
    assert np.array_equal(lat.cell_momentum(), momentum.reshape(-1))
    lat.close()


@pytest.mark.parametrize("dx,dy", [(1200, 1024), (2049, 3002), (4096, 2048)])
def test_large_results_arrive_whole(dx, dy):
    """Results on both sides of the size from which several threads copy them,
    with a ragged last chunk, into ordinary and into pinned memory, twice into
    the same arrays, and from two lattices on two threads at once."""
    import threading
    lats = [make(2, dx, dy), make(0, dx, dy)]
    rng = np.random.default_rng(dx)
    n = dx * dy
    states = [rng.integers(0, 1 << Q[m], n, dtype=np.uint8) for m in (2, 0)]
    types = (rng.random(n) < 0.1).astype(np.uint8)
    bad = []

    def check(lat, state, model):
        from lgca_amd import _capi as capi
        for _ in range(2):
            lat.set_cell_types(types)
            lat.set_state_u8(state)
            lat.copy_data_to_output_buffer()
            lat.post_process()
            density, momentum = orc.cell_post_process(model, dx, dy, state)
            pinned = torch.empty(n, dtype=torch.uint8).pin_memory()
            capi.check(capi.lib().lgca_get_state_u8(lat.handle, pinned.data_ptr()), lat.handle)
            for name, got, want in (("state", lat.get_state_u8(), state), ("pinned", pinned.numpy(), state),
                                    ("types", lat.get_cell_types(), types), ("density", lat.cell_density(), density),
                                    ("momentum", lat.cell_momentum(), momentum.reshape(-1))):
                if not np.array_equal(got, want):
                    bad.append((model, name))
            state = state[::-1].copy()

    threads = [threading.Thread(target=check, args=a) for a in zip(lats, states, (2, 0))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    for lat in lats:
        lat.close()


@pytest.mark.parametrize("dy", [34, 1000, 65534])
def test_rows_solid_ranges_reach_the_walks(dy):
    """The launch order is made from every row's range of solid cells: set twice
    and walked against the oracle, up to the most rows there can be."""
    dx, steps = 64, 9
    rng = np.random.default_rng(dy)
    state = rng.integers(0, 1 << Q[2], dx * dy, dtype=np.uint8)
    lat = make(2, dx, dy)
    lat.set_tuning(8, 16)
    for _ in range(2):
        types = np.zeros((dy, dx), dtype=np.uint8)
        types[0], types[-1] = 1, 1
        types[rng.integers(0, dy, max(2, dy // 50)), rng.integers(0, dx, max(2, dy // 50))] = 1
        types = types.reshape(-1)
        lat.set_cell_types(types)
        lat.set_state_u8(state)
        lat.set_step(0)
        lat.step(steps)
        assert np.array_equal(lat.get_state_u8(), orc.run(2, dx, dy, types, state, SEED, 0, steps, None, nthreads=8))
    lat.close()
