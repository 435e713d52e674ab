"""lgca_batch_result around the slots its arrays pass through: sizes below,
at and past one slot and past two, with last bytes that fill no 16; every choice
of arrays; a pinned destination; four threads at once.  The bits must be those
of the single-lattice path, and nothing past an array's end is written."""
import threading

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = [(33, 10, 1), (70, 30, 3), (1024, 512, 256), (1025, 512, 8), (2047, 1026, 1)]


def job(dim_x, dim_y, radius):
    from lgca_amd.batch import Job
    return Job("FHP_II", dim_x, dim_y, 6, seed=dim_x, coarse_radius=radius, fill=0.3)


def alone(j):
    from lgca_amd import Lattice
    lat = Lattice(j.model, dim_x=j.dim_x, dim_y=j.dim_y, coarse_graining_radius=j.coarse_radius, seed=j.seed)
    lat.init_random(j.fill)
    lat.step(j.steps)
    state = lat.get_state_u8().reshape(-1)
    lat.copy_data_to_output_buffer()
    lat.post_process(cells=False)
    got = state.copy(), lat.mean_density().reshape(-1).copy(), lat.mean_momentum().reshape(-1).copy()
    lat.close()
    return got


def fetch(batch, jid, want, take):
    """The arrays in `take`, each with 64 bytes of guard behind it."""
    from lgca_amd import _capi as capi
    bufs = [np.full(w.nbytes + 64, 0xA5, dtype=np.uint8) if t else None for w, t in zip(want, take)]
    ptr = [b.ctypes.data if b is not None else None for b in bufs]
    assert capi.lib().lgca_batch_result(batch._h, jid, *ptr) == 0
    for b, w in zip(bufs, want):
        if b is not None:
            assert np.array_equal(b[:w.nbytes], w.view(np.uint8))
            assert (b[w.nbytes:] == 0xA5).all()


@pytest.mark.parametrize("size", SIZES)
def test_arrays_through_the_slots(size):
    from lgca_amd import _capi as capi
    from lgca_amd.batch import Batch
    j = job(*size)
    want = alone(j)
    with Batch(hbm_budget=10 ** 9) as b:
        i = b.submit(j)
        b.wait()
        for take in [(1, 1, 1), (1, 0, 0), (0, 1, 0), (0, 0, 1), (0, 1, 1), (0, 0, 0)]:
            fetch(b, i, want, take)
        pinned = torch.zeros(want[0].nbytes, dtype=torch.uint8, pin_memory=True)
        md = np.empty_like(want[1])
        assert capi.lib().lgca_batch_result(b._h, i, pinned.data_ptr(), md.ctypes.data, None) == 0
        assert np.array_equal(pinned.numpy(), want[0]) and np.array_equal(md, want[1])


def test_threads_at_once():
    from lgca_amd.batch import Batch
    jobs = [job(*s) for s in SIZES]
    want = [alone(j) for j in jobs]
    failed = []
    with Batch(hbm_budget=10 ** 9) as b:
        ids = [b.submit(j) for j in jobs]
        b.wait()

        def work(t):
            try:
                for r in range(8):
                    k = (t + r) % len(ids)
                    fetch(b, ids[k], want[k], (1, 1, 1))
            except Exception as e:  # noqa: BLE001
                failed.append(repr(e))

        threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    assert not failed, failed
