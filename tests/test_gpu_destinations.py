"""Results fetched into other than ordinary host memory: lgca_post_process with
destinations on the GPU and in pinned memory gives the bits that it gives
ordinary arrays, in any mixture."""
import ctypes as C
import itertools

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_post_process_destinations():
    import torch

    from lgca_amd import Lattice
    from lgca_amd._capi import check, lib
    lat = Lattice(2, dim_x=330, dim_y=128, coarse_graining_radius=8, seed=3)
    lat.init_random(0.3)
    lat.copy_data_to_output_buffer()
    lat.post_process()
    want = [lat.cell_density(), lat.cell_momentum(), lat.mean_density(), lat.mean_momentum()]
    make = {"none": lambda n: None,
            "host": lambda n: torch.zeros(n, dtype=torch.float32),
            "pinned": lambda n: torch.zeros(n, dtype=torch.float32, pin_memory=True),
            "device": lambda n: torch.zeros(n, dtype=torch.float32, device="cuda")}
    for cells, coarse_d, coarse_m in itertools.product(("none", "host", "device"), make, make):
        kinds = (cells, cells, coarse_d, coarse_m)
        print("[post_process]", kinds, flush=True)
        out = [make[k](w.size) for k, w in zip(kinds, want)]
        torch.cuda.synchronize()
        ptr = [C.c_void_p(o.data_ptr()) if o is not None else None for o in out]
        check(lib().lgca_post_process(lat.handle, *ptr), lat.handle)
        for o, w in zip(out, want):
            if o is not None:
                np.testing.assert_array_equal(o.cpu().numpy(), w)
    lat.close()
