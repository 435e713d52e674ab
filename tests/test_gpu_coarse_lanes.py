"""Coarse fields of lattices with many small coarse cells, which a lane each
takes, against the oracle bit for bit: more coarse cells than 64 times the
GPU's CUs, a last wave that is not full, and the wrapped column."""
import pytest

from test_gpu_reductions import test_coarse_fields_bit_exact_at_unit_edges as check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("model", [0, 1, 2])
@pytest.mark.parametrize("dx,dy,r", [(600, 302, 1), (2, 65000, 1), (1203, 902, 2), (3208, 2056, 4)])
def test_coarse_fields_bit_exact_by_lanes(model, dx, dy, r):
    check(model, dx, dy, r)
