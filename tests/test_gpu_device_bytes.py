"""lgca_info.device_bytes: counts the count-mode force's workspace, and shows that
the force windows of a tuned lattice stay within 64 MiB where its passes do."""
import pytest

pytestmark = pytest.mark.gpu


def test_device_bytes_hold_the_force_workspace():
    from lgca_amd import Lattice
    lat = Lattice("FHP_II", dim_x=640, dim_y=400, coarse_graining_radius=1, seed=3)
    lat.init_random(0.3)
    before = lat.info().device_bytes
    lat.apply_body_force_count("x", 1000)
    listed = 16 * 1000 // 256 * 256  # tries listed ahead, 8 bytes each
    grown = lat.info().device_bytes - before
    assert listed * 8 <= grown <= listed * 8 + 8192
    lat.apply_body_force_count("x", 500)  # fits
    assert lat.info().device_bytes - before == grown
    lat.close()


def test_tuning_keeps_force_windows_within_their_cap():
    from lgca_amd import Lattice
    # 4 MB of decisions a step, passes of up to 14 steps: windows of 64 MiB hold them
    lat = Lattice("FHP_II", dim_x=8192, dim_y=4096, coarse_graining_radius=1, seed=3)
    lat.init_random(0.3)
    before = lat.info().device_bytes
    lat.set_forcing("x", 1e-3)
    lat.tune()
    lat.step(60)
    lat.synchronize()
    assert 0 < lat.info().device_bytes - before <= 64 << 20
    lat.close()
