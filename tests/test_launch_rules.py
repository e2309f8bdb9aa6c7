"""The host's launch rules (pippin_amd/csrc/launch_rules.hpp), without a device."""
import pytest

from tests.emu.pyemu import lib


@pytest.mark.parametrize("envs", [1, 7, 1023, 1024, 1025, 5120, 8192, 16384])
@pytest.mark.parametrize("per_cu,cus", [(20, 256), (4, 256), (8, 64)])
def test_the_general_sweeps_fill_the_device(envs, per_cu, cus):
    """Every env of a batch may be left to them: a wavefront each, as far as the device holds them."""
    assert lib().emu_general_sweep_blocks(envs, per_cu, cus) == min(envs, per_cu * cus)
