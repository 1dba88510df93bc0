"""Which kernel a diagonal panel takes (launch_panel, compiled for the CPU with
tests/emu/emu_panel.cpp)."""
import ctypes

import pytest

from test_kernel_order import build


@pytest.fixture(scope="module")
def panel(tmp_path_factory):
    lib = build(tmp_path_factory, "emu_panel")

    def launch(dtype, trmm, n, m, kc=0, bcol=0, unit=0, strip=16, waves=0):
        """(columns per group, threads)"""
        out = ctypes.create_string_buffer(1 << 10)
        assert lib.emu_panel(dtype, trmm, n, ctypes.c_int64(m), kc, bcol, unit, strip, waves, out,
                             ctypes.c_int64(len(out))) == 0
        groups, threads, _ = out.value.decode().split(" ", 2)
        return -(-m // int(groups)), int(threads)
    return launch


@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("trmm", [0, 1])
@pytest.mark.parametrize("n", [64, 192, 512, 768])
@pytest.mark.parametrize("waves", [0, 4, 8])
def test_strip_setting_is_what_runs(panel, dtype, trmm, n, waves):
    """32 columns per group wherever the setting asks for them, but in FP64
    above 512 rows, whose strip does not fit; the waves that were asked for up
    to 512 rows."""
    cols, threads = panel(dtype, trmm, n, 3200, strip=32, waves=waves)
    assert cols == (16 if dtype == 1 and n > 512 else 32)
    assert threads == (256 if waves == 4 or n > 512 else 512)
    cols, threads = panel(dtype, trmm, n, 3200, strip=16, waves=4)
    assert (cols, threads) == (16, 256)
