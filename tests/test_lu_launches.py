"""The launches of nla_getrf2's host side (nla_lu.hip compiled for the CPU,
tests/emu/emu_lu.cpp): how several host threads share a stream's exchange
buffer, and which calls need one."""
import ctypes

import pytest

from test_kernel_order import build


@pytest.fixture(scope="module")
def lu(tmp_path_factory):
    return build(tmp_path_factory, "emu_lu")


def launches(lu, dtype, m, n, threads=1, stream=64, capturing=0):
    """(status, [(thread, groups, kernel)])"""
    out = ctypes.create_string_buffer(1 << 20)
    st = lu.emu_getrf2(dtype, ctypes.c_int64(m), ctypes.c_int64(n), threads, ctypes.c_int64(stream), capturing, out,
                       ctypes.c_int64(len(out)))
    rows = [line.split(" ", 2) for line in out.value.decode().splitlines()]
    return st, [(int(t), int(g), k) for t, g, k in rows]


def is_panel(row):
    """A panel that exchanges rows among several groups."""
    return "lu_panel_kernel" in row[2] and row[1] > 1


@pytest.mark.parametrize("threads", [1, 3])
def test_panel_and_its_recovery_stay_together(lu, threads):
    """A panel of several groups saves its block in the stream's buffer for the
    recovery launch behind it; no other thread's panel may come in between and
    save its own there."""
    st, log = launches(lu, 1, 600, 192, threads)
    assert st == 0
    users = [row for row in log if is_panel(row) or "lu_panel_recover_kernel" in row[2]]
    assert len(users) == 2 * 3 * threads
    for panel, recover in zip(users[::2], users[1::2]):
        assert is_panel(panel) and not is_panel(recover) and panel[0] == recover[0], users
