"""The launches of nla_getrf2's host side (nla_lu.hip compiled for the CPU,
tests/emu/emu_lu.cpp): how several host threads share a stream's exchange
buffer, and which calls need one."""
import ctypes

import numpy as np
import pytest

from test_kernel_order import build, ptr


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


@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("m,n", [(129, 64), (1000, 64), (4096, 33), (4096, 1), (128, 64), (700, 65), (40, 4096)])
def test_thin_factorization_is_captured_on_a_new_stream(lu, dtype, m, n):
    """A captured call on a stream that has factored nothing: no allocation
    (which a capture does not allow) and no launch that uses the stream's
    exchange buffer, so that graphs of such calls may run side by side."""
    before = lu.emu_allocated()
    st, log = launches(lu, dtype, m, n, stream=1000 + m + n, capturing=1)
    assert st == 0 and lu.emu_allocated() == before
    assert not any(is_panel(row) or "recover" in row[2] for row in log)
    assert log


def test_captured_after_a_call_of_its_size(lu):
    """With the stream's buffer there, a wide captured call uses the panels; a
    thin one still shares nothing."""
    assert launches(lu, 1, 1000, 700, stream=5000)[0] == 0
    st, log = launches(lu, 1, 1000, 700, stream=5000, capturing=1)
    assert st == 0 and any(is_panel(row) for row in log)
    st, log = launches(lu, 1, 1000, 64, stream=5000, capturing=1)
    assert st == 0 and not any(is_panel(row) for row in log)
    # a tall thin call has left the buffer of tall blocks only
    assert launches(lu, 1, 5000, 64, stream=5001)[0] == 0
    assert launches(lu, 1, 5000, 2000, stream=5001, capturing=1)[0] == 0


def test_buffer_of_small_factorizations(lu):
    """Up to 4096 rows a stream's buffer stays below 3 MB."""
    before = lu.emu_allocated()
    assert launches(lu, 1, 4096, 100, stream=6000)[0] == 0
    assert 0 < lu.emu_allocated() - before < 3 << 20


def test_threads_have_buffers_of_their_own_for_their_own_streams(lu):
    """hipStreamPerThread is one handle for a different stream in every thread:
    their panels run at the same time and must not share a buffer."""
    before = lu.emu_allocated()
    assert launches(lu, 1, 600, 64, threads=1, stream=7000)[0] == 0
    one = lu.emu_allocated() - before
    assert launches(lu, 1, 600, 64, threads=3, stream=2)[0] == 0
    assert lu.emu_allocated() - before == 4 * one


def pivots(kind, m, b, K, rng):
    k = np.arange(b, b + K)
    p = {"random": lambda: rng.integers(k, m), "same": lambda: np.full(K, m - 1), "next": lambda: np.minimum(k + 1, m - 1),
         "self": lambda: k, "few": lambda: np.maximum(k, rng.choice([m - 1, m // 2, m - 7], K)),
         "near": lambda: np.minimum(k + rng.integers(0, 4, K), m - 1),
         "back": lambda: np.maximum(k, m - 1 - k)}[kind]()
    return p + 1


@pytest.mark.parametrize("m,b,K", [(5, 0, 5), (700, 0, 64), (1500, 100, 1024), (1500, 3, 1025), (3000, 0, 2500)])
@pytest.mark.parametrize("kind", ["random", "same", "next", "self", "few", "near", "back"])
def test_interchanges_composed(lu, kind, m, b, K):
    """The kernel that applies K interchanges as one permutation against the
    swaps one after the other, for scattered, repeated and chained targets."""
    rng = np.random.default_rng(m + K)
    ipiv = np.zeros(m, np.int64)
    ipiv[b:b + K] = pivots(kind, m, b, K, rng)
    ref = np.arange(3 * m, dtype=np.float64).reshape(3, m)
    got = [ref.copy() for _ in range(2)]
    for i in range(b, b + K):
        j = ipiv[i] - 1
        ref[:, [i, j]] = ref[:, [j, i]]
    for rev, g in enumerate(got):
        assert lu.emu_laswp(ctypes.c_int64(3), ptr(g), ctypes.c_int64(m), ctypes.c_int64(b), K, m - b, ptr(ipiv), rev) == 0
        assert np.array_equal(g, ref), kind
