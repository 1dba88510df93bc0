"""Recursive LU with partial pivoting on the device (nla_getrf2, the
reference's getrf2!, src/lu.jl:185-300) against the oracle's restatement,
which is itself pinned to LAPACK dgetrf (tests/test_oracle.py).

FP64: the same pivots as the oracle and factors equal to rounding.  FP32:
P*L*U = A to the bound of the reference tests' check (test/lu.jl:25-28,
relative error of the reconstruction) and |L| <= 1; pivots are not compared
in FP32, where a different summation order can flip a near tie.
"""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda"
SHAPES = [(1, 1), (1, 7), (7, 1), (2, 2), (3, 5), (64, 64), (100, 90), (90, 100), (257, 300), (513, 513),
          (1000, 700)]


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(np.asarray(a).T)).to(DEV).t()


def host(t):
    torch.cuda.synchronize()
    return t.detach().cpu().numpy()


@pytest.mark.parametrize("m,n", SHAPES)
def test_fp64_matches_oracle(nla, m, n):
    rng = np.random.default_rng(m * 1009 + n)
    A = rng.standard_normal((m, n))
    LU, ipiv, info = nla.getrf2_(dev(A))
    ref, ref_piv, ref_info = O.getrf2(A)
    assert info == ref_info == 0
    assert np.array_equal(host(ipiv), ref_piv), (m, n)
    got = host(LU)
    assert np.max(np.abs(got - ref)) <= 1e-11 * max(1.0, np.max(np.abs(ref))), (m, n)
    assert np.linalg.norm(O.lu_reconstruct(got, host(ipiv)) - A) <= 20 * max(m, n) * 2.2e-16 * np.linalg.norm(A)


@pytest.mark.parametrize("m,n", [(64, 64), (300, 257), (257, 300), (1000, 1000)])
def test_fp32_reconstructs(nla, m, n):
    rng = np.random.default_rng(7 + m + n)
    A = rng.standard_normal((m, n)).astype(np.float32)
    LU, ipiv, info = nla.getrf2_(dev(A))
    got, piv = host(LU), host(ipiv)
    assert info == 0
    k = min(m, n)
    assert np.all((piv >= np.arange(1, k + 1)) & (piv <= m))
    assert np.max(np.abs(np.tril(got[:, :k], -1))) <= 1.0 + 1e-6
    err = np.linalg.norm(O.lu_reconstruct(got, piv) - A) / np.linalg.norm(A)
    assert err <= 20 * max(m, n) * 1.2e-7, err


def test_singular_info_and_padded_lda(nla):
    """A zero third column: info = 3 (U(3,3) exactly zero) and the rest of
    the factorization as the oracle's; A inside a larger allocation (lda > m)
    with the rows past m untouched."""
    rng = np.random.default_rng(3)
    A = rng.standard_normal((40, 30))
    A[:, 2] = 0.0
    big = torch.full((30, 48), 7.0, dtype=torch.float64, device=DEV).t()  # 48 x 30, lda 48
    big[:40].copy_(torch.from_numpy(A).to(DEV))
    view = big[:40]
    LU, ipiv, info = nla.getrf2_(view)
    ref, ref_piv, ref_info = O.getrf2(A)
    assert info == ref_info == 3
    assert np.array_equal(host(ipiv), ref_piv)
    assert np.max(np.abs(host(LU) - ref)) <= 1e-12 * np.max(np.abs(ref))
    assert torch.all(big[40:] == 7.0)


def test_empty_and_invalid(nla):
    E = torch.empty((0, 5), dtype=torch.float64, device=DEV)
    _, ipiv, info = nla.getrf2_(E)
    assert info == 0 and ipiv.numel() == 0
    with pytest.raises(ValueError):
        nla.getrf2_(torch.ones(4, 5, dtype=torch.float64, device=DEV))  # row-major
    with pytest.raises(ValueError):
        nla.getrf2_(dev(np.eye(4)), ipiv=torch.empty(2, dtype=torch.int64, device=DEV))
    with pytest.raises(ValueError):
        nla.getrf2_(dev(np.eye(4)).to(torch.int32))


def test_large_fp64_self_certified(nla):
    """n = 4096: P*L*U = A checked on the device in FP64."""
    n = 4096
    g = torch.Generator(device=DEV)
    g.manual_seed(5)
    A0 = torch.empty((n, n), dtype=torch.float64, device=DEV).t().normal_(generator=g)
    A = A0.clone()
    LU, ipiv, info = nla.getrf2_(A)
    assert info == 0
    L = torch.tril(LU, -1) + torch.eye(n, dtype=torch.float64, device=DEV)
    U = torch.triu(LU)
    R = L @ U
    perm = torch.arange(n, device=DEV)
    piv = ipiv.cpu().numpy() - 1
    p = perm.cpu().numpy()
    for i in range(n):  # row i of P*A came from row p[i]
        j = piv[i]
        p[i], p[j] = p[j], p[i]
    PA = A0[torch.from_numpy(p).to(DEV)]
    err = (torch.linalg.norm(R - PA) / torch.linalg.norm(A0)).item()
    assert err <= 1e-13, err
    assert torch.max(torch.abs(torch.tril(LU, -1))).item() <= 1.0


@pytest.fixture
def split_rows():
    """Set the row count from which leaves spread over several work-groups;
    restores the previous value."""
    from nextla_amd import _lib
    olds = []

    def set_(v):
        olds.append(_lib.set_config(_lib.NLA_CFG_LU_SPLIT_ROWS, v))
    yield set_
    if olds:
        _lib.set_config(_lib.NLA_CFG_LU_SPLIT_ROWS, olds[0])


@pytest.mark.parametrize("m,n", SHAPES + [(2049, 8), (4097, 20)])
def test_split_leaf_matches_oracle(nla, split_rows, m, n):
    """Every leaf through the multi-work-group kernel (threshold 1 row): the
    same pivots as the oracle and factors equal to rounding, for the shapes
    above and blocks with a partial last work-group."""
    split_rows(1)
    rng = np.random.default_rng(m * 7919 + n)
    A = rng.standard_normal((m, n))
    LU, ipiv, info = nla.getrf2_(dev(A))
    ref, ref_piv, ref_info = O.getrf2(A)
    assert info == ref_info == 0
    assert np.array_equal(host(ipiv), ref_piv), (m, n)
    assert np.max(np.abs(host(LU) - ref)) <= 1e-11 * max(1.0, np.max(np.abs(ref))), (m, n)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("m,n", [(131072, 8), (131073, 8), (6000, 8), (8192, 64)])
def test_split_leaf_equals_single_group_leaf(nla, split_rows, dtype, m, n):
    """Tall leaves up to the 64-work-group limit (131072 rows; one more row
    takes the one-work-group kernel): the split kernel gives the same pivots
    and the same factors as the one-work-group leaf on the same input."""
    g = torch.Generator(device=DEV)
    g.manual_seed(m + n)
    A0 = torch.empty((n, m), dtype=dtype, device=DEV).normal_(generator=g).t()
    split_rows(0)
    L1, p1, i1 = nla.getrf2_(A0.clone())
    split_rows(1)
    L2, p2, i2 = nla.getrf2_(A0.clone())
    assert i1 == i2 == 0
    assert torch.equal(p1, p2)
    tol = 1e-12 if dtype == torch.float64 else 1e-5
    assert torch.max(torch.abs(L1 - L2)).item() <= tol * torch.max(torch.abs(L1)).item()


@pytest.mark.parametrize("rows,split", [(3000, 1), (5000, 1), (5000, 0)],
                         ids=["one-group-register", "split", "global-memory"])
def test_leaf_singular_and_padded(nla, split_rows, rows, split):
    """A zero column and lda > m through each leaf kernel (m = 5000 with
    split rows 1 takes the multi-work-group kernel for its leaves, 3000 the
    one-work-group register kernel, split rows 0 the global-memory leaf):
    info, pivots and factors as the oracle's, the rows past m untouched."""
    split_rows(split)
    rng = np.random.default_rng(11)
    A = rng.standard_normal((rows, 12))
    A[:, 2] = 0.0
    big = torch.full((12, rows + 100), 7.0, dtype=torch.float64, device=DEV).t()
    big[:rows].copy_(torch.from_numpy(A).to(DEV))
    LU, ipiv, info = nla.getrf2_(big[:rows])
    ref, ref_piv, ref_info = O.getrf2(A)
    assert info == ref_info == 3
    assert np.array_equal(host(ipiv), ref_piv)
    assert np.max(np.abs(host(LU) - ref)) <= 1e-12 * np.max(np.abs(ref))
    assert torch.all(big[rows:] == 7.0)


@pytest.mark.parametrize("rows,split", [(5000, 1), (5000, 0), (2000, 1)])
def test_leaf_all_nan_column(nla, split_rows, rows, split):
    """An all-NaN column: no finite pivot, so its row stays (pivot = the row
    itself, as the oracle's first-maximum rule gives for all-NaN), info 0,
    and the NaNs spread exactly where the oracle's do."""
    split_rows(split)
    rng = np.random.default_rng(12)
    A = rng.standard_normal((rows, 10))
    A[:, 4] = np.nan
    LU, ipiv, info = nla.getrf2_(dev(A))
    ref, ref_piv, ref_info = O.getrf2(A)
    got = host(LU)
    assert info == ref_info == 0
    assert np.array_equal(host(ipiv), ref_piv)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    ok = ~np.isnan(ref)
    assert np.max(np.abs(got[ok] - ref[ok])) <= 1e-12 * np.max(np.abs(ref[ok]))


@pytest.fixture
def spin_limit():
    from nextla_amd import _lib
    olds = []

    def set_(v):
        olds.append(_lib.set_config(_lib.NLA_CFG_LU_SPIN_LIMIT, v))
    yield set_
    if olds:
        _lib.set_config(_lib.NLA_CFG_LU_SPIN_LIMIT, olds[0])


@pytest.mark.parametrize("m,n", [(20000, 8), (9000, 24)])
def test_split_leaf_timeout_is_recovered(nla, split_rows, spin_limit, m, n):
    """A grid-barrier wait of the multi-work-group leaf that runs out (forced
    from the host with a one-poll limit, so work-groups that are merely a
    little behind count as missing): the leaf is redone from its saved copy
    by the one-work-group leaf, and the factorization equals the normal one
    (pivots equal, factors to rounding), singular info included."""
    g = torch.Generator(device=DEV)
    g.manual_seed(m + n)
    A0 = torch.empty((n, m), dtype=torch.float64, device=DEV).normal_(generator=g).t()
    A0[:, 3] = 0.0
    split_rows(1)
    L1, p1, i1 = nla.getrf2_(A0.clone())
    spin_limit(1)
    for _ in range(2):
        L2, p2, i2 = nla.getrf2_(A0.clone())
        assert i1 == i2 == 4
        assert torch.equal(p1, p2)
        assert torch.max(torch.abs(L1 - L2)).item() <= 1e-12 * torch.max(torch.abs(L1)).item()
    spin_limit(0)
    L3, p3, i3 = nla.getrf2_(A0.clone())  # and the normal path after a recovery
    assert i3 == 4 and torch.equal(p1, p3) and torch.equal(L1, L3)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("m,n", [(33, 64), (128, 64), (129, 65), (257, 63), (8192, 17), (8193, 64), (32769, 33),
                                 (65537, 17)])
def test_register_panel_edges(nla, split_rows, dtype, m, n):
    """Panels at the edges of their groups (128 rows, 256 above 8192) and
    column counts (64, 32 above 32768 rows, 16 above 65536), wide and with a
    column more than the panel takes: the pivots and the factors of the
    global-memory leaf, with equal entries in a column (ties go to the first
    row) among the inputs."""
    g = torch.Generator(device=DEV)
    g.manual_seed(3 * m + n)
    A0 = torch.empty((n, m), dtype=dtype, device=DEV).normal_(generator=g).t()
    A0[:, 0] = 1.0  # every row ties for the first pivot
    split_rows(0)
    L1, p1, i1 = nla.getrf2_(A0.clone())
    split_rows(1)
    L2, p2, i2 = nla.getrf2_(A0.clone())
    assert i1 == i2 == 0 and p1[0].item() == 1
    assert torch.equal(p1, p2)
    tol = 1e-12 if dtype == torch.float64 else 1e-5
    assert torch.max(torch.abs(L1 - L2)).item() <= tol * torch.max(torch.abs(L1)).item()


@pytest.mark.parametrize("m,n", [(5000, 5000), (32768, 6656), (38913, 1300)])
def test_interchanges_large(nla, m, n):
    """Interchanges of whole halves at once, in several permutations of one
    block (32768 rows leave room for 3270 swaps at a time) and past the rows a
    permutation takes: P*A = L*U on sampled columns, in float64 (the residual
    of one factorization: a few n eps of |L||U|)."""
    g = torch.Generator(device=DEV)
    g.manual_seed(m)
    A0 = torch.empty((n, m), dtype=torch.float64, device=DEV).normal_(generator=g).t()
    LU, ipiv, info = nla.getrf2_(A0.clone())
    assert info == 0
    p = np.arange(m)
    for i, j in enumerate(ipiv.cpu().numpy() - 1):
        p[i], p[j] = p[j], p[i]
    cols = torch.tensor([0, 63, 64, n // 2, n - 1], device=DEV)
    L = torch.tril(LU, -1)
    L.diagonal().fill_(1.0)
    U = torch.triu(LU[:n])[:, cols]
    err = L @ U - A0[:, cols][torch.from_numpy(p).to(DEV)]
    bound = 4 * n * 2.2e-16 * (L.abs() @ U.abs())
    assert torch.all(err.abs() <= bound)


def test_threads_on_one_stream(nla, split_rows, spin_limit):
    """Three host threads factor matrices of their own on one stream, with and
    without waits that run out (a one-poll limit from the host): every thread's
    factors are its own, as when it is alone."""
    import threading
    from nextla_amd import _lib
    lib = _lib.load()
    split_rows(1)
    g = torch.Generator(device=DEV)
    g.manual_seed(9)
    shapes = [(9000, 24), (700, 130), (3000, 64)]
    A0 = [torch.empty((n, m), dtype=torch.float64, device=DEV).normal_(generator=g).t() for m, n in shapes]
    ref = [nla.getrf2_(a.clone()) for a in A0]
    stream = torch.cuda.Stream()
    for limit in (0, 1):
        spin_limit(limit)
        work = [[a.clone() for _ in range(6)] for a in A0]
        piv = [[torch.zeros(a.shape[1], dtype=torch.int64, device=DEV) for _ in range(6)] for a in A0]
        info = [[torch.zeros(1, dtype=torch.int64, device=DEV) for _ in range(6)] for a in A0]
        torch.cuda.synchronize()
        bad = []

        def run(i):
            m, n = shapes[i]
            for a, p, f in zip(work[i], piv[i], info[i]):
                st = lib.nla_getrf2(_lib.NLA_F64, m, n, a.data_ptr(), m, p.data_ptr(), f.data_ptr(), stream.cuda_stream)
                if st != 0:
                    bad.append(st)
        pool = [threading.Thread(target=run, args=(i,)) for i in range(3)]
        for t in pool:
            t.start()
        for t in pool:
            t.join()
        torch.cuda.synchronize()
        assert not bad
        for i in range(3):
            L, p, inf = ref[i]
            for a, q, f in zip(work[i], piv[i], info[i]):
                assert f.item() == inf == 0 and torch.equal(q, p)
                assert torch.max(torch.abs(a - L)).item() <= 1e-12 * torch.max(torch.abs(L)).item()


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("m,n", [(128, 8), (129, 8), (1024, 8), (1536, 8), (1537, 8), (2048, 5), (4096, 3), (4096, 1),
                                 (4097, 1), (513, 2)])
def test_narrow_blocks(nla, split_rows, dtype, m, n):
    """Few columns, at the edges of the rule between the single group's panel,
    the register leaf and the panel of several groups: the pivots and factors
    of the global-memory leaf, with a tied first column, a zero column and a
    column of NaN among the inputs."""
    g = torch.Generator(device=DEV)
    g.manual_seed(m + n)
    for kind in ("ties", "zero", "nan"):
        A0 = torch.empty((n, m), dtype=dtype, device=DEV).normal_(generator=g).t()
        A0[:, n // 2] = {"ties": 1.0, "zero": 0.0, "nan": float("nan")}[kind]
        split_rows(0)
        L1, p1, i1 = nla.getrf2_(A0.clone())
        split_rows(1)
        L2, p2, i2 = nla.getrf2_(A0.clone())
        assert i1 == i2 == (n // 2 + 1 if kind == "zero" else 0), kind
        assert torch.equal(p1, p2), kind
        assert torch.equal(torch.isnan(L1), torch.isnan(L2)), kind
        tol = 1e-12 if dtype == torch.float64 else 1e-5
        L1, L2 = torch.nan_to_num(L1), torch.nan_to_num(L2)
        assert torch.max(torch.abs(L1 - L2)).item() <= tol * torch.max(torch.abs(L1)).item(), kind


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("m,n", [(16384, 65), (16385, 65), (32768, 33), (32769, 17), (65536, 17), (65537, 9),
                                 (131072, 9)])
def test_tall_panels(nla, split_rows, dtype, m, n):
    """Heights where the panel's columns change (64, 32, 16 and 8), one column
    more than the narrowest of them takes: the pivots and factors of the
    global-memory leaf."""
    g = torch.Generator(device=DEV)
    g.manual_seed(m + n)
    A0 = torch.empty((n, m), dtype=dtype, device=DEV).normal_(generator=g).t()
    split_rows(0)
    L1, p1, i1 = nla.getrf2_(A0.clone())
    split_rows(1)
    L2, p2, i2 = nla.getrf2_(A0.clone())
    assert i1 == i2 == 0
    assert torch.equal(p1, p2)
    tol = 1e-12 if dtype == torch.float64 else 1e-5
    assert torch.max(torch.abs(L1 - L2)).item() <= tol * torch.max(torch.abs(L1)).item()


def test_four_tall_factorizations_at_once(nla):
    """Four streams, one LU each of heights from 9000 to 120000 rows: every
    panel's groups find a place beside the others', so none waits for a group
    that never starts (such a wait ends after about a second, far above the
    whole call), and the results are those of one at a time."""
    import time
    g = torch.Generator(device=DEV)
    g.manual_seed(4)
    from nextla_amd import _lib
    lib = _lib.load()
    shapes = [(20000, 128), (32000, 128), (60000, 64), (120000, 32)]
    A0 = [torch.empty((n, m), dtype=torch.float64, device=DEV).normal_(generator=g).t() for m, n in shapes]
    ref = [nla.getrf2_(a.clone()) for a in A0]
    streams = [torch.cuda.Stream() for _ in shapes]
    took = []
    for _ in range(4):
        work = [a.clone() for a in A0]
        piv = [torch.zeros(n, dtype=torch.int64, device=DEV) for _, n in shapes]
        info = torch.zeros(4, dtype=torch.int64, device=DEV)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for i, (m, n) in enumerate(shapes):
            assert lib.nla_getrf2(_lib.NLA_F64, m, n, work[i].data_ptr(), m, piv[i].data_ptr(), info[i:].data_ptr(),
                                  streams[i].cuda_stream) == 0
        torch.cuda.synchronize()
        took.append(time.perf_counter() - t0)
        for i, (L, p, inf) in enumerate(ref):
            assert info[i].item() == inf == 0 and torch.equal(piv[i], p) and torch.equal(work[i], L)
    assert min(took) < 0.5, took


@pytest.mark.parametrize("m,n", [(1000, 64), (4096, 33), (300, 8), (100, 64)])
def test_thin_graphs_of_one_stream_at_once(nla, m, n):
    """Captured without a call before on a new stream; two graphs of the stream
    replayed at once, with eager factorizations on that stream in between: every
    replay gives the same factors, and the eager pivots."""
    from nextla_amd import _lib
    lib = _lib.load()
    g = torch.Generator(device=DEV)
    g.manual_seed(m * n)
    A0 = [torch.empty((n, m), dtype=torch.float64, device=DEV).normal_(generator=g).t() for _ in range(2)]
    ref = [nla.getrf2_(a.clone()) for a in A0]
    work = [a.clone() for a in A0]
    piv = [torch.zeros(min(m, n), dtype=torch.int64, device=DEV) for _ in A0]
    info = torch.zeros(2, dtype=torch.int64, device=DEV)
    home, other = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    graphs = []
    for i in range(2):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=home):
            work[i].copy_(A0[i])
            assert lib.nla_getrf2(_lib.NLA_F64, m, n, work[i].data_ptr(), m, piv[i].data_ptr(), info[i:].data_ptr(),
                                  torch.cuda.current_stream().cuda_stream) == 0
        graphs.append(graph)
    first = None
    for rep in range(6):
        for i, st in enumerate((home, other)):
            with torch.cuda.stream(st):
                graphs[i].replay()
        torch.cuda.synchronize()
        if first is None:
            first = [w.clone() for w in work]
        for i in range(2):
            assert info[i].item() == 0 and torch.equal(piv[i], ref[i][1]) and torch.equal(work[i], first[i])
            scale = torch.max(torch.abs(ref[i][0])).item()
            assert torch.max(torch.abs(work[i] - ref[i][0])).item() <= 1e-12 * scale
        with torch.cuda.stream(home):
            nla.getrf2_(A0[0].clone())


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("m,n", [(128, 64), (100, 33), (65, 64), (33, 40), (2, 2)])
@pytest.mark.parametrize("value", [0.0, float("nan")])
def test_single_group_panel_without_a_pivot(nla, split_rows, dtype, m, n, value):
    """Up to 128 rows and 64 columns, one work-group: a column of zeros or of
    NaN, the first and a later one: the info, pivots, factors and NaNs of the
    global-memory leaf."""
    g = torch.Generator(device=DEV)
    g.manual_seed(m + n)
    for col in (0, min(m, n) - 1):
        A0 = torch.empty((n, m), dtype=dtype, device=DEV).normal_(generator=g).t()
        A0[:, col] = value
        split_rows(0)
        L1, p1, i1 = nla.getrf2_(A0.clone())
        split_rows(1)
        L2, p2, i2 = nla.getrf2_(A0.clone())
        assert i1 == i2 == (col + 1 if value == 0.0 else 0) and torch.equal(p1, p2)
        assert torch.equal(torch.isnan(L1), torch.isnan(L2))
        tol = 1e-12 if dtype == torch.float64 else 1e-4
        L1, L2 = torch.nan_to_num(L1), torch.nan_to_num(L2)
        assert torch.max(torch.abs(L1 - L2)).item() <= tol * max(1.0, torch.max(torch.abs(L1)).item())
