"""GEMM update (nla_gemm, the reference's GEMM_ADD!/GEMM_SUB!,
src/matmul.jl:69-80) at the edges of its kernels' tiles and of the rule that
chooses between them, against the product in float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def mat(rows, cols, dtype, row_major, pad, g):
    shape = (rows, cols + pad) if row_major else (cols, rows + pad)
    t = torch.empty(shape, dtype=dtype, device=DEV).normal_(generator=g)
    return t[:, :cols] if row_major else t[:, :rows].t()


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (32, 32, 16), (33, 31, 15), (31, 65, 17), (64, 96, 200), (5, 300, 67),
                                   (300, 8, 1030), (1024, 1025, 64), (1024, 1025, 127), (1025, 1025, 128),
                                   (1667, 1800, 129), (768, 769, 40)])
def test_every_orientation(nla, dtype, m, n, k):
    """All four orientations of X and Y, odd leading dimensions: C -= X*Y and
    C := alpha*X*Y over a C of NaN (beta = 0 reads nothing).  Elementwise
    error at most (k + 3) eps (|C| + |X||Y|): k + 1 roundings of the sum in
    any order, one each of alpha and the update."""
    g = torch.Generator(device=DEV)
    g.manual_seed(m + 7 * n + 31 * k)
    eps = torch.finfo(dtype).eps
    from nextla_amd import _lib
    lib = _lib.load()
    for xt in (False, True):
        for yt in (False, True):
            for pad in (0, 3):
                X, Y, C = mat(m, k, dtype, xt, pad, g), mat(k, n, dtype, yt, pad, g), mat(m, n, dtype, False, pad, g)
                P, A = X.double() @ Y.double(), X.double().abs() @ Y.double().abs()
                ref, bound = C.double() - P, (k + 3) * eps * (C.double().abs() + A)
                nla.GEMM_SUB_(C, X, Y)
                assert torch.all((C.double() - ref).abs() <= bound), (xt, yt, pad)
                C.fill_(float("nan"))
                st = lib.nla_gemm(_lib.NLA_F64 if dtype == torch.float64 else _lib.NLA_F32, b"T" if xt else b"N",
                                  b"T" if yt else b"N", m, n, k, 1.5, X.data_ptr(), X.stride(0 if xt else 1),
                                  Y.data_ptr(), Y.stride(0 if yt else 1), 0.0, C.data_ptr(), C.stride(1),
                                  torch.cuda.current_stream().cuda_stream)
                assert st == 0
                assert torch.all((C.double() - 1.5 * P).abs() <= 1.5 * (k + 3) * eps * A), (xt, yt, pad, "beta 0")


def check(nla, dtype, m, n, k, pads):
    """C -= X*Y in every orientation, within (k + 3) eps (|C| + |X||Y|)."""
    g = torch.Generator(device=DEV)
    g.manual_seed(m + 7 * n + 31 * k)
    eps = torch.finfo(dtype).eps
    for xt in (False, True):
        for yt in (False, True):
            for pad in pads:
                X, Y, C = mat(m, k, dtype, xt, pad, g), mat(k, n, dtype, yt, pad, g), mat(m, n, dtype, False, pad, g)
                Xd, Yd, Cd = X.double(), Y.double(), C.double()
                ref, bound = Cd - Xd @ Yd, (k + 3) * eps * (Cd.abs() + Xd.abs() @ Yd.abs())
                nla.GEMM_SUB_(C, X, Y)
                assert torch.all((C.double() - ref).abs() <= bound), (xt, yt, pad)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("m,n,k", [(20001, 24, 100), (24, 20001, 100), (597, 864, 8), (768, 769, 1024), (1408, 1408, 192),
                                   (1152, 1152, 192), (1024, 1024, 48)])
def test_between_the_kernels(nla, dtype, m, n, k):
    """Shapes near the line between the K-splitting and the tiled kernels,
    long and narrow ones among them."""
    check(nla, dtype, m, n, k, (0, 3))


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("m,n,k", [(4095, 4095, 1501), (4093, 4090, 1504)])
def test_largest_tiles_ragged(nla, dtype, m, n, k):
    """Sizes that take the largest tiles (FP64 256 x 128, FP32 256 x 256 with a
    loop of its own), ragged in M and N, with whole and partial k steps, odd
    leading dimensions."""
    check(nla, dtype, m, n, k, (0, 3))
