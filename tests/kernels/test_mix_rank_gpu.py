"""Short bf16 products (csrc/kernels/mix_rank.hip) against 64-bit sums: rows and columns around the
tiles, column slices of wider rows, the forms that stay with the library, infinities, derivatives."""
import pytest
import torch

from replisense_rfq_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _check(x, w, out_dtype):
    y = ops.matmul_nt(x, w, out_dtype)
    assert y.dtype == (out_dtype or torch.bfloat16) and y.is_contiguous()
    xd, wd = x.double().cpu(), w.double().cpu()
    want, size = xd @ wd.t(), xd.abs() @ wd.abs().t()
    # products of bf16 are exact in fp32, each of K sums rounds a part of `size` to 2^-24; bf16: half
    # a step of 2^-8 of the value more
    tol = x.shape[1] * 2.0 ** -24 * size + (2.0 ** -8 * want.abs() if y.dtype == torch.bfloat16 else 0)
    assert bool(((y.double().cpu() - want).abs() <= tol).all())


# 512 x 4,096 is the largest, one row more stays with the library
@pytest.mark.parametrize("M,N", [(1, 4), (15, 60), (16, 64), (17, 260), (64, 2048), (129, 68), (512, 4096), (513, 4096)])
@pytest.mark.parametrize("K", [32, 64, 96, 128, 40])          # 40: the library
@pytest.mark.parametrize("out_dtype", [None, torch.float32])
def test_short_products(M, N, K, out_dtype):
    g = torch.Generator().manual_seed(M + K)
    wide, w = torch.randn(M, K + 16, generator=g).to(DEV, torch.bfloat16), torch.randn(N, K, generator=g).to(DEV, torch.bfloat16)
    _check(wide[:, 8:8 + K], w, out_dtype)
    _check(wide[:, 3:3 + K], w, out_dtype)                    # rows that begin at odd addresses
    if N % 4 == 0 and N > 4:
        _check(wide[:, :K], w[:N - 1], out_dtype)             # columns that are no multiple of four


def test_infinities_stay_in_their_row_and_column():
    x, w = torch.ones(20, 64, device=DEV, dtype=torch.bfloat16), torch.ones(72, 64, device=DEV, dtype=torch.bfloat16)
    x[3, 5], w[70, 9] = float("inf"), float("nan")
    y = ops.matmul_nt(x, w, torch.float32)
    want = torch.full((20, 72), 64.0)
    want[3], want[:, 70] = float("inf"), float("nan")
    torch.testing.assert_close(y.cpu(), want, atol=0, rtol=0, equal_nan=True)


def test_derivatives_are_the_library_products():
    x, w = (torch.randn(n, 64, device=DEV, dtype=torch.bfloat16) for n in (8, 12))
    x.requires_grad_()
    ops.matmul_nt(x, w).sum().backward()
    torch.testing.assert_close(x.grad, w.sum(0, keepdim=True).expand(8, 64), atol=0.05, rtol=0.02)
    with torch.no_grad():
        assert ops.matmul_nt(x, w).shape == (8, 12)


def _check_f32(x, w):
    y = ops.matmul_nt(x, w)
    assert y.dtype == torch.float32 and y.is_contiguous()
    xd, wd = x.double().cpu(), w.double().cpu()
    # each of K sums rounds a part of the sum of sizes to 2^-24; what the parts leave out is less than 2^-24 of every product
    tol = (x.shape[1] + 1) * 2.0 ** -24 * (xd.abs() @ wd.abs().t())
    assert bool(((y.double().cpu() - xd @ wd.t()).abs() <= tol).all())


# a wave with 16, 32 (from 641 tiles of 64 x 16 on) and 64 columns (1,536), one block of rows and several (2,048); tiles that
# are cut, columns slices of wider rows, rows at odd addresses (there the library, or a copy)
@pytest.mark.parametrize("M,N", [(1, 4), (17, 60), (64, 2048), (129, 68), (645, 1028), (1540, 1030 * 2), (2100, 2052), (9000, 1024)])
@pytest.mark.parametrize("K", [32, 64, 96, 128, 40])
def test_short_fp32_products(M, N, K):
    g = torch.Generator().manual_seed(M + K)
    wide, w = torch.randn(M, K + 12, generator=g).to(DEV), torch.randn(N, K, generator=g).to(DEV)
    _check_f32(wide[:, 4:4 + K], w)
    if M < 200:
        _check_f32(wide[:, 3:3 + K], w)
        _check_f32(torch.frombuffer(bytearray(4 * M * K + 4), dtype=torch.float32)[1:].view(M, K).to(DEV), w[:N - 1])


@pytest.mark.parametrize("value", [float("inf"), float("nan"), 3.4e38, 1e-38])
def test_fp32_products_at_the_ends_of_the_range(value):
    x, w = torch.full((40, 64), 0.25, device=DEV), torch.full((72, 64), 0.5, device=DEV)
    w[:, 7] = -0.5
    x[3, 5], w[70, 9] = value, value
    y = ops.matmul_nt(x, w)
    want = x.cpu() @ w.cpu().t()
    torch.testing.assert_close(y.cpu(), want, atol=0, rtol=1e-6, equal_nan=True)


def test_fp32_products_keep_autocast_and_derivatives():
    x, w = (torch.randn(n, 64, device=DEV) for n in (8, 12))
    with torch.autocast("cuda", torch.bfloat16):
        assert ops.matmul_nt(x, w).dtype == torch.bfloat16
    x.requires_grad_()
    ops.matmul_nt(x, w).sum().backward()
    torch.testing.assert_close(x.grad, w.sum(0, keepdim=True).expand(8, 64), atol=1e-4, rtol=1e-4)
    y = torch.func.vmap(lambda a: ops.matmul_nt(a, w))(torch.ones(3, 5, 64, device=DEV))
    torch.testing.assert_close(y, w.sum(1).expand(3, 5, 12), atol=1e-4, rtol=1e-4)
