"""The split-operand GEMM (gemm_split.h: fp32 operands as three bf16 pieces)
and the choice between its tiles and the short-K fp32 kernel."""
import numpy as np
import pytest
import torch

from annc_amd import EPI_RELU
from annc_amd import device as dev
from tests.gpu_util import device, note

pytestmark = pytest.mark.gpu

# sizes one past or short of a tile, a 32-column panel, a k-block and a stage;
# together they reach every tile, with whole and partial last panels
CASES = [(1, 8195, 1024, 545), (1, 8193, 1001, 577), (1, 4099, 992, 865), (1, 2049, 1000, 1024),
         (1, 4097, 512, 1023), (1, 2050, 301, 845), (1, 2047, 512, 1055), (1, 1023, 512, 1024),
         (1, 16390, 16, 1023), (1, 8200, 96, 97), (1, 3000, 70, 33), (1, 4096, 96, 20),
         (1, 1025, 1024, 256), (1, 4096, 64, 512), (5, 300, 288, 577), (3, 65, 2080, 129)]


def _operands(batch, m, n, k, lda_pad, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    shape = (m, k + lda_pad) if batch == 1 else (batch, m, k + lda_pad)
    a = torch.randn(shape, generator=g, device="cuda").relu_()[..., :k]
    b = torch.randn(shape[:-2] + (k, n), generator=g, device="cuda") * 0.1
    return a, b


def _check(got, a, b, bias):
    """|error| <= 2 * (K/16 + 32) * 2^-24 * |A||B|: the large products round
    once per 16 k (by up to one unit, as the matrix units truncate), their
    corrections are 2^-8 of them, and at most 32 roundings more (pieces left
    out, groups added, bias)."""
    ref = a.double() @ b.double() + bias.double()
    k = a.shape[-1]
    bound = 2 * (k / 16 + 32) * 2.0 ** -24 * (a.double().abs() @ b.double().abs() + bias.abs())
    # (short K runs the fp32 instruction: one rounding per k pair, K <= 512)
    if k <= 512:
        bound = bound * (1 + k / 2 / (k / 16 + 32))
    err = (got.double() - ref.relu()).abs() - bound
    assert err.max().item() <= 0, f"{(err > 0).sum().item()} out of bounds, worst {err.max().item()}"


@pytest.mark.parametrize("batch,m,n,k", CASES)
@pytest.mark.parametrize("lda_pad,ldb_pad", [(0, 0), (3, 1)])
def test_split_gemm_edges(batch, m, n, k, lda_pad, ldb_pad):
    """Every tile at its edges, rows of any alignment, within the bound of the
    64-bit product; packed and row-major B give the same bits."""
    note(f"split GEMM {batch}x{m}x{n}x{k} lda+{lda_pad} ldb+{ldb_pad}")
    device()
    a, b = _operands(batch, m, n, k, lda_pad, m + n + k)
    bias = torch.randn(n, device="cuda")
    wide = torch.zeros(b.shape[:-1] + (n + ldb_pad,), device="cuda")
    wide[..., :n] = b
    got = dev.gemm(a, wide[..., :n], bias=bias, epilogue=EPI_RELU)
    _check(got, a, b, bias)
    if batch == 1:
        packed = dev.gemm(a, dev.pack_weight(b), bias=bias, epilogue=EPI_RELU)
        assert torch.equal(got, packed)


@pytest.mark.parametrize("m,n,k", [(1025, 512, 1024), (4096, 512, 1000), (8192, 1000, 640)])
def test_split_gemm_values_its_pieces_cannot_hold(m, n, k):
    """Infinite, NaN, largest and smallest operands: what the products of the
    pieces cannot represent is recomputed with the fp32 instruction."""
    note(f"split GEMM special values {m}x{n}x{k}")
    device()
    a, b = _operands(1, m, n, k, 0, 7)
    b[:, 5] = b[:, 5].abs() + 0.01
    big = torch.finfo(torch.float32).max
    a[3, 1] = float("inf")
    a[70, k - 1] = float("-inf")
    a[130, 2] = float("nan")
    a[200] = 0
    a[200, 4] = big            # rounds past bf16's range
    a[201] = a[201] * 2.0 ** -120   # pieces below bf16's smallest value
    a[202] = 2.0 ** -140            # denormal
    b[9, 40] = float("inf")
    a[:, 9] = a[:, 9].abs() + 0.5
    a[200, 9] = 0.5
    a[201, 9] = 2.0 ** -121
    a[202, 9] = 2.0 ** -140
    zero = torch.zeros(n, device="cuda")
    got = dev.gemm(a, b)
    ref = a.double() @ b.double()
    for r in (3, 70, 130, 200):
        # (a sum of -inf and inf terms is NaN in both)
        assert torch.equal(torch.isnan(got[r]), torch.isnan(ref[r])), r
        fin = torch.isfinite(ref[r]) & (ref[r].abs() < big)
        assert torch.equal(torch.isinf(got[r]) & ~fin, torch.isinf(ref[r].float()) & ~fin), r
    assert torch.isinf(got[:, 40]).sum() + torch.isnan(got[:, 40]).sum() == m
    keep = torch.ones(n, dtype=torch.bool, device="cuda")
    keep[40] = False
    for r, tol in ((200, 1e-6), (201, 3e-6), (202, 0.0)):
        x, y = got[r][keep].double(), ref[r][keep]
        # row 202: denormal products, one 2^-149 step per term is all fp32 has
        bound = tol * (a[r].double().abs() @ b.double().abs())[keep] + k * 2.0 ** -149
        assert ((x - y).abs() <= bound).all(), r
    ok = torch.ones(m, dtype=torch.bool, device="cuda")
    ok[[3, 70, 130, 200, 201, 202]] = False
    _check(got[ok][:, keep].relu(), a[ok], b[:, keep], zero[keep])


def test_row_stride_past_32_bit_offsets():
    """A rows 2^25 floats apart (past the split kernel's 32-bit row offsets):
    the tile kernel, packed and row-major."""
    note("GEMM with a row stride of 2^25 floats")
    device()
    m, k, lda = 33, 48, 1 << 25
    store = torch.empty((m - 1) * lda + k, device="cuda")
    a = store.as_strided((m, k), (lda, 1))
    for n in (4256, 3000):  # more and fewer than 256 32x32 blocks
        src, b = _operands(1, m, n, k, 0, 3)
        a.copy_(src)
        bias = torch.randn(n, device="cuda")
        for w in (b, dev.pack_weight(b)):
            _check(dev.gemm(a, w, bias=bias, epilogue=EPI_RELU), src, b, bias)


# 16x16 blocks (at most 256 of them): one row, row and column edges, K tails,
# K < 32, partial panels of 1-31 columns, K split over workgroups (K >= 2048)
TINY_CASES = [(1, 1, 512, 1024), (1, 17, 33, 64), (1, 16, 47, 545), (1, 15, 8, 20), (1, 256, 256, 31),
              (1, 100, 300, 845), (3, 40, 64, 96), (2, 33, 50, 77), (1, 4096, 16, 1024),
              (1, 1, 1024, 4096), (1, 64, 500, 2049), (1, 16, 31, 2600), (1, 128, 512, 2559),
              # 32x32 blocks (the small kernel): edges, K tails and K < 32, fewer k-blocks
              # than waves and more than its ring of 8 x 4, K split over workgroups
              (1, 257, 1000, 1024), (1, 500, 500, 31), (1, 290, 260, 65), (1, 300, 300, 1311),
              (3, 100, 480, 100), (1, 8190, 17, 320), (1, 128, 1000, 3100),
              # from K = 2048 up to 128 blocks (and not at 2047, nor past them)
              (1, 217, 448, 2048), (1, 217, 448, 2047), (4, 33, 500, 2081), (1, 300, 448, 2048)]


@pytest.mark.parametrize("batch,m,n,k", TINY_CASES)
@pytest.mark.parametrize("lda_pad", [0, 1])
def test_few_block_gemm_edges(batch, m, n, k, lda_pad):
    """Few blocks, K split over 16 or 8 waves: within the fp32 bound of the 64-bit
    product (one rounding per k), packed and row-major B bit-identical."""
    note(f"few-block GEMM {batch}x{m}x{n}x{k} lda+{lda_pad}")
    device()
    a, b = _operands(batch, m, n, k, lda_pad, m + n + k)
    bias = torch.randn(n, device="cuda")
    got = dev.gemm(a, b, bias=bias, epilogue=EPI_RELU)
    ref = (a.double() @ b.double() + bias.double()).relu()
    bound = (k + 32) * 2.0 ** -24 * (a.double().abs() @ b.double().abs() + bias.abs())
    assert ((got.double() - ref).abs() <= bound).all()
    if batch == 1:
        assert torch.equal(got, dev.gemm(a, dev.pack_weight(b), bias=bias, epilogue=EPI_RELU))


@pytest.mark.parametrize("m,n,k", [(478, 960, 672), (478, 960, 685), (204, 1952, 673)])
def test_fp32_pipeline_past_k_512(m, n, k):
    """A grid of at most one round of 64x32 tiles takes the fp32 pipeline also
    for longer K: _check's bound with one rounding per k pair; packed and
    row-major B give the same bits."""
    note(f"fp32 pipeline {m}x{n}x{k}")
    device()
    a, b = _operands(1, m, n, k, 0, m + n + k)
    bias = torch.randn(n, device="cuda")
    got = dev.gemm(a, b, bias=bias, epilogue=EPI_RELU)
    ref = a.double() @ b.double() + bias.double()
    bound = 2 * (k / 2 + k / 16 + 32) * 2.0 ** -24 * (a.double().abs() @ b.double().abs() + bias.abs())
    assert ((got.double() - ref.relu()).abs() <= bound).all()
    assert torch.equal(got, dev.gemm(a, dev.pack_weight(b), bias=bias, epilogue=EPI_RELU))
