"""The split-operand GEMM (gemm_split.h: fp32 operands as three bf16 pieces),
the fp32 pipeline beside it, the choice between their tiles, and the kernels
for few blocks."""
import pytest
import torch

from annc_amd import EPI_RELU, _lib
from annc_amd import device as dev
from tests.gpu_util import device, note

pytestmark = pytest.mark.gpu

# (batch, m, n, k) and the tile that runs it: 0-4 split 256x128, 128x128, 128x64,
# 64x64, 64x32; 5-7 fp32 64x64, 64x32, 128x64; + 8: the tail columns in a second
# launch.  Sizes one past or short of a tile, a 32-column panel, a k-block and a
# stage: every tile with whole and ragged K and N, one product and batches
# (128x128 takes whole panels only).  The first sixteen have longer K.
CASES = [
    (1, 8195, 1024, 545, 2), (1, 8193, 1001, 577, 2), (1, 4099, 992, 865, 0),
    (1, 2049, 1000, 1024, 9), (1, 4097, 512, 1023, 1), (1, 2050, 301, 845, 3),
    (1, 2047, 512, 1055, 3), (1, 1023, 512, 1024, 4), (1, 16390, 16, 1023, 6),
    (1, 8200, 96, 97, 6), (1, 3000, 70, 33, 6), (1, 4096, 96, 20, 6), (1, 1025, 1024, 256, 2),
    (5, 300, 288, 577, 6), (3, 65, 2080, 129, 5), (1, 4100, 96, 1000, 4),
    (1, 2689, 1536, 32, 0), (1, 16385, 197, 64, 0), (1, 3327, 1280, 33, 0), (1, 14080, 257, 33, 0),
    (7, 897, 640, 32, 0), (3, 3587, 321, 64, 0), (5, 515, 1536, 33, 0), (7, 1923, 261, 33, 0),
    (1, 4099, 640, 128, 1), (1, 6147, 512, 33, 1), (3, 707, 1152, 128, 1), (7, 257, 1408, 33, 1),
    (1, 769, 1280, 192, 2), (1, 3587, 257, 192, 2), (1, 2179, 704, 97, 2), (1, 1539, 645, 161, 2),
    (3, 451, 704, 192, 2), (7, 193, 577, 192, 2), (5, 259, 1024, 97, 2), (7, 65, 1157, 165, 2),
    (1, 705, 704, 384, 3), (1, 513, 897, 256, 3), (1, 1345, 384, 225, 3), (1, 2691, 165, 193, 3),
    (7, 65, 640, 512, 3), (3, 67, 1428, 256, 3), (3, 65, 1408, 357, 3), (3, 131, 916, 225, 3),
    (1, 385, 640, 640, 4), (1, 1153, 193, 128, 4), (1, 323, 768, 353, 4), (1, 1153, 193, 101, 4),
    (2, 384, 352, 768, 4), (2, 579, 193, 128, 4), (3, 385, 197, 97, 4),
    (1, 515, 1024, 32, 5), (1, 4097, 101, 32, 5), (1, 323, 1536, 33, 5), (1, 8963, 33, 33, 5),
    (5, 65, 896, 32, 5), (3, 131, 901, 32, 5), (2, 129, 1408, 33, 5), (7, 65, 660, 37, 5),
    (1, 897, 288, 32, 6), (1, 2049, 97, 32, 6), (1, 195, 1280, 33, 6), (1, 3073, 65, 33, 6),
    (2, 451, 288, 32, 6), (3, 1535, 33, 32, 6), (5, 195, 256, 33, 6), (5, 963, 33, 37, 6),
    (1, 2943, 896, 32, 7), (1, 11007, 129, 32, 7), (1, 11521, 288, 33, 7), (1, 12547, 212, 33, 7),
    (3, 707, 1152, 32, 7), (7, 2816, 69, 32, 7), (5, 3583, 192, 33, 7), (7, 1791, 193, 37, 7),
    (1, 6657, 1183, 33, 8), (5, 640, 1281, 33, 9), (1, 2819, 709, 97, 10), (7, 65, 1172, 709, 11),
    (1, 1089, 468, 896, 12), (5, 257, 1285, 33, 13), (3, 129, 927, 325, 14), (1, 2563, 1537, 32, 15)]


def _tile(batch, m, n, k):
    return _lib.lib().annc_hip_gemm_tile(batch, m, n, k)


def _operands(batch, m, n, k, lda_pad, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    shape = (m, k + lda_pad) if batch == 1 else (batch, m, k + lda_pad)
    a = torch.randn(shape, generator=g, device="cuda").relu_()[..., :k]
    b = torch.randn(shape[:-2] + (k, n), generator=g, device="cuda") * 0.1
    return a, b


def _check(got, a, b, bias, tile):
    """|error| <= 2 * R * 2^-24 * |A||B|.  Split tiles: R = K/16 + 32, the large
    products round once per 16 k (by up to one unit, as the matrix units
    truncate), their corrections are 2^-8 of them, and at most 32 roundings
    more (pieces left out, groups added, bias).  The fp32 instruction rounds
    once per k pair (per k in the tail columns' kernel): R = K/2 + 32 (K + 32)."""
    ref = a.double() @ b.double() + bias.double()
    k = a.shape[-1]
    roundings = 32 + (k if tile >= 8 else k / 16 if tile < 5 else k / 2)
    bound = 2 * roundings * 2.0 ** -24 * (a.double().abs() @ b.double().abs() + bias.abs())
    err = (got.double() - ref.relu()).abs() - bound
    assert err.max().item() <= 0, f"{(err > 0).sum().item()} out of bounds, worst {err.max().item()}"


@pytest.mark.parametrize("batch,m,n,k,tile", CASES)
@pytest.mark.parametrize("lda_pad,ldb_pad", [(0, 0), (3, 1)])
def test_split_gemm_edges(batch, m, n, k, tile, lda_pad, ldb_pad):
    """Every tile at its edges, rows of any alignment, within the bound of the
    64-bit product; packed and row-major B give the same bits."""
    note(f"split GEMM {batch}x{m}x{n}x{k} lda+{lda_pad} ldb+{ldb_pad}")
    device()
    assert _tile(batch, m, n, k) == tile, "the case has left its tile: take another size"
    a, b = _operands(batch, m, n, k, lda_pad, m + n + k)
    bias = torch.randn(n, device="cuda")
    wide = torch.zeros(b.shape[:-1] + (n + ldb_pad,), device="cuda")
    wide[..., :n] = b
    got = dev.gemm(a, wide[..., :n], bias=bias, epilogue=EPI_RELU)
    _check(got, a, b, bias, tile)
    if batch == 1:
        packed = dev.gemm(a, dev.pack_weight(b), bias=bias, epilogue=EPI_RELU)
        assert torch.equal(got, packed)


# one of each split tile, ragged
@pytest.mark.parametrize("m,n,k,tile", [(4099, 992, 865, 0), (4097, 512, 1023, 1), (8193, 1001, 577, 2),
                                        (2050, 301, 845, 3), (1153, 193, 101, 4)])
def test_one_product_an_output(m, n, k, tile):
    """Rows of A with one nonzero: of the nine products of the pieces, m*l, l*m
    and l*l are left out, up to 2^-24 of the operands' product together, and
    the sum of the others is rounded once: within 2^-23 (the fp32 instruction:
    2^-24)."""
    note(f"split GEMM of one nonzero a row {m}x{n}x{k}")
    device()
    assert _tile(1, m, n, k) == tile
    g = torch.Generator(device="cuda").manual_seed(m)
    a = torch.zeros((m, k), device="cuda")
    a[torch.arange(m, device="cuda"), torch.randint(k, (m,), generator=g, device="cuda")] = \
        torch.rand(m, generator=g, device="cuda") + 1
    b = torch.rand((k, n), generator=g, device="cuda") + 1
    ref = a.double() @ b.double()
    for w in (b, dev.pack_weight(b)):
        assert ((dev.gemm(a, w).double() - ref).abs() <= 2.0 ** -23 * ref).all()


@pytest.mark.parametrize("m,n,k", [(1025, 512, 1024), (4096, 512, 1000), (8192, 1000, 640),
                                   (2050, 301, 845), (385, 640, 640), (4097, 512, 1023)])
@pytest.mark.parametrize("layout", ["row-major", "packed", "batched"])
def test_split_gemm_values_its_pieces_cannot_hold(m, n, k, layout):
    """Infinite, NaN, largest and smallest operands: what the products of the
    pieces cannot represent is recomputed with the fp32 instruction, on packed
    and row-major B with and without tails, and in every batch."""
    note(f"split GEMM special values {m}x{n}x{k} {layout}")
    device()
    batch = 3 if layout == "batched" else 1
    tile = _tile(batch, m, n, k)
    assert tile < 5
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
    if layout == "batched":  # the values in the middle one
        a3, b3 = torch.ones((3, m, k), device="cuda"), torch.ones((3, k, n), device="cuda")
        a3[1], b3[1] = a, b
        got = dev.gemm(a3, b3)
        assert (got[0] == k).all() and (got[2] == k).all()
        got = got[1]
    else:
        got = dev.gemm(a, dev.pack_weight(b) if layout == "packed" else b)
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
    _check(got[ok][:, keep].relu(), a[ok], b[:, keep], zero[keep], tile)


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
            _check(dev.gemm(a, w, bias=bias, epilogue=EPI_RELU), src, b, bias, 5)


def test_b_row_stride_past_32_bit_offsets():
    """Row-major B with rows 2^27 floats apart: the tile kernel."""
    note("GEMM with a row stride of B of 2^27 floats")
    device()
    m, n, k, ldb = 300, 1000, 4, 1 << 27
    a, src = _operands(1, m, n, k, 0, 4)
    b = torch.empty((k - 1) * ldb + n, device="cuda").as_strided((k, n), (ldb, 1))
    b.copy_(src)
    bias = torch.randn(n, device="cuda")
    _check(dev.gemm(a, b, bias=bias, epilogue=EPI_RELU), a, src, bias, 5)


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
    assert _tile(1, m, n, k) == 6
    a, b = _operands(1, m, n, k, 0, m + n + k)
    bias = torch.randn(n, device="cuda")
    got = dev.gemm(a, b, bias=bias, epilogue=EPI_RELU)
    ref = a.double() @ b.double() + bias.double()
    bound = 2 * (k / 2 + k / 16 + 32) * 2.0 ** -24 * (a.double().abs() @ b.double().abs() + bias.abs())
    assert ((got.double() - ref.relu()).abs() <= bound).all()
    assert torch.equal(got, dev.gemm(a, dev.pack_weight(b), bias=bias, epilogue=EPI_RELU))
