"""Large GEMMs over the whole range of fp32 operands: each operand is split
into three bf16 pieces, which hold it exactly from 2^-110 on; products of
smaller ones have to come out as the fp32 instruction gives them."""
import pytest
import torch

from annc_amd import _lib
from annc_amd import device as dev
from tests.gpu_util import device, note

pytestmark = pytest.mark.gpu


def _denormal_row(a, b):
    """One row of A denormal: products that are denormal themselves."""
    a[..., 40, :] *= 2.0 ** -140


def _denormal_column(a, b):
    b[..., 70] *= 2.0 ** -135


def _zero_pieces(a, b):
    """One nonzero operand in a row, below half of bf16's least value: all its
    pieces are 0, the product is not."""
    a[..., 40, :] = 0
    a[..., 40, 11] = 2.0 ** -140
    b[..., 11, 33] = 2.0 ** 100


EXPONENTS = (-112, -118, -125, -130, -138)


def _hidden_in_an_ordinary_sum(a, b):
    """A small operand of A times a large one of B, and one ordinary term of
    the same size."""
    k = a.shape[-1]
    for i, e in enumerate(EXPONENTS):
        a[..., 40 + 64 * i, :] = 0
        a[..., 40 + 64 * i, 5] = 2.0 ** (e + 110)
        a[..., 40 + 64 * i, k - 3] = 1.2345678 * 2.0 ** e
        b[..., k - 3, 33 + i] = 1.7654321 * 2.0 ** 110


def _large_a_small_b(a, b):
    k = a.shape[-1]
    for i, e in enumerate(EXPONENTS):
        b[..., 33 + i] = 0
        b[..., k - 3, 33 + i] = 2.0 ** (e + 110)
        b[..., 2, 33 + i] = 1.2345678 * 2.0 ** e
        a[..., 40 + 64 * i, 2] = 1.7654321 * 2.0 ** 110


def _small_by_ordinary(a, b):
    """Rows and columns scaled down, everything else ordinary: sums from 2^-60
    down to denormal."""
    for i, e in enumerate((-55, -70, -90, -108, -111, -116, -123)):
        a[..., 40 + 32 * i, :] *= 2.0 ** e
        b[..., 3 + i] *= 2.0 ** -(3 * i)


PLANTS = [_denormal_row, _denormal_column, _zero_pieces, _hidden_in_an_ordinary_sum,
          _large_a_small_b, _small_by_ordinary]


# each split tile (256x128 ... 64x32), whole and ragged in K and N, two batched
@pytest.mark.parametrize("batch,m,n,k,tile", [
    (1, 16384, 512, 1056, 0), (1, 4096, 1024, 1024, 1), (1, 8195, 1000, 1023, 2),
    (1, 3000, 544, 1055, 2), (1, 2047, 301, 845, 3), (1, 1025, 512, 1024, 3),
    (1, 4100, 96, 1000, 4), (3, 451, 704, 192, 2), (3, 512, 612, 577, 3)])
@pytest.mark.parametrize("plant", PLANTS)
def test_small_and_large_operands(plant, batch, m, n, k, tile):
    note(f"GEMM operand range {plant.__name__} {batch}x{m}x{n}x{k}")
    device()
    assert _lib.lib().annc_hip_gemm_tile(batch, m, n, k) == tile
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    shape = (m, k) if batch == 1 else (batch, m, k)
    a = torch.randn(shape, generator=g, device="cuda").relu_()
    b = torch.randn(shape[:-2] + (k, n), generator=g, device="cuda") * 0.1
    plant(a, b)
    a64, b64 = a.double(), b.double()
    ref = a64 @ b64
    # fp32 sums: one rounding per k pair of the fp32 instruction (up to one
    # unit), 32 more for the parts that are added up; a denormal result has
    # one unit of 2^-149 per term
    bound = 2 * (k / 2 + 32) * 2.0 ** -24 * (a64.abs() @ b64.abs()) + k * 2.0 ** -149
    weights = [b] if batch > 1 else [b, dev.pack_weight(b)]
    for w in weights:
        err = (dev.gemm(a, w).double() - ref).abs() - bound
        assert err.max().item() <= 0, f"{(err > 0).sum().item()} out of bounds"


@pytest.mark.parametrize("scale", [1e-10, 1e-16])
def test_small_sums_of_exact_pieces(scale):
    """Both sides scaled down, every operand still above 2^-110: the pieces
    are exact and so are their products, whatever the size of the sums."""
    note(f"GEMM of operands scaled by {scale}")
    device()
    m, n, k = 4096, 512, 1000
    g = torch.Generator(device="cuda").manual_seed(3)
    a = torch.randn((m, k), generator=g, device="cuda") * scale
    b = torch.randn((k, n), generator=g, device="cuda") * scale
    ref = a.double() @ b.double()
    bound = 2 * (k / 16 + 32) * 2.0 ** -24 * (a.double().abs() @ b.double().abs()) + k * 2.0 ** -149
    assert ((dev.gemm(a, b).double() - ref).abs() <= bound).all()
