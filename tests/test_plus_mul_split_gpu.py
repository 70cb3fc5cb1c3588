"""plus_mul through three BF16 parts per operand: edges of its tiles and slabs,
both tile sizes, unaligned rows, in-place epilogue, and the values that send a
tile to the FP32 instructions.  Reference: FP64 on the GPU; the bound is one
rounding of 2^-24 of the sum of the terms' magnitudes for each of the six
products of a 16-k slab, and for C."""
import pytest
import torch

import simd2_amd

pytestmark = pytest.mark.gpu


def _check(D, A, B, C=None):
    A, B = A.double(), B.double()
    want, mag = A @ B, A.abs() @ B.abs()
    if C is not None:
        want, mag = want + C.double(), mag + C.double().abs()
    roundings = 6 * ((A.shape[1] + 15) // 16) + 2
    assert bool(((D.double() - want).abs() <= roundings * 2.0 ** -24 * mag + 2.0 ** -149).all())


def _pair(m, n, k, seed=0):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return (torch.randn((m, k), generator=g, device="cuda"),
            torch.randn((k, n), generator=g, device="cuda"),
            torch.randn((m, n), generator=g, device="cuda"))


@pytest.mark.parametrize("m,n,k", [
    (1, 1, 256), (64, 64, 256), (65, 63, 257), (33, 31, 272), (100, 127, 287), (70, 130, 289),
    (1000, 777, 300), (300, 1, 1000),                                            # 64x64
    (1536, 1536, 256), (2048, 1537, 257), (2049, 2048, 271), (2047, 2047, 272),  # 128x128
    (2944, 2944, 256), (3001, 2900, 300), (2817, 3000, 515)])                    # 256x256
def test_edges(m, n, k):
    A, B, C = _pair(m, n, k, m + n + k)
    _check(simd2_amd.srgemm("plus_mul", A, B), A, B)
    _check(simd2_amd.srgemm("plus_mul", A, B, C, True), A, B, C)


def test_padded_rows_and_in_place():
    m, n, k = 2050, 2047, 300
    A, B, C = _pair(m, n, k)
    wa, wb, wc = (torch.full((t.shape[0], t.shape[1] + 3), 7.0, device="cuda") for t in (A, B, C))
    wa[:, :k], wb[:, :n], wc[:, :n] = A, B, C
    st = simd2_amd.lib().cuasr_plusmul_srsgemm(
        n, m, k, wb.data_ptr(), n + 3, wa.data_ptr(), k + 3, wc.data_ptr(), n + 3, wc.data_ptr(),
        True, torch.cuda.current_stream().cuda_stream)
    assert st == 0
    _check(wc[:, :n], A, B, C)
    assert bool((wc[:, n:] == 7.0).all())


@pytest.mark.parametrize("m,n", [(700, 700), (2048, 2048), (2944, 2944)])
def test_values_out_of_range(m, n):
    """Each kind of value in rows of its own; no other row is disturbed."""
    k = 256
    A, B, C = _pair(m, n, k)
    A[5, 7] = float("inf")
    A[150, 9] = -float("inf")
    A[200, 3] = 3.4028234663852886e38     # rounds to infinity in BF16
    A[300, :] *= 2.0 ** -110              # below BF16's range once split
    A[400:410, :] *= 2.0 ** -60           # products below FP32's range
    B[:, 490:500] *= 2.0 ** -60
    A[600, :] = 0.0
    A[601, :] = 1.0e-45                   # denormals
    D = simd2_amd.srgemm("plus_mul", A, B)
    want = A.double() @ B.double()
    big = want.abs() > 3.4e38
    assert bool(big.any()) and torch.equal(D[big], want[big].float())
    keep = torch.ones(m, dtype=torch.bool, device="cuda")
    keep[[5, 150, 200, 601]] = False
    _check(D[keep], A[keep], B)
    assert bool(torch.isfinite(D[keep]).all())
    assert bool((D[601].abs() <= 256 * 1.5e-45 * B.abs().max()).all())


def test_exact_on_integers():
    A, B, C = (t.mul(10).round() for t in _pair(2048, 2048, 1024))
    D = simd2_amd.srgemm("plus_mul", A, B, C, True)
    assert torch.equal(D.double(), A.double() @ B.double() + C.double())


@pytest.mark.parametrize("k", [256, 300, 1024])
def test_tile_sizes_agree(k):
    """A block of a large product equals the block computed by itself."""
    A, B, C = _pair(2944, 2944, k, 3)
    full = simd2_amd.srgemm("plus_mul", A, B, C, True)
    for lo, hi in ((0, 1600), (1000, 1100)):
        part = simd2_amd.srgemm("plus_mul", A[lo:hi].contiguous(), B[:, lo:hi].contiguous(),
                                C[lo:hi, lo:hi].contiguous(), True)
        assert torch.equal(part, full[lo:hi, lo:hi])

