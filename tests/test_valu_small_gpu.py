"""The small forms of the VALU product, bit for bit against the oracle
(minus_square on integers, which are exact): the eight-wave K split (whole tiles
and slabs, K >= 256, at most one 64x64 tile per CU) at the ends of its ranges and
just off them, and rows of any alignment in every form."""
import numpy as np
import pytest
import torch

import oracle
import simd2_amd

pytestmark = pytest.mark.gpu

OPS = ["min_plus", "max_plus", "max_min", "max_mul", "min_mul", "min_max"]


def _inputs(op, m, n, k, seed):
    rng = np.random.default_rng(seed)
    A, B, C = (rng.integers(1, 101, s).astype(np.float32) for s in ((m, k), (k, n), (m, n)))
    hole = np.float32(np.inf) if op.startswith("min") else np.float32(-np.inf)
    if op not in ("minus_square", "max_mul", "min_mul"):
        A[rng.random(A.shape) < 0.3] = hole
        B[rng.random(B.shape) < 0.3] = hole
    return A, B, C


def _padded(x, pad, shift):
    """x on the GPU with `pad` more columns, `shift` floats into its buffer."""
    rows, cols = x.shape
    buf = torch.full((rows * (cols + pad) + shift,), 7.0, device="cuda")
    w = buf[shift:].view(rows, cols + pad)
    w[:, :cols] = torch.from_numpy(x).cuda()
    return w


def _run(op, A, B, C, epi, pads, shift):
    m, k = A.shape
    n = B.shape[1]
    a, b, c = (_padded(x, p, shift) for x, p in zip((A, B, C), pads))
    d = _padded(np.zeros((m, n), np.float32), pads[2], shift)
    st = simd2_amd.cuasr_srsgemm(op, n, m, k, b, n + pads[1], a, k + pads[0],
                                 c if epi else None, n + pads[2], d, epi)
    assert st == 0
    assert bool((d[:, n:] == 7.0).all())
    return d[:, :n].cpu().numpy()


@pytest.mark.parametrize("op", OPS)
@pytest.mark.parametrize("m,n,k", [(64, 64, 256), (64, 64, 240), (128, 64, 272), (64, 128, 271),
                                   (65, 64, 256), (64, 63, 640), (128, 192, 1040),
                                   (1024, 1024, 512)])
def test_eight_waves(op, m, n, k):
    A, B, C = _inputs(op, m, n, k, m + n + k)
    for epi in (False, True):
        want = oracle.srgemm_f32(op, A, B, C, epi)
        assert np.array_equal(_run(op, A, B, C, epi, (0, 0, 0), 0), want)
        assert np.array_equal(_run(op, A, B, C, epi, (3, 1, 5), 1), want)


@pytest.mark.parametrize("op", OPS)
@pytest.mark.parametrize("m,n,k", [(16, 16, 16), (1, 1, 1), (65, 63, 10), (64, 64, 17), (100, 90, 32),
                                   (64, 128, 33), (1500, 1400, 16), (1500, 1400, 32), (64, 64, 128),
                                   (130, 70, 129), (1088, 1024, 192), (1088, 1020, 200)])
def test_groups_by_slabs_and_tiles(op, m, n, k):
    A, B, C = _inputs(op, m, n, k, m + n + k)
    rows = np.unique(np.linspace(0, m - 1, 40).astype(int))
    for epi in (False, True):
        D = _run(op, A, B, C, epi, (1, 0, 2), 1)
        assert np.array_equal(D[rows], oracle.srgemm_f32(op, A[rows], B, C[rows], epi))


@pytest.mark.parametrize("op", ["min_plus", "max_mul", "minus_square"])
@pytest.mark.parametrize("m,n,k", [(64, 64, 64), (70, 61, 33), (100, 129, 17), (1100, 1090, 40),
                                   (1500, 1600, 21), (2500, 2400, 18)])
def test_unaligned_rows(op, m, n, k):
    """Four and two groups, unsplit tiles; padded and shifted operands."""
    A, B, C = _inputs(op, m, n, k, m + k)
    for pads, shift in (((0, 0, 0), 0), ((1, 2, 3), 3)):
        D = _run(op, A, B, C, True, pads, shift)
        rows = np.unique(np.linspace(0, m - 1, 40).astype(int))
        assert np.array_equal(D[rows], oracle.srgemm_f32(op, A[rows], B, C[rows], True))


@pytest.mark.parametrize("n", [512, 515, 1024])
def test_loop_uses_the_change_test(n):
    """The fused loop's flag comes from the eight-wave kernel's epilogue."""
    rng = np.random.default_rng(n)
    X = np.full((n, n), np.inf, np.float32)
    mask = rng.random((n, n)) < 0.02
    X[mask] = rng.integers(1, 101, int(mask.sum()))
    np.fill_diagonal(X, 0)
    Y, itr, st = simd2_amd.converge("min_plus", torch.from_numpy(X).cuda(), check="threshold")
    Z, itr_r, st_r = simd2_amd.converge("min_plus", torch.from_numpy(X).cuda(),
                                        check="threshold", flags=simd2_amd.CONVERGE_REFERENCE)
    assert (st, itr) == (0, itr_r) and st_r == 0 and torch.equal(Y, Z)


@pytest.mark.parametrize("op,m,n,k,cfg", [
    ("minus_square", 8192, 4096, 300, 0), ("minus_square", 5376, 5376, 300, 0),
    ("minus_square", 4608, 4608, 300, 1), ("minus_square", 5120, 5120, 128, 1),
    ("minus_square", 8192, 8192, 64, 1), ("minus_square", 16384, 16384, 128, 0),
    ("min_plus", 3900, 3900, 512, 1), ("min_plus", 4096, 4096, 4096, 2),
    ("max_min", 2048, 8192, 1000, 2), ("max_min", 4100, 4100, 300, 1)])
def test_tile_shape_by_full_rounds(op, m, n, k, cfg):
    """The shape that was fastest there (256 CUs; others round elsewhere)."""
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("measured with 256 CUs")
    assert simd2_amd.lib().simd2_pick_tile_config(simd2_amd.OPS.index(op), n, m, k) == cfg
