"""The FP16 emulation product at the edges of its tiles (32, 64 and 128), its
K split and its slabs (32 and 64 k), with infinities, NaN terms and unaligned
operands, against the sequential restatement, bit for bit."""
import numpy as np
import pytest
import torch

import simd2_amd
from oracle import fp16_emulation

pytestmark = pytest.mark.gpu


def _inputs(op, m, n, k, seed, specials):
    rng = np.random.default_rng(seed)
    if op in ("min_plus", "max_plus", "max_min", "min_max"):
        A, B = rng.integers(1, 101, (m, k)).astype(np.float16), rng.integers(1, 101, (k, n)).astype(np.float16)
    else:
        A, B = rng.standard_normal((m, k)).astype(np.float16), rng.standard_normal((k, n)).astype(np.float16)
    if specials:
        A[rng.random((m, k)) < 0.1] = np.inf
        B[rng.random((k, n)) < 0.1] = np.inf if op.startswith("min") else -np.inf
        if op in ("min_mul", "max_mul"):
            A[rng.random((m, k)) < 0.05] = 0.0     # 0 * inf
    return A, B, rng.standard_normal((m, n)).astype(np.float32)


def _same(D, want):
    return np.array_equal(D.cpu().numpy(), want, equal_nan=True)


SIZES = [(16, 16, 16), (32, 48, 80), (64, 64, 256), (80, 112, 272), (144, 16, 64),
         (528, 512, 48), (512, 528, 144), (784, 1040, 16), (784, 1040, 144), (1040, 1040, 32)]


@pytest.mark.parametrize("op", simd2_amd.OPS)
@pytest.mark.parametrize("m,n,k", SIZES)
def test_tiles(op, m, n, k):
    for specials in (False, True):
        if specials and op in ("plus_mul", "minus_square"):
            continue
        A, B, C = _inputs(op, m, n, k, m + n + k, specials)
        a, b, c = (torch.from_numpy(t).cuda() for t in (A, B, C))
        for epi in (False, True):
            with np.errstate(all="ignore"):
                want = fp16_emulation.tensor_srgemm(A, B, C, op, epi)
            assert _same(simd2_amd.tensor_srgemm(op, a, b, c, epi), want), (specials, epi)


@pytest.mark.parametrize("op", ["min_plus", "max_mul", "plus_mul", "or_and"])
def test_large_tiles(op):
    """128x128 tiles (their count is what chooses them): rows and columns of
    the result against the restatement on those rows and columns."""
    m, n, k = 3088, 2896, 48
    A, B, C = _inputs(op, m, n, k, 5, False)
    a, b, c = (torch.from_numpy(t).cuda() for t in (A, B, C))
    D = simd2_amd.tensor_srgemm(op, a, b, c, True)
    rows, cols = [0, 63, 64, 127, 128, 1500, 3087], [0, 127, 128, 2000, 2815, 2816, 2895]
    with np.errstate(all="ignore"):
        assert _same(D[rows], fp16_emulation.tensor_srgemm(A[rows], B, C[rows], op, True))
        assert _same(D[:, cols], fp16_emulation.tensor_srgemm(A, B[:, cols], C[:, cols], op, True))


@pytest.mark.parametrize("op", ["min_plus", "plus_mul"])
def test_unaligned(op):
    m, n, k = 96, 80, 112
    A, B, C = _inputs(op, m, n, k, 9, False)

    def shifted(x):
        w = torch.empty(x.size + 1, dtype=torch.from_numpy(x).dtype, device="cuda")
        w[1:] = torch.from_numpy(x).cuda().reshape(-1)
        return w[1:].view(x.shape)

    D = simd2_amd.tensor_srgemm(op, shifted(A), shifted(B), shifted(C), True,
                                out=shifted(np.zeros((m, n), np.float32)))
    assert _same(D, fp16_emulation.tensor_srgemm(A, B, C, op, True))
