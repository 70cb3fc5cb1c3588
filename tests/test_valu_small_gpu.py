"""The VALU product on rows of any alignment, in every form (split K in four
and two groups, unsplit tiles), bit for bit against the oracle (minus_square on
integers, which are exact)."""
import numpy as np
import pytest
import torch

import oracle
import simd2_amd

pytestmark = pytest.mark.gpu


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

