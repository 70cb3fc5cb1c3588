"""Packed or_and where A is empty in whole slabs of 128 k: the slabs left out, taken
in order again, taken across several looks ahead (60 slabs each), with K split over
workgroups, in both tile sizes, aligned and not; and the time that leaving them out
saves.  Reference: a float product on the GPU."""
import pytest
import torch

import simd2_amd

pytestmark = pytest.mark.gpu

SLAB = 128
KEPT = {
    "none": lambda s, n: False,
    "first": lambda s, n: s == 0,
    "second": lambda s, n: s == 1,
    "last": lambda s, n: s == n - 1,
    "ends": lambda s, n: s in (0, 1, n - 1),
    "after two": lambda s, n: s != 1 and s != 2,
    "odd pairs": lambda s, n: s % 6 in (3, 4),
    "one of five": lambda s, n: s % 5 == 4,
    "around a look's end": lambda s, n: s in (2, 61, 62, 63, 64, 121, 122, 123),
    "a look's worth": lambda s, n: 2 <= s < 62,
    "empty look": lambda s, n: s < 3 or s > 70,
    "late": lambda s, n: s < n - 4,
}


def _check(m, n, k, kept, density, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    slabs = (k + SLAB - 1) // SLAB
    mask = torch.tensor([kept(q // SLAB, slabs) for q in range(k)], device="cuda")
    A = ((torch.rand((m, k), generator=g, device="cuda") < density) & mask).int()
    B = (torch.rand((k, n), generator=g, device="cuda") < 0.02).int()
    C = (torch.rand((m, n), generator=g, device="cuda") < 0.01).int()
    want = (A.float() @ B.float()) > 0
    a, b, c = (simd2_amd.pack_bits(t) for t in (A, B, C))
    for epilogue in (False, True):
        D = simd2_amd.unpack_bits(simd2_amd.orand_packed(a, b, n, c, epilogue), n)
        assert torch.equal(D > 0, want | (C > 0) if epilogue else want), epilogue


# one 128x128 tile with K split in four, tiles with K whole, 256x256 tiles
@pytest.mark.parametrize("kept", list(KEPT))
@pytest.mark.parametrize("m,n,k", [(100, 120, 128 * 70 + 9), (700, 3000, 128 * 15 - 1),
                                   (2000, 3968, 128 * 130), (4200, 4000, 128 * 125 + 33)])
def test_slabs_left_out(m, n, k, kept):
    print(kept, m, n, k, flush=True)
    _check(m, n, k, KEPT[kept], 0.02, m + k)


@pytest.mark.parametrize("density", [0.0, 1e-6, 1e-5, 1e-4, 1e-3])
@pytest.mark.parametrize("m,n,k", [(2000, 3968, 128 * 130), (4200, 4000, 128 * 80 + 33)])
def test_thin(m, n, k, density):
    _check(m, n, k, lambda s, slabs: True, density, 3)


def test_rows_of_different_slabs():
    """Bands and blocks on the diagonal: every tile has slabs of its own."""
    n = 4608
    i, j = torch.arange(n, device="cuda")[:, None], torch.arange(n, device="cuda")[None, :]
    for A in ((i - j).abs() <= 3, i // 300 == j // 300, (i + j) % 997 == 0, i == n - 1 - j):
        want = (A.float() @ A.float()) > 0
        a = simd2_amd.pack_bits(A.int())
        assert torch.equal(simd2_amd.unpack_bits(simd2_amd.orand_packed(a, a, n), n) > 0, want)


def test_empty_slabs_cost_less():
    n = 8192
    times = []
    for density in (0.0, 0.5):
        a = simd2_amd.pack_bits((torch.rand((n, n), device="cuda") < density).int())
        D = torch.empty_like(a)
        best = float("inf")
        for _ in range(6):
            e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
            e[0].record()
            for _ in range(10):
                simd2_amd.orand_packed(a, a, n, out=D)
            e[1].record()
            torch.cuda.synchronize()
            best = min(best, e[0].elapsed_time(e[1]))
        times.append(best)
    assert times[0] < 0.5 * times[1], times
