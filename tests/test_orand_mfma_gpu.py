"""or_and on the FP4 matrix cores: the packed kernel at the edges of its tiles
(128x128 and 256x256 outputs, 128-k slabs, 32-bit words), its K split, and
the int32 product that packs its operands into the output's rows.  Reference:
the 0/1 product in float32, whose counts are exact integers."""
import numpy as np
import pytest
import torch

import simd2_amd

pytestmark = pytest.mark.gpu


def _bits(shape, density, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return (torch.rand(shape, generator=g, device="cuda") < density).int()


def _want(A, B, C):
    D = (A != 0).float() @ (B != 0).float() > 0
    return (D if C is None else D | (C != 0)).int()


def _wide(P, pad):
    """The rows of P inside a wider buffer, `pad` words of junk behind each."""
    W = torch.full((P.shape[0], P.shape[1] + pad), -1, dtype=torch.int32, device="cuda")
    W[:, :P.shape[1]] = P
    return W[:, :P.shape[1]]


@pytest.mark.parametrize("m,n,k", [
    (1, 1, 1), (31, 33, 32), (128, 128, 128), (129, 127, 129), (64, 2048, 255), (200, 300, 31),
    (4096, 4096, 160), (4099, 4129, 257), (8192, 2080, 33),       # 256x256 tiles
    (64, 64, 8192), (130, 96, 4100)])                             # K split
@pytest.mark.parametrize("pad", [0, 3])
def test_packed_edges(m, n, k, pad):
    A, B = _bits((m, k), 1.5 / k ** 0.5 / 4, m), _bits((k, n), 1.5 / k ** 0.5 / 4, n)
    C = _bits((m, n), 0.05, k)
    pa, pb, pc = (_wide(simd2_amd.pack_bits(t), pad) for t in (A, B, C))
    nw, kw = (n + 31) // 32, (k + 31) // 32
    for epi in (False, True):
        out = torch.full((m, nw + pad), 7, dtype=torch.int32, device="cuda")
        st = simd2_amd.lib().simd2_orand_packed(
            m, n, k, pa.data_ptr(), kw + pad, pb.data_ptr(), nw + pad, pc.data_ptr(), nw + pad,
            out.data_ptr(), nw + pad, int(epi), torch.cuda.current_stream().cuda_stream)
        assert st == 0
        assert torch.equal(simd2_amd.unpack_bits(out[:, :nw], n), _want(A, B, C if epi else None))
        assert bool((out[:, nw:] == 7).all())
        if n % 32:  # the bits past column n stay clear
            assert int((out[:, nw - 1].to(torch.int64) & 0xFFFFFFFF).max()) < 1 << (n % 32)


def test_packed_every_position():
    """One bit at a time: the identity on either side returns the other."""
    n = 320
    eye, M = torch.eye(n, dtype=torch.int32, device="cuda"), _bits((n, n), 0.5, 1)
    pe, pm = simd2_amd.pack_bits(eye), simd2_amd.pack_bits(M)
    assert torch.equal(simd2_amd.unpack_bits(simd2_amd.orand_packed(pe, pm, n), n), M)
    assert torch.equal(simd2_amd.unpack_bits(simd2_amd.orand_packed(pm, pe, n), n), M)


def test_packed_skips_and_dense():
    """Slabs that are empty on one side only, and every term set."""
    m, n, k = 512, 512, 1024
    A, B = _bits((m, k), 0.01, 2), _bits((k, n), 0.01, 3)
    A[:, 128:512] = 0
    A[128:256] = 0
    B[600:900] = 0
    B[:, 256:384] = 0
    for X, Y in ((A, B), (torch.ones_like(A), torch.ones_like(B))):
        P = simd2_amd.orand_packed(simd2_amd.pack_bits(X), simd2_amd.pack_bits(Y), n)
        assert torch.equal(simd2_amd.unpack_bits(P, n), _want(X, Y, None))


@pytest.mark.parametrize("m,n,k", [
    (256, 256, 256), (1024, 1024, 1024), (1025, 1028, 1030), (777, 1000, 300), (333, 515, 67),
    (64, 1024, 512), (100, 2048, 1000),   # k past the rows: bands of packed rows
    (64, 256, 4096), (64, 250, 3001),     # k in parts
    (64, 64, 2048), (7, 9, 5), (2048, 48, 64)])  # too narrow for the packed route
def test_int32_routes(m, n, k):
    A, B = _bits((m, k), 0.03, m) * 5, _bits((k, n), 0.03, n) * -3  # any nonzero is true
    C = _bits((m, n), 0.05, k) * 2
    for epi in (False, True):
        D = simd2_amd.srgemm("or_and", A, B, C, epi)
        assert torch.equal(D, _want(A, B, C if epi else None)), epi
    # C in place, and a padded output whose gap stays untouched
    W = torch.full((m, n + 5), 9, dtype=torch.int32, device="cuda")
    W[:, :n] = C
    L, s = simd2_amd.lib(), torch.cuda.current_stream().cuda_stream
    st = L.cuasr_orand_srsgemm(n, m, k, B.data_ptr(), n, A.data_ptr(), k, W.data_ptr(), n + 5,
                               W.data_ptr(), True, s)
    assert st == 0
    assert torch.equal(W[:, :n], _want(A, B, C))
    assert bool((W[:, n:] == 9).all())


def test_int32_shifted_epilogue():
    """C overlapping D at another offset keeps the unpacked kernel's result
    where rows do not meet: here they are disjoint rows of one buffer."""
    m, n, k = 256, 512, 256
    A, B = _bits((m, k), 0.03, 1), _bits((k, n), 0.03, 2)
    W = torch.zeros((2 * m, n), dtype=torch.int32, device="cuda")
    W[m:] = _bits((m, n), 0.1, 3)
    want = _want(A, B, W[m:])
    D = simd2_amd.srgemm("or_and", A, B, W[m:], True, out=W[:m])
    assert torch.equal(D, want)


def test_int32_captured():
    m, n, k = 512, 640, 384
    A, B, C = _bits((m, k), 0.03, 1), _bits((k, n), 0.03, 2), _bits((m, n), 0.03, 3)
    D = torch.empty((m, n), dtype=torch.int32, device="cuda")
    simd2_amd.srgemm("or_and", A, B, C, True, out=D)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        simd2_amd.srgemm("or_and", A, B, C, True, out=D)
    for i in range(3):
        A.copy_(_bits((m, k), 0.03, 10 + i))
        D.fill_(3)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(D, _want(A, B, C))
