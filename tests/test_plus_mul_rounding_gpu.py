"""plus_mul adds every product at full width with one rounding: a single product is
the rounded product bit for bit, and few or many of them are no further from the
sum in 64 bits than a chain of fused multiply-adds is."""
import pytest
import torch

import simd2_amd

pytestmark = pytest.mark.gpu


def _randn(shape, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.randn(shape, generator=g, device="cuda")


def _sparse(rows, k, terms, seed):
    """`terms` normal values in each row, zeros elsewhere."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    at = torch.rand((rows, k), generator=g, device="cuda").topk(terms, dim=1).indices
    return torch.zeros((rows, k), device="cuda").scatter_(1, at, _randn((rows, terms), seed + 1))


@pytest.mark.parametrize("m,n,k", [(64, 64, 256), (100, 70, 300), (65, 63, 64), (1536, 1537, 257),
                                   (2944, 2950, 256)])
def test_one_product_is_rounded_once(m, n, k):
    for swap in (False, True):
        A, B = _sparse(m, k, 1, m + k), _randn((k, n), n)
        if swap:
            A, B = _randn((m, k), n), _sparse(n, k, 1, m + k).t().contiguous()
        # 24 by 24 bits are exact in 64: one rounding
        want = (A.double() @ B.double()).float()
        D = simd2_amd.srgemm("plus_mul", A, B)
        assert torch.equal(D, want), int((D != want).sum())


@pytest.mark.parametrize("k,terms", [(256, 2), (256, 4), (256, 8), (1000, 3), (1024, 32),
                                     (256, 256), (1024, 1024)])
def test_no_further_off_than_a_chain(k, terms):
    """Against one rounding per product in k order.  Any order of the products
    rounds as often, so the two 2-norms over 512 x 512 outputs agree but for
    chance: 5% is ten times what that leaves."""
    A, B = _sparse(512, k, terms, 7 * k + terms), _randn((k, 512), terms)
    want = A.double() @ B.double()
    chain = torch.zeros((512, 512), device="cuda")
    for q in range(k):
        chain = (chain.double() + A[:, q:q + 1].double() * B[q].double()).float()
    D = simd2_amd.srgemm("plus_mul", A, B)
    off, most = (D - want).norm().item(), (chain - want).norm().item()
    assert off <= 1.05 * most, (off, most)
