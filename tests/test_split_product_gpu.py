"""The tile products that run as six bfloat16 products per float32 product: at the edges of the tiles, exactly where
the result is a float32 number whatever the order of the sums, and against float64 elsewhere."""
import pytest
import torch

from chainerkfac_amd import ops

pytestmark = pytest.mark.gpu


def _signed_permutation(d, gen):
    """A symmetric matrix (as every inverse factor is) with one entry +-2^e per row: products with it are exact."""
    perm = torch.randperm(d, device='cuda', generator=gen)
    i, j = perm[:(d + 1) // 2], perm[d // 2:].flip(0)   # an odd d leaves its middle row to itself
    value = torch.randint(-3, 4, i.shape, device='cuda', generator=gen).float().exp2()
    value *= torch.randint(0, 2, i.shape, device='cuda', generator=gen).float() * 2 - 1
    m = torch.zeros((d, d), device='cuda')
    m[i, j] = value
    m[j, i] = value
    return m


@pytest.mark.parametrize('dG, dA', [(1, 2), (31, 33), (64, 65), (127, 129), (130, 256), (257, 1153)])
@pytest.mark.parametrize('bias', [False, True])
def test_all_24_bits_of_an_operand_reach_the_product(dG, dA, bias):
    # Every output has one nonzero term: hi, mid and lo of the operand times a power of two, added up exactly.
    # A plane that is dropped, swapped or taken from another row or k-value changes the bits.
    gen = torch.Generator(device='cuda').manual_seed(dG * 10007 + dA)
    G, A = _signed_permutation(dG, gen), _signed_permutation(dA, gen)
    g = torch.randn((dG, dA), device='cuda', generator=gen)
    gW, gb = (g[:, :-1].contiguous(), g[:, -1].contiguous()) if bias else (g, None)
    kfW, kfb = torch.empty_like(gW), torch.empty_like(gb) if bias else None
    ops.precond_conn(G, A, gW, gb, kfW, kfb)
    want = (G.double() @ g.double() @ A.double()).float()
    got = torch.cat([kfW, kfb[:, None]], 1) if bias else kfW
    assert torch.equal(got, want)


@pytest.mark.parametrize('d', [127, 128, 129, 255, 257, 640, 1025])
def test_inverse_within_the_float32_bound(d):
    # An inverse from float32 Cholesky factors has a relative error of at most a small multiple of d u cond(A)
    # (u = 2^-24); d u cond(A) itself is asked for: the statistical error is smaller by more than sqrt(d).
    gen = torch.Generator(device='cuda').manual_seed(d)
    x = torch.randn((2 * d, d), device='cuda', generator=gen)
    a = x.t() @ x / (2 * d)
    a.diagonal().add_(1e-3)
    a = (a + a.t()) / 2
    out = torch.empty_like(a)
    _, info = ops.spd_inverse_batched([a], outs=[out])
    ref = a.cpu().double()
    want = torch.linalg.inv(ref)
    bound = d * 2.0 ** -24 * float(torch.linalg.cond(ref))
    assert int(info.max()) == 0
    assert torch.equal(out, out.t())
    assert float((out.cpu().double() - want).norm() / want.norm()) <= bound
