"""The tile products that run as six bfloat16 products per float32 product, and their rules and ranges: at the edges of
the tiles, exactly where the result is a float32 number whatever the order of the sums, and against float64 elsewhere."""
import pytest
import torch

from chainerkfac_amd import _lib, ops

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


def _twelve_bits(shape, gen):
    """Numbers of 12 significand bits (two bfloat16 numbers each): a product of two is a float32 number."""
    sign = torch.randint(0, 2, shape, device='cuda', generator=gen) * 2 - 1
    return (torch.randint(2048, 4096, shape, device='cuda', generator=gen) * sign).float() / 2048


# launches of 64-tiles with the float32 instruction, of 64-tiles with split products and of 128-tiles, in both
# products of a layer; loads of one and of four values; several k-slices
@pytest.mark.parametrize('dG, dA', [(10, 101), (256, 257), (768, 577), (513, 1025), (1000, 785), (1100, 1100), (515, 2049)])
@pytest.mark.parametrize('twelve', ['G', 'A'])
def test_products_of_two_planes_are_exact(dG, dA, twelve):
    # One operand pair of every output has mid planes on both sides (mid * mid is 2^-16 of the product), the other
    # factor is a power of two: the result is a float32 number.
    gen = torch.Generator(device='cuda').manual_seed(dG * 10007 + dA)
    G, A = _signed_permutation(dG, gen), _signed_permutation(dA, gen)
    F = G if twelve == 'G' else A
    m = _twelve_bits(F.shape, gen)
    F *= torch.tril(m) + torch.tril(m, -1).t()
    g = _twelve_bits((dG, dA), gen)
    kf, _ = ops.precond_conn(G, A, g)
    assert torch.equal(kf, (G.double() @ g.double() @ A.double()).float())


def _float32_chain(x, slices):
    """x^T x as float32 sums in the order of the k-values, one rounding each, slice by slice."""
    total = None
    for part in x.double().split(slices):
        acc = torch.zeros((x.shape[1], x.shape[1]), device=x.device)
        for row in part:
            acc = (acc.double() + row[:, None] * row[None, :]).float()
        total = acc if total is None else total + acc
    return total


def _rms(got, want, scale):
    return float(((got.double() - want) / scale.clamp_min(1e-300)).pow(2).mean().sqrt())


@pytest.mark.parametrize('route', ['single', 'group', 'macro'])
@pytest.mark.parametrize('d', [60, 300, 700])
@pytest.mark.parametrize('shift', [0.0, 1.0])
def test_covariance_of_rectified_values_as_exact_as_float32_sums(route, d, shift):
    # Rectified activations are the operands that a covariance mostly meets: every product with a zero leaves a
    # float32 sum as it is, so a kernel that rounds its sum whether or not anything is added loses accuracy there.
    # The root mean square of the error over some 1e4 .. 1e5 entries scatters by a few per cent: 1.1 times is asked for.
    gen = torch.Generator(device='cuda').manual_seed(d)
    n, slices = (512, 256) if route == 'macro' else (352, 352)   # as the planners cut these reductions
    x = (torch.randn((n, d), device='cuda', generator=gen) - shift).relu()
    out = torch.empty((d, d), device='cuda')
    if route == 'single':
        ops.cov_linear(x, False, 1.0, out=out)
    else:
        slab = x.view(n // 16, 16, d).transpose(1, 2).contiguous().view(n // 16, d, 4, 4)   # (sample, channel, pixel)
        with _lib.options(group_macro=int(route == 'macro')):
            ops.CovGroup([(ops.COV_SLAB, n // 16, d, 4, 4, 1, 1, 0, 1)]).run([slab], [out], [1.0], [0.0])
    want = x.double().t() @ x.double()
    assert _rms(out, want, want) <= 1.1 * _rms(_float32_chain(x, slices), want, want)


@pytest.mark.parametrize('route', ['linear', 'slab', 'group'])
@pytest.mark.parametrize('n, d', [(1, 31), (1, 700), (5, 65), (31, 129), (128, 300), (33, 4200)])
def test_short_covariances_round_a_product_once(route, n, d):
    # One k-value with anything in it: every entry is one product, and a float32 sum rounds it once.
    gen = torch.Generator(device='cuda').manual_seed(n * 10007 + d)
    x = torch.zeros((n, d), device='cuda')
    x[n // 2] = torch.randn(d, device='cuda', generator=gen)
    out = torch.empty((d + 1, d + 1), device='cuda')
    if route == 'linear':
        ops.cov_linear(x, True, 1.0, out=out)
    elif route == 'slab':
        ops.cov_conv_a(x.view(n, d, 1, 1), 1, 1, 0, True, 1.0, out=out)
    else:
        ops.CovGroup([(ops.COV_LINEAR, n, d, 1, 1, 1, 1, 1, 1)]).run([x], [out], [1.0], [0.0])
    row = x[n // 2].double()
    assert torch.equal(out[:d, :d], (row[:, None] * row[None, :]).float())
    assert torch.equal(out[d, :d], x[n // 2]) and torch.equal(out[:d, d], x[n // 2]) and float(out[d, d]) == n


@pytest.mark.parametrize('dG, dA', [(1, 2), (10, 101), (64, 577), (256, 257), (512, 513)])
def test_small_layers_round_a_product_once(dG, dA):
    # Products with a workgroup per CU or less take the float32 instruction, which rounds a single product once.
    gen = torch.Generator(device='cuda').manual_seed(dG * 10007 + dA)
    G, A = _signed_permutation(dG, gen), _signed_permutation(dA, gen)
    m = torch.rand(G.shape, device='cuda', generator=gen) + 0.5
    G *= torch.tril(m) + torch.tril(m, -1).t()
    g = torch.randn((dG, dA), device='cuda', generator=gen)
    kf, _ = ops.precond_conn(G, A, g)
    assert torch.equal(kf, ((G.double() @ g.double()).float().double() @ A.double()).float())


@pytest.mark.parametrize('shape', [(2, 128, 14, 14), (4, 65, 13, 13), (3, 300, 9, 9)])
@pytest.mark.parametrize('stride', [1, 2])
def test_covariances_of_few_workgroups_round_a_product_once(shape, stride):
    # Several tiles, a workgroup per CU or less, more than 128 k-values; subsampled slabs at any size.
    gen = torch.Generator(device='cuda').manual_seed(shape[1])
    shape = shape[:2] + (shape[2] * stride, shape[3] * stride)
    x = torch.zeros(shape, device='cuda')
    v = torch.randn(shape[1], device='cuda', generator=gen)
    x[1, :, 2 * stride, 5 * stride] = v
    out = ops.cov_conv_a(x, 1, stride, 0, False, 1.0)
    assert torch.equal(out, (v.double()[:, None] * v.double()[None, :]).float())


# one shape per way that operands reach split products: 64- and 128-tiles, whole and ragged, every loader
_COVARIANCES = {
    'linear64': (8192, 320), 'linear64_scalar': (2048, 511), 'linear128': (300, 700), 'linear128_scalar': (300, 701),
    'slab64': (32, 512, 14, 14), 'slab64_scalar': (32, 320, 21, 21), 'slab128': (4, 700, 10, 10),
    'slab128_scalar': (4, 700, 9, 9), 'strided128': (4, 600, 18, 18), 'gather64': (16, 8, 31, 31),
    'gather128': (4, 70, 11, 11), 'group64': (8, 100, 6, 6), 'group64_scalar': (8, 100, 5, 5),
    'group128': (8, 300, 6, 6), 'group128_scalar': (8, 300, 5, 5), 'group_linear64': (200, 100),
    'group_linear128': (200, 300), 'group_linear128_scalar': (200, 301),
}


def _covariance(route, make):
    """(P^T P with a ones column, the patch matrix P) of an input ``make(shape)``; P in float64 on the GPU."""
    shape = _COVARIANCES[route]
    x = make(shape)
    stride = 2 if route.startswith('strided') else 1
    if len(shape) == 2:
        P = x
    elif route.startswith('gather'):
        P = torch.nn.functional.unfold(x, 5).transpose(1, 2).reshape(-1, shape[1] * 25)
    else:
        P = x[:, :, ::stride, ::stride].permute(0, 2, 3, 1).reshape(-1, shape[1])
    d = P.shape[1]
    out = torch.empty((d + 1, d + 1), device='cuda')
    if route.startswith('group'):
        kind, hw = (ops.COV_LINEAR, (1, 1)) if len(shape) == 2 else (ops.COV_SLAB, shape[2:])
        ops.CovGroup([(kind, shape[0], shape[1]) + hw + (1, 1, 1, 1)]).run([x], [out], [1.0], [0.0])
    elif len(shape) == 2:
        ops.cov_linear(x, True, 1.0, out=out)
    else:
        ops.cov_conv_a(x, 5 if route.startswith('gather') else 1, stride, 0, True, 1.0, out=out)
    P = torch.cat([P, torch.ones((P.shape[0], 1), device='cuda')], 1).double()
    return out, P


@pytest.mark.parametrize('at', ['first', 'middle', 'last'])
@pytest.mark.parametrize('route', list(_COVARIANCES))
def test_every_plane_reaches_the_covariance(route, at):
    # One k-value (one pixel of one sample) with anything in it, so that every entry is one product, of a power of two and
    # anything or of two numbers of 12 bits: a float32 number.  A plane that is dropped, swapped, or taken from another
    # row or k-value changes the bits; the ones column holds the value itself.
    gen = torch.Generator(device='cuda').manual_seed(len(route))
    shape = _COVARIANCES[route]
    c = shape[1]
    v = torch.randn(c, device='cuda', generator=gen)
    v[0::3] = torch.randint(-6, 7, v[0::3].shape, device='cuda', generator=gen).float().exp2()
    v[1::3] = _twelve_bits(v[1::3].shape, gen)
    where = {'first': 0.0, 'middle': 0.6, 'last': 1.0}[at]
    stride = 2 if route.startswith('strided') else 1

    def make(shape):
        x = torch.zeros(shape, device='cuda')
        pixel = [int(where * (n - 1)) // stride * stride for n in shape[2:]]
        x[(int(where * (shape[0] - 1)), slice(None)) + tuple(pixel)] = v
        return x

    out, P = _covariance(route, make)
    want = P.t() @ P
    channel = torch.arange(P.shape[1], device='cuda')
    if route.startswith('gather'):
        channel = torch.div(channel, 25, rounding_mode='floor')
    channel[-1] = 0   # the ones column
    kind = channel % 3
    exact = (kind[:, None] == 0) | (kind[None, :] == 0) | ((kind[:, None] == 1) & (kind[None, :] == 1))
    assert torch.equal(out[exact], want.float()[exact])
    # the rest misses mid * lo, lo * mid and lo * lo: 2^-23 together, and the rounding of the sum
    assert bool(((out.double() - want).abs() <= 2.0 ** -22 * want.abs()).all())


def _assert_close_where_finite(got, want, scale, tol):
    """Infinities and NaN as in ``want`` (float64, rounded to float32); elsewhere |difference| <= tol * scale."""
    want32 = want.float()
    assert torch.equal(torch.isnan(got), torch.isnan(want32))
    assert torch.equal(got[torch.isinf(want32)], want32[torch.isinf(want32)])
    fine = torch.isfinite(want32)
    assert bool(torch.isfinite(got[fine]).all())
    error = (got.double() - want).abs()
    assert bool((error <= tol * scale)[fine].all()), float((error / scale)[fine].max())


def _operands(shape, column, kind, gen):
    x = torch.randn(shape, device='cuda', generator=gen)
    if kind == 'inf':
        x[0, column].view(-1)[-1:] = float('inf')
    elif kind == 'nan':
        x[0, column].view(-1)[-1:] = float('nan')
    elif kind == 'huge':      # the last float32 numbers round to infinity as bfloat16
        x *= 2.0 ** -20
        x[0, column].view(-1)[-1:] = -torch.finfo(torch.float32).max
    elif kind == 'both small':
        x *= 2.0 ** -58
    else:                     # a power of two; below 2^-110 a bfloat16 number cannot hold the last bits
        x[:, column] *= 2.0 ** kind
    return x


@pytest.mark.parametrize('kind', ['inf', 'nan', 'huge', 'both small', -105, -109, -112, -120, -135])
@pytest.mark.parametrize('route', list(_COVARIANCES))
def test_covariances_over_the_range_of_float32(route, kind):
    gen = torch.Generator(device='cuda').manual_seed(5)
    column = _COVARIANCES[route][1] * 2 // 3
    out, P = _covariance(route, lambda shape: _operands(shape, column, kind, gen))
    # float32 sums of n products of either sign, to a part of n u (u = 2^-24) of the sum of their magnitudes; results
    # under 2^-126 are held to multiples of 2^-149, once per sum of sixteen k-values or two
    n = P.shape[0]
    scale = P.abs().t() @ P.abs()
    scale = torch.where(torch.isfinite(scale), scale, torch.ones_like(scale)) + n * 2.0 ** -149 / (64 * 2.0 ** -24)
    _assert_close_where_finite(out, P.t() @ P, scale, 64 * 2.0 ** -24)


@pytest.mark.parametrize('kind', ['inf', 'nan', 'huge', 'both small', -105, -109, -112, -120, -135])
@pytest.mark.parametrize('dG, dA, group', [(768, 577, False), (1100, 1100, False), (513, 1025, False), (60, 70, True),
                                           (200, 300, True), (201, 301, True)])
def test_preconditioning_over_the_range_of_float32(dG, dA, group, kind):
    gen = torch.Generator(device='cuda').manual_seed(6)
    G = torch.eye(dG, device='cuda')
    A = torch.randn((dA, dA), device='cuda', generator=gen)
    A = torch.tril(A) + torch.tril(A, -1).t()
    g = _operands((dA, dG), dG // 3, kind, gen).t().contiguous()
    if kind == 'both small':
        A *= 2.0 ** -58
    if kind == 'huge':
        A *= 2.0 ** -20
    if kind in ('inf', 'nan'):
        # the identity's zeros times an infinity are NaN in the whole column of the first product
        G = torch.full((dG, dG), 0.5, device='cuda')
    if group:
        kf = torch.empty_like(g)
        ops.PrecondGroup([(dG, dA, 0)]).run([G], [A], [g], [None], [kf], [None])
    else:
        kf, _ = ops.precond_conn(G, A, g)
    T = G.double() @ g.double()
    scale = (G.double().abs() @ g.double().abs()) @ A.double().abs()
    scale = torch.where(torch.isfinite(scale), scale, torch.ones_like(scale)) + (dG + dA) * 2.0 ** -149 / (64 * 2.0 ** -24)
    _assert_close_where_finite(kf, T @ A.double(), scale, 64 * 2.0 ** -24)
