"""f32 inputs on the bf16 matrix cores (chain_tile_kernel<f32>): the sizes
where its tiles can go wrong, the values that do not split into three bf16
parts, and that it is no further from 64 bits than a f32 product.

Tolerance: each of the (at most K + 8) f32 roundings of a logit's sum is at
most 2^-24 of the sum of its magnitudes S = scale * sum |a b|, the partial
products left out 2^-24 of it (test_f32_layout.py); the softmax turns a logit error d into a
relative one of at most 2 d (its own and the row sum's), to which exp2, the
row sum (N / 128 partial sums) and the final product add a few 2^-22.
"""
from __future__ import annotations

import math

import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

needs_gpu = pytest.mark.skipif(not torch.cuda.is_available(), reason="no GPU")


def _inputs(batch, m, n, k, seed, spread=1.0):
    g = torch.Generator().manual_seed(seed)
    a = torch.randn((batch, m, k), generator=g) * spread / math.sqrt(k)
    b = torch.randn((batch, k, n), generator=g)
    return a, b


def _reference(a, b, scale):
    y = torch.matmul(a.double(), b.double()) * scale
    mag = torch.matmul(a.abs().double(), b.abs().double()) * abs(scale)
    return torch.softmax(y, dim=-1), mag


def _check(out, a, b, scale):
    want, mag = _reference(a, b, scale)
    k, n = b.shape[-2:]
    d = mag.amax(-1, keepdim=True) * (k + 8) * 2.0 ** -24
    bound = want * (2 * d + (4 + n / 128) * 2.0 ** -22) + 1e-37
    err = (out.double().cpu() - want).abs()
    assert bool((err <= bound).all()), float((err / bound).max())


SHAPES = [
    # 64 x 64 tiles, one k-group: a single one, its edges, one past them
    (1, 1, 8, 4), (1, 64, 64, 32), (1, 65, 72, 36), (2, 63, 136, 64), (1, 130, 520, 192),
    # two k-groups: short and ragged K, the ring's first turns
    (1, 64, 64, 196), (1, 70, 200, 224), (3, 129, 64, 260), (1, 200, 264, 1024),
    # more than one tile to a CU (257 .. 512 tiles), ragged
    (1, 2048, 520, 36), (2, 1000, 1000, 196), (1, 64, 4096, 200),
    # 128 x 128 tiles on the exchange path (over 512 tiles of 64) and past it (split)
    (1, 1500, 2000, 68), (1, 2048, 2048, 196), (1, 2100, 2104, 132), (1, 257, 8200, 36),
]


@needs_gpu
@pytest.mark.parametrize("batch,m,n,k", SHAPES)
def test_tile_edges(native_lib, batch, m, n, k):
    from welder_typical_chain_amd.chain import matmul_softmax, read_diagnostics
    print(f"\n[gpu-case] f32 {batch}x{m}x{n}x{k}", flush=True)
    a, b = _inputs(batch, m, n, k, seed=m + n + k, spread=2.0)
    for scale in (0.7, -1.3):
        out = matmul_softmax(a.cuda(), b.cuda(), logit_scale=scale, check=True)
        _check(out, a, b, scale)
    assert read_diagnostics()[0] == 0


@needs_gpu
@pytest.mark.parametrize("path", ["exchange", "split", "unfused"])
@pytest.mark.parametrize("m,n,k", [(130, 200, 100), (130, 200, 300)])
@pytest.mark.parametrize("what", ["tiny", "huge", "zero", "part_subnormal", "probabilities", "tiny_products"])
def test_values_past_the_split(native_lib, path, m, n, k, what):
    """Magnitudes whose bf16 parts would be subnormal or infinite, zeros,
    probabilities (down to 1e-45, recomputed or not the same to f32), and
    products of ordinary values that are themselves tiny."""
    from welder_typical_chain_amd.chain import matmul_softmax
    print(f"\n[gpu-case] f32 {what} {path} {m}x{n}x{k}", flush=True)
    a, b = _inputs(1, m, n, k, seed=5, spread=2.0)
    if what == "tiny":
        a, b = a * 2.0 ** -120, b * 2.0 ** 120
    elif what == "huge":
        a, b = a * 2.0 ** -126, b * 2.0 ** 124
        b[0, 3, 5] = 3.4e38
        a[0, :, 3] *= 2.0 ** -20
    elif what == "zero":
        a[0, 7] = 0.0
        b[0, :, 9] = 0.0
        a[0, :, 40:70] = 0.0
    elif what == "probabilities":
        a = torch.softmax(a * (30.0 * math.sqrt(k)), dim=-1)
        assert bool(((a > 0) & (a < 2.0 ** -100)).any())
    elif what == "tiny_products":
        a, b = a * 2.0 ** -60, b * 2.0 ** -60
    else:
        a[0, 11, 4] = 1.1754944e-38
        b[0, 5, 66] = 1e-42
    scale = {"huge": 4.0, "tiny_products": 2.0 ** 120}.get(what, 1.0)
    out = matmul_softmax(a[0].cuda(), b[0].cuda(), logit_scale=scale, path=path)
    _check(out[None], a, b, scale)


@needs_gpu
@pytest.mark.parametrize("path", ["exchange", "split"])
@pytest.mark.parametrize("k", [64, 260])
def test_infinities_and_nan(native_lib, path, k):
    """A row or column with an infinity or NaN gives what f32 products give;
    the rows without one are not touched by it."""
    from welder_typical_chain_amd.chain import matmul_softmax
    print(f"\n[gpu-case] f32 non-finite {path} k={k}", flush=True)
    m, n = 200, 136
    a, b = _inputs(1, m, n, k, seed=9)
    a, b = a[0], b[0]
    a[3, 10] = math.inf            # logits +-inf: a NaN row
    a[70, 2] = math.nan
    b[5, 100] = -math.inf          # with a[:, 5] > 0 a logit of -inf: probability 0
    a[:, 5] = a[:, 5].abs() + 0.1
    got = matmul_softmax(a.cuda(), b.cuda(), path=path).cpu()
    want = torch.softmax(torch.matmul(a, b), dim=-1)
    assert torch.equal(got.isnan(), want.isnan())
    keep = ~want.isnan().any(-1)
    assert int(keep.sum()) == m - 2 and bool((got[keep, 100] == 0).all())
    assert torch.allclose(got[keep], want[keep], rtol=2e-5, atol=1e-9)


@needs_gpu
@pytest.mark.parametrize("m,n,k", [(512, 512, 1024), (1024, 2048, 260)])
def test_no_further_from_64_bits_than_f32_products(native_lib, m, n, k):
    """Relative 2-norm error of the outputs against a f32 product's (torch's
    CPU one, blocked sums) on the same inputs."""
    from welder_typical_chain_amd.chain import matmul_softmax
    print(f"\n[gpu-case] f32 accuracy {m}x{n}x{k}", flush=True)
    a, b = _inputs(1, m, n, k, seed=2)
    want, _ = _reference(a, b, 1.0)
    f32 = torch.softmax(torch.matmul(a, b).double(), dim=-1)
    got = matmul_softmax(a.cuda(), b.cuda()).double().cpu()
    err = float((got - want).norm() / want.norm())
    # the kernel's own softmax arithmetic (exp2, sums, product) is in f32 too
    assert err <= 1.5 * float((f32 - want).norm() / want.norm()) + 3e-7, err


@needs_gpu
@pytest.mark.parametrize("m,n,k", [(1024, 1024, 1024), (2048, 2048, 512)])
def test_probabilities_take_no_longer(native_lib, m, n, k):
    """Values below 2^-100 beside ones near 1 do not reach a result: no tile is
    recomputed for them (that takes 1.5 times the call, and did three times)."""
    from welder_typical_chain_amd.chain import matmul_softmax
    print(f"\n[gpu-case] f32 time with tiny values {m}x{n}x{k}", flush=True)
    a, b = (x[0].cuda() for x in _inputs(1, m, n, k, seed=3))
    tiny = a.clone()
    tiny[::17, ::13] = 1e-32
    out = torch.empty((m, n), device="cuda")

    def us(x):
        best = math.inf
        for _ in range(5):
            t0, t1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            t0.record()
            for _ in range(50):
                matmul_softmax(x, b, out=out)
            t1.record()
            torch.cuda.synchronize()
            best = min(best, t0.elapsed_time(t1) * 20)
        return best
    us(a)
    plain, with_tiny = us(a), us(tiny)
    assert with_tiny < 1.25 * plain, (with_tiny, plain)


@needs_gpu
@pytest.mark.parametrize("m,n,k", [(256, 512, 64), (512, 512, 1024), (1500, 2000, 256)])
def test_mantissas_at_the_worst_of_the_split(native_lib, m, n, k):
    """All products of one sign, both operands within 3 units in the last place of
    1 + 2^-8 - 2^-17, where the partial products left out are 2^-24 of each
    product: they add up to S 2^-24 per logit (S = 8 here).  Allowed beside it: the
    roundings of a sum that grows to S in t = 6 K / 16 steps, of either sign and
    evenly spread over half a unit (0.29 sqrt(t / 3) of 2^-24 S in the mean
    square), both doubled by the softmax, and its own arithmetic (exp2, sums,
    product)."""
    from welder_typical_chain_amd.chain import matmul_softmax
    print(f"\n[gpu-case] f32 worst mantissas {m}x{n}x{k}", flush=True)
    g = torch.Generator().manual_seed(k)

    def near(shape):
        ulps = torch.randint(-3, 4, shape, generator=g).float()
        return 1.0 + 2.0 ** -8 - 2.0 ** -17 + ulps * 2.0 ** -23
    a, b = near((m, k)), near((k, n))
    scale = 8.0 / k
    want = torch.softmax(torch.matmul(a.double(), b.double()) * scale, dim=-1)
    got = matmul_softmax(a.cuda(), b.cuda(), logit_scale=scale).double().cpu()
    err = float((got - want).norm() / want.norm())
    assert err <= 2 * 8.0 * 2.0 ** -24 * (1 + 0.29 * math.sqrt(6 * k / 16 / 3)) + 5e-7, err
