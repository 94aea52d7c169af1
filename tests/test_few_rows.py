"""The few-row kernel (a batch's rows at most 32, its logits in LDS): its rule
on the CPU, and its results at the edges of its ranges on the GPU against
64-bit torch."""
from __future__ import annotations

import math

import pytest

torch = pytest.importorskip("torch")

from welder_typical_chain_amd import _lib  # noqa: E402

needs_gpu = pytest.mark.skipif(not torch.cuda.is_available(), reason="no GPU")
TYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}


def _grid(batch, m, n, k=128):
    return _lib.plan(batch, m, n, k, _lib.DTYPE_F16, _lib.DTYPE_F16, _lib.PATH_ROWS)["grid"]


def test_rule(native_lib):
    """32 rows and 16384 floats of logits (columns padded to 128, 4 floats more
    a row), else 128-row blocks; both have one workgroup per batch here, so the
    estimate tells them apart."""
    def est(m, n):
        return _lib.plan(64, m, n, 128, _lib.DTYPE_F16, _lib.DTYPE_F16, _lib.PATH_ROWS)["est_us"]
    assert _grid(300, 32, 384) == 300 and _grid(300, 33, 384) == 300 and _grid(3, 129, 384) == 6
    for inside, past in (((32, 384), (33, 384)), ((1, 16256), (1, 16264)), ((8, 1920), (8, 2048)),
                         ((4, 3968), (4, 4096))):
        rows, n = past
        block = est(100, n)  # a 128-row block for certain
        assert abs(est(*past) - block) < 0.05 * block, past  # but for A's and out's bytes
        assert abs(est(*inside) - est(100, inside[1])) > 0.08 * est(*inside), inside


SHAPES = [
    # one row over one tile and less, K from nothing to 128 (one and two units a tile)
    (1, 1, 8, 8), (3, 1, 128, 64), (2, 1, 136, 72), (2, 1, 264, 128), (2, 2, 200, 0),
    # rows per wave: 8, 4, 2, 1 waves a row and more rows than waves
    (5, 2, 1000, 96), (4, 3, 5368, 40), (4, 4, 2048, 128), (3, 5, 3200, 64), (2, 7, 2304, 128),
    (2, 8, 1920, 120), (2, 9, 1792, 16), (3, 32, 384, 128), (2, 31, 504, 56),
    # the longest row
    (2, 1, 16256, 128),
    # two workgroups per CU
    (600, 1, 2048, 64), (513, 3, 1000, 128),
]


@pytest.mark.gpu
@needs_gpu
@pytest.mark.parametrize("in_dtype,out_dtype", [("f16", "f16"), ("bf16", "bf16"), ("bf16", "f32")])
@pytest.mark.parametrize("batch,m,n,k", SHAPES)
def test_few_rows(native_lib, batch, m, n, k, in_dtype, out_dtype):
    """Tolerance: one rounding to the output type, and the f32 sums' error:
    2^-24 (K + 8) of the sum of magnitudes per logit, doubled by the softmax."""
    from welder_typical_chain_amd.chain import matmul_softmax
    print(f"\n[gpu-case] few rows {in_dtype}->{out_dtype} {batch}x{m}x{n}x{k}", flush=True)
    g = torch.Generator().manual_seed(m * n + k)
    a = torch.randn((batch, m, k), generator=g).to(TYPES[in_dtype])
    b = torch.randn((batch, k, n), generator=g).to(TYPES[in_dtype])
    ulp = {"f16": 2.0 ** -11, "bf16": 2.0 ** -8, "f32": 0.0}[out_dtype]
    least = {"f16": 2.0 ** -24, "bf16": 1e-38, "f32": 1e-38}[out_dtype]
    for scale in (1.0 / math.sqrt(max(k, 1)), -0.3):
        out = torch.full((batch, m, n), 7.0, dtype=TYPES[out_dtype], device="cuda")
        matmul_softmax(a.cuda(), b.cuda(), out=out, logit_scale=scale, path="rows")
        y = torch.matmul(a.double(), b.double()) * scale
        want = torch.softmax(y, dim=-1)
        mag = torch.matmul(a.abs().double(), b.abs().double()).amax(-1, keepdim=True) * abs(scale)
        bound = want * (ulp + 2 * mag * (k + 8) * 2.0 ** -24 + 8 * 2.0 ** -22) + least
        err = (out.double().cpu() - want).abs()
        assert bool((err <= bound).all()), float((err / bound).max())


@pytest.mark.gpu
@needs_gpu
@pytest.mark.parametrize("m,n", [(1, 1000), (6, 520)])
def test_non_finite_rows(native_lib, m, n):
    """NaN and infinite logits make their own row NaN, -inf ones are 0."""
    from welder_typical_chain_amd.chain import matmul_softmax
    print(f"\n[gpu-case] few rows non-finite {m}x{n}", flush=True)
    g = torch.Generator().manual_seed(4)
    a = torch.randn((3, m, 64), generator=g).half()
    b = torch.randn((3, 64, n), generator=g).half()
    a[1, m - 1, 3] = math.nan
    a[:, :, 7] = 1.0
    b[0, 7, 11] = -math.inf
    b[2, 7, n - 1] = math.inf
    got = matmul_softmax(a.cuda(), b.cuda(), out_dtype=torch.float32, path="rows").cpu()
    want = torch.softmax(torch.matmul(a.float(), b.float()), dim=-1)
    assert torch.equal(got.isnan(), want.isnan())
    assert bool((got[0, :, 11] == 0).all()) and bool(got[2].isnan().all())
    assert torch.allclose(got[0], want[0], rtol=1e-4, atol=1e-9)
