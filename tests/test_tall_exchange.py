"""The exchange path on 256-row tiles (two entry slots each): its rule on the
CPU, and its results at the edges of its ranges on the GPU against 64-bit
torch."""
from __future__ import annotations

import math

import pytest

torch = pytest.importorskip("torch")

from welder_typical_chain_amd import _lib  # noqa: E402

needs_gpu = pytest.mark.skipif(not torch.cuda.is_available(), reason="no GPU")
TYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32, "fp8": torch.float8_e4m3fn}
TILES = [128, 128, 64, 2, 32]


def _plan(batch, m, n, k=256):
    return _lib.plan(batch, m, n, k, _lib.DTYPE_F16, _lib.DTYPE_F16, _lib.PATH_EXCHANGE)


def test_rule(native_lib):
    """128-row tiles while they fit on 256 CUs, then 256-row tiles while those do,
    for rows of at most 32 column tiles."""
    assert _plan(1, 2048, 2048)["grid"] == 256
    pl = _plan(1, 2049, 2048)
    assert pl["grid"] == 9 * 16 and pl["tiles"] == TILES
    assert _plan(1, 3840, 2048)["grid"] == 15 * 16
    assert _plan(1, 4096, 2048)["grid"] == _plan(1, 2048, 4096)["grid"] == _plan(8, 1024, 1024)["grid"] == 256
    assert _plan(1, 1500, 4096)["grid"] == 6 * 32
    for m, n in ((4097, 2048), (1500, 4104)):
        with pytest.raises(_lib.WtcError):
            _plan(1, m, n)
    # a slot per 128 rows: the entries fit what the workspace holds for them
    pl = _plan(15, 130, 2048)
    assert pl["grid"] == 15 * 16 and pl["workspace_bytes"] >= 256 + 4096 + 2 * pl["grid"] * 1024


SHAPES = [
    # the last row block: 220 rows, 1 row, a full one; two row blocks per batch of 2 rows and 257
    (1, 1500, 3000, 1000), (1, 2049, 2048, 64), (1, 3840, 2048, 136), (15, 130, 2048, 256), (5, 257, 3080, 72),
    # every CU: 256 tiles (with f32 outputs every slot there is)
    (1, 4096, 2048, 72), (8, 1000, 1024, 128),
    # 32 column tiles, the last of 8 columns; no K at all
    (1, 1500, 3976, 320), (1, 2304, 2048, 0),
]


@pytest.mark.gpu
@needs_gpu
@pytest.mark.parametrize("in_dtype,out_dtype", [("f16", "f16"), ("bf16", "bf16"), ("f16", "f32")])
@pytest.mark.parametrize("batch,m,n,k", SHAPES)
def test_tall_exchange(native_lib, batch, m, n, k, in_dtype, out_dtype):
    """Tolerance: one rounding to the output type, and the f32 sums' error:
    2^-24 (K + 8) of the sum of magnitudes per logit, doubled by the softmax.
    Between calls of one shape and the other row heights the slots'
    generations must agree: 128-row calls on the same workspace in between."""
    from welder_typical_chain_amd.chain import matmul_softmax
    print(f"\n[gpu-case] tall exchange {in_dtype}->{out_dtype} {batch}x{m}x{n}x{k}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(m * n + k)
    a = torch.randn((batch, m, k), generator=g, device="cuda").to(TYPES[in_dtype])
    b = torch.randn((batch, k, n), generator=g, device="cuda").to(TYPES[in_dtype])
    ulp = {"f16": 2.0 ** -11, "bf16": 2.0 ** -8, "f32": 0.0}[out_dtype]
    least = {"f16": 2.0 ** -24, "bf16": 1e-38, "f32": 1e-38}[out_dtype]
    for scale in (1.0 / math.sqrt(max(k, 1)), -0.3):
        y = torch.matmul(a.double(), b.double()) * scale
        want = torch.softmax(y, dim=-1)
        mag = torch.matmul(a.abs().double(), b.abs().double()).amax(-1, keepdim=True) * abs(scale)
        bound = want * (ulp + 2 * mag * (k + 8) * 2.0 ** -24 + 8 * 2.0 ** -22) + least
        for rows in (m, min(m, 300), m):
            part = a[:1, :rows].contiguous() if rows < m else a
            ops = (part, b[:1] if rows < m else b)
            out = torch.full((ops[0].shape[0], rows, n), 7.0, dtype=TYPES[out_dtype], device="cuda")
            matmul_softmax(*ops, out=out, logit_scale=scale, path="exchange", tiles=TILES, check=True)
            err = (out.double() - want[:out.shape[0], :rows]).abs()
            assert bool((err <= bound[:out.shape[0], :rows]).all()), rows


def test_slots_of_f32_outputs(native_lib):
    """Two entries a row (max and sum): four slots per tile, in the workspace and within the slots' limit."""
    for m in (2049, 3840, 4096):
        pl = _lib.plan(1, m, 2048, 256, _lib.DTYPE_F16, _lib.DTYPE_F32, _lib.PATH_EXCHANGE)
        assert pl["grid"] == -(-m // 256) * 16 and 4 * pl["grid"] <= 1024
        assert pl["workspace_bytes"] >= 256 + 4096 + 4 * pl["grid"] * 1024
        size = _lib.lib().wtc_matmul_softmax_workspace_size
        for path in (_lib.PATH_AUTO, _lib.PATH_EXCHANGE):
            assert size(1, m, 2048, 256, _lib.DTYPE_F16, _lib.DTYPE_F32, path) >= pl["workspace_bytes"]
    # other paths and smaller tiles ask for no more than with 16-bit outputs
    for path, m in ((_lib.PATH_SPLIT, 2049), (_lib.PATH_EXCHANGE, 2048), (_lib.PATH_ROWS, 2049)):
        wide, half = (_lib.plan(1, m, 2048, 64, _lib.DTYPE_F16, out, path)["workspace_bytes"]
                      for out in (_lib.DTYPE_F32, _lib.DTYPE_F16))
        assert wide == half


@pytest.mark.gpu
@needs_gpu
@pytest.mark.parametrize("in_dtype,batch,m,n,k,deviation", [
    ("f16", 1, 1500, 3000, 64, 1.0), ("bf16", 1, 1500, 3000, 256, 8.0), ("bf16", 15, 130, 2048, 256, 1.0),
    ("f16", 1, 3328, 2048, 128, 32.0), ("fp8", 1, 2304, 2048, 1024, 32.0),
])
def test_f32_outputs_as_close_as_the_split_path(native_lib, in_dtype, batch, m, n, k, deviation):
    """Relative 2-norm error against 64 bits, both paths on the same products:
    row statistics exchanged in less than the split path keeps (max and sum)
    show as 10 to 40 % more; what differs is the last product's rounding."""
    from welder_typical_chain_amd.chain import matmul_softmax
    print(f"\n[gpu-case] tall exchange accuracy {in_dtype} {batch}x{m}x{n}x{k}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(k)
    a = torch.randn((batch, m, k), generator=g, device="cuda").to(TYPES[in_dtype])
    b = torch.randn((batch, k, n), generator=g, device="cuda").to(TYPES[in_dtype])
    scale = deviation / math.sqrt(k)
    want = torch.softmax(torch.matmul(a.float().double(), b.float().double()) * scale, dim=-1)

    def error(path, tiles):
        out = torch.empty((batch, m, n), device="cuda")
        matmul_softmax(a, b, out=out, logit_scale=scale, path=path, tiles=tiles, check=True)
        return float((out.double() - want).norm() / want.norm())
    k_tile = 128 if in_dtype == "fp8" else 64
    split = error("split", [256, 128, k_tile, 2, 32])
    exchange = error("exchange", [128, 128, k_tile, 2, 32])
    assert exchange <= 1.02 * split, (exchange, split)
