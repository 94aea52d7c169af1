"""The forms of the exchange path beside its 128-row tiles: 256-row tiles (two
entry slots each, with f32 outputs four) and f32 inputs on 64 x 64 tiles, two
workgroups to a CU.

* Waits that run out (a limit of 2 ticks set from the host: every wait is
  bounded and every kernel exits normally) are reported, and the next call on
  the same workspace is right.
* A captured call replays to the eager output, with other inputs each time.
* A call that needs the largest workspace of the path runs under capture on a
  stream whose default workspace an earlier, small call made.
* fp8 inputs: the same as the split path's tiles of the same products.
"""
from __future__ import annotations

import math

import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

needs_gpu = pytest.mark.skipif(not torch.cuda.is_available(), reason="no GPU")
TYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32, "fp8": torch.float8_e4m3fn}
CODES = {"f32": 0, "f16": 1, "bf16": 2, "fp8": 3}
ROUNDING = {"f16": 2.0 ** -11, "bf16": 2.0 ** -8, "f32": 0.0}

# in, out, m, n, workgroups: 256-row tiles on some and on all CUs, 64 x 64 tiles
FORMS = [("f16", "f16", 3300, 2048, 208), ("bf16", "f32", 4096, 2048, 256), ("f32", "f32", 2048, 1024, 512)]


def _operands(in_dtype, m, n, k, seed, batch=1):
    g = torch.Generator(device="cuda").manual_seed(seed)
    a = torch.randn((batch, m, k), generator=g, device="cuda")
    b = torch.randn((batch, k, n), generator=g, device="cuda")
    return a.to(TYPES[in_dtype]), b.to(TYPES[in_dtype])


def _check(out, a, b, scale, out_dtype):
    """One rounding to the output type, and 2^-24 (K + 8) of a logit's magnitudes."""
    k = a.shape[-1]
    y = torch.matmul(a.double(), b.double()) * scale
    want = torch.softmax(y, dim=-1)
    mag = torch.matmul(a.abs().double(), b.abs().double()).amax(-1, keepdim=True) * abs(scale)
    bound = want * (ROUNDING[out_dtype] + 2 * mag * (k + 8) * 2.0 ** -24 + 8 * 2.0 ** -22) + 2.0 ** -24
    assert bool(((out.double() - want).abs() <= bound).all())


@needs_gpu
@pytest.mark.parametrize("in_dtype,out_dtype,m,n,grid", FORMS)
def test_waits_that_run_out_are_reported(native_lib, in_dtype, out_dtype, m, n, grid):
    from welder_typical_chain_amd import _lib
    from welder_typical_chain_amd.chain import (check_status, matmul_softmax, new_workspace, read_diagnostics,
                                                set_exchange_wait_limit, workspace_size)
    print(f"\n[gpu-case] exchange wait limit of 2 ticks, {in_dtype}->{out_dtype} {m}x{n}", flush=True)
    k = 4096 if in_dtype != "f32" else 2048  # a long K loop spreads the tiles' publications
    assert _lib.plan(1, m, n, k, CODES[in_dtype], CODES[out_dtype], _lib.PATH_EXCHANGE)["grid"] == grid
    a, b = _operands(in_dtype, m, n, k, 3)
    scale = 1.0 / math.sqrt(k)
    ws = new_workspace(workspace_size(1, m, n, k, CODES[in_dtype], CODES[out_dtype], "exchange"))
    out = torch.empty((1, m, n), dtype=TYPES[out_dtype], device="cuda")

    def call(**kw):
        return matmul_softmax(a, b, out=out, logit_scale=scale, path="exchange", workspace=ws, **kw)
    reported = False
    try:
        set_exchange_wait_limit(2)
        for _ in range(8):
            call()
            try:
                check_status()
            except _lib.WtcError as e:
                assert e.code == _lib.WTC_ERR_TIMEOUT, e
                reported = True
                break
    finally:
        set_exchange_wait_limit(0)
    flags, _, timeouts = read_diagnostics(ws)
    assert reported and flags & 1 and timeouts > 0
    for _ in range(2):
        out.fill_(7.0)
        call(check=True)
        _check(out, a, b, scale, out_dtype)
    assert read_diagnostics(ws)[0] == 0


@needs_gpu
@pytest.mark.parametrize("in_dtype,out_dtype,m,n,grid", FORMS)
def test_replays_match_eager_calls(native_lib, in_dtype, out_dtype, m, n, grid):
    from welder_typical_chain_amd.chain import matmul_softmax, new_workspace, workspace_size
    print(f"\n[gpu-case] graph of the exchange path, {in_dtype}->{out_dtype} {m}x{n}", flush=True)
    k = 256
    a, b = _operands(in_dtype, m, n, k, 5)
    ws = new_workspace(workspace_size(1, m, n, k, CODES[in_dtype], CODES[out_dtype], "exchange"))
    out = torch.empty((1, m, n), dtype=TYPES[out_dtype], device="cuda")
    eager = torch.empty_like(out)

    def call(dst):
        matmul_softmax(a, b, out=dst, logit_scale=1.0 / 16, path="exchange", workspace=ws)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        call(out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        call(out)
        call(out)
    for rep in range(4):
        new_a, new_b = _operands(in_dtype, m, n, k, 50 + rep)
        a.copy_(new_a)
        b.copy_(new_b)
        call(eager)
        torch.cuda.synchronize()
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager), f"replay {rep}"
        _check(out, a, b, 1.0 / 16, out_dtype)


@needs_gpu
def test_largest_exchange_fits_a_small_calls_default_workspace(native_lib):
    """f32 outputs on 256 tiles of 256 rows take every slot; the default workspace
    that a small call makes holds them, so that the call runs under capture."""
    from welder_typical_chain_amd.chain import matmul_softmax, release_stream
    print("\n[gpu-case] largest exchange call captured after a small one", flush=True)
    a, b = _operands("f16", 4096, 2048, 64, 9)
    out = torch.empty((1, 4096, 2048), device="cuda")
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        matmul_softmax(a[:, :64].contiguous(), b, path="exchange")
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        matmul_softmax(a, b, out=out, logit_scale=0.125, path="exchange")
    for _ in range(2):
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        _check(out, a, b, 0.125, "f32")
    release_stream(s)


@needs_gpu
@pytest.mark.parametrize("out_dtype", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("batch,m,n,k", [(1, 2049, 2048, 64), (1, 1500, 3976, 320), (8, 1000, 1024, 144),
                                         (1, 3840, 2048, 1040), (1, 4096, 2048, 0)])
def test_fp8_as_the_split_path(native_lib, batch, m, n, k, out_dtype):
    """256-row tiles of both paths run the same products; the outputs differ by
    the roundings to the output type (the split path's two) and the softmax's
    own f32 arithmetic."""
    from welder_typical_chain_amd.chain import matmul_softmax
    print(f"\n[gpu-case] tall exchange fp8->{out_dtype} {batch}x{m}x{n}x{k}", flush=True)
    a, b = _operands("fp8", m, n, k, m + k, batch)
    for scale in (1.0 / math.sqrt(max(k, 1)), -0.3):
        got, split = (torch.full((batch, m, n), 7.0, dtype=TYPES[out_dtype], device="cuda") for _ in range(2))
        matmul_softmax(a, b, out=got, logit_scale=scale, path="exchange", tiles=[128, 128, 128, 2, 32], check=True)
        matmul_softmax(a, b, out=split, logit_scale=scale, path="split", tiles=[256, 128, 128, 2, 32])
        x, y = got.double(), split.double()
        least = {"f16": 2.0 ** -23, "bf16": 2.0 ** -30, "f32": 1e-37}[out_dtype]
        bound = y * (3 * ROUNDING[out_dtype] + 2.0 ** -18) + least
        assert bool(((x - y).abs() <= bound).all()), float(((x - y).abs() / bound).max())
