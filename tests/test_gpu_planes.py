"""The several-token matmul over activation planes (gemm_planes.hip): every
format and every tile it is built in, at the edges of the tiles (tokens and
rows that fill none, one and a part of them; one, two, three and more
superblocks, so both buffers and the last step), against the dequantized
weights in float64.

The bar is derived: each input is x to 22 bits (2^-22; Q4_K, whose record it
is, the other formats hold every bit), and the products of
a row are added in float32 in at most K / 16 + 24 roundings, each within
2^-24 of the sum of the absolute products.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GGUF = ["Q8_0", "Q4_0", "Q4_1", "Q4_K", "Q5_K", "Q6_K"]
QM = [(4, 32), (4, 64), (4, 128), (4, 256), (4, 0), (8, 32), (8, 64), (8, 128), (8, 0)]


def dev(torch, a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def matrix(lm, ctx, orc, fmt, n, k, rng):
    """(the device matrix, its weights in float64 [n, k])."""
    if isinstance(fmt, str):
        from llm_mojo_amd import synth

        t = orc.GGML[fmt]
        blocks = synth.gguf_blocks(t, n, k, seed=n + k)
        return lm.HipGGUFMatrix.from_blocks(ctx, t, blocks, n, k), orc.gguf_dequant(t, blocks, n, k).astype(np.float64)
    w = rng.normal(0, 0.05, (k, n)).astype(np.float32)
    o = orc.QuantMatrix.from_f32(w, *fmt, False, False)
    return lm.HipQuantMatrix.from_f32(ctx, w, *fmt, False, False), o.dequant().astype(np.float64)


def check(got, x, w, add=0.0):
    want = x.astype(np.float64) @ w.T + add
    size = np.abs(x).astype(np.float64) @ np.abs(w).T + np.abs(add)
    bar = (2.0 ** -22 + (x.shape[1] / 16 + 24) * 2.0 ** -24) * size
    assert np.all(np.abs(got - want) <= bar), np.max(np.abs(got - want) / bar)


@pytest.mark.parametrize("tile", range(7))
@pytest.mark.parametrize("fmt", GGUF + QM, ids=str)
def test_planes_tiles(gpu, orc, fmt, tile, monkeypatch):
    torch, lm, ctx = gpu
    monkeypatch.setenv("LLMQ_PLANES_TILE", str(tile))
    for t, n, k in ((64, 70, 256), (65, 256, 512), (129, 300, 768), (17, 1000, 1280)):
        if fmt == "Q4_K" and t < 64:
            continue  # (its own kernel)
        print("planes", fmt, tile, t, n, k, flush=True)
        rng = np.random.default_rng(t + n + k)
        g, w = matrix(lm, ctx, orc, fmt, n, k, rng)
        x = rng.normal(0, 1, (t, k)).astype(np.float32)
        out = torch.full((t, n), float("nan"), device="cuda")
        lm.linear(ctx, out, dev(torch, x), g)
        torch.cuda.synchronize()
        check(out.cpu().numpy(), x, w)
        g.free()


@pytest.mark.parametrize("fmt", ["Q8_0", "Q5_K", "Q6_K", (8, 0), (4, 32)], ids=str)
def test_planes_epilogue_and_scales(gpu, orc, fmt, monkeypatch):
    """Bias and residual; tokens of scale 0, 1e-30, 1e30, mixed 1e4 / 1e-4
    inputs, one whose sub-block sums pass float32's range, and an input that
    is not 16-byte aligned."""
    torch, lm, ctx = gpu
    rng = np.random.default_rng(5)
    t, n, k = 70, 200, 512
    g, w = matrix(lm, ctx, orc, fmt, n, k, rng)
    x = rng.normal(0, 1, (t, k)).astype(np.float32)
    x[0] = 0
    x[1] *= 1e-30
    x[2] *= 1e30
    x[3] *= np.where(np.arange(k) % 3 == 0, 1e4, 1e-4)
    if fmt not in ("Q5_K", "Q6_K"):  # (their test weights reach 10: the results would pass the range too)
        x[4] = 1.2e37 * (np.arange(k) < 64)
    b = rng.normal(0, 1, n).astype(np.float32)
    res = rng.normal(0, 1, (t, n)).astype(np.float32)
    flat = torch.empty(t * k + 1, device="cuda")
    xd = flat[1:].view(t, k)
    xd.copy_(dev(torch, x))
    out = dev(torch, res)
    monkeypatch.setenv("LLMQ_PLANES_TILE", "3")
    print("planes epilogue", fmt, flush=True)
    lm.linear(ctx, out, xd, g, dev(torch, b), resid=True)
    torch.cuda.synchronize()
    check(out.cpu().numpy(), x, w, b + res.astype(np.float64))
    g.free()


@pytest.mark.parametrize("fmt", ["Q8_0", "Q4_0", (8, 0)], ids=str)
def test_planes_infinite_inputs(gpu, orc, fmt, monkeypatch):
    """An infinite or NaN input changes its own token's outputs only, and
    those to what the fp32 kernel gives (LLMQ_GEMM_H16=0)."""
    torch, lm, ctx = gpu
    rng = np.random.default_rng(6)
    t, n, k = 66, 130, 512
    g, w = matrix(lm, ctx, orc, fmt, n, k, rng)
    x = rng.normal(0, 1, (t, k)).astype(np.float32)
    x[3, 7], x[20, 300], x[21, 5] = np.inf, -np.inf, np.nan
    got = []
    for h16 in ("1", "0"):
        monkeypatch.setenv("LLMQ_GEMM_H16", h16)
        monkeypatch.setenv("LLMQ_PLANES_TILE", "3")
        out = torch.zeros((t, n), device="cuda")
        print("planes inf", fmt, h16, flush=True)
        lm.linear(ctx, out, dev(torch, x), g)
        torch.cuda.synchronize()
        got.append(out.cpu().numpy())
    live = np.isfinite(x).all(1)
    assert np.isfinite(got[0][live]).all()
    assert np.array_equal(np.nan_to_num(got[0][~live], nan=7.0), np.nan_to_num(got[1][~live], nan=7.0))
    check(got[0][live], x[live], w)
    g.free()


def test_planes_parts_and_capture(gpu, orc):
    """llmq_linear_noalloc of a long prompt gives llmq_linear's bits; under
    graph capture the replays stay within the bar."""
    torch, lm, ctx = gpu
    from llm_mojo_amd._lib import check as ok, lib

    rng = np.random.default_rng(7)
    t, n, k = 700, 96, 4096
    g, w = matrix(lm, ctx, orc, "Q8_0", n, k, rng)
    x = rng.normal(0, 1, (t, k)).astype(np.float32)
    xd, a, b = dev(torch, x), torch.zeros((t, n), device="cuda"), torch.zeros((t, n), device="cuda")
    print("planes parts", flush=True)
    lm.linear(ctx, a, xd, g)
    ok(lib().llmq_linear_noalloc(ctx.h, b.data_ptr(), xd.data_ptr(), g.h, None, t, k, n, 0))
    torch.cuda.synchronize()
    assert torch.equal(a, b)
    check(a.cpu().numpy(), x, w)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        ctx.set_stream(stream)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream, capture_error_mode="thread_local"):
            lm.linear(ctx, b, xd, g)
    try:
        for _ in range(3):
            b.zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            check(b.cpu().numpy(), x, w)
    finally:
        ctx.set_stream(None)
    g.free()


def test_planes_two_streams(gpu, orc):
    """Calls on alternating streams of one context: each gives what it gives
    alone."""
    torch, lm, ctx = gpu
    rng = np.random.default_rng(8)
    t, n, k = 512, 512, 4096
    g, w = matrix(lm, ctx, orc, "Q8_0", n, k, rng)
    xs = [dev(torch, rng.normal(0, 1, (t, k)).astype(np.float32)) for _ in range(2)]
    outs = [[torch.zeros((t, n), device="cuda") for _ in range(6)] for _ in range(2)]
    ref = [torch.zeros((t, n), device="cuda") for _ in range(2)]
    for x, r in zip(xs, ref):
        lm.linear(ctx, r, x, g)
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]
    print("planes streams", flush=True)
    try:
        for i in range(6):
            for s in range(2):
                ctx.set_stream(streams[s])
                lm.linear(ctx, outs[s][i], xs[s], g)
    finally:
        ctx.set_stream(None)
    torch.cuda.synchronize()
    for s in range(2):
        for o in outs[s]:
            assert torch.equal(o, ref[s])
    g.free()


@pytest.mark.parametrize("tile", [1, 2, 3, 4])
@pytest.mark.parametrize("fmt", [(4, 64), (4, 128), (4, 256), (4, 0), (8, 32), (8, 64), (8, 128), (8, 512), (8, 0)], ids=str)
def test_planes_int16_activations(gpu, fmt, tile, monkeypatch):
    """The same kernel over int16 activation codes: the int8-MFMA form's bits
    (LLMQ_MFMA_F16=0) in every tile, with ragged tokens, the n % 32 rows
    left to rows_i16, bias, GELU, residual and LayerNorm, and codes and
    weights at their extremes (every partial sum then at its largest)."""
    torch, lm, ctx = gpu
    bits, group = fmt
    rng = np.random.default_rng(bits + group)
    for t, n, k, big in ((2, 64, 512, True), (17, 70, 512, False), (65, 300, 1024, False), (130, 96, 1536, True)):
        w = rng.normal(0, 0.05, (k, n)).astype(np.float32)
        x = rng.normal(0, 1, (t, k)).astype(np.float32)
        if big:  # codes near +-32767 against u - zp at its ends
            w = np.where(rng.random((k, n)) < 0.97, 0.1, -1e-4).astype(np.float32)
            x = (rng.uniform(0.999, 1.0, (t, k)) * np.where(np.arange(t)[:, None] % 2, -1, 1)).astype(np.float32)
        g = lm.HipQuantMatrix.from_f32(ctx, w, bits, group, False, True)
        b, res = dev(torch, rng.normal(0, 1, n).astype(np.float32)), rng.normal(0, 1, (t, n)).astype(np.float32)
        ln = (dev(torch, rng.uniform(0.5, 1.5, k).astype(np.float32)), dev(torch, rng.normal(0, 0.1, k).astype(np.float32)))
        got = []
        for env in ({"LLMQ_MFMA_F16": "0"}, {"LLMQ_MFMA_F16": "1", "LLMQ_PLANES_TILE": str(tile)}):
            for name, v in env.items():
                monkeypatch.setenv(name, v)
            for opt in ({"gelu": True}, {"resid": True}, {} if big else {"ln": ln}):
                print("planes a16", fmt, tile, t, n, k, env, opt.keys(), flush=True)
                out = dev(torch, res)
                lm.linear(ctx, out, dev(torch, x), g, b, **opt)
                torch.cuda.synchronize()
                got.append(out.cpu().numpy().view(np.uint32))
        for i in range(3):
            assert np.array_equal(got[i], got[3 + i]), (t, n, k, i)
        g.free()
