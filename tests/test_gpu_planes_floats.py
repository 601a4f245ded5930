"""Several tokens of float activations (gemm_planes.hip over x itself): what
the float32 inputs may hold, and that a call needs no memory of the library's.

Every input is held to its last bit in three bf16 planes, whatever its
neighbours are, so the bars are those of float32 sums: at most K / 16 + 24
roundings of 2^-24 of the sum of the absolute products.
"""
import numpy as np
import pytest

from tests.test_gpu_planes import GGUF, QM, dev, matrix

pytestmark = pytest.mark.gpu

FLOATS = [f for f in GGUF if f != "Q4_K"] + QM  # (Q4_K's activations go through its fp16 record)
SOME = ["Q8_0", "Q4_0", "Q4_1", "Q5_K", "Q6_K", (4, 32), (4, 128), (8, 0)]


def run(torch, lm, ctx, g, x, n, **opt):
    out = torch.full((x.shape[0], n), float("nan"), device="cuda")
    lm.linear(ctx, out, dev(torch, x), g, **opt)
    torch.cuda.synchronize()
    return out.cpu().numpy()


def bar(x, w):
    return (x.shape[1] / 16 + 24) * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(w).T)


@pytest.mark.parametrize("tile", ["0", "1", "2", "4"])
@pytest.mark.parametrize("fmt", ["Q8_0", "Q4_0", "Q6_K", (4, 32), (4, 128), (8, 64), (8, 0)], ids=str)
def test_zero_weight_under_a_large_input(gpu, orc, fmt, tile, monkeypatch):
    """One input 2^20 to 2^60 times its neighbours, in rows whose weight there
    is 0: the neighbours' sum is the whole result, and exact to float32 sums."""
    torch, lm, ctx = gpu
    monkeypatch.setenv("LLMQ_PLANES_TILE", tile)
    rng = np.random.default_rng(11)
    t, n, k = 66, 2000, 512
    g, w = matrix(lm, ctx, orc, fmt, n, k, rng)
    at = 37
    rows = np.flatnonzero(w[:, at] == 0)
    assert len(rows) >= 3
    x = rng.normal(0, 1, (t, k)).astype(np.float32)
    x[:, at] = (2.0 ** np.linspace(20, 60, t)).astype(np.float32)
    print("zero weight", fmt, tile, len(rows), flush=True)
    got = run(torch, lm, ctx, g, x, n)[:, rows]
    live = np.delete(x, at, 1)
    wl = np.delete(w[rows], at, 1)
    err = np.abs(got - live.astype(np.float64) @ wl.T)
    assert np.all(err <= bar(live, wl)), np.max(err / bar(live, wl))
    g.free()


@pytest.mark.parametrize("fmt", FLOATS, ids=str)
def test_error_no_larger_than_fp32_matrix_cores(gpu, orc, fmt, monkeypatch):
    """Against float64, over rows of a residual stream (a few channels much
    larger) and rows after a GELU (values down to 1e-9 of the largest): no
    further off than the fp32 matrix-core kernel."""
    torch, lm, ctx = gpu
    rng = np.random.default_rng(12)
    t, n, k = 96, 320, 2048
    g, w = matrix(lm, ctx, orc, fmt, n, k, rng)
    x = rng.normal(0, 1, (t, k))
    x[:, rng.integers(0, k, k // 256)] *= 8.0
    h = rng.normal(0, 2, (t, k))
    h = 0.5 * h * (1 + np.tanh(np.sqrt(2 / np.pi) * (h + 0.044715 * h ** 3)))
    for name, v in (("stream", x), ("gelu", h)):
        v = v.astype(np.float32)
        want = v.astype(np.float64) @ w.T
        err = []
        for h16, tile in (("0", "0"), ("1", "0"), ("1", "1"), ("1", "2"), ("1", "3"), ("1", "4")):
            monkeypatch.setenv("LLMQ_GEMM_H16", h16)
            monkeypatch.setenv("LLMQ_PLANES_TILE", tile)
            got = run(torch, lm, ctx, g, v, n)
            err.append(np.linalg.norm(got - want) / np.linalg.norm(want))
            drift = float(np.mean(got - want) / np.mean(np.abs(want)))
            # 30720 outputs about 1e-7 off: a mean of 1e-9 by chance; products cut downwards leave 5e-8 and more
            assert h16 == "0" or abs(drift) < 2.5e-8, (tile, drift)
        print("error", fmt, name, " ".join(f"{e:.2e}" for e in err), flush=True)
        assert max(err[1:]) <= err[0]
    g.free()


def test_few_tokens_keep_the_exacter_kernel(gpu, orc):
    """A call near the line to the fp32 matrix cores, which are 3.5e-7 off
    there: it stays with the planes (1e-7)."""
    torch, lm, ctx = gpu
    rng = np.random.default_rng(16)
    t, n, k = 10, 7224, 1280
    g, w = matrix(lm, ctx, orc, "Q4_1", n, k, rng)
    x = rng.normal(0, 1, (t, k)).astype(np.float32)
    print("few tokens", flush=True)
    got, want = run(torch, lm, ctx, g, x, n), x.astype(np.float64) @ w.T
    assert np.linalg.norm(got - want) <= 1.8e-7 * np.linalg.norm(want)
    g.free()


@pytest.mark.parametrize("tile", ["0", "1", "2", "4"])
@pytest.mark.parametrize("fmt", SOME, ids=str)
def test_infinite_nan_and_extreme_inputs(gpu, orc, fmt, tile, monkeypatch):
    """An infinite or NaN input changes its own token's outputs only, and
    those to what the fp32 kernel gives; inputs near float32's ends, and
    chunks of nothing but tiny ones, keep their bits."""
    torch, lm, ctx = gpu
    rng = np.random.default_rng(13)
    t, n, k = 66, 130, 512
    g, w = matrix(lm, ctx, orc, fmt, n, k, rng)
    x = rng.normal(0, 1, (t, k)).astype(np.float32)
    x[3, 7], x[20, 300], x[21, 5], x[65, 511] = np.inf, -np.inf, np.nan, np.inf
    x[40] *= 1e-33
    x[41, 64:96] *= 1e-34
    x[42, 100] = 3e36
    x[43] *= np.float32(1e30)
    x[44, 256:] = 0
    x[45, 0], x[45, 40] = np.inf, 1e35
    got = []
    for h16 in ("1", "0"):
        monkeypatch.setenv("LLMQ_GEMM_H16", h16)
        monkeypatch.setenv("LLMQ_PLANES_TILE", tile)
        print("extremes", fmt, tile, h16, flush=True)
        got.append(run(torch, lm, ctx, g, x, n))
    live = np.isfinite(x).all(1)
    assert np.isfinite(got[0][live]).all()
    a, b = got[0][~live], got[1][~live]
    assert np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(np.isposinf(a), np.isposinf(b))
    assert np.array_equal(np.isneginf(a), np.isneginf(b))
    size = np.abs(w)
    if fmt in ("Q4_1", "Q5_K"):  # (code and offset are separate products: each as large as the row's largest weight)
        size = np.broadcast_to(2 * size.max(1, keepdims=True), w.shape)
    err = np.abs(got[0][live] - x[live].astype(np.float64) @ w.T)
    assert np.all(err <= bar(x[live], size) + 2.0 ** -149), np.max(err / (bar(x[live], size) + 2.0 ** -149))
    g.free()


@pytest.mark.parametrize("fmt", FLOATS, ids=str)
def test_noalloc_uses_no_scratch(gpu, orc, fmt):
    """llmq_linear_noalloc of these types gives llmq_linear's bits and leaves
    the per-GPU scratch alone: two contexts' calls that overlap on two
    streams, one of them of a type that does use it, do not meet."""
    torch, lm, ctx = gpu
    from llm_mojo_amd._lib import check as ok, lib

    rng = np.random.default_rng(14)
    t, n, k = 300, 256, 1024
    g, w = matrix(lm, ctx, orc, fmt, n, k, rng)
    q, _ = matrix(lm, ctx, orc, "Q4_K", n, k, rng)
    x = dev(torch, rng.normal(0, 1, (t, k)).astype(np.float32))
    ref, rq = torch.zeros((t, n), device="cuda"), torch.zeros((t, n), device="cuda")
    lm.linear(ctx, ref, x, g)
    lm.linear(ctx, rq, x, q)
    torch.cuda.synchronize()
    other = lm.Context(0)
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    outs = [(torch.zeros((t, n), device="cuda"), torch.zeros((t, n), device="cuda")) for _ in range(8)]
    torch.cuda.synchronize()
    print("noalloc", fmt, flush=True)
    try:
        ctx.set_stream(a)
        other.set_stream(b)
        for o, oq in outs:
            ok(lib().llmq_linear_noalloc(ctx.h, o.data_ptr(), x.data_ptr(), g.h, None, t, k, n, 0))
            ok(lib().llmq_linear_noalloc(other.h, oq.data_ptr(), x.data_ptr(), q.h, None, t, k, n, 0))
    finally:
        ctx.set_stream(None)
        other.set_stream(None)
    torch.cuda.synchronize()
    for o, oq in outs:
        assert torch.equal(o, ref) and torch.equal(oq, rq)
    other.close()
    g.free()
    q.free()


@pytest.mark.parametrize("fmt", ["Q8_0", "Q5_K", (8, 0)], ids=str)
def test_captured_calls_give_the_same_bits(gpu, orc, fmt):
    torch, lm, ctx = gpu
    rng = np.random.default_rng(15)
    t, n, k = 300, 256, 1024
    g, w = matrix(lm, ctx, orc, fmt, n, k, rng)
    x = dev(torch, rng.normal(0, 1, (t, k)).astype(np.float32))
    ref, out = torch.zeros((t, n), device="cuda"), torch.zeros((t, n), device="cuda")
    lm.linear(ctx, ref, x, g)
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    print("captured", fmt, flush=True)
    with torch.cuda.stream(stream):
        ctx.set_stream(stream)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream, capture_error_mode="thread_local"):
            lm.linear(ctx, out, x, g)
    try:
        for _ in range(3):
            out.zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, ref)
    finally:
        ctx.set_stream(None)
    g.free()
