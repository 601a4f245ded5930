"""The context's workspaces are shared by every stream the context is given:
work that takes one waits for the stream that used one last, whichever
streams the context had in between."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

T, N, K = 256, 512, 2048


def dev(torch, a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def matrix(lm, ctx, orc, fmt, rng):
    if fmt == "Q4_K":
        from llm_mojo_amd import synth

        return lm.HipGGUFMatrix.from_blocks(ctx, orc.GGML[fmt], synth.gguf_blocks(orc.GGML[fmt], N, K, seed=3), N, K)
    return lm.HipQuantMatrix.from_f32(ctx, rng.normal(0, 0.05, (K, N)).astype(np.float32), *fmt)


@pytest.mark.parametrize("between", ["none", "idle", "own", "captured", "back"])
@pytest.mark.parametrize("fmt", ["Q4_K", (8, 0, False, True)], ids=str)
def test_workspace_order_over_streams(gpu, orc, fmt, between):
    """Stream a: a long wait, then a prompt that uses the workspace.  The
    context goes to c (directly, by an idle stream, by its own stream, by a
    stream that is being captured, or by way of a again) and another prompt:
    it may not run ahead of the one on a, and both give their own results."""
    torch, lm, ctx = gpu
    rng = np.random.default_rng(4)
    g = matrix(lm, ctx, orc, fmt, rng)
    xs = [dev(torch, rng.normal(0, 1, (T, K)).astype(np.float32)) for _ in range(2)]
    ref = [torch.zeros((T, N), device="cuda") for _ in range(2)]
    out = [torch.zeros((T, N), device="cuda") for _ in range(2)]
    for x, r in zip(xs, ref):
        lm.linear(ctx, r, x, g)
    far = torch.zeros(1 << 26, device="cuda")
    buf = torch.zeros(16, device="cuda")
    torch.cuda.synchronize()
    a, b, c = (torch.cuda.Stream() for _ in range(3))
    print("workspace order", fmt, between, flush=True)
    graph = None
    try:
        if between == "captured":
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.stream(b):
                graph.capture_begin(capture_error_mode="thread_local")
                buf.add_(1.0)
        ctx.set_stream(a)
        with torch.cuda.stream(a):
            for _ in range(500):
                far.add_(1.0)
        lm.linear(ctx, out[0], xs[0], g)
        ea, ec = torch.cuda.Event(), torch.cuda.Event()
        ea.record(a)
        if between == "idle":
            ctx.set_stream(b)
        elif between == "own":
            ctx.set_stream(None)
        elif between == "captured":
            ctx.set_stream(b)
        elif between == "back":
            ctx.set_stream(b)
            ctx.set_stream(a)
        ctx.set_stream(c)
        if graph is not None:
            with torch.cuda.stream(b):
                graph.capture_end()
        lm.linear(ctx, out[1], xs[1], g)
        ec.record(c)
        waited = 0
        while not ea.query():
            early = ec.query()
            if early and not ea.query():
                raise AssertionError("the second prompt ran ahead of the first")
            waited += 1
            time.sleep(0.001)
        assert waited > 1, "the first stream was done too soon to tell"
    finally:
        ctx.set_stream(None)
        torch.cuda.synchronize()
    for o, r in zip(out, ref):
        assert torch.equal(o, r)
    g.free()
