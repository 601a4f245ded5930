"""The config-4 decoder (llm_mojo_amd/llama.py) on the GPU against its NumPy
statement (tests/llama_ref.py).  The reference has no such model, so these
pin our own definition (model-level parity unpinned); the GGUF, cache and
int16-head parts come from the oracle."""
import numpy as np
import pytest

from tests.llama_ref import NumpyLlama

pytestmark = pytest.mark.gpu

SMALL = dict(n_layer=2, dim=256, n_head=4, n_kv=2, head_dim=64, ffn=512, vocab=1000, max_t=96, batch=2,
             layer_type=12, head_type=14, embd_type=12, eps=1e-5, theta=10000.0)


def rel(a, b):
    return float(np.max(np.abs(a - b)) / np.max(np.abs(b)))


def test_llama_forward_matches_numpy(gpu):
    """Prefill of 20 tokens, then 3 more on the same cache: last-token
    logits within 1e-3 of max |logit|."""
    torch, lm, ctx = gpu
    from llm_mojo_amd import synth

    tensors = synth.llama_tensors(SMALL, 5)
    toks = synth.llama_prompts(5, 1, 23, SMALL["vocab"])[0]
    print("llama forward", flush=True)
    m = lm.Llama(ctx, SMALL, tensors)
    ref = NumpyLlama(SMALL, tensors)
    got = m.forward(0, toks[:20], 0)
    want = ref.forward(0, toks[:20], 0)
    assert rel(got, want) < 1e-3, rel(got, want)
    got = m.forward(0, toks[20:], 20)
    want = ref.forward(0, toks[20:], 20)
    assert rel(got, want) < 1e-3, rel(got, want)
    m.free()


@pytest.mark.parametrize("head_type,B", [(14, 2), (14, 1), (8, 1), (12, 2), (12, 1)])
def test_llama_generate_matches_numpy_greedy(gpu, head_type, B):
    """B sequences, 12-token prompts, 6 greedy tokens each (5 decode steps
    through the captured graph) against NumPy greedy decoding; a step whose
    NumPy top-2 margin is under 1e-3 of max |logit| ends the comparison of
    that sequence.  Q6_K / Q8_0 heads take the int16 head with argmax
    partials and the pick-and-embed kernel, Q4_K the float head and the full
    argmax; batch 1 stages the attention splits in the Wo GEMV, batch 2 runs
    the combine kernel."""
    torch, lm, ctx = gpu
    from llm_mojo_amd import synth

    cfg = dict(SMALL, head_type=head_type)
    tensors = synth.llama_tensors(cfg, 6)
    prompts = synth.llama_prompts(6, B, 12, cfg["vocab"])
    print("llama generate", head_type, B, flush=True)
    m = lm.Llama(ctx, cfg, tensors)
    toks, pre_ms, dec_ms = m.generate(prompts, 6)
    assert toks.shape == (6, B)
    ref = NumpyLlama(cfg, tensors, n_seq=B)
    for b in range(B):
        logits = ref.forward(b, prompts[b], 0)
        for i in range(6):
            top = np.sort(logits)[-2:]
            want = int(np.argmax(logits))
            if top[1] - top[0] < 1e-3 * np.max(np.abs(logits)):
                break
            assert toks[i, b] == want, (b, i, toks[:, b], want)
            logits = ref.forward(b, [want], 12 + i)
    m.free()


@pytest.mark.parametrize("B", [1, 2])
def test_llama_grouped_query_attention_matches_numpy(gpu, B):
    """Eight query heads a key / value head (the TinyLlama grouping): batch 1
    takes the per-head split kernel, batch 2 the kernel that serves the 8
    heads of a group from one read of the cache.  270-token prompts (two
    256-position splits, the new position in the second), 6 greedy tokens,
    against NumPy greedy decoding (the margin rule); the same prompt twice in
    the batch gives the same tokens in both rows."""
    torch, lm, ctx = gpu
    from llm_mojo_amd import synth

    cfg = dict(SMALL, dim=512, n_head=8, n_kv=1, max_t=300)
    tensors = synth.llama_tensors(cfg, 12)
    prompts = synth.llama_prompts(12, 1, 270, cfg["vocab"])
    prompts = np.repeat(prompts, B, axis=0)
    print("llama grouped attention", B, flush=True)
    m = lm.Llama(ctx, cfg, tensors)
    toks, _, _ = m.generate(prompts, 6)
    m.free()
    for b in range(1, B):
        assert np.array_equal(toks[:, b], toks[:, 0])
    n = greedy_vs_numpy(toks[:, 0], NumpyLlama(cfg, tensors), 0, prompts[0], 0)
    assert n >= 2, n


def test_llama_batch_rows_are_independent(gpu):
    """The same prompt in both sequences of a batch gives the same tokens,
    equal to a one-sequence run; a second call (graph replayed) repeats them."""
    torch, lm, ctx = gpu
    from llm_mojo_amd import synth

    tensors = synth.llama_tensors(SMALL, 7)
    p = synth.llama_prompts(7, 1, 10, SMALL["vocab"])
    print("llama batch", flush=True)
    m = lm.Llama(ctx, SMALL, tensors)
    two, _, _ = m.generate(np.concatenate([p, p]), 8)
    one, _, _ = m.generate(p, 8)
    again, _, _ = m.generate(p, 8)
    assert np.array_equal(two[:, 0], two[:, 1])
    assert np.array_equal(two[:, 0], one[:, 0])
    assert np.array_equal(one, again)
    m.free()


def test_llama_rejects_bad_shapes(gpu):
    torch, lm, ctx = gpu
    from llm_mojo_amd import synth

    bad = dict(SMALL, n_kv=3)
    with pytest.raises(lm.LlmqError, match="unsupported shape"):
        lm.Llama(ctx, bad, synth.llama_tensors(SMALL, 1))
    m = lm.Llama(ctx, SMALL, synth.llama_tensors(SMALL, 1))
    with pytest.raises(lm.LlmqError, match="capacity"):
        m.generate(np.zeros((3, 4), np.int64), 2)
    with pytest.raises(lm.LlmqError, match="beyond"):
        m.forward(0, np.zeros(4, np.int64), SMALL["max_t"] - 2)
    m.free()


def test_llama_long_context_decode(gpu):
    """Decode attention past 1024 positions (three positions a thread of the
    512-thread workgroup): a 1026-token prompt, then 3 greedy tokens, against
    NumPy greedy decoding (the same margin rule)."""
    torch, lm, ctx = gpu
    from llm_mojo_amd import synth

    cfg = dict(SMALL, max_t=1100, batch=1)
    tensors = synth.llama_tensors(cfg, 8)
    prompt = synth.llama_prompts(8, 1, 1026, cfg["vocab"])
    print("llama long context", flush=True)
    m = lm.Llama(ctx, cfg, tensors)
    toks, _, _ = m.generate(prompt, 4)
    ref = NumpyLlama(cfg, tensors)
    logits = ref.forward(0, prompt[0], 0)
    for i in range(4):
        top = np.sort(logits)[-2:]
        want = int(np.argmax(logits))
        if top[1] - top[0] < 1e-3 * np.max(np.abs(logits)):
            break
        assert toks[i, 0] == want, (i, toks[:, 0], want)
        logits = ref.forward(0, [want], 1026 + i)
    m.free()


def greedy_vs_numpy(toks, ref, seq, prompt, pos0, logits=None):
    """Compare greedy tokens with NumPy greedy decoding from `prompt` (whose
    logits, if given, ref has already computed); a step whose NumPy top-2
    margin is under 1e-3 of max |logit| ends the comparison.  Returns the
    number of tokens compared."""
    if logits is None:
        logits = ref.forward(seq, prompt, pos0)
    for i in range(len(toks)):
        top = np.sort(logits)[-2:]
        want = int(np.argmax(logits))
        if top[1] - top[0] < 1e-3 * np.max(np.abs(logits)):
            return i
        assert toks[i] == want, (i, list(toks), want)
        logits = ref.forward(seq, [want], pos0 + len(prompt) + i)
    return len(toks)


PROMPT_1024 = 1024  # a 1024-token prompt, then greedy tokens
# The full-shape tests below use zero-mean Q4_K weights (synth centered=True):
# with uniform codes and random mins every weight row shares a positive
# offset, the residual stream turns input-independent after a few layers and
# every prompt yields the same tokens, which would let a batch kernel that
# mixed up its sequences pass.


def top1_ok(got, want):
    """Same top-1, unless the NumPy top-2 margin is within the logit bar
    (then either pick is within tolerance)."""
    top = np.sort(want)[-2:]
    if top[1] - top[0] < 2e-3 * np.max(np.abs(want)):
        return True
    return int(np.argmax(got)) == int(np.argmax(want))


@pytest.mark.timeout(300)
def test_llama_full_width_prompt_1024(gpu):
    """Two layers at the TinyLlama width (d 2048, 32 query / 4 key-value
    heads, FFN 5632, Q4_K) under its 32000 x 2048 Q6_K int16 head, at config
    4's own context: a 1024-token prompt in one call (the LDS-staged Q4_K
    matmul for 64+ tokens at the 2560 / 2048 / 11264 / 5632-input widths, the
    grouped prompt attention over 1024 positions), then 8 decode positions
    on the same cache (attention over 4-5 splits of 256 positions): logits
    within 1e-3 of max |logit| and the same top-1 at each of the 9."""
    torch, lm, ctx = gpu
    from llm_mojo_amd import synth
    from llm_mojo_amd.llama import TINYLLAMA

    cfg = dict(TINYLLAMA, n_layer=2, max_t=1152)
    tensors = synth.llama_tensors(cfg, 9, centered=True)
    toks = synth.llama_prompts(9, 1, PROMPT_1024 + 8, cfg["vocab"])[0]
    print("llama full width, 1024-token prompt: load", flush=True)
    m = lm.Llama(ctx, cfg, tensors)
    ref = NumpyLlama(cfg, tensors)
    spans = [(0, PROMPT_1024)] + [(PROMPT_1024 + i, PROMPT_1024 + i + 1) for i in range(8)]
    errs = []
    for lo, hi in spans:
        got = m.forward(0, toks[lo:hi], lo)
        want = ref.forward(0, toks[lo:hi], lo)
        errs.append(rel(got, want))
        print(f"llama full width: tokens {lo}..{hi} rel err {errs[-1]:.2e}", flush=True)
        assert errs[-1] < 1e-3, (lo, errs[-1])
        assert top1_ok(got, want), (lo, int(np.argmax(got)), int(np.argmax(want)))
    m.free()


@pytest.mark.timeout(600)
def test_llama_full_depth_prompt_1024_greedy(gpu):
    """All 22 layers of the TinyLlama shape at config 4's context: the
    1024-token prompt's logits within 1e-3 of NumPy's, then 16 greedy tokens
    from the device loop against NumPy greedy decoding (the margin rule
    above), at least 8 of them compared."""
    torch, lm, ctx = gpu
    from llm_mojo_amd import synth
    from llm_mojo_amd.llama import TINYLLAMA

    cfg = dict(TINYLLAMA, max_t=1152)
    tensors = synth.llama_tensors(cfg, 11, centered=True)
    prompt = synth.llama_prompts(11, 1, PROMPT_1024, cfg["vocab"])
    print("llama full depth: load", flush=True)
    m = lm.Llama(ctx, cfg, tensors)
    print("llama full depth: prompt", flush=True)
    got = m.forward(0, prompt[0], 0)
    toks, _, _ = m.generate(prompt, 16)
    m.free()
    print("llama full depth: numpy", flush=True)
    ref = NumpyLlama(cfg, tensors)
    want = ref.forward(0, prompt[0], 0)
    print(f"llama full depth: prompt logits rel err {rel(got, want):.2e}", flush=True)
    assert rel(got, want) < 1e-3 and top1_ok(got, want)
    n = greedy_vs_numpy(toks[:, 0], ref, 0, prompt[0], 0, logits=want)
    print("llama full depth: tokens compared", n, flush=True)
    assert n >= 8


@pytest.mark.timeout(300)
def test_llama_batch16_full_context_equals_batch1(gpu):
    """Batch 16 at config 4's workload: 16 different 1024-token prompts, 128
    greedy tokens each through the captured batch-16 step (the batched
    Q4_K matmuls and grouped attention on the fp16 matrix cores, up to 1152
    positions); each sequence's tokens equal its own batch-1 run (the "many
    == one" pattern of tests/gguf_int_head.mojo:49-54)."""
    torch, lm, ctx = gpu
    from llm_mojo_amd import synth
    from llm_mojo_amd.llama import TINYLLAMA

    cfg = dict(TINYLLAMA, batch=16, max_t=1152)
    tensors = synth.llama_tensors(cfg, 10, centered=True)
    prompts = synth.llama_prompts(10, 16, PROMPT_1024, cfg["vocab"])
    print("llama batch 16, 1024-token prompts: load", flush=True)
    m = lm.Llama(ctx, cfg, tensors)
    many, _, _ = m.generate(prompts, 128)
    assert many.shape == (128, 16)
    for b in range(16):
        one, _, _ = m.generate(prompts[b:b + 1], 128)
        assert np.array_equal(one[:, 0], many[:, b]), (b, one[:, 0].tolist(), many[:, b].tolist())
        print(f"llama batch 16: sequence {b} equals its batch-1 run", flush=True)
    distinct = len({tuple(many[:, b]) for b in range(16)})
    print(f"llama batch 16: {distinct} distinct token sequences", flush=True)
    assert distinct >= 12  # (zero-mean weights: each prompt leads its own way)
    m.free()


@pytest.mark.parametrize("B", [2, 3, 16, 20])
def test_llama_batch_fused_records_match_numpy(gpu, monkeypatch, B):
    """The batch-decode chain whose Q4_K matmul epilogues write the next
    matmul's input record (h16s: a scale per 16 inputs; the RMSNorm as a
    factor on the reading matmul's outputs from the record's sums of
    squares, SwiGLU in the gate / up epilogue): two layers at the TinyLlama
    width, B sequences with their own 40-token prompts (B = 2, 3: a padded
    token tile; B = 20: two token tiles), 10 greedy tokens each against NumPy greedy decoding (the
    margin rule), and the tokens of the chain with the record kernels
    (LLMQ_FUSE_REC=0) up to the first NumPy near-tie."""
    torch, lm, ctx = gpu
    from llm_mojo_amd import synth
    from llm_mojo_amd.llama import TINYLLAMA

    cfg = dict(TINYLLAMA, n_layer=2, batch=B, max_t=64)
    tensors = synth.llama_tensors(cfg, 21, centered=True)
    prompts = synth.llama_prompts(21, B, 40, cfg["vocab"])
    print("llama fused batch records", B, flush=True)
    m = lm.Llama(ctx, cfg, tensors)
    fused, _, _ = m.generate(prompts, 10)
    m.free()
    monkeypatch.setenv("LLMQ_FUSE_REC", "0")
    m = lm.Llama(ctx, cfg, tensors)
    plain, _, _ = m.generate(prompts, 10)
    m.free()
    ref = NumpyLlama(cfg, tensors, n_seq=B)
    compared = []
    for b in range(B):
        n = greedy_vs_numpy(fused[:, b], ref, b, prompts[b], 0)
        assert np.array_equal(fused[:n, b], plain[:n, b]), (b, fused[:, b], plain[:, b])
        compared.append(n)
    print("llama fused batch records: tokens compared", compared, flush=True)
    assert sum(compared) >= 6 * B, compared


@pytest.mark.parametrize("group", [2, 8])
def test_llama_one_token_forwards_match_numpy(gpu, group):
    """forward of single tokens (the decode step's split attention) on the
    second of two sequences, across a split's edge (256 positions) and from
    an empty cache, against NumPy; the first sequence's cache stays as it
    was."""
    torch, lm, ctx = gpu
    from llm_mojo_amd import synth

    cfg = dict(SMALL, max_t=300, n_head=4 if group == 2 else 8, n_kv=2 if group == 2 else 1,
               dim=256 if group == 2 else 512)
    tensors = synth.llama_tensors(cfg, 9, centered=True)
    toks = synth.llama_prompts(9, 2, 262, cfg["vocab"])
    m = lm.Llama(ctx, cfg, tensors)
    ref = NumpyLlama(cfg, tensors, n_seq=2)
    print("llama one-token forwards", group, flush=True)
    first = m.forward(0, toks[0][:40], 0)
    for i in range(3):  # from an empty cache
        assert rel(m.forward(1, toks[1][i:i + 1], i), ref.forward(1, toks[1][i:i + 1], i)) < 1e-3, i
    m.forward(1, toks[1][3:254], 3)
    ref.forward(1, toks[1][3:254], 3)
    for i in range(254, 262):
        assert rel(m.forward(1, toks[1][i:i + 1], i), ref.forward(1, toks[1][i:i + 1], i)) < 1e-3, i
    assert np.array_equal(m.forward(0, toks[0][38:40], 38), m.forward(0, toks[0][38:40], 38))
    ref.forward(0, toks[0][:40], 0)
    assert rel(first, ref.forward(0, toks[0][38:40], 38)) < 1e-3
    assert rel(m.forward(0, toks[0][40:41], 40), ref.forward(0, toks[0][40:41], 40)) < 1e-3
    m.free()
