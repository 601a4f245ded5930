"""One-token float attention at the edges of its kernel: chains of 16
positions padded with -0.0, 64-position waves (the last of which also forms
the total), 512-position passes, caches too long for the columns form, and
the fused store of the decode step, bit for bit against the oracle."""
import numpy as np
import pytest

from tests.test_gpu_exact import dev, same_bits

pytestmark = pytest.mark.gpu

POS = [0, 1, 14, 15, 16, 17, 31, 32, 47, 62, 63, 64, 65, 127, 128, 255, 256, 447, 448, 449, 510, 511, 512, 513, 600,
       1022, 1023]


@pytest.mark.parametrize("MT,poss", [(1024, POS), (70, [0, 33, 68, 69]), (2200, [100, 2199]), (3000, [2999])])
def test_one_token_attention_bit_exact(gpu, orc, MT, poss):
    torch, lm, ctx = gpu
    rng = np.random.default_rng(MT)
    NH, C = 4, 256
    qkv = rng.normal(0, 1, (MT, 3 * C)).astype(np.float32)
    qkv[:, :C] *= 3.0
    qkv[5 % MT, C:2 * C] = 0.0
    kv, okv = lm.QuantKV8(ctx, 1, MT, NH, 64), orc.QuantKV8(1, MT, NH, 64)
    kv.store(0, 0, dev(torch, qkv))
    for p in range(MT):
        okv.store(0, p, qkv[p, C:2 * C], qkv[p, 2 * C:])
    out = torch.zeros((1, C), device="cuda")
    for p in poss:
        print("one-token attention", MT, p, flush=True)
        kv.attend(out, dev(torch, qkv[p:p + 1]), 0, p)
        torch.cuda.synchronize()
        same_bits(out.cpu().numpy(), okv.attend(qkv[p:p + 1], 0, 1, p))
    kv.free()


@pytest.mark.parametrize("p0", [0, 445, 509])
def test_decode_steps_bit_exact(gpu, orc, p0):
    """GPT-2 one-token forwards (the store fused into the attention) across
    positions p0 .. p0 + 5, logits bit for bit, and the device's greedy loop
    over the same positions."""
    torch, lm, ctx = gpu
    from llm_mojo_amd import gpt2, synth

    tensors = synth.gpt2_tensors(11)
    model, ref = lm.GPT2(ctx, tensors), orc.GPT2(gpt2.params_list(tensors))
    prompt = synth.prompt_ids(12, max(p0, 1))
    print("decode steps", p0, flush=True)
    lo = ref.forward(prompt, 0)
    same_bits(model.forward(prompt, 0), lo)
    toks = []
    for i in range(6):
        toks.append(int(orc.argmax(lo)))
        lo = ref.forward([toks[-1]], len(prompt) + i)
        same_bits(model.forward([toks[-1]], len(prompt) + i), lo)
    toks.append(int(orc.argmax(lo)))
    assert list(model.generate(prompt, 7)[0]) == toks
    model.free()
