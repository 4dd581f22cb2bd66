"""GPU parity on the other benchmark configurations.

Each case runs the HIP path on the full workload of one attention layer (or one
whole model) and checks oracle slices: the float64 oracle estimator on the
device's packed planes (reference attention.py:419-461, compressors.py:186-189),
the softmax / P.V tail (families/qwen2.py:110-117, llama.py:107-122) and
value decompression (compressors.py:311-317), within rel-err 1e-3 and cosine
0.9999 per output row.

  Qwen2.5-3B attention: 16 query / 2 kv heads, causal prefill of
              2048 / 4096 / 8192 tokens, bits 2 / 3 / 4; and the 36-layer
              random-init model's bf16 forward at 2048 tokens
  Llama-3.1-8B attention: 32 / 8 heads, 4 sequences x 32768 tokens,
              bits 4: causal prefill and one decode step
  DeepSeek-LLM-7B MHA: 32 / 32 heads, bits 2, Student-t(5) keys:
              8 x 16384 (decode and causal prefill) and 1 x 131072 (decode)
"""

import copy
import math

import numpy as np
import pytest
import torch

from oracle import tq_oracle as O
from test_gpu_kernels import _np
from turboquant_pytorch import _native, compressed_attention
from turboquant_pytorch.compressors import TurboQuantCompressorMSE, TurboQuantCompressorV2

pytestmark = pytest.mark.gpu
DEV = "cuda"
REL = 1e-3


def _case(**kw):
    print("case:", kw, flush=True)


def _head_planes(kc, vc, ck, cv, row0, sk):
    """Oracle-side planes of the sk rows starting at row0 (one (batch, kv head) sequence)."""
    d = kc.head_dim
    r = slice(row0, row0 + sk)
    codes = O.unpack_bits(_np(ck["packed_key_indices"][r]), kc.mse_bits, d)
    signs = O.unpack_bits(_np(ck["packed_qjl_signs"][r]), 1, d)
    rn = _np(ck["residual_norm"].reshape(-1)[r])
    vn = _np(ck["vec_norms"].reshape(-1)[r])
    codes_v = O.unpack_bits(_np(cv["packed_indices"][r]), vc.bits, d)
    vals = O.value_decompress(codes_v, _np(cv["vec_norms"][r]), vc.Pi.cpu().numpy(), vc.centroids.cpu().numpy())
    return codes, signs, rn, vn, vals


def _check_rows(out, q, kc, vc, ck, cv, hkv, picks, causal):
    """out [B, Sq, Hq, d] against the oracle for picks = [(b, h, rows)]."""
    B, hq, Sq, d = q.shape
    Sk = ck["shape"][2]
    g = hq // hkv
    cent16 = kc.centroids.cpu().numpy().astype(np.float16)
    s_eff16 = kc._dev_tables.s_eff16.cpu().numpy()
    worst = 0.0
    cache = {}
    for b, h, rows in picks:
        kv = b * hkv + h // g
        if kv not in cache:
            cache = {kv: _head_planes(kc, vc, ck, cv, kv * Sk, Sk)}
        codes, signs, rn, vn, vals = cache[kv]
        q_rot, q_proj = O.query_prep(q[b, h, rows].float().cpu().numpy(), kc.Pi.cpu().numpy(), s_eff16)
        sc = O.scores_packed(q_rot, q_proj, codes, signs, rn, vn, cent16, O.COEFF(d))
        for t, i in enumerate(rows):
            lim = i + (Sk - Sq) if causal else Sk - 1
            ref = O.attention(sc[t:t + 1, : lim + 1], vals[: lim + 1], 1 / math.sqrt(d))[0]
            got = _np(out[b, i, h])
            err = O.rel_err(got, ref)
            worst = max(worst, err)
            assert err < REL and O.cosine(got, ref) > 0.9999, (b, h, i, err)
    print(f"worst rel-err over {sum(len(r) for _, _, r in picks)} rows: {worst:.2e}", flush=True)


def _compressors(d, bits):
    return (TurboQuantCompressorV2(d, bits, seed=42, device=DEV),
            TurboQuantCompressorMSE(d, bits, seed=10042, device=DEV))


def _randn(shape, seed, dtype=torch.bfloat16):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(*shape, device=DEV, generator=g).to(dtype)


# ---------------------------------------------------------------- Qwen2.5-3B

@pytest.mark.parametrize("bits", [2, 3, 4])
@pytest.mark.parametrize("S", [2048, 4096, 8192])
def test_qwen25_3b_layer_prefill(S, bits):
    _case(config=2, S=S, bits=bits)
    hq, hkv, d = 16, 2, 128
    q = _randn((1, hq, S, d), S + bits)
    k = _randn((1, hkv, S, d), 2 * S + bits)
    v = _randn((1, hkv, S, d), 3 * S + bits)
    kc, vc = _compressors(d, bits)
    ck, cv = kc.compress(k), vc.compress(v)
    out = compressed_attention(q, kc, vc, ck, cv, causal=True, out_dtype=torch.float32)
    torch.cuda.synchronize()
    assert torch.isfinite(out).all()
    rows = [0, 1, 63, S // 2, S - 1]
    _check_rows(out, q, kc, vc, ck, cv, hkv, [(0, h, rows) for h in (0, 7, 8, 15)], causal=True)


def test_qwen25_3b_model_forward_bf16():
    """The whole 36-layer Qwen2.5-3B-shaped random-init model, bf16, 2048 tokens, bits 3,
    apply_turboquant's defaults: finite logits; for the first and last layer, the module's
    output equals the fused kernel on its own q/k/v (recomputed from the captured inputs),
    that kernel output matches the oracle on the device's planes, and the layer agrees with
    its CPU path (the reference's PyTorch branch, f32) fed the same inputs."""
    _case(config=2, what="36-layer model, 2048 tokens")
    from transformers import Qwen2Config, Qwen2ForCausalLM
    from transformers_turboquant import apply_turboquant

    cfg = Qwen2Config(vocab_size=151936, hidden_size=2048, intermediate_size=11008, num_hidden_layers=36,
                      num_attention_heads=16, num_key_value_heads=2, max_position_embeddings=32768,
                      tie_word_embeddings=True)
    torch.manual_seed(0)
    with torch.device(DEV):
        model = Qwen2ForCausalLM(cfg)
    model = model.to(torch.bfloat16).eval()
    apply_turboquant(model, bits=3, seed=42)
    captured = {}

    def hook(i):
        def fn(mod, args, kwargs, output):
            captured[i] = (args, kwargs, output[0].detach())
        return fn

    layers = model.model.layers
    handles = [layers[i].self_attn.register_forward_hook(hook(i), with_kwargs=True) for i in (0, 35)]
    ids = torch.randint(0, cfg.vocab_size, (1, 2048), generator=torch.Generator().manual_seed(0)).to(DEV)
    with torch.no_grad():
        logits = model(input_ids=ids).logits
    torch.cuda.synchronize()
    for h in handles:
        h.remove()
    assert logits.shape == (1, 2048, cfg.vocab_size) and torch.isfinite(logits).all()

    def to_cpu(x):
        if isinstance(x, torch.Tensor):
            return x.detach().to("cpu", torch.float32)
        if isinstance(x, (tuple, list)):
            return type(x)(to_cpu(y) for y in x)
        return x

    for i in (0, 35):
        args, kwargs, gpu_out = captured[i]
        attn = layers[i].self_attn
        hs = kwargs["hidden_states"] if "hidden_states" in kwargs else args[0]
        B, T, _ = hs.shape
        with torch.no_grad():
            q = attn.q_proj(hs).view(B, T, 16, 128).transpose(1, 2)
            k = attn.k_proj(hs).view(B, T, 2, 128).transpose(1, 2)
            v = attn.v_proj(hs).view(B, T, 2, 128).transpose(1, 2)
            q, k = type(attn).apply_rotary(q, k, *kwargs["position_embeddings"])
            kc, vc = attn.key_compressor, attn.val_compressor
            ck, cv = kc.compress(k), vc.compress(v)
            out = compressed_attention(q, kc, vc, ck, cv, out_dtype=torch.float32)
            again = attn.o_proj(out.to(torch.bfloat16).reshape(B, T, -1))
        assert torch.equal(again, gpu_out), i
        _check_rows(out, q, kc, vc, ck, cv, 2, [(0, h, [0, 1, 1023, 2047]) for h in (0, 9, 15)], causal=False)
        cpu_attn = copy.deepcopy(attn).to("cpu", torch.float32)
        with torch.no_grad():
            cpu_out = cpu_attn(*to_cpu(args), **{kk: to_cpu(vv) for kk, vv in kwargs.items()})[0]
        cos = O.cosine(gpu_out.float().cpu().numpy(), cpu_out.numpy())
        print(f"layer {i}: GPU bf16 vs CPU f32 attention output cosine {cos:.6f}", flush=True)
        # bf16 projections and the packed format's f16 key centroids against f32 and the
        # unpacked format; the random-init attention is nearly uniform over 2048 keys, so
        # its output is a small mean of many values and carries those differences relatively
        assert cos > 0.99, (i, cos)


# ---------------------------------------------------------------- Llama-3.1-8B

def test_llama31_8b_layer_prefill_and_decode():
    _case(config=3, B=4, S=32768, bits=4)
    B, hq, hkv, S, d, bits = 4, 32, 8, 32768, 128, 4
    k = _randn((B, hkv, S, d), 31)
    v = _randn((B, hkv, S, d), 32)
    kc, vc = _compressors(d, bits)
    ck, cv = kc.compress(k), vc.compress(v)
    del k, v
    q = _randn((B, hq, S, d), 33)
    out = compressed_attention(q, kc, vc, ck, cv, causal=True, out_dtype=torch.float32)
    torch.cuda.synchronize()
    assert torch.isfinite(out).all()
    rows = [0, 1, 4095, 16384, S - 1]
    _check_rows(out, q, kc, vc, ck, cv, hkv, [(b, h, rows) for b in (0, 3) for h in (0, 17, 31)], causal=True)
    del out
    # one decode step: a new query row per sequence against the whole cache (split-K kernels)
    qd = q[:, :, -1:].contiguous()
    assert _native.lib().tq_attention_workspace_size(B, hq, hkv, 1, S, d, bits) > 0
    outd = compressed_attention(qd, kc, vc, ck, cv, out_dtype=torch.float32)
    torch.cuda.synchronize()
    _check_rows(outd, qd, kc, vc, ck, cv, hkv, [(b, h, [0]) for b in (0, 3) for h in range(hq)], causal=False)


# ---------------------------------------------------------------- DeepSeek-7B MHA

def _student_t(shape, seed):
    torch.manual_seed(seed)
    t = torch.distributions.StudentT(torch.tensor(5.0, device=DEV)).sample(shape)
    return t.to(torch.bfloat16)


def test_deepseek_7b_mha_8x16384():
    _case(config=4, B=8, S=16384, bits=2)
    B, h, S, d, bits = 8, 32, 16384, 128, 2
    k = _student_t((B, h, S, d), 2)
    v = _randn((B, h, S, d), 3)
    kc, vc = _compressors(d, bits)
    ck, cv = kc.compress(k), vc.compress(v)
    del k, v
    q = _randn((B, h, S, d), 4)
    qd = q[:, :, -1:].contiguous()
    assert _native.lib().tq_attention_workspace_size(B, h, h, 1, S, d, bits) > 0
    outd = compressed_attention(qd, kc, vc, ck, cv, out_dtype=torch.float32)
    torch.cuda.synchronize()
    _check_rows(outd, qd, kc, vc, ck, cv, h, [(b, hh, [0]) for b in (0, 7) for hh in (0, 5, 19, 31)],
                causal=False)
    out = compressed_attention(q, kc, vc, ck, cv, causal=True, out_dtype=torch.float32)
    torch.cuda.synchronize()
    assert torch.isfinite(out).all()
    rows = [0, 1, 8191, S - 1]
    _check_rows(out, q, kc, vc, ck, cv, h, [(b, hh, rows) for b in (0, 7) for hh in (0, 31)], causal=True)


def test_deepseek_7b_mha_131072_decode():
    _case(config=4, B=1, S=131072, bits=2)
    B, h, S, d, bits = 1, 32, 131072, 128, 2
    k = _student_t((B, h, S, d), 5)
    v = _randn((B, h, S, d), 6)
    kc, vc = _compressors(d, bits)
    ck, cv = kc.compress(k), vc.compress(v)
    del k, v
    q = _randn((B, h, 1, d), 7)
    assert _native.lib().tq_attention_workspace_size(B, h, h, 1, S, d, bits) > 0
    out = compressed_attention(q, kc, vc, ck, cv, out_dtype=torch.float32)
    scores = kc.asymmetric_attention_scores(q, ck)
    torch.cuda.synchronize()
    _check_rows(out, q, kc, vc, ck, cv, h, [(0, hh, [0]) for hh in (0, 11, 31)], causal=False)
    # materialised decode scores on the same planes
    cent16 = kc.centroids.cpu().numpy().astype(np.float16)
    for hh in (0, 31):
        codes, signs, rn, vn, _ = _head_planes(kc, vc, ck, cv, hh * S, S)
        q_rot, q_proj = O.query_prep(q[0, hh].float().cpu().numpy(), kc.Pi.cpu().numpy(),
                                     kc._dev_tables.s_eff16.cpu().numpy())
        ref = O.scores_packed(q_rot, q_proj, codes, signs, rn, vn, cent16, O.COEFF(d))
        assert O.rel_err(_np(scores[0, hh]), ref) < REL, hh
