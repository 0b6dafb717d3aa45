"""FP8 (OCP e4m3) KV cache: quantization round trip, CPU engine path
through the reference ops, and GPU kernel numerics (marked gpu)."""
import pytest
import torch

import llmlb_amd.ops as ops
from llmlb_amd.ops import reference
from llmlb_amd.backend.engine import Engine, EngineConfig
from llmlb_amd.backend.sampler import SamplingParams
from llmlb_amd.models.llama import LlamaConfig


def test_quantize_round_trip_cpu():
    x = torch.randn(8, 4, 128) * 3
    q, scale = reference.quantize_fp8(x)
    deq = q.view(torch.float8_e4m3fn).float() * scale.unsqueeze(-1)
    rel = (deq - x).abs().max() / x.abs().max()
    assert rel < 0.07, rel.item()     # e4m3 step ~6% of amax


def test_fp8_engine_cpu():
    """Engine with fp8 KV on CPU (reference ops): prefill is exact (it
    attends dense K/V), decode reads the dequantized cache."""
    cfg = EngineConfig(model=LlamaConfig.tiny(), device="cpu",
                       dtype="float32", kv_cache_blocks=64,
                       kv_dtype="fp8_e4m3", seed=5)
    eng = Engine(cfg)
    assert eng.kv.fp8
    p = SamplingParams(temperature=0.0)
    out = eng.generate_sync([2, 7, 1, 8, 2, 8], 12, p).token_ids
    assert len(out) == 12
    ref_eng = Engine(EngineConfig(model=LlamaConfig.tiny(), device="cpu",
                                  dtype="float32", kv_cache_blocks=64,
                                  seed=5))
    ref = ref_eng.generate_sync([2, 7, 1, 8, 2, 8], 12, p).token_ids
    # the first token depends only on the exact dense prefill
    assert out[0] == ref[0]
    # and the stream stays plausible (same vocab, mostly agrees for a
    # tiny model whose margins are wide)
    agree = sum(a == b for a, b in zip(out, ref))
    assert agree >= 8, (out, ref)


@pytest.mark.gpu
def test_fp8_append_and_attention_gpu():
    torch.manual_seed(2)
    dev = "cuda:0"
    T, nkv, nq, D, BS, nb = 48, 2, 8, 128, 16, 8
    k = torch.randn(T, nkv, D, dtype=torch.bfloat16, device=dev)
    v = torch.randn(T, nkv, D, dtype=torch.bfloat16, device=dev)
    kc = torch.zeros(nb, nkv, BS, D, dtype=torch.uint8, device=dev)
    vc = torch.zeros_like(kc)
    ks = torch.zeros(nb, nkv, BS, dtype=torch.float32, device=dev)
    vs = torch.zeros_like(ks)
    slots = torch.arange(16, 16 + T, dtype=torch.int32, device=dev)
    ops.kv_append(kc, vc, k, v, slots, k_scale=ks, v_scale=vs)
    # quantization matches the torch e4m3 reference within 1 ULP
    kc_ref = torch.zeros_like(kc).cpu()
    vc_ref = torch.zeros_like(vc).cpu()
    ks_ref = torch.zeros_like(ks).cpu()
    vs_ref = torch.zeros_like(vs).cpu()
    reference.kv_append_fp8(kc_ref, vc_ref, ks_ref, vs_ref, k.cpu(),
                            v.cpu(), slots.cpu(), BS)
    assert torch.allclose(ks.cpu(), ks_ref, rtol=1e-6)
    deq_gpu = reference.dequant_fp8_cache(kc, ks).cpu().float()
    deq_ref = reference.dequant_fp8_cache(kc_ref, ks_ref).float()
    assert (deq_gpu - deq_ref).abs().max() < 0.05

    # attention over the fp8 cache vs SDPA on the dequantized values
    S = 3
    bt = torch.tensor([[1, 2], [2, 3], [3, 4]], dtype=torch.int32,
                      device=dev)
    sl = torch.tensor([20, 30, 17], dtype=torch.int32, device=dev)
    q = torch.randn(S, nq, D, dtype=torch.bfloat16, device=dev)
    out = ops.paged_attn_decode(q, kc, vc, bt, sl, D ** -0.5,
                                k_scale=ks, v_scale=vs)
    kd = reference.dequant_fp8_cache(kc, ks)
    vd = reference.dequant_fp8_cache(vc, vs)
    ref = reference.paged_attn_decode(q.float().cpu(),
                                      kd.cpu().float(),
                                      vd.cpu().float(),
                                      bt.cpu(), sl.cpu(), D ** -0.5)
    rel = (out.cpu().float() - ref).abs().max() / ref.abs().max()
    assert rel < 0.02, rel.item()


@pytest.mark.gpu
def test_fp8_engine_gpu_decode():
    """End-to-end fp8-KV engine on GPU: greedy decode runs through the
    fp8 kernels (graphs on) and stays close to the bf16-KV engine."""
    # fp8 KV needs heads of 128 on GPU, up to 16 to a key/value head
    cfg = LlamaConfig(hidden=512, layers=4, q_heads=4, kv_heads=2,
                      head_dim=128, inter=1024, vocab=4096, max_pos=1024,
                      name="fp8-test")
    p = SamplingParams(temperature=0.0)
    outs = {}
    for kvd in ("bfloat16", "fp8_e4m3"):
        eng = Engine(EngineConfig(model=cfg, device="cuda:0",
                                  dtype="bfloat16", kv_cache_blocks=256,
                                  kv_dtype=kvd, seed=3))
        outs[kvd] = eng.generate_sync(list(range(24)), 16, p).token_ids
        del eng
        torch.cuda.empty_cache()
    assert len(outs["fp8_e4m3"]) == 16
    assert outs["fp8_e4m3"][0] == outs["bfloat16"][0]
    agree = sum(a == b for a, b in zip(outs["fp8_e4m3"],
                                       outs["bfloat16"]))
    assert agree >= 10, outs


@pytest.mark.gpu
def test_fp8_weight_gemm_gpu():
    """W8 arm of the v2 decode GEMM vs fp32 reference on dequantized
    weights (exact math target) and vs the bf16 kernel (quant noise)."""
    torch.manual_seed(4)
    dev = "cuda:0"
    for N, M, K in ((64, 4096, 14336), (16, 28672, 4096),
                    (64, 6144, 4096)):
        x = (torch.randn(N, K, device=dev) * 0.5).to(torch.bfloat16)
        w = (torch.randn(M, K, device=dev) * 0.02).to(torch.bfloat16)
        w8, scale = ops.quantize_fp8_weight(w)
        out = ops.decode_gemm_v2(x, w8, w_scale=scale)
        wd = (w8.view(torch.float8_e4m3fn).float()
              * scale[:, None]).to(torch.float32)
        ref = x.float() @ wd.T
        rel = (out.float() - ref).abs().max() / ref.abs().max()
        assert rel < 0.02, (N, M, K, rel.item())


@pytest.mark.gpu
def test_fp8_weights_engine_gpu():
    """LLMLB_FP8_WEIGHTS engine end-to-end: greedy decode mostly
    agrees with the bf16-weight engine (W8A16 quantization noise)."""
    import importlib
    import llmlb_amd.ops as ops_mod
    from llmlb_amd.backend.engine import Engine, EngineConfig
    from llmlb_amd.backend.sampler import SamplingParams
    from llmlb_amd.models.llama import LlamaConfig
    # real 8B-shaped layers so every projection passes the fp8
    # dispatch legality (K >= 4096, M % 128 == 0)
    cfg = LlamaConfig(hidden=4096, layers=2, q_heads=32, kv_heads=8,
                      head_dim=128, inter=14336, vocab=8192,
                      max_pos=1024, name="w8-test")
    p = SamplingParams(temperature=0.0)
    outs = {}
    for arm in (False, True):
        ops_mod._FP8_WEIGHTS = arm
        try:
            eng = Engine(EngineConfig(model=cfg, device="cuda:0",
                                      dtype="bfloat16",
                                      kv_cache_blocks=128, seed=3))
            outs[arm] = eng.generate_sync(list(range(24)), 16,
                                          p).token_ids
            del eng
            torch.cuda.empty_cache()
        finally:
            ops_mod._FP8_WEIGHTS = False
    assert len(outs[True]) == 16
    # random-init weights have razor-thin logit margins, so greedy
    # token agreement is not a meaningful quality metric here; kernel
    # numerics are covered by test_fp8_weight_gemm_gpu.  Check sanity.
    assert all(0 <= t < cfg.vocab for t in outs[True])
    assert len(outs[False]) == 16


def test_fp8_with_prefix_and_spec_cpu():
    """Feature interplay on CPU: fp8 KV + prefix caching + speculative
    decoding together stay self-consistent (repeatable greedy)."""
    cfg = EngineConfig(model=LlamaConfig.tiny(), device="cpu",
                       dtype="float32", kv_cache_blocks=96,
                       kv_dtype="fp8_e4m3", spec_ngram=4, seed=9)
    p = SamplingParams(temperature=0.0)
    prompt = [3, 1, 3, 1, 3, 1] + list(range(20))
    eng = Engine(cfg)
    a = eng.generate_sync(prompt, 12, p).token_ids
    b = eng.generate_sync(prompt, 12, p).token_ids   # prefix-cache hit
    assert a == b
    assert len(a) == 12
    if eng.prefix:
        assert eng.prefix.hit_tokens > 0


@pytest.mark.gpu
def test_fp8_group8_engine_gpu():
    """fp8 KV with GQA group 8 (the 70B shape): the tiled attention's
    8-bit pages end to end."""
    from llmlb_amd.backend.engine import Engine, EngineConfig
    from llmlb_amd.backend.sampler import SamplingParams
    from llmlb_amd.models.llama import LlamaConfig
    cfg = LlamaConfig(hidden=2048, layers=2, q_heads=16, kv_heads=2,
                      head_dim=128, inter=4096, vocab=8192,
                      max_pos=1024, name="fp8-g8-test")
    eng = Engine(EngineConfig(model=cfg, device="cuda:0",
                              dtype="bfloat16", kv_cache_blocks=256,
                              kv_dtype="fp8_e4m3", seed=6))
    p = SamplingParams(temperature=0.0)
    out = eng.generate_sync(list(range(40)), 12, p).token_ids
    assert len(out) == 12
    assert all(0 <= t < cfg.vocab for t in out)
    out2 = eng.generate_sync(list(range(40)), 12, p).token_ids
    assert out == out2
