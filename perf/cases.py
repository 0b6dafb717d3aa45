"""What the serving backend does for its users, as cases to measure.

The backend reads prompts, generates token by token, and embeds texts, for
the Llama family and four hybrid families.  Sizes are those of
``python bench.py --hybrid``: layers of width 1024, 2048 and 4096 (s, m and
l; l: those of an 8B model), with equal parameters in all families; hybrid
models have 8 of them.  Llama, whose layers are all alike, has 4: on its
16-bit residual stream more would round too much to compare by.  A case is
one model call of a serving process:

work "step"   hybrid families, ``Engine.run_batch``: one token of each of
              ``batch`` sequences that have ``context`` tokens behind them,
              beside ``prompts`` new prompts of about ``length`` tokens
work "token"  Llama: one token of each of ``batch`` sequences through the
              model's layers and the paged cache, captured in a graph as the
              serving loop does; ``kv`` is the cache's storage type
work "embed"  Llama: hidden states of ``batch`` texts of ``length`` tokens

Weights are random and the same for every seed, as a server's are for every
request; tokens, cached keys and values come from the seed.
"""
import math
import random

import torch

from llmlb_amd import ops
from llmlb_amd.backend.engine import Engine, EngineConfig
from llmlb_amd.backend.kv_cache import BLOCK_SIZE, KVCache
from llmlb_amd.models.dibelix import DibelixConfig, DibelixForCausalLM
from llmlb_amd.models.fidepel import FidepelConfig, FidepelForCausalLM
from llmlb_amd.models.llama import LlamaConfig, LlamaForCausalLM
from llmlb_amd.models.rasodra import RasodraConfig, RasodraForCausalLM
from llmlb_amd.models.taletar import TaletarConfig, TaletarForCausalLM

DEVICE = "cuda:0"
F64 = torch.float64
VOCAB, MAX_POS, WINDOW, CHUNK = 32000, 8192, 1024, 2048

#        width heads head_dim kv_heads inter
SIZES = {"s": (1024, 16, 64, 4, 2816),
         "m": (2048, 16, 128, 4, 5632),
         "l": (4096, 32, 128, 8, 14336)}
# feed-forward widths at which all families have Llama's parameters
FF = {"dibelix": {"s": 3584, "m": 7168, "l": 19456},
      "taletar": {"s": 2176, "m": 4352, "l": 11904},
      "fidepel": {"s": 256, "m": 512, "l": 1280},
      "rasodra": {"s": 3328, "m": 6784, "l": 18304}}
CLASSES = {"llama": LlamaForCausalLM, "dibelix": DibelixForCausalLM,
           "taletar": TaletarForCausalLM, "fidepel": FidepelForCausalLM,
           "rasodra": RasodraForCausalLM}


# -- the cases -------------------------------------------------------------

def _step(model, size, batch=0, context=0, prompts=0, length=0,
          dtype="bfloat16"):
    return {"work": "step", "model": model, "size": size, "dtype": dtype,
            "batch": batch, "context": context, "prompts": prompts,
            "length": length}


def _token(size, batch, context, kv="bfloat16"):
    return {"work": "token", "model": "llama", "size": size, "batch": batch,
            "context": context, "kv": kv}


def _embed(size, batch, length):
    return {"work": "embed", "model": "llama", "size": size, "batch": batch,
            "length": length}


def listed():
    named = {
        # one user chatting with a small model: launches and latency
        "token s 1x100": _token("s", 1, 100),
        # a loaded 8B replica generating: the serving benchmark's batch
        "token l 64x1024": _token("l", 64, 1024),
        # the same with the 8-bit cache that long contexts are served with
        "token l fp8 32x2048": _token("l", 32, 2048, kv="fp8_e4m3"),
        # embedding a batch of documents
        "embed l 8x2048": _embed("l", 8, 2048),
        # a wave of long prompts, one per hybrid family
        "prompts dibelix m 8x2048": _step("dibelix", "m", 0, 0, 8, 2048),
        "prompts taletar l 8x2048": _step("taletar", "l", 0, 0, 8, 2048),
        "prompts fidepel m 8x2048": _step("fidepel", "m", 0, 0, 8, 2048),
        # hybrid replicas generating at their benchmark's batch
        "decode dibelix l 64x1024": _step("dibelix", "l", 64, 1024),
        "decode taletar s 64x1024": _step("taletar", "s", 64, 1024),
        "decode fidepel l 61x777": _step("fidepel", "l", 61, 777),
        # continuous batching: prompts of uneven length are read while
        # others generate
        "mixed rasodra m 24x700 3x517": _step("rasodra", "m", 24, 700, 3,
                                              517),
        # the 32-bit type of trace replays
        "prompts rasodra s fp32 2x300": _step("rasodra", "s", 0, 0, 2, 300,
                                              "float32"),
    }
    return [dict(case, name=name) for name, case in named.items()]


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread over its logarithm."""
    return min(hi, int(math.exp(rng.uniform(math.log(lo),
                                            math.log(hi + 1)))))


def draw(rng):
    model = rng.choice(["llama", "llama", *FF])
    size = rng.choice("sml")
    most = {"s": 16384, "m": 16384, "l": 12288}[size]
    if model == "llama":
        if rng.random() < 0.35:
            length = _log(rng, 9, 4096)
            return _embed(size, _log(rng, 1, min(32, most // length)),
                          length)
        context = _log(rng, 16, 4096)
        kv = "bfloat16"
        if SIZES[size][2] == 128 and rng.random() < 0.3:
            kv = "fp8_e4m3"
        return _token(size, _log(rng, 1, min(128, 65536 // context)),
                      context, kv)
    kind = rng.choice(["prompts", "decode", "decode", "mixed", "fp32"])
    if kind == "fp32":
        length = _log(rng, 9, 400)
        return _step(model, "s", 0, 0, rng.randint(1, 4), length, "float32")
    batch = context = prompts = length = 0
    if kind != "decode":
        length = _log(rng, 16, 4096)
        prompts = _log(rng, 1, min(16, most // length))
    if kind != "prompts":
        context = _log(rng, 16, 2048)
        batch = _log(rng, 1, min(96, 49152 // context))
    return _step(model, size, batch, context, prompts, length)


# -- models ----------------------------------------------------------------

def _config(model, size):
    w, h, d, kv, inter = SIZES[size]
    common = dict(vocab=VOCAB, width=w, max_pos=MAX_POS)
    if model == "llama":
        return LlamaConfig(hidden=w, layers=4, q_heads=h, kv_heads=kv,
                           head_dim=d, inter=inter, vocab=VOCAB,
                           max_pos=MAX_POS, name=f"llama-{size}")
    ff = FF[model][size]
    if model == "dibelix":
        return DibelixConfig.build(
            "LDDS" * 2, ff=ff, heads=h, dim=d, rot_dim=d // 2, vdim=d,
            kv_rank=4 * d, window=WINDOW, delta_heads=h, delta_kv_heads=h,
            delta_dim=d, delta_vdim=d, low_rank=d, **common)
    if model == "taletar":
        return TaletarConfig.build(
            "AGMG" * 2, ff=ff, heads=h, kv_heads=kv, dim=d // 2, vdim=d,
            gla_heads=h, gla_dim=d, gla_vdim=d, low_rank=d, ssm_heads=h,
            ssm_vdim=d, state=d, groups=kv, norm_groups=kv, **common)
    if model == "fidepel":
        return FidepelConfig.build(
            8, heads=h, kv_heads=kv, dim=d, vdim=d, window=WINDOW, ff=ff,
            experts=16, top=4, groups=4, keep=2, shared_ff=ff,
            residual_mult=0.4, **common)
    return RasodraConfig.build(
        "AMLM" * 2, ff=ff, heads=h, kv_heads=kv, dim=d, chunk=CHUNK,
        latent_heads=h, latent_dim=d, rot_dim=d // 2, latent_vdim=d,
        kv_rank=4 * d, memory_heads=h, memory_dim=d, memory_vdim=d, **common)


def _clear_routing(embed, routers):
    """Experts are chosen as clearly as a trained router does: every token
    carries the directions of four experts of two groups, which the routers
    read.  (Where random weights choose, rounding decides for some tokens,
    and no two implementations agree on those.)"""
    vocab, width = embed.shape
    g = torch.Generator(device=embed.device).manual_seed(1)
    order = torch.rand(vocab, 4, generator=g, device=embed.device).argsort(1)
    place = torch.rand(vocab, 4, 4, generator=g,
                       device=embed.device).argsort(2)[..., :2]
    experts = (4 * order[:, :2, None]
               + place.gather(1, order[:, :2, None].expand(-1, -1, 2)))
    rows = torch.randn(16, width, generator=g, device=embed.device)
    share = torch.tensor([1.6, 1.2, 1.4, 1.0], device=embed.device)
    carried = (rows[experts.flatten(1)] * share[:, None]).sum(1)
    noise = torch.randn(vocab, width, generator=g, device=embed.device)
    embed.copy_(carried + noise)
    for r in routers:
        r.copy_(rows * (4.0 / width))


def _lengths(case):
    """Prompt lengths of a step: even waves where nothing else runs, uneven
    prompts beside decoding sequences."""
    n, most = case["prompts"], case["length"]
    if not case["batch"]:
        return [most] * n
    return [max(1, most - i * most // 7) for i in range(n)]


def _contexts(case):
    """Tokens behind each of Llama's sequences: requests that have come in
    at different times."""
    c = case["context"]
    return [max(1, c - i * 13 % (c // 4 + 1)) for i in range(case["batch"])]


def _tokens(case, seed):
    """(tokens of the decoding sequences, the next one last; prompts)."""
    g = torch.Generator().manual_seed(seed)

    def some(n):
        return torch.randint(1, VOCAB, (n,), generator=g).tolist()

    return ([some(case["context"] + 1) for _ in range(case["batch"])],
            [some(n) for n in _lengths(case)])


def _prepare_step(case, seed):
    live, prompts = _tokens(case, seed)
    held = [len(t) + BLOCK_SIZE for t in live + prompts]
    engine = Engine(EngineConfig(
        model=_config(case["model"], case["size"]), device=DEVICE,
        dtype=case["dtype"],
        kv_cache_blocks=8 + sum(-(-n // BLOCK_SIZE) for n in held)))
    if case["model"] == "fidepel":
        _clear_routing(engine.model.embed.data,
                       [layer.ff.w_router.data
                        for layer in engine.model.layers_])
    sequences = [engine.open_sequence() for _ in live]
    behind = [(s, t[:-1], []) for s, t in zip(sequences, live)]
    at_once = max(1, 16384 // max(case["context"], 1))
    for i in range(0, len(behind), at_once):
        engine.run_batch(behind[i:i + at_once])
    return {"engine": engine, "sequences": sequences,
            "next": [t[-1] for t in live], "prompts": prompts}


def _run_step(state):
    engine, sequences = state["engine"], state["sequences"]
    fresh = [engine.open_sequence() for _ in state["prompts"]]
    work = [(s, [t], [0]) for s, t in zip(sequences, state["next"])]
    work += [(s, p, [len(p) - 1]) for s, p in zip(fresh, state["prompts"])]
    logits = engine.run_batch(work)
    # the next pass is the same step: the token's place is taken again
    for s in sequences:
        s.length -= 1
    for s in reversed(fresh):
        engine.close_sequence(s)
    n = len(work)
    return {"logits": logits,
            "state": {f"{i:02d}": t[:n]
                      for i, t in engine.kv.state.items()}}


def _prepare_token(case, seed):
    cfg = _config("llama", case["size"])
    model = LlamaForCausalLM(cfg, device=DEVICE)
    lens = _contexts(case)
    pages = [n // BLOCK_SIZE + 1 for n in lens]
    total = sum(pages)
    kv = KVCache(cfg.layers, 1 + total, cfg.kv_heads, cfg.head_dim, DEVICE,
                 kv_dtype=case["kv"])
    # pages come and go with requests: no sequence has its own in order
    mixed = kv.allocate(total)
    random.Random(seed).shuffle(mixed)
    table = torch.zeros(len(lens), MAX_POS // BLOCK_SIZE, dtype=torch.int32)
    for i, n in enumerate(pages):
        table[i, :n] = torch.tensor(mixed[:n])
        mixed = mixed[n:]
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    slots = torch.arange(BLOCK_SIZE, (1 + total) * BLOCK_SIZE, device=DEVICE)
    std = 0.02 * cfg.hidden ** 0.5        # as the projections make them
    for li in range(cfg.layers):
        k, v = torch.randn(2, len(slots), cfg.kv_heads, cfg.head_dim,
                           generator=g, device=DEVICE).mul_(std).bfloat16()
        ops.kv_append(
            kv.k[li], kv.v[li], k, v, slots,
            k_scale=kv.k_scale[li] if kv.fp8 else None,
            v_scale=kv.v_scale[li] if kv.fp8 else None)
    at = torch.tensor(lens)
    state = {
        "model": model, "kv": kv, "table": table.to(DEVICE),
        "ids": torch.randint(1, VOCAB, (len(lens),), generator=g,
                             device=DEVICE),
        "lens": at.int().to(DEVICE), "seq_lens": (at + 1).int().to(DEVICE),
        "slots": (table.gather(1, at[:, None] // BLOCK_SIZE)[:, 0]
                  * BLOCK_SIZE + at % BLOCK_SIZE).int().to(DEVICE)}
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _forward_token(state)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    state["graph"] = torch.cuda.CUDAGraph()
    with torch.cuda.graph(state["graph"]):
        state["logits"] = _forward_token(state)
    return state


def _forward_token(s):
    model, kv = s["model"], s["kv"]
    ops.set_decode_phase(True)
    try:
        h, residual = model.embed_tokens(s["ids"]), None
        for li in range(model.cfg.layers):
            scales = dict(k_scale=kv.k_scale[li], v_scale=kv.v_scale[li]) \
                if kv.fp8 else {}
            q, k, v, residual = model.layer_attn_prelude(
                li, h, residual, s["lens"], quant_ok=True,
                kv_sink=None if kv.fp8 else (kv.k[li], kv.v[li],
                                             s["slots"]))
            if kv.fp8:
                ops.kv_append(kv.k[li], kv.v[li], k, v, s["slots"], **scales)
            attn = ops.paged_attn_decode(
                q, kv.k[li], kv.v[li], s["table"], s["seq_lens"],
                model.cfg.head_dim ** -0.5, **scales)
            h, residual = model.layer_attn_epilogue(li, attn, residual,
                                                    quant_ok=True)
        return model.final(h, residual, quant_ok=True)
    finally:
        ops.set_decode_phase(False)


def _prepare_embed(case, seed):
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    return {"model": LlamaForCausalLM(_config("llama", case["size"]),
                                      device=DEVICE),
            "ids": torch.randint(1, VOCAB, (case["batch"], case["length"]),
                                 generator=g, device=DEVICE)}


@torch.inference_mode()
def prepare(case, seed):
    make = {"step": _prepare_step, "token": _prepare_token,
            "embed": _prepare_embed}[case["work"]]
    return dict(make(case, seed), work=case["work"])


def run(state):
    if state["work"] == "step":
        return _run_step(state)
    if state["work"] == "token":
        state["graph"].replay()
        return state["logits"]
    return state["model"].forward_dense(state["ids"])


# -- what a pass needs -----------------------------------------------------

def _pairs(n, context, window=None, chunk=None):
    """(query, key) pairs of n queries behind ``context`` tokens."""
    if chunk:
        return sum((context + i) % chunk + 1 for i in range(n))
    first, last = context + 1, context + n
    if window is None or last <= window:
        return (first + last) * n // 2
    return sum(min(context + i + 1, window) for i in range(n))


def _work_llama(case):
    cfg = _config("llama", case["size"])
    q, kv = cfg.q_heads * cfg.head_dim, cfg.kv_heads * cfg.head_dim
    layers = cfg.layers * cfg.hidden * (2 * q + 2 * kv + 3 * cfg.inter)
    if case["work"] == "embed":
        n, L = case["batch"], case["length"]
        return {"bytes": 2 * layers + n * L * (4 * cfg.hidden + 8),
                "flops": 2 * n * L * layers
                + 4 * cfg.layers * q * n * _pairs(L, 0)}
    lens = _contexts(case)
    head = cfg.vocab * cfg.hidden
    per_token = 2 * (kv + 4 * cfg.kv_heads) if case["kv"] != "bfloat16" \
        else 4 * kv
    return {"bytes": 2 * (layers + head) + cfg.layers * per_token
            * sum(n + 1 for n in lens)
            + len(lens) * (2 * cfg.vocab + 2 * cfg.hidden),
            "flops": 2 * len(lens) * (layers + head)
            + 4 * cfg.layers * q * sum(n + 1 for n in lens)}


def _work_step(case):
    cfg = _config(case["model"], case["size"])
    shapes = CLASSES[case["model"]](cfg, device="meta",
                                    init_weights=False).weight_shapes()
    size = 4 if case["dtype"] == "float32" else 2
    runs = [(1, case["context"])] * case["batch"] \
        + [(n, 0) for n in _lengths(case)]
    T, n_out = sum(n for n, _ in runs), len(runs)
    layers = sum(math.prod(s) for k, s in shapes.items()
                 if k not in ("embed", "head"))
    used = layers                       # parameters that a token meets
    experts = sum(math.prod(s) for k, s in shapes.items() if ".mlp.e" in k)
    if experts:
        used -= experts * 12 // 16
        layers -= int(experts * (12 / 16) ** T)      # none of whose tokens
    head = math.prod(shapes["head"])
    nbytes = size * (layers + head + T * cfg.width) + 4 * n_out * cfg.vocab
    flops = 2 * T * used + 2 * n_out * head
    for layer in cfg.layers:
        m = layer["mixer"]
        H = m["heads"]
        if "attention" in layer["type"]:
            mask = (m.get("mask") or {}).get("size")
            rank, rot = m.get("kv_rank"), m.get("rot_dim", 0)
            maps = 2 if "diff" in m else 1
            row = rank + rot if rank else \
                m["kv_heads"] * (maps * m["dim"] + m["vdim"])
            chunk = mask if case["model"] == "rasodra" and not rank else None
            for n, context in runs:
                seen = _pairs(n, context, None if chunk else mask, chunk)
                flops += 2 * H * seen * maps * (m["dim"] + rot + m["vdim"])
                keys = _pairs(1, context, None if chunk else mask, chunk) \
                    if context else n
                nbytes += size * row * keys
            continue
        D = m.get("state") or m["dim"]
        flops += 4 * T * H * D * m["vdim"]
        nbytes += 4 * H * D * m["vdim"] * (2 * case["batch"]
                                           + case["prompts"])
    return {"bytes": nbytes, "flops": flops}


def work(case):
    return _work_step(case) if case["work"] == "step" else _work_llama(case)


def tolerance(case):
    """16-bit runs are 0.0025 to 0.020 from ``exact``, 32-bit runs 6e-7 to
    5e-6; four times that, and at most 0.03."""
    return {"rel": 2e-5 if case.get("dtype") == "float32" else 0.03}


# -- the same in 64 bits ---------------------------------------------------

def _rms(x, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)


def _layer_norm(x, w, eps):
    d = x - x.mean(-1, keepdim=True)
    return d * torch.rsqrt(d.square().mean(-1, keepdim=True) + eps) * w


def _rotate(x, pos, base, n, neighbours=False):
    """x [B, T, heads, D]: the first n numbers of each head turned at
    positions ``pos`` ([T] or [B, T]); pairs are neighbours or n/2 apart."""
    i = torch.arange(n // 2, dtype=F64, device=x.device)
    a = pos.to(F64)[..., None, None] * base ** (-2.0 * i / n)
    cos, sin = a.cos(), a.sin()
    out = x.clone()
    u, v = (slice(0, n, 2), slice(1, n, 2)) if neighbours else \
        (slice(0, n // 2), slice(n // 2, n))
    out[..., u] = x[..., u] * cos - x[..., v] * sin
    out[..., v] = x[..., v] * cos + x[..., u] * sin
    return out


def _attend(q, k, v, scale, window=None, chunk=None, cap=None, sink=None):
    """Causal attention: q [B, T, H, D], k [B, T, G, D], v [B, T, G, V]."""
    B, T, H, _ = q.shape
    G = k.shape[2]
    at = torch.arange(T, device=q.device)
    back = at[:, None] - at[None]
    seen = back >= 0
    if window is not None:
        seen &= back < window
    if chunk is not None:
        seen &= at[:, None] // chunk == at[None] // chunk
    out = []
    for b in range(B):
        qb = q[b].view(T, G, H // G, -1).permute(1, 2, 0, 3)
        s = qb.reshape(G, H // G * T, -1) @ k[b].permute(1, 2, 0) * scale
        if cap:
            s = cap * torch.tanh(s / cap)
        s = s.view(G, H // G, T, T).masked_fill(~seen, -math.inf)
        if sink is not None:
            s = torch.cat([s, sink.view(G, H // G, 1, 1).expand(
                G, H // G, T, 1)], -1)
        p = torch.softmax(s, -1)[..., :T]
        o = p.reshape(G, H // G * T, T) @ v[b].transpose(0, 1)
        out.append(o.view(G, H // G, T, -1).permute(2, 0, 1, 3).reshape(
            T, H, -1))
    return torch.stack(out)


def _conv(x, taps, bias=None):
    """Causal convolution per channel, then silu; taps [C, K]."""
    T, K = x.shape[1], taps.shape[1]
    pad = torch.nn.functional.pad(x, (0, 0, K - 1, 0))
    y = sum(pad[:, i:i + T] * taps[:, i] for i in range(K))
    return torch.nn.functional.silu(y if bias is None else y + bias)


def _scan(q, k, v, g):
    """S <- diag(g) S + v k^T, o = S q, with S [B, H, V, D]."""
    B, T, H, D = q.shape
    S = q.new_zeros(B, H, v.shape[-1], D)
    out = torch.empty_like(v)
    for t in range(T):
        S.mul_(g[:, t, :, None]).add_(v[:, t, ..., None] * k[:, t, :, None])
        out[:, t] = (S @ q[:, t, ..., None])[..., 0]
    return out, S


def _latent(h, w, m, eps, kept=None, neighbours=False):
    B, T, _ = h.shape
    H, D, R = m["heads"], m["dim"], m["rot_dim"]
    pos, base = torch.arange(T, device=h.device), m["rot"]["base"]
    if kept is None:
        c, kr = torch.split(h @ w["dkv"].T, [m["kv_rank"], R], -1)
        kept = (_rms(c, eps) * w["dkv.norm"],
                _rotate(kr[:, :, None], pos, base, R, neighbours))
    c, kr = kept
    q = (h @ w["q"].T).view(B, T, H, D + R)
    q = torch.cat([q[..., :D],
                   _rotate(q[..., D:], pos, base, R, neighbours)], -1)
    k = torch.cat([(c @ w["uk"].T).view(B, T, H, D),
                   kr.expand(B, T, H, R)], -1)
    o = _attend(q, k, (c @ w["uv"].T).view(B, T, H, -1), m["scale"],
                (m.get("mask") or {}).get("size"), sink=w.get("sink"))
    o = o.flatten(2)
    if "g" in w:
        o = o * torch.sigmoid(h @ w["g"].T)
    return o @ w["o"].T, kept


def _delta(h, w, m, eps):
    B, T, _ = h.shape
    H, KH, D, V = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
    q, k, v = (_conv(h @ w[n].T, w[n + ".conv"]).view(B, T, -1, d)
               for n, d in (("q", D), ("k", D), ("v", V)))
    q, k = (t * torch.rsqrt(t.square().sum(-1, keepdim=True) + 1e-6)
            for t in (q, k))
    q, k = (t.repeat_interleave(H // KH, 2) for t in (q * D ** -0.5, k))
    z = ((h @ w["a1"].T) @ w["a2"].T + w["dt_bias"]).view(B, T, H, D)
    g = torch.exp(-w["A_log"].exp()[:, None]
                  * torch.nn.functional.softplus(z, threshold=50.0))
    beta = torch.sigmoid(h @ w["b"].T)[..., None]
    S = q.new_zeros(B, H, V, D)
    o = torch.empty_like(v)
    for t in range(T):
        S.mul_(g[:, t, :, None])
        u = beta[:, t] * (v[:, t] - (S @ k[:, t, ..., None])[..., 0])
        S.add_(u[..., None] * k[:, t, :, None])
        o[:, t] = (S @ q[:, t, ..., None])[..., 0]
    gate = torch.sigmoid((h @ w["g1"].T) @ w["g2"].T).view(B, T, H, V)
    o = _rms(o, eps) * w["norm"] * gate
    return o.flatten(2) @ w["o"].T, S


def _dibelix(x, w, cfg):
    kept, states = {}, {}
    for i, layer in enumerate(cfg.layers):
        m, mix, mlp = layer["mixer"], w.part(f"l{i}.mix."), \
            w.part(f"l{i}.mlp.")
        if layer["type"] == "latent_attention":
            y, c = _latent(x, mix, m, cfg.eps, kept.get(m.get("kv_from")))
            kept[i] = c
        else:
            y, states[i] = _delta(x, mix, m, cfg.eps)
        x = x + _rms(y, cfg.eps) * (1.0 + w[f"l{i}.norm1"])
        u = torch.nn.functional.gelu(x @ mlp["up"].T, approximate="tanh")
        x = x + _rms(u @ mlp["down"].T, cfg.eps) * (1.0 + w[f"l{i}.norm2"])
    z = (_rms(x[:, -1], cfg.eps) * (1.0 + w["final.norm"])) @ w["head"].T
    return cfg.logit_softcap * torch.tanh(z / cfg.logit_softcap), states


def _pair(h, w, m, eps):
    B, T, _ = h.shape
    H, G, D, V = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
    q = (h @ w["q"].T).view(B, T, H, 2, D)
    k = (h @ w["k"].T).view(B, T, G, 2, D)
    v = (h @ w["v"].T).view(B, T, G, V)
    p = torch.arange(1, T + 1, dtype=F64, device=h.device)
    temp = 1.0 + m["q_temp"]["coef"] * torch.log(
        torch.floor(p / m["q_temp"]["every"]) + 1.0)
    q = q * temp[:, None, None, None]
    a, b = (_attend(q[..., n, :], k[..., n, :], v, m["scale"],
                    cap=m["softcap"]) for n in (0, 1))
    lam = (w["lq1"] * w["lk1"]).sum().exp() \
        - (w["lq2"] * w["lk2"]).sum().exp() + m["diff"]
    o = _rms(a - lam * b, eps) * (1.0 - m["diff"])
    return o.flatten(2) * torch.sigmoid(h @ w["g"].T)


def _gla(h, w, m, eps):
    B, T, _ = h.shape
    H, D, V = m["heads"], m["dim"], m["vdim"]
    q = (h @ w["q"].T).view(B, T, H, D) * D ** -0.5
    k = (h @ w["k"].T).view(B, T, H, D)
    v = (h @ w["v"].T).view(B, T, H, V)
    z = (h @ w["a1"].T) @ w["a2"].T + w["a2.b"]
    o, S = _scan(q, k, v, (torch.sigmoid(z) ** (1.0 / m["tau"])).view(
        B, T, H, D))
    o = (_rms(o, eps) * w["norm"]).flatten(2)
    return o * torch.nn.functional.silu(h @ w["g"].T), S


def _mamba(h, w, m, eps):
    B, T, _ = h.shape
    H, V, N, G = m["heads"], m["vdim"], m["state"], m["groups"]
    z, xbc, dt = torch.split(h @ w["in"].T,
                             [H * V, H * V + 2 * G * N, H], -1)
    x, b, c = torch.split(_conv(xbc, w["conv"], w["conv.b"]),
                          [H * V, G * N, G * N], -1)
    x = x.view(B, T, H, V)
    b, c = (t.view(B, T, G, N).repeat_interleave(H // G, 2) for t in (b, c))
    dt = torch.nn.functional.softplus(dt + w["dt_bias"])[..., None]
    y, S = _scan(c, b, dt * x, torch.exp(-w["A_log"].exp()[:, None] * dt)
                 .expand(B, T, H, N))
    y = (y + w["D"][:, None] * x).flatten(2) * torch.nn.functional.silu(z)
    y = _rms(y.view(B, T, m["norm_groups"], -1), eps).flatten(2)
    return y * w["norm"], S


def _taletar(x, w, cfg):
    states = {}
    for i, layer in enumerate(cfg.layers):
        mix, mlp = w.part(f"l{i}.mix."), w.part(f"l{i}.mlp.")
        n = _rms(x, cfg.eps)
        h, limit = n * w[f"l{i}.norm1"], layer["mlp"]["limit"]
        if layer["type"] == "attention":
            y = _pair(h, mix, layer["mixer"], cfg.eps)
        else:
            y, states[i] = (_gla if layer["type"] == "gla" else _mamba)(
                h, mix, layer["mixer"], cfg.eps)
        h = n * w[f"l{i}.norm2"]
        g = (h @ mlp["gate"].T).clamp(max=limit)
        u = (h @ mlp["up"].T).clamp(-limit, limit)
        u = g * torch.sigmoid(1.702 * g) * (u + 1.0)
        x = x + y @ mix["o"].T + u @ mlp["down"].T
    return (_rms(x[:, -1], cfg.eps) * w["final.norm"]) @ w["head"].T, states


def _experts(h, w, mlp):
    """Routed and shared experts of h [T, W]."""
    r = mlp["router"]
    E, count, keep = r["experts"], r["groups"]["count"], r["groups"]["keep"]
    p = torch.softmax(h @ w["router"].T, -1)
    best = p.view(-1, count, E // count).amax(-1)
    kept = torch.zeros_like(best, dtype=torch.bool).scatter_(
        1, best.topk(keep, -1).indices, True)
    chosen = p.masked_fill(~kept.repeat_interleave(E // count, 1), -1.0)
    top, index = chosen.topk(r["top"], -1)
    weight = torch.zeros_like(p).scatter_(
        1, index, top / (top.sum(-1, keepdim=True) + 1e-20) * r["scale"])

    def one(t, name):
        u = (t @ w[name + ".up"].T).clamp(min=0.0)
        return u.square() @ w[name + ".down"].T

    y = one(h, "shared")
    for e in range(E):
        rows = weight[:, e].nonzero()[:, 0]
        y[rows] += weight[rows, e, None] * one(h[rows], f"e{e}")
    return y


def _fidepel(x, w, cfg):
    B, T, W = x.shape
    pos = torch.arange(T, device=x.device)
    for i, layer in enumerate(cfg.layers):
        m, mix, mlp = layer["mixer"], w.part(f"l{i}.mix."), \
            w.part(f"l{i}.mlp.")
        h = _rms(x, cfg.eps) * w[f"l{i}.norm1"]
        q, k = (_rotate((_rms(h @ mix[n].T, cfg.eps) * mix[n + ".norm"])
                        .view(B, T, -1, m["dim"]), pos, m["rot"]["base"],
                        m["rot"]["dims"]) for n in ("q", "k"))
        o = _attend(q * mix["temp"][:, None], k,
                    (h @ mix["v"].T).view(B, T, -1, m["vdim"]), m["scale"],
                    m["mask"]["size"])
        o = (o * torch.sigmoid(h @ mix["g"].T)[..., None]).flatten(2)
        y = _experts(h.view(-1, W), mlp, layer["mlp"]).view(B, T, W)
        x = x + cfg.residual_mult * (o @ mix["o"].T + y)
    return (_rms(x[:, -1], cfg.eps) * w["final.norm"]) @ w["head"].T, {}


def _memory(h, w, m, eps):
    B, T, _ = h.shape
    H, D, V, cap = m["heads"], m["dim"], m["vdim"], m["gate_cap"]
    q = (h @ w["q"].T).view(B, T, H, D) * D ** -0.5
    k = (h @ w["k"].T).view(B, T, H, D)
    v = (h @ w["v"].T).view(B, T, H, V)
    li = cap * torch.tanh((h @ w["i"].T + w["i.b"]) / cap)
    lf = torch.nn.functional.logsigmoid(
        cap * torch.tanh((h @ w["f"].T + w["f.b"]) / cap))
    S, n = q.new_zeros(B, H, V, D), q.new_zeros(B, H, D)
    top = q.new_zeros(B, H)
    o = torch.empty_like(v)
    for t in range(T):
        new = torch.maximum(lf[:, t] + top, li[:, t])
        keep = torch.exp(lf[:, t] + top - new)[..., None]
        put = torch.exp(li[:, t] - new)[..., None] * k[:, t]
        S.mul_(keep[..., None]).add_(v[:, t, ..., None] * put[:, :, None])
        n, top = keep * n + put, new
        den = torch.maximum((n * q[:, t]).sum(-1).abs(), torch.exp(-top))
        o[:, t] = (S @ q[:, t, ..., None])[..., 0] / (den + 1e-6)[..., None]
    o = _rms(o, eps).flatten(2) * w["norm"]
    return (o * torch.sigmoid(h @ w["g"].T)) @ w["o"].T, S


def _rasodra(x, w, cfg):
    B, T, _ = x.shape
    pos, states = torch.arange(T, device=x.device), {}
    for i, layer in enumerate(cfg.layers):
        m, mix, mlp = layer["mixer"], w.part(f"l{i}.mix."), \
            w.part(f"l{i}.mlp.")
        h = _layer_norm(x, w[f"l{i}.norm1"], cfg.eps)
        if layer["type"] == "mlstm":
            y, states[i] = _memory(h, mix, m, cfg.eps)
        elif layer["type"] == "latent_attention":
            y, _ = _latent(h, mix, m, cfg.eps, neighbours=True)
        else:
            q, v = ((h @ mix[n].T + mix[n + ".b"]).view(B, T, -1, m["dim"])
                    for n in ("q", "k"))
            q, k = (_rotate(_rms(t, cfg.eps) * mix[n], pos, m["rot"]["base"],
                            m["rot"]["dims"], True)
                    for t, n in ((q, "q.norm"), (v, "k.norm")))
            y = _attend(q, k, v, m["scale"], chunk=m["mask"]["size"]) \
                .flatten(2) @ mix["o"].T
        x = x + _layer_norm(y, w[f"l{i}.norm1b"], cfg.eps)
        h = _layer_norm(x, w[f"l{i}.norm2"], cfg.eps)
        u = (h @ mlp["up"].T).clamp(min=0.0).square()
        x = x + _layer_norm(u @ mlp["down"].T, w[f"l{i}.norm2b"], cfg.eps)
    return _layer_norm(x[:, -1], w["final.norm"], cfg.eps) @ w["head"].T, \
        states


class _Weights(dict):
    """Tensors by name, widened to 64 bits as they are used."""

    def __getitem__(self, name):
        return super().__getitem__(name).to(F64)

    def get(self, name, default=None):
        return self[name] if name in self else default

    def part(self, prefix):
        return _Weights({k[len(prefix):]: t for k, t in self.items()
                         if k.startswith(prefix)})


def _given_weights(case):
    """The random weights that an engine of this case serves, by name, as
    it stores them: matrices in the storage type, the rest in 32 bits."""
    dtype = getattr(torch, case["dtype"])
    model = CLASSES[case["model"]](
        _config(case["model"], case["size"]), dtype=dtype, device=DEVICE,
        init_weights=False)
    shapes = model.weight_shapes()
    g = torch.Generator(device=DEVICE).manual_seed(EngineConfig.seed)
    drawn = {}

    def take(name):
        t = model.random_tensor(name, torch.randn(
            shapes[name], generator=g, device=DEVICE))
        drawn[name] = t.to(dtype) \
            if t.dim() == 2 and not name.endswith("conv") else t
        return t

    model._assign(take)
    if case["model"] == "fidepel":       # drawn twice, of which this is used
        for i, layer in enumerate(model.layers_):
            drawn[f"l{i}.mix.o"] = layer.w_out[:, :layer.mix.out_width]
        _clear_routing(drawn["embed"], [
            drawn[f"l{i}.mlp.router"] for i in range(len(model.layers_))])
    return model.cfg, _Weights(drawn)


def _exact_step(case, seed):
    cfg, w = _given_weights(case)
    live, prompts = _tokens(case, seed)
    every = live + prompts
    forward = {"dibelix": _dibelix, "taletar": _taletar,
               "fidepel": _fidepel, "rasodra": _rasodra}[case["model"]]
    logits, states = [None] * len(every), {}
    # sequences of one length at a time, as many as memory has room for
    for n in sorted({len(t) for t in every}):
        rows = [i for i, t in enumerate(every) if len(t) == n]
        at_once = max(1, 32768 // n)
        for j in range(0, len(rows), at_once):
            part = rows[j:j + at_once]
            ids = torch.tensor([every[i] for i in part], device=DEVICE)
            z, found = forward(w["embed"][ids], w, cfg)
            for r, i in enumerate(part):
                logits[i] = z[r]
                for li, s in found.items():
                    states.setdefault(li, [None] * len(every))[i] = s[r]
    return {"logits": torch.stack(logits),
            "state": {f"{li:02d}": torch.stack(s)
                      for li, s in states.items()}}


def _exact_llama(case, seed):
    s = prepare(case, seed)
    model, cfg = s["model"], s["model"].cfg
    eps, D, B = cfg.norm_eps, cfg.head_dim, s["ids"].shape[0]
    nq, nkv = cfg.q_heads, cfg.kv_heads
    token = case["work"] == "token"
    T = 1 if token else case["length"]
    pos = s["lens"][:, None] if token else torch.arange(T, device=DEVICE)
    x = model.embed[s["ids"]].to(F64).view(B, T, -1)
    for li, layer in enumerate(model.layers_):
        h = _rms(x, eps) * layer.input_norm_w.to(F64)
        q, k, v = (h @ layer.qkv.weight.to(F64).T).view(
            B, T, nq + 2 * nkv, D).split([nq, nkv, nkv], 2)
        q, k = (_rotate(t, pos, cfg.rope_theta, D) for t in (q, k))
        if token:
            o = _paged(q[:, 0], k[:, 0], v[:, 0], s, li)[:, None]
        else:
            o = _attend(q, k, v, D ** -0.5)
        x = x + o.flatten(2) @ layer.o_proj.weight.to(F64).T
        h = _rms(x, eps) * layer.post_norm_w.to(F64)
        g, u = (h @ layer.gate_up.weight.to(F64).T).chunk(2, -1)
        x = x + (torch.nn.functional.silu(g) * u) \
            @ layer.down.weight.to(F64).T
    x = _rms(x, eps) * model.final_norm_w.to(F64)
    return x[:, 0] @ model.lm_head.to(F64).T if token else x


def _paged(q, k_new, v_new, s, li):
    """Attention of one new token of every sequence over its pages."""
    kv, out = s["kv"], []
    for b, n in enumerate(s["lens"].tolist()):
        pages = s["table"][b, :n // BLOCK_SIZE + 1].long()
        keys, values = (_cached(store[li][pages], None if not kv.fp8
                                else scale[li][pages], n)
                        for store, scale in ((kv.k, kv.k_scale),
                                             (kv.v, kv.v_scale)))
        keys = torch.cat([keys, k_new[b][:, None]], 1)       # [G, n + 1, D]
        values = torch.cat([values, v_new[b][:, None]], 1)
        qb = q[b].view(len(keys), -1, q.shape[-1])
        p = torch.softmax(qb @ keys.transpose(1, 2) * q.shape[-1] ** -0.5,
                          -1)
        out.append((p @ values).reshape(q.shape[1], -1))
    return torch.stack(out)


def _cached(pages, scale, n):
    """The first n tokens of pages [P, G, 16, D] as [G, n, D]."""
    if scale is not None:
        pages = pages.view(torch.float8_e4m3fn).to(F64) \
            * scale.to(F64)[..., None]
    return pages.to(F64).transpose(0, 1).flatten(1, 2)[:, :n]


@torch.inference_mode()
def exact(case, seed):
    if case["work"] == "step":
        return _exact_step(case, seed)
    return _exact_llama(case, seed)
