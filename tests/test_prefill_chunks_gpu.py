"""Prompts as they are served, in chunks and behind cached prefixes, at the
head sizes of the tiled attention kernels: what the engine hands over (layout,
strides, scale, pages) against one pass without a cache."""
import pytest
import torch

import llmlb_amd.ops as ops
from llmlb_amd.backend.engine import Engine, EngineConfig
from llmlb_amd.backend.sampler import SamplingParams
from llmlb_amd.models.llama import LlamaConfig

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LENGTH, CHUNK, NEW = 200, 64, 5


class _Watch:
    """Logits and attention routes of an engine's steps."""

    def __init__(self, engine, monkeypatch):
        self.logits, self.tiled = [], []
        final, tiled = engine.model.final, ops.prompt_attn_tiled

        def watched_final(*args, **kw):
            out = final(*args, **kw)
            self.logits.append(out.float())
            return out

        def watched_tiled(q, k, v):
            self.tiled.append((q.shape[1], k.shape[1], tiled(q, k, v)))
            return self.tiled[-1][2]

        monkeypatch.setattr(engine.model, "final", watched_final)
        monkeypatch.setattr(ops, "prompt_attn_tiled", watched_tiled)


def _serve(engine, prompts, monkeypatch):
    """The first tokens' logits [B, vocab], all tokens, routes."""
    with monkeypatch.context() as patch:
        watch = _Watch(engine, patch)
        sinks = [engine.submit(p, SamplingParams(
            temperature=0.0, max_new_tokens=NEW))[1] for p in prompts]
        for _ in range(100):
            if not engine.step():
                break
    tokens = []
    for sink in sinks:
        tokens.append([])
        while len(tokens[-1]) < NEW:
            tokens[-1].append(sink.get_nowait()[0])
    return watch.logits[0], tokens, watch.tiled


def _whole(model, prompts):
    """Logits of the last tokens by one pass over whole prompts."""
    h = model.forward_dense(torch.tensor(prompts, device=DEV))
    return torch.nn.functional.linear(h[:, -1].float(),
                                      model.lm_head.float())


# Logits of two bf16 layers in another order are 2^-7 apart; keys and values
# in e4m3 are 2^-4 of themselves off each, which attention over a hundred
# tokens averages.  Heads, tokens or pages in the wrong place change logits by
# as much as they are.
@pytest.mark.parametrize("dim,kv,tol", [(64, "bfloat16", 0.03),
                                        (128, "bfloat16", 0.03),
                                        (128, "fp8_e4m3", 0.1)])
@pytest.mark.parametrize("batch", [1, 3])
def test_chunks_and_prefixes(dim, kv, tol, batch, monkeypatch):
    cfg = LlamaConfig(hidden=256, layers=2, q_heads=6, kv_heads=2,
                      head_dim=dim, inter=512, vocab=1024, max_pos=512,
                      name=f"llama-{dim}")
    engine = Engine(EngineConfig(
        model=cfg, device=DEV, dtype="bfloat16", kv_cache_blocks=256,
        prefill_chunk=CHUNK, enable_prefix_cache=True, kv_dtype=kv, seed=21))
    g = torch.Generator().manual_seed(dim + batch)
    prompts = torch.randint(1, cfg.vocab, (batch, LENGTH),
                            generator=g).tolist()
    want = _whole(engine.model, prompts)

    def close(got):
        off = (got - want).norm() / want.norm()
        assert off < tol, float(off)

    first, tokens, routes = _serve(engine, prompts, monkeypatch)
    close(first)
    # all chunks, the later ones behind the cached tokens of those before
    seen = {(new, keys) for new, keys, _ in routes}
    assert seen == {(CHUNK, CHUNK), (CHUNK, 2 * CHUNK), (CHUNK, 3 * CHUNK),
                    (LENGTH - 3 * CHUNK, LENGTH)}
    assert all(tiled for _, _, tiled in routes)

    hits = engine.prefix.hit_tokens
    again, same, routes = _serve(engine, prompts, monkeypatch)
    close(again)
    cached = (engine.prefix.hit_tokens - hits) // batch
    assert cached >= LENGTH - CHUNK
    assert {(new, keys) for new, keys, _ in routes} == {
        (LENGTH - cached, LENGTH)}
    assert all(tiled for _, _, tiled in routes)

    # Decoding reads what the chunks stored: its tokens are the best, but for
    # those that errors of logits (four times the rms at most, both ways)
    # may exchange.
    assert same == tokens or kv != "bfloat16"
    for i in range(NEW):
        z = _whole(engine.model, [p + t[:i] for p, t in zip(prompts, tokens)])
        chosen = z.gather(1, torch.tensor([[t[i]] for t in tokens],
                                          device=DEV))
        gap = z.amax(1, keepdim=True) - chosen
        assert (gap <= 8 * tol * z.square().mean(1, keepdim=True).sqrt()
                ).all(), (i, gap)
