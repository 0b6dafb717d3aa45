"""Queries, keys and values rotated and appended in the product's launch
(row_gemm.hip) against the product and the launches that follow it."""
import pytest
import torch

import llmlb_amd.ops as ops
from llmlb_amd.ops.reference import build_cos_sin_table

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _inputs(N, n_q, n_kv, D, K, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed + N + K)
    x = torch.randn(N, K + 8, generator=g, device=DEV).bfloat16()[:, :K]
    w = torch.randn((n_q + 2 * n_kv) * D, K, generator=g, device=DEV).bfloat16()
    pos = torch.randint(0, 500, (N,), generator=g, device=DEV)
    slots = torch.randperm(256, generator=g, device=DEV)[:N].int()
    return x, w, pos, slots


def _views(t, n_q, n_kv, D):
    q, k, v = t.split([n_q * D, n_kv * D, n_kv * D], dim=1)
    return q.unflatten(1, (n_q, D)), k.unflatten(1, (n_kv, D)), \
        v.unflatten(1, (n_kv, D))


# one row and all tiles of rows; heads smaller than a tile of outputs, of its
# size and larger; fewer pieces of the depth than waves, and a remainder
@pytest.mark.parametrize("n_q,n_kv,D,K", [
    (1, 1, 8, 8), (3, 1, 16, 72), (16, 4, 64, 1024), (14, 2, 64, 264),
    (32, 8, 128, 520), (5, 5, 256, 136)])
@pytest.mark.parametrize("N", [1, 16, 17, 40, 64, 97, 128])
@pytest.mark.parametrize("sink", [True, False])
def test_as_launches_of_their_own(N, n_q, n_kv, D, K, sink):
    x, w, pos, slots = _inputs(N, n_q, n_kv, D, K)
    slots[N // 2] = -1                         # a token without a place
    cs = build_cos_sin_table(512, D, 1e4, device=DEV)
    still = torch.cat([torch.ones(512, D // 2, device=DEV),
                       torch.zeros(512, D // 2, device=DEV)], 1)
    plain = ops.linear_rotary(x, w, n_q, n_kv, D, still, pos)
    x64, w64 = x.double(), w.double()
    ref = x64 @ w64.T
    bound = ref.abs() * 2.0 ** -8 \
        + (x64.abs() @ w64.abs().T) * K * 2.0 ** -24
    assert ((plain.double() - ref).abs() <= bound + 1e-30).all()

    caches = [torch.full((17, n_kv, 16, D), 7.0, device=DEV).bfloat16()
              for _ in range(4)]
    out = ops.linear_rotary(x, w, n_q, n_kv, D, cs, pos,
                            (caches[0], caches[1], slots) if sink else None)
    q, k, v = _views(plain, n_q, n_kv, D)
    if sink and D % 16 == 0:
        ops.rope_kv_append(q, k, v, cs, pos, caches[2], caches[3], slots)
    elif D % 16 == 0:
        ops.rope_apply(q, k, cs, pos)
    else:                                      # heads their kernel refuses
        half = D // 2
        c, s = cs[pos][:, None, :half], cs[pos][:, None, half:]
        for t in (q, k):
            a, b = t.float().chunk(2, -1)
            t.copy_(torch.cat([a * c - b * s, b * c + a * s], -1))
        assert (out.float() - plain.float()).abs().max() \
            <= plain.float().abs().max() * 2.0 ** -8
        return
    assert torch.equal(out, plain)
    assert torch.equal(caches[0], caches[2])
    assert torch.equal(caches[1], caches[3])


def test_other_operands_take_several_launches():
    x, w, pos, slots = _inputs(4, 4, 2, 64, 256)
    cs = build_cos_sin_table(512, 64, 1e4, device=DEV)
    kc = torch.zeros(17, 2, 16, 64, device=DEV).bfloat16()

    def go(x=x, w=w, n=(4, 2, 64), cs=cs, pos=pos, sink=(kc, kc, slots)):
        return ops.linear_rotary(x, w, *n, cs, pos, sink)

    assert go() is not None and go(sink=None) is not None
    assert go(n=(5, 2, 64)) is None                     # other heads
    assert go(n=(8, 4, 32)) is None                     # another table
    assert go(cs=cs.double()) is None
    assert go(pos=pos[:3]) is None
    assert go(x=x[:, :252], w=w[:, :252].contiguous()) is None
    assert go(w=w.float()) is None
    assert go(sink=(kc.float(), kc.float(), slots)) is None
    assert go(sink=(kc, kc[:16], slots)) is None
    assert go(sink=(kc[:, :1], kc[:, :1], slots)) is None
    wide = torch.randn(129, 256, device=DEV).bfloat16()
    assert go(x=wide, pos=pos.repeat(33)[:129], sink=None) is None


def test_a_model_with_hooks_calls_its_modules():
    from llmlb_amd.models.llama import LlamaConfig, LlamaForCausalLM
    model = LlamaForCausalLM(LlamaConfig.tiny(), device=DEV)
    h = model.embed_tokens(torch.arange(5, device=DEV))
    pos = torch.arange(5, device=DEV)
    with torch.inference_mode():
        before = model.layer_attn_prelude(0, h.clone(), None, pos)
        seen = []
        model.layers_[0].qkv.register_forward_hook(
            lambda *a: seen.append(a[2].shape))
        after = model.layer_attn_prelude(0, h.clone(), None, pos)
    assert seen
    for a, b in zip(before, after):
        assert (a.float() - b.float()).norm() <= 0.01 * b.float().norm()
