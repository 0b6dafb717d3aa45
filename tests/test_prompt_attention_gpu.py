"""Prompt attention of the Llama family (flash_attention.hip) against 64
bits, at the edges of its tiles of queries and keys."""
import pytest
import torch

import llmlb_amd.ops as ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _check(q, k, v, scale):
    B, Lq, H, D = q.shape
    Lk, G = k.shape[1:3]
    out = ops.prompt_attention(q, k, v, scale)
    assert out.shape == (B * Lq, H, D) and out.is_contiguous()
    qd, kd, vd = (t.double().transpose(1, 2) for t in (q, k, v))
    kd, vd = (t.repeat_interleave(H // G, 1) for t in (kd, vd))
    at = torch.arange(Lk, device=DEV)
    s = (qd @ kd.transpose(2, 3) * scale).masked_fill(
        at[None] > at[Lk - Lq:, None], -float("inf"))
    p = torch.softmax(s, -1)
    ref = (p @ vd).transpose(1, 2).reshape(out.shape)
    # weights enter the second product rounded to bf16 (2^-9 each), scores
    # are float sums of D products, the result is rounded once
    off = 2.0 ** -8 + (qd.abs() @ kd.abs().transpose(2, 3)).amax() \
        * scale * D * 2.0 ** -24
    bound = (p @ vd.abs() * off).transpose(1, 2).reshape(out.shape) \
        + ref.abs() * 2.0 ** -8
    assert ((out.double() - ref).abs() <= bound + 1e-30).all()


@pytest.mark.parametrize("H,G,D", [(4, 4, 128), (8, 2, 128), (14, 2, 64),
                                   (6, 6, 64), (128, 1, 64)])
@pytest.mark.parametrize("B,Lq,Lk", [(1, 1, 1), (3, 5, 5), (1, 63, 64),
                                     (2, 65, 65), (9, 33, 200),
                                     (1, 128, 1000), (2, 300, 300),
                                     (1, 700, 700)])
def test_prompt_attention(B, Lq, Lk, H, G, D):
    g = torch.Generator(device=DEV).manual_seed(B + Lq + H)
    # rows of a wider matrix, as the stacked projection leaves them
    wide = torch.randn(B, Lk, (H + 2 * G) * D + 8, generator=g,
                       device=DEV).bfloat16()
    q, k, v = wide[:, :, 8:].split([H * D, G * D, G * D], 2)
    q = q[:, Lk - Lq:].unflatten(2, (H, D))
    k, v = (t.unflatten(2, (G, D)) for t in (k, v))
    assert ops.prompt_attn_tiled(q, k, v)
    _check(q, k, v, D ** -0.5)


@pytest.mark.parametrize("shift", [-300.0, 0.0, 40.0])
def test_maximum_that_moves(shift):
    """Scores that rise along the keys, far below and above zero: the
    running maximum has to follow, and its first value to be the row's."""
    g = torch.Generator(device=DEV).manual_seed(3)
    B, L, H, D = 1, 400, 4, 128
    q = torch.randn(B, L, H, D, generator=g, device=DEV)
    k, v = torch.randn(2, B, L, H, D, generator=g, device=DEV)
    q[..., 0] = 8.0
    k[..., 0] = (torch.arange(L, device=DEV)[None, :, None] * 0.25 + shift)
    _check(q.bfloat16(), k.bfloat16(), v.bfloat16(), D ** -0.5)


def test_other_sizes_go_to_the_library():
    q = torch.randn(2, 20, 4, 96, device=DEV).bfloat16()
    k = torch.randn(2, 30, 2, 96, device=DEV).bfloat16()
    assert not ops.prompt_attn_tiled(q, k, k)
    _check(q, k, k, 0.1)
