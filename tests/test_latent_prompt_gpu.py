"""Prompt attention over expanded latents (latent_prompt_kernel) against 64
bits."""
import pytest
import torch

from llmlb_amd.backend.ragged import RaggedBatch
from llmlb_amd.ops import hybrid as hy
from llmlb_amd.ops.hybrid import _check, _f, _i, _ptr, _stream

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# outputs and the weights before the second product are bf16 numbers
TOL = 2.0 ** -7


# portions at the start and behind others, edges of 16, 64 and 128 queries
@pytest.mark.parametrize("window", [1, 50, 200, 2 ** 30])
@pytest.mark.parametrize("sink", [None, -3.0, 40.0, -3e38, float("-inf")])
@pytest.mark.parametrize("H,D,R,V", [(3, 64, 32, 64), (2, 128, 64, 128),
                                     (5, 96, 0, 64), (1, 136, 56, 128)])
def test_latent_prompt(H, D, R, V, sink, window):
    g = torch.Generator(device=DEV).manual_seed(H + D)
    runs = [(0, 0, [1] * 9), (2, 37, [1] * 64), (1, 300, [1] * 129),
            (3, 0, [1] * 200)]
    b = RaggedBatch.build(runs, torch.zeros(4, 1, dtype=torch.int32,
                                            device=DEV))
    blocks, items, n_blocks, n_items = b.long_plan(window)
    rn = lambda *s: torch.randn(*s, generator=g, device=DEV)
    T, n, gate = b.n_tok, 64 * n_blocks, H * (D + R)
    ld = gate + H * V
    # some scores far above those before them
    proj = rn(T, ld).bfloat16()
    kx, kr = rn(n, H * D).bfloat16(), rn(n, R).bfloat16()
    kx[::41] *= 12.0
    vx = rn(n, H * V).bfloat16()
    sinks = None if sink is None else torch.full((H,), sink, device=DEV)
    scale = (D + R) ** -0.5
    gated = sink != 40.0
    out = torch.full((T, H * V), 7.0, device=DEV, dtype=torch.bfloat16)
    _check(hy.native().hy_latent_prompt(
        _ptr(out), _ptr(proj), _i(ld), _ptr(kx), _ptr(kr), _ptr(vx),
        _ptr(items), _i(n_items), _i(H), _i(D), _i(R), _i(V), _i(window),
        _f(scale), None if sinks is None else _ptr(sinks),
        _i(gate if gated else -1), _stream()), "hy_latent_prompt")
    at = 0
    for start, length, pos, row in b.entries:
        first, end = max(0, pos - window + 1), pos + length
        rows = slice(at, at + end - first)
        at += -(-(end - first) // 64) * 64
        k = torch.cat([kx[rows].double().view(-1, H, D), kr[rows].double()[
            :, None].expand(-1, H, R)], 2)
        q = proj[start:start + length, :gate].double().view(-1, H, D + R)
        s = torch.matmul(q.transpose(0, 1), k.permute(1, 2, 0).contiguous()) \
            * scale
        age = (torch.arange(pos, end, device=DEV)[:, None]
               - torch.arange(first, end, device=DEV))
        s = s.masked_fill((age < 0) | (age >= window), float("-inf"))
        if sink is not None:
            s = torch.cat([s, torch.full_like(s[..., :1], sink)], 2)
        p = torch.softmax(s, 2)[..., :end - first]
        want = torch.matmul(p, vx[rows].double().view(-1, H, V).transpose(
            0, 1).contiguous()).transpose(0, 1).reshape(length, H * V)
        if gated:
            want = want * proj[start:start + length, gate:].double().sigmoid()
        got = out[start:start + length].double()
        # weights are off by 2^-9 of themselves each, and the result by 2^-9
        off = (got - want).abs().max() / vx.double().abs().max()
        assert off < TOL, (row, float(off))
