"""Decode attention over pages on the matrix cores (page_attention.hip)
against the same attention in 64 bits, at the edges of pages, pairs of
pages, parts and tiles of heads."""
import pytest
import torch

import llmlb_amd.ops as ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LENS = [1, 2, 15, 16, 17, 31, 32, 33, 127, 128, 129, 255, 257, 512, 513, 1100]


def _exact(q, k, v, bt, lens, scale):
    """(result, error that float sums and one rounding to bf16 may add)"""
    out, bound = [], []
    for s, n in enumerate(lens.tolist()):
        pages = bt[s, :-(-n // 16)].long()
        ks, vs = (t[pages].double().transpose(0, 1).flatten(1, 2)[:, :n]
                  for t in (k, v))                      # [G, n, D]
        qs = q[s].double().view(ks.shape[0], -1, q.shape[-1])
        p = torch.softmax(qs @ ks.transpose(1, 2) * scale, -1)
        out.append((p @ vs).flatten(0, 1))
        # scores are off by about 2^-24 of the sum of magnitudes, weights
        # by as much and by 2^-17 where they enter the product
        off = (qs.abs() @ ks.abs().transpose(1, 2)).amax(-1, keepdim=True) \
            * scale * 2.0 ** -22 + 2.0 ** -16
        bound.append(((p @ vs.abs()) * off).flatten(0, 1))
    out, bound = torch.stack(out), torch.stack(bound)
    return out, bound + out.abs() * 2.0 ** -8


def _case(heads, kv, D, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    lens = torch.tensor(LENS, dtype=torch.int32, device=DEV)
    per = [-(-n // 16) for n in LENS]
    ids = torch.randperm(sum(per), generator=g, device=DEV).int() + 1
    bt = torch.zeros(len(LENS), 80, dtype=torch.int32, device=DEV)
    at = 0
    for s, n in enumerate(per):
        bt[s, :n] = ids[at:at + n]
        at += n
    wide = torch.randn(len(LENS), heads * D + 64, generator=g,
                       device=DEV).bfloat16()
    q = wide[:, 64:].unflatten(1, (heads, D))     # rows of a wider matrix
    k, v = torch.randn(2, sum(per) + 1, kv, 16, D, generator=g, device=DEV)
    return q, k, v, bt, lens, per


@pytest.mark.parametrize("parts", [None, 1, 3, 16])
@pytest.mark.parametrize("heads,kv,D", [(4, 4, 128), (32, 8, 128),
                                        (14, 2, 64), (16, 1, 64),
                                        (34, 2, 128)])
def test_page_attention(heads, kv, D, parts):
    q, k, v, bt, lens, per = _case(heads, kv, D, heads + D)
    k, v = k.bfloat16(), v.bfloat16()
    ref, bound = _exact(q, k, v, bt, lens, D ** -0.5)
    # what an earlier sequence left behind a sequence's end is not read
    for s, n in enumerate(LENS):
        if n % 16:
            k[bt[s, per[s] - 1].long(), :, n % 16:] = float("nan")
            v[bt[s, per[s] - 1].long(), :, n % 16:] = float("nan")
    out = ops.paged_attn_decode(q, k, v, bt, lens, D ** -0.5, n_parts=parts)
    assert ((out.double() - ref).abs() <= bound).all()


@pytest.mark.parametrize("shift,gap", [(4, 0), (0, 4), (1, 3)])
@pytest.mark.parametrize("D", [64, 128])
def test_queries_of_any_alignment(D, shift, gap):
    q, k, v, bt, lens, _ = _case(8, 2, D, 5)
    k, v = k.bfloat16(), v.bfloat16()
    n = 8 * D
    rows = torch.zeros(len(LENS), shift + n + gap, device=DEV).bfloat16()
    rows[:, shift:shift + n] = q.flatten(1)
    loose = rows[:, shift:shift + n].unflatten(1, (8, D))
    assert loose.stride(0) % 8 or loose.data_ptr() % 16
    want = ops.paged_attn_decode(q, k, v, bt, lens, D ** -0.5)
    assert torch.equal(
        ops.paged_attn_decode(loose, k, v, bt, lens, D ** -0.5), want)


@pytest.mark.parametrize("parts", [1, 4])
@pytest.mark.parametrize("heads,kv", [(32, 8), (16, 1)])
def test_page_attention_fp8(heads, kv, parts):
    q, k, v, bt, lens, per = _case(heads, kv, 128, heads)
    caches, scales, wide = [], [], []
    for t in (k, v):
        s = torch.rand(t.shape[:3], device=DEV) * 0.01 + 0.001
        b = (t / s[..., None]).clamp(-448, 448).to(torch.float8_e4m3fn)
        wide.append(b.double() * s[..., None].double())
        caches.append(b.view(torch.uint8))
        scales.append(s)
    ref, bound = _exact(q, *wide, bt, lens, 128 ** -0.5)
    for s, n in enumerate(LENS):
        if n % 16:
            page = bt[s, per[s] - 1].long()
            for c, sc in zip(caches, scales):
                c[page, :, n % 16:] = 0x7F              # not a number
                sc[page, :, n % 16:] = float("nan")
    out = ops.paged_attn_decode(q, *caches, bt, lens, 128 ** -0.5,
                                n_parts=parts, k_scale=scales[0],
                                v_scale=scales[1])
    assert ((out.double() - ref).abs() <= bound).all()


def test_no_tokens_give_zeros():
    q, k, v, bt, lens, _ = _case(8, 2, 128, 3)
    out = ops.paged_attn_decode(q, k.bfloat16(), v.bfloat16(), bt,
                                torch.zeros_like(lens), 0.1)
    assert (out == 0).all()


@pytest.mark.parametrize("fp8", [False, True], ids=["bf16", "fp8"])
@pytest.mark.parametrize("D", [64, 128])
def test_weights_are_floats(D, fp8):
    """Pairs of keys whose weights differ by 2^-12 and whose values cancel,
    beside one that takes the rest: what is left shows the weights' last
    bits.  exp2, the scores, two scalings and the sums are good to about
    2^-24 each, eight such together; weights of 16 bits would be off by
    2^-18."""
    if fp8 and D == 64:
        pytest.skip("8-bit caches have heads of 128")
    S, lo = 64, 2.0 ** -12
    lens = torch.full((S,), 3, dtype=torch.int32, device=DEV)
    bt = torch.arange(S, dtype=torch.int32, device=DEV)[:, None]
    q = torch.zeros(S, 16, D, device=DEV)
    q[..., 0] = torch.linspace(-1.5, -0.1, S, device=DEV)[:, None]
    q[..., 1], q[..., 2] = 1.0, lo
    k, v = torch.zeros(2, S, 1, 16, D, device=DEV)
    k[:, :, :2, 0], k[:, :, 1, 2] = 1.0, 1.0
    v[:, :, 0], v[:, :, 1] = 1.0, -1.0
    q = q.bfloat16()
    scales = {}
    if fp8:
        ones = torch.ones(S, 1, 16, device=DEV)
        scales = dict(k_scale=ones, v_scale=ones)
        caches = [t.to(torch.float8_e4m3fn).view(torch.uint8)
                  for t in (k, v)]
    else:
        caches = [t.bfloat16() for t in (k, v)]
    out = ops.paged_attn_decode(q, *caches, bt, lens, 1.0, **scales)
    ref, _ = _exact(q, k, v, bt, lens, 1.0)
    bound = ref.abs() * 2.0 ** -8 + 8 * 2.0 ** -24
    assert ((out.double() - ref).abs() <= bound).all()


# one part of eight waves (144 and 256 workgroups) or two of four (128 and
# 320), of sequences with fewer pages than waves and with more; 400: one, but
# two of bf16 heads of 128
@pytest.mark.parametrize("kv", [8, 9, 16, 20, 25])
@pytest.mark.parametrize("D", [64, 128])
def test_two_parts(kv, D):
    q, k, v, bt, lens, _ = _case(2 * kv, kv, D, kv + D)
    k, v = k.bfloat16(), v.bfloat16()
    ref, bound = _exact(q, k, v, bt, lens, D ** -0.5)
    out = ops.paged_attn_decode(q, k, v, bt, lens, D ** -0.5, n_parts=2)
    assert ((out.double() - ref).abs() <= bound).all()
    if D == 128:
        test_page_attention_fp8(2 * kv, kv, 2)


# A wave looks up the pages of 32 pairs at a time: tokens just before, at and behind
# its second and third look, 4096 apart for four waves and 8192 for eight (144
# workgroups that would be two parts); the first waves look, and the others do not
@pytest.mark.parametrize("D,fp8", [(64, False), (128, False), (128, True)])
@pytest.mark.parametrize("kv,parts,lens", [
    (1, 1, [4096, 4097, 4129, 4225, 4240, 8190, 8193, 8400, 40]),
    (2, 1, [12289, 3, 5000]), (16, 2, [8192, 8193, 8450, 70, 1, 16385, 300, 33,
                                       9000]),
    (1, 3, [12288, 12289, 12400, 24577])])
def test_pages_of_long_sequences(D, fp8, kv, parts, lens):
    heads = 2 * kv
    g = torch.Generator(device=DEV).manual_seed(D + kv)
    per = [-(-n // 16) for n in lens]
    ids = torch.randperm(sum(per), generator=g, device=DEV).int() + 1
    bt = torch.zeros(len(lens), max(per) + 3, dtype=torch.int32, device=DEV)
    for s, part in enumerate(ids.split(per)):
        bt[s, :per[s]] = part
    shape = (sum(per) + 1, kv, 16, D)
    q = torch.randn(len(lens), heads, D, generator=g, device=DEV).bfloat16()
    caches, scales, wide = [], [], []
    for _ in range(2):
        t = torch.randn(shape, generator=g, device=DEV)
        if fp8:
            s = torch.rand(shape[:3], generator=g, device=DEV) * 0.01 + 0.001
            t = (t / s[..., None]).clamp(-448, 448).to(torch.float8_e4m3fn)
            wide.append(t.float() * s[..., None])
            caches.append(t.view(torch.uint8))
            scales.append(s)
        else:
            caches.append(t.bfloat16())
            wide.append(caches[-1])
    n = torch.tensor(lens, dtype=torch.int32, device=DEV)
    ref, bound = _exact(q, *wide, bt, n, D ** -0.5)
    for s, tokens in enumerate(lens):           # nothing behind the end is read
        if tokens % 16:
            page = bt[s, per[s] - 1].long()
            for c in caches:
                c[page, :, tokens % 16:] = 0x7F if fp8 else float("nan")
            for c in scales:
                c[page, :, tokens % 16:] = float("nan")
    more = dict(k_scale=scales[0], v_scale=scales[1]) if fp8 else {}
    out = ops.paged_attn_decode(q, *caches, bt, n, D ** -0.5, n_parts=parts,
                                **more)
    assert ((out.double() - ref).abs() <= bound).all()
