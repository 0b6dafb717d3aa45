"""What the delta rule takes of a packed batch (convolutions, unit norms,
decays), whose tokens are walked four at a time, against float64."""
import pytest
import torch
import torch.nn.functional as F

from llmlb_amd.ops import _ptr, _stream
from llmlb_amd.ops import hybrid as hy

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# lengths of sequences that begin before, at and behind a group of four and
# the 16 tokens of a workgroup; positions within and past the taps
SEQUENCES = [(1, 0), (2, 7), (3, 0), (4, 1), (5, 2), (16, 3), (17, 0), (31, 4),
             (1, 2), (7, 0)]


def _wants(proj, b_off, dec, ring, w, a_log, bias, KH, H, D, V, taps):
    """q, k, decays, v, beta of every token."""
    C, rows = 2 * KH * D + H * V, []
    t = 0
    for slot, (n, pos) in enumerate(SEQUENCES):
        past = [ring[slot, (pos - b) % taps] if pos - b >= 0
                else torch.zeros(C, dtype=torch.float64)
                for b in range(taps - 1, 0, -1)]
        x = torch.cat([torch.stack(past), proj[t:t + n, :C]])
        rows.append(sum(x[b:b + n] * w[b] for b in range(taps)))
        t += n
    y = torch.cat(rows)
    y = y * torch.sigmoid(y)
    q, k = (y[:, i * KH * D:][:, :KH * D].reshape(t, KH, D) for i in (0, 1))
    q, k = (z / (z.square().sum(-1, keepdim=True) + 1e-6).sqrt()
            for z in (q, k))
    rate = a_log.exp().repeat_interleave(D)
    return (q * D ** -0.5, k, (-rate * F.softplus(dec + bias)).exp(),
            y[:, 2 * KH * D:], torch.sigmoid(proj[:, b_off:b_off + H]))


# 32 lanes a head (128, 256) and 16, whole vectors and not, fewer taps; the
# last heads of a workgroup are not there
@pytest.mark.parametrize("KH, H, D, V", [(3, 6, 128, 72), (9, 9, 256, 128),
                                         (3, 3, 64, 64), (17, 17, 24, 20),
                                         (2, 4, 100, 36), (1, 1, 200, 8)])
@pytest.mark.parametrize("taps", [2, 4])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32],
                         ids=["bf16", "fp32"])
def test_delta_prep(KH, H, D, V, taps, dtype):
    g = torch.Generator().manual_seed(D + taps)
    T, C = sum(n for n, _ in SEQUENCES), 2 * KH * D + H * V
    b_off = C + -C % 8
    ld = b_off + H + -H % 8

    def rand(*shape):
        return torch.randn(shape, generator=g).to(dtype)

    proj, dec = rand(T, ld), rand(T, H * D) * 4
    ring, w = rand(len(SEQUENCES), taps, C), rand(taps, C).float()
    a_log, bias = rand(H).float(), rand(H * D).float()
    pos, row, start, t = [], [], [], 0
    for slot, (n, first) in enumerate(SEQUENCES):
        pos += range(first, first + n)
        row += [slot] * n
        start += [t] * n
        t += n
    wants = _wants(*(z.double() if torch.is_tensor(z) else z for z in (
        proj, b_off, dec, ring, w, a_log, bias)), KH, H, D, V, taps)
    on = [z.to(DEV) for z in (proj, dec, ring, w, a_log, bias)]
    at = [torch.tensor(z, dtype=torch.int32, device=DEV)
          for z in (pos, row, start)]
    lib, sizes = hy.native(), [hy._i(n) for n in (KH, H, D, V)]
    ws = torch.full((T, int(lib.hy_delta_ws_floats(*sizes))), 7.0, device=DEV)
    assert lib.hy_delta_prep(
        _ptr(ws), _ptr(on[0]), hy._i(ld), hy._i(b_off), *map(_ptr, on[1:]),
        *map(_ptr, at), hy._i(T), *sizes, hy._i(taps), hy._f(D ** -0.5),
        hy._dt(dtype), _stream()) == 0
    ws = ws.double().cpu()
    q, k, decay, v, beta = wants
    first = 0
    for want in (q.flatten(1), k.flatten(1), decay, v,
                 (q * k).sum(-1), beta):
        got = ws[:, first:first + want.shape[1]]
        first += want.shape[1]
        # a few roundings to 24 bits each, of terms no larger than 30; the
        # hardware's exponential and logarithm are off by 2^-22 of themselves,
        # an exponent of up to 90 by 90 * 2^-23
        assert (got - want).abs().max() <= 2.0 ** -16 * max(
            1.0, want.abs().max())
        assert (got - want).norm() <= 1e-6 * want.norm()


def _place(tokens, sequences):
    """pos, row and first token of each, of equal sequences."""
    at = torch.arange(tokens, dtype=torch.int32, device=DEV)
    row = at // (tokens // sequences)
    first = row * (tokens // sequences)
    return at - first, row, first


def _prep(proj, dec, ring, where, w, a_log, bias, size, taps):
    ws = torch.full((len(proj), int(hy.native().hy_delta_ws_floats(
        *map(hy._i, size)))), float("nan"), device=DEV)
    pos, row, first = where
    assert hy.native().hy_delta_prep(
        _ptr(ws), _ptr(proj), hy._i(proj.stride(0)),
        hy._i(2 * size[0] * size[2] + size[1] * size[3]), _ptr(dec),
        _ptr(ring), _ptr(w), _ptr(a_log), _ptr(bias), _ptr(pos), _ptr(row),
        _ptr(first), hy._i(len(proj)), *map(hy._i, size), hy._i(taps),
        hy._f(0.1), hy._dt(proj.dtype), _stream()) == 0
    return ws


# 4100 tokens of 16 and 32 heads of 128 write more than 128 and 256 MB, whose
# workgroups are in another order than those of the sequences one by one
@pytest.mark.parametrize("heads, dtype", [(32, torch.bfloat16),
                                          (16, torch.float32)])
def test_many_tokens(heads, dtype):
    T, n, taps, size = 4100, 4, 4, (heads, heads, 128, 128)
    g = torch.Generator(device=DEV).manual_seed(heads)

    def rand(*shape):
        return torch.randn(shape, generator=g, device=DEV)

    C = 3 * heads * 128
    proj, dec = rand(T, C + heads).to(dtype), rand(T, heads * 128).to(dtype)
    ring = rand(n, taps, C).to(dtype)
    rest = rand(taps, C), rand(heads), rand(heads * 128), size, taps
    got = _prep(proj, dec, ring, _place(T, n), *rest)
    each = T // n
    for s in range(n):
        part = slice(s * each, (s + 1) * each)
        want = _prep(proj[part], dec[part], ring[s:s + 1], _place(each, 1),
                     *rest)
        used = 3 * heads * 128 + heads * 128 + 2 * heads
        assert torch.equal(got[part, :used], want[:, :used])
        assert not want[:, :used].isnan().any()


# 11000 tokens of 6144 channels are more than 256 MB read and written
@pytest.mark.parametrize("T", [11000, 1000])
def test_state_space_convolution(T):
    C, H, n, taps, dtype = 6144, 8, 4, 4, torch.bfloat16
    g = torch.Generator(device=DEV).manual_seed(T)
    proj = torch.randn(T, C + H, generator=g, device=DEV).to(dtype)
    ring = torch.randn(n, taps, C, generator=g, device=DEV).to(dtype)
    w = torch.randn(taps, C, generator=g, device=DEV)
    b = torch.randn(C, generator=g, device=DEV)
    heads = torch.randn(3, H, generator=g, device=DEV)

    def prep(proj, ring, where):
        out = torch.full((len(proj), C), float("nan"), dtype=dtype,
                         device=DEV)
        assert hy.native().hy_ssm_prep(
            _ptr(out), None, _ptr(proj), hy._i(C + H), hy._i(C), _ptr(ring),
            _ptr(w), _ptr(b), _ptr(heads), *map(_ptr, where),
            hy._i(len(proj)), hy._i(C), hy._i(H), hy._i(taps), hy._i(0),
            _stream()) == 0
        return out

    got, each = prep(proj, ring, _place(T, n)), T // n
    for s in range(n):
        part = slice(s * each, (s + 1) * each)
        want = prep(proj[part], ring[s:s + 1], _place(each, 1))
        assert torch.equal(got[part], want)
        assert not want.isnan().any()


# more than 256 MB read and written, in whole parts of rows and not, and less
@pytest.mark.parametrize("T, C", [(11000, 4096), (11000, 4104), (9000, 6144),
                                  (300, 4096), (70, 2050)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_gated_linear_decays(T, C, dtype):
    g = torch.Generator(device=DEV).manual_seed(C)
    dec = torch.randn(T, C, generator=g, device=DEV).to(dtype) * 3
    bias = torch.randn(C, generator=g, device=DEV)
    out = torch.full((T, C), float("nan"), device=DEV)
    assert hy.native().hy_gla_decay(
        _ptr(out), _ptr(dec), _ptr(bias), hy._i(T), hy._i(C),
        hy._f(1 / 16), hy._dt(dtype), _stream()) == 0
    want = torch.sigmoid(dec.double() + bias.double()) ** (1 / 16)
    # the sum, a logarithm and an exponential in 24 bits; the hardware's are off
    # by 2^-22 of themselves, and a sixteenth of the logarithm is at most one
    assert (out.double() - want).abs().max() <= 2.0 ** -20
