"""Recurrences in chunks (chunk_scan.hip, the state-space part of
memory_mfma.hip) against the recurrences themselves, token by token in 64
bits."""
import pytest
import torch

from llmlb_amd.ops import hybrid as hy
from llmlb_amd.ops.hybrid import _check, _f, _i, _ptr, _stream

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
F64 = torch.float64
# All is float (the state-space part's weights and state take three bf16
# numbers each): numbers good to 2^-24, sums of up to 256 products, products
# of up to 16 decays, three such products behind each other and through the
# state.  Errors of that size add up like noise.
TOL = 2.0 ** -19


def entries(lens, resume):
    start, at = [], 0
    for n in lens:
        start.append(at)
        at += n
    pos = [5 * (resume and i % 2) for i in range(len(lens))]
    row = [len(lens) - 1 - i for i in range(len(lens))]
    return at, start, pos, row, [
        torch.tensor(x, dtype=torch.int32, device=DEV)
        for x in (start, lens, pos, row)]


def close(got, want):
    err = (got.double() - want).abs().max() / want.abs().max()
    assert err < TOL, float(err)


def run(delta, lens, G, H, D, V, logs, resume=True, reset=None):
    """logs: (lowest, highest) logarithm of two of a decay; reset: tokens
    whose decays are 2^-90 and after which inputs are 2^-20 of those before,
    for 2 tokens."""
    g = torch.Generator(device=DEV).manual_seed(sum(lens) + D + V)
    T, start, pos, row, e = entries(lens, resume)
    kind = torch.float32 if delta else torch.bfloat16
    qo, ko, vo = 0, G * D, 2 * G * D
    width = (2 * G * D + H * V + 2 * H + 15) // 8 * 8
    x = torch.randn(T, width, generator=g, device=DEV)
    if delta:
        x[:, :2 * G * D] = torch.nn.functional.normalize(
            x[:, :2 * G * D].unflatten(1, (2 * G, D)), dim=2).flatten(1)
        x[:, vo + H * V:] = x[:, vo + H * V:].sigmoid()
    lo, hi = logs
    f = (torch.rand(T, H, D, generator=g, device=DEV) * (hi - lo) + lo).neg_()
    f[:, :, ::3] *= 2.0 ** -6      # channels that remember
    for t in reset or ():
        f[t] = -90.0
        x[t:t + 3, G * D:vo + H * V] *= 2.0 ** -20      # k and v
    x = x.to(kind)
    state = torch.randn(len(lens), H, V, D, generator=g, device=DEV)
    want_S = state.double()
    o = torch.full((T, H * V), 7.0, device=DEV)
    beta = x[:, vo + H * V:] if delta else None
    want = torch.empty(T, H, V, dtype=F64, device=DEV)
    q, k = (x[:, at:at + G * D].double().view(T, G, D).repeat_interleave(
        H // G, 1) for at in (qo, ko))
    v = x[:, vo:vo + H * V].double().view(T, H, V)
    for s, n, p, r in zip(start, lens, pos, row):
        S = want_S[r] if p else torch.zeros_like(want_S[r])
        for t in range(s, s + n):
            S = S * f[t].exp2().double()[:, None]
            u = v[t]
            if delta:
                b = beta[t, :H].double()[:, None]
                u = b * (u - torch.matmul(S, k[t][:, :, None])[..., 0])
            S = S + u[:, :, None] * k[t][:, None]
            want[t] = torch.matmul(S, q[t][:, :, None])[..., 0] * 0.5
        want_S[r] = S
    _check(hy.native().hy_chunk_scan(
        _ptr(o), _ptr(state), _ptr(x), _i(width), _i(qo), _i(ko), _i(vo),
        _ptr(f.exp2()), _i(H * D), None if beta is None else _ptr(beta),
        *(_ptr(t) for t in e), _i(len(lens)), _i(G), _i(H), _i(D), _i(V),
        _f(0.5), _i(int(delta)), _stream()), "hy_chunk_scan")
    close(o.view(T, H, V), want)
    close(state, want_S)
    for t in reset or ():          # tokens of their own size
        for n in range(t, t + 3):
            close(o.view(T, H, V)[n], want[n])


@pytest.mark.parametrize("D,V", [(8, 1), (40, 24), (64, 64), (72, 70),
                                 (128, 128)])
@pytest.mark.parametrize("delta", [False, True], ids=["linear", "delta"])
def test_sizes(delta, D, V):
    run(delta, [1, 7, 8, 9, 15, 16, 17, 33, 100], 2, 4, D, V, (0.0, 0.5))


@pytest.mark.parametrize("logs", [(0.0, 2.0 ** -8), (0.0, 4.0), (3.0, 20.0),
                                  (0.0, 60.0), (200.0, 400.0)], ids=str)
@pytest.mark.parametrize("delta", [False, True], ids=["linear", "delta"])
def test_decays(delta, logs):
    run(delta, [70, 64], 2, 2, 128, 64, logs)


@pytest.mark.parametrize("delta", [False, True], ids=["linear", "delta"])
def test_resets(delta):
    """What a reset leaves of the state is nothing beside inputs however
    small: places in a chunk, in a half, quarter and pair of tokens, and the
    last of one chunk."""
    run(delta, [70, 64], 2, 2, 128, 64, (0.0, 0.1),
        reset=[5, 12, 24, 31, 47, 70 + 19, 70 + 40])


def test_repeated_keys():
    """Steps that undo each other: L is far from small."""
    D = V = 64
    T, start, pos, row, e = entries([48], False)
    x = torch.randn(T, 2 * D + V + 4, device=DEV,
                    generator=torch.Generator(device=DEV).manual_seed(1))
    x[:, :2 * D] = torch.nn.functional.normalize(x[0, :D], dim=0).repeat(2)
    x[:, 2 * D + V] = 1.0
    f = torch.ones(T, D, device=DEV)
    o = torch.empty(T, V, device=DEV)
    state = torch.zeros(1, 1, V, D, device=DEV)
    _check(hy.native().hy_chunk_scan(
        _ptr(o), _ptr(state), _ptr(x), _i(x.shape[1]), _i(0), _i(D),
        _i(2 * D), _ptr(f), _i(D), _ptr(x[:, 2 * D + V:]),
        *(_ptr(t) for t in e), _i(1), _i(1), _i(1), _i(D), _i(V), _f(1.0),
        _i(1), _stream()), "hy_chunk_scan")
    close(o, x[:, 2 * D:2 * D + V].double())   # each step forgets the last


@pytest.mark.parametrize("rate", [1e-3, 1.0, 30.0, 3e4])
@pytest.mark.parametrize("D,V", [(16, 16), (40, 72), (128, 128), (256, 24)])
def test_state_space(D, V, rate):
    G, H = 2, 4
    lens = [1, 5, 63, 64, 65, 150]
    T, start, pos, row, e = entries(lens, True)
    g = torch.Generator(device=DEV).manual_seed(D + V)
    C = H * V + 2 * G * D
    x = torch.randn(T, C, generator=g, device=DEV).bfloat16()
    dt_in = torch.randn(T, H, generator=g, device=DEV).bfloat16()
    head = torch.stack([torch.linspace(-2, 1, H), torch.full((H,), rate),
                        torch.linspace(0.1, 1, H)]).to(DEV)
    state = torch.randn(len(lens), H, V, D, generator=g, device=DEV)
    want_S = state.double()
    dt = torch.nn.functional.softplus(dt_in.double() + head[0].double(),
                                      threshold=60.0)
    v = x[:, :H * V].double().view(T, H, V)
    k, q = (x[:, at:at + G * D].double().view(T, G, D).repeat_interleave(
        H // G, 1) for at in (H * V, H * V + G * D))
    want = torch.empty(T, H, V, dtype=F64, device=DEV)
    for s, n, p, r in zip(start, lens, pos, row):
        S = want_S[r] if p else torch.zeros_like(want_S[r])
        for t in range(s, s + n):
            S = S * torch.exp(-head[1].double() * dt[t])[:, None, None] \
                + (dt[t][:, None] * v[t])[:, :, None] * k[t][:, None]
            want[t] = torch.matmul(S, q[t][:, :, None])[..., 0] \
                + head[2].double()[:, None] * v[t]
        want_S[r] = S
    o = torch.full((T, H * V), 7.0, device=DEV)
    gates = torch.empty(3, T, H, device=DEV)
    _check(hy.native().hy_ssm_chunk(
        _ptr(o), _ptr(gates), _ptr(state), _ptr(x), _i(C),
        _i(H * V + G * D), _i(H * V), _ptr(dt_in), _i(H), _i(0), _ptr(head),
        *(_ptr(t) for t in e), _i(len(lens)), _i(max(lens)), _i(T), _i(G),
        _i(H), _i(D), _i(V), _stream()), "hy_ssm_chunk")
    close(o.view(T, H, V), want)
    close(state, want_S)
