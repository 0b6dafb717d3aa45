"""Attention of float models in float matrix products (float_rows.h) against
64 bits."""
import pytest
import torch

from llmlb_amd.ops import hybrid as hy
from llmlb_amd.ops.hybrid import _check, _f, _i, _ptr, _stream

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
F64 = torch.float64
# rows of up to 1000 keys: sums in float and one exponential's rounding
TOL = 5e-6
# All in all: a number passes about sixteen roundings (parts of a score and
# their sum, scaling, exponential, weights' and values' sums, quotient), each
# 2^-24 / sqrt(3) off.  That makes 4 / sqrt(3) * 2^-24; not more than 3.
RMS = 3 * 2.0 ** -24
PAGES, BLOCKS = 70, 64


def close(got, want):
    off = got.double() - want
    err = off.abs().max() / want.abs().max()
    assert err < TOL, float(err)
    rms = off.norm() / want.norm()
    assert rms < RMS, float(rms)


def tokens(N, g):
    pos = torch.randint(0, BLOCKS * 16, (N,), generator=g, device=DEV,
                        dtype=torch.int32)
    pos[:4] = torch.tensor([0, 15, 16, BLOCKS * 16 - 1])[:N]
    row = torch.randint(0, 3, (N,), generator=g, device=DEV,
                        dtype=torch.int32)
    tables = torch.stack([torch.randperm(PAGES, generator=g,
                                         device=DEV)[:BLOCKS]
                          for _ in range(3)]).int()
    return pos, row, tables


def attend(q, k, v, sink=None):
    """q [H, W] in powers of two; k, v [n, ...]."""
    s = q @ k.T * 0.6931471805599453
    if sink is not None:
        s = torch.cat([s, sink[:, None]], 1)
    p = torch.softmax(s, 1)
    return p[:, :len(k)] @ v


# few workgroups and many, every number of value tiles, remainders of 16
@pytest.mark.parametrize("N", [4, 70])
@pytest.mark.parametrize("H,rank,R,window,sink", [
    (16, 256, 32, 10 ** 6, False), (5, 60, 4, 37, True),
    (21, 128, 64, 200, True), (3, 512, 64, 500, False), (1, 4, 8, 1, False)])
def test_latent(N, H, rank, R, window, sink):
    g = torch.Generator(device=DEV).manual_seed(H + rank)
    D = 8
    pos, row, tables = tokens(N, g)
    rn = lambda *s: torch.randn(*s, generator=g, device=DEV)
    cache, qa = rn(PAGES, 16, rank + R), rn(H, N, rank)
    proj, ld = rn(N, H * (D + R) + 4), H * (D + R) + 4
    sinks = rn(H) if sink else None
    scale = (rank + R) ** -0.5
    out = torch.full_like(qa, 7.0)
    _check(hy.native().hy_latent_rows(
        _ptr(out), _ptr(qa), _ptr(proj), _i(ld), _i(H), _i(D), _i(R),
        _i(rank), _ptr(cache), _ptr(pos), _ptr(row), _ptr(tables),
        _i(BLOCKS), _i(window), _f(scale),
        None if sinks is None else _ptr(sinks), _i(N), _i(1), _stream()),
        "hy_latent_rows")
    want = torch.empty(H, N, rank, dtype=F64, device=DEV)
    for t in range(N):
        keys = cache[tables[row[t]].long()].double().flatten(0, 1)
        keys = keys[max(0, int(pos[t]) - window + 1):int(pos[t]) + 1]
        q = torch.cat([qa[:, t], proj[t, :H * (D + R)].view(H, D + R)[:, D:]],
                      1).double() * (scale * 1.4426950408889634)
        want[:, t] = attend(q, keys, keys[:, :rank],
                            None if sinks is None else sinks.double())
    close(out, want)


@pytest.mark.parametrize("N", [4, 70])
@pytest.mark.parametrize("H,G,D,V,window,chunk,gate", [
    (16, 4, 64, 64, 10 ** 6, 0, False), (20, 1, 20, 68, 100, 0, True),
    (6, 2, 132, 4, 64, 1, True), (4, 4, 16, 300, 17, 0, False),
    (3, 1, 256, 512, 300, 1, False)])
def test_window(N, H, G, D, V, window, chunk, gate):
    g = torch.Generator(device=DEV).manual_seed(H + D + V)
    pos, row, tables = tokens(N, g)
    rn = lambda *s: torch.randn(*s, generator=g, device=DEV)
    cache = rn(PAGES, G, 16, D + V)
    proj, ld = rn(N, H * D + H), H * D + H
    proj[:, :H * D] *= D ** -0.5
    wide = torch.full((N, H * V + 8), 7.0, device=DEV)
    out = wide[:, 4:4 + H * V]
    _check(hy.native().hy_window_rows(
        _ptr(out), _i(wide.shape[1]), _ptr(proj), _i(ld),
        _i(H * D if gate else -1), _ptr(cache), _ptr(pos), _ptr(row),
        _ptr(tables), _i(BLOCKS), _i(H), _i(G), _i(D), _i(V), _i(window),
        _i(chunk), _i(N), _i(1), _stream()), "hy_window_rows")
    want = torch.empty(N, H, V, dtype=F64, device=DEV)
    for t in range(N):
        p = int(pos[t])
        first = p // window * window if chunk else max(0, p - window + 1)
        rows = cache[tables[row[t]].long()].double()
        for kv in range(G):
            kvs = rows[:, kv].flatten(0, 1)[first:p + 1]
            hs = slice(kv * (H // G), (kv + 1) * (H // G))
            want[t, hs] = attend(proj[t, :H * D].double().view(H, D)[hs],
                                 kvs[:, :D], kvs[:, D:])
    if gate:
        want *= proj[:, H * D:].double().sigmoid()[:, :, None]
    close(out.reshape(N, H, V), want)
    assert (wide[:, :4] == 7).all() and (wide[:, 4 + H * V:] == 7).all()
