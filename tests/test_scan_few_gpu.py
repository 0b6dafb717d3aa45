"""The scan of few sequences in 32 bits at the edges of its blocks of 16
tokens, with 1 to 8 rows of the state a lane."""
import pytest
import torch

import rasodra_util as R
import taletar_util as U

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
F32 = torch.float32
# after which the sequence goes on: whole blocks, one token less and more
CUTS = [1, 3, 18, 34, 49, 64, 81, 112, 145, 176]


def check(got, want):
    # T steps of a decaying sum of D products each: 5e-5 of the largest, as
    # the same recurrences are tested with elsewhere
    err = (got.double() - want).abs().max() / want.abs().max()
    assert err < 5e-5, float(err)


@pytest.mark.parametrize("ly", [
    U.gla(2, 16, 16), U.gla(8, 32, 48), U.gla(3, 64, 64), U.gla(2, 128, 16),
    U.mamba2(2, 16, 16), U.mamba2(8, 48, 32, 2), U.mamba2(3, 64, 64),
    U.mamba2(4, 16, 128, 2)], ids=str)
def test_edges(ly):
    width = 48
    oracle, m, w = U.case(ly, width, 3)
    h = U.inputs(CUTS[-1], width, 2)
    run = U.MixerRun(U.mixer(ly["type"], m, w, 1e-4, width, DEV, F32), 2,
                     len(h))
    for cuts in ([], CUTS[:-1]):
        run.restart(1)
        check(run.cuts(1, h, cuts), oracle(h, w, "", m, 1e-4))


@pytest.mark.parametrize("ly", [
    R.memory(2, 16, 16), R.memory(8, 32, 48), R.memory(3, 64, 64, cap=4.0),
    R.memory(2, 128, 16)], ids=str)
def test_memory_edges(ly):
    op = R.memory_op(ly, 3, DEV, F32)
    x = op.rows(CUTS[-1], 2)
    run = R.MixerRun(op, 2, len(x))
    for cuts in ([], CUTS[:-1]):
        run.restart(1)
        check(run.cuts(1, x, cuts), op.oracle(x))


def test_unequal_lengths_together():
    """Entries end in different blocks, and in different places of them."""
    width = 40
    ly = U.gla(4, 64, 32)
    oracle, m, w = U.case(ly, width, 1)
    hs = [U.inputs(n, width, n) for n in (16, 1, 33, 47)]
    run = U.MixerRun(U.mixer(ly["type"], m, w, 1e-5, width, DEV, F32), 4, 64)
    got = run.step(list(enumerate(hs)))
    for i, h in enumerate(hs):
        check(got[i], oracle(h, w, "", m, 1e-5))


# 512, 1024 and 1984 waves of the 2047 at most
@pytest.mark.parametrize("kind", ["channel", "head", "memory"])
@pytest.mark.parametrize("E, H, D, V", [(3, 2, 16, 16), (2, 16, 64, 64),
                                        (4, 8, 128, 128), (31, 16, 32, 16)])
def test_sixteen_bits(kind, E, H, D, V):
    """The same numbers in either type: all sums are of floats in the same
    order, but a product may be rounded before it is added or not, 33 + D
    times 2^-24 at most, 1e-5."""
    from llmlb_amd.ops import hybrid as hy
    from llmlb_amd.ops.hybrid import _f, _i, _p, _ptr, _stream
    g = torch.Generator(device=DEV).manual_seed(D + E)
    rand = lambda *s: torch.rand(*s, generator=g, device=DEV)
    lens = [(1, 15, 16, 17, 33)[i % 5] for i in range(E)]
    T, ld = sum(lens), 2 * H * D + H * V
    rows = (2 * rand(T, ld) - 1).bfloat16()
    decay = 0.9 + 0.1 * rand(T, H * (D if kind == "channel" else 1))
    dt = None if kind == "channel" else rand(T, H)
    skip = None if kind == "channel" else 0.5 + rand(T, H)
    n0 = rand(E, H, D) if kind == "memory" else None
    ints = lambda l: torch.tensor(l, dtype=torch.int32, device=DEV)
    runs = (ints([sum(lens[:i]) for i in range(E)]), ints(lens),
            ints([i % 2 for i in range(E)]), ints(list(range(E))[::-1]))
    first = rand(E, H, V, D)
    got = []
    for x in (rows, rows.float()):
        o, state = torch.zeros(T, H * V, device=DEV), first.clone()
        extra = torch.zeros(E, H, hy.memory_extra(D), device=DEV)
        rc = hy.native().hy_linear_scan(
            _ptr(o), _ptr(state), _ptr(x), _i(ld), _i(0), _i(H * D),
            _i(2 * H * D), _ptr(decay), _p(dt), _p(skip), *map(_ptr, runs),
            _i(E), _i(H), _i(H), _i(D), _i(V), _f(D ** -0.5), _p(n0),
            _ptr(extra) if kind == "memory" else None, hy._dt(x.dtype),
            _stream())
        assert rc == 0
        got.append((o, state, extra))
    for a, b in zip(*got):
        assert (a - b).abs().max() <= 1e-5 * b.abs().max()
    assert got[0][0].abs().max() > 0
