"""The decays' low-rank projection inside a decoding step's kernel: the
same step with the projection given, and the plain implementation."""
import types

import pytest
import torch

from llmlb_amd.ops import hybrid as hy
from llmlb_amd.ops import reference_hybrid as ref

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
F32, B16 = torch.float32, torch.bfloat16


def batch(n, dev):
    """The last sequence is new: its state is whatever was there."""
    pos = [5] * (n - 1) + [0]
    return types.SimpleNamespace(
        decode=True, n_tok=n, entries=[(i, 1, p, i)
                                       for i, p in enumerate(pos)],
        pos=torch.tensor(pos, dtype=torch.int32, device=dev),
        row=torch.arange(n, dtype=torch.int32, device=dev))


# heads, dim, vdim, rank: one load a lane and fewer lanes than four, a
# remainder of 32, whole ones, more channels than a pass has and fewer
@pytest.mark.parametrize("sizes", [
    (2, 16, 16, 8), (3, 11, 24, 40), (4, 64, 64, 64), (2, 100, 36, 24),
    (2, 128, 128, 128), (1, 200, 50, 136), (1, 512, 16, 32)], ids=str)
@pytest.mark.parametrize("n", [1, 5])
@pytest.mark.parametrize("dtype", [B16, F32], ids=["bf16", "f32"])
def test_projection_in_the_step(sizes, n, dtype):
    H, D, V, R = sizes
    up = lambda a: a + -a % 8
    k_off = up(H * D)
    v_off = k_off + up(H * D)
    g_off = v_off + up(H * V)
    low = g_off + up(H * V)
    g = torch.Generator().manual_seed(H + D + R)
    proj = torch.randn(n, low + R, generator=g).to(dtype)
    w = (torch.randn(H * D, R, generator=g) * R ** -0.5).to(dtype)
    bias = torch.randn(H * D, generator=g)
    norm = torch.randn(V, generator=g)
    state = torch.randn(n, H, V, D, generator=g)
    # whole sums of 64 bits, rounded once: what the projection's launch
    # returns but for sums that lie on the edge between two numbers
    dec = (proj[:, low:].double() @ w.double().t()).to(dtype)

    def run(dev, dec, fn, **more):
        out = torch.zeros(n, H * V, dtype=dtype, device=dev)
        st = state.clone().to(dev)
        fn(out, proj.to(dev), k_off, v_off, g_off, dec, bias.to(dev), st,
           batch(n, dev), norm.to(dev), H, D, V, 16.0, 1e-5, **more)
        return out.float().cpu(), st.cpu()

    wd = w.to(DEV)
    assert hy.decays_in_step(proj.to(DEV), low, wd, D, batch(n, DEV)) \
        == (D * R <= 4096)
    got, st = run(DEV, None, hy.gated_linear, low=(low, wd))
    given, st_given = run(DEV, dec.to(DEV), hy.gated_linear)
    want, st_want = run("cpu", dec, ref.gated_linear)
    # Another order of a float sum: R steps of 2^-24 of |dec| < 6, through
    # a sigmoid's power of 1/16 (slope <= 1/16) into the decays.  In
    # bfloat16 a sum may round to the neighbour, 2^-7 of |dec|.
    step = (6 * 2 ** -7 if dtype == B16 else 6 * R * 2 ** -24) / 16
    scale = state.abs().max()
    assert (st - st_given).abs().max() <= (step + 1e-6) * scale
    assert (st - st_want).abs().max() <= (step + 1e-5) * scale
    tol = (2 ** -7 if dtype == B16 else 2e-5) + 4 * step
    for other in (given, want):
        assert (got - other).abs().max() <= tol * want.abs().max()


def test_unfit_operands_keep_their_launch():
    b = batch(2, DEV)
    proj = torch.zeros(2, 64, dtype=B16, device=DEV)
    w = torch.zeros(16, 16, dtype=B16, device=DEV)
    assert hy.decays_in_step(proj, 16, w, 16, b)
    assert not hy.decays_in_step(proj, 12, w, 16, b)
    assert not hy.decays_in_step(proj[:, :60].contiguous(), 16, w, 16, b)
    assert not hy.decays_in_step(proj, 16, w[:, :12].contiguous(), 16, b)
    assert not hy.decays_in_step(proj, 16, w.float(), 16, b)
    assert not hy.decays_in_step(proj, 16, w.t(), 16, b)
    assert not hy.decays_in_step(proj, 16, w, 264, b)
    b.decode = False
    assert not hy.decays_in_step(proj, 16, w, 16, b)


@pytest.mark.parametrize("mode", ["0", "off", "1"])
def test_the_librarys_product_where_it_is_asked_for(mode, monkeypatch):
    import llmlb_amd.ops as ops
    proj = torch.zeros(2, 64, dtype=B16, device=DEV)
    w = torch.zeros(16, 16, dtype=B16, device=DEV)
    assert hy.decays_in_step(proj, 16, w, 16, batch(2, DEV))
    monkeypatch.setattr(ops, "_USE_CUSTOM_DECODE_GEMM", mode)
    assert not hy.decays_in_step(proj, 16, w, 16, batch(2, DEV))
