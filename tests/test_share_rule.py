"""In how many shares a product is taken whose shares a norm adds up: the rule is
the host's, and needs no GPU."""
import ctypes

import pytest
import torch

import llmlb_amd.ops as ops

pytestmark = pytest.mark.skipif(not ops.native_available(),
                                reason="kernels are not built")


def shares(N, M, K, plan="joined"):
    return getattr(ops._lib, f"ll_row_gemm_{plan}")(
        *(ctypes.c_int(n) for n in (N, M, K)))


def workgroups(N, M, n):
    """Of tiles of 64 outputs where they are enough, else of 32."""
    for outputs in (64, 32):
        few = -(-M // 32) * 2 * n <= 256
        blocks = -(-M // outputs) * n * (2 if N > 64 or (N > 32 and few)
                                         else 1)
        if outputs == 32 or blocks >= 176:
            return blocks


@pytest.mark.parametrize("K", [2816, 3072, 4096, 4104, 6144, 12288, 28672])
def test_one_round_of_workgroups(K):
    """Where the norm's adding up alone makes shares gain, a second round of
    workgroups on 256 compute units would cost more."""
    for N in (1, 8, 12, 16, 17, 32, 33, 48, 64, 65, 96, 128):
        for M in range(768, 4097, 4):
            n = shares(N, M, K)
            if n > 1 and shares(N, M, K, "shares") == 1:
                assert workgroups(N, M, n) <= 256, (N, M, K, n)


# rows, outputs, depth; on both sides of every line
@pytest.mark.parametrize("N, M, K, n", [
    (1, 1024, 2808, 1), (1, 1024, 2816, 4), (64, 1536, 2816, 4),
    (64, 2048, 2816, 1), (64, 2048, 3072, 4), (65, 2048, 2816, 2),
    (65, 2048, 4104, 4), (65, 1024, 2816, 4), (97, 1280, 6400, 2),
    (65, 1280, 6400, 1), (36, 1280, 4096, 1), (36, 1280, 4608, 4),
    (49, 1280, 4096, 4), (36, 1408, 4096, 4),
    (64, 2560, 4096, 2), (64, 2560, 8000, 2), (65, 2560, 4096, 1),
    (64, 4096, 3064, 1), (64, 4096, 3072, 2), (64, 4096, 4096, 2),
    (48, 4096, 6144, 4), (65, 4096, 4088, 1), (65, 4096, 4096, 2),
    (11, 4096, 6144, 1), (12, 4096, 6144, 2), (16, 4096, 12288, 4),
    (8, 4096, 14336, 1), (64, 764, 4096, 1), (64, 4100, 4096, 1),
    (64, 2046, 4096, 1), (129, 2048, 4096, 1), (0, 2048, 4096, 1)])
def test_lines(N, M, K, n):
    assert shares(N, M, K) == n


@pytest.mark.parametrize("K", [64, 2816, 4104, 24576])
@pytest.mark.parametrize("joined", [True, False])
def test_kept_counts_are_the_rule(K, joined):
    for N in (1, 16, 33, 64, 128):
        for M in (764, 1024, 2048, 4096):
            want = shares(N, M, K, "joined" if joined else "shares")
            for _ in range(2):
                assert ops._share_count(N, M, K, joined) == want


@pytest.mark.parametrize("rows, dtype, asked", [
    (128, torch.bfloat16, True), (129, torch.bfloat16, False),
    (5, torch.float32, False)])
def test_prompts_and_floats_are_not_asked(monkeypatch, rows, dtype, asked):
    """Their products never come in shares, and asking each sublayer costs a
    step that waits for the host 3% of its time."""
    from llmlb_amd.models import mixers

    class Part(mixers.Projected):
        def __init__(self):
            super().__init__()
            self.w_o = mixers._param(torch.ones(8, 8, dtype=dtype))

        def before(self, x):
            return x

    seen = []
    monkeypatch.setattr(mixers, "linear_shares",
                        lambda *a, **k: seen.append(1))
    part, x = Part(), torch.ones(rows, 8, dtype=dtype)
    call = mixers.for_norm(part) if mixers.few_rows(rows, dtype) else part
    assert torch.equal(call(x), x * 8) and len(seen) == asked
