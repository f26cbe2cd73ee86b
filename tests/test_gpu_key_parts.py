"""Range forward and dQ with a row group's keys in parts (launches of few
workgroups), against the float64 oracle: lengths whose grids take 1, 2 and 4
parts (test_part_counts.py holds them to that), key counts that leave parts
without a tile or with a ragged one, rows without any key, every head dim, flat
rows and head chunks; one sequence alone and in a batch whose launch takes
another part count; and the finishing layer against the same launches by
branch."""

import pytest
import torch

from oracle import nsa_oracle as O
from nsa_testlib import assert_close, log, make_block_idx, randn, require_gpu, to64

pytestmark = pytest.mark.gpu
BF, F32 = torch.bfloat16, torch.float32

# T, window, l, d
SIZES = [(40, 200, 16, 8), (129, 97, 16, 16), (1000, 130, 32, 16), (2500, 512, 64, 64)]
HEADS = [(4, 1, 16), (5, 1, 32), (12, 2, 64), (16, 1, 64), (16, 1, 128), (20, 1, 128), (64, 4, 128)]


def case_sizes(size, heads):
    """The case's sizes with T cut down for the oracle."""
    T, window, l, d = size
    return (600 if heads[0] * T > 50000 else T), window, l, d


@pytest.mark.parametrize("dtype", [F32, BF], ids=["f32", "bf16"])
@pytest.mark.parametrize("heads", HEADS, ids=lambda h: "Hq%d-Hkv%d-D%d" % h)
@pytest.mark.parametrize("size", SIZES, ids=lambda s: "T%d-w%d-l%d-d%d" % s)
def test_parts_match_oracle(size, heads, dtype):
    import nsa_fused_kernel as nfk
    import nsa_hip_ops as ops
    dev = require_gpu()
    T, window, l, d = case_sizes(size, heads)
    Hq, Hkv, D = heads
    log(f"key parts T{T} w{window} l{l} d{d} Hq{Hq} Hkv{Hkv} D{D} {dtype}")
    q, do = randn((1, Hq, T, D), 1, dtype), randn((1, Hq, T, D), 4, dtype)
    for mode in ("window", "compress"):
        n = T if mode == "window" else ops.n_cmp_tokens(T, l, d)
        k, v = randn((1, Hkv, n, D), 2, dtype), randn((1, Hkv, n, D), 3, dtype)
        xs = [t.to(dev).requires_grad_() for t in (q, k, v)]
        o = nfk.window_attn_triton(*xs, window) if mode == "window" else nfk.compression_attn_triton(*xs, l, d)
        o.backward(do.to(dev))
        torch.cuda.synchronize()
        ref = [t.requires_grad_() for t in to64(q, k, v)]
        o_r, lse_r = (O.window_attention(*ref, window) if mode == "window" else O.compression_attention(*ref, l, d))
        o_r.backward(do.double())
        assert_close(o, o_r, dtype, f"{mode} o")
        assert_close(xs[0].grad, ref[0].grad, dtype, f"{mode} dq")


# T, Hq, Hkv, D, and a batch whose launches take fewer parts than the sequence alone
ALONE = [(700, 4, 1, 64, 20), (500, 16, 1, 64, 20), (900, 6, 1, 32, 20), (600, 16, 1, 128, 32), (1000, 4, 1, 16, 40)]


def part_counts(lib, B, T, Hq, Hkv, D, window, n, dtype):
    """Key parts of (forward, dQ) of the window and the compression."""
    code = 1 if dtype == BF else 0
    return [lib.nsa_range_key_parts(p, m, B, Hq, Hkv, T, L, D, window, code, None)
            for m, L in ((0, T), (1, n)) for p in (0, 1)]


@pytest.mark.parametrize("dtype", [F32, BF], ids=["f32", "bf16"])
@pytest.mark.parametrize("c", ALONE, ids=str)
def test_alone_and_in_a_batch(c, dtype):
    """The same sequence in launches of different part counts: float32 results
    apart by the order of their sums, bf16 ones also by P's rounding, which is
    relative to another maximum."""
    import nsa_fused_kernel as nfk
    import nsa_hip_ops as ops
    dev = require_gpu()
    T, Hq, Hkv, D, B = c
    window = 300
    for mode in ("window", "compress"):
        n = T if mode == "window" else ops.n_cmp_tokens(T, 32, 4)
        one = [randn((1, Hq, T, D), 1, dtype), randn((1, Hkv, n, D), 2, dtype), randn((1, Hkv, n, D), 3, dtype)]
        do = randn((1, Hq, T, D), 4, dtype)
        got = []
        for b in (1, B):
            log(f"key parts {c} {dtype} {mode} batch {b}")
            xs = [x.repeat(b, 1, 1, 1).to(dev).requires_grad_() for x in one]
            o = nfk.window_attn_triton(*xs, window) if mode == "window" else nfk.compression_attn_triton(*xs, 32, 4)
            o.backward(do.repeat(b, 1, 1, 1).to(dev))
            torch.cuda.synchronize()
            got.append((o.detach()[0].double(), xs[0].grad[0].double()))
        for a, b, what in zip(*got, ("o", "dq")):
            # sums of up to `window` or n terms, twice as long for dQ's chain through dS
            eps = 2.0 ** -7 if dtype == BF else 8 * 2.0 ** -24 * max(window, n) ** 0.5
            err = float((a - b).norm() / b.norm())
            assert err <= eps, f"{mode} {what}: {err:.2e} apart"


@pytest.mark.parametrize("dtype", [F32, BF], ids=["f32", "bf16"])
@pytest.mark.parametrize("c", [(300, 16, 1, 128), (1000, 12, 2, 64), (1301, 64, 4, 128), (500, 4, 1, 32)], ids=str)
def test_finished_rows_match_branches(c, dtype):
    """The layer (window forward merging and gating, both dQs in one launch)
    against the branches composed in torch."""
    import nsa_fused_kernel as nfk
    dev = require_gpu()
    T, Hq, Hkv, D = c
    idx = make_block_idx(1, Hkv, T, 32, 8).to(dev)
    ins = [randn((1, Hq, T, D), 1, dtype)] + [randn((1, Hkv, T, D), 2 + i, dtype) for i in range(6)]
    ins.append(randn((1, Hq, T, 3), 9, dtype))
    do = randn((1, Hq, T, D), 10, dtype).to(dev)
    got = []
    for fn in (nfk.nsa_fused_forward, nfk.nsa_fused_forward_composed):
        xs = [x.to(dev).requires_grad_() for x in ins]
        out = fn(*xs, idx, 32, 200)
        out.backward(do)
        torch.cuda.synchronize()
        got.append([out.detach(), xs[0].grad, xs[7].grad])
    for a, b, what in zip(*got, ("out", "dq", "dgate")):
        # two bf16 (float32) evaluations of the same layer
        assert_close(a, b.double(), dtype, what)
