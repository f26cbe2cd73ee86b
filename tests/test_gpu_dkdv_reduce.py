"""The launch that sums the range dK/dV's partial rows, against the float64
oracle: windows whose key blocks take 7, 8 and 10 parts (eight is where eight
threads begin to share a run of 4 floats), key counts and head dims whose runs
end inside a workgroup, one pooled key in all, two batches."""

import pytest
import torch

from oracle import nsa_oracle as O
from nsa_testlib import assert_close, log, randn, require_gpu, to64

pytestmark = pytest.mark.gpu

# T, window, span l, stride d
SIZES = [(300, 192, 32, 16), (301, 193, 64, 64), (299, 257, 16, 4), (287, 40, 287, 16)]
HEADS = [(2, 1, 16), (8, 4, 64)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("heads", HEADS, ids=lambda h: "Hq%d-Hkv%d-D%d" % h)
@pytest.mark.parametrize("size", SIZES, ids=lambda s: "T%d-w%d-l%d-d%d" % s)
def test_reduce_matches_oracle(size, heads, dtype):
    import nsa_fused_kernel as nfk
    import nsa_hip_ops as ops
    dev = require_gpu()
    T, window, l, d = size
    Hq, Hkv, D = heads
    log(f"dkdv reduce T{T} w{window} l{l} d{d} Hq{Hq} Hkv{Hkv} D{D} {dtype}")
    n = ops.n_cmp_tokens(T, l, d)
    q, do = randn((2, Hq, T, D), 1, dtype), randn((2, Hq, T, D), 4, dtype)
    for mode in ("window", "compress"):
        L = T if mode == "window" else n
        k, v = randn((2, Hkv, L, D), 2, dtype), randn((2, Hkv, L, D), 3, dtype)

        def gpu():
            xs = [t.to(dev).requires_grad_() for t in (q, k, v)]
            o = nfk.window_attn_triton(*xs, window) if mode == "window" else nfk.compression_attn_triton(*xs, l, d)
            o.backward(do.to(dev))
            torch.cuda.synchronize()
            return xs[1].grad, xs[2].grad
        got, again = gpu(), gpu()
        xs = [t.requires_grad_() for t in to64(q, k, v)]
        o, _ = (O.window_attention(*xs, window) if mode == "window" else O.compression_attention(*xs, l, d))
        o.backward(do.double())
        for i, what in enumerate(("dk", "dv")):
            assert torch.equal(got[i], again[i]), f"{mode} {what}: not the same twice"
            if not (i == 0 and L == 1):   # the dK of one key is 0: no scale to compare against
                assert_close(got[i], xs[1 + i].grad, dtype, f"{mode} {what}")
