"""Range dK/dV with a key block's queries in several parts (short sequences,
where the key blocks alone leave CUs idle), against the float64 oracle and
the launch that takes each key block whole.

Sizes put the parts' edges inside and past the key blocks' query ranges:
windows of 3 (of 1, dK is 0) and past the sequence's end, lengths of one key block and one
more, the last block nearly empty; groups with flat rows (G < 16, float32 and
bf16; up to G = 8 in float32 at D = 128) and with head chunks."""

import pytest
import torch

from oracle import nsa_oracle as O
from nsa_testlib import assert_close, log, randn, require_gpu, to64

pytestmark = pytest.mark.gpu

# T, window, span l, stride d
SIZES = [(64, 3, 16, 16), (65, 40, 16, 8), (257, 700, 32, 16), (1000, 100, 64, 64), (1301, 512, 32, 16)]
HEADS = [(4, 1, 64), (12, 2, 32), (16, 1, 128), (20, 1, 64), (8, 1, 128), (9, 1, 128), (15, 1, 128), (15, 1, 64)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("heads", HEADS, ids=lambda h: "Hq%d-Hkv%d-D%d" % h)
@pytest.mark.parametrize("size", SIZES, ids=lambda s: "T%d-w%d-l%d-d%d" % s)
def test_parts_match_oracle_and_whole_blocks(size, heads, dtype, monkeypatch):
    import nsa_fused_kernel as nfk
    import nsa_hip_ops as ops
    dev = require_gpu()
    T, window, l, d = size
    Hq, Hkv, D = heads
    log(f"dkdv parts T{T} w{window} l{l} d{d} Hq{Hq} Hkv{Hkv} D{D} {dtype}")
    n = ops.n_cmp_tokens(T, l, d)
    q, do = randn((1, Hq, T, D), 1, dtype), randn((1, Hq, T, D), 4, dtype)
    for mode in ("window", "compress"):
        L = T if mode == "window" else n
        k, v = randn((1, Hkv, L, D), 2, dtype), randn((1, Hkv, L, D), 3, dtype)

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
        with monkeypatch.context() as m:   # without a partial buffer a window key block has one workgroup
            m.setattr(ops, "DETERMINISTIC_DKDV", False)
            whole = gpu()
        for i, what in enumerate(("dk", "dv")):
            assert torch.equal(got[i], again[i]), f"{mode} {what}: not the same twice"
            assert_close(got[i], xs[1 + i].grad, dtype, f"{mode} {what}")
            # the same T G float32 terms in another order (their errors add like a
            # random walk), and one bf16 unit where the output's rounding flips
            eps = 4 * 2.0 ** -24 * (T * Hq // Hkv) ** 0.5 + (2.0 ** -7 if dtype == torch.bfloat16 else 0.0)
            ref = whole[i].float()
            err = float((got[i].float() - ref).abs().max())
            assert err <= eps * max(1.0, float(ref.abs().max())), f"{mode} {what}: {err:.2e} from whole blocks"
