"""Range dK/dV with a window past the sequence ("no limit", up to 2^31 - 1) and
with a compression span or stride past it: the same bits as with the sequence's
length in their place.  Groups with flat rows, whose bounds are products with
the group size, and with head chunks."""

import pytest
import torch

from nsa_testlib import log, randn, require_gpu

pytestmark = pytest.mark.gpu
HEADS = [(2, 1, 64), (4, 1, 32), (6, 1, 128), (15, 1, 16), (16, 1, 64)]
LONG = [1 << 28, 1 << 29, 1 << 30, (1 << 31) - 1]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("heads", HEADS, ids=lambda h: "Hq%d-Hkv%d-D%d" % h)
def test_bounds_past_the_sequence(heads, dtype):
    import nsa_fused_kernel as nfk
    import nsa_hip_ops as ops
    dev = require_gpu()
    Hq, Hkv, D = heads
    T, n = 130, 70
    q, do = randn((1, Hq, T, D), 1, dtype).to(dev), randn((1, Hq, T, D), 4, dtype).to(dev)

    def grads(kind, L, a, b):
        xs = [q.clone()] + [randn((1, Hkv, L, D), 2 + i, dtype).to(dev) for i in range(2)]
        xs = [x.requires_grad_() for x in xs]
        log(f"long window {kind} {a} {b} {heads} {dtype}")
        o = (nfk.window_attn_triton(*xs, a) if kind == "window"
             else ops.RangeAttnHIP.apply(*xs, ops.MODE_COMPRESS, 0, a, b))
        o.backward(do)
        torch.cuda.synchronize()
        return [o.detach()] + [x.grad for x in xs]

    for kind, L, short, long in (
            [("window", T, (T, 0), (w, 0)) for w in LONG] +
            [("span", n, (T + 1, 16), (w, w)) for w in LONG] +        # no key is seen
            [("stride", n, (1, T), (1, w)) for w in LONG]):           # key 0 is seen by all
        ref, got = grads(kind, L, *short), grads(kind, L, *long)
        for a, b, what in zip(ref, got, ("o", "dq", "dk", "dv")):
            assert torch.equal(a, b), f"{kind} {long}: {what} differs from {short}"
        assert kind == "span" or float(ref[3].abs().max()) > 0
