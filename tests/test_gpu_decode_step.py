"""NSADecodeCache.step in one library call: the bits of append then attend,
and appended pooled tokens that are the pooling kernel's bit for bit (spans
shorter, longer and no multiple of the rows staged at a time)."""

import pytest
import torch

from nsa_testlib import randn, require_gpu

pytestmark = pytest.mark.gpu
BF, F32 = torch.bfloat16, torch.float32

# (l, d, l', n, w), Hq, Hkv, D
CASES = [((32, 16, 64, 16, 128), 16, 1, 128), ((16, 16, 16, 4, 32), 8, 2, 64), ((48, 8, 48, 3, 40), 6, 2, 32),
         ((64, 64, 64, 2, 64), 4, 4, 16), ((40, 20, 32, 5, 50), 40, 1, 128), ((1, 1, 16, 2, 8), 4, 2, 64)]


@pytest.mark.parametrize("dtype", [F32, BF], ids=["f32", "bf16"])
@pytest.mark.parametrize("c", CASES, ids=str)
def test_step_is_append_then_attend(c, dtype):
    import nsa_decode
    import nsa_hip_ops as ops
    dev = require_gpu()
    (l, d, ls, n, w), Hq, Hkv, D = c
    geom = ops.NSAGeometry(l, d, ls, n, w)
    cap, T0, steps = 200, 90, 112           # past the capacity: full caches stay as they are
    lens = [T0, 1, 63]
    B = len(lens)
    prompt = [randn((B, Hkv, T0, D), 10 + i, dtype).to(dev) for i in range(6)]
    both = [nsa_decode.NSADecodeCache(B, Hkv, D, cap, geom, dtype=dtype) for _ in range(2)]
    for cache in both:
        cache.prefill(*prompt, lens=lens)
    one, two = both
    for s in range(steps):
        q, gate = randn((B, Hq, D), 100 + s, dtype).to(dev), randn((B, Hq, 3), 300 + s, dtype).to(dev)
        rows = [randn((B, Hkv, D), 1000 + 6 * s + i, dtype).to(dev) for i in range(6)]
        out, idx = one.step(q, gate, rows)
        two.append(*rows)
        ref, ref_idx = two.attend(q, gate)
        assert torch.equal(out, ref) and torch.equal(idx, ref_idx) and torch.equal(one.lens, two.lens)
    torch.cuda.synchronize()
    assert one.lens.tolist() == [min(x + steps, cap) for x in lens]
    for a, b in zip((*one.caches(), one.k_cmp, one.v_cmp), (*two.caches(), two.k_cmp, two.v_cmp)):
        assert torch.equal(a, b)
    for b, x in enumerate(lens):
        L = min(x + steps, cap)
        m = ops.n_cmp_tokens(L, l, d)
        for src, got in ((one.kc, one.k_cmp), (one.vc, one.v_cmp)):
            assert torch.equal(ops.pool_fwd(src[b:b + 1, :, :L], l, d), got[b:b + 1, :, :m])
