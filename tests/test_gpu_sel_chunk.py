"""Selection work items of the sizes that short sequences take: the forward's
partials and the dQ do not depend on how a block's queries are cut, dK / dV
only through the order of their float32 sums."""

import pytest
import torch

from nsa_testlib import make_block_idx, randn, require_gpu

BF, F32 = torch.bfloat16, torch.float32


def test_chunk_rule():
    import _nsa_lib
    lib = _nsa_lib.load()
    for fn, lo, hi in ((lib.nsa_sel_fwd_chunk, 16, 128), (lib.nsa_sel_dkdv_chunk, 32, 512)):
        last = 0
        for T in (1, 64, 600, 1024, 2048, 4096, 12000, 32768, 131072):
            c = fn(1, 4, T, 16, 64)
            assert lo <= c <= hi and c & (c - 1) == 0 and c >= last
            last = c
        assert last == hi
        assert fn(0, 4, 64, 16, 64) == 0


# B, Hq, Hkv, D, T, block, S: groups of 16 heads, packed groups, two passes, a ragged last block
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [F32, BF], ids=["f32", "bf16"])
@pytest.mark.parametrize("c", [(1, 16, 1, 128, 300, 64, 4), (2, 8, 2, 64, 1000, 32, 16), (1, 6, 1, 64, 517, 128, 3)],
                         ids=str)
def test_items_of_any_size_agree(c, dtype, monkeypatch):
    import nsa_hip_ops as ops
    import nsa_selection_backward as nsb
    dev = require_gpu()
    B, Hq, Hkv, D, T, bs, S = c
    idx = make_block_idx(B, Hkv, T, bs, S).to(dev)
    q, do = randn((B, Hq, T, D), 1, dtype), randn((B, Hq, T, D), 4, dtype)
    k, v = randn((B, Hkv, T, D), 2, dtype), randn((B, Hkv, T, D), 3, dtype)

    def gpu():
        xs = [t.to(dev).requires_grad_() for t in (q, k, v)]
        o = nsb.selection_attn_triton(*xs, idx, bs)
        o.backward(do.to(dev))
        torch.cuda.synchronize()
        return [o.detach()] + [x.grad for x in xs]
    got = gpu()
    for small in (2, 10):
        with monkeypatch.context() as m:
            m.setattr(ops, "SEL_FWD_CHUNK", small)
            m.setattr(ops, "SEL_DKDV_CHUNK", small)
            other = gpu()
        assert torch.equal(got[0], other[0]) and torch.equal(got[1], other[1]), "o or dq depends on the items"
        for i, what in ((2, "dk"), (3, "dv")):
            # T G float32 terms in another order (a random walk of their errors),
            # and one bf16 unit where the output's rounding flips
            eps = 4 * 2.0 ** -24 * (T * Hq // Hkv) ** 0.5 + (2.0 ** -7 if dtype == BF else 0.0)
            ref = got[i].float()
            err = float((other[i].float() - ref).abs().max())
            assert err <= eps * max(1.0, float(ref.abs().max())), f"{what}: {err:.2e}"
