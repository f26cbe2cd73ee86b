"""The sums over a row's selection slots at slot counts around a batch of 16,
every head dim (2 to 16 lanes a row), two passes per block, with NaN in the
slots that hold no pair."""

import pytest
import torch

from nsa_testlib import assert_close, make_block_idx, randn, require_gpu

pytestmark = pytest.mark.gpu
BF, F32 = torch.bfloat16, torch.float32


@pytest.mark.parametrize("dtype", [F32, BF], ids=["f32", "bf16"])
@pytest.mark.parametrize("D", [16, 32, 64, 128])
@pytest.mark.parametrize("S,bs", [(1, 16), (15, 16), (16, 16), (17, 16), (33, 16), (9, 128)])
def test_merge_and_dq_sum(S, bs, D, dtype):
    import _nsa_lib as L
    import nsa_hip_ops as ops
    from nsa_selection_kernel import selection_forward_reference
    dev = require_gpu()
    T, Hq, Hkv = 300 if bs == 16 else 600, 6, 2
    G = Hq // Hkv
    idx = make_block_idx(1, Hkv, T, bs, S, seed=S).to(dev)
    idx[:, :, ::7, S // 2:] = -1
    idx[:, :, 5] = -1                                         # a row with no pair at all
    q = randn((1, Hq, T, D), 1, dtype).to(dev)
    k, v = (randn((1, Hkv, T, D), s, dtype).to(dev) for s in (2, 3))
    (o_part, ml), _ = ops.sel_fwd_partials(q, k, v, idx, bs)
    npass = int(L.load().nsa_sel_partial_slots(S, bs)) // S
    t = torch.arange(T, device=dev)[:, None]
    ok = ((idx >= 0) & (idx * bs <= t)).repeat_interleave(npass, dim=-1)      # [1, Hkv, T, NS]
    o_part.masked_fill_(~ok[..., None, None], float("nan"))
    ml.masked_fill_(~ok[..., None, None], float("nan"))
    o, lse = ops.sel_merge(idx, (o_part, ml), q.shape, Hkv, bs)
    ref = selection_forward_reference(q.double().cpu(), k.double().cpu(), v.double().cpu(), idx.cpu(), bs)
    assert_close(o, ref, dtype, "o")
    none = ~ok.any(-1).repeat_interleave(G, dim=1)
    assert (lse[none] == -1e9).all() and (lse[~none] > -1e8).all()
    part = randn((1, Hkv, T, S * npass, G, D), 7, dtype).to(dev)
    want = part.double().masked_fill(~ok[..., None, None], 0.0).sum(3).transpose(2, 3).reshape(1, Hq, T, D)
    got = ops.sel_dq_reduce(idx, part.masked_fill(~ok[..., None, None], float("nan")), None, bs, dtype)
    # float32 sums of S terms of size ~1, rounded to the dtype once
    eps = S * npass * 2.0 ** -23 + (2.0 ** -8 if dtype == BF else 0.0)
    assert float((got.double() - want).abs().max()) <= eps * max(1.0, float(want.abs().max()))


@pytest.mark.parametrize("dtype", [F32, BF], ids=["f32", "bf16"])
@pytest.mark.parametrize("D", [16, 32, 64, 128])
def test_infinite_value_of_a_slot_without_weight(D, dtype):
    """A selected block whose weight underflows to 0 beside the row's maximum
    still passes an infinite or NaN value on (0 x inf is NaN, as in torch):
    in the merge of its own and in the layer's window forward."""
    import nsa_fused_kernel as nfk
    import nsa_selection_backward as nsb
    dev = require_gpu()
    T, Hq, bs = 256, 4, 64
    q, k = torch.ones(1, Hq, T, D), torch.zeros(1, 1, T, D)
    k[:, :, :bs] = 400.0 / D ** 0.5      # scores of 400 in block 0, 0 elsewhere: exp(-400) is 0
    v = randn((1, 1, T, D), 1, F32)
    idx = torch.arange(T // bs).expand(1, 1, T, T // bs).clone().to(torch.int32)
    idx[idx * bs > torch.arange(T)[:, None]] = -1
    others = [randn((1, 1, T, D), 2 + i, F32) for i in range(4)]
    gate = torch.zeros(1, Hq, T, 3)
    for bad in (float("inf"), float("nan")):
        vb = v.clone()
        vb[:, :, 130] = bad              # block 2: the queries from 130 on see it
        qd, kd, vd, *od, gd = (x.to(dev, dtype) for x in (q, k, vb, *others, gate))
        o = nsb.selection_attn_triton(qd, kd, vd, idx.to(dev), bs)
        layer = nfk.nsa_fused_forward(qd, od[0], od[1], kd, vd, od[2], od[3], gd, idx.to(dev), bs, 32)
        for x, what in ((o, "selection"), (layer, "layer")):
            assert x[:, :, :128].isfinite().all(), f"{what}: {bad} reached a query that has not selected it"
            assert not x[:, :, 130:].isfinite().any(), f"{what}: {bad} lost"
