"""The layer's two routes (C entry points, Python sequence of calls): which
calls take which, and the same bits from both."""

import pytest
import torch

from nsa_testlib import make_block_idx, randn, require_gpu

BF, F32 = torch.bfloat16, torch.float32


def _takes(T, geom, block_idx=None, Hq=4, Hkv=2, D=64):
    import nsa_hip_ops as ops
    return ops._capi_takes(torch.empty(1, Hq, T, D), torch.empty(1, Hkv, T, D), geom, block_idx)


def test_route_rule(monkeypatch):
    import nsa_hip_ops as ops
    g = ops.NSAGeometry(32, 16, 64, 16, 512)
    assert _takes(64, g) and _takes(1000, g)
    assert not _takes(63, g) and not _takes(31, g) and not _takes(0, g)
    assert not _takes(1000, ops.NSAGeometry(32, 16, 64, 0, 512))
    assert not _takes(1000, ops.NSAGeometry(32, 16, 64, 16, 512, False, -1))
    idx = torch.zeros(1, 2, 1000, 15, dtype=torch.int32)
    assert _takes(1000, g, idx)                                         # min(16, 1000 // 64) = 15
    assert not _takes(1000, g, torch.zeros(1, 2, 1000, 16, dtype=torch.int32))
    assert not ops._capi_takes(torch.empty(4, 64), torch.empty(1, 2, 64, 64), g, None)
    for name, value in (("OVERLAP_SEL_BWD", True), ("SEPARATE_SEL_DQ", True), ("FUSE_RANGE_DQ", False),
                        ("DETERMINISTIC_DKDV", False), ("SEL_FWD_CHUNK", 64), ("SEL_DKDV_CHUNK", 64),
                        ("LAYER_CAPI", False), ("_TIMER", ops.LaunchTimer())):
        with monkeypatch.context() as m:
            m.setattr(ops, name, value)
            assert not _takes(1000, g), name


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [F32, BF], ids=["f32", "bf16"])
@pytest.mark.parametrize("T,given", [(64, False), (65, True), (333, False), (700, "wide")])
def test_routes_give_the_same_bits(T, given, dtype, monkeypatch):
    import nsa_fused_kernel as nfk
    import nsa_hip_ops as ops
    dev = require_gpu()
    Hq, Hkv, D = 8, 2, 64
    geom = ops.NSAGeometry.aligned(32, 6, 100)
    n = min(6, T // 32)
    idx = make_block_idx(1, Hkv, T, 32, 32 if given == "wide" else n).to(dev) if given else None
    ins = [randn((1, Hq, T, D), 1, dtype)] + [randn((1, Hkv, T, D), 2 + i, dtype) for i in range(6)]
    ins.append(randn((1, Hq, T, 3), 9, dtype))
    do = randn((1, Hq, T, D), 10, dtype).to(dev)

    def step():
        # q and the gate logits come as strided views, as a caller's projections may
        xs = [x.to(dev).transpose(1, 2).contiguous().transpose(1, 2).requires_grad_() for x in ins]
        out, picked = nfk.nsa_attention(*xs, geom, block_idx=idx)
        out.backward(do)
        with torch.no_grad():
            again, _ = nfk.nsa_attention(*xs, geom, block_idx=idx)
        torch.cuda.synchronize()
        assert torch.equal(out, again)
        return [out.detach(), picked] + [x.grad for x in xs]
    one = step()
    with monkeypatch.context() as m:
        m.setattr(ops, "LAYER_CAPI", False)
        two = step()
    for a, b in zip(one, two):
        assert a.shape == b.shape and torch.equal(a, b)
