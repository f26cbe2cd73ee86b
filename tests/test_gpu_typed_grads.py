"""dK / dV and the selection output written in the inputs' dtype by the
kernels that sum them: the float32 result rounded once, bit for bit."""

import pytest
import torch

from nsa_testlib import make_block_idx, randn, require_gpu

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


# T, block, S, D, Hq, Hkv: one item per block, several batches of items (chunk
# 2), a ragged last block; window split (short) and whole
@pytest.mark.parametrize("c", [(100, 32, 3, 64, 4, 2), (700, 64, 8, 128, 16, 1), (333, 128, 2, 32, 6, 1)], ids=str)
@pytest.mark.parametrize("chunk", [2, 512])
def test_rounded_once(c, chunk, monkeypatch):
    import _nsa_lib as L
    import nsa_hip_ops as ops
    dev = require_gpu()
    T, bs, S, D, Hq, Hkv = c
    monkeypatch.setattr(ops, "SEL_DKDV_CHUNK", chunk)
    q, do = (randn((1, Hq, T, D), s, BF).to(dev) for s in (1, 4))
    k, v = (randn((1, Hkv, T, D), s, BF).to(dev) for s in (2, 3))
    idx = make_block_idx(1, Hkv, T, bs, S).to(dev)
    (o, o32), lse, csr = ops.sel_fwd_fsa(q, k, v, idx, bs, o_both=True)
    assert torch.equal(o, o32.to(BF))
    assert torch.equal(o, ops.sel_fwd_fsa(q, k, v, idx, bs)[0])
    dot, coff = ops.delta_of(do, o32, lse)
    f = ops.sel_dkdv(q, k, v, do, coff, dot, idx, bs, csr=csr, want_dq=True)
    b = ops.sel_dkdv(q, k, v, do, coff, dot, idx, bs, csr=csr, want_dq=True, out_dtype=BF)
    for x, y in zip(f[:2], b[:2]):
        assert y.dtype == BF and torch.equal(x.to(BF), y)
    lib = L.load()
    for mode, L_, win, l, d in ((ops.MODE_WINDOW, T, 50, 1, 1), (ops.MODE_COMPRESS, T // 16, 0, 16, 16)):
        kk, vv = k[:, :, :L_].contiguous(), v[:, :, :L_].contiguous()
        o, lse = ops.range_fwd(mode, q, kk, vv, win, l, d, o_f32=True)
        dot, coff = ops.delta_of(do, o, lse)
        x32 = ops.range_dkdv(mode, q, kk, vv, do, coff, dot, win, l, d)
        span, step = (win, 1) if mode == ops.MODE_WINDOW else (l, d)
        n = int(lib.nsa_range_dkdv_partial_bytes(mode, 1, Hkv, T, L_, D, span, step, L.stream_of(q)))
        for parts in ((n,) if mode == ops.MODE_COMPRESS else (n, 0)):
            part = torch.empty(max(n, 4) // 4, device=dev, dtype=torch.float32)
            y = [torch.empty(1, Hkv, L_, D, device=dev, dtype=BF) for _ in range(2)]
            rc = lib.nsa_range_dkdv_as(mode, L.ptr(q), L.ptr(kk), L.ptr(vv), L.ptr(do), L.ptr(coff), L.ptr(dot),
                                       L.ptr(y[0]), L.ptr(y[1]), L.ptr(part) if parts else None, parts, 1, Hq, Hkv, T,
                                       L_, D, win, l, d, L.NSA_BF16, L.NSA_BF16, L.stream_of(q))
            assert rc == 0
            torch.cuda.synchronize()
            if parts == n:
                assert all(torch.equal(a.to(BF), b_) for a, b_ in zip(x32, y))
            else:   # whole key blocks: the same sums in another order
                for a, b_ in zip(x32, y):
                    assert float((a - b_.float()).abs().max()) <= 2.0 ** -7 * float(a.abs().max())
    # a bf16 result of several workgroups needs the partial rows
    assert lib.nsa_range_dkdv_as(ops.MODE_COMPRESS, L.ptr(q), L.ptr(k), L.ptr(v), L.ptr(do), L.ptr(coff), L.ptr(dot),
                                 L.ptr(y[0]), L.ptr(y[1]), None, 0, 1, Hq, Hkv, T, T // 16, D, 0, 16, 16, L.NSA_BF16,
                                 L.NSA_BF16, L.stream_of(q)) == L.NSA_ERR_ARG
