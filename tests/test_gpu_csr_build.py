"""The counting CSR build and the work items over sizes around their
workgroups: lists around 64 (one a lane) and 4096 (one pass over the totals),
chunks around 16 and 256 (the scan's waves and batches), no pair at all, empty
blocks, rows that hold a block twice -- against a stable sort."""

import pytest
import torch

from nsa_testlib import make_block_idx, require_gpu

pytestmark = pytest.mark.gpu


def _csr(idx, bs, n_blk, packed):
    """(q_of_block, offsets [B * Hkv, n_blk + 1], pair_bh) by a stable sort of the keys."""
    B, Hkv, T, S = idx.shape
    t = torch.arange(T)[None, None, :, None].expand_as(idx)
    bh = torch.arange(B * Hkv).view(B, Hkv, 1, 1).expand_as(idx)
    ok = ((idx >= 0) & (idx < n_blk) & (idx.long() * bs <= t)).reshape(-1)
    key = (bh * n_blk + idx.long()).reshape(-1)[ok]
    key, order = torch.sort(key, stable=True)
    bits = max(0, (S - 1).bit_length())
    slot = torch.arange(S).expand_as(idx)
    val = ((t << bits) | slot if packed else t).reshape(-1)[ok][order]
    counts = torch.bincount(key, minlength=B * Hkv * n_blk).view(B * Hkv, n_blk)
    ends = counts.reshape(-1).cumsum(0).view(B * Hkv, n_blk)
    start = (ends - counts)
    return val, torch.cat([start, ends[:, -1:]], 1), key // n_blk


# B, Hkv, T, block, S
SIZES = [(1, 1, 1, 16, 1), (5, 64, 600, 16, 2), (1, 2, 64, 16, 4), (2, 3, 65, 16, 5), (1, 4, 1025, 16, 16),
         (3, 2, 1040, 16, 3), (1, 1, 16500, 64, 2), (1, 3, 17000, 256, 4), (2, 32, 1100, 16, 2), (70, 2, 500, 16, 2)]


@pytest.mark.parametrize("c", SIZES, ids=str)
@pytest.mark.parametrize("kind", ["random", "none", "one", "twice"])
def test_csr_is_the_stable_sort(c, kind):
    import nsa_hip_ops as ops
    dev = require_gpu()
    B, Hkv, T, bs, S = c
    idx = make_block_idx(B, Hkv, T, bs, S, seed=S)
    if kind == "none":
        idx.fill_(-1)
    elif kind == "one":
        idx.fill_(0)                      # every slot of every row on block 0
    elif kind == "twice":
        idx[..., -1] = idx[..., 0]
    n_blk = -(-T // bs)
    for packed in (True, False):
        q, off, bh, count = ops.csr_device(idx.to(dev), bs, pack_slot=packed)
        torch.cuda.synchronize()
        val, want, pbh = _csr(idx, bs, n_blk, packed)
        n = val.numel()
        assert int(count) == n
        assert torch.equal(off.view(-1, n_blk + 1).cpu().long(), want)
        assert torch.equal(q[:n].cpu().long(), val.long()) and (q[n:idx.numel()] == -1).all()
        assert torch.equal(bh[:n].cpu().long(), pbh) and (bh[n:idx.numel()] == -1).all()


@pytest.mark.parametrize("chunk", [2, 16, 1000])
@pytest.mark.parametrize("c", [(1, 1, 33, 16, 2), (1, 4, 1025, 16, 16), (2, 2, 17000, 16, 2), (40, 4, 600, 16, 1)],
                         ids=str)
def test_items_cover_every_pair_in_order(c, chunk):
    """nsa_sel_dkdv's work items (read back from its workspace): each block's
    entries in consecutive runs of `chunk`, blocks in order, `first` the
    blocks' first items."""
    import _nsa_lib as L
    import nsa_hip_ops as ops
    dev = require_gpu()
    B, Hkv, T, bs, S = c
    idx = make_block_idx(B, Hkv, T, bs, S, seed=3).to(dev)
    q_of_block, off, _, count = ops.csr_device(idx, bs, pack_slot=True)
    D, n_blk = 16, -(-T // bs)
    z = torch.zeros(B, Hkv, T, D, device=dev)
    c0, d0 = torch.full((B * Hkv * T,), float("inf"), device=dev), torch.zeros(B * Hkv * T, device=dev)
    lib = L.load()
    ws = torch.full((int(lib.nsa_sel_dkdv_workspace(B, Hkv, T, S, bs, chunk)) // 4,), -7, device=dev, dtype=torch.int32)
    dk, dv = torch.empty_like(z), torch.empty_like(z)
    rc = lib.nsa_sel_dkdv(L.ptr(z), L.ptr(z), L.ptr(z), None, L.ptr(z), L.ptr(c0), L.ptr(d0), L.ptr(q_of_block), 1,
                          L.ptr(off), L.ptr(count), L.ptr(dk), L.ptr(dv), None, 0, None, L.ptr(ws), ws.numel() * 4, B,
                          Hkv, Hkv, T, D, S, bs, chunk, L.NSA_F32, L.stream_of(z))
    assert rc == 0
    torch.cuda.synchronize()
    nb = B * Hkv * n_blk
    rows = off.view(-1, n_blk + 1).cpu().long()
    beg, end = rows[:, :-1].reshape(-1), rows[:, 1:].reshape(-1)
    n = (end - beg + chunk - 1) // chunk
    first = torch.cat([torch.zeros(1, dtype=torch.long), n.cumsum(0)])
    total = int(first[-1])
    cap = nb + (B * Hkv * T * S + chunk - 1) // chunk + 1
    w = ws.cpu().long()
    assert int(w[4 * cap]) == total
    assert torch.equal(w[4 * cap + 64:4 * cap + 64 + nb + 1], first)
    e = torch.repeat_interleave(torch.arange(nb), n)
    s0 = beg[e] + (torch.arange(total) - first[e]) * chunk
    want = torch.stack([e, s0, torch.minimum(s0 + chunk, end[e]), torch.zeros_like(e)], 1)
    assert torch.equal(w[:4 * total].view(total, 4), want)
