"""The decode step's block choice against a plain sort of its own scores:
candidate counts around a wave and a workgroup, picks from one to all, random
scores, scores that all tie (the lower block first, down to the last digit of
the selection's keys) and scores in a few tied groups."""

import pytest
import torch

from nsa_testlib import randn, require_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_sel", [1, 16, 64])
@pytest.mark.parametrize("T", [16, 1024, 1040, 1041, 9600, 40000])       # 1, 64, 65, 66, 600 and 2500 candidates
@pytest.mark.parametrize("kind", ["random", "tied", "groups"])
def test_picks_are_the_sorted_scores(T, n_sel, kind):
    import nsa_hip_ops as ops
    dev = require_gpu()
    geom = ops.NSAGeometry(16, 16, 16, n_sel, 32, kind == "groups", 0)
    Hq, Hkv, D = 6, 2, 32
    lens = [T, max(1, T - 5)]
    caches = [randn((2, Hkv, T, D), 5 + i, torch.float32).to(dev) for i in range(6)]
    q = randn((2, Hq, D), 1, torch.float32).to(dev)
    if kind != "random":
        q.zero_()                        # every pooled token weighs the same
    if kind == "groups":                 # ... or one of three weights
        q.fill_(1.0)
        caches[0].copy_((torch.arange(T, device=dev) // 16 % 3).float()[None, None, :, None].expand_as(caches[0]) / 8)
    gate = randn((2, Hq, 3), 2, torch.float32).to(dev)
    k_cmp, v_cmp = (ops.pool_fwd(c, 16, 16) for c in caches[:2])
    _, idx, ex = ops.decode_fwd(q, k_cmp, v_cmp, *caches[2:], gate, torch.tensor(lens, dtype=torch.int32, device=dev),
                                geom, return_scores=True)
    torch.cuda.synchronize()
    for b, n in enumerate(lens):
        ncand = (n - 1) // 16 + 1
        sc = ex["scores"][b, :, :ncand].double().cpu()
        j = torch.arange(ncand)
        sc = sc.masked_fill(((j + 1) * 16 > n)[None, :], torch.finfo(torch.float32).min)
        if kind == "groups":
            sc[:, 0] = float("inf")
        S = min(n_sel, ncand)
        want = torch.sort(sc, dim=-1, descending=True, stable=True).indices[:, :S]
        assert torch.equal(want, idx[b, :, :S].cpu().long()), f"T {n} n_sel {n_sel} {kind}"
        assert (idx[b, :, S:] == -1).all()
