"""GPU parity of the compression phi at the edges of its tiles: the weight
gradients' 32-token chunks and 8-token runs (few tokens per sequence, so that a
chunk or a run crosses several sequences; one token in all; a remainder), every
hidden width and a partial 128-column group.  Against the float64 oracle at the
strict bound."""

import pytest
import torch

from oracle import nsa_oracle as O
from nsa_testlib import assert_strict, log, randn, require_gpu

pytestmark = pytest.mark.gpu

BF, F32 = torch.bfloat16, torch.float32

# dtype, B, H, T, D, hidden, l, d
CASES = [
    (BF, 1, 1, 4, 64, 32, 4, 4),         # one token
    (F32, 3, 5, 4, 64, 64, 4, 2),        # one token per sequence: a run crosses 8 sequences
    (BF, 2, 9, 21, 128, 128, 3, 3),      # 7 tokens per sequence, 126 in all
    (BF, 1, 3, 40, 64, 128, 1, 1),       # l = 1, 40 tokens per sequence
    (F32, 1, 1, 65, 128, 32, 1, 2),      # 33 tokens
    (BF, 1, 2, 270, 64, 64, 13, 1),      # l D = 832: a partial column group
    (F32, 1, 2, 90, 128, 128, 5, 3),     # 29 tokens per sequence
]


def case_id(c):
    return f"{str(c[0])[6:]}-B{c[1]}H{c[2]}T{c[3]}D{c[4]}h{c[5]}l{c[6]}d{c[7]}"


@pytest.mark.parametrize("case", CASES, ids=case_id)
def test_phi_edges(case):
    import nsa_hip_ops as ops
    dev = require_gpu()
    dtype, B, H, T, D, Hd, l, d = case
    log(f"phi edges {case}")

    def rounded(t):   # the kernels take W1 / W2 in the operand dtype
        return t.to(dtype).float()

    x = randn((B, H, T, D), 1, dtype)
    pos = 0.3 * randn((l, D), 2, F32)
    w1 = rounded(randn((Hd, l * D), 3, F32) * (l * D) ** -0.5)
    b1 = 0.1 * randn((Hd,), 4, F32)
    w2 = rounded(randn((D, Hd), 5, F32) * Hd ** -0.5)
    b2 = 0.1 * randn((D,), 6, F32)
    dout = randn((B, H, O.n_cmp_tokens(T, l, d), D), 7, dtype)
    leaves = [t.to(dev).requires_grad_() for t in (x, pos, w1, b1, w2, b2)]
    out = ops.phi_compress(*leaves, l, d)
    out.backward(dout.to(dev))
    torch.cuda.synchronize()
    ref_leaves = [t.double().requires_grad_() for t in (x, pos, w1, b1, w2, b2)]
    ref = O.phi_compress(*ref_leaves, l, d)
    ref.backward(dout.double())
    assert_strict(out.float().cpu(), ref, dtype, "out")
    for name, got, r in zip(["dx", "dpos", "dW1", "db1", "dW2", "db2"], leaves, ref_leaves):
        assert_strict(got.grad.float().cpu(), r.grad, dtype, name)
