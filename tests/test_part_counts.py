"""CPU checks that the sizes of the GPU tests take the launches they mean to:
the key parts of the range forward and dQ (test_gpu_key_parts.py) and the parts
of a window key block's queries in the dK/dV (test_gpu_dkdv_parts.py).  Without
a device the rules count 256 compute units, as an MI355X has."""

import os

import pytest
import torch

import test_gpu_dkdv_parts
import test_gpu_key_parts as kp


def _lib():
    import _nsa_lib
    if not os.path.exists(_nsa_lib.LIB_PATH):
        pytest.skip("libnsa_hip.so not built")
    return _nsa_lib.load()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
def test_key_part_sizes_cover_every_count(dtype):
    import nsa_hip_ops as ops
    lib, seen = _lib(), [set(), set()]
    for size in kp.SIZES:
        for heads in kp.HEADS:
            T, window, l, d = kp.case_sizes(size, heads)
            parts = kp.part_counts(lib, 1, T, *heads, window, ops.n_cmp_tokens(T, l, d), dtype)
            seen[0] |= {parts[0], parts[2]}
            seen[1] |= {parts[1], parts[3]}
    assert seen[0] >= {1, 2, 4} and seen[1] >= {1, 2, 4}, seen


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("c", kp.ALONE, ids=str)
def test_batched_sequences_take_other_part_counts(c, dtype):
    import nsa_hip_ops as ops
    T, Hq, Hkv, D, B = c
    n = ops.n_cmp_tokens(T, 32, 4)
    alone = kp.part_counts(_lib(), 1, T, Hq, Hkv, D, 300, n, dtype)
    batch = kp.part_counts(_lib(), B, T, Hq, Hkv, D, 300, n, dtype)
    assert all(x in (1, 2, 4) for x in alone + batch)
    # two parts of a float32 dQ's tiles do not fit LDS at D = 128
    fewer = (0, 2) if dtype == torch.float32 and D == 128 else range(4)
    assert all(alone[i] > batch[i] for i in fewer), (alone, batch)


def test_dkdv_part_sizes_split_the_window():
    lib, split = _lib(), 0
    for T, window, _, _ in test_gpu_dkdv_parts.SIZES:
        for _, Hkv, D in test_gpu_dkdv_parts.HEADS:
            split += lib.nsa_range_dkdv_partial_bytes(0, 1, Hkv, T, T, D, window, 1, None) > 0
    assert split == len(test_gpu_dkdv_parts.SIZES) * len(test_gpu_dkdv_parts.HEADS)


def test_key_part_query_refuses_what_the_launch_refuses():
    lib = _lib()
    good = (0, 0, 1, 4, 1, 256, 256, 64, 100, 0, None)
    assert lib.nsa_range_key_parts(*good) in (1, 2, 4)
    for i, bad in ((0, 3), (1, 7), (2, 0), (4, 3), (5, 0), (7, 48), (8, 0), (9, 9)):
        assert lib.nsa_range_key_parts(*good[:i], bad, *good[i + 1:]) < 0, i
