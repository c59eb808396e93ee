"""Sizes at which a dispatch rule changes its mind, through the ops, against the dense fp32 product of the unpacked
weights.  Tolerance: the inputs are exact on both sides and the sums are fp32, so what is left is the fp16 rounding of the
result (2^-11 of a value at most, 2.1e-4 in the Frobenius norm) and the order of the sums (1e-6)."""
import pytest
import torch

from triteia_amd.python import ops
from triteia_amd.python.ops.utils.sparsity import unpack_2_4
from triteia_amd.workloads import random_activations, random_packed_deltas

pytestmark = pytest.mark.gpu
REL = 4e-4


def dense(q, meta, s):
    return unpack_2_4(q, meta, None, torch.float32) * s.float().reshape(1, -1)


def check(got, ref, what):
    err = float((got.float() - ref).norm() / ref.norm())
    assert err <= REL, f"{what}: relative Frobenius error {err:.2e}"


# last tokens of a long uniform batch: in the 64-token launch where that adds no workgroup to the busiest CU (1), in a
# launch of the narrow kernel where it does (4104 rows on 4096 columns: a full round and one tile)
@pytest.mark.parametrize("T,k,m", [(4000, 128, 11008), (2000, 256, 11008), (4104, 128, 4096), (2056, 128, 11008), (2060, 128, 14336)])
def test_last_tokens_of_a_long_batch(T, k, m):
    q, meta, s = (t[0] for t in random_packed_deltas(1, k, m, T, "cuda"))
    x = random_activations(T, k, T + 1, "cuda")
    check(ops.matmul_4bit_2_4(q, x, meta, s), x.float() @ dense(q, meta, s), f"T={T} k={k} m={m}")
