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


# (tokens, deltas, k, m, share of tokens without a delta): column shares of at most 16 tokens, weights requested ahead of
# the routing, routed first, several passes per delta, a plan of narrow and of wide tiles, nothing routed at all
@pytest.mark.parametrize("T,n,k,m,none", [(1, 2, 128, 128, 1.0), (13, 32, 256, 384, 0.5), (16, 64, 512, 4096, 0.3), (64, 16, 256, 4096, 0.2),
                                          (40, 33, 256, 640, 0.5), (256, 16, 256, 384, 0.4), (65, 64, 256, 128, 0.3), (300, 70, 128, 256, 0.3),
                                          (1000, 8, 256, 512, 0.3), (1500, 3, 128, 2048, 1.0)])
def test_rows_without_a_delta_are_cleared_by_the_launch(T, n, k, m, none):
    from triteia_amd.python.capi import _ffi, routed_workspace, sbmm_2_4_routed
    g = torch.Generator().manual_seed(T + n)
    idx = torch.randint(0, n, (T,), generator=g) + 5
    out = torch.rand(T, generator=g) < none
    idx[out] = torch.randint(0, 2, (int(out.sum()),), generator=g) * (n + 6) - 1        # below and past the deltas' range
    idx = idx.to(torch.int32).cuda()
    q, meta, s = random_packed_deltas(n, k, m, T, "cuda")
    x = random_activations(T, k, T + 1, "cuda")
    want = torch.zeros((T, m), dtype=torch.float16, device="cuda")
    sbmm_2_4_routed(x, q, meta, want, s, idx, index_offset=5)
    got = torch.full_like(want, float("nan"))
    ws = routed_workspace(T, n, x.device)
    err = _ffi.lib().triteia_hip_sbmm_2_4_routed(
        *(_ffi.ptr(t) for t in (x, q, meta, got, s, idx)), 5, n, m, T, k, _ffi.ptr(ws), ws.numel() * ws.element_size(), 2,
        _ffi.device_index(x), _ffi.stream_of(x))
    assert err == 0 and torch.equal(got, want)
