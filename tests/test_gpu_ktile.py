"""Uniform groups on the tiles whose wavefronts split K (sparse24_ktile_kernel): against the oracle and against the streaming
kernel, at the edges of its tiles, steps and shares of K."""
import pytest
import torch

from oracle import triteia_oracle as orc
from tests.helpers import activations, check_close, make_deltas, setknob, to_gpu
from triteia_amd.python import ops
from triteia_amd.python.capi import _ffi, mul_2_4

pytestmark = pytest.mark.gpu


def _case(b, t, k, m, seed=5):
    qw, meta, s = make_deltas(b, k, m, seed)
    x = activations(b * t, k, seed + 1).reshape(b, t, k)
    return qw, meta, s, x


# tokens either side of a 16-, 32-, 48- and 64-token tile, and tiles whose last 16 tokens start inside the tile before; one token to a
# matrix; fewer steps of K than wavefronts (k = 128: one), steps that do not divide among them (9, 11), K split over workgroups
# (long K, few columns) and not
@pytest.mark.parametrize("b,t,k,m", [
    (64, 17, 128, 512), (24, 25, 384, 640), (17, 1, 8192, 512), (33, 2, 128, 512), (4, 16, 2048, 640), (8, 12, 1408, 384), (3, 16, 8192, 128), (2, 31, 1152, 2048),
    (1, 32, 4096, 1152), (1, 33, 4096, 1152), (2, 48, 1152, 2048), (2, 49, 1152, 2048), (1, 63, 8192, 512), (1, 65, 8192, 640), (5, 64, 896, 1024),
    (1, 129, 4096, 1152), (1, 300, 1024, 4224), (1, 1100, 512, 384), (1, 37, 11008, 512),
])
def test_against_the_oracle(monkeypatch, b, t, k, m):
    qw, meta, s, x = _case(b, t, k, m)
    gq, gm, gs, gx = to_gpu(qw, meta, s, x)
    call = (lambda: ops.matmul_4bit_2_4(gq[0], gx[0], gm[0], gs[0])[None]) if b == 1 else (lambda: ops.bmm_4bit_2_4(gq, gx, gm, gs))
    out = call()
    check_close(out, orc.bmm_4bit_2_4(qw, x, meta, s), what=f"ktile {b} x {t} tokens, {k} x {m}")
    assert torch.equal(call(), out)
    setknob(monkeypatch, "TRITEIA_HIP_KTILE", 0)
    other = call()
    # (the same exact products added up in another order, in fp32, and rounded once: a few results in a thousand differ in their last bit)
    assert ((out.float() - other.float()).norm() / other.float().norm()).item() < 1e-4


def test_without_a_scratch_and_in_a_graph():
    """mul_2_4 has no room for shares of K: the same launch unsplit.  A captured split replays."""
    t, k, m = 37, 11008, 512
    qw, meta, s, x = _case(1, t, k, m)
    gq, gm, gs, gx = to_gpu(qw[0], meta[0], s[0], x[0])
    lib = _ffi.lib()
    assert lib.triteia_hip_uniform_kernel(m, 1, t, k, 1) > 1000 and lib.triteia_hip_uniform_kernel(m, 1, t, k, 0) == 0
    split = ops.matmul_4bit_2_4(gq, gx, gm, gs)
    plain = torch.zeros((t, m), dtype=torch.float16, device="cuda")
    mul_2_4(gx, gq, gm, plain, gs, torch.zeros(m // 128 * 16, dtype=torch.int32, device="cuda"))
    assert ((plain.float() - split.float()).norm() / split.float().norm()).item() < 1e-4
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        y = ops.matmul_4bit_2_4(gq, gx, gm, gs)
    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, split)
        assert torch.equal(ops.matmul_4bit_2_4(gq, gx, gm, gs), split)


def test_rows_that_are_not_aligned():
    """Activations that start inside 16 bytes stay with the kernels that took them before."""
    t, k, m = 40, 4096, 1152
    qw, meta, s, x = _case(1, t, k, m)
    gq, gm, gs, gx = to_gpu(qw[0], meta[0], s[0], x[0])
    shifted = torch.empty(t * k + 4, dtype=torch.float16, device="cuda")[4:].view(t, k)
    shifted.copy_(gx)
    a, b = ops.matmul_4bit_2_4(gq, shifted, gm, gs), ops.matmul_4bit_2_4(gq, gx, gm, gs)
    assert ((a.float() - b.float()).norm() / b.float().norm()).item() < 1e-4


@pytest.mark.parametrize("b,t,k,m", [(1, 37, 17024, 1536), (3, 31, 23296, 768)])
def test_rows_that_are_not_aligned_keep_their_split(monkeypatch, b, t, k, m):
    """The scratch is for the shares of K of either kernel: more of them on the streaming kernel here than on the tiles."""
    qw, meta, s, x = _case(b, t, k, m)
    gq, gm, gs, gx = to_gpu(qw, meta, s, x)
    shifted = torch.empty(b * t * k + 4, dtype=torch.float16, device="cuda")[4:].view(b, t, k)
    shifted.copy_(gx)
    out = ops.bmm_4bit_2_4(gq, shifted, gm, gs)
    setknob(monkeypatch, "TRITEIA_HIP_KTILE", 0)
    assert torch.equal(out, ops.bmm_4bit_2_4(gq, gx, gm, gs))
