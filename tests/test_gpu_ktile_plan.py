"""Routed batches on the tiles whose wavefronts split K (sparse24_ktile_plan_kernel): against the oracle, and to the bit against the
streaming kernel, at the edges of its tiles, steps and parts of the columns."""
import numpy as np
import pytest
import torch

from oracle import triteia_oracle as orc
from tests.helpers import activations, check_close, make_deltas, setknob, to_gpu
from triteia_amd.python import ops
from triteia_amd.python.capi import _ffi

pytestmark = pytest.mark.gpu


def _counts_to_indices(counts, none, seed):
    idx = np.concatenate([np.full(c, d, dtype=np.int32) for d, c in enumerate(counts)] + [np.full(none, -1, dtype=np.int32)])
    return np.random.default_rng(seed).permutation(idx)


def _streaming(monkeypatch, call):
    for name, value in (("PLAN_KTILE", 0), ("MID", 0), ("WIDE", 0), ("FUSED_ROUTE", 0)):
        setknob(monkeypatch, "TRITEIA_HIP_" + name, value)
    return call()


# tokens of a delta: none, one, either side of 16, 32, 48 and 64 and of several tiles; one step of K, fewer than wavefronts, odd numbers, and a
# walk that starts elsewhere for every delta (narrow layers); one column block, fewer than parts, and 29 / 45 of them (4, 8 parts); lists of
# 16- / 32-token tiles and of 64-token ones
@pytest.mark.parametrize("k,m,counts,none", [
    (128, 128, [1, 0, 15, 16, 17, 31, 32, 33], 3), (384, 1152, [63, 64, 65, 0, 47, 48, 49, 1], 0), (640, 384, [129, 0, 0, 200, 2], 7),
    (1408, 3712, [40, 33, 70, 1], 1), (256, 5760, [90, 100, 81, 64, 65], 2), (4096, 1024, [5] * 40, 4), (2176, 640, [300, 700, 64, 130], 0),
    (128, 256, [0, 0, 2049, 1], 0), (896, 512, [17] * 64, 0),
])
@pytest.mark.parametrize("base", [False, True])
def test_against_the_oracle_and_the_streaming_kernel(monkeypatch, k, m, counts, none, base):
    qw, meta, s = make_deltas(len(counts), k, m, 3)
    idx = _counts_to_indices(counts, none, 4)
    x = activations(len(idx), k, 5)
    w = (np.random.default_rng(6).standard_normal((m, k)) * 0.02).astype(np.float16) if base else None
    gq, gm, gs, gx, gi = to_gpu(qw, meta, s, x, idx)
    gw = to_gpu(w)[0] if base else None
    call = lambda: ops.sbmm_4bit_2_4_native(gq, gx, gm, gs, gi, base_weight=gw)
    setknob(monkeypatch, "TRITEIA_HIP_PLAN_KTILE", 2)
    setknob(monkeypatch, "TRITEIA_HIP_FUSED_ROUTE", 0)
    assert _ffi.lib().triteia_hip_planned_ktile(len(idx), len(counts), m, k) in (16, 32, 64)
    assert _ffi.lib().triteia_hip_routed_in_kernel(len(idx), len(counts), m, k) == 0
    out = call()
    if not base:
        check_close(out, orc.sbmm_4bit_2_4(qw, x, meta, s, idx), what=f"planned ktile {k} x {m}, {counts}")
        assert bool((out[gi < 0] == 0).all())
    assert torch.equal(call(), out)
    assert torch.equal(_streaming(monkeypatch, call), out)


def test_a_batch_that_a_plan_serves_better_still_runs_without_a_workspace():
    n, t, k, m = 2, 64, 8192, 256
    qw, meta, s = make_deltas(n, k, m, 3)
    idx = (np.arange(t) % (n + 1) - 1).astype(np.int32)
    gq, gm, gs, gx, gi = to_gpu(qw, meta, s, activations(t, k, 5), idx)
    lib = _ffi.lib()
    assert lib.triteia_hip_routed_in_kernel(t, n, m, k) == 0 and lib.triteia_hip_planned_ktile(t, n, m, k) > 0
    want = ops.sbmm_4bit_2_4_native(gq, gx, gm, gs, gi)
    out = torch.full((t, m), 9.0, dtype=torch.float16, device="cuda")
    args = lambda ws, size: (gx.data_ptr(), gq.data_ptr(), gm.data_ptr(), out.data_ptr(), gs.data_ptr(), gi.data_ptr(), 0, n, m, t, k, ws, size, 2, 0,
                             torch.cuda.current_stream().cuda_stream)
    ws = torch.empty(lib.triteia_hip_sbmm_routed_workspace_bytes(t, n) + 16, dtype=torch.uint8, device="cuda")
    for call in (lib.triteia_hip_sbmm_2_4_routed, lib.triteia_hip_sbmm_2_4_routed_own):
        # (none, not aligned, too small: routed in the kernel)
        for ptr, size in ((None, 0), (ws.data_ptr() + 4, ws.numel() - 16), (ws.data_ptr(), ws.numel() - 32)):
            out.fill_(9.0)
            assert call(*args(ptr, size)) == 0
            assert torch.equal(out, want)
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        y = ops.sbmm_4bit_2_4_native(gq, gx, gm, gs, gi)
    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
        assert torch.equal(ops.sbmm_4bit_2_4_native(gq, gx, gm, gs, gi), want)


@pytest.mark.parametrize("n,t,k,m", [(2, 64, 8192, 256), (1, 32, 11008, 512), (4, 256, 4096, 256)])
def test_a_workspace_that_other_calls_may_share_stays_untouched(n, t, k, m):
    """triteia_hip_sbmm_2_4_routed routes such a batch in the kernel whatever workspace it is given; triteia_hip_sbmm_2_4_routed_own plans it."""
    qw, meta, s = make_deltas(n, k, m, 3)
    idx = (np.arange(t) % (n + 1) - 1).astype(np.int32)
    x = activations(t, k, 5)
    gq, gm, gs, gx, gi = to_gpu(qw, meta, s, x, idx)
    lib = _ffi.lib()
    assert lib.triteia_hip_routed_leaves_workspace(t, n, m, k) == 1 and lib.triteia_hip_routed_in_kernel(t, n, m, k) == 0
    outs = []
    for call, touched in ((lib.triteia_hip_sbmm_2_4_routed, False), (lib.triteia_hip_sbmm_2_4_routed_own, True)):
        out = torch.full((t, m), 9.0, dtype=torch.float16, device="cuda")
        ws = torch.full((lib.triteia_hip_sbmm_routed_workspace_bytes(t, n),), 0x5a, dtype=torch.uint8, device="cuda")
        assert call(gx.data_ptr(), gq.data_ptr(), gm.data_ptr(), out.data_ptr(), gs.data_ptr(), gi.data_ptr(), 0, n, m, t, k, ws.data_ptr(), ws.numel(), 2, 0,
                    torch.cuda.current_stream().cuda_stream) == 0
        assert bool((ws != 0x5a).any()) is touched
        outs.append(out)
    assert torch.equal(*outs)
    check_close(outs[0], orc.sbmm_4bit_2_4(qw, x, meta, s, idx), what=f"routed {n} deltas, {t} tokens, {k} x {m}")


@pytest.mark.parametrize("k,m,counts", [(384, 1152, [63, 64, 65, 0, 47, 48, 49, 1]), (4096, 1024, [5] * 40)])
def test_infinities_and_nan(monkeypatch, k, m, counts):
    """They stay in their own rows (a tile's padding is its last token again) and meet the same weights as on the streaming kernel."""
    qw, meta, s = make_deltas(len(counts), k, m, 3)
    idx = _counts_to_indices(counts, 2, 4)
    gq, gm, gs, gx, gi = to_gpu(qw, meta, s, activations(len(idx), k, 5), idx)
    call = lambda: ops.sbmm_4bit_2_4_native(gq, gx, gm, gs, gi)
    setknob(monkeypatch, "TRITEIA_HIP_PLAN_KTILE", 2)
    setknob(monkeypatch, "TRITEIA_HIP_FUSED_ROUTE", 0)
    assert _ffi.lib().triteia_hip_planned_ktile(len(idx), len(counts), m, k) > 0
    clean = call()
    rows = [int(np.flatnonzero(idx == d)[-1]) for d in (0, 2, 7)]
    for row, column, value in zip(rows, (5, k // 2, k - 1), (float("inf"), float("-inf"), float("nan"))):
        gx[row, column] = value
    out = call()
    kept = torch.ones(len(idx), dtype=torch.bool, device="cuda")
    kept[rows] = False
    assert torch.equal(out[kept], clean[kept])
    other = _streaming(monkeypatch, call)
    assert bool((~torch.isfinite(out[rows])).any(-1).all())
    assert torch.equal(out.isnan(), other.isnan()) and torch.equal(out[~out.isnan()], other[~out.isnan()])


def test_activations_that_are_not_aligned_stay_with_the_kernels_before():
    n, t, k, m = 3, 300, 1024, 512
    qw, meta, s = make_deltas(n, k, m, 3)
    idx = (np.arange(t) % n).astype(np.int32)
    gq, gm, gs, gx, gi = to_gpu(qw, meta, s, activations(t, k, 5), idx)
    shifted = torch.empty(t * k + 4, dtype=torch.float16, device="cuda")[4:].view(t, k)
    shifted.copy_(gx)
    a, b = (ops.sbmm_4bit_2_4_native(gq, v, gm, gs, gi) for v in (shifted, gx))
    # (the same exact products added up in another order, in fp32, and rounded once)
    assert ((a.float() - b.float()).norm() / b.float().norm()).item() < 1e-4


def test_a_plan_for_small_batches_asks_for_aligned_activations():
    """A batch that triteia_hip_sbmm_2_4_routed_own plans for the K-splitting tiles is routed in the kernel, the workspace untouched, if its
    activations start inside 16 bytes: it is their address that counts, not the weights'."""
    n, t, k, m = 2, 64, 8192, 256
    qw, meta, s = make_deltas(n, k, m, 3)
    idx = (np.arange(t) % (n + 1) - 1).astype(np.int32)
    gq, gm, gs, gx, gi = to_gpu(qw, meta, s, activations(t, k, 5), idx)
    shifted = torch.empty(t * k + 4, dtype=torch.float16, device="cuda")[4:].view(t, k)
    shifted.copy_(gx)
    lib = _ffi.lib()
    assert lib.triteia_hip_planned_ktile(t, n, m, k) > 0 and gx.data_ptr() % 16 == 0 == gq.data_ptr() % 16
    outs = []
    for x in (gx, shifted):
        out = torch.full((t, m), 9.0, dtype=torch.float16, device="cuda")
        ws = torch.full((lib.triteia_hip_sbmm_routed_workspace_bytes(t, n),), 0x5a, dtype=torch.uint8, device="cuda")
        assert lib.triteia_hip_sbmm_2_4_routed_own(x.data_ptr(), gq.data_ptr(), gm.data_ptr(), out.data_ptr(), gs.data_ptr(), gi.data_ptr(), 0, n, m, t, k,
                                                   ws.data_ptr(), ws.numel(), 2, 0, torch.cuda.current_stream().cuda_stream) == 0
        assert bool((ws != 0x5a).any()) is (x is gx)
        outs.append(out)
    assert torch.equal(*outs)
