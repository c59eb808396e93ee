"""The LoRA product in one launch (triteia_hip_lora) against the oracle, at the edges of its tiles, steps and pieces of columns."""
import numpy as np
import pytest
import torch

from oracle import triteia_oracle as orc
from tests.helpers import setknob
from triteia_amd.python import ops
from triteia_amd.python.capi import _ffi

pytestmark = pytest.mark.gpu


@pytest.fixture
def always(monkeypatch):
    """Every call that can run in one launch does."""
    setknob(monkeypatch, "TRITEIA_HIP_LORA_FUSED", 2)


@pytest.mark.parametrize("T,M,k,r,m", [
    (1, 1, 64, 8, 8),             # smallest: one step of one wavefront, half a rank tile, one 16-byte piece of output
    (17, 3, 576, 16, 264),        # nine steps for eight wavefronts; a tile and one token; a last piece of 8 columns
    (70, 2, 1088, 24, 520),       # 32-token tiles and a rest; a rank that is no power of two
    (130, 3, 4160, 64, 256),      # more steps than are in flight
    (200, 70, 512, 32, 4680),     # more than 64 bins, more than eight tiles; pieces of columns that do not divide among the wavefronts
    (300, 4, 640, 40, 5000),      # the widest tile, several turns of pieces a wavefront
    (4096, 5, 128, 64, 72),       # the largest batch
    (90, 1024, 64, 8, 64),        # the most adapters
])
@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
def test_one_launch_against_the_oracle(always, T, M, k, r, m, dtype):
    rng = np.random.default_rng(T * k + m)
    A = (rng.standard_normal((M, k, r)) * 0.1).astype(np.float16)
    B = (rng.standard_normal((M, r, m)) * 0.1).astype(np.float16)
    x = rng.standard_normal((T, k)).astype(np.float16)
    idx = rng.integers(-1, M, size=T)
    idx[rng.random(T) < 0.3] = M - 1                          # a hot adapter
    if dtype == "bf16":
        A, B, x = (orc.round_bf16(v) for v in (A, B, x))
    ref = orc.lora(A, B, x, idx, intermediate=dtype) if dtype == "bf16" else orc.lora(A, B, x, idx)
    tdt = torch.bfloat16 if dtype == "bf16" else torch.float16
    gA, gB, gx = (torch.from_numpy(np.ascontiguousarray(v)).cuda().to(tdt) for v in (A, B, x))
    assert _ffi.lib().triteia_hip_lora_ok(T, M, k, r, m)
    # one rounding of the intermediate and one of the result: 2^-11 (2^-8) relative each, and the oracle's own
    tol = 2e-2 if dtype == "bf16" else 2e-3
    scale = max(1e-6, float(np.sqrt(np.mean(np.square(ref.astype(np.float64))))))
    for gi in (torch.from_numpy(idx.astype(np.int32)).cuda(), torch.from_numpy(idx.astype(np.int64)).cuda()):
        y = ops.lora_bgmv(gA, gB, gx, gi)
        assert y.dtype == tdt and bool((y[gi < 0] == 0).all())
        err = np.linalg.norm(y.float().cpu().numpy().astype(np.float64) - ref) / (scale * np.sqrt(ref.size))
        assert err <= tol, err
        assert torch.equal(y, ops.lora_bgmv(gA, gB, gx, gi))
    # added to a base product: rows without an adapter keep the base's bits
    base = torch.from_numpy((rng.standard_normal((m, k)) * 0.05).astype(np.float16)).cuda().to(tdt)
    gi = torch.from_numpy(idx.astype(np.int32)).cuda()
    y = ops.lora_bgmv(gA, gB, gx, gi, base_weight=base, scale=0.5)
    plain = ops.lora_bgmv(gA, gB, gx, torch.full_like(gi, -1), base_weight=base)
    assert torch.equal(y[gi < 0], plain[gi < 0])
    want = plain.double() + 0.5 * torch.from_numpy(np.ascontiguousarray(ref.astype(np.float64))).cuda()
    assert float((y.double() - want).norm() / want.norm()) <= tol


@pytest.mark.parametrize("r", [8, 24, 40, 56])
def test_infinite_weight_beside_the_padding_of_the_rank(always, r):
    """The rank is padded to 16, 32 or 64: an infinity in the last rank row stays one in its column alone."""
    A = torch.ones((1, 64, r), dtype=torch.float16, device="cuda")
    B = torch.ones((1, r, 16), dtype=torch.float16, device="cuda")
    B[0, r - 1, 3] = float("inf")
    x = torch.ones((5, 64), dtype=torch.float16, device="cuda")
    assert _ffi.lib().triteia_hip_lora_ok(5, 1, 64, r, 16)
    y = ops.lora_bgmv(A, B, x, torch.zeros(5, dtype=torch.int32, device="cuda"))
    want = torch.full((5, 16), 64.0 * r, dtype=torch.float16, device="cuda")
    want[:, 3] = float("inf")
    assert torch.equal(y, want)


def test_which_calls_run_in_one_launch():
    ok = _ffi.lib().triteia_hip_lora_ok
    assert ok(1, 8, 1024, 16, 4096) and ok(100, 32, 1536, 16, 11008) and ok(600, 8, 2048, 32, 2048)
    assert not ok(1, 8, 4096, 16, 4096)                     # a workgroup would read more than the pair's second launch costs
    assert not ok(16, 8, 448, 16, 4096)                     # fewer steps than wavefronts
    assert not ok(16, 8, 1024, 128, 4096) and not ok(16, 8, 1056, 16, 4096) and not ok(4097, 8, 1024, 16, 4096) and not ok(16, 8, 1024, 16, 0)


@pytest.mark.parametrize("base", [False, True])
def test_refusals_of_the_entry_point(base):
    lib = _ffi.lib()
    t = torch.zeros(1 << 16, dtype=torch.float16, device="cuda")
    p = t.data_ptr()
    call = lambda y=p, x=p, T=4, k=64, r=8, m=64, xs=64: lib.triteia_hip_lora(y, m, x, xs, p, p, p, 0, T, 2, k, r, m, 1.0, int(base), 0, 0, None)
    assert call() == 0 and call(T=0) == 0 and call(m=0) == 0
    assert call(k=96) == _ffi.ERR_KERN_SHAPE and call(r=72, k=128) == _ffi.ERR_KERN_SHAPE and call(m=12) == _ffi.ERR_KERN_SHAPE
    assert call(x=p + 2) == _ffi.ERR_ARGUMENT and call(y=p + 8) == _ffi.ERR_ARGUMENT and call(xs=68) == _ffi.ERR_ARGUMENT and call(x=None) == _ffi.ERR_ARGUMENT
    torch.cuda.synchronize()
