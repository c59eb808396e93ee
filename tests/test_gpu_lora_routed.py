"""The LoRA pair that routes by itself (lora_shrink / lora_expand) against the oracle, at the edges of its tiles, splits
and layouts.  (Its product in one launch, which takes small calls otherwise, is off.)"""
import numpy as np
import pytest
import torch

from oracle import triteia_oracle as orc
from tests.helpers import setknob
from triteia_amd.python import ops
from triteia_amd.python.capi import _ffi, lora_scratch, lora_shrink
from triteia_amd.python.capi._native import native

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def pair(monkeypatch):
    setknob(monkeypatch, "TRITEIA_HIP_LORA_FUSED", 0)


@pytest.mark.parametrize("T,M,k,r,m", [
    (1, 1, 32, 8, 8),             # smallest: one step of k, half a rank tile, one 16-byte piece of output
    (17, 3, 96, 16, 264),         # a tile and one token; an output block of 8 columns
    (65, 2, 512, 24, 520),        # 64-token tiles and a rest; a rank that is no power of two (no swizzle)
    (130, 3, 1056, 64, 256),      # steps of k that do not divide among the splits
    (200, 70, 256, 32, 128),      # more than 64 bins; most adapters with a handful of tokens
    (300, 4, 4128, 128, 640),     # 32-token tiles of the widest rank
    (4096, 5, 128, 40, 72),       # the largest batch it takes
    (90, 1024, 64, 8, 64),        # the most adapters it takes
])
@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
def test_lora_pair_against_the_oracle(T, M, k, r, m, dtype):
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
    assert lora_scratch(T, gA) is not None and not _ffi.lib().triteia_hip_lora_ok(T, M, k, r, m)
    # one rounding of the intermediate and one of the result: 2^-11 (2^-8) relative each, and the oracle's own
    tol = 2e-2 if dtype == "bf16" else 2e-3
    scale = max(1e-6, float(np.sqrt(np.mean(np.square(ref.astype(np.float64))))))
    for gi in (torch.from_numpy(idx.astype(np.int32)).cuda(), torch.from_numpy(idx.astype(np.int64)).cuda()):
        for fn in (ops.lora_bgmv, ops.lora_sgmv, ops.lora_sgmv_routed):
            y = fn(gA, gB, gx, gi)
            assert y.dtype == tdt and bool((y[gi < 0] == 0).all())
            err = np.linalg.norm(y.float().cpu().numpy().astype(np.float64) - ref) / (scale * np.sqrt(ref.size))
            assert err <= tol, (fn.__name__, err)
    # added to a base product: rows without an adapter keep the base's bits
    base = torch.from_numpy((rng.standard_normal((m, k)) * 0.05).astype(np.float16)).cuda().to(tdt)
    gi = torch.from_numpy(idx.astype(np.int32)).cuda()
    plain = torch.matmul(gx, base.t())
    y = ops.lora_bgmv(gA, gB, gx, gi, base_weight=base, scale=0.5)
    assert torch.equal(y[gi < 0], plain[gi < 0])
    want = plain.double() + 0.5 * torch.from_numpy(np.ascontiguousarray(ref.astype(np.float64))).cuda()
    assert float((y.double() - want).norm() / want.norm()) <= tol


def test_lora_shapes_it_leaves_to_the_other_kernels():
    A = torch.zeros((2, 4096, 16), dtype=torch.float16, device="cuda")
    assert lora_scratch(4097, A) is None                                  # more tokens than indices fit in LDS
    assert lora_scratch(8, A[:, :4088]) is None                           # k no multiple of 32
    assert lora_scratch(8, A[:, :, :12]) is None                          # r no multiple of 8


def test_lora_tensors_inside_a_16_byte_word():
    """Views that start inside 16 bytes are left to the kernels of the other interfaces, with the same values."""
    g = torch.Generator(device="cuda").manual_seed(3)
    A, B, x = (torch.randn(s, generator=g, device="cuda").to(torch.float16) * 0.1 for s in ((3, 64, 16), (3, 16, 72), (20, 64)))
    idx = torch.arange(20, device="cuda").remainder(4).sub(1).sort().values.to(torch.int32)
    want = ops.lora_forloop(A, B, x, idx)

    def shifted(t):
        buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
        buf[1:].copy_(t.reshape(-1))
        return buf[1:].view(t.shape)
    for args in ((shifted(A), B, x), (A, shifted(B), x), (A, B, shifted(x))):
        assert native().lora(*args, idx, None, 1.0) is None
    y = ops.lora_bgmv(A, B, shifted(x), idx)
    assert float((y - want).float().norm() / want.float().norm()) <= 2e-3     # as above
    with pytest.raises(RuntimeError, match="16-byte aligned"):
        lora_shrink(shifted(x), A, idx, lora_scratch(20, A), False)


@pytest.mark.parametrize("r", [8, 24, 40, 72])
def test_lora_infinite_weight_beside_the_padding_of_the_rank(r):
    """The rank is padded to 16, 32, 64 or 128: an infinity in the last rank row stays one in its column alone."""
    A = torch.ones((1, 32, r), dtype=torch.float16, device="cuda")
    B = torch.ones((1, r, 16), dtype=torch.float16, device="cuda")
    B[0, r - 1, 3] = float("inf")
    x = torch.ones((5, 32), dtype=torch.float16, device="cuda")
    y = ops.lora_bgmv(A, B, x, torch.zeros(5, dtype=torch.int32, device="cuda"))
    want = torch.full((5, 16), 32.0 * r, dtype=torch.float16, device="cuda")
    want[:, 3] = float("inf")
    assert torch.equal(y, want)
