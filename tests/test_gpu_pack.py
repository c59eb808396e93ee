"""The packing kernel against the torch codec, byte for byte (the CPU tests hold the codec exact against the oracle)."""
import pytest
import torch

from triteia_amd.python.capi._native import native
from triteia_amd.python.ops.utils.generator import fp16_to_sparse
from triteia_amd.python.ops.utils.sparsity import mask_creator, prune_pack_2_4, unpack_nibbles

pytestmark = pytest.mark.gpu


# edges: half a column block (m % 128 = 64), a single packed row, packed rows that leave wavefronts of a block idle
@pytest.mark.parametrize("k,m", [(32, 64), (64, 192), (288, 128), (512, 320), (4096, 1024)])
@pytest.mark.parametrize("values", ["normal", "ties", "special"])
def test_pack_kernel_gives_the_codecs_bytes(k, m, values):
    g = torch.Generator().manual_seed(k * m)
    w = torch.randn((k, m), generator=g).to(torch.float16)
    s = (w.abs().amax(0, keepdim=True) * (2 / 15))
    if values == "ties":               # few distinct magnitudes of either sign, zeros among them: ties in most groups
        w = torch.randint(-3, 4, (k, m), generator=g).to(torch.float16)
        s = torch.full((1, m), 0.5, dtype=torch.float16)
    elif values == "special":          # what a broken checkpoint holds: zero scales, infinities, NaNs, tiny and huge values
        pool = torch.tensor([0.0, -0.0, 1.0, -65504.0, 6e-8, float("inf"), float("-inf"), float("nan")], dtype=torch.float16)
        w = pool[torch.randint(0, len(pool), (k, m), generator=g)]
        s[:, ::3] = 0.0
    w, s = w.cuda(), s.cuda()
    got = prune_pack_2_4(w, s)
    # (an explicit mask takes the codec's own steps on the same device)
    want = prune_pack_2_4(w, s, mask=mask_creator(w.t().contiguous()))
    for a, b, name in zip(got, want, ("qweight", "meta", "scales", "meta_raw")):
        assert a.dtype == b.dtype and a.shape == b.shape
        # (the scales are handed through: compared as bytes, for their NaNs)
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8)), name


def test_packing_inside_a_trace():
    """A trace follows torch's operations: it records the codec, and answers for other weights than those it was made with."""
    g = torch.Generator(device="cuda").manual_seed(5)
    # (whole multiples of the scale: torch's fuser may leave out the rounding of the quotient to fp16)
    first, second = ((torch.randint(-8, 8, (64, 128), generator=g, device="cuda") * 0.5).half() for _ in range(2))
    scale = torch.full((1, 128), 0.5, dtype=torch.float16, device="cuda")
    traced = torch.jit.trace(prune_pack_2_4, (first, scale))
    for w in (first, second):
        for got, want in zip(traced(w, scale), prune_pack_2_4(w, scale)):
            assert torch.equal(got, want)
    assert native().pack(first, scale) is not None         # (the kernel, outside a trace)


def _quantised(w, s):
    """The codec's integers 0 .. 15 of weights [k, m] and scales [1, m]."""
    return (torch.round(w / s).to(torch.int64) + 8).clamp(0, 15).to(torch.uint8)


@pytest.mark.parametrize("scales", ["negative", "infinite", "nan", "subnormal", "zero"])
def test_pack_kernel_on_unusual_scales(scales):
    g = torch.Generator().manual_seed(9)
    w = torch.randn((128, 192), generator=g).to(torch.float16)
    w[::7] *= 6e-8                                                     # (subnormal weights among the others)
    w[5::16] = float("inf")
    w[6::16] = float("nan")
    s = {"negative": -w.abs().nan_to_num(1.0, 1.0).amax(0, keepdim=True) * (2 / 15), "infinite": torch.full((1, 192), float("inf")),
         "nan": torch.full((1, 192), float("nan")), "subnormal": torch.randint(1, 1024, (1, 192), generator=g) * 2.0 ** -24,
         "zero": torch.zeros((1, 192))}[scales].to(torch.float16)
    if scales in ("infinite", "zero"):
        s[:, ::2] = -s[:, ::2]
    w, s = w.cuda(), s.cuda()
    got, want = prune_pack_2_4(w, s), prune_pack_2_4(w, s, mask=mask_creator(w.t().contiguous()))
    for a, b in zip(got, want):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


def test_pack_kernels_quotient_on_every_pair_of_fp16_values():
    """Every weight with every scale, both all 2^16 bit patterns: two weights a group behind two zeros, so that the weights
    are the two kept (a tie keeps the later)."""
    every = torch.arange(65536, device="cuda", dtype=torch.int32).to(torch.int16).view(torch.float16)
    s = every.reshape(1, -1)
    rows = 1024                                                        # weights per pass: 2048 dense k x 65536 columns, 256 MB
    for first in range(0, 65536, rows):
        v = every[first:first + rows].reshape(rows // 2, 2)
        w = torch.cat([torch.zeros_like(v), v], 1).reshape(-1, 1).expand(-1, 65536).contiguous()
        qweight, _, _ = native().pack(w, s)
        got = unpack_nibbles(qweight)
        want = _quantised(every[first:first + rows].reshape(-1, 1), s)
        assert torch.equal(got, want), f"weights {first} .. {first + rows - 1}"
        print(f"[pairs] weights {first} .. {first + rows - 1}", flush=True)


@pytest.mark.parametrize("shape", [(96,), (1, 192), (192, 1)])
def test_fp16_to_sparse_in_one_call_and_step_by_step(shape):
    """What the one native call answers is what the moves, views and the packing give one by one, and it answers for plain tensors on
    the current GPU only."""
    g = torch.Generator(device="cuda").manual_seed(9)
    m = max(shape) // 64 * 64
    w = (torch.randn((160, m), generator=g, device="cuda") * 0.02).half()
    s = (w.abs().amax(0) * (2 / 15)).reshape([m if d > 1 else 1 for d in shape])
    got = fp16_to_sparse(w, s)
    packed = prune_pack_2_4(w, s.reshape(1, -1))
    assert got[0] is w and got[2].data_ptr() == s.data_ptr()
    for a, b in zip(got, (w, packed[0], packed[2], packed[1], packed[3])):
        assert a.shape == b.shape and a.dtype == b.dtype and torch.equal(a, b)
    assert native().sparse(w, s) is not None
    wide = torch.zeros((160, 2 * m), dtype=torch.float16, device="cuda")
    wide[:, :m] = w
    for args in ((wide[:, :m], s), (w.float(), s), (w, s.float()), (w.cpu(), s), (w, s.cpu()), (w, s[:-1] if s.dim() == 1 else s.flatten()[:-1]),
                 (w[:-1], s), (w, s.clone().requires_grad_())):
        assert native().sparse(*args) is None
    for a, b in zip(fp16_to_sparse(wide[:, :m], s.cpu()), got):
        assert torch.equal(a, b)


def test_fp16_to_sparse_follows_function_modes():
    class Seen(torch.overrides.TorchFunctionMode):
        calls = 0

        def __torch_function__(self, func, types, args=(), kwargs=None):
            Seen.calls += 1
            return func(*args, **(kwargs or {}))

    w, s = torch.ones((64, 128), dtype=torch.float16, device="cuda"), torch.ones((1, 128), dtype=torch.float16, device="cuda")
    want = fp16_to_sparse(w, s)
    with Seen():
        got = fp16_to_sparse(w, s)
    assert Seen.calls > 0
    for a, b in zip(got, want):
        assert torch.equal(a, b)
