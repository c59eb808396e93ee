"""The dense base product of the routed ops against the same product in 64 bits."""
import pytest
import torch

from tests.helpers import make_deltas, setknob, to_gpu
from triteia_amd.python import ops
from triteia_amd.python.capi import _ffi

pytestmark = pytest.mark.gpu


def _operands(tokens, k, m, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed + tokens * k + m)
    x = torch.randn((tokens, k), generator=g, device="cuda").half()
    w = (torch.randn((m, k), generator=g, device="cuda") * 0.05).half()
    return x, w


def _packed(k, m):
    return to_gpu(*make_deltas(1, k, m, 3))


def _base_only(x, w, packed):
    """All tokens without a delta: the op's result is the base product."""
    q, meta, s = packed
    none = torch.full((x.shape[0],), -1, dtype=torch.int32, device="cuda")
    return ops.sbmm_4bit_2_4_native(q, x, meta, s, none, base_weight=w)


def _check(y, x, w):
    want = x.double() @ w.double().t()
    # the result's rounding to fp16 (2^-11 of it, 2^-25 below the normal range) and k roundings of fp32 partial sums, each at most
    # 2^-24 of the sum of the magnitudes
    bound = want.abs() * 2.0 ** -11 + 2.0 ** -25 + (x.double().abs() @ w.double().abs().t()) * (x.shape[1] * 2.0 ** -24)
    worst = ((y.double() - want).abs() / bound).max().item()
    assert worst <= 1.0, worst


def _dense(x, w):
    """triteia_hip_dense itself; columns of any multiple of 8."""
    lib = _ffi.lib()
    (tokens, k), m = x.shape, w.shape[0]
    size = lib.triteia_hip_dense_scratch_bytes(tokens, m, k)
    scratch = torch.empty(max(size, 16), dtype=torch.uint8, device="cuda")
    y = torch.full((tokens + 1, m), 9.0, dtype=torch.float16, device="cuda")
    assert lib.triteia_hip_dense(x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), y.data_ptr(), tokens, m, k, scratch.data_ptr() if size else None, size, 0,
                                 torch.cuda.current_stream().cuda_stream) == 0
    assert bool((y[tokens] == 9.0).all())
    return y[:tokens]


# Every tile (tokens x features), K split over workgroups or not, walks over K that start at the first chunk or spread around its
# chunks (from 2^24 weights on), with a last tile and a last feature group that are partly empty
@pytest.mark.parametrize("tile,split,spread,tokens,k,m", [
    ((16, 32), False, False, 2, 1152, 912), ((16, 32), False, True, 8, 2368, 7152), ((16, 32), True, False, 1, 2880, 368), ((16, 32), True, True, 13, 6592, 2704),
    ((16, 64), False, False, 2, 128, 8248), ((16, 64), False, True, 5, 1600, 10576), ((16, 64), True, False, 1, 3200, 744), ((16, 64), True, True, 15, 3648, 4600),
    ((32, 32), False, False, 17, 64, 8), ((32, 32), False, True, 20, 2112, 7952), ((32, 32), True, False, 17, 1408, 8), ((32, 32), True, True, 18, 6336, 2704),
    ((32, 64), False, False, 17, 64, 8296), ((32, 64), False, True, 17, 1600, 10536), ((32, 64), True, False, 23, 2048, 1400), ((32, 64), True, True, 17, 6336, 2656),
    ((64, 32), False, False, 33, 64, 8), ((64, 32), False, True, 33, 2432, 6920), ((64, 32), True, False, 34, 1152, 8),
    ((64, 64), False, False, 131, 64, 2736), ((64, 64), False, True, 37, 1920, 8752), ((64, 64), True, False, 67, 3072, 328), ((64, 64), True, True, 37, 4480, 3752),
    ((64, 96), False, False, 195, 64, 4120), ((64, 96), True, False, 194, 3456, 648), ((64, 96), True, True, 33, 5632, 2984),
    ((128, 64), False, False, 66, 64, 8200), ((128, 64), True, False, 66, 3072, 696), ((128, 64), True, True, 65, 6528, 2576),
    ((128, 96), False, False, 129, 64, 8384), ((128, 96), True, False, 131, 5056, 1400), ((128, 96), True, True, 67, 2752, 6136),
    ((128, 128), False, False, 129, 64, 12336), ((128, 128), True, False, 131, 7360, 1552), ((128, 128), True, True, 138, 7360, 2280),
    # whole tiles
    ((16, 64), True, True, 16, 8192, 8192), ((32, 64), True, True, 32, 4096, 4096), ((64, 96), True, True, 64, 4096, 11008), ((128, 96), False, False, 256, 4096, 11008),
])
def test_every_tile(tile, split, spread, tokens, k, m):
    code = _ffi.lib().triteia_hip_dense_tile(tokens, m, k)
    assert (code % 1000, code // 1000 % 1000) == tile and (code // 2000000 > 1, bool(code // 1000000 & 1)) == (split, spread), code
    x, w = _operands(tokens, k, m)
    y = _dense(x, w)
    _check(y, x, w)
    assert torch.equal(y, _dense(x, w))


# through the op: the smallest and largest batches, a single chunk of K, K split over workgroups (few columns or a long K) and not, columns that leave
# the last feature group partly empty (96 features, m a multiple of 128)
@pytest.mark.parametrize("tokens,k,m", [(17, 4096, 256), (32, 192, 128), (33, 2048, 128), (64, 4160, 384),
                                        (65, 512, 1408), (128, 8192, 128), (129, 64, 128), (200, 1088, 3200), (256, 2048, 11008),
                                        (13, 11008, 4096), (256, 13824, 512), (1, 1024, 1024)])
def test_base_product(tokens, k, m):
    assert _ffi.lib().triteia_hip_dense_ok(tokens, m, k)
    x, w = _operands(tokens, k, m)
    y = _base_only(x, w, _packed(k, m))
    _check(y, x, w)
    assert torch.equal(y, _dense(x, w))


@pytest.mark.parametrize("tokens,k,m", [(1, 64, 128), (16, 128, 384), (257, 256, 128), (160, 8192, 16384)])
def test_base_product_that_stays_with_torch(tokens, k, m):
    """Up to 16 tokens on less than 2^20 weights, more than 256 tokens, and where its library is ahead."""
    assert not _ffi.lib().triteia_hip_dense_ok(tokens, m, k)
    x, w = _operands(tokens, k, m)
    assert torch.equal(_base_only(x, w, _packed(k, m)), torch.matmul(x, w.t()))


def test_the_knob_gives_the_product_to_torch(monkeypatch):
    tokens, k, m = 13, 11008, 512                          # (K split over workgroups: other bits than torch's)
    x, w = _operands(tokens, k, m)
    packed = _packed(k, m)
    own = _base_only(x, w, packed)
    setknob(monkeypatch, "TRITEIA_HIP_DENSE", 0)
    assert torch.equal(_base_only(x, w, packed), torch.matmul(x, w.t())) and not torch.equal(own, torch.matmul(x, w.t()))


def test_rows_do_not_depend_on_the_batch_where_nothing_is_split_or_spread():
    k, m = 1024, 8448                                      # (33 feature groups of 256 and more: unsplit; less than 2^24 weights)
    x, w = _operands(256, k, m)
    lib = _ffi.lib()
    batches = [t for t in range(1, 257) if lib.triteia_hip_dense_tile(t, m, k) // 1000000 == 2]
    assert len({lib.triteia_hip_dense_tile(t, m, k) for t in batches}) > 3
    whole = _dense(x, w) if 256 in batches else None
    assert whole is not None
    for t in batches[::13]:
        assert torch.equal(_dense(x[:t], w), whole[:t]), t


@pytest.mark.parametrize("tokens,k,m", [(13, 11008, 512), (33, 2048, 1288), (131, 5056, 1400), (200, 1088, 3200)])
def test_infinities_and_nan(tokens, k, m):
    """They stay in their own rows and columns: the rows and features that pad a tile are others again."""
    x, w = _operands(tokens, k, m)
    clean = _dense(x, w)
    x[0, 3], x[tokens - 1, k - 1], x[tokens // 2, k // 2] = float("inf"), float("nan"), float("-inf")
    w[m - 1, 7] = float("nan")
    w[5, k - 2] = float("inf")
    y, want = _dense(x, w), x.double() @ w.double().t()
    assert torch.equal(y.isnan(), want.isnan()) and torch.equal(y.isposinf(), want.isposinf()) and torch.equal(y.isneginf(), want.isneginf())
    rows = torch.ones(tokens, dtype=torch.bool, device="cuda")
    rows[[0, tokens - 1, tokens // 2]] = False
    columns = torch.ones(m, dtype=torch.bool, device="cuda")
    columns[[m - 1, 5]] = False
    assert torch.equal(y[rows][:, columns], clean[rows][:, columns])


def test_base_product_of_views():
    """Rows with a gap between them run as they lie; rows and tensors that are not aligned to 16 bytes go to torch."""
    tokens, k, m = 24, 320, 256
    x, w = _operands(tokens, k, m)
    packed = _packed(k, m)
    wide = torch.full((m, k + 40), float("nan"), dtype=torch.float16, device="cuda")
    for gap in (slice(0, k), slice(8, 8 + k), slice(3, 3 + k)):
        wide[:, gap] = w
        _check(_base_only(x, wide[:, gap], packed), x, w)
    odd = torch.full((m, k + 1), float("nan"), dtype=torch.float16, device="cuda")
    odd[:, 1:] = w
    _check(_base_only(x, odd[:, 1:], packed), x, w)
    columns = w.t().contiguous().t()                      # the weight stored [k, m]
    _check(_base_only(x, columns, packed), x, w)
    shifted = torch.empty(tokens * k + 1, dtype=torch.float16, device="cuda")[1:].view(tokens, k)
    shifted.copy_(x)
    _check(_base_only(shifted, w, packed), x, w)
    _check(_base_only(x.t().contiguous().t(), w, packed), x, w)


def test_base_product_with_a_gradient():
    """Autograd records torch's product, as it always has."""
    tokens, k, m = 24, 256, 128
    assert _ffi.lib().triteia_hip_dense_ok(tokens, m, k)
    x, w = _operands(tokens, k, m)
    w.requires_grad_(True)
    y = _base_only(x, w, _packed(k, m))
    assert y.requires_grad
    y.sum().backward()
    assert torch.allclose(w.grad.float(), x.float().sum(0).expand(m, k), rtol=1e-2, atol=1e-2)
    with torch.no_grad():
        assert not _base_only(x, w, _packed(k, m)).requires_grad


def test_base_product_in_a_graph():
    tokens, k, m = 20, 4096, 256                           # (two launches: K is split)
    x, w = _operands(tokens, k, m)
    packed = _packed(k, m)
    want = _base_only(x, w, packed)
    none = torch.full((tokens,), -1, dtype=torch.int32, device="cuda")
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        y = ops.sbmm_4bit_2_4_native(packed[0], x, packed[1], packed[2], none, base_weight=w)
    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
        assert torch.equal(_base_only(x, w, packed), want)


def test_base_product_under_tunable_op(tmp_path):
    """A process that has torch tune its products gets torch's, tuned or not."""
    tokens, k, m = 13, 11008, 512                          # (K split over workgroups: other bits than torch's)
    x, w = _operands(tokens, k, m)
    packed = _packed(k, m)
    tunable = torch.cuda.tunable
    assert not tunable.is_enabled()
    plain = _base_only(x, w, packed)
    tuning = tunable.tuning_is_enabled()
    tunable.set_filename(str(tmp_path / "results.csv"))    # (read when it is switched on; not the working folder's)
    tunable.tuning_enable(False)
    tunable.enable(True)
    try:
        y, want = _base_only(x, w, packed), torch.matmul(x, w.t())
    finally:
        tunable.enable(False)
        tunable.tuning_enable(tuning)
    assert torch.equal(y, want)
    assert not torch.equal(plain, want)
    assert torch.equal(_base_only(x, w, packed), plain)
