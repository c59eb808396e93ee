"""The dense base product of the routed ops against the same product in 64 bits."""
import pytest
import torch

from tests.helpers import make_deltas, to_gpu
from triteia_amd.python import ops

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


# either side of each tile's tokens, a single chunk of K, K split over workgroups (few columns or a long K) and not, columns that
# leave the last feature group partly empty (96 features, m a multiple of 128), and the first batch that torch takes
@pytest.mark.parametrize("tokens,k,m", [(1, 64, 128), (16, 128, 384), (17, 4096, 256), (32, 192, 128), (33, 2048, 128), (64, 4160, 384),
                                        (65, 512, 1408), (128, 8192, 128), (129, 64, 128), (200, 1088, 3200), (256, 2048, 11008),
                                        (13, 11008, 4096), (256, 13824, 512), (257, 256, 128), (1, 1024, 1024)])
def test_base_product(tokens, k, m):
    x, w = _operands(tokens, k, m)
    _check(_base_only(x, w, _packed(k, m)), x, w)


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
    tokens, k, m = 16, 256, 128
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
