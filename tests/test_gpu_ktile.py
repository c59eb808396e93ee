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


# Every build (tile of 16 tokens on eight and on four wavefronts, of 32, 48 and 64), K split over workgroups (`kernel` // 1000 shares) and not; whole
# tiles, last tiles of fewer 16-token tiles than the others, and last 16 tokens that start inside the tile before; one and two tokens to a
# matrix; fewer steps of K than wavefronts (k = 128: one) and steps that do not divide among them (9, 11)
@pytest.mark.parametrize("b,t,k,m,kernel", [
    (2, 13, 2688, 128, 1017), (1, 50, 10752, 1408, 4017), (1, 64, 11136, 1408, 4017), (17, 1, 8192, 512, 3017), (33, 2, 8192, 512, 1017),
    (1, 32, 4096, 1152, 1017), (1, 33, 4096, 1152, 1017),
    (2, 12, 128, 128, 1016), (4, 16, 2048, 640, 1016), (8, 12, 1408, 384, 1016), (2, 48, 1152, 2048, 1016), (2, 31, 1152, 2048, 1016), (3, 16, 8192, 128, 16016),
    (1, 63, 8192, 512, 8016),
    (64, 17, 128, 512, 1032), (20, 25, 384, 896, 1032), (5, 64, 896, 2048, 1032), (1, 129, 4096, 1152, 1032), (1, 1100, 512, 512, 1032), (1, 65, 8192, 640, 8032),
    (1, 611, 4352, 128, 3032),
    (1, 300, 1024, 4224, 1048), (1, 864, 896, 1280, 1048), (1, 740, 128, 1408, 1048), (1, 552, 9472, 640, 4048),
    (1, 530, 896, 5504, 1064), (1, 832, 896, 1920, 1064), (1, 913, 128, 1664, 1064), (1, 687, 11392, 768, 3064),
])
def test_against_the_oracle(monkeypatch, b, t, k, m, kernel):
    assert _ffi.lib().triteia_hip_uniform_ktile(m, b, t, k, 1) == kernel
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


@pytest.mark.parametrize("b,t,k,m", [(1, 37, 11008, 512), (3, 16, 8192, 128), (1, 687, 11392, 768)])
def test_without_room_for_the_shares_of_k(b, t, k, m):
    """No scratch, one that is too small and one that is not aligned: the tile that is best unsplit, whose sums the oracle checks and which are
    the same all three times; with room for them, the shares."""
    qw, meta, s, x = _case(b, t, k, m)
    gq, gm, gs, gx = to_gpu(qw, meta, s, x)
    lib = _ffi.lib()
    need = lib.triteia_hip_bmm_scratch_bytes(m, b, t, k)
    assert lib.triteia_hip_uniform_ktile(m, b, t, k, 1) > 2000 > lib.triteia_hip_uniform_ktile(m, b, t, k, 0) > 1000
    room = torch.empty(need + 256, dtype=torch.uint8, device="cuda")
    want = orc.bmm_4bit_2_4(qw, x, meta, s)

    def call(scratch, size):
        out = torch.full((b, t, m), 9.0, dtype=torch.float16, device="cuda")
        assert lib.triteia_hip_bmm_2_4_tokens_scratch(gx.data_ptr(), gq.data_ptr(), gm.data_ptr(), out.data_ptr(), gs.data_ptr(), m, b, t, k, scratch, size, 0,
                                                      torch.cuda.current_stream().cuda_stream) == 0
        check_close(out, want, what=f"ktile {b} x {t} tokens, {k} x {m}, scratch of {size} bytes")
        return out

    shares = lib.triteia_hip_uniform_ktile(m, b, t, k, 1) // 1000
    split = call(room.data_ptr(), need)
    unsplit = [call(None, 0), call(room.data_ptr(), 4 * shares * b * t * m - 1), call(room.data_ptr() + 4, need)]
    assert torch.equal(unsplit[0], unsplit[1]) and torch.equal(unsplit[0], unsplit[2])
    assert torch.equal(split, ops.bmm_4bit_2_4(gq, gx, gm, gs))
    # (the same exact products added up in another order, in fp32, and rounded once)
    assert ((unsplit[0].float() - split.float()).norm() / split.float().norm()).item() < 1e-4


def test_mul_2_4_and_a_graph():
    """mul_2_4 splits through a scratch of its binding's, as the op does.  A captured split replays."""
    t, k, m = 37, 11008, 512
    qw, meta, s, x = _case(1, t, k, m)
    gq, gm, gs, gx = to_gpu(qw[0], meta[0], s[0], x[0])
    split = ops.matmul_4bit_2_4(gq, gx, gm, gs)
    plain = torch.zeros((t, m), dtype=torch.float16, device="cuda")
    mul_2_4(gx, gq, gm, plain, gs, torch.zeros(m // 128 * 16, dtype=torch.int32, device="cuda"))
    assert torch.equal(plain, split)
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


@pytest.mark.parametrize("b,t,k,m", [(2, 31, 1152, 2048), (1, 63, 8192, 512), (1, 300, 1024, 4224), (1, 530, 896, 5504)])
def test_infinities_and_nan(monkeypatch, b, t, k, m):
    """They stay in their own rows (the rows that pad a tile are other tokens' again) and meet the same weights as on the streaming kernel."""
    qw, meta, s, x = _case(b, t, k, m)
    gq, gm, gs, gx = to_gpu(qw, meta, s, x)
    assert _ffi.lib().triteia_hip_uniform_ktile(m, b, t, k, 1) > 0
    clean = ops.bmm_4bit_2_4(gq, gx, gm, gs)
    rows = [0, t // 2, t - 1]
    gx[-1, rows[0], 5] = float("inf")
    gx[-1, rows[1], k - 1] = float("nan")
    gx[-1, rows[2], k // 2] = float("-inf")
    out = ops.bmm_4bit_2_4(gq, gx, gm, gs)
    kept = torch.ones((b, t), dtype=torch.bool, device="cuda")
    kept[-1, rows] = False
    assert torch.equal(out[kept], clean[kept])
    setknob(monkeypatch, "TRITEIA_HIP_KTILE", 0)
    other = ops.bmm_4bit_2_4(gq, gx, gm, gs)
    assert bool((~torch.isfinite(out[~kept])).any(-1).all())
    assert torch.equal(out.isnan(), other.isnan()) and torch.equal(out.isposinf(), other.isposinf()) and torch.equal(out.isneginf(), other.isneginf())


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
