"""What the native op binding must leave to the ops' Python path, and how it fails."""
import pytest
import torch

from triteia_amd.python import ops
from triteia_amd.python.capi._native import native
from triteia_amd.python.nn.linear import multi_delta_linear
from triteia_amd.workloads import random_activations, random_packed_deltas

pytestmark = pytest.mark.gpu
K, M_OUT, N, T, RANK = 128, 256, 3, 20, 8


@pytest.fixture(scope="module")
def layer():
    g = torch.Generator(device="cuda").manual_seed(1)
    rand = lambda *shape: (torch.randn(shape, generator=g, device="cuda") * 0.1).half()
    q, meta, s = random_packed_deltas(N, K, M_OUT, 2, "cuda")
    return dict(q=q, meta=meta, s=s, x=random_activations(T, K, 3, "cuda"), A=rand(N, K, RANK), B=rand(N, RANK, M_OUT), base=rand(M_OUT, K),
                idx=torch.arange(T, device="cuda", dtype=torch.int32) % (N + 1) - 1)


def calls(t, base):
    return {"sbmm": lambda: ops.sbmm_4bit_2_4_native(t["q"], t["x"], t["meta"], t["s"], t["idx"], base_weight=base),
            "lora": lambda: ops.lora_bgmv(t["A"], t["B"], t["x"], t["idx"], base_weight=base),
            "ldmm": lambda: ops.ldmm(t["idx"], t["x"], t["A"], t["B"], t["q"], t["meta"], t["s"], base_weight=base)}


@pytest.mark.parametrize("name", ["sbmm", "lora", "ldmm"])
def test_base_product_of_another_type_under_autocast(layer, name):
    """Autocast gives the base product its own type.  One that is not the activations' is refused, as by the ops' Python
    path; without a base weight, and where the types agree, autocast changes nothing."""
    plain, based = calls(layer, None)[name], calls(layer, layer["base"])[name]
    want, want_based = plain(), based()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        with pytest.raises(RuntimeError, match="float16"):
            based()
        assert torch.equal(plain(), want)
    with torch.autocast("cuda", dtype=torch.float16):
        assert torch.equal(based(), want_based)


def test_bf16_adapters_under_fp16_autocast(layer):
    t = {n: v.bfloat16() if n in ("x", "A", "B", "base") else v for n, v in layer.items()}
    based = calls(t, t["base"])["lora"]
    want = based()
    with torch.autocast("cuda", dtype=torch.float16):
        with pytest.raises(RuntimeError, match="float16"):
            based()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert torch.equal(based(), want)


def test_module_with_a_base_under_autocast(layer):
    mod = multi_delta_linear(K, M_OUT, N, with_base=True).cuda()
    for i in range(N):
        mod.load_delta(i, layer["q"][i], layer["meta"][i], layer["s"][i])
    mod.base.copy_(layer["base"])
    want = mod(layer["x"], layer["idx"])
    assert torch.equal(want, calls(layer, layer["base"])["sbmm"]())
    with torch.autocast("cuda", dtype=torch.bfloat16):
        with pytest.raises(RuntimeError, match="float16"):
            mod(layer["x"], layer["idx"])


def test_failed_launch_raises(layer):
    """An error that the HIP runtime reports for a launch (here one that the host has left behind: no such device) is
    raised by the op; the call after it works."""
    import ctypes

    from triteia_amd.python.capi import _ffi
    hip = ctypes.CDLL(_ffi.LIB_PATH)      # (symbols of the runtime that it is linked to)
    t = layer
    w = (torch.randn(64, 128, device="cuda") * 0.1).half()
    scale = torch.full((1, 128), 0.02, dtype=torch.float16, device="cuda")
    ops_ = dict(calls(t, None), matmul=lambda: ops.matmul_4bit_2_4(t["q"][0], t["x"], t["meta"][0], t["s"][0]),
                bmm=lambda: ops.bmm_4bit_2_4(t["q"], t["x"][:N].unsqueeze(1), t["meta"], t["s"]),
                pack=lambda: native().pack(w, scale)[0])
    for name, op in ops_.items():
        want = op()
        torch.cuda.synchronize()
        assert hip.hipSetDevice(1000) != 0
        with pytest.raises(RuntimeError, match="triteia_hip error 4"):
            op()
        assert torch.equal(op(), want), name


def test_more_deltas_than_a_plan_takes_are_refused_ahead_of_every_launch(layer):
    n = 8193
    q, meta, s = (torch.zeros(shape, dtype=dt, device="cuda") for shape, dt in
                  (((n, K // 32, 2 * M_OUT), torch.int32), ((n, M_OUT, K // 16), torch.int16), ((n, 1, M_OUT), torch.float16)))
    for base in (None, layer["base"]):
        assert native().sbmm(q, layer["x"], meta, s, layer["idx"], base) is None
        assert native().ldmm(layer["idx"], layer["x"], layer["A"], layer["B"], q, meta, s, base) is None
        with pytest.raises(RuntimeError, match="8192"):
            ops.sbmm_4bit_2_4_native(q, layer["x"], meta, s, layer["idx"], base_weight=base)


@pytest.mark.parametrize("accumulate", [False, True])
def test_capi_wrappers_of_the_lora_pair_and_the_packer(layer, accumulate):
    """capi.lora_scratch / lora_shrink / lora_expand and capi.pack_2_4: the same launches as the ops, hence the same bits."""
    from triteia_amd.python.capi import lora_expand, lora_scratch, lora_shrink, pack_2_4
    t = layer
    y = torch.matmul(t["x"], t["base"].t()) if accumulate else torch.empty((T, M_OUT), dtype=torch.float16, device="cuda")
    scratch = lora_scratch(T, t["A"])
    lora_shrink(t["x"], t["A"], t["idx"], scratch, accumulate)
    lora_expand(y, t["B"], scratch, K, accumulate, scale=0.5)
    assert torch.equal(y, ops.lora_bgmv(t["A"], t["B"], t["x"], t["idx"], base_weight=t["base"] if accumulate else None, scale=0.5))
    with pytest.raises(RuntimeError, match="lora_shrink"):
        lora_expand(y, t["B"], scratch, K, not accumulate)
    w = (torch.randn(96, 192, device="cuda") * 0.1).half()
    scale = torch.full((1, 192), 0.02, dtype=torch.float16, device="cuda")
    for got, want in zip(pack_2_4(w, scale), native().pack(w, scale)):
        assert torch.equal(got, want)
    odd = torch.empty(96 * 192 + 1, dtype=torch.float16, device="cuda")[1:].view(96, 192)     # starts inside a pair: copied
    odd.copy_(w)
    assert all(torch.equal(got, want) for got, want in zip(pack_2_4(odd, scale), native().pack(w, scale)))


def test_ldmm_with_the_lora_pair_on_a_second_stream():
    """A large batch with a base weight forks outside a capture and runs on one stream inside it: the same bits, call after
    call on new inputs; a launch that fails between the fork and the join raises, and the calls after it are right."""
    import ctypes

    from triteia_amd.python.capi import _ffi
    tokens, k, m, models, rank = 2049, 4096, 4096, 3, 16              # (the smallest batch of this layer, and one token)
    g = torch.Generator(device="cuda").manual_seed(2)
    rand = lambda *shape: (torch.randn(shape, generator=g, device="cuda") * 0.02).half()
    q, meta, s = random_packed_deltas(models, k, m, 4, "cuda")
    A, B, base = rand(models, k, rank), rand(models, rank, m), rand(m, k)
    x = torch.empty((tokens, k), dtype=torch.float16, device="cuda")
    idx = torch.empty(tokens, dtype=torch.int32, device="cuda")
    inputs = [(random_activations(tokens, k, 10 + i, "cuda"),
               torch.randint(-1, 2 * models, (tokens,), generator=g, device="cuda", dtype=torch.int32)) for i in range(4)]
    call = lambda: native().ldmm(idx, x, A, B, q, meta, s, base)

    def load(i):
        x.copy_(inputs[i][0])
        idx.copy_(inputs[i][1])

    load(0)
    call()
    torch.cuda.synchronize()
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.stream(stream), torch.cuda.graph(graph, stream=stream):
        captured = call()
    want = []
    for i in range(4):
        load(i)
        graph.replay()
        want.append(captured.clone())
    plain = torch.matmul(x, base.t())
    assert torch.equal(want[3][idx < 0], plain[idx < 0]) and not torch.equal(want[3], plain)
    for _ in range(3):                       # (nothing waits between the calls: each follows the copies and the call before it)
        got = []
        for i in range(4):
            load(i)
            got.append(call())
        for i in range(4):
            assert torch.equal(got[i], want[i]), i
    hip = ctypes.CDLL(_ffi.LIB_PATH)
    torch.cuda.synchronize()
    assert hip.hipSetDevice(1000) != 0       # (an error that the host has left behind)
    with pytest.raises(RuntimeError, match="triteia_hip error 4"):
        call()
    assert torch.equal(call(), want[3])
