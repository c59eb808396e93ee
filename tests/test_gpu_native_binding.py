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
