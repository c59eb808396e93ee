"""CPU-side checks of the C-ABI library: it loads, exports every declared symbol, and rejects
bad problems before touching the GPU."""
import ctypes
import os
import re

import pytest

from tests.helpers import setknob
from triteia_amd.python.capi import _ffi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols():
    text = open(os.path.join(ROOT, "include", "triteia_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(triteia_hip_\w+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    names = declared_symbols()
    assert len(names) >= 12
    handle = ctypes.CDLL(_ffi.LIB_PATH)
    for n in names:
        assert hasattr(handle, n), f"{n} declared in include/triteia_hip.h but not exported"
    assert set(names) == set(_ffi.SIGNATURES), "ctypes table and header disagree"


def test_version_and_error_text():
    lib = _ffi.lib()
    assert lib.triteia_hip_version() >= 1000
    assert isinstance(_ffi.last_error(), str)


@pytest.mark.parametrize("m,n,k,gs,code", [
    (100, 16, 4096, -1, _ffi.ERR_PROB_SHAPE),      # m not a multiple of 128
    (4096, 16, 100, -1, _ffi.ERR_PROB_SHAPE),      # k not a multiple of 64
    (4096, 16, 4096, 32, _ffi.ERR_KERN_SHAPE),     # scale groups other than 128 dense k (groupsize 64) have no kernel
    (4096, 0, 4096, -1, 0),                        # empty problem is a no-op
])
def test_shape_errors_do_not_need_a_gpu(m, n, k, gs, code):
    lib = _ffi.lib()
    null = ctypes.c_void_p(0)
    rc = lib.triteia_hip_mul_2_4(null, null, null, null, null, m, n, k, null, gs, 0, null, -1, -1, -1, 16)
    assert rc == code
    if code:
        assert _ffi.last_error() != ""
    rc = lib.triteia_hip_bmm_2_4(null, null, null, null, null, m, n, k, null, gs, 0, null, -1, -1, -1, 16)
    assert rc == code


def test_grouped_scales_are_for_the_single_matrix_product():
    """groupsize 64 (scales per column and 128 dense k, marlin_nm.cu:68,102-111) is taken by mul_2_4; the batched and
    routed launchers, whose group iteration the reference itself has commented out (triteia_nm_bmm.cu:69-71,
    triteia_nm_sbmm.cu:70-72), answer ERR_KERN_SHAPE; K must be whole groups."""
    lib = _ffi.lib()
    null = ctypes.c_void_p(0)
    assert lib.triteia_hip_mul_2_4(null, null, null, null, null, 4096, 0, 4096, null, 64, 0, null, -1, -1, -1, 16) == 0
    assert lib.triteia_hip_mul_2_4(null, null, null, null, null, 4096, 16, 4096, null, 64, 0, null, -1, -1, -1, 16) == _ffi.ERR_ARGUMENT
    assert lib.triteia_hip_mul_2_4(null, null, null, null, null, 4096, 16, 4160, null, 64, 0, null, -1, -1, -1, 16) == _ffi.ERR_PROB_SHAPE
    assert lib.triteia_hip_bmm_2_4(null, null, null, null, null, 4096, 16, 4096, null, 64, 0, null, -1, -1, -1, 16) == _ffi.ERR_KERN_SHAPE
    assert lib.triteia_hip_sbmm_2_4(*([null] * 8), 4096, 16, 4096, 1, null, 64, 0, null, -1, -1, -1, 16) == _ffi.ERR_KERN_SHAPE


def test_other_argument_errors():
    lib = _ffi.lib()
    null = ctypes.c_void_p(0)
    # bgmv: narrow side too wide / not a multiple of 8
    assert lib.triteia_hip_bgmv(null, null, null, null, 4, 4096, 256, 1, 0, 1.0, 0, null) == _ffi.ERR_KERN_SHAPE
    assert "No suitable kernel" in _ffi.last_error()
    assert lib.triteia_hip_bgmv(null, null, null, null, 4, 4096, 12, 1, 0, 1.0, 0, null) == _ffi.ERR_KERN_SHAPE
    assert lib.triteia_hip_bgmv(null, null, null, null, 4, 4096, 16, 1, 3, 1.0, 0, null) == _ffi.ERR_PROB_SHAPE
    # routed sbmm: workspace too small, too many deltas
    need = lib.triteia_hip_sbmm_routed_workspace_bytes(64, 16)
    assert need == 4 * (8 + 4 * (16 + 64 // 16) + 4 * (64 // 33 + 1) + 64 + 4 * (16 + 64 // 16) + 4 * (16 + 64 // 64))
    assert lib.triteia_hip_plan_tile_tokens(8, 8) == 16
    assert lib.triteia_hip_plan_tile_tokens(64, 16) == 16       # at most 4 tokens per delta on average
    assert lib.triteia_hip_plan_tile_tokens(256, 16) == 32
    assert lib.triteia_hip_plan_tile_tokens(4096, 4) == 64
    assert lib.triteia_hip_planned_tile_kernel(256, 32, 11008, 4096) == 32      # cfg3: wide layer, 32-token tiles
    assert lib.triteia_hip_planned_tile_kernel(256, 16, 4096, 4096) == 0        # narrow layer: not on the wide kernel ...
    assert lib.triteia_hip_planned_ktile(256, 16, 4096, 4096) == 32             # ... the K-splitting tiles
    assert lib.triteia_hip_planned_ktile(256, 32, 11008, 4096) == 0
    assert lib.triteia_hip_planned_tile_kernel(2048, 32, 11008, 4096) == 64
    assert lib.triteia_hip_planned_tile_kernel(2048, 64, 28672, 8192) == 64     # 64-token tiles on a long K as well
    # 1024 tokens over 8 deltas: the plan is cut in 32-token tiles and lists 64-token tiles beside them for wide layers
    assert lib.triteia_hip_plan_tile_tokens(1024, 8) == 32
    assert lib.triteia_hip_planned_tile_kernel(1024, 8, 11008, 4096) == 64
    assert lib.triteia_hip_planned_tile_kernel(1024, 8, 4096, 4096) == 32
    assert lib.triteia_hip_planned_tile_kernel(1024, 32, 11008, 4096) == 32     # 32 tokens per delta: no 64-token tiles
    one = ctypes.c_void_p(16)
    assert lib.triteia_hip_route_plan(one, 0, 16, 64, one, need - 1, 0, null) == _ffi.ERR_ARGUMENT
    assert lib.triteia_hip_route_plan(one, 0, 100000, 64, one, 1 << 30, 0, null) == _ffi.ERR_KERN_SHAPE
    assert lib.triteia_hip_sgmv_tmp_size(7) == 420
    assert lib.triteia_hip_sgmv(null, null, null, null, null, 0, 4096, 16, 0, 0, null) == 0


def test_python_wrappers_refuse_cpu_tensors():
    import torch
    from triteia_amd.python.ops import matmul_4bit_2_4
    x = torch.zeros(2, 128, dtype=torch.float16)
    with pytest.raises(RuntimeError, match="GPU tensor"):
        matmul_4bit_2_4(torch.zeros(4, 512, dtype=torch.int32), x, torch.zeros(256, 8, dtype=torch.int16),
                        torch.ones(1, 256, dtype=torch.float16))


def test_product_code_never_reaches_for_the_oracle():
    """The CPU restatement is the checker: nothing in the package, its import alias, the C sources
    or the header may import, read or mention it."""
    import pathlib
    root = pathlib.Path(__file__).resolve().parents[1]
    offenders = []
    for top in ("triteia_amd", "triteia", "include"):
        for path in (root / top).rglob("*"):
            if path.suffix in (".py", ".h", ".hip") and "oracle" in path.read_text(errors="replace"):
                offenders.append(str(path.relative_to(root)))
    assert not offenders, offenders


def test_dispatch_queries_at_the_documented_points():
    """Which kernel a call would run is a pure host-side function of the shapes and the knobs: the answers at the
    benchmark's points, as the documentation states them (no GPU involved)."""
    lib = _ffi.lib()
    _ffi.reload_env()
    uniform = lib.triteia_hip_uniform_kernel          # (m, batch, tokens, k, with_scratch)
    tiles = lib.triteia_hip_uniform_ktile
    assert uniform(4096, 1, 16, 4096, 1) == 16         # cfg0: K of 4096 is too short for a split across workgroups; 16-column shares
    assert uniform(4096, 1, 17, 4096, 1) == 0          # more than one 16-token pass: column blocks of 128 ...
    assert tiles(4096, 1, 17, 4096, 1) == 1017         # ... on K-splitting tiles of 16 tokens, eight wavefronts
    assert uniform(11008, 1, 16, 4096, 1) == 16        # 86 column blocks: shares of 64 columns
    assert uniform(28672, 1, 16, 4096, 1) == 0         # 224 column blocks: the streaming kernel
    assert tiles(28672, 1, 16, 4096, 1) == 0
    assert uniform(4096, 8, 1, 4096, 1) == 0           # cfg1: a workgroup per CU already
    assert tiles(4096, 8, 1, 4096, 1) == 0
    assert uniform(8192, 1, 16, 8192, 1) == 1004       # long K, few workgroups: K split in 4 ...
    assert uniform(8192, 1, 16, 8192, 0) == 16         # ... only with a scratch buffer (without: shares of 32 columns)
    assert lib.triteia_hip_bmm_scratch_bytes(8192, 1, 16, 8192) == 4 * 16 * 8192 * 4
    assert lib.triteia_hip_bmm_scratch_bytes(4096, 1, 16, 4096) == 0
    assert uniform(4096, 1, 1024, 4096, 1) == 33       # 32-token tiles on eight wavefronts (one workgroup per CU)
    assert uniform(4096, 1, 1536, 4096, 1) == 65       # 64-token tiles on eight wavefronts
    assert uniform(4096, 1, 4096, 4096, 1) == 64       # 64-token tiles, two workgroups per CU
    assert uniform(2048, 1, 8192, 4096, 1) == 256      # a narrow layer: one round of 256-token tiles
    assert uniform(28672, 1, 4096, 8192, 1) == 64      # several rounds: 64-token tiles, two workgroups per CU
    assert uniform(4096, 1, 128, 4096, 1) == 0 and tiles(4096, 1, 128, 4096, 1) == 0   # 256 16-token passes: the streaming kernel
    assert tiles(4096, 1, 129, 4096, 1) == 1032 and tiles(4096, 1, 768, 4096, 1) == 1048 and tiles(4096, 1, 1024, 4096, 1) == 0
    assert uniform(4096, 1, 37, 11008, 1) == 1004 and tiles(4096, 1, 37, 11008, 1) == 4032   # long K, few workgroups: K split ...
    assert uniform(4096, 1, 37, 11008, 0) == 0 and tiles(4096, 1, 37, 11008, 0) == 1017      # ... only with a scratch buffer
    assert tiles(4096, 1, 11, 8192, 1) == 0 and tiles(4096, 1, 16, 4096, 1) == 0             # a single matrix of 16 tokens and fewer
    assert tiles(2048, 4, 11, 2048, 1) == 0 and tiles(2048, 4, 12, 2048, 1) > 0              # several: from 12 on ...
    assert tiles(2048, 4, 2, 8192, 1) == 0 and tiles(5120, 2, 1, 13824, 1) > 0               # ... with fewer on a long K past 64 column blocks
    assert tiles(1024, 1, 599, 1024, 1) == 0 and tiles(1024, 1, 640, 1024, 1) > 0            # less than 2^22 weights: from 600 tokens on
    assert tiles(11008, 1, 256, 4096, 1) > 0 and tiles(8192, 1, 769, 8192, 1) == 0           # 832 tiles of 64 tokens x 128 columns
    assert tiles(4096, 1, 129, 4160, 1) == 0           # half a K step of 128 at the end
    assert uniform(100, 1, 16, 4096, 1) == -1          # not a legal shape
    routed = lib.triteia_hip_routed_in_kernel          # (tokens, deltas, m, k)
    assert routed(64, 16, 4096, 4096) == 1             # cfg2: one launch, no plan
    assert routed(256, 16, 4096, 4096) == 1
    assert routed(65, 17, 4096, 4096) == 0             # above 64 tokens only up to 16 deltas
    assert routed(64, 32, 4096, 4096) == 1             # a small layer: the plan's launch would not pay
    assert routed(64, 32, 11008, 4096) == 0            # 33 .. 64 tokens over many deltas of a large layer: planned ...
    assert lib.triteia_hip_plan_tile_tokens(64, 32) == 32   # ... in 32-token tiles (a skewed batch's hot delta in one tile)
    assert routed(32, 32, 11008, 4096) == 1
    assert routed(1, 16, 4096, 4096) == 2              # one token: column shares, routed in the kernel
    assert routed(4, 16, 4096, 4096) == 2              # at most four deltas in use: 128 column blocks on the bound
    assert routed(8, 16, 4096, 4096) == 1              # up to eight: the streaming kernel
    assert routed(16, 4, 4096, 4096) == 1              # four tokens per delta: weights requested ahead of the routing
    assert routed(256, 32, 11008, 4096) == 0           # cfg3: planned ...
    assert lib.triteia_hip_planned_tile_kernel(256, 32, 11008, 4096) == 32   # ... and its 32-token tiles go to the wide kernel
    assert lib.triteia_hip_planned_tile_kernel(256, 16, 4096, 4096) == 0     # a narrow layer does not
    assert lib.triteia_hip_planned_tile_kernel(1024, 16, 4096, 4096) == 32   # except for a thousand tokens in full tiles ...
    planned = lib.triteia_hip_planned_ktile            # (tokens, deltas, m, k): first of all
    assert planned(1024, 16, 4096, 4096) == 64         # ... which at 768 tiles of 64 tokens x 128 columns the K-splitting tiles have
    assert planned(1024, 16, 4096, 2048) == 0 and planned(1024, 16, 8192, 4096) == 0 and planned(1024, 40, 4096, 4096) == 0
    assert planned(1500, 16, 5120, 4480) == 0 and planned(1500, 16, 5120, 4608) == 64   # up to 1536 from k = 4500 on
    assert planned(500, 22, 1024, 8192) == 32 and planned(279, 5, 4096, 11008) == 32
    assert planned(256, 32, 11008, 4096) == 0 and planned(1000, 32, 11008, 4096) == 0   # the wide kernel
    assert lib.triteia_hip_plan_tile_tokens(64, 16) == 16
    assert lib.triteia_hip_plan_tile_tokens(4096, 16) == 64


def test_the_plans_k_splitting_tiles_have_an_upper_end():
    """triteia_hip_planned_ktile (tokens, deltas, m, k): batches that the streaming kernel would take alone at any size; of those whose hot
    deltas the wide kernel takes, by column groups of the layer, tokens per delta and units of 64 tokens x 128 columns."""
    lib = _ffi.lib()
    _ffi.reload_env()
    ktile = lib.triteia_hip_planned_ktile
    assert ktile(513, 32, 4096, 4096) == 32 and ktile(1536, 4, 4096, 4096) > 0
    for tokens in (4096, 8192, 32768, 65536):            # eight and twelve column groups
        assert ktile(tokens, 16, 4096, 4096) == 0 and ktile(tokens, 4, 4096, 4096) == 0 and ktile(tokens, 4, 6144, 8192) == 0
    assert ktile(32768, 16, 1536, 4096) == 64            # three column groups: at any number of tokens
    assert ktile(4096, 64, 4096, 4096) == 64             # 64 tokens per delta
    assert ktile(6000, 64, 4096, 4096) == 64 and ktile(6200, 64, 4096, 4096) == 0   # either side of 96
    # over 8 deltas, units of tokens and half a tile per delta x column blocks: up to 4096 on 28 blocks (seven groups), 3072 on 33 and 60
    for blocks, units in ((28, 4096), (33, 3072), (60, 3072)):
        most = units * 64 // blocks - 32 * 8
        assert ktile(most, 8, 128 * blocks, 4096) == 64 and ktile(most + 64, 8, 128 * blocks, 4096) == 0, blocks


def test_small_batches_leave_the_workspace():
    """triteia_hip_routed_leaves_workspace (tokens, deltas, m, k): what callers that share a workspace over streams may rely on."""
    lib = _ffi.lib()
    _ffi.reload_env()
    for k, m in ((4096, 4096), (11008, 4096), (13824, 13824)):
        for tokens in (1, 16, 32, 33, 64):
            for deltas in (1, 2, 16, 17, 64):
                planned = tokens > 32 and deltas > 16 and k * m >= 1 << 25
                assert lib.triteia_hip_routed_leaves_workspace(tokens, deltas, m, k) == (not planned), (tokens, deltas, m, k)
    assert lib.triteia_hip_routed_leaves_workspace(256, 16, 4096, 4096) == 1 and lib.triteia_hip_routed_leaves_workspace(257, 16, 4096, 4096) == 0
    assert lib.triteia_hip_routed_leaves_workspace(65, 17, 4096, 4096) == 0
    # a plan that only a workspace of the call's own allows
    assert lib.triteia_hip_routed_in_kernel(32, 1, 4096, 11008) == 0 and lib.triteia_hip_routed_in_kernel(64, 16, 4096, 4096) == 1


def test_the_scratch_of_uniform_launches_is_enough_for_either_kernel(monkeypatch):
    """triteia_hip_bmm_scratch_bytes knows nothing of the activations' alignment, which decides between the K-splitting tiles and the kernels
    before: it holds the shares of K of both."""
    lib = _ffi.lib()
    shapes = [(m, batch, tokens, k) for m in (128, 512, 768, 1536, 2560) for batch in (1, 2, 3, 8) for tokens in (1, 12, 17, 24, 31, 37, 64, 200)
              for k in (4096, 8192, 11008, 14592, 17024, 23296)]
    _ffi.reload_env()
    both = [lib.triteia_hip_bmm_scratch_bytes(*shape) for shape in shapes]
    setknob(monkeypatch, "TRITEIA_HIP_KTILE", 0)
    before = [lib.triteia_hip_bmm_scratch_bytes(*shape) for shape in shapes]
    assert all(a >= b for a, b in zip(both, before)) and sum(b > 0 for b in before) > 100


def test_which_base_products_the_library_takes(monkeypatch):
    """triteia_hip_dense_ok (tokens, m, k): not where the library that torch calls measures ahead, and not at all under DENSE = 0."""
    lib = _ffi.lib()
    _ffi.reload_env()
    ok = lib.triteia_hip_dense_ok
    taken = [(13, 4096, 11008), (256, 11008, 4096), (256, 5120, 13824), (200, 4096, 4096), (128, 28672, 8192), (32, 2048, 2048), (17, 128, 64),
             (128, 2048, 2048), (128, 9728, 5888), (193, 9728, 5888), (160, 4096, 11008), (256, 13824, 8192)]
    left = [(129, 9728, 5888), (192, 9728, 5888), (160, 28672, 8192), (256, 28672, 8192), (129, 16384, 8192),       # the library is ahead
            (257, 4096, 4096), (16, 512, 512), (13, 4096, 96)]                                                      # the kernel cannot or never did
    assert all(ok(*shape) for shape in taken) and not any(ok(*shape) for shape in left)
    setknob(monkeypatch, "TRITEIA_HIP_DENSE", 0)
    assert not any(ok(*shape) for shape in taken)
    setknob(monkeypatch, "TRITEIA_HIP_DENSE", 2)
    assert [ok(*shape) for shape in left] == [1] * 5 + [0] * 3


def test_which_lora_calls_take_one_launch():
    """triteia_hip_lora_ok (tokens, adapters, k, r, m): not where a workgroup's columns are many, however little it reads for the first product."""
    ok = _ffi.lib().triteia_hip_lora_ok
    _ffi.reload_env()
    taken = [(16, 16, 1024, 16, 2048), (600, 8, 2048, 32, 2048), (100, 32, 1536, 16, 11008), (16, 16, 1024, 16, 12928), (1375, 46, 1280, 64, 4096),
             (4, 64, 512, 8, 13824), (600, 8, 2048, 32, 13824)]
    left = [(62, 62, 1024, 16, 12928), (63, 62, 1024, 16, 12928), (60, 54, 768, 8, 10496), (101, 58, 896, 8, 13824),     # few tokens an adapter
            (1375, 46, 1280, 64, 13312), (1334, 45, 2432, 8, 13056), (307, 62, 1536, 64, 13440), (1603, 60, 1152, 8, 11648)]
    assert [c for c in taken if not ok(*c)] == [] and [c for c in left if ok(*c)] == []


def test_bench_refuses_more_than_one_gpu():
    import subprocess
    import sys
    res = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"], capture_output=True, text=True)
    assert res.returncode == 2
    assert "ONE GPU" in res.stderr


def test_sizes_past_a_grid_are_refused_before_the_launch():
    lib = _ffi.lib()
    null = ctypes.c_void_p(0)
    expand = lambda m: lib.triteia_hip_lora_expand(null, m, null, null, 1, 1, 32, 8, m, 1.0, 0, 0, 0, null)
    assert expand(65535 * 256) == _ffi.ERR_ARGUMENT             # (null pointers come after the sizes)
    assert expand(65535 * 256 + 8) == _ffi.ERR_KERN_SHAPE
    pack = lambda k, m: lib.triteia_hip_pack_2_4(null, null, null, null, null, k, m, 0, null)
    assert pack(32, 2 ** 30 - 128) == _ffi.ERR_ARGUMENT
    assert pack(32, 2 ** 30) == _ffi.ERR_PROB_SHAPE


def test_environment_is_read_in_one_place():
    """The knobs' table is the only reader: no kernel is picked by a variable that it does not list."""
    csrc = os.path.join(ROOT, "triteia_amd", "csrc")
    calls = {f: len(re.findall(r"\bgetenv\s*\(", open(os.path.join(csrc, f)).read())) for f in sorted(os.listdir(csrc))}
    assert {f: n for f, n in calls.items() if n} == {"triteia_hip.hip": 1}


def test_every_entry_point_has_a_caller():
    """What the library exports is called by the binding, the tests or the benchmark."""
    text = ""
    for folder in (os.path.join(ROOT, "triteia_amd"), os.path.join(ROOT, "tests"), ROOT):
        for base, _, files in os.walk(folder):
            if folder == ROOT and base != ROOT:
                continue
            for f in files:
                if f.endswith((".py", ".cpp")):
                    source = open(os.path.join(base, f)).read()
                    text += source.split("_lib = None")[1] if f == "_ffi.py" else source      # (not the table itself)
    unused = [n for n in _ffi.SIGNATURES if not re.search(n + r"\b", text) and not (n.endswith("_bf16") and n[:-5] in text)]
    assert not unused
