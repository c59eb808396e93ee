"""The wide and the tile kernels turn their results through LDS into whole rows: token counts at the edges of a 16-token group, of a
tile and of a workgroup, a last group of column blocks that is not full, and the memory behind the last row."""
import numpy as np
import pytest
import torch

from oracle import triteia_oracle as orc
from tests.helpers import activations, check_close, make_deltas, setknob, to_gpu
from triteia_amd.python import capi
from triteia_amd.python.capi import _ffi

pytestmark = pytest.mark.gpu
ALWAYS, NEVER = "1000000000", "0"
# kernel -> the most units of 32-token tiles, the most that split K inside a workgroup (of 32 and 64 tokens), the tile kernel
KERNELS = {"wide64": (NEVER, NEVER, NEVER, "0"), "wide64ks": (NEVER, NEVER, ALWAYS, "0"), "wide32": (ALWAYS, NEVER, NEVER, "0"),
           "wide32ks": (ALWAYS, ALWAYS, NEVER, "0"), "tile256": (NEVER, NEVER, NEVER, "2")}


@pytest.mark.parametrize("kernel", sorted(KERNELS))
def test_rows_and_what_lies_behind_them(monkeypatch, kernel):
    most32, split32, split64, tile256 = KERNELS[kernel]
    for name, value in (("WIDE_MIN_UNITS", "1"), ("WIDE32_MIN_UNITS", "1"), ("WIDE32_MAX_UNITS", most32), ("WIDE32_KSPLIT_MAX_UNITS", split32),
                        ("WIDE64_KSPLIT_MAX_UNITS", split64), ("TILE256", tile256), ("TILE256_MIN_UNITS", "1"), ("KTILE", "0")):
        setknob(monkeypatch, "TRITEIA_HIP_" + name, value)
    k, m = 384, 640
    qw, meta, s = make_deltas(1, k, m, 61)
    gq, gm, gs = to_gpu(qw[0], meta[0], s[0])
    workspace = torch.zeros(m // 128 * 16, dtype=torch.int32, device="cuda")
    for n in (64, 65, 79, 80, 81, 112, 127, 128, 129, 255, 257):
        print(f"row stores {kernel} n={n}", flush=True)
        x = activations(n, k, 62 + n)
        out = torch.full((n + 16, m), 7.0, dtype=torch.float16, device="cuda")
        capi.mul_2_4(to_gpu(x)[0], gq, gm, out[:n], gs, workspace)
        torch.cuda.synchronize()
        check_close(out[:n], orc.matmul_4bit_2_4(qw[0], x, meta[0], s[0]), what=f"{kernel} n={n}")
        assert bool((out[n:] == 7.0).all()), f"{kernel} n={n}: written behind the last row"


# builds that a plan launches -> knobs, what triteia_hip_planned_tile_kernel says (0: the plan's wide tiles on the 64-token build and the rest on
# the streaming kernel; ALL64: one list of 64-token tiles)
PLANS = {"plan32": (dict(MID_DEPTH=1, PLAN_BIG=0), 32), "plan32deep": (dict(MID_DEPTH=2, PLAN_BIG=0), 32), "plan64": (dict(MID_DEPTH=1, PLAN_BIG=2), 64),
         "wide": (dict(MID=0, PLAN_WIDE_MIN_UNITS=1, PLAN_ALL64=0), 0), "wide_all": (dict(MID=0, PLAN_WIDE_MIN_UNITS=1, PLAN_ALL64=1), 0)}


@pytest.mark.parametrize("build", sorted(PLANS))
def test_rows_that_are_added_to(monkeypatch, build):
    """The builds that a plan launches, added to what the rows hold: old values turn the other way, and slots behind a delta's last token repeat its row."""
    knobs, tile = PLANS[build]
    for name, value in dict(PLAN_KTILE=0, MID_MIN_UNITS=1, MID_MIN_COLUMN_GROUPS=1, MID_MIN_HALF_TOKENS=0, **knobs).items():
        setknob(monkeypatch, "TRITEIA_HIP_" + name, value)
    k, m, counts = 384, 640, [1, 15, 16, 17, 0, 33, 63, 64, 65, 130]
    idx = np.concatenate([np.full(c, d, dtype=np.int32) for d, c in enumerate(counts)] + [np.full(9, -1, dtype=np.int32)])
    idx = np.random.default_rng(71).permutation(idx)
    n = len(idx)
    lib = _ffi.lib()
    assert lib.triteia_hip_planned_ktile(n, len(counts), m, k) == 0 and lib.triteia_hip_planned_tile_kernel(n, len(counts), m, k) == tile
    qw, meta, s = make_deltas(len(counts), k, m, 72)
    x, old = activations(n, k, 73), activations(n + 16, m, 74)
    gq, gm, gs, gx, gi, out = to_gpu(qw, meta, s, x, idx, old)
    before = out.clone()
    plan = capi.route_plan(gi, len(counts))
    print(f"row stores {build}, added", flush=True)
    capi.sbmm_2_4_planned(gx, gq, gm, out[:n], gs, plan, accumulate=True)
    torch.cuda.synchronize()
    want = old[:n].astype(np.float64) + orc.sbmm_4bit_2_4(qw, x, meta, s, idx)
    for d in range(len(counts)):
        if counts[d]:
            check_close(out[:n][gi == d], want[idx == d], what=f"{build}, delta {d} of {counts[d]} tokens")
    assert torch.equal(out[:n][gi < 0], before[:n][gi < 0]) and torch.equal(out[n:], before[n:])
