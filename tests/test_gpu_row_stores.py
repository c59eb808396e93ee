"""The wide and the tile kernels turn their results through LDS into whole rows: token counts at the edges of a 16-token group, of a
tile and of a workgroup, a last group of column blocks that is not full, and the memory behind the last row."""
import pytest
import torch

from oracle import triteia_oracle as orc
from tests.helpers import activations, check_close, make_deltas, setknob, to_gpu
from triteia_amd.python import capi

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
