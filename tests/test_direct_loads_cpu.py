"""Direct loads from global memory to LDS in the built library's own machine code: a scalar write of M0, which holds the LDS address,
needs one wait state ahead of the load that uses it, and a scalar base written by the vector unit five."""
import os
import re
import shutil
import subprocess

import pytest

from triteia_amd import build

OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")


def _kernels(tmp_path):
    """{kernel: its instructions} of the built library."""
    if not os.path.exists(OBJDUMP):
        pytest.skip(f"{OBJDUMP} is not installed")
    build.ensure_built()
    lib = shutil.copy(build.LIB, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", lib], cwd=tmp_path, check=True, capture_output=True)
    objects = [p for p in tmp_path.iterdir() if p.name.endswith("gfx950")]
    assert len(objects) == 1, objects
    text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(objects[0])], check=True, capture_output=True, text=True).stdout
    kernels, name = {}, None
    for line in text.splitlines():
        head = re.match(r"^[0-9a-f]+ <(.*)>:", line)
        if head:
            name = kernels.setdefault(head.group(1), [])
        elif name is not None and line.startswith("\t"):
            name.append(line.split("//")[0].strip())
    return kernels


def test_wait_states_ahead_of_direct_loads(tmp_path):
    seen, early, base = set(), [], []
    for kernel, code in _kernels(tmp_path).items():
        for i, instruction in enumerate(code):
            if not instruction.startswith("global_load_lds"):
                continue
            seen.add(kernel)
            before = code[max(0, i - 5):i]
            if re.match(r"\S+ m0\b", before[-1]):
                early.append((kernel, before[-1], instruction))
            scalars = re.search(r"s\[(\d+):(\d+)\]", instruction)
            if scalars:
                base += [(kernel, b, instruction) for b in before if re.match(rf"v_\S+ s(\[?)({scalars.group(1)}|{scalars.group(2)})\b", b)]
    assert not early, f"{len(early)} loads right behind their write of M0: {early[0]}"
    assert not base, f"{len(base)} loads within five instructions of their base: {base[0]}"
    # (the kernels that bring their tiles this way are all in there)
    for part in ("sparse24_wide_kernel", "sparse24_tile256_kernel", "sparse24_ktile_kernel", "sparse24_ktile_plan_kernel", "dense_base_kernel", "lora_shrink_kernel",
                 "lora_fused_kernel"):
        assert any(part in kernel for kernel in seen), part
