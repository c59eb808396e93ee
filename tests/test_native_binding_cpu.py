"""The native op binding with arguments that it leaves to the Python path: anything that is not exactly a torch tensor,
in any position, comes back as None (no GPU needed: the arguments are looked at before anything else)."""
import numpy as np
import pytest
import torch

from triteia_amd.python import ops
from triteia_amd.python.capi._native import native


class Subclass(torch.Tensor):
    """Any subclass: it may give every operation another meaning."""


# function -> its tensor arguments, and what follows them
FUNCTIONS = {"matmul": (4, ()), "bmm": (4, ()), "sbmm": (5, (None,)), "lora": (4, (None, 1.0)), "ldmm": (7, (None,)), "pack": (2, ()),
             "sparse": (2, ())}
STRANGE = {"none": None, "list": [0, 1], "array": np.zeros(3, dtype=np.int32), "number": 3, "text": "x", "object": object(),
           "subclass": torch.zeros(2, 2).as_subclass(Subclass)}


@pytest.mark.parametrize("what", sorted(STRANGE))
@pytest.mark.parametrize("name", sorted(FUNCTIONS))
def test_arguments_that_are_no_plain_tensors(name, what):
    tensors, rest = FUNCTIONS[name]
    fn = getattr(native(), name)
    plain = [torch.zeros(2, 2) for _ in range(tensors)] + list(rest)
    assert fn(*plain) is None                                   # (tensors of the CPU)
    for i in range(len(plain)):
        assert fn(*plain[:i], STRANGE[what], *plain[i + 1:]) is None
    assert fn(*[STRANGE[what]] * len(plain)) is None


@pytest.mark.parametrize("count", [0, 1, 3, 7, 9, 40])
def test_other_numbers_of_arguments(count):
    for name in FUNCTIONS:
        for arg in (None, torch.zeros(2, 2), 1.0):
            if count != FUNCTIONS[name][0] + len(FUNCTIONS[name][1]):
                assert getattr(native(), name)(*[arg] * count) is None


def test_ops_raise_for_arguments_of_another_kind():
    t = torch.zeros(2, 64, dtype=torch.float16)
    q, meta, s = torch.zeros(1, 2, 256, dtype=torch.int32), torch.zeros(1, 128, 4, dtype=torch.int16), torch.zeros(1, 1, 128, dtype=torch.float16)
    for indices in ([1, 2], np.zeros(2, dtype=np.int32), None):
        with pytest.raises((AttributeError, TypeError)):
            ops.sbmm_4bit_2_4_native(q, t, meta, s, indices)
    with pytest.raises((AttributeError, TypeError)):
        ops.matmul_4bit_2_4(q[0], [0.0], meta[0], s[0])
    with pytest.raises(RuntimeError, match="GPU tensor"):
        ops.matmul_4bit_2_4(q[0], t.as_subclass(Subclass), meta[0], s[0])
