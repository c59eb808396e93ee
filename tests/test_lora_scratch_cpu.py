"""What capi.lora_expand accepts as its scratch (checked on the host, ahead of the device)."""
import pytest
import torch

from triteia_amd.python.capi import lora_expand


@pytest.mark.parametrize("left_by", [None, (5, 2, 64, 8, True), (4, 3, 64, 8, True), (4, 2, 96, 8, True), (4, 2, 64, 16, True), (4, 2, 64, 8, False)])
def test_scratch_of_other_sizes_is_refused(left_by):
    y, b = torch.zeros(4, 128, dtype=torch.float16), torch.zeros(2, 8, 128, dtype=torch.float16)
    scratch = torch.zeros(1 << 16, dtype=torch.uint8)
    if left_by:
        scratch.lora_pair = left_by
    with pytest.raises(RuntimeError, match="lora_shrink"):
        lora_expand(y, b, scratch, 64, True)


def test_scratch_of_the_same_sizes_reaches_the_device_check():
    y, b = torch.zeros(4, 128, dtype=torch.float16), torch.zeros(2, 8, 128, dtype=torch.float16)
    scratch = torch.zeros(1 << 16, dtype=torch.uint8)
    scratch.lora_pair = (4, 2, 64, 8, True)
    with pytest.raises(RuntimeError, match="GPU tensor"):
        lora_expand(y, b, scratch, 64, True)
