"""Host-side contract of the masked attention API (no GPU): rejections before any launch."""

import dataclasses

import pytest
import torch

from systems_for_llms_amd.attention import _validated_schedule, attention
from systems_for_llms_amd.masks import BlockSchedule, MaskSpec, compile_mask


def test_dispatch_rejections_before_launch():
    # attention_lab/test_interval_kernel.py:53-62
    with pytest.raises(ValueError, match="document"):
        attention(None, None, None, None, MaskSpec(same_document=True), implementation="interval")
    with pytest.raises(ValueError, match="implementation"):
        attention(None, None, None, None, MaskSpec(), implementation="other")
    with pytest.raises(TypeError, match="use_full_blocks"):
        attention(None, None, None, None, MaskSpec(), use_full_blocks=1)
    with pytest.raises(TypeError, match="spec"):
        attention(None, None, None, None, {"causal": True})


def test_cpu_tensors_rejected():
    q = torch.zeros(1, 1, 8, 64, dtype=torch.bfloat16)
    with pytest.raises(ValueError, match="same CUDA device"):
        attention(q, q, q, compile_mask(8, MaskSpec(causal=True)), MaskSpec(causal=True))


def test_schedule_validation():
    good = compile_mask(5, MaskSpec(causal=True), 16, 16)
    _validated_schedule(good)
    with pytest.raises(ValueError, match="block_q"):
        _validated_schedule(BlockSchedule(5, 24, 16, [0, 1], [0], [False]))
    with pytest.raises(ValueError, match="invalid CSR"):
        _validated_schedule(BlockSchedule(5, 16, 16, [0, 2], [0], [False]))
    with pytest.raises(ValueError, match="sorted"):
        _validated_schedule(BlockSchedule(40, 16, 16, [0, 2, 2, 2], [1, 0], [False, False]))
    with pytest.raises(TypeError, match="bool"):
        _validated_schedule(BlockSchedule(5, 16, 16, [0, 1], [0], [1]))


def test_schedule_entry_types_are_told_apart():
    good = BlockSchedule(40, 16, 16, [0, 1, 2, 3], [0, 1, 2], [False, True, True])
    _validated_schedule(good)
    for field, value, error in (("row_ptr", True, TypeError), ("col_idx", 1.0, TypeError), ("col_idx", True, TypeError),
                                ("full_blocks", 1, TypeError), ("col_idx", 1 << 31, ValueError)):
        entries = list(getattr(good, field))
        entries[1] = value
        with pytest.raises(error):
            _validated_schedule(dataclasses.replace(good, **{field: entries}))
