"""_lib.operand hands a kernel the elements that reshape(shape).to(dtype).contiguous()
would, for every stride, type and shape, and refuses what that refuses."""

from __future__ import annotations

import math

import pytest
import torch

from FlagOS_mhc import _lib

BASE = torch.arange(2 * 3 * 4 * 6, dtype=torch.float32)


def _cases():
    t = BASE.view(2, 3, 4, 6)
    return [t, t.view(6, 4, 6), t.transpose(2, 3), t[:, :, ::2], t[:, 1:], t.permute(3, 0, 2, 1), t.expand(2, 3, 4, 6),
            BASE[:24].view(1, 24).expand(6, 24), t.to(torch.bfloat16), t.to(torch.float16).transpose(0, 1),
            t.double(), BASE[1:].as_strided((2, 5), (7, 1)), BASE[:0].view(0, 4)]


@pytest.mark.parametrize("i", range(len(_cases())))
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_operand_holds_the_same_elements(i, dtype):
    t = _cases()[i]
    shape = (t.numel(),) if i % 2 else (t.shape[0], -1) if t.numel() else (0, 4)
    shape = tuple(t.numel() // max(1, t.shape[0]) if s == -1 else s for s in shape)
    got, want = _lib.operand(t, shape, dtype), t.reshape(shape).to(dtype).contiguous()
    assert got.is_contiguous() and got.dtype == dtype and got.numel() == math.prod(shape)
    assert torch.equal(got.reshape(-1), want.reshape(-1))


def test_operand_refuses_other_sizes():
    for t in _cases():
        with pytest.raises(RuntimeError):
            _lib.operand(t, (t.numel() + 1,), t.dtype)
