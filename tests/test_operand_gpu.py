"""The plan calls' operand checks: the short path and the full one agree on
every kind of tensor (what they return, or the error)."""
import numpy as np
import pytest

from helpers import capi

pytestmark = pytest.mark.gpu


def _tensors(torch):
    base = torch.zeros(128, 96, dtype=torch.bfloat16, device="cuda")
    return {
        "whole": base, "wider": base[:, :64], "offset": base[3:, 32:], "one row": base[:1], "every other row": base[::2],
        "transposed": base.t(), "column step": base[:, ::2], "expanded": base[:1].expand(128, 96),
        "flat": base.view(-1), "flat short": base.view(-1)[:1000], "flat step": base.view(-1)[::2],
        "3-D": base.view(4, 32, 96), "scalar": base[0, 0], "empty": base[:0],
        "f32": torch.zeros(128, 96, device="cuda"), "host": torch.zeros(128, 96, dtype=torch.bfloat16),
        "parameter": torch.nn.Parameter(base), "numpy": np.zeros((128, 96), np.uint16), "none": None, "address": 1 << 20,
    }


@pytest.mark.parametrize("rows,cols,ld", [(128, 96, None), (64, 64, None), (128, 96, 96), (64, 64, 96), (64, 64, 64),
                                          (1, 96, None), (1, 12288, 12288), (0, 0, None), (1, 64, 128), (64, 96, 192)])
def test_short_and_full_checks_agree(rows, cols, ld):
    import torch
    capi.load()
    for name, t in _tensors(torch).items():
        got = []
        for fn in (capi._operand, capi._operand_checked):
            try:
                got.append(fn(t, "x", 2, rows, cols, ld, 0))
            except (TypeError, ValueError, IndexError) as e:
                got.append((type(e), str(e)))
        assert got[0] == got[1], (name, rows, cols, ld, got)
