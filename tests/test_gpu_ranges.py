"""GPU parity at the sizes where launch plans change: remainders of tiles,
splits and waves, and the smallest and largest of each plan's range, against
the CPU oracle (tests/util.py's tolerances) or a float64 product of the same
operands."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import oracle as orc
from rxq4 import capi
from tests import util

pytestmark = pytest.mark.gpu


def dev(a: np.ndarray) -> torch.Tensor:
    a = np.ascontiguousarray(a)
    return torch.from_numpy(a.view(np.int16) if a.dtype == np.uint16 else a).cuda()


def host16(t: torch.Tensor) -> np.ndarray:
    return t.cpu().view(torch.int16).numpy().view(np.uint16)


# ------------------------------------------------- long rows, idle last waves
# Rows of more than 64 slots whose waves hold more than 16 KB: the rows of the
# ranges give 1022, 1021 and 1022 waves, so the last workgroup of four has
# waves without rows (they must not read past range 0).
@pytest.mark.parametrize("rows,K", [((2503, 2604), 13824), ((5101,), 13824), ((1, 5099, 3), 13824)])
def test_long_rows_with_idle_waves(rows, K):
    x = util.x_f16(7001, K)
    Ws = [util.weights(7002 + i, M, K) for i, M in enumerate(rows)]
    ys = [torch.empty(M, dtype=torch.float16, device="cuda") for M in rows]
    capi.gemv_multi_f16([(y, dev(W), M) for y, W, M in zip(ys, Ws, rows)], dev(x), K)
    for y, W, M in zip(ys, Ws, rows):
        pick = np.unique(np.r_[0, M // 2, max(0, M - 40):M])
        ref = orc.gemv_f64(np.ascontiguousarray(W[pick]), K, orc.bits_f16(x).astype(np.float32))
        assert util.rounded_ok(host16(y)[pick], ref).all(), (rows, M)
