"""The int8 RMSNorm on the device (rmsnorm_lane in forward.hip) against the oracle's, bit for bit, over
every element value beside every rms that a row holding it can have."""
import math

import numpy as np
import pytest
import torch

import jero_hip as J
import pyoracle as O

pytestmark = pytest.mark.gpu


def rows_of(r, rng):
    """Rows whose isqrt(mean square) is r, and in them every value that such a row can hold."""
    lo, hi = 512 * r * r, 512 * (r + 1) ** 2 - 1
    todo = [v for v in range(-128, 128) if v * v <= hi]
    rows = []
    while todo:
        take, ss = [], 0
        # as many values as still leave the sum of squares within reach of the others
        while todo and ss + todo[0] ** 2 <= hi and ss + todo[0] ** 2 + (511 - len(take)) * 16384 >= lo:
            ss += todo[0] ** 2
            take.append(todo.pop(0))
        if not take:
            todo.pop(0)  # only rows of r that hold nothing else hold it: none
            continue
        m = 512 - len(take)
        rest = min(max((lo + hi) // 2 - ss, 0), m * 16384)
        f = math.isqrt(rest // m) if m else 0
        more = (rest - m * f * f) // (2 * f + 1) if f < 128 else 0
        row = np.array(take + [-(f + 1)] * more + [-f] * (m - more), np.int64)
        assert lo <= int((row * row).sum()) <= hi
        rows.append(rng.permutation(row).astype(np.int8))
    return rows


def test_every_value_and_rms(dev):
    rng = np.random.default_rng(1)
    rows, pairs = [], 0
    for r in range(129):
        of_r = rows_of(r, rng) if r < 128 else [np.full(512, -128, np.int8)]
        pairs += len(np.unique(np.stack(of_r)))
        rows += of_r
    x = np.stack(rows)
    # rms 0 and 1 hold |v| <= 22 and 45, 2: 67, 3: 90, 4: 113, above that all 256 values
    assert pairs >= 45 + 91 + 135 + 181 + 227 + 123 * 256 + 1
    d = torch.from_numpy(x).to(dev)
    y = torch.full_like(d, 77)
    J.ForwardModel.rmsnorm(d, y)
    torch.cuda.synchronize()
    assert np.array_equal(y.cpu().numpy(), O.fwd_rmsnorm(x))
