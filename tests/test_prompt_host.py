"""Host logic of the prompt GEMM (no GPU): the slot order of a weight's row tiles."""
from __future__ import annotations

import numpy as np
import pytest

from tilequant_amd import _native as nat


def _slots(counts, n_tc):
    rp = np.concatenate(([0], np.cumsum(counts))).astype(np.int32)
    out = np.full(len(counts) + 3, 77, np.int32)
    n = nat.load().tq_gemm_row_order(rp.ctypes.data, len(counts), n_tc, out.ctypes.data, out.size)
    return out[:n].tolist(), out[n:].tolist()


@pytest.mark.parametrize("seed", range(6))
def test_row_order_covers_every_row_tile_and_groups_the_heavy_ones(seed):
    rng = np.random.default_rng(seed)
    n_tr, n_tc = int(rng.integers(1, 60)), int(rng.integers(1, 80))
    counts = rng.integers(0, max(1, n_tc // 2), n_tr)
    counts[rng.random(n_tr) < 0.1 * seed] = n_tc
    slots, rest = _slots(counts, n_tc)
    heavy = [r for r in range(n_tr) if 3 * counts[r] >= 2 * n_tc]
    whole = -(-len(heavy) // 4) * 4
    assert len(slots) == n_tr + whole - len(heavy) and set(rest) <= {77}
    assert sorted(s for s in slots if s >= 0) == list(range(n_tr))
    assert sorted(s for s in slots[:whole] if s >= 0) == heavy and all(s >= 0 for s in slots[whole:])
    ordered = [counts[s] for s in slots if s >= 0]
    assert ordered == sorted(ordered, reverse=True)


def test_row_order_rejects_bad_arguments():
    lib = nat.load()
    rp, out = np.zeros(5, np.int32), np.zeros(7, np.int32)
    assert lib.tq_gemm_row_order(None, 4, 4, out.ctypes.data, 7) == -1
    assert lib.tq_gemm_row_order(rp.ctypes.data, 4, 4, out.ctypes.data, 6) == -1
    assert lib.tq_gemm_row_order(rp.ctypes.data, 0, 4, out.ctypes.data, 7) == -1


def test_prompt_entries_reject_bad_arguments_before_any_launch():
    lib = nat.load()
    assert lib.tq_act_quant_blocked(None, 64, 0, 0, 64, None, None, None, 0, None) == -1
    assert lib.tq_act_quant_blocked(1 << 20, 100, 0, 4, 100, 1 << 20, 1 << 20, None, 0, None) == -1
    assert lib.tq_act_quant_blocked(1 << 20, 68, 0, 100, 64, 1 << 20, 1 << 20, None, 0, None) == -3
    assert lib.tq_act_quant_blocked(1 << 20, 64, 0, 600, 64, 1 << 20, 1 << 20, None, 0, None) == -4
    fake = 1 << 20
    args = [fake, fake, fake, fake, fake, fake, fake, 128, 0, None, None, None, fake, 64, 0, None, 100, 64, 128, 1, 2, 1,
            None, 0, None, 0, 0, None]
    for at, value, code in ((16, -1, -1), (18, 100, -1), (8, 7, -2), (21, 5, -2), (13, 60, -1), (0, fake + 8, -3),
                            (2, fake + 4, -3), (5, None, -1)):
        bad = list(args)
        bad[at] = value
        assert lib.tq_gemm_mixed_blocked(*bad) == code, (at, value)
    assert lib.tq_gemm_mixed_blocked(*[fake if i == 22 else a for i, a in enumerate(args)]) == -1   # no slots
    assert lib.tq_prompt_forward(None) == -1
