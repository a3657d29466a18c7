"""How the 64-head MLA attention's workgroups are dealt to the chip (vx_mla_attn64_item), on the CPU."""
import ctypes as C

import pytest

XCDS, CUS = 8, 32


def _deal(hiplib, splits, batch, groups):
    f, out = hiplib.vx_mla_attn64_deal, (C.c_uint32 * 3)()
    f.argtypes, f.restype = [C.c_uint32] * 4 + [C.POINTER(C.c_uint32)], None
    items = []
    for block in range((splits * batch * groups + 7) // 8 * 8):
        f(block, splits, batch, groups, out)
        items.append(tuple(out))
    return items


def _makespan(cost):
    """Workgroup i of `cost` goes to XCD i % 8, there to the CU that is free first (a CU holds one)."""
    free = [[0.0] * CUS for _ in range(XCDS)]
    for i, c in enumerate(cost):
        x = free[i % XCDS]
        x[x.index(min(x))] += c
    return max(max(x) for x in free)


@pytest.mark.parametrize("splits,batch,groups", [(1, 1, 1), (8, 16, 2), (7, 17, 2), (9, 28, 1), (14, 19, 1), (64, 5, 1),
                                                 (28, 5, 2), (64, 32, 2), (3, 43, 2)])
def test_every_item_is_dealt_once(hiplib, splits, batch, groups):
    got = [it for it in _deal(hiplib, splits, batch, groups) if it[0] < splits]
    assert sorted(got) == [(s, b, g) for s in range(splits) for b in range(batch) for g in range(groups)]


@pytest.mark.parametrize("batch", range(1, 33))
@pytest.mark.parametrize("s_max,shortest", [(3401, 0.5), (3401, 0.1), (801, 0.5)])
def test_unequal_lengths_past_one_round(hiplib, batch, s_max, shortest):
    """Lengths from s_max down to `shortest` of it, DeepSeek-V3's two head groups, splits of 256 or more workgroups:
    the longest CU takes no longer than with the grid dealt split by split within sequence by sequence of each head
    group, as a plain (splits, sequences, groups) grid is. An item costs 13 us and 1.4 per 32-position chunk, an
    empty one 4."""
    groups = 2
    splits = min(64, -(-256 // (batch * groups)))
    chunk = (-(-s_max // splits) + 31) // 32 * 32
    lengths = [s_max - int((1 - shortest) * s_max * b / max(1, batch - 1)) for b in range(batch)]

    def cost(it):
        n = min(lengths[it[1]] - it[0] * chunk, chunk) if it[0] < splits else 0
        return 13 + 1.4 * -(-n // 32) if n > 0 else 4.0

    plain = _makespan([cost((s, b, g)) for g in range(groups) for b in range(batch) for s in range(splits)])
    assert _makespan([cost(it) for it in _deal(hiplib, splits, batch, groups)]) <= plain * 1.001
