"""The lane offsets of the MN-major GEMMs' loads, 32-bit and modulo 2^32, over row strides: up to kMaxDescLd the descriptor's
range alone leaves out the K rows past the last (and the lanes that start past M or N), and the loads masked lane by lane,
which take over there, leave them out at any stride the entry points take."""
import os
import re

import pytest

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nano-gpic_amd", "csrc", "gemm.hip")
OOB = 1 << 31


def _max_desc_ld():
    m = re.search(r"constexpr int64_t kMaxDescLd = int64_t\(1\) << (\d+);", open(SRC).read())
    assert m, "gemm.hip states the longest row stride whose K tail the descriptor masks"
    return 1 << int(m.group(1))


def _read(K, ld, el, masked):
    """(rows of the first K tile whose load is in range for a lane that starts inside M, for one that starts at kOOB)."""
    tile, step = 128 // el, 16 // el
    num = K * ld * el
    inside, outside = [], []
    for row in range(tile):
        i, m = divmod(row, step)   # load i, the lane's row of it
        base, rest = m * ld * el, i * step * ld * el
        if masked and row >= K:
            offs = OOB, OOB
        else:
            offs = (base + rest) % 2 ** 32, (OOB + rest) % 2 ** 32
        if offs[0] < num:
            inside.append(row)
        if offs[1] < num:
            outside.append(row)
    return inside, outside


@pytest.mark.parametrize("el", [1, 2])
def test_k_rows_past_the_end(el):
    limit = _max_desc_ld()
    for ld in (16, 4096, limit // 3 // 16 * 16, limit - 16, limit, limit + 16, 1 << 25, 1 << 26, (1 << 26) + 16, 1 << 27, 1 << 29):
        most = ((1 << 31) - 1) // (ld * el)   # K x ld x el < 2^31
        for K in {1, 2, 15, 16, 63, 64, 100, 127, most} - {0}:
            K = min(K, most, 128 // el)
            if K == 0:
                continue
            assert _read(K, ld, el, masked=ld > limit) == (list(range(K)), []), (K, ld)


def test_longer_rows_need_the_lane_masks():
    # 16 rows of 2^26 bytes: rows 64..79 wrap to rows 0..15
    assert _read(16, 1 << 26, 1, masked=False)[0] == [*range(16), *range(64, 80)]
