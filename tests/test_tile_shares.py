"""How a decode launch deals its tiles out to workgroups (tiles_of_workgroup in csrc/ntc_decode_kernel.h, on the host)."""
import ctypes as C
import os

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.parametrize("by_die", [0, 1])
@pytest.mark.parametrize("workgroups", [1, 7, 8, 9, 255, 256, 257, 304, 512])
@pytest.mark.parametrize("total", ["none over", 1, 7, 8, 9, "half over", "one short", 1 << 30])
def test_shares_cover_the_list_and_differ_by_one_tile(by_die, workgroups, total):
    path = os.path.join(HERE, "libexact_decode.so")
    if not os.path.exists(path):
        pytest.skip("run __graft_entry__.build() (make -C tests)")
    lib = C.CDLL(path)
    tiles = {"none over": 3 * workgroups, "half over": 21 * workgroups + workgroups // 2, "one short": 6 * workgroups - 1}.get(total)
    tiles = workgroups + total if tiles is None else tiles
    ranges, out = [], (C.c_int * 2)()
    for w in range(workgroups):
        lib.tiles_of_workgroup(by_die, tiles, workgroups, w, out)
        ranges.append((out[0], out[1]))
    sizes = [b - a for a, b in ranges]
    assert sorted(set(sizes)) in ([tiles // workgroups], [tiles // workgroups, tiles // workgroups + 1])
    assert sizes == sorted(sizes, reverse=True)              # the longer ones first
    ordered = sorted(ranges)
    assert ordered[0][0] == 0 and ordered[-1][1] == tiles and all(x[1] == y[0] for x, y in zip(ordered, ordered[1:]))
    if by_die and workgroups % 8 == 0:                       # a die's workgroups hold neighbouring shares, in order
        for die in range(8):
            mine = ranges[die::8]
            assert all(x[1] == y[0] for x, y in zip(mine, mine[1:]))
