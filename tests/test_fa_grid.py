"""Which sequence a workgroup of the attention kernels serves (fa_grid.h), on the
CPU: the header built as host C++."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "teco-ops_amd", "csrc")
XCDS, SLOTS, ROWS = 8, 32, 64  # 8 XCDs of 4 shader engines


@pytest.fixture(scope="module")
def grid(tmp_path_factory):
    d = tmp_path_factory.mktemp("grid")
    (d / "grid.cpp").write_text("""#include "fa_grid.h"
extern "C" int place(int place, int row, int turn, int batch) {
    return tecoops::fa::turned_place(place, row, turn, batch);
}
extern "C" int turn(int units, int batch) { return tecoops::fa::turn_shift(units, batch); }
extern "C" int turn_of(int units, int batch, int longest, long long rows) {
    return tecoops::fa::turn_shift(units, batch, longest, rows);
}
""")
    subprocess.run(["g++", "-std=c++17", "-fPIC", "-shared", "-I", CSRC, str(d / "grid.cpp"), "-o",
                    str(d / "grid.so")], check=True)
    return ctypes.CDLL(str(d / "grid.so"))


# kv heads times head groups of the calls in use: 1 (one kv head) to 40
@pytest.mark.parametrize("units", [1, 2, 4, 5, 8, 10, 16, 32, 40])
@pytest.mark.parametrize("first", [0, 37])
def test_sequences_go_round(grid, units, first):
    """Every sequence once in every row, and over 64 rows on all slots alike (half
    as often again at most); units that are a multiple of 8 keep each to its XCD."""
    for batch in (1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 12, 16, 20, 24, 31, 48, 96):
        turn = grid.turn(units, batch)
        met = [[0] * SLOTS for _ in range(batch)]
        xcds = [set() for _ in range(batch * units)]
        for row in range(first, first + ROWS):
            served = [grid.place(place, row, turn, batch) for place in range(batch)]
            assert sorted(served) == list(range(batch))
            for place, b in enumerate(served):
                for u in range(units):
                    n = (row * batch + place) * units + u
                    met[b][n % SLOTS] += 1
                    xcds[b * units + u].add(n % XCDS)
        for slots in met:
            mean = ROWS * units / SLOTS
            assert 0.5 * mean <= min(slots) and max(slots) <= 1.5 * mean, (batch, slots)
        if units % XCDS == 0:
            assert all(len(x) == 1 for x in xcds)


@pytest.mark.parametrize("units", [1, 4, 8])
def test_sequences_alike_stay(grid, units):
    for batch in (1, 2, 3, 8, 24):
        assert grid.turn_of(units, batch, 512, ctypes.c_longlong(512 * batch)) == 31
        assert grid.turn_of(units, batch, 512, ctypes.c_longlong(448 * batch)) == 31
        assert grid.turn_of(units, batch, 512, ctypes.c_longlong(447 * batch)) == grid.turn(units, batch)
        assert grid.turn_of(units, batch, 1 << 20, ctypes.c_longlong(1 << 20)) == grid.turn(units, batch)
