"""Offsets of the rows that the full sum over strips stores through a buffer descriptor, on the host: what lanes without a state store has to
fall behind the descriptor's end, whichever row of the last block it is for."""
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "i6_native_ops_amd", "csrc")
PROGRAM = r"""
#include "strip_rows.h"
#include <cstdio>
#include <cstdlib>
// taken in the full sum, in the best path, lowest offset of a lane without a state, highest of one with a state, end of the rows, for L = T
int main(int argc, char** argv) {
    for (int i = 1; i + 1 < argc; i += 2) {
        const int T = atoi(argv[i]), SP = atoi(argv[i + 1]);
        unsigned low = ~0u, high = 0;
        for (long long t = 0; t < (T + 7LL) / 8 * 8; t++) {
            const unsigned none = strip_row_offset(STRIP_NO_COLUMN, (int)t, SP), last = strip_row_offset(4u * (SP - 1), (int)t, SP);
            low = none < low ? none : low;
            if (t < T) high = last > high ? last : high;
        }
        printf("%d %d %u %u %lld\n", (int)strip_rows_taken(false, T, SP), (int)strip_rows_taken(true, T, SP), low, high, 4LL * T * SP);
    }
    return 0;
}
"""


@pytest.fixture(scope="module")
def rows(tmp_path_factory):
    where = tmp_path_factory.mktemp("rows")
    (where / "rows.cpp").write_text(PROGRAM)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-I", CSRC, str(where / "rows.cpp"), "-o", str(where / "rows")])

    def run(sizes):
        out = subprocess.run([str(where / "rows")] + [str(x) for size in sizes for x in size], capture_output=True, text=True, check=True).stdout
        return np.array([line.split() for line in out.splitlines()], dtype=np.int64)
    return run


@pytest.mark.parametrize("SP", [16, 64, 1552, 1760, 4016, 4080, 4096])
def test_rows_at_the_limit(rows, SP):
    limit = 2 ** 29 // SP                       # rows of SP floats in 2 GiB
    sizes = [(T, SP) for T in range(max(1, limit - 17), limit + 10)] + [(8, SP), (1, SP)]
    if SP >= 1552:                              # (every row is walked over)
        sizes += [(345921, 1552), (133681, 4016), (131586, 4080)]
    got = rows(sizes)
    for (T, sp), (fits, path, low, high, end) in zip(sizes, got):
        assert bool(fits) == (4 * -(-T // 8) * 8 * sp < 2 ** 31)
        assert path                             # (stores no such rows)
        if fits:
            assert high == end - 4              # the last state of the last row is the last word
            assert low >= end                   # and a lane without a state is never in front of it
    wrapped = [low < end for (_, _, low, _, end) in got]
    assert SP < 1552 or any(wrapped)            # (there are such sizes)
