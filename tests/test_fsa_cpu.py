"""What the CTC builder reads and counts of a row of labels, on the host: elements from target_lens[b] on need not exist
(rows of different lengths packed one behind the other), so the last label here is the last word before a page that
cannot be read."""
import os
import subprocess

import numpy as np
import pytest

from i6_native_ops_amd.fbw.workloads import _ctc

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "i6_native_ops_amd", "csrc")
PROGRAM = r"""
#include "fsa_counts.h"
#include <cstdio>
#include <cstdlib>
#include <sys/mman.h>
int main(int argc, char** argv) {
    const int L = argc - 2, Lmax = atoi(argv[1]);
    char* page = (char*)mmap(nullptr, 1 << 17, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
    if (page == MAP_FAILED || mprotect(page + (1 << 16), 1 << 16, PROT_NONE) != 0) return 2;
    int32_t* lab = (int32_t*)(page + (1 << 16)) - L;
    int repeats = 0, sum = L ? 0 : CTC_EMPTY_EDGES;
    for (int i = 0; i < L; i++) { lab[i] = atoi(argv[2 + i]); repeats += i > 0 && lab[i] == lab[i - 1]; }
    for (int i = 0; i < Lmax; i++) sum += ctc_label_edges(lab, i, L);
    printf("%d %d\n", sum, ctc_edges(L, repeats, L > 1 && lab[L - 1] == lab[L - 2]));
    return 0;
}
"""


@pytest.fixture(scope="module")
def counter(tmp_path_factory):
    where = tmp_path_factory.mktemp("fsa")
    (where / "count.cpp").write_text(PROGRAM)
    subprocess.check_call(["g++", "-O0", "-std=c++17", "-I", CSRC, str(where / "count.cpp"), "-o", str(where / "count")])
    return str(where / "count")


@pytest.mark.parametrize("L", [0, 1, 2, 3, 17])
def test_counts_and_reads_stay_within_the_row(counter, L):
    rng = np.random.default_rng(L)
    for rep in range(8):
        labels = rng.integers(1, 3, size=L).tolist()
        run = subprocess.run([counter, str(L + 9)] + [str(x) for x in labels], capture_output=True, text=True)
        assert run.returncode == 0, f"read behind the {L} labels of the row"
        want = len(_ctc(labels).frm)
        assert [int(x) for x in run.stdout.split()] == [want, want]
