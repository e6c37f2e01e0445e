// Edge counts of the CTC automata (fsa_builders.inc); plain C++, so that a host program can check what they read.
#pragma once
#include <cstdint>

#ifdef __HIPCC__
#define I6_COUNT_FN __host__ __device__ __forceinline__
#else
#define I6_COUNT_FN inline
#endif

// Edges of a sequence of L labels, of which `repeats` equal the one before: a loop and an edge from the
// previous state into each of the 2L + 1 states (from the start state into the first), start state -> first label, the
// skips between different labels; and once more those into the last label and the last blank.
constexpr int CTC_EMPTY_EDGES = 4;
I6_COUNT_FN int ctc_edges(const int L, const int repeats, const bool last_repeats) {
    if (L == 0) return CTC_EMPTY_EDGES;
    return 2 * (2 * L + 1) + 1 + (L - 1 - repeats) + 2 + (L == 1 ? 3 : (last_repeats ? 2 : 3));
}
// The share of label i in that number: two states with two edges each and (behind the first label) the skip into it; the
// last label adds the rest.  0 for i >= L, where the row need not have an element: nothing is read there.
I6_COUNT_FN int ctc_label_edges(const int32_t* lab, const int i, const int L) {
    if (i >= L) return 0;
    const bool rep = i > 0 && lab[i] == lab[i - 1];
    int edges = 4 + (i > 0 && !rep ? 1 : 0);
    if (i == L - 1) edges += 2 + 1 + 2 + (L == 1 ? 3 : (rep ? 2 : 3));
    return edges;
}
