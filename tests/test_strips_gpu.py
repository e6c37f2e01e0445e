"""The strip kernels (automata whose edges lead from a state to itself or up to four numbers upward) against the oracle,
at the sizes where they can go wrong: strips of 60 states, workgroups of four strips, blocks of eight frames, back-pointer
windows of 64 states, and every kind of edge they take or leave to the other kernels."""
import numpy as np
import pytest
import torch

from i6_native_ops_amd import cabi
from tests.test_viterbi_gpu import assert_identical, run_cabi_viterbi

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def stage_after_stage():
    cabi.set_overlap(0)
    yield
    cabi.set_overlap(-1)


def automata(rng, sizes, F, kind, permute=False):
    """Left-to-right automata of the given numbers of states.  kind: "chain" loops and steps; "optional" some states can be
    passed over; "ctc" emission on the target state and several edges into the last state; "wide" edges of up to four
    states upward, some of them twice; "far" one edge of five (not for the strips); "mixed" that in the last sequence only;
    "sparse" like wide, but few of those edges, and "passing" like optional, but few such states (2.05 and 2.3 edges per state at
    most, what the full sum leaves to the strips); "own" and "own skip" like chain and passing, but every edge has an emission of
    its own, with "end" an end state that no edge leaves, entered by five edges from up to four states below.  Weights are multiples of 1/2, so ties are common."""
    frm, to, emis, seq, w = [], [], [], [], []
    ends = []
    off = 0
    for b, n in enumerate(sizes):
        state_emis = rng.integers(0, F, size=n)

        def edge(u, v, e):
            frm.append(off + u); to.append(off + v); emis.append(int(e)); seq.append(b)
            w.append(-0.5 * int(rng.integers(0, 4)))

        for u in range(n):
            by_target = kind in ("ctc", "wide")
            steps = [0, 1]
            if kind in ("optional", "ctc") and rng.random() < 0.4:
                steps.append(2)
            if kind == "passing" and rng.random() < 0.2:
                steps.append(2)
            if kind.startswith("own skip") and rng.random() < (0.2 if n > 600 else 0.01):
                steps.append(2)
            if kind == "sparse" and (u % 60 in (1, 56, 57) or u in (235, 236, 239)) and (u // 60) % 2 == 0:
                steps.append(int(rng.choice([1, 3, 4, 2])))
            if kind == "wide":
                steps += [int(x) for x in rng.integers(1, 5, size=rng.integers(0, 2))]
            if (kind == "far" or (kind == "mixed" and b == len(sizes) - 1)) and u == n // 3:
                steps.append(5)
            for k in steps:
                if u + k < n and not (kind.endswith(("ctc", "end")) and u + k == n - 1 and k == 0):
                    edge(u, u + k, rng.integers(0, F) if kind.startswith("own") else state_emis[u + k] if by_target else state_emis[u])
        if kind == "ctc" and n >= 5:
            for u, v in ((n - 2, n - 2), (n - 3, n - 2), (n - 4, n - 2), (n - 2, n - 3)):
                edge(u, n - 1, state_emis[v])
        if kind.endswith("end") and n >= 5:
            for u in (n - 2, n - 3, n - 4, n - 5):
                edge(u, n - 1, rng.integers(0, F))
        ends.append(off + n - 1)
        off += n
    starts = np.concatenate([[0], np.cumsum(sizes)[:-1]])
    edges = np.array([frm, to, emis, seq], dtype=np.int32)
    start_end = np.array([starts, ends], dtype=np.int32)
    if permute:
        # ids that do not follow the automaton, each sequence within its own range
        new = np.concatenate([s + rng.permutation(n) for s, n in zip(starts, sizes)]).astype(np.int32)
        edges[:2] = new[edges[:2]]
        start_end = new[start_end].astype(np.int32)
    order = rng.permutation(edges.shape[1])
    return edges[:, order].copy(), np.array(w, dtype=np.float32)[order].copy(), start_end, off


CASES = [
    # sizes, frames, lengths, classes, kind
    ([56, 57, 59, 60, 61, 63, 64, 65], 96, [96, 95, 91, 90, 89, 88, 81, 65], 40, "chain"),       # around one strip
    ([116, 117, 119, 120, 121, 125], 200, [200, 199, 193, 192, 191, 126], 23, "optional"),
    ([232, 236, 237, 240, 241, 245], 400, [400, 399, 393, 385, 384, 243], 97, "chain"),          # around one workgroup
    ([480, 476, 481, 477], 700, [700, 697, 480, 699], 300, "optional"),                          # two of them; just enough frames
    ([1, 2, 3, 4, 5, 8], 24, [24, 1, 7, 8, 9, 17], 5, "chain"),                                  # the smallest
    ([6, 61, 125, 242, 300], 330, [330, 200, 329, 328, 327], 60, "ctc"),                         # strips with edges of any kind
    ([70, 130, 250, 64], 180, [180, 179, 177, 64], 31, "wide"),
    ([70, 130, 250, 64], 280, [280, 279, 277, 64], 31, "far"),                                   # the other kernels
    ([70, 130, 250, 64], 280, [280, 279, 277, 64], 31, "mixed"),                                 # for the whole batch
    ([300, 200, 100], 150, [150, 100, 99], 50, "chain"),                                         # the end is out of reach for two of them
    ([1900, 1100], 2304, [2301, 1100], 700, "optional"),                                         # many workgroups, several passes of the gather
]


@pytest.mark.parametrize("permute", [False, True], ids=["in_order", "permuted"])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_best_path(oracle, case, permute):
    sizes, T, lens, F, kind = CASES[case]
    rng = np.random.default_rng(100 + case)
    edges, weights, start_end, n = automata(rng, sizes, F, kind, permute)
    am = -0.25 * rng.integers(0, 12, size=(T, len(sizes), F)).astype(np.float32)      # multiples of 1/4: ties
    seq_lens = np.array(lens, dtype=np.int32)
    args = (am, edges, weights, start_end, seq_lens, n)
    align, scores, _ = run_cabi_viterbi(*args)
    assert_identical((align, scores), oracle.viterbi_oracle(*args))


OWN = ["own", "own skip", "own end", "own skip end"]


@pytest.mark.parametrize("kind", OWN)
@pytest.mark.parametrize("sizes,T", [([61, 125, 180, 301, 59], 420), ([60, 121, 241, 5], 256), ([900, 640, 1201], 1300)])
def test_best_path_with_a_score_per_edge(oracle, kind, sizes, T):
    """No state has one score: a score per class of edge in the strips' table, two or three classes; with and without an end state whose edges are
    left out of its strip; one strip and many, short sequences and chunks."""
    rng = np.random.default_rng(len(kind) + T)
    edges, weights, start_end, n = automata(rng, sizes, 300, kind, permute=T == 420)
    lens = np.array([T - k for k in (0, 7, 2, 5, 4)[:len(sizes)]], dtype=np.int32)
    for am in (rng.normal(size=(T, len(sizes), 300)).astype(np.float32), -0.25 * rng.integers(0, 12, size=(T, len(sizes), 300)).astype(np.float32)):
        args = (am, edges, weights, start_end, lens, n)
        want = oracle.viterbi_oracle(*args)
        assert_identical(run_cabi_viterbi(*args)[:2], want)
    assert np.isfinite(want[1]).all()
    if max(sizes) > 240:        # (a wait between workgroups that runs out, which only the strips have: they were there)
        cabi.set_spin_limit(1)
        try:
            assert run_cabi_viterbi(*args, check=False)[2] == -15
        finally:
            cabi.set_spin_limit(0)


# sequences, frames, states from .. to, kind: what follows the paths is a matter of these (best_path_walk)
WALKS = [
    (100, 300, 60, 160, "chain"),           # one workgroup a sequence
    (64, 512, 66, 70, "own end"),           # the same, in pieces, with bytes
    (60, 449, 40, 80, "ctc"),               # with an end state looked up apart
    (2, 500, 10, 30, "ctc"),
    (3, 130, 125, 200, "optional"),         # few frames of many states: chunks in the search's kernel
    (100, 520, 60, 120, "optional"),        # a kernel of their own
    (60, 450, 100, 200, "ctc"),
    (60, 450, 100, 200, "own skip end"),
    (60, 600, 290, 300, "chain"),
]


@pytest.mark.parametrize("case", range(len(WALKS)))
def test_best_path_whoever_follows_it(oracle, case):
    B, T, lo, hi, kind = WALKS[case]
    rng = np.random.default_rng(600 + case)
    edges, weights, start_end, n = automata(rng, rng.integers(lo, hi + 1, size=B).tolist(), 50, kind)
    lens = rng.integers(max(hi, T // 2), T + 1, size=B).astype(np.int32) if hi < T // 2 else rng.integers(T - 9, T + 1, size=B).astype(np.int32)
    for am in (rng.normal(size=(T, B, 50)).astype(np.float32), -0.25 * rng.integers(0, 12, size=(T, B, 50)).astype(np.float32)):
        args = (am, edges, weights, start_end, lens, n)
        assert_identical(run_cabi_viterbi(*args)[:2], oracle.viterbi_oracle(*args))
    if lo > 240:        # a wait between workgroups that runs out: no path and no score (and the strips were there)
        cabi.set_spin_limit(1)
        try:
            align, scores, code = run_cabi_viterbi(*args, check=False)
        finally:
            cabi.set_spin_limit(0)
        assert code == -15 and np.isnan(scores).all() and not align.any()


def test_best_path_over_many_chunks(oracle):
    """Where the paths lead over a chunk of 64 frames is written by one workgroup and read by another, in the same kernel and, for most numbers of states,
    from cache lines that several have written: other scores in the same workspace, again and again."""
    rng = np.random.default_rng(41)
    sizes = [30, 70, 100, 130, 175, 250, 330, 10]
    edges, weights, start_end, n = automata(rng, sizes, 50, "optional")
    for rep in range(6):
        am = rng.normal(size=(1500, len(sizes), 50)).astype(np.float32)
        args = (am, edges, weights, start_end, rng.integers(1300, 1501, size=len(sizes)).astype(np.int32), n)
        assert_identical(run_cabi_viterbi(*args)[:2], oracle.viterbi_oracle(*args))


def test_best_path_beyond_the_rows_of_the_full_sum(oracle):
    """131100 frames of 4090 states: more than 2 GiB of the rows that only the full sum stores, so no reason to leave the strips out.  (That they
    are there is seen from a wait that runs out: the search that would take their place has none.)"""
    rng = np.random.default_rng(42)
    edges, weights, start_end, n = automata(rng, [4090], 8, "chain")
    am = rng.normal(size=(131100, 1, 8)).astype(np.float32)
    args = (am, edges, weights, start_end, np.array([131093], dtype=np.int32), n)
    assert_identical(run_cabi_viterbi(*args)[:2], oracle.viterbi_oracle(*args))
    cabi.set_spin_limit(1)
    try:
        _, scores, code = run_cabi_viterbi(*args, check=False)
    finally:
        cabi.set_spin_limit(0)
    assert code == -15 and np.isnan(scores[0])


@pytest.mark.parametrize("B", [1, 8])
@pytest.mark.parametrize("n_frames", [9, 16, 23, 50, 64, 127, 200, 249, 256])
def test_best_path_of_short_ctc_automata(oracle, n_frames, B):
    """Few frames of few states: one workgroup follows the path as a whole (chunks where there are more), from an end state whose edges are looked up apart from the others': last frames
    everywhere in a block, short sequences behind long ones, repeated labels at the end, scores with and without ties."""
    from i6_native_ops_amd.fsa import ctc_fsa
    rng = np.random.default_rng(10 * n_frames + B)
    F = 29
    for rep in range(4):
        # (one sequence: another residue on every turn; eight of them: all residues at once)
        lens = np.array([max(1, n_frames - (b + 2 * rep) % 8) if b < 6 or rep % 2 else n_frames // 4 + b // 2 for b in range(B)], dtype=np.int32)
        n_labels = np.array([rng.integers(1, max(2, n // 2)) for n in lens], dtype=np.int32)
        targets = rng.integers(1, F, size=(B, int(n_labels.max()))).astype(np.int32)
        for b in range(0, B, 3):
            if n_labels[b] > 1:
                targets[b, n_labels[b] - 2] = targets[b, n_labels[b] - 1]
        am = rng.normal(size=(n_frames, B, F)).astype(np.float32)
        if rep >= 2:
            am = np.round(2 * am) / 4
        n, edges, weights, start_end = (x.cpu().numpy() if torch.is_tensor(x) else x for x in
                                        ctc_fsa(torch.from_numpy(targets).cuda(), torch.from_numpy(n_labels).cuda()))
        there = edges[3] >= 0
        got = run_cabi_viterbi(am, edges, weights, start_end, lens, int(n))
        assert_identical(got[:2], oracle.viterbi_oracle(am, edges[:, there].copy(), weights[there].copy(), start_end, lens, int(n)))


@pytest.mark.parametrize("n_frames", [257, 320, 321, 385])
def test_best_path_of_ctc_automata_that_end_with_a_chunk(oracle, n_frames):
    """Chunks of 64 frames: sequences that end with one, with the first frame of the next, and all around that."""
    from i6_native_ops_amd.fsa import ctc_fsa
    rng = np.random.default_rng(n_frames)
    F = 29
    lens = np.array([max(1, n_frames - d) for d in (0, 1, 2, 7, 8, 63, 64, 65, 66, 128, 129, 250)], dtype=np.int32)
    n_labels = np.array([rng.integers(1, max(2, n // 2)) for n in lens], dtype=np.int32)
    targets = rng.integers(1, F, size=(lens.size, int(n_labels.max()))).astype(np.int32)
    n, edges, weights, start_end = (x.cpu().numpy() if torch.is_tensor(x) else x for x in
                                    ctc_fsa(torch.from_numpy(targets).cuda(), torch.from_numpy(n_labels).cuda()))
    there = edges[3] >= 0
    for rep in range(2):
        am = rng.normal(size=(n_frames, lens.size, F)).astype(np.float32)
        if rep == 1:
            am = np.round(2 * am) / 4
        got = run_cabi_viterbi(am, edges, weights, start_end, lens, int(n))
        assert_identical(got[:2], oracle.viterbi_oracle(am, edges[:, there].copy(), weights[there].copy(), start_end, lens, int(n)))


def test_scores_that_are_not_numbers():
    """A NaN never wins, -inf closes an edge, a class of +inf takes everything: as in the other kernels (the reference's
    compare-and-swap does something else with a NaN)."""
    rng = np.random.default_rng(7)
    edges, weights, start_end, n = automata(rng, [90, 61, 130], 20, "optional")
    am = rng.normal(size=(150, 3, 20)).astype(np.float32)
    am[rng.random(am.shape) < 0.05] = np.nan
    am[rng.random(am.shape) < 0.05] = -np.inf
    am[40, 1, 3] = np.inf
    args = (am, edges, weights, start_end, np.array([150, 149, 141], dtype=np.int32), n)
    got = run_cabi_viterbi(*args)
    cabi.set_overlap(1)
    want = run_cabi_viterbi(*args)
    assert_identical(got[:2], want[:2])
    assert np.isfinite(got[1][0]) and np.isposinf(got[1][1]) and np.isneginf(got[1][2])


def test_replayed_graph(oracle):
    """Counters and tables start afresh on every replay of a captured call."""
    rng = np.random.default_rng(11)
    edges, weights, start_end, n = automata(rng, [300, 250], 40, "optional")
    am = rng.normal(size=(420, 2, 40)).astype(np.float32)
    seq_lens = np.array([420, 400], dtype=np.int32)
    dev = torch.device("cuda:0")
    d = [torch.from_numpy(np.ascontiguousarray(x)).to(dev) for x in (am, edges, weights, start_end, seq_lens)]
    T, B, F = am.shape
    E = edges.shape[1]
    align = torch.empty((T, B), dtype=torch.int32, device=dev)
    scores = torch.empty((B,), dtype=torch.float32, device=dev)
    ws = torch.empty(cabi.workspace_size(T, B, F, E, n), dtype=torch.uint8, device=dev)

    def call():
        cabi.viterbi(d[0].data_ptr(), d[0].stride(0), d[0].stride(1), d[1].data_ptr(), d[1].stride(0), d[2].data_ptr(), d[3].data_ptr(),
                     d[3].stride(0), d[4].data_ptr(), T, B, F, E, n, align.data_ptr(), align.stride(0), align.stride(1), scores.data_ptr(),
                     ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream)

    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for i in range(4):
        am = rng.normal(size=am.shape).astype(np.float32)
        d[0].copy_(torch.from_numpy(am))
        align.fill_(-1)
        graph.replay()
        torch.cuda.synchronize()
        assert_identical((align.cpu().numpy(), scores.cpu().numpy()), oracle.viterbi_oracle(am, edges, weights, start_end, seq_lens, n))


FULL_SUM = [
    ([119, 120, 121, 176, 180, 181], 264, [264, 263, 257, 256, 199, 264], 40, "chain"),      # borders of strips, of blocks, of the last block
    ([236, 240, 244, 480], 600, [600, 599, 593, 592], 97, "chain"),                          # borders of workgroups
    ([300, 290, 20], 304, [301, 290, 5], 50, "chain"),                                       # just enough frames; an end out of reach
    ([700, 650, 1200], 1288, [1288, 1281, 1250], 300, "passing"),                            # large, three sources per state
    ([180, 247, 300, 121], 304, [304, 303, 301, 297], 50, "sparse"),                         # strips with edges of any kind
    ([700, 650, 1200], 808, [808, 801, 790], 300, "passing"),                                # the same, fewer frames than states
]


def run_without_strips(am, edges, weights, start_end, seq_lens, n_states, out_mode):
    """The same call in a workspace that ends before the strips' tables."""
    from tests.gpu_util import DeviceProblem
    P = DeviceProblem(am, edges, weights, start_end, seq_lens, n_states)
    P.ws_bytes -= 256
    out, loss = P.run(out_mode)
    return out.cpu().numpy(), loss.cpu().numpy()


def check_full_sum(oracle, args, strips=True):
    """Both output modes; losses to 1e-5 and posteriors to 1e-4 of the oracle's, the bars of the other full-sum tests.  Other bits
    than without strips show that the strips were there."""
    from tests.gpu_util import run_cabi
    from tests.helpers import posterior
    want_out, want_loss = oracle.fbw_oracle(*args, threads=4)
    out, loss = run_cabi(*args)
    np.testing.assert_allclose(loss, want_loss, rtol=1e-5, atol=1e-6)
    np.testing.assert_allclose(posterior(out), posterior(want_out), rtol=0, atol=1e-4)
    assert (np.isposinf(out) == np.isposinf(want_out)).all()
    prob, loss = run_cabi(*args, out_mode=cabi.OUT_PROB)
    np.testing.assert_allclose(loss, want_loss, rtol=1e-5, atol=1e-6)
    np.testing.assert_allclose(prob, posterior(want_out), rtol=0, atol=1e-4)
    other, _ = run_without_strips(*args, cabi.OUT_PROB)
    assert strips != np.array_equal(prob, other)


@pytest.mark.parametrize("permute", [False, True], ids=["in_order", "permuted"])
@pytest.mark.parametrize("case", range(len(FULL_SUM)))
def test_full_sum(oracle, case, permute):
    sizes, T, lens, F, kind = FULL_SUM[case]
    rng = np.random.default_rng(300 + case)
    edges, weights, start_end, n = automata(rng, sizes, F, kind, permute)
    am = rng.uniform(0.1, 9.0, size=(T, len(sizes), F)).astype(np.float32)
    args = (am, edges, -weights, start_end, np.array(lens, dtype=np.int32), n)
    # (ids that do not follow a small automaton are only renumbered where it is tightly aligned, and its batch goes elsewhere then)
    check_full_sum(oracle, args, strips=not (permute and case in (0, 1, 4)))


@pytest.mark.parametrize("kind", OWN)
@pytest.mark.parametrize("sizes,T", [([177, 180, 240, 296], 312), ([700, 650, 1201], 1288)])
def test_full_sum_with_a_score_per_edge(oracle, kind, sizes, T):
    rng = np.random.default_rng(len(kind) + T)
    edges, weights, start_end, n = automata(rng, sizes, 300, kind)
    am = rng.uniform(0.1, 9.0, size=(T, len(sizes), 300)).astype(np.float32)
    check_full_sum(oracle, (am, edges, -weights, start_end, np.array([T - k for k in (0, 7, 2, 5)[:len(sizes)]], dtype=np.int32), n))


@pytest.mark.parametrize("n_frames", [257, 258, 263, 264])
def test_full_sum_last_state_alone_in_a_strip(oracle, n_frames):
    """Backward strips hold the states from 60 j - 4 on: with 57 states more than a multiple of 60 the end state has the last one to
    itself, and a value in a single row."""
    rng = np.random.default_rng(500 + n_frames)
    edges, weights, start_end, n = automata(rng, [117, 177, 237], 40, "chain")
    am = rng.uniform(0.1, 9.0, size=(264, 3, 40)).astype(np.float32)
    check_full_sum(oracle, (am, edges, -weights, start_end, np.array([n_frames, 264, n_frames], dtype=np.int32), n))


@pytest.mark.parametrize("labels", [(27, 30, 28, 29), (57, 58, 87, 60), (119, 147, 118, 120), (260, 300, 297, 290)])
def test_full_sum_ctc(oracle, labels):
    """CTC automata as ctc_fsa leaves them (arrays at their capacity): an end state with five entering edges, alone in a strip or beside others; a
    repeated label at the end."""
    from i6_native_ops_amd.fsa import ctc_fsa
    from tests.gpu_util import DeviceProblem
    from tests.helpers import posterior
    rng = np.random.default_rng(sum(labels))
    F, T = 23, max(272, 5 * max(labels) // 2)
    lens = np.array([T, T - 3, T - 8, T - 9], dtype=np.int32)
    targets = rng.integers(1, F, size=(4, max(labels))).astype(np.int32)
    targets[2, labels[2] - 2] = targets[2, labels[2] - 1]
    am = rng.uniform(0.1, 9.0, size=(T, 4, F)).astype(np.float32)
    n, edges, weights, start_end = (x.cpu().numpy() if torch.is_tensor(x) else x for x in
                                    ctc_fsa(torch.from_numpy(targets).cuda(), torch.from_numpy(np.array(labels, dtype=np.int32)).cuda()))
    there = edges[3] >= 0
    want_out, want_loss = oracle.fbw_oracle(am, edges[:, there].copy(), weights[there].copy(), start_end, lens, int(n), threads=4)
    P = DeviceProblem(am, edges, weights, start_end, lens, n)
    strips = P.run(cabi.OUT_PROB)[0].cpu().numpy()
    np.testing.assert_allclose(P.loss.cpu().numpy(), want_loss, rtol=1e-5, atol=1e-6)
    np.testing.assert_allclose(strips, posterior(want_out), rtol=0, atol=1e-4)
    P.ws_bytes -= 256       # without the strips' tables: other bits show that they were there
    assert not np.array_equal(strips, P.run(cabi.OUT_PROB)[0].cpu().numpy())


@pytest.mark.parametrize("label", [28, 59, 147])
def test_full_sum_ctc_last_frames(oracle, label):
    """Last frames everywhere in a block: beta leaves the end state there, in the first block of its walk or into the next one."""
    from i6_native_ops_amd.fsa import ctc_fsa
    from tests.gpu_util import DeviceProblem
    from tests.helpers import posterior
    rng = np.random.default_rng(label)
    B, F, T = 9, 23, max(272, 5 * label // 2)
    lens = np.array([T - b for b in range(B)], dtype=np.int32)
    targets = rng.integers(1, F, size=(B, label + 1)).astype(np.int32)
    targets[1::3, label - 1] = targets[1::3, label - 2]
    n_labels = np.array([label + (b % 2) for b in range(B)], dtype=np.int32)
    am = rng.uniform(0.1, 9.0, size=(T, B, F)).astype(np.float32)
    n, edges, weights, start_end = (x.cpu().numpy() if torch.is_tensor(x) else x for x in ctc_fsa(torch.from_numpy(targets).cuda(), torch.from_numpy(n_labels).cuda()))
    there = edges[3] >= 0
    want_out, want_loss = oracle.fbw_oracle(am, edges[:, there].copy(), weights[there].copy(), start_end, lens, int(n), threads=4)
    P = DeviceProblem(am, edges, weights, start_end, lens, n)
    strips = P.run(cabi.OUT_PROB)[0].cpu().numpy()
    np.testing.assert_allclose(P.loss.cpu().numpy(), want_loss, rtol=1e-5, atol=1e-6)
    np.testing.assert_allclose(strips, posterior(want_out), rtol=0, atol=1e-4)
    P.ws_bytes -= 256       # without the strips' tables: other bits show that they were there
    assert not np.array_equal(strips, P.run(cabi.OUT_PROB)[0].cpu().numpy())


def test_full_sum_over_impossible_scores(oracle):
    """Scores of +inf (probability 0): scattered ones, a class that is never possible, a frame that lets nothing pass."""
    rng = np.random.default_rng(31)
    for kind, sizes, T in (("chain", [200, 130, 190], 424), ("passing", [700, 610, 660], 960)):
        edges, weights, start_end, n = automata(rng, sizes, 60, kind)
        am = rng.uniform(0.1, 9.0, size=(T, 3, 60)).astype(np.float32)
        am[rng.random(am.shape) < 0.005] = np.inf      # (a chain over 60 classes finds no way through 0.02)
        am[:, 1, 7] = np.inf
        am[T // 2, 2, :] = np.inf
        check_full_sum(oracle, (am, edges, -weights, start_end, np.array([T, T - 5, T - 9], dtype=np.int32), n))


def test_full_sum_scores_that_are_not_numbers_stay_in_their_sequence(oracle):
    """(What they make of their own sequence is not pinned: the reference skips some and loses the sequence over others.)"""
    from tests.gpu_util import run_cabi
    rng = np.random.default_rng(32)
    for bad in (np.nan, -np.inf):
        for kind, sizes, T in (("chain", [200, 130, 190], 424), ("passing", [700, 610, 660], 960)):
            edges, weights, start_end, n = automata(rng, sizes, 60, kind)
            am = rng.uniform(0.1, 9.0, size=(T, 3, 60)).astype(np.float32)
            args = [am, edges, -weights, start_end, np.array([T, T - 5, T - 9], dtype=np.int32), n]
            want, want_loss = run_cabi(*args, out_mode=cabi.OUT_PROB)
            args[0] = am.copy()
            args[0][:, 1][rng.random((T, 60)) < 0.01] = bad
            out, loss = run_cabi(*args, out_mode=cabi.OUT_PROB)
            for b in (0, 2):
                np.testing.assert_array_equal(out[:, b], want[:, b])
                np.testing.assert_array_equal(loss[:, b], want_loss[:, b])


@pytest.mark.parametrize("n_edges", [4095, 4096, 4097, 4607, 4608, 4609])
def test_row_writer_staging_area(oracle, n_edges):
    """One automaton on both sides of what the row writer keeps in registers (4096 edges) and of what it stages at once (4608),
    behind the strips and behind the other recursion; a small one beside it."""
    from tests.helpers import posterior
    rng = np.random.default_rng(n_edges)
    S, T = 2040, 2304
    edges, weights, start_end, n = automata(rng, [S, 30], 700, "optional")
    frm, to, emis, seq = edges
    spare = np.flatnonzero((seq == 0) & (to - frm == 2))            # states that can be passed over: as many as it takes
    drop = int((seq == 0).sum()) - n_edges
    assert 0 <= drop <= spare.size
    keep = np.ones(edges.shape[1], dtype=bool)
    keep[spare[:drop]] = False
    keep[(seq == 1) & (to - frm == 2)] = False          # (the small one a chain: more than 2.3 edges per state would keep the strips out)
    edges, weights = edges[:, keep].copy(), weights[keep].copy()
    assert (edges[3] == 0).sum() == n_edges
    am = rng.uniform(0.1, 9.0, size=(T, 2, 700)).astype(np.float32)
    args = (am, edges, -weights, start_end, np.array([2301, 300], dtype=np.int32), n)
    check_full_sum(oracle, args, strips=n_edges <= 23 * S // 10)
    other, loss = run_without_strips(*args, cabi.OUT_PROB)
    want_out, want_loss = oracle.fbw_oracle(*args, threads=4)
    np.testing.assert_allclose(loss, want_loss, rtol=1e-5, atol=1e-6)
    np.testing.assert_allclose(other, posterior(want_out), rtol=0, atol=1e-4)


@pytest.mark.parametrize("B", [16, 160])
def test_batches_with_more_strips_than_compute_units(oracle, B):
    """The full sum leaves them to the other recursion, which needs no second round of workgroups (same bits as without strips)."""
    rng = np.random.default_rng(B)
    edges, weights, start_end, n = automata(rng, rng.integers(120, 200, size=B).tolist(), 20, "chain")
    am = rng.uniform(0.1, 9.0, size=(256, B, 20)).astype(np.float32)
    check_full_sum(oracle, (am, edges, -weights, start_end, rng.integers(210, 257, size=B).astype(np.int32), n), strips=B == 16)


def test_replayed_graph_of_the_full_sum(oracle):
    """Progress counters, marks and offsets start afresh on every replay of a captured call."""
    from tests.gpu_util import DeviceProblem
    from tests.helpers import posterior
    rng = np.random.default_rng(12)
    edges, weights, start_end, n = automata(rng, [300, 250], 40, "chain")
    seq_lens = np.array([420, 400], dtype=np.int32)
    am = rng.uniform(0.1, 9.0, size=(420, 2, 40)).astype(np.float32)
    P = DeviceProblem(am, edges, -weights, start_end, seq_lens, n)
    P.run(cabi.OUT_PROB)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        P.run(cabi.OUT_PROB, check=False)
    for i in range(4):
        am = rng.uniform(0.1, 9.0, size=am.shape).astype(np.float32)
        P.am.copy_(torch.from_numpy(am))
        P.out.fill_(-1)
        graph.replay()
        torch.cuda.synchronize()
        out, loss = P.out.cpu().numpy().copy(), P.loss.cpu().numpy().copy()
        want_out, want_loss = oracle.fbw_oracle(am, edges, -weights, start_end, seq_lens, n, threads=4)
        np.testing.assert_allclose(loss, want_loss, rtol=1e-5, atol=1e-6)
        np.testing.assert_allclose(out, posterior(want_out), rtol=0, atol=1e-4)
        eager, _ = P.run(cabi.OUT_PROB)
        np.testing.assert_array_equal(out, eager.cpu().numpy())


def test_last_block_of_a_tight_sequence(oracle):
    """The last strip holds nothing but the end state, which no row of the last block needs; the frames of that block behind
    the sequence's end are in nobody's score table (more than 1024 classes: four frames a pass), so they hold what
    the workspace held.  Neither may show in the results."""
    from tests.gpu_util import DeviceProblem
    from tests.helpers import posterior
    sizes, T, F = [1141, 701], 1140, 12000
    rng = np.random.default_rng(12)
    edges, weights, start_end, n = automata(rng, sizes, F, "chain")
    am = rng.uniform(0.1, 9.0, size=(T, 2, F)).astype(np.float32)
    args = (am, edges, -weights, start_end, np.array([1140, 700], dtype=np.int32), n)
    want_out, want_loss = oracle.fbw_oracle(*args, threads=4)
    P = DeviceProblem(*args)
    for fill in (-1e30, 1e30):
        P.ws.view(torch.float32).fill_(fill)
        out, loss = P.run(cabi.OUT_PROB)
        np.testing.assert_allclose(loss.cpu().numpy(), want_loss, rtol=1e-5, atol=1e-6)
        np.testing.assert_allclose(out.cpu().numpy(), posterior(want_out), rtol=0, atol=1e-4)


@pytest.mark.parametrize("writer", [0, 1], ids=["rows", "flat"])
def test_waits_that_run_out_leave_nan_and_a_status(writer):
    """Strips that give up waiting for the strip in front of them (a poll limit of one from the host; every wave still walks to its
    end): the call reports it, rows hold NaN or what they should, and the next call is as ever."""
    from tests.gpu_util import DeviceProblem
    rng = np.random.default_rng(5)
    sizes, T, F = [500, 130, 30], 560, 2500
    edges, weights, start_end, n = automata(rng, sizes, F, "chain")
    am = rng.uniform(0.1, 9.0, size=(T, 3, F)).astype(np.float32)
    P = DeviceProblem(am, edges, -weights, start_end, np.array([560, 551, 540], dtype=np.int32), n)
    good_out, good_loss = [x.cpu().numpy().copy() for x in P.run(cabi.OUT_PROB)]
    stream = torch.cuda.current_stream().cuda_stream
    cabi.set_dense_writer(writer)
    cabi.set_spin_limit(1)
    try:
        P.out.fill_(-7.0)
        P.loss.fill_(-7.0)
        P.run(cabi.OUT_PROB, check=False)
        code, _ = cabi.read_status(P.ws.data_ptr(), P.B, stream)
    finally:
        cabi.set_spin_limit(0)
        cabi.set_dense_writer(-1)
    out, loss = P.out.cpu().numpy(), P.loss.cpu().numpy()
    assert code == -15
    assert np.isnan(out[:, 0]).all() and np.isnan(loss[:, 0]).all()
    for got, good in ((out, good_out), (loss, good_loss)):
        np.testing.assert_allclose(got[~np.isnan(got)], good[~np.isnan(got)], rtol=1e-6, atol=1e-6)
    out, loss = P.run(cabi.OUT_PROB)
    np.testing.assert_array_equal(out.cpu().numpy(), good_out)
    np.testing.assert_array_equal(loss.cpu().numpy(), good_loss)


def test_best_path_waits_that_run_out(oracle):
    rng = np.random.default_rng(6)
    edges, weights, start_end, n = automata(rng, [500, 130, 30], 40, "optional")
    am = rng.normal(size=(560, 3, 40)).astype(np.float32)
    args = (am, edges, weights, start_end, np.array([560, 551, 540], dtype=np.int32), n)
    want = oracle.viterbi_oracle(*args)
    cabi.set_spin_limit(1)
    try:
        align, scores, code = run_cabi_viterbi(*args, check=False)
    finally:
        cabi.set_spin_limit(0)
    assert code == -15 and np.isnan(scores[0])
    for b in range(3):
        if np.isnan(scores[b]):
            assert (align[:, b] == 0).all()
        else:
            assert_identical((align[:, b], scores[b:b + 1]), (want[0][:, b], want[1][b:b + 1]))
    assert_identical(run_cabi_viterbi(*args)[:2], want)


@pytest.mark.parametrize("kind", ["chain", "mixed"])
def test_a_batch_goes_through_the_strips_as_a_whole(oracle, kind):
    """One sequence that they cannot take, and the others go with it: the two recursions one behind the other would take as
    long as both.  (Seen by the bits, which are those of a call without strips then.)"""
    from tests.gpu_util import run_cabi
    from tests.helpers import posterior
    rng = np.random.default_rng(21)
    edges, weights, start_end, n = automata(rng, [200, 250, 190], 40, kind)
    am = rng.uniform(0.1, 9.0, size=(420, 3, 40)).astype(np.float32)
    args = (am, edges, -weights, start_end, np.array([420, 411, 300], dtype=np.int32), n)
    out, loss = run_cabi(*args, out_mode=cabi.OUT_PROB)
    want_out, want_loss = oracle.fbw_oracle(*args, threads=4)
    np.testing.assert_allclose(loss, want_loss, rtol=1e-5, atol=1e-6)
    np.testing.assert_allclose(out, posterior(want_out), rtol=0, atol=1e-4)
    other, _ = run_without_strips(*args, cabi.OUT_PROB)
    assert np.array_equal(out, other) == (kind == "mixed")


@pytest.mark.parametrize("writer", [0, 1], ids=["rows", "flat"])
@pytest.mark.parametrize("kind", ["passing", "mixed"])
def test_large_automata_overlapped_or_in_strips(oracle, kind, writer):
    """Calls whose sizes ask for the overlapped schedule: enqueued both ways, the preparation decides."""
    from tests.gpu_util import run_cabi
    from tests.helpers import posterior
    rng = np.random.default_rng(22)
    T, B, F = 1025, 5, 13100
    assert T * B * F >= 1 << 26
    edges, weights, start_end, n = automata(rng, rng.integers(590, 650, size=B).tolist(), F, kind)
    am = rng.uniform(0.1, 9.0, size=(T, B, F)).astype(np.float32)
    lens = rng.integers(660, T + 1, size=B).astype(np.int32)
    lens[1] = T
    args = (am, edges, -weights, start_end, lens, n)
    want_out, want_loss = oracle.fbw_oracle(*args, threads=8)
    cabi.set_dense_writer(writer)
    try:
        cabi.set_overlap(-1)
        out, loss = run_cabi(*args, out_mode=cabi.OUT_PROB)
        cabi.set_overlap(1)         # (leaves the strips out)
        overlapped, _ = run_cabi(*args, out_mode=cabi.OUT_PROB)
    finally:
        cabi.set_dense_writer(-1)
    np.testing.assert_allclose(loss, want_loss, rtol=1e-5, atol=1e-6)
    np.testing.assert_allclose(out, posterior(want_out), rtol=0, atol=1e-4)
    assert np.array_equal(out, overlapped) == (kind == "mixed")


@pytest.mark.parametrize("kind", ["optional", "mixed", "far"])
def test_best_path_overlapped_or_in_strips(oracle, kind):
    rng = np.random.default_rng(23)
    T, B, F = 800, 13, 6500
    assert T * B * F >= 1 << 26
    cabi.set_overlap(-1)
    edges, weights, start_end, n = automata(rng, rng.integers(60, 200, size=B).tolist(), F, kind, permute=True)
    am = -0.25 * rng.integers(0, 12, size=(T, B, F)).astype(np.float32)
    args = (am, edges, weights, start_end, rng.integers(300, T + 1, size=B).astype(np.int32), n)
    for rep in range(2):
        assert_identical(run_cabi_viterbi(*args)[:2], oracle.viterbi_oracle(*args))
