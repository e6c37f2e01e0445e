"""The calls whose speed this repository looks after.

Three operations, through the package's public functions only: a training step with the full-sum loss
(``fbw_loss`` and its backward), the same sum in the form the reference's extension module returns it
(``fbw.core.fbw``, -log posteriors over (T, B, F)), and forced alignment (``align_viterbi``).
The automata are the ones such programs have: HMM chains with three states per label, with or without optional
silence, handed over as finished tuples (built by a data loader on the host), or chains and CTC
topologies built on the GPU from the labels of the batch in every step (``hmm_fsa``, ``ctc_fsa``).
"""
import math

import numpy as np
import torch

from i6_native_ops_amd import fbw
from i6_native_ops_amd.fast_viterbi import align_viterbi
from i6_native_ops_amd.fbw.workloads import make_workload
from i6_native_ops_amd.fsa import ctc_fsa, hmm_fsa

STATES = 3                      # HMM states per label
HALF = math.log(0.5)            # log transition probability of the chains built from labels

# T frames, B sequences (the longest has T frames, the shortest at least shortest * T), F emission classes,
# between lo and hi labels per sequence.
#   topology "chain":   HMM chain built with hmm_fsa in the pass
#            "tied":    HMM chain over tied states with a weight for every transition, handed over
#            "silence": HMM chain with optional silence between the labels, handed over
#            "ctc":     built with ctc_fsa in the pass


def listed():
    return [
        # the smallest training step: two short utterances, a handful of classes; launches and host work
        dict(name="tiny", op="loss", topology="chain", T=50, B=2, F=10, lo=5, hi=5, shortest=0.8),
        # one utterance aligned on its own, as an interactive tool does
        dict(name="align_utterance", op="align", topology="chain", T=713, B=1, F=129, lo=40, hi=60, shortest=1.0),
        # hybrid HMM with monophone states
        dict(name="monophone", op="loss", topology="silence", T=500, B=32, F=264, lo=40, hi=60, shortest=0.8),
        # forced alignment of a batch with the same model
        dict(name="align_monophone", op="align", topology="silence", T=500, B=32, F=264, lo=40, hi=60, shortest=0.8),
        # CTC over characters: short rows, long label sequences, ragged lengths
        dict(name="ctc_chars", op="loss", topology="ctc", T=1203, B=64, F=61, lo=100, hi=300, shortest=0.5),
        # CTC over subword units: large batch after subsampling
        dict(name="ctc_units", op="loss", topology="ctc", T=200, B=256, F=5001, lo=20, hi=60, shortest=0.75),
        # CTC over a large vocabulary
        dict(name="ctc_words", op="loss", topology="ctc", T=300, B=16, F=50000, lo=20, hi=60, shortest=0.6),
        # hybrid HMM with tied triphone states, the headline workload of bench.py
        dict(name="cart", op="loss", topology="tied", T=1000, B=32, F=12001, lo=100, hi=150, shortest=0.8),
        # the same kind of model through the extension module, an odd and ragged batch
        dict(name="cart_neg_log", op="neg_log", topology="tied", T=437, B=19, F=4499, lo=40, hi=70, shortest=0.6),
        # forced alignment with tied triphone states
        dict(name="align_cart", op="align", topology="tied", T=1000, B=32, F=12001, lo=100, hi=150, shortest=0.8),
        # recordings of many minutes
        dict(name="longform", op="loss", topology="silence", T=4000, B=8, F=12001, lo=400, hi=600, shortest=0.5),
        # and their alignment with a small model
        dict(name="align_longform", op="align", topology="silence", T=4000, B=8, F=264, lo=400, hi=600, shortest=0.5),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choices(("loss", "align", "neg_log"), (6, 4, 2))[0]
    topology = rng.choice(("chain", "tied", "silence", "ctc"))
    T = _log_uniform(rng, 50, 4000)
    B = _log_uniform(rng, 1, min(256, 76000 // T))
    F = _log_uniform(rng, 30, 50000) if topology == "ctc" else _log_uniform(rng, 10, 12001)
    F = max(10, min(F, 380_000_000 // (T * B)))
    shortest = round(rng.uniform(0.5, 1.0), 2)
    per_label = 2 if topology == "ctc" else STATES      # frames that a label cannot do without
    hi = max(1, min(600, int(T * shortest * rng.uniform(0.2, 0.75) / per_label)))
    lo = max(1, int(hi * rng.uniform(0.4, 1.0)))
    return dict(op=op, topology=topology, T=T, B=B, F=F, lo=lo, hi=hi, shortest=shortest)


def prepare(case, seed):
    T, B, F = case["T"], case["B"], case["F"]
    dev = torch.device("cuda")
    rng = np.random.default_rng(seed)
    lens = rng.integers(max(1, int(case["shortest"] * T)), T + 1, size=B)
    lens[rng.integers(B)] = T
    state = {"op": case["op"], "topology": case["topology"], "lens": torch.from_numpy(lens.astype(np.int32)).to(dev)}

    # scores of a network that is being trained: log softmax of normal logits
    gen = torch.Generator(device=dev).manual_seed(int(seed))
    batch_first = case["op"] != "neg_log"
    scores = torch.randn((B, T, F) if batch_first else (T, B, F), generator=gen, device=dev)
    scores = torch.log_softmax(scores.mul_(2.0), dim=-1)
    if not batch_first:
        scores = scores.neg_()
    state["scores"] = scores.requires_grad_(case["op"] == "loss")

    if case["topology"] in ("tied", "silence"):
        kind = "cart" if case["topology"] == "tied" else "monophone"
        W = make_workload(kind, seed=int(rng.integers(1 << 31)), T=T, B=B, F=F, with_am=False, n_labels=(case["lo"], case["hi"]))
        # the alignment maximises: log probabilities in place of their negatives
        weights = -W.weights if case["op"] == "align" else W.weights
        state["fsa"] = (W.n_states, torch.from_numpy(W.edges).to(dev), torch.from_numpy(weights).to(dev),
                        torch.from_numpy(W.start_end_states).to(dev))
    else:
        n_labels = rng.integers(case["lo"], case["hi"] + 1, size=B)
        first, last = (1, F) if case["topology"] == "ctc" else (0, max(1, F // STATES))
        labels = rng.integers(first, last, size=(B, int(n_labels.max())))
        state["labels"] = torch.from_numpy(labels.astype(np.int32)).to(dev)
        state["n_labels"] = torch.from_numpy(n_labels.astype(np.int32)).to(dev)
    return state


def run(state):
    op = state["op"]
    if state["topology"] == "ctc":
        fsa = ctc_fsa(state["labels"], state["n_labels"])
    elif state["topology"] == "chain":
        weight = HALF if op == "align" else -HALF
        fsa = hmm_fsa(state["labels"], state["n_labels"], STATES, weight, weight)
    else:
        fsa = state["fsa"]

    if op == "align":
        return align_viterbi(state["scores"], fsa, state["lens"])
    if op == "neg_log":
        num_states, edges, weights, start_end = fsa
        return fbw.core.fbw(state["scores"], edges, weights, start_end, state["lens"], num_states)
    log_probs = state["scores"]
    log_probs.grad = None
    loss = fbw.fbw_loss(log_probs, fsa, state["lens"])
    loss[0].sum().backward()
    return loss, log_probs.grad


def _edges(case):
    """Edges per sequence, on average."""
    labels = (case["lo"] + case["hi"]) / 2
    return {"chain": 2 * STATES, "tied": 2 * STATES, "silence": 2 * STATES + 1.5, "ctc": 5}[case["topology"]] * labels


def work(case):
    """Of the scores, those of the sequence's own emission classes in the frames it has; of the automaton,
    what is handed over: edges of 20 bytes, or labels of 4.  The results are dense."""
    T, B, F = case["T"], case["B"], case["F"]
    frames = B * T * (1 + case["shortest"]) / 2
    labels = (case["lo"] + case["hi"]) / 2
    # distinct classes among the ones drawn for a sequence
    pool = F if case["topology"] in ("ctc", "tied") else max(1, F // STATES)
    drawn = STATES * labels if case["topology"] == "tied" else labels
    classes = pool * (1 - (1 - 1 / pool) ** drawn)
    if case["topology"] in ("chain", "silence"):
        classes *= STATES
    classes += case["topology"] in ("silence", "ctc")
    edges = _edges(case)
    automaton = B * (20 * edges if case["topology"] in ("tied", "silence") else 4 * labels) + 12 * B
    scores = 4 * frames * classes
    if case["op"] == "align":
        # an addition of the weight, one of the score and a comparison for every edge and frame
        return {"bytes": scores + automaton + 4 * T * B + 4 * B, "flops": 3 * frames * edges}
    # the same in both directions with exponentials, and the edge's posterior
    return {"bytes": scores + automaton + 4 * T * B * F + 4 * T * B, "flops": 12 * frames * edges}


def tolerance(case):
    """Four times the distance from the same sums in 64 bits, over the cases above and a dozen drawn ones:
    loss 4e-8, gradient up to 9.4e-6 (2-norm) and 2.1e-4 (single values) where float rows of a thousand and more
    frames are added up; -log posteriors 4.3e-7 and 2.6e-6.  Alignments are the reference's bit for bit."""
    if case["op"] == "align":
        return "exact"
    return {"rel": 3e-5, "max": 8e-4} if case["op"] == "loss" else {"rel": 2e-6, "max": 1e-5}
