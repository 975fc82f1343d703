"""What the split kernel's exchange lines keep from call to call on one
handle: calls of every kind of row and several lengths (chunk counts) after
one another, across the points where an epoch's shortened tags come round
again.  Every call's ids equal the oracle's on its own inputs."""
import os
import shutil
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpu_sim"))

V3 = 12289  # three chunks of one row


def _call(oracle, kind, V=V3, B=1, seed=0, epoch=None):
    """One call's inputs.  The distributions differ from call to call, so
    that buckets and lists left by one are wrong for the next."""
    g = np.random.default_rng(seed)
    x = (g.standard_normal((B, V)) * g.choice([0.3, 3.0, 6.0], (B, 1))).astype(np.float32)
    p = oracle.make_params(B, temperature=0.8, top_k=0, top_p=0.9, mask_state=-1)
    if kind == "list":
        p["top_k"] = 40
    elif kind == "wide":
        p["top_k"] = 2000
    elif kind == "greedy":
        p["temperature"] = 0.0
    elif kind == "masked":
        p["mask_state"] = 0
    elif kind == "invalid":
        p["temperature"] = np.nan
    u = (g.integers(0, 1 << 24, B) / (1 << 24)).astype(np.float32)
    return dict(x=x, p=p, u=u, epoch=epoch)


def _table(V):
    return np.zeros((1, (V + 31) // 32), np.uint32)  # one state, nothing allowed


def _ids(oracle, c):
    V = c["x"].shape[1]
    return oracle.sample_batch(c["x"], c["p"], c["u"], mask_table=_table(V), nthreads=8)["ids"]


def _run(oracle, calls):
    import sim as S

    S.build()
    got = S.run_sequence(calls, mask_table=_table(max(c["x"].shape[1] for c in calls)))
    for i, (ids, c) in enumerate(zip(got, calls)):
        np.testing.assert_array_equal(ids, _ids(oracle, c), err_msg=f"call {i}")


sim = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")


@sim
@pytest.mark.parametrize("before", ["list", "greedy", "masked"])
def test_decision_tag_comes_round_unwritten(oracle, before):
    """A row's first histogram call is its 2^24-th call: no call before it had
    a decision to publish."""
    _run(oracle, [_call(oracle, before, seed=1, epoch=(1 << 24) - 2), _call(oracle, "topp", seed=2)])


@sim
@pytest.mark.parametrize("between", ["list", "greedy", "masked"])
def test_decision_tag_comes_round(oracle, between):
    """2^24 calls after a published decision, all but the last without one."""
    _run(oracle, [_call(oracle, "topp", seed=3), _call(oracle, between, seed=4, epoch=(1 << 24) - 1),
                  _call(oracle, "topp", seed=5), _call(oracle, "wide", seed=6)])


@sim
@pytest.mark.parametrize("word", [None, (1 << 14) - 4, (1 << 24) - 4, (1 << 32) - 5])
def test_kinds_and_lengths_alternate(oracle, word):
    """Rows of every kind and one to four chunks in turn on the same lines,
    also across the wraps of the maxima's, the decision's and the epoch's own
    tags."""
    kinds = ["topp", "list", "topp", "masked", "wide", "greedy", "topp", "invalid", "topp"]
    lengths = [V3, 16384, 8200, V3, 16384, 4200, V3, V3, 16384]
    calls = [_call(oracle, k, V, seed=20 + i) for i, (k, V) in enumerate(zip(kinds, lengths))]
    calls[0]["epoch"] = word
    _run(oracle, calls)


@sim
def test_done_words_come_round(oracle):
    """Lists published 2^32 - 1 calls ago, all between without any: they are
    not taken for the current call's."""
    _run(oracle, [_call(oracle, "topp", seed=40), _call(oracle, "greedy", seed=41, epoch=(1 << 32) - 2),
                  _call(oracle, "topp", seed=42)])


@pytest.mark.gpu
@pytest.mark.parametrize("B", [1, 9])
def test_kinds_and_lengths_alternate_on_the_gpu(oracle, B):
    """The same on the device, with up to 16 chunks per row."""
    import gpu_harness as H
    import tinygpt_amd as tg

    s = tg.Sampler(device=0, max_batch=B, max_vocab=151936, max_hist=1)
    kinds = ["topp", "list", "topp", "masked", "wide", "greedy", "topp", "invalid", "topp", "list", "masked", "topp"]
    lengths = [128256, 50001, 8200, 128256, 151936, 4200, 33000, 128256, 50001, 16384, 151936, 128256]
    for i, (kind, V) in enumerate(zip(kinds, lengths)):
        c = _call(oracle, kind, V, B=B, seed=60 + i)
        H.log(f"case split state call {i} {kind} V={V} B={B}")
        r = H.run_gpu(s, c["x"], c["p"], c["u"], mask_table=_table(V), kept_cap=8, post=False)
        np.testing.assert_array_equal(r["ids"], _ids(oracle, c), err_msg=f"call {i}")
    s.close()
