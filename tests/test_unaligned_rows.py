"""Rows that start at any element alignment (odd vocabularies) through the
paths that read whole 16-byte vectors there: token log-probabilities and
speculative verification, both element types, lengths around a vector, a
block and a chunk."""
import os
import shutil
import sys

import numpy as np
import pytest

import gpu_harness as H

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpu_sim"))

# log-probability of V ids: fp32 terms of 2^-23 relative exponent error
# (|x - m| log2(e) <= 64 here, so 64 ulp of 1 is 8e-6) and sums of at most V / 256
# terms per thread and 8 + 16 merges, each 6e-8 relative: under 1e-5 in all
ATOL = 2e-5


def _bits(x, bf16):
    from tinygpt_amd import workloads as W

    return W.f32_to_bf16_bits(x) if bf16 else x


def _logprob_case(V, bf16, pad):
    g = np.random.default_rng(V)
    B = 9
    x = g.normal(0.0, 3.0, (B, V + pad)).astype(np.float32)
    x[1, :V] = -np.inf
    x[2, V - 1] = np.nan
    x[3, V // 2] = np.inf
    x[4, :max(V - 1, 1)] = -np.inf
    x[4, V - 1] = 0.5
    x[:, V:] = 1e30  # past the row: never read into the sum
    tok = g.integers(0, V, B).astype(np.int32)
    tok[4], tok[5], tok[6] = V - 1, V, -1
    return _bits(x, bf16), tok


def _close(got, ref):
    nan = np.isnan(ref)
    np.testing.assert_array_equal(np.isnan(got), nan)
    np.testing.assert_array_less(np.abs(got[~nan].astype(np.float64) - ref[~nan]), ATOL)


LP = [(1, 0), (3, 0), (7, 2), (9, 0), (1031, 0), (2049, 6), (4103, 0), (8205, 0), (12293, 4)]


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("V,pad", LP[:7])
def test_logprob_in_the_simulation(oracle, V, pad, bf16):
    import sim as S

    S.build()
    x, tok = _logprob_case(V, bf16, pad)
    lp, lse = S.run_logprob(x, tok, V=V)
    r_lp, r_lse = oracle.token_logprobs(x, tok, V=V)
    _close(lp, r_lp)
    _close(lse, r_lse)


@pytest.mark.gpu
@pytest.mark.parametrize("bf16", [False, True])
def test_logprob_on_the_gpu(sampler, oracle, bf16):
    import torch

    for V, pad in LP:
        H.log(f"case logprob V={V} pad={pad} bf16={bf16}")
        x, tok = _logprob_case(V, bf16, pad)
        xd = (torch.from_numpy(x.view(np.int16)).to("cuda:0").view(torch.bfloat16) if bf16
              else torch.from_numpy(x).to("cuda:0"))[:, :V]
        lse = torch.empty(x.shape[0], dtype=torch.float32, device="cuda:0")
        lp = sampler.token_logprobs(xd, torch.from_numpy(tok).to("cuda:0"), lse=lse)
        torch.cuda.synchronize()
        r_lp, r_lse = oracle.token_logprobs(x, tok, V=V)
        _close(lp.cpu().numpy(), r_lp)
        _close(lse.cpu().numpy(), r_lse)


def _spec_case(V, bf16):
    g = np.random.default_rng(V + 1)
    B, k = 5, 3
    t = g.normal(0.0, 3.0, (B, k + 1, V)).astype(np.float32)
    d = (t[:, :k] + g.normal(0.0, 1.0, (B, k, V))).astype(np.float32)
    if V > 20:
        t[2, :, ::5] = -np.inf
        d[2, 1, 3] = np.nan
        t[1, 1, V - 1] = 14.0
    u = lambda *s: (g.integers(0, 1 << 24, s) / (1 << 24)).astype(np.float32)  # noqa: E731
    tok = g.integers(0, V, (B, k)).astype(np.int32)
    tok[3] = d[3].argmax(-1)
    T = np.array([1.0, 0.7, 1.3, 1.0, 0.0], np.float32)
    return _bits(t, bf16), _bits(d, bf16), tok, T, u(B, k), u(B)


SPEC = [1, 5, 1023, 1025, 2053, 3079]


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("V", SPEC[:5])
def test_spec_in_the_simulation(oracle, V, bf16):
    import sim as S

    S.build()
    c = _spec_case(V, bf16)
    o = oracle.spec_verify_batch(*c, nthreads=4)
    n_acc, out = S.run_spec(*c)
    np.testing.assert_array_equal(n_acc, o["n_acc"])
    np.testing.assert_array_equal(out, o["out"])


@pytest.mark.gpu
@pytest.mark.parametrize("bf16", [False, True])
def test_spec_on_the_gpu(sampler, oracle, bf16):
    import torch

    for V in SPEC:
        H.log(f"case spec V={V} bf16={bf16}")
        c = _spec_case(V, bf16)
        o = oracle.spec_verify_batch(*c, nthreads=4)
        n_acc, out = sampler.spec_verify(*[H.to_dev(x) for x in c])
        torch.cuda.synchronize()
        np.testing.assert_array_equal(n_acc.cpu().numpy(), o["n_acc"])
        np.testing.assert_array_equal(out.cpu().numpy(), o["out"])
