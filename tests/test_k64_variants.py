"""The fused top_k <= 64 kernel's instantiations at the sizes where the choice
between them changes: one wave up to two vectors per lane, four waves for more
rows than CUs up to eight vectors per thread, eight waves one or two
workgroups per CU; with history, masks, ragged rows and both element types,
bit-exact against the oracle."""
import os
import shutil
import sys

import numpy as np
import pytest

import gpu_harness as H

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpu_sim"))


def _batch(oracle, B, V, bf16, mask, seed):
    from tinygpt_amd import workloads as W

    g = np.random.default_rng(seed)
    x = (g.standard_normal((B, V)) * 3.0).astype(np.float32)
    x[1::7] = np.round(x[1::7])  # ties
    x[2::7] -= 30.0  # negative rows
    x[3::7, ::3] = -np.inf
    p = oracle.make_params(B, temperature=g.choice([0.7, 1.0, 0.0], B), top_k=g.integers(1, 65, B),
                           top_p=g.choice([0.9, 1.0], B), presence=0.5, frequency=0.3)
    table = None
    if mask:
        words = (V + 31) // 32
        table = np.packbits(g.random((8, words * 32)) < g.choice([0.01, 0.3, 0.9], (8, 1)), axis=1,
                            bitorder="little").view(np.uint32)
        p["mask_state"] = g.integers(-1, 8, B)
    h = g.integers(0, V, (B, 48)).astype(np.int32)
    hl = g.integers(0, 49, B).astype(np.int32)
    u = (g.integers(0, 1 << 24, B) / (1 << 24)).astype(np.float32)
    return (W.f32_to_bf16_bits(x) if bf16 else x), p, u, h, hl, table


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
@pytest.mark.parametrize("B,V,bf16,mask,block", [(3, 512, False, True, 64), (3, 1021, True, True, 64),
                                                 (257, 520, False, True, 256), (257, 1030, True, False, 256)])
def test_small_variants_in_the_simulation(oracle, B, V, bf16, mask, block):
    import sim as S

    import tinygpt_amd as tg

    S.build()
    x, p, u, h, hl, table = _batch(oracle, B, V, bf16, mask, V)
    r = S.run_sample(x, p, u, h, hl, mask_table=table, kept_cap=64, hint=tg.batch_hint(p, V))
    assert r["launches"] == [(B, block)]
    o = oracle.sample_batch(x, p, u, hist=h, hist_len=hl, mask_table=table, kept_cap=64, want_post=True, nthreads=8)
    H.compare(r, o, p, V, what="fused kernel")


@pytest.mark.gpu
@pytest.mark.parametrize("bf16,mask", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("B,V", [(4, 512), (4, 516), (4, 1024), (4, 1032), (260, 513), (260, 1025), (260, 8192),
                                 (260, 8196), (260, 16384), (260, 16392), (24, 151936), (65, 131072), (70, 40000),
                                 (129, 50001)])
def test_variants(sampler, oracle, B, V, bf16, mask):
    x, p, u, h, hl, table = _batch(oracle, B, V, bf16, mask, B + V)
    H.log(f"case fused kernel B={B} V={V} bf16={bf16} mask={mask}")
    post = B * V < 4_000_000
    r = H.run_gpu(sampler, x, p, u, h, hl, mask_table=table, kept_cap=64, hint="auto", post=post)
    o = oracle.sample_batch(x, p, u, hist=h, hist_len=hl, mask_table=table, kept_cap=64, want_post=post, nthreads=8)
    H.compare(r, o, p, V, what="fused kernel", check_post=post)
