"""Rows over several workgroups (longer than one workgroup's registers): no
top-k and every kind of top-k, ragged and padded lengths, both element types,
penalties, masks, greedy and invalid rows, ties past the ranked capacity,
top-p off and near zero, infinities and NaN; bit-exact against the oracle.  On the CPU every
workgroup of the launch runs at once (the exchange) or one after another
(every poll runs out: the fallbacks)."""
import os
import shutil
import sys

import numpy as np
import pytest

import gpu_harness as H

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpu_sim"))


def _rows(oracle, V, seed, bf16=False, mask=False, hist=64):
    """One row of each kind the kernel tells apart."""
    from tinygpt_amd import workloads as W

    g = np.random.default_rng(seed)
    kinds = ["plain", "flat", "greedy", "special", "coarse", "inf", "none", "invalid"]
    B = len(kinds)
    x = (g.standard_normal((B, V)) * 3.0).astype(np.float32)
    p = oracle.make_params(B, temperature=0.8, top_k=0, top_p=0.9, repetition=1.1, presence=0.2, frequency=0.1)
    p["temperature"][3], p["temperature"][4] = 1.0, 0.5
    p["top_p"][[3, 4]] = [1.0, 1e-9]
    p["top_k"][[0, 3]] = [-1, V + 3]
    x[1] = 0.75  # every id in one bucket, more than the lists and the ranking hold
    x[1, ::3] = 0.7
    p["temperature"][2] = 0.0
    x[3, g.choice(V, V // 20, replace=False)] = np.nan
    x[3, g.choice(V, V // 20, replace=False)] = -np.inf
    x[4] = np.round(x[4])
    x[5, [5, V - 1]] = np.inf
    x[6] = -np.inf
    p["temperature"][7] = np.nan
    table = None
    if mask:
        words = (V + 31) // 32
        table = g.integers(0, 1 << 32, (3, words), dtype=np.uint64).astype(np.uint32)
        table[1] = 0
        table[1, [0, words // 2, words - 1]] = 1
        table[:, -1] &= np.uint32((1 << (V - 32 * (words - 1))) - 1) if V % 32 else np.uint32(0xFFFFFFFF)
        p["mask_state"] = [0, 1, 2, -1, 0, 1, 2, 0]
    h = g.integers(-2, V + 2, (B, hist)).astype(np.int32) if hist else None
    hl = g.integers(0, hist + 1, B).astype(np.int32) if hist else None
    u = (g.integers(0, 1 << 24, B) / (1 << 24)).astype(np.float32)
    return (W.f32_to_bf16_bits(x) if bf16 else x), p, u, h, hl, table


def _oracle(oracle, x, p, u, h, hl, table):
    return oracle.sample_batch(x, p, u, hist=h, hist_len=hl, mask_table=table, kept_cap=8, want_post=True, nthreads=8)


def _topk_rows(oracle, V, seed, bf16=False, mask=False, hist=64):
    """_rows with a top-k on every sampling row (but the invalid one), and
    more of them: small and large k, k past the allowed ids of a sparse mask,
    k that ends in ties, in the mass-0 bucket, above 1024."""
    x, p, u, h, hl, table = _rows(oracle, V, seed, bf16, mask, hist)
    p["top_k"] = [50, 1000, 0, 700, 64, 3, 5, 9]
    g = np.random.default_rng(seed + 1)
    n = 6
    rows = [0, 4, 0, 0, 1, 0]
    x2, p2 = x[rows].copy(), p[rows].copy()
    p2["top_k"] = [1, 513, 2000, 1024, 7, 512]
    p2["temperature"] = [1.0, 0.7, 1.3, 0.01, 1.0, 0.6]
    p2["top_p"] = [0.5, 1.0, 0.8, 1.0, 0.9, 0.999]
    cat = np.concatenate
    u2 = (g.integers(0, 1 << 24, n) / (1 << 24)).astype(np.float32)
    return (cat([x, x2]), cat([p, p2]), cat([u, u2]), None if h is None else cat([h, h[rows]]),
            None if hl is None else cat([hl, hl[rows]]), table)


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
@pytest.mark.parametrize("rows,V,bf16,mask,concurrent", [
    ([0, 1], 32769, False, False, True), ([3, 4], 33001, True, True, True), ([9, 12], 36864, True, False, True),
    ([8, 10], 32800, False, True, True), ([11, 13], 33000, True, False, True), ([0, 1, 9, 10], 33003, True, False, False),
    ([4, 11], 33002, False, True, False)])
def test_topk_rows_in_the_simulation(oracle, rows, V, bf16, mask, concurrent):
    import sim as S

    S.build()
    x, p, u, h, hl, table = _topk_rows(oracle, V, 9 + V, bf16, mask)
    x, p, u, h, hl = x[rows], p[rows], u[rows], h[rows], hl[rows]
    r = S.run_sample(x, p, u, h, hl, mask_table=table, kept_cap=1025, concurrent=concurrent,
                     env_extra={"TGS_KEY_SPINS": "100000"} if concurrent else None)
    assert [blk for _, blk in r["launches"]] == [512]  # one launch for every kind of row
    o = oracle.sample_batch(x, p, u, hist=h, hist_len=hl, mask_table=table, kept_cap=1025, want_post=True, nthreads=8)
    H.compare(r, o, p, V, what="split top-k")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
@pytest.mark.parametrize("rows,V,bf16,mask,concurrent", [
    ([0, 1], 32769, False, False, True), ([2, 3], 33001, True, True, True), ([4, 5], 36864, False, True, True),
    ([6, 7], 32800, True, False, True), ([6, 5], 32800, True, False, False),
    ([0, 1, 2, 4], 33003, True, False, False), ([3, 5], 33002, False, True, False)])
def test_split_rows_in_the_simulation(oracle, rows, V, bf16, mask, concurrent):
    import sim as S

    import tinygpt_amd as tg

    S.build()
    x, p, u, h, hl, table = _rows(oracle, V, 7 + V, bf16, mask)
    x, p, u, h, hl = x[rows], p[rows], u[rows], h[rows], hl[rows]
    hint = tg.batch_hint(p, V)
    r = S.run_sample(x, p, u, h, hl, mask_table=table, kept_cap=8, hint=hint, concurrent=concurrent,
                     repeat=2 if concurrent else 1, env_extra={"TGS_KEY_SPINS": "100000"} if concurrent else None)
    assert all(blk == 512 and grid > len(rows) for grid, blk in r["launches"])
    H.compare(r, _oracle(oracle, x, p, u, h, hl, table), p, V, what="split top-p")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_slabs_of_the_static_workspace(oracle):
    """A batch of 276 chunks takes one launch on the allocation-free entry
    point's workspace too (all but one of its rows greedy)."""
    import sim as S

    import tinygpt_amd as tg

    S.build()
    B, V = 92, 32769
    g = np.random.default_rng(92)
    x = np.tile((g.standard_normal((1, V)) * 3.0).astype(np.float32), (B, 1))
    x[np.arange(B), g.integers(0, V, B)] = 20.0
    p = oracle.make_params(B, temperature=0.0, top_p=0.9)
    p["temperature"][50] = 0.8
    u = np.full(B, 0.75, np.float32)
    r = S.run_sample(x, p, u, hint=tg.batch_hint(p, V), post=False, kept_cap=8, noalloc=True)
    assert [n for n in r["launches"] if n[1] == 512] == [(3 * B, 512)]
    np.testing.assert_array_equal(r["ids"], oracle.sample_batch(x, p, u, nthreads=8)["ids"])


@pytest.mark.gpu
@pytest.mark.parametrize("V,bf16,mask,hist", [
    (32769, False, False, 64), (32776, True, True, 64), (50001, True, False, 0), (65536, False, True, 1000),
    (128256, False, False, 64), (128256, True, True, 0), (151936, True, False, 256), (151935, False, True, 64)])
def test_split_rows(sampler, oracle, V, bf16, mask, hist):
    x, p, u, h, hl, table = _rows(oracle, V, V, bf16, mask, hist)
    o = _oracle(oracle, x, p, u, h, hl, table)
    for hint in ("auto", None):  # top-p rows and greedy rows alone, and every kind of row
        H.log(f"case split top-p V={V} bf16={bf16} mask={mask} hint={hint}")
        r = H.run_gpu(sampler, x, p, u, h, hl, mask_table=table, kept_cap=8, hint=hint)
        H.compare(r, o, p, V, what="split top-p")


@pytest.mark.gpu
@pytest.mark.parametrize("B", [1, 3, 33, 200])
def test_split_batches(sampler, oracle, B):
    """Chunk counts from the most to the fewest, and a batch over several
    launches (its slabs outnumber the workspace's)."""
    V = 128256
    g = np.random.default_rng(B)
    x = (g.standard_normal((B, V)) * 3.0).astype(np.float32)
    p = oracle.make_params(B, temperature=g.choice([0.7, 1.0, 1.3], B), top_k=0, top_p=g.choice([0.3, 0.9, 1.0], B))
    u = (g.integers(0, 1 << 24, B) / (1 << 24)).astype(np.float32)
    o = _oracle(oracle, x, p, u, None, None, None)
    for _ in range(2):
        H.log(f"case split top-p batch B={B}")
        r = H.run_gpu(sampler, x, p, u, kept_cap=8, hint="auto")
        H.compare(r, o, p, V, what="split top-p")


@pytest.mark.gpu
@pytest.mark.parametrize("V,bf16,mask,hist", [
    (32769, False, False, 64), (32776, True, True, 64), (50001, True, False, 0), (65536, False, True, 1000),
    (128256, False, False, 64), (128256, True, True, 0), (151935, True, False, 256)])
def test_topk_rows(sampler, oracle, V, bf16, mask, hist):
    """Without a hint, with the kept lists and without them (their rows take
    other lists)."""
    x, p, u, h, hl, table = _topk_rows(oracle, V, V + 3, bf16, mask, hist)
    o = oracle.sample_batch(x, p, u, hist=h, hist_len=hl, mask_table=table, kept_cap=1025, want_post=True, nthreads=8)
    H.log(f"case split top-k V={V} bf16={bf16} mask={mask}")
    H.compare(H.run_gpu(sampler, x, p, u, h, hl, mask_table=table, kept_cap=1025), o, p, V, what="split top-k")
    import torch

    import tinygpt_amd as tg

    got = {k: torch.zeros(s, dtype=t, device="cuda:0") for k, s, t in
           (("counts", (len(p), 2), torch.int32), ("mass", (len(p), 2), torch.int64), ("cut_ids", (len(p),), torch.int32))}
    ids = sampler.sample(H.to_dev(x), tg.params_to_device(p, "cuda:0"), H.to_dev(u), hist=H.to_dev(h),
                         hist_len=H.to_dev(hl), vocab=V, debug=got)
    np.testing.assert_array_equal(ids.cpu().numpy(), o["ids"])
    ok = o["ids"] != -2
    np.testing.assert_array_equal(got["counts"].cpu().numpy()[ok], np.stack([o["res"]["n_topk"], o["res"]["n_topp"]], 1)[ok])
    np.testing.assert_array_equal(got["mass"].cpu().numpy().view(np.uint64)[ok],
                                  np.stack([o["res"]["mass_k"], o["res"]["mass_p"]], 1)[ok])
    np.testing.assert_array_equal(got["cut_ids"].cpu().numpy()[ok], o["res"]["cut_id"][ok])


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
@pytest.mark.parametrize("rows,V,bf16,mask,chunks", [
    ([0, 1, 2, 3, 4, 5, 6, 7], 4097, False, False, 1), ([0, 8, 9, 10, 11, 12, 13], 4099, True, True, 1),
    ([1, 9, 11, 13], 8192, True, False, 2), ([0, 3, 10], 16383, False, False, 3), ([2, 4, 8, 12], 12289, True, True, 3),
    ([0, 1, 2, 3, 4, 5, 6, 8, 9], 8200, False, False, 2)])
def test_short_rows_in_the_simulation(oracle, rows, V, bf16, mask, chunks):
    """Rows that one workgroup's registers could hold, batches of every kind:
    one chunk or a few."""
    import sim as S

    S.build()
    x, p, u, h, hl, table = _topk_rows(oracle, V, 9 + V, bf16, mask)
    x, p, u, h, hl = x[rows], p[rows], u[rows], h[rows], hl[rows]
    o = oracle.sample_batch(x, p, u, hist=h, hist_len=hl, mask_table=table, kept_cap=1025, want_post=True, nthreads=8)
    for kept_cap in (1025, 0):  # with the kept lists and without them
        r = S.run_sample(x, p, u, h, hl, mask_table=table, kept_cap=kept_cap, concurrent=True, repeat=2,
                         env_extra={"TGS_KEY_SPINS": "100000"})
        assert r["launches"] == [(len(rows) * chunks, 512)] * 2
        if kept_cap:
            H.compare(r, o, p, V, what="short rows")
        else:
            np.testing.assert_array_equal(r["ids"], o["ids"])


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
@pytest.mark.parametrize("top_k", [0, 2000])
def test_rows_that_lds_does_not_hold(oracle, top_k):
    """A device whose LDS holds the top-p kernel's tail but not the split
    kernel's: rows beyond one workgroup's registers are refused before
    anything is launched, shorter ones go to the kernels that fit."""
    import sim as S

    import tinygpt_amd as tg

    S.build()
    g = np.random.default_rng(44)
    for V in (33000, 8000):
        x = (g.standard_normal((1, V)) * 3.0).astype(np.float32)
        p = oracle.make_params(1, temperature=0.8, top_k=top_k, top_p=0.9)
        u = np.full(1, 0.5, np.float32)
        run = lambda hint: S.run_sample(x, p, u, post=False, kept_cap=8, hint=hint, env_extra={"TGS_SIM_LDS": "44000"})  # noqa: E731
        for hint in (tg.batch_hint(p, V), None):
            if V == 33000:
                with pytest.raises(RuntimeError, match=r"sample -5 .*\(top-p rows\)"):
                    run(hint)
            else:
                np.testing.assert_array_equal(run(hint)["ids"], oracle.sample_batch(x, p, u)["ids"])


def _floor_rows(oracle, V, seed, bf16):
    """Rows that leave a floor below too many of a chunk's ids: in order, all
    equal, all but one equal, of a few values around 0 of both signs, infinite
    at more ids than k, and allowed in one stretch or at few ids only; and one
    whose largest ids lie two to a thread of the first chunk, so that its k-th
    is hardly above the floor."""
    from tinygpt_amd import workloads as W

    g = np.random.default_rng(seed)
    n = np.sort(g.standard_normal(V) * 3.0)
    x = np.stack([n, n[::-1], np.full(V, 0.75), np.full(V, -1e4), g.choice([-1e-40, -0.0, 0.0, 1e-40], V),
                  g.standard_normal(V), g.standard_normal(V), g.standard_normal(V),
                  g.uniform(-6.0, -5.0, V)]).astype(np.float32)
    x[3, V // 3] = 5.0
    first = np.arange(min(512, V // 16)) * (8 if bf16 else 4)
    x[8, first], x[8, first + 1] = g.uniform(10.0, 11.0, len(first)), g.uniform(5.0, 6.0, len(first))
    x[5, g.choice(V, V // 2, replace=False)] = np.inf
    B, words = len(x), (V + 31) // 32
    bits = np.zeros((2, words * 32), bool)
    bits[0, V // 8:V // 3] = True
    bits[1, g.choice(V, 600, replace=False)] = True
    p = oracle.make_params(B, temperature=0.8, top_p=[0.9, 1.0, 0.5, 0.99, 0.9, 0.7, 0.95, 0.9, 1.0],
                           mask_state=[-1, -1, -1, -1, -1, -1, 0, 1, -1])
    p["top_k"] = [1000, 1024, 513, 700, 900, 600, 1023, 1000, 1000]
    u = (g.integers(0, 1 << 24, B) / (1 << 24)).astype(np.float32)
    return (W.f32_to_bf16_bits(x) if bf16 else x), p, u, np.packbits(bits, axis=1, bitorder="little").view(np.uint32)


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
@pytest.mark.parametrize("rows,V,bf16,split,concurrent", [
    ([0, 1, 2, 3, 4, 5, 6, 7], 4609, False, None, True), ([0, 2, 8], 12289, True, None, True),
    ([1, 3, 8], 12289, False, None, True), ([4, 5], 8200, True, None, True), ([6, 7], 16384, False, 5, True), ([0, 4, 6], 8200, False, None, False)])
def test_floors_in_the_simulation(oracle, rows, V, bf16, split, concurrent):
    import sim as S

    S.build()
    x, p, u, table = _floor_rows(oracle, V, V, bf16)
    x, p, u = x[rows], p[rows], u[rows]
    r = S.run_sample(x, p, u, mask_table=table, kept_cap=1025, split=split, concurrent=concurrent,
                     env_extra={"TGS_KEY_SPINS": "100000"} if concurrent else None)
    assert [blk for _, blk in r["launches"]] == [512]
    o = oracle.sample_batch(x, p, u, mask_table=table, kept_cap=1025, want_post=True, nthreads=8)
    H.compare(r, o, p, V, what="floors")


@pytest.mark.gpu
@pytest.mark.parametrize("V,bf16", [(4609, True), (12289, False), (32000, True), (128256, False), (151935, True)])
@pytest.mark.parametrize("copies", [1, 33])
def test_floors(sampler, oracle, V, bf16, copies):
    x, p, u, table = _floor_rows(oracle, V, V + 1, bf16)
    o = oracle.sample_batch(x, p, u, mask_table=table, kept_cap=1025, want_post=False, nthreads=8)
    rep = lambda t: np.concatenate([t] * copies)  # noqa: E731
    H.log(f"case floors V={V} bf16={bf16} B={copies * len(p)}")
    r = H.run_gpu(sampler, rep(x), rep(p), rep(u), mask_table=table, kept_cap=1025, post=False)
    for i in range(copies):
        part = {k: (None if v is None else v[i * len(p):(i + 1) * len(p)]) for k, v in r.items()}
        H.compare(part, o, p, V, what="floors", check_post=False)


def _large_k_rows(oracle, V, seed):
    """Rows with 1024 < top_k < V whose sets end inside buckets of a few, of
    many and of nearly all ids; top-p on, off and near zero."""
    g = np.random.default_rng(seed)
    x = np.concatenate([np.round(g.standard_normal((3, V)) * 2.0), np.full((2, V), 0.75), g.standard_normal((4, V)) * 3.0])
    x[4, ::3] = 0.74
    B = len(x)
    p = oracle.make_params(B, temperature=0.8, top_p=[0.9, 1.0, 0.5, 0.6, 1.0, 0.99, 1.0, 1e-9, 0.9])
    p["top_k"] = [V // 2, 1100, V - 1, 3000, V // 2, V // 2, 3000, V // 3, 1025]
    return x.astype(np.float32), p, (g.integers(0, 1 << 24, B) / (1 << 24)).astype(np.float32)


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
@pytest.mark.parametrize("rows,V,concurrent", [([0, 3, 5], 12289, True), ([1, 4, 6], 8200, True),
                                               ([2, 7, 8], 8200, True), ([0, 1, 2, 3, 4, 5, 6, 7, 8], 4100, True),
                                               ([0, 4, 6], 8200, False)])
def test_large_k_in_the_simulation(oracle, rows, V, concurrent):
    import sim as S

    S.build()
    x, p, u = (t[rows] for t in _large_k_rows(oracle, V, V))
    r = S.run_sample(x, p, u, kept_cap=8, concurrent=concurrent,
                     env_extra={"TGS_KEY_SPINS": "100000"} if concurrent else None)
    assert [blk for _, blk in r["launches"]] == [512]
    H.compare(r, oracle.sample_batch(x, p, u, kept_cap=8, want_post=True, nthreads=8), p, V, what="large k")


@pytest.mark.gpu
@pytest.mark.parametrize("V", [4100, 12289, 50001, 128256])
@pytest.mark.parametrize("copies", [1, 29])
def test_large_k(sampler, oracle, V, copies):
    x, p, u = (np.concatenate([t] * copies) for t in _large_k_rows(oracle, V, V))
    o = oracle.sample_batch(x, p, u, kept_cap=8, want_post=False, nthreads=8)
    H.log(f"case large k V={V} B={len(p)}")
    H.compare(H.run_gpu(sampler, x, p, u, kept_cap=8, post=False), o, p, V, what="large k", check_post=False)


@pytest.mark.gpu
@pytest.mark.parametrize("V,bf16,mask,hist", [
    (4097, False, False, 64), (4104, True, True, 0), (7325, True, False, 64), (11008, False, True, 1000),
    (16384, False, False, 64), (16385, True, True, 64), (32768, True, False, 0)])
@pytest.mark.parametrize("copies", [1, 30])
def test_short_rows(sampler, oracle, V, bf16, mask, hist, copies):
    """Few rows over several chunks each, and more rows than CUs (one chunk up
    to 16,384 ids)."""
    x, p, u, h, hl, table = _topk_rows(oracle, V, V + 5, bf16, mask, hist)
    rep = lambda t: None if t is None else np.concatenate([t] * copies)  # noqa: E731
    x, p, u, h, hl = (rep(t) for t in (x, p, u, h, hl))
    o = oracle.sample_batch(x, p, u, hist=h, hist_len=hl, mask_table=table, kept_cap=1025, want_post=True, nthreads=8)
    H.log(f"case short rows V={V} bf16={bf16} mask={mask} B={len(p)}")
    H.compare(H.run_gpu(sampler, x, p, u, h, hl, mask_table=table, kept_cap=1025), o, p, V, what="short rows")
    import torch

    import tinygpt_amd as tg

    got = {"counts": torch.zeros(len(p), 2, dtype=torch.int32, device="cuda:0"),
           "mass": torch.zeros(len(p), 2, dtype=torch.int64, device="cuda:0"),
           "cut_ids": torch.zeros(len(p), dtype=torch.int32, device="cuda:0")}
    ids = sampler.sample(H.to_dev(x), tg.params_to_device(p, "cuda:0"), H.to_dev(u), hist=H.to_dev(h),
                         hist_len=H.to_dev(hl), vocab=V, debug=got)
    np.testing.assert_array_equal(ids.cpu().numpy(), o["ids"])
    ok = o["ids"] != -2
    res = o["res"]
    np.testing.assert_array_equal(got["counts"].cpu().numpy()[ok], np.stack([res["n_topk"], res["n_topp"]], 1)[ok])
    np.testing.assert_array_equal(got["mass"].cpu().numpy().view(np.uint64)[ok],
                                  np.stack([res["mass_k"], res["mass_p"]], 1)[ok])
    np.testing.assert_array_equal(got["cut_ids"].cpu().numpy()[ok], res["cut_id"][ok])
