"""The sampler's measured workloads: what a decode loop, a scoring job or a
constrained-generation server calls through the public entry points, from one
byte-level row to a thousand rows of a large vocabulary.

Logits follow the benchmark's distributions (N(0, 3^2), eight spikes per row),
histories are Zipf-like token ids, uniforms are multiples of 2^-24, mask rows
have a log-uniform density.  Every state keeps its own sampler handle, as a
serving process keeps one, and the batch hint where the caller computes one.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

import tinygpt_amd as tg
from tinygpt_amd import grammar as G

DEV = "cuda:0"
DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16}
ITEM = {"fp32": 4, "bf16": 2}
MASK_STATES = 64   # mask rows a state keeps (one per live grammar state)
REPORT = 20        # alternatives reported per row when a caller asks for them


# ------------------------------------------------------------------ the cases

def _sample(name, B, V, dtype, policy, hist=0, mask=False, hint=True, report=False):
    return {"name": name, "kind": "sample", "B": B, "V": V, "dtype": dtype, "policy": policy, "hist": hist,
            "mask": mask, "hint": hint, "report": report}


def listed():
    return [
        # one decode step of a byte-level model: the smallest call there is
        _sample("byte_step", 1, 256, "fp32", "topk", hist=64),
        # one chat user, nucleus sampling over a large vocabulary (no top-k)
        _sample("chat_topp", 1, 151936, "bf16", "topp", hist=256),
        # the benchmark's headline batch: penalties, top-k 50, top-p 0.9
        _sample("batch_topk", 64, 128256, "fp32", "topk", hist=512),
        # a batch of nucleus-sampling requests
        _sample("batch_topp", 32, 128256, "fp32", "topp"),
        # grammar-constrained decoding, half of the rows greedy
        _sample("grammar_topp", 128, 32000, "fp32", "grammar", mask=True),
        # a large serving batch with per-request top-k up to 1024
        _sample("large_topk", 1024, 151936, "bf16", "wide", hist=256),
        # requests of every kind in one batch: greedy, small and large top-k, top-p only
        _sample("mixed_requests", 96, 128256, "bf16", "mixed", hist=256),
        # a caller without a hint, odd batch and odd vocabulary (rows not 16-byte aligned)
        _sample("ragged_plain", 17, 50001, "fp32", "topk", hist=100, hint=False),
        # speculative verification of a batch, eight draft tokens each
        {"name": "spec_batch", "kind": "spec", "B": 32, "k": 8, "V": 128256, "dtype": "fp32", "T": 1.0},
        # speculative verification for one user
        {"name": "spec_single", "kind": "spec", "B": 1, "k": 4, "V": 128256, "dtype": "bf16", "T": 0.7},
        # teacher-forced scoring of a 2048-token context
        {"name": "score_context", "kind": "logprob", "B": 2048, "V": 128256, "dtype": "bf16"},
        # 64 new grammar states: their mask rows, then the batch sampled under them
        {"name": "constrained_step", "kind": "constrained", "B": 64, "V": 151936, "dtype": "fp32"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sample", "sample", "sample", "sample", "spec", "logprob", "constrained"])
    dtype = rng.choice(["fp32", "bf16"])
    V = _log_int(rng, 2000, 151936)
    if rng.random() < 0.5:
        V = max(2048, V // 64 * 64)  # padded vocabularies are as common as odd ones
    if kind == "sample":
        policy = rng.choice(["topk", "topk", "topp", "topp", "grammar", "wide", "mixed"])
        most = 96e6 if policy in ("topk", "topp", "grammar") else 48e6
        B = _log_int(rng, 1, max(1, min(1024, int(most / (V * ITEM[dtype])))))
        hist = rng.choice([0, 0, _log_int(rng, 16, 1000)])
        mask = policy == "grammar" or rng.random() < 0.2
        hint = rng.random() < 0.8
        report = policy == "topk" and rng.random() < 0.3
        c = _sample("", B, V, dtype, policy, hist, mask, hint, report)
        del c["name"]
        return c
    if kind == "spec":
        k = rng.randint(1, 8)
        B = _log_int(rng, 1, max(1, min(64, int(200e6 / ((2 * k + 1) * V * ITEM[dtype])))))
        return {"kind": kind, "B": B, "k": k, "V": V, "dtype": dtype, "T": rng.choice([1.0, 0.7, 1.3])}
    if kind == "logprob":
        return {"kind": kind, "B": _log_int(rng, 1, max(1, min(4096, int(400e6 / (V * ITEM[dtype]))))), "V": V,
                "dtype": dtype}
    return {"kind": kind, "B": _log_int(rng, 1, MASK_STATES), "V": V, "dtype": dtype}


# ------------------------------------------------------------------ inputs

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _uniform(g, *shape):
    return torch.randint(0, 1 << 24, shape, generator=g, device=DEV).float() * 2.0**-24


def _logits(g, B, V, dtype, sigma=3.0, spikes=8):
    x = torch.randn(B, V, generator=g, device=DEV) * sigma
    if spikes:
        x.scatter_(1, torch.randint(0, V, (B, spikes), generator=g, device=DEV), 4 * sigma)
    return x.to(DTYPES[dtype])


def _history(g, B, H, V):
    u = torch.rand(B, H, generator=g, device=DEV)
    return (torch.exp(u * math.log(V)) - 1).to(torch.int32).clamp_(0, V - 1)


def _params(policy, B, V, hist, seed, states):
    r = np.random.default_rng(seed)
    p = tg.make_params(B, temperature=0.7, top_k=50, top_p=0.9, mask_state=states)
    if hist:
        p["presence"], p["frequency"] = 0.5, 0.3
    if policy == "topk":
        p["top_k"] = 50 if B == 64 else r.integers(20, 65, B)
    elif policy == "topp":
        p["temperature"], p["top_k"], p["top_p"] = 0.8, 0, r.choice([0.9, 0.95, 1.0], B)
        if hist:
            p["repetition"], p["presence"], p["frequency"] = 1.1, 0.0, 0.0
    elif policy == "grammar":
        p["temperature"], p["top_k"], p["top_p"] = 1.0, 0, 0.95
        p["temperature"][: B // 2] = 0.0
    elif policy == "wide":
        p["temperature"], p["top_k"] = r.uniform(0.3, 1.5, B), r.integers(1, min(1024, V - 1) + 1, B)
        p["top_p"] = r.uniform(0.5, 1.0, B)
        if hist:
            p["repetition"], p["presence"], p["frequency"] = r.uniform(1.05, 1.3, B), 0.0, 0.0
    elif policy == "mixed":
        which = r.random(B)
        p["temperature"] = np.where(which < 0.15, 0.0, r.uniform(0.3, 1.5, B))
        p["top_k"] = np.where(which < 0.55, r.integers(20, 65, B), np.where(which < 0.7, r.integers(65, 1025, B), 0))
        p["top_p"] = r.uniform(0.7, 1.0, B)
    return p


def _mask_table(g, V):
    """MASK_STATES rows of allowed-token bits, density log-uniform in [0.1%, 30%]."""
    words = (V + 31) // 32
    dens = torch.exp(torch.empty(MASK_STATES, 1, device=DEV).uniform_(math.log(1e-3), math.log(0.3), generator=g))
    bits = torch.rand(MASK_STATES, words * 32, generator=g, device=DEV) < dens
    bits[torch.arange(MASK_STATES), torch.randint(0, V, (MASK_STATES,), generator=g, device=DEV).cpu()] = True
    bits[:, V:] = False
    weight = 2 ** torch.arange(32, device=DEV, dtype=torch.int64)
    return (bits.view(MASK_STATES, words, 32) * weight).sum(-1).cpu().numpy().astype(np.uint32)


@functools.lru_cache(maxsize=None)
def _grammar():
    d = G.compile_gbnf(G.PACE_TOOL_TAGS)
    return d, d.byte_classes(), np.nonzero(~d.complete)[0]


@functools.lru_cache(maxsize=4)
def _vocabulary(V):
    """Token bytes as a server holds them: words, tag pieces, some UTF-8."""
    r = np.random.default_rng(31)
    pieces = [b"[", b"]", b"POINT", b":", b"none", b",", b"CLICK", b"TYPE", b"SCROLL", b"up", b"KEY", b"+",
              b"OPEN_APP", b" ", b"_", b"-", b"12", b"9"]
    text = np.frombuffer(b"abcdefghijklmnopqrstuvwxyzABCDEFGHIJ etaoinshr.,", np.uint8)[
        r.integers(0, 48, V + 16)].tobytes()
    kind, length, pick = r.random(V), r.integers(1, 13, V), r.integers(0, len(pieces), (V, 2))
    toks = [b""]
    for v in range(1, V):
        if kind[v] < 0.7:
            toks.append(text[v:v + length[v]])
        elif kind[v] < 0.9:
            toks.append(pieces[pick[v, 0]] + pieces[pick[v, 1]])
        else:
            toks.append("".join(chr(0xC0 + 31 * int(c)) for c in pick[v]).encode())
    return G.token_csr(toks)


def prepare(case, seed):
    g = _gen(seed)
    B, V, dtype = case["B"], case["V"], case["dtype"]
    kind = case["kind"]
    if kind == "sample":
        hist = case["hist"]
        sampler = tg.Sampler(device=0, max_batch=B, max_vocab=V, max_hist=max(hist, 1))
        states = -1
        if case["mask"]:
            sampler.set_mask_table(_mask_table(g, V), V)
            states = np.random.default_rng(seed + 1).integers(0, MASK_STATES, B)
        p = _params(case["policy"], B, V, hist, seed, states)
        s = {"sampler": sampler, "logits": _logits(g, B, V, dtype), "params": tg.params_to_device(p, DEV),
             "u": _uniform(g, B), "hist": None, "hist_len": None, "debug": None,
             "hint": tg.batch_hint(p, V) if case["hint"] else None}
        if hist:
            s["hist"] = _history(g, B, hist, V)
            s["hist_len"] = torch.full((B,), hist, dtype=torch.int32, device=DEV)
        if case["report"]:
            s["debug"] = {"kept_ids": torch.empty(B, REPORT, dtype=torch.int32, device=DEV),
                          "kept_probs": torch.empty(B, REPORT, device=DEV)}
    elif kind == "spec":
        k = case["k"]
        sampler = tg.Sampler(device=0, max_batch=B, max_vocab=V, max_hist=1)
        sampler.reserve_spec(B, k)
        target = torch.randn(B, k + 1, V, generator=g, device=DEV) * 3.0
        draft = target[:, :k] + torch.randn(B, k, V, generator=g, device=DEV)
        tok = torch.multinomial(torch.softmax(draft / case["T"], -1).view(B * k, V), 1, generator=g)
        s = {"sampler": sampler, "target": target.to(DTYPES[dtype]), "draft": draft.to(DTYPES[dtype]),
             "tok": tok.view(B, k).to(torch.int32), "T": torch.full((B,), case["T"], device=DEV),
             "u_acc": _uniform(g, B, k), "u_res": _uniform(g, B)}
    elif kind == "logprob":
        s = {"sampler": tg.Sampler(device=0, max_batch=1, max_vocab=V, max_hist=1),
             "logits": _logits(g, B, V, dtype),
             "tokens": torch.randint(0, V, (B,), generator=g, device=DEV).to(torch.int32)}
    else:
        d, (bc, ct), live = _grammar()
        off, data = _vocabulary(V)
        sampler = tg.Sampler(device=0, max_batch=B, max_vocab=V, max_hist=1)
        sampler.set_mask_table(np.zeros((B, (V + 31) // 32), np.uint32), V)
        up = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(DEV)  # noqa: E731
        p = tg.make_params(B, temperature=0.8, top_k=40, top_p=0.95, mask_state=np.arange(B))
        s = {"sampler": sampler, "logits": _logits(g, B, V, dtype), "params": tg.params_to_device(p, DEV),
             "u": _uniform(g, B), "hint": tg.batch_hint(p, V), "byte_class": up(bc), "trans": up(ct),
             "complete": up(d.complete.astype(np.uint8)), "off": up(off), "data": up(data),
             "states": up(np.random.default_rng(seed).choice(live, B).astype(np.int32)),
             "rows": torch.arange(B, dtype=torch.int32, device=DEV),
             "debug": {"kept_ids": torch.empty(B, 40, dtype=torch.int32, device=DEV)}}
    s["case"] = case
    return s


# ------------------------------------------------------------------ one pass

def run(s):
    kind = s["case"]["kind"]
    if kind == "sample":
        ids = s["sampler"].sample(s["logits"], s["params"], s["u"], hist=s["hist"], hist_len=s["hist_len"],
                                  hint=s["hint"], debug=s["debug"])
        return {"ids": ids, **(s["debug"] or {})}
    if kind == "spec":
        n_acc, out = s["sampler"].spec_verify(s["target"], s["draft"], s["tok"], s["T"], s["u_acc"], s["u_res"])
        return {"n_acc": n_acc, "out": out}
    if kind == "logprob":
        lse = torch.empty(s["logits"].shape[0], device=DEV)
        return {"logprob": s["sampler"].token_logprobs(s["logits"], s["tokens"], lse=lse), "lse": lse}
    s["sampler"].mask_rows_from_dfa(s["byte_class"], s["trans"], s["complete"], s["off"], s["data"], s["states"],
                                    s["rows"])
    ids = s["sampler"].sample(s["logits"], s["params"], s["u"], hint=s["hint"], debug=s["debug"])
    return {"ids": ids, **s["debug"]}


# ------------------------------------------------------------------ what a pass needs, and how exact it is

def work(case):
    """Each input read once, each output written once (floating-point work is
    not what any of these paths is sized by)."""
    B, V, item = case["B"], case["V"], ITEM[case["dtype"]]
    kind = case["kind"]
    if kind == "sample":
        row = V * item + 4 * case["hist"] + 32 + 4 + 4 + ((V + 7) // 8 if case["mask"] else 0)
        return {"bytes": B * (row + (8 * REPORT if case["report"] else 0)), "flops": 0}
    if kind == "spec":
        return {"bytes": B * ((2 * case["k"] + 1) * V * item + 16 * case["k"] + 16), "flops": 0}
    if kind == "logprob":
        return {"bytes": B * (V * item + 12), "flops": 0}
    # token offsets and bytes (about 6), the table written and read once, the logits
    return {"bytes": V * 10 + B * (V * item + 2 * ((V + 7) // 8) + 208), "flops": 0}


def tolerance(case):
    # token ids are whole numbers fixed by the sampling contract; the log-probabilities are fp32 sums
    # (3.5e-8 relative against 64 bits over these cases), the reported probabilities fp32 ratios (1.5e-7)
    if case["kind"] == "logprob":
        return {"rel": 1.5e-7, "max": 2e-6}
    if case["kind"] == "sample" and case["report"]:
        return {"rel": 6e-7, "max": 1e-5}
    return "exact"


def exact(case, seed):
    if case["kind"] == "logprob":
        s = prepare(case, seed)
        lp, lse = [], []
        for i in range(0, case["B"], 64):  # 64 rows at a time in 64 bits
            x = s["logits"][i:i + 64].double()
            z = torch.logsumexp(x, -1)
            lse.append(z)
            lp.append(x.gather(1, s["tokens"][i:i + 64].long().unsqueeze(1)).squeeze(1) - z)
        return {"logprob": torch.cat(lp), "lse": torch.cat(lse)}
    if case["kind"] == "sample" and case["report"]:
        return {"ids": None, "kept_ids": None, "kept_probs": _exact_probs(case, seed)}
    return None


def _exact_probs(case, seed):
    """The reported probabilities of a top-k, top-p row in 64 bits."""
    s = prepare(case, seed)
    B, V, H = case["B"], case["V"], case["hist"]
    p = np.frombuffer(s["params"].cpu().numpy().tobytes(), dtype=tg.make_params(1).dtype)
    z = s["logits"].double().cpu().numpy()
    words = None
    if case["mask"]:
        words = _mask_table(_gen(seed), V)
    out = np.zeros((B, REPORT))
    for b in range(B):
        r, y = p[b], z[b].copy()
        if H:
            ids, n = np.unique(s["hist"][b].cpu().numpy(), return_counts=True)
            y[ids] = y[ids] - float(r["frequency"]) * n - float(r["presence"])
        if words is not None:
            bits = np.unpackbits(words[r["mask_state"]].view(np.uint8), bitorder="little")[:V].astype(bool)
            y[~bits] = -np.inf
        y /= float(r["temperature"])
        k = min(int(r["top_k"]), int(np.isfinite(y).sum()))
        top = np.sort(y)[::-1][:k]
        w = np.exp(top - top[0])
        c = np.cumsum(w)
        n = int(np.searchsorted(c, float(r["top_p"]) * c[-1])) + 1
        got = (w / c[min(n, k) - 1])[:min(n, k, REPORT)]
        out[b, :len(got)] = got
    return torch.from_numpy(out)
