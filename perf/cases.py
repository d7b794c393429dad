"""Performance cases of the tree-verification path: what a serving loop calls.

A target model that verifies draft trees calls, per layer, the K/V append and
the fused tree verify over its (paged or dense) cache, around it plain decode
and chunked-prefill attention, and after the last layer the lm_head and the
acceptance walk, then commits the accepted rows to the cache.  Each kind of
call is one ``kind`` below; the listed cases are the sizes it meets most, and
``draw`` gives others of the same ranges.

    kind     entry points
    verify   tree_verify (with bundle_row_order_device when bundles > 0)
    flash    flash_attn_with_kvcache (decode and causal chunked prefill)
    bundle   FusedBundleVerifier.verify_bundle / PagedBundleVerifier.verify_bundle_paged
    step     append_tree_kv + tree_verify per layer, tree_accept, kv_commit
    accept   tree_accept, greedy and typical
    sample   tree_accept, sampling
    lmhead   lmhead_tree_accept
"""

from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

# The package lives in a subfolder of the working folder (the repository root).
_PKG = os.path.join(os.getcwd(), "specdiff-ae_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from diffspec_mi355x import workloads as wl  # noqa: E402
from diffspec_mi355x.core.bundle_scheduler import bundle_row_order_device  # noqa: E402
from diffspec_mi355x.draft.tree_verification import kv_commit, lmhead_tree_accept, tree_accept  # noqa: E402
from diffspec_mi355x.runtime.attention_compat import flash_attn_with_kvcache  # noqa: E402
from diffspec_mi355x.runtime.bundle_verifier import FusedBundleVerifier, PagedBundleVerifier  # noqa: E402
from diffspec_mi355x.runtime.cache_state import append_tree_kv  # noqa: E402
from diffspec_mi355x.runtime.tree_attention import tree_verify  # noqa: E402

_DTYPE = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
_BYTES = {"bf16": 2, "f16": 2, "f32": 4}
_DEV = "cuda"
# Bounds of a drawn case: what the largest listed cases do (flops of fp32
# cases count 16 times, the ratio of the 16-bit to the fp32 matrix rate).
_MAX_BYTES = 1.11e9
_MAX_FLOPS = 2.8e11


# ----------------------------------------------------------------------------
# The cases
# ----------------------------------------------------------------------------

def listed():
    return [
        # One layer of a short chat turn: a small tree over a 1000-token paged
        # prefix.  Launches and latency.
        dict(name="verify_short", kind="verify", B=1, M=16, N=1000, H=32, Hk=8, D=128, page=16, dtype="bf16", bundles=0),
        # Eight requests verified together, small odd trees over dense caches, f16.
        dict(name="verify_batch", kind="verify", B=8, M=24, N=4099, H=32, Hk=8, D=128, page=0, dtype="f16", bundles=0),
        # The repository's headline step: 64 nodes against a 64K paged prefix.
        dict(name="verify_64k", kind="verify", B=1, M=64, N=65536, H=32, Hk=8, D=128, page=16, dtype="bf16", bundles=0),
        # 128K prefix, 128 nodes packed in bundle order (computed on the device
        # in the same pass).
        dict(name="verify_128k_bundles", kind="verify", B=1, M=128, N=131072, H=32, Hk=8, D=128, page=16, dtype="bf16",
             bundles=8),
        # fp32 models: the 4096-token fp32 configuration, dense cache.
        dict(name="verify_f32", kind="verify", B=1, M=64, N=4096, H=32, Hk=8, D=128, page=0, dtype="f32", bundles=0),
        # Plain decode of a batch with ragged lengths (one token per sequence).
        dict(name="decode_ragged", kind="flash", B=32, M=1, N=8192, H=32, Hk=8, D=128, dtype="bf16", causal=False,
             ragged=True),
        # A 2048-token prefill chunk at the end of an 8192-token context.
        dict(name="prefill_chunk", kind="flash", B=1, M=2048, N=8192, H=32, Hk=8, D=128, dtype="bf16", causal=True,
             ragged=False),
        # The bundle verifier at the reference microbenchmark's shape: K/V in
        # the expanded 32-head form, fp16, a byte mask over all 32000 keys.
        dict(name="bundle_masked", kind="bundle", B=1, M=48, N=32000, H=32, Hk=32, D=128, page=0, dtype="f16"),
        # The library's part of a whole verification step over four layers:
        # append, verify, greedy acceptance, commit.
        dict(name="step_4_layers", kind="step", layers=4, M=48, N=8192, H=32, Hk=8, D=128, page=16, dtype="bf16", V=32000),
        # Typical acceptance of eight 64-node trees over a 128256-token vocabulary.
        dict(name="accept_typical", kind="accept", mode="typical", T=8, M=64, V=128256, dtype="bf16"),
        # Sampling acceptance with the usual temperature and top-p.
        dict(name="accept_sample", kind="sample", T=4, M=64, V=128256, dtype="bf16", temperature=0.8, top_p=0.9, top_k=0),
        # lm_head and greedy acceptance of three trees (192 rows), with logits.
        dict(name="lmhead_3_trees", kind="lmhead", mode="greedy", T=3, M=64, V=128256, hidden=4096),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw(rng):
    kind = rng.choice(["verify", "verify", "verify", "flash", "flash", "bundle", "step", "accept", "sample", "lmhead"])
    H, Hk = rng.choice([(32, 8), (32, 8), (32, 8), (32, 32), (16, 4), (12, 4), (8, 8), (8, 2), (4, 1)])
    D = rng.choice([128, 128, 128, 64])
    if kind == "verify":
        dtype = rng.choice(["bf16", "bf16", "f16", "f32"])
        M = _logint(rng, 3, 300)
        return dict(kind=kind, B=rng.choice([1, 1, 1, 2, 3, 8]), M=M, N=_logint(rng, 200, 131072), H=H, Hk=Hk, D=D,
                    page=rng.choice([0, 16, 16, 32, 64]), dtype=dtype, bundles=rng.choice([0, 0, 8]))
    if kind == "flash":
        dtype = rng.choice(["bf16", "f16"])
        if rng.random() < 0.5:  # decode
            return dict(kind=kind, B=_logint(rng, 1, 64), M=rng.choice([1, 1, 1, 2, 4, 7]), N=_logint(rng, 200, 32768),
                        H=H, Hk=Hk, D=D, dtype=dtype, causal=True, ragged=rng.random() < 0.7)
        M = _logint(rng, 128, 4096)  # prefill: a chunk at the end of N keys
        return dict(kind=kind, B=rng.choice([1, 1, 2, 4]), M=M, N=M + rng.choice([0, _logint(rng, 16, 16384)]), H=H, Hk=Hk,
                    D=D, dtype=dtype, causal=True, ragged=False)
    if kind == "bundle":
        return dict(kind=kind, B=rng.choice([1, 1, 2]), M=_logint(rng, 4, 128), N=_logint(rng, 500, 40000), H=H, Hk=Hk, D=D,
                    page=rng.choice([0, 16]), dtype=rng.choice(["bf16", "f16"]))
    V = rng.choice([32000, 50257, 128256])
    if kind == "step":
        return dict(kind=kind, layers=rng.randint(1, 6), M=_logint(rng, 8, 128), N=_logint(rng, 500, 32768), H=H, Hk=Hk, D=D,
                    page=rng.choice([16, 16, 32]), dtype=rng.choice(["bf16", "f16"]), V=V)
    dtype = rng.choice(["bf16", "bf16", "f16", "f32"])
    T, M = rng.choice([1, 1, 2, 4, 8]), _logint(rng, 8, 128)
    if kind == "accept":
        return dict(kind=kind, mode=rng.choice(["greedy", "typical"]), T=T, M=M, V=V, dtype=dtype)
    if kind == "sample":
        top_p, top_k = rng.choice([(1.0, 0), (0.9, 0), (0.95, 0), (0.9, 50), (1.0, 50)])
        return dict(kind=kind, T=T, M=M, V=V, dtype=dtype, temperature=rng.choice([0.7, 0.8, 1.0]), top_p=top_p, top_k=top_k)
    return dict(kind=kind, mode=rng.choice(["greedy", "greedy", "typical"]), T=T, M=M, V=V,
                hidden=rng.choice([2048, 4096, 4096]))


def draw(rng):
    while True:
        case = _draw(rng)
        w = work(case)
        flops = w["flops"] * (16 if case.get("dtype") == "f32" and case["kind"] == "verify" else 1)
        if w["bytes"] <= _MAX_BYTES and flops <= _MAX_FLOPS:
            return case


# ----------------------------------------------------------------------------
# Inputs
# ----------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=_DEV)
    g.manual_seed(int(seed) % (1 << 62))
    return g


def _randn(g, shape, scale, dtype):
    """N(0, scale) in ``dtype``, made in pieces so that no fp32 copy of a large tensor exists."""
    out = torch.empty(shape, dtype=dtype, device=_DEV)
    flat = out.view(-1)
    step = 1 << 26
    for i in range(0, flat.numel(), step):
        part = flat[i:i + step]
        part.copy_(torch.randn(part.numel(), generator=g, device=_DEV) * scale)
    return out


def _np_rng(seed):
    return np.random.default_rng(int(seed) % (1 << 31))


def _tree(M, seed):
    return wl.make_tree(M, max_depth=12, max_outdeg=6, seed=int(seed) % (1 << 31))


def _pool(g, rng, c, layers, tokens):
    """A page pool [layers, 2, P, Hk, page, D] and page tables [B, n] (or [n] for one sequence)."""
    n = -(-tokens // c["page"])
    B = c.get("B", 1)
    pool = _randn(g, (layers, 2, B * n, c["Hk"], c["page"], c["D"]), 1.0, _DTYPE[c["dtype"]])
    pt = rng.permutation(B * n).astype(np.int32).reshape(B, n)
    return pool, torch.from_numpy(pt[0] if B == 1 else pt).to(_DEV)


# Query scale: scores q.k / sqrt(D) of standard deviation 1.5, softmax weights
# that concentrate on a part of the keys, as a trained model's do.
_QS = 1.5


def _prepare_verify(c, seed):
    g, rng = _gen(seed), _np_rng(seed)
    B, M, N, H, Hk, D, dt = c["B"], c["M"], c["N"], c["H"], c["Hk"], c["D"], _DTYPE[c["dtype"]]
    s = dict(c=c, q=_randn(g, (B, M, H, D), _QS, dt), pt=None)
    if c["page"]:
        s["pool"], s["pt"] = _pool(g, rng, c, 1, N + M)
        s["k"], s["v"] = s["pool"][0, 0], s["pool"][0, 1]
    else:
        s["k"], s["v"] = _randn(g, (B, N + M, Hk, D), 1.0, dt), _randn(g, (B, N + M, Hk, D), 1.0, dt)
    s["trees"] = [_tree(M, seed * 131 + b)[0] for b in range(B)]
    par = torch.tensor(s["trees"], dtype=torch.int64, device=_DEV)
    s["parent"] = par[0] if B == 1 else par
    s["parent0"] = par[0].contiguous()  # the packing order is one tree's
    return s


def _prepare_flash(c, seed):
    g, rng = _gen(seed), _np_rng(seed)
    B, M, N, H, Hk, D, dt = c["B"], c["M"], c["N"], c["H"], c["Hk"], c["D"], _DTYPE[c["dtype"]]
    lens = None
    if c["ragged"]:
        lens = np.clip(np.round(N * rng.uniform(0.1, 1.0, B)).astype(np.int64), M, N)
        lens[rng.integers(B)] = N
        lens = torch.from_numpy(lens.astype(np.int32)).to(_DEV)
    return dict(c=c, q=_randn(g, (B, M, H, D), _QS, dt), k=_randn(g, (B, N, Hk, D), 1.0, dt),
                v=_randn(g, (B, N, Hk, D), 1.0, dt), lens=lens)


def _prepare_bundle(c, seed):
    g, rng = _gen(seed), _np_rng(seed)
    B, M, N, H, Hk, D, dt = c["B"], c["M"], c["N"], c["H"], c["Hk"], c["D"], _DTYPE[c["dtype"]]
    s = dict(c=c, q=_randn(g, (B, M, H, D), _QS, dt), pt=None)
    if c["page"]:
        s["pool"], s["pt"] = _pool(g, rng, c, 1, N)
    else:
        s["k"], s["v"] = _randn(g, (B, N, Hk, D), 1.0, dt), _randn(g, (B, N, Hk, D), 1.0, dt)
    mask = np.ones((M, N), dtype=np.int8)  # the shared prefix, then the bundle's tree
    T = min(M, N)
    mask[:, N - T:] = wl.ancestor_mask(_tree(M, seed)[0])[:, :T]
    s["mask"] = torch.from_numpy(mask).to(_DEV)
    s["ver"] = (PagedBundleVerifier if c["page"] else FusedBundleVerifier)(bundle_size=3, device=_DEV)
    return s


def _rope(M, D, pos, dt):
    inv = 1.0 / (5e5 ** (torch.arange(0, D, 2, device=_DEV, dtype=torch.float32) / D))
    ang = pos.float()[:, None] * inv[None, :]
    return torch.cat([ang.cos()] * 2, -1).to(dt), torch.cat([ang.sin()] * 2, -1).to(dt)


def _prepare_step(c, seed):
    g, rng = _gen(seed), _np_rng(seed)
    L, M, N, H, Hk, D, dt = c["layers"], c["M"], c["N"], c["H"], c["Hk"], c["D"], _DTYPE[c["dtype"]]
    a = wl.make_accept_inputs(T=1, M=M, V=c["V"], dtype=dt, seed=int(seed) % (1 << 20), device=_DEV, max_outdeg=6,
                              max_depth=12)
    pool, pt = _pool(g, rng, dict(c, B=1), L, N + M)
    # The fused QKV projection's output of each layer: q, k, v are views of it.
    qkv = _randn(g, (L, M, (H + 2 * Hk) * D), 1.0, dt)
    pos = torch.tensor([N + d for d in a.depths[0]], dtype=torch.int64, device=_DEV)
    cos, sin = _rope(M, D, pos, dt)
    return dict(c=c, pool=pool, pt=pt, acc=a, pos=pos, cos=cos, sin=sin, tree=a.parents[0],
                parent=torch.tensor(a.parents[0], dtype=torch.int64, device=_DEV), hops=min(max(a.depths[0]) + 2, M),
                q=[x[:, :H * D].view(M, H, D) for x in qkv], k=[x[:, H * D:(H + Hk) * D].view(M, Hk, D) for x in qkv],
                v=[x[:, (H + Hk) * D:].view(M, Hk, D) for x in qkv])


def _prepare_accept(c, seed):
    a = wl.make_accept_inputs(T=c["T"], M=c["M"], V=c["V"], dtype=_DTYPE[c["dtype"]], seed=int(seed) % (1 << 20),
                              max_depth=12, max_outdeg=6, device=_DEV)
    return dict(c=c, a=a, hops=min(14, c["M"]))


def _prepare_sample(c, seed):
    """Rows of three sorts, as a language model's next-token rows are: sure of
    one token, undecided between some tens, and open (a few hundred to a few
    thousand tokens share the mass)."""
    g, rng = _gen(seed), _np_rng(seed)
    s = _prepare_accept(c, seed)
    T, M, V = c["T"], c["M"], c["V"]
    sort = torch.from_numpy(rng.choice(3, size=(T, M), p=[0.65, 0.25, 0.1])).to(_DEV)
    sigma = torch.from_numpy(rng.uniform(2.5, 3.5, size=(T, M)).astype(np.float32)).to(_DEV)
    rungs = 40
    ids = torch.from_numpy(rng.integers(0, V, size=(T, M, rungs))).to(_DEV)
    ladder = 17.0 - 0.25 * torch.arange(rungs, device=_DEV, dtype=torch.float32)
    for t in range(T):
        x = s["a"].logits[t]
        own = torch.randn((M, V), generator=g, device=_DEV) * sigma[t][:, None]
        tens = own.clone().scatter_(1, ids[t], ladder.expand(M, rungs))
        x.copy_(torch.where((sort[t] == 1)[:, None], tens, torch.where((sort[t] == 2)[:, None], own, x.float())))
    s["seed"] = int(rng.integers(1 << 62))
    return s


def _prepare_lmhead(c, seed):
    """Unit-RMS hidden rows (after the final norm) that lean towards one
    token's weight row by a margin that differs from row to row."""
    g, rng = _gen(seed), _np_rng(seed)
    T, M, V, Dm = c["T"], c["M"], c["V"], c["hidden"]
    W = _randn(g, (V, Dm), 0.02, torch.bfloat16)
    top = torch.from_numpy(rng.integers(0, V, size=(T, M))).to(_DEV)
    lean = torch.from_numpy(rng.uniform(5.0, 10.0, size=(T, M, 1)).astype(np.float32)).to(_DEV) * math.sqrt(4096 / Dm)
    x = torch.randn((T, M, Dm), generator=g, device=_DEV) + lean * W[top].float()
    x = (x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True))).to(torch.bfloat16)
    draft = rng.integers(0, V, size=(T, M))
    pref, pos = [], []
    for t in range(T):  # a root path of each tree agrees with the target
        parent, depth = _tree(M, seed * 131 + t)
        node, tt = int(rng.integers(M)), top[t].cpu().numpy()
        while node > 0:
            draft[t, node] = tt[parent[node]]
            node = parent[node]
        pref.append(wl.parent_to_reference(parent))
        pos.append(depth)
    return dict(c=c, h=x, W=W, draft=torch.from_numpy(draft).to(_DEV), hops=min(14, M),
                parent=torch.tensor(pref, dtype=torch.int64, device=_DEV).reshape(T, M - 1),
                pos=torch.tensor(pos, dtype=torch.int64, device=_DEV))


_PREPARE = dict(verify=_prepare_verify, flash=_prepare_flash, bundle=_prepare_bundle, step=_prepare_step,
                accept=_prepare_accept, sample=_prepare_sample, lmhead=_prepare_lmhead)


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, int(seed))


# ----------------------------------------------------------------------------
# One pass
# ----------------------------------------------------------------------------

def _run_verify(s, c):
    perm = bundle_row_order_device(s["parent0"], num_bundles=c["bundles"]) if c["bundles"] else None
    out, lse = tree_verify(s["q"], s["k"], s["v"], c["N"], s["parent"], page_table=s["pt"], row_perm=perm,
                           check_row_perm=False)
    return {"out": out, "lse": lse}


def _run_flash(s, c):
    out, lse = flash_attn_with_kvcache(s["q"], s["k"], s["v"], causal=c["causal"], cache_seqlens=s["lens"],
                                       return_softmax_lse=True)
    return {"out": out, "lse": lse}


def _run_bundle(s, c):
    prefix = max(0, c["N"] - c["M"])
    if c["page"]:
        out, lse = s["ver"].verify_bundle_paged(s["q"], s["pool"], s["pt"], [s["mask"]], shared_prefix_len=prefix)
    else:
        out, lse = s["ver"].verify_bundle(s["q"], s["k"], s["v"], [s["mask"]], shared_prefix_len=prefix)
    return {"out": out, "lse": lse}


def _run_step(s, c):
    pool, pt, N = s["pool"], s["pt"], c["N"]
    outs, lses = [], []
    for l in range(c["layers"]):
        q = append_tree_kv(s["k"][l], s["v"][l], pool[l, 0], pool[l, 1], N, cos=s["cos"], sin=s["sin"], page_table=pt,
                           q=s["q"][l])
        out, lse = tree_verify(q.unsqueeze(0), pool[l, 0], pool[l, 1], N, s["parent"], page_table=pt)
        outs.append(out)
        lses.append(lse)
    a = s["acc"]
    r = tree_accept(a.logits, a.draft, a.parent_ref, a.pos, s["hops"])
    kv_commit(pool, N, r["path"], r["info"], page_table=pt)
    return {"out": outs, "lse": lses, "pool": pool, "path": r["path"], "tokens": r["tokens"], "info": r["info"]}


def _run_accept(s, c):
    a = s["a"]
    return tree_accept(a.logits, a.draft, a.parent_ref, a.pos, s["hops"], mode=c["mode"], return_next=True)


def _run_sample(s, c):
    a = s["a"]
    return tree_accept(a.logits, a.draft, a.parent_ref, a.pos, s["hops"], mode="sample", temperature=c["temperature"],
                       top_p=c["top_p"], top_k=c["top_k"], seed=s["seed"], return_next=True)


def _run_lmhead(s, c):
    return lmhead_tree_accept(s["h"], s["W"], s["draft"], s["parent"], s["pos"], s["hops"], mode=c["mode"],
                              return_next=True, return_logits=True)


_RUN = dict(verify=_run_verify, flash=_run_flash, bundle=_run_bundle, step=_run_step, accept=_run_accept,
            sample=_run_sample, lmhead=_run_lmhead)


def run(state):
    c = state["c"]
    return _RUN[c["kind"]](state, c)


# ----------------------------------------------------------------------------
# Work and tolerances
# ----------------------------------------------------------------------------

def _attn_work(c, keys, pairs):
    """``keys``: K/V rows read per KV head over all batches; ``pairs``: visible
    (query row, key) pairs per query head."""
    es = _BYTES[c["dtype"]]
    rows = c.get("B", 1) * c["M"]
    b = 2 * keys * c["Hk"] * c["D"] * es + 2 * rows * c["H"] * c["D"] * es + 4 * rows * c["H"]
    return {"bytes": b, "flops": 4 * pairs * c["H"] * c["D"]}


def work(case):
    c = case
    kind = c["kind"]
    if kind == "verify":
        # Tree keys count as one per node pair of the dense M x M block.
        return _attn_work(c, c["B"] * (c["N"] + c["M"]), c["B"] * c["M"] * (c["N"] + c["M"]))
    if kind == "flash":
        # Ragged lengths average 0.55 N; causal chunks see half of their own block.
        n = c["N"] * (0.55 if c["ragged"] else 1.0)
        seen = max(n - (c["M"] - 1) / 2, 1.0) if c["causal"] else n
        return _attn_work(c, c["B"] * n, c["B"] * c["M"] * seen)
    if kind == "bundle":
        w = _attn_work(c, c["B"] * c["N"], c["B"] * c["M"] * c["N"])
        return {"bytes": w["bytes"] + c["M"] * c["N"], "flops": w["flops"]}
    if kind == "step":
        es = _BYTES[c["dtype"]]
        w = _attn_work(c, c["N"] + c["M"], c["M"] * (c["N"] + c["M"]))
        append = 2 * c["M"] * (c["H"] + 2 * c["Hk"]) * c["D"] * es
        return {"bytes": c["layers"] * (w["bytes"] + append) + c["M"] * c["V"] * es, "flops": c["layers"] * w["flops"]}
    if kind in ("accept", "sample"):
        return {"bytes": c["T"] * c["M"] * c["V"] * _BYTES[c["dtype"]], "flops": 0}
    R = c["T"] * c["M"]
    return {"bytes": 2 * c["V"] * c["hidden"] + 2 * R * c["hidden"] + 2 * R * c["V"], "flops": 2 * R * c["V"] * c["hidden"]}


def tolerance(case):
    kind = case["kind"]
    if kind in ("accept", "sample"):
        return "exact"  # tokens and node ids only, defined bit for bit
    if kind == "lmhead":
        # bf16 logits (half a step is 2^-9 of the value); a token may differ
        # where two logits round to neighbouring bf16 values.
        return {"rel": 8e-3, "max": 3e-2, "differ": 2e-2}
    # 16-bit probabilities, split results and outputs, about four times what the
    # path shows against float64: 0.0029 in bf16 (0.0037 with the 16-bit RoPE of
    # a step before it) and 0.0017 in f16 and f32 (bf16 split results).
    if kind == "step":
        return {"rel": 1.5e-2, "max": 1e-1}
    return {"rel": 1.2e-2 if case["dtype"] == "bf16" else 7e-3, "max": 8e-2 if case["dtype"] == "bf16" else 5e-2}


# ----------------------------------------------------------------------------
# Plain float64 results
# ----------------------------------------------------------------------------

def _attend(q, k, v, keep=None):
    """q [M, H, D], k, v [N, Hk, D] float64, keep [M, N] bool or None -> out [M, H, D], lse [M, H]."""
    M, H, D = q.shape
    Hk = k.shape[1]
    out = torch.empty((M, H, D), dtype=torch.float64, device=q.device)
    lse = torch.empty((M, H), dtype=torch.float64, device=q.device)
    for h in range(H):
        kk, vv = k[:, h // (H // Hk)].contiguous(), v[:, h // (H // Hk)].contiguous()
        for m0 in range(0, M, 512):
            sc = q[m0:m0 + 512, h].contiguous() @ kk.t().contiguous() / math.sqrt(D)
            if keep is not None:
                sc.masked_fill_(~keep[m0:m0 + 512], -math.inf)
            l = torch.logsumexp(sc, dim=1)
            sc = torch.exp(sc - torch.where(torch.isinf(l), torch.zeros_like(l), l)[:, None])
            out[m0:m0 + 512, h] = sc @ vv
            lse[m0:m0 + 512, h] = l
    return out, lse


def _logical(pages, pt, n, page):
    tok = torch.arange(n, device=_DEV)
    return pages[pt.long()[tok // page], :, tok % page].double()


def _ancestors(parent):
    keep = torch.zeros((len(parent), len(parent)), dtype=torch.bool)
    for i in range(len(parent)):
        j = i
        while j >= 0:
            keep[i, j] = True
            j = parent[j]
    return keep.to(_DEV)


def _tree_keep(parent, N):
    M = len(parent)
    return torch.cat([torch.ones((M, N), dtype=torch.bool, device=_DEV), _ancestors(parent)], dim=1)


def _exact_verify(s, c):
    outs, lses = [], []
    for b in range(c["B"]):
        if c["page"]:
            pt = s["pt"] if s["pt"].dim() == 1 else s["pt"][b]
            k, v = (_logical(x, pt, c["N"] + c["M"], c["page"]) for x in (s["k"], s["v"]))
        else:
            k, v = s["k"][b].double(), s["v"][b].double()
        o, l = _attend(s["q"][b].double(), k, v, _tree_keep(s["trees"][b], c["N"]))
        outs.append(o)
        lses.append(l)
    return {"out": torch.stack(outs), "lse": torch.stack(lses)}


def _exact_flash(s, c):
    outs, lses = [], []
    for b in range(c["B"]):
        n = int(s["lens"][b]) if s["lens"] is not None else c["N"]
        keep = None
        if c["causal"]:
            keep = (torch.arange(n, device=_DEV)[None, :]
                    <= n - c["M"] + torch.arange(c["M"], device=_DEV)[:, None])
        o, l = _attend(s["q"][b].double(), s["k"][b, :n].double(), s["v"][b, :n].double(), keep)
        outs.append(o)
        lses.append(l.t())
    return {"out": torch.stack(outs), "lse": torch.stack(lses)}


def _exact_bundle(s, c):
    outs, lses = [], []
    for b in range(c["B"]):
        if c["page"]:
            pt = s["pt"] if s["pt"].dim() == 1 else s["pt"][b]
            k, v = (_logical(s["pool"][0, x], pt, c["N"], c["page"]) for x in (0, 1))
        else:
            k, v = s["k"][b].double(), s["v"][b].double()
        o, l = _attend(s["q"][b].double(), k, v, s["mask"] != 0)
        outs.append(o)
        lses.append(l)
    return {"out": torch.stack(outs), "lse": torch.stack(lses)}


def _exact_step(s, c):
    M, N, page, pt = c["M"], c["N"], c["page"], s["pt"].long()
    cos, sin = s["cos"].double()[:, None], s["sin"].double()[:, None]

    def rope(x):
        x = x.double()
        a, b = x.chunk(2, -1)
        return x * cos + torch.cat([-b, a], -1) * sin

    pool = s["pool"].double()
    tok = N + torch.arange(M, device=_DEV)
    outs, lses = [], []
    keep = _tree_keep(s["tree"], N)
    for l in range(c["layers"]):
        pool[l, 0][pt[tok // page], :, tok % page] = rope(s["k"][l])
        pool[l, 1][pt[tok // page], :, tok % page] = s["v"][l].double()
        o, ls = _attend(rope(s["q"][l]), _logical(pool[l, 0], pt, N + M, page), _logical(pool[l, 1], pt, N + M, page), keep)
        outs.append(o[None])
        lses.append(ls[None])
    # The accepted path: the deepest node whose root path agrees with the argmax.
    nxt = s["acc"].logits[0].float().argmax(-1).tolist()
    draft, depth, tree = s["acc"].draft[0].tolist(), s["acc"].depths[0], s["tree"]
    ok = [True] * M
    for i in range(1, M):  # parents precede children
        ok[i] = ok[tree[i]] and draft[i] == nxt[tree[i]]
    node = max((i for i in range(M) if ok[i]), key=lambda i: (depth[i], -i))
    path = []
    while node >= 0:
        path.append(node)
        node = tree[node]
    src, dst = tok[torch.tensor(path[::-1], device=_DEV)], tok[:len(path)]
    for l in range(c["layers"]):
        for x in (0, 1):
            pool[l, x][pt[dst // page], :, dst % page] = pool[l, x][pt[src // page], :, src % page]
    return {"out": outs, "lse": lses, "pool": pool, "path": None, "tokens": None, "info": None}


def _exact_lmhead(s, c):
    h = s["h"].reshape(-1, c["hidden"]).double()
    logits = torch.empty((h.shape[0], c["V"]), dtype=torch.float64, device=_DEV)
    for i in range(0, c["V"], 16384):
        logits[:, i:i + 16384] = h @ s["W"][i:i + 16384].double().t().contiguous()
    return {"path": None, "tokens": None, "info": None, "next": None, "logits": logits.view(c["T"], c["M"], c["V"])}


_EXACT = dict(verify=_exact_verify, flash=_exact_flash, bundle=_exact_bundle, step=_exact_step, lmhead=_exact_lmhead)


def exact(case, seed):
    if case["kind"] not in _EXACT:
        return None
    return _EXACT[case["kind"]](prepare(case, seed), case)
