"""Sampling, 16-bit logits: heads and the count of a row's values (one workgroup per row).

Where it can go wrong: a counter that overflows (more than 65535 entries of one
value), a top-p cut or a k-th value whose y several logits share (a high
temperature merges logits), ragged and unaligned rows, rows of -inf, NaN and
+inf, k beyond the finite entries, more distinct values than the counts' list
holds, rows that a head decides beside rows that it does not or that do not try,
and the ways into the kernel (all rows, the rows that their head leaves open,
the rows that the select kernel leaves open).  Every draw is compared bit for
bit with the oracle's.
"""

import numpy as np
import pytest
import torch

from oracle import sampling as sp
from diffspec_mi355x import workloads as wl
from diffspec_mi355x.draft.tree_verification import tree_accept

pytestmark = pytest.mark.gpu

DT = {torch.bfloat16: "bf16", torch.float16: "f16"}


def _run(logits, temperature, top_p, top_k, seed):
    T, M, V = logits.shape
    a = wl.make_accept_inputs(T=T, M=M, V=V, device="cuda", seed=3)
    r = tree_accept(logits, a.draft, a.parent_ref, a.pos, min(14, M), mode="sample", temperature=temperature, top_p=top_p,
                    top_k=top_k, seed=seed, return_next=True)
    torch.cuda.synchronize()
    lg = logits.float().cpu().numpy()
    for t in range(T):
        draws = sp.sample_walk(lg[t], DT[logits.dtype], a.draft[t].cpu().numpy(), a.parent_ref[t].cpu().tolist(),
                               a.pos[t].cpu().numpy(), 12, temperature, top_p, top_k, seed, tree=t)[-1]
        assert r["next"][t].tolist() == draws.tolist(), f"tree {t}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,V", [(33, 4099), (5, 4099), (40, 1), (34, 9)])
@pytest.mark.parametrize("temperature,top_p,top_k", [(1.0, 0.9, 0), (37.0, 0.6, 0), (0.3, 0.95, 20), (1.7, 1.0, 5),
                                                     (250.0, 0.5, 900)])
def test_value_counts(gpu, dtype, M, V, temperature, top_p, top_k):
    print(f"[sample values] {dtype} M={M} V={V} T={temperature} p={top_p} k={top_k}", flush=True)
    g = torch.Generator().manual_seed(M * V)
    lg = (torch.randn((1, M, V), generator=g) * 3.0).to(dtype)
    lg[0, 1] = float("-inf")
    lg[0, 2, V // 2] = float("inf")
    lg[0, 3, ::3] = float("nan")
    lg[0, 4] = -lg[0, 4].abs() - 5.0
    _run(lg.to(gpu), temperature, top_p, top_k, seed=17)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_value_counters_overflow_and_large_kept_sets(gpu, dtype):
    M, V = 32, 70001
    print(f"[sample values] overflow {dtype}", flush=True)
    lg = torch.zeros((1, M, V), dtype=dtype)  # one value 70001 times
    lg[0, 1] = 1.5
    lg[0, 1, 69999:] = 9.0
    lg[0, 2:] = (torch.randn((M - 2, V), generator=torch.Generator().manual_seed(1)) * 0.1).to(dtype)  # flat
    _run(lg.to(gpu), 0.8, 0.9, 0, seed=5)
    _run(lg.to(gpu), 0.8, 1.0, 66000, seed=6)


# Rows sure of a token, undecided between tens, with a tie at the top, and open to
# different degrees: some are decided by their head, some try in vain, some do
# not try; odd V (unaligned rows), V around the 1024 vectors of a block, short and
# long.
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("V", [8191, 8193, 16384, 20011])
@pytest.mark.parametrize("temperature,top_p,top_k", [(0.8, 0.9, 0), (1.0, 0.95, 0), (1.0, 0.999, 0), (0.8, 0.9, 50), (0.8, 1.0, 50),
                                                     (1.0, 1.0, 1030)])
def test_heads_and_counts(gpu, dtype, V, temperature, top_p, top_k):
    M = 42
    print(f"[sample values] heads {dtype} V={V} T={temperature} p={top_p} k={top_k}", flush=True)
    g = torch.Generator().manual_seed(V + top_k)
    lg = torch.randn((1, M, V), generator=g) * (2.0 + 0.05 * torch.arange(M)[:, None])
    for m in range(M):
        ids = torch.randperm(V, generator=g)
        if m % 4 == 0:
            lg[0, m, ids[0]] = 25.0
        elif m % 4 == 1:
            lg[0, m, ids[:40]] = 17.0 - 0.25 * torch.arange(40)
        elif m % 8 == 2:
            lg[0, m, ids[:1500]] = 11.0
    _run(lg.to(dtype).to(gpu), temperature, top_p, top_k, seed=23)


@pytest.mark.parametrize("dtype,temperature", [(torch.bfloat16, 1.5e38), (torch.float16, 2.5e4)])
def test_more_distinct_values_than_the_list(gpu, dtype, temperature):
    M = 6
    print(f"[sample values] distinct {dtype}", flush=True)
    bits = torch.arange(65536, dtype=torch.int32)
    inf = 0x7F80 if dtype == torch.bfloat16 else 0x7C00
    bits = bits[(bits & 0x7FFF) < inf].to(torch.int16)  # every finite value once, all of a mass within e^-6 of the largest
    lg = torch.stack([bits[torch.randperm(len(bits), generator=torch.Generator().manual_seed(m))] for m in range(M)])
    lg = lg.view(dtype)[None].to(gpu)
    for top_p, top_k in ((0.9, 0), (1.0, 40000), (0.02, 0), (0.9, 40000)):
        _run(lg, temperature, top_p, top_k, seed=7)


def test_long_rows_of_most_cus(gpu):
    M, V = 200, 65600  # bf16, three quarters of 256 CUs: straight to the counts
    print("[sample values] long rows", flush=True)
    lg = torch.randn((1, M, V), generator=torch.Generator().manual_seed(4)) * 3.0
    lg[0, ::2, 77] = 25.0
    _run(lg.to(torch.bfloat16).to(gpu), 0.8, 0.9, 0, seed=9)
