"""Sampling, 16-bit logits: the count of a row's values (one workgroup per row).

Where it can go wrong: a counter that overflows (more than 65535 entries of one
value), a top-p cut or a k-th value whose y several logits share (a high
temperature merges logits), ragged and unaligned rows, rows of -inf, NaN and
+inf, k beyond the finite entries, and both ways into the kernel (all rows, or
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
@pytest.mark.parametrize("M,V", [(33, 4099), (5, 4099), (40, 1), (34, 9)])  # all rows at once from 32 rows on
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
