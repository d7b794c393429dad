"""Dense attention of one split: the kernel writes the output and the LSE itself.

Sizes at the edges of its row blocks (256 rows of query heads x nodes) and of
the causal cut (rows that see few or no keys), with per-batch lengths; the
reference is float64 attention, the bounds those of the other attention tests.
Batch 16 x 16 KV heads fill the GPU, so that every call is one split.
"""

import pytest
import torch

from diffspec_mi355x.runtime.attention_compat import flash_attn_with_kvcache

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,D", [(1, 33, 128), (70, 200, 64), (128, 128, 128), (129, 300, 128), (300, 310, 64)])
@pytest.mark.parametrize("causal", [True, False])
def test_one_split_output(gpu, dtype, M, N, D, causal):
    B, H, Hk = 16, 32, 16
    print(f"[direct output] {dtype} M={M} N={N} D={D} causal={causal}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(M + N)
    q, k, v = (torch.randn(s, generator=g, device=gpu).to(dtype) for s in ((B, M, H, D), (B, N, Hk, D), (B, N, Hk, D)))
    lens = torch.randint(0, N + 1, (B,), generator=torch.Generator().manual_seed(N))
    lens[0], lens[1] = N, 0
    out, lse = flash_attn_with_kvcache(q, k, v, causal=causal, cache_seqlens=lens.to(gpu), return_softmax_lse=True)
    torch.cuda.synchronize()
    for b in range(B):
        n = int(lens[b])
        keep = torch.ones((M, n), dtype=torch.bool, device=gpu)
        if causal:
            keep = torch.arange(n, device=gpu)[None, :] <= n - M + torch.arange(M, device=gpu)[:, None]
        for h in range(0, H, 5):
            s = (q[b, :, h].double() @ k[b, :n, h // 2].double().t().contiguous()) / D ** 0.5
            s = s.masked_fill(~keep, float("-inf"))
            l = torch.logsumexp(s, dim=1) if n else torch.full((M,), float("-inf"), device=gpu, dtype=torch.float64)
            p = torch.exp(s - torch.where(torch.isinf(l), 0.0, l)[:, None])
            o = p @ v[b, :n, h // 2].double().contiguous()
            seen = ~torch.isinf(l)
            assert torch.equal(torch.isinf(lse[b, h]), ~seen) and (out[b, ~seen, h] == 0).all()
            if seen.any():
                rel = ((out[b, seen, h].double() - o[seen]).norm() / o[seen].norm()).item()
                err = (lse[b, h, seen].double() - l[seen]).abs().max().item()
                assert rel <= 1e-2 and err <= 2e-3, (b, h, rel, err)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("D", [64, 128])
def test_rows_without_keys_beside_nonfinite_values(gpu, dtype, bad, D):
    B, M, H, Hk, N = 16, 70, 32, 16, 96
    print(f"[direct output] rows without keys {dtype} {bad} D={D}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(D)
    q, k, v = (torch.randn(s, generator=g, device=gpu).to(dtype) for s in ((B, M, H, D), (B, N, Hk, D), (B, N, Hk, D)))
    v[:, 3] = bad
    lens = torch.arange(B, device=gpu) * 5 + 1  # up to 76: the first M - len rows see nothing
    out, lse = flash_attn_with_kvcache(q, k, v, causal=True, cache_seqlens=lens, return_softmax_lse=True)
    torch.cuda.synchronize()
    for b in range(B):
        n = int(lens[b])
        first = max(0, M - n)  # row m sees keys up to n - M + m
        assert (out[b, :first] == 0).all() and torch.isneginf(lse[b, :, :first]).all(), f"batch {b}"
        assert torch.isfinite(lse[b, :, first:]).all(), f"batch {b}"
        sees = n - M + torch.arange(M, device=gpu) >= 3
        assert not torch.isfinite(out[b, sees]).any(), f"batch {b}"
