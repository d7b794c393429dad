"""Dense attention of one split: the kernel writes the output and the LSE itself.

Sizes at the edges of its row blocks (256 rows of query heads x nodes) and of
the causal cut (rows that see few or no keys), with per-batch lengths; the
reference is float64 attention, the bounds those of the other attention tests.
Batch x KV heads x row blocks fill the GPU, so that every call is one split (which
the workspace's size shows).
"""

import pytest
import torch

from diffspec_mi355x import _ext
from diffspec_mi355x.runtime.attention_compat import flash_attn_with_kvcache

pytestmark = pytest.mark.gpu


def _one_split_bytes(B, M, H, Hk, D, N):
    """The call's workspace, one split's."""
    ws = _ext.load().dsv_attn_workspace_bytes(B, M, H, Hk, D, N, 0, 0)
    assert ws == -(-B * H * M * D * 2 // 256) * 256 + -(-B * H * M * 8 // 256) * 256, "the plan has more than one split"
    return ws


def _check_rows(out, lse, q, k, v, lens, causal, heads):
    """out [B, M, H, D], lse [B, H, M] against float64 attention; rows without keys are zero."""
    B, M, H, D = q.shape
    G = H // k.shape[2]
    dev = q.device
    for b in range(B):
        n = int(lens[b])
        keep = torch.ones((M, n), dtype=torch.bool, device=dev)
        if causal:
            keep = torch.arange(n, device=dev)[None, :] <= n - M + torch.arange(M, device=dev)[:, None]
        for h in heads:
            s = (q[b, :, h].double() @ k[b, :n, h // G].double().t().contiguous()) / D ** 0.5
            s = s.masked_fill(~keep, float("-inf"))
            l = torch.logsumexp(s, dim=1) if n else torch.full((M,), float("-inf"), device=dev, dtype=torch.float64)
            o = torch.exp(s - torch.where(torch.isinf(l), 0.0, l)[:, None]) @ v[b, :n, h // G].double().contiguous()
            seen = ~torch.isinf(l)
            assert torch.equal(torch.isinf(lse[b, h]), ~seen) and (out[b, ~seen, h] == 0).all()
            if seen.any():
                rel = ((out[b, seen, h].double() - o[seen]).norm() / o[seen].norm()).item()
                err = (lse[b, h, seen].double() - l[seen]).abs().max().item()
                assert rel <= 1e-2 and err <= 2e-3, (b, h, rel, err)


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
    _one_split_bytes(B, M, H, Hk, D, N)
    _check_rows(out, lse, q, k, v, lens, causal, range(0, H, 5))


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


# Row blocks sorted longest first: within one round of 256 CUs (33 x 4, 8 x 20
# blocks) and dealt over the XCDs beyond (65 x 5, 15 x 20, 1 x 264), 3, 5 and 33 query
# heads per KV head, blocks that span two query heads, fewer keys than rows.
@pytest.mark.parametrize("B,M,H,Hk,D,N", [(11, 300, 9, 3, 128, 333), (13, 400, 15, 5, 64, 401), (2, 1000, 20, 4, 64, 900),
                                         (3, 1000, 25, 5, 128, 1000), (1, 2048, 33, 1, 64, 2100)])
def test_sorted_row_blocks(gpu, B, M, H, Hk, D, N):
    print(f"[direct output] sorted B={B} M={M} H={H}/{Hk} D={D} N={N}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(M + H)
    q, k, v = (torch.randn(s, generator=g, device=gpu).to(torch.bfloat16) for s in ((B, M, H, D), (B, N, Hk, D), (B, N, Hk, D)))
    out, lse = flash_attn_with_kvcache(q, k, v, causal=True, return_softmax_lse=True)
    torch.cuda.synchronize()
    _one_split_bytes(B, M, H, Hk, D, N)
    _check_rows(out, lse, q, k, v, [N] * B, True, sorted({0, H // 2, H - 1}))


# (heads apart, elements before the first row): rows on 16-byte boundaries are
# written by the attention kernel, which leaves the workspace alone; others go
# through partials and the merge.
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("pad,off,direct", [(8, 0, True), (64, 8, True), (4, 0, False), (0, 1, False), (8, 4, False)])
def test_strided_and_unaligned_outputs(gpu, dtype, pad, off, direct):
    B, M, H, Hk, D, N = 16, 37, 32, 16, 64, 150
    print(f"[direct output] strided {dtype} pad={pad} off={off}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(pad + off)
    q, k, v = (torch.randn(s, generator=g, device=gpu).to(dtype) for s in ((B, M, H, D), (B, N, Hk, D), (B, N, Hk, D)))
    lib, nb = _ext.load(), _one_split_bytes(B, M, H, Hk, D, N)
    buf = torch.full((off + B * M * H * (D + pad),), 7.5, dtype=dtype, device=gpu)
    out = buf[off:].view(B, M, H, D + pad)[..., :D]
    lse = torch.empty((B, H, M), dtype=torch.float32, device=gpu)
    ws = torch.full((nb,), 0x5A, dtype=torch.uint8, device=gpu)
    rc = lib.dsv_flash_attn_with_kvcache(_ext.desc(q), _ext.desc(k), _ext.desc(v), _ext.desc(None), N, 1, _ext.desc(out),
                                         _ext.desc(lse), ws.data_ptr(), nb, _ext.stream_of(gpu))
    _ext.check(rc, "flash_attn_with_kvcache")
    torch.cuda.synchronize()
    assert bool((ws == 0x5A).all()) == direct, "which kernel wrote the output"
    _check_rows(out, lse, q, k, v, [N] * B, True, range(0, H, 7))
    rest = buf.clone()
    rest[off:].view(B, M, H, D + pad)[..., :D] = 7.5
    assert (rest == 7.5).all(), "elements between the rows"


@pytest.mark.parametrize("over", ["q", "k", "v"])
def test_output_over_an_input(gpu, over):
    B, M, H, D = 16, 300, 16, 128
    print(f"[direct output] out over {over}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(3)
    t = {n: torch.randn((B, M, H, D), generator=g, device=gpu).to(torch.bfloat16) for n in ("q", "k", "v")}
    want, want_lse = flash_attn_with_kvcache(t["q"], t["k"], t["v"], causal=True, return_softmax_lse=True)
    lib, nb = _ext.load(), _ext.load().dsv_attn_workspace_bytes(B, M, H, H, D, M, 0, 0)
    ws = torch.empty(nb, dtype=torch.uint8, device=gpu)
    lse = torch.empty_like(want_lse)
    rc = lib.dsv_flash_attn_with_kvcache(_ext.desc(t["q"]), _ext.desc(t["k"]), _ext.desc(t["v"]), _ext.desc(None), M, 1,
                                         _ext.desc(t[over]), _ext.desc(lse), ws.data_ptr(), nb, _ext.stream_of(gpu))
    _ext.check(rc, "flash_attn_with_kvcache")
    torch.cuda.synchronize()
    # (bf16 partials of one split, merged, round to the directly written row)
    assert torch.equal(t[over], want) and torch.equal(lse, want_lse)
