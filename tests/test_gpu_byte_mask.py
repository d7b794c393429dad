"""Byte-masked attention: the keep-bit window of the split-K kernel.

The kernel packs each query row's mask bytes into one word per 32-key tile,
a window of tiles at a time.  The sizes are the edges of that packing: masks
that end inside a tile, rows at odd byte offsets, strided masks, a window
that is refilled, several row blocks, and masks shorter than the keys.
The reference is float64 masked attention; the bounds are those of the other
attention tests (16-bit probabilities and split results: relative 1e-2).
"""

import pytest
import torch

from diffspec_mi355x import _ext
from diffspec_mi355x.runtime.bundle_verifier import FusedBundleVerifier, PagedBundleVerifier

pytestmark = pytest.mark.gpu


def _reference(q, k, v, keep):
    """q [B, M, H, D], k / v [B, N, Hk, D], keep [Bm, M, N] bool -> out, lse in float64."""
    B, M, H, D = q.shape
    G = H // k.shape[2]
    out = torch.zeros((B, M, H, D), dtype=torch.float64, device=q.device)
    lse = torch.zeros((B, M, H), dtype=torch.float64, device=q.device)
    for b in range(B):
        kp = keep[b if keep.shape[0] > 1 else 0]
        for h in range(H):
            kk = k[b, :, h // G].double().contiguous()
            s = (q[b, :, h].double() @ kk.t().contiguous()) / D ** 0.5
            s = s.masked_fill(~kp, float("-inf"))
            lse[b, :, h] = torch.logsumexp(s, dim=1)
            p = torch.exp(s - torch.where(torch.isinf(lse[b, :, h]), 0.0, lse[b, :, h])[:, None])
            out[b, :, h] = p @ v[b, :, h // G].double().contiguous()
    return out, lse


def _check(got, want, what):
    o, l = got
    o_ref, l_ref = want
    rel = ((o.double() - o_ref).norm() / o_ref.norm().clamp_min(1e-30)).item()
    inf = torch.isinf(l_ref)
    assert torch.equal(torch.isinf(l), inf), f"{what}: -inf pattern"
    err = (l.double() - l_ref)[~inf].abs().max().item() if (~inf).any() else 0.0
    assert rel <= 1e-2 and err <= 2e-3, f"{what}: rel {rel:.2e} lse {err:.2e}"
    assert (o[inf] == 0).all(), f"{what}: rows that keep nothing are zero"


def _mask(shape, seed, dev, kind):
    g = torch.Generator().manual_seed(seed)
    m = torch.ones(shape, dtype=torch.uint8)
    if kind == "random":
        m = (torch.rand(shape, generator=g) < 0.5).to(torch.uint8) * 255
    else:  # whole tiles kept and dropped, a ragged end
        m[..., shape[-1] // 2:] = (torch.rand(shape[:-1] + (shape[-1] - shape[-1] // 2,), generator=g) < 0.3).to(torch.uint8) * 2
        m[..., 0, :] = 0
    return m.to(dev)


@pytest.mark.parametrize("B,M,H,Hk,D,N", [(1, 1, 4, 4, 64, 31), (1, 5, 8, 2, 128, 33), (2, 33, 8, 8, 128, 95),
                                         (1, 64, 8, 2, 128, 1007), (1, 300, 4, 4, 64, 129), (2, 70, 16, 2, 64, 640),
                                         (16, 64, 64, 16, 64, 2597)])  # the last one refills the window
@pytest.mark.parametrize("kind", ["random", "prefix"])
def test_byte_mask_sizes(gpu, B, M, H, Hk, D, N, kind):
    print(f"[byte mask] B={B} M={M} H={H}/{Hk} D={D} N={N} {kind}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(N)
    q, k, v = (torch.randn(s, generator=g, device=gpu).to(torch.float16) for s in
               ((B, M, H, D), (B, N, Hk, D), (B, N, Hk, D)))
    mask = _mask((1, M, N), N + M, gpu, kind)
    if N == 2597:  # one split of 82 tiles, windows of 76 (20480 words for 256 rows)
        ws = _ext.load().dsv_attn_workspace_bytes(B, M, H, Hk, D, N, 0, 0)
        assert ws == B * H * M * (D * 2 + 8), "the plan has more than one split: the window is not refilled"
    got = FusedBundleVerifier(device="cuda").verify_bundle(q, k, v, [mask])
    _check(got, _reference(q, k, v, mask != 0), f"N={N} {kind}")


@pytest.mark.parametrize("form", ["odd offset", "strided keys", "per batch", "short", "bool"])
def test_byte_mask_forms(gpu, form):
    B, M, H, Hk, D, N, ps = 2, 24, 8, 4, 128, 500, 16
    print(f"[byte mask] {form}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(9)
    q = torch.randn((B, M, H, D), generator=g, device=gpu).to(torch.bfloat16)
    npg = -(-N // ps)
    pool = torch.randn((1, 2, B * npg, Hk, ps, D), generator=g, device=gpu).to(torch.bfloat16)
    pt = torch.randperm(B * npg, generator=torch.Generator().manual_seed(5)).reshape(B, npg).to(gpu)
    tok = torch.arange(N, device=gpu)
    k, v = (torch.stack([pool[0, x][pt[b][tok // ps], :, tok % ps] for b in range(B)]) for x in (0, 1))
    nm = N - 45 if form == "short" else N
    if form == "odd offset":
        mask = _mask((1, M, N + 3), 1, gpu, "prefix")[:, :, 3:]
    elif form == "strided keys":
        mask = _mask((1, M, 2 * N), 2, gpu, "random")[:, :, ::2]
    elif form == "per batch":
        mask = _mask((B, M, N), 3, gpu, "random")
    else:
        mask = _mask((1, M, nm), 4, gpu, "random")
    if form == "bool":
        mask = mask != 0
    keep = torch.zeros((mask.shape[0], M, N), dtype=torch.bool, device=gpu)
    keep[:, :, :nm] = mask != 0  # keys past a short mask are dropped
    ver = PagedBundleVerifier(device="cuda")
    dense = ver.verify_bundle(q, k, v, [mask])
    _check(dense, _reference(q, k, v, keep), form)
    if form != "short":  # the paged call's keys are the mask's
        paged = ver.verify_bundle_paged(q, pool, pt, [mask])
        assert torch.equal(paged[0], dense[0]) and torch.equal(paged[1], dense[1])
