"""Attention rows whose score jumps inside a split, past the lagging row maximum.

The exponentials run against a maximum that may lag behind the true one, so a
probability can lie far above 1 before it is rounded to 16 bits; it must stay
in that type's range (f16: below 65520, 2^16 rounds to infinity).  Every call
is one split of five tiles.  The first tile's scores are 0, one key of the
third tile lies ``jump`` log2 units higher and the other keys of its tile 12
units lower, so that they add nothing to the tile's sum.  The reference is
float64; the bounds are those of the other attention tests.
"""

import math

import pytest
import torch

from diffspec_mi355x import _ext
from diffspec_mi355x.runtime.attention_compat import flash_attn_with_kvcache
from diffspec_mi355x.runtime.bundle_verifier import FusedBundleVerifier, PagedBundleVerifier
from diffspec_mi355x.runtime.tree_attention import tree_verify

pytestmark = pytest.mark.gpu

# Below the range of a probability, at its end (in f16 2^15.9998 rounds to
# infinity, and 2^16 is the next value that a sum of 2^16 would let through), above.
JUMPS = [8.5, 14.9, 15.2, 15.9, 15.9998, 16.1]
B, M, H, N = 16, 3, 16, 160  # B x H = 256 units: one split on 256 CUs or fewer


def _inputs(gpu, D, dtype, jump):
    ws = _ext.load().dsv_attn_workspace_bytes(B, M, H, H, D, N, 0, 0)
    assert ws == B * H * M * (D * 2 + 8), "the plan has more than one split"
    unit = math.sqrt(D) / math.log2(math.e)  # a score of one log2 unit
    q = torch.zeros((B, M, H, D), device=gpu)
    q[..., 0] = q[..., 1] = 1.0
    k = torch.zeros((B, N, H, D), device=gpu)
    k[:, 64:96, :, 0] = -12.0 * unit
    k[:, 96:, :, 0] = -3.0 * unit
    hi = math.floor(jump * unit * 16) / 16  # in two 16-bit parts
    k[:, 77, :, 0], k[:, 77, :, 1] = hi, jump * unit - hi
    v = torch.randn((B, N, H, D), generator=torch.Generator(device=gpu).manual_seed(7), device=gpu)
    v[:, 77, :, 5] = 0.0  # (infinity times 0 is not a number)
    return q.to(dtype), k.to(dtype), v.to(dtype)


def _reference(q, k, v):
    s = (q.permute(0, 2, 1, 3).double().contiguous() @ k.permute(0, 2, 3, 1).double().contiguous()) / q.shape[-1] ** 0.5
    out = torch.softmax(s, dim=-1) @ v.permute(0, 2, 1, 3).double().contiguous()
    return out.permute(0, 2, 1, 3), torch.logsumexp(s, dim=-1).permute(0, 2, 1)


def _check(out, lse, want, what):
    o, l = want
    assert torch.isfinite(out).all() and torch.isfinite(lse).all(), f"{what}: not finite"
    rel = ((out.double() - o).norm() / o.norm()).item()
    err = (lse.double() - l).abs().max().item()
    assert rel <= 1e-2 and err <= 2e-3, f"{what}: rel {rel:.2e} lse {err:.2e}"


def _paged(k, v, ps=16):
    """k, v [B, N, Hk, D] as a page pool [1, 2, B * n, Hk, ps, D] and its tables [B, n]."""
    n = k.shape[1] // ps
    pages = [x.reshape(B * n, ps, H, x.shape[-1]).transpose(1, 2) for x in (k, v)]
    return torch.stack(pages)[None].contiguous(), torch.arange(B * n, device=k.device).reshape(B, n)


@pytest.mark.parametrize("jump", JUMPS)
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_byte_mask_jump(gpu, dtype, D, jump):
    print(f"[score jump] byte mask {dtype} D={D} jump={jump}", flush=True)
    q, k, v = _inputs(gpu, D, dtype, jump)
    want = _reference(q, k, v)
    mask = torch.ones((M, N), dtype=torch.int8, device=gpu)  # every tile kept whole
    ver = PagedBundleVerifier(device="cuda")
    _check(*FusedBundleVerifier(device="cuda").verify_bundle(q, k, v, [mask]), want, "dense")
    pool, pt = _paged(k, v)
    _check(*ver.verify_bundle_paged(q, pool, pt, [mask]), want, "paged")


@pytest.mark.parametrize("jump", JUMPS)
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_unmasked_jump(gpu, dtype, D, jump):
    print(f"[score jump] tree, flash {dtype} D={D} jump={jump}", flush=True)
    q, k, v = _inputs(gpu, D, dtype, jump)
    out, lse = flash_attn_with_kvcache(q, k, v, return_softmax_lse=True)
    _check(out, lse.transpose(1, 2), _reference(q, k, v), "flash")
    # The same prefix with a chain of M nodes after it, dense and paged; node 0
    # sees the prefix and itself.
    kt, vt = (torch.cat([x, x[:, :M]], dim=1) for x in (k, v))
    parent = torch.arange(-1, M - 1, device=gpu)
    want = [torch.cat(x, dim=1) for x in zip(*(_reference(q[:, m:m + 1], kt[:, :N + m + 1], vt[:, :N + m + 1])
                                               for m in range(M)))]
    _check(*tree_verify(q, kt, vt, N, parent.expand(B, M).contiguous()), want, "tree dense")
    pad = (0, 0, 0, 0, 0, 16 - M)
    pool, pt = _paged(*(torch.nn.functional.pad(x, pad) for x in (kt, vt)))
    _check(*tree_verify(q, pool[0, 0], pool[0, 1], N, parent.expand(B, M).contiguous(), page_table=pt), want, "tree paged")
