"""Dry run (CPU) of one-split attention and of the byte mask's LDS window.

The emulation walks what the kernel does there with the kernel's own index
functions: the order of the row blocks (each once), every block's last key of
a causal call, and the keep-bit words of every row block.
"""

import ctypes

import pytest

from diffspec_mi355x import _ext
from test_dry_run import Alloc, dry, none, ok, paged_case, tensor, view  # noqa: F401  (dry: the fixture)


def _flash(lib, B, M, H, Hk, D, N, causal, dt=_ext.DSV_BF16, out=None):
    a = Alloc()
    q, k, v = tensor(a, (B, M, H, D), dt), tensor(a, (B, N, Hk, D), dt), tensor(a, (B, N, Hk, D), dt)
    o = out(a) if out else tensor(a, (B, M, H, D), dt)
    lse = tensor(a, (B, H, M), _ext.DSV_F32)
    ws = lib.dsv_attn_workspace_bytes(B, M, H, Hk, D, N, 0, 0)
    rc = lib.dsv_flash_attn_with_kvcache(ctypes.byref(q), ctypes.byref(k), ctypes.byref(v), ctypes.byref(none()), N,
                                         int(causal), ctypes.byref(o), ctypes.byref(lse), a.take(ws), ws, None)
    return rc, ws


# Row blocks per KV head below, at and above the query heads of one (the sorted
# order), one round of 256 CUs and more (dealt), rows that end inside a block,
# blocks that span two query heads, more rows than keys.
SHAPES = [(16, 128, 32, 16, 64, 130), (11, 300, 9, 3, 128, 333), (13, 400, 15, 5, 64, 401), (2, 1000, 20, 4, 64, 1100),
          (3, 1000, 25, 5, 128, 1000), (1, 1029, 33, 1, 64, 1040), (2, 700, 28, 4, 64, 600), (1, 2048, 17, 17, 64, 2048),
          (1, 2048, 33, 33, 64, 2100), (1, 4096, 32, 1, 64, 4100)]


@pytest.mark.parametrize("B,M,H,Hk,D,N", SHAPES)
@pytest.mark.parametrize("causal", [False, True])
def test_one_split(dry, B, M, H, Hk, D, N, causal):
    rc, ws = _flash(dry, B, M, H, Hk, D, N, causal)
    ok(dry, rc, "flash")
    rows = B * H * M
    align = lambda x: -(-x // 256) * 256  # noqa: E731
    assert ws == align(rows * D * 2) + align(rows * 8), "the plan has more than one split"


@pytest.mark.parametrize("dt", [_ext.DSV_BF16, _ext.DSV_F16])
@pytest.mark.parametrize("pad,off", [(0, 0), (8, 0), (4, 0), (0, 1), (8, 3)])  # direct where both are multiples of 8
def test_one_split_strided_and_unaligned_output(dry, dt, pad, off):
    B, M, H, Hk, D, N = 16, 40, 32, 16, 64, 64

    def out(a):
        base = tensor(a, (B * M * H * (D + pad) + off,), dt)
        return view(base, off, (B, M, H, D), (M * H * (D + pad), H * (D + pad), D + pad, 1))

    rc, _ = _flash(dry, B, M, H, Hk, D, N, True, dt, out)
    ok(dry, rc, "flash")


def test_outputs_over_inputs_take_the_merge(dry):
    """The attention kernel's blocks read q, k and v until the last one ends: an output
    that overlaps them is written by the merge, as one of unaligned rows is (the number
    of checked accesses tells the two apart)."""
    B, M, H, D = 16, 40, 16, 64
    lib = dry

    def checks(out_of, lse_of, off=0):
        a = Alloc()
        t = {n: tensor(a, (B, M, H, D)) for n in ("q", "k", "v", "out")}
        lse = tensor(a, (B, H, M), _ext.DSV_F32)
        if lse_of:
            lse.data = t[lse_of].data
        t[out_of].data += off
        ws = lib.dsv_attn_workspace_bytes(B, M, H, H, D, M, 0, 0)
        rc = lib.dsv_flash_attn_with_kvcache(ctypes.byref(t["q"]), ctypes.byref(t["k"]), ctypes.byref(t["v"]), ctypes.byref(none()),
                                             M, 1, ctypes.byref(t[out_of]), ctypes.byref(lse), a.take(ws), ws, None)
        ok(lib, rc, f"out over {out_of}, lse over {lse_of}")
        return lib.dsv_dry_run_checks()

    direct, merged = checks("out", None), checks("out", None, 2)
    assert direct != merged
    for out_of, lse_of in (("q", None), ("k", None), ("v", None), ("out", "q"), ("out", "v")):
        assert checks(out_of, lse_of) == merged, (out_of, lse_of)


# Row blocks of 1 to 8 waves, several blocks, more tiles than a window holds.
@pytest.mark.parametrize("B,M,H,Hk,D,N", [(1, 1, 1, 1, 64, 31), (1, 40, 4, 4, 128, 700), (1, 65, 2, 1, 64, 333), (2, 100, 4, 2, 64, 999),
                                         (1, 150, 1, 1, 128, 400), (1, 180, 1, 1, 64, 100), (1, 200, 1, 1, 64, 129),
                                         (1, 256, 1, 1, 64, 64), (1, 300, 2, 1, 64, 200), (16, 64, 64, 16, 64, 2597)])
def test_byte_mask_window(dry, B, M, H, Hk, D, N):
    a = Alloc()
    q, k, v = tensor(a, (B, M, H, D)), tensor(a, (B, N, Hk, D)), tensor(a, (B, N, Hk, D))
    mask = tensor(a, (1, M, N), _ext.DSV_I8)
    out, lse = tensor(a, (B, M, H, D)), tensor(a, (B, M, H), _ext.DSV_F32)
    ws = dry.dsv_attn_workspace_bytes(B, M, H, Hk, D, N, 0, 0)
    rc = dry.dsv_verify_bundle(ctypes.byref(q), ctypes.byref(k), ctypes.byref(v), ctypes.byref(mask), ctypes.byref(out),
                               ctypes.byref(lse), a.take(ws), ws, None)
    ok(dry, rc, "verify_bundle")
    pool, pt, _ = paged_case(a, N, Hk=Hk, D=D, ps=16, layers=1, spare=1)
    ws = dry.dsv_attn_workspace_bytes(B, M, H, Hk, D, N, 16, 0)
    rc = dry.dsv_verify_bundle_paged(ctypes.byref(q), ctypes.byref(pool), ctypes.byref(pt), 0, ctypes.byref(mask),
                                     ctypes.byref(out), ctypes.byref(lse), a.take(ws), ws, None)
    ok(dry, rc, "verify_bundle_paged")
