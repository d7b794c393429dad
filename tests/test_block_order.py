"""Order of the causal row blocks of one-split attention, on the CPU.

The kernel's own index functions (dsv_attn_geo.h), compiled for the host:
every (head, row block) is met once, each head's longest blocks come first,
and the XCDs (dispatch ids round-robin) get equal shares of the keys.
"""

import ctypes
import subprocess

import pytest

from diffspec_mi355x import _build

SRC = """
#include "dsv_attn_geo.h"
extern "C" void order(int dealt, int heads, int n_rb, int G, int* head, int* rb) {
  for (int p = 0; p < heads * n_rb; ++p) {
    int i;
    if (dealt) {
      dsv::deal_block(p, heads, n_rb, head[p], i);
    } else {
      head[p] = p / n_rb;
      i = p % n_rb;
    }
    rb[p] = dsv::long_first_rb(i, n_rb, G);
  }
}
"""


@pytest.fixture(scope="module")
def order(tmp_path_factory):
    d = tmp_path_factory.mktemp("order")
    (d / "order.hip").write_text(SRC)
    subprocess.run([_build._hipcc(), "--offload-host-only", "-O1", "-std=c++17", "-shared", "-fPIC", f"-I{_build.CSRC_DIR}",
                    f"-I{_build.INCLUDE_DIR}", str(d / "order.hip"), "-o", str(d / "order.so")], check=True,
                   capture_output=True)
    lib = ctypes.CDLL(str(d / "order.so"))

    def call(dealt, heads, n_rb, G):
        h, r = (ctypes.c_int * (heads * n_rb))(), (ctypes.c_int * (heads * n_rb))()
        lib.order(dealt, heads, n_rb, G, h, r)
        return list(h), list(r)

    return call


@pytest.mark.parametrize("dealt", [0, 1])
@pytest.mark.parametrize("heads", [1, 2, 3, 7, 8, 9, 12, 16, 28, 33])
@pytest.mark.parametrize("G,n_rb", [(1, 2), (1, 64), (3, 4), (4, 5), (4, 64), (7, 43), (32, 33), (32, 512)])
def test_every_block_once(order, dealt, heads, G, n_rb):
    h, r = order(dealt, heads, n_rb, G)
    assert sorted(zip(h, r)) == [(a, b) for a in range(heads) for b in range(n_rb)]


# (B x KV heads, query heads per KV head, rows = keys)
@pytest.mark.parametrize("heads,G,M", [(1, 32, 4096), (2, 4, 16384), (4, 4, 8192), (3, 4, 4096), (6, 4, 4096), (8, 4, 4096),
                                       (12, 2, 4096), (4, 7, 4096)])
def test_xcds_share_the_keys(order, heads, G, M):
    n_rb = -(-G * M // 256)
    h, r = order(1, heads, n_rb, G)
    keys = [min((b * 256 + 255) % M, M - 1) + 1 for b in range(n_rb)]  # (256 divides M: no block spans two query heads)
    for x in range(8):
        own = list(zip(h[x::8], r[x::8]))
        share = sum(keys[b] for _, b in own) * 8 / (heads * sum(keys))
        assert 0.9 <= share <= 1.1, f"XCD {x}: {share:.2f} of the mean"
        for head in range(heads):  # longest first
            seen = [keys[b] for a, b in own if a == head]
            assert seen == sorted(seen, reverse=True)
