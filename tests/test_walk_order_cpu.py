"""The order in which forward and dQ blocks visit their key tiles (KeyTiles and KeyWalk of attn_common.h, built for the
host): every tile that a row sees comes once, and in an order that does not depend on the rows its block holds besides."""
import ctypes
import importlib.util
import os
import subprocess

import numpy as np
import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ring-sliding-window-attention_amd")
spec = importlib.util.spec_from_file_location("rswa_build", os.path.join(PKG, "build.py"))
build = importlib.util.module_from_spec(spec)
spec.loader.exec_module(build)

SOURCE = """
#include "attn_common.h"
using namespace rswa;
// Tiles of the block of rows i0 .. i_last in their order, then three more places of the cursor.
extern "C" int walk(int wl, int wr, int n_sink, int shift, int len_q, int len_k, int i0, int i_last, int branch, int* out) {
  AttnArgs a{};
  a.wl = wl, a.wr = wr, a.n_sink = n_sink, a.shift_explicit = 1, a.shift_val = shift;
  a.by_walk = walk_period(a, 256, 64);
  const KeyTiles t = key_tiles<64>(a, i0, i_last, len_q, len_k);
  const int n = t.n_sink + t.n_band;
  KeyWalk w(a, t);
  for (int i = 0; i < n + 3; i++) {
    out[i] = w.tile;
    if (branch) w.next<true>();
    else w.next<false>();
  }
  return n;
}
"""


@pytest.fixture(scope="module")
def walk(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("walk")
    (tmp / "walk.hip").write_text(SOURCE)
    flags = ["--cuda-host-only", "-O1", "-std=c++17", "-fPIC", "-shared", "-nogpulib", "-I" + os.path.join(PKG, "csrc")]
    subprocess.run([build._hipcc(), *flags, str(tmp / "walk.hip"), "-o", str(tmp / "walk.so")], check=True,
                   capture_output=True)
    fn = ctypes.CDLL(str(tmp / "walk.so")).walk
    out = np.empty(1 << 16, dtype=np.int32)

    def call(*args):
        n = fn(*args, out.ctypes.data_as(ctypes.c_void_p))
        return out[:n].tolist(), out[n:n + 3].tolist()

    return call


def _rows_order(walk, wl, wr, n_sink, shift, len_q, len_k, block, first):
    """Per row of [0, len_q), the tiles that it sees as its block of `block` rows visits them; the blocks are those of
    the rows from `first` on, a view whose shift is as much larger."""
    orders = []
    for i0 in range(0, len_q - first, block):
        i_last = min(i0 + block, len_q - first) - 1
        args = (wl, wr, n_sink, shift + first, len_q - first, len_k, i0, i_last)
        tiles, beyond = walk(*args, 0)
        assert (tiles, beyond) == walk(*args, 1)
        assert len(set(tiles)) == len(tiles) and (not tiles or set(beyond) <= set(tiles))
        for i in range(i0, i_last + 1):
            at = i + first + shift
            hi = min(len_k - 1, at + wr) if wr >= 0 else len_k - 1
            lo = max(0, at - wl) if wl >= 0 else 0
            sees = set(range(lo // 64, hi // 64 + 1)) if hi >= lo else set()
            sees |= set(range((max(0, min(n_sink, hi + 1, lo)) + 63) // 64))
            assert sees <= set(tiles), (i, first)
            orders.append([t for t in tiles if t in sees])
    return orders


@pytest.mark.parametrize("wl,wr,n_sink", [
    (0, 0, 0), (63, 0, 0), (100, 0, 0), (350, 0, 0), (447, 0, 0), (500, 70, 0), (1000, 0, 0), (1950, 0, 0), (2000, 0, 4),
    (300, 0, 64), (300, 0, 65), (900, 10, 200), (190, 0, 1000), (-1, 0, 0), (500, -1, 0), (-1, 0, 100)])
def test_a_rows_tiles_have_one_order(walk, wl, wr, n_sink):
    for len_q, len_k, shift in ((2600, 2600, 0), (1100, 2900, 1800), (1300, 700, 0), (900, 2000, -200)):
        want = _rows_order(walk, wl, wr, n_sink, shift, len_q, len_k, 64, 0)
        for block, first in ((128, 0), (256, 0), (64, 40), (128, 1), (256, 200)):
            got = _rows_order(walk, wl, wr, n_sink, shift, len_q, len_k, block, first)
            assert got == want[first:], (len_q, len_k, shift, block, first)
