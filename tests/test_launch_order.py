"""The launch order of the attention kernels: what decode_block gives with the operands block_order prepares, against plain divisions."""
import ctypes as C
import pathlib
import shutil
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]

PROGRAM = r"""
#include "fox_kernels.hpp"
#include <cstdio>
using namespace fox;
int main() {
  const int dividends[] = {0, 1, 2, 127, 128, 65535, 1 << 24, (1 << 25) - 1, 1 << 30, 2147483646, 2147483647};
  for (int d : {1, 2, 3, 5, 7, 12, 60, 127, 128, 129, 641, 65535, 65537, (1 << 25) - 1, 1 << 30, (1 << 30) + 1, 2147483647})
    for (int n : dividends)
      for (int near = -1; near <= 1; ++near) {   // also on either side of a multiple of d
        const int64_t x = near ? (int64_t)(n / d) * d + near : n;
        if (x >= 0 && x <= 2147483647 && divide((int)x, divisor(d)) != (int)x / d) return std::printf("%lld / %d\n", (long long)x, d), 1;
      }
  // pairs that 8 divides or not, one group, several of one or two sizes, one pair a group, resident grids or not
  const int shapes[][4] = {{1, 12, 1, 1}, {1, 12, 4, 1}, {3, 5, 7, 1}, {4, 16, 128, 4}, {4, 15, 64, 60}, {5, 16, 33, 3}, {7, 9, 10, 5}, {1, 1, 4096, 1}, {2, 16, 16, 2}, {8, 64, 3, 64}, {4, 12, 8, 1}};
  for (auto& s : shapes)
    for (int v = 0; v < 4; ++v) {
      const int B = s[0], H = s[1], tiles = s[2], groups = s[3], n_bh = B * H;
      const bool fold = v & 1, last_first = v & 2, by_xcd = n_bh % 8 == 0;
      const int nb = by_xcd ? n_bh / 8 : n_bh, cus = by_xcd ? 32 : 256, total = nb * tiles;
      const BlockOrder o = block_order(B, H, tiles, groups, fold);
      for (int xcd = 0; xcd < (by_xcd ? 8 : 1); ++xcd) {
        int place = 0;
        for (int first = 0, g = 0; g < groups; ++g) {   // the order in words: group by group, heaviest tile first, the pairs of the group in turn
          const int size = nb / groups + (g < nb % groups);
          for (int tile = tiles - 1; tile >= 0; --tile)
            for (int pair = first; pair < first + size; ++pair, ++place) {
              const int r = fold && total <= 2 * cus && place >= cus ? total - 1 - (place - cus) : place;   // (folding is its own inverse)
              int bh, t;
              decode_block(by_xcd ? r * 8 + xcd : r, o, last_first, bh, t);
              const int want = last_first ? nb - 1 - pair : pair;
              if (t != tile || bh != (by_xcd ? want * 8 + xcd : want) || divide(bh, o.by_heads) != bh / H)
                return std::printf("B%d H%d tiles %d groups %d variant %d place %d\n", B, H, tiles, groups, v, r), 1;
            }
          first += size;
        }
        if (place != total) return 1;
      }
    }
  // one-launch backward: as many workgroups as there are tiles, each tile once, the heaviest of either kind first
  for (int keys = 1; keys < 20; ++keys)
    for (int queries = 1; queries <= keys; ++queries) {
      int next_query = queries - 1, next_key = 0;
      for (int t = keys + queries - 1; t >= 0; --t) {
        const BothTile w = both_tile(t, keys, queries);
        if (w.tile != (w.query ? next_query-- : next_key++)) return std::printf("%d key tiles, %d query tiles, place %d\n", keys, queries, t), 1;
      }
      if (next_query != -1 || next_key != keys) return 1;
    }
}
"""


def test_launch_order_without_divisions(tmp_path):
    hipcc = shutil.which("hipcc") or shutil.which("/opt/rocm/bin/hipcc")
    if hipcc is None:
        pytest.skip("no hipcc")
    src, exe = tmp_path / "order.hip", tmp_path / "order"
    src.write_text(PROGRAM)
    csrc = ROOT / "forgetting-transformer_amd" / "csrc"
    subprocess.run([hipcc, "-std=c++17", "-O1", "--offload-arch=gfx950", "-Wno-unused-command-line-argument", f"-I{csrc}", str(src), "-o", str(exe)], check=True)
    done = subprocess.run([str(exe)], capture_output=True, text=True)
    assert done.returncode == 0, done.stdout


@pytest.mark.parametrize("B,H,M,N,D,pruned,yes", [
    (4, 12, 512, 512, 64, False, 1), (2, 32, 1000, 1000, 64, True, 1), (2, 16, 2048, 2048, 64, True, 1), (16, 16, 257, 257, 64, False, 0), (1, 1, 100, 100, 128, False, 0),
    (3, 32, 1000, 1000, 32, True, 1), (1, 6, 16384, 16384, 16, False, 1), (49, 16, 100, 100, 32, False, 0), (48, 16, 100, 100, 32, True, 1),
    # long rows: room on the chip, more of it under a threshold
    (1, 10, 4096, 4096, 64, True, 1), (1, 11, 4096, 4096, 64, True, 0), (1, 15, 4096, 4096, 64, False, 1), (1, 16, 4096, 4096, 64, False, 0),
    (1, 2, 16384, 16384, 32, True, 1), (1, 4, 16384, 16384, 32, True, 0), (1, 12, 8192, 8192, 32, True, 1),
    (1, 16, 300, 4096, 64, True, 1), (1, 16, 2048, 4096, 64, True, 0), (1, 16, 2048, 4096, 64, False, 1)])
def test_grids_of_the_one_launch_backward(B, H, M, N, D, pruned, yes):
    from forgetting_transformer.ops import _lib
    x = 1 << 20   # (never read: host arithmetic only)
    got = C.c_int32(-1)
    view = _lib.View(x, H * N * D, N * D, D)
    args = _lib.BwdArgs(_lib.Dims(B, H, M, N, D, 0), *[view] * 8, x, x, None, x if pruned else None, 0.1, x, x + 64, x, x, 0, 0, 0, None, None)
    _lib.check(_lib.load().fox_attn_bwd_one_launch(C.byref(args), C.byref(got)), "fox_attn_bwd_one_launch")
    assert got.value == yes


@pytest.mark.parametrize("B,H,M,N,D,pruned,yes", [
    (1, 1, 2, 3584, 64, False, 0), (2, 16, 2048, 2048, 128, False, 1), (2, 16, 2048, 2048, 64, False, 0), (2, 16, 2048, 2048, 64, True, 1), (2, 9, 3583, 3583, 16, False, 1),
    (4, 32, 500, 500, 32, False, 1), (8, 32, 400, 1000, 64, True, 0),
    # several query tiles behind many keys repeat the row, one does not
    (8, 32, 130, 1200, 64, True, 1), (8, 32, 130, 1600, 64, True, 0), (8, 32, 130, 1600, 128, False, 0), (16, 32, 128, 3500, 64, True, 1), (8, 32, 130, 1500, 64, True, 1),
    # more than two workgroups per CU
    (4, 28, 1000, 1000, 64, False, 1), (4, 32, 1000, 1000, 64, False, 0), (4, 32, 1000, 1000, 64, True, 1), (16, 32, 256, 256, 128, False, 1), (8, 24, 500, 500, 128, False, 0),
    (3, 16, 1536, 1536, 64, True, 0), (32, 33, 128, 128, 64, True, 0)])
def test_grids_that_form_their_own_sums(B, H, M, N, D, pruned, yes):
    from forgetting_transformer.ops import _lib
    got = C.c_int32(-1)
    _lib.check(_lib.load().fox_attn_fwd_takes_gates(C.byref(_lib.Dims(B, H, M, N, D, 0)), pruned, C.byref(got)), "fox_attn_fwd_takes_gates")
    assert got.value == yes


@pytest.mark.parametrize("B,H,N,D,counters", [(1, 12, 1500, 64, 12), (1, 64, 1000, 64, 64), (1, 64, 1200, 64, 0), (1, 4, 8192, 128, 4), (1, 5, 8192, 128, 0), (1, 5, 700, 32, 0),
                                              (1, 128, 600, 64, 0), (1, 128, 1500, 16, 128), (1, 129, 1500, 16, 0), (16, 16, 32768, 128, 0),
                                              # several batches of keys a wave: up to two, and with half a chip of workgroups
                                              (1, 4, 8193, 128, 0), (1, 2, 8193, 128, 2), (1, 2, 16384, 128, 2), (1, 1, 16385, 128, 0), (1, 2, 32768, 64, 2), (1, 3, 32768, 64, 0)])
def test_counters_of_a_generation_step(B, H, N, D, counters):
    from forgetting_transformer.ops import _lib
    got = C.c_int32(-1)
    _lib.check(_lib.load().fox_attn_decode_counters(C.byref(_lib.Dims(B, H, 1, N, D, 0)), C.byref(got)), "fox_attn_decode_counters")
    assert got.value == counters <= 128
    assert _lib.load().fox_attn_decode_counters(C.byref(_lib.Dims(B, H, 2, N, D, 0)), C.byref(got)) == -1


@pytest.mark.parametrize("B,H,M,N,D,yes", [(1, 17, 4096, 4096, 128, 0), (1, 18, 4096, 4096, 128, 1), (8, 22, 700, 700, 32, 0), (8, 23, 700, 700, 32, 1),
                                           (4, 64, 128, 32768, 16, 1), (1, 64, 128, 32768, 16, 0)])
def test_thresholds_with_the_scan_beside_the_norms(B, H, M, N, D, yes):
    from forgetting_transformer.ops import _lib
    got = C.c_int32(-1)
    _lib.check(_lib.load().fox_auto_threshold_scan_one_launch(C.byref(_lib.Dims(B, H, M, N, D, 0)), C.byref(got)), "fox_auto_threshold_scan_one_launch")
    assert got.value == yes
