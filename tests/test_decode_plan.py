"""The key splits of a generation step, on the host: the scratch that the query asks for holds what any call launches, and a call with less
scratch than that launches no more than fits; counters are touched where the query asks for them."""
import pathlib
import shutil
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]

PROGRAM = r"""
#include "fox_decode_plan.hpp"
#include <algorithm>
#include <cstdio>
using namespace fox;
int main() {
  int more[2] = {0, 0};   // shapes where the call without padding, and the one with it, has the more splits
  for (int bh = 1; bh <= 2100; bh += bh < 1100 ? 1 : 4)
    for (int D : {16, 32, 64, 128})
      for (int64_t batch = 1; batch <= 512; batch += batch < 140 ? 1 : 5)
        for (int past = 0; past <= 1; ++past) {
          const int N = (int)(batch * 16384 / D) + past;
          if ((int64_t)bh * ((N + 63) / 64) * 64 > 0x7fffffffLL) continue;
          const int64_t room = decode_workspace_bytes(1, bh, N, D);
          int splits[2];
          for (int padded = 0; padded <= 1; ++padded) {
            const DecodePlan p = decode_plan(1, bh, N, D, padded);
            const int64_t need = decode_bytes(1, bh, D, p.least);
            // the number before it was made even: at most 2048 workgroups, which is what a caller's scratch always had to hold at most
            const int64_t even = std::min(std::min((2048 + bh - 1) / (int64_t)bh, decode_batches(N, D)), (int64_t)kDecodeMaxSplits);
            const bool whole = decode_batches(N, D) <= 1 || decode_one_workgroup(bh, decode_batches(N, D), D);
            if (p.splits < 1 || p.splits > kDecodeMaxSplits || p.least < 1 || p.least > (whole ? 1 : even) || (even == 1 && p.splits > 1) || need > room || (whole && room))
              return std::printf("%d pairs N%d D%d padded %d: %d splits, %d at least, room %lld\n", bh, N, D, padded, p.splits, p.least, (long long)room), 1;
            splits[padded] = p.splits;
            // padded rows give up splits only where four are left and every CU has as many pairs as the others
            if (padded && p.splits < even && (bh % kCus || p.splits < 4) && !whole) return std::printf("%d pairs N%d D%d: %d splits of %lld\n", bh, N, D, p.splits, (long long)even), 1;
            for (const int64_t bytes : {room, need, room - 1, (need + room) / 2, decode_bytes(1, bh, D, (int)even)}) {
              if (bytes < need) continue;   // refused
              const int n = decode_splits(1, bh, N, D, padded, bytes);
              if (decode_bytes(1, bh, D, n) > bytes || (bytes >= room && n != p.splits) || (n != p.splits && n != p.least))
                return std::printf("%d pairs N%d D%d padded %d: %d splits in %lld bytes\n", bh, N, D, padded, n, (long long)bytes), 1;
              if (decode_merges(1, bh, N, D, n) && (decode_counters(1, bh, N, D) != bh || bh > 128))
                return std::printf("%d pairs N%d D%d padded %d: %d splits merge, %d counters\n", bh, N, D, padded, n, decode_counters(1, bh, N, D)), 1;
            }
          }
          more[0] += splits[0] > splits[1];
          more[1] += splits[1] > splits[0];
        }
  return !more[0] || !more[1];   // the query has to look at both
}
"""


def test_scratch_of_a_generation_step_holds_its_splits(tmp_path):
    hipcc = shutil.which("hipcc") or shutil.which("/opt/rocm/bin/hipcc")
    if hipcc is None:
        pytest.skip("no hipcc")
    src, exe = tmp_path / "plan.hip", tmp_path / "plan"
    src.write_text(PROGRAM)
    csrc = ROOT / "forgetting-transformer_amd" / "csrc"
    subprocess.run([hipcc, "-std=c++17", "-O1", "--offload-arch=gfx950", "-Wno-unused-command-line-argument", f"-I{csrc}", str(src), "-o", str(exe)], check=True)
    done = subprocess.run([str(exe)], capture_output=True, text=True)
    assert done.returncode == 0, done.stdout
