// How a generation step (launch_decode_gates) is cut up: host arithmetic only, for the launch, for the queries of its scratch and for the
// check of what a caller brings.
#pragma once

#include "fox_kernels.hpp"

namespace fox {

inline int64_t decode_batches(int N, int D) { return ((int64_t)N * D + 16383) / 16384; }   // batches of keys, four waves each

// Whether one workgroup of sixteen waves takes a (batch, head) whole, which saves the merge of splits and its launch.  The line
// lies where a CU's share of the bandwidth costs more than the merge: D 64, splits of four waves and merge against one
// workgroup, us: B1 H12 N300 (2 batches) 7.9 / 6.8, N1500 (6 batches) 8.2 / 12.0.  With half a workgroup per CU or more the
// splits share those CUs anyway: B8 H16 N700 (3) 10.7 / 9.5, B16 H16 N700 13.6 / 11.7, B8 H16 N2048 (8) 17.0 / 17.5.
// Head dim 16 needs one register more than sixteen waves leave a lane.
inline bool decode_one_workgroup(int64_t bh, int64_t batches, int D) {
  return D >= 32 && bh < 2 * kCus && batches > 1 && batches <= (bh >= kCus / 2 ? 4 : 2);
}

// Key splits of launch_decode_gates: about eight workgroups per CU, a wave's run being a whole number `per` of batches of keys, and as many splits as the runs of a row without
// padding need.  (More than that are not just idle: consecutive workgroups go round the XCDs, so with twelve of sixteen splits in use four of the eight XCDs got two
// thirds of the rows.)  us, 2048 workgroups whatever the row / now:
// - A run of a few batches: the number with which the CUs get the most even share of them, one batch a wave where that is no worse, so that no wave waits for its second.
//   D 128, 128 pairs N3000 41.6 / 35.0 (twelve splits of two batches 36.1), 64 pairs N5000 32.6 / 29.7, D 64, 128 pairs N5000 33.2 / 29.0.  Not from one split, which needs no merge
//   (2048 pairs N1700 D16, padded by up to a quarter, one split 35.4, two 44.1).
// - One split, and no merge, where every CU, or three of four, has one pair, or all have nearly the same number: one workgroup a CU asks for as much as the memory gives.
//   D 128, 192 pairs N1700 31.3 / 28.9, N32768 491 / 448, 256 pairs N1700 42.9 / 35.6, N15000 298 / 286, D 64, 512 pairs N500 13.7 / 10.5, N15000 301 / 289.  128 pairs
//   N24000 (243 / 295) and 320 (582 / 688) lose, and so do 192 pairs of head dims below 64 (D 16 N15000 36.5 / 41.1); those gain
//   from nine tenths of the CUs on: D 32, 231 pairs N5000 30.6 / 27.2, N32768 163 / 150, 256 pairs N5000 43.7 / 29.2, 512 pairs N32768 348 / 328, D 16, 231 pairs N1700 11.8 / 9.2, N32768 86.5 / 81.9,
//   256 pairs N12000 46.8 / 36.6, 768 pairs N28000 222 / 219, N50000 384 / 380; only rows of N32768, each a power of two away from the next, lose there (256 pairs 92.4 / 93.3, 768 pairs 255 / 267).  Not with padding, which differs from row to row: the longest row would be left to one CU.
// - With padding the rows' own lengths decide what a split gets, and the number is not made even (D 128, 128 pairs N15000, padded by up to all of it, 16 / 15 splits 90.8 / 95.0).
// - With padding, long rows, the same number of pairs on every CU and four splits left of eight: half as many workgroups; they start and end less often, and are still few batches of
//   the whole (D 128, 256 pairs N32768, padded by up to a quarter 577 / 567, by up to all of it 398 / 372; shorter rows lose the balance: N5000 54.9 / 56.7, 512 pairs N5000 99 / 104).
//   Not where the CUs' shares become less even (N32768 D 64, 320 pairs, seven splits / four, 349 / 361, D 128 padded by up to all of it 323 / 353, 1040 pairs N20000, two / one, 1324 / 1379 and 783 / 889),
//   nor with fewer than four pieces of a row (512 pairs N20000 D 128 padded by up to all of it, four / two, 412 / 462; N32768 513 / 482).
struct DecodePlan {
  int splits;   // what a call takes
  int least;    // what its scratch must have room for: before the number is made even, which may take more
};
inline DecodePlan decode_plan(int B, int H, int N, int D, bool padded) {
  const int64_t bh = (int64_t)B * H, batches = decode_batches(N, D), rounds = (bh + kCus - 1) / kCus;
  if (batches <= 1 || decode_one_workgroup(bh, batches, D)) return {1, 1};
  const int64_t most = batches < kDecodeMaxSplits ? batches : kDecodeMaxSplits;
  auto of = [&](int64_t wgs) { const int64_t even = (wgs + bh - 1) / bh; return even < most ? even : most; };
  const int64_t fewer = of(bh >= kCus && batches >= 128 ? 4 * kCus : 8 * kCus), splits = padded && bh % kCus == 0 && fewer >= 4 ? fewer : of(8 * kCus);
  if (!padded && (bh <= kCus && D >= 64 ? 4 * bh >= 3 * kCus : 10 * bh >= 9 * rounds * kCus)) return {1, (int)fewer};
  int64_t per = (batches + splits - 1) / splits;
  auto runs = [&](int64_t p) { return (batches + p - 1) / p; };
  auto heaviest = [&](int64_t p) { return p * ((bh * runs(p) + kCus - 1) / kCus); };   // CU's share, in batches a wave
  if (splits > 1 && per <= 4)
    for (int64_t p = per - 1; p >= 1 && runs(p) <= most && bh * runs(p) <= 16 * kCus; --p)
      if (heaviest(p) < heaviest(per) || (p == 1 && heaviest(p) == heaviest(per))) per = p;
  return {(int)(padded && per > 1 ? splits : runs(per)), (int)fewer};
}

// Scratch of a call with that many splits: partial accumulators, then a DecodePartial each.
inline int64_t decode_bytes(int B, int H, int D, int splits) {
  return splits <= 1 ? 0 : (int64_t)splits * B * H * (int64_t)(D * sizeof(float) + sizeof(DecodePartial));
}
// Scratch for the shape, left padding or none: neither of the two plans has more splits than the other everywhere.
inline int64_t decode_workspace_bytes(int B, int H, int N, int D) {
  const int a = decode_plan(B, H, N, D, false).splits, b = decode_plan(B, H, N, D, true).splits;
  return decode_bytes(B, H, D, a > b ? a : b);
}
// Splits of a call that has `bytes` of scratch, at least those of `least` splits.  Scratch that the evened number outgrows holds the number it came from.
inline int decode_splits(int B, int H, int N, int D, bool padded, int64_t bytes) {
  const DecodePlan p = decode_plan(B, H, N, D, padded);
  return p.splits > 1 && bytes < decode_bytes(B, H, D, p.splits) ? p.least : p.splits;
}

// Whether the split that arrives last merges the others, where there are counters.  The kernels take longer that way (partials past the L2, a counter,
// partials back: three round trips to memory against a launch boundary), but the call is a launch and 4.5 us of host time shorter, and a generation step of one
// user waits for the host.  GPU, two launches / one, us: B1 H12 N1500 D64 8.0 / 8.3, B1 H4 N8192 D128 8.3 / 11.5, with more workgroups than CUs B4 H12 N3000 D64
// 11.0 / 12.2, B1 H16 N8000 D128 14.1 / 26.2.  A token, cache append and attention call: B1 H12 N1200 D64 14.2 / 12.3, H2 N32000 14.3 / 13.3, D128 H12 N2000
// 14.7 / 13.6, H4 N8000 14.2 / 14.2, H1 N16000 14.6 / 13.4.  Where the splits have several batches of keys a wave the step is the GPU's again: D128 H1
// N24000 14.4 / 14.4, H4 N12000 14.3 / 14.9, H4 N24000 15.4 / 17.7, D64 H4 N32000 14.4 / 14.8.  (Calls back to back with nothing between them are the GPU's
// as well: up to 0.5 us more at head dims up to 64 with few workgroups, 1 to 3 us at 128.)
inline bool decode_merge_pays(int B, int H, int N, int D, int splits) {
  const int64_t wgs = (int64_t)B * H * splits, batches = decode_batches(N, D);
  return splits > 1 && wgs <= kCus && (batches <= kDecodeMaxSplits || (2 * wgs <= kCus && batches <= 2 * kDecodeMaxSplits));
}
// Counters that a shape's calls may touch.  A few shapes pay without left padding only (3 pairs of 16385 to 21504 keys at head dim 64), and stay with two launches.
inline int decode_counters(int B, int H, int N, int D) {
  return decode_merge_pays(B, H, N, D, decode_plan(B, H, N, D, true).splits) ? B * H : 0;
}
inline bool decode_merges(int B, int H, int N, int D, int splits) {
  return decode_merge_pays(B, H, N, D, splits) && decode_counters(B, H, N, D) > 0;
}

}  // namespace fox
