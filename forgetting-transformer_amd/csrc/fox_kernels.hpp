// Kernel argument blocks and launcher declarations shared by the C ABI layer and
// the kernel translation units.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace fox {

struct View {
  const uint16_t* ptr;
  int64_t sb, sh, st;
};

// Optional epilogue of the forward: the gated per-head RMS norm of the output rows (see store_rows_norm_gate).
// Off when y.ptr is null.  gate and y are (B, H, M, D) views like o; w is (H*D) fp32; rstd is (B, M, H) fp32.
struct FwdEpilogue {
  View gate, y;
  const float* w;
  float* rstd;
  float eps;
  int act;
};

// Gates of a forward that forms their cumulative sums itself (fwd_body).
struct GateK {
  const void* g;       // log gates (fp32), or logits
  int64_t sb, sh, sn;  // element strides
  int kind;            // kGateLog, or the dtype of the logits
  float* c;            // (B,H,N) or null: the cumulative sums, for a backward
  float* log_fgate;    // (B,H,N) or null: the log gates of logits
};
enum : int { kGateLog = -1 };            // else 0 bf16, 1 fp16, 2 fp32 logits
constexpr int kOwnScanMaxKeys = 3584;    // what fits beside the tiles in LDS at every head dim and occupancy

// Division by a number that is fixed for a launch, n / d = n * mul >> shift, exact for 0 <= n < 2^31: mul is 2^shift / d rounded up, by less than
// one, so the quotient is too large by less than n / 2^shift <= 1 / d.  (A division of scalars is some twenty dependent instructions.)
struct Divisor {
  uint32_t mul;
  int32_t shift;
};
constexpr Divisor divisor(int32_t d) {
  int32_t shift = 31;
  while (((int64_t)1 << (shift - 31)) < d) ++shift;
  return {(uint32_t)((((uint64_t)1 << shift) + d - 1) / d), shift};
}
__host__ __device__ __forceinline__ int divide(int n, Divisor d) { return (int)(((uint64_t)(uint32_t)n * d.mul) >> d.shift); }

// Launch order of the attention kernels, made by block_order(), read by decode_block().
struct BlockOrder {
  int32_t tiles;              // of a (batch, head) pair
  int32_t nb;                 // pairs per XCD, or of the launch where 8 does not divide them
  int32_t size, extra;        // groups of pairs: the first `extra` hold size + 1, the others size
  Divisor by_size[2], by_group[2];   // by the pairs and by the workgroups of a group; [1]: of a larger one
  Divisor by_heads;           // pair -> batch
  int32_t by_xcd, fold;
};

struct FwdK {
  View q, k, v, o;
  const float* c;
  float* lse;
  const int64_t* seq_start;
  const float* thr;
  int32_t* first_block;
  int B, H, M, N;
  float sm_scale;
  int n_mtiles;
  int splits;      // key splits of the forward (1 = none)
  BlockOrder order;
  Divisor by_splits;
  bool pair;       // two groups of waves share every query tile's walk (fwd_pairs)
  float* ws_o;     // (splits, B, H, M, D) partial accumulators
  float* ws_ml;    // (splits, B, H, M, 2) partial row maximum and row sum
  FwdEpilogue epi; // only for splits == 1 and M > 1 (the launcher rejects it otherwise)
  bool stream;     // K and V tiles are read once and not again soon: load them with the non-temporal hint
  GateK gates;     // launch_fwd_gates only, which does not read c
};

// Single-query forward from the log gates (decode_gates_kernel).
struct DecodePartial {   // of one key split: sum of its gates, maximum (log2 domain, relative to its last key) and row sum
  double g;
  float m, l;
};
struct DecodeK {
  View q, k, v, o;
  const float* g;            // log gates, element strides below
  int64_t g_sb, g_sh, g_sn;
  float* lse;                // (B,H) or null
  const int64_t* seq_start;
  int B, H, N;
  float sm_scale;
  int splits;
  Divisor by_splits, by_heads;
  float* ws_o;               // (B, H, splits, D) partial accumulators
  DecodePartial* ws_p;       // (B, H, splits)
  uint32_t* arrived;         // null, or (B, H) zeros: the split that arrives last merges them and leaves a zero
};
constexpr int kDecodeMaxSplits = 64;                     // one lane of a wave each in the merge
template <int D> constexpr int kDecodeBatchKeys = 4096 / D;   // keys a wave holds in flight: 8 KiB of K and 8 KiB of V

// New tokens into a layer's key, value and gate buffers: rows old .. old + T - 1 of every (batch, head).
struct CacheAppendK {
  View k, v, k_buf, v_buf;
  const float* g;
  float* g_buf;
  int64_t g_sb, g_sh, g_sn, gb_sb, gb_sh, gb_sn, old;
  int H, T, D;
  uint32_t total;   // 16-byte pieces of K: B * H * T * D / 8
};

struct BwdK {
  View q, k, v, o, d_o, dq, dk, dv;
  const float* c;
  const float* lse;
  const int64_t* seq_start;
  const float* thr;
  float* delta;   // (B,H,M): rowsum(o * do), written by the dQ kernel
  float* drow;    // (B,H,M): row sums of dS, written by the dQ kernel, read by the dK/dV kernel
  float* dc;
  int B, H, M, N;
  float sm_scale;
  int n_tiles;
  BlockOrder order;   // set by the launchers
  bool last_first;    // dQ: pairs from the last to the first, set by its launcher
  int cls;         // kClassAll, or the class of key tiles this dK/dV launch handles (fox_common.hpp)
  int light_limit; // distance from the diagonal, in keys, that separates the two classes
  int32_t* q_first_block;  // optional (B,H,ceil(M/kFwdBM)): first key block (of kFwdBN keys) each query tile of the dQ kernel visits
  int32_t* kv_end_row;     // optional (B,H,ceil(N/kKvUnit)): per unit of kKvUnit keys, the query row at which the dK/dV kernel stops
};

constexpr int kKvUnit = 64;  // granularity of kv_end_row: the smallest key tile any dK/dV variant uses

// Token shift: x, out, dout, dx are (B, T, H, D) 16-bit with shared element strides; the weights and
// their gradients are (B, T, H) fp32 with shared element strides.
struct ShiftK {
  const uint16_t* x;
  uint16_t* out;
  const uint16_t* dout;
  uint16_t* dx;
  const float* prev_w;
  const float* curr_w;
  float* dprev_w;
  float* dcurr_w;
  int64_t x_sb, x_st, x_sh, w_sb, w_st, w_sh;
  int B, T, H;
  int strip;   // time steps per thread, set by the launcher
};

// Gated per-head RMS norm: x, g, y, dy, dx, dg are (R rows, G heads, D) 16-bit, heads and head dim
// contiguous, each with its own row stride; w, dw are (G*D) fp32; rstd is (R, G) fp32.
struct NormGateK {
  const uint16_t* x;
  const uint16_t* g;
  uint16_t* y;
  const uint16_t* dy;
  uint16_t* dx;
  uint16_t* dg;
  const float* w;
  float* rstd;
  float* dw;
  float* dw_partial;
  int64_t x_sr, g_sr, y_sr, dy_sr, dx_sr, dg_sr;
  int64_t R;
  int G;
  float eps;
  int cols, rows_per_lane;   // how the backward is cut (norm_bwd_plan), set by the launcher
};

// Tile sizes (see fox_tile_config in the public header)
constexpr int kXcds = 8, kCus = 256;
constexpr int kFwdBM = 128;
constexpr int kFwdBN = 64;
constexpr int kKvBN = 128;   // key rows per workgroup in the dK/dV kernel
constexpr int kKvBM = 128;   // query rows per step in the dK/dV kernel

// Groups of (batch, head) pairs in the launch order of the attention kernels (decode_block).  A group ends with its
// lightest tiles, so the larger the last group, the less of the chip idles while the final heavy tiles finish; the
// smaller a group, the better its K and V stay in an XCD's 4 MiB L2.  The line lies at 8 MiB of K and V per group and XCD,
// with at least two pairs.  Forward time against one pair after the other, D = 128, B*H = 64, for 2 / 4 / 8 pairs a group:
// T = 4096 (2 MiB a pair) 0.890 / 0.877 / 0.886, T = 8192 0.971 / 0.968 / 0.994, T = 16384 0.971 / 0.986 / 1.064; D = 64, B*H = 128,
// T = 1024, for 4 / 8 / 16: 0.842 / 0.789 / 0.781.  With many more keys than queries the tiles weigh about the same and
// only the caches count: one pair after the other (dK/dV at M = 128, N = 32768: 2.52 ms, in groups of two 2.65 ms).
// Below D = 64 with the heads of a token side by side, a row is a part of a 128-byte line that it shares with the heads next to it.
// - Without a threshold a row counts as the whole line, whose other heads run on other XCDs: by its own bytes D = 16, B4 T4096 H64 got 32
//   pairs a group, forward 478 -> 600 us and backward 1.09 -> 1.37 ms against one pair after the other (now 435 us and 1.04 ms).  Under a
//   threshold the walks are short and large groups cost nothing (D = 16, B8 H16 T2048 "auto", groups by bytes over one pair after the
//   other: forward 1.10, backward 1.12 of its rate).
// - Where 8 does not divide the pairs, one pair after the other puts tile t of pair b on XCD (b * tiles + t) % 8: pairs 8 / gcd(tiles, 8) apart
//   meet on an XCD, and when they share lines that is worth more than groups can give to the short walks under a threshold.  At -10, groups
//   over that order, forward / backward rate: D = 16 with 64 tiles B4 H15 0.83 / 0.65, with 60 (every second pair) B9 H12 0.85 / 0.69, with 54 1.02 / 1.01;
//   D = 32 with 64 tiles B4 H15 0.90 / 0.81, with 60 1.07 / 1.05.  Up to four tiles per CU groups are the faster ones anyway.
constexpr bool even_tiles(int M, int N) { return (int64_t)2 * M < N; }
constexpr int order_groups(int n_bh, int tiles, int M, int N, int D, int64_t row_stride, bool pruned) {
  const bool by_xcd = n_bh % 8 == 0;
  const int nb = by_xcd ? n_bh / 8 : n_bh;
  const int64_t line = row_stride < 64 ? row_stride : 64;   // in elements
  if (pruned && !by_xcd && (int64_t)tiles * n_bh > 4 * 256) {
    const int apart = tiles % 8 == 0 ? 1 : tiles % 4 == 0 ? 2 : tiles % 2 == 0 ? 4 : 8;
    if (apart * D < line) return nb;
  }
  const int64_t row = pruned || D > line ? D : line;
  int64_t per = ((int64_t)8 << 20) / (N * row * 4);
  if (per < 2) per = 2;
  if (even_tiles(M, N)) per = 1;
  const int64_t groups = nb / (by_xcd ? per : per * 8);
  return groups < 1 ? 1 : (int)groups;
}
// The divisions of decode_block and their operands.  `fold` asks for the folded order, which a grid gets that is resident at once.
constexpr BlockOrder block_order(int B, int H, int tiles, int groups, bool fold) {
  BlockOrder o{};
  const int n_bh = B * H;
  o.tiles = tiles;
  o.by_xcd = n_bh % kXcds == 0;
  o.nb = o.by_xcd ? n_bh / kXcds : n_bh;
  o.size = o.nb / groups;
  o.extra = o.nb % groups;
  for (int i = 0; i < 2; ++i) {
    o.by_size[i] = divisor(o.size + i);
    o.by_group[i] = divisor((o.size + i) * tiles);
  }
  o.by_heads = divisor(H);
  o.fold = fold && (int64_t)tiles * o.nb <= 2 * (o.by_xcd ? kCus / kXcds : kCus);
  return o;
}

// Workgroup id -> (bh, tile).  Every tile of one (batch, head) goes to one XCD when the count allows it (the hardware
// deals consecutive workgroup ids round-robin over the 8 XCDs, each with its own L2).  Within an XCD the (batch, head)
// pairs are taken in groups of nearly equal size, and inside a group the tiles come heaviest first (largest index
// under a causal mask) with the pairs of the group in turn.  One pair after the other would start the last pair's
// heaviest tile when the chip is about to run empty; all pairs at once would stream more K and V than an L2 holds.
// order_groups() picks the number of groups, block_order() makes the operands.
// Folded: when the whole grid is resident at two workgroups per CU, the second workgroup of a CU is the one that arrives
// kCus ids after the first.  Taken in the same order both would be heavy on one CU and both light on another; from
// workgroup kCus on the list is therefore walked from its light end (forward B1 H16 T4096 D128: 109 -> 84 us, dQ 152 -> 116 us).
// `last_first`: the pairs from the last to the first.  The dQ kernel takes them so (with one exception, dq_t), between a forward and a dK/dV kernel that start with the
// first: each of the three then opens on the tensors its predecessor touched last, which are still in the 256 MiB last-level cache.
// Backward with dQ ascending / descending: B4 T16384 H16 D128 "auto" 731 / 710 us, B16 H16 T4096 D64 "auto" 516 / 491,
// B4 H32 T4096 D64 at -10 240 / 229, without a threshold 963 / 953.
// What is divided by is the same for a whole launch: six divisions by Divisor instead of the compiler's take some 130 instructions off the front of a
// kernel, which is what a workgroup of a pruned walk and one that finds nothing to do notice (at -10: the dK/dV class without a tile, B4 T4096 H16 D128, 6.9 -> 5.6 us, forward
// B4 T4096 H32 D64 57.9 -> 56.5; other kernels and dense walks within the runs' spread).
__host__ __device__ __forceinline__ void decode_block(uint32_t wid, const BlockOrder& o, bool last_first, int& bh, int& tile) {
  int r = (int)(o.by_xcd ? wid / kXcds : wid);
  const int cus = o.by_xcd ? kCus / kXcds : kCus;
  if (o.fold && r >= cus) r = o.tiles * o.nb - 1 - (r - cus);
  const int big_pairs = o.extra * (o.size + 1);
  const int big = r < big_pairs * o.tiles, size = o.size + big;
  const Divisor by_group = big ? o.by_group[1] : o.by_group[0], by_size = big ? o.by_size[1] : o.by_size[0];
  const int q = big ? r : r - big_pairs * o.tiles, grp = divide(q, by_group), in = q - grp * size * o.tiles, t = divide(in, by_size);
  int b = (big ? 0 : big_pairs) + grp * size + in - t * size;
  tile = o.tiles - 1 - t;
  if (last_first) b = o.nb - 1 - b;
  bh = o.by_xcd ? b * kXcds + (int)(wid % kXcds) : b;
}

// blockIdx.x, once the lines of the argument block that a kernel opens with are there.  Left to the compiler the order's operands are loaded first and the
// sizes only where they are needed, a round trip to memory further on, which a short walk notices (sizes later / together: dQ B1 H8 T2870 D128 68.4 / 67.5 us, B2 H3 T3000
// 71.2 / 70.2, forward B1 H8 T7200 D64 at -10 12.1 / 11.8).  Not in the paired and the split forward and the one with its own sums, which lose by
// it (B2 H3 T1794 D128 25.1 / 25.5, B1 H12 T77 D64 6.5 / 6.6).
template <typename K>
__device__ __forceinline__ uint32_t block_id(const K& a) {
  uint32_t id = blockIdx.x;
  asm volatile("" : "+s"(id) : "s"(a.order.tiles), "s"(a.seq_start), "s"(a.M));
  return id;
}

// Tile t of a (batch, head) pair in the one-launch backward (dq_kernel with BOTH), which holds key_tiles + query_tiles of them (M <= N, so there are at
// least as many of the former).  From the last to the first: query and key tiles in turn, heaviest first, then the key tiles left over.
struct BothTile {
  bool query;
  int tile;
};
__host__ __device__ __forceinline__ BothTile both_tile(int t, int key_tiles, int query_tiles) {
  const int rest = key_tiles - query_tiles, u = t - rest;
  if (u >= 0 && (u & 1)) return {true, u >> 1};
  const int rank = u < 0 ? t : rest + (u >> 1);   // of the key tile, from the one with the fewest rows to walk
  return {false, key_tiles - 1 - rank};
}

hipError_t launch_fwd(const FwdK& a, int D, int dtype, hipStream_t s);
hipError_t launch_fwd_gates(const FwdK& a, int D, int dtype, hipStream_t s);   // unsplit, at most kOwnScanMaxKeys keys, M > 1
bool fwd_can_scan(int B, int H, int M, int N, int splits);
bool fwd_scans(int B, int H, int M, int N, int D, bool pruned, int splits);
int fwd_key_splits(int B, int H, int M, int N, int D);
bool fwd_pairs(int B, int H, int M, int N, int D, bool pruned, int splits);
hipError_t launch_bwd_delta(const BwdK& a, int D, int dtype, hipStream_t s);
hipError_t launch_bwd_dkdv(const BwdK& a, int D, int dtype, hipStream_t s);   // a.cls selects the variant and its tiles
bool dkdv_split_supports(int D);   // head dims the split (kClassLight) variant of the dK/dV kernel exists for
bool bwd_together(const BwdK& a, int D);
hipError_t launch_bwd(const BwdK& a, int D, int dtype, hipStream_t s);   // dq_kernel's and dkdv_kernel's work in one launch
hipError_t launch_bwd_dq(const BwdK& a, int D, int dtype, hipStream_t s);
hipError_t launch_fwd_decode(const FwdK& a, int D, int dtype, hipStream_t s);  // M == 1, without the merge of the splits
hipError_t launch_decode_gates(const DecodeK& a, int D, int dtype, hipStream_t s);
hipError_t launch_cache_append(const CacheAppendK& a, hipStream_t s);
hipError_t launch_norm_gate(const NormGateK& a, int D, int dtype, bool bwd, int act, hipStream_t s);  // act: FOX_ACT_*
int64_t norm_gate_workspace_rows(int64_t rows);
hipError_t launch_shift_fwd(const ShiftK& a, int D, int dtype, hipStream_t s);
hipError_t launch_shift_bwd(const ShiftK& a, int D, int dtype, hipStream_t s);
hipError_t launch_cumsum_fwd(const float* g, int64_t sb, int64_t sh, int64_t sn, const int64_t* seq_start, float* c, int B,
                             int H, int N, hipStream_t s);
hipError_t launch_gate_cumsum_fwd(const void* logits, int dtype, int64_t sb, int64_t sh, int64_t sn, const int64_t* seq_start,
                                  float* log_fgate, float* c, int B, int H, int N, hipStream_t s);
// drow: null (dc is only read), or (B,H,M) added to the last M of dc, in memory as well
hipError_t launch_gate_cumsum_bwd(float* dc, const void* logits, int dtype, int64_t sb, int64_t sh, int64_t sn,
                                  const int64_t* seq_start, void* dlogits, int64_t db, int64_t dh, int64_t dn, int B, int H, int N,
                                  const float* drow, int M, hipStream_t s);
hipError_t launch_cumsum_bwd(float* dc, float* dg, int64_t db, int64_t dh, int64_t dn, const int64_t* seq_start, int B, int H,
                             int N, const float* drow, int M, hipStream_t s);
hipError_t launch_mfma_probe(const void* operands, float* sink, int workgroups, int iters, hipStream_t s);  // fox_probe.hip
hipError_t launch_qk_norm_threshold(const float* wq, const float* wk, int H, int D, double seq_len, double tolerance, float* thr, hipStream_t s);
hipError_t launch_auto_threshold(const View& q, const View& k, int B, int H, int M, int N, int D, int dtype, float sm_scale,
                                 float* thr, uint32_t* scratch, const GateK* t, const int64_t* seq_start, hipStream_t s);   // t: null, or scanned as well
bool threshold_scans(int B, int H, int M, int N, int D);

}  // namespace fox
