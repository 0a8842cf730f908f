// Forward kernel of Forgetting Attention for gfx950.
//
// One workgroup (4 waves) owns 128 query rows of one (batch, head); wave w owns
// rows 32w..32w+31 and keeps them in registers as the B operand of
// S^T = K Q^T (32x32x16 MFMA).  With the scores transposed, lane (g, i) holds one
// query row i and 16 key columns per 32-column block, so the online-softmax row
// statistics are lane-local plus one exchange between the two 32-lane halves, and
// the probabilities are already laid out as the B operand of O^T = V^T P^T.
//
// K and V tiles of 64 keys go from HBM straight into LDS (buffer loads with the
// LDS bit: no registers, no ds_write; out-of-range rows read as zero), into two
// alternating buffers, so the loads of the next tile fly while the current one is
// consumed and there is one barrier per tile.  V^T is read with the transposing
// LDS load.
// When a (batch, head) has a single query tile nobody reads a K or V tile twice, and the
// loads carry the non-temporal hint (the STREAM instantiation).
//
// Key tiles are walked from the diagonal backwards.  Under a forget gate the
// scores shrink with distance, so the running row maximum is set by the first
// tiles; it is only raised when a tile exceeds it by more than 2^8, which keeps
// every exponent <= 8 (exact in fp32/bf16 terms, the factor cancels in o = acc/l)
// and makes the rescale of the accumulator a rare, wave-uniform branch.
//
// The decay bias enters relative to c_ref = c[first query row of the tile]:
//   x = (q.k) * sm_scale*log2e - (c_n - c_ref)*log2e          (per score)
// and the row term (c_m - c_ref)*log2e, constant along a row, is only added to the
// stored log-normaliser.  Columns left of seq_start (and beyond N) get
// (c_n - c_ref) = +inf, which makes x = -inf without a compare in the loop; only
// tiles crossing the diagonal run the causal compare (separate code path).
#include <stddef.h>

#include "fox_common.hpp"
#include "fox_kernels.hpp"

namespace fox {

constexpr float kLazyMaxLog2 = 8.0f;
constexpr int kMinPipelinedTiles = 4;   // interior tiles below which the software-pipelined path is not entered

template <typename Tr, int D>
__device__ __forceinline__ void fwd_tile(const char* k_tile, const char* v_tile, const float* cn_s, const u32x4 (&qreg)[D / 16],
                                f32x16 (&oacc)[(D + 31) / 32], float& m_i, float& l_i, int n0, int a_m, float qk_scale,
                                int lane, bool diag) {
  constexpr int BN = kFwdBN, KK = D / 16, DB = (D + 31) / 32, NB = BN / 32;
  const int g = lane >> 5, i = lane & 31;

  // S^T = K Q^T + key term
  f32x16 s[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    u32x4 ka[KK];
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) ka[kk] = lds_row_operand<D>(k_tile, 32 * nb + i, 2 * kk + g);
    s[nb] = acc_init(cn_s, 32 * nb, g);
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) s[nb] = Tr::mfma32(ka[kk], qreg[kk], s[nb]);
  }

  // scores in the log2 domain and their maximum
  float mloc = -INFINITY;
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int r = 0; r < 16; ++r) s[nb][r] *= qk_scale;
  if (diag) {  // causal compare, only on tiles that cross the diagonal
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int n = n0 + 32 * nb + c_row(r, g);
        s[nb][r] = (n > a_m) ? -INFINITY : s[nb][r];
      }
  }
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int r = 0; r < 16; ++r) mloc = fmaxf(mloc, s[nb][r]);
  mloc = half_max(mloc);
  const bool raise = mloc > m_i + kLazyMaxLog2;
  if (__any(raise)) {  // rare: rescale what has been accumulated so far
    const float m_new = raise ? mloc : m_i;
    const float alpha = __builtin_amdgcn_exp2f(m_i - m_new);
    m_i = m_new;
    l_i *= alpha;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) oacc[db][r] *= alpha;
  }
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int r = 0; r < 16; ++r) s[nb][r] = __builtin_amdgcn_exp2f(s[nb][r] - m_i);

  // O^T += V^T P^T.  The row sum is taken over the probabilities as rounded for the MFMA (the weights that
  // multiply V then add up to exactly l), two at a time: per-lane partial sum, the two halves are added in the epilogue.
  float rsum = 0.f;
#pragma unroll
  for (int sl = 0; sl < BN / 16; ++sl) {
    const u32x4 pb = pack8<Tr>(s[sl >> 1], 8 * (sl & 1));
#pragma unroll
    for (int e = 0; e < 4; ++e) rsum = Tr::add_pair(pb[e], rsum);
    u32x4 va[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) va[db] = lds_col_operand<D>(v_tile, 16 * sl, db, lane);
#pragma unroll
    for (int db = 0; db < DB; ++db) oacc[db] = Tr::mfma32(va[db], pb, oacc[db]);
  }
  l_i += rsum;
}

// Interior tile (no key of the tile is right of any query row of the workgroup): branch-free and
// software-pipelined across tiles.  While the vector ALU turns the scores of the current tile into
// probabilities, the matrix pipe already computes the scores of the next tile (from k_next) and then
// accumulates the current tile's P V (from v_cur).  s_cur holds the raw scores of the current tile
// on entry; s_next holds those of the next tile on exit.  Work is issued in small chunks separated
// by scheduling fences so that MFMA and vector instructions alternate in the instruction stream.
// dma(u) issues chunk u's share of the global loads of the tiles after next: spread over the tile they
// do not hold the wave's issue slot back to back right after the barrier.
template <typename Tr, int D, typename Dma>
__device__ __forceinline__ void fwd_tile_pipelined(const char* k_next, const char* v_cur, const float* cn_next,
                                                  const u32x4 (&qreg)[D / 16], f32x16 (&oacc)[(D + 31) / 32], float& m_i,
                                                  float& l_i, float qk_scale, int lane, f32x16 (&s_cur)[kFwdBN / 32],
                                                  f32x16 (&s_next)[kFwdBN / 32], Dma dma) {
  constexpr int BN = kFwdBN, KK = D / 16, DB = (D + 31) / 32, NB = BN / 32, NSL = BN / 16;
  constexpr int SPC = 16 * NB / KK;  // scores handled per chunk of phase A
  static_assert(16 * NB % KK == 0 && SPC % 4 == 0, "whole float4 groups of scores per chunk");
  const int g = lane >> 5, i = lane & 31;

  // Phase A: scores of the next tile  ||  maximum of the current tile's raw scores (sm_scale > 0 here)
  float mloc = -INFINITY;
  u32x4 ka[NB][KK + 1];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    ka[nb][0] = lds_row_operand<D>(k_next, 32 * nb + i, g);
    s_next[nb] = acc_init(cn_next, 32 * nb, g);
  }
  static_for<0, KK>([&](auto uc) {
    constexpr int u = decltype(uc)::value;
    dma(u);  // this chunk's share of the global loads of the tiles after next
    if constexpr (u + 1 < KK) {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) ka[nb][u + 1] = lds_row_operand<D>(k_next, 32 * nb + i, 2 * (u + 1) + g);
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) s_next[nb] = Tr::mfma32(ka[nb][u], qreg[u], s_next[nb]);
#pragma unroll
    for (int e = 0; e < SPC; ++e) {
      const int idx = u * SPC + e;
      mloc = fmaxf(mloc, s_cur[idx >> 4][idx & 15]);
    }
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, (SPC / 2 + NB - 1) / NB, 0);  // the chunk's v_max3 dealt out over its MFMAs
    }
    __builtin_amdgcn_sched_barrier(0);
  });
  mloc = half_max(mloc) * qk_scale;
  const bool raise = mloc > m_i + kLazyMaxLog2;
  if (__any(raise)) {  // rare: rescale what has been accumulated so far
    const float m_new = raise ? mloc : m_i;
    const float alpha = __builtin_amdgcn_exp2f(m_i - m_new);
    m_i = m_new;
    l_i *= alpha;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) oacc[db][r] *= alpha;
  }

  // Phase B: p = exp2(s*scale - m), row sums, pack  ||  O^T += V^T P^T, one 16-key slice behind
  const float neg_m = -m_i;
  float rsum = 0.f;
  u32x4 pb[NSL];
  u32x4 va[NSL][DB];
#pragma unroll
  for (int c = 0; c <= NSL; ++c) {
    if (c < NSL) {
#pragma unroll
      for (int db = 0; db < DB; ++db) va[c][db] = lds_col_operand<D>(v_cur, 16 * c, db, lane);
    }
    if (c >= 1) {
#pragma unroll
      for (int db = 0; db < DB; ++db) oacc[db] = Tr::mfma32(va[c - 1][db], pb[c - 1], oacc[db]);
    }
    if (c < NSL) {
      const int nb = c >> 1, r0 = 8 * (c & 1);
#pragma unroll
      for (int e = 0; e < 8; ++e) s_cur[nb][r0 + e] = __builtin_amdgcn_exp2f(fmaf(s_cur[nb][r0 + e], qk_scale, neg_m));
      pb[c] = pack8<Tr>(s_cur[nb], r0);
#pragma unroll
      for (int e = 0; e < 4; ++e) rsum = Tr::add_pair(pb[c][e], rsum);  // row sum of the rounded probabilities
    }
    if (c >= 1 && c < NSL) {
#pragma unroll
      for (int k = 0; k < DB; ++k) {  // a slice has 16 vector and 8 exp instructions: dealt out over its DB MFMAs
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 16 / DB, 0);
        __builtin_amdgcn_sched_group_barrier(0x400, 8 / DB, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  l_i += rsum;
}

// The global loads of a K tile and a V tile, dealt out over the D/16 chunks of a pipelined tile:
// dma(u) issues chunk u's share.
template <int D, int AUX>
struct TileDma {
  static constexpr int KK = D / 16, PER = DirectTileLoader<D, kFwdBN, 4, AUX>::PER, PER_CHUNK = (2 * PER + KK - 1) / KK;
  const DirectTileLoader<D, kFwdBN, 4, AUX>& kld;
  const DirectTileLoader<D, kFwdBN, 4, AUX>& vld;
  const uint16_t* k_src;
  const uint16_t* v_src;
  int k_bytes, v_bytes;
  char* k_fill;
  char* v_fill;
  __device__ __forceinline__ void all() const {
#pragma unroll
    for (int j = 0; j < PER; ++j) kld.issue_one(j, k_src, k_bytes, k_fill);
#pragma unroll
    for (int j = 0; j < PER; ++j) vld.issue_one(j, v_src, v_bytes, v_fill);
  }
  __device__ __forceinline__ void operator()(int u) const {  // u is a constant at every call site
#pragma unroll
    for (int r = 0; r < PER_CHUNK; ++r) {
      const int idx = u * PER_CHUNK + r;
      if (idx < PER) kld.issue_one(idx, k_src, k_bytes, k_fill);
      else if (idx < 2 * PER) vld.issue_one(idx - PER, v_src, v_bytes, v_fill);
    }
  }
};

// Cumulative sums c[n] = sum of the gates of keys seq .. n (zero left of seq) for n < hi, into LDS.  As in scan_row: coalesced through LDS,
// consecutive keys per thread, fp64, rounded once.  Positions from `first` to hi are also stored for the backward, as are the log gates of
// logits.  fetch() requests the gates: it comes before the tile loads, which the counter of loads in flight retires in order, and the barriers
// below wait for LDS only, so the tiles and Q arrive while the sums are formed.
template <int NT>
struct OwnScan {
  static constexpr int MAX = (kOwnScanMaxKeys / NT + 1) | 1;   // keys per thread: odd, so that a wave's reads fall on different banks
  float g[MAX];

  static __device__ __forceinline__ void barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
  template <int KIND>
  __device__ __forceinline__ void fetch_as(const GateK& t, int64_t row, int hi, int tid) {
#pragma unroll
    for (int e = 0; e < MAX; ++e) {
      if (e * NT >= hi) break;
      const int64_t i = row + min(e * NT + tid, hi - 1) * t.sn;
      if constexpr (KIND == kGateLog) g[e] = reinterpret_cast<const float*>(t.g)[i];
      else g[e] = load_logit<KIND>(t.g, i);
    }
  }
  __device__ __forceinline__ void fetch(const GateK& t, int b, int h, int hi, int tid) {
    const int64_t row = b * t.sb + h * t.sh;
    if (t.kind == kGateLog) fetch_as<kGateLog>(t, row, hi, tid);
    else if (t.kind == 0) fetch_as<0>(t, row, hi, tid);
    else if (t.kind == 1) fetch_as<1>(t, row, hi, tid);
    else fetch_as<2>(t, row, hi, tid);
  }
  __device__ __forceinline__ void run(const GateK& t, float* c_s, int64_t out_row, int hi, int seq, int first, int tid) {
    __shared__ double wave_tot[NT / kWave];
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
#pragma unroll
    for (int e = 0; e < MAX; ++e) {
      if (e * NT >= hi) break;
      const int n = e * NT + tid;
      if (t.kind != kGateLog) {
        g[e] = log_sigmoid(g[e]);
        if (t.log_fgate && n >= first && n < hi) t.log_fgate[out_row + n] = g[e];
      }
      if (n < hi) c_s[n] = n >= seq ? g[e] : 0.f;
    }
    barrier();
    const int per = ((hi + NT - 1) / NT) | 1, n0 = tid * per;
    double v[MAX], sum = 0.0;
#pragma unroll
    for (int e = 0; e < MAX; ++e) {
      if (e >= per) break;
      sum += n0 + e < hi ? (double)c_s[n0 + e] : 0.0;
      v[e] = sum;
    }
    const double incl = wave_scan(sum);
    if (lane == kWave - 1) wave_tot[wave] = incl;
    barrier();
    double before = lane_before(incl);
    for (int w = 0; w < wave; ++w) before += wave_tot[w];
#pragma unroll
    for (int e = 0; e < MAX; ++e) {
      if (e >= per) break;
      if (n0 + e < hi) c_s[n0 + e] = (float)(before + v[e]);
    }
    barrier();
    if (t.c)
      for (int n = first + tid; n < hi; n += NT) t.c[out_row + n] = c_s[n];
  }
};

// EPI: the variant whose epilogue also applies the layer's output norm and gate (a.epi); a variant of its own so
// that the plain kernel's register allocation is not touched by it.
// Waves per SIMD the forward is compiled for: the register budget that goes with it (512 / waves) holds the
// kernel to the occupancy its head dim allows.
template <int D>
constexpr int kFwdWaves = D <= 64 ? 3 : 2;

// STREAM: the variant for shapes with a single query tile per (batch, head): every K and V tile is read by exactly one
// workgroup, so the tile loads carry the non-temporal hint (with it the chunked-prefill shape B16 M128 N32768 H16 D128
// takes 0.62 ms instead of 0.71).  Where tiles are shared by the workgroups of several query tiles the hint costs 16-28 %.
//
// PAIR: the variant for grids of few query tiles (fwd_pairs below).  A workgroup has two groups of four waves with their own
// tile buffers; they take the key tiles of the same 128 query rows in turn, each with its own running maximum and sum, and group 0
// merges the two states from LDS before the epilogue.  The walk of the heaviest tile, which is what such a grid waits for, is half
// as long, and a CU with a single query tile has two waves per SIMD (B1 H16 T3001 D128, scan included: 67.7 -> 57.6 us).  Both groups pass the same barriers: the trip counts of
// the loops are those of group 0, and a step for which group 1 has no tile left moves and computes nothing.
//
// SCAN: the workgroup forms the cumulative sums of its row itself, from the log gates or their logits, up to its last key, and keeps them in
// LDS; each writes the part of its own rows for the backward.  Every workgroup of a row repeats the sum of what lies in front of it, so this is for
// grids of few workgroups per CU (fwd_scans, with the times), where it takes the scan's launch out of the chain.
template <typename Tr, int D, bool SPLIT, bool EPI, bool STREAM, bool PAIR, bool SCAN>
__device__ __forceinline__ void fwd_body(const FwdK& a) {   // a: the kernel's only argument
  static_assert(!(PAIR && (SPLIT || STREAM)), "the paired variant is for whole walks over shared tiles");
  static_assert(!PAIR || D >= 32, "group 1's accumulators are handed over in its tile buffers");
  constexpr int GROUPS = PAIR ? 2 : 1;
  static_assert(!(SPLIT && EPI), "partial results of a key split are not normalised");
  static_assert(!(STREAM && EPI), "no streaming variant with the epilogue");
  static_assert(!(SCAN && (SPLIT || STREAM)), "own sums are for whole walks over shared tiles");
  constexpr int AUX = STREAM ? kLoadNonTemporal : 0;
  constexpr int BM = kFwdBM, BN = kFwdBN;
  constexpr int KK = D / 16, DB = (D + 31) / 32, NB = BN / 32;
  static_assert(BM == 128, "four waves of 32 rows");
  __shared__ __align__(16) char k_tile0_s[GROUPS * Tile<D>::bytes(BN)];
  __shared__ __align__(16) char k_tile1_s[GROUPS * Tile<D>::bytes(BN)];
  __shared__ __align__(16) char v_tile0_s[GROUPS * Tile<D>::bytes(BN)];
  __shared__ __align__(16) char v_tile1_s[GROUPS * Tile<D>::bytes(BN)];
  __shared__ __align__(16) float cn_s0_s[GROUPS * BN];
  __shared__ __align__(16) float cn_s1_s[GROUPS * BN];

  const int wave_id = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), grp = PAIR ? wave_id >> 2 : 0;
  const int tid = PAIR ? threadIdx.x & 255 : threadIdx.x, wave = PAIR ? wave_id & 3 : wave_id;   // within the group
  const int lane = tid & 63, g = lane >> 5, i = lane & 31;
  char *k_tile0 = k_tile0_s + grp * Tile<D>::bytes(BN), *k_tile1 = k_tile1_s + grp * Tile<D>::bytes(BN);
  char *v_tile0 = v_tile0_s + grp * Tile<D>::bytes(BN), *v_tile1 = v_tile1_s + grp * Tile<D>::bytes(BN);
  float *cn_s0 = cn_s0_s + grp * BN, *cn_s1 = cn_s1_s + grp * BN;
  int bh, mt, sp = 0;
  if constexpr (SPLIT) {  // (query tile, key split) pairs take the place of query tiles
    int mts;
    decode_block(blockIdx.x, a.order, false, bh, mts);
    mt = divide(mts, a.by_splits);
    sp = mts - mt * a.splits;
  } else {
    decode_block(PAIR || SCAN ? blockIdx.x : block_id(a), a.order, false, bh, mt);
  }
  const int b = divide(bh, a.order.by_heads), h = bh - b * a.H;
  const int M = a.M, N = a.N, p_seq = N - M;
  const int m0 = mt * BM;
  __shared__ float c_s[SCAN ? kOwnScanMaxKeys : 1];
  const float* c_row = SCAN ? c_s : a.c + (int64_t)bh * N;   // (own sums: [0, hi))
  const uint16_t* qp = a.q.ptr + b * a.q.sb + h * a.q.sh;
  const uint16_t* kp = a.k.ptr + b * a.k.sb + h * a.k.sh;
  const uint16_t* vp = a.v.ptr + b * a.v.sb + h * a.v.sh;
  uint16_t* op = const_cast<uint16_t*>(a.o.ptr) + b * a.o.sb + h * a.o.sh;

  const int a0 = p_seq + m0;  // key position of the tile's first query row
  const int hi = min(N, a0 + BM);
  int seq = 0;
  if (a.seq_start) {
    const int64_t s64 = a.seq_start[b];
    seq = (int)(s64 < 0 ? 0 : (s64 > N ? N : s64));
  }
  const int m = m0 + 32 * wave + i;  // this lane's query row
  const int a_m = p_seq + m;
  const int a_w0 = a0 + 32 * wave;   // key position of the wave's first row
  const float qk_scale = nonzero_scale(a.sm_scale * kLog2e), inv_scale = 1.0f / qk_scale;
  // Everything the workgroup needs first is requested before anything is waited for.  The first tile to
  // visit (the one under the end of the diagonal) does not depend on the pruning bound, so it goes
  // first; then Q, then the per-row and per-key terms; the bound search's loads queue behind them.
  OwnScan<GROUPS * 256> scan;
  if constexpr (SCAN) scan.fetch(a.gates, b, h, hi, threadIdx.x);
  const DirectTileLoader<D, BN, 4, AUX> kld(a.k.st, wave, lane), vld(a.v.st, wave, lane);
  int n0_first = hi > 0 ? ((hi - 1) / BN) * BN : 0;
  bool early = !SPLIT && hi > (min(seq, hi) / BN) * BN && (n0_first + BN - 1 > a0 || !(qk_scale > 0.f));
  // The tile before it is requested as well when nothing can exclude it: it still reaches the workgroup's first row
  // (the pruning bound never cuts there) and lies right of seq_start.  Under pruning a workgroup visits two or
  // three tiles, and every round trip taken out of that chain counts.
  const int n0_second = n0_first - BN;
  bool early2 = early && n0_second >= (a0 / BN) * BN && n0_second >= (min(seq, hi) / BN) * BN &&
                      (n0_second + BN - 1 > a0 || !(qk_scale > 0.f));
  if constexpr (PAIR) {   // group 1's first tile is the second of the walk
    if (grp) {
      early = early2;
      n0_first = n0_second;
    }
    early2 = false;
  }
  if (early) {
    kld.issue(kp, a.k.st, n0_first, N, k_tile0);
    vld.issue(vp, a.v.st, n0_first, N, v_tile0);
  }
  if (early2) {
    kld.issue(kp, a.k.st, n0_second, N, k_tile1);
    vld.issue(vp, a.v.st, n0_second, N, v_tile1);
  }
  u32x4 qreg[KK];
  load_row_operand_regs<D>(qreg, qp, a.q.st, m, M, g);
  if constexpr (SCAN) scan.run(a.gates, c_s, (int64_t)bh * N, hi, seq, mt == 0 ? 0 : a0, threadIdx.x);
  const float c_ref = c_row[a0];
  const float c_m = c_row[min(a_m, (SCAN ? hi : N) - 1)];
  // Under pruning the third tile of the walk (the look-back tile, which is also the next query tile's upper diagonal
  // tile) is wanted more often than not, but its LDS buffer is busy until the first tile is done.  One dword per cache
  // line brings it into L2 now, while the neighbour fetches it as well (pruned forward 0.253 -> 0.246 ms at B4 T16384
  // H16 D128; the same in the dQ and dK/dV kernels costs 2-4 %, so only here).
  int l2_touch = 0;
  if (a.thr && early2) {
    const int n0_third = n0_second - BN;
    if (n0_third >= 0 && n0_third + BN > seq) {
      constexpr int LPR = (2 * D + 127) / 128;   // cache lines per row
      const int idx = tid & 127, row = idx / LPR, part = idx % LPR;
      if (row < BN) {
        const uint16_t* src = (tid < 128 ? kp + (int64_t)(n0_third + row) * a.k.st : vp + (int64_t)(n0_third + row) * a.v.st) + part * 64;
        l2_touch = *reinterpret_cast<const int*>(src);
      }
    }
  }

  // Key terms of a tile: the load is requested here, the arithmetic on it is done where the value goes to
  // LDS (a tile later), so that nothing waits for the load in between.  Masked keys get -inf through the
  // subtraction.
  // (Own sums are in LDS already: only the tile is kept.)
  float cn_raw = 0.f;
  bool cn_ok = false;
  int cn_n0 = 0;
  auto issue_cn = [&](int n0) {
    cn_n0 = n0;
    if (!SCAN && tid < BN) {
      const int n = n0 + tid;
      cn_ok = (n < N) & (n >= seq);
      cn_raw = c_row[min(n, N - 1)];
    }
  };
  auto cn_term = [&]() {
    if constexpr (SCAN) {
      const int n = cn_n0 + tid;
      return (c_ref - (n < N && n >= seq ? c_s[min(n, hi - 1)] : INFINITY)) * kLog2e * inv_scale;
    } else {
      return (c_ref - (cn_ok ? cn_raw : INFINITY)) * kLog2e * inv_scale;
    }
  };
  auto issue = [&](int n0, char* kt, char* vt) {
    issue_cn(n0);  // small load first: vmcnt retires in order, so it must not queue behind the tile loads
    kld.issue(kp, a.k.st, n0, N, kt);
    vld.issue(vp, a.v.st, n0, N, vt);
  };
  if (early) issue_cn(n0_first);
  float cn_raw2 = 0.f;   // key terms of the second early tile: handed to cn_raw once the first tile's are in LDS
  bool cn_ok2 = false;
  if (!SCAN && early2 && tid < BN) {
    const int n = n0_second + tid;
    cn_ok2 = (n < N) & (n >= seq);
    cn_raw2 = c_row[min(n, N - 1)];
  }
  const float cm2 = (m < M) ? (c_m - c_ref) * kLog2e : 0.f;

  f32x16 oacc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) oacc[db][r] = 0.f;
  float m_i = -3.0e38f, l_i = 0.f;  // finite floor: a row that has seen no valid key yet yields exp2(-inf) = 0

  int lo = min(seq, hi);
  if (a.thr) {
    const int t = acp_first_kept_block(c_row, c_ref, a.thr[bh], N, BN, a0 / BN, lane);
    lo = max(lo, t * BN);
  }
  lo = (lo / BN) * BN;
  if (a.first_block && tid == 0 && sp == 0) a.first_block[(int64_t)bh * a.n_mtiles + mt] = lo / BN;
  int n_tiles = (hi - lo + BN - 1) / BN;  // walked from the last (diagonal) tile down to lo
  if constexpr (SPLIT) {  // this workgroup's contiguous share of the key tiles
    const int per = divide(n_tiles + a.splits - 1, a.by_splits);
    const int t0 = min(n_tiles, sp * per), t1 = min(n_tiles, t0 + per);
    lo += t0 * BN;
    n_tiles = t1 - t0;
  }

  // A wave whose 32 rows all lie beyond M (decode and other short query blocks) still moves its share
  // of every tile but computes nothing.
  const bool wave_has_rows = m0 + 32 * wave < M;
  auto compute = [&](int n0, const char* kt, const char* vt, const float* cn) {
    if (n0 > a_w0 + 31 || !wave_has_rows) return;  // tile entirely above this wave's rows
    fwd_tile<Tr, D>(kt, vt, cn, qreg, oacc, m_i, l_i, n0, a_m, qk_scale, lane, n0 + BN - 1 > a_w0);
  };

  // Phase 1: the tiles that reach the workgroup's diagonal (the last ceil(BM/BN) + 1 at most), with
  // the masking code, double-buffered.  Phase 2: interior tiles, software-pipelined across tiles.
  // The pipelined code takes the row maximum on the raw accumulators, which needs sm_scale > 0;
  // otherwise every tile goes through phase 1.
  int n_diag = 0;
  while (n_diag < n_tiles && lo + (n_tiles - 1 - n_diag) * BN + BN - 1 > a0) ++n_diag;
  if (!(qk_scale > 0.f)) n_diag = n_tiles;
  // The pipelined path starts with two round trips of its own (K of its first tile, then V): worth it for a long
  // walk only.  With a few interior tiles (the usual case under pruning) they go through phase 1 as well.
  if (n_tiles - n_diag < kMinPipelinedTiles) n_diag = n_tiles;
  const int t_stop = n_tiles - n_diag;
  auto tile_n0 = [&](int t) { return lo + t * BN; };   // start of the tile at loop position t
  if (n_diag > 0) {
    if (!early && n_tiles - 1 - grp >= t_stop) issue(tile_n0(n_tiles - 1 - grp), k_tile0, v_tile0);
    if (tid < BN) cn_s0[tid] = cn_term();
    if (early2) { cn_raw = cn_raw2; cn_ok = cn_ok2; cn_n0 = n0_second; }
  }
  bool requested = early2;  // buffers 1 already hold (or await) the next tile
  for (int tu = n_tiles - 1; tu >= t_stop; tu -= 2 * GROUPS) {
    const int t = tu - grp, t1 = t - GROUPS, t2 = t - 2 * GROUPS;   // this group's tile and its next two
    // even step: consume buffers 0, fill buffers 1
    wait_vmem_all();
    __syncthreads();
    if (t1 >= t_stop && !requested) issue(tile_n0(t1), k_tile1, v_tile1);
    requested = false;
    if (!PAIR || t >= t_stop) compute(tile_n0(t), k_tile0, v_tile0, cn_s0);
    if (tu - GROUPS < t_stop) break;
    if (tid < BN) cn_s1[tid] = cn_term();
    // odd step: consume buffers 1, fill buffers 0
    wait_vmem_all();
    __syncthreads();
    if (t2 >= t_stop) issue(tile_n0(t2), k_tile0, v_tile0);
    if (!PAIR || t1 >= t_stop) compute(tile_n0(t1), k_tile1, v_tile1, cn_s1);
    if (t2 >= t_stop && tid < BN) cn_s0[tid] = cn_term();
  }

  if (t_stop > 0) {
    // this group's interior tile j (0 = nearest to the diagonal); n_steps is the count of group 0, the larger one
    const int n_int = (t_stop - grp + GROUPS - 1) / GROUPS, n_steps = (t_stop + GROUPS - 1) / GROUPS;
    auto int_n0 = [&](int j) { return lo + (t_stop - 1 - grp - GROUPS * j) * BN; };
    auto issue_k = [&](int j, char* kt) {
      const int n0 = int_n0(j);
      issue_cn(n0);
      kld.issue(kp, a.k.st, n0, N, kt);
    };
    auto issue_v = [&](int j, char* vt) { vld.issue(vp, a.v.st, int_n0(j), N, vt); };
    // K runs one tile ahead of V: iteration j computes S(j+1) and P(j) V(j).
    static_assert(kMinPipelinedTiles >= GROUPS, "every group has an interior tile here");
    __syncthreads();  // phase 1 is done with every buffer
    issue_k(0, k_tile0);
    if (tid < BN) cn_s0[tid] = cn_term();
    wait_vmem_all();
    __syncthreads();
    if (n_int > 1) issue_k(1, k_tile1);
    issue_v(0, v_tile0);
    f32x16 s_a[NB], s_b[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      if (!wave_has_rows) break;
      s_a[nb] = acc_init(cn_s0, 32 * nb, g);
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) s_a[nb] = Tr::mfma32(lds_row_operand<D>(k_tile0, 32 * nb + i, 2 * kk + g), qreg[kk], s_a[nb]);
    }
    // Iteration j: S(j+1) from k_nx, P(j) V(j) from v_cur; meanwhile K(j+2) is requested into k_fill and
    // V(j+1) into v_fill, one load instruction per chunk of the tile (an empty extent when there is no such
    // tile: the loads then write zeros into the free buffer).
    auto pipelined_tile = [&](int j, const char* k_nx, const char* v_cur, const float* cn_nx, char* k_fill, char* v_fill,
                              f32x16 (&s_cur)[NB], f32x16 (&s_nx)[NB]) {
      if (PAIR && j >= n_int) return;   // group 0 has one tile more
      const bool more_k = j + 2 < n_int, more_v = j + 1 < n_int;
      const int nk = more_k ? int_n0(j + 2) : lo, nv = more_v ? int_n0(j + 1) : lo;
      if (more_k) issue_cn(nk);
      const uint16_t *k_src = kp + (int64_t)nk * a.k.st, *v_src = vp + (int64_t)nv * a.v.st;
      const int k_bytes = kld.extent(a.k.st, nk, more_k ? N : nk), v_bytes = vld.extent(a.v.st, nv, more_v ? N : nv);
      const TileDma<D, AUX> dma{kld, vld, k_src, v_src, k_bytes, v_bytes, k_fill, v_fill};
      if (wave_has_rows) fwd_tile_pipelined<Tr, D>(k_nx, v_cur, cn_nx, qreg, oacc, m_i, l_i, qk_scale, lane, s_cur, s_nx, dma);
      else dma.all();  // a wave without query rows only moves its share of the tiles
    };
    for (int j = 0; j < n_steps; j += 2) {
      // even iteration: K(j+1) in k_tile1 with its key terms in cn_s1, V(j) in v_tile0.  The key
      // terms of tile j+1 go to LDS before the barrier: their buffer was last read two iterations ago.
      wait_vmem_all();
      if (j + 1 < n_int && tid < BN) cn_s1[tid] = cn_term();
      __syncthreads();
      pipelined_tile(j, k_tile1, v_tile0, cn_s1, k_tile0, v_tile1, s_a, s_b);
      if (j + 1 >= n_steps) break;
      // odd iteration: K(j+2) in k_tile0 with its key terms in cn_s0, V(j+1) in v_tile1
      wait_vmem_all();
      if (j + 2 < n_int && tid < BN) cn_s0[tid] = cn_term();
      __syncthreads();
      pipelined_tile(j + 1, k_tile0, v_tile1, cn_s0, k_tile1, v_tile0, s_b, s_a);
    }
  }

  // epilogue
  float l_tot = half_sum(l_i);
  if constexpr (PAIR) {   // group 1 leaves its state in its tile buffers (one per wave), group 0 takes it up and goes on alone
    __shared__ float pair_m[256], pair_l[256];
    static_assert(16 * DB * kWave * 4 <= Tile<D>::bytes(BN), "a wave's accumulators fit one tile buffer");
    const int next = Tile<D>::bytes(BN);
    float* there = reinterpret_cast<float*>((wave == 0 ? k_tile0_s : wave == 1 ? k_tile1_s : wave == 2 ? v_tile0_s : v_tile1_s) + next);
    wait_vmem_all();
    __syncthreads();
    if (grp) {
      pair_m[tid] = m_i;
      pair_l[tid] = l_tot;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) there[(16 * db + r) * kWave + lane] = oacc[db][r];
    }
    __syncthreads();
    if (grp) return;   // (no barrier below)
    const float m2 = pair_m[tid], mx = fmaxf(m_i, m2);
    const float w0 = __builtin_amdgcn_exp2f(m_i - mx), w1 = __builtin_amdgcn_exp2f(m2 - mx);
    m_i = mx;
    l_tot = l_tot * w0 + pair_l[tid] * w1;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) oacc[db][r] = oacc[db][r] * w0 + there[(16 * db + r) * kWave + lane] * w1;
  }
  if constexpr (SPLIT) {
    // partial result of this key split: unnormalised accumulator, row maximum (log2 domain,
    // including the row term) and row sum; fox::combine_kernel merges the splits
    if (m < M) {
      const int64_t row = ((int64_t)sp * a.B * a.H + bh) * M + m;
      float* wo = a.ws_o + row * D;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
          const int d = 32 * db + 8 * q4 + 4 * g;
          if (d < D) {
            f32x4 w = {oacc[db][4 * q4 + 0], oacc[db][4 * q4 + 1], oacc[db][4 * q4 + 2], oacc[db][4 * q4 + 3]};
            *reinterpret_cast<f32x4*>(wo + d) = w;
          }
        }
      if (g == 0) {
        a.ws_ml[2 * row] = m_i + cm2;
        a.ws_ml[2 * row + 1] = l_tot;
      }
    }
    return;
  }
  const bool empty = a_m < seq;
  const float inv = empty ? 0.f : 1.0f / l_tot;
  if (m < M && g == 0) a.lse[(int64_t)bh * M + m] = empty ? -INFINITY : (m_i + cm2) * kLn2 + __logf(l_tot);
  // o leaves through LDS (the tile buffers are free now, one per wave) so that the global stores are whole rows
  static_assert(kStoreStageBytes<D> <= Tile<D>::bytes(BN), "one wave stages in one tile buffer");
  if constexpr (!PAIR) {
    wait_vmem_all();  // whatever was requested last (possibly an empty tile) has landed
    __syncthreads();  // every wave is done with the last tile
  }
  char* stage = wave == 0 ? k_tile0 : wave == 1 ? k_tile1 : wave == 2 ? v_tile0 : v_tile1;
  if constexpr (EPI) {  // the layer's output norm and gate, applied while the rows are on their way out
    // The epilogue's arguments are fetched from the kernel argument block only here, through a pointer the
    // compiler cannot see through: loaded at kernel entry they would occupy scalar registers across the key loop.
    typedef const char __attribute__((address_space(4)))* kernarg_bytes;
    typedef const FwdEpilogue __attribute__((address_space(4)))* kernarg_epilogue;
    kernarg_epilogue ep = (kernarg_epilogue)((kernarg_bytes)__builtin_amdgcn_kernarg_segment_ptr() + offsetof(FwdK, epi));
    asm volatile("" : "+s"(ep));
    const uint16_t* gp = ep->gate.ptr ? ep->gate.ptr + b * ep->gate.sb + h * ep->gate.sh : nullptr;
    uint16_t* yp = const_cast<uint16_t*>(ep->y.ptr) + b * ep->y.sb + h * ep->y.sh;
    store_rows_norm_gate<Tr, D>(stage, oacc, inv, a.o.ptr ? op : nullptr, a.o.st, gp, ep->gate.st, yp, ep->y.st,
                                ep->w + h * D, ep->rstd + (int64_t)b * M * a.H + h, a.H, ep->eps, ep->act, m0 + 32 * wave,
                                M, lane);
  } else {
    store_rows_via_lds<Tr, D>(stage, oacc, inv, op, a.o.st, m0 + 32 * wave, M, lane);
  }
  asm volatile("" ::"v"(l2_touch));   // the value is never used; this keeps the load
}

// (the bodies for the device pass only: on the host side a kernel is a stub, and the tile code's device builtins do not resolve there)
template <typename Tr, int D, bool SPLIT, bool EPI = false, bool STREAM = false>
__global__ __launch_bounds__(256, kFwdWaves<D>) void fwd_kernel(const FwdK a) {
#ifdef __HIP_DEVICE_COMPILE__
  fwd_body<Tr, D, SPLIT, EPI, STREAM, false, false>(a);
#endif
}
template <typename Tr, int D, bool EPI>
__global__ __launch_bounds__(512, 2) void fwd_pair_kernel(const FwdK a) {
#ifdef __HIP_DEVICE_COMPILE__
  fwd_body<Tr, D, false, EPI, false, true, false>(a);
#endif
}
// The same two with their own cumulative sums
template <typename Tr, int D, bool EPI>
__global__ __launch_bounds__(256, kFwdWaves<D>) void fwd_scan_kernel(const FwdK a) {
#ifdef __HIP_DEVICE_COMPILE__
  fwd_body<Tr, D, false, EPI, false, false, true>(a);
#endif
}
template <typename Tr, int D, bool EPI>
__global__ __launch_bounds__(512, 2) void fwd_scan_pair_kernel(const FwdK a) {
#ifdef __HIP_DEVICE_COMPILE__
  fwd_body<Tr, D, false, EPI, false, true, true>(a);
#endif
}

// Merge the partial results of the key splits of one query row:
//   m = max_s m_s,  l = sum_s l_s 2^(m_s - m),  o = sum_s acc_s 2^(m_s - m) / l,  lse = m ln2 + ln l.
// One thread per (row, 4 head-dim elements).
template <typename Tr, int D, int U>
__global__ __launch_bounds__(256) void combine_kernel(const FwdK a) {
  constexpr int TPR = D / 4;  // threads per row
  const int64_t n_rows = (int64_t)a.B * a.H * a.M;
  const int64_t row = ((int64_t)blockIdx.x * 256 + threadIdx.x) / TPR;
  const int d = (threadIdx.x % TPR) * 4;
  if (row >= n_rows) return;
  const int bh = (int)(row / a.M), m = (int)(row % a.M), b = bh / a.H, h = bh % a.H;
  // U splits' partials in flight, the first ones' accumulators before the maximum is known: one after the other each split was a round trip to memory of
  // its own (B1 H12 M64 N16384 D64, 32 splits, the whole call 41.2 -> 30.5 us).  U follows the number of splits, since one more is one more read (two splits, 34 MB of them: 20.5 us
  // with U = 8, 11 to 13 with 2 and before).
  auto split = [&](int sp) { return min(sp, a.splits - 1) * n_rows + row; };   // splits past the end repeat the last one
  float mx = -INFINITY, l = 0.f;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  f32x4 o[U];
  auto fetch = [&](int sp0) {
#pragma unroll
    for (int u = 0; u < U; ++u) o[u] = *reinterpret_cast<const f32x4*>(a.ws_o + split(sp0 + u) * D + d);
  };
  fetch(0);
  for (int sp0 = 0; sp0 < a.splits; sp0 += U) {
#pragma unroll
    for (int u = 0; u < U; ++u) mx = fmaxf(mx, a.ws_ml[2 * split(sp0 + u)]);
  }
  for (int sp0 = 0; sp0 < a.splits; sp0 += U) {
    if (sp0) fetch(sp0);
    float ms[U], ls[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      ms[u] = a.ws_ml[2 * split(sp0 + u)];
      ls[u] = a.ws_ml[2 * split(sp0 + u) + 1];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (sp0 + u < a.splits) {
        const float w = __builtin_amdgcn_exp2f(ms[u] - mx);
        l += ls[u] * w;
        acc += o[u] * w;
      }
    }
  }
  int seq = 0;
  if (a.seq_start) {
    const int64_t s64 = a.seq_start[b];
    seq = (int)(s64 < 0 ? 0 : (s64 > a.N ? a.N : s64));
  }
  const bool empty = (a.N - a.M + m) < seq;
  const float inv = empty ? 0.f : 1.0f / l;
  uint16_t* op = const_cast<uint16_t*>(a.o.ptr) + b * a.o.sb + h * a.o.sh + (int64_t)m * a.o.st + d;
  u32x2 w;
  w[0] = Tr::pack2(acc[0] * inv, acc[1] * inv);
  w[1] = Tr::pack2(acc[2] * inv, acc[3] * inv);
  *reinterpret_cast<u32x2*>(op) = w;
  if (d == 0) a.lse[row] = empty ? -INFINITY : mx * kLn2 + __logf(l);
}

// Query tiles per (batch, head) up to which the forward's K and V tile loads may carry the non-temporal hint
// (FwdK::stream asks for it).
constexpr int kStreamMaxQueryTiles = 1;

// explicit instantiations: every (dtype, head dim) pair the dispatcher can reach
#define FOX_INSTANTIATE_FWD(TR)                                          \
  template __global__ void fwd_kernel<TR, 16, false>(const FwdK);        \
  template __global__ void fwd_kernel<TR, 32, false>(const FwdK);        \
  template __global__ void fwd_kernel<TR, 64, false>(const FwdK);        \
  template __global__ void fwd_kernel<TR, 128, false>(const FwdK);       \
  template __global__ void fwd_kernel<TR, 16, false, true>(const FwdK);  \
  template __global__ void fwd_kernel<TR, 32, false, true>(const FwdK);  \
  template __global__ void fwd_kernel<TR, 64, false, true>(const FwdK);  \
  template __global__ void fwd_kernel<TR, 128, false, true>(const FwdK); \
  template __global__ void fwd_kernel<TR, 16, true>(const FwdK);         \
  template __global__ void fwd_kernel<TR, 32, true>(const FwdK);         \
  template __global__ void fwd_kernel<TR, 64, true>(const FwdK);         \
  template __global__ void fwd_kernel<TR, 128, true>(const FwdK);        \
  template __global__ void fwd_kernel<TR, 16, false, false, true>(const FwdK);  \
  template __global__ void fwd_kernel<TR, 32, false, false, true>(const FwdK);  \
  template __global__ void fwd_kernel<TR, 64, false, false, true>(const FwdK);  \
  template __global__ void fwd_kernel<TR, 128, false, false, true>(const FwdK); \
  template __global__ void fwd_kernel<TR, 16, true, false, true>(const FwdK);   \
  template __global__ void fwd_kernel<TR, 32, true, false, true>(const FwdK);   \
  template __global__ void fwd_kernel<TR, 64, true, false, true>(const FwdK);   \
  template __global__ void fwd_kernel<TR, 128, true, false, true>(const FwdK);  \
  template __global__ void fwd_pair_kernel<TR, 32, false>(const FwdK);   \
  template __global__ void fwd_pair_kernel<TR, 64, false>(const FwdK);   \
  template __global__ void fwd_pair_kernel<TR, 128, false>(const FwdK);  \
  template __global__ void fwd_pair_kernel<TR, 32, true>(const FwdK);    \
  template __global__ void fwd_pair_kernel<TR, 64, true>(const FwdK);    \
  template __global__ void fwd_pair_kernel<TR, 128, true>(const FwdK);   \
  template __global__ void fwd_scan_kernel<TR, 16, false>(const FwdK);   \
  template __global__ void fwd_scan_kernel<TR, 32, false>(const FwdK);   \
  template __global__ void fwd_scan_kernel<TR, 64, false>(const FwdK);   \
  template __global__ void fwd_scan_kernel<TR, 128, false>(const FwdK);  \
  template __global__ void fwd_scan_kernel<TR, 16, true>(const FwdK);    \
  template __global__ void fwd_scan_kernel<TR, 32, true>(const FwdK);    \
  template __global__ void fwd_scan_kernel<TR, 64, true>(const FwdK);    \
  template __global__ void fwd_scan_kernel<TR, 128, true>(const FwdK);   \
  template __global__ void fwd_scan_pair_kernel<TR, 32, false>(const FwdK);  \
  template __global__ void fwd_scan_pair_kernel<TR, 64, false>(const FwdK);  \
  template __global__ void fwd_scan_pair_kernel<TR, 128, false>(const FwdK); \
  template __global__ void fwd_scan_pair_kernel<TR, 32, true>(const FwdK);   \
  template __global__ void fwd_scan_pair_kernel<TR, 64, true>(const FwdK);   \
  template __global__ void fwd_scan_pair_kernel<TR, 128, true>(const FwdK);
#define FOX_INSTANTIATE_COMBINE(TR, U)                         \
  template __global__ void combine_kernel<TR, 16, U>(const FwdK); \
  template __global__ void combine_kernel<TR, 32, U>(const FwdK); \
  template __global__ void combine_kernel<TR, 64, U>(const FwdK); \
  template __global__ void combine_kernel<TR, 128, U>(const FwdK);
#define FOX_INSTANTIATE_COMBINES(TR) \
  FOX_INSTANTIATE_COMBINE(TR, 2) FOX_INSTANTIATE_COMBINE(TR, 3) FOX_INSTANTIATE_COMBINE(TR, 4) FOX_INSTANTIATE_COMBINE(TR, 6) FOX_INSTANTIATE_COMBINE(TR, 8)
FOX_INSTANTIATE_FWD(Bf16)
FOX_INSTANTIATE_FWD(Fp16)
FOX_INSTANTIATE_COMBINES(Bf16)
FOX_INSTANTIATE_COMBINES(Fp16)

template <typename Tr, int D>
static hipError_t launch_fwd_d(const FwdK& a, int dtype, hipStream_t s) {
  if (a.epi.y.ptr && (a.M == 1 || a.splits > 1)) return hipErrorInvalidValue;  // the epilogue lives in the unsplit kernel only
  const bool stream = a.stream && a.n_mtiles <= kStreamMaxQueryTiles;
  if (a.M == 1) {  // decode step: the streaming kernel, one workgroup per (batch, head, key split)
    const hipError_t e = launch_fwd_decode(a, D, dtype, s);
    if (e != hipSuccess || a.splits <= 1) return e;
  } else if (a.splits <= 1) {
    const dim3 grid((unsigned)(a.n_mtiles * a.B * a.H));
    if constexpr (D >= 32) {
      if (a.pair) {   // (two query tiles at least: never a streaming shape)
        if (a.epi.y.ptr) hipLaunchKernelGGL((fwd_pair_kernel<Tr, D, true>), grid, dim3(512), 0, s, a);
        else hipLaunchKernelGGL((fwd_pair_kernel<Tr, D, false>), grid, dim3(512), 0, s, a);
        return hipGetLastError();
      }
    }
    if (a.epi.y.ptr) hipLaunchKernelGGL((fwd_kernel<Tr, D, false, true>), grid, dim3(256), 0, s, a);
    else if (stream) hipLaunchKernelGGL((fwd_kernel<Tr, D, false, false, true>), grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((fwd_kernel<Tr, D, false>), grid, dim3(256), 0, s, a);
    return hipGetLastError();
  } else {
    const dim3 grid((unsigned)(a.n_mtiles * a.splits * a.B * a.H));
    if (stream) hipLaunchKernelGGL((fwd_kernel<Tr, D, true, false, true>), grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((fwd_kernel<Tr, D, true>), grid, dim3(256), 0, s, a);
  }
  const int64_t threads = (int64_t)a.B * a.H * a.M * (D / 4);
  const dim3 rows((unsigned)((threads + 255) / 256));
  switch (a.splits) {
    case 2: hipLaunchKernelGGL((combine_kernel<Tr, D, 2>), rows, dim3(256), 0, s, a); break;
    case 3: hipLaunchKernelGGL((combine_kernel<Tr, D, 3>), rows, dim3(256), 0, s, a); break;
    case 4: hipLaunchKernelGGL((combine_kernel<Tr, D, 4>), rows, dim3(256), 0, s, a); break;
    case 5: case 6: hipLaunchKernelGGL((combine_kernel<Tr, D, 6>), rows, dim3(256), 0, s, a); break;
    default: hipLaunchKernelGGL((combine_kernel<Tr, D, 8>), rows, dim3(256), 0, s, a);
  }
  return hipGetLastError();
}

template <typename Tr, int D>
static hipError_t launch_fwd_gates_d(const FwdK& a, hipStream_t s) {
  if (a.M == 1 || a.splits > 1 || a.N > kOwnScanMaxKeys) return hipErrorInvalidValue;
  const dim3 grid((unsigned)(a.n_mtiles * a.B * a.H));
  if constexpr (D >= 32) {
    if (a.pair) {
      if (a.epi.y.ptr) hipLaunchKernelGGL((fwd_scan_pair_kernel<Tr, D, true>), grid, dim3(512), 0, s, a);
      else hipLaunchKernelGGL((fwd_scan_pair_kernel<Tr, D, false>), grid, dim3(512), 0, s, a);
      return hipGetLastError();
    }
  }
  if (a.epi.y.ptr) hipLaunchKernelGGL((fwd_scan_kernel<Tr, D, true>), grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL((fwd_scan_kernel<Tr, D, false>), grid, dim3(256), 0, s, a);
  return hipGetLastError();
}
template <typename Tr>
static hipError_t launch_fwd_gates_t(const FwdK& a, int D, hipStream_t s) {
  switch (D) {
    case 16: return launch_fwd_gates_d<Tr, 16>(a, s);
    case 32: return launch_fwd_gates_d<Tr, 32>(a, s);
    case 64: return launch_fwd_gates_d<Tr, 64>(a, s);
    case 128: return launch_fwd_gates_d<Tr, 128>(a, s);
    default: return hipErrorInvalidValue;
  }
}

template <typename Tr>
static hipError_t launch_fwd_t(const FwdK& a, int D, int dtype, hipStream_t s) {
  switch (D) {
    case 16: return launch_fwd_d<Tr, 16>(a, dtype, s);
    case 32: return launch_fwd_d<Tr, 32>(a, dtype, s);
    case 64: return launch_fwd_d<Tr, 64>(a, dtype, s);
    case 128: return launch_fwd_d<Tr, 128>(a, dtype, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_fwd(const FwdK& a, int D, int dtype, hipStream_t s) {
  return dtype == 0 ? launch_fwd_t<Bf16>(a, D, dtype, s) : launch_fwd_t<Fp16>(a, D, dtype, s);
}

hipError_t launch_fwd_gates(const FwdK& a, int D, int dtype, hipStream_t s) {
  return dtype == 0 ? launch_fwd_gates_t<Bf16>(a, D, s) : launch_fwd_gates_t<Fp16>(a, D, s);
}

// What fox_attn_fwd_gates accepts.
bool fwd_can_scan(int B, int H, int M, int N, int splits) {
  const int64_t wgs = (int64_t)((M + kFwdBM - 1) / kFwdBM) * B * H;
  return M > 1 && splits <= 1 && N <= kOwnScanMaxKeys && wgs <= (N <= 1024 ? 4 : 2) * kCus;
}

// Whether the forward forms the cumulative sums itself (fwd_scan_kernel) instead of reading what a scan left.  The scan is a launch and
// 3 to 6 us of one workgroup per row; own sums cost a workgroup 1 to 2 us, most of it while its first tiles arrive, but every workgroup.
// Forward with its scan / with own sums, us, on inputs that the caches hold; on fresh ones the gates of (B, T, H) memory, a line per token and workgroup,
// come from further away and the longest rows gain nothing (B1 T3001 H16 D128).
// - Resident grids (up to two workgroups per CU): B16 H16 N250 D64 12.5 / 10.4, B4 H32 N500 16.1 / 14.6, B2 H12 N2048 D128 43.6 / 42.4, B1 H16 N3500 66.4 / 64.3,
//   at -10 B2 H32 N1000 D64 17.4 / 15.5, B1 H16 N3500 18.8 / 16.6.  Without a threshold the walks of head dims up to 64 hide little of it; they lose on long rows of many
//   heads: B1 H32 N1900 D16 28.9 / 30.2, D32 30.3 / 31.6, D64 33.9 / 34.6 (H16 N2048 24.3 / 24.1, 25.6 / 24.9, 29.0 / 28.7).
// - Fewer queries than keys: every query tile of a pair repeats almost the whole row, B8 H32 M130 N3500 D64 at -10 23.7 / 25.9, M400 B4 22.6 / 24.6, M130 N1600 18.6 /
//   19.2.  The line lies at 2900 keys summed up per CU (B8 H32 M130 N1200 17.9 / 17.8); a pair's only tile repeats nothing
//   (B16 H32 M128 N3500 34.0 / 28.4).
// - Up to four workgroups per CU: short rows, at -10 B4 H32 N1000 D64 25.1 / 24.2, without a threshold up to 3.5 (B4 H28 N1000 30.8 / 29.5, B4 H32 N1000 34.3 / 35.5, B8 H32
//   N500 25.1 / 25.7) or very short ones (B16 H32 N256 20.5 / 20.0, D128 31.3 / 30.2; D128 B8 H24 N500 31.6 / 32.8).  Not long ones (B4 H16 N1500 D128 55.8 / 55.8).
// - Beyond that every round repeats the sums: B8 H12 N2048 D64 70.6 / 71.4, B16 H16 N3500 475 / 499.
bool fwd_scans(int B, int H, int M, int N, int D, bool pruned, int splits) {
  const int64_t pairs = (int64_t)B * H, tiles = (M + kFwdBM - 1) / kFwdBM, wgs = tiles * pairs;
  if (!fwd_can_scan(B, H, M, N, splits)) return false;
  if (tiles > 1 && M < N && wgs * (2 * (int64_t)N - M) > 2 * 2900 * kCus) return false;
  if (wgs <= 2 * kCus) return pruned || D > 64 || N <= 1024 || 4 * wgs <= 5 * kCus || pairs < 24;
  return pruned || N <= 384 || (D <= 64 && 2 * wgs <= 7 * kCus);
}

// Whether the forward takes the paired variant (fwd_pair_kernel): less than two query tiles per CU under a causal triangle, where the
// heaviest tile's walk sets the time.  Measured forward with its scan, us, one group / paired.
// - Unsplit grids beyond one tile per CU lose a little throughput (the merge, one workgroup's start and end with nothing beside it)
//   and gain the tail: worth it from a walk of 16 keys per tile beyond one per CU on.  D 64: 280 tiles N1200 26.0 / 21.8, 322 tiles N2900
//   49.4 / 39.9, 384 tiles N1024 23.3 / 24.1, N3001 48.6 / 39.5.  D 128: 280 tiles N1200 32.3 / 29.1, 384 tiles N1024 31.2 / 34.4, N2048
//   50.2 / 47.3, N3001 67.7 / 57.6.  Two full tiles per CU are balanced by the folded order (D 128 N2048 55.9 / 59.2, N4096 94.1 / 91.7),
//   more make no tail that matters (768 tiles N4096 121 / 129).
// - Smaller grids with fewer keys than are split: from 512 keys on.  D 64: N300 11.6 / 12.0, N512 15.6 / 14.5, N777 19.3 / 17.1.
// - Two key splits cost a pass over fp32 partials and a merge launch, which pays for longer walks only.  D 128 and 64: B2 H12 N1024
//   33.2 / 25.3 and 24.6 / 19.4, B1 H16 N2048 44.3 / 38.2 and 34.3 / 29.3, B1 H10 N2900 53.4 / 55.1 and 38.2 / 39.0.
// - Under a pruning threshold the walks are short whatever the shape; head dim 16 has no room to hand the accumulators over.
bool fwd_pairs(int B, int H, int M, int N, int D, bool pruned, int splits) {
  const int64_t wgs = (int64_t)((M + kFwdBM - 1) / kFwdBM) * B * H;
  if (D < 32 || pruned || even_tiles(M, N) || wgs >= 2 * kCus || N < 512) return false;
  if (splits > 1) return splits == 2 && N <= 2560;
  return N >= 16 * (wgs - kCus);
}

// Number of key splits the forward uses for a shape: 1 unless the grid of query tiles
// alone leaves most of the chip idle while each workgroup has a long key loop (chunked
// prefill, decode).  Splits are sized to give every CU at most two workgroups: one workgroup more would
// run in a second round of its own (B2 H16 M333 N5333 D128: six splits, 576 workgroups, 60 us; five, 480, 50 us).  Between one
// and two tiles per CU, tiles of equal weight are halved (the two rounds then even out what a CU with two tiles and one with a single
// tile differ by); under a causal triangle the folded launch order evens that out already.  Head dims up to 64 hold three workgroups on a CU
// (kFwdWaves): where two splits leave some CUs with a single one, three fill them (B8 H8 M333 N12000 D32 two / three splits 107 / 95 us, N3000 37.9 / 36.5;
// causal B1 H5 T5333 D64 50.5 / 45.0), but for the causal grids of up to 2560 keys that the paired kernel takes.  The streaming
// kernel of the single-query case keeps no tile in LDS and takes about eight per CU, at
// least 512 keys each.
int fwd_key_splits(int B, int H, int M, int N, int D) {
  if (M == 1) {
    const int64_t bh = (int64_t)B * H;
    int64_t splits = (2048 + bh - 1) / bh;
    splits = splits > N / 512 ? N / 512 : splits;
    splits = splits > 64 ? 64 : splits;
    return splits < 1 ? 1 : (int)splits;
  }
  const int64_t wgs = (int64_t)((M + kFwdBM - 1) / kFwdBM) * B * H;
  const int key_tiles = (N + kFwdBN - 1) / kFwdBN;
  if (wgs >= 2 * kCus || key_tiles < 16) return 1;
  int splits = wgs > kCus && even_tiles(M, N) ? 2 : (int)(2 * kCus / wgs);
  if (D <= 64 && splits == 2 && wgs < kCus && (even_tiles(M, N) || N > 2560)) splits = 3;
  splits = splits > key_tiles / 8 ? key_tiles / 8 : splits;
  splits = splits > 32 ? 32 : splits;
  return splits < 1 ? 1 : splits;
}

}  // namespace fox
