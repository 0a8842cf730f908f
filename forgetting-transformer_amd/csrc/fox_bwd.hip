// Backward kernels of Forgetting Attention for gfx950.
//
//   dq_kernel    : one workgroup keeps 128 query rows (Q, dO in registers) and
//                  walks the key tiles like the forward; computes delta_i =
//                  sum_d o_id * do_id for its rows on the way in, writes dq,
//                  delta and the row sums drow[i] = sum_j dS[i,j].
//   dkdv_kernel  : runs after it.  One workgroup keeps 128 key rows (K, V in
//                  registers as MFMA B operands; dK^T, dV^T accumulators) and
//                  walks the query tiles below its diagonal; writes dk, dv and
//                  dc[n] = drow[n - (N - M)] - sum_i dS[i,n].
//   dq_kernel with BOTH : the workgroups of either kind in one launch, for small
//                  grids (bwd_together); dc then lacks drow, which the reverse
//                  scan behind it adds (fox_scan.hip).
//   delta_kernel : delta alone (a stage of its own for callers that want it;
//                  the backward does not launch it).
// Every kernel here only stores: no read-modify-write of anything another kernel wrote,
// so a stage may be repeated or timed alone without changing the result.
//
// Probabilities are rebuilt from the stored log-normaliser:
//   P = exp2( (q.k)*sm_scale*log2e + rowc_i - colc_j ),
//   rowc_i = (c_i - c_ref - lse_i)*log2e   (-inf for rows past M or empty rows),
//   colc_j = (c_j - c_ref)*log2e           (+inf left of seq_start or past N),
// so row/column validity costs nothing in the loop; only tiles that cross the
// diagonal run the causal compare.  In every kernel the first MFMA leaves each
// lane with one index of the dimension that stays free in the second MFMA, so the
// recomputed P / dS feed the second MFMA straight from registers.
#include "fox_common.hpp"
#include "fox_kernels.hpp"

namespace fox {

// ---------------------------------------------------------------------------
template <typename Tr, int D>
__global__ __launch_bounds__(256) void delta_kernel(const BwdK a) {
  constexpr int LPR = D / 8;          // lanes per row
  constexpr int RPP = 256 / LPR;      // rows per pass
  constexpr int ROWS = 128;           // rows per workgroup
  const int tid = threadIdx.x;
  const int bh = blockIdx.y, b = bh / a.H, h = bh % a.H;
  const uint16_t* op = a.o.ptr + b * a.o.sb + h * a.o.sh;
  const uint16_t* dop = a.d_o.ptr + b * a.d_o.sb + h * a.d_o.sh;
  const int ch = tid % LPR;
  // every load of the workgroup's rows is requested before the first one is used (rows past the end repeat the last row)
  constexpr int NP = ROWS / RPP;
  u32x4 x[NP], y[NP];
#pragma unroll
  for (int pass = 0; pass < NP; ++pass) {
    const int m = min(blockIdx.x * ROWS + pass * RPP + tid / LPR, a.M - 1);
    x[pass] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(op + (int64_t)m * a.o.st + ch * 8));
    y[pass] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(dop + (int64_t)m * a.d_o.st + ch * 8));
  }
#pragma unroll
  for (int pass = 0; pass < NP; ++pass) {
    const int m = blockIdx.x * ROWS + pass * RPP + tid / LPR;
    float acc = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) acc += Tr::lo(x[pass][e]) * Tr::lo(y[pass][e]) + Tr::hi(x[pass][e]) * Tr::hi(y[pass][e]);
#pragma unroll
    for (int off = LPR / 2; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
    if (m < a.M && ch == 0) a.delta[(int64_t)bh * a.M + m] = acc;
  }
}

// ---------------------------------------------------------------------------
// One step (BMQ query rows) of the dK/dV kernel for one wave (32 key rows).
// rc_s holds rowc_i / (sm_scale*log2e) and dl_s holds -delta_i.  The wave accumulates the NDB 32-column
// blocks of dK and dV that start at block db0 (all of them, or one half of the head dim when two waves
// share a block of keys).
template <typename Tr, int D, int BMQ = kKvBM, int NDB = (D + 31) / 32>
__device__ __forceinline__ void dkdv_step(const char* q_tile, const char* do_tile, const float* rc_s, const float* dl_s,
                                 const u32x4 (&kreg)[D / 16], const u32x4 (&vreg)[D / 16], f32x16 (&dkacc)[NDB],
                                 f32x16 (&dvacc)[NDB], float& csum, int a_s0, int n, int n_w0, float qk_scale,
                                 float colc, int lane, int db0 = 0) {
  constexpr int KK = D / 16, MB = BMQ / 32;
  const int g = lane >> 5, i = lane & 31;
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int a_b0 = a_s0 + 32 * mb;   // key position of the block's first query row
    if (a_b0 + 31 < n_w0) continue;    // block entirely above the diagonal for this wave
    f32x16 s = acc_init(rc_s, 32 * mb, g), dp = acc_init(dl_s, 32 * mb, g);
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) s = Tr::mfma32(lds_row_operand<D>(q_tile, 32 * mb + i, 2 * kk + g), kreg[kk], s);
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) dp = Tr::mfma32(lds_row_operand<D>(do_tile, 32 * mb + i, 2 * kk + g), vreg[kk], dp);
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = __builtin_amdgcn_exp2f(fmaf(s[r], qk_scale, -colc));
    if (a_b0 < n_w0 + 31) {  // causal compare, only on blocks that cross the diagonal
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = (n > a_b0 + c_row(r, g)) ? 0.f : s[r];
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float ds = s[r] * dp[r];
      dp[r] = ds;
      csum += ds;
    }
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      const u32x4 pb = pack8<Tr>(s, 8 * hh);
      const u32x4 dsb = pack8<Tr>(dp, 8 * hh);
#pragma unroll
      for (int db = 0; db < NDB; ++db) {
        dvacc[db] = Tr::mfma32(lds_col_operand<D>(do_tile, 32 * mb + 16 * hh, db0 + db, lane), pb, dvacc[db]);
        dkacc[db] = Tr::mfma32(lds_col_operand<D>(q_tile, 32 * mb + 16 * hh, db0 + db, lane), dsb, dkacc[db]);
      }
    }
  }
}

// Interior step (every query row of the step sits at or below every key of the
// tile: no causal compare, nothing to skip): branch-free and software-pipelined by
// hand, because the kernel holds one wave per SIMD and nobody else can fill the
// matrix pipe while this wave does its exp/scale arithmetic.  The step is cut
// into slots; slot b issues, interleaved in chunks of 4 MFMAs + 2 scores,
//   * the score MFMAs        S, dP   of block b+1,
//   * the vector arithmetic  P, dS   of block b,
//   * the accumulation MFMAs dV, dK  of block b-1,
// which are mutually independent (one MFMA, then a few vector instructions, four times per chunk, in source order
// between scheduling fences).  The global loads of the next tile are spread over
// the step as well (dma(k) issues the k-th of NDMA instructions): issued back to back
// after the barrier by all four waves they would hold every wave's issue slot, and
// with one wave per SIMD the matrix pipe, for over a thousand cycles per step.
// The LDS operands of a chunk are requested three
// chunks (about twelve MFMAs) ahead, across slot boundaries, so their latency hides
// behind the chunks in between.
template <typename Tr, int D, int NDMA, typename Dma>
__device__ __forceinline__ void dkdv_step_interior(const char* q_tile, const char* do_tile, const float* rc_s, const float* dl_s,
                                          const u32x4 (&kreg)[D / 16], const u32x4 (&vreg)[D / 16],
                                          f32x16 (&dkacc)[(D + 31) / 32], f32x16 (&dvacc)[(D + 31) / 32], float& csum,
                                          float qk_scale, float colc, int lane, Dma dma) {
  constexpr int BMQ = kKvBM, KK = D / 16, DB = (D + 31) / 32, MB = BMQ / 32;
  // chunks per slot: as many as the larger of the two MFMA groups needs (one k-step of S and dP, one accumulation
  // pair of dV and dK per chunk), so that every chunk carries matrix work; the 16 scores per lane of a block are
  // dealt out evenly over them
  constexpr int NCH = KK > 2 * DB ? KK : 2 * DB, SPC = 16 / NCH;
  static_assert(16 % NCH == 0 && (SPC == 2 || SPC == 4 || SPC == 8), "whole scores per chunk, whole operands per 8 scores");
  constexpr int NC = (MB + 2) * NCH;  // chunks of the step: slots -1 .. MB
  constexpr int PF = 3;               // LDS operands are requested this many chunks before their MFMAs
  constexpr int kDmaEvery = (NC - NCH) / (NDMA > 0 ? NDMA : 1) > 0 ? (NC - NCH) / (NDMA > 0 ? NDMA : 1) : 1;
  static_assert(NDMA * kDmaEvery <= NC - NCH, "every load instruction of the next tile finds a chunk");
  static_assert(KK <= NCH && 2 * DB <= NCH, "one k-step and one accumulation pair per chunk");
  const int g = lane >> 5, i = lane & 31;
  f32x16 s[MB], dp[MB];
  u32x4 pb[MB][2], dsb[MB][2];
  u32x4 aq[NC + PF], ado[NC + PF], cq[NC + PF], cdo[NC + PF];  // indexed by chunk; only a few are live at a time
  auto fetch = [&](auto ic) {
    constexpr int c = decltype(ic)::value;
    constexpr int slot = c / NCH - 1, u = c % NCH, bs = slot + 1, bc = slot - 1;
    if constexpr (c < NC && bs < MB && u < KK) {
      aq[c] = lds_row_operand<D>(q_tile, 32 * bs + i, 2 * u + g);
      ado[c] = lds_row_operand<D>(do_tile, 32 * bs + i, 2 * u + g);
    }
    if constexpr (c < NC && slot >= 1 && u < 2 * DB) {
      cdo[c] = lds_col_operand<D>(do_tile, 32 * bc + 16 * (u / DB), u % DB, lane);
      cq[c] = lds_col_operand<D>(q_tile, 32 * bc + 16 * (u / DB), u % DB, lane);
    }
  };
  // the accumulators of block b start from the row terms instead of zero; requested PF chunks early too
  auto init_block = [&](int b) {  // b is a constant at every call site
    if (b < MB) {
      s[b] = acc_init(rc_s, 32 * b, g);
      dp[b] = acc_init(dl_s, 32 * b, g);
    }
  };
  init_block(0);
  static_for<0, PF>([&](auto ic) { fetch(ic); });
  static_for<0, NC>([&](auto ic) {
    constexpr int c = decltype(ic)::value;
    constexpr int slot = c / NCH - 1, u = c % NCH;
    constexpr bool do_s = slot + 1 < MB, do_v = slot >= 0 && slot < MB, do_c = slot >= 1;
    constexpr int bs = slot + 1, bv = slot, bc = slot - 1;
    fetch(std::integral_constant<int, c + PF>{});
    if constexpr (u == (NCH > PF ? NCH - PF : 0)) init_block(bs + 1);
    // the next tile's load instructions, one every kDmaEvery chunks from the second slot on
    if constexpr (c >= NCH && (c - NCH) % kDmaEvery == 0 && (c - NCH) / kDmaEvery < NDMA)
      dma(std::integral_constant<int, (c - NCH) / kDmaEvery>{});
    // The chunk in issue order, every group fenced so that matrix and vector instructions alternate: S MFMA, exp2 of
    // SPC scores, dP MFMA, dS and the column sum of those scores, dV MFMA, pack P (when eight scores are complete),
    // dK MFMA, pack dS.  S and dP accumulate in VGPRs (mfma32_vgpr_acc), so this code keeps the distance between an
    // MFMA that writes s[b] / dp[b] and the first vector instruction that reads them (12 issued instructions).  Block
    // b's last S MFMA opens chunk NCH-1 of slot b-1 and its first score is read in chunk 0 of slot b, after that
    // chunk's S MFMA.  For b >= 1 the instructions in between are the 2*SPC exp2 / fma, the dP MFMA, the 2*SPC multiply
    // / add and the 8 packs of chunk NCH-1 (it completes eight scores), then the next chunk's operand requests and
    // S MFMA: >= 20.  dP's last MFMA is followed by 2*SPC + 8 of those, the requests, the S MFMA and 2*SPC exp2 / fma
    // before dS reads it: >= 18.  Block 0 is computed in a slot without vector work, so its first chunk of vector
    // work starts with explicit wait states.
    constexpr bool mf_s = do_s && u < KK, mf_c = do_c && u < 2 * DB;
    constexpr bool pack_due = do_v && (SPC * (u + 1)) % 8 == 0;   // eight scores complete: one MFMA operand each of P and dS
    constexpr int hh = pack_due ? SPC * (u + 1) / 8 - 1 : 0;
    static_assert(SPC >= 2 && NCH * SPC == 16, "the distances above count on at least two scores per chunk, eight per pack");
    if constexpr (mf_s) Tr::mfma32_vgpr_acc(s[bs], aq[c], kreg[u]);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (do_v && bv == 0 && u == 0) {
      asm volatile("s_nop 11");
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (do_v) {
#pragma unroll
      for (int e = 0; e < SPC; ++e) s[bv][SPC * u + e] = __builtin_amdgcn_exp2f(fmaf(s[bv][SPC * u + e], qk_scale, -colc));
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (mf_s) Tr::mfma32_vgpr_acc(dp[bs], ado[c], vreg[u]);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (do_v) {
#pragma unroll
      for (int e = 0; e < SPC; ++e) {
        const float ds = s[bv][SPC * u + e] * dp[bv][SPC * u + e];
        dp[bv][SPC * u + e] = ds;
        csum += ds;
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (mf_c) dvacc[u % DB] = Tr::mfma32(cdo[c], pb[bc][u / DB], dvacc[u % DB]);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (pack_due) pb[bv][hh] = pack8<Tr>(s[bv], 8 * hh);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (mf_c) dkacc[u % DB] = Tr::mfma32(cq[c], dsb[bc][u / DB], dkacc[u % DB]);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (pack_due) dsb[bv][hh] = pack8<Tr>(dp[bv], 8 * hh);
    __builtin_amdgcn_sched_barrier(0);
  });
}

// DSPLIT: the variant for key tiles that pruning leaves a few query steps (class kClassLight).  Such a workgroup
// is a short chain of loads, a few steps and stores; at one workgroup per CU nothing overlaps with it.  Here two
// waves share 32 keys, each recomputing S and dP and accumulating one half of the head dim of dK and dV, so that
// the kernel fits in 256 registers; a workgroup is 64 keys x 2 halves with query steps of 64 rows, and two
// workgroups (two waves per SIMD) share a CU.
//
// OWN_DELTA: the body forms delta = sum_d o_id * do_id for the rows of a step itself instead of reading what the dQ kernel left, so
// that it can run beside it (dq_kernel with BOTH).  A wave takes the rows whose dO it has brought into LDS: its own wait is enough to read
// them, and the barrier that publishes the step's tiles publishes their delta as well.  The sum is the dQ walk's, bit for bit: the gradient of the
// gates is the difference of the row sums of dS there and the column sums here, and is only as good as the two see one delta.

// Two elements' part of delta.  (One expression for both walks, with the rounding spelled out.)
template <typename Tr>
__device__ __forceinline__ float delta_term(uint32_t o, uint32_t d_o) {
  return __builtin_fmaf(Tr::lo(o), Tr::lo(d_o), Tr::hi(o) * Tr::hi(d_o));
}
template <int D, bool DSPLIT>
struct DkdvLds {
  static constexpr int BMQ = DSPLIT ? 64 : kKvBM;
  char *q_tile0, *q_tile1, *do_tile0, *do_tile1;   // Tile<D>::bytes(BMQ) each
  float *rc_s0, *rc_s1, *dl_s0, *dl_s1;            // BMQ each
};
template <typename Tr, int D, bool DSPLIT, bool OWN_DELTA>
__device__ __forceinline__ void dkdv_body(const BwdK& a, int bh, int nt, const DkdvLds<D, DSPLIT>& lds) {
  constexpr int BN = DSPLIT ? 64 : kKvBN, BMQ = DSPLIT ? 64 : kKvBM;
  constexpr int KK = D / 16, DB = (D + 31) / 32, NDB = DSPLIT ? DB / 2 : DB, DW = DSPLIT ? D / 2 : D;
  static_assert(!DSPLIT || DB % 2 == 0, "the head dim splits into two halves of whole 32-column blocks");
  static_assert(!OWN_DELTA || D <= 64, "the long-loop path and the split variant read delta");
  char *q_tile0 = lds.q_tile0, *q_tile1 = lds.q_tile1, *do_tile0 = lds.do_tile0, *do_tile1 = lds.do_tile1;
  float *rc_s0 = lds.rc_s0, *rc_s1 = lds.rc_s1, *dl_s0 = lds.dl_s0, *dl_s1 = lds.dl_s1;

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 5, i = lane & 31;
  const int kb = DSPLIT ? wave >> 1 : wave;   // block of 32 keys this wave owns
  const int dh = DSPLIT ? wave & 1 : 0;       // half of the head dim it accumulates
  const int b = bh / a.H, h = bh % a.H;
  const int M = a.M, N = a.N, p_seq = N - M;
  const int n0 = nt * BN;
  const float* c_row = a.c + (int64_t)bh * N;
  if (a.cls != kClassAll) {  // the class of the 128-key tile this workgroup's keys belong to decides who handles them
    const int n_last = min(N - 1, (n0 / kKvBN) * kKvBN + kKvBN - 1);
    const bool light = acp_light_k(c_row, c_row[n_last], a.thr ? a.thr[bh] : 0.f, n_last, N, a.light_limit);
    if (light != (a.cls == kClassLight)) return;
  }
  const float* lse_row = a.lse + (int64_t)bh * M;
  const float* delta_row = a.delta + (int64_t)bh * M;
  const uint16_t* op = a.o.ptr + b * a.o.sb + h * a.o.sh;   // (read with OWN_DELTA only)
  const uint16_t* qp = a.q.ptr + b * a.q.sb + h * a.q.sh;
  const uint16_t* kp = a.k.ptr + b * a.k.sb + h * a.k.sh;
  const uint16_t* vp = a.v.ptr + b * a.v.sb + h * a.v.sh;
  const uint16_t* dop = a.d_o.ptr + b * a.d_o.sb + h * a.d_o.sh;
  uint16_t* dkp = const_cast<uint16_t*>(a.dk.ptr) + b * a.dk.sb + h * a.dk.sh;
  uint16_t* dvp = const_cast<uint16_t*>(a.dv.ptr) + b * a.dv.sb + h * a.dv.sh;

  int seq = 0;
  if (a.seq_start) {
    const int64_t s64 = a.seq_start[b];
    seq = (int)(s64 < 0 ? 0 : (s64 > N ? N : s64));
  }
  // query range: rows whose key position reaches this tile, up to the pruning bound
  int m_lo = max(n0 - p_seq, 0);
  m_lo = (m_lo / BMQ) * BMQ;
  const int n_w0 = n0 + 32 * kb;
  const int n = n_w0 + i;  // this lane's key row
  // Everything the workgroup needs first is requested before anything is waited for: the tile of the
  // first diagonal step (it does not depend on the pruning bound), K and V, then the per-row terms.
  const DirectTileLoader<D, BMQ> qld(a.q.st, wave, lane), dold(a.d_o.st, wave, lane);
  // The wave's own rows of a step: its j-th load brings one 1 KiB block of the tile, the rows of which the CH lanes of a row read back chunk by
  // chunk; o is fetched in the same shape (whole rows: operand-shaped loads move a quarter of the bytes per clock).
  constexpr int CH = D / 8, OPER = OWN_DELTA ? DirectTileLoader<D, BMQ>::PER : 0, ORPB = Tile<D>::RPB;
  static_assert(!OWN_DELTA || DirectTileLoader<D, BMQ>::NBLK % 4 == 0, "every wave has whole blocks of the step");
  static_assert(!OWN_DELTA || CH <= 16, "the lanes of a row lie in one DPP row");
  const int o_row = wave * ORPB + lane / CH, o_ch = lane % CH;   // of block 0; the j-th block is 4 * ORPB rows further down each
  u32x4 o_raw[OPER > 0 ? OPER : 1];
  auto issue_o = [&](int ms) {
    if constexpr (OWN_DELTA) {
      const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<uint16_t*>(op + (int64_t)ms * a.o.st), 0, dold.extent(a.o.st, ms, M), 0x00020000);
#pragma unroll
      for (int j = 0; j < OPER; ++j)
        o_raw[j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)((o_row + 4 * ORPB * j) * a.o.st * 2) + 16 * o_ch, 0, 0));
    }
  };
  // After the wave's own loads have landed; rows past M are zeros.  The bits of delta are those of the dQ walk: its two halves of the wave add the
  // terms of the even and of the odd chunks of a row one after the other, and the halves are added last.  Here a chunk is a lane, so the running sum
  // goes from lane to lane, two lanes further with every chunk; the last two lanes of the row end up with the two halves.
  auto store_own_delta = [&](const char* dot, float* dl) {
    if constexpr (OWN_DELTA) {
      // Tile<D>::off() within a block, written out, and here: as a call, or as a value of the function above, it changes what the compiler makes of the
      // addresses in dkdv_kernel at head dims 32 and 64, which does not even come here (25 more additions; B3 H16 T1536 at -60 79.3 -> 80.7 us).
      const int o_at = 16 * ((lane & 48) | ((lane & 15) ^ (lane >> 4 << 2)));
#pragma unroll
      for (int j = 0; j < OPER; ++j) {
        const int row = o_row + 4 * ORPB * j;
        const u32x4 x = *reinterpret_cast<const u32x4*>(dot + (wave + 4 * j) * Tile<D>::BLOCK_BYTES + o_at);
        float part = 0.f;
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
          if (kk > 0) part = dpp_take<0x112>(part);   // row_shr 2
#pragma unroll
          for (int e = 0; e < 4; ++e) part += delta_term<Tr>(o_raw[j][e], x[e]);
        }
        part = row_sum<2>(part);
        if (o_ch == CH - 1) dl[row] = -part;
      }
    }
  };
  const bool early = m_lo < M && p_seq + m_lo < n0 + BN - 1 && !(n0 + BN <= seq);
  if (early) {
    qld.issue(qp, a.q.st, m_lo, M, q_tile1);
    dold.issue(dop, a.d_o.st, m_lo, M, do_tile1);
  }
  u32x4 kreg[KK], vreg[KK];
  // The split variant lives for two or three steps, so the way its K and V rows arrive counts: as register loads
  // every instruction touches 32 rows for 32 bytes each; as tile loads they come in whole rows, through buffer set 0
  // (free until the second step), and go from LDS to the registers like any row operand.
  constexpr bool kStageKV = DSPLIT;
  if constexpr (kStageKV) {
    static_assert(BN == BMQ, "the key rows of a workgroup fill one step tile");
    const DirectTileLoader<D, BN> kld(a.k.st, wave, lane), vld(a.v.st, wave, lane);
    kld.issue(kp, a.k.st, n0, N, q_tile0);
    vld.issue(vp, a.v.st, n0, N, do_tile0);
  } else {
    load_row_operand_regs<D>(kreg, kp, a.k.st, n, N, g);
    load_row_operand_regs<D>(vreg, vp, a.v.st, n, N, g);
  }
  const float c_ref = c_row[n0];
  const float c_key = c_row[min(n, N - 1)];
  const float c_last = c_row[min(N - 1, n0 + BN - 1)];  // for the pruning bound below
  float drow_key = 0.f;   // (the split variant is short: the row sum for its dc is requested here, not waited for at the end)
  if constexpr (DSPLIT) drow_key = a.drow[(int64_t)bh * M + min(max(n - p_seq, 0), M - 1)];
  const float qk_scale = nonzero_scale(a.sm_scale * kLog2e), inv_scale = 1.0f / qk_scale;

  // Per-row terms of a step: the loads are requested here, the arithmetic on them is done where the values
  // go to LDS (a step later), so that nothing waits for the loads in between.  Rows past M and empty rows
  // (lse = -inf) get -inf through the subtraction.
  // The BMQ rows of a step are dealt out evenly over the four waves (their first BMQ/4 lanes each), so that
  // no wave arrives late at the barrier because of them.
  const bool row_lane = lane < BMQ / 4;
  const int row_slot = wave * (BMQ / 4) + lane;
  float l_raw = 0.f, c_raw = 0.f, d_raw = 0.f;
  bool row_ok = false;
  auto issue_rows = [&](int ms) {
    if (row_lane) {
      const int mm = ms + row_slot, mc = min(mm, M - 1);
      row_ok = mm < M;
      l_raw = lse_row[mc];
      c_raw = c_row[p_seq + mc];
      if constexpr (!OWN_DELTA) d_raw = delta_row[mc];
    }
  };
  auto rc_term = [&]() {
    const float l_eff = (row_ok & (l_raw > -INFINITY)) ? l_raw : INFINITY;
    return (c_raw - c_ref - l_eff) * kLog2e * inv_scale;
  };
  auto dl_term = [&]() { return row_ok ? -d_raw : 0.f; };
  auto issue = [&](int ms, char* qt, char* dot) {
    issue_rows(ms);  // small loads first: vmcnt retires in order, so they must not queue behind the tile
    qld.issue(qp, a.q.st, ms, M, qt);
    dold.issue(dop, a.d_o.st, ms, M, dot);
    issue_o(ms);
  };
  if (early) {
    issue_rows(m_lo);
    issue_o(m_lo);
  }
  const float colc = (n < N && n >= seq) ? (c_key - c_ref) * kLog2e : INFINITY;

  f32x16 dkacc[NDB], dvacc[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) { dkacc[db][r] = 0.f; dvacc[db][r] = 0.f; }
  float csum = 0.f;


  int m_hi = M;
  if (a.thr) {
    const int U = (M + BMQ - 1) / BMQ;
    const int u = acp_first_pruned_qblock(c_row, c_last, a.thr[bh], p_seq, BMQ, m_lo / BMQ, U, lane);
    m_hi = min(M, u * BMQ);
  }
  if (n0 + BN <= seq) m_hi = m_lo;  // every key of the tile is left padding
  if (a.kv_end_row && tid < BN / kKvUnit && n0 + tid * kKvUnit < N)  // the bound this workgroup works with, for callers that check it
    a.kv_end_row[(int64_t)bh * ((N + kKvUnit - 1) / kKvUnit) + n0 / kKvUnit + tid] = m_hi;
  const int n_steps = m_hi > m_lo ? (m_hi - m_lo + BMQ - 1) / BMQ : 0;
  if constexpr (kStageKV) {
    wait_vmem_all();
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      kreg[kk] = lds_row_operand<D>(q_tile0, 32 * kb + i, 2 * kk + g);
      vreg[kk] = lds_row_operand<D>(do_tile0, 32 * kb + i, 2 * kk + g);
    }
    // (the barrier in front of the first step frees buffer set 0 for the second step's tiles)
  }

  // The long-loop kernel (head dim 128, one workgroup per CU).  Phase 1: the steps that touch the tile's
  // diagonal (at most BN/BMQ + 1 of them) run one at a
  // time through buffer 1 with the masking code; the first interior tile is requested into
  // buffer 0 before the last of them is computed.  Phase 2: interior steps, double-buffered,
  // from the end of the sequence down: the workgroups of one (batch, head) that run together on
  // an XCD then request the same Q / dO tile at about the same time, and all but the first
  // request hit that XCD's L2.
  int n_diag = 0;
  while (n_diag < n_steps && p_seq + m_lo + n_diag * BMQ < n0 + BN - 1) ++n_diag;
  const int n_int = n_steps - n_diag, m_top = m_lo + (n_steps - 1) * BMQ;
  if constexpr (D <= 64 || DSPLIT) {
    // Small head dims (and the split variant) leave room for two workgroups per CU: the second wave on each SIMD
    // fills the matrix pipe while the first does its vector work, so every step takes the plain code path.  The
    // steps, diagonal ones first (upwards from m_lo), then the interior ones (downwards from m_top), alternate
    // between the two buffer sets, starting with set 1 (which the early request above has filled): the next step's
    // tiles are requested before the current one is computed.
    auto step_rows = [&](int idx) { return idx < n_diag ? m_lo + idx * BMQ : m_top - (idx - n_diag) * BMQ; };
    auto store_rows = [&](const char* dot, float* rc, float* dl) {
      if (row_lane) {
        rc[row_slot] = rc_term();
        if constexpr (!OWN_DELTA) dl[row_slot] = dl_term();
      }
      wait_vmem_all();
      if constexpr (OWN_DELTA) {
        __builtin_amdgcn_sched_barrier(0);   // the reads below stay behind the wait
        store_own_delta(dot, dl);
      }
    };
    if (n_steps > 0) {
      if (!early) issue(step_rows(0), q_tile1, do_tile1);
      store_rows(do_tile1, rc_s1, dl_s1);
    }
    for (int idx = 0; idx < n_steps; ++idx) {
      const bool odd = idx & 1;
      __syncthreads();
      if (idx + 1 < n_steps) issue(step_rows(idx + 1), odd ? q_tile1 : q_tile0, odd ? do_tile1 : do_tile0);
      dkdv_step<Tr, D, BMQ, NDB>(odd ? q_tile0 : q_tile1, odd ? do_tile0 : do_tile1, odd ? rc_s0 : rc_s1, odd ? dl_s0 : dl_s1, kreg,
                                 vreg, dkacc, dvacc, csum, p_seq + step_rows(idx), n, n_w0, qk_scale, colc, lane, dh * NDB);
      if (idx + 1 < n_steps) store_rows(odd ? do_tile1 : do_tile0, odd ? rc_s1 : rc_s0, odd ? dl_s1 : dl_s0);
    }
  } else {
  for (int t = 0; t < n_diag; ++t) {
    const int ms = m_lo + t * BMQ;
    if (!(early && t == 0)) {
      __syncthreads();  // buffer 1 is free again
      issue(ms, q_tile1, do_tile1);
    }
    if (row_lane) { rc_s1[row_slot] = rc_term(); dl_s1[row_slot] = dl_term(); }
    wait_vmem_all();
    __syncthreads();
    if (t == n_diag - 1 && n_int > 0) issue(m_top, q_tile0, do_tile0);
    dkdv_step<Tr, D, BMQ, NDB>(q_tile1, do_tile1, rc_s1, dl_s1, kreg, vreg, dkacc, dvacc, csum, p_seq + ms, n, n_w0, qk_scale, colc,
                               lane, dh * NDB);
  }
  if (n_int > 0) {
    if (n_diag == 0) issue(m_top, q_tile0, do_tile0);
    if (row_lane) { rc_s0[row_slot] = rc_term(); dl_s0[row_slot] = dl_term(); }
  }
  constexpr int PER = DirectTileLoader<D, BMQ>::PER;
  // Every tile below the first interior one is a whole tile, so the source of the loads a step spreads over its chunks
  // is a pointer that moves back by one tile per step and an extent that is either a whole tile's or, when there is no
  // next tile, zero (the loads then write zeros into the free buffer): no address arithmetic per step beyond that.
  const int64_t q_back = (int64_t)BMQ * a.q.st, do_back = (int64_t)BMQ * a.d_o.st;
  const int q_whole = qld.extent(a.q.st, 0, BMQ), do_whole = dold.extent(a.d_o.st, 0, BMQ);
  const uint16_t *q_next = qp + (int64_t)(m_top - BMQ) * a.q.st, *do_next = dop + (int64_t)(m_top - BMQ) * a.d_o.st;
  for (int t = 0; t < n_int; t += 2) {
    wait_vmem_all();
    __syncthreads();
    {  // tile t from buffers 0; tile t+1 (if any) into buffers 1
      const bool more = t + 1 < n_int;
      if (more) issue_rows(m_top - (t + 1) * BMQ);
      const int q_bytes = more ? q_whole : 0, do_bytes = more ? do_whole : 0;
      dkdv_step_interior<Tr, D, 2 * PER>(q_tile0, do_tile0, rc_s0, dl_s0, kreg, vreg, dkacc, dvacc, csum, qk_scale, colc, lane, [&](auto k) {
        constexpr int K = decltype(k)::value;
        if constexpr (K < PER) qld.issue_one(K, q_next, q_bytes, q_tile1);
        else dold.issue_one(K - PER, do_next, do_bytes, do_tile1);
      });
      q_next -= q_back;
      do_next -= do_back;
    }
    if (t + 1 >= n_int) break;
    if (row_lane) { rc_s1[row_slot] = rc_term(); dl_s1[row_slot] = dl_term(); }
    wait_vmem_all();
    __syncthreads();
    {
      const bool more = t + 2 < n_int;
      if (more) issue_rows(m_top - (t + 2) * BMQ);
      const int q_bytes = more ? q_whole : 0, do_bytes = more ? do_whole : 0;
      dkdv_step_interior<Tr, D, 2 * PER>(q_tile1, do_tile1, rc_s1, dl_s1, kreg, vreg, dkacc, dvacc, csum, qk_scale, colc, lane, [&](auto k) {
        constexpr int K = decltype(k)::value;
        if constexpr (K < PER) qld.issue_one(K, q_next, q_bytes, q_tile0);
        else dold.issue_one(K - PER, do_next, do_bytes, do_tile0);
      });
      q_next -= q_back;
      do_next -= do_back;
      if (more && row_lane) { rc_s0[row_slot] = rc_term(); dl_s0[row_slot] = dl_term(); }
    }
  }

  }
  wait_vmem_all();  // whatever was requested last (possibly an empty tile) has landed before the buffers are reused
  const float ctot = half_sum(csum);
  // gradient w.r.t. the cumulative sum: the row sum the dQ kernel left for the query row that sits at this key
  // position (none left of the first query row) minus this key's column sum
  if (n < N && g == 0 && dh == 0) {  // (the two waves of a split pair hold the same column sums)
    float rtot = 0.f;   // (beside the dQ walk: the reverse scan adds it)
    if constexpr (!OWN_DELTA) {
      if (n >= p_seq) rtot = DSPLIT ? drow_key : a.drow[(int64_t)bh * M + (n - p_seq)];
    }
    a.dc[(int64_t)bh * N + n] = rtot - ctot;
  }
  // dK and dV leave through LDS (the tile buffers are free now) so that the global stores are whole rows (of the
  // wave's DW columns)
  static_assert(2 * kStoreStageBytes<DW> <= Tile<D>::bytes(BMQ), "two waves stage in one tile buffer");
  __syncthreads();  // every wave is done with the tiles of the last step
  if constexpr (DSPLIT) {   // both at once, a tile buffer per wave: one pass through LDS instead of two
    static_assert(2 * kStoreStageBytes<DW> <= Tile<D>::bytes(BMQ), "a wave stages both in one tile buffer");
    char* stage = wave == 0 ? q_tile0 : wave == 1 ? q_tile1 : wave == 2 ? do_tile0 : do_tile1;
    stage_rows<Tr, DW>(stage, dkacc, a.sm_scale, lane);
    stage_rows<Tr, DW>(stage + kStoreStageBytes<DW>, dvacc, 1.0f, lane);
    staged_rows_visible();
    store_staged_rows<Tr, DW>(stage, dkp + dh * DW, a.dk.st, n_w0, N, lane);
    store_staged_rows<Tr, DW>(stage + kStoreStageBytes<DW>, dvp + dh * DW, a.dv.st, n_w0, N, lane);
  } else {
    char* stage = (wave < 2 ? q_tile0 : do_tile0) + (wave & 1) * kStoreStageBytes<DW>;
    store_rows_via_lds<Tr, DW>(stage, dkacc, a.sm_scale, dkp + dh * DW, a.dk.st, n_w0, N, lane);
    store_rows_via_lds<Tr, DW>(stage, dvacc, 1.0f, dvp + dh * DW, a.dv.st, n_w0, N, lane);
  }
}

template <typename Tr, int D, bool DSPLIT>
__global__ __launch_bounds__(256, (D <= 64 || DSPLIT) ? 2 : 1) void dkdv_kernel(const BwdK a) {
  constexpr int BMQ = DkdvLds<D, DSPLIT>::BMQ;
  __shared__ __align__(16) char q_tile0[Tile<D>::bytes(BMQ)];
  __shared__ __align__(16) char q_tile1[Tile<D>::bytes(BMQ)];
  __shared__ __align__(16) char do_tile0[Tile<D>::bytes(BMQ)];
  __shared__ __align__(16) char do_tile1[Tile<D>::bytes(BMQ)];
  __shared__ __align__(16) float rc_s0[BMQ];
  __shared__ __align__(16) float rc_s1[BMQ];
  __shared__ __align__(16) float dl_s0[BMQ];
  __shared__ __align__(16) float dl_s1[BMQ];
#ifdef __HIP_DEVICE_COMPILE__
  int bh, nt;
  decode_block(block_id(a), a.order, false, bh, nt);
  nt = a.n_tiles - 1 - nt;  // the first key tiles see the most query rows: start them first
  dkdv_body<Tr, D, DSPLIT, false>(a, bh, nt, {q_tile0, q_tile1, do_tile0, do_tile1, rc_s0, rc_s1, dl_s0, dl_s1});
#endif
}

// ---------------------------------------------------------------------------
// One 64-key tile of the dQ kernel for one wave (32 query rows).
// cn_s holds -colc_j / (sm_scale*log2e), the start value of the score accumulators.
template <typename Tr, int D>
__device__ __forceinline__ void dq_tile(const char* k_tile, const char* v_tile, const float* cn_s, const u32x4 (&qreg)[D / 16],
                               const u32x4 (&doreg)[D / 16], f32x16 (&dqacc)[(D + 31) / 32], float& rsum, int n0, int a_m,
                               int a_w0, float qk_scale, float rowc, float delta, int lane) {
  constexpr int BN = kFwdBN, KK = D / 16, DB = (D + 31) / 32, NB = BN / 32;
  const int g = lane >> 5, i = lane & 31;
  // dP starts from -delta (constant along a query row, i.e. per lane) instead of zero: the matrix pipe does the
  // subtraction.  The sixteen equal registers are loop-invariant for the caller.
  f32x16 neg_delta;
#pragma unroll
  for (int r = 0; r < 16; ++r) neg_delta[r] = -delta;
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const int nb0 = n0 + 32 * nb;
    if (nb0 > a_w0 + 31) continue;  // block entirely above this wave's rows
    f32x16 s = acc_init(cn_s, 32 * nb, g);
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) s = Tr::mfma32(lds_row_operand<D>(k_tile, 32 * nb + i, 2 * kk + g), qreg[kk], s);
    f32x16 dp = Tr::mfma32(lds_row_operand<D>(v_tile, 32 * nb + i, g), doreg[0], neg_delta);
#pragma unroll
    for (int kk = 1; kk < KK; ++kk) dp = Tr::mfma32(lds_row_operand<D>(v_tile, 32 * nb + i, 2 * kk + g), doreg[kk], dp);
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = __builtin_amdgcn_exp2f(fmaf(s[r], qk_scale, rowc));
    if (nb0 + 31 > a_w0) {  // causal compare, only on blocks that cross the diagonal
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = (nb0 + c_row(r, g) > a_m) ? 0.f : s[r];
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float ds = s[r] * dp[r];
      dp[r] = ds;
      rsum += ds;
    }
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      const u32x4 dsb = pack8<Tr>(dp, 8 * hh);
#pragma unroll
      for (int db = 0; db < DB; ++db)
        dqacc[db] = Tr::mfma32(lds_col_operand<D>(k_tile, 32 * nb + 16 * hh, db, lane), dsb, dqacc[db]);
    }
  }
}

// The kernel's argument block behind a pointer the compiler cannot see through: each kind of workgroup loads its arguments where it needs
// them (loaded at entry, those of both would not fit the scalar registers).
__device__ __forceinline__ const BwdK& own_arguments() {
  typedef const BwdK __attribute__((address_space(4)))* kernarg;
  kernarg p = (kernarg)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *(const BwdK*)p;
}

// BOTH: dQ and dK/dV in one launch, for small grids of head dims up to 64 (bwd_together): workgroups of either kind side by side, the heaviest of either
// kind first.  One after the other, each of the two kernels waits for its longest walk on a chip that is mostly idle.  (The dQ walk is part of the
// kernel and not a function both kernels call: that way the compiler put eight more waits for LDS into it, 213 instead of 205, and unpruned dQ at D = 128 took 2 to
// 10 % longer: B4 H16 T4096 365 -> 373 us, B8 H3 T3309 111 -> 119, B2 H16 T2048 67 -> 74.)
template <typename Tr, int D, bool BOTH>
__global__ __launch_bounds__(256, 2) void dq_kernel(const BwdK args) {
  constexpr int BM = kFwdBM, BN = kFwdBN, ROWS = BOTH ? kKvBM : kFwdBN;   // rows of a tile buffer: the dK/dV walk needs the larger ones
  constexpr int KK = D / 16, DB = (D + 31) / 32;
  static_assert(!BOTH || (D <= 64 && kKvBM >= kFwdBN), "two workgroups of either kind per CU; the dQ walk fits the buffers of the dK/dV walk");
  __shared__ __align__(16) char k_tile0[Tile<D>::bytes(ROWS)];
  __shared__ __align__(16) char k_tile1[Tile<D>::bytes(ROWS)];
  __shared__ __align__(16) char v_tile0[Tile<D>::bytes(ROWS)];
  __shared__ __align__(16) char v_tile1[Tile<D>::bytes(ROWS)];
  __shared__ __align__(16) float cn_s0[ROWS];
  __shared__ __align__(16) float cn_s1[ROWS];
  int bh, mt;
  if constexpr (BOTH) {
    __shared__ __align__(16) float row2[ROWS];
    __shared__ __align__(16) float row3[ROWS];
    int t;
    decode_block(blockIdx.x, args.order, false, bh, t);
    const BothTile w = both_tile(t, args.n_tiles, (args.M + BM - 1) / BM);
    if (!w.query) {
#ifdef __HIP_DEVICE_COMPILE__
      dkdv_body<Tr, D, false, true>(own_arguments(), bh, w.tile, {k_tile0, k_tile1, v_tile0, v_tile1, cn_s0, cn_s1, row2, row3});
#endif
      return;
    }
    mt = w.tile;
  } else {
    decode_block(block_id(args), args.order, args.last_first, bh, mt);
  }
  const BwdK& a = BOTH ? own_arguments() : args;

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 5, i = lane & 31;
  const int b = divide(bh, a.order.by_heads), h = bh - b * a.H;
  const int M = a.M, N = a.N, p_seq = N - M;
  const int m0 = mt * BM;
  const float* c_row = a.c + (int64_t)bh * N;
  const uint16_t* qp = a.q.ptr + b * a.q.sb + h * a.q.sh;
  const uint16_t* kp = a.k.ptr + b * a.k.sb + h * a.k.sh;
  const uint16_t* vp = a.v.ptr + b * a.v.sb + h * a.v.sh;
  const uint16_t* dop = a.d_o.ptr + b * a.d_o.sb + h * a.d_o.sh;
  const uint16_t* op = a.o.ptr + b * a.o.sb + h * a.o.sh;
  uint16_t* dqp = const_cast<uint16_t*>(a.dq.ptr) + b * a.dq.sb + h * a.dq.sh;

  const int a0 = p_seq + m0;
  const int hi = min(N, a0 + BM);
  int seq = 0;
  if (a.seq_start) {
    const int64_t s64 = a.seq_start[b];
    seq = (int)(s64 < 0 ? 0 : (s64 > N ? N : s64));
  }
  const int m = m0 + 32 * wave + i;
  const int a_m = p_seq + m;
  const int a_w0 = a0 + 32 * wave;
  const float qk_scale = nonzero_scale(a.sm_scale * kLog2e), inv_scale = 1.0f / qk_scale;
  // Everything the workgroup needs first is requested before anything is waited for: the first tile to
  // visit (it does not depend on the pruning bound), Q and dO, then the per-row and per-key terms.
  const DirectTileLoader<D, BN> kld(a.k.st, wave, lane), vld(a.v.st, wave, lane);
  const int n0_first = hi > 0 ? ((hi - 1) / BN) * BN : 0;
  const bool early = hi > (min(seq, hi) / BN) * BN;
  // The tile before it as well, when neither the pruning bound (it never cuts right of the first row's own
  // position) nor seq_start can exclude it: under pruning a workgroup visits two or three tiles, and every round
  // trip taken out of that chain counts.
  const int n0_second = n0_first - BN;
  const bool early2 = early && n0_second >= (a0 / BN) * BN && n0_second >= (min(seq, hi) / BN) * BN;
  if (early) {
    kld.issue(kp, a.k.st, n0_first, N, k_tile0);
    vld.issue(vp, a.v.st, n0_first, N, v_tile0);
  }
  if (early2) {
    kld.issue(kp, a.k.st, n0_second, N, k_tile1);
    vld.issue(vp, a.v.st, n0_second, N, v_tile1);
  }
  u32x4 qreg[KK], doreg[KK], oreg[KK];
  load_row_operand_regs<D>(qreg, qp, a.q.st, m, M, g);
  load_row_operand_regs<D>(doreg, dop, a.d_o.st, m, M, g);
  load_row_operand_regs<D>(oreg, op, a.o.st, m, M, g);
  const float c_ref = c_row[a0];
  const int mc = min(m, M - 1);
  const float l = a.lse[(int64_t)bh * M + mc], c_m = c_row[min(p_seq + mc, N - 1)];

  // Key terms of a tile: the load is requested here, the arithmetic on it is done where the value goes to
  // LDS (a tile later), so that nothing waits for the load in between.  Masked keys get -inf through the
  // subtraction.
  float cn_raw = 0.f;
  bool cn_ok = false;
  auto issue_cn = [&](int n0) {
    if (tid < BN) {
      const int nn = n0 + tid;
      cn_ok = (nn < N) & (nn >= seq);
      cn_raw = c_row[min(nn, N - 1)];
    }
  };
  auto cn_term = [&]() { return (c_ref - (cn_ok ? cn_raw : INFINITY)) * kLog2e * inv_scale; };
  auto issue = [&](int n0, char* kt, char* vt) {
    issue_cn(n0);  // small load first: vmcnt retires in order, so it must not queue behind the tile loads
    kld.issue(kp, a.k.st, n0, N, kt);
    vld.issue(vp, a.v.st, n0, N, vt);
  };
  if (early) issue_cn(n0_first);
  float cn_raw2 = 0.f;   // key terms of the second early tile: handed to cn_raw once the first tile's are in LDS
  bool cn_ok2 = false;
  if (early2 && tid < BN) {
    const int nn = n0_second + tid;
    cn_ok2 = (nn < N) & (nn >= seq);
    cn_raw2 = c_row[min(nn, N - 1)];
  }

  // The pruning bound: its loads are the last to join the ones above, and the search's first wait is the wait for
  // all of them.  Nothing before this point waits for a load: one round trip covers the whole prologue.
  int lo = min(seq, hi);
  if (a.thr) {
    const int t = acp_first_kept_block(c_row, c_ref, a.thr[bh], N, BN, a0 / BN, lane);
    lo = max(lo, t * BN);
  }
  lo = (lo / BN) * BN;
  if (a.q_first_block && tid == 0) a.q_first_block[(int64_t)bh * ((M + BM - 1) / BM) + mt] = lo / BN;
  const int n_tiles = (hi - lo + BN - 1) / BN;

  // rows past M and empty rows (lse = -inf) get rowc = -inf through the subtraction: no load behind a branch
  const float l_eff = ((m < M) & (l > -INFINITY)) ? l : INFINITY;
  const float rowc = (c_m - c_ref - l_eff) * kLog2e;
  // delta_i = sum_d o_id * do_id (_bwd_preprocess of the reference, :902-943) for this lane's row: each half of
  // the wave holds half of the row's elements.  Rows past M were loaded as zeros.  Stored for the dK/dV kernel.
  float delta;
  {
    float part = 0.f;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
#pragma unroll
      for (int e = 0; e < 4; ++e) part += delta_term<Tr>(oreg[kk][e], doreg[kk][e]);
    delta = half_sum(part);
    if (m < M && g == 0) a.delta[(int64_t)bh * M + m] = delta;
  }

  f32x16 dqacc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) dqacc[db][r] = 0.f;
  float rsum = 0.f;

  const bool wave_has_rows = m0 + 32 * wave < M;  // a wave without query rows only moves tiles
  auto compute = [&](int n0, const char* kt, const char* vt, const float* cn) {
    if (!wave_has_rows) return;
    dq_tile<Tr, D>(kt, vt, cn, qreg, doreg, dqacc, rsum, n0, a_m, a_w0, qk_scale, rowc, delta, lane);
  };

  auto tile_n0 = [&](int t) { return lo + t * BN; };   // start of the tile at loop position t
  if (n_tiles > 0) {
    if (!early) issue(tile_n0(n_tiles - 1), k_tile0, v_tile0);
    if (tid < BN) cn_s0[tid] = cn_term();
    if (early2) { cn_raw = cn_raw2; cn_ok = cn_ok2; }
  }
  bool requested = early2;  // buffers 1 already hold (or await) the next tile
  for (int t = n_tiles - 1; t >= 0; t -= 2) {
    wait_vmem_all();
    __syncthreads();
    if (t >= 1 && !requested) issue(tile_n0(t - 1), k_tile1, v_tile1);
    requested = false;
    compute(tile_n0(t), k_tile0, v_tile0, cn_s0);
    if (t < 1) break;
    if (tid < BN) cn_s1[tid] = cn_term();
    wait_vmem_all();
    __syncthreads();
    if (t >= 2) issue(tile_n0(t - 2), k_tile0, v_tile0);
    compute(tile_n0(t - 1), k_tile1, v_tile1, cn_s1);
    if (t >= 2 && tid < BN) cn_s0[tid] = cn_term();
  }

  const float rtot = half_sum(rsum);
  if (m < M && g == 0) a.drow[(int64_t)bh * M + m] = rtot;  // for dc: the dK/dV kernel, next on this stream, adds it, or with BOTH the reverse scan
  // dQ leaves through LDS (the tile buffers are free now, one per wave) so that the global stores are whole rows
  static_assert(kStoreStageBytes<D> <= Tile<D>::bytes(BN), "one wave stages in one tile buffer");
  __syncthreads();  // every wave is done with the last tile
  char* stage = wave == 0 ? k_tile0 : wave == 1 ? k_tile1 : wave == 2 ? v_tile0 : v_tile1;
  store_rows_via_lds<Tr, D>(stage, dqacc, a.sm_scale, dqp, a.dq.st, m0 + 32 * wave, M, lane);
}

// explicit instantiations: every (dtype, head dim) pair the dispatchers can reach
#define FOX_INSTANTIATE_BWD(KERNEL, TR)                      \
  template __global__ void KERNEL<TR, 16>(const BwdK);       \
  template __global__ void KERNEL<TR, 32>(const BwdK);       \
  template __global__ void KERNEL<TR, 64>(const BwdK);       \
  template __global__ void KERNEL<TR, 128>(const BwdK);
FOX_INSTANTIATE_BWD(delta_kernel, Bf16)
FOX_INSTANTIATE_BWD(delta_kernel, Fp16)
#define FOX_INSTANTIATE_DKDV(TR)                                     \
  template __global__ void dkdv_kernel<TR, 16, false>(const BwdK);   \
  template __global__ void dkdv_kernel<TR, 32, false>(const BwdK);   \
  template __global__ void dkdv_kernel<TR, 64, false>(const BwdK);   \
  template __global__ void dkdv_kernel<TR, 128, false>(const BwdK);  \
  template __global__ void dkdv_kernel<TR, 128, true>(const BwdK);
FOX_INSTANTIATE_DKDV(Bf16)
FOX_INSTANTIATE_DKDV(Fp16)
#define FOX_INSTANTIATE_DQ(TR)                                       \
  template __global__ void dq_kernel<TR, 16, false>(const BwdK);     \
  template __global__ void dq_kernel<TR, 32, false>(const BwdK);     \
  template __global__ void dq_kernel<TR, 64, false>(const BwdK);     \
  template __global__ void dq_kernel<TR, 128, false>(const BwdK);    \
  template __global__ void dq_kernel<TR, 16, true>(const BwdK);      \
  template __global__ void dq_kernel<TR, 32, true>(const BwdK);      \
  template __global__ void dq_kernel<TR, 64, true>(const BwdK);
FOX_INSTANTIATE_DQ(Bf16)
FOX_INSTANTIATE_DQ(Fp16)

// ---------------------------------------------------------------------------
#define FOX_DISPATCH_D(KERNEL, GRID, SMEM)                                                        \
  switch (D) {                                                                                    \
    case 16: hipLaunchKernelGGL((KERNEL<Tr, 16>), GRID, dim3(256), SMEM, s, a); break;            \
    case 32: hipLaunchKernelGGL((KERNEL<Tr, 32>), GRID, dim3(256), SMEM, s, a); break;            \
    case 64: hipLaunchKernelGGL((KERNEL<Tr, 64>), GRID, dim3(256), SMEM, s, a); break;            \
    case 128: hipLaunchKernelGGL((KERNEL<Tr, 128>), GRID, dim3(256), SMEM, s, a); break;          \
    default: return hipErrorInvalidValue;                                                         \
  }

template <typename Tr>
static hipError_t delta_t(const BwdK& a, int D, hipStream_t s) {
  const dim3 grid((unsigned)((a.M + 127) / 128), (unsigned)(a.B * a.H));
  FOX_DISPATCH_D(delta_kernel, grid, 0)
  return hipGetLastError();
}
template <typename Tr>
static hipError_t dkdv_t(const BwdK& a0, int D, hipStream_t s) {
  BwdK a = a0;
  const int groups = order_groups(a.B * a.H, (a.N + kKvBN - 1) / kKvBN, a.M, a.N, D, a.k.st, a.thr != nullptr);
  const bool fold = !even_tiles(a.M, a.N) && (D <= 64 || a.cls == kClassLight);   // (two workgroups per CU)
  if (a.cls == kClassLight) {  // the split variant: 64 keys per workgroup
    if (!dkdv_split_supports(D)) return hipErrorInvalidValue;
    a.n_tiles = (a.N + 63) / 64;
    a.order = block_order(a.B, a.H, a.n_tiles, groups, fold);
    hipLaunchKernelGGL((dkdv_kernel<Tr, 128, true>), dim3((unsigned)(a.n_tiles * a.B * a.H)), dim3(256), 0, s, a);
    return hipGetLastError();
  }
  a.n_tiles = (a.N + kKvBN - 1) / kKvBN;
  a.order = block_order(a.B, a.H, a.n_tiles, groups, fold);
  const dim3 grid((unsigned)(a.n_tiles * a.B * a.H));
  switch (D) {
    case 16: hipLaunchKernelGGL((dkdv_kernel<Tr, 16, false>), grid, dim3(256), 0, s, a); break;
    case 32: hipLaunchKernelGGL((dkdv_kernel<Tr, 32, false>), grid, dim3(256), 0, s, a); break;
    case 64: hipLaunchKernelGGL((dkdv_kernel<Tr, 64, false>), grid, dim3(256), 0, s, a); break;
    case 128: hipLaunchKernelGGL((dkdv_kernel<Tr, 128, false>), grid, dim3(256), 0, s, a); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
template <typename Tr>
static hipError_t dq_t(const BwdK& a0, int D, hipStream_t s) {
  BwdK a = a0;
  a.n_tiles = (a.M + kFwdBM - 1) / kFwdBM;
  a.order = block_order(a.B, a.H, a.n_tiles, order_groups(a.B * a.H, a.n_tiles, a.M, a.N, D, a.k.st, a.thr != nullptr), !even_tiles(a.M, a.N));
  // Not under a threshold on a grid that is resident at once: all pairs start together, and where 8 does not divide them the turned order puts each on another
  // XCD than its forward (turned / not, whole step: B1 H12 T4096 D64 at -10 56.5 / 55.5 us, B1 H6 T8192 57.0 / 56.4; without a threshold B1 H1 T16384 D128 804 / 809).
  a.last_first = !a.thr || a.n_tiles * a.B * a.H > 2 * kCus;
  const dim3 grid((unsigned)(a.n_tiles * a.B * a.H));
  switch (D) {
    case 16: hipLaunchKernelGGL((dq_kernel<Tr, 16, false>), grid, dim3(256), 0, s, a); break;
    case 32: hipLaunchKernelGGL((dq_kernel<Tr, 32, false>), grid, dim3(256), 0, s, a); break;
    case 64: hipLaunchKernelGGL((dq_kernel<Tr, 64, false>), grid, dim3(256), 0, s, a); break;
    case 128: hipLaunchKernelGGL((dq_kernel<Tr, 128, false>), grid, dim3(256), 0, s, a); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <typename Tr>
static hipError_t bwd_t(const BwdK& a0, int D, hipStream_t s) {
  BwdK a = a0;
  a.n_tiles = (a.N + kKvBN - 1) / kKvBN;
  const int q_tiles = (a.M + kFwdBM - 1) / kFwdBM, tiles = a.n_tiles + q_tiles;
  // M < N: the query tiles of all pairs first.  Each has the longest walk there is, and with the pairs one after the other those of the next pair would
  // join those of the one before on their CUs.
  const int groups = q_tiles < a.n_tiles ? 1 : order_groups(a.B * a.H, a.n_tiles, a.M, a.N, D, a.k.st, a.thr != nullptr);
  a.order = block_order(a.B, a.H, tiles, groups, !even_tiles(a.M, a.N));
  const dim3 grid((unsigned)(tiles * a.B * a.H));
  switch (D) {
    case 16: hipLaunchKernelGGL((dq_kernel<Tr, 16, true>), grid, dim3(256), 0, s, a); break;
    case 32: hipLaunchKernelGGL((dq_kernel<Tr, 32, true>), grid, dim3(256), 0, s, a); break;
    case 64: hipLaunchKernelGGL((dq_kernel<Tr, 64, true>), grid, dim3(256), 0, s, a); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

bool dkdv_split_supports(int D) { return D == 128; }

hipError_t launch_bwd_delta(const BwdK& a, int D, int dtype, hipStream_t s) {
  return dtype == 0 ? delta_t<Bf16>(a, D, s) : delta_t<Fp16>(a, D, s);
}
hipError_t launch_bwd_dkdv(const BwdK& a, int D, int dtype, hipStream_t s) {
  return dtype == 0 ? dkdv_t<Bf16>(a, D, s) : dkdv_t<Fp16>(a, D, s);
}
// Whether dQ and dK/dV go out as one launch (dq_kernel with BOTH).  One after the other, each waits for the longest walk of a grid that fills the chip
// once or less; side by side the two waits are one, and so are two launches and the drain between them.  Forward and backward, the latter one after the
// other / together, us: D 64 B2 H12 T2048 117 / 98, B4 H12 T512 43.7 / 36.1, B16 H16 T250 42.2 / 41.6, B1 H16 M256 N4096 114 / 106; D 32 B3 H5 T777 49.7 / 38.1,
// D 16 B16 H16 T250 34.2 / 29.3.  Against it stand delta, formed anew for every step, the row sums that the reverse scan has to add, and the LDS of the
// dK/dV walk, which the dQ walk does not need.
// - With more than 512 tiles of either kind at D 64 it goes either way (backward alone, 768: B12 H16 T500 51.2 / 50.3, B16 H24 T250 38.1 / 40.5; 2048: B8 H32
//   T1000 "auto" 87 / 99; 4096: B4 H32 T4096 980 / 1130).  Head dims up to 32 hold three workgroups per CU: 768 tiles B3 H32 T1000 D32 at -10 57.3 / 52.3 and
//   D16 54.9 / 48.5, 2048 tiles B8 H16 T2048 D16, backward alone, 151 / 200.
// - Long rows.  The reverse scan of few long rows is a chain that the row sums make longer, and under a threshold walks are short and have little to overlap,
//   so that the grid has to leave room: D 64 at -10, T4096 with 320 tiles 53.5 / 53.1, 384 55.2 / 56.1, 448 57.3 / 59.1, 512 55.6 / 59.2; T16384 with 256 59.2 / 57.4,
//   384 60.8 / 65.4, 512 68.1 / 76.0; D 32 T16384 with 256 51.7 / 49.3, 512 61.3 / 64.8.  Rows up to 2048 (D 64) and 8192 are past that: B2 H12 T2048 48.5 / 47.7,
//   D 32 B1 H12 T8192 68.0 / 66.8.  Without a threshold D 64 gains until both kinds fill the chip to the last
//   place: 480 tiles B3 H5 T4000 222 / 197, 510 B1 H10 T6500 346 / 311, 504 B1 H8 T8000 405 / 396, 512 B1 H16 T4000 225 / 223 and 226 / 230, H4 T16384 818 / 833; D 32 gains with 768, 805 / 747.
//   Where M < N the tiles of both kinds count: B1 H16 M300 N4096 at -10 (560 of them) 52.4 / 47.7.
bool bwd_together(const BwdK& a, int D) {
  if (D > 64 || a.o.st <= 0 || ((int64_t)kKvBM * a.o.st + D) * 2 >= (int64_t)1 << 31) return false;   // o through 32-bit offsets
  const int64_t pairs = (int64_t)a.B * a.H, keys = pairs * ((a.N + kKvBN - 1) / kKvBN), both = keys + pairs * ((a.M + kFwdBM - 1) / kFwdBM);
  if (keys > (D == 64 ? 2 : 3) * kCus) return false;
  if (a.N <= (D == 64 ? 2048 : 8192)) return true;
  return a.thr ? 2 * both <= 5 * kCus : D < 64 || both < 4 * kCus;
}
hipError_t launch_bwd(const BwdK& a, int D, int dtype, hipStream_t s) {
  return dtype == 0 ? bwd_t<Bf16>(a, D, s) : bwd_t<Fp16>(a, D, s);
}
hipError_t launch_bwd_dq(const BwdK& a, int D, int dtype, hipStream_t s) {
  return dtype == 0 ? dq_t<Bf16>(a, D, s) : dq_t<Fp16>(a, D, s);
}

}  // namespace fox
