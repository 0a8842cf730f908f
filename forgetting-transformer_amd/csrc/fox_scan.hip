// Row scans and the "auto" pruning threshold for gfx950.
//
//   scan_kernel<kForward> : c[n]  = sum_{l<=n} g[l], with g[l] := 0 for l < seq_start
//   scan_kernel<kReverse> : dg[l] = sum_{n>=l} dc[n]
//   gate_scan_fwd/bwd  : the same two scans fused with logsigmoid of the gate logits and its derivative
//   norm_max_kernel    : the "auto" threshold from the largest row L2 norms of q and k.
//
// One workgroup scans one (batch, head) row.  Partial sums are carried in fp64 and
// rounded once on store, so c is exactly non-increasing whenever g <= 0 (the
// pruning bounds rely on that) and long rows lose no precision to the scan order.
#include "fox_common.hpp"
#include "fox_kernels.hpp"

namespace fox {

// The gradient of a cumulative sum at one position is its row sum of dS minus its column sum.  Where the backward ran in one launch the dK/dV walk
// could not wait for the row sums (drow, of the last M positions of the row): the reverse scan adds them, and stores the sum back into dc, which then
// holds what the dK/dV kernel leaves there on its own.  The loads are a loop of their own, without a branch: in a branch per element every one of them was
// waited for before the next was sent (2 rows of 16384 positions 12.5 us, so 11.2, without row sums 8.6; 48 rows of 512 5.1, 4.0 and 4.0).  A variant
// of its own: as a branch at run time it cost the other scans 0.3 to 0.6 us.
struct RowSums {
  static constexpr bool kAny = true;
  const float* drow;   // (M)
  float* dc;
  int p_seq;
  __device__ __forceinline__ float load(int idx) const {
    const float r = drow[max(idx - p_seq, 0)];
    return idx >= p_seq ? r : 0.f;
  }
  __device__ __forceinline__ void keep(int idx, float x) const { dc[idx] = x; }
};
struct NoRows {
  static constexpr bool kAny = false;
  __device__ __forceinline__ float load(int) const { return 0.f; }
  __device__ __forceinline__ void keep(int, float) const {}
};

// Scan of one row: element idx is produced by load(idx) and the running sum up to and including
// it is handed to store(idx, sum).  REVERSE walks the row from its last element to its first.
// A span of PER x NT elements moves between memory and LDS with consecutive lanes on consecutive
// elements (whole cache lines per wave instruction, whatever the caller's stride), and between LDS and
// registers with PER consecutive elements per thread, the order the scan wants.  The totals of the threads meet by DPP (wave_scan): through
// shuffles, twelve trips through LDS one after the other, 12 rows of 4096 took 5.4 / 4.7 us.
// Bound by latency: one workgroup per row, few rows.  A long row gets the widest workgroup there is; a row that a single span of
// fewer waves covers gets just those (scan_threads), and the barriers between sixteen waves and the chain over their totals go.
// Rows of 77 to 2048 elements: 5.1 us a call with 1024 threads, 3.9 with as many as the row needs.  Rows cut over several
// workgroups, each adding up what lies in front of its piece, were slower wherever there were enough of them to count (64 rows of 16384 8.5 -> 10.4
// us, 256 rows of 32768 17 -> 28 us).
// rows: a second addend of the last M positions (RowSums), or nothing.
template <bool REVERSE, int NT, int PER, typename Load, typename Store, typename Rows = NoRows>
__device__ __forceinline__ void scan_row(int N, Load load, Store store, Rows rows = {}) {
  static_assert(PER % 4 == 0);
  constexpr int SPAN = PER * NT, WAVES = NT / kWave;
  __shared__ double wave_tot[WAVES];
  __shared__ __align__(16) float stage[SPAN];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  double carry = 0.0;
  float x[PER], x_next[PER], r[PER], r_next[PER];   // (r: Rows::kAny only)
  auto fetch = [&](int base, float (&dst)[PER], float (&dst_r)[PER]) {  // element e of a thread sits at position base + e*NT + tid of the scan order
    asm volatile("" : "+s"(base));   // (one address after the other: as pointers that a loop moves on they took 32 registers and spilt)
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const int pos = base + e * NT + tid;
      const int idx = REVERSE ? N - 1 - pos : pos;
      dst[e] = pos < N ? load(idx) : 0.f;
    }
    if constexpr (Rows::kAny) {
#pragma unroll
      for (int e = 0; e < PER; ++e) {
        const int pos = base + e * NT + tid, in = min(pos, N - 1);
        const float y = rows.load(REVERSE ? N - 1 - in : in);
        dst_r[e] = pos < N ? y : 0.f;
      }
    }
  };
  fetch(0, x, r);
  for (int base = 0; base < N; base += SPAN) {
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      if constexpr (Rows::kAny) x[e] += r[e];
      stage[e * NT + tid] = x[e];
    }
    if (base + SPAN < N) fetch(base + SPAN, x_next, r_next);   // in flight while this span is scanned
    __syncthreads();
    f32x4* const own = reinterpret_cast<f32x4*>(stage + tid * PER);
    double v[PER];
    double run = 0.0;
#pragma unroll
    for (int i = 0; i < PER / 4; ++i) {
      const f32x4 y = own[i];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[4 * i + e] = run += (double)y[e];
    }
    // inclusive scan of the per-thread totals across the wave, then across waves
    const double incl = wave_scan(run);
    if (lane == kWave - 1) wave_tot[wave] = incl;
    __syncthreads();
    double before = carry, total = 0.0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const double t = wave_tot[w];
      if (w < wave) before += t;
      total += t;
    }
    before += incl - run;
#pragma unroll
    for (int i = 0; i < PER / 4; ++i) {
      f32x4 y;
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = (float)(before + v[4 * i + e]);
      own[i] = y;   // each thread overwrites the values it read
    }
    carry += total;
    __syncthreads();
    int out = base;
    if constexpr (Rows::kAny) asm volatile("" : "+s"(out));   // (as in fetch; the others have the registers for it)
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const int pos = out + e * NT + tid;
      const int idx = REVERSE ? N - 1 - pos : pos;
      if (pos < N) store(idx, stage[e * NT + tid]);
    }
    if constexpr (Rows::kAny) {
#pragma unroll
      for (int e = 0; e < PER; ++e) {
        const int pos = out + e * NT + tid;
        if (pos < N) rows.keep(REVERSE ? N - 1 - pos : pos, x[e]);
      }
    }
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      x[e] = x_next[e];
      if constexpr (Rows::kAny) r[e] = r_next[e];
    }
    __syncthreads();  // the span has left LDS before the next one is written
  }
}

// Row of a workgroup (rows >= `rows`: none).  Workgroups go round-robin over the 8 XCDs, and so do the rows: where 8 divides their number the attention
// kernels put a pair on the same XCD, whose L2 then still holds what the one wrote for the other.  The gate gradients of a batch's heads share cache
// lines when they lie as (B, T, H): with their rows spread every L2 would write its own part of each line, so those go to one XCD as neighbours
// (`neighbours`; reverse scan, spread / neighbours: B4 T4096 H32 10.8 / 7.6 us, B4 T16384 H16 19.0 / 17.0; strided reads of the forward scan do not gain).
__device__ __forceinline__ int scan_row_of_block(int rows, bool neighbours) {
  const int per = (rows + kXcds - 1) / kXcds, id = blockIdx.x;
  return neighbours ? id % kXcds * per + id / kXcds : id;   // (the grid is 8 * per workgroups)
}
inline unsigned scan_blocks(int rows) { return (unsigned)((rows + kXcds - 1) / kXcds * kXcds); }

template <bool ROWS>
__device__ __forceinline__ auto row_sums(const float* drow, float* dc, int bh, int M, int N) {   // of the row of pair bh
  if constexpr (ROWS) return RowSums{drow + (int64_t)bh * M, dc + (int64_t)bh * N, N - M};
  else return NoRows{};
}

inline int scan_threads(int N) { return N <= 8 * 64 ? 64 : N <= 8 * 256 ? 256 : 1024; }
// Whether a thread of the widest workgroup takes sixteen elements of a span in place of eight: rows of more than 8192 positions have half as
// many spans then, each a chain through LDS, the waves' totals and three barriers.  us, eight and shuffles / sixteen and DPP (a row of one span gains 0.3 to 0.7
// from the latter alone): 15 rows of 12242 forward 7.9 / 6.5, reverse 8.1 / 6.8; 64 rows of 16384 8.5 / 6.9 and 9.1 / 7.7; reverse, 64 rows of 32768, 16.0 / 13.3.
// Against it stand the loads of a row's next span, sent while one is scanned.  Eight / sixteen, both by DPP: forward 64 rows of 20000 9.4 / 10.7, 256 rows of
// 32768 14.7 / 15.4, 512 rows of 16384 16.1 / 17.1; reverse 512 rows of 20000 22.2 / 26.2, 16384 18.6 / 18.6.
inline bool scan_deep(int N, int64_t rows, bool reverse) {
  if (N <= 8 * 1024 || N > 1 << 30) return false;   // (the end of a span stays below 2^31: rows up to 2^31 - 8 * 1024 have always been taken)
  return reverse ? rows <= kCus || N <= 16 * 1024 : rows <= kCus && N <= 16 * 1024;
}

enum : int { kForward = 0, kReverse = 1, kReverseRows = 2 };   // kinds of scan_kernel; the last with row sums to add
template <int KIND, int NT, int PER>
__global__ __launch_bounds__(NT) void scan_kernel(const float* in, int64_t sb, int64_t sh, int64_t sn,
                                                   const int64_t* __restrict__ seq_start, float* __restrict__ out, int64_t ob,
                                                   int64_t oh, int64_t on, int rows, int H, int N, const float* __restrict__ drow, int M,
                                                   float* dc) {
  constexpr bool REVERSE = KIND != kForward;
  const int bh = REVERSE ? scan_row_of_block(rows, on != 1) : blockIdx.x, b = bh / H, h = bh % H;
  if (REVERSE && bh >= rows) return;
  const float* src = in + b * sb + h * sh;
  float* dst = out + b * ob + h * oh;
  int seq = 0;
  if (seq_start) {
    const int64_t s64 = seq_start[b];
    seq = (int)(s64 < 0 ? 0 : (s64 > N ? N : s64));
  }
  // Reverse: the gradient of every gate up to and including position seq is the sum of all dc, zero in exact
  // arithmetic (those gates shift every cumulative sum the kernels see by the same amount, or are zeroed by the
  // forward); it is stored as an exact zero instead of the rounding noise of that sum.
  scan_row<REVERSE, NT, PER>(
      N,
      [&](int idx) { return (REVERSE || idx >= seq) ? src[(int64_t)idx * sn] : 0.f; },
      [&](int idx, float sum) { dst[(int64_t)idx * on] = (REVERSE && idx <= seq) ? 0.f : sum; },
      row_sums<KIND == kReverseRows>(drow, dc, bh, M, N));
}

template <int DT>
__device__ __forceinline__ void store_logit(void* p, int64_t i, float x) {
  if constexpr (DT == 2) reinterpret_cast<float*>(p)[i] = x;
  else if constexpr (DT == 0) reinterpret_cast<uint16_t*>(p)[i] = (uint16_t)(Bf16::pack2(x, 0.f) & 0xffffu);
  else reinterpret_cast<uint16_t*>(p)[i] = (uint16_t)(Fp16::pack2(x, 0.f) & 0xffffu);
}

// c[n] = sum_{seq_start <= l <= n} logsigmoid(x[l]) in one pass over the logits; optionally also
// stores log_fgate[n] = logsigmoid(x[n]) (the decode cache of the FoX layer keeps it).
template <int DT, int NT, int PER>
__global__ __launch_bounds__(NT) void gate_scan_fwd_kernel(const void* __restrict__ logits, int64_t sb, int64_t sh, int64_t sn,
                                                            const int64_t* __restrict__ seq_start,
                                                            float* __restrict__ log_fgate, float* __restrict__ out, int H,
                                                            int N) {
  const int bh = blockIdx.x, b = bh / H, h = bh % H;
  const int64_t base = b * sb + h * sh;
  float* dst = out + (int64_t)bh * N;
  float* lg = log_fgate ? log_fgate + (int64_t)bh * N : nullptr;
  int seq = 0;
  if (seq_start) {
    const int64_t s64 = seq_start[b];
    seq = (int)(s64 < 0 ? 0 : (s64 > N ? N : s64));
  }
  scan_row<false, NT, PER>(
      N,
      [&](int idx) {
        const float x = load_logit<DT>(logits, base + (int64_t)idx * sn);
        const float g = log_sigmoid(x);
        if (lg) lg[idx] = g;
        return idx >= seq ? g : 0.f;
      },
      [&](int idx, float sum) { dst[idx] = sum; });
}

// dlogit[l] = (sum_{n>=l} dc[n]) * d logsigmoid(x_l)/dx = dg[l] * (1 - sigmoid(x_l)), stored in the
// dtype and layout of the logits.
constexpr int kRows = 4;   // with row sums to add
template <int DT_ROWS, int NT, int PER>
__global__ __launch_bounds__(NT) void gate_scan_bwd_kernel(float* dc, const void* __restrict__ logits,
                                                            int64_t sb, int64_t sh, int64_t sn, const int64_t* __restrict__ seq_start,
                                                            void* __restrict__ dlogits, int64_t db, int64_t dh, int64_t dn,
                                                            int rows, int H, int N, const float* __restrict__ drow, int M) {
  constexpr int DT = DT_ROWS & 3;
  const int bh = scan_row_of_block(rows, dn != 1), b = bh / H, h = bh % H;
  if (bh >= rows) return;
  const float* src = dc + (int64_t)bh * N;
  const int64_t lbase = b * sb + h * sh, dbase = b * db + h * dh;
  int seq = 0;
  if (seq_start) {
    const int64_t s64 = seq_start[b];
    seq = (int)(s64 < 0 ? 0 : (s64 > N ? N : s64));
  }
  scan_row<true, NT, PER>(
      N, [&](int idx) { return src[idx]; },
      [&](int idx, float sum) {
        const float x = load_logit<DT>(logits, lbase + (int64_t)idx * sn);
        const float z = __expf(-fabsf(x));
        const float r = __fdividef(z, 1.f + z);              // sigmoid(-|x|)
        // positions up to and including seq: an exact zero, as in scan_kernel
        store_logit<DT>(dlogits, dbase + (int64_t)idx * dn, idx <= seq ? 0.f : sum * (x < 0.f ? 1.f - r : r));
      },
      row_sums<(DT_ROWS & kRows) != 0>(drow, dc, bh, M, N));
}

// KERNEL<ARG, threads for rows of N elements>, BLOCKS workgroups, one per row of the B x H.
#define FOX_LAUNCH_SCAN(KERNEL, ARG, REVERSE, BLOCKS, ...)                                                                      \
  switch (scan_threads(N)) {                                                                                                     \
    case 64: hipLaunchKernelGGL((KERNEL<ARG, 64, 8>), dim3(BLOCKS), dim3(64), 0, s, __VA_ARGS__); break;                         \
    case 256: hipLaunchKernelGGL((KERNEL<ARG, 256, 8>), dim3(BLOCKS), dim3(256), 0, s, __VA_ARGS__); break;                      \
    default:                                                                                                                     \
      if (scan_deep(N, (int64_t)B * H, REVERSE)) hipLaunchKernelGGL((KERNEL<ARG, 1024, 16>), dim3(BLOCKS), dim3(1024), 0, s, __VA_ARGS__);                \
      else hipLaunchKernelGGL((KERNEL<ARG, 1024, 8>), dim3(BLOCKS), dim3(1024), 0, s, __VA_ARGS__);                              \
  }

hipError_t launch_gate_cumsum_fwd(const void* logits, int dtype, int64_t sb, int64_t sh, int64_t sn, const int64_t* seq_start,
                                  float* log_fgate, float* c, int B, int H, int N, hipStream_t s) {
  switch (dtype) {
    case 0: FOX_LAUNCH_SCAN(gate_scan_fwd_kernel, 0, false, (unsigned)(B * H), logits, sb, sh, sn, seq_start, log_fgate, c, H, N) break;
    case 1: FOX_LAUNCH_SCAN(gate_scan_fwd_kernel, 1, false, (unsigned)(B * H), logits, sb, sh, sn, seq_start, log_fgate, c, H, N) break;
    case 2: FOX_LAUNCH_SCAN(gate_scan_fwd_kernel, 2, false, (unsigned)(B * H), logits, sb, sh, sn, seq_start, log_fgate, c, H, N) break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_gate_cumsum_bwd(float* dc, const void* logits, int dtype, int64_t sb, int64_t sh, int64_t sn,
                                  const int64_t* seq_start, void* dlogits, int64_t db, int64_t dh, int64_t dn, int B, int H, int N,
                                  const float* drow, int M, hipStream_t s) {
  switch (drow ? dtype | kRows : dtype) {
    case 0: FOX_LAUNCH_SCAN(gate_scan_bwd_kernel, 0, true, scan_blocks(B * H), dc, logits, sb, sh, sn, seq_start, dlogits, db, dh, dn, B * H, H, N, drow, M) break;
    case 1: FOX_LAUNCH_SCAN(gate_scan_bwd_kernel, 1, true, scan_blocks(B * H), dc, logits, sb, sh, sn, seq_start, dlogits, db, dh, dn, B * H, H, N, drow, M) break;
    case 2: FOX_LAUNCH_SCAN(gate_scan_bwd_kernel, 2, true, scan_blocks(B * H), dc, logits, sb, sh, sn, seq_start, dlogits, db, dh, dn, B * H, H, N, drow, M) break;
    case 0 | kRows: FOX_LAUNCH_SCAN(gate_scan_bwd_kernel, (0 | kRows), true, scan_blocks(B * H), dc, logits, sb, sh, sn, seq_start, dlogits, db, dh, dn, B * H, H, N, drow, M) break;
    case 1 | kRows: FOX_LAUNCH_SCAN(gate_scan_bwd_kernel, (1 | kRows), true, scan_blocks(B * H), dc, logits, sb, sh, sn, seq_start, dlogits, db, dh, dn, B * H, H, N, drow, M) break;
    case 2 | kRows: FOX_LAUNCH_SCAN(gate_scan_bwd_kernel, (2 | kRows), true, scan_blocks(B * H), dc, logits, sb, sh, sn, seq_start, dlogits, db, dh, dn, B * H, H, N, drow, M) break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_cumsum_fwd(const float* g, int64_t sb, int64_t sh, int64_t sn, const int64_t* seq_start, float* c, int B,
                             int H, int N, hipStream_t s) {
  FOX_LAUNCH_SCAN(scan_kernel, kForward, false, (unsigned)(B * H), g, sb, sh, sn, seq_start, c,
                     (int64_t)H * N, (int64_t)N, (int64_t)1, B * H, H, N, nullptr, N, nullptr)
  return hipGetLastError();
}

hipError_t launch_cumsum_bwd(float* dc, float* dg, int64_t db, int64_t dh, int64_t dn, const int64_t* seq_start, int B, int H,
                             int N, const float* drow, int M, hipStream_t s) {
  if (drow) {
    FOX_LAUNCH_SCAN(scan_kernel, kReverseRows, true, scan_blocks(B * H), dc, (int64_t)H * N, (int64_t)N, (int64_t)1,
                       seq_start, dg, db, dh, dn, B * H, H, N, drow, M, dc)
  } else {
    FOX_LAUNCH_SCAN(scan_kernel, kReverse, true, scan_blocks(B * H), dc, (int64_t)H * N, (int64_t)N, (int64_t)1,
                       seq_start, dg, db, dh, dn, B * H, H, N, nullptr, N, nullptr)
  }
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// "auto" threshold
// ---------------------------------------------------------------------------
template <typename Tr>
__device__ __forceinline__ float round16(float x) {  // round to the 16-bit dtype and back
  return Tr::lo(Tr::pack2(x, 0.f));
}

__global__ void zero_u32_kernel(uint32_t* p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0u;
}

// The threshold from the largest norms; every tensor op of the reference rounds to the input dtype.
template <typename Tr>
__device__ __forceinline__ float threshold_of_norms(float qn, float kn, float sm_scale, float log_n) {
  float ub = round16<Tr>(qn * kn);
  ub = round16<Tr>(ub * sm_scale);
  float th = round16<Tr>(2.f * ub);
  th = round16<Tr>(th + log_n);
  th = -th;
  return round16<Tr>(th - 10.f);
}
// Norm of a row of which this lane holds eight elements, its D / 8 lanes the others.
template <typename Tr, int LPR>
__device__ __forceinline__ float row_norm(const u32x4& x) {
  float acc = 0.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) acc += Tr::lo(x[e]) * Tr::lo(x[e]) + Tr::hi(x[e]) * Tr::hi(x[e]);
#pragma unroll
  for (int off = LPR / 2; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
  return round16<Tr>(sqrtf(acc));
}
__device__ __forceinline__ float wave_max(float x) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) x = fmaxf(x, __shfl_xor(x, off));
  return x;
}

// Workgroup `id` of those of all q, w.q_blocks for each (batch, head), and then of all k: kNormRows rows of one of them.  scratch holds, per (batch, head), the two
// running maxima (float bits) and the number of workgroups that have added theirs; the workgroup that arrives last
// turns the maxima into the threshold, so no kernel of its own is needed for that.
constexpr int kNormRows = 512;
struct NormBlocks {
  int pairs, q_blocks, k_blocks;
  Divisor by_q, by_k, by_heads;
};
template <typename Tr, int D>
__device__ __forceinline__ void norm_max(const View& q, const View& k, int H, int M, int N, uint32_t* scratch, float* thr, float sm_scale,
                                         float log_n, int id, const NormBlocks& w) {
  constexpr int LPR = D / 8, RPP = 256 / LPR;
  const int tid = threadIdx.x;
  const int which = id >= w.pairs * w.q_blocks;   // 1: k
  if (which) id -= w.pairs * w.q_blocks;
  const int bh = divide(id, which ? w.by_k : w.by_q), block = id - bh * (which ? w.k_blocks : w.q_blocks), b = divide(bh, w.by_heads), h = bh - b * H;
  const View& t = which ? k : q;
  const int T = which ? N : M;
  const uint16_t* p = t.ptr + b * t.sb + h * t.sh;
  const int ch = tid % LPR;
  float best = 0.f;
  constexpr int U = (kNormRows / RPP) < 8 ? (kNormRows / RPP) : 8;  // rows in flight per thread
  for (int pass = 0; pass < kNormRows / RPP; pass += U) {
    u32x4 x[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int row = min(block * kNormRows + (pass + u) * RPP + tid / LPR, T - 1);  // rows past the end repeat the last one
      x[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p + (int64_t)row * t.st + ch * 8));
    }
#pragma unroll
    for (int u = 0; u < U; ++u) best = fmaxf(best, row_norm<Tr, LPR>(x[u]));
  }
  best = wave_max(best);
  __shared__ float wave_best[4];
  if ((tid & 63) == 0) wave_best[tid >> 6] = best;
  __syncthreads();
  if (tid != 0) return;
  best = fmaxf(fmaxf(wave_best[0], wave_best[1]), fmaxf(wave_best[2], wave_best[3]));
  uint32_t* mine = scratch + bh * 3;
  // Non-negative floats order like uints.  The arrival is counted only after the maximum has been applied: the count's
  // operand depends on the value the first atomic returns, and a returning atomic has been carried out where all
  // workgroups' atomics meet.  (No fence: a device-wide release would write back the whole L2 once per workgroup.)
  const uint32_t before = atomicMax(&mine[which], __float_as_uint(best));
  uint32_t one = 1u;
  asm volatile("" : "+v"(one) : "v"(before));
  if (atomicAdd(&mine[2], one) != (uint32_t)(w.q_blocks + w.k_blocks) - 1u) return;
  // the last workgroup of this (batch, head): every maximum has been added (read through the atomic unit as well)
  const float qn = __uint_as_float(atomicMax(&mine[0], 0u)), kn = __uint_as_float(atomicMax(&mine[1], 0u));
  thr[bh] = threshold_of_norms<Tr>(qn, kn, sm_scale, log_n);
}

template <typename Tr, int D>
__global__ __launch_bounds__(256) void norm_max_kernel(View q, View k, int H, int M, int N, uint32_t* scratch, float* thr, float sm_scale, float log_n, NormBlocks w) {
  norm_max<Tr, D>(q, k, H, M, N, scratch, thr, sm_scale, log_n, blockIdx.x, w);
}

// Short rows: one workgroup takes q and k of a (batch, head) whole, up to 128 KB in flight, and there is nothing to clear, to count or to wait for: a single
// round trip and a reduction (12 pairs T256 D128: 12.7 us for zeroing, norms and atomics, 6.2 now).
template <typename Tr, int D>
__global__ __launch_bounds__(1024) void norm_max_pair_kernel(View q, View k, int H, int M, int N, float* thr, float sm_scale, float log_n) {
  constexpr int LPR = D / 8, RPP = 1024 / LPR, U = RPP >= 128 ? 1024 / RPP : 8;   // (threshold_pairs: 1024 rows at most, and no load beyond them)
  const int tid = threadIdx.x, bh = blockIdx.x, b = bh / H, h = bh % H, ch = tid % LPR;
  const uint16_t *qp = q.ptr + b * q.sb + h * q.sh + ch * 8, *kp = k.ptr + b * k.sb + h * k.sh + ch * 8;
  float best_q = 0.f, best_k = 0.f;
  for (int row0 = tid / LPR; row0 < M + N; row0 += U * RPP) {   // (the lanes of a row together)
    u32x4 x[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int row = min(row0 + u * RPP, M + N - 1);   // rows of q, then those of k
      const uint16_t* p = row < M ? qp + (int64_t)row * q.st : kp + (int64_t)(row - M) * k.st;
      x[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float n = row_norm<Tr, LPR>(x[u]);
      if (row0 + u * RPP < M) best_q = fmaxf(best_q, n);
      else best_k = fmaxf(best_k, n);
    }
  }
  best_q = wave_max(best_q);
  best_k = wave_max(best_k);
  __shared__ float wave_q[16], wave_k[16];
  if ((tid & 63) == 0) {
    wave_q[tid >> 6] = best_q;
    wave_k[tid >> 6] = best_k;
  }
  __syncthreads();
  if (tid >= kWave) return;
  best_q = wave_max(wave_q[tid & 15]);
  best_k = wave_max(wave_k[tid & 15]);
  if (tid == 0) thr[bh] = threshold_of_norms<Tr>(best_q, best_k, sm_scale, log_n);
}

// norm_max_kernel with the forward scan of the gates beside it, one workgroup per row in front of the others: the scan is a chain of one workgroup's barriers
// (20 us in a step at B4 T16384 H16) that needs none of the bandwidth the norms stream at (88 us), and needs no threshold.
// At most six waves a SIMD, which is what the registers leave head dims 64 and 128 as well: with eight all norms of a middling call are resident at once and the scan's
// chain waits behind them.  Eight / six, us: 64 pairs T8192 D32 26.3 / 23.8, 128 pairs T4096 D32 25.4 / 23.3, 512 pairs T16384 D16 287 / 261, T2048 D16 43.7 / 40.7.  Five
// starve the norms of long rows (256 pairs T8192 D64 117 / 123).
template <typename Tr, int D, int KIND>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 6))) void norm_max_scan_kernel(View q, View k, int H, int M, int N, uint32_t* scratch, float* thr, float sm_scale, float log_n,
                                                            GateK t, const int64_t* __restrict__ seq_start, NormBlocks w) {
  if ((int)blockIdx.x >= w.pairs) {
    norm_max<Tr, D>(q, k, H, M, N, scratch, thr, sm_scale, log_n, blockIdx.x - w.pairs, w);
    return;
  }
  const int bh = blockIdx.x, b = bh / H, h = bh % H;
  int seq = 0;
  if (seq_start) {
    const int64_t s64 = seq_start[b];
    seq = (int)(s64 < 0 ? 0 : (s64 > N ? N : s64));
  }
  const int64_t base = b * t.sb + h * t.sh;
  float *dst = t.c + (int64_t)bh * N, *lg = t.log_fgate ? t.log_fgate + (int64_t)bh * N : nullptr;
  scan_row<false, 256, 8>(
      N,
      [&](int idx) {
        if constexpr (KIND == kGateLog) {
          return idx >= seq ? reinterpret_cast<const float*>(t.g)[base + (int64_t)idx * t.sn] : 0.f;
        } else {
          const float g = log_sigmoid(load_logit<KIND>(t.g, base + (int64_t)idx * t.sn));
          if (lg) lg[idx] = g;
          return idx >= seq ? g : 0.f;
        }
      },
      [&](int idx, float sum) { dst[idx] = sum; });
}

// Threshold per head from the QK-norm weights: -(2 * max|w_q| * max|w_k| * sqrt(D) + log T) + tolerance, every operation
// rounded to fp32 in the order of the tensor expression it replaces (eleven launches of which none computes anything to speak of;
// 45 us of a layer's forward at B2 T2048 H12 D64, this kernel 2 us).  One wave per head; shared weights: one head.
__global__ __launch_bounds__(256) void qk_norm_threshold_kernel(const float* __restrict__ wq, const float* __restrict__ wk, int H, int D,
                                                                float sqrt_d, float log_t, float tolerance, float* __restrict__ thr) {
  const int h = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (h >= H) return;
  float mq = 0.f, mk = 0.f;
  bool nan = false;   // a NaN weight gives a NaN threshold, as the tensor maximum would
  for (int d = lane; d < D; d += kWave) {
    const float q = fabsf(wq[(int64_t)h * D + d]), k = fabsf(wk[(int64_t)h * D + d]);
    nan |= q != q || k != k;
    mq = fmaxf(mq, q);
    mk = fmaxf(mk, k);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    mq = fmaxf(mq, __shfl_xor(mq, off));
    mk = fmaxf(mk, __shfl_xor(mk, off));
  }
  if (__any(nan)) mq = NAN;
  if (lane == 0) {
    const float bound = __fmul_rn(__fmul_rn(mq, mk), sqrt_d);
    thr[h] = __fadd_rn(-__fadd_rn(__fmul_rn(2.f, bound), log_t), tolerance);
  }
}

hipError_t launch_qk_norm_threshold(const float* wq, const float* wk, int H, int D, double seq_len, double tolerance, float* thr, hipStream_t s) {
  hipLaunchKernelGGL(qk_norm_threshold_kernel, dim3((unsigned)((H + 3) / 4)), dim3(256), 0, s, wq, wk, H, D, (float)sqrt((double)D),
                     (float)log(seq_len), (float)tolerance, thr);
  return hipGetLastError();
}

// Whether one workgroup takes a (batch, head) whole, where that is no longer a chain than the launch that clears the scratch and the three atomics behind each
// other.  us, with them / whole: D 128 T64 9.8 / 6.0, T512 9.4 .. 11.7 / 9.0 .. 9.5, T1024 9.4 / 15.3, D 64 T512 8.4 / 6.0, T1024 7.9 / 9.1, D 32 T512 6.8 / 4.6, D 16 6.7 / 3.9
// (with loads beyond the last row 6.1 and 5.6; M1 N1000, 64 pairs D 16 6.8 / 5.7, with them 7.1); 512 pairs T512, D 128 26.8 / 23.6, D 32 14.8 / 11.9.
static bool threshold_pairs(int M, int N) { return (int64_t)M + N <= 1024; }

template <typename Tr, int D>
static hipError_t auto_threshold_d(const View& q, const View& k, int B, int H, int M, int N, float sm_scale, float* thr, uint32_t* scratch,
                                   const GateK* t, const int64_t* seq_start, hipStream_t s) {
  const int n_bh = B * H, q_blocks = (M + kNormRows - 1) / kNormRows, k_blocks = (N + kNormRows - 1) / kNormRows;
  const NormBlocks w{n_bh, q_blocks, k_blocks, divisor(q_blocks), divisor(k_blocks), divisor(H)};
  const float log_n = (float)log((double)N);
  if (!t && threshold_pairs(M, N)) {
    hipLaunchKernelGGL((norm_max_pair_kernel<Tr, D>), dim3((unsigned)n_bh), dim3(1024), 0, s, q, k, H, M, N, thr, sm_scale, log_n);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(zero_u32_kernel, dim3((unsigned)((3 * n_bh + 255) / 256)), dim3(256), 0, s, scratch, 3 * n_bh);
  const dim3 norms((unsigned)n_bh * (unsigned)(q_blocks + k_blocks)), grid(norms.x + (unsigned)n_bh);
  if (!t) {
    hipLaunchKernelGGL((norm_max_kernel<Tr, D>), norms, dim3(256), 0, s, q, k, H, M, N, scratch, thr, sm_scale, log_n, w);
    return hipGetLastError();
  }
  switch (t->kind) {
    case kGateLog: hipLaunchKernelGGL((norm_max_scan_kernel<Tr, D, kGateLog>), grid, dim3(256), 0, s, q, k, H, M, N, scratch, thr, sm_scale, log_n, *t, seq_start, w); break;
    case 0: hipLaunchKernelGGL((norm_max_scan_kernel<Tr, D, 0>), grid, dim3(256), 0, s, q, k, H, M, N, scratch, thr, sm_scale, log_n, *t, seq_start, w); break;
    case 1: hipLaunchKernelGGL((norm_max_scan_kernel<Tr, D, 1>), grid, dim3(256), 0, s, q, k, H, M, N, scratch, thr, sm_scale, log_n, *t, seq_start, w); break;
    case 2: hipLaunchKernelGGL((norm_max_scan_kernel<Tr, D, 2>), grid, dim3(256), 0, s, q, k, H, M, N, scratch, thr, sm_scale, log_n, *t, seq_start, w); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
template <typename Tr>
static hipError_t auto_threshold_t(const View& q, const View& k, int B, int H, int M, int N, int D, float sm_scale, float* thr, uint32_t* scratch,
                                   const GateK* t, const int64_t* seq_start, hipStream_t s) {
  switch (D) {
    case 16: return auto_threshold_d<Tr, 16>(q, k, B, H, M, N, sm_scale, thr, scratch, t, seq_start, s);
    case 32: return auto_threshold_d<Tr, 32>(q, k, B, H, M, N, sm_scale, thr, scratch, t, seq_start, s);
    case 64: return auto_threshold_d<Tr, 64>(q, k, B, H, M, N, sm_scale, thr, scratch, t, seq_start, s);
    case 128: return auto_threshold_d<Tr, 128>(q, k, B, H, M, N, sm_scale, thr, scratch, t, seq_start, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_auto_threshold(const View& q, const View& k, int B, int H, int M, int N, int D, int dtype, float sm_scale,
                                 float* thr, uint32_t* scratch, const GateK* t, const int64_t* seq_start, hipStream_t s) {
  return dtype == 0 ? auto_threshold_t<Bf16>(q, k, B, H, M, N, D, sm_scale, thr, scratch, t, seq_start, s)
                    : auto_threshold_t<Fp16>(q, k, B, H, M, N, D, sm_scale, thr, scratch, t, seq_start, s);
}

// Whether the scan goes beside the norms.  There it has 256 threads (2 us and 1 us per 1024 elements), on its own 1024 (about 4 us and 1 us per 2100) and a launch; the norms take 8 us
// and stream at about 6 TB/s.
// - Fewer queries than half the keys: always, but for a row that takes longer than all of that and is alone.  Threshold and scan alone, two launches / one, us: M8 N9000 12 pairs D128
//   21.1 / 12.6, 32 pairs M4 N29333 D64 56 / 45, 128 pairs D16 M8 N4000 16.6 / 13.6, 2 pairs N32768 D16 21.8 / 26.1, 12 pairs N32768 D64 38.1 / 39.7, D128 45.7 / 43.7.
// - Else where the norms stream for longer than the scan's 256 threads take.  "auto" forward, us: B4 T16384 H16 D128 345 / 329, B4 T4096 H32 D64 107 / 99, B2 T8192 H16 D64 68.4 / 62.5,
//   B8 T700 H32 D32 29.6 / 26.9.  Below that line one launch can be the faster one as well (12 pairs D128 M = N = 4096, threshold and scan alone, 17.5 / 12.8), but a host test
//   holds the line at shapes on either side of it, and it has not been swept for another.
bool threshold_scans(int B, int H, int M, int N, int D) {
  const int64_t pairs = (int64_t)B * H, bytes = pairs * ((int64_t)M + N) * D * 2;
  const bool beside = threshold_pairs(M, N) || 2 * (int64_t)M >= N ? bytes >= 6000 * ((int64_t)N + 2000) : bytes >= 6000000 * ((int64_t)N / 1400 - 11);
  return beside && pairs * (1 + 2 * (int64_t)((N + kNormRows - 1) / kNormRows)) < (int64_t)1 << 31;
}

}  // namespace fox
