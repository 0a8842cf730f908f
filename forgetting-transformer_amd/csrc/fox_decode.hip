// Single-query forward (decode step, M == 1) of Forgetting Attention for gfx950.
//
// With one query row per (batch, head) there is nothing for the matrix cores to do: the step is one
// pass over the K and V cache, 4*D flops per 4*D bytes.  Like the reference, which switches to an
// element-wise multiply-and-sum for this case (ops/forgetting_attention.py:148-153, :637-641,
// :665-668), this kernel is dot-free.  It keeps nothing in LDS while it streams: a key row of D
// elements is spread over D/8 lanes (16 bytes each), a wave instruction covers 64/(D/8) consecutive
// keys, and every lane holds eight such loads of K and of V in flight, so that a CU has hundreds of
// KiB outstanding instead of the two 64-key tiles of the tiled kernel.  The lanes of a key row reduce
// the partial dot products with four DPP adds; each row group runs its own online softmax
// (running maximum m, sum l, eight accumulator elements per lane), and the groups of a workgroup are
// merged once at the end.
//
// The key range [lo, N) -- lo = max(seq_start, first block the pruning bound keeps) -- is dealt out
// over `splits` workgroups per (batch, head); with more than one split the partial (m, l, acc) go to
// the same workspace layout as the tiled kernel's key splits and fox::combine_kernel merges them.
#include "fox_common.hpp"
#include "fox_decode_plan.hpp"
#include "fox_kernels.hpp"

namespace fox {

namespace {

template <typename Tr>
__device__ __forceinline__ void unpack8f(const u32x4& v, float (&f)[8]) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    f[2 * e] = Tr::lo(v[e]);
    f[2 * e + 1] = Tr::hi(v[e]);
  }
}

// merge the online-softmax state (m2, l2, acc2) into (m, l, acc)
__device__ __forceinline__ void merge_state(float& m, float& l, float (&acc)[8], float m2, float l2, const float (&acc2)[8]) {
  const float mx = fmaxf(m, m2);
  const float w1 = __builtin_amdgcn_exp2f(m - mx), w2 = __builtin_amdgcn_exp2f(m2 - mx);
  l = l * w1 + l2 * w2;
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = acc[e] * w1 + acc2[e] * w2;
  m = mx;
}

}  // namespace

template <typename Tr, int D>
__global__ __launch_bounds__(256) void decode_kernel(const FwdK a) {
  constexpr int LPR = D / 8;      // lanes per key row
  constexpr int KPL = 64 / LPR;   // keys per wave load instruction
  constexpr int U = 8;            // loads of K and of V in flight per lane
  constexpr int KPB = KPL * U;    // keys per wave and batch
  __shared__ float part_m[4], part_l[4];
  __shared__ __align__(16) float part_acc[4][D];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ch = lane % LPR, r = lane / LPR;
  const int bh = divide(blockIdx.x, a.by_splits), sp = blockIdx.x - bh * a.splits;
  const int b = divide(bh, a.order.by_heads), h = bh - b * a.H;
  const int N = a.N;
  const float* c_row = a.c + (int64_t)bh * N;
  const uint16_t* qp = a.q.ptr + b * a.q.sb + h * a.q.sh;
  const uint16_t* kp = a.k.ptr + b * a.k.sb + h * a.k.sh + ch * 8;
  const uint16_t* vp = a.v.ptr + b * a.v.sb + h * a.v.sh + ch * 8;

  int seq = 0;
  if (a.seq_start) {
    const int64_t s64 = a.seq_start[b];
    seq = (int)(s64 < 0 ? 0 : (s64 > N ? N : s64));
  }
  const int a0 = N - 1;  // key position of the query row
  const float c_ref = c_row[a0];
  int lo = seq;
  if (a.thr) {
    const int t = acp_first_kept_block(c_row, c_ref, a.thr[bh], N, kFwdBN, a0 / kFwdBN, lane);
    lo = max(lo, t * kFwdBN);
  }
  if (a.first_block && tid == 0 && sp == 0) a.first_block[bh] = lo / kFwdBN;

  // this workgroup's share of [lo, N): whole rounds of 4 waves x KPB keys
  const int n_keys = N - lo;
  int per = divide(n_keys + a.splits - 1, a.by_splits);
  per = (per + 4 * KPB - 1) / (4 * KPB) * (4 * KPB);
  const int k0 = min(N, lo + sp * per), k1 = min(N, k0 + per);

  float qf[8];
  {
    const float qk_scale = a.sm_scale * kLog2e;
    unpack8f<Tr>(*reinterpret_cast<const u32x4*>(qp + ch * 8), qf);
#pragma unroll
    for (int e = 0; e < 8; ++e) qf[e] *= qk_scale;
  }
  float m = -3.0e38f, l = 0.f;  // finite floor: a group that has seen no key yet yields exp2(-inf) = 0
  float acc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = 0.f;

  for (int base = k0 + wave * KPB; base < k1; base += 4 * KPB) {
    u32x4 kx[U], vx[U];
    float cn[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int n = min(base + u * KPL + r, N - 1);  // keys past the range read a valid row and are masked below
      kx[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(kp + (int64_t)n * a.k.st));
      cn[u] = c_row[n];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int n = min(base + u * KPL + r, N - 1);
      vx[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(vp + (int64_t)n * a.v.st));
    }
    float s[U];
    float bmax = -INFINITY;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float kf[8];
      unpack8f<Tr>(kx[u], kf);
      float dot = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) dot = fmaf(qf[e], kf[e], dot);
      dot = row_sum<LPR>(dot);
      // log2-domain score: sm_scale*log2e*(q.k) + (c_ref - c_n)*log2e.  The two cumulative sums are subtracted
      // first (they are of similar, possibly large, magnitude; their difference is small and exact to an ulp of
      // itself), then scaled: the order of the reference (:642-643).
      const float x = fmaf(c_ref - cn[u], kLog2e, dot);
      s[u] = (base + u * KPL + r < k1) ? x : -INFINITY;
      bmax = fmaxf(bmax, s[u]);
    }
    const float m_new = fmaxf(m, bmax);
    const float alpha = __builtin_amdgcn_exp2f(m - m_new);
    m = m_new;
    l *= alpha;
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] *= alpha;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float p = __builtin_amdgcn_exp2f(s[u] - m);
      l += p;
      float vf[8];
      unpack8f<Tr>(vx[u], vf);
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] = fmaf(p, vf[e], acc[e]);
    }
  }

  // merge the KPL row groups of the wave, then the four waves
#pragma unroll
  for (int off = LPR; off < 64; off <<= 1) {
    const float m2 = __shfl_xor(m, off), l2 = __shfl_xor(l, off);
    float acc2[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) acc2[e] = __shfl_xor(acc[e], off);
    merge_state(m, l, acc, m2, l2, acc2);
  }
  if (r == 0) {
    if (ch == 0) { part_m[wave] = m; part_l[wave] = l; }
#pragma unroll
    for (int e = 0; e < 8; ++e) part_acc[wave][ch * 8 + e] = acc[e];
  }
  __syncthreads();
  if (tid >= LPR) return;
  m = part_m[0];
  l = part_l[0];
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = part_acc[0][ch * 8 + e];
#pragma unroll
  for (int w = 1; w < 4; ++w) {
    float acc2[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) acc2[e] = part_acc[w][ch * 8 + e];
    merge_state(m, l, acc, part_m[w], part_l[w], acc2);
  }

  if (a.splits > 1) {  // partial result of this key split, in the layout fox::combine_kernel reads (M == 1)
    const int64_t row = (int64_t)sp * a.B * a.H + bh;
    float* wo = a.ws_o + row * D + ch * 8;
    const f32x4 w0 = {acc[0], acc[1], acc[2], acc[3]}, w1 = {acc[4], acc[5], acc[6], acc[7]};
    *reinterpret_cast<f32x4*>(wo) = w0;
    *reinterpret_cast<f32x4*>(wo + 4) = w1;
    if (ch == 0) {
      a.ws_ml[2 * row] = m;
      a.ws_ml[2 * row + 1] = l;
    }
    return;
  }
  const bool empty = a0 < seq;  // every key is left padding: o = 0, lse = -inf (:679-685)
  const float inv = empty ? 0.f : 1.0f / l;
  uint16_t* op = const_cast<uint16_t*>(a.o.ptr) + b * a.o.sb + h * a.o.sh + ch * 8;
  u32x4 w;
#pragma unroll
  for (int e = 0; e < 4; ++e) w[e] = Tr::pack2(acc[2 * e] * inv, acc[2 * e + 1] * inv);
  *reinterpret_cast<u32x4*>(op) = w;
  if (ch == 0) a.lse[bh] = empty ? -INFINITY : m * kLn2 + __logf(l);
}

#define FOX_INSTANTIATE_DECODE(TR)                               \
  template __global__ void decode_kernel<TR, 16>(const FwdK);   \
  template __global__ void decode_kernel<TR, 32>(const FwdK);   \
  template __global__ void decode_kernel<TR, 64>(const FwdK);   \
  template __global__ void decode_kernel<TR, 128>(const FwdK);
FOX_INSTANTIATE_DECODE(Bf16)
FOX_INSTANTIATE_DECODE(Fp16)

template <typename Tr>
static hipError_t launch_decode_t(const FwdK& a, int D, hipStream_t s) {
  const dim3 grid((unsigned)(a.splits * a.B * a.H));
  switch (D) {
    case 16: hipLaunchKernelGGL((decode_kernel<Tr, 16>), grid, dim3(256), 0, s, a); break;
    case 32: hipLaunchKernelGGL((decode_kernel<Tr, 32>), grid, dim3(256), 0, s, a); break;
    case 64: hipLaunchKernelGGL((decode_kernel<Tr, 64>), grid, dim3(256), 0, s, a); break;
    case 128: hipLaunchKernelGGL((decode_kernel<Tr, 128>), grid, dim3(256), 0, s, a); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// The streaming part of a single-query forward; the caller merges the splits (fox::combine_kernel).
hipError_t launch_fwd_decode(const FwdK& a, int D, int dtype, hipStream_t s) {
  return dtype == 0 ? launch_decode_t<Bf16>(a, D, s) : launch_decode_t<Fp16>(a, D, s);
}

// Merge of the splits of decode_gates_kernel by 256 threads per (batch, head), every partial in flight at once (at most
// kDecodeMaxSplits of them, one round trip; a thread that walks the splits one after the other pays one per split).
// AGENT: the partials come from workgroups of the same launch.
template <typename Tr, int D, bool AGENT>
__device__ __forceinline__ void decode_merge(const DecodeK& a, int bh) {
  constexpr int TPR = D / 4, GROUPS = 256 / TPR, PER = (kDecodeMaxSplits + GROUPS - 1) / GROUPS;
  __shared__ float weight[kDecodeMaxSplits];
  __shared__ float l_tot, m_tot;
  __shared__ __align__(16) float part[GROUPS][D];
  const int tid = threadIdx.x, b = divide(bh, a.by_heads), h = bh - b * a.H, splits = a.splits;
  const int grp = tid / TPR, d = (tid % TPR) * 4;
  const float* wo = a.ws_o + (int64_t)bh * splits * D + d;
  f32x4 x[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const float* p = wo + (int64_t)min(grp + i * GROUPS, splits - 1) * D;
    if constexpr (AGENT) x[i] = f32x4{load_agent(p), load_agent(p + 1), load_agent(p + 2), load_agent(p + 3)};
    else x[i] = *reinterpret_cast<const f32x4*>(p);
  }
  if (tid < kWave) {   // one lane per split (counted from the last keys): its maximum moves by the gates of the splits behind it
    const DecodePartial* from = a.ws_p + (int64_t)bh * splits + min(tid, splits - 1);
    const DecodePartial p = AGENT ? DecodePartial{load_agent(&from->g), load_agent(&from->m), load_agent(&from->l)} : *from;
    double incl = tid < splits ? p.g : 0.0;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const double up = __shfl_up(incl, off);
      if (tid >= off) incl += up;
    }
    const double excl = __shfl_up(incl, 1);
    const float m = tid == 0 ? p.m : tid < splits ? p.m + (float)excl * kLog2e : -INFINITY;
    float mx = m;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
    const float w = __builtin_amdgcn_exp2f(m - mx);
    float l = p.l * w;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) l += __shfl_xor(l, off);
    weight[tid] = w;
    if (tid == 0) { l_tot = l; m_tot = mx; }
  }
  __syncthreads();
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < PER; ++i)
    if (grp + i * GROUPS < splits) acc += x[i] * weight[grp + i * GROUPS];
  *reinterpret_cast<f32x4*>(&part[grp][d]) = acc;
  __syncthreads();
  if (tid >= TPR) return;
  acc = *reinterpret_cast<const f32x4*>(&part[0][d]);
  const int used = min(GROUPS, splits);
  for (int i = 1; i < used; ++i) acc += *reinterpret_cast<const f32x4*>(&part[i][d]);
  const bool empty = a.seq_start && a.seq_start[b] >= a.N;
  const float inv = empty ? 0.f : 1.0f / l_tot;
  uint16_t* op = const_cast<uint16_t*>(a.o.ptr) + b * a.o.sb + h * a.o.sh + d;
  u32x2 w;
  w[0] = Tr::pack2(acc[0] * inv, acc[1] * inv);
  w[1] = Tr::pack2(acc[2] * inv, acc[3] * inv);
  *reinterpret_cast<u32x2*>(op) = w;
  if (d == 0 && a.lse) a.lse[bh] = empty ? -INFINITY : m_tot * kLn2 + __logf(l_tot);
}

// ---------------------------------------------------------------------------
// The same step straight from the log forget gates: no cumulative sum of the whole row in front of it.
//
// The score of key n needs the sum of the gates behind it, not the two ends of a sum from the row's start.  Every wave owns
// a contiguous run of keys, walks it from its end and carries that sum (fp64, rounded once per key) relative to the end of
// its own run; the runs' totals then shift the partial maxima where partials are merged: four waves in LDS, splits in
// decode_merge, by the one that arrives last or in a launch of its own.  A gate is read once, by the wave that reads its key; the row scan this replaces (one workgroup per
// row, a chain of barriers per 8192 keys) took 20 us of a 600 us step at B16 H16 N32768 D128 and 5.7 us of 36 at
// B1 H12 N1500 D64.  Bound by HBM where the cache is long, by one round trip per batch where it is short.
template <typename Tr, int D, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void decode_gates_kernel(const DecodeK a) {
  constexpr int LPR = D / 8;      // lanes per key row
  constexpr int KPL = 64 / LPR;   // keys per wave load instruction
  constexpr int U = 8;            // loads of K and of V in flight per lane
  constexpr int KPB = KPL * U;    // keys per wave and batch
  constexpr int GB = (KPB + 63) / 64;   // gates per lane and batch
  static_assert(KPB == kDecodeBatchKeys<D>, "the host counts batches with the same size");
  __shared__ float part_m[WAVES], part_l[WAVES];
  __shared__ double part_g[WAVES];
  __shared__ __align__(16) float part_acc[WAVES][D];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ch = lane % LPR, r = lane / LPR;
  const int bh = divide(blockIdx.x, a.by_splits), sp = blockIdx.x - bh * a.splits;
  const int b = divide(bh, a.by_heads), h = bh - b * a.H;
  const int N = a.N;
  const float* gp = a.g + b * a.g_sb + h * a.g_sh;
  const uint16_t* qp = a.q.ptr + b * a.q.sb + h * a.q.sh;
  const uint16_t* kp = a.k.ptr + b * a.k.sb + h * a.k.sh + ch * 8;
  const uint16_t* vp = a.v.ptr + b * a.v.sb + h * a.v.sh + ch * 8;

  int lo = 0;
  if (a.seq_start) {
    const int64_t s64 = a.seq_start[b];
    lo = (int)(s64 < 0 ? 0 : (s64 > N ? N : s64));
  }
  // run gw of the splits * WAVES runs, counted from the last key: whole batches, the first one excepted
  const int gw = sp * WAVES + wave;
  int per = divide((N - lo + WAVES - 1) / WAVES + a.splits - 1, a.by_splits);
  per = (per + KPB - 1) / KPB * KPB;
  const int64_t back = (int64_t)gw * per;
  const int k1 = back < N - lo ? N - (int)back : lo, k0 = k1 - lo > per ? k1 - per : lo;

  float qf[8];
  {
    const float qk_scale = a.sm_scale * kLog2e;
    unpack8f<Tr>(*reinterpret_cast<const u32x4*>(qp + ch * 8), qf);
#pragma unroll
    for (int e = 0; e < 8; ++e) qf[e] *= qk_scale;
  }
  float m = -3.0e38f, l = 0.f;  // finite floor: a group that has seen no key yet yields exp2(-inf) = 0
  float acc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = 0.f;
  double behind = 0.0;          // sum of the run's gates behind the batch

  for (int end = k1; end > k0; end -= KPB) {   // keys end - KPB .. end - 1, those left of k0 masked
    float gx[GB];
#pragma unroll
    for (int s = 0; s < GB; ++s) {             // lane j of group s holds the gate of key end - 1 - 64 s - j
      const int j = 64 * s + lane, n = end - 1 - j;
      gx[s] = gp[(int64_t)max(n, k0) * a.g_sn];
      if (j >= KPB || n < k0) gx[s] = 0.f;
    }
    u32x4 kx[U], vx[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int n = max(end - KPB + u * KPL + r, k0);   // keys left of the run read its first row and are masked below
      kx[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(kp + (int64_t)n * a.k.st));
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int n = max(end - KPB + u * KPL + r, k0);
      vx[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(vp + (int64_t)n * a.v.st));
    }
    float bias[GB];   // log2e * sum of the gates behind the key whose gate this lane holds
#pragma unroll
    for (int s = 0; s < GB; ++s) {
      double incl = (double)gx[s];
#pragma unroll
      for (int off = 1; off < kWave; off <<= 1) {
        const double up = __shfl_up(incl, off);
        if (lane >= off) incl += up;
      }
      const double excl = __shfl_up(incl, 1);   // (not incl - gate: a gate may be -inf)
      bias[s] = (float)(lane > 0 ? behind + excl : behind) * kLog2e;
      behind += __shfl(incl, kWave - 1);
    }
    float sc[U];
    float bmax = -INFINITY;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float kf[8];
      unpack8f<Tr>(kx[u], kf);
      float dot = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) dot = fmaf(qf[e], kf[e], dot);
      dot = row_sum<LPR>(dot);
      const int j = KPB - 1 - u * KPL;   // key u * KPL + r of the batch sits j - r keys before its end
      const float x = dot + __shfl(bias[j / 64], (j - r) & 63);
      sc[u] = (end - KPB + u * KPL + r >= k0) ? x : -INFINITY;
      bmax = fmaxf(bmax, sc[u]);
    }
    const float m_new = fmaxf(m, bmax);
    const float alpha = __builtin_amdgcn_exp2f(m - m_new);
    m = m_new;
    l *= alpha;
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] *= alpha;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float p = __builtin_amdgcn_exp2f(sc[u] - m);
      l += p;
      float vf[8];
      unpack8f<Tr>(vx[u], vf);
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] = fmaf(p, vf[e], acc[e]);
    }
  }

  // merge the KPL row groups of the wave, then the waves, each shifted by the gates of the runs behind its own
#pragma unroll
  for (int off = LPR; off < 64; off <<= 1) {
    const float m2 = __shfl_xor(m, off), l2 = __shfl_xor(l, off);
    float acc2[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) acc2[e] = __shfl_xor(acc[e], off);
    merge_state(m, l, acc, m2, l2, acc2);
  }
  if (r == 0) {
    if (ch == 0) { part_m[wave] = m; part_l[wave] = l; part_g[wave] = behind; }
#pragma unroll
    for (int e = 0; e < 8; ++e) part_acc[wave][ch * 8 + e] = acc[e];
  }
  __syncthreads();
  if (tid < LPR) {
    m = part_m[0];
    l = part_l[0];
    double shift = part_g[0];
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = part_acc[0][ch * 8 + e];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) {
      float acc2[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) acc2[e] = part_acc[w][ch * 8 + e];
      merge_state(m, l, acc, part_m[w] + (float)shift * kLog2e, part_l[w], acc2);
      shift += part_g[w];
    }

    if (a.splits > 1) {  // partial result of this split: accumulator, maximum and sum relative to its last key, sum of its gates
      const int64_t row = (int64_t)bh * a.splits + sp;
      float* wo = a.ws_o + row * D + ch * 8;
      if (WAVES == 4 && a.arrived) {
#pragma unroll
        for (int e = 0; e < 8; ++e) store_agent(wo + e, acc[e]);
        if (ch == 0) {
          store_agent(&a.ws_p[row].g, shift);
          store_agent(&a.ws_p[row].m, m);
          store_agent(&a.ws_p[row].l, l);
        }
      } else {
        const f32x4 w0 = {acc[0], acc[1], acc[2], acc[3]}, w1 = {acc[4], acc[5], acc[6], acc[7]};
        *reinterpret_cast<f32x4*>(wo) = w0;
        *reinterpret_cast<f32x4*>(wo + 4) = w1;
        if (ch == 0) a.ws_p[row] = DecodePartial{shift, m, l};
      }
    } else {
      const bool empty = lo >= N;  // every key is left padding: o = 0, lse = -inf (:679-685)
      const float inv = empty ? 0.f : 1.0f / l;
      uint16_t* op = const_cast<uint16_t*>(a.o.ptr) + b * a.o.sb + h * a.o.sh + ch * 8;
      u32x4 w;
#pragma unroll
      for (int e = 0; e < 4; ++e) w[e] = Tr::pack2(acc[2 * e] * inv, acc[2 * e + 1] * inv);
      *reinterpret_cast<u32x4*>(op) = w;
      if (ch == 0 && a.lse) a.lse[bh] = empty ? -INFINITY : m * kLn2 + __logf(l);
    }
  }
  if constexpr (WAVES == 4) {   // the last of the splits merges them (decode_merges)
    if (a.splits <= 1 || !a.arrived) return;
    __shared__ bool last;
    if (wave == 0) {   // the wave that stored the partials
      stores_complete();
      if (lane == 0) last = arrive(&a.arrived[bh]) == (uint32_t)a.splits - 1u;
    }
    __syncthreads();
    if (!last) return;
    decode_merge<Tr, D, true>(a, bh);
    if (tid == 0) __hip_atomic_store(&a.arrived[bh], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// decode_merge as a launch of its own
template <typename Tr, int D>
__global__ __launch_bounds__(256) void decode_combine_kernel(const DecodeK a) {
  decode_merge<Tr, D, false>(a, blockIdx.x);
}

template <typename Tr, int D>
static hipError_t launch_decode_gates_d(const DecodeK& a, hipStream_t s) {
  if constexpr (D >= 32) {
    if (decode_one_workgroup((int64_t)a.B * a.H, decode_batches(a.N, D), D)) {
      hipLaunchKernelGGL((decode_gates_kernel<Tr, D, 16>), dim3((unsigned)(a.B * a.H)), dim3(1024), 0, s, a);
      return hipGetLastError();
    }
  }
  hipLaunchKernelGGL((decode_gates_kernel<Tr, D, 4>), dim3((unsigned)(a.splits * a.B * a.H)), dim3(256), 0, s, a);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || a.splits <= 1 || a.arrived) return e;
  hipLaunchKernelGGL((decode_combine_kernel<Tr, D>), dim3((unsigned)(a.B * a.H)), dim3(256), 0, s, a);
  return hipGetLastError();
}

template <typename Tr>
static hipError_t launch_decode_gates_t(const DecodeK& a, int D, hipStream_t s) {
  switch (D) {
    case 16: return launch_decode_gates_d<Tr, 16>(a, s);
    case 32: return launch_decode_gates_d<Tr, 32>(a, s);
    case 64: return launch_decode_gates_d<Tr, 64>(a, s);
    case 128: return launch_decode_gates_d<Tr, 128>(a, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_decode_gates(const DecodeK& a, int D, int dtype, hipStream_t s) {
  return dtype == 0 ? launch_decode_gates_t<Bf16>(a, D, s) : launch_decode_gates_t<Fp16>(a, D, s);
}

// ---------------------------------------------------------------------------
// New tokens into a layer's cache: keys, values and log gates in one launch.  One 16-byte piece of K and the same piece of V per
// thread, the thread with a row's first piece also moves its gate.  For one token per sequence the launches are the cost
// (B1 H12 D64: three strided copies 6.1 us of kernels plus their host time, this kernel 2.3); a prompt is a plain stream.
__global__ __launch_bounds__(256) void cache_append_kernel(const CacheAppendK a) {
  const uint32_t idx = blockIdx.x * 256u + threadIdx.x, pieces = (uint32_t)a.D / 8u;
  if (idx >= a.total) return;
  const uint32_t row = idx / pieces, ch = idx - row * pieces, bh = row / (uint32_t)a.T, t = row - bh * (uint32_t)a.T;
  const uint32_t b = bh / (uint32_t)a.H, h = bh - b * (uint32_t)a.H;
  auto at = [&](const View& v, int64_t t0) { return v.ptr + b * v.sb + h * v.sh + (t0 + t) * v.st + ch * 8; };
  const u32x4 kx = *reinterpret_cast<const u32x4*>(at(a.k, 0)), vx = *reinterpret_cast<const u32x4*>(at(a.v, 0));
  float gx = 0.f;
  if (ch == 0) gx = a.g[b * a.g_sb + h * a.g_sh + t * a.g_sn];
  *reinterpret_cast<u32x4*>(const_cast<uint16_t*>(at(a.k_buf, a.old))) = kx;
  *reinterpret_cast<u32x4*>(const_cast<uint16_t*>(at(a.v_buf, a.old))) = vx;
  if (ch == 0) a.g_buf[b * a.gb_sb + h * a.gb_sh + (a.old + t) * a.gb_sn] = gx;
}

hipError_t launch_cache_append(const CacheAppendK& a, hipStream_t s) {
  hipLaunchKernelGGL(cache_append_kernel, dim3((a.total + 255u) / 256u), dim3(256), 0, s, a);
  return hipGetLastError();
}

}  // namespace fox
