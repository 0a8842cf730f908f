// Per-head RMS normalisation for gfx950, gated or plain: the epilogue the FoX layer applies to the
// attention output before the output projection, and the normalisation of queries and keys in front
// of the attention (QK-norm),
//   y[r,h,:] = x[r,h,:] * rstd[r,h] * w[h,:] * act(g[r,h,:]),   rstd = 1 / sqrt(mean_d x^2 + eps),
// act(g) = sigmoid(g), g*sigmoid(g) (swish) or 1 (no gate tensor), and its backward
//   yn = xhat * w (xhat = x * rstd),  dg = dy * yn * act'(g),  dyn = dy * act(g),
//   dw[h,:] = sum_r dyn * xhat,  dx = (dyn*w - xhat * mean_d(dyn*w*xhat)) * rstd.
// (reference: model/forgetting_transformer/fuse_norm_gate.py:132-206 forward, :309-417 backward, the
// configuration FusedGroupNormGated(num_groups=heads, is_rms_norm=True, activation="sigmoid") of
// modeling_forgetting_transformer.py:243, no bias, no residual; the plain form is layer_norm_fwd_kernel /
// layer_norm_bwd_kernel of layernorm.py:183-254, :328-435 as used by GroupNorm(num_groups=heads,
// is_rms_norm=True) and RMSNorm(head_dim), modeling_forgetting_transformer.py:258-265, :314-325)
//
// Both are pure streams over HBM.  A (row, head) group of D elements is spread over D/8 lanes, 16
// bytes each; the two row reductions are shuffles inside that lane group.  In the backward every
// thread keeps one (head, 8 elements) column and walks rows of a strip, so the weight gradient is
// accumulated in registers and leaves as one partial per workgroup; a second kernel adds the partials in
// a fixed order (no atomics: the result does not depend on scheduling).
#include "fox_common.hpp"
#include "fox_kernels.hpp"

namespace fox {

template <typename Tr>
__device__ __forceinline__ void unpack8v(const u32x4& v, float (&f)[8]) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    f[2 * e] = Tr::lo(v[e]);
    f[2 * e + 1] = Tr::hi(v[e]);
  }
}
template <typename Tr>
__device__ __forceinline__ u32x4 pack8v(const float (&f)[8]) {
  u32x4 r;
#pragma unroll
  for (int e = 0; e < 4; ++e) r[e] = Tr::pack2(f[2 * e], f[2 * e + 1]);
  return r;
}
template <typename Tr, int D, int ACT>
__global__ __launch_bounds__(256) void norm_gate_fwd_kernel(const NormGateK a) {
  constexpr int CH = D / 8;
  const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int chunk = (int)(gid % CH);
  const int64_t grp = gid / CH;             // (row, head) index
  const bool live = grp < (int64_t)a.R * a.G;
  const int64_t row = live ? grp / a.G : 0;
  const int h = live ? (int)(grp % a.G) : 0;
  const int64_t off = h * (int64_t)D + chunk * 8;
  float x[8], g[8], w[8], y[8];
  unpack8v<Tr>(__builtin_nontemporal_load(reinterpret_cast<const u32x4*>(a.x + row * a.x_sr + off)), x);
  if (ACT != kActNone) unpack8v<Tr>(__builtin_nontemporal_load(reinterpret_cast<const u32x4*>(a.g + row * a.g_sr + off)), g);
  {
    const f32x4 w0 = *reinterpret_cast<const f32x4*>(a.w + off), w1 = *reinterpret_cast<const f32x4*>(a.w + off + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) { w[e] = w0[e]; w[4 + e] = w1[e]; }
  }
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) ss += x[e] * x[e];
#pragma unroll
  for (int o = CH / 2; o > 0; o >>= 1) ss += __shfl_xor(ss, o);
  const float rstd = 1.0f / sqrtf(ss / D + a.eps);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    y[e] = x[e] * rstd * w[e];
    if (ACT != kActNone) {
      const float s = sigmoidf(g[e]);
      y[e] *= ACT == kActSwish ? g[e] * s : s;
    }
  }
  if (live) {
    *reinterpret_cast<u32x4*>(a.y + row * a.y_sr + off) = pack8v<Tr>(y);
    if (chunk == 0) a.rstd[grp] = rstd;
  }
}

// Backward.  A workgroup covers the `cols` (head, 8 elements) columns times R = blockDim / cols row lanes,
// and walks `rows_per_lane` rows per lane (every R-th row of its strip), so that a wave reads whole token rows, the weight
// gradient is accumulated in registers over the rows of a lane, through LDS over the R lanes, and leaves as one partial
// row per workgroup.  The kernel streams (5 x 2 bytes per element, 3 x 2 without a gate); what bounds a small call is how much of it is in
// flight, so the rows per lane follow from the size (norm_bwd_plan).  Both launches together: at 32 rows per thread whatever the size,
// 4096 rows of 12 x 64 made 48 workgroups and took 34.4 us gated and 21.0 us plain, now 12.1 and 9.2 us; 65536 rows of 16 x 128
// stay at 32 rows (262 and 150 us, 5.1 and 5.4 TB/s); 1 M rows of one 128-element head 183 -> 142 us (fewer partials).
// More than 256 columns: one row lane, and the (strip, column) pairs are dealt out in order, so that the workgroups of the same rows run
// side by side and no lane idles (workgroups of 256 columns, all strips of the first columns in front: 32768 rows of 32 x 128 303 instead of 263 us).
template <typename Tr, int D, int ACT>
__global__ __launch_bounds__(256) void norm_gate_bwd_kernel(const NormGateK a) {
  constexpr int CH = D / 8;
  __shared__ __align__(16) float dw_s[256][8];
  const int tid = threadIdx.x;
  const bool wide = a.cols > 256;
  const int64_t flat = (int64_t)blockIdx.x * 256 + tid;
  const int64_t strip = wide ? flat / a.cols : blockIdx.x;
  const int rl = wide ? 0 : tid / a.cols;
  const int col = wide ? (int)(flat - strip * a.cols) : tid - rl * a.cols;
  const int R = wide ? 1 : blockDim.x / a.cols;         // row lanes (threads beyond R * cols idle)
  const bool live = rl < R && strip * R * a.rows_per_lane < a.R;
  const int hh = live ? col / CH : 0;
  const int64_t off = live ? (int64_t)col * 8 : 0;
  const int64_t r0 = strip * R * a.rows_per_lane;
  const int64_t r1 = min((int64_t)a.R, r0 + (int64_t)R * a.rows_per_lane);
  float w[8], dw[8];
  {
    const f32x4 w0 = *reinterpret_cast<const f32x4*>(a.w + off), w1 = *reinterpret_cast<const f32x4*>(a.w + off + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) { w[e] = w0[e]; w[4 + e] = w1[e]; }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) dw[e] = 0.f;

  constexpr int U = 4;  // rows in flight
  for (int64_t rb = r0 + rl; live && rb < r1; rb += U * R) {   // (the lanes of a (row, head) group enter and leave together)
    u32x4 xv[U], gv[U], dyv[U];
    float rs[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t r = min(rb + u * R, r1 - 1);
      xv[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(a.x + r * a.x_sr + off));
      if (ACT != kActNone) gv[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(a.g + r * a.g_sr + off));
      dyv[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(a.dy + r * a.dy_sr + off));
      rs[u] = a.rstd[r * a.G + hh];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t r = rb + u * R;
      if (r < r1) {
        float x[8], g[8], dy[8], dx[8], dg[8], wdy[8];
        unpack8v<Tr>(xv[u], x);
        if (ACT != kActNone) unpack8v<Tr>(gv[u], g);
        unpack8v<Tr>(dyv[u], dy);
        float c1 = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float xhat = x[e] * rs[u];
          const float yn = xhat * w[e];
          float dyn = dy[e];
          if (ACT != kActNone) {
            const float s = sigmoidf(g[e]);
            if (ACT == kActSwish) {
              dg[e] = dy[e] * yn * (s + g[e] * s * (1.f - s));
              dyn = dy[e] * g[e] * s;
            } else {
              dg[e] = dy[e] * yn * s * (1.f - s);
              dyn = dy[e] * s;
            }
          }
          dw[e] += dyn * xhat;
          wdy[e] = dyn * w[e];
          c1 += xhat * wdy[e];
          x[e] = xhat;
        }
#pragma unroll
        for (int o = CH / 2; o > 0; o >>= 1) c1 += __shfl_xor(c1, o);
        c1 *= 1.0f / D;
#pragma unroll
        for (int e = 0; e < 8; ++e) dx[e] = (wdy[e] - x[e] * c1) * rs[u];
        // Every input is read once (non-temporal loads above).  With a gate the kernel writes two streams and the
        // non-temporal hint on the stores pays as well (0.277 -> 0.262 ms at B4 T16384 H16 D128); with dx alone it costs.
        if (ACT != kActNone) {
          __builtin_nontemporal_store(pack8v<Tr>(dx), reinterpret_cast<u32x4*>(a.dx + r * a.dx_sr + off));
          __builtin_nontemporal_store(pack8v<Tr>(dg), reinterpret_cast<u32x4*>(a.dg + r * a.dg_sr + off));
        } else {
          *reinterpret_cast<u32x4*>(a.dx + r * a.dx_sr + off) = pack8v<Tr>(dx);
        }
      }
    }
  }
  if (R > 1) {   // add the row lanes in order
#pragma unroll
    for (int e = 0; e < 8; ++e) dw_s[tid][e] = dw[e];
    __syncthreads();
    const float* flat = &dw_s[0][0];
    float* p = a.dw_partial + strip * a.G * D;
    for (int j = tid; j < a.cols * 8; j += blockDim.x) {
      float sum = flat[j];
#pragma unroll 8
      for (int q = 1; q < R; ++q) sum += flat[q * a.cols * 8 + j];
      p[j] = sum;
    }
  } else if (live) {
    float* p = a.dw_partial + strip * a.G * D + off;
    const f32x4 lo = {dw[0], dw[1], dw[2], dw[3]}, hi = {dw[4], dw[5], dw[6], dw[7]};
    *reinterpret_cast<f32x4*>(p) = lo;
    *reinterpret_cast<f32x4*>(p + 4) = hi;
  }
}

// dst[group][j] = sum of src[s][j] over the `per_group` consecutive rows s of the group, in a fixed order: 64 columns per
// workgroup, one per lane, its 16 waves taking every 16th row; the waves' sums are added in order.  Up to kReduceRows rows
// are added in one launch, more in two (groups of kReduceRows, then the groups' sums).
constexpr int kReduceRows = 512;
__global__ __launch_bounds__(1024) void reduce_rows_kernel(const float* __restrict__ src, float* __restrict__ dst, int64_t n_rows,
                                                           int width, int per_group) {
  __shared__ float part[16][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, j = blockIdx.x * 64 + lane;
  const int64_t s0 = (int64_t)blockIdx.y * per_group, s1 = min(n_rows, s0 + per_group);
  float acc = 0.f;
  if (j < width) {
    int64_t s = s0 + wave;
    for (; s + 7 * 16 < s1; s += 8 * 16) {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = src[(s + 16 * u) * width + j];
#pragma unroll
      for (int u = 0; u < 8; ++u) acc += v[u];
    }
    for (; s < s1; s += 16) acc += src[s * width + j];
  }
  part[wave][lane] = acc;
  __syncthreads();
  if (wave == 0 && j < width) {
    for (int q = 1; q < 16; ++q) acc += part[q][lane];
    dst[(int64_t)blockIdx.y * width + j] = acc;
  }
}

#define FOX_NG_INST(TR, DD)                                                   \
  template __global__ void norm_gate_fwd_kernel<TR, DD, kActSigmoid>(const NormGateK); \
  template __global__ void norm_gate_fwd_kernel<TR, DD, kActSwish>(const NormGateK);   \
  template __global__ void norm_gate_fwd_kernel<TR, DD, kActNone>(const NormGateK);    \
  template __global__ void norm_gate_bwd_kernel<TR, DD, kActSigmoid>(const NormGateK); \
  template __global__ void norm_gate_bwd_kernel<TR, DD, kActSwish>(const NormGateK);   \
  template __global__ void norm_gate_bwd_kernel<TR, DD, kActNone>(const NormGateK);
#define FOX_NG_INST_ALL(TR) FOX_NG_INST(TR, 16) FOX_NG_INST(TR, 32) FOX_NG_INST(TR, 64) FOX_NG_INST(TR, 128)
FOX_NG_INST_ALL(Bf16)
FOX_NG_INST_ALL(Fp16)

// How the backward of `rows` rows of G heads is cut: columns, row lanes, rows per lane, strips of lanes * rows_per_lane rows (one partial each).
struct NormBwdPlan {
  int cols, lanes, rows_per_lane;
  int64_t strips;
};
constexpr int kNormRowsPerLane = 32;   // at most
static NormBwdPlan norm_bwd_plan(int64_t rows, int G, int D) {
  NormBwdPlan p;
  p.cols = G * (D / 8);
  p.lanes = p.cols > 256 ? 1 : 256 / p.cols;
  // about four workgroups per CU, at least four rows per lane (what it keeps in flight)
  int64_t per = rows * ((p.cols + 255) / 256) / ((int64_t)p.lanes * 4 * kCus);
  per = per < 4 ? 4 : per > kNormRowsPerLane ? kNormRowsPerLane : per;
  p.rows_per_lane = (int)per;
  p.strips = (rows + p.lanes * per - 1) / (p.lanes * per);
  return p;
}
// Rows of G*D floats the backward needs as workspace, an upper bound over G and D: one per workgroup along the rows (with at least
// kNormRowsPerLane rows each, or about 4 * kCus of them for small calls) plus one per group of kReduceRows of those; what it
// adds for the groups is generous (callers were told one per 32).
int64_t norm_gate_workspace_rows(int64_t rows) {
  int64_t strips = (rows + kNormRowsPerLane - 1) / kNormRowsPerLane;
  const int64_t small = (rows + 3) / 4 < 8 * kCus ? (rows + 3) / 4 : 8 * kCus;
  strips = strips > small ? strips : small;
  return strips + (strips + 31) / 32;
}

template <typename Tr, int D>
static hipError_t norm_gate_d(const NormGateK& a, bool bwd, int act, hipStream_t s) {
  constexpr int CH = D / 8;
  if (!bwd) {
    const int64_t threads = (int64_t)a.R * a.G * CH;
    const dim3 grid((unsigned)((threads + 255) / 256));
    if (act == kActSwish) hipLaunchKernelGGL((norm_gate_fwd_kernel<Tr, D, kActSwish>), grid, dim3(256), 0, s, a);
    else if (act == kActNone) hipLaunchKernelGGL((norm_gate_fwd_kernel<Tr, D, kActNone>), grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((norm_gate_fwd_kernel<Tr, D, kActSigmoid>), grid, dim3(256), 0, s, a);
    return hipGetLastError();
  }
  const NormBwdPlan p = norm_bwd_plan(a.R, a.G, D);
  NormGateK k = a;
  k.cols = p.cols;
  k.rows_per_lane = p.rows_per_lane;
  const bool wide = p.cols > 256;
  const dim3 grid((unsigned)(wide ? (p.strips * p.cols + 255) / 256 : p.strips)), block(wide ? 256u : (unsigned)((p.cols * p.lanes + 63) / 64 * 64));
  if (act == kActSwish) hipLaunchKernelGGL((norm_gate_bwd_kernel<Tr, D, kActSwish>), grid, block, 0, s, k);
  else if (act == kActNone) hipLaunchKernelGGL((norm_gate_bwd_kernel<Tr, D, kActNone>), grid, block, 0, s, k);
  else hipLaunchKernelGGL((norm_gate_bwd_kernel<Tr, D, kActSigmoid>), grid, block, 0, s, k);
  const int width = a.G * D;
  const int64_t groups = (p.strips + kReduceRows - 1) / kReduceRows;
  const dim3 columns((unsigned)((width + 63) / 64));
  if (groups == 1) {
    hipLaunchKernelGGL(reduce_rows_kernel, columns, dim3(1024), 0, s, a.dw_partial, a.dw, p.strips, width, (int)p.strips);
    return hipGetLastError();
  }
  float* stage = a.dw_partial + p.strips * width;  // second part of the workspace
  hipLaunchKernelGGL(reduce_rows_kernel, dim3(columns.x, (unsigned)groups), dim3(1024), 0, s, a.dw_partial, stage, p.strips, width, kReduceRows);
  hipLaunchKernelGGL(reduce_rows_kernel, columns, dim3(1024), 0, s, stage, a.dw, groups, width, (int)groups);
  return hipGetLastError();
}

template <typename Tr>
static hipError_t norm_gate_t(const NormGateK& a, int D, bool bwd, int act, hipStream_t s) {
  switch (D) {
    case 16: return norm_gate_d<Tr, 16>(a, bwd, act, s);
    case 32: return norm_gate_d<Tr, 32>(a, bwd, act, s);
    case 64: return norm_gate_d<Tr, 64>(a, bwd, act, s);
    case 128: return norm_gate_d<Tr, 128>(a, bwd, act, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_norm_gate(const NormGateK& a, int D, int dtype, bool bwd, int act, hipStream_t s) {
  return dtype == 0 ? norm_gate_t<Bf16>(a, D, bwd, act, s) : norm_gate_t<Fp16>(a, D, bwd, act, s);
}

}  // namespace fox
