// RMSNorm forward and backward for gfx950.
//
// Forward takes the place of rmsnorm_twoPassAlgo_e8
// (kernel_src/csrc/rms_norm/rms_norm_cutlass.cu:81-159): out = x * rms * w with
// rms = 1 / sqrt(mean(x^2) + eps) per row, rms kept as float for the backward.
// The reference reads every row twice; here a row stays in registers between
// the sum of squares and the scaling, so it is read once.
//
// Backward takes the place of the tensor expressions of rms_norm.backward
// (src/loquetier_src/kernel_utils.py:169-176):
//   dot = sum_j g*w*x,  dx = (g*w - x*dot*rms^2/n) * rms,  dw = sum_rows x*rms*g
// in float throughout, one pass over x and g; dw is summed per workgroup into a
// float partial and folded by a second launch in fixed order (no atomics).
//
// Both are streaming kernels bound by HBM: 2*n bytes read + 2*n written per
// row forward, 4*n read + 2*n written backward.
#pragma once
#include "smlm_common.hpp"

namespace smlm {

constexpr int kRmsChunks = 8;                       // 512-element chunks a wave keeps in registers
constexpr int kRmsWaveCols = 512 * kRmsChunks;      // columns one wave covers
constexpr int kRmsMaxCols = 4 * kRmsWaveCols;       // four waves per row at most

// Sum over the wave with DPP adds (shifts inside rows of 16 lanes, then the
// row totals); every lane returns the total.
__device__ __forceinline__ float wave_sum_f32(float x) {
#define SMLM_DPP_ADD(ctrl, rmask)                                                                      \
  x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), ctrl, rmask, \
                                                             0xf, false))
  SMLM_DPP_ADD(0x111, 0xf);  // row_shr:1
  SMLM_DPP_ADD(0x112, 0xf);  // row_shr:2
  SMLM_DPP_ADD(0x114, 0xf);  // row_shr:4
  SMLM_DPP_ADD(0x118, 0xf);  // row_shr:8
  SMLM_DPP_ADD(0x142, 0xa);  // row_bcast:15 into rows 1 and 3
  SMLM_DPP_ADD(0x143, 0xc);  // row_bcast:31 into rows 2 and 3
#undef SMLM_DPP_ADD
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), 63));
}

template <int DT>
__device__ __forceinline__ void unpack8(u32x4 v, float (&f)[8]) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    f[2 * e] = Num<DT>::lo(v[e]);
    f[2 * e + 1] = Num<DT>::hi(v[e]);
  }
}

struct RmsFwdArgs {
  uint16_t* out;        // [rows, cols]
  float* rms;           // [rows]
  const uint16_t* x;    // [rows, cols]
  const uint16_t* w;    // [cols]
  int rows, cols;
  float eps;
};

// WPR waves share a row (1: cols <= 4096, 4: cols <= 16384); a workgroup of four
// waves handles 4 / WPR rows at a time and walks rows blockIdx.x * (4 / WPR),
// + gridDim.x * (4 / WPR), ...  Chunk i of wave v covers the 512 columns starting
// at (i * WPR + v) * 512, eight per lane.  When a workgroup has more than one
// turn, the next row is on its way from memory while the current one is
// reduced, scaled and stored.  (Measured: one turn per workgroup is fastest.)
// x is read and the output written non-temporally: both are touched once per launch (the next
// reader of x is the backward, much later; a reader of the output that follows at once still
// finds it in the caches when it fits them).
template <int DT, int WPR, bool ONE_TURN>
__global__ __launch_bounds__(256) void rms_fwd_kernel(RmsFwdArgs a) {
  __shared__ float part[2][4];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int sub = wave % WPR;
  constexpr int kRows = 4 / WPR;
  const u32x4 zero = {0u, 0u, 0u, 0u};

  bool ok[kRmsChunks];
  u32x4 wv[kRmsChunks], xv[kRmsChunks];
#pragma unroll
  for (int i = 0; i < kRmsChunks; ++i) {
    const int col = ((i * WPR + sub) * 64 + lane) * 8;
    ok[i] = col < a.cols;
    wv[i] = ldg16(a.w + (ok[i] ? col : 0));
  }
  auto load_row = [&](int row, u32x4 (&v)[kRmsChunks]) {
    const uint16_t* xr = a.x + (long)(row < a.rows ? row : 0) * a.cols;
#pragma unroll
    for (int i = 0; i < kRmsChunks; ++i) {
      const int col = ((i * WPR + sub) * 64 + lane) * 8;
      v[i] = ldg16_nt(xr + (ok[i] ? col : 0));
    }
  };
  const int step = (int)gridDim.x * kRows;
  int row = (int)blockIdx.x * kRows + wave / WPR;
  load_row(row, xv);
  int parity = 0;
  // WPR == 4: `row` is uniform over the workgroup, so every wave reaches the barrier
  for (; row < a.rows; row += step) {
    u32x4 xn[kRmsChunks];
    if (ONE_TURN) {
#pragma unroll
      for (int i = 0; i < kRmsChunks; ++i) xn[i] = zero;
    } else {
      // unconditional (past the last row it re-reads row 0): a branch around the loads would
      // make the wave wait for everything in flight where the paths join
      load_row(row + step, xn);
    }
    __builtin_amdgcn_sched_barrier(0);  // the next row's loads are issued before this row is used
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < kRmsChunks; ++i) {
      if (!ok[i]) xv[i] = zero;
      float f[8];
      unpack8<DT>(xv[i], f);
#pragma unroll
      for (int e = 0; e < 8; ++e) ss += f[e] * f[e];
    }
    ss = wave_sum_f32(ss);
    if (WPR > 1) {
      if (lane == 0) part[parity][wave] = ss;
      __syncthreads();  // one barrier a row: the two halves of `part` alternate
      ss = (part[parity][0] + part[parity][1]) + (part[parity][2] + part[parity][3]);
      parity ^= 1;
    }
    const float rms = 1.0f / sqrtf(ss / (float)a.cols + a.eps);
    if (lane == 0 && sub == 0) a.rms[row] = rms;
    uint16_t* orow = a.out + (long)row * a.cols;
#pragma unroll
    for (int i = 0; i < kRmsChunks; ++i) {
      const int col = ((i * WPR + sub) * 64 + lane) * 8;
      if (!ok[i]) continue;
      float f[8], g[8];
      unpack8<DT>(xv[i], f);
      unpack8<DT>(wv[i], g);
      u32x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = pack2<DT>(f[2 * e] * rms * g[2 * e], f[2 * e + 1] * rms * g[2 * e + 1]);
      stg16_nt(orow + col, o);
    }
#pragma unroll
    for (int i = 0; i < kRmsChunks; ++i) xv[i] = xn[i];
  }
}

struct RmsBwdArgs {
  uint16_t* dx;         // [rows, cols]
  float* partial;       // [gridDim.x, cols] per-workgroup sums of x*rms*g
  const uint16_t* g;    // [rows, cols] upstream gradient
  const uint16_t* x;    // [rows, cols]
  const uint16_t* w;    // [cols]
  const float* rms;     // [rows]
  int rows, cols;
};

// A workgroup walks the rows R at a time, blockIdx.x * R, + gridDim.x * R, ...; a thread takes 8 columns (CH = 1, up to
// 8192 columns: as many threads as a row has pieces of 8, in whole waves) or 16 (CH = 2: half as many threads) and
// keeps its columns of w and its share of dw in registers.  The dots of the R rows cross the waves through LDS
// together, one barrier for them; the next rows are on their way meanwhile.
// Bound by HBM: three passes of 2 bytes an element.  A thread per column piece keeps a lane's registers few (dw is
// eight floats) and the rows in flight many.  Neighbouring workgroups work on neighbouring rows: with a contiguous
// share each, all of them stand at the same place modulo the share and meet in few HBM channels.  Whole backward with
// its fold, bf16, us, a wave to a row of up to 4096 columns (64 columns a lane, 208 registers) and four waves to a
// wider one / contiguous shares / interleaved: 4096 x 4096 26.0 / 24.3 / 23.2, 8192 x 4096 46.4 / 41.0 / 38.0,
// 8192 x 6144 80.6 / 67.2 / 55.0, 4096 x 12288 66.7 / 70.1 / 57.6, 1000 x 16384 30.4 / 31.1 / 29.8,
// 4096 x 16384 85.6 / 83.0 / 76.7, 300 x 1024 12.0 / 6.5 / 6.3, 4096 x 2048 17.4 / 17.1 / 16.5.
template <int DT, int CH, int R>
__global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(4))) void rms_bwd_kernel(RmsBwdArgs a) {
  typedef float dots_t __attribute__((ext_vector_type(R)));
  __shared__ dots_t part[2][16];  // the rows' dots by wave, two halves in turn
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, nw = (int)blockDim.x >> 6;
  const float inv_n = 1.0f / (float)a.cols;
  const int step = (int)gridDim.x * R;

  int col[CH];
  bool ok[CH];
  u32x4 wv[CH];
  float dw[CH][8];
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    col[i] = ((int)threadIdx.x + i * (int)blockDim.x) * 8;
    ok[i] = col[i] < a.cols;
    if (!ok[i]) col[i] = 0;
    wv[i] = ldg16(a.w + col[i]);
#pragma unroll
    for (int e = 0; e < 8; ++e) dw[i][e] = 0.0f;
  }
  // rows past the last re-read it and are not used
  auto load = [&](int row, u32x4 (&xr)[R][CH], u32x4 (&gr)[R][CH], float (&r)[R]) {
#pragma unroll
    for (int t = 0; t < R; ++t) {
      const int rr = row + t < a.rows ? row + t : a.rows - 1;
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        xr[t][i] = ldg16_nt(a.x + (long)rr * a.cols + col[i]);
        gr[t][i] = ldg16_nt(a.g + (long)rr * a.cols + col[i]);
      }
      r[t] = uload(a.rms, rr);
    }
  };
  u32x4 xv[R][CH], gv[R][CH];
  float rms[R];
  load((int)blockIdx.x * R, xv, gv, rms);
  int parity = 0;
  for (int row = (int)blockIdx.x * R; row < a.rows; row += step) {  // uniform over the workgroup
    u32x4 xn[R][CH], gn[R][CH];
    float rn[R];
    // unconditional (past the end it re-reads these rows): a branch around the loads would make the wave wait
    // for everything in flight where the paths join
    load(row + step < a.rows ? row + step : row, xn, gn, rn);
    __builtin_amdgcn_sched_barrier(0);  // the next rows' loads are issued before these rows are used
    dots_t dots;
#pragma unroll
    for (int t = 0; t < R; ++t) {
      float dot = 0.0f;
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        float xf[8], gf[8], wf[8];
        unpack8<DT>(xv[t][i], xf);
        unpack8<DT>(gv[t][i], gf);
        unpack8<DT>(wv[i], wf);
        float d = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) d += gf[e] * wf[e] * xf[e];
        dot += ok[i] ? d : 0.0f;  // (a column read past the row is column 0, whose g or x may be infinite or NaN)
      }
      dots[t] = wave_sum_f32(dot);
    }
    if (lane == 0) part[parity][wave] = dots;
    __syncthreads();
    dots = part[parity][0];
    for (int v = 1; v < nw; ++v) dots += part[parity][v];
    parity ^= 1;
#pragma unroll
    for (int t = 0; t < R; ++t) {
      if (row + t >= a.rows) break;  // uniform over the workgroup
      const float coef = dots[t] * rms[t] * rms[t] * inv_n;
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        float xf[8], gf[8], wf[8];
        unpack8<DT>(xv[t][i], xf);
        unpack8<DT>(gv[t][i], gf);
        unpack8<DT>(wv[i], wf);
        u32x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          o[e] = pack2<DT>((gf[2 * e] * wf[2 * e] - xf[2 * e] * coef) * rms[t],
                           (gf[2 * e + 1] * wf[2 * e + 1] - xf[2 * e + 1] * coef) * rms[t]);
        if (ok[i]) stg16_nt(a.dx + (long)(row + t) * a.cols + col[i], o);
#pragma unroll
        for (int e = 0; e < 8; ++e) dw[i][e] += xf[e] * rms[t] * gf[e];
      }
    }
#pragma unroll
    for (int t = 0; t < R; ++t) {
#pragma unroll
      for (int i = 0; i < CH; ++i) xv[t][i] = xn[t][i], gv[t][i] = gn[t][i];
      rms[t] = rn[t];
    }
  }

  float* prow = a.partial + (long)blockIdx.x * a.cols;
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    if (!ok[i]) continue;
    *(SMLM_GLOBAL f32x4*)(prow + col[i]) = f32x4{dw[i][0], dw[i][1], dw[i][2], dw[i][3]};
    *(SMLM_GLOBAL f32x4*)(prow + col[i] + 4) = f32x4{dw[i][4], dw[i][5], dw[i][6], dw[i][7]};
  }
}

// ---- rows wider than kRmsMaxCols: the row no longer fits the registers of four waves.  Plain
// two-pass kernels (the reference's own scheme, rms_norm_cutlass.cu:81-159): a workgroup per row
// walks the columns once for the reduction and once more for the output (the second pass mostly
// hits L2).  The backward keeps its share of dw in the float partial rows themselves, read and
// written once per row it handles.  Correct for any width that is a multiple of 8; not tuned.
__device__ __forceinline__ float block_sum_f32(float x, float* red4) {
  x = wave_sum_f32(x);
  __syncthreads();  // red4 is free again
  if ((threadIdx.x & 63) == 0) red4[threadIdx.x >> 6] = x;
  __syncthreads();
  return (red4[0] + red4[1]) + (red4[2] + red4[3]);
}

template <int DT>
__global__ __launch_bounds__(256) void rms_fwd_wide_kernel(RmsFwdArgs a) {
  __shared__ float red4[4];
  for (int row = blockIdx.x; row < a.rows; row += gridDim.x) {
    const uint16_t* xr = a.x + (long)row * a.cols;
    float ss = 0.0f;
    for (int col = threadIdx.x * 8; col < a.cols; col += 256 * 8) {
      float f[8];
      unpack8<DT>(ldg16(xr + col), f);
#pragma unroll
      for (int e = 0; e < 8; ++e) ss += f[e] * f[e];
    }
    ss = block_sum_f32(ss, red4);
    const float rms = 1.0f / sqrtf(ss / (float)a.cols + a.eps);
    if (threadIdx.x == 0) a.rms[row] = rms;
    uint16_t* orow = a.out + (long)row * a.cols;
    for (int col = threadIdx.x * 8; col < a.cols; col += 256 * 8) {
      float f[8], g[8];
      unpack8<DT>(ldg16(xr + col), f);
      unpack8<DT>(ldg16(a.w + col), g);
      u32x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = pack2<DT>(f[2 * e] * rms * g[2 * e], f[2 * e + 1] * rms * g[2 * e + 1]);
      stg16_nt(orow + col, o);
    }
  }
}

template <int DT>
__global__ __launch_bounds__(256) void rms_bwd_wide_kernel(RmsBwdArgs a) {
  __shared__ float red4[4];
  const float inv_n = 1.0f / (float)a.cols;
  float* prow = a.partial + (long)blockIdx.x * a.cols;
  bool first = true;
  for (int row = blockIdx.x; row < a.rows; row += gridDim.x) {
    const long off = (long)row * a.cols;
    float dot = 0.0f;
    for (int col = threadIdx.x * 8; col < a.cols; col += 256 * 8) {
      float xf[8], gf[8], wf[8];
      unpack8<DT>(ldg16(a.x + off + col), xf);
      unpack8<DT>(ldg16(a.g + off + col), gf);
      unpack8<DT>(ldg16(a.w + col), wf);
#pragma unroll
      for (int e = 0; e < 8; ++e) dot += gf[e] * wf[e] * xf[e];
    }
    dot = block_sum_f32(dot, red4);
    const float rms = a.rms[row], coef = dot * rms * rms * inv_n;
    for (int col = threadIdx.x * 8; col < a.cols; col += 256 * 8) {
      float xf[8], gf[8], wf[8];
      unpack8<DT>(ldg16(a.x + off + col), xf);
      unpack8<DT>(ldg16(a.g + off + col), gf);
      unpack8<DT>(ldg16(a.w + col), wf);
      u32x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        o[e] = pack2<DT>((gf[2 * e] * wf[2 * e] - xf[2 * e] * coef) * rms,
                         (gf[2 * e + 1] * wf[2 * e + 1] - xf[2 * e + 1] * coef) * rms);
      stg16_nt(a.dx + off + col, o);
      // this thread's columns of the workgroup's partial row: nobody else touches them
      f32x4 p0 = {0.f, 0.f, 0.f, 0.f}, p1 = p0;
      if (!first) p0 = ldg_f4(prow + col), p1 = ldg_f4(prow + col + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) p0[e] += xf[e] * rms * gf[e], p1[e] += xf[4 + e] * rms * gf[4 + e];
      *(SMLM_GLOBAL f32x4*)(prow + col) = p0;
      *(SMLM_GLOBAL f32x4*)(prow + col + 4) = p1;
    }
    first = false;
  }
  if (first)  // more workgroups than rows never happens (the host sizes the grid), but a partial row must not stay unwritten
    for (int col = threadIdx.x * 4; col < a.cols; col += 256 * 4) *(SMLM_GLOBAL f32x4*)(prow + col) = f32x4{0.f, 0.f, 0.f, 0.f};
}

struct RmsFoldArgs {
  uint16_t* dw;          // [cols]
  const float* partial;  // [n_part, cols]
  int n_part, cols;
};

// grid: ceil(cols / (4 * C4)), block 256: thread (rg = tid / C4, c4 = tid % C4) adds partial rows rg, rg + 256 / C4, ...
// of four columns; the row groups are then added across the lanes of each wave and the four waves through LDS, always
// in the same order.
template <int DT, int C4>
__global__ __launch_bounds__(256) void rms_fold_kernel(RmsFoldArgs a) {
  constexpr int kRmsFoldRows = 256 / C4;
  __shared__ f32x4 red[4][C4];
  const int rg = threadIdx.x / C4, c4 = threadIdx.x % C4, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int col = (int)blockIdx.x * 4 * C4 + c4 * 4;
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
  if (col < a.cols && rg < a.n_part) {
    // eight partial rows are requested at a time; rows past the end re-read row rg and are dropped
    for (int p0 = rg; p0 < a.n_part; p0 += 8 * kRmsFoldRows) {
      f32x4 v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int p = p0 + j * kRmsFoldRows;
        v[j] = ldg_f4(a.partial + (long)(p < a.n_part ? p : rg) * a.cols + col);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (p0 + j * kRmsFoldRows < a.n_part) s += v[j];
    }
  }
#pragma unroll
  for (int d = C4; d < kWaveSize; d *= 2)
#pragma unroll
    for (int e = 0; e < 4; ++e) s[e] += __shfl_xor(s[e], d, kWaveSize);
  if (lane < C4) red[wave][c4] = s;
  __syncthreads();
  if (threadIdx.x < C4 && col < a.cols) {
    const f32x4 t = (red[0][c4] + red[1][c4]) + (red[2][c4] + red[3][c4]);
    u32x2 o;
    o[0] = pack2<DT>(t[0], t[1]);
    o[1] = pack2<DT>(t[2], t[3]);
    *(SMLM_GLOBAL u32x2*)(a.dw + col) = o;
  }
}

}  // namespace smlm
