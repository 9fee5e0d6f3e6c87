// LayerNorm forward/backward and row softmax forward/backward for gfx950.
// All four are HBM-bound: one wave64 (long rows: one workgroup) owns one row, holds
// it in registers as 16-byte chunks (chunk c of the row belongs to lane c % 64), and
// reduces with cross-lane shuffles, so every element is read from HBM exactly once.
// ANY: rows of any length and alignment, in the same chunks (struct Row in rowops.h).  31713 rows of 1021 fp16
// elements: LayerNorm forward 58 -> 31 us (4.2 TB/s), backward 218 -> 55 us (3.5 TB/s) against element-wise
// loads; 4000 fp32 softmax rows of 777: 13.6 -> 7.6 and 11.8 -> 8.3 us.
#include "rowops.h"

namespace tfa {

constexpr int kRowsPerBlock = 4;  // 4 waves per workgroup, one row each
#ifndef TF_LN_FWD_ROWS
#define TF_LN_FWD_ROWS 2
#endif
constexpr int kLnFwdRowsPerWave = TF_LN_FWD_ROWS;  // rows a wave of the forward kernel walks (with the next one in flight)

// ---------------------------------------------------------------------------
// LayerNorm forward.  WPR = waves per row: 1 (a workgroup takes four rows) or 4 (one row); NV = 16-byte
// chunks per lane (row length <= NV * WPR * 64 * 8).
// ---------------------------------------------------------------------------
// sum of one value per lane over the waves of a row; `slot` alternates between consecutive uses, so that one
// barrier per sum is enough (a slot is rewritten two sums later, behind the barrier of the sum in between)
template <int WPR> __device__ __forceinline__ float row_sum(float v, float (*red)[4], int slot) {
  v = wave_sum(v);
  if constexpr (WPR == 1) return v;
  if ((threadIdx.x & 63) == 0) red[slot][threadIdx.x >> 6] = v;
  __syncthreads();
  return (red[slot][0] + red[slot][1]) + (red[slot][2] + red[slot][3]);
}

// Access to the chunks of a LayerNorm or softmax row of NV chunks per lane.  The chunk that crosses the end of a ragged row lies among a
// lane's upper NV / 2 (a row takes NV only if NV / 2 do not hold it): those are fetched as 16 bytes inside the row and
// moved down (Row::settle), so that no wave stands waiting for eight element loads in the midst of its prefetch.  fp16, us:
// backward 31713 x 1021 68.0 -> 46.0 (1024 columns: 42.2), 31713 x 777 60.7 -> 41.8, 20000 x 2051 121 -> 99, 8000 x 8191
// 156 -> 140; forward 31713 x 1021 33.0 -> 30.0, 8000 x 8191 69.7 -> 62.6; softmax 31713 x 1021 forward 26.3 -> 23.7, backward
// 36.5 -> 31.6, 16000 x 3001 41.2 -> 39.1 and 58.5 -> 53.0 (fp32 46.5 -> 44.9, 77 -> 74; forward rows of 257 to 259, where one lane has
// an upper chunk and three elements at the most, lose: 63488 x 259 24.1 -> 25.4, 261 to 511 gain 1 to 6 per cent).
template <typename T, int NV, bool ANY, int FROM = NV / 2> struct RowEnds {
  typedef Row<T, ANY> R;
  static __device__ __forceinline__ u32x4 fetch(const T* row, int c, int i, int n, T fill = (T)0.f) {
    return i >= FROM ? R::template fetch<true>(row, c, n, fill) : R::template fetch<false>(row, c, n, fill);
  }
  static __device__ __forceinline__ u32x4 settle(u32x4 raw, int c, int i, int n, T fill = (T)0.f) {
    return i >= FROM ? R::template settle<true>(raw, c, n, fill) : raw;
  }
  static __device__ __forceinline__ void store(T* row, int c, int i, int n, u32x4 v) {
    if (i >= FROM) R::template store<true>(row, c, n, v);
    else R::template store<false>(row, c, n, v);
  }
  // Elements of gamma or beta.  fp32 ones beyond one chunk per lane are read by elements at the end of the row: eight of them are
  // two accesses with moves each, which took the forward kernels from 101 to 146 registers, four waves per SIMD to three
  // (fp16, us, by elements / with moves / here: 8192 x 1025 12.2 / 15.9 / 12.5, 31713 x 1537 48 / 56 / 47, 2048 x 6001 with a
  // residual 22.0 / 25.8 / 20.9).
  template <typename TP> static __device__ __forceinline__ void load8(const TP* p, int c, int i, int n, float (&v)[8]) {
    if (i >= FROM && (sizeof(TP) == 2 || NV == 1)) load8_row<TP, ANY, true>(p, c, n, v);
    else load8_row<TP, ANY, false>(p, c, n, v);
  }
};

// With ADD the normalised row is s = x + res, rounded to T and also written to `sum`
// (the residual stream after the addition); the statistics are those of the rounded s,
// so the result equals an addition kernel followed by the plain forward.
template <typename T, typename TP, int NV, int WPR, bool ADD, bool ANY, bool ONCE>
__global__ __launch_bounds__(256) void ln_fwd_vec(int64_t rows, int d, const T* __restrict__ x, int64_t ldx,
                                                   const T* __restrict__ res, int64_t ldres,
                                                   T* __restrict__ sum, int64_t ldsum,
                                                   const TP* __restrict__ gamma, const TP* __restrict__ beta,
                                                   float eps, T* __restrict__ y, int64_t ldy,
                                                   float* __restrict__ mean_out, float* __restrict__ rstd_out) {
  // Wave w of workgroup b walks rows (b*4 + w) + k*4*grid.  The raw chunks of the wave's next row
  // are requested before the cross-lane sums of the current one, so that the reads of one row run
  // beside the reductions and the stores of the row before: with one row per wave and every wave
  // of the launch resident at once, the whole launch reads first and writes afterwards, and
  // neither half of the memory system's time is used by the other.
  // The add + LayerNorm instantiation must give the bits of an addition followed by the plain one:
  // no contraction left to the compiler (it may fuse differently per instantiation), the fused
  // operations are spelled out.
#pragma clang fp contract(off)
  typedef Row<T, ANY> R;
  // (four chunks per lane with a residual: 31713 x 1537 88 us by elements, 102 so)
  typedef RowEnds<T, NV, ANY, ADD && NV == 4 && WPR == 1 ? NV : NV / 2> E;
  __shared__ float red[2][4];
  const int lane = WPR == 1 ? threadIdx.x & 63 : threadIdx.x;  // lane within the row
  constexpr int LANES = 64 * WPR, RPB = kRowsPerBlock / WPR;
  const int nchunk = R::chunks(d);
  const int64_t stride = (int64_t)gridDim.x * RPB;
  u32x4 raw_x[NV], raw_r[ADD ? NV : 1];
  auto fetch = [&](int64_t row) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = lane + i * LANES;
      if (c < nchunk) {
        raw_x[i] = E::fetch(x + row * ldx, c, i, d);
        if (ADD) raw_r[i] = E::fetch(res + row * ldres, c, i, d);
      }
    }
  };
  int64_t row = (int64_t)blockIdx.x * RPB + (WPR == 1 ? threadIdx.x >> 6 : 0);
  if (row < rows) fetch(row);
  // ONCE: no wave has a second row.  gamma and beta are then requested here, behind x, and arrive beside it
  float g[NV][8], b[NV][8];
  auto params = [&](int i, int c) {
    E::template load8<TP>(gamma, c, i, d, g[i]);
    E::template load8<TP>(beta, c, i, d, b[i]);
  };
  if (ONCE) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = lane + i * LANES;
      if (c < nchunk) params(i, c);
    }
  }
  for (; row < rows; row += stride) {
    float v[NV][8];
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = lane + i * LANES;
      if (c < nchunk) {
        unpack8<T>(E::settle(raw_x[i], c, i, d), v[i]);
        if (ADD) {
          float r[8];
          unpack8<T>(E::settle(raw_r[i], c, i, d), r);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[i][e] += r[e];
          const u32x4 packed = pack8<T>(v[i]);
          E::store(sum + row * ldsum, c, i, d, packed);
          unpack8<T>(packed, v[i]);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) s += v[i][e];
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[i][e] = 0.f;
      }
    }
    if (!ONCE && row + stride < rows) fetch(row + stride);
    const float mean = row_sum<WPR>(s, red, 0) / (float)d;
    float q = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = lane + i * LANES;
      if (c < nchunk) {
        if (ANY && (c + 1) * 8 > d) {  // the chunk that crosses the end of the row
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float t = c * 8 + e < d ? v[i][e] - mean : 0.f;
            q = __builtin_fmaf(t, t, q);
          }
          continue;
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) { const float t = v[i][e] - mean; q = __builtin_fmaf(t, t, q); }
      }
    }
    const float var = row_sum<WPR>(q, red, 1) / (float)d;
    const float rstd = 1.0f / sqrtf(var + eps);
    if (lane == 0) { mean_out[row] = mean; rstd_out[row] = rstd; }
    T* yr = y + row * ldy;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = lane + i * LANES;
      if (c < nchunk) {
        // (gamma and beta are fetched per row where there are several: held in registers across the rows a wave walks they
        // cost a wave of occupancy, 98 against 86 VGPRs, and the kernel 0.5 us at d = 1024)
        if (!ONCE) params(i, c);
        float o[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          o[e] = __builtin_fmaf((v[i][e] - mean) * rstd, g[i][e], b[i][e]);
          // the fp32 value is pinned before the rounding to 16 bits: left alone, the compiler turns
          // some of these into v_fma_mix*_f16 (one rounding straight to 16 bits) and others not,
          // differently per instantiation, and the two forms differ in one element in 50 000
          asm("" : "+v"(o[e]));
        }
        E::store(yr, c, i, d, pack8<T>(o));
      }
    }
  }
}

// Rows beyond the registers of a workgroup, and ragged ones of few columns: scalar loads, three passes over the row (the
// second and third come from cache).
template <typename T, typename TP, bool ADD>
__global__ __launch_bounds__(256) void ln_fwd_any(int64_t rows, int d, const T* __restrict__ x, int64_t ldx,
                                                   const T* __restrict__ res, int64_t ldres,
                                                   T* __restrict__ sum, int64_t ldsum,
                                                   const TP* __restrict__ gamma, const TP* __restrict__ beta,
                                                   float eps, T* __restrict__ y, int64_t ldy,
                                                   float* __restrict__ mean_out, float* __restrict__ rstd_out) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * kRowsPerBlock + (threadIdx.x >> 6);
  if (row >= rows) return;
  const T* xr = x + row * ldx;
  if (ADD) {
    // every lane re-reads only the columns it wrote itself
    T* sr = sum + row * ldsum;
    for (int c = lane; c < d; c += 64) sr[c] = (T)((float)xr[c] + (float)res[row * ldres + c]);
    xr = sr;
  }
  float s = 0.f;
  for (int c = lane; c < d; c += 64) s += (float)xr[c];
  const float mean = wave_sum(s) / (float)d;
  float q = 0.f;
  for (int c = lane; c < d; c += 64) { const float t = (float)xr[c] - mean; q += t * t; }
  const float rstd = 1.0f / sqrtf(wave_sum(q) / (float)d + eps);
  if (lane == 0) { mean_out[row] = mean; rstd_out[row] = rstd; }
  T* yr = y + row * ldy;
  for (int c = lane; c < d; c += 64)
    yr[c] = (T)__builtin_fmaf(((float)xr[c] - mean) * rstd, (float)gamma[c], (float)beta[c]);
}

// ---------------------------------------------------------------------------
// LayerNorm backward.  Wave w of workgroup b walks rows (b*4 + w) + k*4*grid.
// dx is written per row; dgamma/dbeta partial sums stay in registers, are
// summed over the 4 waves through LDS and land in partial[b][0|1][d].
// The raw 16-byte chunks of the wave's next row are requested before the
// cross-lane sums of the current row, so a wave always has loads in flight.
// With ADD, dsum (the gradient that reaches the normalised tensor by another
// path, e.g. along a residual stream) is added to dx before the rounding.
// ---------------------------------------------------------------------------
template <typename T, typename TP, int NV, int WPR, bool ADD, bool ANY>
__global__ __launch_bounds__(256) void ln_bwd_vec(int64_t rows, int d, const T* __restrict__ dy, int64_t lddy,
                                                   const T* __restrict__ dsum, int64_t lddsum,
                                                   const T* __restrict__ x, int64_t ldx,
                                                   const TP* __restrict__ gamma, const float* __restrict__ mean,
                                                   const float* __restrict__ rstd, T* __restrict__ dx,
                                                   int64_t lddx, float* __restrict__ partial) {
  typedef Row<T, ANY> R;
  // (four chunks per lane with a residual by elements: with the moves it takes 276 registers, one wave per SIMD -- 31713 x 1025
  // 69 us by elements, 81 with them, 8192 x 1537 35 and 39)
  typedef RowEnds<T, NV, ANY, ADD && NV == 4 && WPR == 1 ? NV : NV / 2> E;
  extern __shared__ float dyn[];  // WPR == 1: [4][d] for the sums of the four waves; then [d] for gamma when G_LDS
  __shared__ float red[2][4];
  // Wide rows (NV >= 4) keep gamma in LDS as fp32 and read a chunk where it is used: held in registers its
  // 8 * NV values pushed the kernel past 256 registers, one wave per SIMD and one workgroup per CU, so that
  // the 512 workgroups of a launch ran in two turns (d = 2048: 23.4 us per launch with it, 67 MB).
  constexpr bool G_LDS = NV >= 4;
  constexpr int LANES = 64 * WPR, RPB = kRowsPerBlock / WPR;
  const int lane = WPR == 1 ? threadIdx.x & 63 : threadIdx.x;  // lane within the row
  const int wave = threadIdx.x >> 6;
  const int nchunk = R::chunks(d);
  float* const gam = dyn + (WPR == 1 ? 4 * d : 0);
  float g[G_LDS ? 1 : NV][8], dg[NV][8], db[NV][8];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = lane + i * LANES;
#pragma unroll
    for (int e = 0; e < 8; ++e) { dg[i][e] = 0.f; db[i][e] = 0.f; }
    if constexpr (!G_LDS) {
#pragma unroll
      for (int e = 0; e < 8; ++e) g[i][e] = 0.f;
      if (c < nchunk) E::template load8<TP>(gamma, c, i, d, g[i]);
    }
  }
  if constexpr (G_LDS) {
    for (int c = threadIdx.x; c < nchunk; c += 256) {
      float gv[8];
      load8_row<TP, ANY>(gamma, c, d, gv);
#pragma unroll
      for (int e = 0; e < 8; ++e) gam[c * 8 + e] = gv[e];  // (whole chunks: the buffer is padded to them)
    }
    __syncthreads();
  }
  const float inv_d = 1.0f / (float)d;
  const int64_t stride = (int64_t)gridDim.x * RPB;
  u32x4 raw_x[NV], raw_dy[NV], raw_ds[ADD ? NV : 1];
  float mu_next = 0.f, rs_next = 0.f;
  auto fetch = [&](int64_t row) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = lane + i * LANES;
      if (c < nchunk) {
        raw_x[i] = E::fetch(x + row * ldx, c, i, d);
        raw_dy[i] = E::fetch(dy + row * lddy, c, i, d);
        if (ADD) raw_ds[i] = E::fetch(dsum + row * lddsum, c, i, d);
      }
    }
    mu_next = mean[row];
    rs_next = rstd[row];
  };
  int64_t row = (int64_t)blockIdx.x * RPB + (WPR == 1 ? wave : 0);
  if (row < rows) fetch(row);
  for (; row < rows; row += stride) {
    const float mu = mu_next, rs = rs_next;
    float xh[NV][8], gd[NV][8], ds[ADD ? NV : 1][8];
    float s1 = 0.f, s2 = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = lane + i * LANES;
      if (c < nchunk) {
        float xv[8], dv[8], gl[8];
        unpack8<T>(E::settle(raw_x[i], c, i, d), xv);
        unpack8<T>(E::settle(raw_dy[i], c, i, d), dv);
        if (ADD) unpack8<T>(E::settle(raw_ds[i], c, i, d), ds[i]);
#pragma unroll
        for (int e = 0; e < 8; ++e) gl[e] = G_LDS ? gam[c * 8 + e] : g[G_LDS ? 0 : i][e];
#pragma unroll
        for (int e = 0; e < 8; ++e) {  // (beyond the end of the row dy reads as zero: nothing reaches a sum)
          xh[i][e] = (xv[e] - mu) * rs;
          gd[i][e] = dv[e] * gl[e];
          s1 += gd[i][e] * xh[i][e];
          s2 += gd[i][e];
          dg[i][e] += dv[e] * xh[i][e];
          db[i][e] += dv[e];
        }
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) { xh[i][e] = 0.f; gd[i][e] = 0.f; }
      }
    }
    if (row + stride < rows) fetch(row + stride);
    const float c1 = row_sum<WPR>(s1, red, 0) * inv_d;
    const float c2 = row_sum<WPR>(s2, red, 1) * inv_d;
    T* dxr = dx + row * lddx;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = lane + i * LANES;
      if (c < nchunk) {
        float o[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          o[e] = (gd[i][e] - xh[i][e] * c1 - c2) * rs;
          if (ADD) o[e] += ds[i][e];
        }
        E::store(dxr, c, i, d, pack8<T>(o));
      }
    }
  }
  float* pout = partial + (int64_t)blockIdx.x * 2 * d;
  if constexpr (WPR > 1) {  // every column belongs to one thread of the workgroup
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = lane + i * LANES;
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (c * 8 + e < d) { pout[c * 8 + e] = dg[i][e]; pout[d + c * 8 + e] = db[i][e]; }
    }
    return;
  }
  // cross-wave reduction, dgamma then dbeta, through one [4][d] LDS buffer
#pragma unroll
  for (int which = 0; which < 2; ++which) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = lane + i * LANES;
      if (c < nchunk) {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (!ANY || c * 8 + e < d) dyn[wave * d + c * 8 + e] = which ? db[i][e] : dg[i][e];
      }
    }
    __syncthreads();
    for (int c = threadIdx.x; c < d; c += 256)
      pout[which * d + c] = dyn[c] + dyn[d + c] + dyn[2 * d + c] + dyn[3 * d + c];
  }
}

template <typename T, typename TP, bool ADD>
__global__ __launch_bounds__(256) void ln_bwd_any(int64_t rows, int d, const T* __restrict__ dy, int64_t lddy,
                                                   const T* __restrict__ dsum, int64_t lddsum,
                                                   const T* __restrict__ x, int64_t ldx,
                                                   const TP* __restrict__ gamma, const float* __restrict__ mean,
                                                   const float* __restrict__ rstd, T* __restrict__ dx,
                                                   int64_t lddx, float* __restrict__ partial) {
  // One workgroup per slice of rows; every thread owns columns tid, tid+256, ...
  // so the dgamma/dbeta partials need no cross-thread reduction; the per-row
  // sums are reduced per wave, with all 4 waves walking the same row.
  __shared__ float sred[2][4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const float inv_d = 1.0f / (float)d;
  float* pout = partial + (int64_t)blockIdx.x * 2 * d;
  for (int c = threadIdx.x; c < d; c += 256) { pout[c] = 0.f; pout[d + c] = 0.f; }
  for (int64_t row = blockIdx.x; row < rows; row += gridDim.x) {
    const float mu = mean[row], rs = rstd[row];
    const T* xr = x + row * ldx;
    const T* dyr = dy + row * lddy;
    float s1 = 0.f, s2 = 0.f;
    for (int c = threadIdx.x; c < d; c += 256) {
      const float xh = ((float)xr[c] - mu) * rs, dv = (float)dyr[c], gd = dv * (float)gamma[c];
      s1 += gd * xh;
      s2 += gd;
      pout[c] += dv * xh;
      pout[d + c] += dv;
    }
    s1 = wave_sum(s1);
    s2 = wave_sum(s2);
    __syncthreads();
    if (lane == 0) { sred[0][wave] = s1; sred[1][wave] = s2; }
    __syncthreads();
    const float c1 = (sred[0][0] + sred[0][1] + sred[0][2] + sred[0][3]) * inv_d;
    const float c2 = (sred[1][0] + sred[1][1] + sred[1][2] + sred[1][3]) * inv_d;
    T* dxr = dx + row * lddx;
    for (int c = threadIdx.x; c < d; c += 256) {
      const float xh = ((float)xr[c] - mu) * rs, gd = (float)dyr[c] * (float)gamma[c];
      float o = (gd - xh * c1 - c2) * rs;
      if (ADD) o += (float)dsum[row * lddsum + c];
      dxr[c] = (T)o;
    }
  }
}

// Second stage over partial viewed as a [nparts][2d] matrix (dgamma columns then
// dbeta columns): workgroup = 16 columns x 16 row slices, slices summed in a
// fixed order through LDS.  Four independent running sums per thread keep
// several loads in flight.
template <typename T>
__global__ __launch_bounds__(256) void ln_bwd_reduce(int nparts, int d, const float* __restrict__ partial,
                                                      T* __restrict__ dgamma, T* __restrict__ dbeta) {
  __shared__ float red[16][17];
  const int cl = threadIdx.x & 15, slice = threadIdx.x >> 4;
  const int col = blockIdx.x * 16 + cl;  // 0 .. 2d-1
  float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f;
  if (col < 2 * d) {
    const float* src = partial + col;
    const int64_t ld = 2 * (int64_t)d;
    int p = slice;
    for (; p + 48 < nparts; p += 64) {
      a0 += src[(int64_t)p * ld];
      a1 += src[(int64_t)(p + 16) * ld];
      a2 += src[(int64_t)(p + 32) * ld];
      a3 += src[(int64_t)(p + 48) * ld];
    }
    for (; p < nparts; p += 16) a0 += src[(int64_t)p * ld];
  }
  red[slice][cl] = (a0 + a1) + (a2 + a3);
  __syncthreads();
  if (slice == 0 && col < 2 * d) {
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k) s += red[k][cl];
    if (col < d) dgamma[col] = (T)s;
    else dbeta[col - d] = (T)s;
  }
}

// The same second stage for the partial sums of several LayerNorms in one launch (blockIdx.y = LayerNorm):
// the parameter gradients of a whole backward pass, whose partial sums were left in place by the row passes.
constexpr int kLnReduceBatch = 64;
struct LnReduceItem {
  const float* partial;
  void* dgamma;
  void* dbeta;
  int parts;
};
struct LnReduceBatch { LnReduceItem it[kLnReduceBatch]; };
template <typename T>
__global__ __launch_bounds__(256) void ln_bwd_reduce_batch(LnReduceBatch batch, int d) {
  __shared__ float red[16][17];
  const LnReduceItem r = batch.it[blockIdx.y];
  const int cl = threadIdx.x & 15, slice = threadIdx.x >> 4;
  const int col = blockIdx.x * 16 + cl;  // 0 .. 2d-1
  float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f;
  if (col < 2 * d) {
    const float* src = r.partial + col;
    const int64_t ld = 2 * (int64_t)d;
    int p = slice;
    for (; p + 48 < r.parts; p += 64) {
      a0 += src[(int64_t)p * ld];
      a1 += src[(int64_t)(p + 16) * ld];
      a2 += src[(int64_t)(p + 32) * ld];
      a3 += src[(int64_t)(p + 48) * ld];
    }
    for (; p < r.parts; p += 16) a0 += src[(int64_t)p * ld];
  }
  red[slice][cl] = (a0 + a1) + (a2 + a3);
  __syncthreads();
  if (slice == 0 && col < 2 * d) {
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k) s += red[k][cl];
    if (col < d) ((T*)r.dgamma)[col] = (T)s;
    else ((T*)r.dbeta)[col - d] = (T)s;
  }
}

// ---------------------------------------------------------------------------
// Softmax (T = f16 / bf16 / float).  NV chunks of Chunk<T>::N elements per lane.
// ---------------------------------------------------------------------------
template <typename T> __device__ __forceinline__ void row_floats(u32x4 raw, float (&v)[Chunk<T>::N]) {
  if constexpr (sizeof(T) == 2) unpack8<T>(raw, v);
  else {
    const f32x4 f = __builtin_bit_cast(f32x4, raw);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = f[i];
  }
}
template <typename T, int N> __device__ __forceinline__ u32x4 row_pack(const float (&v)[N]) {
  if constexpr (sizeof(T) == 2) return pack8<T>(v);
  else {
    const f32x4 f = {v[0], v[1], v[2], v[3]};
    return __builtin_bit_cast(u32x4, f);
  }
}

// Sum of a chunk in pairs, as the sums of lanes and waves are, so that the error of a row's sum stays below that of one
// element per lane and step (fp32 rows of 8191: 7.2e-8 of the result with serial sums over chunks and waves, 6.2e-8 by
// elements, 5.2e-8 so).
__device__ __forceinline__ float pair_sum(const float (&v)[4]) { return (v[0] + v[1]) + (v[2] + v[3]); }
__device__ __forceinline__ float pair_sum(const float (&v)[8]) {
  return ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
}

template <typename T, int NV, bool ANY>
__global__ __launch_bounds__(256) void softmax_fwd_vec(int64_t rows, int cols, const T* __restrict__ x,
                                                        int64_t ldx, T* __restrict__ y, int64_t ldy) {
  typedef RowEnds<T, NV, ANY> E;
  constexpr int N = Chunk<T>::N;
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * kRowsPerBlock + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int nchunk = Row<T, ANY>::chunks(cols);
  const T* xr = x + row * ldx;
  float v[NV][N];
  float m = -INFINITY;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = lane + i * 64;
    if (c < nchunk) {
      row_floats<T>(E::settle(E::fetch(xr, c, i, cols, (T)-INFINITY), c, i, cols, (T)-INFINITY), v[i]);
#pragma unroll
      for (int e = 0; e < N; ++e) m = fmaxf(m, v[i][e]);
    }
  }
  m = wave_max(m);
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    if (lane + i * 64 < nchunk) {
#pragma unroll
      for (int e = 0; e < N; ++e) v[i][e] = exp2f((v[i][e] - m) * kLog2e);
      s += pair_sum(v[i]);
    }
  }
  const float inv = 1.0f / wave_sum(s);
  T* yr = y + row * ldy;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = lane + i * 64;
    if (c < nchunk) {
#pragma unroll
      for (int e = 0; e < N; ++e) v[i][e] *= inv;
      E::store(yr, c, i, cols, row_pack<T>(v[i]));
    }
  }
}

template <typename T>
__global__ __launch_bounds__(256) void softmax_fwd_any(int64_t rows, int cols, const T* __restrict__ x,
                                                        int64_t ldx, T* __restrict__ y, int64_t ldy) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * kRowsPerBlock + (threadIdx.x >> 6);
  if (row >= rows) return;
  const T* xr = x + row * ldx;
  float m = -INFINITY;
  for (int c = lane; c < cols; c += 64) m = fmaxf(m, (float)xr[c]);
  m = wave_max(m);
  float s = 0.f;
  for (int c = lane; c < cols; c += 64) s += exp2f(((float)xr[c] - m) * kLog2e);
  const float inv = 1.0f / wave_sum(s);
  T* yr = y + row * ldy;
  for (int c = lane; c < cols; c += 64) yr[c] = (T)(exp2f(((float)xr[c] - m) * kLog2e) * inv);
}

template <typename T, int NV, bool ANY>
__global__ __launch_bounds__(256) void softmax_bwd_vec(int64_t rows, int cols, const T* __restrict__ dy,
                                                        int64_t lddy, const T* __restrict__ y, int64_t ldy,
                                                        T* __restrict__ dx, int64_t lddx) {
  typedef RowEnds<T, NV, ANY> E;
  constexpr int N = Chunk<T>::N;
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * kRowsPerBlock + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int nchunk = Row<T, ANY>::chunks(cols);
  float yv[NV][N], gv[NV][N];
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = lane + i * 64;
    if (c < nchunk) {
      const u32x4 ry = E::fetch(y + row * ldy, c, i, cols), rg = E::fetch(dy + row * lddy, c, i, cols);
      row_floats<T>(E::settle(ry, c, i, cols), yv[i]);
      row_floats<T>(E::settle(rg, c, i, cols), gv[i]);
      float p[N];
#pragma unroll
      for (int e = 0; e < N; ++e) p[e] = yv[i][e] * gv[i][e];
      s += pair_sum(p);
    }
  }
  s = wave_sum(s);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = lane + i * 64;
    if (c < nchunk) {
      float o[N];
#pragma unroll
      for (int e = 0; e < N; ++e) o[e] = yv[i][e] * (gv[i][e] - s);
      E::store(dx + row * lddx, c, i, cols, row_pack<T>(o));
    }
  }
}

template <typename T>
__global__ __launch_bounds__(256) void softmax_bwd_any(int64_t rows, int cols, const T* __restrict__ dy,
                                                        int64_t lddy, const T* __restrict__ y, int64_t ldy,
                                                        T* __restrict__ dx, int64_t lddx) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * kRowsPerBlock + (threadIdx.x >> 6);
  if (row >= rows) return;
  float s = 0.f;
  for (int c = lane; c < cols; c += 64) s += (float)y[row * ldy + c] * (float)dy[row * lddy + c];
  s = wave_sum(s);
  for (int c = lane; c < cols; c += 64)
    dx[row * lddx + c] = (T)((float)y[row * ldy + c] * ((float)dy[row * lddy + c] - s));
}

// ---------------------------------------------------------------------------
// Long rows (beyond the 512 chunks a single wave holds: vocabulary-sized rows): one workgroup of 16
// waves per row, the row in registers as NV 16-byte chunks per thread (chunk c of thread t:
// t + 1024 c), wave sums merged through LDS.  Every element is read once and written once, as in
// the wave-per-row kernels.
// ---------------------------------------------------------------------------
constexpr int kLongRowThreads = 1024;
// all-reduce of one value per thread over the workgroup; `slot` distinguishes consecutive uses
template <bool MAX> __device__ __forceinline__ float block_reduce16(float v, float* red, int slot) {
  v = MAX ? wave_max(v) : wave_sum(v);
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) red[slot * 16 + wave] = v;
  __syncthreads();
  float r[16];
#pragma unroll
  for (int w = 0; w < 16; ++w) r[w] = red[slot * 16 + w];
#pragma unroll
  for (int h = 8; h > 0; h >>= 1)
#pragma unroll
    for (int w = 0; w < h; ++w) r[w] = MAX ? fmaxf(r[w], r[w + h]) : r[w] + r[w + h];
  return r[0];
}

// Exponentials of the non-positive arguments of a chunk.  Whole rows: v_exp_f32 as it is, results below 2^-126 become zero
// (as they always have there).  ANY: a chunk that has such a result takes the library function, which keeps the subnormal
// numbers (taken for every chunk: 4000 x 4097 fp32 28.4 -> 31.4 us, so 29.8).
template <bool ANY, int N> __device__ __forceinline__ void long_exp2(float (&v)[N]) {
  float least = 0.f;
#pragma unroll
  for (int e = 0; e < N; ++e) least = fminf(least, v[e]);
  if (ANY && least < -126.f) {
#pragma unroll
    for (int e = 0; e < N; ++e) v[e] = exp2f(v[e]);
  } else {
#pragma unroll
    for (int e = 0; e < N; ++e) v[e] = __builtin_amdgcn_exp2f(v[e]);
  }
}
// The chunk that crosses the end of a ragged row, fetched as the 16 bytes that end with it.  Called behind a branch that one
// wave of the row takes: the empty statement keeps the moves from being made for every chunk.  Eight tested element loads in
// its place, each waited for, held the row up at the workgroup's reduction (us, forward / backward): fp16 4000 x 5001
// 48.1 -> 28.6 / 37.8 -> 30.0, 2000 x 20001 47.7 -> 38.1 / 52.0 -> 49.1, 4096 x 50257 200 -> 195 / 294 -> 286; fp32 2000 x 33001
// 110 -> 106 / 170 -> 161.  (All loads of the row ahead of the first conversion: the same forward, the backward of 50304
// fp16 columns 212 -> 216 and 2 % slower in ragged rows, fp32 rows of 8 chunks in scratch.)
template <typename T> __device__ __forceinline__ void long_row_end(u32x4& raw, int c, int cols, T fill = (T)0.f) {
  asm volatile("");
  raw = Row<T, true>::template settle<true>(raw, c, cols, fill);
}
template <typename T, int NV, bool ANY>
__global__ __launch_bounds__(kLongRowThreads) void softmax_fwd_long(int cols, const T* __restrict__ x, int64_t ldx,
                                                                    T* __restrict__ y, int64_t ldy) {
  constexpr int N = Chunk<T>::N;
  __shared__ float red[32];
  const int64_t row = blockIdx.x;
  const int nchunk = Row<T, ANY>::chunks(cols);
  const T* xr = x + row * ldx;
  float v[NV][N];
  float m = -INFINITY;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = threadIdx.x + i * kLongRowThreads;
    if (c < nchunk) {
      u32x4 raw = Row<T, ANY>::template fetch<true, true>(xr, c, cols, (T)-INFINITY);
      if (ANY && (c + 1) * N > cols) long_row_end<T>(raw, c, cols, (T)-INFINITY);
      row_floats<T>(raw, v[i]);
#pragma unroll
      for (int e = 0; e < N; ++e) m = fmaxf(m, v[i][e]);
    }
  }
  m = block_reduce16<true>(m, red, 0);
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    if ((int)threadIdx.x + i * kLongRowThreads < nchunk) {
      // (the difference first: x * log2e - m * log2e, one multiply-add, overflows for rows at the type's lowest value,
      // and from |m| of 1e10 on the rounding of m * log2e alone exceeds the range of the exponential.  The operation
      // more shows where few rows leave the memory idle: 100 x 65536 fp32 9.5 -> 9.9 us, 1000 x 8192 fp16 7.3 -> 7.4)
#pragma unroll
      for (int e = 0; e < N; ++e) v[i][e] = (v[i][e] - m) * kLog2e;
      long_exp2<ANY>(v[i]);
      s += pair_sum(v[i]);
    }
  }
  const float inv = 1.0f / block_reduce16<false>(s, red, 1);
  T* yr = y + row * ldy;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = threadIdx.x + i * kLongRowThreads;
    if (c < nchunk) {
#pragma unroll
      for (int e = 0; e < N; ++e) v[i][e] *= inv;
      Row<T, ANY>::store(yr, c, cols, row_pack<T>(v[i]));
    }
  }
}

// y and dy stay in registers as the raw 16-byte chunks (converted where they are used: as floats, 16-bit
// rows would need twice the registers); with HOLD_DY false dy is read a second time instead (from the
// cache: a row is a few hundred KB), for rows whose two operands do not fit the 128 registers of a thread.
template <typename T, int NV, bool HOLD_DY, bool ANY>
__global__ __launch_bounds__(kLongRowThreads) void softmax_bwd_long(int cols, const T* __restrict__ dy, int64_t lddy,
                                                                    const T* __restrict__ y, int64_t ldy,
                                                                    T* __restrict__ dx, int64_t lddx) {
  constexpr int N = Chunk<T>::N;
  __shared__ float red[16];
  const int64_t row = blockIdx.x;
  const int nchunk = Row<T, ANY>::chunks(cols);
  u32x4 ry[NV], rg[HOLD_DY ? NV : 1];
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = threadIdx.x + i * kLongRowThreads;
    if (c < nchunk) {
      ry[i] = Row<T, ANY>::template fetch<true, true>(y + row * ldy, c, cols);
      u32x4 g = Row<T, ANY>::template fetch<true, HOLD_DY>(dy + row * lddy, c, cols);
      if (ANY && (c + 1) * N > cols) {
        long_row_end<T>(ry[i], c, cols);
        long_row_end<T>(g, c, cols);
      }
      if (HOLD_DY) rg[i] = g;
      float yv[N], gv[N];
      row_floats<T>(ry[i], yv);
      row_floats<T>(g, gv);
#pragma unroll
      for (int e = 0; e < N; ++e) s += yv[e] * gv[e];
    }
  }
  s = block_reduce16<false>(s, red, 0);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = threadIdx.x + i * kLongRowThreads;
    if (c < nchunk) {
      u32x4 g = HOLD_DY ? rg[i] : Row<T, ANY>::template fetch<true>(dy + row * lddy, c, cols);
      if (!HOLD_DY && ANY && (c + 1) * N > cols) long_row_end<T>(g, c, cols);
      float yv[N], gv[N], o[N];
      row_floats<T>(ry[i], yv);
      row_floats<T>(g, gv);
#pragma unroll
      for (int e = 0; e < N; ++e) o[e] = yv[e] * (gv[e] - s);
      Row<T, ANY>::store(dx + row * lddx, c, cols, row_pack<T>(o));
    }
  }
}
// chunks per thread of the long-row kernels for a row of `nchunk` chunks (0: beyond them)
template <typename T> static int pick_long_nv(int64_t nchunk) {
  if (nchunk <= 4 * kLongRowThreads) return 4;
  if (nchunk <= 8 * kLongRowThreads) return 8;
  if (nchunk <= 16 * kLongRowThreads && sizeof(T) == 4) return 16;  // 65536 elements of either width
  return 0;
}

// ---------------------------------------------------------------------------
// host dispatch
// ---------------------------------------------------------------------------
static int pick_nv(int64_t nchunk) {
  if (nchunk <= 64) return 1;
  if (nchunk <= 128) return 2;
  if (nchunk <= 256) return 4;
  if (nchunk <= 512) return 8;
  return 0;
}

// Ragged rows of at most one element per lane go by elements: 63488 x 33 fp16, LayerNorm forward 17.0 us against 21.9 in
// chunks, softmax 13.9 against 18.5, softmax backward 10.2 against 14.2.  (LayerNorm backward, whose column sums dominate: 124 in
// elements, 36 in chunks.)
constexpr int64_t kFewCols = 64;

// LayerNorm: 16-byte chunks per lane.  Rows of up to kLnWaveRow elements belong to one wave, longer ones (up to
// 8192) to the four waves of a workgroup: held by one wave, a row of 4096 takes 8 chunks per lane, and the backward
// kernel's five arrays of 64 values do not fit the registers.
constexpr int64_t kLnWaveRow = 2048;
static int ln_pick(int64_t nchunk) {
  if (nchunk <= 64) return 1;
  if (nchunk <= 128) return 2;
  if (nchunk <= 256) return 4;
  if (nchunk <= 512) return 2;
  if (nchunk <= 1024) return 4;
  return 0;
}

template <typename T, typename TP, bool ADD>
static int ln_fwd_launch(hipStream_t st, int64_t rows, int64_t d, const void* x, int64_t ldx, const void* res,
                         int64_t ldres, void* sum, int64_t ldsum, const void* gamma, const void* beta, float eps,
                         void* y, int64_t ldy, float* mean, float* rstd) {
  const dim3 grid((unsigned)ceil_div(rows, kRowsPerBlock)), block(256);
  bool vec = row_vectorizable<T>(x, d, ldx) && row_vectorizable<T>(y, d, ldy) && aligned16(gamma) && aligned16(beta);
  if (ADD) vec = vec && row_vectorizable<T>(res, d, ldres) && row_vectorizable<T>(sum, d, ldsum);
  const int nv = !vec && d <= kFewCols ? 0 : ln_pick((d + 7) / 8), wpr = nv > 0 && d > kLnWaveRow ? 4 : 1;
  // the row-walking kernel: kLnFwdRowsPerWave rows per wave once there are enough rows to fill the chip
  const int64_t rpb = kRowsPerBlock / wpr;
  int64_t walkers = ceil_div(rows, rpb * kLnFwdRowsPerWave);
  const int64_t fill = (int64_t)device_shape().cus * 4;
  if (walkers < fill) walkers = ceil_div(rows, rpb) < fill ? ceil_div(rows, rpb) : fill;
  const dim3 wgrid((unsigned)walkers);
  // One row per wave and at most two workgroups per CU: gamma and beta beside x, not after the statistics, in registers that
  // nobody else needs.  A launch of few rows is a chain of latencies, and this was a whole one.  fp16 with a residual, fp32
  // parameters, us: 128 x 768 3.75 -> 3.09, 128 x 1024 3.69 -> 3.10 (fp16 parameters 3.64 -> 3.21), 960 x 768 4.43 -> 3.83,
  // 512 x 1536 5.21 -> 4.14, 128 x 2048 5.37 -> 3.95, 2048 x 2048 10.5 -> 8.9, 512 x 8192 10.7 -> 9.3.  With four workgroups
  // per CU the registers cost waves: 4096 x 1024 9.05 -> 9.54, 4096 x 2048 16.1 -> 17.5, without a residual 9.3 -> 10.6.  (Both sides
  // with the sums through the LDS crossbar; either is 0.3 shorter with wave_sum as it is.)
  // (One chunk per lane of 16-bit parameters, 960 x 256, 3.22 -> 3.29: as before.)
  const bool once = vec && rows <= walkers * rpb && walkers <= fill / 2;
#define LN_ARGS                                                                                                    \
  (rows, (int)d, (const T*)x, ldx, (const T*)res, ldres, (T*)sum, ldsum, (const TP*)gamma, (const TP*)beta, eps, (T*)y, \
   ldy, mean, rstd)
#define LN_FWD(NV, WPR)                                                        \
  if (once) ln_fwd_vec<T, TP, NV, WPR, ADD, false, (NV > 1 || sizeof(TP) == 4)><<<wgrid, block, 0, st>>>LN_ARGS; \
  else if (vec) ln_fwd_vec<T, TP, NV, WPR, ADD, false, false><<<wgrid, block, 0, st>>>LN_ARGS; \
  else ln_fwd_vec<T, TP, NV, WPR, ADD, true, false><<<wgrid, block, 0, st>>>LN_ARGS
  switch (nv * 10 + wpr) {
    case 11: LN_FWD(1, 1); break;
    case 21: LN_FWD(2, 1); break;
    case 41: LN_FWD(4, 1); break;
    case 24: LN_FWD(2, 4); break;
    case 44: LN_FWD(4, 4); break;
    default: ln_fwd_any<T, TP, ADD><<<grid, block, 0, st>>>LN_ARGS;
  }
#undef LN_FWD
#undef LN_ARGS
  TF_CHECK_LAUNCH();
  return TF_OK;
}

static int ln_bwd_parts(int64_t rows) {
  int64_t g = (rows + kRowsPerBlock - 1) / kRowsPerBlock;
  return (int)(g < 512 ? g : 512);
}

template <typename T, typename TP, bool ADD>
static int ln_bwd_launch(hipStream_t st, int64_t rows, int64_t d, const void* dy, int64_t lddy, const void* dsum,
                         int64_t lddsum, const void* x, int64_t ldx, const void* gamma, const float* mean,
                         const float* rstd, void* dx, int64_t lddx, void* dgamma, void* dbeta, float* partial) {
  const int parts = ln_bwd_parts(rows);
  bool vec = row_vectorizable<T>(x, d, ldx) && row_vectorizable<T>(dy, d, lddy) && row_vectorizable<T>(dx, d, lddx) &&
             aligned16(gamma);
  if (ADD) vec = vec && row_vectorizable<T>(dsum, d, lddsum);
  const int nv = ln_pick((d + 7) / 8), wpr = nv > 0 && d > kLnWaveRow ? 4 : 1;
  // sums of the four waves of a workgroup (not needed where they share their rows); wide rows keep gamma there too
  const size_t lds = (size_t)((wpr == 1 ? 4 * d : 0) + (nv >= 4 ? (d + 7) / 8 * 8 : 0)) * sizeof(float);
#define LN_ARGS                                                                                                   \
  (rows, (int)d, (const T*)dy, lddy, (const T*)dsum, lddsum, (const T*)x, ldx, (const TP*)gamma, mean, rstd, (T*)dx, lddx, \
   partial)
#define LN_BWD(NV, WPR)                                                                   \
  if (vec) ln_bwd_vec<T, TP, NV, WPR, ADD, false><<<dim3(parts), dim3(256), lds, st>>>LN_ARGS; \
  else ln_bwd_vec<T, TP, NV, WPR, ADD, true><<<dim3(parts), dim3(256), lds, st>>>LN_ARGS
  switch (nv * 10 + wpr) {
    case 11: LN_BWD(1, 1); break;
    case 21: LN_BWD(2, 1); break;
    case 41: LN_BWD(4, 1); break;
    case 24: LN_BWD(2, 4); break;
    case 44: LN_BWD(4, 4); break;
    default: ln_bwd_any<T, TP, ADD><<<dim3(parts), dim3(256), 0, st>>>LN_ARGS;
  }
#undef LN_BWD
#undef LN_ARGS
  TF_CHECK_LAUNCH();
  if (!dgamma) return TF_OK;  // the partial sums stay where they are, for tf_layernorm_param_grads
  ln_bwd_reduce<TP><<<dim3(ceil_div(2 * d, 16)), dim3(256), 0, st>>>(parts, (int)d, partial, (TP*)dgamma, (TP*)dbeta);
  TF_CHECK_LAUNCH();
  return TF_OK;
}

template <typename T>
static int softmax_fwd_launch(hipStream_t st, int64_t rows, int64_t cols, const void* x, int64_t ldx, void* y,
                              int64_t ldy) {
  const dim3 grid((unsigned)ceil_div(rows, kRowsPerBlock)), block(256);
  const bool vec = row_vectorizable<T>(x, cols, ldx) && row_vectorizable<T>(y, cols, ldy);
  const int64_t nchunk = ceil_div(cols, Chunk<T>::N);
  const bool few = !vec && cols <= kFewCols;
  const int nv = few ? 0 : pick_nv(nchunk);
#define SM_FWD(NV)                                                                                        \
  if (vec) softmax_fwd_vec<T, NV, false><<<grid, block, 0, st>>>(rows, (int)cols, (const T*)x, ldx, (T*)y, ldy); \
  else softmax_fwd_vec<T, NV, true><<<grid, block, 0, st>>>(rows, (int)cols, (const T*)x, ldx, (T*)y, ldy)
  switch (nv) {
    case 1: SM_FWD(1); break;
    case 2: SM_FWD(2); break;
    case 4: SM_FWD(4); break;
    case 8: SM_FWD(8); break;
    default: {
      const int lnv = !few && rows <= 0x7fffffff ? pick_long_nv<T>(nchunk) : 0;
      const dim3 lgrid((unsigned)rows), lblock(kLongRowThreads);
#define SM_FWD_LONG(TT, NV)                                                                                         \
  do {                                                                                                              \
    if (vec) softmax_fwd_long<TT, NV, false><<<lgrid, lblock, 0, st>>>((int)cols, (const TT*)x, ldx, (TT*)y, ldy);    \
    else softmax_fwd_long<TT, NV, true><<<lgrid, lblock, 0, st>>>((int)cols, (const TT*)x, ldx, (TT*)y, ldy);         \
  } while (0)
      if (lnv == 4) SM_FWD_LONG(T, 4);
      else if (lnv == 8) SM_FWD_LONG(T, 8);
      else if (lnv == 16 && sizeof(T) == 4) SM_FWD_LONG(float, 16);
      else softmax_fwd_any<T><<<grid, block, 0, st>>>(rows, (int)cols, (const T*)x, ldx, (T*)y, ldy);
    }
  }
#undef SM_FWD
#undef SM_FWD_LONG
  TF_CHECK_LAUNCH();
  return TF_OK;
}

template <typename T>
static int softmax_bwd_launch(hipStream_t st, int64_t rows, int64_t cols, const void* dy, int64_t lddy,
                              const void* y, int64_t ldy, void* dx, int64_t lddx) {
  const dim3 grid((unsigned)ceil_div(rows, kRowsPerBlock)), block(256);
  const bool vec =
      row_vectorizable<T>(dy, cols, lddy) && row_vectorizable<T>(y, cols, ldy) && row_vectorizable<T>(dx, cols, lddx);
  const int64_t nchunk = ceil_div(cols, Chunk<T>::N);
  const bool few = !vec && cols <= kFewCols;
  const int nv = few ? 0 : pick_nv(nchunk);
#define SM_ARGS (rows, (int)cols, (const T*)dy, lddy, (const T*)y, ldy, (T*)dx, lddx)
#define SM_BWD(NV)                                                      \
  if (vec) softmax_bwd_vec<T, NV, false><<<grid, block, 0, st>>>SM_ARGS; \
  else softmax_bwd_vec<T, NV, true><<<grid, block, 0, st>>>SM_ARGS
  switch (nv) {
    case 1: SM_BWD(1); break;
    case 2: SM_BWD(2); break;
    case 4: SM_BWD(4); break;
    case 8: SM_BWD(8); break;
    default: {
      const int lnv = !few && rows <= 0x7fffffff ? pick_long_nv<T>(nchunk) : 0;
      const dim3 lgrid((unsigned)rows), lblock(kLongRowThreads);
#define SM_LARGS(TT) ((int)cols, (const TT*)dy, lddy, (const TT*)y, ldy, (TT*)dx, lddx)
#define SM_BWD_LONG(TT, NV, HOLD)                                                           \
  do {                                                                                      \
    if (vec) softmax_bwd_long<TT, NV, HOLD, false><<<lgrid, lblock, 0, st>>>SM_LARGS(TT);     \
    else softmax_bwd_long<TT, NV, HOLD, true><<<lgrid, lblock, 0, st>>>SM_LARGS(TT);          \
  } while (0)
      if (lnv == 4) SM_BWD_LONG(T, 4, true);
      else if (lnv == 8) SM_BWD_LONG(T, 8, true);
      else if (lnv == 16 && sizeof(T) == 4) SM_BWD_LONG(float, 16, false);
      else softmax_bwd_any<T><<<grid, block, 0, st>>>(rows, (int)cols, (const T*)dy, lddy, (const T*)y, ldy, (T*)dx, lddx);
#undef SM_BWD_LONG
#undef SM_LARGS
    }
  }
#undef SM_BWD
#undef SM_ARGS
  TF_CHECK_LAUNCH();
  return TF_OK;
}

static bool bad_rows(int64_t rows, int64_t n, int64_t ld) {
  return rows < 0 || n <= 0 || n > (1 << 30) || ld < n || rows > (int64_t)kRowsPerBlock * 0x7fffffff;
}

}  // namespace tfa

using namespace tfa;

template <bool ADD>
static int ln_fwd_entry(void* stream, int dtype, int param_dtype, int64_t rows, int64_t d, const void* x, int64_t ldx,
                        const void* res, int64_t ldres, void* sum, int64_t ldsum, const void* gamma,
                        const void* beta, float eps, void* y, int64_t ldy, float* mean, float* rstd) {
  if (!x || !gamma || !beta || !y || !mean || !rstd) return TF_EINVAL;
  if (ADD && (!res || !sum || ldres < d || ldsum < d)) return TF_EINVAL;
  if (bad_rows(rows, d, ldx) || ldy < d) return TF_EINVAL;
  if (rows == 0) return TF_OK;
  hipStream_t st = (hipStream_t)stream;
  if (param_dtype != dtype && param_dtype != TF_F32) return TF_EDTYPE;
#define LN_FWD_GO(T, TP) \
  return ln_fwd_launch<T, TP, ADD>(st, rows, d, x, ldx, res, ldres, sum, ldsum, gamma, beta, eps, y, ldy, mean, rstd)
  if (dtype == TF_F16) { if (param_dtype == TF_F32) LN_FWD_GO(f16, float); else LN_FWD_GO(f16, f16); }
  if (dtype == TF_BF16) { if (param_dtype == TF_F32) LN_FWD_GO(bf16, float); else LN_FWD_GO(bf16, bf16); }
#undef LN_FWD_GO
  return TF_EDTYPE;
}

extern "C" int tf_layernorm_fwd(void* stream, int dtype, int param_dtype, int64_t rows, int64_t d, const void* x,
                                int64_t ldx, const void* gamma, const void* beta, float eps, void* y, int64_t ldy,
                                float* mean, float* rstd) {
  return ln_fwd_entry<false>(stream, dtype, param_dtype, rows, d, x, ldx, nullptr, 0, nullptr, 0, gamma, beta, eps, y,
                             ldy, mean, rstd);
}

extern "C" int tf_add_layernorm_fwd(void* stream, int dtype, int param_dtype, int64_t rows, int64_t d, const void* x,
                                    int64_t ldx, const void* res, int64_t ldres, void* sum, int64_t ldsum,
                                    const void* gamma, const void* beta, float eps, void* y, int64_t ldy, float* mean,
                                    float* rstd) {
  return ln_fwd_entry<true>(stream, dtype, param_dtype, rows, d, x, ldx, res, ldres, sum, ldsum, gamma, beta, eps, y,
                            ldy, mean, rstd);
}

extern "C" int64_t tf_layernorm_bwd_partial_bytes(int64_t rows, int64_t d) {
  if (rows <= 0 || d <= 0) return 0;
  return (int64_t)ln_bwd_parts(rows) * 2 * d * (int64_t)sizeof(float);
}

template <bool ADD>
static int ln_bwd_entry(void* stream, int dtype, int param_dtype, int64_t rows, int64_t d, const void* dy,
                        int64_t lddy, const void* dsum, int64_t lddsum, const void* x, int64_t ldx,
                        const void* gamma, const float* mean, const float* rstd, void* dx, int64_t lddx,
                        void* dgamma, void* dbeta, float* partial, int64_t partial_bytes) {
  if (!dy || !x || !gamma || !mean || !rstd || !dx || (dgamma == nullptr) != (dbeta == nullptr)) return TF_EINVAL;
  if (ADD && (!dsum || lddsum < d)) return TF_EINVAL;
  if (bad_rows(rows, d, ldx) || lddy < d || lddx < d || rows == 0) return TF_EINVAL;
  if (!partial || partial_bytes < tf_layernorm_bwd_partial_bytes(rows, d)) return TF_EWORKSPACE;
  hipStream_t st = (hipStream_t)stream;
  if (param_dtype != dtype && param_dtype != TF_F32) return TF_EDTYPE;
#define LN_BWD_GO(T, TP)                                                                                          \
  return ln_bwd_launch<T, TP, ADD>(st, rows, d, dy, lddy, dsum, lddsum, x, ldx, gamma, mean, rstd, dx, lddx, dgamma, \
                                   dbeta, partial)
  if (dtype == TF_F16) { if (param_dtype == TF_F32) LN_BWD_GO(f16, float); else LN_BWD_GO(f16, f16); }
  if (dtype == TF_BF16) { if (param_dtype == TF_F32) LN_BWD_GO(bf16, float); else LN_BWD_GO(bf16, bf16); }
#undef LN_BWD_GO
  return TF_EDTYPE;
}

extern "C" int tf_layernorm_bwd(void* stream, int dtype, int param_dtype, int64_t rows, int64_t d, const void* dy,
                                int64_t lddy, const void* x, int64_t ldx, const void* gamma, const float* mean,
                                const float* rstd, void* dx, int64_t lddx, void* dgamma, void* dbeta,
                                float* partial, int64_t partial_bytes) {
  return ln_bwd_entry<false>(stream, dtype, param_dtype, rows, d, dy, lddy, nullptr, 0, x, ldx, gamma, mean, rstd, dx,
                             lddx, dgamma, dbeta, partial, partial_bytes);
}

extern "C" int tf_add_layernorm_bwd(void* stream, int dtype, int param_dtype, int64_t rows, int64_t d, const void* dy,
                                    int64_t lddy, const void* dsum, int64_t lddsum, const void* x, int64_t ldx,
                                    const void* gamma, const float* mean, const float* rstd, void* dx, int64_t lddx,
                                    void* dgamma, void* dbeta, float* partial, int64_t partial_bytes) {
  return ln_bwd_entry<true>(stream, dtype, param_dtype, rows, d, dy, lddy, dsum, lddsum, x, ldx, gamma, mean, rstd, dx,
                            lddx, dgamma, dbeta, partial, partial_bytes);
}

extern "C" int64_t tf_layernorm_bwd_parts(int64_t rows) { return rows > 0 ? ln_bwd_parts(rows) : 0; }

extern "C" int tf_layernorm_param_grads(void* stream, int param_dtype, int64_t d, int count,
                                        const tf_ln_param_grads* items) {
  if (count < 0 || d <= 0 || d > 0x3fffffff || (count > 0 && !items)) return TF_EINVAL;
  if (param_dtype != TF_F16 && param_dtype != TF_BF16 && param_dtype != TF_F32) return TF_EDTYPE;
  for (int i = 0; i < count; ++i)
    if (!items[i].partial || !items[i].dgamma || !items[i].dbeta || items[i].parts < 1 || items[i].parts > 512)
      return TF_EINVAL;
  hipStream_t st = (hipStream_t)stream;
  for (int base = 0; base < count; base += kLnReduceBatch) {
    const int n = count - base < kLnReduceBatch ? count - base : kLnReduceBatch;
    LnReduceBatch b = {};
    for (int i = 0; i < n; ++i)
      b.it[i] = {items[base + i].partial, items[base + i].dgamma, items[base + i].dbeta, (int)items[base + i].parts};
    const dim3 grid((unsigned)ceil_div(2 * d, 16), (unsigned)n), block(256);
    if (param_dtype == TF_F32) ln_bwd_reduce_batch<float><<<grid, block, 0, st>>>(b, (int)d);
    else if (param_dtype == TF_F16) ln_bwd_reduce_batch<f16><<<grid, block, 0, st>>>(b, (int)d);
    else ln_bwd_reduce_batch<bf16><<<grid, block, 0, st>>>(b, (int)d);
    TF_CHECK_LAUNCH();
  }
  return TF_OK;
}

extern "C" int tf_softmax_fwd(void* stream, int dtype, int64_t rows, int64_t cols, const void* x, int64_t ldx,
                              void* y, int64_t ldy) {
  if (!x || !y) return TF_EINVAL;
  if (bad_rows(rows, cols, ldx) || ldy < cols) return TF_EINVAL;
  if (rows == 0) return TF_OK;
  hipStream_t st = (hipStream_t)stream;
  switch (dtype) {
    case TF_F16: return softmax_fwd_launch<f16>(st, rows, cols, x, ldx, y, ldy);
    case TF_BF16: return softmax_fwd_launch<bf16>(st, rows, cols, x, ldx, y, ldy);
    case TF_F32: return softmax_fwd_launch<float>(st, rows, cols, x, ldx, y, ldy);
  }
  return TF_EDTYPE;
}

extern "C" int tf_softmax_bwd(void* stream, int dtype, int64_t rows, int64_t cols, const void* dy, int64_t lddy,
                              const void* y, int64_t ldy, void* dx, int64_t lddx) {
  if (!dy || !y || !dx) return TF_EINVAL;
  if (bad_rows(rows, cols, ldy) || lddy < cols || lddx < cols) return TF_EINVAL;
  if (rows == 0) return TF_OK;
  hipStream_t st = (hipStream_t)stream;
  switch (dtype) {
    case TF_F16: return softmax_bwd_launch<f16>(st, rows, cols, dy, lddy, y, ldy, dx, lddx);
    case TF_BF16: return softmax_bwd_launch<bf16>(st, rows, cols, dy, lddy, y, ldy, dx, lddx);
    case TF_F32: return softmax_bwd_launch<float>(st, rows, cols, dy, lddy, y, ldy, dx, lddx);
  }
  return TF_EDTYPE;
}
