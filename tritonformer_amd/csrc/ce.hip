// Cross-entropy forward/backward for gfx950.  HBM-bound: the forward streams
// each logits row once (online max / sum-of-exp in the log2 domain), the
// backward streams it once more and writes the gradient, already multiplied by
// the upstream per-row gradient.  ANY: rows of any length and alignment (a vocabulary that
// nobody padded), in the same 16-byte chunks (struct Row in rowops.h): 4095 bf16 rows of 50257 entries
// forward 233 -> 81 us (5.1 TB/s), backward 208 -> 170 us (4.8 TB/s) against element-wise loads.
#include "rowops.h"

namespace tfa {

constexpr int kCeThreads = 256;

// v_exp_f32 as it is: the library exp2f wraps the same instruction in a range check and a rescaling
// (five instructions more per element) that only matter for results below 2^-126, which are
// flushed to zero here -- terms that do not change a sum of exponentials whose largest term is 1.
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
// The probabilities of a gradient chunk, exp2(x * log2e - l2).  ANY: also where they are subnormal numbers, which an
// upstream gradient may lift into the range of the type -- only a chunk that has one takes the library function
// (4095 x 50257 bf16, forward with gradient, as it then was: 246 us without, 276 with that function for every element, 263
// this way).
template <bool ANY> __device__ __forceinline__ void grad_probs(float (&v)[8], float l2) {
  float least = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) { v[e] = v[e] * kLog2e - l2; least = fminf(least, v[e]); }
  if (ANY && least < -126.f) {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = exp2f(v[e]);
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = fast_exp2(v[e]);
  }
}

struct MaxSum {
  float m;  // running max of x*log2e
  float s;  // running sum of exp2(x*log2e - m)
};
__device__ __forceinline__ MaxSum combine(MaxSum a, MaxSum b) {
  const float m = fmaxf(a.m, b.m);
  MaxSum r;
  r.m = m;
  // exp2f(-inf - finite) = 0; both -inf only when both are empty (s = 0).
  r.s = (m == -INFINITY) ? 0.f : a.s * exp2f(a.m - m) + b.s * exp2f(b.m - m);
  return r;
}

__device__ __forceinline__ MaxSum block_combine(MaxSum v, MaxSum* smem) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    MaxSum other;
    other.m = __shfl_xor(v.m, o, 64);
    other.s = __shfl_xor(v.s, o, 64);
    v = combine(v, other);
  }
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) smem[wave] = v;
  __syncthreads();
  MaxSum r = smem[0];
#pragma unroll
  for (int w = 1; w < kCeThreads / 64; ++w) r = combine(r, smem[w]);
  return r;
}

// Row r of the (rows, V) problem lives at (r / inner) * outer + (r % inner) * ld: with
// inner = S-1, ld = V, outer = S*V these are the rows of a (B, S, V) tensor without the
// last position of every sequence, i.e. the shifted logits read in place.
struct RowMap {
  int64_t ld, outer;
  int inner;
  __device__ __forceinline__ int64_t at(int64_t r) const { return (r / inner) * outer + (r % inner) * ld; }
};

template <typename T, bool ANY>
__global__ __launch_bounds__(kCeThreads) void ce_fwd(int V, const T* __restrict__ logits, RowMap map,
                                                      const int64_t* __restrict__ labels, T* __restrict__ loss,
                                                      float* __restrict__ lse) {
  __shared__ MaxSum smem[kCeThreads / 64];
  const int64_t row = blockIdx.x;
  const T* xr = logits + map.at(row);
  MaxSum acc = {-INFINITY, 0.f};
  const int nchunk = Row<T, ANY>::chunks(V);
  constexpr int U = 4;  // 16-byte loads in flight per thread
  for (int c0 = threadIdx.x; c0 < nchunk; c0 += U * kCeThreads) {
    u32x4 raw[U];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (c0 + u * kCeThreads < nchunk) raw[u] = Row<T, ANY>::template load<true>(xr, c0 + u * kCeThreads, V, (T)-INFINITY);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (c0 + u * kCeThreads >= nchunk) break;
      float v[8];
      unpack8<T>(raw[u], v);
      float cm = v[0];
#pragma unroll
      for (int e = 1; e < 8; ++e) cm = fmaxf(cm, v[e]);
      cm *= kLog2e;
      if (cm > acc.m) { acc.s *= exp2f(acc.m - cm); acc.m = cm; }
      // nothing but masked entries so far (-inf, or a lowest value whose multiple is): they count as exp2(-inf - 0),
      // where -inf - (-inf) is NaN
      const float shift = acc.m == -INFINITY ? 0.f : acc.m;
      float part = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) part += fast_exp2(v[e] * kLog2e - shift);
      acc.s += part;
    }
  }
  const MaxSum tot = block_combine(acc, smem);
  if (threadIdx.x == 0) {
    const float l = (tot.m + log2f(tot.s)) * kLn2;  // natural-log logsumexp
    lse[row] = l;
    const int64_t lab = labels[row];
    const float xl = (lab >= 0 && lab < V) ? (float)xr[lab] : 0.f;
    loss[row] = (T)(l - xl);
  }
}

// Forward for rows that fit into the registers of one workgroup (V <= 8 * NCH * kCeThreads): a
// thread requests all of its NCH 16-byte chunks at once -- NCH loads in flight instead of four --
// takes the row maximum first and then the sum of exponentials, both from registers.
// GRAD: the same pass also writes (softmax(row) - onehot(label)) * grad_scale to the row of
// `dlogits` -- the row is still in registers once its log-sum-exp is known, so the gradient of
// the loss with respect to the logits costs one write instead of a second read-and-write pass.
// (Up to 8 chunks: left to itself the compiler interleaves them all in 230 registers, two waves per SIMD, and a launch of
// many short rows takes its workgroups in turns: 8192 x 257 fp16 36 us, 11 with four waves, 14 in a loop over elements;
// 8192 x 8191 85, 28 and 63.)
template <typename T, int NCH, bool GRAD, bool ANY>
__global__ __launch_bounds__(kCeThreads, NCH == 8 ? 4 : 1) void ce_fwd_regs(int V, const T* __restrict__ logits, RowMap map,
                                                           const int64_t* __restrict__ labels, T* __restrict__ loss,
                                                           float* __restrict__ lse, T* __restrict__ dlogits,
                                                           RowMap dmap, float grad_scale) {
  __shared__ float red[2][kCeThreads / 64];
  const int64_t row = blockIdx.x;
  const T* xr = logits + map.at(row);
  const int nchunk = Row<T, ANY>::chunks(V);
  u32x4 raw[NCH];
#pragma unroll
  for (int u = 0; u < NCH; ++u) {
    const int c = threadIdx.x + u * kCeThreads;
    if (c < nchunk) raw[u] = Row<T, ANY>::template fetch<true, true>(xr, c, V, (T)-INFINITY);
  }
  float m = -INFINITY;
#pragma unroll
  for (int u = 0; u < NCH; ++u) {
    // (This test is an unsigned one, the signed one above another to the compiler: made to share it, the kernel of whole rows took
    // 54 registers for 48 and 8192 x 1000 fp16 11.4 us for 10.8, with gradient 16.1 for 15.4.)
    if (threadIdx.x + u * kCeThreads < nchunk) {
      const int c = threadIdx.x + u * kCeThreads;
      // The chunk that crosses the end of the row is the 16 bytes that end with it, moved down -- behind a branch that one
      // wave takes (the empty statement keeps the moves from being made for every chunk).  Eight tested element loads in
      // its place held up the loads in flight.  bf16 with gradient, us: 4095 x 50257 190 -> 173, 2047 x 33001 70.7 -> 58,
      // 8192 x 1001 24.0 -> 20.5; forward alone 8192 x 4097 19.1 -> 16.7, 8192 x 1001 13.3 -> 11.9, 4095 x 50257 82 as before.
      // (Fewer rows than CUs and 33000 columns and more lose a little: with gradient 256 x 50257 fp16 18.4 -> 19.4, 100 x 50257
      // 15.5 -> 16.3; 600 x 33001 27.8 -> 23.9.)
      if (ANY && (c + 1) * 8 > V) {
        asm volatile("");
        raw[u] = Row<T, ANY>::template settle<true>(raw[u], c, V, (T)-INFINITY);
      }
      float v[8];
      unpack8<T>(raw[u], v);
#pragma unroll
      for (int e = 0; e < 8; ++e) m = fmaxf(m, v[e]);
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) red[0][wave] = m;
  __syncthreads();
  m = red[0][0];
#pragma unroll
  for (int w = 1; w < kCeThreads / 64; ++w) m = fmaxf(m, red[0][w]);
  // The later passes convert the row again: bf16 rows kept as floats from one pass to the next took 25 chunks to 290
  // registers, one wave per SIMD (4095 x 50257 bf16, forward with gradient: 263 -> 188 us, 173 since; 50304 193 -> 153).
#pragma unroll
  for (int u = 0; u < NCH; ++u) asm("" : "+v"(raw[u]));
  const float m2 = m * kLog2e;
  float s = 0.f;
#pragma unroll
  for (int u = 0; u < NCH; ++u) {
    if (threadIdx.x + u * kCeThreads < nchunk) {
      float v[8];
      unpack8<T>(raw[u], v);
      float part = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) part += fast_exp2(v[e] * kLog2e - m2);
      s += part;
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  if ((threadIdx.x & 63) == 0) red[1][wave] = s;
  __syncthreads();
  float tot = red[1][0];
#pragma unroll
  for (int w = 1; w < kCeThreads / 64; ++w) tot += red[1][w];
  const float l = (m2 + log2f(tot)) * kLn2;  // natural-log logsumexp
  // back to the log2 domain exactly as the backward kernel does from the stored value: the
  // gradient written here equals the one ce_bwd would produce, bit for bit
  const float l2 = l * kLog2e;
  const int64_t lab = labels[row];
  if (threadIdx.x == 0) {
    lse[row] = l;
    const float xl = (lab >= 0 && lab < V) ? (float)xr[lab] : 0.f;
    loss[row] = (T)(l - xl);
  }
  if constexpr (GRAD) {
#pragma unroll
    for (int u = 0; u < NCH; ++u) asm("" : "+v"(raw[u]));
    T* dr = dlogits + dmap.at(row);
    const int lab_chunk = (lab >= 0 && lab < V) ? (int)(lab >> 3) : -1;
#pragma unroll
    for (int u = 0; u < NCH; ++u) {
      const int c = threadIdx.x + u * kCeThreads;
      if (c < nchunk) {
        float v[8];
        unpack8<T>(raw[u], v);
        grad_probs<ANY>(v, l2);
        if (c == lab_chunk) {
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] -= (e == (int)(lab & 7)) ? 1.0f : 0.0f;
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] *= grad_scale;
        Row<T, ANY>::store(dr, c, V, pack8<T>(v));
      }
    }
  }
}

// How ce_bwd walks its rows; bound by memory.  kCeAligned: whole aligned chunks.  kCeShort: chunks counted from the start of
// the row, wherever it lies.  kCeLines: chunks counted from the 128-byte line in which the row of the gradient starts, so that
// a wave's access covers whole lines instead of leaving a piece of one to the next: 4095 x 50257 bf16 187 -> 170 us
// (4.8 TB/s), 2047 x 32001 50.7 -> 44.3, 8192 x 4097 27.3 -> 24.6, but 8192 x 1001 12.1 -> 12.8 (written through, these
// stores take 183, 53 and 54 us).  The values of the last two are the same bits: an element depends on nothing but itself, and
// where a chunk holds a probability below 2^-126 the library function gives its other elements what v_exp_f32 would.  Whole
// aligned rows flush such probabilities to zero.
enum CeRows { kCeAligned, kCeShort, kCeLines };
constexpr int64_t kCeLinesFrom = 2048;
template <typename T, CeRows FORM>
__global__ __launch_bounds__(kCeThreads) void ce_bwd(int V, const T* __restrict__ logits, RowMap map,
                                                      const int64_t* __restrict__ labels,
                                                      const float* __restrict__ lse, const T* __restrict__ gout,
                                                      int64_t gstride, T* __restrict__ dlogits, RowMap dmap) {
  constexpr bool ANY = FORM != kCeAligned;
  typedef Row<T, ANY> R;
  const int64_t row = blockIdx.x;
  const T* xr = logits + map.at(row);
  T* dr = dlogits + dmap.at(row);
  const float l2 = lse[row] * kLog2e;
  const float g = (float)gout[row * gstride];
  const int lab = (int)labels[row];
  const int before = FORM == kCeLines ? (int)((reinterpret_cast<uintptr_t>(dr) & 127) / sizeof(T)) : 0;  // of the line, ahead of the row
  const int nchunk = FORM == kCeLines ? (V + before + 7) / 8 : R::chunks(V);
  for (int c = threadIdx.x; c < nchunk; c += kCeThreads) {
    int first = c * 8 - before;
    if (FORM == kCeLines && first <= -8) continue;
    // a chunk that crosses an end of the row is taken as the eight elements at that end: its neighbour writes some of
    // them as well, the same bits
    const bool inside = FORM != kCeLines || (first >= 0 && first + 8 <= V);
    if (FORM == kCeLines) first = min(max(first, 0), V - 8);
    float v[8];
    if (FORM == kCeLines) unpack8<T>(ld16_elem<true>(xr + first, std::integral_constant<int, 2>()), v);
    else unpack8<T>(R::template settle<true>(R::template fetch<true, true>(xr, c, V), c, V), v);
    grad_probs<ANY>(v, l2);
    if ((unsigned)(lab - first) < 8u) {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] -= (e == lab - first) ? 1.0f : 0.0f;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] *= g;
    if (FORM != kCeLines) R::template store<true>(dr, c, V, pack8<T>(v));
    else if (inside) *reinterpret_cast<u32x4*>(dr + first) = pack8<T>(v);
    else st16_elem(dr + first, pack8<T>(v), std::integral_constant<int, 2>());
  }
}

template <typename T>
static int ce_fwd_launch(hipStream_t st, int64_t rows, int64_t V, const void* logits, RowMap map,
                         const int64_t* labels, void* loss, float* lse) {
  const dim3 grid((unsigned)rows), block(kCeThreads);
  const RowMap none = {0, 0, 1};
  const bool vec = row_vectorizable<T>(logits, V, map.ld) && map.outer % 8 == 0;
  const int64_t per_thread = ((V + 7) / 8 + kCeThreads - 1) / kCeThreads;  // 16-byte chunks per thread
#define CE_ARGS ((int)V, (const T*)logits, map, labels, (T*)loss, lse, nullptr, none, 0.f)
#define CE_REGS(NCH)                                                              \
  do {                                                                            \
    if (vec) ce_fwd_regs<T, NCH, false, false><<<grid, block, 0, st>>>CE_ARGS;      \
    else ce_fwd_regs<T, NCH, false, true><<<grid, block, 0, st>>>CE_ARGS;           \
  } while (0)
  if (per_thread <= 8) CE_REGS(8);
  else if (per_thread <= 16) CE_REGS(16);
  else if (per_thread <= 25) CE_REGS(25);
  else if (vec) ce_fwd<T, false><<<grid, block, 0, st>>>((int)V, (const T*)logits, map, labels, (T*)loss, lse);
  else ce_fwd<T, true><<<grid, block, 0, st>>>((int)V, (const T*)logits, map, labels, (T*)loss, lse);
#undef CE_REGS
#undef CE_ARGS
  TF_CHECK_LAUNCH();
  return TF_OK;
}

template <typename T>
static int ce_bwd_launch(hipStream_t st, int64_t rows, int64_t V, const void* logits, RowMap map,
                         const int64_t* labels, const float* lse, const void* gout, int64_t gstride,
                         void* dlogits, RowMap dmap) {
  const dim3 grid((unsigned)rows), block(kCeThreads);
  const bool aligned = row_vectorizable<T>(logits, V, map.ld) && row_vectorizable<T>(dlogits, V, dmap.ld) &&
                       map.outer % 8 == 0 && dmap.outer % 8 == 0;
#define CE_BWD(FORM)                                                                                                  \
  ce_bwd<T, FORM><<<grid, block, 0, st>>>((int)V, (const T*)logits, map, labels, lse, (const T*)gout, gstride, (T*)dlogits, \
                                          dmap)
  if (aligned) CE_BWD(kCeAligned);
  else if (V >= kCeLinesFrom && logits != dlogits) CE_BWD(kCeLines);
  else CE_BWD(kCeShort);
#undef CE_BWD
  TF_CHECK_LAUNCH();
  return TF_OK;
}

// Forward that also leaves (softmax - onehot) * grad_scale in dlogits: one kernel when the row fits
// the registers of a workgroup, else the forward followed by the backward kernel with `scale_dev` (one value of T in device memory holding
// grad_scale) as the upstream gradient of every row -- the same values either way.
template <typename T>
static int ce_fwd_grad_launch(hipStream_t st, int64_t rows, int64_t V, const void* logits, RowMap map,
                              const int64_t* labels, void* loss, float* lse, void* dlogits, RowMap dmap,
                              float grad_scale, const void* scale_dev) {
  const dim3 grid((unsigned)rows), block(kCeThreads);
  const int64_t per_thread = ((V + 7) / 8 + kCeThreads - 1) / kCeThreads;
  if (per_thread <= 25) {
    const bool vec = row_vectorizable<T>(logits, V, map.ld) && map.outer % 8 == 0 &&
                     row_vectorizable<T>(dlogits, V, dmap.ld) && dmap.outer % 8 == 0;
#define CE_ARGS ((int)V, (const T*)logits, map, labels, (T*)loss, lse, (T*)dlogits, dmap, grad_scale)
#define CE_REGS(NCH)                                                             \
  do {                                                                           \
    if (vec) ce_fwd_regs<T, NCH, true, false><<<grid, block, 0, st>>>CE_ARGS;      \
    else ce_fwd_regs<T, NCH, true, true><<<grid, block, 0, st>>>CE_ARGS;           \
  } while (0)
    if (per_thread <= 8) CE_REGS(8);
    else if (per_thread <= 16) CE_REGS(16);
    else CE_REGS(25);
#undef CE_REGS
#undef CE_ARGS
    TF_CHECK_LAUNCH();
    return TF_OK;
  }
  if (!scale_dev) return TF_EINVAL;
  const int rc = ce_fwd_launch<T>(st, rows, V, logits, map, labels, loss, lse);
  if (rc != TF_OK) return rc;
  return ce_bwd_launch<T>(st, rows, V, logits, map, labels, lse, scale_dev, 0, dlogits, dmap);
}

}  // namespace tfa

using namespace tfa;

static bool make_map(RowMap& m, int64_t rows, int64_t V, int64_t ld, int64_t inner, int64_t outer) {
  if (inner <= 0) { inner = rows > 0 ? rows : 1; outer = 0; }
  if (ld < V || inner > 0x7fffffff || outer < 0 || (inner < rows && outer < (inner - 1) * ld + V)) return false;
  m.ld = ld; m.outer = outer; m.inner = (int)inner;
  return true;
}

extern "C" int tf_cross_entropy_fwd(void* stream, int dtype, int64_t rows, int64_t V, const void* logits,
                                    int64_t ld, int64_t inner_rows, int64_t outer_stride, const int64_t* labels,
                                    void* loss, float* lse) {
  if (!logits || !labels || !loss || !lse) return TF_EINVAL;
  if (rows < 0 || rows > 0x7fffffff || V <= 0 || V > (1 << 30)) return TF_EINVAL;
  RowMap map;
  if (!make_map(map, rows, V, ld, inner_rows, outer_stride)) return TF_EINVAL;
  if (rows == 0) return TF_OK;
  hipStream_t st = (hipStream_t)stream;
  if (dtype == TF_F16) return ce_fwd_launch<f16>(st, rows, V, logits, map, labels, loss, lse);
  if (dtype == TF_BF16) return ce_fwd_launch<bf16>(st, rows, V, logits, map, labels, loss, lse);
  return TF_EDTYPE;
}

extern "C" int tf_cross_entropy_bwd(void* stream, int dtype, int64_t rows, int64_t V, const void* logits,
                                    int64_t ld, int64_t inner_rows, int64_t outer_stride, const int64_t* labels,
                                    const float* lse, const void* gout, int64_t gout_stride, void* dlogits,
                                    int64_t ldd, int64_t outer_stride_d) {
  if (!logits || !labels || !lse || !gout || !dlogits) return TF_EINVAL;
  if (rows < 0 || rows > 0x7fffffff || V <= 0 || V > (1 << 30) || gout_stride < 0) return TF_EINVAL;
  RowMap map, dmap;
  if (!make_map(map, rows, V, ld, inner_rows, outer_stride)) return TF_EINVAL;
  if (!make_map(dmap, rows, V, ldd, inner_rows, outer_stride_d)) return TF_EINVAL;
  if (rows == 0) return TF_OK;
  hipStream_t st = (hipStream_t)stream;
  if (dtype == TF_F16)
    return ce_bwd_launch<f16>(st, rows, V, logits, map, labels, lse, gout, gout_stride, dlogits, dmap);
  if (dtype == TF_BF16)
    return ce_bwd_launch<bf16>(st, rows, V, logits, map, labels, lse, gout, gout_stride, dlogits, dmap);
  return TF_EDTYPE;
}

extern "C" int tf_cross_entropy_fwd_grad(void* stream, int dtype, int64_t rows, int64_t V, const void* logits,
                                         int64_t ld, int64_t inner_rows, int64_t outer_stride, const int64_t* labels,
                                         void* loss, float* lse, void* dlogits, int64_t ldd, int64_t outer_stride_d,
                                         float grad_scale, const void* grad_scale_dev) {
  if (!logits || !labels || !loss || !lse || !dlogits) return TF_EINVAL;
  if (rows < 0 || rows > 0x7fffffff || V <= 0 || V > (1 << 30)) return TF_EINVAL;
  RowMap map, dmap;
  if (!make_map(map, rows, V, ld, inner_rows, outer_stride)) return TF_EINVAL;
  if (!make_map(dmap, rows, V, ldd, inner_rows, outer_stride_d)) return TF_EINVAL;
  if (dtype != TF_F16 && dtype != TF_BF16) return TF_EDTYPE;
  if (rows == 0) return TF_OK;
  hipStream_t st = (hipStream_t)stream;
  if (dtype == TF_F16)
    return ce_fwd_grad_launch<f16>(st, rows, V, logits, map, labels, loss, lse, dlogits, dmap, grad_scale, grad_scale_dev);
  return ce_fwd_grad_launch<bf16>(st, rows, V, logits, map, labels, loss, lse, dlogits, dmap, grad_scale, grad_scale_dev);
}
