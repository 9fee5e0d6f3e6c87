// Column sums (bias gradient) and the ReLU gradient mask for gfx950; both are
// HBM-bound streaming kernels with 16-byte accesses.
#include <atomic>
#include "rowops.h"

namespace tfa {

// Scratch of the allocation-free column sum (tf_colsum_noalloc): the first-stage partial sums live
// here instead of in a buffer the caller brings.  One copy per GPU the library runs on, held until
// the process ends.  In host code the array's name is only a handle for hipGetSymbolAddress; the
// device address it yields is what kernels and copies are given.
constexpr int64_t kNoAllocScratchBytes = 4 << 20;
static __device__ __align__(256) float scratch[kNoAllocScratchBytes / sizeof(float)];

constexpr int kCsColsPerBlock = 256;  // 32 lanes x 8 elements
constexpr int kCsSlices = 8;          // row slices per workgroup

static int colsum_groups(int64_t rows, int64_t cols) {
  const int64_t col_blocks = (cols + kCsColsPerBlock - 1) / kCsColsPerBlock;
  int64_t want = (2048 + col_blocks - 1) / col_blocks;  // aim for ~2048 workgroups
  const int64_t max_groups = (rows + 4 * kCsSlices - 1) / (4 * kCsSlices);  // >= 4 rows per slice
  if (want > max_groups) want = max_groups;
  if (want < 1) want = 1;
  return (int)want;
}

// Rows whose sums may be made in parts (below) have scratch for sixteen of them, up to where the columns alone fill the chip.
constexpr int64_t kCsFewRows = 1024;
constexpr int kCsFewSlices = 128, kCsParts = 16;
static int colsum_scratch_groups(int64_t rows, int64_t cols) {
  const int groups = colsum_groups(rows, cols);
  return rows > kCsFewRows / 4 && rows <= kCsFewRows && cols <= 32768 && groups < kCsParts ? kCsParts : groups;
}
static bool on_lines(const void* p, int64_t ld) { return reinterpret_cast<uintptr_t>(p) % 128 == 0 && ld % 64 == 0; }  // 16-bit rows

// grid (col_blocks, groups).  Thread (slice, lane32) sums 8 adjacent columns
// over rows  group_begin + slice, + 8, ...; slices are combined through LDS.
// MASK: x is masked by act > 0 first and written to `out` on the way -- the sums take the same values in the same
// order as a mask pass and a sum pass give, without reading the masked matrix back (memory-bound; the two passes took
// 9.6 + 5.7 us at 4113 x 1733 fp16; Linear with bias and ReLU, forward and backward, 182.4 -> 179.1 with this one).
template <typename T, bool ANY, bool MASK>
__global__ __launch_bounds__(256) void colsum_partial(int64_t rows, int cols, const T* __restrict__ x, int64_t ldx,
                                                       float* __restrict__ partial, int rows_per_group,
                                                       const T* __restrict__ act, int64_t lda, T* __restrict__ out,
                                                       int64_t ldo) {
  typedef Row<T, ANY> R;
  __shared__ float red[kCsSlices][kCsColsPerBlock];
  const int lane32 = threadIdx.x & 31;
  const int slice = threadIdx.x >> 5;
  const int col0 = blockIdx.x * kCsColsPerBlock + lane32 * 8;
  const int64_t rbeg = (int64_t)blockIdx.y * rows_per_group;
  int64_t rend = rbeg + rows_per_group;
  if (rend > rows) rend = rows;
  float acc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = 0.f;
  if (col0 < cols) {
    for (int64_t r = rbeg + slice; r < rend; r += kCsSlices) {
      float v[8];
      const u32x4 rx = R::template fetch<true>(x + r * ldx, col0 / 8, cols);
      const u32x4 ra = MASK ? R::template fetch<true>(act + r * lda, col0 / 8, cols) : rx;
      unpack8<T>(R::template settle<true>(rx, col0 / 8, cols), v);
      if constexpr (MASK) {
        float a[8];
        unpack8<T>(R::template settle<true>(ra, col0 / 8, cols), a);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = a[e] > 0.f ? v[e] : 0.f;
        R::template store<true>(out + r * ldo, col0 / 8, cols, pack8<T>(v));
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] += v[e];
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) red[slice][lane32 * 8 + e] = acc[e];
  __syncthreads();
  const int c = blockIdx.x * kCsColsPerBlock + threadIdx.x;
  if (c < cols) {
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < kCsSlices; ++k) s += red[k][threadIdx.x];
    partial[(int64_t)blockIdx.y * cols + c] = s;
  }
}

// Second stage: out[c] = sum over groups of partial[g][c], in a fixed order.  A workgroup takes 32
// columns; its 8 slices of 32 lanes each add up every 8th group, then the slices are combined through LDS.
// Bound by the latency of its loads, sixteen of which are in flight per lane: sums of 16384 rows of 768 and 3072 columns,
// second stage 8.7 us with two in flight, 4.7 now.
template <typename T>
__global__ __launch_bounds__(256) void colsum_final(int groups, int cols, const float* __restrict__ partial,
                                                     T* __restrict__ out) {
  __shared__ float red[8][32];
  const int lane32 = threadIdx.x & 31, slice = threadIdx.x >> 5;
  const int c = blockIdx.x * 32 + lane32;
  float s0 = 0.f, s1 = 0.f;
  if (c < cols) {
    int g = slice;
    const float* p = partial + c;
    for (; g + 120 < groups; g += 128) {  // sixteen loads in flight, added in the order of the loop below
      float v[16];
#pragma unroll
      for (int k = 0; k < 16; ++k) v[k] = p[(int64_t)(g + 8 * k) * cols];
#pragma unroll
      for (int k = 0; k < 16; k += 2) { s0 += v[k]; s1 += v[k + 1]; }
    }
    for (; g + 8 < groups; g += 16) {
      s0 += p[(int64_t)g * cols];
      s1 += p[(int64_t)(g + 8) * cols];
    }
    if (g < groups) s0 += p[(int64_t)g * cols];
  }
  red[slice][lane32] = s0 + s1;
  __syncthreads();
  if (slice == 0 && c < cols) {
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k) s += red[k][lane32];
    out[c] = (T)s;
  }
}

// Up to 1024 rows (512 of ragged columns): 128 slices of every 128th row, eight slices to a part, sixteen parts; slices and parts are
// added in their order by either form, so that a sum has the same bits with and without a mask.  Four rows of a thread are requested
// together.
// WHOLE: a workgroup of 1024 threads takes 64 columns (one line of a row), all slices, and writes the sums.  Bound by the latency of its
// loads; the second launch cost more than the idle CUs do: both stages as they are beyond 1024 rows and this one, us in a graph, fp16: 512 x
// 1024 4.35 -> 2.47, 960 x 768 4.57 -> 3.17, 960 x 3072 5.98 -> 4.92, 1024 x 8192 7.98 -> 5.39.
// !WHOLE: a workgroup of 256 threads takes 256 columns and the slices of one part (blockIdx.y), which it leaves to colsum_parts: where one
// CU has too many bytes to move, and where rows do not start on a line, which makes pieces of 128 bytes two lines each.
template <typename T, typename TO, bool ANY, bool MASK, bool WHOLE>
__global__ __launch_bounds__(WHOLE ? 1024 : 256) void colsum_few(int rows, int cols, const T* __restrict__ x, int64_t ldx,
                                                                 TO* __restrict__ sums, const T* __restrict__ act, int64_t lda,
                                                                 T* __restrict__ out, int64_t ldo) {
  typedef Row<T, ANY> R;
  constexpr int COLS = WHOLE ? 64 : 256, LANES = COLS / 8, PARTS = WHOLE ? kCsParts : 1, PER = kCsFewSlices / kCsParts, SLICES = PARTS * PER;
  __shared__ __align__(16) float red[SLICES][COLS + 4];
  __shared__ float part[PARTS][COLS];
  const int lane8 = threadIdx.x % LANES, local = threadIdx.x / LANES, slice = (WHOLE ? 0 : blockIdx.y * PER) + local;
  const int chunk = blockIdx.x * LANES + lane8;
  float acc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = 0.f;
  if (chunk * 8 < cols) {
    auto add = [&](int r, u32x4 rx, u32x4 ra) {
      float v[8];
      unpack8<T>(R::template settle<true>(rx, chunk, cols), v);
      if constexpr (MASK) {
        float a[8];
        unpack8<T>(R::template settle<true>(ra, chunk, cols), a);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = a[e] > 0.f ? v[e] : 0.f;
        R::template store<true>(out + (int64_t)r * ldo, chunk, cols, pack8<T>(v));
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] += v[e];
    };
    auto fetch_x = [&](int r) { return R::template fetch<true>(x + (int64_t)r * ldx, chunk, cols); };
    auto fetch_a = [&](int r, u32x4 rx) { return MASK ? R::template fetch<true>(act + (int64_t)r * lda, chunk, cols) : rx; };
    int r = slice;
    for (; r + 3 * kCsFewSlices < rows; r += 4 * kCsFewSlices) {
      u32x4 rx[4], ra[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        rx[k] = fetch_x(r + k * kCsFewSlices);
        ra[k] = fetch_a(r + k * kCsFewSlices, rx[k]);
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) add(r + k * kCsFewSlices, rx[k], ra[k]);
    }
    for (; r < rows; r += kCsFewSlices) {
      const u32x4 rx = fetch_x(r);
      add(r, rx, fetch_a(r, rx));
    }
  }
#pragma unroll
  for (int e = 0; e < 8; e += 4) {
    const f32x4 v = {acc[e], acc[e + 1], acc[e + 2], acc[e + 3]};
    *reinterpret_cast<f32x4*>(&red[local][lane8 * 8 + e]) = v;
  }
  __syncthreads();
  const int col = threadIdx.x % COLS, p = threadIdx.x / COLS, c = blockIdx.x * COLS + col;
  float s = 0.f;
#pragma unroll
  for (int k = 0; k < PER; ++k) s += red[p * PER + k][col];
  if constexpr (WHOLE) {
    part[p][col] = s;
    __syncthreads();
    if (p == 0 && c < cols) {
      s = 0.f;
#pragma unroll
      for (int k = 0; k < kCsParts; ++k) s += part[k][col];
      sums[c] = (TO)s;
    }
  } else if (c < cols) {
    sums[(int64_t)blockIdx.y * cols + c] = (TO)s;
  }
}

// The sixteen parts of colsum_few, in their order.
template <typename TO>
__global__ __launch_bounds__(64) void colsum_parts(int cols, const float* __restrict__ parts, TO* __restrict__ sums) {
  const int c = blockIdx.x * 64 + threadIdx.x;
  if (c >= cols) return;
  float v[kCsParts], s = 0.f;
#pragma unroll
  for (int k = 0; k < kCsParts; ++k) v[k] = parts[(int64_t)k * cols + c];
#pragma unroll
  for (int k = 0; k < kCsParts; ++k) s += v[k];
  sums[c] = (TO)s;
}

template <typename T, bool ANY>
__global__ __launch_bounds__(256) void relu_mask_kernel(int64_t rows, int cols, const T* __restrict__ grad,
                                                         int64_t ldg, const T* __restrict__ act, int64_t lda,
                                                         T* __restrict__ out, int64_t ldo) {
  typedef Row<T, ANY> R;
  const int cpr = R::chunks(cols);
  const int64_t total = rows * cpr;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    const int64_t r = i / cpr;
    const int c = (int)(i - r * cpr);
    float g[8], a[8];
    const u32x4 rg = R::template fetch<true>(grad + r * ldg, c, cols), ra = R::template fetch<true>(act + r * lda, c, cols);
    unpack8<T>(R::template settle<true>(rg, c, cols), g);
    unpack8<T>(R::template settle<true>(ra, c, cols), a);
#pragma unroll
    for (int e = 0; e < 8; ++e) g[e] = a[e] > 0.f ? g[e] : 0.f;
    R::template store<true>(out + r * ldo, c, cols, pack8<T>(g));
  }
}

// `masked` non-null: the sums are those of where(act > 0, x, 0), which is written there
template <typename T>
static int colsum_launch(hipStream_t st, int64_t rows, int64_t cols, const void* x, int64_t ldx, void* out,
                         bool out_f32, float* partial, int64_t partial_bytes, const void* act = nullptr, int64_t lda = 0,
                         void* masked = nullptr, int64_t ldm = 0) {
  const bool vec = row_vectorizable<T>(x, cols, ldx) && (!masked || (row_vectorizable<T>(act, cols, lda) && row_vectorizable<T>(masked, cols, ldm)));
  const int groups = colsum_groups(rows, cols);
  // The order of the sums follows from the matrix that is summed alone (its alignment, for the two stages are the faster ones for long
  // ragged columns): the masked one where there is a mask, which a call without one reads.
  const bool few = rows <= (row_vectorizable<T>(masked ? masked : x, cols, masked ? ldm : ldx) ? kCsFewRows : kCsFewRows / 2);
  if (few) {
    // With a mask a row is three pieces.  us on one CU per 64 columns, apart, and in the two stages: 1024 x 3072 7.9, 5.2, 5.8; 1024 x 16384
    // 17.3, 17.8, 20.0; 640 x 1024 5.0, 5.0, 5.4.  Rows that do not start on a line: 1024 x 7208 13.0, 9.7, 10.6; 450 x 3071 7.9, 5.5,
    // 6.2; 400 x 777 4.9, 5.7, 6.6; 300 x 12345 6.8, 7.0, 7.3.  Without a mask: 1024 x 7208 4.7, 4.8, 5.9; 700 x 7208 3.4, 4.5, 4.9.
    const bool lines = vec && on_lines(x, ldx) && on_lines(act, lda) && on_lines(masked, ldm);
    const bool apart = masked && colsum_scratch_groups(rows, cols) >= kCsParts && partial_bytes >= kCsParts * cols * (int64_t)sizeof(float) &&
                       (lines ? rows > 640 && cols <= 8192 : rows > 256 && (rows > 352 || cols > 16384));
    const dim3 grid((unsigned)ceil_div(cols, apart ? 256 : 64), apart ? kCsParts : 1), block(apart ? 256 : 1024);
#define COLSUM_FEW(TO, ANY, MASK, WHOLE, RES)                                                                          \
  colsum_few<T, TO, ANY, MASK, WHOLE><<<grid, block, 0, st>>>((int)rows, (int)cols, (const T*)x, ldx, (TO*)(RES), (const T*)act, lda, \
                                                              (T*)masked, ldm)
#define COLSUM_FEW_FORM(TO, WHOLE, RES)                                                                                \
  do {                                                                                                                 \
    if (!masked) { if (vec) COLSUM_FEW(TO, false, false, true, RES); else COLSUM_FEW(TO, true, false, true, RES); }    \
    else { if (vec) COLSUM_FEW(TO, false, true, WHOLE, RES); else COLSUM_FEW(TO, true, true, WHOLE, RES); }            \
  } while (0)
    if (apart) COLSUM_FEW_FORM(float, false, partial);
    else if (out_f32) COLSUM_FEW_FORM(float, true, out);
    else COLSUM_FEW_FORM(T, true, out);
#undef COLSUM_FEW_FORM
#undef COLSUM_FEW
    TF_CHECK_LAUNCH();
    if (!apart) return TF_OK;
    if (out_f32) colsum_parts<float><<<dim3(ceil_div(cols, 64)), dim3(64), 0, st>>>((int)cols, partial, (float*)out);
    else colsum_parts<T><<<dim3(ceil_div(cols, 64)), dim3(64), 0, st>>>((int)cols, partial, (T*)out);
    TF_CHECK_LAUNCH();
    return TF_OK;
  }
  const int rpg = (int)((rows + groups - 1) / groups);
  const dim3 grid((unsigned)ceil_div(cols, kCsColsPerBlock), (unsigned)groups), block(256);
#define COLSUM(ANY, MASK)                                                                                       \
  colsum_partial<T, ANY, MASK><<<grid, block, 0, st>>>(rows, (int)cols, (const T*)x, ldx, partial, rpg, (const T*)act, \
                                                       lda, (T*)masked, ldm)
  if (!masked) {
    if (vec) COLSUM(false, false);
    else COLSUM(true, false);
  } else if (vec) {
    COLSUM(false, true);
  } else {
    COLSUM(true, true);
  }
#undef COLSUM
  TF_CHECK_LAUNCH();
  if (out_f32) colsum_final<float><<<dim3(ceil_div(cols, 32)), block, 0, st>>>(groups, (int)cols, partial, (float*)out);
  else colsum_final<T><<<dim3(ceil_div(cols, 32)), block, 0, st>>>(groups, (int)cols, partial, (T*)out);
  TF_CHECK_LAUNCH();
  return TF_OK;
}

template <typename T>
static int relu_mask_launch(hipStream_t st, int64_t rows, int64_t cols, const void* grad, int64_t ldg,
                            const void* act, int64_t lda, void* out, int64_t ldo) {
  const bool vec =
      row_vectorizable<T>(grad, cols, ldg) && row_vectorizable<T>(act, cols, lda) && row_vectorizable<T>(out, cols, ldo);
  const int64_t work = rows * ((cols + 7) / 8);
  int64_t blocks = (work + 255) / 256;
  if (blocks > 256 * 32) blocks = 256 * 32;
  if (blocks < 1) blocks = 1;
  if (vec)
    relu_mask_kernel<T, false><<<dim3((unsigned)blocks), dim3(256), 0, st>>>(rows, (int)cols, (const T*)grad, ldg,
                                                                            (const T*)act, lda, (T*)out, ldo);
  else
    relu_mask_kernel<T, true><<<dim3((unsigned)blocks), dim3(256), 0, st>>>(rows, (int)cols, (const T*)grad, ldg,
                                                                             (const T*)act, lda, (T*)out, ldo);
  TF_CHECK_LAUNCH();
  return TF_OK;
}

// ---------------------------------------------------------------------------
// Convert up to four (rows, cols) matrices to 16 bits, side by side in one matrix.
// ---------------------------------------------------------------------------
struct PackSources { const void* p[4]; };

template <typename TI, typename TO, bool VEC>
__global__ __launch_bounds__(256) void cast_pack(PackSources src, int count, int64_t rows, int cols, int64_t ld_src,
                                                  TO* __restrict__ dst, int64_t ld_dst) {
  const int per_row = VEC ? cols >> 3 : cols;  // work items per source row
  const int64_t total = rows * count * per_row;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    const int c = (int)(i % per_row);
    const int64_t rj = i / per_row;
    const int j = (int)(rj % count);
    const int64_t r = rj / count;
    const TI* s = (const TI*)src.p[j] + r * ld_src;
    TO* d = dst + r * ld_dst + (int64_t)j * cols;
    if (VEC) {
      float v[8];
      load8<TI>(s + c * 8, v);
      Chunk<TO>::store(d + c * 8, v);
    } else {
      d[c] = (TO)(float)s[c];
    }
  }
}

template <typename TI, typename TO>
static int cast_pack_launch(hipStream_t st, int count, int64_t rows, int64_t cols, const void* const* srcs,
                            int64_t ld_src, void* dst, int64_t ld_dst) {
  PackSources ps = {};
  bool vec = cols % 8 == 0 && ld_src % 8 == 0 && ld_dst % 8 == 0 && aligned16(dst);
  for (int j = 0; j < count; ++j) { ps.p[j] = srcs[j]; vec = vec && aligned16(srcs[j]); }
  const int64_t items = rows * count * (vec ? cols / 8 : cols);
  int64_t blocks = (items + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  if (vec) cast_pack<TI, TO, true><<<dim3((unsigned)blocks), dim3(256), 0, st>>>(ps, count, rows, (int)cols, ld_src, (TO*)dst, ld_dst);
  else cast_pack<TI, TO, false><<<dim3((unsigned)blocks), dim3(256), 0, st>>>(ps, count, rows, (int)cols, ld_src, (TO*)dst, ld_dst);
  TF_CHECK_LAUNCH();
  return TF_OK;
}

}  // namespace tfa

using namespace tfa;

// what a call cannot do without; with what tf_colsum_partial_bytes answers it may take the faster form
static int64_t colsum_least_bytes(int64_t rows, int64_t cols) { return (int64_t)colsum_groups(rows, cols) * cols * (int64_t)sizeof(float); }

extern "C" int64_t tf_colsum_partial_bytes(int64_t rows, int64_t cols) {
  if (rows <= 0 || cols <= 0) return 0;
  return (int64_t)colsum_scratch_groups(rows, cols) * cols * (int64_t)sizeof(float);
}

extern "C" int tf_colsum(void* stream, int dtype, int out_dtype, int64_t rows, int64_t cols, const void* x,
                         int64_t ldx, void* out, float* partial, int64_t partial_bytes) {
  if (!x || !out) return TF_EINVAL;
  if (rows <= 0 || cols <= 0 || cols > (1 << 30) || ldx < cols) return TF_EINVAL;
  if (dtype != TF_F16 && dtype != TF_BF16) return TF_EDTYPE;
  if (out_dtype != dtype && out_dtype != TF_F32) return TF_EDTYPE;
  if (!partial || partial_bytes < colsum_least_bytes(rows, cols)) return TF_EWORKSPACE;
  hipStream_t st = (hipStream_t)stream;
  if (dtype == TF_F16) return colsum_launch<f16>(st, rows, cols, x, ldx, out, out_dtype == TF_F32, partial, partial_bytes);
  return colsum_launch<bf16>(st, rows, cols, x, ldx, out, out_dtype == TF_F32, partial, partial_bytes);
}

// Device address of `scratch` on the current device, looked up once per device (with that device
// current) and kept.  Returns null if the runtime refuses.
static float* noalloc_scratch() {
  constexpr int kMaxDevices = 64;
  static std::atomic<float*> ptrs[kMaxDevices];
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
  float* p = ptrs[dev].load(std::memory_order_acquire);
  if (!p) {
    void* addr = nullptr;
    if (hipGetSymbolAddress(&addr, HIP_SYMBOL(scratch)) != hipSuccess || !addr) {
      (void)hipGetLastError();
      return nullptr;
    }
    p = static_cast<float*>(addr);
    ptrs[dev].store(p, std::memory_order_release);  // every thread finds the same address
  }
  return p;
}

extern "C" int64_t tf_colsum_noalloc_max_partial_bytes(void) { return kNoAllocScratchBytes; }

extern "C" int tf_colsum_noalloc(void* stream, int dtype, int out_dtype, int64_t rows, int64_t cols, const void* x,
                                 int64_t ldx, void* out) {
  if (!x || !out) return TF_EINVAL;
  if (rows <= 0 || cols <= 0 || cols > (1 << 30) || ldx < cols) return TF_EINVAL;
  if (dtype != TF_F16 && dtype != TF_BF16) return TF_EDTYPE;
  if (out_dtype != dtype && out_dtype != TF_F32) return TF_EDTYPE;
  if (colsum_least_bytes(rows, cols) > kNoAllocScratchBytes) return TF_EWORKSPACE;  // beyond the fixed scratch
  float* partial = noalloc_scratch();
  if (!partial) return TF_ELAUNCH;
  hipStream_t st = (hipStream_t)stream;
  // every partial sum the second stage reads is written by the first stage of the same call:
  // nothing has to start at zero, whatever an earlier (larger) call left behind
  if (dtype == TF_F16) return colsum_launch<f16>(st, rows, cols, x, ldx, out, out_dtype == TF_F32, partial, kNoAllocScratchBytes);
  return colsum_launch<bf16>(st, rows, cols, x, ldx, out, out_dtype == TF_F32, partial, kNoAllocScratchBytes);
}

extern "C" int tf_relu_mask(void* stream, int dtype, int64_t rows, int64_t cols, const void* grad, int64_t ldg,
                            const void* act, int64_t lda, void* out, int64_t ldo) {
  if (!grad || !act || !out) return TF_EINVAL;
  if (rows < 0 || cols <= 0 || cols > (1 << 30) || ldg < cols || lda < cols || ldo < cols) return TF_EINVAL;
  if (rows == 0) return TF_OK;
  hipStream_t st = (hipStream_t)stream;
  if (dtype == TF_F16) return relu_mask_launch<f16>(st, rows, cols, grad, ldg, act, lda, out, ldo);
  if (dtype == TF_BF16) return relu_mask_launch<bf16>(st, rows, cols, grad, ldg, act, lda, out, ldo);
  return TF_EDTYPE;
}

extern "C" int tf_relu_mask_colsum(void* stream, int dtype, int out_dtype, int64_t rows, int64_t cols, const void* grad,
                                   int64_t ldg, const void* act, int64_t lda, void* masked, int64_t ldm, void* sums,
                                   float* partial, int64_t partial_bytes) {
  if (!grad || !act || !masked || !sums) return TF_EINVAL;
  if (rows <= 0 || cols <= 0 || cols > (1 << 30) || ldg < cols || lda < cols || ldm < cols) return TF_EINVAL;
  if (dtype != TF_F16 && dtype != TF_BF16) return TF_EDTYPE;
  if (out_dtype != dtype && out_dtype != TF_F32) return TF_EDTYPE;
  if (!partial || partial_bytes < colsum_least_bytes(rows, cols)) return TF_EWORKSPACE;
  hipStream_t st = (hipStream_t)stream;
  if (dtype == TF_F16)
    return colsum_launch<f16>(st, rows, cols, grad, ldg, sums, out_dtype == TF_F32, partial, partial_bytes, act, lda, masked, ldm);
  return colsum_launch<bf16>(st, rows, cols, grad, ldg, sums, out_dtype == TF_F32, partial, partial_bytes, act, lda, masked, ldm);
}

extern "C" int tf_cast_pack(void* stream, int src_dtype, int dst_dtype, int count, int64_t rows, int64_t cols,
                            const void* const* srcs, int64_t ld_src, void* dst, int64_t ld_dst) {
  if (!srcs || !dst || count < 1 || count > 4) return TF_EINVAL;
  for (int j = 0; j < count; ++j)
    if (!srcs[j]) return TF_EINVAL;
  if (rows < 0 || cols <= 0 || cols > (1 << 30) || ld_src < cols || ld_dst < count * cols) return TF_EINVAL;
  if (dst_dtype != TF_F16 && dst_dtype != TF_BF16) return TF_EDTYPE;
  if (src_dtype != TF_F32 && src_dtype != dst_dtype) return TF_EDTYPE;
  if (rows == 0) return TF_OK;
  hipStream_t st = (hipStream_t)stream;
  if (dst_dtype == TF_F16)
    return src_dtype == TF_F32 ? cast_pack_launch<float, f16>(st, count, rows, cols, srcs, ld_src, dst, ld_dst)
                               : cast_pack_launch<f16, f16>(st, count, rows, cols, srcs, ld_src, dst, ld_dst);
  return src_dtype == TF_F32 ? cast_pack_launch<float, bf16>(st, count, rows, cols, srcs, ld_src, dst, ld_dst)
                             : cast_pack_launch<bf16, bf16>(st, count, rows, cols, srcs, ld_src, dst, ld_dst);
}
