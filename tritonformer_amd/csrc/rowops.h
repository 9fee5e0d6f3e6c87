// Row-wise helpers shared by the bandwidth-bound kernels: 16-byte chunks of a
// row converted to fp32, for 16-bit and 32-bit element types.
#pragma once
#include "common.h"

namespace tfa {

template <typename T> struct Chunk {  // 16-bit types: 8 elements per 16 bytes
  static constexpr int N = 8;
  static __device__ __forceinline__ void load(const T* p, float (&v)[8]) { unpack8<T>(ld16(p), v); }
  static __device__ __forceinline__ void load_stream(const T* p, float (&v)[8]) { unpack8<T>(ld16_stream(p), v); }
  static __device__ __forceinline__ void store(T* p, const float (&v)[8]) { st16(p, pack8<T>(v)); }
};
template <> struct Chunk<float> {
  static constexpr int N = 4;
  static __device__ __forceinline__ void load(const float* p, float (&v)[4]) {
    f32x4 r = *reinterpret_cast<const f32x4*>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = r[i];
  }
  static __device__ __forceinline__ void load_stream(const float* p, float (&v)[4]) {
    f32x4 r = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p));
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = r[i];
  }
  static __device__ __forceinline__ void store(float* p, const float (&v)[4]) {
    f32x4 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = v[i];
    store_out(p, r);
  }
};

// 8 consecutive elements as fp32; TP = a 16-bit type or float (fp32 master parameters are
// read as they are, no 16-bit copy is made first).
template <typename TP> __device__ __forceinline__ void load8(const TP* p, float (&v)[8]) { Chunk<TP>::load(p, v); }
template <> __device__ __forceinline__ void load8<float>(const float* p, float (&v)[8]) {
  float a[4], b[4];
  Chunk<float>::load(p, a);
  Chunk<float>::load(p + 4, b);
#pragma unroll
  for (int i = 0; i < 4; ++i) { v[i] = a[i]; v[4 + i] = b[i]; }
}

// Rows of any length starting at any element.  The vector memory path takes 16-byte accesses at any
// element address at the rate of aligned ones (copy of 32768 rows of 1016 16-bit elements: 5.98 TB/s at a
// pitch of 1024 elements, 5.58 at 1021, 5.69 at 1022), so a ragged row is read and written in the same
// 16-byte chunks as an aligned one; only the chunk that crosses the end of the row goes by elements.
// ANY = false: the caller has checked that rows are aligned and whole chunks (row_vectorizable).
typedef u32x4 u32x4_a2 __attribute__((aligned(2)));
typedef u32x4 u32x4_a4 __attribute__((aligned(4)));
template <bool STREAM> __device__ __forceinline__ u32x4 ld16_elem(const void* p, std::integral_constant<int, 2>) {
  const u32x4_a2* q = reinterpret_cast<const u32x4_a2*>(p);
  return STREAM ? __builtin_nontemporal_load(q) : *q;
}
template <bool STREAM> __device__ __forceinline__ u32x4 ld16_elem(const void* p, std::integral_constant<int, 4>) {
  const u32x4_a4* q = reinterpret_cast<const u32x4_a4*>(p);
  return STREAM ? __builtin_nontemporal_load(q) : *q;
}
__device__ __forceinline__ void st16_elem(void* p, u32x4 v, std::integral_constant<int, 2>) { *reinterpret_cast<u32x4_a2*>(p) = v; }
__device__ __forceinline__ void st16_elem(void* p, u32x4 v, std::integral_constant<int, 4>) { *reinterpret_cast<u32x4_a4*>(p) = v; }

template <typename T, bool ANY> struct Row {
  static constexpr int N = 16 / (int)sizeof(T);  // elements per chunk
  typedef std::integral_constant<int, (int)sizeof(T)> size_t_;
  static __device__ __forceinline__ int chunks(int n) { return ANY ? (n + N - 1) / N : n / N; }
  // chunk c of a row of n elements; elements beyond the row read as `fill` (put there once, at the load: tested per
  // element where the values are used the register-resident cross-entropy forward took 120 us instead of 94 at 4095 x 50257)
  template <bool STREAM = false> static __device__ __forceinline__ u32x4 load(const T* row, int c, int n, T fill = (T)0.f) {
    const T* p = row + c * N;
    if constexpr (!ANY) return STREAM ? ld16_stream(p) : ld16(p);
    if ((c + 1) * N <= n) return ld16_elem<STREAM>(p, size_t_());
    struct alignas(16) { T v[N]; } t;
#pragma unroll
    for (int e = 0; e < N; ++e) t.v[e] = c * N + e < n ? p[e] : fill;
    return __builtin_bit_cast(u32x4, t);
  }
  static __device__ __forceinline__ void store(T* row, int c, int n, u32x4 v) {
    T* p = row + c * N;
    if constexpr (!ANY) { st16(p, v); return; }
    if ((c + 1) * N <= n) {  // lines are filled by neighbouring lanes and stores: write-back, see st16
      st16_elem(p, v, size_t_());
      return;
    }
    struct alignas(16) Elems { T v[N]; };
    const Elems t = __builtin_bit_cast(Elems, v);
#pragma unroll
    for (int e = 0; e < N; ++e)
      if (c * N + e < n) p[e] = t.v[e];
  }
};
// eight elements from index 8 c on of a vector of n elements (16-bit or fp32) as fp32, zero beyond its end
template <typename TP, bool ANY> __device__ __forceinline__ void load8_row(const TP* p, int c, int n, float (&v)[8]) {
  if constexpr (!ANY) {
    load8<TP>(p + c * 8, v);
  } else if constexpr (sizeof(TP) == 2) {
    unpack8<TP>(Row<TP, true>::load(p, c, n), v);
  } else {
    const f32x4 a = __builtin_bit_cast(f32x4, Row<float, true>::load(p, 2 * c, n));
    f32x4 b = {};
    if (8 * c + 4 < n) b = __builtin_bit_cast(f32x4, Row<float, true>::load(p, 2 * c + 1, n));
#pragma unroll
    for (int i = 0; i < 4; ++i) { v[i] = a[i]; v[4 + i] = b[i]; }
  }
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// True when rows of `n` elements of T starting at p with leading dimension ld
// can be read as whole 16-byte chunks.
template <typename T> inline bool row_vectorizable(const void* p, int64_t n, int64_t ld) {
  const int per = 16 / (int)sizeof(T);
  return aligned16(p) && (n % per == 0) && (ld % per == 0);
}

#define TF_CHECK_LAUNCH()                                      \
  do {                                                         \
    if (hipGetLastError() != hipSuccess) return TF_ELAUNCH;    \
  } while (0)

}  // namespace tfa
