// Row-wise helpers shared by the bandwidth-bound kernels: 16-byte chunks of a
// row converted to fp32, for 16-bit and 32-bit element types.
#pragma once
#include "common.h"

namespace tfa {

template <typename T> struct Chunk {  // 16-bit types: 8 elements per 16 bytes
  static constexpr int N = 8;
  static __device__ __forceinline__ void load(const T* p, float (&v)[8]) { unpack8<T>(ld16(p), v); }
  static __device__ __forceinline__ void store(T* p, const float (&v)[8]) { st16(p, pack8<T>(v)); }
};
template <> struct Chunk<float> {
  static constexpr int N = 4;
  static __device__ __forceinline__ void load(const float* p, float (&v)[4]) {
    f32x4 r = *reinterpret_cast<const f32x4*>(p);
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
typedef u32x2 u32x2_a2 __attribute__((aligned(2)));
typedef uint32_t u32_a2 __attribute__((aligned(2)));
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
  // The same in two halves for SHORT rows, one chunk per lane, where every wave has a chunk that crosses the end and the
  // tested element loads above, each waited for, are most of the time: `fetch` takes the 16 bytes that end with the row
  // in its place, `settle` moves their elements down.  (63488 x 71 fp16, LayerNorm forward: 28.5 us with
  // element loads, 22.5 so, 22.1 in a loop over elements; with a residual 40.2, 28.9 and 31.2.  In longer rows the moves, made
  // for every chunk, cost more than the element loads of the one: 8192 x 1537 14.4 -> 18.3.)
  template <bool SHORT, bool STREAM = false>
  static __device__ __forceinline__ u32x4 fetch(const T* row, int c, int n, T fill = (T)0.f) {
    if (!ANY || !SHORT || n < N) return load<STREAM>(row, c, n, fill);
    return ld16_elem<STREAM>(row + min(c * N, n - N), size_t_());
  }
  template <bool SHORT> static __device__ __forceinline__ u32x4 settle(u32x4 raw, int c, int n, T fill = (T)0.f) {
    if (!ANY || !SHORT || n < N || (c + 1) * N <= n) return raw;
    const int up = ((c + 1) * N - n) * (int)sizeof(T) * 8;  // bits to move down by, 16 to 112
    struct Words { uint64_t lo, hi; };
    Words w = __builtin_bit_cast(Words, raw);
    w.lo = up >= 64 ? w.hi >> (up & 63) : w.lo >> up | w.hi << (64 - up);
    w.hi = up >= 64 ? 0 : w.hi >> up;
    struct { T v[8 / sizeof(T)]; } f8;
#pragma unroll
    for (int e = 0; e < 8 / (int)sizeof(T); ++e) f8.v[e] = fill;
    const uint64_t f = __builtin_bit_cast(uint64_t, f8);
    if (f != 0) {
      w.hi |= up >= 64 ? f : f << (64 - up);
      if (up > 64) w.lo |= f << (128 - up);
    }
    return __builtin_bit_cast(u32x4, w);
  }
  template <bool SHORT = false> static __device__ __forceinline__ void store(T* row, int c, int n, u32x4 v) {
    T* p = row + c * N;
    if constexpr (!ANY) { st16(p, v); return; }
    if ((c + 1) * N <= n) {  // lines are filled by neighbouring lanes and stores: write-back, see st16
      st16_elem(p, v, size_t_());
      return;
    }
    if constexpr (!SHORT) {
      struct alignas(16) Elems { T v[N]; };
      const Elems t = __builtin_bit_cast(Elems, v);
#pragma unroll
      for (int e = 0; e < N; ++e)
        if (c * N + e < n) p[e] = t.v[e];
      return;
    }
    // SHORT: what is left of the row in pieces of 8, 4 and 2 bytes
    char* q = reinterpret_cast<char*>(p);
    const int left = (n - c * N) * (int)sizeof(T);
    if (left & 8) {
      *reinterpret_cast<u32x2_a2*>(q) = u32x2{v[0], v[1]};
      q += 8;
      v[0] = v[2], v[1] = v[3];
    }
    if (left & 4) {
      *reinterpret_cast<u32_a2*>(q) = v[0];
      q += 4;
      v[0] = v[1];
    }
    if (sizeof(T) == 2 && (left & 2)) *reinterpret_cast<uint16_t*>(q) = (uint16_t)v[0];
  }
};
// eight elements from index 8 c on of a vector of n elements (16-bit or fp32) as fp32, zero beyond its end
template <typename TP, bool ANY, bool SHORT = false>
__device__ __forceinline__ void load8_row(const TP* p, int c, int n, float (&v)[8]) {
  if constexpr (!ANY) {
    load8<TP>(p + c * 8, v);
  } else if constexpr (sizeof(TP) == 2) {
    typedef Row<TP, true> R;
    unpack8<TP>(R::template settle<SHORT>(R::template fetch<SHORT>(p, c, n), c, n), v);
  } else {
    typedef Row<float, true> R;
    const f32x4 a = __builtin_bit_cast(f32x4, R::template settle<SHORT>(R::template fetch<SHORT>(p, 2 * c, n), 2 * c, n));
    f32x4 b = {};
    if (8 * c + 4 < n) b = __builtin_bit_cast(f32x4, R::template settle<SHORT>(R::template fetch<SHORT>(p, 2 * c + 1, n), 2 * c + 1, n));
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
