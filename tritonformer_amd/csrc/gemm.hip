// Dense contraction C[M,N] = epilogue(sum_k A(m,k) B(n,k)) on gfx950 MFMA.
//
// One workgroup owns a BM x BN tile of C (or one slice of its contraction).  Two
// kernel families share the tiling and the MFMA code:
//  * gemm_dma_kernel / gemm_dma_group_kernel, the ones a training step runs: per
//    BK-wide step the A and B panels go HBM -> LDS directly (global_load_lds_dwordx4,
//    no VGPR round trip) into two LDS stages; the LDS operand reads, the loads of the
//    next step and the MFMAs are interleaved by hand (bare s_barrier, explicit
//    s_waitcnt); the result leaves through a wave-private LDS slab so that every
//    global store covers whole 128-byte lines;
//  * gemm_reg_kernel, for anything those cannot take (ragged extents, unaligned pointers,
//    a contraction that is not a multiple of BK): the same loop and write-out with the
//    operands staged through registers in 16-byte chunks at any element address.
// Both use v_mfma_f32_16x16x32_{f16,bf16} with fp32 accumulators.  Real data holds the clock of the matrix pipes down (power),
// and the smaller instruction needs less of it: it moves half the accumulators per multiplication.  The MFMA stream
// of a 256x256x64 step alone on normal fp16 data: 1.29 us with 32x32x16, 1.13 with 16x16x32 (bf16 1.20 and 1.06); equal on zeros.
// The results are the same bits.  Products on operands from HBM, fp16, with 32x32x16 and now: 8192 x 1024 x 4096 71.2 -> 64.9 us,
// 8192 x 4096 x 1024 73.5 -> 69.9, 4096 x 8192 x 2048 125.2 -> 115.9, 8192 x 50304 x 1024 819 -> 772; 4096 x 4096 x 8192 225 -> 204:
// the clock rises from 1.51 to 1.64 GHz and more, the matrix pipes are busy for three quarters of the cycles either way.
//
// Either operand may be stored with the contraction dimension contiguous
// ("K-major": read from LDS with ds_read_b128) or strided ("K-minor": read with
// the gfx950 transposing ds_read_b64_tr_b16), so X.W, dY.W^T and X^T.dY all run
// from the tensors as PyTorch holds them, without transposed copies.  LDS
// tiles are XOR-swizzled at 16-byte granularity to keep both access patterns
// free of bank conflicts.
//
// The MFMA is issued as D^T = B_frag x A_frag, so a lane ends up holding four
// consecutive n for one m: bias, ReLU and rounding need no cross-lane traffic.
//
// Workgroup ids are remapped so that each XCD (which receive ids round-robin)
// works on a compact block of neighbouring tiles and shares the A/B panels
// through its own L2.  The number of XCDs and of CUs is read from the device.
#include <algorithm>
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <type_traits>
#include "rowops.h"


namespace tfa {

struct GemmParams {
  const void* A;
  const void* B;
  void* C;
  const void* bias;  // of type T, or fp32 (bias_f32: an fp32 master, rounded to T where it is read)
  float* partial;
  int M, N, K;
  int64_t lda, ldb, ldc;
  int relu;
  int bias_f32;
  int splits, k_per_split;
  int tiles_m, tiles_n;
  int flags;  // bit 0: skip the XCD remap (set by the diagnostic entry point only)
  int xcds;   // XCDs of the device (workgroup ids are dealt to them round-robin)
  int out_f32;  // C holds fp32 instead of T
  const void* mask;  // optional (M, N) activation of type T: C = mask > 0 ? C : 0
  int64_t ldmask;
  // One bit per element, rows of ldsign bytes, bit n % 8 of byte n / 8 (direct-to-LDS kernels only):
  // sign_out receives C > 0 (with the ReLU epilogue: the gradient mask of the activation, at a
  // sixteenth of its size); sign_in zeroes C where its bit is clear.
  void* sign_out;
  const void* sign_in;
  int64_t ldsign;
  // Output split into column blocks of chunk_n columns, each its own (M, chunk_n) matrix
  // with leading dimension ldc, chunk_skip + chunk_n elements after the previous one.
  // One matrix: chunk_n = N, chunk_skip = 0.
  int chunk_n;
  int64_t chunk_skip;
  // Optional factor on the whole product, one fp32 value in DEVICE memory (null = 1): it is applied
  // to the fp32 sums before bias / rounding.  A pointer, so that a value computed on the GPU (the
  // upstream gradient of a mean loss) needs no host round trip.
  const float* alpha;
  // B as up to three matrices side by side (K-minor, leading dimension ldb): columns [i * b_each, (i + 1) * b_each) are
  // those of B, B1, B2; b_each is a multiple of the tile's width, so a tile reads one of them.  0: B alone.
  const void* B1 = nullptr;
  const void* B2 = nullptr;
  int b_each = 0;
};

// Round-robin XCD dispatch -> compact per-XCD ranges, then grouped raster.
__device__ __forceinline__ int remap_xcd(int pid, int n, int X) {
  const int xcd = pid % X, local = pid / X;
  const int q = n / X, r = n % X;
  return xcd * q + (xcd < r ? xcd : r) + local;
}

// ---------------------------------------------------------------------------
// Fast path: HBM -> LDS directly (global_load_lds_dwordx4, no VGPR round trip),
// STAGES LDS buffers, loads issued STAGES-1 steps ahead of their use.
// A wave-level load writes 64 x 16 bytes to consecutive LDS addresses, so the
// chunk swizzle is applied on the GLOBAL side: the lane that owns LDS slot
// (row, c') fetches chunk c = c' ^ swz(row).  Rows / columns beyond M / N are
// clamped to valid memory (their products only reach C entries that are never
// stored); the contraction extent must be a multiple of BK.
// ---------------------------------------------------------------------------
typedef __attribute__((address_space(1))) const void gptr_void;

// s_waitcnt lgkmcnt(n): at most n LDS reads (the youngest) may still be in flight.
template <int N> __device__ __forceinline__ void wait_lgkmcnt() {
  __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4) | ((N & 15) << 8));
}

// LDS operand reads issued as volatile asm: the compiler neither reorders them nor
// waits for them, so the kernel decides how far ahead of their MFMAs they run
// (every consumer sits behind an explicit wait_lgkmcnt + scheduling barrier).
template <bool KMAJOR> struct FragRegs;
template <> struct FragRegs<true> {
  u32x4 q;
  template <typename V8> __device__ __forceinline__ V8 get() const { return __builtin_bit_cast(V8, q); }
};
template <> struct FragRegs<false> {
  u32x2 lo, hi;
  template <typename V8> __device__ __forceinline__ V8 get() const {
    const u32x4 v = {lo[0], lo[1], hi[0], hi[1]};
    return __builtin_bit_cast(V8, v);
  }
};



// A wave-uniform address plus a lane's 32-bit offset, as one instruction takes them.  The empty statement keeps the
// extension of the offset to 64 bits next to its use: hoisted out of the loop it costs a second register per offset and a
// 64-bit addition per access.
__device__ __forceinline__ const char* at_offset(const char* origin, uint32_t off) {
  asm volatile("" : "+v"(off));
  return origin + off;
}
__device__ __forceinline__ const char* at_offset(const char* origin, uint64_t off) { return origin + off; }

template <typename T, int R, int BK, bool KMAJOR, int NW>
struct DmaPanel {
  static constexpr int CPR = KMAJOR ? BK / 8 : R / 8;
  static constexpr int LROWS = KMAJOR ? R : BK;
  static constexpr int NCHUNK = LROWS * CPR;
  static constexpr int BYTES = NCHUNK * 16;
  static constexpr int WLOADS = NCHUNK / 64;   // wave-level loads per panel
  static constexpr int PER_WAVE = WLOADS / NW;
  static_assert(WLOADS % NW == 0 && PER_WAVE >= 1, "panel must divide evenly over the waves");
  static_assert(KMAJOR ? (CPR == 4 || CPR == 8) : (CPR >= 8), "the swizzle stays within the row");

  // K-major: 16 rows of one chunk column fill the banks once.  K-minor: a transposing read takes 32 bytes of each of four
  // neighbouring rows per 16 lanes, and of the four rows eight further on in the next 16.  Rows of 256 bytes and more begin
  // at the same bank, rows of 128 bytes at every other half of them.
  static __device__ __forceinline__ int swz(int lrow, int c) {
    if constexpr (KMAJOR) return c ^ ((lrow / (16 / CPR)) % CPR);
    else if constexpr (CPR >= 16) return c ^ ((lrow & 3) << 2) ^ ((lrow >> 2) & 2);
    else return c ^ ((lrow & 3) << 1) ^ ((lrow >> 2) & 2);
  }

  // Byte offset of each of this lane's chunks from the panel's first element of a step (row row0, contraction index kbeg):
  // the address is wave-uniform but for these 32 bits (64 for rows beyond kMaxPitch), which no step changes.
  static __device__ __forceinline__ const char* origin(const T* base, int64_t ld, int row0, int kbeg) {
    return (const char*)(KMAJOR ? base + (int64_t)row0 * ld + kbeg : base + (int64_t)kbeg * ld + row0);
  }
  template <typename Off>
  static __device__ __forceinline__ void init(Off (&offs)[PER_WAVE], int64_t ld, int row0, int rmax, int wave, int lane) {
#pragma unroll
    for (int j = 0; j < PER_WAVE; ++j) {
      const int slot = (wave * PER_WAVE + j) * 64 + lane;
      const int lrow = slot / CPR;
      const int c = swz(lrow, slot % CPR);
      if (KMAJOR) offs[j] = ((Off)(min(row0 + lrow, rmax - 1) - row0) * (Off)ld + (Off)(c * 8)) * 2;
      else offs[j] = ((Off)lrow * (Off)ld + (Off)(row0 + c * 8 < rmax ? c * 8 : 0)) * 2;
    }
  }
  template <typename Off>
  static __device__ __forceinline__ void issue_one(const char* org, const Off (&offs)[PER_WAVE], char* lds, int wave, int j) {
    __builtin_amdgcn_global_load_lds((gptr_void*)at_offset(org, offs[j]), (lds_void*)(lds + (wave * PER_WAVE + j) * 1024), 16, 0, 0);
  }
  template <typename Off>
  static __device__ __forceinline__ void issue(const char* org, const Off (&offs)[PER_WAVE], char* lds, int wave) {
#pragma unroll
    for (int j = 0; j < PER_WAVE; ++j) issue_one(org, offs, lds, wave, j);
  }
  // bytes from one step's panel to the next one's
  static __device__ __forceinline__ int64_t stride(int64_t ld) { return (KMAJOR ? (int64_t)BK : (int64_t)BK * ld) * 2; }

  static constexpr int READS_PER_FRAG = KMAJOR ? 1 : 2;
  // MFMA operands: fragment F holds the 16 rows from rb0 + 16 F on (rb0: first row of the wave's tile) for the 32-wide
  // contraction step KS, lane l elements (row l % 16, k = KS * 32 + (l / 16) * 8 + 0..7), read with volatile asm.
  // frag_lane: the lane's part of the address; the swizzle and F share bits of it, the rest is the instruction's offset.
  static __device__ __forceinline__ uint32_t frag_lane(int rb0, int lane) {
    if constexpr (KMAJOR) {
      const int row = rb0 + (lane & 15);
      return (uint32_t)(row * CPR + swz(row, lane >> 4)) * 16u;
    } else {
      const int i = lane & 15, lrow = 8 * (lane >> 4) + (i >> 2);
      return (uint32_t)(lrow * CPR + swz(lrow, rb0 / 8 + ((i >> 1) & 1))) * 16u + (uint32_t)(i & 1) * 8u;
    }
  }
  template <int F, int KS> static __device__ __forceinline__ void frag_issue(FragRegs<KMAJOR>& f, uint32_t base, uint32_t lane_part) {
    static_assert(BK == 64, "offsets of a 64-wide step");
    if constexpr (KMAJOR) {
      lds_read128_at<F * 16 * CPR * 16>(f.q, base + (lane_part ^ (uint32_t)(KS * 64)));
    } else {
      const uint32_t a = base + (lane_part ^ (uint32_t)(F % 8 * 32));
      lds_read64_tr_at<F / 8 * 256 + KS * 32 * CPR * 16>(f.lo, a);
      lds_read64_tr_at<F / 8 * 256 + (KS * 32 + 4) * CPR * 16>(f.hi, a);
    }
  }
};

// Where the LDS reads of the next 32-wide step go among the TM x TN MFMAs of a step (row by row): B's fragments (items 0 to
// TN - 1), which every row needs, into a second set of registers behind the first MFMAs; A's (the items after them) into the
// registers that the row just multiplied has left.  `from`: first MFMA that may carry reads (behind a hand-over to the next
// stage: then two at a time).
template <int TM, int TN> struct ReadSlots {
  int slot[TN + TM];  // ascending
  constexpr ReadSlots(int from) : slot() {
    int at = from, n = 0;
    for (int q = 0; q < TN + TM; ++q) {
      const int earliest = q < TN ? 0 : TN * (q - TN) + TN - 1, most = q < TN && from == 0 ? 1 : 2;
      if (at < earliest) { at = earliest; n = 0; }
      if (n == most && at < TM * TN - 1) { ++at; n = 0; }
      ++n;
      slot[q] = at;
    }
  }
  constexpr int before(int m) const {  // items that go behind MFMAs ahead of m
    int q = 0;
    while (q < TN + TM && slot[q] < m) ++q;
    return q;
  }
};
// MFMA rows of a stage's last step that come ahead of the hand-over to the next stage
constexpr int hand_rows(int tm) { return tm >= 8 ? 5 : tm >= 4 ? 2 : 1; }

// bias[n .. n + 3] in T
template <typename T> __device__ __forceinline__ typename Vec<T>::v4 bias4(const GemmParams& p, int n) {
  if (!p.bias_f32) return *reinterpret_cast<const typename Vec<T>::v4*>((const T*)p.bias + n);
  const f32x4 b = *reinterpret_cast<const f32x4*>((const float*)p.bias + n);
  typename Vec<T>::v4 r;
#pragma unroll
  for (int e = 0; e < 4; ++e) r[e] = (T)b[e];
  return r;
}
template <typename T> __device__ __forceinline__ T bias1(const void* bias, int f32, int n) {
  return f32 ? (T)((const float*)bias)[n] : ((const T*)bias)[n];
}

// Epilogue of the direct-to-LDS kernel.  Each wave rounds its accumulators (after
// bias / ReLU), parks one 32-row block at a time in a private LDS region and
// reads it back row-contiguously, so every global store instruction writes whole
// 16-byte chunks of complete row segments (8 rows x 128 B for a 64-wide wave
// tile) instead of 32 scattered 16-byte pieces.
// PLAIN: the caller knows that there is no bias, ReLU, mask or sign-bit work (most launches of a
// training step): the write-out is then straight-line code without the tests for them.
// ANY: rows of C, the bias and the mask start at any element and N is any number (register-staged kernel):
// the same 16-byte accesses at element alignment, the chunk that crosses the end of a row by elements.
template <typename T, typename TO, int TM, int TN, int WTM, int WTN, bool PLAIN = false, bool FULL = false, bool ANY = false>
__device__ __forceinline__ void gemm_epilogue_lds(const GemmParams& p, f32x4 (&acc)[TM][TN], char* smem, int m0,
                                                  int n0, int wm, int wn, int wave, int lane,
                                                  const uint8_t (*sign_bytes)[4] = nullptr) {
  constexpr int ES = (int)sizeof(TO);
  constexpr int ROWB = WTN * ES + 16;     // padded row pitch in bytes
  constexpr int CH = WTN * ES / 16;       // 16-byte chunks per row
  constexpr int RPI = 64 / CH;            // rows covered by one wave-wide access
  constexpr int EPC = 16 / ES;            // elements per chunk
  char* mine = smem + wave * (32 * ROWB);
  const void* bias = PLAIN ? nullptr : p.bias;
  const bool relu = !PLAIN && p.relu;
  const void* mask = PLAIN ? nullptr : p.mask;
  const void* sign_in = PLAIN ? nullptr : p.sign_in;
  void* sign_out = PLAIN ? nullptr : p.sign_out;
  const float alpha = (!PLAIN && p.alpha) ? *p.alpha : 1.f;
  TO* C = (TO*)p.C;
  const int nbase = n0 + wn * WTN;
  // this lane stores the same 16-byte column chunk of every row it handles: the column part of the
  // address (with its division by the chunk width) is computed once, not per store (-0.2 ms per
  // step of the 410M model: the store loop is where short-contraction launches spend their time)
  const int n_lane = nbase + (lane % CH) * EPC;
  const int64_t col_off = n_lane + (int64_t)(n_lane / p.chunk_n) * p.chunk_skip;
  // ... and so is the row part of its first store; the others lie whole multiples of ldc further on
  TO* const row0 = C + (int64_t)(m0 + wm * WTM + lane / CH) * p.ldc + col_off;
  // this lane's bias values: the same for every 32-row block, requested once ahead of the loop
  typename Vec<T>::v4 bvals[TN] = {};
  if (bias) {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int nl = j * 16 + (lane >> 4) * 4;
      if constexpr (ANY) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (nbase + nl + e < p.N) bvals[j][e] = bias1<T>(bias, p.bias_f32, nbase + nl + e);
      } else {
        if (nbase + nl < p.N) bvals[j] = bias4<T>(p, nbase + nl);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < TM / 2; ++i) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int r = h * 16 + (lane & 15), nl = j * 16 + (lane >> 4) * 4;
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = acc[i * 2 + h][j][e];
        if (!PLAIN) {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] *= alpha;
        }
        if (bias) {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] += (float)bvals[j][e];
        }
        if (relu) {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = fmaxf(v[e], 0.f);
        }
        if (ES == 4) {
          f32x4 o = {v[0], v[1], v[2], v[3]};
          *reinterpret_cast<f32x4*>(mine + r * ROWB + nl * 4) = o;
        } else {
          typename Vec<T>::v4 o;
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = (T)v[e];
          *reinterpret_cast<typename Vec<T>::v4*>(mine + r * ROWB + nl * 2) = o;
        }
      }
    }
    // all row segments of the block are requested from the slab before the first store: each store
    // then waits for its own read only (a read followed at once by its store exposes the LDS
    // latency once per store)
    u32x4 vals[32 / RPI];
#pragma unroll
    for (int rr = 0; rr < 32 / RPI; ++rr) vals[rr] = lds_ld16(mine, (rr * RPI + lane / CH) * ROWB + (lane % CH) * 16);
#pragma unroll
    for (int rr = 0; rr < 32 / RPI; ++rr) {
      const int r = rr * RPI + lane / CH, c = lane % CH;
      u32x4 val = vals[rr];
      const int m = m0 + wm * WTM + i * 32 + r, n = nbase + c * EPC;
      if (FULL || (m < p.M && n < p.N)) {
        if (mask) {  // ReLU gradient mask fused into the write-out: zero where the activation is not positive
          const T* mk = (const T*)mask + (int64_t)m * p.ldmask + n;
          if constexpr (ES == 2 && ANY) {
            const typename Vec<T>::v8 mv = __builtin_bit_cast(typename Vec<T>::v8, Row<T, true>::load(mk, 0, p.N - n));
            typename Vec<T>::v8 cv = __builtin_bit_cast(typename Vec<T>::v8, val);
#pragma unroll
            for (int e = 0; e < 8; ++e)
              if (!((float)mv[e] > 0.f)) cv[e] = (T)0.f;
            val = __builtin_bit_cast(u32x4, cv);
          } else if constexpr (ANY) {
            f32x4 cv = __builtin_bit_cast(f32x4, val);
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (n + e < p.N && !((float)mk[e] > 0.f)) cv[e] = 0.f;
            val = __builtin_bit_cast(u32x4, cv);
          } else if constexpr (ES == 2) {
            const typename Vec<T>::v8 mv = __builtin_bit_cast(typename Vec<T>::v8, ld16(mk));
            typename Vec<T>::v8 cv = __builtin_bit_cast(typename Vec<T>::v8, val);
#pragma unroll
            for (int e = 0; e < 8; ++e)
              if (!((float)mv[e] > 0.f)) cv[e] = (T)0.f;
            val = __builtin_bit_cast(u32x4, cv);
          } else {
            const typename Vec<T>::v4 mv = *reinterpret_cast<const typename Vec<T>::v4*>(mk);
            f32x4 cv = __builtin_bit_cast(f32x4, val);
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (!((float)mv[e] > 0.f)) cv[e] = 0.f;
            val = __builtin_bit_cast(u32x4, cv);
          }
        }
        if (!ANY && sign_in) {  // the same mask from one bit per element
          unsigned bits;
          if constexpr (ES == 2) bits = sign_bytes[i][rr];  // requested before the main loop
          else bits = ((const uint8_t*)sign_in)[(int64_t)m * p.ldsign + (n >> 3)] >> (n & 7);
          if constexpr (ES == 2) {
            typename Vec<T>::v8 cv = __builtin_bit_cast(typename Vec<T>::v8, val);
#pragma unroll
            for (int e = 0; e < 8; ++e)
              if (!((bits >> e) & 1u)) cv[e] = (T)0.f;
            val = __builtin_bit_cast(u32x4, cv);
          } else {
            f32x4 cv = __builtin_bit_cast(f32x4, val);
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (!((bits >> e) & 1u)) cv[e] = 0.f;
            val = __builtin_bit_cast(u32x4, cv);
          }
        }
        if constexpr (ES == 2) {
          if (!ANY && sign_out) {  // a chunk is 8 elements: one byte
            const typename Vec<T>::v8 cv = __builtin_bit_cast(typename Vec<T>::v8, val);
            unsigned bits = 0;
#pragma unroll
            for (int e = 0; e < 8; ++e) bits |= ((float)cv[e] > 0.f ? 1u : 0u) << e;
            ((uint8_t*)sign_out)[(int64_t)m * p.ldsign + (n >> 3)] = (uint8_t)bits;
          }
        }
        TO* const dst = row0 + (int64_t)(i * 32 + rr * RPI) * p.ldc;
        if constexpr (ANY && FULL) st16_elem(dst, val, std::integral_constant<int, ES>());
        else if constexpr (ANY) Row<TO, true>::store(dst, 0, p.N - n, val);
        else st16(dst, val);
      }
    }
  }
}

// One bit per element of a chunk of eight 16-bit values none of which is negative (a ReLU output;
// -0 counts as zero): bit e set where element e is positive.  Word arithmetic on the packed
// halves: h & 0x7fff is 0 or at least 1, so (h & 0x7fff) + 0x7fff carries into bit 15 exactly
// for the positive ones (and never into the neighbouring half).
__device__ __forceinline__ unsigned positive_bits8(u32x4 v) {
  unsigned b = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const unsigned t = ((v[k] & 0x7fff7fffu) + 0x7fff7fffu) >> 15 & 0x00010001u;  // elements 2k (bit 0), 2k+1 (bit 16)
    b |= t << (2 * k);
  }
  return (b | b >> 15) & 0xffu;
}
// ... and the reverse: the chunk with every element whose bit is clear set to zero
__device__ __forceinline__ u32x4 keep_by_bits8(u32x4 v, unsigned bits) {
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const unsigned lo = (unsigned)__builtin_amdgcn_sbfe((int)bits, 2 * k, 1);      // 0 or 0xffffffff
    const unsigned hi = (unsigned)__builtin_amdgcn_sbfe((int)bits, 2 * k + 1, 1);
    v[k] &= __builtin_amdgcn_perm(hi, lo, 0x05040100u);  // bytes: lo.0 lo.1 hi.0 hi.1
  }
  return v;
}

// Write-out of a full tile with the ReLU sign bits, 16-bit result, no tests in the store loop.
//  BITS_OUT: C = relu(acc + bias), bits = (C > 0).  A lane's bit bytes go to an LDS image of the
//            tile's bits (BM rows of BN / 8 bytes) and leave it as whole 16-byte pieces after a
//            barrier: stored from the loop they would be 64 single bytes per store instruction,
//            eight to a row, a partial write of eight lines each.
//  !BITS_OUT: C = bit ? acc : 0, the bytes requested before the main loop (sign_bytes).
template <typename T, int BM, int BN, int TM, int TN, int WTM, int WTN, bool BITS_OUT>
__device__ __forceinline__ void gemm_epilogue_bits(const GemmParams& p, f32x4 (&acc)[TM][TN], char* smem, int m0, int n0,
                                                   int wm, int wn, int wave, int lane, const uint8_t (*sign_bytes)[4]) {
  constexpr int ROWB = WTN * 2 + 16, CH = WTN * 2 / 16, RPI = 64 / CH;
  constexpr int NW = (BM / WTM) * (BN / WTN);
  constexpr int IMG = NW * 32 * ROWB;  // the bit image lies behind the waves' slabs
  static_assert(BN / 8 % 16 == 0, "rows of the bit image are whole 16-byte pieces");
  char* mine = smem + wave * (32 * ROWB);
  T* C = (T*)p.C;
  const int nbase = n0 + wn * WTN;
  const int n_lane = nbase + (lane % CH) * 8;
  T* const row0 = C + (int64_t)(m0 + wm * WTM + lane / CH) * p.ldc + n_lane + (int64_t)(n_lane / p.chunk_n) * p.chunk_skip;
  typename Vec<T>::v4 bvals[TN] = {};
  if (BITS_OUT && p.bias) {
#pragma unroll
    for (int j = 0; j < TN; ++j) bvals[j] = bias4<T>(p, nbase + j * 16 + (lane >> 4) * 4);
  }
#pragma unroll
  for (int i = 0; i < TM / 2; ++i) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        typename Vec<T>::v4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float v = acc[i * 2 + h][j][e];
          if (BITS_OUT) v = fmaxf(v + (float)bvals[j][e], 0.f);
          o[e] = (T)v;
        }
        *reinterpret_cast<typename Vec<T>::v4*>(mine + (h * 16 + (lane & 15)) * ROWB + (j * 16 + (lane >> 4) * 4) * 2) = o;
      }
    u32x4 vals[32 / RPI];
#pragma unroll
    for (int rr = 0; rr < 32 / RPI; ++rr) vals[rr] = lds_ld16(mine, (rr * RPI + lane / CH) * ROWB + (lane % CH) * 16);
#pragma unroll
    for (int rr = 0; rr < 32 / RPI; ++rr) {
      u32x4 val = vals[rr];
      if (BITS_OUT) {
        const int row = wm * WTM + i * 32 + rr * RPI + lane / CH;  // in the tile
        smem[IMG + row * (BN / 8) + wn * (WTN / 8) + lane % CH] = (char)positive_bits8(val);
      } else {
        val = keep_by_bits8(val, sign_bytes[i][rr]);
      }
      st16(row0 + (int64_t)(i * 32 + rr * RPI) * p.ldc, val);
    }
  }
  if (BITS_OUT) {
    __syncthreads();
    constexpr int PIECES = BM * (BN / 8) / 16, PPR = BN / 8 / 16;  // 16-byte pieces of the image, per row
    uint8_t* out = (uint8_t*)p.sign_out + (int64_t)m0 * p.ldsign + n0 / 8;
    for (int q = threadIdx.x; q < PIECES; q += NW * 64)
      *reinterpret_cast<u32x4*>(out + (int64_t)(q / PPR) * p.ldsign + (q % PPR) * 16) = lds_ld16(smem, IMG + q * 16);
  }
}

// NS: pipeline stages in LDS.  2: ping-pong -- the loads of a stage are requested while the stage before it is
// being multiplied, and have one stage's time to arrive.  3: a stage's loads are requested two stages ahead
// and have two stages' time: for tiles whose stage is short (256x128: half the MFMAs of 256x256 per stage)
// one stage's time does not cover the latency of operands that come from HBM rather than from the L2.
template <typename T, int BM, int BN, int BK, int WM, int WN, bool A_KMAJOR, bool B_KMAJOR, int NS = 2, typename Off = uint32_t>
__device__ __forceinline__ void gemm_dma_body(const GemmParams& p, const int pid) {
  static_assert(NS == 2 || NS == 3, "two or three pipeline stages");
  constexpr int NW = WM * WN;
  constexpr int WTM = BM / WM, WTN = BN / WN;
  constexpr int TM = WTM / 16, TN = WTN / 16;
  constexpr int GROUP_M = 8;
  constexpr int KSTEPS = BK / 32;
  typedef DmaPanel<T, BM, BK, A_KMAJOR, NW> PA;
  typedef DmaPanel<T, BN, BK, B_KMAJOR, NW> PB;
  typedef typename Vec<T>::v8 v8;
  constexpr int STAGE = PA::BYTES + PB::BYTES;      // two stages, ping-pong
  constexpr int LPS = PA::PER_WAVE + PB::PER_WAVE;  // loads per wave per stage
  constexpr int NEARLY = LPS / 2;  // loads of a stage issued right after the hand-over to the stage before it
  static_assert(KSTEPS == 2, "B's fragments alternate between two sets of registers");
  extern __shared__ __attribute__((aligned(16))) char smem[];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform: LDS slab addresses stay scalar
  const int wm = wave / WN, wn = wave % WN;

  const int tiles = p.tiles_m * p.tiles_n;
  const int split = pid / tiles;
  const int t = pid - split * tiles;
  const int per_group = GROUP_M * p.tiles_n;
  const int group = t / per_group;
  const int first_m = group * GROUP_M;
  const int gsz = min(p.tiles_m - first_m, GROUP_M);
  const int tm = first_m + (t % per_group) % gsz;
  const int tn = (t % per_group) / gsz;
  const int m0 = tm * BM, n0 = tn * BN;
  const int kbeg = split * p.k_per_split;
  const int kend = min(p.K, kbeg + p.k_per_split);
  const int nk = (kend - kbeg) / BK;

  Off oa[PA::PER_WAVE], ob[PB::PER_WAVE];
  PA::init(oa, p.lda, m0, p.M, wave, lane);
  const T* B = (const T*)p.B;
  int nb = n0, nend = p.N;  // the tile's columns in B
  if (!B_KMAJOR && p.b_each) {
    const int i = n0 / p.b_each;
    B = (const T*)(i == 0 ? p.B : i == 1 ? p.B1 : p.B2);
    nb = n0 - i * p.b_each;
    nend = p.b_each;
  }
  PB::init(ob, p.ldb, nb, nend, wave, lane);
  const char* pa = PA::origin((const T*)p.A, p.lda, m0, kbeg);
  const char* pb = PB::origin(B, p.ldb, nb, kbeg);
  const int64_t sa = PA::stride(p.lda), sb = PB::stride(p.ldb);
  const uint32_t la = PA::frag_lane(wm * WTM, lane), lb = PA::BYTES + PB::frag_lane(wn * WTN, lane);

  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.f;

  // Mask bits of a 16-bit result: this lane's bytes (one per 8-element chunk it will store, in the
  // order of the write-out) are requested here, a whole main loop ahead of their use -- loaded in
  // the write-out they would sit between every LDS read and the store that needs both.
  static_assert(WTN == 64 || WTN == 32, "four or two wave-wide stores per 32-row block of a 16-bit result");
  uint8_t sign_bytes[TM / 2][4] = {};
  if (p.sign_in && !p.out_f32) {
    constexpr int CH16 = WTN * 2 / 16, RPI16 = 64 / CH16;
#pragma unroll
    for (int i = 0; i < TM / 2; ++i)
#pragma unroll
      for (int rr = 0; rr < 32 / RPI16; ++rr) {
        const int m = m0 + wm * WTM + i * 32 + rr * RPI16 + lane / CH16, n = n0 + wn * WTN + (lane % CH16) * 8;
        if (m < p.M && n < p.N) sign_bytes[i][rr] = ((const uint8_t*)p.sign_in)[(int64_t)m * p.ldsign + (n >> 3)];
      }
  }

  // Bare s_barrier everywhere in the pipeline: __syncthreads() adds a fence that would
  // drain every outstanding direct-to-LDS load.  The waits that matter are explicit.
  auto barrier = [&]() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  FragRegs<A_KMAJOR> fa[TM];
  FragRegs<B_KMAJOR> fb[2][TN];
  const uint32_t lds0 = lds_address(smem);
  // operand fragment for 32-wide step KS of the stage at LDS offset `at`: item q < TN is B's (into set KS), the others A's
  auto read_item = [&](uint32_t at, auto ks_c, auto q_c) {
    constexpr int ks = decltype(ks_c)::value, q = decltype(q_c)::value;
    if constexpr (q < TN) PB::template frag_issue<q, ks>(fb[ks][q], lds0 + at, lb);
    else PA::template frag_issue<q - TN, ks>(fa[q - TN], lds0 + at, la);
  };
  auto load_item = [&](uint32_t at, int q) {
    if (q < PA::PER_WAVE) PA::issue_one(pa, oa, smem + at, wave, q);
    else PB::issue_one(pb, ob, smem + at + PA::BYTES, wave, q - PA::PER_WAVE);
  };
  auto load_all = [&](uint32_t at) {
    PA::issue(pa, oa, smem + at, wave);
    PB::issue(pb, ob, smem + at + PA::BYTES, wave);
    pa += sa;
    pb += sb;
  };

  // ---- prologue: step 0 into stage 0, then its first operands and the head of step 1
  if (nk > 0) {
    load_all(0);
    // the head of step 1 goes out before step 0 is waited for: the two travel together through
    // the cold start instead of one after the other
    if constexpr (NS == 3) {
      // three buffers: all of step 1 and the head of step 2
      if (nk > 1) {
        load_all(STAGE);
        if (nk > 2) {
#pragma unroll
          for (int q = 0; q < NEARLY; ++q) load_item(2 * STAGE, q);
          wait_vmcnt<LPS + NEARLY>();  // loads complete in order: all but the youngest LPS + NEARLY = step 0
        } else {
          wait_vmcnt<LPS>();
        }
      } else {
        wait_vmcnt<0>();
      }
    } else if (nk > 1) {
#pragma unroll
      for (int q = 0; q < NEARLY; ++q) load_item(STAGE, q);
      wait_vmcnt<NEARLY>();  // loads complete in order: all but the NEARLY youngest = step 0
    } else {
      wait_vmcnt<0>();
    }
    barrier();
    static_for<TN + TM>([&](auto q_c) { read_item(0, std::integral_constant<int, 0>(), q_c); });
  }

  // ---- main loop.  Every LDS read and load sits behind an MFMA, pinned there by scheduling barriers: the matrix pipe is
  // busy for 16 cycles per MFMA and the wave is free to issue meanwhile.  A stage is two steps of 32, a step TM x TN MFMAs,
  // row by row and back and forth along the rows, so that every MFMA has one operand in common with the one before it (the
  // MFMA stream alone draws less power that way: 1.13 -> 1.10 us per 256x256x64); ReadSlots says where the reads of the next step go.  An LDS read has most of a step to land: ahead of row i
  // the wait leaves in flight what was requested after A's fragment i (B's are older).  Of the next stage's loads the first
  // half goes out behind the hand-over (wait for this wave's loads and reads, barrier), into the buffer everyone has just
  // left, the rest at the head of step 0.
  constexpr int NMFMA = TM * TN;
  constexpr int HAND = hand_rows(TM) * TN;  // MFMAs of the last step ahead of the hand-over
  constexpr int RA = PA::READS_PER_FRAG, RB = PB::READS_PER_FRAG;
  static_assert(LPS % 2 == 0, "loads go out in two halves");
  // One 64-wide stage.  MORE: another stage follows (hand over to it); MORE2: and one after that
  // (its first loads go out).  Compile-time, so the steady state of the loop has no branch.
  // With three buffers (NS == 3) everything that is loaded lies one stage further ahead: step 0 sends the
  // rest of the stage after the next one into the third buffer `far`, the last step the head of the stage
  // after that into `cur`; MORE3: that stage exists.  The hand-over then waits for all but the youngest
  // stage's loads.
  auto stage = [&](uint32_t cur, uint32_t nxt, uint32_t far, auto more_c, auto more2_c, auto more3_c) {
    constexpr bool MORE = decltype(more_c)::value, MORE2 = decltype(more2_c)::value, MORE3 = decltype(more3_c)::value;
    constexpr bool LOAD0 = NS == 3 ? MORE2 : MORE;    // step 0 has loads to send
    constexpr bool LOADL = NS == 3 ? MORE3 : MORE2;   // the last step has
    const uint32_t dst0 = NS == 3 ? far : nxt;
    static_for<KSTEPS>([&](auto ks_c) {
      constexpr int ks = decltype(ks_c)::value;
      constexpr bool last = ks + 1 == KSTEPS, hands = last && MORE;
      typedef std::integral_constant<int, last ? 0 : ks + 1> next_ks;
      constexpr ReadSlots<TM, TN> slots(hands ? HAND : 0);
      static_for<NMFMA>([&](auto m_c) {
        constexpr int m = decltype(m_c)::value, i = m / TN, j = i % 2 ? TN - 1 - m % TN : m % TN;
        if constexpr (hands && m == HAND) {
          wait_lgkmcnt<0>();  // this wave has read the last operands of `cur`
          wait_vmcnt<(NS == 3 && MORE2) ? LPS : 0>();  // its loads of the next stage have landed
          barrier();                                   // ... and everyone's
          __builtin_amdgcn_sched_barrier(0);
        } else if constexpr (m % TN == 0 && (!hands || m < HAND)) {
          constexpr int flying = (TM - 1 - i) * RA + (last || i == 0 ? 0 : TN * RB + i * RA);
          wait_lgkmcnt<(flying < 15 ? flying : 15)>();
          __builtin_amdgcn_sched_barrier(0);
        }
        acc[i][j] = mfma16(fb[ks][j].template get<v8>(), fa[i].template get<v8>(), acc[i][j]);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (!last || MORE) {
          constexpr int q0 = slots.before(m), q1 = slots.before(m + 1);
          static_for<q1 - q0>([&](auto q) {
            read_item(last ? nxt : cur, next_ks(), std::integral_constant<int, q0 + decltype(q)::value>());
          });
        }
        if constexpr (ks == 0 && LOAD0) {  // the rest of the next stage (NS == 3: of the one after it)
#pragma unroll
          for (int q = 0; q < LPS - NEARLY; ++q)
            if (TN + 2 * q == m || (TN + 2 * q > m && m == NMFMA - 1)) load_item(dst0, NEARLY + q);
        }
        if constexpr (last && LOADL) {     // first half of the stage after the next one (NS == 3: one further)
          if constexpr (m == HAND) { pa += sa; pb += sb; }
#pragma unroll
          for (int q = 0; q < NEARLY; ++q)
            if (HAND + 4 + 2 * q == m || (HAND + 4 + 2 * q > m && m == NMFMA - 1)) load_item(cur, q);
        }
        __builtin_amdgcn_sched_barrier(0);
      });
    });
  };
  typedef std::integral_constant<bool, true> yes_t;
  typedef std::integral_constant<bool, false> no_t;
  int kt = 0;
  if constexpr (NS == 3) {
    uint32_t o0 = 0, o1 = STAGE, o2 = 2 * STAGE;   // buffers of this stage, the next one and the one after it
    auto rotate = [&]() { const uint32_t t = o0; o0 = o1; o1 = o2; o2 = t; ++kt; };
    for (; kt + 3 < nk; rotate()) stage(o0, o1, o2, yes_t(), yes_t(), yes_t());
    if (kt + 2 < nk) { stage(o0, o1, o2, yes_t(), yes_t(), no_t()); rotate(); }
    if (kt + 1 < nk) { stage(o0, o1, o2, yes_t(), no_t(), no_t()); rotate(); }
    if (kt < nk) stage(o0, o1, o2, no_t(), no_t(), no_t());
  } else {
    for (; kt + 2 < nk; ++kt) stage((kt & 1) * STAGE, (~kt & 1) * STAGE, 0, yes_t(), yes_t(), no_t());
    if (kt + 1 < nk) {
      stage((kt & 1) * STAGE, (~kt & 1) * STAGE, 0, yes_t(), no_t(), no_t());
      ++kt;
    }
    if (kt < nk) stage((kt & 1) * STAGE, (~kt & 1) * STAGE, 0, no_t(), no_t(), no_t());
  }

  static_assert(NW * 32 * (WTN * 4 + 16) <= NS * STAGE, "epilogue staging must fit in the pipeline LDS");
  static_assert(NW * 32 * (WTN * 2 + 16) + BM * BN / 8 <= NS * STAGE, "... and so must the image of a tile's sign bits behind it");
  const bool full = m0 + BM <= p.M && n0 + BN <= p.N;  // no row or column of the tile lies outside C: stores need no test
  if (p.splits > 1) {
    // fp32 partial of this contraction slice: a plain (M, N) matrix, written like an fp32 result
    GemmParams q = p;
    q.C = p.partial + (int64_t)split * p.M * p.N;
    q.ldc = p.N;
    q.bias = nullptr;
    q.relu = 0;
    q.mask = nullptr;
    q.sign_out = nullptr;
    q.sign_in = nullptr;
    q.alpha = nullptr;
    q.chunk_n = p.N;
    q.chunk_skip = 0;
    __syncthreads();  // all waves are done reading the last pipeline stage
    if (full) gemm_epilogue_lds<T, float, TM, TN, WTM, WTN, true, true>(q, acc, smem, m0, n0, wm, wn, wave, lane);
    else gemm_epilogue_lds<T, float, TM, TN, WTM, WTN, true>(q, acc, smem, m0, n0, wm, wn, wave, lane);
  } else {
    __syncthreads();  // all waves are done reading the last pipeline stage
    const bool plain = !p.bias && !p.relu && !p.mask && !p.sign_in && !p.sign_out && !p.alpha;
    if (p.out_f32) {
      if (plain && full) gemm_epilogue_lds<T, float, TM, TN, WTM, WTN, true, true>(p, acc, smem, m0, n0, wm, wn, wave, lane);
      else if (plain) gemm_epilogue_lds<T, float, TM, TN, WTM, WTN, true>(p, acc, smem, m0, n0, wm, wn, wave, lane);
      else gemm_epilogue_lds<T, float, TM, TN, WTM, WTN>(p, acc, smem, m0, n0, wm, wn, wave, lane);
    } else {
      // the two sign-bit launches of a fused MLP, on full tiles of a plain (unchunked) result whose bit rows take
      // 16-byte pieces: write-outs of their own, nothing tested per store
      const bool bits_fast = BN >= 128 && full && !p.mask && !p.alpha && p.chunk_skip == 0 && p.ldsign % 16 == 0 &&
                             ((reinterpret_cast<uintptr_t>(p.sign_out) | reinterpret_cast<uintptr_t>(p.sign_in)) & 15) == 0;
      if (plain && full) return gemm_epilogue_lds<T, T, TM, TN, WTM, WTN, true, true>(p, acc, smem, m0, n0, wm, wn, wave, lane);
      if (plain) return gemm_epilogue_lds<T, T, TM, TN, WTM, WTN, true>(p, acc, smem, m0, n0, wm, wn, wave, lane);
      if constexpr (BN >= 128) {
        if (bits_fast && p.sign_out && p.relu) return gemm_epilogue_bits<T, BM, BN, TM, TN, WTM, WTN, true>(p, acc, smem, m0, n0, wm, wn, wave, lane, sign_bytes);
        if (bits_fast && p.sign_in && !p.bias && !p.relu) return gemm_epilogue_bits<T, BM, BN, TM, TN, WTM, WTN, false>(p, acc, smem, m0, n0, wm, wn, wave, lane, sign_bytes);
      }
      gemm_epilogue_lds<T, T, TM, TN, WTM, WTN>(p, acc, smem, m0, n0, wm, wn, wave, lane, sign_bytes);
    }
  }
}

template <typename T, int BM, int BN, int BK, int WM, int WN, int WPE, bool A_KMAJOR, bool B_KMAJOR, int NS = 2>
__global__ __launch_bounds__(WM* WN * 64, WPE) void gemm_dma_kernel(GemmParams p) {
  const int pid = (p.flags & 1) ? (int)blockIdx.x : remap_xcd(blockIdx.x, p.tiles_m * p.tiles_n * p.splits, p.xcds);
  gemm_dma_body<T, BM, BN, BK, WM, WN, A_KMAJOR, B_KMAJOR, NS>(p, pid);
}

// Operands with rows beyond kMaxPitch: 64-bit offsets, which the 128x128 tile has the registers for.  Same steps, same order of
// sums as any other tile of these kernels.
template <typename T, bool A_KMAJOR, bool B_KMAJOR>
__global__ __launch_bounds__(256, 2) void gemm_wide_kernel(GemmParams p) {
  const int pid = (p.flags & 1) ? (int)blockIdx.x : remap_xcd(blockIdx.x, p.tiles_m * p.tiles_n * p.splits, p.xcds);
  gemm_dma_body<T, 128, 128, 64, 2, 2, A_KMAJOR, B_KMAJOR, 2, uint64_t>(p, pid);
}

// ---------------------------------------------------------------------------
// Anything the direct-to-LDS kernel cannot take: extents, leading dimensions and pointers of any
// element alignment, contractions that are not a multiple of BK.  The same tiles, LDS layout, MFMA
// order and write-out; a panel travels HBM -> registers -> LDS in 16-byte loads at element alignment
// (direct-to-LDS loads are kept to aligned addresses).  The loads of a stage are requested two
// stages ahead of its MFMAs: they stay in registers for one stage and are parked in the LDS buffer
// the other stage has just left, behind the MFMAs of the next.
// Only a slice's last stage tests extents: every stage before it reads whole chunks without a test --
// rows beyond M / N are clamped, a chunk that crosses the end of a contraction-strided row reads on
// into the row after it, which exists (its products reach only entries of C that are not stored).
// Rows shorter than a chunk could run past the last row that way: all their stages are tested.
// Bound by the matrix pipe and the LDS traffic around it like the direct-to-LDS kernel, 25-35 % behind it by the
// stores through the registers.  Against the kernel before it (chunks fetched one stage ahead with a test each, result
// stored from the accumulators, 4 and 2 bytes per lane and row): 4113 x 1733 x 2051 fp16 forward 112 -> 57 us, input
// gradient 103 -> 56, weight gradient 121 -> 59; 8192 x 50257 x 1024 forward 4232 -> 1057 (of the element-wise one),
// 798 TFLOP/s; 8192 x 1024 x 2056 (all aligned, K % 64 != 0) 58 -> 46.
// ---------------------------------------------------------------------------
template <typename T, int R, int BK, bool KMAJOR, int NW, typename Off>
struct RegPanel {
  typedef DmaPanel<T, R, BK, KMAJOR, NW> D;
  static constexpr int PER = D::PER_WAVE;  // chunks per thread
  static constexpr int NT = NW * 64;
  static constexpr int ROWS = NT / D::CPR;  // LDS rows between a thread's chunks
  static_assert(NT % D::CPR == 0 && D::NCHUNK == PER * NT, "panel must divide evenly over the threads");
  static_assert(KMAJOR ? (ROWS / (16 / D::CPR)) % D::CPR == 0 : ROWS % 16 == 0, "a thread's chunks share one swizzle");

  // Thread t owns the LDS slots t, t + NT, ... and fetches the chunk that the swizzle puts there.
  // Offsets in bytes from D::origin.
  static __device__ __forceinline__ void init(Off (&offs)[PER], int64_t ld, int row0, int rmax) {
    const int t = threadIdx.x, lrow = t / D::CPR, c = D::swz(lrow, t % D::CPR);
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      if (KMAJOR) offs[j] = ((Off)(min(row0 + lrow + j * ROWS, rmax - 1) - row0) * (Off)ld + (Off)(c * 8)) * 2;
      else offs[j] = ((Off)(lrow + j * ROWS) * (Off)ld + (Off)(row0 + c * 8 < rmax ? c * 8 : 0)) * 2;
    }
  }
  static __device__ __forceinline__ u32x4 fetch(const T* ptr) {
    return ld16_elem<false>(ptr, std::integral_constant<int, 2>());
  }
  // chunk j of the stage that starts at contraction index k0, zero from kend on
  static __device__ __forceinline__ u32x4 fetch_tested(const T* ptr, int j, int k0, int kend, int row0, int rmax) {
    const int t = threadIdx.x, lrow = t / D::CPR, c = D::swz(lrow, t % D::CPR);
    u32x4 v = {0u, 0u, 0u, 0u};
    if (KMAJOR) {
      const int left = kend - (k0 + c * 8);
      if (left > 0) v = Row<T, true>::load(ptr, 0, left);
    } else if (k0 + lrow + j * ROWS < kend) {
      const int gr = row0 + c * 8 < rmax ? row0 + c * 8 : row0;
      v = Row<T, true>::load(ptr, 0, rmax - gr);
    }
    return v;
  }
};

template <typename T, int BM, int BN, int BK, int WM, int WN, int WPE, bool A_KMAJOR, bool B_KMAJOR>
__global__ __launch_bounds__(WM* WN * 64, WPE) void gemm_reg_kernel(GemmParams p) {
  constexpr int NW = WM * WN, NT = NW * 64;
  constexpr int WTM = BM / WM, WTN = BN / WN;
  constexpr int TM = WTM / 16, TN = WTN / 16;
  constexpr int GROUP_M = 8;
  constexpr int KSTEPS = BK / 32;
  // the tiles of 256 rows keep 32-bit offsets (kMaxPitch): 64 bits are eight registers more, and 256x256 has none left.  It holds all
  // 256, and where just one operand is contraction-strided it parks seven in scratch around the stages that test extents, not in
  // the loop over whole stages
  typedef std::conditional_t<(BM > 128), uint32_t, uint64_t> Off;
  typedef RegPanel<T, BM, BK, A_KMAJOR, NW, Off> PA;
  typedef RegPanel<T, BN, BK, B_KMAJOR, NW, Off> PB;
  typedef typename Vec<T>::v8 v8;
  constexpr int STAGE = PA::D::BYTES + PB::D::BYTES;
  constexpr int LPS = PA::PER + PB::PER;  // chunks per thread per stage
  static_assert(KSTEPS == 2, "stores, loads and hand-over are dealt over two contraction steps");
  extern __shared__ __attribute__((aligned(16))) char smem[];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WN, wn = wave % WN;

  const int tiles = p.tiles_m * p.tiles_n;
  const int pid = (p.flags & 1) ? (int)blockIdx.x : remap_xcd(blockIdx.x, tiles * p.splits, p.xcds);
  const int split = pid / tiles;
  const int t = pid - split * tiles;
  const int per_group = GROUP_M * p.tiles_n;
  const int group = t / per_group;
  const int first_m = group * GROUP_M;
  const int gsz = min(p.tiles_m - first_m, GROUP_M);
  const int tm = first_m + (t % per_group) % gsz;
  const int tn = (t % per_group) / gsz;
  const int m0 = tm * BM, n0 = tn * BN;
  const int kbeg = split * p.k_per_split;
  const int kend = min(p.K, kbeg + p.k_per_split);
  const int nk = (kend - kbeg + BK - 1) / BK;
  // stages that need no test: all but the last one, none where a row may be shorter than a chunk
  const int nfree = (A_KMAJOR || p.lda >= 8) && (B_KMAJOR || p.ldb >= 8) ? nk - 1 : 0;

  Off oa[PA::PER], ob[PB::PER];
  PA::init(oa, p.lda, m0, p.M);
  PB::init(ob, p.ldb, n0, p.N);
  const char* pa = PA::D::origin((const T*)p.A, p.lda, m0, kbeg);
  const char* pb = PB::D::origin((const T*)p.B, p.ldb, n0, kbeg);
  const int64_t sa = PA::D::stride(p.lda), sb = PB::D::stride(p.ldb);

  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.f;

  u32x4 regs[LPS];
  // chunk q of the next stage to be fetched (which starts at contraction index k0) into its register
  auto load_item = [&](int q, int k0, auto tested_c) {
    constexpr bool TESTED = decltype(tested_c)::value;
    if (q < PA::PER) {
      const T* ptr = (const T*)at_offset(pa, oa[q]);
      regs[q] = TESTED ? PA::fetch_tested(ptr, q, k0, kend, m0, p.M) : PA::fetch(ptr);
    } else {
      const T* ptr = (const T*)at_offset(pb, ob[q - PA::PER]);
      regs[q] = TESTED ? PB::fetch_tested(ptr, q - PA::PER, k0, kend, n0, p.N) : PB::fetch(ptr);
    }
    if (q == LPS - 1) {
      pa += sa;
      pb += sb;
    }
  };
  auto store_item = [&](char* dst, int q) {
    if (q < PA::PER) lds_st16(dst, (int)threadIdx.x * 16 + q * NT * 16, regs[q]);
    else lds_st16(dst, PA::D::BYTES + (int)threadIdx.x * 16 + (q - PA::PER) * NT * 16, regs[q]);
  };
  auto barrier = [&]() {  // bare: __syncthreads() would wait for the loads in flight as well
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  FragRegs<A_KMAJOR> fa[TM];
  FragRegs<B_KMAJOR> fb[2][TN];
  const uint32_t lds0 = lds_address(smem);
  const uint32_t la = PA::D::frag_lane(wm * WTM, lane), lb = PA::D::BYTES + PB::D::frag_lane(wn * WTN, lane);
  auto read_item = [&](uint32_t at, auto ks_c, auto q_c) {
    constexpr int ks = decltype(ks_c)::value, q = decltype(q_c)::value;
    if constexpr (q < TN) PB::D::template frag_issue<q, ks>(fb[ks][q], lds0 + at, lb);
    else PA::D::template frag_issue<q - TN, ks>(fa[q - TN], lds0 + at, la);
  };
  typedef std::integral_constant<bool, true> yes_t;
  typedef std::integral_constant<bool, false> no_t;

  // ---- prologue: stage 0 into LDS, stage 1 into the registers, the first operands
#pragma unroll
  for (int q = 0; q < LPS; ++q) {
    if (nfree > 0) load_item(q, kbeg, no_t());
    else load_item(q, kbeg, yes_t());
  }
#pragma unroll
  for (int q = 0; q < LPS; ++q) store_item(smem, q);
  if (nk > 1) {
#pragma unroll
    for (int q = 0; q < LPS; ++q) {
      if (nfree > 1) load_item(q, kbeg + BK, no_t());
      else load_item(q, kbeg + BK, yes_t());
    }
  }
  wait_lgkmcnt<0>();
  barrier();
  static_for<TN + TM>([&](auto q_c) { read_item(0, std::integral_constant<int, 0>(), q_c); });

  // ---- one stage, as in the direct-to-LDS kernel: everything that is not an MFMA sits behind one, pinned by scheduling
  // barriers.  MORE: another stage follows (its chunks are in the registers: stored behind the MFMAs of step 0); LOAD: and one
  // after that, whose chunks are requested into the registers a store has left (TESTED: by extents).  The waits for
  // fragments count reads alone: with stores among them they leave less in flight than they might, never more.
  constexpr int NMFMA = TM * TN;
  constexpr int HAND = hand_rows(TM) * TN;
  constexpr int RA = PA::D::READS_PER_FRAG, RB = PB::D::READS_PER_FRAG;
  auto stage = [&](uint32_t cur, uint32_t nxt, int k2, auto more_c, auto load_c, auto tested_c) {
    constexpr bool MORE = decltype(more_c)::value, LOAD = decltype(load_c)::value, TESTED = decltype(tested_c)::value;
    static_for<KSTEPS>([&](auto ks_c) {
      constexpr int ks = decltype(ks_c)::value;
      constexpr bool last = ks + 1 == KSTEPS, hands = last && MORE;
      typedef std::integral_constant<int, last ? 0 : ks + 1> next_ks;
      constexpr ReadSlots<TM, TN> slots(hands ? HAND : 0);
      static_for<NMFMA>([&](auto m_c) {
        constexpr int m = decltype(m_c)::value, i = m / TN, j = i % 2 ? TN - 1 - m % TN : m % TN;
        if constexpr (hands && m == HAND) {
          wait_lgkmcnt<0>();  // this wave's stores of the next stage are in, it has read the last operands of `cur`
          barrier();          // ... and everyone
          __builtin_amdgcn_sched_barrier(0);
          if constexpr (LOAD && TESTED) {  // branches: here, where no read is in flight whose register a branch might move
#pragma unroll
            for (int q = 0; q < LPS; ++q) load_item(q, k2, tested_c);
            __builtin_amdgcn_sched_barrier(0);
          }
        } else if constexpr (m % TN == 0 && (!hands || m < HAND)) {
          constexpr int flying = (TM - 1 - i) * RA + (last || i == 0 ? 0 : TN * RB + i * RA);
          wait_lgkmcnt<(flying < 15 ? flying : 15)>();
          __builtin_amdgcn_sched_barrier(0);
        }
        acc[i][j] = mfma16(fb[ks][j].template get<v8>(), fa[i].template get<v8>(), acc[i][j]);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (!last || MORE) {
          constexpr int q0 = slots.before(m), q1 = slots.before(m + 1);
          static_for<q1 - q0>([&](auto q) {
            read_item(last ? nxt : cur, next_ks(), std::integral_constant<int, q0 + decltype(q)::value>());
          });
        }
        // step 0: store and load of chunk q, the load half a step behind its store where the step is long enough; the loads
        // that are left in the last step
        constexpr int T0 = m * LPS / NMFMA, T1 = (m + 1) * LPS / NMFMA;
        static_for<T1 - T0>([&](auto q_c) {
          constexpr int q = T0 + decltype(q_c)::value;
          if constexpr (!last && MORE) store_item(smem + nxt, q);
          if constexpr (!last && LOAD && !TESTED && q >= LPS / 2) load_item(q - LPS / 2, k2, tested_c);
          if constexpr (last && LOAD && !TESTED && q < LPS / 2) load_item(q + LPS / 2, k2, tested_c);
        });
        __builtin_amdgcn_sched_barrier(0);
      });
    });
  };
  static_assert(LPS % 2 == 0, "halves of a stage's chunks");
  int kt = 0;
  auto cur = [&]() { return (uint32_t)((kt & 1) * STAGE); };
  auto nxt = [&]() { return (uint32_t)((~kt & 1) * STAGE); };
  for (; kt + 2 < nfree; ++kt) stage(cur(), nxt(), 0, yes_t(), yes_t(), no_t());
  for (; kt + 2 < nk; ++kt) stage(cur(), nxt(), kbeg + (kt + 2) * BK, yes_t(), yes_t(), yes_t());
  if (kt + 1 < nk) {
    stage(cur(), nxt(), 0, yes_t(), no_t(), no_t());
    ++kt;
  }
  stage(cur(), nxt(), 0, no_t(), no_t(), no_t());

  __syncthreads();  // all waves are done reading the last pipeline stage
  const bool full = m0 + BM <= p.M && n0 + BN <= p.N;
  if (p.splits > 1) {
    // fp32 partial of this contraction slice: a plain (M, N) matrix, written like an fp32 result
    GemmParams q = p;
    q.C = p.partial + (int64_t)split * p.M * p.N;
    q.ldc = p.N;
    q.bias = nullptr;
    q.relu = 0;
    q.mask = nullptr;
    q.alpha = nullptr;
    q.chunk_n = p.N;
    q.chunk_skip = 0;
    if (full) gemm_epilogue_lds<T, float, TM, TN, WTM, WTN, true, true, true>(q, acc, smem, m0, n0, wm, wn, wave, lane);
    else gemm_epilogue_lds<T, float, TM, TN, WTM, WTN, true, false, true>(q, acc, smem, m0, n0, wm, wn, wave, lane);
  } else if (p.out_f32) {
    gemm_epilogue_lds<T, float, TM, TN, WTM, WTN, false, false, true>(p, acc, smem, m0, n0, wm, wn, wave, lane);
  } else {
    const bool plain = !p.bias && !p.relu && !p.mask && !p.alpha;
    if (plain && full) gemm_epilogue_lds<T, T, TM, TN, WTM, WTN, true, true, true>(p, acc, smem, m0, n0, wm, wn, wave, lane);
    else gemm_epilogue_lds<T, T, TM, TN, WTM, WTN, false, false, true>(p, acc, smem, m0, n0, wm, wn, wave, lane);
  }
}

// Up to sixteen independent products of one operand layout in ONE launch: workgroup ids
// [first[i], first[i+1]) belong to problem i.  Used for weight gradients, whose output has
// few tiles: side by side they fill the chip with fewer, longer contraction slices.
constexpr int kMaxGroup = 16;
struct GemmGroup {
  GemmParams p[kMaxGroup];
  int first[kMaxGroup + 1];
  int count;
};
static_assert(sizeof(GemmGroup) <= 4000, "the group travels as a kernel argument (4 KB of them at most)");
template <typename T, int BM, int BN, int BK, int WM, int WN, int WPE, bool A_KMAJOR, bool B_KMAJOR>
__global__ __launch_bounds__(WM* WN * 64, WPE) void gemm_dma_group_kernel(GemmGroup g) {
  // (a group with a split tail keeps the ids as dealt, round-robin over the XCDs: whole tiles first, on every
  // XCD alike, then the short slices of the tail -- the remap would hand all of the tail to the last XCDs)
  const int pid = (g.p[0].flags & 1) ? (int)blockIdx.x : remap_xcd(blockIdx.x, g.first[g.count], g.p[0].xcds);
  int i = 0;
#pragma unroll
  for (int k = 1; k < kMaxGroup; ++k)
    if (k < g.count && pid >= g.first[k]) i = k;
  gemm_dma_body<T, BM, BN, BK, WM, WN, A_KMAJOR, B_KMAJOR>(g.p[i], pid - g.first[i]);
}

// Sum the split-contraction partials in a fixed order and apply the epilogue.
//  kReduceRows: N and ldc multiples of 4, 16-byte aligned partials, 8-byte aligned C: four columns of a row at a time
//  kReduceFlat: C is one dense (M, N) matrix and there is no bias, so partials and result are the same flat sequence,
//               taken four elements at a time whatever N is (2051 x 1733 x 4113 in four slices, both passes: 65 -> 61 us)
//  kReduceAny:  element by element
enum ReduceMode { kReduceAny, kReduceRows, kReduceFlat };
template <typename T, typename TO, ReduceMode MODE>
__global__ __launch_bounds__(256) void gemm_reduce(int M, int N, int splits, const float* __restrict__ partial,
                                                    const void* __restrict__ bias, int bias_f32, int relu, TO* __restrict__ C,
                                                    int64_t ldc, int chunk_n, int64_t chunk_skip,
                                                    const float* __restrict__ alpha_ptr) {
  const int64_t total = (int64_t)M * N;
  const float alpha = alpha_ptr ? *alpha_ptr : 1.f;
  if (MODE != kReduceAny) {
    struct alignas(sizeof(TO) * 4) Quad { TO v[4]; };
    const int64_t quads = total >> 2;
    for (int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x; q < quads; q += (int64_t)gridDim.x * 256) {
      const int64_t i = q * 4;
      auto part = [&](int k) {  // a slice of an odd number of elements starts at any of them
        const float* src = partial + (int64_t)k * total + i;
        if (MODE == kReduceRows) return *reinterpret_cast<const f32x4*>(src);
        return __builtin_bit_cast(f32x4, ld16_elem<false>(src, std::integral_constant<int, 4>()));
      };
      f32x4 s = part(0);
      for (int k = 1; k < splits; ++k) s += part(k);
      const int m = MODE == kReduceRows ? (int)(i / N) : 0, n = MODE == kReduceRows ? (int)(i - (int64_t)m * N) : 0;
      Quad qd;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x = s[e] * alpha + (MODE == kReduceRows && bias ? (float)bias1<T>(bias, bias_f32, n + e) : 0.f);
        qd.v[e] = (TO)(relu ? fmaxf(x, 0.f) : x);
      }
      if (MODE == kReduceRows) store_out(C + (int64_t)m * ldc + n + (int64_t)(n / chunk_n) * chunk_skip, qd);
      else store_out(C + i, qd);
    }
    if (MODE == kReduceFlat && blockIdx.x == 0 && threadIdx.x < (total & 3)) {
      const int64_t i = (quads << 2) + threadIdx.x;
      float s = 0.f;
      for (int k = 0; k < splits; ++k) s += partial[(int64_t)k * total + i];
      s *= alpha;
      C[i] = (TO)(relu ? fmaxf(s, 0.f) : s);
    }
  } else {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
      float s = 0.f;
      for (int k = 0; k < splits; ++k) s += partial[(int64_t)k * total + i];
      const int m = (int)(i / N), n = (int)(i - (int64_t)m * N);
      s *= alpha;
      if (bias) s += (float)bias1<T>(bias, bias_f32, n);
      C[(int64_t)m * ldc + n + (int64_t)(n / chunk_n) * chunk_skip] = (TO)(relu ? fmaxf(s, 0.f) : s);
    }
  }
}

// The same second pass for up to kMaxGroup products of one grouped launch at once (blockIdx.y = product;
// no bias, no ReLU): one launch instead of one per product.
struct ReduceItem {
  const float* partial;
  void* C;
  int64_t ldc, chunk_skip;
  int M, N, splits, chunk_n;
};
struct ReduceBatch { ReduceItem it[kMaxGroup]; };
template <typename TO, bool VEC4>
__global__ __launch_bounds__(256) void gemm_reduce_group(ReduceBatch batch) {
  const ReduceItem r = batch.it[blockIdx.y];
  if (r.splits <= 1) return;
  const int64_t total = (int64_t)r.M * r.N;
  TO* C = (TO*)r.C;
  if (VEC4) {
    const int64_t quads = total >> 2;
    for (int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x; q < quads; q += (int64_t)gridDim.x * 256) {
      f32x4 s = *reinterpret_cast<const f32x4*>(r.partial + q * 4);
      for (int k = 1; k < r.splits; ++k) s += *reinterpret_cast<const f32x4*>(r.partial + (int64_t)k * total + q * 4);
      const int64_t i = q * 4;
      const int m = (int)(i / r.N), n = (int)(i - (int64_t)m * r.N);
      struct alignas(sizeof(TO) * 4) Quad { TO v[4]; };
      Quad qd;
#pragma unroll
      for (int e = 0; e < 4; ++e) qd.v[e] = (TO)s[e];
      store_out(C + (int64_t)m * r.ldc + n + (int64_t)(n / r.chunk_n) * r.chunk_skip, qd);
    }
  } else {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
      float s = 0.f;
      for (int k = 0; k < r.splits; ++k) s += r.partial[(int64_t)k * total + i];
      const int m = (int)(i / r.N), n = (int)(i - (int64_t)m * r.N);
      C[(int64_t)m * r.ldc + n + (int64_t)(n / r.chunk_n) * r.chunk_skip] = (TO)s;
    }
  }
}

// ---------------------------------------------------------------------------
// host side: tile choice, contraction split, launch
// ---------------------------------------------------------------------------
struct GemmPlan {
  int cfg;
  int bm, bn, bk;
  int tiles_m, tiles_n, splits, k_per_split;
};

struct TileCfg { int bm, bn, bk, waves, dma; };  // dma: direct-to-LDS kernel
// index = cfg id used by launch_cfg below
static const TileCfg kCfgs[] = {
    {256, 256, 64, 8, 0},  // 0: register-staged, wave tile 128x64, any shape / alignment
    {128, 128, 64, 4, 0},  // 1: register-staged, wave tile 64x64, any shape / alignment
    {256, 256, 64, 8, 1},  // 2: direct-to-LDS, 128 KB LDS, one workgroup per CU, wave tile 128x64
    {128, 128, 64, 4, 1},  // 3: direct-to-LDS, 64 KB LDS, two workgroups per CU, wave tile 64x64
    {256, 128, 64, 8, 1},  // 4: direct-to-LDS, three stages = 144 KB LDS, waves 4x2, wave tile 64x64
    {128, 256, 64, 8, 1},  // 5: direct-to-LDS, three stages = 144 KB LDS, waves 2x4, wave tile 64x64
    {64, 64, 64, 4, 1},    // 6: direct-to-LDS, three stages = 48 KB LDS, waves 2x2, wave tile 32x32: few tiles
    {128, 64, 64, 4, 1},   // 7: direct-to-LDS, three stages = 72 KB LDS, waves 4x1, wave tile 32x64: few tiles
    {256, 128, 64, 8, 0},  // 8: register-staged, waves 4x2, wave tile 64x64, any shape / alignment
};
constexpr int kNumCfgs = (int)(sizeof(kCfgs) / sizeof(kCfgs[0]));

// What the diagnostic entry point may impose on ONE call (nothing is kept between calls):
// a tile configuration (index into kCfgs, -1 = chosen by the cost model), a contraction
// split (0 = chosen), and flag bits -- 1: no XCD remap of the workgroup ids; 64: never cut
// a product along N.  Every product entry point passes kNoForce.
struct GemmForce { int cfg, splits, flags; };
constexpr GemmForce kNoForce = {-1, 0, 0};

// Tile shape, contraction split and the rough cost (microseconds) of running
// M x N x K with tile configuration `cfg`.  The cost constants are fits to
// rocprofv3 kernel durations on MI355X: one "round" of workgroups (one per CU)
// costs a fixed part (launch, cold first loads, result write-out) plus a part
// per 64-wide contraction step.
static GemmPlan plan_for(int64_t cus, int cfg, int64_t M, int64_t N, int64_t K, double* cost_us, bool allow_split,
                         int force_splits = 0) {
  GemmPlan pl;
  pl.cfg = cfg;
  pl.bm = kCfgs[cfg].bm;
  pl.bn = kCfgs[cfg].bn;
  pl.bk = kCfgs[cfg].bk;
  pl.tiles_m = (int)((M + pl.bm - 1) / pl.bm);
  pl.tiles_n = (int)((N + pl.bn - 1) / pl.bn);
  const int64_t tiles = (int64_t)pl.tiles_m * pl.tiles_n;
  const int64_t ksteps = (K + pl.bk - 1) / pl.bk;
  const int wg_per_cu = pl.bm * pl.bn <= 128 * 128 ? 2 : 1;
  const int64_t slots = cus * wg_per_cu;
  // Split the contraction only when the tiles alone leave most CUs idle (weight
  // gradients: few output tiles, long contraction); never beyond one full round of
  // workgroups, and every slice keeps at least 16 steps so that the fp32 partial
  // traffic stays small.
  // Microseconds of a round of workgroups beside its steps and per 64-wide step (`alone`: of a round with one workgroup per CU at
  // the most, where two of 128x128 share one otherwise), by configuration.  Found over 2300 products of 2 to 16384 rows, 64 to 8192
  // columns and contractions of 64 to 16384, all layouts, odd extents and whole multiples of 8 and 64, shapes of decoders among them,
  // operands from HBM, every tile timed with and without slices; over 1400 others the tile taken is 1.0 per cent slower than the best of
  // those at hand (geometric mean; 0.5 where the contraction is not split), 0.2 to 0.4 with operands of any alignment.
  // With the figures of the 32x32x16 kernels (2: 10 and 1.65, 4: 7 and 1.0, 3: 7 and 1.1, 0: 10 and 2.25, 1: 7 and 1.6, no 8) it
  // is 1.3, 0.9 and 0.6 to 0.7.  A step of 256x128 tiles at 0.78 us, what it is where a contraction is short, took long ones to them:
  // 14976 x 1984 x 12800 643 us on 256x256 tiles and 768 on 256x128, 8192 x 2048 x 12288 319 and 348.
  // Register-staged 256x128 tiles pay where 128x128 tiles are more than one and less than two per CU: 1563 x 2665 x 5116 106 us on
  // these and 82, but with fewer than one per CU 1509 x 105 x 7035 119 and 179.
  static const struct { double fixed, per_step, alone; } rates[] = {
      {13.9, 1.93, 1.93}, {5.1, 1.47, 1.25}, {10.8, 1.55, 1.55}, {5.8, 1.09, 1.09}, {7.3, 0.88, 0.88},
      {7.3, 0.88, 0.88},  {5.8, 1.09, 1.09}, {5.8, 1.09, 1.09},  {8.7, 1.31, 1.31}};
  static_assert(sizeof(rates) / sizeof(rates[0]) == sizeof(kCfgs) / sizeof(kCfgs[0]), "rates for each configuration");
  auto cost_of = [&](int64_t nsplit, int64_t steps) {
    const int64_t wgs = tiles * nsplit, rounds = (wgs + slots - 1) / slots;
    double c = (double)rounds * (rates[cfg].fixed + rates[cfg].per_step * (double)steps);
    if (wgs - (rounds - 1) * slots <= cus) c -= (rates[cfg].per_step - rates[cfg].alone) * (double)steps;
    if (nsplit > 1) c += 3.0 + (nsplit + 0.5) * (double)M * (double)N * 4.0 / 5.0e6;
    return c;
  };
  int64_t splits = 1;
  if (tiles <= slots / 2) {
    splits = slots / tiles;
    const int64_t max_by_k = ksteps / 16 > 0 ? ksteps / 16 : 1;
    if (splits > max_by_k) splits = max_by_k;
    if (splits > 16) splits = 16;
  }
  // A long contraction whose tiles leave part of a round idle (0.75 of a round: the LM-head input gradient
  // of a narrow model) may be cheaper in more, shorter slices that fill whole rounds: by the cost model,
  // among slice counts that keep 16 steps per slice, and only when it wins by a tenth.
  if (allow_split && force_splits <= 0 && tiles % slots != 0 && ksteps >= 256) {
    double best = cost_of(splits, (ksteps + splits - 1) / splits) * 0.9;
    for (int64_t sp = 2; sp <= 16 && ksteps / sp >= 16; ++sp) {
      const double c = cost_of(sp, (ksteps + sp - 1) / sp);
      if (c < best) { best = c; splits = sp; }
    }
  }
  if (force_splits > 0) splits = force_splits;
  if (!allow_split) splits = 1;
  if (splits > ksteps) splits = ksteps > 0 ? ksteps : 1;
  const int64_t steps_per = (ksteps + splits - 1) / splits;
  pl.k_per_split = (int)(steps_per * pl.bk);
  pl.splits = (int)((ksteps + steps_per - 1) / steps_per);
  if (pl.splits < 1) pl.splits = 1;
  if (cost_us) *cost_us = cost_of(pl.splits, steps_per);
  return pl;
}

// Time (microseconds) of a direct-to-LDS launch that leaves CUs or their second workgroup idle, where the cost above --
// made for whole rounds -- is 1.3 to 2 times too high: a fixed part plus a time per 64-wide step that rises with the
// workgroups per CU (`fill`), since operands come faster and the clock is higher while few CUs work.  Fits to the products above
// that leave CUs idle.  Over 300 others (16 to 8192 rows and columns, contractions of 64 to 8192, all layouts) the tile taken has 1.47 times
// the speed of the large one (geometric mean) and is 0.6 per cent slower than the best of the five (1.5 with the fit named below).  The
// few that are slower, by up to a fifth, are long contractions on just over one workgroup per CU (192 x 1536 x 6144 in six slices 18.4 us
// on 64x64 and 21.9 on 128x64 tiles), where two of a CU take longer than `fill` of them would; counted as two they would cost others more.
// A first fit to these kernels (2.8 and 0.26 for 64x64 tiles, 2.6 and 0.36 for 128x64), to operands that lay in the caches, took products of
// a step or two and products of 256x128 tiles to 128x64: 40 x 1536 x 64 2.8 us on 64x64 and 3.6, 7296 x 560 x 832 13.7 on 256x128 and 17.1.
static double part_round_us(int64_t cus, const GemmPlan& pl, int64_t M, int64_t N) {
  const double steps = (double)(pl.k_per_split / pl.bk);
  const double fill = (double)((int64_t)pl.tiles_m * pl.tiles_n * pl.splits) / (double)cus;
  auto rise = [](double x, double from, double to) { return x <= from ? 0.0 : x >= to ? 1.0 : (x - from) / (to - from); };
  const double more = std::max(0.0, fill - 1);  // further workgroups of a CU: their start and write-out
  double c = 0;
  switch (pl.cfg) {
    case 2: c = 5.14 + steps * (0.82 + 0.71 * rise(fill, 0.35, 0.84)); break;
    case 3: c = 3.38 + steps * (0.717 + 0.407 * rise(fill, 0.654, 2.19)); break;
    case 4: c = 4.04 + steps * (0.588 + 0.36 * rise(fill, 0.16, 1.05)); break;
    case 6: c = 2.59 + more * 0.6 + steps * std::max(0.277 + 0.05 * rise(fill, 0.5, 1), 0.306 * fill); break;
    case 7: c = 2.84 + more * 0.7 + steps * std::max(0.322 + 0.138 * rise(fill, 0.5, 1), 0.378 * fill); break;
  }
  if (pl.splits > 1) c += 3.0 + (pl.splits + 0.5) * (double)M * (double)N * 4.0 / 5.0e6;
  return c;
}

static GemmPlan make_plan(int64_t cus, int64_t M, int64_t N, int64_t K, bool vec, bool allow_split = true,
                          double* cost_us = nullptr, const GemmForce& force = kNoForce) {
  const bool dma = vec && K % 64 == 0;
  if (cost_us) *cost_us = -1.0;  // stays negative when the configuration is forced
  if (force.cfg >= 0 && force.cfg < kNumCfgs) {
    int cfg = force.cfg;
    if (kCfgs[cfg].dma && !dma) cfg = kCfgs[cfg].bm * kCfgs[cfg].bn >= 256 * 256 ? 0 : 1;  // register-staged twin
    return plan_for(cus, cfg, M, N, K, nullptr, allow_split, force.splits);
  }
  // candidates: 256x256, 256x128 and 128x128 tiles, direct-to-LDS kernels when their
  // preconditions hold, the register-staged twins otherwise
  const int cand_dma[3] = {2, 4, 3};
  const int cand_reg[3] = {0, 8, 1};
  const int* cand = dma ? cand_dma : cand_reg;
  GemmPlan best = plan_for(cus, cand[0], M, N, K, nullptr, allow_split, force.splits);
  double best_cost = 1e30;
  for (int i = 0; i < 3; ++i) {
    double c;
    const GemmPlan pl = plan_for(cus, cand[i], M, N, K, &c, allow_split, force.splits);
    if (c < best_cost) { best_cost = c; best = pl; }
  }
  // Tiles that do not fill one round of workgroups: smaller ones occupy more CUs.  A 256x128 tile's step takes 0.64 us on
  // an idle chip, a 64x64 one's 0.27, and start and write-out shrink with the tile: 128 x 1024 x 1024 14.4 -> 6.9 us,
  // 960 x 768 x 768 12.1 -> 6.3, 2048 x 1024 x 1024 15.1 -> 9.5.  Beyond one round the larger tiles are the better ones
  // throughout (2048 x 4096 x 1024: 21 against 29 us).  The slices of the contraction stay those of the larger tile: the
  // same sums in the same order, whatever the tile.  The cost handed back stays the larger tile's: the cuts below compare it
  // with that of whole rounds, and the two scales are not comparable (mixed, 247 of 400 000 products were cut otherwise: 1920 x
  // 8512 x 2304 79 us for 86 but 3968 x 4160 x 512 25.2 for 24.0 and 384 x 35840 x 2048 83.9 for 80.5, 16 of them with other
  // slices and so with sums in another order).
  const int64_t wgs = (int64_t)best.tiles_m * best.tiles_n * best.splits;
  if (dma && wgs <= cus * (best.cfg == 3 ? 2 : 1)) {
    const GemmPlan best_large = best;
    double best_us = 0.95 * part_round_us(cus, best, M, N);
    for (int cfg : {6, 7}) {
      const GemmPlan pl = plan_for(cus, cfg, M, N, K, nullptr, allow_split, best_large.splits);
      const double us = part_round_us(cus, pl, M, N);
      if (us < best_us) { best_us = us; best = pl; }
    }
  }
  if (cost_us) *cost_us = best_cost;
  return best;
}

// Diagnostic: GEMM kernel launches since the library was loaded (reduce passes not counted).
static std::atomic<int64_t> g_gemm_launches{0};

template <typename K>
static void allow_big_lds(K kernel, int bytes) {
  if (bytes > 64 * 1024)
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
}

template <typename K>
static int launch_tiles(hipStream_t st, K kernel, int threads, int lds, const GemmParams& p) {
  const unsigned grid = (unsigned)(p.tiles_m * p.tiles_n * p.splits);
  kernel<<<dim3(grid), dim3(threads), lds, st>>>(p);
  TF_CHECK_LAUNCH();
  g_gemm_launches.fetch_add(1, std::memory_order_relaxed);
  return TF_OK;
}

template <typename T, int BM, int BN, int BK, int WM, int WN, int WPE, bool AK, bool BKM>
static int launch_reg(hipStream_t st, const GemmParams& p) {
  constexpr int lds = 2 * (BM + BN) * BK * 2;
  auto kernel = gemm_reg_kernel<T, BM, BN, BK, WM, WN, WPE, AK, BKM>;
  static bool once = (allow_big_lds(kernel, lds), true);
  (void)once;
  return launch_tiles(st, kernel, WM * WN * 64, lds, p);
}

template <typename T, int BM, int BN, int BK, int WM, int WN, int WPE, bool AK, bool BKM, int NS = 2>
static int launch_dma(hipStream_t st, const GemmParams& p) {
  constexpr int lds = NS * (BM + BN) * BK * 2;
  static_assert(lds <= 160 * 1024, "LDS budget");
  auto kernel = gemm_dma_kernel<T, BM, BN, BK, WM, WN, WPE, AK, BKM, NS>;
  static bool once = (allow_big_lds(kernel, lds), true);
  (void)once;
  return launch_tiles(st, kernel, WM * WN * 64, lds, p);
}

// Whatever the plan's tiles: the same slices on 128x128 tiles, whose kernels take rows of any pitch.
template <typename T, bool AK, bool BKM>
static int launch_any_pitch(hipStream_t st, bool dma, const GemmParams& p) {
  GemmParams q = p;
  q.tiles_m = (q.M + 127) / 128;
  q.tiles_n = (q.N + 127) / 128;
  if ((int64_t)q.tiles_m * q.tiles_n * q.splits > 0x7fffffff) return TF_EINVAL;
  if (dma) return launch_tiles(st, gemm_wide_kernel<T, AK, BKM>, 256, 2 * (128 + 128) * 64 * 2, q);
  return launch_reg<T, 128, 128, 64, 2, 2, 2, AK, BKM>(st, q);
}

// The register-staged kernel handles everything (ragged extents, unaligned
// pointers); the direct-to-LDS kernel needs the vector conditions and a
// contraction extent that is a multiple of its BK.
// Leading dimensions up to which a lane's part of an operand address (255 rows and a chunk) fits 32 bits, by half.
constexpr int64_t kMaxPitch = 1 << 22;

constexpr int kStagesNarrow = 3;  // LDS stages of the configurations below 256x256 but 128x128

template <typename T, bool AK, bool BKM>
static int launch_cfg(hipStream_t st, bool vec, const GemmPlan& pl, const GemmParams& p) {
  const bool dma = kCfgs[pl.cfg].dma && vec && p.K % pl.bk == 0;
  if (p.lda > kMaxPitch || p.ldb > kMaxPitch) return launch_any_pitch<T, AK, BKM>(st, dma, p);
  if (dma) {
    switch (pl.cfg) {
      case 2: return launch_dma<T, 256, 256, 64, 2, 4, 2, AK, BKM>(st, p);
      case 3: return launch_dma<T, 128, 128, 64, 2, 2, 2, AK, BKM>(st, p);
      case 4: return launch_dma<T, 256, 128, 64, 4, 2, 2, AK, BKM, kStagesNarrow>(st, p);
      case 5: return launch_dma<T, 128, 256, 64, 2, 4, 2, AK, BKM, kStagesNarrow>(st, p);
      case 6: return launch_dma<T, 64, 64, 64, 2, 2, 2, AK, BKM, kStagesNarrow>(st, p);
      case 7: return launch_dma<T, 128, 64, 64, 4, 1, 2, AK, BKM, kStagesNarrow>(st, p);
    }
  }
  if (pl.bm == 256 && pl.bn == 256) return launch_reg<T, 256, 256, 64, 2, 4, 2, AK, BKM>(st, p);
  if (pl.bm == 256 && pl.bn == 128) return launch_reg<T, 256, 128, 64, 4, 2, 2, AK, BKM>(st, p);
  if (pl.bm == 128 && pl.bn == 128) return launch_reg<T, 128, 128, 64, 2, 2, 2, AK, BKM>(st, p);
  return TF_EINVAL;
}

// Second pass of a split contraction (no-op when the contraction was not split).
template <typename T>
static int launch_reduce(hipStream_t st, const GemmParams& p) {
  if (p.splits <= 1) return TF_OK;
  const int64_t total = (int64_t)p.M * p.N;
  const bool c16 = (reinterpret_cast<uintptr_t>(p.C) & 15) == 0;
  const bool rows = c16 && p.N % 4 == 0 && p.ldc % 4 == 0 && p.chunk_n % 4 == 0 && p.chunk_skip % 4 == 0;
  const bool flat = c16 && !p.bias && p.ldc == p.N && p.chunk_n == p.N;
  int64_t blocks = ((rows || flat ? total / 4 : total) + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  if (blocks < 1) blocks = 1;
  const dim3 g((unsigned)blocks), b(256);
#define REDUCE(TO, MODE) \
  gemm_reduce<T, TO, MODE><<<g, b, 0, st>>>(p.M, p.N, p.splits, p.partial, p.bias, p.bias_f32, p.relu, (TO*)p.C, p.ldc, p.chunk_n, \
                                            p.chunk_skip, p.alpha)
#define REDUCE_MODE(TO) \
  do { if (rows) REDUCE(TO, kReduceRows); else if (flat) REDUCE(TO, kReduceFlat); else REDUCE(TO, kReduceAny); } while (0)
  if (p.out_f32) REDUCE_MODE(float);
  else REDUCE_MODE(T);
#undef REDUCE_MODE
#undef REDUCE
  TF_CHECK_LAUNCH();
  return TF_OK;
}

template <typename T>
static int gemm_dispatch(hipStream_t st, int la, int lb, bool vec, const GemmPlan& pl, const GemmParams& p) {
  const bool ak = la == TF_OP_KMAJOR, bk = lb == TF_OP_KMAJOR;
  int rc;
#define GO(AK, BKM) rc = launch_cfg<T, AK, BKM>(st, vec, pl, p)
  if (ak && bk) GO(true, true);
  else if (ak && !bk) GO(true, false);
  else if (!ak && bk) GO(false, true);
  else GO(false, false);
#undef GO
  if (rc != TF_OK) return rc;
  return launch_reduce<T>(st, p);
}

// One launch for a group of weight-gradient style products (both operands contraction-strided),
// 256x256 tiles, direct-to-LDS kernel; then one reduce pass per problem.
template <typename T>
static int gemm_group_dispatch(hipStream_t st, const GemmGroup& g) {
  constexpr int lds = 2 * (256 + 256) * 64 * 2;
  auto kernel = gemm_dma_group_kernel<T, 256, 256, 64, 2, 4, 2, false, false>;
  static bool once = (allow_big_lds(kernel, lds), true);
  (void)once;
  kernel<<<dim3((unsigned)g.first[g.count]), dim3(512), lds, st>>>(g);
  TF_CHECK_LAUNCH();
  g_gemm_launches.fetch_add(1, std::memory_order_relaxed);
  // second pass of the split contractions: all products of the group in one launch
  ReduceBatch rb = {};
  bool any = false, v4 = true;
  int64_t most = 0;
  for (int i = 0; i < g.count; ++i) {
    const GemmParams& p = g.p[i];
    rb.it[i] = {p.partial, p.C, p.ldc, p.chunk_skip, p.M, p.N, p.splits, p.chunk_n};
    if (p.splits <= 1) continue;
    any = true;
    v4 = v4 && p.N % 4 == 0 && p.ldc % 4 == 0 && p.chunk_n % 4 == 0 && p.chunk_skip % 4 == 0 &&
         (reinterpret_cast<uintptr_t>(p.C) & 15) == 0;
    const int64_t total = (int64_t)p.M * p.N;
    if (total > most) most = total;
  }
  if (!any) return TF_OK;
  int64_t blocks = ((v4 ? most / 4 : most) + 255) / 256;
  blocks = blocks > 4096 ? 4096 : (blocks < 1 ? 1 : blocks);
  const dim3 grid((unsigned)blocks, (unsigned)g.count), block(256);
  const bool f32 = g.p[0].out_f32 != 0;
  if (f32) { if (v4) gemm_reduce_group<float, true><<<grid, block, 0, st>>>(rb); else gemm_reduce_group<float, false><<<grid, block, 0, st>>>(rb); }
  else { if (v4) gemm_reduce_group<T, true><<<grid, block, 0, st>>>(rb); else gemm_reduce_group<T, false><<<grid, block, 0, st>>>(rb); }
  TF_CHECK_LAUNCH();
  return TF_OK;
}

}  // namespace tfa

using namespace tfa;

extern "C" int64_t tf_diag_gemm_launch_count(void) { return g_gemm_launches.load(std::memory_order_relaxed); }

// Tile columns (of 256x256 tiles) per whole number of rounds of workgroups, one per CU.
static int64_t round_unit(int64_t tiles_m, int64_t cus) {
  int64_t a = tiles_m, b = cus;
  while (b) { const int64_t t = a % b; a = b; b = t; }
  return cus / a;
}

// A product whose 256x256 tiles fill a whole number of rounds of workgroups plus a small
// remainder is cut in two along N: the columns that make whole rounds, and a narrow tail
// that runs as a split contraction on the otherwise idle CUs instead of a nearly empty last
// round (LM-head weight gradient: 4 x 197 tiles = 3 rounds + 20 tiles).  Returns the number
// of tail columns, 0 for no cut.
static int64_t tail_columns(int64_t cus, int64_t M, int64_t N, int64_t K, const GemmPlan& pl) {
  if (K < 32 * 64) return 0;
  const int64_t tiles_m = (M + 255) / 256, tiles_n = (N + 255) / 256;
  const int64_t unit = round_unit(tiles_m, cus);
  const int64_t tn1 = (tiles_n / unit) * unit;
  if (tn1 <= 0 || tn1 * 256 >= N) return 0;
  if (pl.cfg == 2 && pl.splits == 1) {
    const int64_t tiles = tiles_m * tiles_n;
    const int64_t rem = tiles % cus;
    if (tiles > cus && rem != 0 && rem <= cus / 4) return N - tn1 * 256;
  }
  return 0;
}

// The same cut for a short contraction, by the cost model: whole rounds of 256x256 tiles, then
// the remaining columns as a product of their own with whatever tiling suits them, when the two
// together are cheaper than the best single launch (q/k/v projection 8192 x 3072 x 1024: one
// round of 256x256 tiles + 1024 columns of 128x128 tiles, 0.2 ms per training step less than
// three rounds of 128x128 tiles).
static int64_t round_cut_columns(int64_t cus, int64_t M, int64_t N, int64_t K, bool vec, bool allow_split, double uncut) {
  if (!(vec && K % 64 == 0) || uncut < 0) return 0;
  double whole, rest;
  const int64_t tiles_m = (M + 255) / 256, tiles_n = (N + 255) / 256;
  if (tiles_m * tiles_n <= cus) return 0;
  const int64_t unit = round_unit(tiles_m, cus);
  const int64_t tn1 = (tiles_n / unit) * unit;
  if (tn1 <= 0 || tn1 * 256 >= N) return 0;
  (void)plan_for(cus, 2, M, tn1 * 256, K, &whole, false);
  (void)make_plan(cus, M, N - tn1 * 256, K, vec, allow_split, &rest);
  if (rest < 0) return 0;
  return whole + rest + 3.0 < uncut ? N - tn1 * 256 : 0;
}

// How a product is run: cut along N (`tail` columns, 0 = uncut) or as `plan`.  Cut along N only where the result is one
// matrix and no mask rides on it; split only where neither a mask nor sign bits do.
enum RouteKind { kRoutePlain, kRouteSigns, kRouteMask, kRouteChunked };
struct Route {
  GemmPlan plan;
  int64_t tail;
};
static Route find_route(int64_t cus, int64_t M, int64_t N, int64_t K, bool vec, RouteKind kind) {
  const bool split = kind == kRoutePlain || kind == kRouteChunked;
  double uncut;
  Route r = {make_plan(cus, M, N, K, vec, split, &uncut), 0};
  if (kind == kRoutePlain) r.tail = tail_columns(cus, M, N, K, r.plan);
  if (r.tail == 0 && (kind == kRoutePlain || kind == kRouteSigns)) r.tail = round_cut_columns(cus, M, N, K, vec, split, uncut);
  if (r.tail > 0 && kind == kRouteSigns) {
    // the bits of both parts have to be served (a cut at a multiple of 256 columns keeps whole bytes and the 16-byte
    // pieces of the bit rows)
    const GemmPlan p1 = make_plan(cus, M, N - r.tail, K, vec, false), p2 = make_plan(cus, M, r.tail, K, vec, false);
    if (!(kCfgs[p1.cfg].dma && kCfgs[p2.cfg].dma && K % p1.bk == 0 && K % p2.bk == 0)) r.tail = 0;
  }
  return r;
}
// The route follows from these figures alone and takes 1 to 4 us to find -- as long as a launch -- several times per
// product (workspace, both alignments, parts of a cut): each thread keeps the last ones it found, 256 at most.
static Route route(int64_t M, int64_t N, int64_t K, bool vec, RouteKind kind) {
  struct Entry {
    int64_t M, N, K, tag;
    Route r;
  };
  static thread_local Entry cache[256];  // all zero at first: no product has M = 0
  const int64_t cus = device_shape().cus, tag = cus * 8 + kind * 2 + (vec ? 1 : 0);
  const uint64_t h = ((uint64_t)M * 0x9e3779b97f4a7c15u + (uint64_t)N * 0xc2b2ae3d27d4eb4fu + (uint64_t)K * 0x165667b19e3779f9u + (uint64_t)tag) *
                     0x9e3779b97f4a7c15u;
  Entry& e = cache[h >> 56];
  if (e.M != M || e.N != N || e.K != K || e.tag != tag) e = {M, N, K, tag, find_route(cus, M, N, K, vec, kind)};
  return e.r;
}

static int64_t plan_need(const GemmPlan& pl, int64_t M, int64_t N) {
  return pl.splits > 1 ? (int64_t)pl.splits * M * N * (int64_t)sizeof(float) : 0;
}

extern "C" int64_t tf_gemm_workspace_bytes(int layout_a, int layout_b, int64_t M, int64_t N, int64_t K) {
  (void)layout_a;
  (void)layout_b;
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  // the caller's alignment is unknown here: cover both kernel families
  int64_t need = 0;
  for (int vec = 0; vec < 2; ++vec) {
    const Route r = route(M, N, K, vec != 0, kRoutePlain);
    need = std::max(need, plan_need(r.plan, M, N));
    if (r.tail > 0)
      for (int64_t n : {N - r.tail, r.tail}) need = std::max(need, plan_need(route(M, n, K, vec != 0, kRouteChunked).plan, M, n));
  }
  return need;
}

extern "C" int tf_gemm(void* stream, int dtype, int layout_a, int layout_b, int64_t M, int64_t N, int64_t K,
                       const void* A, int64_t lda, const void* B, int64_t ldb, void* C, int64_t ldc,
                       const void* bias, int relu, void* workspace, int64_t workspace_bytes) {
  return tf_gemm_out(stream, dtype, dtype, layout_a, layout_b, M, N, K, A, lda, B, ldb, C, ldc, bias, relu, nullptr, 0,
                     workspace, workspace_bytes);
}

extern "C" int tf_gemm_out(void* stream, int dtype, int out_dtype, int layout_a, int layout_b, int64_t M, int64_t N,
                           int64_t K, const void* A, int64_t lda, const void* B, int64_t ldb, void* C, int64_t ldc,
                           const void* bias, int relu, const void* mask_act, int64_t ld_mask, void* workspace,
                           int64_t workspace_bytes) {
  return tf_gemm_out_chunked(stream, dtype, out_dtype, layout_a, layout_b, M, N, K, A, lda, B, ldb, C, ldc, 0, 0, bias,
                             relu, mask_act, ld_mask, workspace, workspace_bytes);
}

static int gemm_entry(void* stream, int dtype, int out_dtype, int layout_a, int layout_b, int64_t M, int64_t N,
                      int64_t K, const void* A, int64_t lda, const void* B, int64_t ldb, void* C, int64_t ldc,
                      int64_t chunk_n, int64_t chunk_stride, const void* bias, int relu, const void* mask_act,
                      int64_t ld_mask, void* workspace, int64_t workspace_bytes, void* sign_out, const void* sign_in,
                      int64_t ld_sign, const GemmForce& force = kNoForce, const float* alpha = nullptr,
                      bool bias_f32 = false, bool like_signs = false) {
  if (!A || !B || !C) return TF_EINVAL;
  if (bias_f32 && (reinterpret_cast<uintptr_t>(bias) & 3)) return TF_EALIGN;
  if (alpha && (reinterpret_cast<uintptr_t>(alpha) & 3)) return TF_EALIGN;
  const bool signs = sign_out || sign_in || like_signs;  // like_signs: the launches of a product with sign bits, none written
  if (signs) {
    if ((sign_out && sign_in) || mask_act || N % 8 != 0 || ld_sign < N / 8 || (chunk_n != 0 && chunk_n < N)) return TF_EINVAL;
    if (sign_out && (!relu || out_dtype != dtype)) return TF_EINVAL;
    if (sign_in && (bias || relu)) return TF_EINVAL;
  }
  if (chunk_n < 0 || chunk_stride < 0) return TF_EINVAL;
  if (mask_act && (bias || relu || ld_mask < N)) return TF_EINVAL;
  if (out_dtype != dtype && out_dtype != TF_F32) return TF_EDTYPE;
  if (M <= 0 || N <= 0 || K <= 0 || M > 0x7fffff00 || N > 0x7fffff00 || K > 0x7fffff00) return TF_EINVAL;
  if (chunk_n == 0 || chunk_n >= N) { chunk_n = N; chunk_stride = N; }
  else if (N % chunk_n != 0 || chunk_n % 8 != 0 || chunk_stride % 8 != 0 ||
           chunk_stride < (M - 1) * ldc + chunk_n) return TF_ESHAPE;
  if ((layout_a != TF_OP_KMAJOR && layout_a != TF_OP_KMINOR) || (layout_b != TF_OP_KMAJOR && layout_b != TF_OP_KMINOR))
    return TF_EINVAL;
  if (dtype != TF_F16 && dtype != TF_BF16) return TF_EDTYPE;
  const int64_t a_contig = layout_a == TF_OP_KMAJOR ? K : M;
  const int64_t b_contig = layout_b == TF_OP_KMAJOR ? K : N;
  if (lda < a_contig || ldb < b_contig || ldc < chunk_n) return TF_ESHAPE;
  if ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B) | reinterpret_cast<uintptr_t>(C) |
       reinterpret_cast<uintptr_t>(bias)) & 1)
    return TF_EALIGN;

  const bool vec = aligned16(A) && aligned16(B) && aligned16(C) && (!bias || aligned16(bias)) && a_contig % 8 == 0 &&
                   b_contig % 8 == 0 && lda % 8 == 0 && ldb % 8 == 0 && N % 8 == 0 && ldc % 8 == 0 &&
                   (!mask_act || (aligned16(mask_act) && ld_mask % 8 == 0));
  const bool forced = force.cfg >= 0 || force.splits > 0 || (force.flags & 64);
  Route rt;
  if (forced) rt = {make_plan(device_shape().cus, M, N, K, vec, mask_act == nullptr && !signs, nullptr, force), 0};
  else rt = route(M, N, K, vec, mask_act ? kRouteMask : signs ? kRouteSigns : chunk_n != N ? kRouteChunked : kRoutePlain);
  if (rt.tail > 0) {  // whole rounds first, then the narrow remainder as a split contraction
    const int64_t tail = rt.tail, n1 = N - tail;
    const int64_t osz = out_dtype == TF_F32 ? 4 : 2;
    const char* b2 = (const char*)B + (layout_b == TF_OP_KMAJOR ? n1 * ldb : n1) * 2;
    const void* bias2 = bias ? (const char*)bias + n1 * (bias_f32 ? 4 : 2) : nullptr;
    void* so2 = sign_out ? (char*)sign_out + n1 / 8 : nullptr;
    const void* si2 = sign_in ? (const char*)sign_in + n1 / 8 : nullptr;
    const int rc = gemm_entry(stream, dtype, out_dtype, layout_a, layout_b, M, n1, K, A, lda, B, ldb, C, ldc, 0, 0, bias,
                              relu, nullptr, 0, workspace, workspace_bytes, sign_out, sign_in, ld_sign, force, alpha, bias_f32,
                              like_signs);
    if (rc != TF_OK) return rc;
    return gemm_entry(stream, dtype, out_dtype, layout_a, layout_b, M, tail, K, A, lda, b2, ldb, (char*)C + n1 * osz,
                      ldc, 0, 0, bias2, relu, nullptr, 0, workspace, workspace_bytes, so2, si2, ld_sign, force, alpha,
                      bias_f32, like_signs);
  }
  const GemmPlan pl = rt.plan;
  // the sign bits exist in the write-out of the direct-to-LDS kernels only
  // (TF_ESHAPE, so that a caller can tell "this product is not served, use the activation as mask"
  // from a malformed call)
  if (signs && !(kCfgs[pl.cfg].dma && vec && K % pl.bk == 0 && pl.splits == 1)) return TF_ESHAPE;
  const int64_t need = plan_need(pl, M, N);
  if (need > 0 && (!workspace || workspace_bytes < need)) return TF_EWORKSPACE;
  if (need > 0 && !aligned16(workspace)) return TF_EALIGN;
  if ((int64_t)pl.tiles_m * pl.tiles_n * pl.splits > 0x7fffffff) return TF_EINVAL;

  GemmParams p;
  p.A = A; p.B = B; p.C = C; p.bias = bias; p.partial = (float*)workspace;
  p.M = (int)M; p.N = (int)N; p.K = (int)K;
  p.lda = lda; p.ldb = ldb; p.ldc = ldc;
  p.relu = relu ? 1 : 0;
  p.bias_f32 = bias_f32 ? 1 : 0;
  p.splits = pl.splits; p.k_per_split = pl.k_per_split;
  p.tiles_m = pl.tiles_m; p.tiles_n = pl.tiles_n;
  p.flags = force.flags;
  p.xcds = device_shape().xcds;
  p.out_f32 = out_dtype == TF_F32 ? 1 : 0;
  p.mask = mask_act;
  p.ldmask = ld_mask;
  p.sign_out = sign_out;
  p.sign_in = sign_in;
  p.ldsign = ld_sign;
  p.chunk_n = (int)chunk_n;
  p.chunk_skip = chunk_stride - chunk_n;
  p.alpha = alpha;
  hipStream_t st = (hipStream_t)stream;
  if (dtype == TF_F16) return gemm_dispatch<f16>(st, layout_a, layout_b, vec, pl, p);
  return gemm_dispatch<bf16>(st, layout_a, layout_b, vec, pl, p);
}

extern "C" int tf_gemm_out_chunked(void* stream, int dtype, int out_dtype, int layout_a, int layout_b, int64_t M,
                                   int64_t N, int64_t K, const void* A, int64_t lda, const void* B, int64_t ldb,
                                   void* C, int64_t ldc, int64_t chunk_n, int64_t chunk_stride, const void* bias,
                                   int relu, const void* mask_act, int64_t ld_mask, void* workspace,
                                   int64_t workspace_bytes) {
  return gemm_entry(stream, dtype, out_dtype, layout_a, layout_b, M, N, K, A, lda, B, ldb, C, ldc, chunk_n,
                    chunk_stride, bias, relu, mask_act, ld_mask, workspace, workspace_bytes, nullptr, nullptr, 0);
}

extern "C" int tf_gemm_relu_bits(void* stream, int dtype, int out_dtype, int layout_a, int layout_b, int64_t M,
                                 int64_t N, int64_t K, const void* A, int64_t lda, const void* B, int64_t ldb,
                                 void* C, int64_t ldc, const void* bias, void* bits_out, const void* bits_in,
                                 int64_t ld_bits) {
  if (!bits_out && !bits_in) return TF_EINVAL;
  return gemm_entry(stream, dtype, out_dtype, layout_a, layout_b, M, N, K, A, lda, B, ldb, C, ldc, 0, 0, bias,
                    bits_out ? 1 : 0, nullptr, 0, nullptr, 0, bits_out, bits_in, ld_bits);
}

extern "C" int tf_gemm_relu(void* stream, int dtype, int layout_a, int layout_b, int64_t M, int64_t N, int64_t K, const void* A,
                            int64_t lda, const void* B, int64_t ldb, void* C, int64_t ldc, const void* bias) {
  return gemm_entry(stream, dtype, dtype, layout_a, layout_b, M, N, K, A, lda, B, ldb, C, ldc, 0, 0, bias, 1, nullptr, 0, nullptr, 0,
                    nullptr, nullptr, N / 8, kNoForce, nullptr, false, true);
}

extern "C" int tf_gemm_master_bias(void* stream, int dtype, int layout_a, int layout_b, int64_t M, int64_t N, int64_t K,
                                   const void* A, int64_t lda, const void* B, int64_t ldb, void* C, int64_t ldc,
                                   const float* bias, int relu, void* bits_out, int64_t ld_bits, void* workspace,
                                   int64_t workspace_bytes) {
  if (!bias) return TF_EINVAL;
  return gemm_entry(stream, dtype, dtype, layout_a, layout_b, M, N, K, A, lda, B, ldb, C, ldc, 0, 0, bias, relu, nullptr, 0,
                    workspace, workspace_bytes, bits_out, nullptr, ld_bits, kNoForce, nullptr, true);
}

extern "C" int tf_gemm_scaled(void* stream, int dtype, int out_dtype, int layout_a, int layout_b, int64_t M, int64_t N,
                              int64_t K, const void* A, int64_t lda, const void* B, int64_t ldb, void* C, int64_t ldc,
                              const float* alpha, void* workspace, int64_t workspace_bytes) {
  if (!alpha) return TF_EINVAL;
  return gemm_entry(stream, dtype, out_dtype, layout_a, layout_b, M, N, K, A, lda, B, ldb, C, ldc, 0, 0, nullptr, 0,
                    nullptr, 0, workspace, workspace_bytes, nullptr, nullptr, 0, kNoForce, alpha);
}

extern "C" int tf_gemm_side_by_side(void* stream, int dtype, int64_t M, int64_t each, int count, int64_t K, const void* A,
                                    int64_t lda, const void* const* B, int64_t ldb, void* C, int64_t ldc, void* workspace,
                                    int64_t workspace_bytes) {
  if (!A || !B || !C || M <= 0 || each <= 0 || K <= 0 || count < 1 || count > 3) return TF_EINVAL;
  if (M > 0x7fffff00 || each > 0x7fffff00 / 3 || K > 0x7fffff00) return TF_EINVAL;
  if (dtype != TF_F16 && dtype != TF_BF16) return TF_EDTYPE;
  const int64_t N = each * count;
  bool vec = lda <= kMaxPitch && ldb <= kMaxPitch && aligned16(A) && aligned16(C) && K % 8 == 0 && each % 8 == 0 && lda % 8 == 0 &&
             ldb % 8 == 0 && ldc % 8 == 0;
  for (int i = 0; i < count; ++i) {
    if (!B[i]) return TF_EINVAL;
    vec = vec && aligned16(B[i]);
  }
  if (lda < K || ldb < each || ldc < N || !vec) return TF_ESHAPE;
  const Route rt = route(M, N, K, true, kRoutePlain);
  const GemmPlan& pl = rt.plan;
  if (rt.tail > 0 || !kCfgs[pl.cfg].dma || K % pl.bk != 0 || each % pl.bn != 0) return TF_ESHAPE;
  const int64_t need = plan_need(pl, M, N);
  if (need > 0 && (!workspace || workspace_bytes < need)) return TF_EWORKSPACE;
  if (need > 0 && !aligned16(workspace)) return TF_EALIGN;
  if ((int64_t)pl.tiles_m * pl.tiles_n * pl.splits > 0x7fffffff) return TF_EINVAL;
  GemmParams p = {};
  p.A = A; p.B = B[0]; p.C = C; p.partial = (float*)workspace;
  p.B1 = B[count > 1 ? 1 : 0]; p.B2 = B[count > 2 ? 2 : 0]; p.b_each = (int)each;
  p.M = (int)M; p.N = (int)N; p.K = (int)K;
  p.lda = lda; p.ldb = ldb; p.ldc = ldc;
  p.splits = pl.splits; p.k_per_split = pl.k_per_split;
  p.tiles_m = pl.tiles_m; p.tiles_n = pl.tiles_n;
  p.xcds = device_shape().xcds;
  p.chunk_n = (int)N;
  hipStream_t st = (hipStream_t)stream;
  if (dtype == TF_F16) return gemm_dispatch<f16>(st, TF_OP_KMAJOR, TF_OP_KMINOR, true, pl, p);
  return gemm_dispatch<bf16>(st, TF_OP_KMAJOR, TF_OP_KMINOR, true, pl, p);
}

// Diagnostic twin of tf_gemm_out_chunked: the same call with a tile configuration, a contraction
// split and flag bits imposed on THIS call only (no state is kept).
extern "C" int tf_diag_gemm(void* stream, int cfg, int splits, int flags, int dtype, int out_dtype, int layout_a,
                            int layout_b, int64_t M, int64_t N, int64_t K, const void* A, int64_t lda, const void* B,
                            int64_t ldb, void* C, int64_t ldc, const void* bias, int relu, void* workspace,
                            int64_t workspace_bytes) {
  if (cfg >= kNumCfgs || splits < 0 || (flags & ~(1 | 64))) return TF_EINVAL;
  const GemmForce force = {cfg < 0 ? -1 : cfg, splits, flags};
  return gemm_entry(stream, dtype, out_dtype, layout_a, layout_b, M, N, K, A, lda, B, ldb, C, ldc, 0, 0, bias, relu,
                    nullptr, 0, workspace, workspace_bytes, nullptr, nullptr, 0, force);
}
extern "C" int tf_diag_gemm_relu_bits(void* stream, int cfg, int dtype, int out_dtype, int layout_a, int layout_b, int64_t M,
                                      int64_t N, int64_t K, const void* A, int64_t lda, const void* B, int64_t ldb, void* C,
                                      int64_t ldc, const void* bias, void* bits_out, const void* bits_in, int64_t ld_bits) {
  if (cfg >= kNumCfgs || (!bits_out && !bits_in)) return TF_EINVAL;
  const GemmForce force = {cfg < 0 ? -1 : cfg, 0, 0};
  return gemm_entry(stream, dtype, out_dtype, layout_a, layout_b, M, N, K, A, lda, B, ldb, C, ldc, 0, 0, bias,
                    bits_out ? 1 : 0, nullptr, 0, nullptr, 0, bits_out, bits_in, ld_bits, force);
}
// The launches of a product, in the order in which gemm_entry makes them: rows of {columns, configuration, slices,
// contraction elements per slice} from `at` on.  Returns the rows there are then, -1 where `room` does not hold them.
static int route_launches(int64_t cus, int64_t M, int64_t N, int64_t K, bool vec, RouteKind kind, int64_t (*rows)[4], int at,
                          int room) {
  const Route r = find_route(cus, M, N, K, vec, kind);
  if (r.tail > 0) {
    at = route_launches(cus, M, N - r.tail, K, vec, kind, rows, at, room);
    return at < 0 ? at : route_launches(cus, M, r.tail, K, vec, kind, rows, at, room);
  }
  if (at >= room) return -1;
  const int64_t row[4] = {N, r.plan.cfg, r.plan.splits, r.plan.k_per_split};
  std::copy(row, row + 4, rows[at]);
  return at + 1;
}
extern "C" int tf_diag_gemm_route(int cus, int64_t M, int64_t N, int64_t K, int vec, int kind, int64_t* launches, int room) {
  if (cus < 1 || M <= 0 || N <= 0 || K <= 0 || kind < 0 || kind > kRouteChunked || !launches || room < 1) return TF_EINVAL;
  return route_launches(cus, M, N, K, vec != 0, (RouteKind)kind, reinterpret_cast<int64_t(*)[4]>(launches), 0, room);
}
extern "C" int64_t tf_diag_gemm_workspace_bytes(int cfg, int splits, int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0 || cfg >= kNumCfgs) return 0;
  if (cfg < 0 && splits <= 0) return tf_gemm_workspace_bytes(0, 0, M, N, K);
  const GemmForce force = {cfg < 0 ? -1 : cfg, splits, 0};
  int64_t need = 0;
  for (int vec = 0; vec < 2; ++vec) {
    need = std::max(need, plan_need(make_plan(device_shape().cus, M, N, K, vec != 0, true, nullptr, force), M, N));
  }
  return need;
}

// ---- grouped products -------------------------------------------------------
namespace {

struct GroupPlan {
  bool grouped;   // one launch for all problems (otherwise: one tf_gemm_out_chunked call each)
  int splits;
  int64_t need;   // workspace bytes
  // Tiles that make whole rounds of workgroups plus a remainder: the last `cut_cols` tile columns of problem
  // `cut_problem` (-1: none) become a member of the group of their own whose contraction is cut into
  // `tail_splits` slices, so that the remainder fills one short round of all CUs instead of a whole round of
  // a few (what the N-cut of a single product does for the LM-head weight gradient).
  int cut_problem;
  int cut_cols;
  int tail_splits;
};

bool group_problem_ok(const tf_gemm_problem& q) {
  return q.A && q.B && q.C && q.M > 0 && q.N > 0 && q.K > 0 && q.M <= 0x7fffff00 && q.N <= 0x7fffff00 &&
         q.K <= 0x7fffff00;
}

// Fast-path preconditions of the direct-to-LDS kernel for a (K-minor, K-minor) problem.
bool group_problem_fast(const tf_gemm_problem& q) {
  const int64_t cn = (q.chunk_n <= 0 || q.chunk_n >= q.N) ? q.N : q.chunk_n;
  return q.lda <= kMaxPitch && q.ldb <= kMaxPitch && aligned16(q.A) && aligned16(q.B) && aligned16(q.C) && q.M % 8 == 0 && q.N % 8 == 0 && q.lda % 8 == 0 &&
         q.ldb % 8 == 0 && q.ldc % 8 == 0 && q.K % 64 == 0 && q.lda >= q.M && q.ldb >= q.N && q.ldc >= cn &&
         q.N % cn == 0 && cn % 8 == 0 && (cn == q.N || (q.chunk_stride % 8 == 0 && q.chunk_stride >= (q.M - 1) * q.ldc + cn));
}

GroupPlan plan_group(int la, int lb, int count, const tf_gemm_problem* pr) {
  GroupPlan gp = {false, 1, 0, -1, 0, 1};
  bool fast = count >= 2 && count <= kMaxGroup && la == TF_OP_KMINOR && lb == TF_OP_KMINOR;
  const int64_t cus = device_shape().cus;
  int64_t tiles = 0, min_ksteps = INT64_MAX;
  for (int i = 0; i < count && fast; ++i) {
    fast = group_problem_ok(pr[i]) && group_problem_fast(pr[i]);
    if (!fast) break;
    tiles += ((pr[i].M + 255) / 256) * ((pr[i].N + 255) / 256);
    const int64_t ks = pr[i].K / 64;
    if (ks < min_ksteps) min_ksteps = ks;
  }
  if (fast && tiles < 0x7fffff) {
    // same rule as for a single product: split only when the tiles alone leave most CUs idle,
    // never beyond one round of workgroups, slices of at least 16 steps
    int64_t splits = 1;
    if (tiles <= cus / 2) {
      splits = cus / tiles;
      const int64_t max_by_k = min_ksteps / 16 > 0 ? min_ksteps / 16 : 1;
      if (splits > max_by_k) splits = max_by_k;
      if (splits > 16) splits = 16;
    }
    gp.grouped = true;
    gp.splits = (int)splits;
    if (splits > 1)
      for (int i = 0; i < count; ++i) gp.need += splits * pr[i].M * pr[i].N * (int64_t)sizeof(float);
    // More tiles than CUs and a remainder: look for a cut.  Costs in 64-wide contraction steps of a round of
    // workgroups; the split tail pays its fp32 partials and the reduce pass (about six steps' worth).
    bool same_k = true;
    for (int i = 1; i < count; ++i) same_k = same_k && pr[i].K == pr[0].K;
    if (splits == 1 && tiles > cus && tiles % cus != 0 && same_k && count < kMaxGroup) {
      const int64_t ksteps = pr[0].K / 64;
      const int64_t rounds_whole = tiles / cus;
      int64_t best = ((tiles + cus - 1) / cus) * ksteps * 9 / 10;  // a cut must win by a tenth
      for (int i = 0; i < count; ++i) {
        const bool unchunked = pr[i].chunk_n <= 0 || pr[i].chunk_n >= pr[i].N;
        if (!unchunked || pr[i].M % 256 || pr[i].N % 256) continue;
        const int64_t tm = pr[i].M / 256, tn = pr[i].N / 256;
        for (int64_t c = 1; c < tn; ++c) {
          const int64_t tail = c * tm;
          if (tiles - tail > rounds_whole * cus) continue;  // the whole tiles must fit the whole rounds
          int64_t s = cus / tail;
          if (s > ksteps / 8) s = ksteps / 8;               // slices of at least 8 steps
          if (s > 16) s = 16;
          if (s < 2) break;
          const int64_t per = (ksteps + s - 1) / s;
          const int64_t cost = rounds_whole * ksteps + per + 6;
          if (cost < best) {
            best = cost;
            gp.cut_problem = i;
            gp.cut_cols = (int)c;
            gp.tail_splits = (int)((ksteps + per - 1) / per);
          }
        }
      }
      if (gp.cut_problem >= 0)
        gp.need = (int64_t)gp.tail_splits * pr[gp.cut_problem].M * gp.cut_cols * 256 * (int64_t)sizeof(float);
    }
    return gp;
  }
  for (int i = 0; i < count; ++i) {
    if (!group_problem_ok(pr[i])) continue;
    const int64_t n = tf_gemm_workspace_bytes(la, lb, pr[i].M, pr[i].N, pr[i].K);
    if (n > gp.need) gp.need = n;
  }
  return gp;
}

}  // namespace

extern "C" int64_t tf_gemm_group_workspace_bytes(int layout_a, int layout_b, int count, const tf_gemm_problem* problems) {
  if (!problems || count < 1 || count > kMaxGroup) return 0;
  return plan_group(layout_a, layout_b, count, problems).need;
}

extern "C" int tf_gemm_group(void* stream, int dtype, int out_dtype, int layout_a, int layout_b, int count,
                             const tf_gemm_problem* problems, void* workspace, int64_t workspace_bytes) {
  if (!problems || count < 1 || count > kMaxGroup) return TF_EINVAL;
  if (dtype != TF_F16 && dtype != TF_BF16) return TF_EDTYPE;
  if (out_dtype != dtype && out_dtype != TF_F32) return TF_EDTYPE;
  const GroupPlan gp = plan_group(layout_a, layout_b, count, problems);
  if (gp.need > 0 && (!workspace || workspace_bytes < gp.need)) return TF_EWORKSPACE;
  if (!gp.grouped) {
    for (int i = 0; i < count; ++i) {
      const tf_gemm_problem& q = problems[i];
      const int rc = tf_gemm_out_chunked(stream, dtype, out_dtype, layout_a, layout_b, q.M, q.N, q.K, q.A, q.lda, q.B,
                                         q.ldb, q.C, q.ldc, q.chunk_n, q.chunk_stride, nullptr, 0, nullptr, 0,
                                         workspace, workspace_bytes);
      if (rc != TF_OK) return rc;
    }
    return TF_OK;
  }
  if (gp.need > 0 && !aligned16(workspace)) return TF_EALIGN;
  // members of the launch: the problems as given, except that a cut problem keeps its leading columns and a
  // further member takes its last tile columns with a split contraction
  tf_gemm_problem mem[kMaxGroup];
  int mem_splits[kMaxGroup];
  int members = 0;
  for (int i = 0; i < count; ++i) {
    mem[members] = problems[i];
    mem_splits[members] = gp.splits;
    if (i == gp.cut_problem) mem[members].N -= (int64_t)gp.cut_cols * 256;
    ++members;
  }
  if (gp.cut_problem >= 0) {
    const tf_gemm_problem& q = problems[gp.cut_problem];
    const int64_t n1 = q.N - (int64_t)gp.cut_cols * 256;
    const int64_t osz = out_dtype == TF_F32 ? 4 : 2;
    tf_gemm_problem t = q;
    t.N = q.N - n1;
    t.B = (const char*)q.B + n1 * 2;  // (K, N) row-major: the columns from n1 on
    t.C = (char*)q.C + n1 * osz;
    t.chunk_n = 0;
    t.chunk_stride = 0;
    mem[gp.cut_problem].chunk_n = 0;  // (only unchunked problems are cut)
    mem[gp.cut_problem].chunk_stride = 0;
    mem[members] = t;
    mem_splits[members] = gp.tail_splits;
    ++members;
  }
  GemmGroup g;
  g.count = members;
  g.first[0] = 0;
  char* ws = (char*)workspace;
  for (int i = 0; i < kMaxGroup; ++i) {
    const tf_gemm_problem& q = mem[i < members ? i : 0];
    const int want = mem_splits[i < members ? i : 0];
    GemmParams& p = g.p[i];
    const int64_t cn = (q.chunk_n <= 0 || q.chunk_n >= q.N) ? q.N : q.chunk_n;
    p.A = q.A; p.B = q.B; p.C = q.C; p.bias = nullptr; p.partial = (float*)ws;
    p.M = (int)q.M; p.N = (int)q.N; p.K = (int)q.K;
    p.lda = q.lda; p.ldb = q.ldb; p.ldc = q.ldc;
    p.relu = 0;
    p.bias_f32 = 0;
    p.tiles_m = (int)((q.M + 255) / 256); p.tiles_n = (int)((q.N + 255) / 256);
    const int64_t ksteps = q.K / 64;
    const int64_t steps_per = (ksteps + want - 1) / want;
    p.k_per_split = (int)(steps_per * 64);
    p.splits = (int)((ksteps + steps_per - 1) / steps_per);
    p.flags = gp.cut_problem >= 0 ? 1 : 0;
    p.xcds = device_shape().xcds;
    p.out_f32 = out_dtype == TF_F32 ? 1 : 0;
    p.mask = nullptr; p.ldmask = 0;
    p.sign_out = nullptr; p.sign_in = nullptr; p.ldsign = 0;
    p.chunk_n = (int)cn;
    p.chunk_skip = (cn == q.N ? q.N : q.chunk_stride) - cn;
    p.alpha = nullptr;
    if (i < members) {
      g.first[i + 1] = g.first[i] + p.tiles_m * p.tiles_n * p.splits;
      if (p.splits > 1) ws += (int64_t)want * q.M * q.N * (int64_t)sizeof(float);
    }
  }
  hipStream_t st = (hipStream_t)stream;
  if (dtype == TF_F16) return gemm_group_dispatch<f16>(st, g);
  return gemm_group_dispatch<bf16>(st, g);
}
