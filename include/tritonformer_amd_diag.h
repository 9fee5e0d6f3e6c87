/*
 * tritonformer_amd_diag.h -- diagnostics, NOT part of the drop-in boundary.
 *
 * Nothing here has a counterpart in the reference (its nearest relative is Triton's
 * autotuner, tritonformer/kernels/gemm.py:15-79, which times tile configurations per
 * shape).  No operator of the package calls these; they exist for the benchmark, for
 * tests that want every tile configuration exercised on small shapes, and for kernel
 * work.  All of them are stateless except the launch counter, which is a relaxed atomic.
 *
 * tf_diag_gemm* live in libtritonformer_amd.so (they need the GEMM's internals);
 * tf_diag_mfma_rate* live in libtritonformer_amd_diag.so, a library of its own.
 */
#ifndef TRITONFORMER_AMD_DIAG_H
#define TRITONFORMER_AMD_DIAG_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* tf_gemm_out (include/tritonformer_amd.h) with the tile choice imposed on THIS call:
 *   cfg    -1 = cost model; 0 / 1 = register-staged 256x256 / 128x128;
 *          2..7 = direct-to-LDS 256x256, 128x128, 256x128, 128x256, 64x64, 128x64; 8 = register-staged 256x128
 *          (a direct-to-LDS cfg falls back to its register-staged twin when the operands
 *          do not meet its preconditions);
 *   splits 0 = chosen by the library, n > 0 = contraction cut into n slices;
 *   flags  bit 0: workgroup ids are not remapped to XCDs; bit 6 (64): the product is never
 *          cut along N into whole rounds + tail.  Other bits are refused.
 * Results are those of tf_gemm_out up to the fp32 summation order of a split contraction.
 * workspace: tf_diag_gemm_workspace_bytes(cfg, splits, M, N, K) bytes. */
int tf_diag_gemm(void* stream, int cfg, int splits, int flags, int dtype, int out_dtype,
                 int layout_a, int layout_b, int64_t M, int64_t N, int64_t K,
                 const void* A, int64_t lda, const void* B, int64_t ldb, void* C, int64_t ldc,
                 const void* bias, int relu, void* workspace, int64_t workspace_bytes);
/* tf_gemm_relu_bits with the tile choice imposed in the same way. */
int tf_diag_gemm_relu_bits(void* stream, int cfg, int dtype, int out_dtype, int layout_a, int layout_b,
                           int64_t M, int64_t N, int64_t K,
                           const void* A, int64_t lda, const void* B, int64_t ldb, void* C, int64_t ldc,
                           const void* bias, void* bits_out, const void* bits_in, int64_t ld_bits);
int64_t tf_diag_gemm_workspace_bytes(int cfg, int splits, int64_t M, int64_t N, int64_t K);

/* The launches that a product becomes on a device of `cus` compute units; nothing is launched and no device is needed.
 *   vec   1: the preconditions of the direct-to-LDS kernels other than K % 64 == 0 hold;
 *   kind  0 = tf_gemm, tf_gemm_out, tf_gemm_scaled; 1 = tf_gemm_relu_bits; 2 = with mask_act;
 *         3 = column blocks (tf_gemm_out_chunked with 0 < chunk_n < N).
 * Each launch is a row of four in `launches` (HOST memory, `room` rows): columns, configuration (as cfg above),
 * slices of the contraction, elements of the contraction per slice.  Returns their number. */
int tf_diag_gemm_route(int cus, int64_t M, int64_t N, int64_t K, int vec, int kind, int64_t* launches, int room);

/* GEMM kernels launched by libtritonformer_amd.so since it was loaded (the reduce passes of
 * split contractions are not counted; one tf_gemm* call may launch two kernels when the
 * product is cut along N).  bench.py divides its event times by the difference of two reads. */
int64_t tf_diag_gemm_launch_count(void);

/* The MFMA instruction stream of the 256x256x64 GEMM step alone: `workgroups` workgroups of 8
 * waves, no memory traffic, `iters` steps each, operands taken once from `operands`
 * (8*6*64*8 = 24576 elements of `dtype`, device memory); `sink`: workgroups*512 floats.  Time
 * the call and divide tf_diag_mfma_rate_flops(iters, workgroups) by it: the sustained rate
 * depends on the operand values (the clock drops under the switching activity of random data). */
int tf_diag_mfma_rate(void* stream, int dtype, const void* operands, int iters, int workgroups,
                      float* sink);
int64_t tf_diag_mfma_rate_flops(int iters, int workgroups);

#ifdef __cplusplus
}
#endif
#endif /* TRITONFORMER_AMD_DIAG_H */
