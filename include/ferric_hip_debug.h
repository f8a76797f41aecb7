/* Measurement and test aids of libferric_hip.so. They are exported by the same library but are no part of the interface a
 * caller of the quantized-linear path binds (include/ferric_hip.h): none of them has a counterpart in the reference. */
#ifndef FERRIC_HIP_DEBUG_H
#define FERRIC_HIP_DEBUG_H

#include "ferric_hip.h"

#ifdef __cplusplus
extern "C" {
#endif

/* Debugging and tests: on != 0 sends every mat-vec to the shape-complete f32 kernel instead of the streaming one (process-wide,
 * not thread-safe against concurrent launches). No counterpart in the reference. */
int fhip_debug_generic_matvec(int on);

/* Debugging and tests: pins the workgroup tile of the matrix-core GEMM (fhip_gemm_q_bf16, fhip_matmul_q_coop, fhip_ffn_coop)
 * for launches of more than 32 rows: 0, 1, 2 = 64, 128, 256 activation rows x 256 outputs, 3 = 256 x 160, 4, 5 = 128, 64 rows x
 * 128 outputs, 6 = 128 x 160, 7, 8 = 128, 64 x 96, 9 = 64 x 160, 10, 11 = 64, 128 x 64, 12 = 64 x 32; -1 (the default) lets the cost estimate choose. Returns the value before the call. Process-wide, not thread-safe against concurrent
 * launches; fhip_workspace_bytes_coop follows it; run sums (fhip_gemm_q_bf16_run_sums) do not. No counterpart in the reference. */
int fhip_debug_gemm_tile(int tile);

/* Debugging and tests: on == 0 keeps batches of three and more rows off the kernels that multiply on the 4 x 4 x 4 (Q4_K / Q5_K / Q6_K /
 * Q8_0) and 16 x 16 x 32 (the 32-value formats) int8 matrix instructions, so that the mat-vec entry points run them on the dot-product kernel
 * a few rows at a time (they give the same bits; the tests compare them this way). Returns the setting before the call (1 = on, the default).
 * Process-wide, not thread-safe against concurrent launches. No counterpart in the reference. */
int fhip_debug_quad_matvec(int on);

/* Tests: the launches fhip_matmul_q makes of a call with these arguments, one after the other: kernels[i] multiplies rows[i] activation
 * rows. *n: how many there are (the first `cap` are stored). Nothing is launched and no operand is read. No counterpart in the reference. */
#define FHIP_ROUTE_DOT 0         /* the dot-product mat-vec, up to four rows a pass over the weight */
#define FHIP_ROUTE_QUAD 1        /* four rows a pass, 4 x 4 x 4 int8 matrix instruction */
#define FHIP_ROUTE_WIDE 2        /* up to sixteen, 16 x 16 x 32 int8 matrix instruction */
#define FHIP_ROUTE_HELD 3        /* f16 hi / lo: a weight row's whole K inside one workgroup */
#define FHIP_ROUTE_OWN_ROWS 4    /* f16 hi / lo: operand rows made by the workgroups that multiply them */
#define FHIP_ROUTE_PREPARED 5    /* f16 hi / lo: operand rows made by a launch in front */
#define FHIP_ROUTE_CUT 8         /* with the last two: weight rows are cut along K between workgroups */
int fhip_debug_matmul_route(const fhip_weight* w, const float* d_x, size_t rows_x, const float* d_y, int* kernels, size_t* rows, size_t cap, size_t* n);

/* Tests: fhip_matmul_q of one group of rows by the f16 hi / lo kernel named (FHIP_ROUTE_HELD, _OWN_ROWS or _PREPARED), whichever fhip_matmul_q itself would pick; the
 * weight's batch policy says how the sums are made. FHIP_ERR_ARG where that kernel cannot do it. No counterpart in the reference. */
int fhip_debug_matmul_by(const fhip_weight* w, int kernel, const float* d_x, size_t rows_x, float* d_y, void* stream);

/* Measurement aid: one launch that reads nbytes at d_src (16-byte loads over the whole chip) and does nothing else; d_sink is
 * one device word that is practically never written. Timed beside a mat-vec of the same size it gives the time a perfect reader
 * needs for those bytes on this device. No counterpart in the reference (its matvec_roofline example prints bytes / time of the
 * kernel itself, crates/ferric-tensor/examples/matvec_roofline.rs:85-100). */
int fhip_debug_read_probe(const void* d_src, size_t nbytes, uint32_t* d_sink, void* stream);

/* Measurement aid: one launch of matrix instructions only (v_mfma_f32_32x32x16_bf16 on register-resident operands with random
 * mantissas; one workgroup of eight waves per CU, `iters` rounds of four instructions per wave). *flops (may be NULL) receives
 * the floating-point operations of the launch: 2 * 32 * 32 * 16 per instruction. Timed, it is what the matrix pipe gives on this
 * device at the clock its power limit allows, the ceiling the dequant-GEMM is priced against. d_sink is one device float that
 * is practically never written. No counterpart in the reference. */
int fhip_debug_mfma_probe(int iters, float* d_sink, double* flops, void* stream);

/* Measurement aid: `launches` one-row calls of fhip_matmul_q (swiglu != 0: fhip_matmul_q_swiglu) enqueued back to back from
 * native code, launch i on weight ws[i % n_weights], all with the same x and y. A profiler run that cannot replay graphs gets
 * the same steady stream of launches from it that a captured graph gives. No counterpart in the reference. */
int fhip_debug_matmul_q_loop(const fhip_weight* const* ws, size_t n_weights, size_t launches, const float* d_x, int swiglu, float* d_y,
                             void* stream);

#ifdef __cplusplus
}
#endif

#endif /* FERRIC_HIP_DEBUG_H */
