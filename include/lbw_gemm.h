/*
 * FP8 GEMM of the FP8 linear layers on gfx950: the products behind lingbot/layers/linear.py:23-29 (rowwise) and
 * :53-73 (MXFP8), with the bias in the epilogue. Conventions of lbw_attn.h: device pointers, int64 sizes, a hipStream_t
 * as void*, an int status; nothing is allocated and nothing synchronises, so every call can be captured in a HIP graph.
 */
#ifndef LBW_GEMM_H
#define LBW_GEMM_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/*
 * out[m][n] = bf16((sum_k x8[m][k] w8[n][k] * w_scale[n]) * x_scale[m] + bias[n]): e4m3 operands with packed rows
 * (x8 [m][k], w8 [n][k]), fp32 sums and scales, each operation in this order rounded to fp32 (as hipBLASLt's rowwise GEMM
 * does), then one rounding to bf16; bias bf16 [n] or null; out [m][n] packed.
 * n and k multiples of 16 (n, k <= 2^22, m <= 2^30); x8, w8 and out 16-byte, the others 4-byte aligned.
 */
int lbw_gemm_fp8_rows(const uint8_t* x8, const float* x_scale, const uint8_t* w8, const float* w_scale,
                      const uint16_t* bias, int64_t m, int64_t n, int64_t k, uint16_t* out, void* stream);

/*
 * The same with one E8M0 scale per 32 values along K of each operand, applied by the matrix instruction:
 * out[m][n] = bf16(trunc_bf16(sum_k (x8 * 2^(ex - 127))[m][k] (w8 * 2^(ew - 127))[n][k]) + bias[n]), the product cut to bf16
 * toward zero before the bias is added, as hipBLASLt's MX GEMM and a separate addition give it. The scales are laid out as
 * [k / 128][rows][4] (lbw_quant_mx_fp8_t writes them so). k a multiple of 128.
 */
int lbw_gemm_fp8_mx(const uint8_t* x8, const uint8_t* x_scale_t, const uint8_t* w8, const uint8_t* w_scale_t,
                    const uint16_t* bias, int64_t m, int64_t n, int64_t k, uint16_t* out, void* stream);

/*
 * lbw_quant_mx_fp8 with its scales written as [cols / 128][rows_pad][4] (cols a multiple of 128): the same bytes in
 * the order lbw_gemm_fp8_mx reads them (which wants them 4-byte aligned).
 */
int lbw_quant_mx_fp8_t(const void* x, int x_is_fp32, int64_t rows, int64_t rows_pad, int64_t cols, int64_t s_row,
                       uint8_t* x8, uint8_t* scale_t, void* stream);

/*
 * lbw_quant_mx_fp8_t, and in the same launch the scales of the other operand, w_scale_e8m0 [w_rows][cols / 32] as
 * lbw_quant_mx_fp8 writes them, reordered into w_scale_t [cols / 128][w_rows][4]. Both 4-byte aligned.
 */
int lbw_quant_mx_fp8_tw(const void* x, int x_is_fp32, int64_t rows, int64_t rows_pad, int64_t cols, int64_t s_row,
                        uint8_t* x8, uint8_t* scale_t, const uint8_t* w_scale_e8m0, int64_t w_rows, uint8_t* w_scale_t,
                        void* stream);

#ifdef __cplusplus
}
#endif

#endif
