/*
 * tk_attention_images.h — softmax(scale Q K^T) V of an encoder layer in one kernel, on the exact fp32 MFMA: the bits of the three launches
 * (Q K^T, softmax_rows, P V; csrc/common/tk_whisper_graph.h: attention) without their score matrix in HBM.
 * Q and K are operand images over all rows of the batch (csrc/nn/tk_gemm_tiled.h), V is row-major, the output is the operand image of the
 * layer behind it.  Heads of 64.
 */
#ifndef TK_ATTENTION_IMAGES_H
#define TK_ATTENTION_IMAGES_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#define TK_AIM_MAX_KEYS 1536 /* a wave holds a quarter of 16 rows' scores in registers: 4 per tile of 16 keys */

static inline bool tk_attention_images_fits(int Tq, int Tk, int d, int nh) {
    return Tq >= 1 && Tk >= 1 && Tk <= TK_AIM_MAX_KEYS && nh >= 1 && d == nh * 64;
}
/* q_img [B Tq][d], k_img [B Tk][d], out_img [B Tq][d]: images; v [B Tk][d] rows.  false (nothing launched): sizes it does not take */
bool tk_launch_attention_images(const float* q_img, const float* k_img, const float* v, float* out_img, int B, int nh, int Tq, int Tk, int d, hipStream_t s);

#endif
