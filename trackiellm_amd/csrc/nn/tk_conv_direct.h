/*
 * tk_conv_direct.h — a convolution whose input patch lies in the LDS: the detector's layers on the exact fp32 MFMA chain.
 *
 * A workgroup takes a tile of output pixels of one image and 16 output channels a wave.  The input pixels under the tile, halo included, are loaded
 * once, all channels, in the order in which the MFMA wants them; then every tap of every 16-channel group is an LDS read at a fixed distance, so that the whole
 * k chain runs without a barrier and without decoding an address per value.  Per output the arithmetic is that of the GEMM over the column matrix
 * (tk_gemm_desc.h): one fma chain over k = (ky kw + kx) C + c ascending from zero, padding taken as zero, v = act(acc + bias) + residual: the same bits.
 *
 * Weights are laid out once: per 16 output channels and 16 k one piece of 64 lanes x 4 values, lane (n = l % 16, g = l / 16) holding k = 16 j + 4 t + g,
 * t = 0 .. 3; channels beyond N are zero.
 */
#ifndef TK_CONV_DIRECT_H
#define TK_CONV_DIRECT_H

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

struct TkConvSource {
    const float* p; /* NHWC */
    int ld;         /* floats between pixels */
    int shift;      /* 1: the map has half the height and width and is read as its 2 x nearest upsampling */
};

struct TkConvDirect {
    TkConvSource src[2]; /* channels [0, c_split) come from src[0], the rest from src[1]; c_split == C: one source */
    int c_split;
    int B, H, W, C;      /* input as the convolution sees it */
    int k, stride, pad;
    int Ho, Wo, N;
    const float* w;      /* tk_launch_conv_weights */
    const float* bias;   /* [N] */
    const float* residual; /* [B][Ho][Wo] of pitch ldr, added behind the activation; or null */
    int ldr;
    float* y;            /* [B][Ho][Wo] of pitch ldy */
    int ldy;
    int act;             /* TK_ACT_NONE or TK_ACT_SILU */
};

/* how a launch is cut; tk_conv_direct_plan() */
struct TkConvPlan {
    int mt;      /* 16-pixel tiles a wave: 1, 2 or 4 */
    int wm, wn;  /* waves of a workgroup along pixels and along channels */
    int th, tw;  /* output pixels of a tile */
};

/* 3 x 3 or 1 x 1, stride 1 or 2, channels (and the split) a multiple of 16, pitches of 4, bases 16-byte aligned */
bool tk_conv_direct_takes(const TkConvDirect& c);
/* the quickest cut by the costs beside it; false: no patch of this layer fits the LDS */
bool tk_conv_direct_plan(const TkConvDirect& c, TkConvPlan* plan);
/* whether a cut is one that tk_launch_conv_direct can launch for these operands */
bool tk_conv_plan_ok(const TkConvDirect& c, const TkConvPlan& plan);
bool tk_launch_conv_direct(const TkConvDirect& c, const TkConvPlan& plan, hipStream_t s);

/* up to TK_CONV_SET convolutions of one batch size that do not depend on each other, in one launch (cuts with the same tiles a wave and number of waves) */
enum { TK_CONV_SET = 6 };
bool tk_conv_direct_plan_set(const TkConvDirect* c, int n, TkConvPlan* plans);
bool tk_launch_conv_direct_set(const TkConvDirect* c, const TkConvPlan* plans, int n, hipStream_t s);

/* [N][K] row-major weights (device) -> pieces; K = k k C, a multiple of 16 */
size_t tk_conv_weight_floats(int N, int K);
void tk_launch_conv_weights(const float* w, int N, int K, float* pieces, hipStream_t s);
/* opts the kernels into their LDS on the calling thread's current device; idempotent, thread-safe */
bool tk_conv_direct_prepare_device();

#endif
