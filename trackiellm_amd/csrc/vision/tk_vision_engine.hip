#include "tk_vision_engine.h"
#include "tk_onnx_weights.h"

#include <stdio.h>
#include <string.h>

#include <algorithm>

#include "../nn/tk_nn_kernels.h"

/* Every stream of the library keeps the default priority: work on streams of different priorities has been seen to hang. */
static inline hipError_t tk_create_perception_stream(hipStream_t* s) { return hipStreamCreateWithFlags(s, hipStreamNonBlocking); }

#define HIPQ(expr)                                                                              \
    do {                                                                                        \
        hipError_t e__ = (expr);                                                                \
        if (e__ != hipSuccess) {                                                                \
            char b__[256];                                                                      \
            snprintf(b__, sizeof b__, "%s failed: %s (%s:%d)", #expr, hipGetErrorString(e__), __FILE__, __LINE__); \
            error = b__;                                                                        \
            return false;                                                                       \
        }                                                                                       \
    } while (0)

/* ------------------------------------------------------------------------------------------
 * pre-processing: the reference CPU formula, op for op (scalar branch):
 *   ratio = (orig - 1) / target ; g = ratio * o ; i = (int)g ; d = g - i
 *   v = p1*(1-dx)*(1-dy) + p2*dx*(1-dy) + p3*(1-dx)*dy + p4*dx*dy      (left to right)
 *   out = (v / 255 - mean) / std
 * compiled with -ffp-contract=off; bit-identical to the compiled reference object (tests).
 * One thread per output pixel, all three channels; u8 reads are served by L2 (the 4 taps of
 * neighbouring pixels overlap), fp32 writes are coalesced per plane.  HBM-bound: 1.23 MB in, 4.92 MB out.
 * ------------------------------------------------------------------------------------------ */
/* the three channels of output pixel (ox, oy) */
__device__ __forceinline__ void preprocess_pixel(const TkPreprocessArgs& a, const uint8_t* src, float x_ratio, float y_ratio, uint32_t ox, uint32_t oy, float out[3]) {
    const float gx = x_ratio * (float)ox, gy = y_ratio * (float)oy;
    const int x = (int)gx, y = (int)gy;
    const float xd = gx - (float)x, yd = gy - (float)y;
    const int x1 = x + 1 < (int)a.in_w ? x + 1 : x, y1 = y + 1 < (int)a.in_h ? y + 1 : y; /* reference reads x+1/y+1 (always in range for w,h >= 2) */
    const uint8_t* r0 = src + (size_t)y * a.in_stride;
    const uint8_t* r1 = src + (size_t)y1 * a.in_stride;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const float p1 = (float)r0[x * a.bpp + c], p2 = (float)r0[x1 * a.bpp + c];
        const float p3 = (float)r1[x * a.bpp + c], p4 = (float)r1[x1 * a.bpp + c];
        float v = (p1 * (1.0f - xd)) * (1.0f - yd);
        v = v + (p2 * xd) * (1.0f - yd);
        v = v + (p3 * (1.0f - xd)) * yd;
        v = v + (p4 * xd) * yd;
        out[c] = tk_divf(tk_divf(v, 255.0f) - a.mean[c], a.std_dev[c]);
    }
}
__global__ void k_preprocess(TkPreprocessArgs a) {
    const uint32_t ox = blockIdx.x * blockDim.x + threadIdx.x, oy = blockIdx.y * blockDim.y + threadIdx.y;
    if (ox >= a.out_w || oy >= a.out_h) return;
    const float x_ratio = tk_divf((float)a.in_w - 1.0f, (float)a.out_w);
    const float y_ratio = tk_divf((float)a.in_h - 1.0f, (float)a.out_h);
    const size_t np = (size_t)a.out_w * a.out_h, pix = (size_t)oy * a.out_w + ox;
    float o[3];
    preprocess_pixel(a, a.src, x_ratio, y_ratio, ox, oy, o);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        if (a.nhwc) a.dst[pix * 3 + c] = o[c];
        else a.dst[c * np + pix] = o[c];
    }
}

void tk_launch_preprocess(const TkPreprocessArgs& a, hipStream_t s) {
    dim3 block(64, 4);
    dim3 grid((a.out_w + 63) / 64, (a.out_h + 3) / 4);
    hipLaunchKernelGGL(k_preprocess, grid, block, 0, s, a);
}

/*
 * The detector's stem, 3 -> 16 channels, 3 x 3, stride 2, padding 1: a thread per output pixel, all 16 channels as the GEMM's chain — acc = fma(a[k], w[n][k], acc) over
 * k = (ky 3 + kx) 3 + c ascending from +0, padding as a = 0 — then bias and SiLU.  The input pixels under a tile of 32 x 8 outputs go through the LDS; from camera
 * frames they are pre-processed on the way, so that the network's input tensor is never written or read.  Weights are read through the scalar cache ([27][16]).
 * Vector instructions bound it (per output 432 fmas and 16 SiLUs, per input pixel ~110): one frame 15 us (pre-processing and stem as launches of their own:
 * 24), 32 frames 546 -> 160 us.  All byte loads of a thread ahead of their use: 178 at 32 frames, no gain at one.
 */
#define TK_STEM_TW 32
#define TK_STEM_TH 8
template <bool FRAMES>
__global__ __launch_bounds__(256) void k_stem(TkPreprocessArgs a, size_t frame_bytes, const float* tensor, int H, int W, int Ho, int Wo, const float* __restrict__ wt,
                                              const float* __restrict__ bias, int silu, float* y, int ldy) {
    constexpr int PW = 2 * TK_STEM_TW + 1, PH = 2 * TK_STEM_TH + 1, PN = PW * PH;
    __shared__ float px[3 * PN];
    const int tid = threadIdx.x, b = blockIdx.z;
    const int iy0 = 2 * (int)blockIdx.y * TK_STEM_TH - 1, ix0 = 2 * (int)blockIdx.x * TK_STEM_TW - 1;
    const float x_ratio = FRAMES ? tk_divf((float)a.in_w - 1.0f, (float)a.out_w) : 0.0f, y_ratio = FRAMES ? tk_divf((float)a.in_h - 1.0f, (float)a.out_h) : 0.0f;
    const uint8_t* src = FRAMES ? a.src + frame_bytes * (size_t)b : nullptr;
    for (int e = tid; e < PN; e += 256) {
        const int py = e / PW, iy = iy0 + py, ix = ix0 + e - py * PW;
        float v[3] = {0.0f, 0.0f, 0.0f};
        if (iy >= 0 && iy < H && ix >= 0 && ix < W) {
            if (FRAMES) preprocess_pixel(a, src, x_ratio, y_ratio, (uint32_t)ix, (uint32_t)iy, v);
            else {
                const float* p = tensor + (((int64_t)b * H + iy) * W + ix) * 3;
                v[0] = p[0]; v[1] = p[1]; v[2] = p[2];
            }
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) px[c * PN + e] = v[c];
    }
    __syncthreads();
    const int ly = tid / TK_STEM_TW, lx = tid % TK_STEM_TW;
    const int oy = blockIdx.y * TK_STEM_TH + ly, ox = blockIdx.x * TK_STEM_TW + lx;
    float acc[16];
#pragma unroll
    for (int n = 0; n < 16; ++n) acc[n] = 0.0f;
    const float* p = px + 2 * ly * PW + 2 * lx;
#pragma unroll
    for (int k = 0; k < 27; ++k) {
        const float v = p[(k % 3) * PN + (k / 9) * PW + k / 3 % 3];
#pragma unroll
        for (int n = 0; n < 16; ++n) acc[n] = __builtin_fmaf(v, wt[k * 16 + n], acc[n]);
    }
    if (oy >= Ho || ox >= Wo) return;
#pragma unroll
    for (int n = 0; n < 16; ++n) acc[n] = acc[n] + bias[n];
    if (silu) tk_silu_all<16>(acc);
    float4* o = (float4*)(y + (((int64_t)b * Ho + oy) * Wo + ox) * ldy);
#pragma unroll
    for (int n = 0; n < 16; n += 4) o[n >> 2] = make_float4(acc[n], acc[n + 1], acc[n + 2], acc[n + 3]);
}
/* [16][27] -> [27][16] */
__global__ void k_stem_weights(const float* w, float* wt) {
    for (int i = threadIdx.x; i < 432; i += blockDim.x) wt[i] = w[(i % 16) * 27 + i / 16];
}

/* ------------------------------------------------------------------------------------------ model */

TkYoloModel::~TkYoloModel() {
    (void)hipSetDevice(device);
    for (auto p : w) if (p) (void)hipFree(p);
    for (auto p : b) if (p) (void)hipFree(p);
    for (auto p : wp) if (p) (void)hipFree(p);
}

bool TkYoloModel::init(int dev, int n_classes) {
    device = dev;
    nc = n_classes;
    if (nc < 1 || nc > 1024) { error = "class count out of range"; return false; }
    struct Dummy {};
    specs = TkYoloV8n<Dummy>::specs(nc);
    HIPQ(hipSetDevice(device));
    w.assign(specs.size(), nullptr);
    b.assign(specs.size(), nullptr);
    wp.assign(specs.size(), nullptr);
    for (size_t i = 0; i < specs.size(); ++i) {
        const TkConvSpec& s = specs[i];
        HIPQ(hipMalloc((void**)&w[i], (size_t)s.cout * s.k * s.k * s.cin * 4));
        HIPQ(hipMalloc((void**)&b[i], (size_t)s.cout * 4));
        const bool stem = i == 0 && s.cin == 3 && s.cout == 16 && s.k == 3 && s.s == 2;
        if (stem || s.cin % 16 == 0) {
            const size_t n = stem ? 432 * 4 : tk_conv_weight_floats(s.cout, s.k * s.k * s.cin) * 4;
            HIPQ(hipMalloc((void**)&wp[i], n));
            HIPQ(hipMemset(wp[i], 0, n)); /* what lies behind the last piece is requested, not used */
        }
    }
    return true;
}

size_t TkYoloModel::param_count() const {
    size_t n = 0;
    for (const auto& s : specs) n += (size_t)s.cout * s.k * s.k * s.cin + s.cout;
    return n;
}

bool TkYoloModel::set_layer(int idx, const float* w_host, const float* b_host) {
    if (idx < 0 || idx >= (int)specs.size()) { error = "layer index out of range"; return false; }
    const TkConvSpec& s = specs[idx];
    HIPQ(hipSetDevice(device));
    HIPQ(hipMemcpy(w[idx], w_host, (size_t)s.cout * s.k * s.k * s.cin * 4, hipMemcpyHostToDevice));
    HIPQ(hipMemcpy(b[idx], b_host, (size_t)s.cout * 4, hipMemcpyHostToDevice));
    if (wp[idx]) {
        if (s.cin == 3) hipLaunchKernelGGL(k_stem_weights, dim3(1), dim3(64), 0, nullptr, w[idx], wp[idx]);
        else tk_launch_conv_weights(w[idx], s.cout, s.k * s.k * s.cin, wp[idx], nullptr);
        HIPQ(hipGetLastError());
        HIPQ(hipStreamSynchronize(nullptr)); /* the engines' streams do not wait for the null stream */
    }
    return true;
}

bool TkYoloModel::fill_synthetic(uint64_t seed, float cls_bias) {
    std::vector<float> hw, hb;
    const int n = (int)specs.size();
    for (int i = 0; i < n; ++i) {
        const TkConvSpec& s = specs[i];
        const int fan = s.k * s.k * s.cin;
        hw.resize((size_t)s.cout * fan);
        hb.resize(s.cout);
        /* the last class conv of each scale: layers n-13, n-7, n-1 (6 convs per scale, class 1x1 last) */
        const bool cls_out = (i == n - 1 || i == n - 7 || i == n - 13);
        for (size_t j = 0; j < hw.size(); ++j) hw[j] = tk_yolo_synth_w(seed, i, (int64_t)j, fan);
        for (int j = 0; j < s.cout; ++j) hb[j] = tk_yolo_synth_b(seed, i, j, cls_out, cls_bias);
        if (!set_layer(i, hw.data(), hb.data())) return false;
    }
    return true;
}

bool TkYoloModel::load_file(const char* path) {
    FILE* f = fopen(path, "rb");
    if (!f) { error = std::string("cannot open ") + path; return false; }
    char magic[8];
    int32_t hdr[2];
    bool ok = fread(magic, 1, 8, f) == 8 && memcmp(magic, "TKYOLO1", 8) == 0 && fread(hdr, 4, 2, f) == 2 && hdr[0] == (int)specs.size() && hdr[1] == nc;
    std::vector<float> hw, hb;
    for (size_t i = 0; ok && i < specs.size(); ++i) {
        const TkConvSpec& s = specs[i];
        int32_t d[4];
        ok = fread(d, 4, 4, f) == 4 && d[0] == s.cin && d[1] == s.cout && d[2] == s.k && d[3] == s.s;
        hw.resize((size_t)s.cout * s.k * s.k * s.cin);
        hb.resize(s.cout);
        ok = ok && fread(hw.data(), 4, hw.size(), f) == hw.size() && fread(hb.data(), 4, hb.size(), f) == hb.size();
        ok = ok && set_layer((int)i, hw.data(), hb.data());
    }
    fclose(f);
    if (!ok && error.empty()) error = "not a TKYOLO1 container for this geometry";
    return ok;
}

/* a YOLO-class file that is not the YOLOv8n topology: accepted when its graph is one the executor can run — every op supported, one float image
 * input [N, 3, H, W], a first output [N, 4 + nc, anchors] (checked against the engine's geometry at the first run) */
static bool yolo_generic_graph(const char* path, TkYoloModel* m, const std::string& why_not_v8n) {
    TkOnnxGraph g;
    if (!g.load(path)) { m->error = why_not_v8n + "; and as a graph: " + g.error; return false; }
    std::string err;
    if (!TkOnnxExec::ops_supported(g, &err)) { m->error = why_not_v8n + "; and the graph executor cannot run it: " + err; return false; }
    std::string in;
    for (const auto& vi : g.inputs) {
        if (g.init.count(vi.name) == 0 && (vi.elem_type == 1 || vi.elem_type == 0)) { /* (the reader already leaves initialisers out of `inputs`) */ if (!in.empty()) { m->error = why_not_v8n + "; and the graph has more than one float input"; return false; } in = vi.name; }
    }
    if (in.empty() || g.outputs.empty()) { m->error = why_not_v8n + "; and the graph has no float image input / no output"; return false; }
    m->generic = true;
    m->onnx_path = path;
    m->graph_in = in;
    m->graph_out = g.outputs[0].name;
    return true;
}

bool TkYoloModel::load_onnx(const char* path) {
    TkOnnxWeights ox;
    /* the Conv-initialiser reader only understands what a YOLOv8n export holds; a file it cannot read may still be a graph the executor runs */
    if (!ox.load(path)) return yolo_generic_graph(path, this, "as a YOLOv8n weight file: " + ox.error);
    /* 63 graph convolutions, optionally followed by the DFL projection conv [1][16][1][1] */
    size_t n = ox.convs.size();
    if (n == specs.size() + 1 && ox.convs.back().cout == 1 && ox.convs.back().cin == TK_YOLO_REG_MAX && ox.convs.back().kh == 1) --n;
    if (n != specs.size())
        return yolo_generic_graph(path, this, "the ONNX graph has " + std::to_string(ox.convs.size()) + " Conv nodes, YOLOv8n has " + std::to_string(specs.size()) + " (+ DFL)");
    for (size_t i = 0; i < n; ++i) { /* the hard-wired graph is the fast path: only a file that IS that topology takes it */
        const TkConvSpec& s = specs[i];
        const TkOnnxConv& c = ox.convs[i];
        if (c.cout != s.cout || c.cin != s.cin || c.kh != s.k || c.kw != s.k)
            return yolo_generic_graph(path, this, "Conv " + std::to_string(i) + " is [" + std::to_string(c.cout) + "][" + std::to_string(c.cin) + "][" + std::to_string(c.kh) + "][" +
                                                      std::to_string(c.kw) + "], the YOLOv8n graph expects [" + std::to_string(s.cout) + "][" + std::to_string(s.cin) + "][" +
                                                      std::to_string(s.k) + "][" + std::to_string(s.k) + "]");
    }
    std::vector<float> hw;
    for (size_t i = 0; i < n; ++i) {
        const TkConvSpec& s = specs[i];
        const TkOnnxConv& c = ox.convs[i];
        if (c.cout != s.cout || c.cin != s.cin || c.kh != s.k || c.kw != s.k) {
            error = "Conv " + std::to_string(i) + " does not match the YOLOv8n graph";
            return false;
        }
        hw.resize(c.w.size());
        for (int o = 0; o < s.cout; ++o) /* [cout][cin][kh][kw] -> [cout][kh][kw][cin] */
            for (int ci = 0; ci < s.cin; ++ci)
                for (int k = 0; k < s.k * s.k; ++k) hw[((size_t)o * s.k * s.k + k) * s.cin + ci] = c.w[((size_t)o * s.cin + ci) * s.k * s.k + k];
        if (!set_layer((int)i, hw.data(), c.b.data())) return false;
    }
    return true;
}

/* ------------------------------------------------------------------------------------------ graph ops on the GPU */

struct TkGpuOps {
    TkDetector* d;
    hipStream_t s;
    TkT alloc(int B, int H, int W, int C) {
        TkT t;
        t.B = B; t.H = H; t.W = W; t.C = C; t.ld = C;
        size_t n = ((size_t)B * H * W * C + 63) & ~(size_t)63;
        t.p = d->arena + d->arena_used;
        d->arena_used += n;
        return t;
    }
    const TkPreprocessArgs* frames = nullptr;
    size_t frame_bytes = 0;
    bool stem(const TkT& x, const TkT& y) {
        const TkConvSpec& sp = d->model->specs[0];
        if (!d->model->wp[0] || sp.cin != 3 || (y.ld & 3) || (((uintptr_t)y.p) & 15) || y.B > 65535) return false;
        const dim3 grid((y.W + TK_STEM_TW - 1) / TK_STEM_TW, (y.H + TK_STEM_TH - 1) / TK_STEM_TH, y.B);
        const TkPreprocessArgs a = frames ? *frames : TkPreprocessArgs{};
        if (frames) hipLaunchKernelGGL((k_stem<true>), grid, dim3(256), 0, s, a, frame_bytes, x.p, x.H, x.W, y.H, y.W, d->model->wp[0], d->model->b[0], sp.act, y.p, y.ld);
        else hipLaunchKernelGGL((k_stem<false>), grid, dim3(256), 0, s, a, frame_bytes, x.p, x.H, x.W, y.H, y.W, d->model->wp[0], d->model->b[0], sp.act, y.p, y.ld);
        return true;
    }
    /* the network's input tensor, of frames that no stem kernel takes */
    void preprocess(const TkT& x) {
        for (int b = 0; frames && b < x.B; ++b) {
            TkPreprocessArgs f = *frames;
            f.src += frame_bytes * b;
            f.dst = x.p + (size_t)b * x.H * x.W * 3;
            tk_launch_preprocess(f, s);
        }
    }
    /* A concatenation's copied and upsampled parts are not written: the convolution behind it reads them where they are (two sources).  Any other reader has them
     * written first. */
    struct Part { TkT x, y; int shift; };
    std::vector<Part> parts;
    static bool meets(const TkT& a, const TkT& b) {
        auto end = [](const TkT& t) { return t.p + ((size_t)t.B * t.H * t.W - 1) * t.ld + t.C; };
        return a.p < end(b) && b.p < end(a);
    }
    void settle(const TkT& x) {
        for (size_t i = 0; i < parts.size();) {
            if (!meets(parts[i].y, x)) { ++i; continue; }
            const Part q = parts[i];
            parts.erase(parts.begin() + i);
            if (q.shift) tk_launch_upsample2x(q.x.p, q.x.B, q.x.H, q.x.W, q.x.C, q.x.ld, q.y.p, q.y.ld, s);
            else tk_launch_copy_cols(q.x.p, q.x.B * q.x.H * q.x.W, q.x.C, q.x.ld, q.y.p, q.y.ld, s);
        }
    }
    /* the sources of x: itself, or with parts at its front and back; false: parts that do not make two sources */
    bool sources(const TkT& x, TkConvDirect* c) const {
        const Part *front = nullptr, *back = nullptr;
        for (const Part& q : parts) {
            if (!meets(q.y, x)) continue;
            if (q.y.ld != x.ld) return false;
            if (q.y.p == x.p && q.y.C < x.C && !front) front = &q;
            else if (q.y.p + q.y.C == x.p + x.C && q.y.p > x.p && !back) back = &q;
            else return false;
        }
        c->src[0] = TkConvSource{x.p, x.ld, 0};
        c->c_split = x.C;
        if (!front && !back) return true;
        c->c_split = front ? front->y.C : x.C - back->y.C;
        if (front && back && front->y.C + back->y.C != x.C) return false;
        c->src[1] = TkConvSource{x.p + c->c_split, x.ld, 0};
        if (front) c->src[0] = TkConvSource{front->x.p, front->x.ld, front->shift};
        if (back) c->src[1] = TkConvSource{back->x.p, back->x.ld, back->shift};
        return true;
    }
    /* false: not a layer for the direct kernel */
    bool describe(const TkT& x, int idx, const TkT& y, const TkT* res, TkConvDirect* out) const {
        const TkConvSpec& sp = d->model->specs[idx];
        if (d->fast || idx == 0 || !d->model->wp[idx]) return false;
        TkConvDirect& c = *out;
        c = TkConvDirect{};
        if (!sources(x, &c)) return false;
        c.B = x.B; c.H = x.H; c.W = x.W; c.C = x.C; c.k = sp.k; c.stride = sp.s; c.pad = sp.k / 2; c.Ho = y.H; c.Wo = y.W; c.N = sp.cout;
        c.w = d->model->wp[idx]; c.bias = d->model->b[idx];
        c.residual = res ? res->p : nullptr; c.ldr = res ? res->ld : 0;
        c.y = y.p; c.ldy = y.ld; c.act = sp.act ? TK_ACT_SILU : TK_ACT_NONE;
        return tk_conv_direct_takes(c);
    }
    bool direct(const TkT& x, int idx, const TkT& y, const TkT* res) {
        TkConvDirect c;
        if (!describe(x, idx, y, res, &c)) return false;
        /* 1 x 1: the GEMM kernels are as quick or quicker (32 frames, 80 x 80 x 64: 31.9 us, 36.2 here) unless a copy and an upsampling fall away (5 us each and more) */
        if (c.k == 1 && c.c_split == x.C) return false;
        TkConvPlan& plan = d->plans[x.B][idx];
        if (plan.mt == 0 && !tk_conv_direct_plan(c, &plan)) { plan.mt = 0; return false; }
        if (res) settle(*res);
        return tk_launch_conv_direct(c, plan, s);
    }
    /* The last 18 layers are six chains of three, box and class branch of each scale: their first layers in one launch, then the second, then the third.  One frame:
     * 18 launches of 170 us, now three of 73.  Up to eight frames' worth of an 80 x 80 map: where each layer fills the chip, the largest patch (256 channels) of one launch
     * sets how many workgroups a CU holds (32 frames: 1055 us for the first layers, 676 one by one).  Calls in sets / one by one: 640 x 640, 1 frame 491 / 565 us, 4 frames
     * 938 / 1035, 8 frames 1553 / 1653, 16 frames 2764 / 2861; 1280 x 736, 2 frames 1070 / 1147, 6 frames 2390 / 2333, 16 frames 5853 / 5428. */
    struct Layer { TkT x, y; int idx; };
    std::vector<Layer> heads[3];
    bool defer(const TkT& x, int idx, const TkT& y, const TkT* res) {
        const int at = idx - ((int)d->model->specs.size() - 18);
        if (at < 0 || res) return false;
        heads[at % 3].push_back(Layer{x, y, idx});
        if (at == 17) {
            for (auto& stage : heads) {
                TkConvDirect c[TK_CONV_SET];
                bool ok = stage.size() == TK_CONV_SET;
                for (size_t i = 0; ok && i < stage.size(); ++i) ok = describe(stage[i].x, stage[i].idx, stage[i].y, nullptr, &c[i]);
                ok = ok && (int64_t)c[0].B * c[0].H * c[0].W <= 8 * 6400;
                TkConvPlan p[TK_CONV_SET];
                if (ok && d->plans[x.B][stage[0].idx].mt == 0) {
                    ok = tk_conv_direct_plan_set(c, TK_CONV_SET, p);
                    for (int i = 0; ok && i < TK_CONV_SET; ++i) d->plans[x.B][stage[i].idx] = p[i];
                } else {
                    for (int i = 0; ok && i < TK_CONV_SET; ++i) p[i] = d->plans[x.B][stage[i].idx];
                }
                if (ok && tk_launch_conv_direct_set(c, p, TK_CONV_SET, s)) continue;
                for (const Layer& l : stage) run(l.x, l.idx, l.y, nullptr);
            }
        }
        return true;
    }
    void conv(const TkT& x, int idx, const TkT& y, const TkT* res) {
        pool();
        if (!defer(x, idx, y, res)) run(x, idx, y, res);
    }
    void run(const TkT& x, int idx, const TkT& y, const TkT* res) {
        const TkConvSpec& sp = d->model->specs[idx];
        if (idx == 0) {
            if (stem(x, y)) return;
            preprocess(x);
        }
        if (direct(x, idx, y, res)) return;
        settle(x);
        if (res) settle(*res);
        TkGemm g{};
        g.M = y.B * y.H * y.W; g.N = sp.cout; g.K = sp.k * sp.k * sp.cin;
        if (sp.k == 1 && sp.s == 1) { g.A = x.p; g.lda = x.ld; }
        else if (tk_gemm_im2col_ok(x.p, x.C, x.ld, d->model->w[idx])) { /* the GEMM addresses the input directly: no column matrix */
            g.A = x.p; g.lda = 0;
            g.im_C = x.C; g.im_H = x.H; g.im_W = x.W; g.im_ldx = x.ld; g.im_kw = sp.k; g.im_stride = sp.s; g.im_pad = sp.k / 2;
            g.im_Ho = y.H; g.im_Wo = y.W;
        } else {
            tk_launch_im2col(x.p, x.B, x.H, x.W, x.C, x.ld, sp.k, sp.k, sp.s, sp.k / 2, d->col, s);
            g.A = d->col; g.lda = g.K;
        }
        g.B = d->model->w[idx]; g.ldb = g.K; g.b_kn = 0;
        g.C = y.p; g.ldc = y.ld;
        g.bias = d->model->b[idx];
        g.residual = res ? res->p : nullptr; g.ldr = res ? res->ld : 0;
        g.act = sp.act ? TK_ACT_SILU : TK_ACT_NONE;
        g.alpha = 1.0f; g.batch = 1;
        g.fast = d->fast ? 1 : 0;
        tk_launch_gemm(g, s);
    }
    /* three poolings, each of the one before: one launch */
    struct Pool { TkT x, y; };
    std::vector<Pool> pools;
    void maxpool5(const TkT& x, const TkT& y) {
        if (!pools.empty() && (x.p != pools.back().y.p || x.C != y.C || x.ld != pools.back().y.ld || y.ld != x.ld)) pool();
        if (pools.empty()) settle(x);
        pools.push_back(Pool{x, y});
        if (pools.size() == 3) pool();
    }
    void pool() {
        const TkT x = pools.empty() ? TkT{} : pools[0].x;
        const bool chain = pools.size() == 3 && tk_launch_maxpool5_chain(x.p, x.B, x.H, x.W, x.C, x.ld, pools[0].y.p, pools[1].y.p, pools[2].y.p, pools[0].y.ld, s);
        if (!chain)
            for (const Pool& q : pools) tk_launch_maxpool5(q.x.p, q.x.B, q.x.H, q.x.W, q.x.C, q.x.ld, q.y.p, q.y.ld, s);
        pools.clear();
    }
    void upsample2x(const TkT& x, const TkT& y) { pool(); settle(x); parts.push_back(Part{x, y, 1}); }
    void copy(const TkT& x, const TkT& y) { pool(); settle(x); parts.push_back(Part{x, y, 0}); }
};

/* sizing pass: same graph, counts arena floats and the largest im2col matrix */
struct TkSizeOps {
    const std::vector<TkConvSpec>* specs;
    size_t used = 0, col = 0;
    TkT alloc(int B, int H, int W, int C) {
        TkT t;
        t.B = B; t.H = H; t.W = W; t.C = C; t.ld = C;
        used += ((size_t)B * H * W * C + 63) & ~(size_t)63;
        return t;
    }
    void conv(const TkT&, int idx, const TkT& y, const TkT*) {
        const TkConvSpec& sp = (*specs)[idx];
        if (!(sp.k == 1 && sp.s == 1)) { size_t n = (size_t)y.B * y.H * y.W * sp.k * sp.k * sp.cin; col = n > col ? n : col; }
    }
    void maxpool5(const TkT&, const TkT&) {}
    void upsample2x(const TkT&, const TkT&) {}
    void copy(const TkT&, const TkT&) {}
};

/* ------------------------------------------------------------------------------------------ decode + NMS kernels */

/* one lane of each anchor says whether it is a candidate: those of a wave are appended to the frame's list, in any order, as keys whose order is (score desc, anchor
 * asc) from the largest down */
__device__ __forceinline__ void append_candidate(bool is, float score, int anchor, uint64_t* list, int32_t* n_list) {
    const uint64_t all = __ballot(is);
    if (all == 0) return;
    const int lane = threadIdx.x & 63, first = __builtin_ctzll(all);
    int base = 0;
    if (lane == first) base = atomicAdd(n_list, __popcll(all));
    base = __shfl(base, first, 64);
    const uint32_t u = tk_f32_bits(score + 0.0f), up = u >> 31 ? ~u : u | 0x80000000u; /* (-0 counts as +0) */
    if (is) list[base + __popcll(all & ((1ull << lane) - 1ull))] = (uint64_t)up << 32 | (uint32_t)~(uint32_t)anchor;
}

/* Four lanes per anchor: lane q takes side q of the box and of every 16 classes the four from 4 q on (first class on ties, as tk_yolo_decode_anchor).  One thread per
 * anchor was a chain of 64 + nc exponentials on a tenth of the chip: 29 us for the 8400 anchors of one 640 x 640 frame, now 8. */
__global__ __launch_bounds__(256) void k_yolo_decode(TkT h0, TkT h1, TkT h2, int nc, int n_anchors, float conf, tk_yolo_cand_t* cand, uint64_t* list, int32_t* n_list) {
    const int at = (blockIdx.x * 256 + threadIdx.x) >> 2, q = threadIdx.x & 3, b = blockIdx.y;
    const int a = at < n_anchors ? at : n_anchors - 1; /* past the end: not stored */
    const int n0 = h0.H * h0.W, n1 = h1.H * h1.W;
    const TkT* h;
    int local;
    float stride;
    if (a < n0) { h = &h0; local = a; stride = 8.0f; }
    else if (a < n0 + n1) { h = &h1; local = a - n0; stride = 16.0f; }
    else { h = &h2; local = a - n0 - n1; stride = 32.0f; }
    const float ax = (float)(local % h->W) + 0.5f, ay = (float)(local / h->W) + 0.5f;
    const float* o = h->p + ((size_t)b * h->H * h->W + local) * h->ld;
    float side[16];
    float best = -1.0f;
    int bi = 0;
    auto score = [&](float l, int k) {
        const float s = tk_sigmoidf(l);
        if (s > best) { best = s; bi = k; }
    };
    if ((nc & 3) == 0) { /* pixels of 64 + nc floats: every group of four is aligned */
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float4 t = ((const float4*)(o + 16 * q))[i];
            side[4 * i] = t.x; side[4 * i + 1] = t.y; side[4 * i + 2] = t.z; side[4 * i + 3] = t.w;
        }
        for (int k = 4 * q; k < nc; k += 16) {
            const float4 t = *(const float4*)(o + 64 + k);
            score(t.x, k); score(t.y, k + 1); score(t.z, k + 2); score(t.w, k + 3);
        }
    } else {
#pragma unroll
        for (int i = 0; i < 16; ++i) side[i] = o[16 * q + i];
        for (int k = q; k < nc; k += 4) score(o[64 + k], k);
    }
    const float d = tk_yolo_dfl(side);
#pragma unroll
    for (int w = 1; w <= 2; w <<= 1) {
        const float os = __shfl_xor(best, w, 64);
        const int oi = __shfl_xor(bi, w, 64);
        if (os > best || (os == best && oi < bi)) { best = os; bi = oi; }
    }
    const float from = q & 1 ? ay : ax, edge = (q < 2 ? from - d : from + d) * stride; /* x1 y1 x2 y2 */
    const bool is = at < n_anchors && best > conf;
    if (at < n_anchors) {
        tk_yolo_cand_t* c = cand + (size_t)b * n_anchors + a;
        (&c->x1)[q] = edge;
        if (q == 0) { c->score = best; c->cls = is ? bi : -1 /* not a candidate */; c->anchor = a; }
    }
    append_candidate(is && q == 0, best, a, list + (size_t)b * n_anchors, n_list + b);
}

/* a YOLO-class graph's own output [4 + nc][anchors] (Ultralytics export: box centre / size in input pixels, class probabilities already through
 * the sigmoid): xyxy = centre -/+ size / 2, score = max_c p_c (first class on ties), candidate iff score > confidence_threshold */
__global__ void k_yolo_decode_out(const float* out, int nc, int n_anchors, float conf, tk_yolo_cand_t* cand, uint64_t* list, int32_t* n_list) {
    const int at = blockIdx.x * blockDim.x + threadIdx.x, a = at < n_anchors ? at : n_anchors - 1;
    tk_yolo_cand_t c;
    tk_yolo_decode_out_anchor(out + a, n_anchors, nc, &c);
    c.anchor = a;
    const bool is = at < n_anchors && c.score > conf;
    if (!is) c.cls = -1;
    if (at < n_anchors) cand[a] = c;
    append_candidate(is, c.score, a, list, n_list);
}

/* rank of every candidate among the candidates; the best MAX_CAND are kept.  Most anchors fall below the confidence threshold and are not in the list.  A workgroup
 * takes 64 candidates, one a lane, and each of its waves a quarter of the list (1 000 candidates of 8 400 anchors: 20 us when every workgroup looked through all anchors,
 * 13 with a lane that walked the whole list, now 6). */
__global__ __launch_bounds__(256) void k_yolo_rank(const uint64_t* list, const int32_t* n_list, int n_anchors, int32_t* order, int32_t* n_cand) {
    const int b = blockIdx.y, n = n_list[b], lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i = blockIdx.x * 64 + lane;
    if (blockIdx.x == 0 && threadIdx.x == 0) n_cand[b] = n < TK_YOLO_MAX_CAND ? n : TK_YOLO_MAX_CAND;
    if (blockIdx.x * 64 >= n) return;
    const uint64_t* lb = list + (size_t)b * n_anchors;
    __shared__ __attribute__((aligned(16))) uint64_t tile[1024];
    __shared__ int part[4][64];
    const uint64_t own = lb[i < n ? i : n - 1];
    int rank = 0;
    for (int base = 0; base < n; base += 1024) {
        if (base) __syncthreads();
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int j = (int)threadIdx.x + u * 256;
            tile[j] = base + j < n ? lb[base + j] : 0; /* below every candidate */
        }
        __syncthreads();
        const int nt = n - base < 1024 ? n - base : 1024;
        for (int k = wave * 8; k < nt; k += 32) { /* the waves take turns: eight keys each */
            uint64_t o[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) o[u] = tile[k + u];
#pragma unroll
            for (int u = 0; u < 8; ++u) rank += o[u] > own ? 1 : 0;
        }
    }
    part[wave][lane] = rank;
    __syncthreads();
    if (wave != 0 || i >= n) return;
    rank = part[0][lane] + part[1][lane] + part[2][lane] + part[3][lane];
    if (rank < TK_YOLO_MAX_CAND) order[(size_t)b * TK_YOLO_MAX_CAND + rank] = (int32_t)~(uint32_t)own;
}

/* suppression bit matrix: bit j of mask[i] set iff j > i, same class, IoU > thr.  A wave holds 64 candidates j, one a lane, and takes 32 rows i: a row's
 * word is the ballot.  (A thread per word, which fetched its 64 candidates one after the other: 27 us for some tens of candidates, now 10.) */
__global__ __launch_bounds__(256) void k_yolo_mask(const tk_yolo_cand_t* cand, int n_anchors, const int32_t* order, const int32_t* n_cand, float iou_thr, uint64_t* mask) {
    __shared__ tk_yolo_cand_t rows[32];
    const int b = blockIdx.z, lane = threadIdx.x & 63, wj = blockIdx.x * 4 + (threadIdx.x >> 6), i0 = blockIdx.y * 32;
    const int n = n_cand[b];
    if (i0 >= n || blockIdx.x * 256 >= n) return;
    const tk_yolo_cand_t* cb = cand + (size_t)b * n_anchors;
    const int32_t* ob = order + (size_t)b * TK_YOLO_MAX_CAND;
    if (threadIdx.x < 32 && i0 + (int)threadIdx.x < n) rows[threadIdx.x] = cb[ob[i0 + threadIdx.x]];
    const int j = wj * 64 + lane;
    const tk_yolo_cand_t cj = cb[ob[j < n ? j : n - 1]];
    __syncthreads();
    if (wj * 64 >= n) return;
    for (int i = i0; i < n && i < i0 + 32; ++i) {
        const tk_yolo_cand_t ci = rows[i - i0];
        const uint64_t bits = __ballot(j > i && j < n && cj.cls == ci.cls && tk_yolo_iou(&ci, &cj) > iou_thr);
        if (lane == 0) mask[((size_t)b * TK_YOLO_MAX_CAND + i) * (TK_YOLO_MAX_CAND / 64) + wj] = bits;
    }
}

/* greedy scan, one wave per frame: 64 candidates at a time, whose words among themselves are in the lanes, so that a kept one costs a few scalar steps and
 * no trip to memory (44 us for some tens of kept boxes, now 8); the later words take the kept rows eight loads at a time */
__global__ __launch_bounds__(64) void k_yolo_scan(const tk_yolo_cand_t* cand, int n_anchors, const int32_t* order, const int32_t* n_cand, const uint64_t* mask,
                                                  TkDetection* kept, int32_t* n_kept, int32_t* n_list) {
    const int b = blockIdx.x, lane = threadIdx.x;
    if (lane == 0) n_list[b] = 0; /* for the next pass */
    constexpr int WORDS = TK_YOLO_MAX_CAND / 64;
    static_assert(WORDS <= 64, "a lane per word");
    const int n = n_cand[b];
    const int words = (n + 63) / 64;
    const tk_yolo_cand_t* cb = cand + (size_t)b * n_anchors;
    const int32_t* ob = order + (size_t)b * TK_YOLO_MAX_CAND;
    const uint64_t* mb = mask + (size_t)b * TK_YOLO_MAX_CAND * WORDS;
    uint64_t removed = 0; /* lane w: word w */
    int nk = 0;
    auto lane_of = [](uint64_t v, int l) {
        return (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, l) | (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), l) << 32;
    };
    for (int w = 0; w < words && nk < TK_OBJECT_DETECTOR_MAX_DETECTIONS; ++w) {
        const int i = w * 64 + lane;
        const uint64_t mine = i < n ? mb[(size_t)i * WORDS + w] : 0;
        const tk_yolo_cand_t c = cb[ob[i < n ? i : n - 1]];
        uint64_t left = ~lane_of(removed, w) & (n - w * 64 >= 64 ? ~0ull : (1ull << (n - w * 64)) - 1ull), keep = 0;
        while (left != 0) {
            const int k = __builtin_ctzll(left);
            keep |= 1ull << k;
            left &= ~(1ull << k) & ~lane_of(mine, k); /* a row marks later candidates only */
        }
        const int at = nk + __popcll(keep & ((1ull << lane) - 1ull));
        if ((keep >> lane & 1) && at < TK_OBJECT_DETECTOR_MAX_DETECTIONS) {
            TkDetection dt{c.x1, c.y1, c.x2, c.y2, c.score, c.cls, c.anchor};
            kept[(size_t)b * TK_OBJECT_DETECTOR_MAX_DETECTIONS + at] = dt;
        }
        nk += __popcll(keep);
        if (w + 1 < words) {
            const int word = lane < words ? lane : words - 1;
            while (keep != 0) {
                uint64_t r[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) { /* past the last kept one: it again */
                    const int k = __builtin_ctzll(keep);
                    r[u] = mb[(size_t)(w * 64 + k) * WORDS + word];
                    const uint64_t rest = keep & (keep - 1);
                    keep = u < 7 && rest == 0 ? keep : rest;
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) removed |= r[u];
            }
        }
    }
    if (lane == 0) n_kept[b] = nk < TK_OBJECT_DETECTOR_MAX_DETECTIONS ? nk : TK_OBJECT_DETECTOR_MAX_DETECTIONS;
}

/* ------------------------------------------------------------------------------------------ detector */

TkDetector::~TkDetector() {
    if (model) (void)hipSetDevice(model->device);
    if (upload_stream) (void)hipStreamSynchronize(upload_stream);
    if (stream) (void)hipStreamSynchronize(stream);
    void* ptrs[] = {frame_dev, arena, col, input, cand, order, n_cand, mask, results, list, n_list, attr_dev};
    for (void* p : ptrs) if (p) (void)hipFree(p);
    if (results_host) (void)hipHostFree(results_host);
    if (exec) exec->unload(); /* before its stream goes */
    if (stream) (void)hipStreamDestroy(stream);
    if (upload_stream) (void)hipStreamDestroy(upload_stream);
    if (uploaded) (void)hipEventDestroy(uploaded);
}

bool TkDetector::init(TkYoloModel* m, int w, int h, int mb) {
    model = m; in_w = w; in_h = h; max_batch = mb;
    if (!m || w <= 0 || h <= 0 || (w % 32) || (h % 32)) { error = "detector input must be a positive multiple of 32"; return false; }
    if (mb < 1 || mb > 256) { error = "max_batch must be in [1,256]"; return false; }
    HIPQ(hipSetDevice(m->device));
    HIPQ(tk_create_perception_stream(&stream));
    n_anchors = (h / 8) * (w / 8) + (h / 16) * (w / 16) + (h / 32) * (w / 32);
    if (m->generic) {
        /* the file's own graph, one frame per run: every node's output of a run lives in the executor's arena (a YOLO-nano-class graph at 640 x 640
         * holds ~25 M activation floats + im2col scratch; 320 floats per input pixel leaves a wide margin and is checked by the executor) */
        exec.reset(new TkOnnxExec());
        if (!exec->load(m->onnx_path.c_str(), m->device, stream, (size_t)320 * h * w + (1u << 22))) { error = "detector graph: " + exec->error; return false; }
    } else {
        TkSizeOps so{&m->specs};
        TkT x = so.alloc(mb, h, w, 3);
        so.used = 0;
        TkT o[3];
        TkYoloV8n<TkSizeOps>::forward(so, x, o, m->nc);
        arena_floats = so.used + 1024;
        col_floats = so.col + 1024;
        HIPQ(hipMalloc((void**)&arena, arena_floats * 4));
        HIPQ(hipMalloc((void**)&col, col_floats * 4));
    }
    plans.resize((size_t)mb + 1);
    HIPQ(hipMalloc((void**)&input, (size_t)mb * h * w * 3 * 4));
    HIPQ(hipMalloc((void**)&cand, (size_t)mb * n_anchors * sizeof(tk_yolo_cand_t)));
    HIPQ(hipMalloc((void**)&order, (size_t)mb * TK_YOLO_MAX_CAND * 4));
    HIPQ(hipMalloc((void**)&n_cand, (size_t)mb * 4));
    HIPQ(hipMalloc((void**)&mask, (size_t)mb * TK_YOLO_MAX_CAND * (TK_YOLO_MAX_CAND / 64) * 8));
    HIPQ(hipMalloc((void**)&list, (size_t)mb * n_anchors * 8));
    HIPQ(hipMalloc((void**)&n_list, (size_t)mb * 4));
    kept_at = ((size_t)mb * 4 + 255) & ~(size_t)255;
    HIPQ(hipMalloc((void**)&results, kept_at + (size_t)mb * TK_OBJECT_DETECTOR_MAX_DETECTIONS * sizeof(TkDetection)));
    n_kept = (int32_t*)results;
    kept = (TkDetection*)(results + kept_at);
    HIPQ(hipHostMalloc((void**)&results_host, kept_at + (size_t)mb * TK_OBJECT_DETECTOR_MAX_DETECTIONS * sizeof(TkDetection), hipHostMallocDefault));
    return true;
}

/* generic models: frame by frame through the file's graph (exports carry a batch dimension of one), each frame's output decoded before the next
 * run reuses the arena (same stream: in order) */
bool TkDetector::run_graph(int B, float* host_out) {
    for (int b = 0; b < B; ++b) {
        exec->begin();
        TkOnnxExec::Val in;
        in.d = input + (size_t)b * 3 * in_h * in_w;
        in.shape = {1, 3, in_h, in_w};
        exec->bind(model->graph_in, in);
        if (!exec->run()) { error = "detector graph: " + exec->error; return false; }
        const TkOnnxExec::Val* o = exec->value(model->graph_out);
        if (!o || !o->d || o->is_int) { error = "detector graph: no float output"; return false; }
        /* [1, 4 + nc, anchors] (or [4 + nc, anchors]) with this engine's anchor count */
        const size_t r = o->shape.size();
        if (r < 2 || o->shape[r - 1] != n_anchors || o->shape[r - 2] != 4 + model->nc || o->count() != (int64_t)(4 + model->nc) * n_anchors) {
            std::string sh;
            for (int64_t d : o->shape) sh += (sh.empty() ? "" : ", ") + std::to_string(d);
            error = "detector graph: output [" + sh + "], expected [1, " + std::to_string(4 + model->nc) + ", " + std::to_string(n_anchors) + "] (4 + class_count rows, " +
                    std::to_string(in_w) + " x " + std::to_string(in_h) + " at strides 8 / 16 / 32)";
            return false;
        }
        hipLaunchKernelGGL(k_yolo_decode_out, dim3((n_anchors + 255) / 256), dim3(256), 0, stream, o->d, model->nc, n_anchors, conf, cand + (size_t)b * n_anchors, list + (size_t)b * n_anchors, n_list + b);
        if (host_out) HIPQ(hipMemcpyAsync(host_out + (size_t)b * o->count(), o->d, (size_t)o->count() * 4, hipMemcpyDeviceToHost, stream)); /* before the next run reuses the arena */
    }
    return true;
}

bool TkDetector::forward_graph(int B, const float* nchw_host, std::vector<float>* out) {
    if (!model->generic) { error = "forward_graph is the graph-executor path's hook (this model runs the hard-wired YOLOv8n graph: forward_tensor)"; return false; }
    if (B < 1 || B > max_batch) { error = "batch larger than the detector was created for"; return false; }
    HIPQ(hipSetDevice(model->device));
    HIPQ(hipMemcpyAsync(input, nchw_host, (size_t)B * 3 * in_h * in_w * 4, hipMemcpyHostToDevice, stream));
    out->assign((size_t)B * (4 + model->nc) * n_anchors, 0.0f);
    last_B = 0;
    if (!begin_list() || !run_graph(B, out->data())) return false;
    hipLaunchKernelGGL(k_yolo_rank, dim3((n_anchors + 63) / 64, B), dim3(256), 0, stream, list, n_list, n_anchors, order, n_cand);
    hipLaunchKernelGGL(k_yolo_mask, dim3(TK_YOLO_MAX_CAND / 256, TK_YOLO_MAX_CAND / 32, B), dim3(256), 0, stream, cand, n_anchors, order, n_cand, iou, mask);
    hipLaunchKernelGGL(k_yolo_scan, dim3(B), dim3(64), 0, stream, cand, n_anchors, order, n_cand, mask, kept, n_kept, n_list);
    HIPQ(hipGetLastError());
    list_clear = true;
    HIPQ(hipStreamSynchronize(stream));
    return true;
}

/* a pass that did not come to its end may have left counts behind */
bool TkDetector::begin_list() {
    if (!list_clear) HIPQ(hipMemsetAsync(n_list, 0, (size_t)max_batch * 4, stream));
    list_clear = false;
    return true;
}

bool TkDetector::network(int first, int B, const TkPreprocessArgs* frames) {
    TkT x;
    x.p = input; x.B = B; x.H = in_h; x.W = in_w; x.C = 3; x.ld = 3;
    if (plans[B].empty()) plans[B].assign(model->specs.size(), TkConvPlan{});
    TkGpuOps ops;
    ops.d = this; ops.s = stream;
    ops.frames = frames;
    ops.frame_bytes = frames ? (size_t)frames->in_stride * frames->in_h : 0;
    arena_used = 0;
    TkYoloV8n<TkGpuOps>::forward(ops, x, heads, model->nc);
    const size_t at = (size_t)first * n_anchors;
    hipLaunchKernelGGL(k_yolo_decode, dim3((n_anchors + 63) / 64, B), dim3(256), 0, stream, heads[0], heads[1], heads[2], model->nc, n_anchors, conf, cand + at, list + at, n_list + first);
    HIPQ(hipGetLastError());
    return true;
}

bool TkDetector::suppress(int B) {
    hipLaunchKernelGGL(k_yolo_rank, dim3((n_anchors + 63) / 64, B), dim3(256), 0, stream, list, n_list, n_anchors, order, n_cand);
    hipLaunchKernelGGL(k_yolo_mask, dim3(TK_YOLO_MAX_CAND / 256, TK_YOLO_MAX_CAND / 32, B), dim3(256), 0, stream, cand, n_anchors, order, n_cand, iou, mask);
    hipLaunchKernelGGL(k_yolo_scan, dim3(B), dim3(64), 0, stream, cand, n_anchors, order, n_cand, mask, kept, n_kept, n_list);
    HIPQ(hipGetLastError());
    list_clear = true;
    return true;
}

bool TkDetector::enqueue(int B, const TkPreprocessArgs* frames) {
    return begin_list() && (model->generic ? run_graph(B, nullptr) : network(0, B, frames)) && suppress(B);
}

int tk_detector_first_part(int B, size_t frame_bytes, int in_w, int in_h) {
    const float up = (float)frame_bytes * (1.0f / 24.5e3f), per = 117.0f * ((float)in_w * (float)in_h / (640.0f * 640.0f));
    auto net = [&](int n) { return 380.0f + per * (float)n; };
    int best = B;
    float least = 0.95f * (up * (float)B + net(B));
    for (int f = 4; f < B; f += 4) {
        const float us = up * (float)f + std::max(net(f), 100.0f /* launches */ + up * (float)(B - f)) + net(B - f);
        if (us < least) { least = us; best = f; }
    }
    return best;
}

/* frames first .. first + n - 1 to their places on the device */
bool TkDetector::upload(const uint8_t* const* frames, size_t frame_bytes, int first, int n, hipStream_t s) {
    for (int b = first; b < first + n; ++b) HIPQ(hipMemcpyAsync(frame_dev + frame_bytes * b, frames[b], frame_bytes, hipMemcpyHostToDevice, s));
    return true;
}

bool TkDetector::detect(int B, const uint8_t* const* frames, uint32_t w, uint32_t h, uint32_t stride, uint32_t bpp, std::vector<std::vector<TkDetection>>* out) {
    if (B < 1 || B > max_batch) { error = "batch larger than the detector was created for"; return false; }
    if (w < 2 || h < 2 || stride < w * bpp) { error = "frame geometry invalid (need w,h >= 2 and stride >= w*bpp)"; return false; }
    HIPQ(hipSetDevice(model->device));
    const size_t fb = (size_t)stride * h;
    if (fb * B > frame_cap) { /* once per frame geometry: room for the engine's whole batch, so a wider job later never re-allocates (hipFree synchronises the device) */
        if (frame_dev) (void)hipFree(frame_dev);
        frame_dev = nullptr;
        HIPQ(hipMalloc((void**)&frame_dev, fb * max_batch));
        frame_cap = fb * max_batch;
    }
    TkPreprocessArgs a{};
    a.src = frame_dev; a.in_w = w; a.in_h = h; a.in_stride = stride; a.bpp = bpp;
    a.dst = input; a.out_w = in_w; a.out_h = in_h; a.nhwc = model->generic ? 0 : 1; /* a file's graph takes planar NCHW */
    for (int c = 0; c < 3; ++c) { a.mean[c] = mean[c]; a.std_dev[c] = std_dev[c]; }
    last_w = w; last_h = h; last_stride = stride; last_B = B;
    if (model->generic) {
        if (!upload(frames, fb, 0, B, stream)) return false;
        for (int b = 0; b < B; ++b) {
            TkPreprocessArgs f = a;
            f.src = frame_dev + fb * b;
            f.dst = input + (size_t)b * in_h * in_w * 3;
            tk_launch_preprocess(f, stream);
        }
        return enqueue(B) && fetch(B, out);
    }
    const int part = tk_detector_first_part(B, fb, in_w, in_h); /* the network takes the frames (TkGpuOps::run) */
    if (part == B) return upload(frames, fb, 0, B, stream) && enqueue(B, &a) && fetch(B, out);
    if (!upload_stream) {
        HIPQ(tk_create_perception_stream(&upload_stream));
        HIPQ(hipEventCreateWithFlags(&uploaded, hipEventDisableTiming));
    }
    if (!upload(frames, fb, 0, part, stream) || !begin_list() || !network(0, part, &a)) return false;
    const bool there = upload(frames, fb, part, B - part, upload_stream);
    if (!there || hipEventRecord(uploaded, upload_stream) != hipSuccess || hipStreamWaitEvent(stream, uploaded, 0) != hipSuccess) {
        (void)hipStreamSynchronize(upload_stream); /* nothing reads the caller's frames any more */
        if (there) error = "frames: the wait for their second part could not be enqueued";
        return false;
    }
    a.src = frame_dev + fb * part;
    if (!network(part, B - part, &a) || !suppress(B)) { (void)hipStreamSynchronize(upload_stream); return false; }
    return fetch(B, out);
}

/* ------------------------------------------------------------------------------------------
 * Per-box attributes (reference: src/vision/tk_attribute_classifier.c, run per detection by tk_vision_pipeline.c:462-485).
 * One workgroup per box; both classifiers are byte / integer histograms over the box's pixels, so the counts are exact whatever
 * the order the threads visit them in, and the fp32 / fp64 arithmetic of the HSV test is the reference's, operation for operation:
 *   r,g,b = u8 / 255.0f;  v = max, delta = max - min, s = delta / max  (s = 0 when max = 0)
 *   h = 60 * ((g - b) / delta | 2 + (b - r) / delta | 4 + (r - g) / delta), + 360 when negative   (the constants are doubles in the
 *   reference: a float op double op rounds once more on the store to float, reproduced with explicit double arithmetic)
 *   s < 0.1 (double compare): black (v < 0.1) / white (v > 0.9) / gray, else six 60-degree hue bins starting at 330.
 * Dominant colour = first bin with the maximum count.  Like the reference the frame is read as tightly packed RGB8
 * (row pitch = 3 * width, :56); pixels outside the frame are skipped (:54).
 * Door state: count interior pixels whose luminance (integer 299/587/114 per mille) differs by more than 100 between the rows above
 * and below; closed when count / (w * h) > 0.1.  The reference does not bounds-check this loop (:113-117); out-of-frame pixels are
 * skipped here.
 * ------------------------------------------------------------------------------------------ */
__device__ __forceinline__ int tk_color_bin(uint8_t R, uint8_t G, uint8_t B) {
    const float r = tk_divf((float)R, 255.0f), g = tk_divf((float)G, 255.0f), b = tk_divf((float)B, 255.0f);
    const float mx = fmaxf(r, fmaxf(g, b)), mn = fminf(r, fminf(g, b));
    const float delta = mx - mn, v = mx;
    float s = 0.0f, h = 0.0f;
    if ((double)mx > 0.0) {
        s = tk_divf(delta, mx);
        if (r >= mx) h = tk_divf(g - b, delta);
        else if (g >= mx) h = (float)(2.0 + (double)tk_divf(b - r, delta));
        else h = (float)(4.0 + (double)tk_divf(r - g, delta));
        h = (float)((double)h * 60.0);
        if ((double)h < 0.0) h = (float)((double)h + 360.0);
    }
    if ((double)s < 0.1) return (double)v < 0.1 ? 6 : ((double)v > 0.9 ? 7 : 8);
    if (h < 30.0f || h >= 330.0f) return 0;
    if (h < 90.0f) return 1;
    if (h < 150.0f) return 2;
    if (h < 210.0f) return 3;
    if (h < 270.0f) return 4;
    if (h < 330.0f) return 5;
    return -1; /* NaN hue: the reference counts the pixel in no bin */
}

__device__ __forceinline__ int tk_luma(const uint8_t* p) { return (int)(uint8_t)((p[0] * 299 + p[1] * 587 + p[2] * 114) / 1000); }

__global__ __launch_bounds__(256) void k_box_attributes(const uint8_t* frame, int W, int H, const int32_t* rects, int32_t* out) {
    __shared__ int bins[9];
    __shared__ int edges;
    const int box = blockIdx.x, t = threadIdx.x;
    const int bx = rects[4 * box], by = rects[4 * box + 1], bw = rects[4 * box + 2], bh = rects[4 * box + 3];
    if (t < 9) bins[t] = 0;
    if (t == 0) edges = 0;
    __syncthreads();
    const int64_t npix = (bw > 0 && bh > 0) ? (int64_t)bw * bh : 0;
    for (int64_t i = t; i < npix; i += 256) {
        const int x = bx + (int)(i % bw), y = by + (int)(i / bw);
        if (x < 0 || x >= W || y < 0 || y >= H) continue;
        const uint8_t* p = frame + ((int64_t)y * W + x) * 3;
        const int c = tk_color_bin(p[0], p[1], p[2]);
        if (c >= 0) atomicAdd(&bins[c], 1);
        const int lx = x - bx, ly = y - by; /* door-state loop: interior of the box, rows above / below inside the frame */
        if (lx >= 1 && lx < bw - 1 && ly >= 1 && ly < bh - 1 && y >= 1 && y < H - 1) {
            const int d = tk_luma(p - (int64_t)W * 3) - tk_luma(p + (int64_t)W * 3);
            if ((d < 0 ? -d : d) > 100) atomicAdd(&edges, 1);
        }
    }
    __syncthreads();
    if (t == 0) {
        int best = 0;
        for (int i = 1; i < 9; ++i)
            if (bins[i] > bins[best]) best = i;
        out[2 * box] = best;
        const float density = tk_divf((float)edges, (float)(bw * bh));
        out[2 * box + 1] = (double)density > 0.1 ? 1 : 0;
    }
}

bool TkDetector::run_attributes(const uint8_t* frame, uint32_t w, uint32_t h, int n, const int32_t* rects, int32_t* color, int32_t* door_closed) {
    if (n <= 0) return true;
    if (n > attr_cap) { /* at least the detector's own cap of boxes at the first use: no regrowth afterwards */
        const int want = n > TK_OBJECT_DETECTOR_MAX_DETECTIONS ? n : TK_OBJECT_DETECTOR_MAX_DETECTIONS;
        if (attr_dev) (void)hipFree(attr_dev);
        attr_dev = nullptr;
        attr_cap = 0;
        HIPQ(hipMalloc((void**)&attr_dev, (size_t)want * 6 * 4));
        attr_cap = want;
    }
    int32_t* res = attr_dev + (size_t)attr_cap * 4;
    HIPQ(hipMemcpyAsync(attr_dev, rects, (size_t)n * 16, hipMemcpyHostToDevice, stream));
    hipLaunchKernelGGL(k_box_attributes, dim3(n), dim3(256), 0, stream, frame, (int)w, (int)h, attr_dev, res);
    std::vector<int32_t> hr((size_t)n * 2);
    HIPQ(hipMemcpyAsync(hr.data(), res, (size_t)n * 8, hipMemcpyDeviceToHost, stream));
    HIPQ(hipStreamSynchronize(stream));
    for (int i = 0; i < n; ++i) {
        if (color) color[i] = hr[2 * i];
        if (door_closed) door_closed[i] = hr[2 * i + 1];
    }
    return true;
}

bool TkDetector::classify_boxes(int b, int n, const int32_t* rects, int32_t* color, int32_t* door_closed) {
    if (b < 0 || b >= last_B || !frame_dev) { error = "no frame of that index is resident (call detect first)"; return false; }
    if (last_stride != last_w * 3) { error = "attribute classification reads tightly packed RGB8 frames, as the reference does"; return false; }
    HIPQ(hipSetDevice(model->device));
    return run_attributes(frame_dev + (size_t)last_stride * last_h * b, last_w, last_h, n, rects, color, door_closed);
}

bool tk_classify_boxes_host(int device, const uint8_t* frame, uint32_t w, uint32_t h, int n, const int32_t* rects, int32_t* color,
                            int32_t* door_closed, std::string* error) {
    if (n <= 0) return true;
    uint8_t* df = nullptr;
    int32_t* dr = nullptr;
    const size_t fb = (size_t)w * h * 3;
    bool ok = hipSetDevice(device) == hipSuccess && hipMalloc((void**)&df, fb) == hipSuccess && hipMalloc((void**)&dr, (size_t)n * 6 * 4) == hipSuccess;
    std::vector<int32_t> hr((size_t)n * 2);
    if (ok) ok = hipMemcpy(df, frame, fb, hipMemcpyHostToDevice) == hipSuccess && hipMemcpy(dr, rects, (size_t)n * 16, hipMemcpyHostToDevice) == hipSuccess;
    if (ok) {
        hipLaunchKernelGGL(k_box_attributes, dim3(n), dim3(256), 0, nullptr, df, (int)w, (int)h, dr, dr + (size_t)n * 4);
        ok = hipGetLastError() == hipSuccess && hipMemcpy(hr.data(), dr + (size_t)n * 4, (size_t)n * 8, hipMemcpyDeviceToHost) == hipSuccess;
    }
    if (df) (void)hipFree(df);
    if (dr) (void)hipFree(dr);
    if (!ok) { if (error) *error = "HIP error in the attribute classifier"; return false; }
    for (int i = 0; i < n; ++i) {
        if (color) color[i] = hr[2 * i];
        if (door_closed) door_closed[i] = hr[2 * i + 1];
    }
    return true;
}

bool TkDetector::fetch(int B, std::vector<std::vector<TkDetection>>* out) {
    /* counts and boxes in one copy to pinned memory (two to pageable memory were staged and waited for one by one) */
    HIPQ(hipMemcpyAsync(results_host, results, kept_at + (size_t)B * TK_OBJECT_DETECTOR_MAX_DETECTIONS * sizeof(TkDetection), hipMemcpyDeviceToHost, stream));
    HIPQ(hipStreamSynchronize(stream));
    const int32_t* nk = (const int32_t*)results_host;
    const TkDetection* hk = (const TkDetection*)(results_host + kept_at);
    out->assign(B, {});
    for (int b = 0; b < B; ++b) (*out)[b].assign(hk + (size_t)b * TK_OBJECT_DETECTOR_MAX_DETECTIONS, hk + (size_t)b * TK_OBJECT_DETECTOR_MAX_DETECTIONS + nk[b]);
    return true;
}

bool TkDetector::forward_tensor(int B, const float* nhwc_host, std::vector<float>* raw_out) {
    if (model->generic) { error = "raw head maps exist on the hard-wired YOLOv8n path only; this model runs its file's graph (forward_graph)"; return false; }
    if (B < 1 || B > max_batch) { error = "batch larger than the detector was created for"; return false; }
    HIPQ(hipSetDevice(model->device));
    HIPQ(hipMemcpyAsync(input, nhwc_host, (size_t)B * in_h * in_w * 3 * 4, hipMemcpyHostToDevice, stream));
    if (!enqueue(B)) return false;
    const int no = 64 + model->nc;
    raw_out->resize((size_t)B * n_anchors * no);
    size_t off = 0;
    for (int b = 0; b < B; ++b)
        for (int i = 0; i < 3; ++i) {
            const size_t n = (size_t)heads[i].H * heads[i].W * no;
            HIPQ(hipMemcpyAsync(raw_out->data() + off, heads[i].p + (size_t)b * n, n * 4, hipMemcpyDeviceToHost, stream));
            off += n;
        }
    HIPQ(hipStreamSynchronize(stream));
    return true;
}
