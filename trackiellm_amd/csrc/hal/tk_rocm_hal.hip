/*
 * tk_rocm_hal.hip — dispatcher + kernel launchers of the reference's ROCm HAL surface
 * (src/gpu/rocm/tk_rocm_dispatch.hpp:83-217, src/gpu/rocm/tk_rocm_kernels.hpp:96,133,176).
 */
#include <hip/hip_runtime.h>
#include <stdlib.h>

#include <vector>

#include "../common/tk_exact_math.h"
#include "tk/tk_mi355x_ext.h"

#include "../vision/tk_vision_engine.h"
#include "tk/tk_rocm_hal.h"
#include "../nn/tk_gemm_image.h"
#include "../nn/tk_gemm_tiled.h"
#include "../nn/tk_conv_direct.h"
#include "../nn/tk_nn_kernels.h"

struct tk_gpu_buffer_s {
    void* dptr;
    size_t size;
};

struct tk_rocm_dispatcher_s {
    int device;
    hipStream_t compute, h2d, d2h; /* three non-blocking streams, as the reference dispatcher */
    hipEvent_t ev_upload, ev_compute;
};

/* out = raw * scale + shift  (src/gpu/rocm/tk_rocm_kernels.cpp:148-163), grid-stride, float4-free: the maps are tiny */
__global__ void k_postprocess_depth(tk_postprocess_depth_params_t p) {
    const size_t n = (size_t)p.width * p.height;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        p.d_metric_depth_map[i] = p.d_raw_depth_map[i] * p.scale + p.shift;
}

/* pinhole unprojection (src/gpu/rocm/tk_rocm_kernels.cpp:176-202): depth <= 0 -> origin */
__global__ void k_depth_to_points(tk_depth_to_points_params_t p) {
    const size_t n = (size_t)p.width * p.height;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const float d = p.d_metric_depth_map[i];
        tk_float3 o = {0.0f, 0.0f, 0.0f};
        if (d > 0.0f) {
            const float u = (float)(i % p.width), v = (float)(i / p.width);
            o.x = tk_divf((u - p.cx) * d, p.fx);
            o.y = tk_divf((v - p.cy) * d, p.fy);
            o.z = d;
        }
        p.d_point_cloud[i] = o;
    }
}

/* multiply-by-scale variant of the canonical pre-processor for scale != 1/255 */
__global__ void k_preprocess_scaled(TkPreprocessArgs a, float scale) {
    const uint32_t ox = blockIdx.x * blockDim.x + threadIdx.x, oy = blockIdx.y * blockDim.y + threadIdx.y;
    if (ox >= a.out_w || oy >= a.out_h) return;
    const float x_ratio = tk_divf((float)a.in_w - 1.0f, (float)a.out_w), y_ratio = tk_divf((float)a.in_h - 1.0f, (float)a.out_h);
    const float gx = x_ratio * (float)ox, gy = y_ratio * (float)oy;
    const int x = (int)gx, y = (int)gy;
    const float xd = gx - (float)x, yd = gy - (float)y;
    const int x1 = x + 1 < (int)a.in_w ? x + 1 : x, y1 = y + 1 < (int)a.in_h ? y + 1 : y;
    const uint8_t* r0 = a.src + (size_t)y * a.in_stride;
    const uint8_t* r1 = a.src + (size_t)y1 * a.in_stride;
    const size_t np = (size_t)a.out_w * a.out_h, pix = (size_t)oy * a.out_w + ox;
    for (int c = 0; c < 3; ++c) {
        float v = ((float)r0[x * a.bpp + c] * (1.0f - xd)) * (1.0f - yd);
        v = v + ((float)r0[x1 * a.bpp + c] * xd) * (1.0f - yd);
        v = v + ((float)r1[x * a.bpp + c] * (1.0f - xd)) * yd;
        v = v + ((float)r1[x1 * a.bpp + c] * xd) * yd;
        a.dst[c * np + pix] = tk_divf(v * scale - a.mean[c], a.std_dev[c]);
    }
}

static tk_error_code_t launch_status() { return hipGetLastError() == hipSuccess ? TK_SUCCESS : TK_ERROR_GPU_KERNEL_LAUNCH; }

extern "C" {

tk_error_code_t tk_kernels_preprocess_image(const tk_preprocess_params_t* p, tk_hip_stream_t stream) {
    if (!p || !p->d_input_image || !p->d_output_tensor || p->output_width == 0 || p->output_height == 0) return TK_ERROR_INVALID_ARGUMENT;
    if (p->input_width < 2 || p->input_height < 2 || p->input_stride_bytes < p->input_width * 3) return TK_ERROR_INVALID_ARGUMENT;
    TkPreprocessArgs a{};
    a.src = p->d_input_image; a.in_w = p->input_width; a.in_h = p->input_height; a.in_stride = p->input_stride_bytes; a.bpp = 3;
    a.dst = p->d_output_tensor; a.out_w = p->output_width; a.out_h = p->output_height; a.nhwc = 0;
    a.mean[0] = p->mean.x; a.mean[1] = p->mean.y; a.mean[2] = p->mean.z;
    a.std_dev[0] = p->std_dev.x; a.std_dev[1] = p->std_dev.y; a.std_dev[2] = p->std_dev.z;
    if (p->scale == 1.0f / 255.0f || p->scale == 0.0f) tk_launch_preprocess(a, (hipStream_t)stream);
    else hipLaunchKernelGGL(k_preprocess_scaled, dim3((a.out_w + 63) / 64, (a.out_h + 3) / 4), dim3(64, 4), 0, (hipStream_t)stream, a, p->scale);
    return launch_status();
}

tk_error_code_t tk_kernels_preprocess_image_generic(const tk_preprocess_params_generic_t* g, tk_hip_stream_t stream) {
    if (!g) return TK_ERROR_INVALID_ARGUMENT;
    tk_preprocess_params_t p;
    p.d_input_image = (const unsigned char*)g->d_input_image; p.input_width = g->input_width; p.input_height = g->input_height;
    p.input_stride_bytes = g->input_stride_bytes; p.d_output_tensor = (float*)g->d_output_tensor; p.output_width = g->output_width;
    p.output_height = g->output_height; p.mean = tk_float3{g->mean.x, g->mean.y, g->mean.z}; p.std_dev = tk_float3{g->std_dev.x, g->std_dev.y, g->std_dev.z};
    p.scale = 1.0f / 255.0f;
    return tk_kernels_preprocess_image(&p, stream);
}

tk_error_code_t tk_kernels_postprocess_depth_map(const tk_postprocess_depth_params_t* p, tk_hip_stream_t stream) {
    if (!p || !p->d_raw_depth_map || !p->d_metric_depth_map || p->width == 0 || p->height == 0) return TK_ERROR_INVALID_ARGUMENT;
    const size_t n = (size_t)p->width * p->height;
    size_t blocks = (n + 255) / 256;
    if (blocks > 2048) blocks = 2048;
    hipLaunchKernelGGL(k_postprocess_depth, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, *p);
    return launch_status();
}

tk_error_code_t tk_kernels_softmax(const tk_softmax_params_t* p, tk_hip_stream_t stream) {
    if (!p || !p->d_input_tensor || !p->d_output_tensor || p->num_rows == 0 || p->num_cols == 0) return TK_ERROR_INVALID_ARGUMENT;
    if (p->d_output_tensor != p->d_input_tensor &&
        hipMemcpyAsync(p->d_output_tensor, p->d_input_tensor, (size_t)p->num_rows * p->num_cols * sizeof(float), hipMemcpyDeviceToDevice,
                       (hipStream_t)stream) != hipSuccess)
        return TK_ERROR_GPU_ROCM_ERROR;
    tk_launch_softmax_rows((float*)p->d_output_tensor, (int)p->num_rows, (int)p->num_cols, (int)p->num_cols, (hipStream_t)stream);
    return launch_status();
}

tk_error_code_t tk_mi355x_gemm_pair(int device, int M, int N, int K, const float* a, const float* w, const float* bias, const float* residual, int act,
                                    int f16, float* c_staged, float* c_tiled) {
    if (M <= 0 || N <= 0 || K <= 0 || K % 128 || !a || !w || !c_staged || !c_tiled || act < 0 || act > 3) return TK_ERROR_INVALID_ARGUMENT;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) return TK_ERROR_GPU_DEVICE_NOT_FOUND;
    if (device < 0 || device >= n || hipSetDevice(device) != hipSuccess) return TK_ERROR_INVALID_ARGUMENT;
    if (!tk_nn_prepare_device() || !tk_gemm_tiled_prepare_device()) return TK_ERROR_GPU_ROCM_ERROR;
    const size_t na = (size_t)M * K, nw = (size_t)N * K, nc = (size_t)M * N;
    const int64_t blk = M >= 256 ? 256 : (M > 128 ? 256 : M > 64 ? 128 : M > 32 ? 64 : M > 16 ? 32 : 16);
    const size_t nimg = (size_t)(((int64_t)M + blk - 1) / blk * blk) * K;
    float *da = nullptr, *dw = nullptr, *db = nullptr, *dr = nullptr, *dc = nullptr, *dimg = nullptr;
    uint16_t* dwh = nullptr;
    uint8_t* dt = nullptr;
    bool ok = hipMalloc((void**)&da, na * 4) == hipSuccess && hipMalloc((void**)&dw, nw * 4) == hipSuccess && hipMalloc((void**)&dc, nc * 4) == hipSuccess &&
              hipMalloc((void**)&dimg, nimg * 4) == hipSuccess && hipMalloc((void**)&dt, tk_tiled_weight_bytes(N, K, f16 ? 2 : 4)) == hipSuccess &&
              (!bias || hipMalloc((void**)&db, (size_t)N * 4) == hipSuccess) && (!residual || hipMalloc((void**)&dr, nc * 4) == hipSuccess) &&
              (!f16 || hipMalloc((void**)&dwh, nw * 2) == hipSuccess);
    ok = ok && hipMemcpy(da, a, na * 4, hipMemcpyHostToDevice) == hipSuccess && hipMemcpy(dw, w, nw * 4, hipMemcpyHostToDevice) == hipSuccess &&
         (!bias || hipMemcpy(db, bias, (size_t)N * 4, hipMemcpyHostToDevice) == hipSuccess) &&
         (!residual || hipMemcpy(dr, residual, nc * 4, hipMemcpyHostToDevice) == hipSuccess) && hipMemset(dimg, 0, nimg * 4) == hipSuccess;
    if (ok) {
        std::vector<uint16_t> wh;
        if (f16) { /* the f16 checkpoint's weights; the staged kernel reads the same values through its f16 B operand */
            wh.resize(nw);
            for (size_t i = 0; i < nw; ++i) wh[i] = tk_f32_to_f16(w[i]);
            ok = hipMemcpy(dwh, wh.data(), nw * 2, hipMemcpyHostToDevice) == hipSuccess;
        }
        /* staged kernel: with f16 the activations must already be f16-rounded values, as the LLM's producers write them */
        std::vector<float> ar;
        if (ok && f16) {
            ar.resize(na);
            for (size_t i = 0; i < na; ++i) ar[i] = tk_f16_to_f32(tk_f32_to_f16(a[i]));
            ok = hipMemcpy(da, ar.data(), na * 4, hipMemcpyHostToDevice) == hipSuccess;
        }
        if (ok) {
            TkGemm g{};
            g.A = da; g.B = f16 ? (const float*)dwh : dw; g.C = dc; g.bias = db; g.residual = dr;
            g.M = M; g.N = N; g.K = K; g.lda = K; g.ldb = K; g.ldc = N; g.ldr = N; g.act = act; g.alpha = 1.0f; g.batch = 1; g.b_f16 = f16 ? 1 : 0;
            tk_launch_gemm(g, nullptr);
            ok = hipMemcpy(c_staged, dc, nc * 4, hipMemcpyDeviceToHost) == hipSuccess && hipMemset(dc, 0, nc * 4) == hipSuccess;
        }
        if (ok) {
            tk_launch_tile_weights(f16 ? (const void*)dwh : (const void*)dw, f16 ? 2 : 4, N, K, dt, nullptr);
            tk_launch_pack_a(da, M, K, K, 0, dimg, nullptr); /* da already holds the f16-rounded values in the f16 case */
            TkTiledGemm t{};
            t.tiles[0] = dt; t.row_tiles[0] = (N + 15) / 16; t.nseg = 1; t.wbytes = f16 ? 2 : 4;
            t.K = K; t.ks = 1; t.ldc = N; t.n_valid = N; t.nrows = M; t.a_img = dimg; t.a_ts = (size_t)K * 16; t.out = dc;
            t.bias = db; t.residual = dr; t.ldr = N; t.act = act; t.add_zero_bias = 1;
            ok = tk_launch_gemm_tiled(t, nullptr) && hipGetLastError() == hipSuccess && hipMemcpy(c_tiled, dc, nc * 4, hipMemcpyDeviceToHost) == hipSuccess;
        }
    }
    void* ptrs[] = {da, dw, db, dr, dc, dimg, dwh, dt};
    for (void* q : ptrs) if (q) (void)hipFree(q);
    return ok ? TK_SUCCESS : TK_ERROR_GPU_ROCM_ERROR;
}

/* false: sizes that do not belong together */
static bool gemm_f32_sizes(TkGemm& g, int M, int N, int K, int lda, int ldb, const int* conv) {
    if (M <= 0 || N <= 0 || K <= 0 || ldb < K || (!conv && lda < K)) return false;
    g.M = M; g.N = N; g.K = K; g.lda = lda; g.ldb = ldb; g.ldc = N; g.ldr = N; g.alpha = 1.0f; g.batch = 1;
    if (!conv) return true;
    for (int i = 0; i < 9; ++i)
        if (conv[i] < (i == 6 ? 0 : 1) || conv[i] > 16384) return false;
    g.im_C = conv[0]; g.im_H = conv[1]; g.im_W = conv[2]; g.im_ldx = conv[3]; g.im_kw = conv[4]; g.im_stride = conv[5]; g.im_pad = conv[6]; g.im_Ho = conv[7]; g.im_Wo = conv[8];
    /* taps of the last output pixel that lie inside the image: nothing else is read */
    return g.im_C % 4 == 0 && g.im_ldx % 4 == 0 && g.im_ldx >= g.im_C && (int64_t)K == (int64_t)g.im_kw * g.im_kw * g.im_C && ldb % 4 == 0 && M % (g.im_Ho * g.im_Wo) == 0;
}

tk_error_code_t tk_mi355x_gemm_f32(int device, int form, int M, int N, int K, int lda, int ldb, const float* a, const float* w, const float* bias, const float* residual, int act,
                                   const int conv[9], float* c) {
    TkGemm g{};
    if (!a || !w || !c || act < 0 || act > 3 || !gemm_f32_sizes(g, M, N, K, lda, ldb, conv) || !tk_gemm_form_takes(g, form)) return TK_ERROR_INVALID_ARGUMENT;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) return TK_ERROR_GPU_DEVICE_NOT_FOUND;
    if (device < 0 || device >= n || hipSetDevice(device) != hipSuccess) return TK_ERROR_INVALID_ARGUMENT;
    const size_t na = conv ? (size_t)(M / (g.im_Ho * g.im_Wo)) * g.im_H * g.im_W * g.im_ldx : (size_t)M * lda, nw = (size_t)N * ldb, nc = (size_t)M * N;
    float *da = nullptr, *dw = nullptr, *db = nullptr, *dr = nullptr, *dc = nullptr;
    auto put = [](float** d, const float* h, size_t n) { return hipMalloc((void**)d, n * 4) == hipSuccess && hipMemcpy(*d, h, n * 4, hipMemcpyHostToDevice) == hipSuccess; };
    bool ok = tk_nn_prepare_device() && put(&da, a, na) && put(&dw, w, nw) && (!bias || put(&db, bias, N)) && (!residual || put(&dr, residual, nc)) &&
              hipMalloc((void**)&dc, nc * 4) == hipSuccess;
    if (ok) {
        g.A = da; g.B = dw; g.C = dc; g.bias = db; g.residual = dr; g.act = act;
        tk_launch_gemm_form(g, form, nullptr);
        ok = hipGetLastError() == hipSuccess && hipMemcpy(c, dc, nc * 4, hipMemcpyDeviceToHost) == hipSuccess;
    }
    float* ptrs[] = {da, dw, db, dr, dc};
    for (float* q : ptrs) if (q) (void)hipFree(q);
    return ok ? TK_SUCCESS : TK_ERROR_GPU_ROCM_ERROR;
}

tk_error_code_t tk_mi355x_gemm_f32_form(int M, int N, int K, int lda, int ldb, int batch, const int conv[9], int* form, int block[2]) {
    TkGemm g{};
    if (!form || !block || batch < 1 || (conv && batch > 1) || !gemm_f32_sizes(g, M, N, K, lda, ldb, conv)) return TK_ERROR_INVALID_ARGUMENT;
    g.batch = batch; g.sA = (int64_t)M * lda; g.sB = (int64_t)N * ldb; g.sC = (int64_t)M * N;
    *form = tk_gemm_f32_form(g, block);
    return TK_SUCCESS;
}

tk_error_code_t tk_mi355x_conv_direct(int device, const int shape[15], const int* cut, const float* x0, const float* x1, const float* w, const float* bias, const float* residual,
                                      float* y, int* used) {
    if (!shape || !x0 || !w || !y) return TK_ERROR_INVALID_ARGUMENT;
    for (int i = 0; i < 15; ++i)
        if (shape[i] < 0 || shape[i] > 16384) return TK_ERROR_INVALID_ARGUMENT;
    TkConvDirect c{};
    c.B = shape[0]; c.H = shape[1]; c.W = shape[2]; c.C = shape[3]; c.c_split = shape[7] > 0 ? shape[4] : c.C;
    c.k = shape[9]; c.stride = shape[10]; c.pad = c.k / 2; c.N = shape[11]; c.ldy = shape[12]; c.ldr = shape[13]; c.act = shape[14];
    if (c.stride < 1 || c.H < 1 || c.W < 1 || c.B < 1 || c.C < 16 || c.N < 1 || c.c_split > c.C || c.ldy < c.N || (residual && c.ldr < c.N) || (c.c_split < c.C && !x1) ||
        shape[5] < c.c_split || (c.c_split < c.C && shape[7] < c.C - c.c_split) || shape[6] > 1 || shape[8] > 1)
        return TK_ERROR_INVALID_ARGUMENT;
    c.Ho = (c.H + 2 * c.pad - c.k) / c.stride + 1; c.Wo = (c.W + 2 * c.pad - c.k) / c.stride + 1;
    const size_t pixels = (size_t)c.B * c.H * c.W, outs = (size_t)c.B * c.Ho * c.Wo, K = (size_t)c.k * c.k * c.C;
    const size_t n0 = (pixels >> (2 * shape[6])) * shape[5], n1 = c.c_split < c.C ? (pixels >> (2 * shape[8])) * shape[7] : 0;
    c.src[0] = TkConvSource{x0, shape[5], shape[6]}; c.src[1] = TkConvSource{x1, shape[7], shape[8]};
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) return TK_ERROR_GPU_DEVICE_NOT_FOUND;
    if (device < 0 || device >= n || hipSetDevice(device) != hipSuccess) return TK_ERROR_INVALID_ARGUMENT;
    float *d0 = nullptr, *d1 = nullptr, *dw = nullptr, *dp = nullptr, *db = nullptr, *dr = nullptr, *dy = nullptr;
    auto put = [](float** d, const float* h, size_t n) { return hipMalloc((void**)d, n * 4) == hipSuccess && hipMemcpy(*d, h, n * 4, hipMemcpyHostToDevice) == hipSuccess; };
    bool ok = put(&d0, x0, n0) && (n1 == 0 || put(&d1, x1, n1)) && put(&dw, w, K * c.N) && (!bias || put(&db, bias, c.N)) && (!residual || put(&dr, residual, outs * c.ldr)) &&
              put(&dy, y, outs * c.ldy) && hipMalloc((void**)&dp, tk_conv_weight_floats(c.N, (int)K) * 4) == hipSuccess;
    bool fits = true;
    if (ok) {
        c.src[0].p = d0; c.src[1].p = d1; c.w = dp; c.bias = db; c.residual = dr; c.y = dy;
        TkConvPlan plan{};
        if (cut) plan = TkConvPlan{cut[0], cut[1], cut[2], cut[3], cut[4]};
        fits = tk_conv_direct_takes(c) && (cut || tk_conv_direct_plan(c, &plan)) && tk_conv_plan_ok(c, plan);
        if (fits) {
            tk_launch_conv_weights(dw, c.N, (int)K, dp, nullptr);
            ok = tk_launch_conv_direct(c, plan, nullptr) && hipGetLastError() == hipSuccess && hipMemcpy(y, dy, outs * c.ldy * 4, hipMemcpyDeviceToHost) == hipSuccess;
            if (used) { used[0] = plan.mt; used[1] = plan.wm; used[2] = plan.wn; used[3] = plan.th; used[4] = plan.tw; }
        }
    }
    float* ptrs[] = {d0, d1, dw, dp, db, dr, dy};
    for (float* q : ptrs) if (q) (void)hipFree(q);
    return !fits ? TK_ERROR_INVALID_ARGUMENT : ok ? TK_SUCCESS : TK_ERROR_GPU_ROCM_ERROR;
}

static __global__ __launch_bounds__(256) void k_f32_to_f16(const float* __restrict__ x, int n, uint16_t* __restrict__ bits) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) bits[i] = tk_f32_to_f16(x[i]);
}

tk_error_code_t tk_mi355x_f32_to_f16(int device, const float* x, int n, uint16_t* bits) {
    if (!x || !bits || n < 1 || n > 1 << 28) return TK_ERROR_INVALID_ARGUMENT;
    int have = 0;
    if (hipGetDeviceCount(&have) != hipSuccess || have <= 0) return TK_ERROR_GPU_DEVICE_NOT_FOUND;
    if (device < 0 || device >= have || hipSetDevice(device) != hipSuccess) return TK_ERROR_INVALID_ARGUMENT;
    float* dx = nullptr;
    uint16_t* db = nullptr;
    bool ok = hipMalloc((void**)&dx, (size_t)n * 4) == hipSuccess && hipMalloc((void**)&db, (size_t)n * 2) == hipSuccess &&
              hipMemcpy(dx, x, (size_t)n * 4, hipMemcpyHostToDevice) == hipSuccess;
    if (ok) {
        hipLaunchKernelGGL(k_f32_to_f16, dim3((n + 255) / 256), dim3(256), 0, nullptr, dx, n, db);
        ok = hipGetLastError() == hipSuccess && hipMemcpy(bits, db, (size_t)n * 2, hipMemcpyDeviceToHost) == hipSuccess;
    }
    if (dx) (void)hipFree(dx);
    if (db) (void)hipFree(db);
    return ok ? TK_SUCCESS : TK_ERROR_GPU_ROCM_ERROR;
}

tk_error_code_t tk_mi355x_gemm_image(int device, int f32, int rows, int N, int K, int max_slabs, const float* x, const float* w, float* out, int* slabs) {
    if (rows < 1 || N < 1 || K < 1 || rows > 16384 || N > 65536 || K > 65536 || max_slabs < 1 || max_slabs > 8 || !x || !w || !out || !slabs) return TK_ERROR_INVALID_ARGUMENT;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) return TK_ERROR_GPU_DEVICE_NOT_FOUND;
    if (device < 0 || device >= n || hipSetDevice(device) != hipSuccess) return TK_ERROR_INVALID_ARGUMENT;
    const int type = f32 ? TK_IMG_F32 : TK_IMG_BF16, kp = tk_img_pad_k(type, K), np = (N + 15) / 16 * 16;
    const size_t slab = ((size_t)rows * N + 3) / 4 * 4;
    TkImgGemm g{};
    g.type = type; g.K = kp; g.N = np; g.nrows = rows; g.ldc = g.n_valid = N; g.max_slabs = max_slabs; g.slab_floats = slab;
    float *dx = nullptr, *dw = nullptr, *dy = nullptr;
    void *ix = nullptr, *iw = nullptr;
    auto put = [](float** d, const float* h, size_t n) { return hipMalloc((void**)d, n * 4) == hipSuccess && hipMemcpy(*d, h, n * 4, hipMemcpyHostToDevice) == hipSuccess; };
    auto image = [&](void** img, const float* src, int64_t r) {
        const size_t bytes = tk_img_bytes(type, r, K);
        if (hipMalloc(img, bytes) != hipSuccess || hipMemset(*img, 0, bytes) != hipSuccess) return false;
        tk_launch_put_image(type, src, 1, r, K, *img, kp / tk_img_kt(type), 0, 0, -1, nullptr);
        return hipGetLastError() == hipSuccess;
    };
    bool ok = put(&dx, x, (size_t)rows * K) && put(&dw, w, (size_t)N * K) && image(&ix, dx, rows) && image(&iw, dw, N) &&
              hipMalloc((void**)&dy, slab * max_slabs * 4) == hipSuccess && !tk_gemm_image_prepare_device();
    if (ok) {
        g.w = iw; g.a = ix; g.out = dy;
        ok = !tk_launch_gemm_image(g, nullptr, slabs) && hipGetLastError() == hipSuccess && hipDeviceSynchronize() == hipSuccess;
        for (int i = 0; ok && i < *slabs; ++i) ok = hipMemcpy(out + (size_t)i * rows * N, dy + i * slab, (size_t)rows * N * 4, hipMemcpyDeviceToHost) == hipSuccess;
    }
    void* ptrs[] = {dx, dw, dy, ix, iw};
    for (void* q : ptrs) if (q) (void)hipFree(q);
    return ok ? TK_SUCCESS : TK_ERROR_GPU_ROCM_ERROR;
}

tk_error_code_t tk_mi355x_gemm_image_form(int f32, int rows, int N, int K, int swiglu, int experts, int top, int max_slabs, int form[4]) {
    if (rows <= 0 || N <= 0 || K <= 0 || experts < 0 || (experts > 0 && (top < 1 || top > experts)) || !form) return TK_ERROR_INVALID_ARGUMENT;
    const int to = swiglu ? 32 : 16;
    TkImgGemm g{};
    g.type = f32 ? TK_IMG_F32 : TK_IMG_BF16; g.K = tk_img_pad_k(g.type, K); g.N = (N + to - 1) / to * to; g.n_valid = N; g.nrows = rows; g.swiglu = swiglu != 0; g.max_slabs = max_slabs;
    if (experts) tk_img_expert_blocks(rows, rows, top, experts, &g);
    tk_gemm_image_form(g, form);
    return TK_SUCCESS;
}

tk_error_code_t tk_kernels_depth_to_point_cloud(const tk_depth_to_points_params_t* p, tk_hip_stream_t stream) {
    if (!p || !p->d_metric_depth_map || !p->d_point_cloud || p->width == 0 || p->height == 0 || p->fx == 0.0f || p->fy == 0.0f)
        return TK_ERROR_INVALID_ARGUMENT;
    const size_t n = (size_t)p->width * p->height;
    size_t blocks = (n + 255) / 256;
    if (blocks > 2048) blocks = 2048;
    hipLaunchKernelGGL(k_depth_to_points, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, *p);
    return launch_status();
}

tk_error_code_t tk_rocm_dispatch_create(tk_rocm_dispatcher_t** out, const tk_rocm_dispatcher_config_t* config) {
    if (!out || !config) return TK_ERROR_INVALID_ARGUMENT;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) return TK_ERROR_GPU_DEVICE_NOT_FOUND;
    if (config->device_id < 0 || config->device_id >= n) return TK_ERROR_INVALID_ARGUMENT;
    tk_rocm_dispatcher_s* d = (tk_rocm_dispatcher_s*)calloc(1, sizeof *d);
    if (!d) return TK_ERROR_OUT_OF_MEMORY;
    d->device = config->device_id;
    if (hipSetDevice(d->device) != hipSuccess || hipStreamCreateWithFlags(&d->compute, hipStreamNonBlocking) != hipSuccess ||
        hipStreamCreateWithFlags(&d->h2d, hipStreamNonBlocking) != hipSuccess || hipStreamCreateWithFlags(&d->d2h, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreateWithFlags(&d->ev_upload, hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&d->ev_compute, hipEventDisableTiming) != hipSuccess) {
        free(d);
        return TK_ERROR_GPU_ROCM_ERROR;
    }
    *out = d;
    return TK_SUCCESS;
}

void tk_rocm_dispatch_destroy(tk_rocm_dispatcher_t** dispatcher) {
    if (!dispatcher || !*dispatcher) return;
    tk_rocm_dispatcher_s* d = *dispatcher;
    (void)hipSetDevice(d->device);
    (void)hipDeviceSynchronize();
    (void)hipStreamDestroy(d->compute); (void)hipStreamDestroy(d->h2d); (void)hipStreamDestroy(d->d2h);
    (void)hipEventDestroy(d->ev_upload); (void)hipEventDestroy(d->ev_compute);
    free(d);
    *dispatcher = NULL;
}

tk_error_code_t tk_rocm_dispatch_malloc(tk_rocm_dispatcher_t* d, tk_gpu_buffer_t* out_buffer, size_t size_bytes) {
    if (!d || !out_buffer || size_bytes == 0) return TK_ERROR_INVALID_ARGUMENT;
    if (hipSetDevice(d->device) != hipSuccess) return TK_ERROR_GPU_ROCM_ERROR;
    tk_gpu_buffer_s* b = (tk_gpu_buffer_s*)calloc(1, sizeof *b);
    if (!b) return TK_ERROR_OUT_OF_MEMORY;
    if (hipMalloc(&b->dptr, size_bytes) != hipSuccess) { free(b); return TK_ERROR_GPU_MEMORY; }
    b->size = size_bytes;
    *out_buffer = b;
    return TK_SUCCESS;
}

void tk_rocm_dispatch_free(tk_rocm_dispatcher_t* d, tk_gpu_buffer_t* buffer) {
    if (!d || !buffer || !*buffer) return;
    (void)hipSetDevice(d->device);
    (void)hipFree((*buffer)->dptr);
    free(*buffer);
    *buffer = NULL;
}

void* tk_rocm_dispatch_buffer_ptr(tk_gpu_buffer_t buffer) { return buffer ? buffer->dptr : NULL; }

tk_error_code_t tk_rocm_dispatch_upload_async(tk_rocm_dispatcher_t* d, tk_gpu_buffer_t dst, const void* src, size_t n) {
    if (!d || !dst || !src || n > dst->size) return TK_ERROR_INVALID_ARGUMENT;
    if (hipSetDevice(d->device) != hipSuccess) return TK_ERROR_GPU_ROCM_ERROR;
    if (hipMemcpyAsync(dst->dptr, src, n, hipMemcpyHostToDevice, d->h2d) != hipSuccess) return TK_ERROR_GPU_MEMORY;
    /* kernels enqueued afterwards must see the data */
    if (hipEventRecord(d->ev_upload, d->h2d) != hipSuccess || hipStreamWaitEvent(d->compute, d->ev_upload, 0) != hipSuccess) return TK_ERROR_GPU_ROCM_ERROR;
    return TK_SUCCESS;
}

tk_error_code_t tk_rocm_dispatch_download_async(tk_rocm_dispatcher_t* d, void* dst, tk_gpu_buffer_t src, size_t n) {
    if (!d || !dst || !src || n > src->size) return TK_ERROR_INVALID_ARGUMENT;
    if (hipSetDevice(d->device) != hipSuccess) return TK_ERROR_GPU_ROCM_ERROR;
    if (hipEventRecord(d->ev_compute, d->compute) != hipSuccess || hipStreamWaitEvent(d->d2h, d->ev_compute, 0) != hipSuccess) return TK_ERROR_GPU_ROCM_ERROR;
    if (hipMemcpyAsync(dst, src->dptr, n, hipMemcpyDeviceToHost, d->d2h) != hipSuccess) return TK_ERROR_GPU_MEMORY;
    return TK_SUCCESS;
}

tk_error_code_t tk_rocm_dispatch_synchronize(tk_rocm_dispatcher_t* d) {
    if (!d) return TK_ERROR_INVALID_ARGUMENT;
    if (hipSetDevice(d->device) != hipSuccess) return TK_ERROR_GPU_ROCM_ERROR;
    if (hipStreamSynchronize(d->h2d) != hipSuccess || hipStreamSynchronize(d->compute) != hipSuccess || hipStreamSynchronize(d->d2h) != hipSuccess)
        return TK_ERROR_GPU_ROCM_ERROR;
    return TK_SUCCESS;
}

tk_error_code_t tk_rocm_dispatch_get_stream(tk_rocm_dispatcher_t* d, tk_hip_stream_t* stream) {
    if (!d || !stream) return TK_ERROR_INVALID_ARGUMENT;
    *stream = (tk_hip_stream_t)d->compute;
    return TK_SUCCESS;
}

tk_error_code_t tk_rocm_dispatch_preprocess_image(tk_rocm_dispatcher_t* d, const tk_preprocess_params_t* params) {
    if (!d) return TK_ERROR_INVALID_ARGUMENT;
    if (hipSetDevice(d->device) != hipSuccess) return TK_ERROR_GPU_ROCM_ERROR;
    return tk_kernels_preprocess_image(params, (tk_hip_stream_t)d->compute);
}

tk_error_code_t tk_rocm_dispatch_depth_to_point_cloud(tk_rocm_dispatcher_t* d, const tk_depth_to_points_params_t* params) {
    if (!d) return TK_ERROR_INVALID_ARGUMENT;
    if (hipSetDevice(d->device) != hipSuccess) return TK_ERROR_GPU_ROCM_ERROR;
    return tk_kernels_depth_to_point_cloud(params, (tk_hip_stream_t)d->compute);
}

} /* extern "C" */
