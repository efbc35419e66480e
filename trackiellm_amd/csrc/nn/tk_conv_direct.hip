/* tk_conv_direct.hip — see tk_conv_direct.h */
#include "tk_conv_direct.h"

#include <algorithm>
#include <atomic>
#include <math.h>
#include <mutex>

#include "../common/tk_exact_math.h"
#include "../common/tk_gemm_desc.h"

typedef float v4f __attribute__((ext_vector_type(4)));
typedef int v4i __attribute__((ext_vector_type(4)));

#define TK_CD_LDS 163840 /* bytes a workgroup may have */
#define TK_CD_MAX_WAVES 8
#define TK_CD_MAX_PF 8
#define TK_CD_TABLE_PAD 16 /* entries behind the last group: operands and entries are read ahead */

/* n / d by one multiplication, for n d < 2^31: by = ceil(2^31 / d) */
static uint32_t cd_div(int d) { return (uint32_t)((0x80000000ull + (uint32_t)d - 1) / (uint32_t)d); }
__device__ __forceinline__ int cd_quot(int n, uint32_t by) { return (int)__umulhi(2u * (uint32_t)n, by); }

struct CdArgs {
    TkConvDirect c;
    int wn, th, tw, pw, ph;      /* waves along channels; tile; patch */
    int vec;                     /* output, residual: four channels of a pixel are an aligned 16 bytes */
    int tiles_x, tiles;          /* spatial tiles of a row, of an image */
    int cp4;                     /* float4 of a pixel in the LDS: C / 4 + 1 */
    uint32_t by_c4[2], by_pw, by_tw, by_wn, by_cj, by_tiles_x; /* cd_div() of a source's float4 of a pixel, ... */
};

/* up to P convolutions of one batch in a launch: block x counts through the (tile, channel group) pairs of the first, then of the second, ... */
template <int P> struct CdSet {
    int n, first[P];
    uint32_t by_tiles[P];
    CdArgs a[P];
};

template <int V> struct CdCount { static constexpr int value = V; };

/*
 * What bounds it.  Few tiles (one frame): the chain, about 46 cycles an MFMA where the wave has nothing else to issue, behind one trip to memory for the patch and the
 * first weights (40 x 40 x 64, 576 k: 7.0 us, of which 2.8 are the chain; k_gemm_f32_t16 10.4, whose slabs are a trip each).  Many: the fp32 pipe, which vector
 * instructions share: 73 % of it at 80 x 80 x 64 x 32 frames (136 us; the GEMM kernels 162), 60 % at 40 x 40 (41 us; 54), where patches and epilogues are a larger part.
 * Weights come from the L2 once per tile of pixels, operands from the LDS: a padding of 16 bytes a pixel turns 16 pixels into 16 different groups of banks.
 */
template <int P, int MT /* 16-pixel tiles a wave */, int PF /* pieces of weights in flight, even: operands are read a group ahead, into two sets */>
__global__ __launch_bounds__(64 * TK_CD_MAX_WAVES) void k_conv_direct(CdSet<P> set) {
    extern __shared__ __attribute__((aligned(16))) float cd_lds[];
    int pi = 0;
#pragma unroll
    for (int i = 1; i < P; ++i) pi += i < set.n && (int)blockIdx.x >= set.first[i] ? 1 : 0;
    const CdArgs& a = set.a[pi];
    const int local = (int)blockIdx.x - set.first[pi], by = cd_quot(local, set.by_tiles[pi]), bx = local - by * a.tiles;
    const TkConvDirect& c = a.c;
    const int tid = threadIdx.x, nthreads = blockDim.x, lane = tid & 63, r = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = cd_quot(wave, a.by_wn), wn = wave - wm * a.wn;
    const int b = blockIdx.z, ty = cd_quot(bx, a.by_tiles_x), tx = bx - ty * a.tiles_x;
    const int oy0 = ty * a.th, ox0 = tx * a.tw;
    const int cj = c.C >> 4, G = c.k * c.k * cj; /* 16-k groups: of a tap, in all */
    const int ntile = by * a.wn + wn;
    const bool active = ntile * 16 < c.N;

    /* the first weights travel under the patch; requests past the chain read what lies behind it (tk_conv_weight_floats) */
    const char* wp = (const char*)c.w + (size_t)(active ? ntile : 0) * G * 1024;
    v4f w[PF];
#pragma unroll
    for (int i = 0; i < PF; ++i) w[i] = *(const v4f*)(wp + (size_t)i * 1024 + lane * 16);

    /* where the operands of a group lie, bytes from the tile's own pixel (past the chain: its last group).  A lone wave issues an instruction every
     * five cycles, four MFMAs take 160: counters of taps and channels beside them cost as much as the chain */
    const v4i* table = (const v4i*)(cd_lds + (size_t)a.ph * a.pw * a.cp4 * 4);
    for (int q = tid; q < G + TK_CD_TABLE_PAD; q += nthreads) {
        const int qq = q < G ? q : G - 1, tap = cd_quot(qq, a.by_cj), ky = c.k == 3 ? (tap * 11) >> 5 : 0, kx = tap - ky * c.k;
        ((int*)table)[q] = (ky * a.pw + kx) * a.cp4 * 16 + (qq - tap * cj) * 64;
    }
    { /* patch, source by source: float4 e = (pixel, four channels); channel 4 t + g of a 16-group goes to place 4 g + t */
        const int iy0 = oy0 * c.stride - c.pad, ix0 = ox0 * c.stride - c.pad;
#pragma unroll 1
        for (int si = 0; si < (c.c_split < c.C ? 2 : 1); ++si) {
            const TkConvSource& s = c.src[si];
            const int c4 = (si == 0 ? c.c_split : c.C - c.c_split) >> 2, total = a.ph * a.pw * c4, sh = s.shift;
            const int hs = c.H >> sh, ws = c.W >> sh, H = c.H, W = c.W, pw = a.pw, cp4 = a.cp4;
            const uint32_t ld = (uint32_t)s.ld, by_pw = a.by_pw;
            const uint32_t by_c4 = a.by_c4[si];
            const float* image = s.p + (int64_t)b * hs * ws * s.ld;
            float* to = cd_lds + (si == 0 ? 0 : c.c_split);
            auto batch = [&](auto count, int e0) { /* past the end: the last float4 again */
                constexpr int U = decltype(count)::value;
                v4f v[U];
                int at[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    int e = e0 + u * nthreads + tid;
                    e = e < total ? e : total - 1;
                    const int pix = cd_quot(e, by_c4), q = e - __mul24(pix, c4);
                    const int py = cd_quot(pix, by_pw), px = pix - __mul24(py, pw);
                    const int iy = iy0 + py, ix = ix0 + px;
                    const bool in = (int)((uint32_t)iy < (uint32_t)H) & (int)((uint32_t)ix < (uint32_t)W);
                    const uint32_t off = ((uint32_t)((iy >> sh) * ws + (ix >> sh)) * ld + 4u * (uint32_t)q) & (0u - (uint32_t)in); /* outside: the first value, not used */
                    const v4f t = *(const v4f*)((const char*)image + off * 4u);
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[u][i] = in ? t[i] : 0.0f;
                    at[u] = (__mul24(pix, cp4) + (q & ~3)) * 4 + (q & 3);
                }
#pragma unroll
                for (int u = 0; u < U; ++u)
#pragma unroll
                    for (int i = 0; i < 4; ++i) to[at[u] + 4 * i] = v[u][i];
            };
            int e0 = 0;
            for (; total - e0 > 4 * nthreads; e0 += 8 * nthreads) batch(CdCount<8>{}, e0);
            if (total - e0 > 2 * nthreads) batch(CdCount<4>{}, e0);
            else if (total - e0 > 0) batch(CdCount<2>{}, e0);
        }
    }
    __syncthreads();
    if (!active) return;

    const char* base[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int p = (wm * MT + m) * 16 + r, pp = p < a.th * a.tw ? p : 0;
        const int py = cd_quot(pp, a.by_tw), px = pp - py * a.tw;
        base[m] = (const char*)cd_lds + ((py * a.pw + px) * c.stride * a.cp4 + g) * 16;
    }
    v4f acc[MT], op[2][MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    auto read = [&](int set, int at) {
#pragma unroll
        for (int m = 0; m < MT; ++m) op[set][m] = *(const v4f*)(base[m] + at);
    };
    auto group = [&](int u, int next) { /* operand set u % 2, weights w[u]; next: where the next group's operands lie */
        read((u + 1) % 2, next);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int m = 0; m < MT; ++m) acc[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[u][t], op[u % 2][m][t], acc[m], 0, 0, 0);
    };
    int q = 0;
    v4i at = table[0], at_next = table[1];
    read(0, at[0]);
    for (; q + PF <= G; q += PF) {
#pragma unroll
        for (int u = 0; u < PF; ++u) {
            const int next = at[(u + 1) & 3];
            if (((u + 1) & 3) == 3) { at = at_next; at_next = table[(q + u + 6) >> 2]; }
            group(u, next);
            w[u] = *(const v4f*)(wp + (size_t)(q + u + PF) * 1024 + lane * 16);
        }
    }
#pragma unroll
    for (int u = 0; u < PF - 1; ++u)
        if (q + u < G) {
            const int next = at[(u + 1) & 3];
            if (((u + 1) & 3) == 3) { at = at_next; at_next = table[(q + u + 6) >> 2]; }
            group(u, next);
        }

    /* The weights are the rows of the MFMAs, so that a lane ends with four channels, 4 g .. 4 g + 3, of one pixel, r, of a tile: an address and a store instead of four, where
     * vector instructions share the pipe */
    const int n = ntile * 16 + 4 * g;
    if (n >= c.N) return;
    const bool silu = c.act == TK_ACT_SILU;
    float bias[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) bias[i] = c.bias && n + i < c.N ? c.bias[n + i] : 0.0f;
    const int64_t image = (int64_t)b * c.Ho * c.Wo;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int p = (wm * MT + m) * 16 + r;
        const int py = cd_quot(p, a.by_tw), px = p - py * a.tw;
        const int oy = oy0 + py, ox = ox0 + px;
        if (py >= a.th || oy >= c.Ho || ox >= c.Wo) continue;
        const int64_t pix = image + oy * c.Wo + ox;
        float* y = c.y + pix * c.ldy + n;
        const float* res = c.residual ? c.residual + pix * c.ldr + n : nullptr;
        v4f before = {0.0f, 0.0f, 0.0f, 0.0f};
        if (res && a.vec) before = *(const v4f*)res;
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = acc[m][i] + bias[i];
        if (silu) tk_silu_all<4>(v);
        if (a.vec) {
            v4f o;
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = res ? v[i] + before[i] : v[i];
            *(v4f*)y = o;
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (n + i < c.N) y[i] = res ? v[i] + res[i] : v[i];
        }
    }
}

__global__ void k_conv_weights(const float* w, int N, int K, float* pieces) {
    const int lane = threadIdx.x, j = blockIdx.x, nt = blockIdx.y, n = nt * 16 + (lane & 15), g = lane >> 4;
    float* dst = pieces + (((size_t)nt * (K >> 4) + j) * 64 + lane) * 4;
#pragma unroll
    for (int t = 0; t < 4; ++t) dst[t] = n < N ? w[(size_t)n * K + 16 * j + 4 * t + g] : 0.0f;
}

/* and the pieces that are requested past the last chain */
size_t tk_conv_weight_floats(int N, int K) { return (size_t)((N + 15) / 16 * 16) * (size_t)K + TK_CD_MAX_PF * 256; }
void tk_launch_conv_weights(const float* w, int N, int K, float* pieces, hipStream_t s) {
    hipLaunchKernelGGL(k_conv_weights, dim3(K / 16, (N + 15) / 16), dim3(64), 0, s, w, N, K, pieces);
}

bool tk_conv_direct_takes(const TkConvDirect& c) {
    if (c.B < 1 || c.H < 1 || c.W < 1 || c.N < 1 || c.C < 16 || (c.C & 15) || (c.c_split & 15) || c.c_split < 16 || c.c_split > c.C) return false;
    if (!((c.k == 3 && c.pad == 1) || (c.k == 1 && c.pad == 0)) || c.stride < 1 || c.stride > 2) return false;
    if (c.act != TK_ACT_NONE && c.act != TK_ACT_SILU) return false;
    if (c.Ho != (c.H + 2 * c.pad - c.k) / c.stride + 1 || c.Wo != (c.W + 2 * c.pad - c.k) / c.stride + 1) return false;
    if (c.Ho > 32768 || c.Wo > 32768 || c.B > 65535 || (int64_t)c.Ho * c.Wo > (1 << 30)) return false;
    for (int i = 0; i < (c.c_split < c.C ? 2 : 1); ++i) {
        const TkConvSource& s = c.src[i];
        if (!s.p || (((uintptr_t)s.p) & 15) || (s.ld & 3) || s.shift < 0 || s.shift > 1) return false;
        if (s.shift && ((c.H | c.W) & 1)) return false;
        if ((int64_t)c.H * c.W * s.ld >= (1 << 29)) return false; /* 32-bit offsets in an image */
    }
    return c.w && !(((uintptr_t)c.w) & 15) && c.y;
}

static int64_t cd_lds_bytes(const TkConvDirect& c, int ph, int pw) { return (int64_t)ph * pw * (c.C / 4 + 1) * 16 + (c.k * c.k * (c.C / 16) + TK_CD_TABLE_PAD + 3) / 4 * 16; }
static bool cd_fill(const TkConvDirect& c, const TkConvPlan& p, CdArgs* a) {
    if ((p.mt != 1 && p.mt != 2 && p.mt != 4) || p.wm < 1 || p.wn < 1 || p.wm * p.wn > TK_CD_MAX_WAVES || p.th < 1 || p.tw < 1) return false;
    if (p.th * p.tw > 16 * p.mt * p.wm) return false;
    a->c = c;
    auto whole = [](const void* q, int ld) { return !(((uintptr_t)q) & 15) && !(ld & 3); };
    a->vec = !(c.N & 3) && whole(c.y, c.ldy) && whole(c.residual, c.residual ? c.ldr : 0);
    a->wn = p.wn; a->th = p.th; a->tw = p.tw;
    a->ph = (p.th - 1) * c.stride + c.k; a->pw = (p.tw - 1) * c.stride + c.k;
    a->tiles_x = (c.Wo + p.tw - 1) / p.tw;
    a->tiles = a->tiles_x * ((c.Ho + p.th - 1) / p.th);
    a->cp4 = c.C / 4 + 1;
    /* (a patch has fewer than 10240 float4, a divisor is at most 10240) */
    a->by_c4[0] = cd_div(c.c_split / 4); a->by_c4[1] = cd_div(c.c_split < c.C ? (c.C - c.c_split) / 4 : 1);
    a->by_pw = cd_div(a->pw); a->by_tw = cd_div(p.tw); a->by_wn = cd_div(p.wn); a->by_cj = cd_div(c.C / 16); a->by_tiles_x = cd_div(a->tiles_x);
    /* pairs of tile and channel group: their quotients by the tiles too */
    if ((int64_t)a->tiles * ((c.N + 15) / 16) * a->tiles >= 0x7fffffff) return false;
    return cd_lds_bytes(c, a->ph, a->pw) <= TK_CD_LDS;
}
bool tk_conv_plan_ok(const TkConvDirect& c, const TkConvPlan& plan) {
    CdArgs a;
    return tk_conv_direct_takes(c) && cd_fill(c, plan, &a);
}

/* Costs in cycles, fitted to 8 000 launches (the detector's 3 x 3 layers at 1, 8, 24 and 32 frames, every cut): the choice takes 1.1 % more than the best cut in the
 * mean, 9 % at most; at 4, 12 and 16 frames, which were not fitted, 0.5, 1.7 and 2.4 %, the largest 24.  A workgroup's latency is its patch, its chains (32 cycles an MFMA) and
 * its epilogue; the CU's further ones take turns on the pipe, which their vector instructions share, and hide no more of a latency than there are of them: a patch that leaves
 * room for one workgroup is paid whole (64 -> 80 channels of 80 x 80, 32 frames: 246 us with 16 x 16 pixels, 185 with 16 x 8).  Five, six or seven waves load the SIMDs unevenly
 * (the same layer: 247 us with five, 190 with four).  Two, four and five channel tiles a wave, which read the patch once for all of them, are no quicker (1 - 2 % at 80
 * channels) but at 20 x 20 x 256 -> 80 (69 / 56 us).  The layers fitted are those of a network of 640 x 640; whole calls of others, by the GEMM kernels / here before this fit:
 * 320 x 320, 1 and 16 frames 779 / 405, 1914 / 1249 us; 512 x 288, 1 and 6 766 / 418, 1207 / 733; 416 x 416, 2 and 16 847 / 496, 2269 / 1690; 1280 x 736, 1 and 16
 * 1095 / 624, 8167 / 5361. */
static float cd_plan(const TkConvDirect& c, int only_mt, int only_waves, TkConvPlan* plan) {
    const int ntiles = (c.N + 15) / 16;
    const float G = (float)(c.k * c.k * c.C / 16);
    float best = 3e38f;
    const int mts[3] = {1, 2, 4}, wns[5] = {1, 2, 3, 4, 8};
    const int widths[10] = {4, 5, 8, 10, 16, 20, 32, 40, 64, 80};
    for (int wn : wns) {
        if (wn > ntiles) break;
        for (int wm = 1; wm * wn <= TK_CD_MAX_WAVES; wm *= 2) {
            const int w = wm * wn;
            if ((w > 4 && w < 8) || (w < 2 && ntiles > 1) || (only_waves && w != only_waves)) continue;
            for (int mt : mts) {
                if (only_mt && mt != only_mt) continue;
                const int rows = 16 * mt * wm;
                for (int tw0 : widths) {
                    const int tw = tw0 < c.Wo ? tw0 : c.Wo;
                    if (tw > rows) break;
                    const int th = rows / tw < c.Ho ? rows / tw : c.Ho;
                    const int64_t lds = cd_lds_bytes(c, (th - 1) * c.stride + c.k, (tw - 1) * c.stride + c.k);
                    if (lds > TK_CD_LDS) continue;
                    const float rounds = (float)((c.Wo + tw - 1) / tw) * (float)((c.Ho + th - 1) / th) * (float)c.B * (float)((ntiles + wn - 1) / wn) * (1.0f / 256.0f);
                    const int side_by_side = (int)(TK_CD_LDS / lds) < 16 / w ? (int)(TK_CD_LDS / lds) : 16 / w;
                    const float per = (float)((w + 3) / 4 * mt), share = 0.25f * (float)(w * mt), kib = (float)lds * (1.0f / 1024.0f);
                    const float latency = 370.0f + 57.0f * kib + per * (G * 4.0f * 32.0f + 33.0f), work = share * (G * 4.0f * 34.3f + 37.0f) + 9.7f * kib + 79.0f * (float)w;
                    float turns = side_by_side > 1 ? 0.32f * rounds + 0.68f * ceilf(rounds) : ceilf(rounds);
                    turns = turns > 1.0f ? turns - 1.0f : 0.0f;
                    const float alone = latency / (float)side_by_side; /* what is not hidden under the others' */
                    const float cost = latency + turns * (work > alone ? work : alone);
                    if (cost < best) {
                        best = cost;
                        *plan = TkConvPlan{mt, wm, wn, th, tw};
                    }
                }
            }
        }
    }
    return best;
}
bool tk_conv_direct_plan(const TkConvDirect& c, TkConvPlan* plan) { return cd_plan(c, 0, 0, plan) < 3e38f; }
/* one form for all: four waves, the tiles a wave that cost least in the sum */
bool tk_conv_direct_plan_set(const TkConvDirect* c, int n, TkConvPlan* plans) {
    float best = 3e38f;
    for (int mt = 1; mt <= 4; mt *= 2) {
        TkConvPlan p[TK_CONV_SET];
        float sum = 0.0f;
        for (int i = 0; i < n && i < TK_CONV_SET; ++i) sum += cd_plan(c[i], mt, 4, &p[i]);
        if (sum < best) {
            best = sum;
            for (int i = 0; i < n && i < TK_CONV_SET; ++i) plans[i] = p[i];
        }
    }
    return best < 3e38f;
}

static std::atomic<bool> g_cd_opted[64];
static std::mutex g_cd_mu;
bool tk_conv_direct_prepare_device() {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return false;
    if (g_cd_opted[dev].load(std::memory_order_acquire)) return true;
    std::lock_guard<std::mutex> lk(g_cd_mu);
    const void* fns[6] = {(const void*)k_conv_direct<1, 1, 8>, (const void*)k_conv_direct<1, 2, 8>, (const void*)k_conv_direct<1, 4, 4>,
                          (const void*)k_conv_direct<TK_CONV_SET, 1, 8>, (const void*)k_conv_direct<TK_CONV_SET, 2, 8>, (const void*)k_conv_direct<TK_CONV_SET, 4, 4>};
    for (const void* f : fns)
        if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, TK_CD_LDS) != hipSuccess) return false;
    g_cd_opted[dev].store(true, std::memory_order_release);
    return true;
}

template <int P>
static bool cd_launch(const TkConvDirect* c, const TkConvPlan* p, int n, hipStream_t s) {
    CdSet<P> set;
    set.n = n;
    int blocks = 0, order[P];
    size_t lds = 0;
    for (int i = 0; i < P; ++i) order[i] = i;
    std::stable_sort(order, order + n, [&](int i, int j) { return c[i].k * c[i].k * c[i].C > c[j].k * c[j].C * c[j].k; });
    for (int i = 0; i < P; ++i) {
        const int j = order[i < n ? i : 0];
        CdArgs& a = set.a[i];
        if (!tk_conv_direct_takes(c[j]) || !cd_fill(c[j], p[j], &a) || c[j].B != c[0].B || p[j].mt != p[0].mt || p[j].wm * p[j].wn != p[0].wm * p[0].wn) return false;
        set.first[i] = blocks;
        set.by_tiles[i] = cd_div(a.tiles);
        if (i >= n) continue;
        blocks += a.tiles * (((c[j].N + 15) / 16 + p[j].wn - 1) / p[j].wn);
        const size_t l = (size_t)cd_lds_bytes(c[j], a.ph, a.pw);
        lds = l > lds ? l : lds;
    }
    if (!tk_conv_direct_prepare_device()) return false;
    const dim3 grid(blocks, 1, c[0].B), block(64 * p[0].wm * p[0].wn);
    switch (p[0].mt) {
        case 1: hipLaunchKernelGGL((k_conv_direct<P, 1, 8>), grid, block, lds, s, set); break;
        case 2: hipLaunchKernelGGL((k_conv_direct<P, 2, 8>), grid, block, lds, s, set); break;
        default: hipLaunchKernelGGL((k_conv_direct<P, 4, 4>), grid, block, lds, s, set); break;
    }
    return true;
}
bool tk_launch_conv_direct(const TkConvDirect& c, const TkConvPlan& p, hipStream_t s) { return cd_launch<1>(&c, &p, 1, s); }
bool tk_launch_conv_direct_set(const TkConvDirect* c, const TkConvPlan* p, int n, hipStream_t s) {
    if (n < 1 || n > TK_CONV_SET) return false;
    return n == 1 ? cd_launch<1>(c, p, 1, s) : cd_launch<TK_CONV_SET>(c, p, n, s);
}
