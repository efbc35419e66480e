/* tk_attention_images.hip — see tk_attention_images.h */
#include "tk_attention_images.h"

#include "../common/tk_exact_math.h"

typedef float v4f __attribute__((ext_vector_type(4)));

/*
 * A workgroup of four waves makes 16 rows of one head.  Wave w owns the keys 256 u + 64 w .. + 63, u = 0 .. U - 1: the partial sums
 * 64 w .. 64 w + 63 of the canonical order (partial = key % 256, ascending), which is one quarter of its tree.
 *   scores: S^T = K Q^T a tile of 16 keys at a time, K's rows handed over in the order 4 b + a for row 4 a + b, so that the accumulator a
 *     lane gets back (rows 4 g .. 4 g + 3 of its column) is keys 4 t + g, t = 0 .. 3, of its query: the layout of P as an operand of P V.
 *     They stay in registers (4 U float4 a lane) until the product needs them.
 *   softmax: the tree's levels 32 .. 4 are inside a lane, 2 and 1 between the four lanes of a query, the quarters meet in LDS.  Scores are
 *     held unscaled: the scale 1 / 8 is a power of two, so (x / 8) - m rounds once, as one fma (a subnormal x / 8 does too, up to differences
 *     below 2^-100, whose exponential is 1 either way).  Division by the row's sum: y = RN(1 / sum), yl what is missing of it, q = e y + e yl
 *     within an ulp, and q + y (e - q sum) rounds correctly: Markstein's theorem (1990) for a correctly rounded reciprocal and an exact remainder.
 *     That is so as long as no remainder is subnormal (e >= 2^-100); the division itself otherwise.
 *   output: P goes through LDS 256 keys at a time, two buffers; wave w makes columns 16 w .. 16 w + 15, one chain over all keys.
 * Bound by the fp32 matrix pipe, which vector instructions share: at 16 rows x 1500 keys 24.3 k cycles of MFMA and 2400 vector instructions of
 * four cycles per SIMD, nearly all of them exponentials and divisions: 97 % of its time.  32 clips of 1500 positions x 6 heads take 1205 us (three
 * launches: 797 + 736 + 574), of which the products alone are 725 us at the rate of a large one.  With two corrections a division, a scale and a
 * vector address for each tile of K, 1240 us; two forms of the exponential, one without the test for values below -87, cost more than they save.
 */
template <int U>
__global__ __launch_bounds__(256, U > 4 ? 3 : 4) void k_attention_images(const float* q_img, const float* k_img, const float* v, float* out_img, int nh, int Tq, int Tk, int d,
                                                                         int tiles, int total, int per_xcd) {
    __shared__ v4f ring[2][16 * 64];
    __shared__ float top[4][16], sum[4][16];
    constexpr float scale = 0.125f; /* 1 / sqrt(64) */
    /* consecutive workgroups go to different XCDs: each XCD takes a run of them, so that a head's K and V (768 KB) are read into few L2s */
    const int id = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    if (id >= total) return;
    const int pair = id / tiles, q0 = (id - pair * tiles) * 16;
    const int b = pair / nh, h = pair - b * nh;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n = lane & 15, g = lane >> 4;
    const size_t group = (size_t)16 * d; /* floats of an image's 16 rows */
    const int col = (4 * h * 64 + g * 16) * 4;

    v4f qf[4];
    {
        const int64_t r = (int64_t)b * Tq + (q0 + n < Tq ? q0 + n : Tq - 1);
        const float* p = q_img + (size_t)(r >> 4) * group + col + (int)(r & 15) * 4;
#pragma unroll
        for (int j = 0; j < 4; ++j) qf[j] = *(const v4f*)(p + j * 256);
    }
    const int64_t k0 = (int64_t)b * Tk;
    const __amdgpu_buffer_rsrc_t kr = __builtin_amdgcn_make_buffer_rsrc((void*)(k_img + (size_t)(k0 >> 4) * group), 0, (unsigned)((k0 + Tk + 15) / 16 - (k0 >> 4)) * (unsigned)group * 4u, 0x00020000);
    const int k_odd = (int)(k0 & 15), key_of_row = 4 * (n & 3) + (n >> 2), k_first = 16 * (4 * wave) + key_of_row;
    auto k_place = [&](int key) { key += k_odd; return (unsigned)(key >> 4) * (unsigned)(64 * d) + (unsigned)(key & 15) * 16u + (unsigned)g * 256u; };
    const unsigned k_at = k_place(k_first);
    auto load_k = [&](int i, v4f* f) { /* tile i of the wave: 16 keys on is 16 rows of the image on */
        const int step = 16 * (i >> 2) + (i & 3);
        unsigned at = k_at, from = 4 * h * 1024 + (unsigned)step * (unsigned)(64 * d);
        if (i >= 4 * U - 4) {
            const int key = k_first + 16 * step;
            at = k_place(key < Tk ? key : Tk - 1);
            from = 4 * h * 1024;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) f[j] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(kr, at + j * 1024, from, 0));
    };
    v4f sc[4 * U];
    float m = -INFINITY, low = INFINITY;
    {
        v4f kf[2][4];
        load_k(0, kf[0]);
#pragma unroll
        for (int i = 0; i < 4 * U; ++i) {
            if (i + 1 < 4 * U) load_k(i + 1, kf[(i + 1) & 1]);
            v4f a = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int t = 0; t < 4; ++t) a = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[i & 1][j][t], qf[j][t], a, 0, 0, 0);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                float x = a[t];
                if (i >= 4 * U - 4) { /* keys that are not there: exp is 0 */
                    const bool there = 16 * (16 * (U - 1) + 4 * wave + (i & 3)) + 4 * t + g < Tk;
                    low = __builtin_fminf(low, there ? x : INFINITY);
                    x = there ? x : -INFINITY;
                } else {
                    low = __builtin_fminf(low, x);
                }
                sc[i][t] = x;
                m = __builtin_fmaxf(m, x); /* (a NaN among the scores makes the sum one) */
            }
            __builtin_amdgcn_sched_barrier(0); /* one tile at a time: the registers hold the scores, one tile of K and the next */
        }
    }
    m = tk_fmaxf(m, __shfl_xor(m, 16, 64));
    m = tk_fmaxf(m, __shfl_xor(m, 32, 64));
    if (lane < 16) top[wave][lane] = m;
    __syncthreads();
    m = tk_fmaxf(tk_fmaxf(top[0][n], top[1][n]), tk_fmaxf(top[2][n], top[3][n])) * scale;

    /* every e of the wave is 2^-100 or more (or none: the keys that are not there) */
    const bool tame = __all(low * scale - m >= -69.0f);
    v4f part[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v4f s = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const float e = tk_expf_below(tk_fmaf(sc[4 * u + i][t], scale, -m));
                sc[4 * u + i][t] = e;
                s[t] = s[t] + e;
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        part[i] = s;
    }
    float quarter;
    {
        float a[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) a[t] = (part[0][t] + part[2][t]) + (part[1][t] + part[3][t]);
        quarter = (a[0] + a[2]) + (a[1] + a[3]);
    }
    quarter = quarter + __shfl_xor(quarter, 32, 64);
    quarter = quarter + __shfl_xor(quarter, 16, 64);
    if (lane < 16) sum[wave][lane] = quarter;
    __syncthreads();
    const float tot = ((sum[0][n] + sum[1][n]) + sum[2][n]) + sum[3][n];
    const float inv = tk_divf(1.0f, tot), rest = inv * tk_fmaf(-tot, inv, 1.0f);

    auto put = [&](int u) { /* the wave's four tiles of 256 keys */
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v4f p;
            if (__builtin_expect(tame, 1)) {
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const float e = sc[4 * u + i][t];
                    const float x = tk_fmaf(e, inv, e * rest);
                    p[t] = tk_fmaf(tk_fmaf(-tot, x, e), inv, x);
                }
            } else {
#pragma unroll
                for (int t = 0; t < 4; ++t) p[t] = tk_divf(sc[4 * u + i][t], tot);
            }
            ring[u & 1][(4 * wave + i) * 64 + lane] = p;
        }
    };
    const unsigned pitch = 4u * (unsigned)d, v_lane = (unsigned)g * pitch + (unsigned)(h * 64 + wave * 16 + n) * 4u;
    const __amdgpu_buffer_rsrc_t vr = __builtin_amdgcn_make_buffer_rsrc((void*)(v + (size_t)b * Tk * d), 0, (unsigned)Tk * pitch, 0x00020000);
    auto load_v = [&](int q, float (*f)[4]) { /* keys 64 q .. 64 q + 63 */
        if (q < 4 * (U - 1) || 64 * q + 64 <= Tk) {
#pragma unroll
            for (int i = 0; i < 16; ++i) f[i >> 2][i & 3] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(vr, v_lane, (unsigned)(64 * q + 4 * i) * pitch, 0));
        } else { /* the last keys */
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int key = 64 * q + 4 * i, over = key + g - (Tk - 1);
                const float x = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(vr, v_lane + (unsigned)(over > 0 ? key - over : key) * pitch, 0, 0));
                f[i >> 2][i & 3] = over > 0 ? 0.0f : x;
            }
        }
    };
    v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
    float vf[2][4][4];
    load_v(0, vf[0]);
    put(0);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < U; ++u) {
        if (u + 1 < U) put(u + 1);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int q = 4 * u + c;
            if (u == U - 1 && 64 * q >= Tk) break;
            if (q + 1 < 4 * U) load_v(q + 1, vf[(q + 1) & 1]);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const v4f p = ring[u & 1][(4 * c + i) * 64 + lane];
#pragma unroll
                for (int t = 0; t < 4; ++t) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(p[t], vf[q & 1][i][t], acc, 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (u + 1 < U) __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = q0 + 4 * g + i;
        if (row < Tq) {
            const int64_t r = (int64_t)b * Tq + row;
            out_img[(size_t)(r >> 4) * group + ((4 * h + wave) * 64 + (n & 3) * 16 + (int)(r & 15)) * 4 + (n >> 2)] = acc[i] + 0.0f;
        }
    }
}

bool tk_launch_attention_images(const float* q_img, const float* k_img, const float* v, float* out_img, int B, int nh, int Tq, int Tk, int d, hipStream_t s) {
    if (B < 1 || !tk_attention_images_fits(Tq, Tk, d, nh)) return false;
    const int tiles = (Tq + 15) / 16;
    const int64_t total = (int64_t)B * nh * tiles, per = (total + 7) / 8;
    if (per * 8 > 0x7fffffff) return false;
#define TK_AIM(U) hipLaunchKernelGGL((k_attention_images<U>), dim3((unsigned)(per * 8)), dim3(256), 0, s, q_img, k_img, v, out_img, nh, Tq, Tk, d, tiles, (int)total, (int)per)
    switch ((Tk + 255) / 256) {
        case 1: TK_AIM(1); break;
        case 2: TK_AIM(2); break;
        case 3: TK_AIM(3); break;
        case 4: TK_AIM(4); break;
        case 5: TK_AIM(5); break;
        default: TK_AIM(6); break;
    }
#undef TK_AIM
    return true;
}
