#include "tk_audio_engine.h"
#include "tk_whisper_ggml.h"

#include <stdio.h>
#include <string.h>

#include <type_traits>

#include "../nn/tk_attention_images.h"
#include "../nn/tk_gemm_tiled.h"
#include "../nn/tk_nn_kernels.h"
#include "../nn/tk_image_device.h"

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

/* ---------------------------------------------------------------- log-mel front end kernels */

/* frame t, tap n: s16 -> f32 (/32768, as the reference's VAD does, src/sensors/tk_vad_silero.c:78-82), reflect padding of
 * n_fft/2 at both ends of the zero-padded 30 s window, times the Hann window */
__global__ void k_frames(const int16_t* pcm, int n_samples, int pcm_stride, int n_total, int T, const float* window, float* out) {
    const int b = blockIdx.z;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)T * TK_WH_NFFT) return;
    const int t = (int)(i / TK_WH_NFFT), n = (int)(i % TK_WH_NFFT);
    int j = t * TK_WH_HOP + n - TK_WH_NFFT / 2;
    if (j < 0) j = -j;
    if (j >= n_total) j = 2 * (n_total - 1) - j;
    const float x = j < n_samples ? tk_divf((float)pcm[(int64_t)b * pcm_stride + j], 32768.0f) : 0.0f;
    out[((int64_t)b * T + t) * TK_WH_NFFT + n] = x * window[n];
}

__global__ void k_power(const float* ri, int64_t rows, int nb, float* out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= rows * nb) return;
    const int64_t r = i / nb;
    const int f = (int)(i % nb);
    const float re = ri[r * 2 * nb + f], im = ri[r * 2 * nb + nb + f];
    out[i] = tk_fmaf(re, re, im * im);
}

/* log10(max(x, 1e-10)); clamp to (max over the utterance) - 8; (x + 4) / 4.  The logarithms bound it: TK_MEL_PARTS workgroups per utterance take them and
 * leave a maximum each, the second launch joins those (a maximum does not depend on the order) and clamps.  240 000 values of one utterance: 129 us in
 * one workgroup, now 7 + 4. */
#define TK_MEL_PARTS 64
__device__ __forceinline__ float mel_block_max(float mx, float* red) { /* 256 threads */
    mx = tk_wave_max(mx);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
    __syncthreads();
    return tk_fmaxf(tk_fmaxf(red[0], red[1]), tk_fmaxf(red[2], red[3]));
}
__global__ __launch_bounds__(256) void k_logmel_log(float* mel, int per_b, float* part) {
    __shared__ float red[4];
    float* m = mel + (int64_t)blockIdx.y * per_b;
    float mx = -INFINITY;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < per_b; i += TK_MEL_PARTS * 256) {
        const float v = tk_log10f(tk_fmaxf(m[i], 1e-10f));
        m[i] = v;
        mx = tk_fmaxf(mx, v);
    }
    mx = mel_block_max(mx, red);
    if (threadIdx.x == 0) part[blockIdx.y * TK_MEL_PARTS + blockIdx.x] = mx;
}
__global__ __launch_bounds__(256) void k_logmel_clamp(float* mel, int per_b, const float* part) {
    __shared__ float red[4];
    float* m = mel + (int64_t)blockIdx.y * per_b;
    const float floor_v = mel_block_max(part[blockIdx.y * TK_MEL_PARTS + (threadIdx.x & (TK_MEL_PARTS - 1))], red) - 8.0f;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < per_b; i += TK_MEL_PARTS * 256) m[i] = (tk_fmaxf(m[i], floor_v) + 4.0f) * 0.25f;
}

/* ---------------------------------------------------------------- decoder-step attention, fused

 * One query row per (sequence, head): scores, softmax and the value contraction in one launch or two, with exactly the arithmetic of the
 * three-launch form it replaces (tk_whisper_graph.h: attention()): score = (fp32 fma chain over the head dimension, ascending) * scale
 * + 0.0f (the GEMM epilogue's bias slot); softmax as k_softmax_rows evaluates it (256 strided partial maxima / sums, shuffle tree,
 * ((w0 + w1) + w2) + w3); output = one fp32 fma chain over the keys in ascending order, + 0.0f.  */
/* What bounds it: the value contraction is one fp32 chain over the keys per output, 8 cycles a key on the 16 x 16 x 4 MFMA (1500 keys: 5 us), and
 * what one CU can fetch (about 40 KB a us).  So the chain must never wait for memory, and a head's K and V come in through several CUs:
 *  - a workgroup takes hd / split outputs of one head, with its part of V only: few sequences leave most CUs idle, so the split grows while the
 *    grid stays within the chip.  16 outputs are one wave's chain; its MFMAs take the weights as 16 equal rows of A.
 *  - V goes through registers, requested before the scores are known (all of 1500 keys x 16 outputs; more in rounds, the next one under way during
 *    a round's chain), into LDS in the order of four MFMAs' operands: a wave gets one LDS read in about 18 cycles, whatever its width, so it
 *    must need few: 2 for 16 keys.
 *  - over long contexts (cross attention) the scores come from a kernel of their own, 64 keys per wave over the whole chip; up to 512 keys
 *    (self attention) every workgroup makes them itself, 64 keys per wave: a launch costs more.
 * Scores: a key per lane.  K comes by LDS-DMA, 16 floats of each key per slot of 4 KiB (rows 64 bytes apart, their 16-byte units swapped by
 * row so that the 64 lanes' reads spread over all banks).
 * Cross attention of one sequence (6 heads, 1500 keys of 64): 18 us (4 + 14); with one workgroup of 4 waves per head, whose lanes read whole rows of K
 * (64 lines per load) and whose chain ran on one vector unit: 49 us.  32 sequences: 42 us against 77.  Contexts beyond 2048 keys read their
 * scores twice and keep the weights in LDS only: a decoder step of four layers over 6000 keys, 16 sequences: 0.65 ms, 1.30 in three launches. */
#define TK_AT1_NW 8             /* waves */
#define TK_AT1_RING (16 * 1024) /* bytes per wave: 64 keys of K in four slots of 16 floats */
#define TK_AT1_SELF 512         /* longest context whose scores are made in the same kernel: 64 keys per wave */
#define TK_AT1_HELD 2048        /* longest context whose scores stay in registers: 8 per thread */
#define TK_AT1_MAX_KEYS 12288   /* a round of V and the weights in the LDS */
typedef float at1_f32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void at1_wait_vm0() { __builtin_amdgcn_s_waitcnt(0x0F70); } /* s_waitcnt vmcnt(0) alone */
__device__ __forceinline__ void at1_dma(const float* src, uint8_t* lds) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src, (__attribute__((address_space(3))) void*)lds, 16, 0, 0);
}
/* the score of key 64 blk + lane (of the last key where there is none); q [hd] in LDS, hd * 256 bytes of ring per wave or 16 KiB, whichever is less */
__device__ __forceinline__ float at1_score(const float* kp, int blk, int Tk, int64_t kv_row, int hd, float scale, const float* qs, uint8_t* ring, int lane) {
    const int unit = (lane & 3) ^ ((lane >> 4) & 3), nsl = hd >> 4;
    const float* src[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        int row = blk * 64 + p * 16 + (lane >> 2);
        row = row < Tk ? row : Tk - 1;
        src[p] = kp + row * kv_row + unit * 4;
    }
    float a = 0.0f;
    for (int s0 = 0; s0 < nsl; s0 += 4) {
        for (int sl = s0; sl < s0 + 4 && sl < nsl; ++sl)
#pragma unroll
            for (int p = 0; p < 4; ++p) at1_dma(src[p] + sl * 16, ring + (sl & 3) * 4096 + p * 1024);
        at1_wait_vm0();
        for (int sl = s0; sl < s0 + 4 && sl < nsl; ++sl) {
            const uint8_t* slot = ring + (sl & 3) * 4096 + lane * 64;
            float4 kk[4], qq[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) { kk[i] = *(const float4*)(slot + ((i ^ ((lane >> 2) & 3)) << 4)); qq[i] = *(const float4*)(qs + sl * 16 + 4 * i); }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                a = tk_fmaf(qq[i].x, kk[i].x, a); a = tk_fmaf(qq[i].y, kk[i].y, a); a = tk_fmaf(qq[i].z, kk[i].z, a); a = tk_fmaf(qq[i].w, kk[i].w, a);
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); /* the ring is read out */
    }
    a = a * scale;
    return a + 0.0f;
}

/* scores [rows][heads][pitch] of a long context: grid (64-key blocks / 4, heads, rows), a block of keys per wave; row i `group` + b is a row of sequence b */
__global__ __launch_bounds__(256) void k_attend1_scores(const float* q, const float* k, float* scores, int Tk, int pitch, int64_t q_bstride, int64_t kv_bstride, int64_t kv_row, int hd,
                                                        int group, float scale) {
    extern __shared__ __attribute__((aligned(16))) uint8_t att1_lds[];
    const int h = blockIdx.y, row = blockIdx.z, b = (int)gridDim.z > group ? (int)((unsigned)row % (unsigned)group) : row, lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    float* qs = (float*)(att1_lds + 4 * TK_AT1_RING);
    for (int i = threadIdx.x; i < hd; i += 256) qs[i] = q[(int64_t)row * q_bstride + (int64_t)h * hd + i];
    __syncthreads();
    const int blk = blockIdx.x * 4 + wave;
    if (blk * 64 >= Tk) return;
    const float a = at1_score(k + (int64_t)b * kv_bstride + (int64_t)h * hd, blk, Tk, kv_row, hd, scale, qs, att1_lds + wave * TK_AT1_RING, lane);
    if (blk * 64 + lane < Tk) scores[((int64_t)row * gridDim.y + h) * pitch + blk * 64 + lane] = a;
}

/* tasks of a thread in a round of V (kernel below), and what a round takes of C columns: the whole of a self attention's usual context at once */
constexpr int at1_tasks(bool self) { return self ? 1 : 3; }
__host__ __device__ constexpr int at1_round_blocks(bool self, int C) { return at1_tasks(self) * 64 * TK_AT1_NW / C; }
/* place of key k's weight in LDS: 16 keys' weights in the order in which four MFMAs take them, so that a lane's four are one read */
__device__ __forceinline__ int at1_place(int k) { return (k & ~15) | (k & 3) << 2 | (k >> 2 & 3); }

/* where the scores are: made here; read from memory once and held; read from memory twice */
enum { AT1_SELF, AT1_HELD, AT1_LONG };
template <int FORM>
__global__ __launch_bounds__(64 * TK_AT1_NW) void k_attend1(const float* q, const float* k, const float* v, const float* scores, int pitch, float* out, int Tk,
                                                           int64_t q_bstride, int64_t kv_bstride, int64_t kv_row, int d, int hd, int split, float scale, int sc_at /* bytes */,
                                                           int more /* keys that each position of a span sees beyond the one before */,
                                                           float* img /* optional: out also as the tiled GEMM's operand image [rows][K = d] */) {
    extern __shared__ __attribute__((aligned(16))) uint8_t att1_lds[];
    /* grid (heads * split, sequences, positions) */
    const int h = blockIdx.x / split, part = blockIdx.x % split, b = blockIdx.y, row = blockIdx.z * gridDim.y + b, t0 = threadIdx.x, lane = t0 & 63;
    Tk += (int)blockIdx.z * more;
    const int wave = __builtin_amdgcn_readfirstlane(t0 >> 6);
    float* vbuf = (float*)att1_lds;         /* a round of V; before it the waves' rings of K */
    float* sc = (float*)(att1_lds + sc_at); /* [Tk rounded up to 16] */
    float* qs = sc + ((Tk + 15) & ~15);     /* [hd] */
    float* red = qs + hd;                   /* [8] */
    const int C = hd / split;               /* this workgroup's outputs: a multiple of 16 */
    const float* vp = v + (int64_t)b * kv_bstride + (int64_t)h * hd + part * C;

    /* 256 threads hold the scores: thread t those of keys t, t + 256, ...: the canonical partials */
    constexpr bool SELF = FORM == AT1_SELF;
    constexpr int NS = SELF ? TK_AT1_SELF / 256 : TK_AT1_HELD / 256;
    float e[NS];
    const float* sp = scores + ((int64_t)row * (gridDim.x / split) + h) * pitch;
    auto load_scores = [&](int k0) {
#pragma unroll
        for (int j = 0; j < NS; ++j) { const int t = k0 + (t0 & 255) + 256 * j; e[j] = sp[t < Tk ? t : Tk - 1]; }
    };
    if (FORM == AT1_HELD) load_scores(0);
    /* V in rounds of 16 * rb keys.  A thread's task: keys 16 kb + 4 t + g, t = 0 .. 3, of four neighbouring columns.  LDS: [block of 16 keys]
     * [16 columns][g][column ^ g][t], 1 KiB a tile (the XOR spreads the four g's writes over the banks) */
    constexpr int NT = at1_tasks(SELF);
    const int cu = C >> 2, nt = C >> 4, rb = at1_round_blocks(SELF, C), nblk = (Tk + 15) >> 4;
    at1_f32x4 vv[NT][4];
    auto load_v = [&](int kb0) { /* past the round or the last key: read again, not used */
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            const int id = t0 + 64 * TK_AT1_NW * i, kq = id / cu, x = id - kq * cu;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                int row = (kb0 + (kq >> 2)) * 16 + 4 * t + (kq & 3);
                row = row < Tk ? row : Tk - 1;
                vv[i][t] = *(const at1_f32x4*)(vp + row * kv_row + 4 * x);
            }
        }
    };
    auto store_v = [&](int blocks) {
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            const int id = t0 + 64 * TK_AT1_NW * i, kq = id / cu, x = id - kq * cu, g = kq & 3;
#pragma unroll
            for (int t = 0; t < 4; ++t) asm volatile("" : "+v"(vv[i][t])); /* as loaded up to here: else the loads are turned, and waited for, where they are issued */
            float* dst = vbuf + ((kq >> 2) * nt + (x >> 2)) * 256 + g * 64 + (x & 3) * 16;
            if ((kq >> 2) < blocks) {
                *(at1_f32x4*)(dst + (0 ^ g) * 4) = at1_f32x4{vv[i][0].x, vv[i][1].x, vv[i][2].x, vv[i][3].x};
                *(at1_f32x4*)(dst + (1 ^ g) * 4) = at1_f32x4{vv[i][0].y, vv[i][1].y, vv[i][2].y, vv[i][3].y};
                *(at1_f32x4*)(dst + (2 ^ g) * 4) = at1_f32x4{vv[i][0].z, vv[i][1].z, vv[i][2].z, vv[i][3].z};
                *(at1_f32x4*)(dst + (3 ^ g) * 4) = at1_f32x4{vv[i][0].w, vv[i][1].w, vv[i][2].w, vv[i][3].w};
            }
        }
    };
    load_v(0);
    __builtin_amdgcn_sched_barrier(0);
    if (SELF) {
        const float* qp = q + (int64_t)row * q_bstride + (int64_t)h * hd;
        for (int i = t0; i < hd; i += 64 * TK_AT1_NW) qs[i] = qp[i];
        __syncthreads();
        if (wave * 64 < Tk) {
            const float a = at1_score(k + (int64_t)b * kv_bstride + (int64_t)h * hd, wave, Tk, kv_row, hd, scale, qs, att1_lds + wave * TK_AT1_RING, lane);
            if (t0 < Tk) sc[t0] = a;
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < NS; ++j) { const int t = (t0 & 255) + 256 * j; e[j] = sc[t < Tk ? t : Tk - 1]; }
    }
    const int tk = t0 & 255; /* threads 256 .. 511 do the same again: no wave waits for another's branch */
    const int rounds = FORM == AT1_LONG ? (Tk + TK_AT1_HELD - 1) / TK_AT1_HELD * TK_AT1_HELD : 1;
    float m = -INFINITY;
    for (int k0 = 0; k0 < rounds; k0 += TK_AT1_HELD) {
        if (FORM == AT1_LONG) load_scores(k0);
#pragma unroll
        for (int j = 0; j < NS; ++j)
            if (k0 + tk + 256 * j < Tk) m = tk_fmaxf(m, e[j]);
    }
    m = tk_wave_max(m);
    if (lane == 0) red[wave & 3] = m;
    __syncthreads();
    m = tk_fmaxf(tk_fmaxf(red[0], red[1]), tk_fmaxf(red[2], red[3]));
    float s = 0.0f;
    for (int k0 = 0; k0 < rounds; k0 += TK_AT1_HELD) {
        if (FORM == AT1_LONG) load_scores(k0);
#pragma unroll
        for (int j = 0; j < NS; ++j)
            if (k0 + tk + 256 * j < Tk) {
                e[j] = tk_expf(e[j] - m);
                s = s + e[j];
                if (FORM == AT1_LONG && wave < 4) sc[at1_place(k0 + tk + 256 * j)] = e[j];
            }
    }
    s = tk_wave_butterfly_sum(s);
    if (lane == 0) red[4 + (wave & 3)] = s;
    __syncthreads();
    const float tot = ((red[4] + red[5]) + red[6]) + red[7];
    if (wave < 4) {
        if (FORM == AT1_LONG) {
            for (int t = t0; t < Tk; t += 256) sc[at1_place(t)] = tk_divf(sc[at1_place(t)], tot); /* its own */
        } else {
#pragma unroll
            for (int j = 0; j < NS; ++j)
                if (t0 + 256 * j < Tk) sc[at1_place(t0 + 256 * j)] = tk_divf(e[j], tot);
        }
        if (t0 < (-Tk & 15)) sc[at1_place(Tk + t0)] = 0.0f;
    }

    at1_f32x4 acc[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}}; /* outputs 16 wave .. and 16 (wave + 8) .. */
    const int g = lane >> 4, col = lane & 15;
    for (int kb0 = 0; kb0 < nblk; kb0 += rb) {
        if (kb0) __syncthreads(); /* everybody is done with the round before */
        const int nb = nblk - kb0 < rb ? nblk - kb0 : rb, n = Tk - kb0 * 16;
        store_v(nb);
        __syncthreads();
        if (kb0 + rb < nblk) load_v(kb0 + rb);
        const float* pc = sc + kb0 * 16;
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            const int tile = wave + TK_AT1_NW * w;
            if (tile >= nt) break;
            struct Stage { at1_f32x4 p[2], v[2]; } x, y; /* 32 keys */
            const float* vt = vbuf + tile * 256 + g * 64 + (col ^ g) * 4;
            auto read = [&](Stage& o, int u) { /* blocks u, u + 1 of 16 keys; the last one again past it */
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const int kb = u + i < nb ? u + i : nb - 1;
                    o.p[i] = *(const at1_f32x4*)(pc + kb * 16 + 4 * g);
                    o.v[i] = *(const at1_f32x4*)(vt + kb * nt * 256);
                }
                __builtin_amdgcn_sched_barrier(0);
            };
            auto multiply = [&](Stage& o, int u, auto tail) {
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    if (tail.value) {
                        if (u + i >= nb) break;
#pragma unroll
                        for (int j = 0; j < 4; ++j) o.v[i][j] = (u + i) * 16 + 4 * j + g < n ? o.v[i][j] : 0.0f; /* keys past the last add 0 x 0 */
                    }
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc[w] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.p[i][j], o.v[i][j], acc[w], 0, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            };
            read(x, 0);
            int u = 0;
            for (; u + 4 < nb; u += 4) {
                read(y, u + 2);
                multiply(x, u, std::false_type{});
                read(x, u + 4);
                multiply(y, u + 2, std::false_type{});
            }
            read(y, u + 2);
            multiply(x, u, std::true_type{});
            multiply(y, u + 2, std::true_type{});
        }
    }
#pragma unroll
    for (int w = 0; w < 2; ++w) {
        const int c0 = (wave + TK_AT1_NW * w) * 16 + col;
        if (c0 - col >= C || g != 0) break;
        const int kk = h * hd + part * C + c0;
        const float r = acc[w][0] + 0.0f;
        out[(int64_t)row * q_bstride + kk] = r;
        if (img) img[(int64_t)(row >> 4) * 16 * d + (int64_t)(kk >> 4) * 256 + (kk & 3) * 64 + (row & 15) * 4 + ((kk & 15) >> 2)] = r;
    }
}
/* bytes in front of the weights: the rings of K or a round of V, whichever is more */
static int at1_buffer(int Tk, int C) {
    const bool self = Tk <= TK_AT1_SELF;
    const int blocks = (Tk + 15) / 16, rb = at1_round_blocks(self, C), round = (blocks < rb ? blocks : rb) * 64 * C, rings = self ? (Tk + 63) / 64 * TK_AT1_RING : 0;
    return round > rings ? round : rings;
}
static bool at1_prepare_device() {
    const int most = 160 * 1024;
    return hipFuncSetAttribute((const void*)k_attend1<AT1_SELF>, hipFuncAttributeMaxDynamicSharedMemorySize, most) == hipSuccess &&
           hipFuncSetAttribute((const void*)k_attend1<AT1_HELD>, hipFuncAttributeMaxDynamicSharedMemorySize, most) == hipSuccess &&
           hipFuncSetAttribute((const void*)k_attend1<AT1_LONG>, hipFuncAttributeMaxDynamicSharedMemorySize, most) == hipSuccess &&
           hipFuncSetAttribute((const void*)k_attend1_scores, hipFuncAttributeMaxDynamicSharedMemorySize, most) == hipSuccess;
}
/* n positions of B sequences, rows position by position; the first sees Tk keys, each next one `more` further ones (0, or 1 with at most TK_AT1_SELF keys for the last).
 * scores: scratch [B n][nh][pitch] */
static bool at1_launch(const float* q, const float* k, const float* v, float* scores, int pitch, float* out, int B, int n, int Tk, int more, int64_t q_bstride, int64_t kv_bstride, int64_t kv_row,
                       int d, int nh, float* img, hipStream_t s) {
    const int hd = d / nh, most = Tk + (n - 1) * more;
    if (n < 1 || (more != 0 && (more != 1 || most > TK_AT1_SELF))) return false;
    const float scale = tk_divf(1.0f, tk_sqrtf((float)hd));
    int split = 1; /* workgroups per head: 16 outputs each at least, while all of them run at once */
    while (hd % (32 * split) == 0 && 2 * split * nh * B * n <= 256) split *= 2;
    const dim3 grid(nh * split, B, n), block(64 * TK_AT1_NW);
    const int sc_at = at1_buffer(most, hd / split);
    const size_t lds = (size_t)sc_at + (size_t)(((most + 15) & ~15) + hd + 8) * 4; /* <= 128 KiB + 3 KiB, 96 KiB + 10 KiB, 96 KiB + 50 KiB */
#define TK_AT1(FORM) hipLaunchKernelGGL((k_attend1<FORM>), grid, block, lds, s, q, k, v, scores, pitch, out, Tk, q_bstride, kv_bstride, kv_row, d, hd, split, scale, sc_at, more, img)
    if (most <= TK_AT1_SELF) {
        TK_AT1(AT1_SELF);
    } else {
        hipLaunchKernelGGL(k_attend1_scores, dim3(((Tk + 63) / 64 + 3) / 4, nh, B * n), dim3(256), 4 * TK_AT1_RING + (size_t)hd * 4, s, q, k, scores, Tk, pitch, q_bstride, kv_bstride, kv_row, hd, B, scale);
        if (Tk <= TK_AT1_HELD) TK_AT1(AT1_HELD); else TK_AT1(AT1_LONG);
#undef TK_AT1
    }
    return true;
}

/* ---------------------------------------------------------------- GPU ops for the shared graph */

/* shapes the tiled GEMM takes: a plain linear layer C = act(A W^T + b) + R with K a multiple of 128 */
static inline bool tk_tiled_gemm_applies(const TkGemm& g) {
    return g.b_kn == 0 && g.batch <= 1 && g.batch_inner == 0 && g.alpha == 1.0f && !g.b_f16 && g.ldb == g.K && g.K % 128 == 0 && g.M > 0;
}
/* floats of the activation image: whole row blocks (16 M-tiles, or the M-tile count of a short pass) */
static inline size_t tk_tiled_gemm_scratch(const TkGemm& g) {
    const int rows_blk = g.M < TK_TW_MAX_BLOCK_ROWS ? g.M : TK_TW_MAX_BLOCK_ROWS;
    const int mt = rows_blk > 128 ? 16 : rows_blk > 64 ? 8 : rows_blk > 32 ? 4 : rows_blk > 16 ? 2 : 1;
    const int64_t blk = (int64_t)mt * 16, padded = ((int64_t)g.M + blk - 1) / blk * blk;
    return (size_t)padded * (size_t)g.K;
}

struct TkAudioGpuOps {
    TkAsr* a;
    hipStream_t s;
    /* set by the engine around the per-utterance long passes (log-mel, encoder, cross keys / values): there the opt-in fast contraction applies.
     * The decode steps never take it — a choice by the row count of a launch would make an utterance's result depend on its batch */
    bool long_ok = false;
    /* the operand image of the last packed activation matrix: consecutive linear layers on the same input (q / k / v, cross k / v) pack it
     * once.  It sits on top of the arena and is dropped — its space handed back — by every other op, by any allocation of the graph and
     * by a GEMM that writes into the matrix it was made from. */
    struct { const float* A = nullptr; int M = 0, K = 0, lda = 0; float* img = nullptr; size_t mark = 0; bool live = false; } pk;
    /* Decoder steps of few sequences: a norm is not launched; the linear layers on it make it themselves (TkTiledGemm::ln_x).  pk then names its output, which nobody else
     * reads, and has no image.  A layer that cannot take it has it launched first.  Up to TK_TW_LN_ROWS sequences: calls of 40 steps for 1, 2, 4, 6, 8, 16 clips, norms
     * launched / in the products: 13.36 / 12.34, 14.39 / 13.28, 16.08 / 15.45, 17.31 / 17.27, 18.92 / 19.24, 23.65 / 26.00 ms. */
    /* Other norms of a whole number of 128 columns wait for their first reader: a layer with tiles gets an operand image and no rows (48 000 rows of 384 columns: 70 -> 28 us),
     * anything else the rows. */
    struct { const float *x = nullptr, *w = nullptr, *b = nullptr; float* y = nullptr; bool live = false, used = false, in_products = false; } norm;
    static bool norm_fits(int rows, int D) { return rows <= TK_TW_LN_ROWS && D <= TK_TW_LN_MAX && D % 128 == 0; }
    void make_norm(bool image) { /* as a launch after all */
        const int M = pk.M, K = pk.K;
        norm.live = pk.live = false;
        if (image) tk_launch_layernorm_image(norm.x, M, K, norm.w, norm.b, TK_WH_LN_EPS, image_for(norm.y, M, K, K), s);
        else tk_launch_layernorm(norm.x, M, K, norm.w, norm.b, TK_WH_LN_EPS, norm.y, s);
    }
    /* columns of a convolution wait for their reader in the same way */
    struct { const float* x = nullptr; int B = 0, T = 0, C = 0, ldx = 0, kw = 0, stride = 0, pad = 0; float* col = nullptr; } cols;
    void make_columns() {
        if (cols.col) tk_launch_im2col1d(cols.x, cols.B, cols.T, cols.C, cols.ldx, cols.kw, cols.stride, cols.pad, cols.col, s);
        cols.col = nullptr;
    }
    /* linear layers on the SAME packed input (q / k / v of a layer, the cross keys and values) are collected — up to three — and go out as ONE
     * launch with a destination per segment (q | k | v: the query buffer and row p of the two caches); anything else flushes the batch first */
    struct { TkTiledGemm t{}; int n = 0; } pend;
    void flush() {
        if (pend.n == 0) return;
        pend.t.nseg = pend.n;
        int cols = 0;
        for (int i = 0; i < pend.n; ++i) cols += pend.t.row_tiles[i] * 16;
        pend.t.n_valid = cols;
        if (!tk_launch_gemm_tiled(pend.t, s)) a->launch_error = "tiled GEMM launch refused (batched decoder layers)";
        pend.n = 0;
    }
    void drop_image() {
        flush();
        make_columns();
        if (norm.live && !norm.used) make_norm(false); /* (its readers are not linear layers) */
        if (pk.live && !norm.live) a->arena_used = pk.mark;
        pk.live = norm.live = false;
    }
    float* alloc(size_t n) {
        drop_image();
        return raw_alloc(n);
    }
    float* raw_alloc(size_t n) {
        n = (n + 63) & ~(size_t)63;
        if (a->arena_used + n > a->arena_floats) { /* tk_asr_arena_floats() counts every allocation: not reached */
            a->launch_error = "ASR arena too small";
            return a->arena;
        }
        float* p = a->arena + a->arena_used;
        a->arena_used += n;
        return p;
    }
    int32_t* alloc_i32(size_t n) { return (int32_t*)alloc(n); }
    static bool short_pass(int M) { return M <= TK_TW_MAX_BLOCK_ROWS; }
    /* the packed image of a matrix a producer kernel is about to write (layer norm, decoder attention): lives on top of the arena like
     * the image gemm() packs itself, and is found there by the linear layers that follow */
    float* image_for(const float* A, int M, int K, int lda) {
        pk.mark = a->arena_used;
        TkGemm g{};
        g.M = M; g.K = K;
        pk.img = raw_alloc(tk_tiled_gemm_scratch(g));
        pk.A = A; pk.M = M; pk.K = K; pk.lda = lda; pk.live = true;
        return pk.img;
    }
    /* a linear layer whose weights have tiles runs on the tiled GEMM (same k-ascending fp32 chain, bit-identical, ~3x the rate of the
     * LDS-staged kernel on these shapes and one short launch instead of a latency chain for the decoder's few rows) */
    void gemm(const TkGemm& g) {
        if (a->fast && long_ok) { /* opt-in fast contraction of the long passes (TkAsr::fast): row-major operands, split-f16 MFMA where the shape allows */
            drop_image();
            TkGemm f = g;
            f.fast = 1;
            tk_launch_gemm(f, s);
            return;
        }
        const int idx = tk_tiled_gemm_applies(g) ? a->model->tensor_of(g.B) : -1;
        if (idx < 0 || !a->model->wt[(size_t)idx]) {
            if (norm.live) make_norm(false);
            drop_image();
            tk_launch_gemm(g, s);
            return;
        }
        if (norm.live && !(pk.A == g.A && pk.M == g.M && pk.K == g.K && pk.lda == g.lda)) drop_image();
        if (!(pk.live && pk.A == g.A && pk.M == g.M && pk.K == g.K && pk.lda == g.lda)) {
            const bool columns = cols.col == g.A && g.K == cols.kw * cols.C && g.lda == g.K && cols.C % 16 == 0;
            if (columns) cols.col = nullptr;
            drop_image();
            pk.mark = a->arena_used;
            pk.img = raw_alloc(tk_tiled_gemm_scratch(g));
            if (columns) tk_launch_im2col1d_image(cols.x, cols.B, cols.T, cols.C, cols.ldx, cols.kw, cols.stride, cols.pad, pk.img, s);
            else tk_launch_pack_a(g.A, g.M, g.K, g.lda, 0, pk.img, s);
            pk.A = g.A; pk.M = g.M; pk.K = g.K; pk.lda = g.lda; pk.live = true;
        } else if (norm.live && !norm.in_products) {
            make_norm(true);
        }
        /* does the output overlap the packed matrix (an in-place layer)?  Then the image is stale once the launch has run */
        const float* c0 = g.C;
        const float* c1 = g.C + (size_t)(g.M - 1) * g.ldc + g.N;
        const float* a0 = g.A;
        const float* a1 = g.A + (size_t)(g.M - 1) * g.lda + g.K;
        const bool in_place = c0 < a1 && a0 < c1;
        const bool plain = !g.residual && !g.c_feeds_linear && g.N % 16 == 0 && !in_place; /* an in-place layer never joins a batch: it runs alone below */
        if (plain) { /* joins (or opens) the batch of layers on this input */
            if (pend.n > 0 && (pend.t.a_img != (norm.live ? nullptr : pk.img) || pend.t.ln_x != (norm.live ? norm.x : nullptr) || pend.t.K != g.K || pend.t.nrows != g.M || pend.t.act != g.act)) flush();
            TkTiledGemm& t = pend.t;
            if (pend.n == 0) {
                t = TkTiledGemm{};
                t.wbytes = 4; t.K = g.K; t.ks = 1; t.nrows = g.M; t.slab_rows = 0; t.a_img = norm.live ? nullptr : pk.img; t.a_ts = (size_t)g.K * 16;
                t.act = g.act; t.add_zero_bias = 1; t.per_seg = 1;
                use_norm(t);
            }
            const int i = pend.n++;
            t.tiles[i] = a->model->wt[(size_t)idx]; t.row_tiles[i] = g.N / 16;
            t.seg_out[i] = g.C; t.seg_ldc[i] = g.ldc; t.seg_bias[i] = g.bias; t.seg_n[i] = g.N; t.seg_img[i] = g.c_image;
            if (pend.n == 3) flush();
            return; /* none of these layers writes into its own input: `plain` excludes in-place layers */
        }
        flush();
        TkTiledGemm t{};
        t.tiles[0] = a->model->wt[(size_t)idx]; t.row_tiles[0] = (g.N + 15) / 16; t.nseg = 1; t.wbytes = 4;
        t.K = g.K; t.ks = 1; t.ldc = g.ldc; t.n_valid = g.N; t.nrows = g.M; t.slab_rows = 0;
        t.a_img = norm.live ? nullptr : pk.img; t.a_ts = (size_t)g.K * 16; t.out = g.C;
        use_norm(t);
        t.bias = g.bias; t.residual = g.residual; t.ldr = g.ldr; t.act = g.act; t.add_zero_bias = 1;
        /* fc1: its output is only ever the input of fc2 — written as fc2's operand image as well (on top of fc1's own), on long (encoder) passes
         * too: there the second image replaces a k_pack_a launch over B x 1500 x 4 d values (9.8 -> 9.4 ms per call, profiles/r04_perception.txt) */
        const bool emit_img = g.c_feeds_linear && g.N % 128 == 0 && g.ldc == g.N && !g.residual && !in_place;
        float* cimg = nullptr;
        if (emit_img) {
            TkGemm nx{};
            nx.M = g.M; nx.K = g.N;
            if (norm.live) pk.mark = a->arena_used; /* (the norm has no image below it) */
            cimg = raw_alloc(tk_tiled_gemm_scratch(nx));
            t.c_img = cimg;
            t.out = nullptr; /* (fc2 has tiles: its K is a multiple of 128) */
        }
        if (!tk_launch_gemm_tiled(t, s)) a->launch_error = "tiled GEMM launch refused"; /* not reached: tk_tiled_gemm_applies() admits only shapes the launcher takes */
        if (emit_img) { /* the image pair stays allocated from pk.mark up; the upper one is now the live image */
            pk.img = cimg; pk.A = g.C; pk.M = g.M; pk.K = g.N; pk.lda = g.ldc; pk.live = true;
            norm.live = false;
            return;
        }
        if (in_place) drop_image(); /* the output overwrote the packed matrix: the image is stale */
    }
    void use_norm(TkTiledGemm& t) {
        if (!norm.live) return;
        norm.used = true;
        t.ln_x = norm.x; t.ln_w = norm.w; t.ln_b = norm.b; t.ln_eps = TK_WH_LN_EPS;
    }
    void im2col1d(const float* x, int B, int T, int C, int ldx, int kw, int stride, int pad, float* col) {
        drop_image();
        cols.x = x; cols.B = B; cols.T = T; cols.C = C; cols.ldx = ldx; cols.kw = kw; cols.stride = stride; cols.pad = pad; cols.col = col;
    }
    void layernorm(const float* x, int rows, int D, const float* w, const float* b, float* y) {
        drop_image();
        if (D % 128) { tk_launch_layernorm(x, rows, D, w, b, TK_WH_LN_EPS, y, s); return; }
        norm.x = x; norm.w = w; norm.b = b; norm.y = y; norm.live = true; norm.used = false;
        norm.in_products = !long_ok && norm_fits(rows, D); /* a decoder step's */
        pk.A = y; pk.M = rows; pk.K = D; pk.lda = D; pk.img = nullptr; pk.mark = a->arena_used; pk.live = true;
    }
    void settle() { drop_image(); }
    void softmax_rows(float* x, int rows, int cols, int ld) { drop_image(); tk_launch_softmax_rows(x, rows, cols, ld, s); }
    bool attend1(const float* q, const float* k, const float* v, float* out, int B, int Tk, int64_t q_bstride, int64_t kv_bstride, int kv_row, int d, int nh, float* scores, int pitch) {
        drop_image();
        const int hd = d / nh;
        if (hd > 256 || (hd & 15) || (d & 3) || Tk < 1 || Tk > TK_AT1_MAX_KEYS) return false; /* the three-launch form takes what does not fit */
        float* img = (short_pass(B) && d % 128 == 0 && q_bstride == d) ? image_for(out, B, d, d) : nullptr; /* the output projection's input, packed on the way out */
        return at1_launch(q, k, v, scores, pitch, out, B, 1, Tk, 0, q_bstride, kv_bstride, kv_row, d, nh, img, s);
    }
    /* positions of a prompt that one pass takes: as many as make TK_ASR_SPAN_ROWS rows.  0, for one by one as they are decoded, where a layer's widths are not those of the
     * kernels that know of several, or where the span's keys need scores from a launch of their own */
    static int span(const TkWhisperHP& h, int B) {
        const int dt = h.n_text_state, hd = dt / h.n_text_head;
        if (dt % 128 || hd > 256 || (hd & 15) || h.n_text_ctx > TK_AT1_SELF || h.n_audio_ctx > TK_AT1_MAX_KEYS) return 0;
        return B < TK_ASR_SPAN_ROWS ? TK_ASR_SPAN_ROWS / B : 1;
    }
    void attend_span(const float* q, const float* k, const float* v, float* out, int B, int n, int Tk, bool causal, int64_t q_bstride, int64_t kv_bstride, int kv_row, int d, int nh, float* scores, int pitch) {
        drop_image();
        float* img = image_for(out, B * n, d, d);
        if (!at1_launch(q, k, v, scores, pitch, out, B, n, Tk, causal ? 1 : 0, q_bstride, kv_bstride, kv_row, d, nh, img, s)) a->launch_error = "decoder attention launch refused";
    }
    /* an encoder layer's attention on operand images: 16 rows of a head in one workgroup, no score matrix.  All contexts it has registers for take it (three launches
     * and their score matrix else): at 1500 positions and six heads 97 -> 56 us a layer for one clip, 2106 -> 1194 us for 32 */
    bool takes_images(const float* q_w, const float* k_w, const float* o_w, int Tc, int d, int nh) {
        if ((a->fast && long_ok) || !long_ok || d % 128 || !tk_attention_images_fits(Tc, Tc, d, nh)) return false;
        for (const float* w : {q_w, k_w, o_w}) {
            const int i = a->model->tensor_of(w);
            if (i < 0 || !a->model->wt[(size_t)i]) return false;
        }
        return true;
    }
    void attend_images(const float* q, const float* k, const float* v, float* out, int B, int Tc, int d, int nh) {
        drop_image();
        float* img = image_for(out, B * Tc, d, d);
        if (!tk_launch_attention_images(q, k, v, img, B, nh, Tc, Tc, d, s)) a->launch_error = "attention launch refused";
    }
    /* the opt-in fast contraction's attention (TkAsr::fast): Q K^T, softmax and P V of a long pass in one kernel, no score matrix in HBM */
    bool attend_fused(const float* q, const float* k, const float* v, float* out, int B, int Tq, int Tk, int64_t q_bstride, int64_t kv_bstride, int d, int nh) {
        if (!a->fast || !long_ok || Tq < 2 || nh < 1 || d != nh * 64) return false;
        drop_image();
        return tk_launch_attention_h3(q, k, v, out, B, nh, Tq, Tk, q_bstride, kv_bstride, d, tk_divf(1.0f, tk_sqrtf(64.0f)), s);
    }
    void add_rows(float* x, const float* add, int rows, int D, int add_rows) { drop_image(); tk_launch_add_rows(x, add, rows, D, add_rows, s); }
    void embed_rows(const float* table, const float* pos, const int32_t* idx, const int32_t* pos_idx, int rows, int D, float* out) {
        drop_image();
        tk_launch_embed_rows(table, pos, idx, pos_idx, rows, D, out, s);
    }
    void argmax_rows(const float* x, int rows, int cols, int ld, int32_t* out) {
        drop_image();
        if (!a->pick.on) { tk_launch_argmax_rows(x, rows, cols, ld, out, s); return; }
        /* whisper.cpp's decoding policy: the step's token by temperature, its log-probability noted (step p of the decode loop, row b: slot p * B + b) */
        TkPick pk{a->pick.temp, a->pick.seed, (uint32_t)(a->pick.step * rows), a->pick.logprob ? a->pick.logprob + (size_t)a->pick.step * rows : nullptr};
        if (a->pick.filtered) {
            /* prompt positions before the last one produce logits nobody samples from: the rows' decode state must not move there */
            if (a->pick.step >= a->pick.first_step) {
                TkWhFilter f{a->pick.suppress, a->pick.state, a->pick.beg, a->pick.eot, a->pick.tid0};
                tk_launch_pick_rows_filtered(x, rows, cols, ld, out, pk, f, s);
            }
        } else {
            tk_launch_pick_rows(x, rows, cols, ld, out, pk, s);
        }
    }
    void frames(const int16_t* pcm, int B, int n_samples, int pcm_stride, int n_total, int T, const float* window, float* out) {
        drop_image();
        const int64_t per = (int64_t)T * TK_WH_NFFT;
        hipLaunchKernelGGL(k_frames, dim3((unsigned)((per + 255) / 256), 1, B), dim3(256), 0, s, pcm, n_samples, pcm_stride, n_total, T, window, out);
    }
    void power(const float* ri, int rows, int nb, float* out) {
        drop_image();
        const int64_t n = (int64_t)rows * nb;
        hipLaunchKernelGGL(k_power, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, ri, (int64_t)rows, nb, out);
    }
    void logmel_finish(float* mel, int B, int per_b) {
        float* part = alloc((size_t)B * TK_MEL_PARTS);
        hipLaunchKernelGGL(k_logmel_log, dim3(TK_MEL_PARTS, B), dim3(256), 0, s, mel, per_b, part);
        hipLaunchKernelGGL(k_logmel_clamp, dim3(TK_MEL_PARTS, B), dim3(256), 0, s, mel, per_b, part);
    }
};

/* sizing twin of the ops (counts arena floats for a given batch) */
struct TkAudioSizeOps {
    size_t used = 0, peak = 0;
    float* alloc(size_t n) { used += (n + 63) & ~(size_t)63; if (used > peak) peak = used; return nullptr; }
    int32_t* alloc_i32(size_t n) { return (int32_t*)alloc(n); }
    void gemm(const TkGemm& g) { /* the tiled path's activation image is scratch on top of the live allocations; fc1 adds fc2's image */
        if (!tk_tiled_gemm_applies(g)) return;
        size_t top = used + ((tk_tiled_gemm_scratch(g) + 63) & ~(size_t)63);
        if (g.c_feeds_linear) { TkGemm nx{}; nx.M = g.M; nx.K = g.N; top += (tk_tiled_gemm_scratch(nx) + 63) & ~(size_t)63; }
        if (top > peak) peak = top;
    }
    void image(int M, int K) { /* a producer's packed output (layer norm, decoder attention) */
        TkGemm g{};
        g.M = M; g.K = K;
        const size_t top = used + ((tk_tiled_gemm_scratch(g) + 63) & ~(size_t)63);
        if (top > peak) peak = top;
    }
    void im2col1d(const float*, int, int, int, int, int, int, int, float*) {}
    void layernorm(const float*, int rows, int D, const float*, const float*, float*) { image(rows, D); }
    void settle() {}
    void softmax_rows(float*, int, int, int) {}
    bool attend1(const float*, const float*, const float*, float*, int B, int, int64_t, int64_t, int, int d, int, float*, int) { image(B, d); return true; }
    bool takes_images(const float*, const float*, const float*, int, int, int) { return false; }
    void attend_images(const float*, const float*, const float*, float*, int, int, int, int) {}
    void attend_span(const float*, const float*, const float*, float*, int B, int n, int, bool, int64_t, int64_t, int, int d, int, float*, int) { image(B * n, d); }
    bool attend_fused(const float*, const float*, const float*, float*, int, int, int, int64_t, int64_t, int, int) { return false; } /* sized for the exact form */
    void add_rows(float*, const float*, int, int, int) {}
    void embed_rows(const float*, const float*, const int32_t*, const int32_t*, int, int, float*) {}
    void argmax_rows(const float*, int, int, int, int32_t*) {}
    void frames(const int16_t*, int, int, int, int, int, const float*, float*) {}
    void power(const float*, int, int, float*) {}
    void logmel_finish(float*, int B, int) { alloc((size_t)B * TK_MEL_PARTS); }
};

/* ---------------------------------------------------------------- model */

TkWhisperModel::~TkWhisperModel() {
    (void)hipSetDevice(device);
    for (auto p : w) if (p) (void)hipFree(p);
    for (auto p : wt) if (p) (void)hipFree(p);
}

int TkWhisperModel::tensor_of(const float* dev_ptr) const {
    for (size_t i = 0; i < w.size(); ++i) if (w[i] == dev_ptr) return (int)i;
    return -1;
}

bool TkWhisperModel::prepare_tiles() {
    HIPQ(hipSetDevice(device));
    if (wt.size() != man.t.size()) wt.assign(man.t.size(), nullptr);
    for (size_t i = 0; i < man.t.size(); ++i) {
        const bool linear = man.t[i].kind == TK_WK_LINEAR_W || (int)i == man.tok_emb; /* the token embedding is also the logits matrix */
        if (!linear || man.t[i].cols % 128 || man.t[i].rows < 16 || wt[i]) continue;
        HIPQ(hipMalloc((void**)&wt[i], tk_tiled_weight_bytes(man.t[i].rows, man.t[i].cols, 4)));
        tk_launch_tile_weights(w[i], 4, man.t[i].rows, man.t[i].cols, wt[i], nullptr);
    }
    HIPQ(hipDeviceSynchronize());
    return true;
}

bool TkWhisperModel::init(const TkWhisperHP& h, int dev) {
    hp = h;
    device = dev;
    if (h.n_audio_state % h.n_audio_head || h.n_text_state % h.n_text_head || h.n_audio_state % 2 || h.n_mels <= 0 || h.n_audio_ctx <= 0 ||
        h.n_text_ctx <= 0 || h.n_vocab <= 0) { error = "invalid Whisper hyper-parameters"; return false; }
    man = tk_whisper_manifest(h);
    HIPQ(hipSetDevice(device));
    w.assign(man.t.size(), nullptr);
    for (size_t i = 0; i < man.t.size(); ++i) HIPQ(hipMalloc((void**)&w[i], (size_t)man.t[i].rows * man.t[i].cols * 4));
    return true;
}

bool TkWhisperModel::set_tensor(int idx, const float* host, size_t n) {
    if (idx < 0 || idx >= (int)man.t.size() || n != (size_t)man.t[idx].rows * man.t[idx].cols) { error = "tensor index / size mismatch"; return false; }
    HIPQ(hipSetDevice(device));
    HIPQ(hipMemcpy(w[idx], host, n * 4, hipMemcpyHostToDevice));
    if ((size_t)idx < wt.size() && wt[(size_t)idx]) { /* keep the tiled twin current */
        tk_launch_tile_weights(w[idx], 4, man.t[idx].rows, man.t[idx].cols, wt[(size_t)idx], nullptr);
        HIPQ(hipDeviceSynchronize());
    }
    return true;
}

bool TkWhisperModel::fill_synthetic(uint64_t seed) {
    std::vector<float> buf;
    for (size_t i = 0; i < man.t.size(); ++i) {
        buf.resize((size_t)man.t[i].rows * man.t[i].cols);
        tk_whisper_fill_tensor(hp, man, (int)i, seed, buf.data());
        if (!set_tensor((int)i, buf.data(), buf.size())) return false;
    }
    return true;
}

bool TkWhisperModel::load_file(const char* path) {
    FILE* f = fopen(path, "rb");
    if (!f) { error = std::string("cannot open ") + path; return false; }
    char magic[8];
    int32_t n = 0;
    bool ok = fread(magic, 1, 8, f) == 8 && memcmp(magic, "TKWHSP1", 8) == 0 && fread(&n, 4, 1, f) == 1 && n == (int)man.t.size();
    std::vector<float> buf;
    /* the three frontend tables and the sinusoidal positions may be omitted (rows == 0 in the file): they are recomputed */
    for (int i = 0; ok && i < n; ++i) {
        int64_t d[2];
        ok = fread(d, 8, 2, f) == 2;
        if (!ok) break;
        if (d[0] == 0) {
            buf.resize((size_t)man.t[i].rows * man.t[i].cols);
            tk_whisper_fill_tensor(hp, man, i, 0, buf.data());
        } else {
            ok = d[0] == man.t[i].rows && d[1] == man.t[i].cols;
            buf.resize((size_t)d[0] * d[1]);
            ok = ok && fread(buf.data(), 4, buf.size(), f) == buf.size();
        }
        ok = ok && set_tensor(i, buf.data(), buf.size());
    }
    fclose(f);
    if (!ok && error.empty()) error = "not a TKWHSP1 container for this geometry";
    return ok;
}

bool TkWhisperModel::load_ggml(TkWhisperGgml& g) {
    std::vector<float> buf;
    for (int i = 0; i < (int)man.t.size(); ++i) {
        bool found = false;
        if (!g.read(man, i, &buf, &found)) {
            if (found) { error = g.error; return false; }
            if (i != man.hann && i != man.dft) { error = "tensor " + man.t[i].name + " is missing from the checkpoint"; return false; }
            buf.resize((size_t)man.t[i].rows * man.t[i].cols);
            tk_whisper_fill_tensor(hp, man, i, 0, buf.data()); /* analysis window and DFT twiddles are computed, not stored */
        }
        if (!set_tensor(i, buf.data(), buf.size())) return false;
    }
    return true;
}

/* ---------------------------------------------------------------- ASR */

TkAsr::~TkAsr() {
    if (model) (void)hipSetDevice(model->device);
    if (stream) (void)hipStreamSynchronize(stream);
    if (arena) (void)hipFree(arena);
    if (pcm_dev) (void)hipFree(pcm_dev);
    if (suppress_dev) (void)hipFree(suppress_dev);
    if (lp_dev) (void)hipFree(lp_dev);
    if (wh_state) (void)hipFree(wh_state);
    if (aux_stream) (void)hipStreamSynchronize(aux_stream);
    if (aux_host) (void)hipHostFree(aux_host);
    if (aux_ready) (void)hipEventDestroy(aux_ready);
    for (hipEvent_t e : aux_done) if (e) (void)hipEventDestroy(e);
    if (aux_stream) (void)hipStreamDestroy(aux_stream);
    if (stream) (void)hipStreamDestroy(stream);
}

/* all that a transcription of `mb` clips has in the arena at any time: the long passes, then the decode loop's token / position / arg-max tables and the
 * operand images of a step on top of what the long passes leave */
size_t tk_asr_arena_floats(const TkWhisperHP& hp, const TkWhManifest& man, int mb) {
    TkAudioSizeOps so;
    std::vector<float*> nullw(man.t.size(), nullptr);
    TkWhisperGraph<TkAudioSizeOps> g{hp, man, nullw.data()};
    float* ml = g.mel(so, nullptr, mb, 0, 0);
    float* enc = g.encode(so, ml, mb);
    const int rows = mb > TK_ASR_SPAN_ROWS ? mb : TK_ASR_SPAN_ROWS;
    auto st = g.begin_decode(so, enc, mb, rows);
    so.alloc_i32((size_t)3 * hp.n_text_ctx * mb);
    st.B = rows; /* a pass's widest images */
    g.decode_step(so, st, 0);
    return so.peak + 4096;
}

bool TkAsr::init(TkWhisperModel* m, int mb) {
    model = m;
    max_batch = mb;
    if (!m || mb < 1 || mb > 256) { error = "max_batch must be in [1,256]"; return false; }
    HIPQ(hipSetDevice(m->device));
    HIPQ(tk_create_perception_stream(&stream));
    arena_floats = tk_asr_arena_floats(m->hp, m->man, mb);
    if (!m->prepare_tiles()) { error = m->error; return false; }
    if (!tk_gemm_tiled_prepare_device() || !at1_prepare_device()) { error = "LDS opt-in of the tiled GEMM or of the decoder's attention failed"; return false; }
    HIPQ(hipMalloc((void**)&arena, arena_floats * 4));
    return true;
}

bool TkAsr::transcribe_policy(int B, const int16_t* pcm, int n_samples, const int32_t* prompt, int n_prompt, int n_steps, float temperature, uint64_t seed,
                              int32_t* tokens_out, float* logprobs_out) {
    if (!(temperature >= 0.0f) || model->hp.n_vocab > 65536) { error = "temperature must be >= 0 and the vocabulary at most 65536 tokens"; return false; }
    const int total = n_prompt + n_steps - 1;
    if (B < 1 || total < 1) { error = "nothing to decode"; return false; }
    if (hipSetDevice(model->device) != hipSuccess) { error = "hipSetDevice failed"; return false; }
    if (!ensure_decode_buffers()) return false;
    if (total > model->hp.n_text_ctx || B > max_batch) { error = "prompt + steps exceed the text context"; return false; }
    float* d_lp = lp_dev;
    pick.on = true; pick.temp = temperature; pick.seed = seed; pick.logprob = d_lp; pick.step = 0;
    const bool ok = transcribe(B, pcm, n_samples, prompt, n_prompt, n_steps, tokens_out, nullptr, nullptr, nullptr); /* synchronises the stream */
    pick.on = false;
    bool copied = true;
    if (ok && logprobs_out) {
        pick_logprobs.resize((size_t)total * B);
        copied = hipMemcpyAsync(pick_logprobs.data(), d_lp, pick_logprobs.size() * sizeof(float), hipMemcpyDeviceToHost, stream) == hipSuccess &&
                 hipStreamSynchronize(stream) == hipSuccess;
        for (int step = 0; copied && step < n_steps; ++step)
            for (int b = 0; b < B; ++b) logprobs_out[(size_t)b * n_steps + step] = pick_logprobs[(size_t)(n_prompt - 1 + step) * B + b];
    }
    pick.logprob = nullptr;
    if (ok && !copied) error = "copy of the log-probabilities failed";
    return ok && copied;
}

/* the decode's small device buffers, allocated ONCE per engine: nothing on a call's path allocates or frees device memory or uses the null stream —
 * hipFree synchronises the whole device and, issued while another host thread captures a hipGraph (the LLM's passes are captured at first use of
 * every row count), was the prime suspect of an intermittent process-wide stall on cold boxes (round 6, 64 cortices) */
bool TkAsr::ensure_decode_buffers() {
    const TkWhisperHP& h = model->hp;
    if (!lp_dev) HIPQ(hipMalloc((void**)&lp_dev, (size_t)max_batch * h.n_text_ctx * sizeof(float)));
    if (!suppress_dev) HIPQ(hipMalloc((void**)&suppress_dev, (size_t)h.n_vocab));
    if (!wh_state) HIPQ(hipMalloc((void**)&wh_state, (size_t)max_batch * TK_WH_STATE_INTS * sizeof(int32_t)));
    return true;
}

bool TkAsr::transcribe_ref(int B, const int16_t* pcm, int n_samples, const int32_t* n_samples_row, const int32_t* prompt, int n_prompt, int n_steps, float temperature,
                           uint64_t seed, const uint8_t* suppress, int32_t token_beg, int32_t token_eot, int32_t* tokens_out, float* logprobs_out, int32_t* result_len,
                           int32_t* status) {
    const TkWhisperHP& h = model->hp;
    if (!(temperature >= 0.0f) || h.n_vocab > 65536) { error = "temperature must be >= 0 and the vocabulary at most 65536 tokens"; return false; }
    if (B < 1 || B > max_batch || !suppress || !n_samples_row || token_beg <= token_eot || token_beg >= h.n_vocab) { error = "bad arguments to the reference-parameter decode"; return false; }
    const int total = n_prompt + n_steps - 1;
    if (total < 1) { error = "nothing to decode"; return false; }
    if (hipSetDevice(model->device) != hipSuccess) { error = "hipSetDevice failed"; return false; }
    if (!ensure_decode_buffers()) return false;
    if (total > h.n_text_ctx) { error = "prompt + steps exceed the text context"; return false; }
    if (suppress_host.size() != (size_t)h.n_vocab || memcmp(suppress_host.data(), suppress, (size_t)h.n_vocab) != 0) {
        HIPQ(hipStreamSynchronize(stream)); /* the previous decode may still read the table */
        suppress_host.assign(suppress, suppress + h.n_vocab);
        HIPQ(hipMemcpyAsync(suppress_dev, suppress_host.data(), (size_t)h.n_vocab, hipMemcpyHostToDevice, stream));
    }
    std::vector<int32_t> st0((size_t)B * TK_WH_STATE_INTS, 0);
    for (int b = 0; b < B; ++b) st0[(size_t)b * TK_WH_STATE_INTS + 7] = n_samples_row[b] / TK_WH_HOP; /* seek_end: the utterance in 10 ms frames */
    HIPQ(hipMemcpyAsync(wh_state, st0.data(), st0.size() * sizeof(int32_t), hipMemcpyHostToDevice, stream));
    float* d_lp = lp_dev;
    HIPQ(hipMemsetAsync(d_lp, 0, (size_t)total * B * sizeof(float), stream));
    pick.on = true; pick.temp = temperature; pick.seed = seed; pick.logprob = d_lp; pick.step = 0;
    pick.filtered = true; pick.first_step = n_prompt - 1; pick.suppress = suppress_dev; pick.state = wh_state; pick.beg = token_beg; pick.eot = token_eot;
    pick.tid0 = 50; /* max_initial_ts 1.0 s / (30 s / 1500 positions) */
    const bool ok = transcribe(B, pcm, n_samples, prompt, n_prompt, n_steps, tokens_out, nullptr, nullptr, nullptr); /* synchronises the stream */
    pick.on = false; pick.filtered = false;
    bool copied = true;
    std::vector<int32_t> st1((size_t)B * TK_WH_STATE_INTS);
    if (ok) {
        pick_logprobs.resize((size_t)total * B);
        copied = hipMemcpyAsync(pick_logprobs.data(), d_lp, pick_logprobs.size() * sizeof(float), hipMemcpyDeviceToHost, stream) == hipSuccess &&
                 hipMemcpyAsync(st1.data(), wh_state, st1.size() * sizeof(int32_t), hipMemcpyDeviceToHost, stream) == hipSuccess &&
                 hipStreamSynchronize(stream) == hipSuccess;
        for (int b = 0; copied && b < B; ++b) {
            const int32_t* sb = &st1[(size_t)b * TK_WH_STATE_INTS];
            if (status) status[b] = sb[6];
            /* n_steps reached before the row ended: every sampled token counts (whisper.cpp would go on to n_text_ctx / 2 - 4 tokens) */
            if (result_len) result_len[b] = sb[6] == 0 ? sb[0] : sb[5];
            for (int step = 0; logprobs_out && step < n_steps; ++step) logprobs_out[(size_t)b * n_steps + step] = pick_logprobs[(size_t)(n_prompt - 1 + step) * B + b];
        }
    }
    pick.logprob = nullptr;
    if (ok && !copied) error = "copy of the decode state failed";
    return ok && copied;
}

/* pinned memory for a call's outputs beside its tokens: kept, so that it is pinned a few times in a context's life, and 64 MB at most; calls that have more to copy take it
 * in turns (aux_copy) */
bool TkAsr::aux_reserve(size_t floats) {
    if (!aux_stream) HIPQ(tk_create_perception_stream(&aux_stream));
    if (!aux_ready) HIPQ(hipEventCreateWithFlags(&aux_ready, hipEventDisableTiming));
    for (hipEvent_t& e : aux_done)
        if (!e) HIPQ(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    size_t want = TK_ASR_AUX_MIN;
    while (want < floats && want < TK_ASR_AUX_MAX) want *= 2;
    if (want <= aux_floats) return true;
    if (aux_host) (void)hipHostFree(aux_host);
    aux_host = nullptr;
    aux_floats = 0;
    HIPQ(hipHostMalloc((void**)&aux_host, want * 4, hipHostMallocDefault));
    aux_floats = want;
    return true;
}

/* device arrays to the caller's memory through two halves of `room` pinned floats: one is on its way while the other is emptied */
bool TkAsr::aux_copy(const Copy* parts, int n, float* through, size_t room) {
    const size_t half = room / 2;
    Copy busy[2] = {};
    int slot = 0;
    auto empty = [&](int i) {
        if (busy[i].n == 0) return true;
        HIPQ(hipEventSynchronize(aux_done[i]));
        memcpy(busy[i].to, busy[i].from, busy[i].n * 4);
        busy[i].n = 0;
        return true;
    };
    for (int p = 0; p < n; ++p)
        for (size_t at = 0; at < parts[p].n; at += half, slot ^= 1) {
            if (!empty(slot)) return false;
            const size_t count = parts[p].n - at < half ? parts[p].n - at : half;
            float* mid = through + slot * half;
            HIPQ(hipMemcpyAsync(mid, parts[p].from + at, count * 4, hipMemcpyDeviceToHost, aux_stream));
            HIPQ(hipEventRecord(aux_done[slot], aux_stream));
            busy[slot] = Copy{parts[p].to + at, mid, count};
        }
    return empty(slot) && empty(slot ^ 1);
}

bool TkAsr::transcribe(int B, const int16_t* pcm, int n_samples, const int32_t* prompt, int n_prompt, int n_steps, int32_t* tokens_out,
                       float* mel_out, float* enc_out, float* first_logits) {
    const TkWhisperHP& h = model->hp;
    if (B < 1 || B > max_batch) { error = "batch larger than the ASR context was created for"; return false; }
    if (n_samples < 0 || n_samples > h.n_samples()) { error = "audio longer than the model window"; return false; }
    if (n_prompt < 1 || n_prompt + n_steps > h.n_text_ctx) { error = "prompt + steps exceed the text context"; return false; }
    HIPQ(hipSetDevice(model->device));
    const size_t n_mel = mel_out ? (size_t)B * h.n_frames() * h.n_mels : 0, n_enc = enc_out ? (size_t)B * h.n_audio_ctx * h.n_audio_state : 0, n_lg = first_logits ? (size_t)B * h.n_vocab : 0;
    if (n_mel + n_enc + n_lg > 0 && aux_host && !aux_reserve(n_mel + n_enc + n_lg)) return false; /* (may give memory back, which waits for the device) */
    size_t need = (size_t)B * (n_samples > 0 ? n_samples : 1);
    if (need > pcm_cap) need = (size_t)max_batch * (size_t)h.n_samples(); /* once: the engine's whole batch of full windows (0.96 MB each) */
    if (need > pcm_cap) {
        if (pcm_dev) (void)hipFree(pcm_dev);
        pcm_dev = nullptr;
        HIPQ(hipMalloc((void**)&pcm_dev, need * 2));
        pcm_cap = need;
    }
    if (n_samples > 0) HIPQ(hipMemcpyAsync(pcm_dev, pcm, (size_t)B * n_samples * 2, hipMemcpyHostToDevice, stream));
    arena_used = 0;
    launch_error.clear();
    TkAudioGpuOps ops{this, stream};
    TkWhisperGraph<TkAudioGpuOps> g{h, model->man, model->w.data()};
    ops.long_ok = true;
    float* ml = g.mel(ops, pcm_dev, B, n_samples, n_samples);
    float* enc = g.encode(ops, ml, B);
    auto st = g.begin_decode(ops, enc, B, B > TK_ASR_SPAN_ROWS ? B : TK_ASR_SPAN_ROWS);
    ops.long_ok = false;
    HIPQ(hipGetLastError());
    /* The mel, the encoder's output and the first logits travel to pinned memory on a stream of their own, and from there to the caller while the decoder's steps run:
     * copies to pageable memory in between held back the launches behind them (one clip: 0.5 ms of 7).  What does not fit goes in pieces once the steps are enqueued; logits
     * that take more than half of the pinned memory go straight to the caller's. */
    if (n_mel + n_enc + n_lg > 0 && !aux_reserve(n_mel + n_enc + n_lg)) return false; /* the first time: pinned while the encoder runs */
    float* const lg_at = n_lg <= aux_floats / 2 ? aux_host : first_logits;
    float* const mel_at = aux_host + (lg_at == aux_host ? n_lg : 0);
    const size_t room = aux_floats - (size_t)(mel_at - aux_host);
    const bool whole = n_mel + n_enc <= room;
    struct Wait { TkAsr* a; ~Wait() { if (a->aux_stream) (void)hipStreamSynchronize(a->aux_stream); } } wait{this}; /* whatever happens below */
    if (n_mel + n_enc > 0) {
        HIPQ(hipEventRecord(aux_ready, stream));
        HIPQ(hipStreamWaitEvent(aux_stream, aux_ready, 0));
        if (whole) {
            if (n_mel) HIPQ(hipMemcpyAsync(mel_at, ml, n_mel * 4, hipMemcpyDeviceToHost, aux_stream));
            if (n_enc) HIPQ(hipMemcpyAsync(mel_at + n_mel, enc, n_enc * 4, hipMemcpyDeviceToHost, aux_stream));
            HIPQ(hipEventRecord(aux_done[0], aux_stream));
        }
    }
    /* The whole greedy loop is enqueued without touching the host: prompt tokens and positions sit in device tables uploaded once, step p
     * reads its token from the prompt table or from the previous step's arg-max slot and writes its own arg-max into slot p of an output
     * table; one copy and one synchronisation at the end.  (A synchronisation and three small copies per step made the 16 steps of 32
     * utterances 1.2 ms each on a 0.3 ms GPU workload.) */
    const int total = n_prompt + n_steps - 1; /* the last generated token is not fed back */
    const size_t tab_ints = ((size_t)n_prompt + 2 * (size_t)total) * B;
    ops.drop_image();
    if (arena_used + tab_ints + 64 > arena_floats) { error = "ASR arena too small for the decode tables"; return false; }
    int32_t* tab = ops.alloc_i32(tab_ints); /* [n_prompt][B] prompt tokens, [total][B] positions, [total][B] arg-max slots */
    int32_t* tok_tab = tab;
    int32_t* pos_tab = tab + (size_t)n_prompt * B;
    int32_t* out_tab = pos_tab + (size_t)total * B;
    std::vector<int32_t> host_tab(((size_t)n_prompt + total) * B);
    for (int p = 0; p < n_prompt; ++p)
        for (int b = 0; b < B; ++b) host_tab[(size_t)p * B + b] = prompt[p];
    for (int p = 0; p < total; ++p)
        for (int b = 0; b < B; ++b) host_tab[((size_t)n_prompt + p) * B + b] = p;
    HIPQ(hipMemcpyAsync(tok_tab, host_tab.data(), host_tab.size() * 4, hipMemcpyHostToDevice, stream));
    int steps_run = n_steps; /* sampled positions really enqueued */
    std::vector<int32_t> st_host;
    /* the prompt's positions several at a time (a pass is bound by its chains and launches, whose number this halves for a prompt of two: 17 positions
     * of one clip 230 us less of 4.8 ms, of 32 clips 320 us of 6.5); logits of the sampled position alone */
    const int span = TkAudioGpuOps::span(h, B);
    for (int p = 0; p < total; ++p) {
        st.tok = p < n_prompt ? tok_tab + (size_t)p * B : out_tab + (size_t)(p - 1) * B;
        st.pos = pos_tab + (size_t)p * B;
        const int left = (n_prompt < total ? n_prompt : total) - p, n = left < span ? left : span;
        const int at = n > 1 ? p + n - 1 : p; /* the pass's last position */
        st.next = out_tab + (size_t)at * B;
        pick.step = at;
        if (n > 1 || (n == 1 && at < n_prompt - 1)) g.prompt_span(ops, st, p, n, at == n_prompt - 1);
        else g.decode_step(ops, st, p);
        p = at;
        if (p == n_prompt - 1 && first_logits) {
            ops.flush();
            HIPQ(hipMemcpyAsync(lg_at, st.logits, n_lg * 4, hipMemcpyDeviceToHost, stream)); /* (the next step writes them again) */
        }
        /* the reference-parameter decode ends where the rows' own bookkeeping says (whisper.cpp: up to n_text_ctx / 2 - 4 tokens): every 16 sampled
         * positions the rows' status words are read; once every row has completed or failed nothing more is enqueued — a finished row emits eot and
         * stands still anyway (k_pick_rows_filtered), so stopping early changes no token */
        const int step = p - (n_prompt - 1);
        if (pick.filtered && step >= 0 && (step + 1) % 16 == 0 && p + 1 < total) {
            ops.flush();
            st_host.resize((size_t)B * TK_WH_STATE_INTS);
            HIPQ(hipMemcpyAsync(st_host.data(), pick.state, st_host.size() * sizeof(int32_t), hipMemcpyDeviceToHost, stream));
            HIPQ(hipStreamSynchronize(stream));
            bool all_done = true;
            for (int b = 0; b < B; ++b) all_done = all_done && st_host[(size_t)b * TK_WH_STATE_INTS + 6] != 0;
            if (all_done) { steps_run = step + 1; break; }
        }
    }
    ops.flush();
    if (!whole) {
        const Copy parts[2] = {{mel_out, ml, n_mel}, {enc_out, enc, n_enc}};
        if (!aux_copy(parts, 2, mel_at, room)) return false;
    } else if (n_mel + n_enc > 0) {
        HIPQ(hipEventSynchronize(aux_done[0]));
        if (n_mel) memcpy(mel_out, mel_at, n_mel * 4);
        if (n_enc) memcpy(enc_out, mel_at + n_mel, n_enc * 4);
    }
    std::vector<int32_t> outs((size_t)steps_run * B);
    HIPQ(hipMemcpyAsync(outs.data(), out_tab + (size_t)(n_prompt - 1) * B, outs.size() * 4, hipMemcpyDeviceToHost, stream));
    HIPQ(hipStreamSynchronize(stream)); /* host_tab and outs live until here */
    if (n_lg && lg_at != first_logits) memcpy(first_logits, lg_at, n_lg * 4);
    for (int step = 0; step < n_steps; ++step)
        for (int b = 0; b < B; ++b) tokens_out[(size_t)b * n_steps + step] = step < steps_run ? outs[(size_t)step * B + b] : pick.eot;
    HIPQ(hipGetLastError());
    if (!launch_error.empty()) { error = launch_error; return false; }
    return true;
}

/* ---------------------------------------------------------------- VAD */

TkVadModel::~TkVadModel() {
    (void)hipSetDevice(device);
    if (stream) (void)hipStreamSynchronize(stream);
    float* ptrs[] = {w1, b1, w2, b2};
    for (float* q : ptrs) if (q) (void)hipFree(q);
    for (Slot& s : slots) {
        if (s.x) (void)hipHostFree(s.x);
        if (s.done) (void)hipEventDestroy(s.done);
    }
    if (stream) (void)hipStreamDestroy(stream);
}

bool TkVadModel::init(int dev, int win, int hid) {
    device = dev; window = win; hidden = hid;
    if (win < 4 || (win & 3) || hid < 1 || hid > 64) { error = "VAD windows are whole groups of four samples, its hidden layer has at most 64 units"; return false; }
    HIPQ(hipSetDevice(device));
    HIPQ(hipMalloc((void**)&w1, (size_t)win * hid * 4));
    HIPQ(hipMalloc((void**)&b1, (size_t)hid * 4));
    HIPQ(hipMalloc((void**)&w2, (size_t)hid * 4));
    HIPQ(hipMalloc((void**)&b2, 4));
    return true;
}

bool TkVadModel::fill_synthetic(uint64_t seed) {
    std::vector<float> a((size_t)hidden * window), b(hidden), c(hidden), d(1);
    tk_vad_synth(seed, window, hidden, a.data(), b.data(), c.data(), d.data());
    /* [hidden][window] -> [window / 4][hidden][4]: a lane per hidden unit reads four of its weights at a time */
    std::vector<float> t(a.size());
    for (int h = 0; h < hidden; ++h)
        for (int k = 0; k < window; ++k) t[((size_t)(k >> 2) * hidden + h) * 4 + (k & 3)] = a[(size_t)h * window + k];
    HIPQ(hipSetDevice(device));
    HIPQ(hipMemcpy(w1, t.data(), t.size() * 4, hipMemcpyHostToDevice));
    HIPQ(hipMemcpy(b1, b.data(), b.size() * 4, hipMemcpyHostToDevice));
    HIPQ(hipMemcpy(w2, c.data(), c.size() * 4, hipMemcpyHostToDevice));
    HIPQ(hipMemcpy(b2, d.data(), 4, hipMemcpyHostToDevice));
    return true;
}

/* A workgroup per window, a lane per hidden unit: its chain over the window, relu, then one lane's chain over the hidden units.  Windows are read from, and probabilities
 * written to, pinned host memory: one launch and one wait make a call.  What is left is the launch, the trip over the bus and the chain of `window` fmas. */
/* Windows of up to 480 samples (16 kHz): NW waves of P groups of four.  The chain goes from wave to wave: each has its P groups of four weights, all asked for at once, and then its share of the window in
 * registers before its turn, so that a turn is its fmas and a hand-over through LDS.  One wave that fetched all weights had 40 groups in flight and read the window from LDS beside
 * the chain (k_vad_long): load, chain, end 3.0, 6.6, 0.9 us of a window of 480, here 2.4, 1.8, 1.0; 33 windows from call to result 23.0 -> 17.8 us, 256 34.4 -> 30.8.  Weights in
 * LDS 19.8 (an LDS read holds the wave's issue as long as four fmas), all 480 in one wave's registers, half of them accumulation registers, 19.8; five waves of 26 groups 18.05,
 * eight of 16 18.3. */
__global__ __launch_bounds__(256) void k_vad(const float* x, int window, int hidden, const float* __restrict__ w1, const float* __restrict__ b1, const float* __restrict__ w2,
                                             const float* __restrict__ b2, float* prob) {
    constexpr int NW = 4, P = 30;
    __shared__ __attribute__((aligned(16))) float win[4 * NW * P], sums[64], w2s[64];
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), groups = window >> 2, unit = lane < hidden ? lane : hidden - 1;
    const int g0 = wave * P;
    at1_f32x4 mine = {0.0f, 0.0f, 0.0f, 0.0f};
    if (t < groups) mine = ((const at1_f32x4*)(x + (int64_t)blockIdx.x * window))[t];
    float w2v = 0.0f, b1v = 0.0f, b2v = 0.0f;
    if (wave == 0) w2v = w2[unit];
    if (wave == NW - 1) { b1v = b1[unit]; b2v = b2[0]; }
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc((void*)w1, 0, (unsigned)(window * hidden * 4), 0x00020000);
    at1_f32x4 w[P], v[P];
#pragma unroll
    for (int i = 0; i < P; ++i) /* past the window: its last group again */
        w[i] = __builtin_bit_cast(at1_f32x4, __builtin_amdgcn_raw_buffer_load_b128(wr, unit * 16, (g0 + i < groups ? g0 + i : groups - 1) * hidden * 16, 0));
    if (t < NW * P) ((at1_f32x4*)win)[t] = mine;
    if (wave == 0) w2s[lane] = w2v;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < P; ++i) v[i] = ((const at1_f32x4*)win)[g0 + i];
    float acc = 0.0f;
#pragma unroll 1
    for (int s = 0; s < NW; ++s) {
        if (s == wave) {
            if (s) acc = sums[lane];
            if (g0 + P <= groups) {
#pragma unroll
                for (int i = 0; i < P; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc = tk_fmaf(v[i][j], w[i][j], acc);
            } else {
#pragma unroll
                for (int i = 0; i < P; ++i)
                    if (g0 + i < groups)
#pragma unroll
                        for (int j = 0; j < 4; ++j) acc = tk_fmaf(v[i][j], w[i][j], acc);
            }
            if (s == NW - 1) acc = tk_fmaxf(acc + b1v, 0.0f);
            sums[lane] = acc;
        }
        if (s < NW - 1) __syncthreads();
    }
    if (wave < NW - 1) return;
    float a = 0.0f;
#pragma unroll
    for (int k0 = 0; k0 < 64; k0 += 16) {
        at1_f32x4 hv[4], wv[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) { hv[i] = ((const at1_f32x4*)sums)[k0 / 4 + i]; wv[i] = ((const at1_f32x4*)w2s)[k0 / 4 + i]; }
#pragma unroll
        for (int i = 0; i < 16; ++i)
            if (k0 + i < hidden) a = tk_fmaf(hv[i >> 2][i & 3], wv[i >> 2][i & 3], a);
    }
    if (lane == 0) prob[blockIdx.x] = tk_sigmoidf(a + b2v);
}

/* windows of more than 480 samples (48 kHz): three waves a SIMD hold no such shares */
#define TK_VAD_AHEAD 20 /* groups of four weights on their way, twice */
__global__ __launch_bounds__(64) void k_vad_long(const float* x, int window, int hidden, const float* __restrict__ w1, const float* __restrict__ b1, const float* __restrict__ w2,
                                                 const float* __restrict__ b2, float* prob) {
    extern __shared__ __attribute__((aligned(16))) float vad_lds[];
    float* hs = vad_lds + window; /* [hidden] behind the window */
    const int t = threadIdx.x, groups = window >> 2, unit = t < hidden ? t : hidden - 1;
    const at1_f32x4* wp = (const at1_f32x4*)w1 + unit;
    at1_f32x4 w[2][TK_VAD_AHEAD];
    auto load = [&](int set, int g0) { /* past the end: the last group again */
#pragma unroll
        for (int i = 0; i < TK_VAD_AHEAD; ++i) w[set][i] = wp[(g0 + i < groups ? g0 + i : groups - 1) * hidden];
    };
    load(0, 0);
    const at1_f32x4* row = (const at1_f32x4*)(x + (int64_t)blockIdx.x * window);
    for (int i = t; i < groups; i += 64) ((at1_f32x4*)vad_lds)[i] = row[i];
    __syncthreads();
    float acc = 0.0f;
    for (int g0 = 0; g0 < groups; g0 += 2 * TK_VAD_AHEAD) {
#pragma unroll
        for (int set = 0; set < 2; ++set) {
            const int base = g0 + set * TK_VAD_AHEAD;
            load(set ^ 1, base + TK_VAD_AHEAD);
#pragma unroll
            for (int i = 0; i < TK_VAD_AHEAD; ++i)
                if (base + i < groups) {
                    const at1_f32x4 v = ((const at1_f32x4*)vad_lds)[base + i];
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc = tk_fmaf(v[j], w[set][i][j], acc);
                }
        }
    }
    if (t < hidden) hs[t] = tk_fmaxf(acc + b1[unit], 0.0f);
    __syncthreads();
    if (t == 0) {
        float a = 0.0f;
        for (int k = 0; k < hidden; ++k) a = tk_fmaf(hs[k], w2[k], a);
        prob[blockIdx.x] = tk_sigmoidf(a + b2[0]);
    }
}

/* pinned memory for one slot's windows and, behind them, their probabilities */
bool TkVadModel::reserve(Slot& s, int n) {
    if (n > s.cap) {
        if (s.x) (void)hipHostFree(s.x); /* (a slot grows between calls or before its first use) */
        s.x = nullptr;
        s.cap = 0;
        const int want = n < 128 ? 128 : n;
        HIPQ(hipHostMalloc((void**)&s.x, (size_t)want * (window + 1) * 4, hipHostMallocDefault));
        s.cap = want;
    }
    if (!s.done) HIPQ(hipEventCreateWithFlags(&s.done, hipEventDisableTiming));
    return true;
}

bool TkVadModel::infer(const float* windows_host, int n, float* prob_host) {
    if (n <= 0) return true;
    HIPQ(hipSetDevice(device));
    if (!stream) HIPQ(tk_create_perception_stream(&stream));
    auto launch = [&](Slot& s, int count) {
        float* prob = s.x + (size_t)s.cap * window;
        if (window <= 480) hipLaunchKernelGGL(k_vad, dim3(count), dim3(256), 0, stream, s.x, window, hidden, w1, b1, w2, b2, prob);
        else hipLaunchKernelGGL(k_vad_long, dim3(count), dim3(64), (size_t)(window + hidden) * 4, stream, s.x, window, hidden, w1, b1, w2, b2, prob);
        return hipGetLastError();
    };
    if (n <= TK_VAD_CHUNK) {
        Slot& s = slots[0];
        if (!reserve(s, n)) return false;
        memcpy(s.x, windows_host, (size_t)n * window * 4);
        HIPQ(launch(s, n));
        HIPQ(hipStreamSynchronize(stream));
        memcpy(prob_host, s.x + (size_t)s.cap * window, (size_t)n * 4);
        return true;
    }
    /* many windows: in turn through two slots, so that one is filled while the other is worked on */
    int from[2] = {0, 0}, count[2] = {0, 0};
    auto fetch = [&](int i) {
        HIPQ(hipEventSynchronize(slots[i].done));
        memcpy(prob_host + from[i], slots[i].x + (size_t)slots[i].cap * window, (size_t)count[i] * 4);
        count[i] = 0;
        return true;
    };
    int at = 0, i = 0;
    for (; at < n; at += TK_VAD_CHUNK, i ^= 1) {
        Slot& s = slots[i];
        if ((count[i] > 0 && !fetch(i)) || !reserve(s, TK_VAD_CHUNK)) { (void)hipStreamSynchronize(stream); return false; }
        from[i] = at;
        count[i] = n - at < TK_VAD_CHUNK ? n - at : TK_VAD_CHUNK;
        memcpy(s.x, windows_host + (size_t)at * window, (size_t)count[i] * window * 4);
        const hipError_t e = launch(s, count[i]);
        if (e != hipSuccess || hipEventRecord(s.done, stream) != hipSuccess) { (void)hipStreamSynchronize(stream); error = "launching the VAD failed"; return false; }
    }
    for (int k = 0; k < 2; ++k)
        if (count[k] > 0 && !fetch(k)) { (void)hipStreamSynchronize(stream); return false; }
    return true;
}
