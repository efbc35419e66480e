/* tk_gemm_image.hip — see tk_gemm_image.h */
#include "tk_gemm_image.h"

#include <algorithm>
#include <atomic>
#include <mutex>
#include <type_traits>

#include "tk_image_device.h"

namespace {

__device__ __forceinline__ tk_v4u ldg16(const uint8_t* p) { return *(const tk_v4u*)p; }
__device__ __forceinline__ tk_v4u ldg16_stream(const uint8_t* p) { return __builtin_nontemporal_load((const tk_v4u*)p); }

/* one accumulator tile (lane: row = l % 16 of the M-tile, columns n .. n + 3) to its f32 destination */
template <typename T>
__device__ __forceinline__ void store_f32(const TkImgGemm& a, int64_t row, int n, tk_v4f v) {
    float* o = a.out + row * a.ldc + n;
    if (n + 3 < a.n_valid && (a.ldc & 3) == 0) *(tk_v4f*)o = v;
    else
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (n + r < a.n_valid) o[r] = v[r];
    if (a.copy_img && n + 3 >= a.copy0 && n < a.copy1)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (n + r >= a.copy0 && n + r < a.copy1) tk_img_put((T*)a.copy_img, row, n + r - a.copy0, a.copy_ktiles, v[r]);
}

/* gate and up tiles of the same 16 columns -> the gated activation in the next product's operand image: M-tile mt, columns 16 ct .. 16 ct + 15, both the same for all lanes, so that
 * the address is a scalar one and a lane's constant offset (row and column of a lane through tk_img_index are two 64-bit products each: 2047 x 28672 x 4096
 * (gate | up) 429 -> 426 us).
 * expf and the division, some forty instructions of an element that becomes bf16 next, stand between a block's last product and the next block's first.  The hardware's exponential and
 * reciprocal would take 21 us off that product, but with the exponent's rounding they are up to |z| units of 2^-24 off. */
template <typename T>
__device__ __forceinline__ void store_act(const TkImgGemm& a, int mt, int ct, int lane, tk_v4f gate, tk_v4f up) {
    constexpr int PER = TkImg<T>::KT / 16, EP = TkImg<T>::EP; /* tiles of 16 columns in a k tile */
    const int n = ct * 16 + 4 * (lane >> 4);
    tk_v4f h;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        float y;
        if (a.act_clamped) {
            const float g = fminf(gate[r], a.act_limit), u = fminf(fmaxf(up[r], -a.act_limit), a.act_limit);
            y = g * tk_sigmoid32(a.act_slope * g) * (u + a.act_shift);
        } else {
            y = tk_silu32(gate[r]) * up[r];
        }
        h[r] = n + r < a.act_valid ? y : 0.0f;
    }
    T* const tile = (T*)a.act_img + ((size_t)mt * a.act_ktiles + ct / PER) * (1024 / sizeof(T)) + ct % PER * 256;
    if (n < a.act_valid) tk_img_put4_at(tile + ((lane & 15) + 16 * ((lane >> 4) * 4 / EP)) * EP + (lane >> 4) * 4 % EP, h);
}

/* ---- skinny: MT M-tiles of rows, NT column tiles per workgroup, K interleaved over the waves in pieces of U tiles ----
 * Loads of three M-tiles are three (33 .. 48 rows; four, one of them twice: 40 rows x 2048 x 16384 gate and up 17.2 -> 15.8 us, x 32000 34.2 -> 28.6).
 * PARTS = 2: the waves of a column tile in two workgroups (skinny_parts), each wave with two pieces on their way.  The first workgroup adds its waves up in slab 0, each wave
 * of the second has a slab of its own: added in ascending order, they are the sum that one workgroup of all waves makes.
 * CHAINS = 2: each wave makes the sums of two waves one behind the other, so that four waves give the bits of eight. */
template <typename T, int MT, int NT, int WAVES, int PARTS, int CHAINS, bool SWIGLU, bool GROUPED>
__global__ __launch_bounds__(64 * WAVES) void k_gemm_skinny(TkImgGemm a) {
    static_assert(PARTS == 1 || (PARTS == 2 && !SWIGLU && !GROUPED), "slabs are of plain products");
    static_assert(CHAINS == 1 || (CHAINS == 2 && PARTS == 1), "two chains a wave: of products in one part");
    constexpr int U = MT >= 3 ? 2 : 4, STEP = PARTS * CHAINS * WAVES * U, AHEAD = PARTS;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ktiles = a.K / TkImg<T>::KT;
    int m0 = blockIdx.y * MT, mlive = (a.nrows + 15) / 16 - m0;
    const uint8_t* wbase = (const uint8_t*)a.w;
    if (GROUPED) {
        if ((int)blockIdx.y >= *a.n_blocks) return;
        const TkImgBlock b = a.blocks[blockIdx.y];
        m0 = b.tile0; mlive = b.ntiles;
        wbase += (size_t)b.group * a.group_bytes;
    }
    if (mlive > MT) mlive = MT;
    const int ntot = a.N / 16, n0 = blockIdx.x * NT;
    const uint8_t* wp[NT];
    const uint8_t* ap[MT];
#pragma unroll
    for (int n = 0; n < NT; ++n) wp[n] = wbase + (size_t)(n0 + n < ntot ? n0 + n : ntot - 1) * ktiles * 1024 + lane * 16;
#pragma unroll
    for (int m = 0; m < MT; ++m) ap[m] = (const uint8_t*)a.a + (size_t)(m0 + (m < mlive ? m : 0)) * ktiles * 1024 + lane * 16;
    tk_v4f acc[NT][MT];
    auto clear = [&] {
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int m = 0; m < MT; ++m) acc[n][m] = tk_v4f{0.0f, 0.0f, 0.0f, 0.0f};
    };
    clear();
    const tk_v4u zero = {0, 0, 0, 0};
    tk_v4u wq[AHEAD][U][NT], aq[AHEAD][U][MT];
    /* tiles past the end re-read the last one against a zero activation: no branch around a load */
    auto load = [&](int p, int c) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int kt = c + u < ktiles ? c + u : ktiles - 1;
#pragma unroll
            for (int n = 0; n < NT; ++n) wq[p][u][n] = ldg16_stream(wp[n] + (size_t)kt * 1024);
#pragma unroll
            for (int m = 0; m < MT; ++m) aq[p][u][m] = ldg16(ap[m] + (size_t)kt * 1024);
        }
    };
    int c = ((PARTS > 1 ? (int)blockIdx.z * WAVES : 0) + wave) * U;
#pragma unroll
    for (int p = 0; p < AHEAD; ++p)
        if (PARTS > 1 || c < ktiles) load(p, c + p * STEP);
    auto walk = [&](int c, int after /* where the next chain starts */) {
        while (c < ktiles) {
#pragma unroll
            for (int p = 0; p < AHEAD; ++p) {
                tk_v4u w0[U][NT], a0[U][MT];
#pragma unroll
                for (int u = 0; u < U; ++u) {
#pragma unroll
                    for (int n = 0; n < NT; ++n) w0[u][n] = wq[p][u][n];
#pragma unroll
                    for (int m = 0; m < MT; ++m) a0[u][m] = c + u < ktiles ? aq[p][u][m] : zero;
                }
                const int next = c + AHEAD * STEP;
                if (PARTS > 1 || next < ktiles) load(p, next);
                else if (CHAINS > 1 && after < ktiles) load(p, after);
#pragma unroll
                for (int u = 0; u < U; ++u)
#pragma unroll
                    for (int n = 0; n < NT; ++n)
#pragma unroll
                        for (int m = 0; m < MT; ++m) acc[n][m] = TkImg<T>::mma(w0[u][n], a0[u][m], acc[n][m]);
                c += STEP;
                if (c >= ktiles) break;
            }
        }
    };
    if (CHAINS == 1) walk(c, ktiles);
    if (PARTS > 1 && blockIdx.z) {
        a.out += (size_t)(1 + wave) * a.slab_floats;
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const int64_t row = (int64_t)(m0 + m) * 16 + (lane & 15);
                if (m < mlive && row < a.nrows && n0 + n < ntot) store_f32<T>(a, row, (n0 + n) * 16 + 4 * (lane >> 4), acc[n][m]);
            }
        return;
    }
    /* partial sums of the waves, ascending */
    tk_v4f* red = (tk_v4f*)lds;
    auto put = [&] {
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int m = 0; m < MT; ++m) red[((wave * NT + n) * MT + m) * 64 + lane] = acc[n][m];
        __syncthreads();
    };
    auto fold = [&](tk_v4f s, int w, int n, int m) {
        for (; w < WAVES; ++w) s += red[((w * NT + n) * MT + m) * 64 + lane];
        return s;
    };
    constexpr int HALVES = SWIGLU ? 2 : 1, UNITS = NT / HALVES * MT, MINE = (UNITS + WAVES - 1) / WAVES;
    tk_v4f first[CHAINS > 1 ? MINE : 1][HALVES]; /* the sum of the first chains */
    if (CHAINS == 1) put();
    else {
#pragma unroll 1
        for (int r = 0; r < CHAINS; ++r) {
            walk(c, r + 1 < CHAINS ? c + WAVES * U : ktiles);
            if (r) __syncthreads();
            put();
            if (r + 1 == CHAINS) break;
#pragma unroll
            for (int j = 0; j < MINE; ++j) {
                const int i = wave + j * WAVES < UNITS ? wave + j * WAVES : 0;
#pragma unroll
                for (int h = 0; h < HALVES; ++h) first[CHAINS > 1 ? j : 0][h] = fold(red[((HALVES * (i / MT) + h) * MT + i % MT) * 64 + lane], 1, HALVES * (i / MT) + h, i % MT);
            }
            clear();
            c += WAVES * U;
        }
    }
#pragma unroll
    for (int j = 0; j < MINE; ++j) {
        const int i = wave + j * WAVES, n = i / MT, m = i % MT;
        if (i >= UNITS) break;
        const int64_t row = (int64_t)(m0 + m) * 16 + (lane & 15);
        if (m >= mlive || (!GROUPED && row >= a.nrows)) continue;
        auto total = [&](int h) {
            return CHAINS > 1 ? fold(first[CHAINS > 1 ? j : 0][h], 0, HALVES * n + h, m) : fold(red[((HALVES * n + h) * MT + m) * 64 + lane], 1, HALVES * n + h, m);
        };
        if (SWIGLU) {
            if (n0 + 2 * n < ntot) store_act<T>(a, m0 + m, n0 / 2 + n, lane, total(0), total(HALVES - 1));
        } else if (n0 + n < ntot) {
            store_f32<T>(a, row, (n0 + n) * 16 + 4 * (lane >> 4), total(0));
        }
    }
}

/* s_waitcnt vmcnt(N): all but this wave's N youngest vector-memory requests are done */
template <int N> __device__ __forceinline__ void wait_vm() { __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | (N >> 4) << 14); }

/* ---- wide: 16 MBT rows x 16 NBT columns per workgroup of WM x WN waves, two k tiles per stage, a ring of LDS stages filled by LDS-DMA ----
 * A block of R x C reads (R + C) k operands for R C k products, so large blocks are what the L2s can feed; a wave of MW x NW tiles takes (MW + NW) KiB of
 * LDS for MW NW MFMAs.  What is left is latency: all waves of a CU meet at the same barrier, and whatever stands between it and the next MFMA is lost
 * by all of them.  So a k tile's operands are read while the tile before it is multiplied, the requests for a later stage are spread between MFMAs, and
 * the loop over them has no branch.  2047 x 28672 x 4096 (gate | up), launches in a row with weights from memory: 494 us with 128 x 128 blocks read and
 * multiplied in turn, 414 with 256 x 256 ones, 379 (1.27 PF/s; 390 - 412 inside a prompt) with the reads and requests between the MFMAs;
 * 2047 x 4096 x 14336 (down): 239 -> 190 us (1.27 PF/s).  Experts (the grouped form), 2047 rows to 8 of 64, 2048 x 2048: 254 -> 243 us. */
constexpr int wide_stage(int mbt, int nbt) { return (mbt + nbt) * 2048; }
template <typename T, int MBT, int NBT, int WM, int WN, int RING, bool SWIGLU, bool GROUPED>
__global__ __launch_bounds__(64 * WM * WN) void k_gemm_wide(TkImgGemm a, int nblk_n, int nblk_m, int ks) {
    constexpr int NW = NBT / WN, MW = MBT / WM; /* tiles of one wave */
    constexpr int STAGE = wide_stage(MBT, NBT);
    static_assert(!SWIGLU || NW % 2 == 0, "a wave has gate and up tiles in pairs");
    static_assert(MW >= 1 && NW >= 1 && (MBT + NBT) * 2 % (WM * WN) == 0, "every wave has tiles, and as many pieces of a stage as the others");
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    /* workgroups go to the eight XCDs in turn: give each XCD a contiguous range of blocks (row blocks fastest) so that it re-reads the same
     * columns of W from its own L2 */
    int id = blockIdx.x;
    const int total = nblk_n * nblk_m * ks;
    {
        const int per = total / 8, rem = total % 8, x = id % 8, i = id / 8;
        id = x * per + (x < rem ? x : rem) + i;
    }
    const int slab = id / (nblk_n * nblk_m), bn = id / nblk_m % nblk_n, bm = id % nblk_m;
    const int ktiles = a.K / TkImg<T>::KT, s0 = (int)((int64_t)(ktiles / 2) * slab / ks), stages = (int)((int64_t)(ktiles / 2) * (slab + 1) / ks) - s0;
    a.out += slab * a.slab_floats;
    int m0 = bm * MBT, mlive = (a.nrows + 15) / 16 - m0;
    const uint8_t* wbase = (const uint8_t*)a.w;
    if (GROUPED) {
        if (bm >= *a.n_blocks) return;
        const TkImgBlock b = a.blocks[bm];
        m0 = b.tile0; mlive = b.ntiles;
        wbase += (size_t)b.group * a.group_bytes;
    }
    if (mlive > MBT) mlive = MBT;
    const int ntot = a.N / 16, n0 = bn * NBT;
    constexpr int PPW = (MBT + NBT) * 2 / (WM * WN); /* pieces of a stage per wave */
    const uint8_t* src[PPW]; /* the same for all lanes */
#pragma unroll
    for (int i = 0; i < PPW; ++i) { /* piece p: tile p / 2 (M-tiles first, then column tiles), k tile p % 2 of the stage */
        const int p = wave * PPW + i, t = p >> 1, k0 = 2 * s0 + (p & 1);
        if (t < MBT) src[i] = (const uint8_t*)a.a + ((size_t)(m0 + (t < mlive ? t : 0)) * ktiles + k0) * 1024;
        else {
            const int nt = n0 + t - MBT < ntot ? n0 + t - MBT : ntot - 1;
            src[i] = wbase + ((size_t)nt * ktiles + k0) * 1024;
        }
    }
    const int lane16 = lane * 16;
    auto stage = [&](int buf) {
#pragma unroll
        for (int i = 0; i < PPW; ++i) {
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src[i] + lane16),
                                             (__attribute__((address_space(3))) void*)(lds + buf * STAGE + (wave * PPW + i) * 1024), 16, 0, 0);
            src[i] += 2048;
        }
    };
    const int wm = wave % WM * MW, wn = wave / WM * NW;
    tk_v4f acc[NW][MW];
#pragma unroll
    for (int n = 0; n < NW; ++n)
#pragma unroll
        for (int m = 0; m < MW; ++m) acc[n][m] = tk_v4f{0.0f, 0.0f, 0.0f, 0.0f};
    struct Ops { tk_v4u a[MW], w[NW]; } x, y;
    auto read = [&](Ops& o, int buf, int k) {
        const uint8_t* b = lds + buf * STAGE + lane16;
#pragma unroll
        for (int n = 0; n < NW; ++n) o.w[n] = *(const tk_v4u*)(b + ((MBT + wn + n) * 2 + k) * 1024);
#pragma unroll
        for (int m = 0; m < MW; ++m) o.a[m] = *(const tk_v4u*)(b + ((wm + m) * 2 + k) * 1024);
    };
    auto multiply = [&](const Ops& o) {
#pragma unroll
        for (int m = 0; m < MW; ++m)
#pragma unroll
            for (int n = 0; n < NW; ++n) acc[n][m] = TkImg<T>::mma(o.w[n], o.a[m], acc[n][m]);
    };
    /* a k tile's operands are read, and `dma` pieces of a later stage requested, between the MFMAs of the tile before it */
    auto weave = [&](auto dma) {
        constexpr int READS = MW + NW, MFMAS = MW * NW * (sizeof(T) == 4 ? 4 : 1), EACH = MFMAS / READS;
#pragma unroll
        for (int i = 0; i < READS; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x8, EACH, 0);
            if (i < dma.value) __builtin_amdgcn_sched_group_barrier(0x10, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        if (MFMAS % READS) __builtin_amdgcn_sched_group_barrier(0x8, MFMAS % READS, 0);
    };
    /* stages s + 1 .. s + RING - 1 are in flight while stage s is multiplied; a stage's place is free once every wave has its operands in registers */
    for (int s = 0; s < RING && s < stages; ++s) stage(s);
    if (stages >= RING) wait_vm<(RING - 1) * PPW>();
    else wait_vm<0>();
    asm volatile("s_barrier" ::: "memory");
    read(x, 0, 0);
    int cur = 0;
    auto step = [&](auto more) {
        const int next = cur + 1 < RING ? cur + 1 : 0;
        read(y, cur, 1);
        multiply(x);
        weave(std::integral_constant<int, 0>{});
        if (more.value) wait_vm<(RING - 2) * PPW>(); /* the next stage: all but the RING - 2 after it */
        else wait_vm<0>();
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); /* the next stage is there, and this one is in everybody's registers */
        if (more.value) stage(cur);
        read(x, next, 0);
        multiply(y);
        weave(std::integral_constant<int, more.value ? PPW : 0>{});
        cur = next;
    };
    int s = 0;
#pragma unroll 1
    for (; s + RING < stages; ++s) step(std::true_type{});
#pragma unroll 1
    for (; s + 1 < stages; ++s) step(std::false_type{});
    read(y, cur, 1);
    multiply(x);
    weave(std::integral_constant<int, 0>{});
    multiply(y);
#pragma unroll
    for (int m = 0; m < MW; ++m) {
        const int64_t row = (int64_t)(m0 + wm + m) * 16 + (lane & 15);
        if (wm + m >= mlive || (!GROUPED && row >= a.nrows)) continue;
        if (SWIGLU) {
#pragma unroll
            for (int n = 0; n < NW / 2; ++n)
                if (n0 + wn + 2 * n < ntot) store_act<T>(a, m0 + wm + m, (n0 + wn) / 2 + n, lane, acc[2 * n][m], acc[2 * n + 1 < NW ? 2 * n + 1 : 0][m]);
        } else {
#pragma unroll
            for (int n = 0; n < NW; ++n)
                if (n0 + wn + n < ntot) store_f32<T>(a, row, (n0 + wn + n) * 16 + 4 * (lane >> 4), acc[n][m]);
        }
    }
}

template <typename T>
__global__ void k_put_image(const void* src, int src_f32, int64_t N, int64_t K, T* img, int ktiles, int64_t n0, int64_t k0, int interleave) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N * K) return;
    const int64_t n = i / K;
    const int k = (int)(i % K);
    const float v = src_f32 ? ((const float*)src)[i] : tk_bf16_float(((const uint16_t*)src)[i]);
    const int64_t row = interleave < 0 ? n0 + n : (2 * (n / 16) + interleave) * 16 + n % 16;
    tk_img_put(img, row, (int)k0 + k, ktiles, v);
}

/* The forms of the wide kernel and what they cost, fitted to products of 100 .. 2047 rows and k = 256 .. 14336
 * whose weights come from memory.  Large blocks where they fill the chip once or several times, smaller ones where larger would leave CUs idle.
 * bf16 (the choice costs 0.4 % on average over the best one; 171 products): rounds of workgroups x (their start and end + k x time per k).  Of forms that run two to a CU a last round of at most 256 runs one
 * to a CU.
 * f32 (within 11 %): four MFMAs for 16 k where bf16 takes one for 32, so the matrix pipe is all there is, two workgroups of a CU take twice the time, and
 * what counts is the blocks of the fullest CU: the first one's start and end once, + per further one, + k x time per k each. */
struct WideForm {
    int mb, nb, ring; /* tiles, stages */
    int per_cu; float start, k, start2, k2;  /* bf16: us, ns per k of a round with one workgroup per CU, and with two */
    float f32_start, f32_more, f32_k;        /* f32 */
};
constexpr WideForm wide_forms[] = {
    /* bf16 1750 x 28672 x 4096: 372 us (next best 379); f32 2047 x 7552 x 4096: 942 us (947) */
    {16, 16, 2, 1, 22.0f, 17.5f, 0.0f, 0.0f, 16.0f, 15.0f, 221.3f},
    /* bf16 2047 x 4096 x 14336: 182 us (242); f32 256 x 16384 x 2048: as the next two, 0.25 us */
    {16, 8, 3, 1, 8.0f, 12.0f, 0.0f, 0.0f, 12.0f, 6.0f, 115.7f},
    /* bf16 1100 x 28672 x 4096: 248 us (271); f32 1303 x 7552 x 4096: 715 us (256 x 256: 940, which bf16's constants would take) */
    {8, 8, 2, 2, 3.0f, 11.8f, 6.4f, 14.1f, 9.5f, 0.3f, 58.7f},
    /* bf16 1750 x 2048 x 8192: 68 us (93); f32 900 x 4096 x 14336: 846 us (873) */
    {8, 8, 4, 1, 4.6f, 7.3f, 0.0f, 0.0f, 9.5f, 4.0f, 58.6f},
    /* bf16 600 x 2048 x 8192: 50 us (64); f32 2047 x 3072 x 2048: 202 us (128 x 128: 251) */
    {8, 4, 3, 2, 3.4f, 5.3f, 3.8f, 9.8f, 8.5f, 0.5f, 31.2f},
    /* bf16 200 x 4096 x 14336: 61 us (84); f32 1303 x 2048 x 8192: 422 us (128 x 128: 487) */
    {8, 2, 4, 2, 3.2f, 4.0f, 2.8f, 7.4f, 7.5f, 1.0f, 17.1f},
};
float wide_us(const WideForm& w, bool f32, int64_t blocks, float k /* thousands */) {
    if (f32) return w.f32_start + (float)((blocks + 255) / 256 - 1) * w.f32_more + (float)((blocks + 255) / 256) * w.f32_k * k;
    const float one = w.start + w.k * k, two = w.start2 + w.k2 * k;
    if (w.per_cu == 1) return (float)((blocks + 255) / 256) * one;
    return (float)(blocks / 512) * two + (blocks % 512 == 0 ? 0.0f : blocks % 512 <= 256 ? one : two);
}
/* rows and row blocks whose sums a launch makes (TkImgGemm::as_rows) */
int order_rows(const TkImgGemm& g) { return std::max(g.nrows, g.as_rows); }
int order_tiles(const TkImgGemm& g, bool grouped) { return grouped ? g.block_tiles : (order_rows(g) + 15) / 16; }

struct WidePick { int form, ks; };
/* ks: parts of k, 0 for its own choice.  A row's sums depend on the parts alone, not on the blocks */
WidePick pick_wide(const TkImgGemm& g, bool swiglu, bool grouped, int rows, int parts) {
    const int ntiles = g.N / 16, mtiles = (rows + 15) / 16;
    /* k in parts whose sums the consumer adds, at least 16 k tiles each: it reads, and this kernel writes, a slab more per part */
    const int kt = tk_img_kt(g.type), most = parts ? parts : swiglu || grouped || g.max_slabs < 1 ? 1 : g.max_slabs;
    const float slab_us = (float)((double)rows * g.n_valid * 8e-6 / 5.0);
    /* f32: no fewer parts than bring 128 x 128 blocks to two a CU, also where fewer would be a little quicker (0 - 20 us a product): shorter chains of sums,
     * 3 - 4 % less error in the logits of prompts of 150 - 300 rows */
    int fewest = parts ? parts : 1;
    const int64_t full = (int64_t)((mtiles + 7) / 8) * ((ntiles + 7) / 8);
    if (!parts && g.type == TK_IMG_F32 && most > 1 && full < 256) fewest = (int)std::max<int64_t>(1, std::min<int64_t>({512 / full, most, g.K / kt / 16}));
    const int row_blocks = g.live_blocks > 0 && g.live_blocks < g.max_blocks ? g.live_blocks : g.max_blocks;
    WidePick best{2, fewest};
    float least = 1e30f;
    for (int f = 0; f < (int)(sizeof wide_forms / sizeof wide_forms[0]); ++f) {
        const WideForm& w = wide_forms[f];
        if ((grouped && w.mb > 8) || (swiglu && w.nb < 4)) continue;
        for (int ks = fewest; ks <= most && (ks == fewest || g.K / kt / ks >= 16); ++ks) {
            const int64_t blocks = (int64_t)(grouped ? row_blocks : (mtiles + w.mb - 1) / w.mb) * ((ntiles + w.nb - 1) / w.nb) * ks;
            const float us = (float)(ks - 1) * slab_us + wide_us(w, g.type == TK_IMG_F32, blocks, 1e-3f * (float)g.K / (float)ks);
            if (us < least) { least = us; best = WidePick{f, ks}; }
        }
    }
    return best;
}
WidePick pick_wide(const TkImgGemm& g, bool swiglu, bool grouped) {
    const WidePick whole = pick_wide(g, swiglu, grouped, order_rows(g), 0);
    return grouped || order_rows(g) == g.nrows ? whole : pick_wide(g, swiglu, grouped, g.nrows, whole.ks);
}

/* A product of few rows by two workgroups a column tile, in TK_SKINNY_SLABS slabs, where its column tiles leave half of the CUs idle and there is work for every wave:
 * 40 rows x 2048 x 8192 19.7 -> 13.9 us, x 2048 7.2 -> 6.1.  Steps of an eight-layer model 2048 wide with one workgroup / two: 1 row 539 / 529 us, 16 rows 599 / 590, 40 rows
 * 816 / 781, 64 rows 894 / 836; three and four pieces of a wave on their way are no quicker than two.  256 column tiles (4096 wide), one tile a workgroup: 1 row 531 / 546, 40 rows 822 / 838; from 17 rows
 * on in workgroups of two tiles, which read the rows' activations half as often: the products of a step of a four-layer model 4096 wide at 40 and 60 rows 550 / 532 and 606 / 590 us.
 * The slabs add up to the bits of one workgroup, so a row's result does not depend on which it was. */
#define TK_SKINNY_WAVES 8
#define TK_SKINNY_SLABS (1 + TK_SKINNY_WAVES / 2)
int skinny_parts(const TkImgGemm& g, bool swiglu, bool grouped) {
    const int most = order_rows(g) > 16 && g.K / tk_img_kt(g.type) >= 128 ? 256 : 128;
    return !swiglu && !grouped && g.max_slabs >= TK_SKINNY_SLABS && g.N / 16 <= most && g.K / tk_img_kt(g.type) >= 64 ? 2 : 1;
}

template <typename T, bool SWIGLU, bool GROUPED>
const char* launch(const TkImgGemm& g, hipStream_t s, int* slabs) {
    const int ntiles = g.N / 16;
    const int mtiles = order_tiles(g, GROUPED);
    if (mtiles <= 4) {
        /* GROUPED: one block per table entry; the waves of a workgroup, which share k out, by the whole pass's */
        const int blocks = GROUPED ? g.max_blocks : 1, gy = GROUPED ? std::max(g.max_blocks, g.as_blocks) : 1;
        const int parts = skinny_parts(g, SWIGLU, GROUPED);
        if (slabs) *slabs = parts > 1 ? TK_SKINNY_SLABS : 1;
#define TK_SKC(MT, NT, WV, P, C) hipLaunchKernelGGL((k_gemm_skinny<T, MT, NT, WV, P, C, SWIGLU, GROUPED>), dim3((ntiles + NT - 1) / NT, blocks, P), dim3(64 * WV), (size_t)WV * NT * MT * 1024, s, g)
#define TK_SK(MT, NT, WV, P) TK_SKC(MT, NT, WV, P, 1)
#define TK_SKM2(NT, WV, P) do { if (mtiles <= 2) TK_SK(2, NT, WV, P); else if (mtiles <= 3) TK_SK(3, NT, WV, P); else TK_SK(4, NT, WV, P); } while (0)
#define TK_SKM(NT, WV, P) do { if (mtiles <= 1) TK_SK(1, NT, WV, P); else TK_SKM2(NT, WV, P); } while (0)
        /* Column tiles of a workgroup: every workgroup reads its rows' activations again, which from two M-tiles on is more than its weights and comes from the L2s.  So two from 384
         * on: 4096 x 7440 with one / two at 1, 20, 40, 60 rows 16.3 / 14.0, 19.0 / 15.9, 22.1 / 17.2, 25.1 / 19.0 us.  Four where workgroups of two are more than run at once (768
         * of eight waves), at two M-tiles as long as those of four do (512 of four waves): 4096 x 24576, 28672, 32000 with two / four at 20 rows 39.2 / 42.8, 49.0 / 45.2,
         * 50.2 / 47.4, at 60 rows 50.8 / 51.8, 63.8 / 55.6, 67.5 / 59.9; x 40960 59.2 / 61.6, 80.6 / 74.2.  Three M-tiles ask for less at a time and gain less, with two chains a wave and a
         * long k nothing in the end: 4096 x 27648, 30720, 32000 at 40 rows 52.6 / 50.5, 54.5 / 55.2, 55.2 / 57.4, 2048 x 32000 29.4 / 27.4.
         * Below 2048 tiles k is shared out in eight chains, from there on in four, whatever the rows: a row's sums are those of a step of fewer. */
        const bool four = !GROUPED && mtiles >= 2 && ntiles > 1536 && (mtiles == 2 ? ntiles <= 2048 : mtiles > 3 || ntiles >= 2048 || ntiles <= 1792 || g.K <= 2048);
        if (four) {
            if constexpr (!GROUPED) {
                if (ntiles >= 2048) TK_SKM2(4, 4, 1);
                else if (mtiles <= 2) TK_SKC(2, 4, 4, 1, 2);
                else if (mtiles <= 3) TK_SKC(3, 4, 4, 1, 2);
                else TK_SKC(4, 4, 4, 1, 2);
            }
        } else if (!GROUPED && !SWIGLU && ntiles >= 384 && ntiles < 1024) {
            if constexpr (!GROUPED) TK_SKM(2, 8, 1);
        } else if (SWIGLU || ntiles * gy >= 1024) {
            if (ntiles * gy >= 2048) TK_SKM(2, 4, 1); else TK_SKM(2, 8, 1);
        } else if (parts > 1) {
            if constexpr (!SWIGLU && !GROUPED) {
                if (ntiles > 128) TK_SKM2(2, TK_SKINNY_WAVES / 2, 2); else TK_SKM(1, TK_SKINNY_WAVES / 2, 2);
            }
        } else {
            TK_SKM((SWIGLU ? 2 : 1), TK_SKINNY_WAVES, 1);
        }
#undef TK_SKM
#undef TK_SKM2
#undef TK_SK
#undef TK_SKC
        return nullptr;
    }
    const WidePick pick = pick_wide(g, SWIGLU, GROUPED);
    if (slabs) *slabs = pick.ks;
#define TK_WD(MB, NB, WM, WN, RING) do { const int nbn = (ntiles + NB - 1) / NB, nbm = GROUPED ? g.max_blocks : ((g.nrows + 15) / 16 + MB - 1) / MB; \
        hipLaunchKernelGGL((k_gemm_wide<T, MB, NB, WM, WN, RING, SWIGLU, GROUPED>), dim3(nbn * nbm * pick.ks), dim3(64 * WM * WN), (size_t)RING * wide_stage(MB, NB), s, g, nbn, nbm, pick.ks); } while (0)
    switch (pick.form) {
        case 0: if constexpr (!GROUPED) TK_WD(16, 16, 4, 2, 2); break;
        case 1: if constexpr (!GROUPED) TK_WD(16, 8, 4, 2, 3); break;
        case 2: TK_WD(8, 8, 2, 4, 2); break;
        case 3: TK_WD(8, 8, 2, 4, 4); break;
        case 4: TK_WD(8, 4, 4, 2, 3); break;
        default: if constexpr (!SWIGLU) TK_WD(8, 2, 4, 1, 4);
    }
#undef TK_WD
    return nullptr;
}

} // namespace

void tk_gemm_image_form(const TkImgGemm& g, int form[4]) {
    const bool grouped = g.max_blocks > 0;
    form[0] = 64; form[1] = form[2] = 0; form[3] = 1;
    if (order_tiles(g, grouped) <= 4) { form[3] = skinny_parts(g, g.swiglu != 0, grouped); return; }
    const WidePick p = pick_wide(g, g.swiglu != 0, grouped);
    const WideForm& w = wide_forms[p.form];
    form[0] = 16 * w.mb; form[1] = 16 * w.nb; form[2] = w.ring; form[3] = p.ks;
}

const char* tk_launch_gemm_image(const TkImgGemm& g, hipStream_t s, int* slabs) {
    if (slabs) *slabs = 1;
    if (g.type != TK_IMG_BF16 && g.type != TK_IMG_F32) return "gemm_image: unknown element type";
    if (!g.w || !g.a || g.K <= 0 || g.K % (2 * tk_img_kt(g.type))) return "gemm_image: K is not a multiple of two tiles";
    if (g.N <= 0 || g.N % (g.swiglu ? 32 : 16)) return "gemm_image: N is not a multiple of its tile";
    if (g.swiglu ? (!g.act_img || g.act_ktiles * tk_img_kt(g.type) < g.N / 2) : (!g.out || g.n_valid > g.N || g.ldc < g.n_valid)) return "gemm_image: output does not fit";
    if (g.copy_img && g.copy_ktiles * tk_img_kt(g.type) < g.copy1 - g.copy0) return "gemm_image: copied columns do not fit their image";
    if (g.max_slabs > 1 && (!slabs || g.swiglu || g.copy_img || g.slab_floats % 4)) return "gemm_image: this product cannot be split over k";
    if (g.blocks ? (!g.n_blocks || g.max_blocks < 1 || g.block_tiles < 1 || g.block_tiles > 8) : g.nrows < 1) return "gemm_image: no rows";
#define TK_GI(T) (g.swiglu ? (g.blocks ? launch<T, true, true>(g, s, slabs) : launch<T, true, false>(g, s, slabs)) : (g.blocks ? launch<T, false, true>(g, s, slabs) : launch<T, false, false>(g, s, slabs)))
    return g.type == TK_IMG_F32 ? TK_GI(float) : TK_GI(TkBf16);
#undef TK_GI
}

template <typename T>
static hipError_t opt_in_wide() {
    hipError_t e = hipSuccess;
#define TK_OPT(MB, NB, WM, WN, RING, S, G) if (e == hipSuccess) e = hipFuncSetAttribute((const void*)k_gemm_wide<T, MB, NB, WM, WN, RING, S, G>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024)
#define TK_OPT4(MB, NB, WM, WN, RING) TK_OPT(MB, NB, WM, WN, RING, false, false); TK_OPT(MB, NB, WM, WN, RING, false, true); TK_OPT(MB, NB, WM, WN, RING, true, false); TK_OPT(MB, NB, WM, WN, RING, true, true)
    TK_OPT(16, 16, 4, 2, 2, false, false); TK_OPT(16, 16, 4, 2, 2, true, false);
    TK_OPT(16, 8, 4, 2, 3, false, false); TK_OPT(16, 8, 4, 2, 3, true, false);
    TK_OPT4(8, 8, 2, 4, 2);
    TK_OPT4(8, 8, 2, 4, 4);
    TK_OPT4(8, 4, 4, 2, 3);
    TK_OPT(8, 2, 4, 1, 4, false, false); TK_OPT(8, 2, 4, 1, 4, false, true);
#undef TK_OPT4
#undef TK_OPT
    return e;
}

const char* tk_gemm_image_prepare_device() {
    static std::atomic<bool> done[64];
    static std::mutex mu;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return "no current device";
    if (done[dev].load(std::memory_order_acquire)) return nullptr;
    std::lock_guard<std::mutex> lk(mu);
    hipError_t e = opt_in_wide<TkBf16>();
    if (e == hipSuccess) e = opt_in_wide<float>();
    if (e != hipSuccess) return hipGetErrorString(e);
    done[dev].store(true, std::memory_order_release);
    return nullptr;
}

void tk_launch_put_image(int type, const void* src, int src_f32, int64_t N, int64_t K, void* img, int ktiles, int64_t n0, int64_t k0, int interleave, hipStream_t s) {
    const unsigned blocks = (unsigned)((N * K + 255) / 256);
    if (type == TK_IMG_F32) hipLaunchKernelGGL((k_put_image<float>), dim3(blocks), dim3(256), 0, s, src, src_f32, N, K, (float*)img, ktiles, n0, k0, interleave);
    else hipLaunchKernelGGL((k_put_image<TkBf16>), dim3(blocks), dim3(256), 0, s, src, src_f32, N, K, (TkBf16*)img, ktiles, n0, k0, interleave);
}
