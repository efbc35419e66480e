/* tk_gemm_tiled.hip — see tk_gemm_tiled.h */
#include "tk_gemm_tiled.h"

#include <math.h>

#include <atomic>
#include <mutex>
#include <type_traits>

#include "../common/tk_exact_math.h"
#include "tk_image_device.h"

typedef _Float16 tw_v8h __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));

#define TK_TW_SLOT_BYTES 65536

__device__ __forceinline__ uint4 tw_ldg_nt(const uint8_t* p) {
    const v4u v = __builtin_nontemporal_load((const v4u*)p);
    return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ float tw_f16(uint32_t h) { return (float)__builtin_bit_cast(_Float16, (uint16_t)h); }

/* s_waitcnt vmcnt(n) alone: until all but this wave's n youngest vector-memory operations are done (LDS-DMA pieces and weight requests
 * count together, in issue order) */
__device__ __forceinline__ void tw_wait_vmcnt(int n) {
#define TK_VMW(k) case k: __builtin_amdgcn_s_waitcnt(0x0F70 | ((k) & 15) | (((k) >> 4) << 14)); break;
    switch (n) {
        TK_VMW(0) TK_VMW(1) TK_VMW(2) TK_VMW(3) TK_VMW(4) TK_VMW(5) TK_VMW(6) TK_VMW(7) TK_VMW(8) TK_VMW(16)
        default: __builtin_amdgcn_s_waitcnt(0x0F70); break;
    }
#undef TK_VMW
}

__device__ __forceinline__ float tw_act(float v, int act) {
    switch (act) {
        case TK_ACT_SILU: return tk_siluf(v);
        case TK_ACT_GELU: return tk_geluf(v);
        case TK_ACT_SIGMOID: return tk_sigmoidf(v);
        default: return v;
    }
}

template <int N> __device__ __forceinline__ void tw_act_all(float* v, int act) {
    if (act == TK_ACT_SILU) {
        tk_silu_all<N>(v);
    } else if (act == TK_ACT_GELU) {
#pragma unroll
        for (int i = 0; i < N; ++i) v[i] = tk_geluf(v[i]);
    } else if (act == TK_ACT_SIGMOID) {
#pragma unroll
        for (int i = 0; i < N; ++i) v[i] = tk_sigmoidf(v[i]);
    }
}

/* WB = bytes per weight value (2: f16, 4: f32); MT = M-tiles per workgroup.
 * What bounds few rows: the chain, 8 cycles a k and M-tile, as long as weights and operands are there in time.  One LDS read takes a wave about 130
 * cycles, so operands are read one pair of tiles ahead, also across the chunks of 32 k.  With a ring the compiler cannot count what is in flight
 * behind the staging and lets the first weights of every PF chunks wait for all requests; where the activations of the whole K range fit the LDS
 * (ONE: multiples of 128 k, up to 2048 at one M-tile, 1024 at two) there is no staging in the loop, and four pieces of weights stay in flight, eight
 * where k is a multiple of 256 from 512 on.
 * REG (the launcher's rules say when): a wave shares no activations, it fetches its operands as it does its weights, straight into registers, by scalar offsets, and its
 * chain starts with the first of both instead of behind a whole image in LDS and a barrier; nothing waits for another wave, and no LDS read takes a turn from the MFMAs.
 * f16: conversions in front of a piece's products, not between them, and the next operands' requests behind them (scattered, 8192 columns of 4096 k at 24 rows take 39.6 us,
 * in order 35.7).  4096 x 28672 at 1, 24, 48 rows, ring -> here: 61 -> 42, 83 -> 68, 142 -> 97 us (floor of the weights 45, of the fp32 MFMAs on two tiles a SIMD 55 and 82).
 * In LDS, cold weights, N x K at 1 row: 384 x 384 5.4 -> 4.5 us and 51872 x 384 24.0 -> 22.0 with four, 384 x 1536 13.9 -> 10.2 with eight; at 32 rows
 * 8.6 -> 7.9, 30.0 -> 27.0 with four, 20.8 -> 18.9 (ring).  Twelve pieces: 384 x 384 at 1 row 5.6 (a wave's requests queue in front of the activations
 * of the others). */
/*
 * Layer norm of the workgroup's rows into the one slot of activations (TkTiledGemm::ln_x): a wave a row, k_layernorm's arithmetic in its order — 256 partial sums over
 * columns p, p + 256, ..., folded within groups of 64 by halves, the four groups left to right — with the four groups side by side in a wave's lanes.  A decoder step of
 * one sequence has 13 norms; as launches of their own they took 2.9 us each, and the 12 products behind them waited for a trip to memory more.  Registers and requests for
 * no more columns than the form is for: 384 columns in the form for 1024 6.4 us a product of a step and 21.9 one of 51 864 columns, in that for 512 6.1 and 19.5.
 */
template <int NV /* times 256 columns, at most */>
__device__ __forceinline__ void tw_layernorm(const TkTiledGemm& a, int row0, int rows, float* image, int wave, int nw, int lane) {
    const int D = a.K;
    auto fold = [&](float (&s)[4]) {
#pragma unroll
        for (int w = 0; w < 4; ++w) s[w] = tk_wave_butterfly_sum(s[w]);
        return ((s[0] + s[1]) + s[2]) + s[3];
    };
    for (int r = wave; r < rows; r += nw) {
        const float* xr = a.ln_x + (size_t)(row0 + r) * D;
        float v[NV][4], wv[NV][4], bv[NV][4];
#pragma unroll
        for (int u = 0; u < NV; ++u)
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                int i = 256 * u + 64 * w + lane;
                i = i < D ? i : D - 1;
                v[u][w] = xr[i]; wv[u][w] = a.ln_w[i]; bv[u][w] = a.ln_b[i];
            }
        float s[4];
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            s[w] = 0.0f;
#pragma unroll
            for (int u = 0; u < NV; ++u)
                if (256 * u + 64 * w + lane < D) s[w] = s[w] + v[u][w];
        }
        const float mean = tk_divf(fold(s), (float)D);
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            s[w] = 0.0f;
#pragma unroll
            for (int u = 0; u < NV; ++u)
                if (256 * u + 64 * w + lane < D) { const float d = v[u][w] - mean; s[w] = tk_fmaf(d, d, s[w]); }
        }
        const float var = tk_divf(fold(s), (float)D);
        const float rstd = tk_divf(1.0f, tk_sqrtf(var + a.ln_eps));
#pragma unroll
        for (int u = 0; u < NV; ++u)
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const int i = 256 * u + 64 * w + lane;
                if (i < D) image[(i >> 4) * 256 + (i & 3) * 64 + r * 4 + ((i & 15) >> 2)] = ((v[u][w] - mean) * rstd) * wv[u][w] + bv[u][w];
            }
    }
}

template <int MT, int WB, bool ONE /* the whole K range in one slot */, int PF /* weight pieces in flight per wave; a ring slot holds a multiple of PF chunks (the launcher's rk), so piece c sits in register set c % PF */,
          int LN = 0 /* the activations are made here, norms of up to LN times 256 columns (MT = 1, ONE) */, bool REG = false /* and each wave fetches its own into registers, like its weights (ONE; f16: up to four M-tiles) */>
__global__ __launch_bounds__(512) void k_gemm_tiled(TkTiledGemm a, int groups, int total_row_tiles, int rk /* k per ring slot */, int slot_bytes /* ring slot pitch */) {
    constexpr int LPC = WB == 4 ? 2 : 1; /* 16-byte requests per piece and lane */
    constexpr int PIECE = 512 * WB;      /* bytes of one (row tile, 32 k) piece */
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nw = blockDim.x >> 6;
    const int Kr = a.K / a.ks;
    /* REG: the row blocks of a unit one behind the other on one XCD, which then has their weights */
    const int unit = REG ? (int)(blockIdx.y * 8 + (blockIdx.x & 7)) : (int)blockIdx.x, block = REG ? (int)(blockIdx.x >> 3) : (int)blockIdx.y;
    const int ksi = unit % a.ks;
    const int k0 = ksi * Kr;
    const int nslots = Kr / rk, cps = rk / 32, gps = rk / 16;
    /* grid y: the block of MT M-tiles this workgroup covers */
    const int row0 = block * MT * TK_TW_ROWS_PER_TILE;
    const float* a_img = a.a_img + (size_t)block * MT * a.a_ts;
    const int rows_here = a.nrows - row0 < MT * TK_TW_ROWS_PER_TILE ? a.nrows - row0 : MT * TK_TW_ROWS_PER_TILE;

    int rt = unit / a.ks + wave * groups;
    const bool active = (!REG || unit < groups * a.ks) && rt < total_row_tiles;
    if (!active) rt = 0;
    /* The segment by comparisons and selects, without an index into the arguments, and all that the end takes from them here: an argument is asked for
     * where it is used else, and each new line of them is a trip to memory of a chain of its own, in front of the weights and behind the sums (with bias and
     * residual early: 17 decoder steps of one clip 45 us less of 4.85 ms, of 32 clips 340 us of 6.9 ms) */
    int seg = 0, col_base = 0;
    const int rt0 = a.row_tiles[0], rt1 = a.row_tiles[1];
    if (a.nseg > 1 && rt >= rt0) { rt -= rt0; col_base = rt0 * TK_TW_ROWS_PER_TILE; seg = 1; }
    if (a.nseg > 2 && seg == 1 && rt >= rt1) { rt -= rt1; col_base += rt1 * TK_TW_ROWS_PER_TILE; seg = 2; }
    auto of = [&](const auto& three) { return seg == 0 ? three[0] : seg == 1 ? three[1] : three[2]; };
    const int nchunk_total = a.K / 32, nchunk = Kr / 32;
    const uint8_t* wbase = of(a.tiles) + ((size_t)rt * nchunk_total + k0 / 32) * PIECE + lane * (8 * WB);
    const bool split = a.ks > 1, per_seg = !split && a.per_seg;
    const int end_n = (per_seg ? 0 : col_base) + rt * TK_TW_ROWS_PER_TILE + (lane & 15), end_cols = per_seg ? of(a.seg_n) : a.n_valid;
    float* const end_out = per_seg ? of(a.seg_out) : a.out;
    const int end_ldc = per_seg ? of(a.seg_ldc) : a.ldc, act = a.act;
    const float* const end_bias = split ? nullptr : per_seg ? of(a.seg_bias) : a.bias;
    const float* const end_res = split || per_seg ? nullptr : a.residual;
    const bool end_img = WB == 4 && per_seg && of(a.seg_img), add_bias = end_bias || a.add_zero_bias;
    float* const c_img = split || per_seg ? nullptr : a.c_img;

    const int ppslot = gps * MT;
    const uint32_t voff = lane * 16;
    auto stage = [&](int s, int slot) { /* slot s of the range: [16-k group j][M-tile m] pieces of 1 KiB, piece p = j * MT + m dealt to wave p % nw */
        for (int p = wave; p < ppslot; p += nw) {
            const int j = p / MT, m = p % MT;
            const uint8_t* src = (const uint8_t*)(a_img + (size_t)m * a.a_ts + ((size_t)(k0 + s * rk) / 16 + j) * 256);
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src + voff),
                                             (__attribute__((address_space(3))) void*)(lds + (size_t)slot * slot_bytes + (size_t)p * 1024), 16, 0, 0);
        }
    };

    float acc[MT][4];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[m][r] = 0.0f;

    /* bias and residual are on their way while the products run: one trip to memory less behind them (few rows: registers for all of it) */
    constexpr bool EARLY = MT <= 2;
    float bias = 0.0f, res[EARLY ? MT : 1][4] = {};
    auto load_end = [&]() {
        const int n = end_n < end_cols ? end_n : end_cols - 1;
        if (end_bias) bias = end_bias[n];
        if (EARLY && end_res) {
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int row = m * TK_TW_ROWS_PER_TILE + 4 * (lane >> 4) + r;
                    res[m][r] = end_res[(size_t)(row0 + (row < rows_here ? row : rows_here - 1)) * a.ldr + n];
                }
        }
    };
    /* REG: operands of chunk c, two 16-k groups of each M-tile; rows that are not there: the last one again.  Scalar offsets walk k: no vector instruction beside the products. */
    v4f aq[REG ? PF : 1][REG ? MT : 1][2];
    const int tiles_here = (rows_here + TK_TW_ROWS_PER_TILE - 1) / TK_TW_ROWS_PER_TILE;
    const __amdgpu_buffer_rsrc_t ar = __builtin_amdgcn_make_buffer_rsrc((void*)(a_img + (size_t)k0 * 16), 0, ((unsigned)(tiles_here - 1) * (unsigned)a.a_ts + (unsigned)Kr * 16u) * 4u, 0x00020000);
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc((void*)(of(a.tiles) + ((size_t)rt * nchunk_total + k0 / 32) * PIECE), 0, (unsigned)nchunk * PIECE, 0x00020000);
    unsigned a_at[REG ? MT : 1];
#pragma unroll
    for (int m = 0; m < (REG ? MT : 0); ++m) {
        const int t = m < tiles_here ? m : tiles_here - 1, rows = rows_here - t * TK_TW_ROWS_PER_TILE, last = rows < TK_TW_ROWS_PER_TILE ? rows - 1 : TK_TW_ROWS_PER_TILE - 1;
        a_at[m] = (unsigned)t * (unsigned)a.a_ts * 4u + (unsigned)((lane & 48) + ((lane & 15) < last ? lane & 15 : last)) * 16u;
    }
    /* a request past the range re-reads the last piece: no branch around a load, static wait counts */
    uint4 wq[PF][LPC];
    auto wload = [&](int c, uint4* dst) {
        if (REG) {
#pragma unroll
            for (int i = 0; i < LPC; ++i) dst[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(wr, lane * (8 * WB) + 16 * i, (unsigned)(c < nchunk ? c : nchunk - 1) * PIECE, 2));
            return;
        }
        const uint8_t* p = wbase + (size_t)(c < nchunk ? c : nchunk - 1) * PIECE;
        dst[0] = tw_ldg_nt(p);
        if (LPC == 2) dst[LPC - 1] = tw_ldg_nt(p + 16);
    };
    auto aload = [&](int c, v4f (*dst)[2]) {
        const unsigned at = (unsigned)(c < nchunk ? c : nchunk - 1) * 2048u;
#pragma unroll
        for (int m = 0; m < (REG ? MT : 0); ++m)
#pragma unroll
            for (int h = 0; h < 2; ++h) dst[m][h] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(ar, a_at[m] + h * 1024, at, 0));
    };
    if (REG) {
        if (!active) return;
#pragma unroll
        for (int i = 0; i < PF; ++i) { aload(i, aq[REG ? i : 0]); wload(i, wq[i]); }
        load_end();
    } else if (LN) {
        if (active) {
#pragma unroll
            for (int i = 0; i < PF; ++i) wload(i, wq[i]);
            load_end();
        }
        tw_layernorm<LN ? LN : 1>(a, row0, rows_here, (float*)lds, wave, nw, lane);
        __syncthreads();
        if (!active) return;
    } else {
        stage(0, 0);
    }
    if (!LN && !REG && !active) { /* no tile of its own: its share of the staging */
        for (int s = 0; s < nslots; ++s) {
            tw_wait_vmcnt(0);
            __syncthreads();
            if (s + 1 < nslots) stage(s + 1, (s + 1) & 1);
        }
        return;
    }
    if (!LN && !REG) {
        load_end();
#pragma unroll
        for (int i = 0; i < PF; ++i) wload(i, wq[i]);
    }

#pragma unroll 1
    for (int s = 0; s < (ONE ? 1 : nslots); ++s) {
        /* slot s has landed once all but the PF * LPC youngest requests are done: those are weight requests issued after its DMA
         * (cps >= PF chunks follow every slot's DMA, the PF initial ones the first) */
        if (!LN && !REG) {
            tw_wait_vmcnt(PF * LPC);
            __syncthreads();
        }
        if (!ONE && s + 1 < nslots) stage(s + 1, (s + 1) & 1);
        const uint8_t* slot = lds + (size_t)(ONE ? 0 : s & 1) * slot_bytes + lane * 16;
        /* operands of M-tiles m, m + 1 (m alone of MT = 1) and chunk cc of the slot; [k half][tile] */
        constexpr int PAIR = MT == 1 ? 1 : REG ? MT : 2, PAIRS = MT / PAIR;
        struct Ops { v4f a[2][PAIR]; } ops[2];
        auto read = [&](Ops& o, int cc, int m) {
            const uint8_t* ap = slot + (size_t)(2 * (cc < cps ? cc : cps - 1)) * MT * 1024 + m * 1024;
#pragma unroll
            for (int i = 0; i < PAIR; ++i)
#pragma unroll
                for (int h = 0; h < 2; ++h) o.a[h][i] = *(const v4f*)(ap + (h * MT + i) * 1024);
        };
        if (!REG) read(ops[0], 0, 0);
#pragma unroll 1
        for (int cc = 0; cc < cps; cc += PF) {
#pragma unroll
            for (int u = 0; u < PF; ++u) {
                const int c = s * cps + cc + u;
                float wf[8];
                if (WB == 2) {
                    const uint4 w = wq[u][0];
                    wf[0] = tw_f16(w.x & 0xffffu); wf[1] = tw_f16(w.x >> 16); wf[2] = tw_f16(w.y & 0xffffu); wf[3] = tw_f16(w.y >> 16);
                    wf[4] = tw_f16(w.z & 0xffffu); wf[5] = tw_f16(w.z >> 16); wf[6] = tw_f16(w.w & 0xffffu); wf[7] = tw_f16(w.w >> 16);
                } else {
                    const uint4 w0 = wq[u][0], w1 = wq[u][LPC - 1];
                    wf[0] = __uint_as_float(w0.x); wf[1] = __uint_as_float(w0.y); wf[2] = __uint_as_float(w0.z); wf[3] = __uint_as_float(w0.w);
                    wf[4] = __uint_as_float(w1.x); wf[5] = __uint_as_float(w1.y); wf[6] = __uint_as_float(w1.z); wf[7] = __uint_as_float(w1.w);
                }
                if (WB == 2 || !ONE) wload(c + PF, wq[u]);
                if (REG && WB == 2) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int p = 0; p < PAIRS; ++p) {
                    /* the next pair's operand reads, the next chunk's behind the last pair, are issued before this pair's MFMAs; of two tiles the
                     * chains alternate (a chain step's 40-cycle dependent latency hides behind the other chain's MFMA) */
                    const int step = u * PAIRS + p, m = p * PAIR;
                    Ops& o = ops[step & 1];
                    if (REG) {
#pragma unroll
                        for (int i = 0; i < PAIR; ++i)
#pragma unroll
                            for (int h = 0; h < 2; ++h) o.a[h][i] = aq[REG ? u : 0][REG ? m + i : 0][h];
                    } else if (p + 1 < PAIRS) {
                        read(ops[(step + 1) & 1], cc + u, m + PAIR);
                    } else {
                        read(ops[(step + 1) & 1], cc + u + 1, 0);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    {
                        v4f d[PAIR];
#pragma unroll
                        for (int i = 0; i < PAIR; ++i) d[i] = v4f{acc[m + i][0], acc[m + i][1], acc[m + i][2], acc[m + i][3]};
#pragma unroll
                        for (int t = 0; t < 8; ++t)
#pragma unroll
                            for (int i = 0; i < PAIR; ++i) d[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.a[t >> 2][i][t & 3], wf[t], d[i], 0, 0, 0);
#pragma unroll
                        for (int i = 0; i < PAIR; ++i)
#pragma unroll
                            for (int r = 0; r < 4; ++r) acc[m + i][r] = d[i][r];
                    }
                }
                if (WB == 4 && ONE) wload(c + PF, wq[u]);
                if (REG) aload(c + PF, aq[REG ? u : 0]);
                if (REG && WB == 2) __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    const int g = lane >> 4, n = end_n;
    if (n >= end_cols) return;
    /* operand-image position of column n as k of the next layer: k = 16 j + 4 t + g2 -> [M-tile][j][g2][row][t] (tk_gemm_tiled.h) */
    const size_t img_col = (size_t)(n >> 4) * 256 + (size_t)(n & 3) * 64 + ((n & 15) >> 2);
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = m * TK_TW_ROWS_PER_TILE + 4 * g + r;
            if (row >= rows_here) continue;
            float v = acc[m][r];
            if (split) {
                __builtin_nontemporal_store(v, &end_out[((size_t)ksi * a.slab_rows + row0 + row) * end_ldc + n]);
                continue;
            }
            if (add_bias) v = v + bias;
            v = tw_act(v, act);
            const size_t at = (size_t)(row0 + row), tile = (at >> 4) * 16 * end_cols + img_col + (at & 15) * 4;
            if (end_img) { /* per segment: a layer of its own, whose output is an operand image */
                end_out[tile] = v;
                continue;
            }
            if (end_res) v = v + (EARLY ? res[EARLY ? m : 0][r] : end_res[at * a.ldr + n]);
            if (WB == 2 || end_out) end_out[at * end_ldc + n] = v;
            if (c_img) c_img[tile] = v;
        }
}

/*
 * Many rows: a wave makes 32 MI x 32 of the output alone, on v_mfma_f32_32x32x2_f32 (the same chain, two k an instruction), both operands from the caches straight
 * into registers, PF stages of KS k in flight: no LDS, no barrier, nothing that waves wait for each other with.  Step s of a 16-k group takes k = 2 s, 2 s + 1: lane half
 * h = l / 32 holds groups g = h and 2 + h of the image and of the weight tiles, a float4 each.  An operand float4 feeds 4 or 4 MI MFMAs of 64 cycles, where the ring
 * kernel above reads LDS once for 4 of 32: fp32 MFMAs and LDS reads take turns on a SIMD.
 * Images are made with the operands exchanged: a lane then holds one row, and lanes l, l + 32 swap halves so that each stores the 16 bytes of a group.
 * f16 weights (K-split parts side by side, the rows of a tile column in one workgroup) are converted in front of each product, on its pipe: 256 rows x 4096 x 28672 533 ->
 * 491 us (393), 136 rows of a 4096-wide layer 1.20 -> 0.77 ms.
 * Form <1, 1> has the smaller tiles, and so more of them; form <2, 1> reads a third less, which counts for matrices that the L2 does not hold (tk_gemm_tiled_plan).
 * 48 000 rows, ring -> here, us (the fp32 MFMAs alone): 384 x 384 183 -> 139 (93), 1152 x 384 475 -> 346 (278), 1536 x 384 with GELU 610 -> 469 (370), 384 x 1536 560 -> 513
 * (370); 1500 rows: 23.2 -> 17.6, 31.6 -> 25.2 and 38.2 -> 30.4 of the last three.  What is left is the last round of tiles and the first requests of each.
 */
template <int WB, int MI, int KS, int PF>
__global__ __launch_bounds__(256, MI == 2 || PF > 2 ? 4 : 5) void k_gemm_wide(TkTiledGemm a, int ncol /* tiles of 32 columns */, int nrow /* tiles of 32 MI rows */, int total /* waves' tiles */,
                                                                                  int per_xcd) {
    constexpr int V = KS / 8;               /* float4 per 32 rows and stage */
    constexpr int WV = WB == 4 ? V : V / 2; /* 16-byte pieces of weights per 32 columns and stage */
    /* consecutive workgroups go to different XCDs: each takes a run of them, whose rows stay in its L2 */
    const int wg = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    const int lane = threadIdx.x & 63, id = wg * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (id >= total) return;
    const int h = lane >> 5, l32 = lane & 31, l16 = lane & 15, up = (lane >> 4) & 1;
    /* f32: the columns of a tile row by row (the weights are small and stay); f16: the rows of a tile column side by side, so that a workgroup's waves share their
     * weights, then the columns, then the parts of k */
    const int blk = WB == 4 ? id / ncol : id % nrow, row0 = blk * 32 * MI;
    const int colk = id / nrow, ksi = WB == 4 ? 0 : colk / ncol;
    int rt = (WB == 4 ? id - blk * ncol : colk - ksi * ncol) * 2, seg = 0, col_base = 0;
    while (seg < a.nseg - 1 && rt >= a.row_tiles[seg]) { rt -= a.row_tiles[seg]; col_base += a.row_tiles[seg] * TK_TW_ROWS_PER_TILE; ++seg; }
    const unsigned a_pitch = (unsigned)a.a_ts * 4u, w_pitch = (unsigned)a.K * 16u * WB; /* bytes of 16 rows */
    const int tiles_here = (a.nrows - row0 + 15) / 16;
    const __amdgpu_buffer_rsrc_t ar = __builtin_amdgcn_make_buffer_rsrc((void*)(a.a_img + (size_t)(row0 / 16) * a.a_ts), 0, (unsigned)(tiles_here < 2 * MI ? tiles_here : 2 * MI) * a_pitch, 0x00020000);
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc((void*)(a.tiles[seg] + (size_t)rt * w_pitch), 0, 2u * w_pitch, 0x00020000);
    unsigned a_at[MI];
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        const int tile = 2 * i + up;
        a_at[i] = (unsigned)(tile < tiles_here ? tile : tiles_here - 1) * a_pitch + (unsigned)(h * 256 + l16 * 16);
    }
    const unsigned w_at = (unsigned)up * w_pitch + (unsigned)((h * 16 + l16) * 8 * WB);

    v4f aq[PF][MI][V], wq[PF][WV];
    const int ns = (WB == 4 ? a.K : a.K / a.ks) / KS, s0 = ksi * ns;
    auto load = [&](int s, v4f (*av)[V], v4f* wv) {
        s = s0 + (s < ns ? s : ns - 1);
#pragma unroll
        for (int v = 0; v < V; ++v) { /* 16-k group v / 2 of the stage, half v % 2 of its groups */
            const unsigned j = (unsigned)(s * (KS / 16) + v / 2);
#pragma unroll
            for (int i = 0; i < MI; ++i) av[i][v] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(ar, a_at[i] + (v & 1) * 512, j * 1024, 0));
            if (WB == 4) wv[v] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(wr, w_at + (v & 1) * 1024, (j >> 1) * 2048 + (j & 1) * 16, 0));
            else if (v % 4 < 2) wv[v / 4 * 2 + v % 2] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(wr, w_at + (v & 1) * 512, (j >> 1) * 1024, 0));
        }
    };
    v16f acc[MI];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][r] = 0.0f;
    const bool image = a.c_img != nullptr || (a.per_seg && a.seg_img[seg]);
    auto products = [&](auto swapped) {
#pragma unroll
        for (int s = 0; s < PF - 1; ++s) load(s, aq[s], wq[s]);
#pragma unroll 1
        for (int s = 0; s < ns; s += PF) {
#pragma unroll
            for (int u = 0; u < PF; ++u) {
                load(s + u + PF - 1, aq[(u + PF - 1) % PF], wq[(u + PF - 1) % PF]);
#pragma unroll
                for (int v = 0; v < V; v += 2)
#pragma unroll
                    for (int t = 0; t < 4; ++t)
#pragma unroll
                        for (int b = 0; b < 2; ++b)
#pragma unroll
                            for (int i = 0; i < MI; ++i) {
                                const float x = aq[u][i][v + b][t];
                                float w;
                                if (WB == 4) w = wq[u][WB == 4 ? v + b : 0][t];
                                else w = (float)__builtin_bit_cast(tw_v8h, wq[u][v / 4 * 2 + b])[4 * (v / 2 % 2) + t]; /* a piece: t of both 16-k groups */
                                acc[i] = swapped.value ? __builtin_amdgcn_mfma_f32_32x32x2f32(w, x, acc[i], 0, 0, 0) : __builtin_amdgcn_mfma_f32_32x32x2f32(x, w, acc[i], 0, 0, 0);
                            }
                /* the requests spread over the products: in front of them they hold these up, behind them (where the compiler puts them) they come late */
#pragma unroll
                for (int i = 0; i < MI * V + WV; ++i) {
                    __builtin_amdgcn_sched_group_barrier(0x008, MI * V * 4 / (MI * V + WV), 0);
                    __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    const int col0 = rt * TK_TW_ROWS_PER_TILE; /* in the segment */
    const float* bias = a.per_seg ? a.seg_bias[seg] : a.bias;
    if (bias && !a.per_seg) bias += col_base;
    const bool add_bias = bias || a.add_zero_bias;
    if (WB == 4 && image) {
        products(std::true_type{});
        float* img = a.per_seg ? a.seg_out[seg] : a.c_img;
        const int cols = a.per_seg ? a.seg_n[seg] : a.n_valid, c0 = a.per_seg ? col0 : col_base + col0;
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            const int row = row0 + 32 * i + l32;
            float v[16];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                v4f b = {0.0f, 0.0f, 0.0f, 0.0f};
                if (bias) b = *(const v4f*)(bias + col0 + 8 * q + 4 * h);
#pragma unroll
                for (int r = 0; r < 4; ++r) v[4 * q + r] = add_bias ? acc[i][4 * q + r] + b[r] : acc[i][4 * q + r];
            }
            tw_act_all<16>(v, a.act);
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int g = 0; g < 4; g += 2) {
                    v4f o;
#pragma unroll
                    for (int b = 0; b < 2; ++b) { /* t = 2 b + h of groups g, g + 1: the lower lanes take g, the upper g + 1 */
                        const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[8 * q + 4 * b + g]), __float_as_uint(v[8 * q + 4 * b + g + 1]), false, false);
                        o[2 * b] = __uint_as_float(x[0]);
                        o[2 * b + 1] = __uint_as_float(x[1]);
                    }
                    if (row < a.nrows) *(v4f*)(img + (size_t)(row >> 4) * 16 * cols + (size_t)(((c0 >> 4) + q) * 256 + (g + h) * 64 + (row & 15) * 4)) = o;
                }
        }
        return;
    }
    products(std::false_type{});
    float* out = a.per_seg ? a.seg_out[seg] + col0 : a.out + (WB == 2 ? (size_t)ksi * a.slab_rows * a.ldc : 0) + col_base + col0;
    const int ldc = a.per_seg ? a.seg_ldc[seg] : a.ldc;
    const float* res = a.residual ? a.residual + col_base + col0 : nullptr;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        const float b = bias ? bias[col0 + l32] : 0.0f;
        float v[16], rs[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int row = row0 + 32 * i + 8 * (r >> 2) + 4 * h + (r & 3);
            if (res) rs[r] = row < a.nrows ? res[(size_t)row * a.ldr + l32] : 0.0f;
            v[r] = add_bias ? acc[i][r] + b : acc[i][r];
        }
        tw_act_all<16>(v, a.act);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int row = row0 + 32 * i + 8 * (r >> 2) + 4 * h + (r & 3);
            if (res) v[r] = v[r] + rs[r];
            if (row < a.nrows) out[(size_t)row * ldc + l32] = v[r];
        }
    }
}

/* ---- operand preparation ---- */

template <typename T>
__global__ void k_tile_weights(const T* src, int64_t N, int64_t K, T* tiles) {
    const int lane = threadIdx.x, n = lane & 15, g = lane >> 4;
    const int64_t chunk = blockIdx.x, rt = blockIdx.y;
    const int64_t row = rt * 16 + n;
    T* dst = tiles + ((rt * (K / 32) + chunk) * 64 + lane) * 8;
#pragma unroll
    for (int t = 0; t < 8; ++t) dst[t] = row < N ? src[row * K + chunk * 32 + 4 * t + g] : (T)0;
}

size_t tk_tiled_weight_bytes(int64_t N, int64_t K, int wbytes) { return (size_t)((N + 15) / 16 * 16) * (size_t)K * (size_t)wbytes; }

void tk_launch_tile_weights(const void* src, int wbytes, int64_t N, int64_t K, uint8_t* tiles, hipStream_t s) {
    const dim3 grid((unsigned)(K / 32), (unsigned)((N + 15) / 16));
    if (wbytes == 2) hipLaunchKernelGGL((k_tile_weights<uint16_t>), grid, dim3(64), 0, s, (const uint16_t*)src, N, K, (uint16_t*)tiles);
    else hipLaunchKernelGGL((k_tile_weights<uint32_t>), grid, dim3(64), 0, s, (const uint32_t*)src, N, K, (uint32_t*)tiles);
}

/* one thread per image element (coalesced 16-byte stores); rows beyond `rows` read as zero */
__global__ void k_pack_a(const float* A, int64_t rows, int K, int lda, int round_f16, float* img) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; /* index of a float4 of the image */
    const int64_t mtiles = (rows + 15) / 16, per_tile = (int64_t)K * 4; /* float4 per M-tile = 16 K / 4 */
    if (i >= mtiles * per_tile) return;
    const int64_t mt = i / per_tile, q = i % per_tile;
    const int64_t j = q / 64;             /* 16-k group */
    const int g = (int)((q % 64) / 16), r = (int)(q % 16);
    const int64_t row = mt * 16 + r;
    v4f v = {0.0f, 0.0f, 0.0f, 0.0f};
    if (row < rows) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const float x = A[row * lda + 16 * j + 4 * t + g];
            v[t] = round_f16 ? tk_f16_to_f32(tk_f32_to_f16(x)) : x;
        }
    }
    *(v4f*)(img + i * 4) = v;
}

size_t tk_a_image_floats(int64_t rows, int64_t K) { return (size_t)((rows + 15) / 16 * 16) * (size_t)K; }

void tk_launch_pack_a(const float* A, int64_t rows, int K, int lda, int round_f16, float* img, hipStream_t s) {
    const int64_t n4 = (rows + 15) / 16 * (int64_t)K * 4;
    hipLaunchKernelGGL(k_pack_a, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, s, A, rows, K, lda, round_f16, img);
}

/* ---- launch ---- */

/* compute units of the calling thread's current device, cached PER DEVICE (the ABI takes a device ordinal per handle; launchers run with
 * the handle's device current and from several host threads) */
static int tk_tiled_num_cu() {
    static std::atomic<int> n[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    int v = n[dev].load(std::memory_order_relaxed);
    if (v > 0) return v;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v < 1) v = 256;
    n[dev].store(v, std::memory_order_relaxed);
    return v;
}

template <typename F>
static hipError_t tw_opt_in(F* fn) { return hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, 2 * TK_TW_SLOT_BYTES); }

static std::atomic<bool> g_tw_opted[64];
static std::mutex g_tw_mu;
bool tk_gemm_tiled_prepare_device() {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return false;
    if (g_tw_opted[dev].load(std::memory_order_acquire)) return true;
    std::lock_guard<std::mutex> lk(g_tw_mu);
    hipError_t e = hipSuccess;
#define TK_TW_OPT(MTV, ONEV, PFV) do { if (e == hipSuccess) e = tw_opt_in(k_gemm_tiled<MTV, 2, ONEV, PFV>); if (e == hipSuccess) e = tw_opt_in(k_gemm_tiled<MTV, 4, ONEV, PFV>); } while (0)
    TK_TW_OPT(1, true, 4); TK_TW_OPT(1, true, 8); TK_TW_OPT(2, true, 4); TK_TW_OPT(2, true, 8);
    TK_TW_OPT(1, false, 4); TK_TW_OPT(2, false, 4); TK_TW_OPT(4, false, 4); TK_TW_OPT(8, false, 4); TK_TW_OPT(16, false, 2); TK_TW_OPT(8, false, 2); TK_TW_OPT(6, false, 2);
#undef TK_TW_OPT
    if (e == hipSuccess) e = tw_opt_in(k_gemm_tiled<1, 4, true, 4, 2>);
    if (e == hipSuccess) e = tw_opt_in(k_gemm_tiled<1, 4, true, 8, 2>);
    if (e == hipSuccess) e = tw_opt_in(k_gemm_tiled<1, 4, true, 4, 4>);
    if (e == hipSuccess) e = tw_opt_in(k_gemm_tiled<1, 4, true, 8, 4>);
    if (e != hipSuccess) return false;
    g_tw_opted[dev].store(true, std::memory_order_release);
    return true;
}

static bool tw_valid(const TkTiledGemm& a) {
    if (a.nseg < 1 || a.nseg > 3 || a.ks < 1 || a.K <= 0 || a.K % (32 * a.ks) || a.nrows <= 0 || (a.wbytes != 2 && a.wbytes != 4) || (a.ks > 1 && a.nrows > a.slab_rows)) return false;
    if ((a.per_seg || a.c_img) && a.ks != 1) return false;
    if (a.per_seg && (a.residual || a.c_img)) return false;
    if (!a.per_seg && !a.out && (!a.c_img || a.wbytes == 2)) return false;
    if (a.per_seg && a.wbytes == 2 && (a.seg_img[0] || a.seg_img[1] || a.seg_img[2])) return false;
    if (a.ln_x && (a.ks != 1 || a.wbytes != 4 || a.K > TK_TW_LN_MAX || a.nrows > TK_TW_LN_ROWS || a.K % 128)) return false;
    return !(a.c_img && (a.n_valid % 16 || a.nseg != 1));
}
static int tw_row_tiles(const TkTiledGemm& a) {
    int n = 0;
    for (int i = 0; i < a.nseg; ++i) n += a.row_tiles[i];
    return n;
}

/* the rest of a cut, M-tiles of a workgroup and its waves given; false: no staging of this k range */
static bool tw_plan(const TkTiledGemm& a, int mt, int waves, TkTiledPlan* p) {
    if ((mt != 1 && mt != 2 && mt != 4 && mt != 6 && mt != 8 && mt != 16) || waves < 1 || waves > 8) return false;
    const int row_tiles = tw_row_tiles(a), Kr = a.K / a.ks;
    *p = TkTiledPlan{};
    p->mt = mt;
    p->waves = waves;
    p->groups = (row_tiles + waves - 1) / waves;
    p->ny = (a.nrows + mt * TK_TW_ROWS_PER_TILE - 1) / (mt * TK_TW_ROWS_PER_TILE);
    /* k per ring slot: the largest multiple of 32 PF that divides the K range and fits a 64 KiB slot (rk / 16 * mt KiB) — a whole short
     * range in one slot (`one`, up to 128 KiB) needs no ring.
     * Many row blocks of 128 rows (of products that are none of k_gemm_wide's): 32 KiB slots and two weight pieces in flight instead, so
     * that TWO workgroups share a CU and one's ring fill and epilogue run under the other's MFMAs. */
    const bool twin = p->ny > 1 && (mt == 8 || mt == 6) && Kr % 64 == 0;
    p->reg = mt == 1 && waves == 1 && Kr % 128 == 0 && a.wbytes == 4 && !a.ln_x; /* a wave by itself shares nothing */
    p->one = p->reg || (mt <= 2 && Kr % 128 == 0 && (size_t)Kr * mt * 64 <= 2 * TK_TW_SLOT_BYTES);
    /* whole range: eight pieces of weights in flight where they divide it, but not all of it at once: 51872 x 256, f32, 1 and 32 rows 14.9 and 18.9 us with
     * four, 18.2 and 22.6 with eight */
    p->pf = mt == 16 || mt == 6 || twin ? 2 : p->one && Kr % 256 == 0 && Kr > 256 ? 8 : 4;
    const int slot_kib = twin ? 32 : 64;
    p->rk = p->one ? Kr : 0;
    for (int c = (slot_kib * 16 / mt) / (32 * p->pf) * (32 * p->pf); p->rk == 0 && c >= 32 * p->pf; c -= 32 * p->pf)
        if (Kr % c == 0) p->rk = c;
    if (p->rk == 0) return false;
    p->slot_bytes = twin ? slot_kib * 1024 : TK_TW_SLOT_BYTES;
    p->lds = p->reg ? 0 : p->one ? (size_t)Kr * mt * 64 : (size_t)2 * p->slot_bytes;
    return true;
}

/* What a launch costs, in cycles: a workgroup's staging (its whole activations, or a slot and the waits for the further ones), its chains of 8 cycles a k and M-tile, then the
 * CU's further workgroups on the same pipe; or the weights, which every block of rows fetches from the L2 again, whichever is longer.  Fitted to 1 700 launches
 * of 1 .. 48 000 rows against 384 x 384 .. 51 872 x 384. */
static float tw_cost(const TkTiledGemm& a, const TkTiledPlan& p) {
    const int row_tiles = tw_row_tiles(a), Kr = a.K / a.ks;
    const float rounds = (float)p.groups * (float)p.ny * (float)a.ks * (1.0f / 256.0f), up = ceilf(rounds);
    int side_by_side = (int)(163840 / (p.lds + 1)) < 16 / p.waves ? (int)(163840 / p.lds) : 16 / p.waves;
    if (side_by_side < 1) side_by_side = 1;
    const int per = (p.waves + 3) / 4;
    const float kib = (float)p.lds * (1.0f / 1024.0f), waits = p.one ? 0.0f : (float)(Kr / p.rk) * 1012.0f;
    const float lone = (float)side_by_side < up ? (float)side_by_side : up;
    const float chain = (float)(per * p.mt * Kr) * ((float)(per * p.mt) * lone <= 1.0f ? 6.0f : 8.6f);
    float turns = side_by_side > 1 ? 0.61f * rounds + 0.39f * up : up;
    turns = turns > 1.0f ? turns - 1.0f : 0.0f;
    const float again = 0.25f * (float)(p.waves * p.mt) * (float)Kr * 10.3f + 21.0f * (float)(p.waves * p.mt) + 0.5f * waits / (float)side_by_side + (p.one ? 24.0f * kib : 0.0f);
    const float pipe = 1100.0f + (p.one ? 158.0f * kib : 1030.0f) + chain + waits + turns * again;
    const float weights = 1100.0f + (float)p.ny * (float)row_tiles * 16.0f * (float)a.K * (float)a.wbytes * (1.0f / 4100.0f);
    return pipe > weights ? pipe + 0.15f * weights : weights + 0.15f * pipe;
}

/*
 * f16 weights, operands in registers: how many M-tiles a wave makes (1 .. 4) and how many waves share a workgroup.  The chip's SIMDs take (tile columns x parts of k x row
 * blocks) in rounds; a wave of m M-tiles takes m + 1 units of time (its products, and the weights' way and conversion once), a lone one of four a quarter more; of equal
 * ones the larger.  What that chooses is within 7 % of the best measured of m = 1 .. 4 with one, four and a CU's share of waves, for 16 matrices of 256 .. 8192 k at 1, 16, 24,
 * 33, 64, 96, 128 rows, but for 1024 x 5632 at 128 rows (20.1 us; m = 1 18.7, the ring 25.7).  Ring or one LDS image / this, us: 4096 x 28672 at 1, 16, 24, 33, 64 rows 61 / 42, 52.7 / 50.6, 83 / 68, 142 / 97, 142 / 131;
 * 14336 x 4096 in seven parts 25.4 / 24.2, (25.2 / 26.4), 43.5 / 35.7, 73 / 51, 74 / 70; 4096 x 4096 35 / 20, 36 / 21, 52 / 21, 84 / 22, 85 / 23; 2048 x 2048 in four parts
 * 6.2 / 5.1, 6.5 / 5.4, 6.8 / 5.8, 9.0 / 7.7, 9.5 / 7.8; 256 x 768 4.4 / 3.8 .. 4.9 / 4.3.  The one in brackets stays with the image in LDS: rows that all 16 of a tile hold
 * and parts of more than 1024 k, whose operands a CU's waves no longer find in its L1 (8192 x 28672 in four parts at 12 rows 98 / 103; at 8 rows 96 / 89).
 * 65 .. 128 rows: up to one and a half tile columns a SIMD (4096 x 6144 in four parts at 96 rows 54 / 43; beyond, 4096 x 28672 at 96 and 128 rows 203 / 198 and 250 / 255).
 * 49 .. 64 rows: behind k_gemm_wide's rule, where both are alike (4096 x 65536 269 / 268, x 40960 195 / 197).
 */
static int tk_tiled_num_cu();
static bool tw_reg_plan(const TkTiledGemm& a, bool behind_wide, TkTiledPlan* p) {
    const int Kr = a.K / a.ks, tiles = (a.nrows + TK_TW_ROWS_PER_TILE - 1) / TK_TW_ROWS_PER_TILE, row_tiles = tw_row_tiles(a);
    if (a.wbytes != 2 || a.ln_x || Kr % 128 || tiles > 8 || (!behind_wide && tiles > 3)) return false;
    const int64_t cus = tk_tiled_num_cu(), simds = 4 * cus, units = (int64_t)row_tiles * a.ks;
    if (units > 400000 || (tiles > 4 && 2 * units > 3 * simds)) return false;
    if (a.nrows > 8 && tiles == 1 && a.ks > 1 && Kr > 1024 && Kr <= 2048 && 2 * units > 3 * simds) return false;
    int mt = 0;
    int64_t least = 0;
    for (int m = 1; m <= 4 && m <= tiles; ++m) {
        const int64_t rounds = (units * ((tiles + m - 1) / m) + simds - 1) / simds, cost = rounds * (m + 1) * (m == 4 && rounds == 1 ? 5 : 4);
        if (mt == 0 || cost <= least) { mt = m; least = cost; }
    }
    *p = TkTiledPlan{};
    p->mt = mt;
    p->ny = (tiles + mt - 1) / mt;
    p->reg = p->one = true;
    p->rk = Kr;
    /* more waves than SIMDs and one row block: as many workgroups as CUs, whose waves share the operands that they find in its L1 (4096 x 28672 at 1 row 42.3 us, single
     * waves 45.2); else a wave a workgroup, which spreads them evenly (4096 x 8192 at 24 rows 22.5, in twos 37.1) */
    p->waves = 1;
    p->groups = row_tiles;
    if (p->ny == 1 && units > simds) {
        int groups = (int)(cus / a.ks);
        groups = groups < 1 ? 1 : groups > row_tiles ? row_tiles : groups;
        while ((row_tiles + groups - 1) / groups > 8) groups *= 2;
        p->waves = (row_tiles + groups - 1) / groups;
        p->groups = groups;
    }
    /* one M-tile, no more waves than SIMDs: eight pieces of weights in flight (4096 x 4096 at 1 row 22.4 -> 19.9 us; 4096 x 6144 in four parts, 1536 waves, 11.9 -> 12.9) */
    p->pf = mt == 1 && units * p->ny <= simds && Kr % 256 == 0 ? 8 : 4;
    return true;
}
static bool tw_usual(const TkTiledGemm& a, TkTiledPlan* p);
bool tk_gemm_wide_plan(const TkTiledGemm& a, int form, TkTiledPlan* p);
bool tk_gemm_tiled_plan(const TkTiledGemm& a, int mt, int waves, TkTiledPlan* p) {
    if (!tw_valid(a)) return false;
    if (mt > 0) return tw_plan(a, mt, waves, p);
    /* Many rows: tiles of 32 x 32 without LDS, from 544 of them on (a chip has 1024 SIMDs).  Ring / wide time, 22 matrices at 260 .. 2000 rows: up to 384 tiles 0.4 .. 0.9
     * (1152 x 384 1.2), 432 .. 576 0.8 .. 1.3, from 640 on 1.1 .. 1.6.  Form 2 where the weights are more than an XCD's L2 holds and there are tiles to spare: 5120 x 1280
     * at 1500 and 12 000 rows 203 -> 179 and 1395 -> 1150 us; 512 rows 74 -> 86, 1536 x 384 at 48 000 rows 469 -> 485. */
    /* f16 weights, from 33 rows on, where the chip's SIMDs get two tiles each; beyond 64 rows, which the ring kernel reads more than once, one and a half, or two and a half of
     * short parts of k.  By ring / wide time of 400 products, 512 .. 5120 wide, 33 .. 256 rows: up to 64 rows 0.34 .. 1.02 below the line, 1.06 .. 1.35 above; beyond 0.35 ..
     * 1.00 and 0.93 .. 2.3.  Layers' products by the ring / as chosen: 1536 wide at 33 rows 47 / 47 us (all in wide tiles 55), 2048 at 96 143 / 127, 4096 at 64 296 / 296 (314),
     * at 160 1026 / 682.  Form 2
     * does a step of its 64 rows in 0.96 of the time that two tiles of form 1 take, but has half as many tiles to spread: 256 rows x 4096, 6144, 28672 columns 72.7, 105.5,
     * 530 us against 76.8, 109.1, 491. */
    if (tw_reg_plan(a, false, p)) return true;
    if (a.wbytes == 2 && a.nrows > 2 * TK_TW_ROWS_PER_TILE) {
        const int64_t cols = (int64_t)(tw_row_tiles(a) / 2) * a.ks, simds = 4 * (int64_t)tk_tiled_num_cu();
        const int64_t one = (a.nrows + 31) / 32 * cols, two = (a.nrows + 63) / 64 * cols;
        const int form = 1.92f * (float)((two + simds - 1) / simds) < (float)((one + simds - 1) / simds) ? 2 : 1;
        const int64_t least = a.nrows <= 64 ? 2 * simds : a.K / a.ks >= 512 ? simds * 3 / 2 : simds * 5 / 2;
        if (one >= least && tk_gemm_wide_plan(a, form, p)) return true;
        if (tw_reg_plan(a, true, p)) return true;
    }
    if (a.wbytes == 4 && a.nrows > TK_TW_MAX_BLOCK_ROWS) {
        const int64_t tiles = (int64_t)((a.nrows + 31) / 32) * (tw_row_tiles(a) / 2);
        const bool large = (size_t)tw_row_tiles(a) * 16 * (size_t)a.K * 4 > (4u << 20);
        if (tiles >= 544 && tk_gemm_wide_plan(a, large && tiles >= 3840 ? 2 : 1, p)) return true;
    }
    /* Up to five tiles of 16 x 16 for eight SIMDs: a wave each, operands in registers.  LDS (the best of 1, 2, 4, 8 waves) / registers, us, cold weights: 1 row x 384, 1152,
     * 1536 columns of 384 k 4.9, 5.2, 5.2 / 4.3, 4.4, 4.4, x 384 of 1536 k 11.0 / 9.1, x 1280 of 1280 9.9 / 8.1, x 5120 of 1280 (320 tiles) 10.2 / 9.5; 32 rows 5.7, 5.8, 5.8 / 5.0,
     * 5.1, 5.2, 11.7 / 9.7, 10.4 / 8.8, 15.1 / 14.6 (640 tiles); beyond, 128 rows x 1536 of 384 (768) 6.4 / 6.7, x 2048 of 512 (1024) 8.1 / 9.7, 48 x 5120 of 1280 (960) 14.9 / 17.8. */
    if (a.wbytes == 4 && !a.ln_x && a.ks == 1) {
        const int64_t tiles = (int64_t)((a.nrows + TK_TW_ROWS_PER_TILE - 1) / TK_TW_ROWS_PER_TILE) * tw_row_tiles(a);
        if (2 * tiles <= 5 * (int64_t)tk_tiled_num_cu() && tw_plan(a, 1, 1, p) && p->reg) return true;
    }
    if (!tw_usual(a, p)) return false;
    /* As many rows as possible behind one reading of the weights is what counts where these are large.  Small matrices (up to 24 MB: they come from the caches) of few
     * tiles leave most of the chip idle that way: fewer M-tiles a workgroup, where that is clearly quicker by the costs, measured 384 x 384 at 32, 256 and 1500 rows
     * 7.8 -> 5.6, 41 -> 5.4, 26.5 -> 10.4 us, 384 x 1536 at 32 and 256 20.3 -> 11.9, 123 -> 12.0.  No cut reads rows of the image that the usual one does not. */
    const TkTiledPlan usual = *p;
    if ((size_t)tw_row_tiles(a) * 16 * (size_t)a.K * (size_t)a.wbytes > 24000000u || (int64_t)tw_row_tiles(a) * usual.ny * a.ks >= 4096) return true;
    float least = 0.93f * tw_cost(a, usual);
    const int mts[5] = {1, 2, 4, 6, 8}, wvs[3] = {2, 4, 8};
    for (int m : mts)
        for (int w : wvs) {
            TkTiledPlan q;
            if (!tw_plan(a, m, w, &q) || (m == 1 && !q.one) || q.ny * q.mt > usual.ny * usual.mt || q.ny > 65535) continue;
            const float c = tw_cost(a, q);
            if (c < least) { least = c; *p = q; }
        }
    return true;
}
static bool tw_usual(const TkTiledGemm& a, TkTiledPlan* p) {
    int mt, waves;
    const int row_tiles = tw_row_tiles(a);
    const int rows_blk = a.nrows < TK_TW_MAX_BLOCK_ROWS ? a.nrows : TK_TW_MAX_BLOCK_ROWS;
    mt = rows_blk > 128 ? 16 : rows_blk > 64 ? 8 : rows_blk > 32 ? 4 : rows_blk > 16 ? 2 : 1;
    if (mt == 16 && a.nrows > TK_TW_MAX_BLOCK_ROWS && (a.K / a.ks) % 64 == 0) {
        /* many row blocks: two workgroups per CU (below), 512 at a time on the chip; of 128- and 96-row blocks the one whose last round
         * wastes less (N = 376 at 48 000 rows: 1 125 workgroups = 3 rounds of 8 M-tiles against 1 500 = 3 rounds of 6) */
        const long wg_per_blk = (row_tiles + 7) / 8;
        const long slots = 2L * tk_tiled_num_cu();
        const long c8 = (((a.nrows + 127) / 128) * wg_per_blk + slots - 1) / slots * 8;
        const long c6 = (((a.nrows + 95) / 96) * wg_per_blk + slots - 1) / slots * 6;
        mt = c6 < c8 ? 6 : 8;
    }
    const int ny = (a.nrows + mt * TK_TW_ROWS_PER_TILE - 1) / (mt * TK_TW_ROWS_PER_TILE);
    /* one pass of <= 256 rows (the LLM): spread the row tiles over the CUs, K-split ranges side by side; many row blocks: eight tiles
     * per workgroup share one activation ring */
    if (ny == 1) {
        int groups = 256 / a.ks;
        if (groups < 1) groups = 1;
        if (groups > row_tiles) groups = row_tiles;
        waves = (row_tiles + groups - 1) / groups;
        while (waves > 8) { groups *= 2; waves = (row_tiles + groups - 1) / groups; }
        if (waves == 1 && row_tiles >= 4) { /* fewer tiles than CUs: one-tile waves that share a workgroup's staging.  More of them ask one CU for more weights at a time,
             * fewer stage more each: 384 x 1536 at 1 row 10.9, 10.2, 10.8 us with 1, 2, 4 waves, at 32 rows 24.8, 20.7, 18.9 */
            waves = mt == 1 ? 2 : 4;
            groups = (row_tiles + waves - 1) / waves;
        }
        if (!tw_plan(a, mt, waves, p)) return false;
        p->groups = groups;
        return true;
    }
    return tw_plan(a, mt, row_tiles < 8 ? row_tiles : 8, p);
}

/* the cut of k_gemm_wide's form 1 (32 x 32 of the output a wave) or 2 (64 x 32); false: not a product it takes */
bool tk_gemm_wide_plan(const TkTiledGemm& a, int form, TkTiledPlan* p) {
    if (!tw_valid(a) || form < 1 || form > 2 || (a.wbytes == 4 && a.ks != 1) || a.ln_x || (a.c_img && (a.wbytes == 2 || a.out || a.residual)) || a.K % (128 * a.ks)) return false;
    if (a.ks > 1 && (a.bias || a.residual || a.act || a.add_zero_bias)) return false; /* parts of k are sums alone */
    for (int i = 0; i < a.nseg; ++i)
        if (a.row_tiles[i] % 2 || (a.per_seg && a.seg_n[i] != a.row_tiles[i] * 16)) return false;
    if (!a.per_seg && a.n_valid != tw_row_tiles(a) * 16) return false;
    *p = TkTiledPlan{};
    p->wide = form;
    p->groups = tw_row_tiles(a) / 2;
    p->ny = (a.nrows + 32 * form - 1) / (32 * form);
    return (int64_t)p->groups * p->ny * a.ks < 0x7fffff00;
}
bool tk_launch_gemm_tiled_plan(const TkTiledGemm& a, const TkTiledPlan& p, hipStream_t s) {
    if (p.wide) {
        TkTiledPlan w; /* (the cut follows from the form) */
        if (!tk_gemm_wide_plan(a, p.wide, &w)) return false;
        const int total = w.groups * w.ny * a.ks, per = ((total + 3) / 4 + 7) / 8;
        const dim3 wgrid((unsigned)per * 8);
#define TK_TW_WIDE(WBV, MIV, KSV, PFV) hipLaunchKernelGGL((k_gemm_wide<WBV, MIV, KSV, PFV>), wgrid, dim3(256), 0, s, a, w.groups, w.ny, total, per)
        if (a.wbytes == 2) {
            if (p.wide == 1) TK_TW_WIDE(2, 1, 32, 4);
            else TK_TW_WIDE(2, 2, 32, 2);
        } else if (p.wide == 1) TK_TW_WIDE(4, 1, 32, 2);
        else TK_TW_WIDE(4, 2, 16, 2);
#undef TK_TW_WIDE
        return true;
    }
    const int row_tiles = tw_row_tiles(a);
    if (a.ln_x) {
        if (p.mt != 1 || !p.one) return false;
#define TK_TW_LN(PFV, NV) hipLaunchKernelGGL((k_gemm_tiled<1, 4, true, PFV, NV>), dim3(p.groups, p.ny), dim3(64 * p.waves), p.lds, s, a, p.groups, row_tiles, p.rk, p.slot_bytes)
        if (a.K <= 512) { if (p.pf == 8) TK_TW_LN(8, 2); else TK_TW_LN(4, 2); }
        else { if (p.pf == 8) TK_TW_LN(8, 4); else TK_TW_LN(4, 4); }
#undef TK_TW_LN
        return true;
    }
#define TK_TW_LAUNCH(MTV, WBV, ONEV, PFV) hipLaunchKernelGGL((k_gemm_tiled<MTV, WBV, ONEV, PFV>), dim3(p.groups * a.ks, p.ny), dim3(64 * p.waves), p.lds, s, a, p.groups, row_tiles, p.rk, p.slot_bytes)
#define TK_TW_LAUNCH_REG(MTV, WBV, PFV) hipLaunchKernelGGL((k_gemm_tiled<MTV, WBV, true, PFV, 0, true>), dim3(8 * p.ny, (p.groups * a.ks + 7) / 8), dim3(64 * p.waves), 0, s, a, p.groups, row_tiles, p.rk, p.slot_bytes)
#define TK_TW_REG(MTV, PFV) do { if (a.wbytes == 2) TK_TW_LAUNCH_REG(MTV, 2, PFV); else TK_TW_LAUNCH_REG(MTV, 4, PFV); } while (0)
#define TK_TW_WB(MTV, ONEV, PFV) do { if (a.wbytes == 2) TK_TW_LAUNCH(MTV, 2, ONEV, PFV); else TK_TW_LAUNCH(MTV, 4, ONEV, PFV); } while (0)
    switch (p.mt) {
        case 1: if (p.reg) { if (p.pf == 8) TK_TW_REG(1, 8); else TK_TW_REG(1, 4); }
                else if (p.one) { if (p.pf == 8) TK_TW_WB(1, true, 8); else TK_TW_WB(1, true, 4); } else TK_TW_WB(1, false, 4); break;
        case 2: if (p.reg) TK_TW_LAUNCH_REG(2, 2, 4);
                else if (p.one) { if (p.pf == 8) TK_TW_WB(2, true, 8); else TK_TW_WB(2, true, 4); } else TK_TW_WB(2, false, 4); break;
        case 3: if (!p.reg) return false;
                TK_TW_LAUNCH_REG(3, 2, 4); break;
        case 4: if (p.reg) TK_TW_LAUNCH_REG(4, 2, 4); else TK_TW_WB(4, false, 4); break;
        case 6: TK_TW_WB(6, false, 2); break;
        case 8: if (p.pf == 2) TK_TW_WB(8, false, 2); else TK_TW_WB(8, false, 4); break;
        default: TK_TW_WB(16, false, 2); break;
    }
#undef TK_TW_WB
#undef TK_TW_REG
#undef TK_TW_LAUNCH_REG
#undef TK_TW_LAUNCH
    return true;
}
bool tk_launch_gemm_tiled(const TkTiledGemm& a, hipStream_t s) {
    TkTiledPlan p;
    return tk_gemm_tiled_plan(a, 0, 0, &p) && tk_launch_gemm_tiled_plan(a, p, s);
}
