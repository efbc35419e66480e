/* tk_decoder.hip — see tk_decoder.h */
#include "tk_decoder.h"

#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <system_error>
#include <thread>
#include <vector>

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

std::mutex& tk_capture_mutex() {
    static std::mutex mu;
    return mu;
}

bool TkDecodeSession::graphs_enabled() {
    /* TK_MI355X_NO_GRAPH=1: eager launches, for profilers that cannot follow hipGraphLaunch */
    const char* ng = getenv("TK_MI355X_NO_GRAPH");
    return !(ng && ng[0] == '1');
}

bool TkDecodeSession::init_tables(int device, int vocab, int row_cap, size_t extra, int32_t** extra_tab) {
    device_ = device;
    vocab_ = vocab;
    row_cap_ = row_cap;
    HIPQ(hipSetDevice(device));
    HIPQ(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
    const size_t ints = 3 * (size_t)row_cap + extra;
    HIPQ(hipMalloc((void**)&d_block_, ints * 4));
    HIPQ(hipMemset(d_block_, 0, ints * 4));
    d_seq = d_block_;
    d_pos = d_seq + row_cap;
    d_tok = d_pos + row_cap;
    if (extra_tab) *extra_tab = d_tok + row_cap;
    HIPQ(hipMalloc((void**)&logits, (size_t)TK_MAX_ROWS * vocab * 4));
    if ((size_t)TK_MAX_ROWS * vocab * 4 > TK_OUT_DIRECT) {
        /* here, and not with the first large copy, of whose call it took 0.06 .. 0.7 ms.  None to be had: those copies are plain ones */
        if (hipHostMalloc((void**)&out_ring_, TK_OUT_PIECES * (TK_OUT_PIECE + 4), hipHostMallocDefault) == hipSuccess) {
            memset(out_ring_ + TK_OUT_PIECES * TK_OUT_PIECE, 0, TK_OUT_PIECES * 4);
        } else {
            out_ring_ = nullptr;
            (void)hipGetLastError();
        }
        HIPQ(hipMalloc((void**)&d_out_done_, TK_OUT_PIECES * 4));
        HIPQ(hipMemset(d_out_done_, 0, TK_OUT_PIECES * 4));
    }
    HIPQ(hipMalloc((void**)&d_nsteps, TK_MAX_ROWS * 4));
    HIPQ(hipMemset(d_nsteps, 0, TK_MAX_ROWS * 4));
    hist_cap = max_ctx;
    HIPQ(hipMalloc((void**)&d_hist, (size_t)hist_cap * TK_MAX_ROWS * 4));
    HIPQ(hipMalloc((void**)&d_mask, (size_t)TK_MAX_ROWS * (((size_t)vocab + 31) / 32) * 4));
    HIPQ(hipMalloc((void**)&d_mask_row, TK_MAX_ROWS * 4));
    HIPQ(hipMemset(d_mask_row, 0xFF, TK_MAX_ROWS * 4));
    mask_rows_dirty = false;
    HIPQ(hipMalloc((void**)&d_samp, TK_MAX_ROWS * sizeof(TkSampleRow)));
    HIPQ(hipMemset(d_samp, 0, TK_MAX_ROWS * sizeof(TkSampleRow))); /* temp 0: every row samples greedily */
    samp_dirty = false;
    return true;
}

TkDecodeSession::~TkDecodeSession() {
    if (!stream && !d_block_) return;
    (void)hipSetDevice(device_);
    void* ptrs[] = {d_block_, logits, d_out_done_, d_nsteps, d_hist, d_mask, d_mask_row, d_samp};
    for (void* p : ptrs) if (p) (void)hipFree(p);
    if (out_ring_) (void)hipHostFree(out_ring_);
    if (stream) (void)hipStreamDestroy(stream);
}

/* floats of `dev` to pinned memory, in pieces of TK_OUT_PIECE; whoever finishes a piece says so in there[piece].  `done` counts a piece's workgroups and is zero between launches */
__global__ __launch_bounds__(256) void k_send_out(const float* __restrict__ dev, float* __restrict__ host, int64_t n, unsigned* done, unsigned* there, unsigned epoch) {
    constexpr int PER = TK_OUT_PIECE / 4 / TK_OUT_GROUPS; /* floats of a workgroup */
    const int piece = blockIdx.x / TK_OUT_GROUPS;
    const int64_t at = (int64_t)blockIdx.x * PER;
    typedef float v4f __attribute__((ext_vector_type(4)));
    if (at + PER <= n) {
        v4f v[PER / 1024];
#pragma unroll
        for (int k = 0; k < PER / 1024; ++k) v[k] = *(const v4f*)(dev + at + 1024 * k + 4 * threadIdx.x);
#pragma unroll
        for (int k = 0; k < PER / 1024; ++k) *(v4f*)(host + at + 1024 * k + 4 * threadIdx.x) = v[k];
    } else {
        for (int64_t i = at + threadIdx.x; i < n && i < at + PER; i += 256) host[i] = dev[i];
    }
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0 && __hip_atomic_fetch_add(done + piece, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == TK_OUT_GROUPS - 1) {
        __hip_atomic_store(done + piece, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(there + piece, epoch, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

/* A copy to pageable memory goes through the runtime's own staging a MiB at a time, 20 us on the bus and 50 .. 70 us of host memcpy in turn: 0.3 .. 0.4 ms for 40 rows x 32 000
 * logits, behind a step of 0.65 ms.  Here a kernel writes them to pinned memory (55 GB/s), and the caller and up to three threads, started when the first piece is there, take
 * each piece to its place as it arrives.  Copies with an event a piece instead cost 13 us a piece on the stream.  The pinned memory is the session's and bounded (two halves,
 * one being filled while the other is taken away); nothing of it is handed out. */
bool TkDecodeSession::copy_out(void* host, const void* dev, size_t bytes) {
    if (bytes <= TK_OUT_DIRECT || !out_ring_ || bytes % 4) {
        HIPQ(hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, stream));
        return true;
    }
    constexpr size_t HALF = TK_OUT_PIECES / 2;
    const size_t n = (bytes + TK_OUT_PIECE - 1) / TK_OUT_PIECE;
    std::atomic<size_t> next{0}; /* pieces taken by a thread */
    std::vector<std::atomic<unsigned>> left((n + HALF - 1) / HALF); /* pieces of each half-ring not yet taken away */
    std::vector<std::atomic<bool>> on_way(left.size()); /* of each by itself: they are sent in the order in which threads free their places, which is any order */
    for (auto& w : on_way) w.store(false, std::memory_order_relaxed);
    std::atomic<int> failed{hipSuccess};
    unsigned* const there = (unsigned*)(out_ring_ + TK_OUT_PIECES * TK_OUT_PIECE);
    const unsigned epoch0 = out_epoch_;
    out_epoch_ += (unsigned)left.size();
    auto send = [&](size_t g) { /* the pieces [g HALF, (g + 1) HALF) */
        const size_t b0 = g * HALF * TK_OUT_PIECE, len = std::min(HALF * TK_OUT_PIECE, bytes - b0), pieces = (len + TK_OUT_PIECE - 1) / TK_OUT_PIECE, slot = (g & 1) * HALF;
        left[g].store((unsigned)pieces);
        hipLaunchKernelGGL(k_send_out, dim3((unsigned)(pieces * TK_OUT_GROUPS)), dim3(256), 0, stream, (const float*)dev + b0 / 4, (float*)(out_ring_ + slot * TK_OUT_PIECE), (int64_t)(len / 4),
                           d_out_done_ + slot, there + slot, epoch0 + (unsigned)g);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) { failed.store(e); return; }
        on_way[g].store(true, std::memory_order_release);
    };
    auto arrived = [&](size_t i) { return on_way[i / HALF].load(std::memory_order_acquire) && __atomic_load_n(there + i % TK_OUT_PIECES, __ATOMIC_ACQUIRE) == epoch0 + (unsigned)(i / HALF); };
    auto wait = [&](size_t i) { /* as the runtime waits: actively, and politely once it takes long; a stream that has ended without the piece has failed */
        const auto t0 = std::chrono::steady_clock::now();
        for (unsigned spin = 1; !arrived(i); ++spin) {
            if (failed.load() != hipSuccess) return false;
            std::this_thread::yield();
            if (spin % 256) continue;
            if (on_way[i / HALF].load()) {
                const hipError_t e = hipStreamQuery(stream);
                if (e != hipErrorNotReady && !arrived(i)) { failed.store(e == hipSuccess ? hipErrorUnknown : e); return false; }
            }
            if (std::chrono::steady_clock::now() - t0 > std::chrono::milliseconds(5)) std::this_thread::sleep_for(std::chrono::microseconds(20));
        }
        return true;
    };
    auto take = [&] {
        (void)hipSetDevice(device_);
        for (size_t i; (i = next.fetch_add(1)) < n && wait(i);) {
            memcpy((uint8_t*)host + i * TK_OUT_PIECE, out_ring_ + i % TK_OUT_PIECES * TK_OUT_PIECE, std::min(TK_OUT_PIECE, bytes - i * TK_OUT_PIECE));
            const size_t g = i / HALF;
            if (left[g].fetch_sub(1) == 1 && g + 2 < left.size()) send(g + 2); /* its half is free: the one behind the other half's */
        }
    };
    send(0);
    if (left.size() > 1 && failed.load() == hipSuccess) send(1);
    std::thread more[3];
    if (wait(0)) {
        try {
            for (size_t t = 0; t < 3 && 2 * (t + 1) < n; ++t) more[t] = std::thread(take);
        } catch (const std::system_error&) { /* no thread to be had: fewer do it */
        }
        take();
    }
    for (std::thread& t : more) if (t.joinable()) t.join();
    const hipError_t e = (hipError_t)failed.load();
    if (e != hipSuccess) (void)hipStreamSynchronize(stream); /* nothing of it may still be on its way into the ring */
    HIPQ(e);
    return true;
}

bool TkDecodeSession::reset() {
    HIPQ(hipSetDevice(device_));
    HIPQ(hipMemsetAsync(d_nsteps, 0, TK_MAX_ROWS * 4, stream));
    HIPQ(hipStreamSynchronize(stream));
    return true;
}

bool TkDecodeSession::rows_in_range(int nrows, const int32_t* seq, const int32_t* pos, const int32_t* tok) {
    for (int r = 0; r < nrows; ++r)
        if (seq[r] < 0 || seq[r] >= max_seq || pos[r] < 0 || pos[r] >= max_ctx || tok[r] < 0 || tok[r] >= vocab_) {
            error = "row out of range (sequence id, position or token id)";
            return false;
        }
    return true;
}

bool TkDecodeSession::stage_sampling(int n, const int32_t* rows, const uint32_t* const* row_masks, const TkSampleRow* row_samp) {
    /* per-row sampling masks: the masks of the constrained rows, compacted, + the row -> mask table the arg max kernel reads */
    int32_t rowtab[TK_MAX_ROWS];
    int nmask = 0;
    const size_t words = ((size_t)vocab_ + 31) / 32;
    for (int r = 0; r < TK_MAX_ROWS; ++r) rowtab[r] = -1;
    for (int i = 0; i < n; ++i) {
        const int r = rows ? rows[i] : i;
        if (row_masks && row_masks[r]) {
            HIPQ(hipMemcpyAsync(d_mask + (size_t)nmask * words, row_masks[r], words * 4, hipMemcpyHostToDevice, stream));
            rowtab[i] = nmask++;
        }
    }
    if (nmask > 0 || mask_rows_dirty) {
        HIPQ(hipMemcpyAsync(d_mask_row, rowtab, TK_MAX_ROWS * 4, hipMemcpyHostToDevice, stream)); /* whole table (a wider pass may have left entries); pageable source: staged before the call returns */
        mask_rows_dirty = nmask > 0;
    }
    /* per-row sampling state (temp <= 0: greedy): data of the pass like the masks, so sampled and greedy rows share passes and graphs */
    bool any_samp = false;
    for (int i = 0; i < n && row_samp; ++i) any_samp = any_samp || row_samp[rows ? rows[i] : i].temp > 0.0f;
    if (any_samp) {
        if (vocab_ > 65536) { error = "stochastic sampling supports vocabularies of at most 65536 tokens"; return false; }
        TkSampleRow tab[TK_MAX_ROWS] = {};
        for (int i = 0; i < n; ++i) tab[i] = row_samp[rows ? rows[i] : i];
        HIPQ(hipMemcpyAsync(d_samp, tab, sizeof tab, hipMemcpyHostToDevice, stream));
        samp_dirty = true;
    } else if (samp_dirty) {
        HIPQ(hipMemsetAsync(d_samp, 0, TK_MAX_ROWS * sizeof(TkSampleRow), stream));
        samp_dirty = false;
    }
    return true;
}

bool TkDecodeSession::capture(hipGraphExec_t* slot, const std::function<void()>& enqueue) {
    if (*slot) return true;
    const auto t_cap = std::chrono::steady_clock::now();
    struct Tally { TkDecodeSession* s; std::chrono::steady_clock::time_point t0; ~Tally() { s->n_captures++; s->capture_ms += std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count(); } } tally{this, t_cap};
    std::lock_guard<std::mutex> lk(tk_capture_mutex());
    hipGraph_t g = nullptr;
    HIPQ(hipStreamBeginCapture(stream, hipStreamCaptureModeRelaxed));
    launch_error.clear();
    enqueue();
    /* from here on the stream must leave capture mode and the graph must be freed whatever fails */
    const hipError_t e_end = hipStreamEndCapture(stream, &g);
    hipError_t e_inst = hipSuccess;
    if (e_end == hipSuccess && launch_error.empty()) e_inst = hipGraphInstantiate(slot, g, nullptr, nullptr, 0);
    if (g) (void)hipGraphDestroy(g);
    if (e_end != hipSuccess || e_inst != hipSuccess || !launch_error.empty()) {
        if (*slot && e_inst != hipSuccess) { (void)hipGraphExecDestroy(*slot); }
        *slot = nullptr;
        (void)hipGetLastError();
        error = !launch_error.empty() ? launch_error
                : std::string("graph capture of a pass failed: ") + hipGetErrorString(e_end != hipSuccess ? e_end : e_inst);
        return false;
    }
    return true;
}

bool TkDecodeSession::decode(int nrows, int n_steps, int32_t* out_tokens_host) {
    if (nrows <= 0 || nrows > TK_MAX_ROWS) { error = "nrows must be in [1,256]"; return false; }
    if (n_steps <= 0 || n_steps > hist_cap) { error = "n_steps exceeds the session context"; return false; }
    HIPQ(hipSetDevice(device_));
    /* positions must stay inside the cache for the whole loop */
    int32_t hpos[TK_MAX_ROWS];
    HIPQ(hipMemcpyAsync(hpos, d_pos, nrows * 4, hipMemcpyDeviceToHost, stream));
    HIPQ(hipStreamSynchronize(stream));
    for (int r = 0; r < nrows; ++r)
        if (hpos[r] + n_steps > max_ctx) { error = "decode would run past max_ctx"; return false; }
    if (!begin_decode(nrows, hpos, n_steps)) return false;
    const bool use_graph = graphs_enabled();
    int top0 = 0;
    for (int r = 0; r < nrows; ++r) top0 = hpos[r] > top0 ? hpos[r] : top0;
    HIPQ(hipMemsetAsync(d_nsteps, 0, TK_MAX_ROWS * 4, stream));
    if (mask_rows_dirty) { HIPQ(hipMemsetAsync(d_mask_row, 0xFF, TK_MAX_ROWS * 4, stream)); mask_rows_dirty = false; } /* the loop samples unconstrained */
    hipEvent_t e0, e1;
    HIPQ(hipEventCreate(&e0));
    HIPQ(hipEventCreate(&e1));
    HIPQ(hipEventRecord(e0, stream));
    int done = 0;
    bool ok = true;
    launch_error.clear();
    for (; done < n_steps && ok; ++done) {
        hipGraphExec_t* slot = decode_slot(nrows, top0 + done); /* positions advance on the device; the host knows where the loop stands */
        if (use_graph) {
            ok = capture(slot, [&] { enqueue_decode(nrows); });
            if (ok && hipGraphLaunch(*slot, stream) != hipSuccess) { error = "graph launch of a decode step failed"; ok = false; }
        } else {
            enqueue_decode(nrows);
            if (!launch_error.empty()) { error = launch_error; ok = false; }
        }
        if (!ok) break;
    }
    end_decode(nrows, done);
    launch_error.clear();
    if (!ok) { (void)hipStreamSynchronize(stream); (void)hipEventDestroy(e0); (void)hipEventDestroy(e1); return false; }
    HIPQ(hipGetLastError());
    HIPQ(hipEventRecord(e1, stream));
    if (out_tokens_host) HIPQ(hipMemcpyAsync(out_tokens_host, d_hist, (size_t)n_steps * TK_MAX_ROWS * 4, hipMemcpyDeviceToHost, stream));
    HIPQ(hipStreamSynchronize(stream));
    float ms = 0.0f;
    HIPQ(hipEventElapsedTime(&ms, e0, e1));
    last_step_ms = ms / n_steps;
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    return true;
}
