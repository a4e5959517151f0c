// reduce.hip -- greedy argmax and exact top-16 over vocabulary logits.
//
// Grid (ceil(nvocab / CHUNK), T).  Each 256-thread workgroup owns CHUNK = 2048 logits of a row
// (8 per thread, coalesced), finds its chunk's best candidate (argmax) or best 16 (top-16) and writes
// them as partials.  The last workgroup to finish a row (arrival counter, reset by that workgroup)
// merges the partials the same way.  Order: larger value first, ties -> lower vocab index; a NaN is
// never selected.  The top-16 is exact: every global top-16 element is a top-16 element of its own
// chunk.
// reference: row_argmax_multi_kernel / row_top16_multi_kernel (src/wzy_kernels_v2.cuh:1873-1984).
#include "wzy_device.h"
#include "wzy_host.h"
#include "wzy_reduce.h"

using namespace wzy;

namespace {
constexpr int RD_THREADS = 256;
constexpr int RD_PER_THREAD = 8;
constexpr int RD_CHUNK = RD_THREADS * RD_PER_THREAD;   // 2048

constexpr int RD_NONE = 0x7fffffff;                     // index of an empty slot

// Best (value, index) of the block's 8 values per thread; every thread gets it.
WZY_DEV void block_best(const float (&v)[RD_PER_THREAD], const int (&ix)[RD_PER_THREAD], float& gv, int& gi, float* sv,
                        int* si) {
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    float bv = -INFINITY;
    int bi = RD_NONE;
#pragma unroll
    for (int j = 0; j < RD_PER_THREAD; ++j) amax_merge(bv, bi, v[j], ix[j]);
    wave_argmax(bv, bi);
    if (lane == 0) { sv[w] = bv; si[w] = bi; }
    __syncthreads();
    gv = sv[0];
    gi = si[0];
#pragma unroll
    for (int k = 1; k < RD_THREADS / 64; ++k) amax_merge(gv, gi, sv[k], si[k]);
    __syncthreads();
}

// (value, index) as one key, larger = better: the value's bits in numeric order (both zeros alike), then
// the inverted index.  A NaN gives the empty slot's key, (-inf, RD_NONE).
WZY_DEV uint64_t rd_key(float v, int i) {
    const bool none = v != v;
    const uint32_t b = __builtin_bit_cast(uint32_t, none ? -INFINITY : v + 0.0f);
    const uint32_t o = (b & 0x80000000u) ? ~b : b | 0x80000000u;
    return ((uint64_t) o << 32) | (uint32_t) ~(none ? RD_NONE : i);
}
WZY_DEV int rd_index(uint64_t k) { return (int) ~(uint32_t) k; }

// The block's 16 best of 8 keys per thread into s_out, best first.  Each lane sorts its eight, each wave
// takes its 16 best from the lane heads (a DPP maximum per round, no barrier), and 64 lanes rank the four
// waves' candidates against each other.  (16 rounds of a block-wide argmax, two barriers each, took 14 us a
// pass: the top-16 of 151,936 logits 31 -> 17 us.)
WZY_DEV void block_top16(uint64_t (&k)[8], uint64_t* s_cand, uint64_t* s_out) {
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    auto ce = [&](int a, int b) {                       // larger first
        const bool sw = k[b] > k[a];
        const uint64_t x = sw ? k[b] : k[a], y = sw ? k[a] : k[b];
        k[a] = x;
        k[b] = y;
    };
    // odd-even merge sort of eight
    ce(0, 1); ce(2, 3); ce(4, 5); ce(6, 7);
    ce(0, 2); ce(1, 3); ce(4, 6); ce(5, 7);
    ce(1, 2); ce(5, 6);
    ce(0, 4); ce(1, 5); ce(2, 6); ce(3, 7);
    ce(2, 4); ce(3, 5);
    ce(1, 2); ce(3, 4); ce(5, 6);
    const uint64_t none = rd_key(-INFINITY, RD_NONE);
    uint64_t mine = none;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        // the largest value among the lane heads; the index decides only where several lanes hold it
        const uint32_t hi = (uint32_t) (k[0] >> 32), lo = (uint32_t) k[0], mh = wave_max_u32(hi);
        const uint64_t at = __ballot(hi == mh);
        uint32_t ml;
        if (__popcll(at) == 1) ml = (uint32_t) __builtin_amdgcn_readlane((int) lo, __ffsll((unsigned long long) at) - 1);
        else ml = wave_max_u32(hi == mh ? lo : 0u);
        const uint64_t m = ((uint64_t) mh << 32) | ml;
        mine = lane == r ? m : mine;
        const bool won = k[0] == m;                     // keys differ, empty ones apart
#pragma unroll
        for (int j = 0; j < 7; ++j) k[j] = won ? k[j + 1] : k[j];
        k[7] = won ? none : k[7];
    }
    if (lane < 16) s_cand[16 * w + lane] = mine;
    if (tid < 16) s_out[tid] = none;
    __syncthreads();
    if (w == 0) {
        const uint64_t c = s_cand[lane];
        int rank = 0;
#pragma unroll
        for (int j = 0; j < 64; ++j) rank += s_cand[j] > c ? 1 : 0;
        if (rank < 16 && c != none) s_out[rank] = c;
    }
    __syncthreads();
}

// Publish a chunk's partials (written by this workgroup before) and tell whether it is the row's last.
WZY_DEV bool last_of_row(unsigned* cnt, int nchunk, int* s_last) {
    __threadfence();
    __syncthreads();
    if (threadIdx.x == 0) *s_last = (atomicAdd(cnt, 1u) == (unsigned) (nchunk - 1));
    __syncthreads();
    if (!*s_last) return false;
    __threadfence();
    return true;
}
}  // namespace

__global__ void __launch_bounds__(RD_THREADS) row_argmax_kernel(const float* __restrict__ logits, int nvocab,
                                                                float* __restrict__ part_v, int* __restrict__ part_i,
                                                                unsigned* __restrict__ row_cnt,
                                                                int* __restrict__ greedy) {
    __shared__ float sv[RD_THREADS / 64];
    __shared__ int si[RD_THREADS / 64];
    __shared__ int s_last;
    const int tid = threadIdx.x;
    const int row = blockIdx.y, nchunk = gridDim.x;
    const float* l = logits + (size_t) row * nvocab;

    float v[RD_PER_THREAD], gv;
    int ix[RD_PER_THREAD], gi;
    const int base = blockIdx.x * RD_CHUNK;
#pragma unroll
    for (int j = 0; j < RD_PER_THREAD; ++j) {
        const int i = base + j * RD_THREADS + tid;
        v[j] = i < nvocab ? l[i] : -INFINITY;
        ix[j] = i < nvocab ? i : RD_NONE;
    }
    block_best(v, ix, gv, gi, sv, si);
    if (tid == 0) {
        part_v[(size_t) row * nchunk + blockIdx.x] = gv;
        part_i[(size_t) row * nchunk + blockIdx.x] = gi;
    }
    if (!last_of_row(&row_cnt[row], nchunk, &s_last)) return;

    // merge the partials (at most RD_CHUNK of them)
    const float* av = part_v + (size_t) row * nchunk;
    const int* ai = part_i + (size_t) row * nchunk;
#pragma unroll
    for (int j = 0; j < RD_PER_THREAD; ++j) {
        const int k = j * RD_THREADS + tid;
        v[j] = k < nchunk ? av[k] : -INFINITY;
        ix[j] = k < nchunk ? ai[k] : RD_NONE;
    }
    block_best(v, ix, gv, gi, sv, si);
    if (tid == 0) {
        if (greedy) greedy[row] = gi;
        row_cnt[row] = 0u;
    }
}

__global__ void __launch_bounds__(RD_THREADS) row_top16_kernel(const float* __restrict__ logits, int nvocab,
                                                               uint64_t* __restrict__ part, unsigned* __restrict__ row_cnt,
                                                               int* __restrict__ greedy, float* __restrict__ top_v,
                                                               int* __restrict__ top_i) {
    __shared__ uint64_t s_cand[64], s_out[16];
    __shared__ int s_last;
    const int tid = threadIdx.x;
    const int row = blockIdx.y, nchunk = gridDim.x;
    const float* l = logits + (size_t) row * nvocab;
    const uint64_t none = rd_key(-INFINITY, RD_NONE);

    uint64_t k[RD_PER_THREAD];
    const int base = blockIdx.x * RD_CHUNK;
#pragma unroll
    for (int j = 0; j < RD_PER_THREAD; ++j) {
        const int i = base + j * RD_THREADS + tid;
        const float v = l[min(i, nvocab - 1)];
        k[j] = i < nvocab ? rd_key(v, i) : none;
    }
    block_top16(k, s_cand, s_out);
    uint64_t* ap = part + (size_t) row * nchunk * 16;
    if (tid < 16) ap[blockIdx.x * 16 + tid] = s_out[tid];
    if (!last_of_row(&row_cnt[row], nchunk, &s_last)) return;

    // merge nchunk * 16 partials (at most RD_CHUNK of them)
    const int n = nchunk * 16;
#pragma unroll
    for (int j = 0; j < RD_PER_THREAD; ++j) {
        const int i = j * RD_THREADS + tid;
        const uint64_t c = ap[min(i, n - 1)];
        k[j] = i < n ? c : none;
    }
    block_top16(k, s_cand, s_out);
    if (tid < 16) {
        const int i = rd_index(s_out[tid]);
        if (top_v) top_v[row * 16 + tid] = i == RD_NONE ? -INFINITY : l[i];
        if (top_i) top_i[row * 16 + tid] = i;
        if (tid == 0) {
            if (greedy) greedy[row] = i;
            row_cnt[row] = 0u;
        }
    }
}

namespace wzy {

size_t reduce_ws_bytes(int nvocab, int T) {
    const int nchunk = (nvocab + RD_CHUNK - 1) / RD_CHUNK;
    return align_up((size_t) T * nchunk * 16 * 8, 256) + 256;
}

// ws layout: [row counters: 64 x u32][partials]
int launch_row_reduce(const float* logits, int nvocab, int T, bool top16, int* greedy, float* top_v, int* top_i,
                      void* ws, hipStream_t st) {
    WZY_REQUIRE(logits && ws && nvocab > 0 && T >= 1 && T <= 64, "row reduce: bad arguments");
    const int nchunk = (nvocab + RD_CHUNK - 1) / RD_CHUNK;
    WZY_REQUIRE((size_t) nchunk * 16 <= (size_t) RD_CHUNK, "row reduce: nvocab too large (%d)", nvocab);
    unsigned* cnt = (unsigned*) ws;
    char* part = (char*) ws + 256;
    if (top16)
        hipLaunchKernelGGL(row_top16_kernel, dim3(nchunk, T), dim3(RD_THREADS), 0, st, logits, nvocab, (uint64_t*) part, cnt,
                           greedy, top_v, top_i);
    else
        hipLaunchKernelGGL(row_argmax_kernel, dim3(nchunk, T), dim3(RD_THREADS), 0, st, logits, nvocab, (float*) part,
                           (int*) part + (size_t) T * nchunk, cnt, greedy);
    WZY_LAUNCH_CHECK();
    return WZY_OK;
}

}  // namespace wzy

// Stand-alone entry points keep a per-device scratch for counters/partials (allocated on first use,
// counters zero-initialised once; every launch leaves them at zero).
static int reduce_scratch(int nvocab, int T, void** out) {
    static void* buf[64] = {nullptr};
    static size_t cap[64] = {0};
    int dev = 0;
    WZY_HIP_TRY(hipGetDevice(&dev));
    WZY_REQUIRE(dev >= 0 && dev < 64, "row reduce: device id out of range");
    const size_t need = reduce_ws_bytes(nvocab, T);
    if (cap[dev] < need) {
        if (buf[dev]) WZY_HIP_TRY(hipFree(buf[dev]));
        buf[dev] = nullptr;
        cap[dev] = 0;
        if (hipMalloc(&buf[dev], need) != hipSuccess) {
            set_error("row reduce: hipMalloc(%zu) failed", need);
            return WZY_ENOMEM;
        }
        WZY_HIP_TRY(hipMemset(buf[dev], 0, need));
        cap[dev] = need;
    }
    *out = buf[dev];
    return WZY_OK;
}

extern "C" int wzy_row_argmax(const float* logits, int nvocab, int T, int* out_ids, void* stream) {
    WZY_REQUIRE(out_ids, "wzy_row_argmax: null output");
    void* ws = nullptr;
    WZY_TRY(reduce_scratch(nvocab, T, &ws));
    return launch_row_reduce(logits, nvocab, T, false, out_ids, nullptr, nullptr, ws, as_stream(stream));
}

extern "C" int wzy_row_top16(const float* logits, int nvocab, int T, int* out_greedy, float* top_v, int* top_i,
                             void* stream) {
    void* ws = nullptr;
    WZY_TRY(reduce_scratch(nvocab, T, &ws));
    return launch_row_reduce(logits, nvocab, T, true, out_greedy, top_v, top_i, ws, as_stream(stream));
}
