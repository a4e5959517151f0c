// prefill.hip -- kernels of the chunked prefill (B prompt cells per launch sequence) on gfx950.
//
//  pf_gemm       every dense projection of the chunk on bf16 MFMA (v_mfma_f32_32x32x16_bf16):
//                128 x 128 or 64 x 64 output tiles, K in steps of 64 through LDS; Q8_0 weights are
//                dequantised (code * fp16 scale, rounded to bf16) on their way into LDS, bf16
//                weights copied.  Workgroups are numbered so that the eight XCDs take interleaved row
//                tiles and each runs all weight tiles of its row tile back to back.  A few bf16
//                weight rows (N <= 16) take pf_skinny instead (fp32 FMA dot products per row).
//  HC read       pf_hc_norm (pending block folded in, per-stream RMSNorm, bf16), GEMMs for inject /
//                down (K split by stream) / up (the stream mean as its epilogue), pf_silu_div; pf_hc_write
//                writes a block into the streams.
//  GDN           pf_gdn_ab (gates), pf_gdn_conv (causal conv + SiLU + L2 of q/k heads over all rows
//                at once), pf_gdn_hist (conv history), pf_gdn_recur (the delta rule, sequential over
//                the rows: 32 lanes per state column, 4 rows each in registers; k, v and gates staged in
//                LDS 32 rows at a time, q in registers), pf_gdn_norm (gated RMS norm, bf16).
//  QSA           pf_qsa_prep (q / k / indexer-q norms + RoPE, INT8 KV append), pf_idx_append (the
//                indexer keys of every block the chunk completes, one workgroup per block, then
//                pf_idx_tail), block scores on fp16 MFMA (pf_score), top-k with the decode kernel,
//                pf_attn (sparse GQA attention on fp16 MFMA, K and V from memory straight into the
//                matrix operands).
// reference: PrefillStageCtx::run_stage_prefill and its kernels (src/wzy_prefill_tc.cuh:20-98,
// 546-1058; src/wzy_qsa_wmma.cuh:5-489), with cuBLAS fp16 GEMMs replaced by bf16 MFMA GEMMs.
#include <algorithm>
#include <type_traits>

#include "wzy_device.h"
#include "wzy_host.h"
#include "wzy_prefill.h"
#include "wzy_qsa.h"
#include "wzy_qsa_dev.h"

using namespace wzy;

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x3_t __attribute__((ext_vector_type(3)));
typedef int i32x2_t __attribute__((ext_vector_type(2)));
typedef int i32x4_t __attribute__((ext_vector_type(4)));

namespace {

WZY_DEV uint16_t f_to_bf16(float f) { return __builtin_bit_cast(uint16_t, (__bf16) f); }   // nearest even
WZY_DEV uint32_t pack_bf16(float a, float b) {                                              // both in one conversion
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{a, b}, bf16x2_t));
}

// ---------------------------------------------------------------------------------------------
// dense GEMM
// ---------------------------------------------------------------------------------------------
constexpr int GK = 64, GLD = GK + 8;                         // k step, LDS row (bf16)

struct GemmArgs {
    PfGemm g;
    int mt, nt;
};

// eight Q8_0 codes times their fp16 scale, rounded to bf16
WZY_DEV uint4 q8_quarter_bf16(uint32_t a, uint32_t b, float sc) {
    return make_uint4(pack_bf16((float) (int8_t) a * sc, (float) (int8_t) (a >> 8) * sc),
                      pack_bf16((float) (int8_t) (a >> 16) * sc, (float) (int8_t) (a >> 24) * sc),
                      pack_bf16((float) (int8_t) b * sc, (float) (int8_t) (b >> 8) * sc),
                      pack_bf16((float) (int8_t) (b >> 16) * sc, (float) (int8_t) (b >> 24) * sc));
}

// UM: the HC up projection with the stream mean as its epilogue.  Tile column n holds stream
// c = n % 4 of position d = n / 4 (weight row c * um_d + d), so a row's four stream gates sit in
// one lane quad and are combined there in stream order.
// T: tile side; a wave holds a quarter of the tile.  An element's sum runs over k in the same order and
// instructions whatever T.
// SB: one LDS buffer (37 KB), so four workgroups share a CU (three with the UM epilogue, whose
// registers allow no more); the next k step still loads into registers during the MFMAs, and a second
// barrier per step guards the buffer.  Launches with at least 512 tiles use it; smaller ones keep two.
// With a thread's 64 bytes of one row per step replaced by whole rows per eight lanes (below), 8,192 x 6,144 x
// 2,048 took 296 -> 261 us from Q8_0 and 276 -> 250 us from bf16 (826 TFLOP/s), 250 x 12,288 x 2,048 50 -> 29.
template <int T, bool UM, bool SB, bool Q8>
__global__ void __launch_bounds__(256, SB ? (UM ? 3 : 4) : T == 64 ? (Q8 ? 4 : 3) : 2) pf_gemm_kernel(GemmArgs ga) {
    constexpr int GM = T, GN = T, NB = T / 64;                     // tile; 32 x 32 blocks per wave and side
    constexpr int NBUF = SB ? 1 : 2, NA = GM / 32, NW = Q8 ? GN / 64 : GN / 32;
    __shared__ __align__(16) uint16_t sAW[NBUF * (GM + GN) * GLD];
    uint16_t (*const sA)[GM][GLD] = (uint16_t (*)[GM][GLD]) sAW;
    uint16_t (*const sW)[GN][GLD] = (uint16_t (*)[GN][GLD]) (sAW + NBUF * GM * GLD);
    constexpr int XS_LD = GN + 8;                                  // UM epilogue: xn tile row stride
    static_assert(GM * XS_LD <= NBUF * (GM + GN) * GLD, "the UM epilogue's xn tile fits the GEMM's LDS");
    const PfGemm& g = ga.g;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, wm = w & 1, wn = w >> 1;
    const int tiles = ga.mt * ga.nt;
    const int ksp = (int) blockIdx.x / tiles;                      // K range of a split launch
    const int b = (int) blockIdx.x - ksp * tiles;
    int mi, ni;
    if ((ga.mt & 7) == 0) {
        const int s = b >> 3;
        mi = (s / ga.nt) * 8 + (b & 7);
        ni = s % ga.nt;
    } else {
        mi = b / ga.nt;
        ni = b % ga.nt;
    }
    const int m0 = mi * GM, n0 = ni * GN;
    const int nk = g.K / GK / max(g.ksplit, 1);                    // k steps of this launch's range
    const size_t k0 = (size_t) ksp * nk * GK;
    // Staging: eight lanes read a row's 128 bytes of a k step (four its 64 Q8_0 codes), so a load touches 8
    // cache lines (16) and not 64.  Thread -> rows tid / 8 + 32 i, k 8 (tid % 8) .. +7 of A and of bf16 weights;
    // rows tid / 4 + 64 i, k 16 (tid % 4) .. +15 of Q8_0 weights.
    const int ar = tid >> 3, ak = (tid & 7) * 8, qr = tid >> 2, qk = (tid & 3) * 16;
    const uint16_t* ap[NA];
    const uint16_t* wbp[NW];
    const int8_t* wqp[NW];
    const uint16_t* wsp[NW];
    auto wrow = [&](int r) {                                       // weight row of tile column r
        const size_t n = (size_t) min(n0 + r, g.N - 1);
        return UM ? (n & 3) * (size_t) g.um_d + (n >> 2) : n;
    };
#pragma unroll
    for (int i = 0; i < NA; ++i) ap[i] = g.a + (size_t) min(m0 + ar + 32 * i, g.M - 1) * g.lda + k0 + ak;
#pragma unroll
    for (int i = 0; i < NW; ++i) {
        if constexpr (Q8) {
            wqp[i] = g.wq + wrow(qr + 64 * i) * g.K + k0 + qk;
            wsp[i] = g.ws + wrow(qr + 64 * i) * (g.K / 32) + (k0 + qk) / 32;
        } else {
            wbp[i] = g.wb + wrow(ar + 32 * i) * g.K + k0 + ak;
        }
    }
    // DEPTH k steps are in flight, in register sets used in turn: small launches leave a SIMD one or two waves,
    // and a step takes as long as its loads unless they left several steps before (250 x 2,048 x 6,144 in bf16
    // on 64-wide tiles: 37 us with two, 26 with three).  Q8_0 gains more from a fourth workgroup per CU than
    // from a third step (the same product from Q8_0: 43 us against 56).
    constexpr int DEPTH = SB ? 1 : Q8 ? 2 : 3;
    u32x4_t ra[DEPTH][NA], rw[DEPTH][NW];
    uint16_t rs[DEPTH][NW];
    auto load = [&](int q, int ks) {                               // past the end the last step again
        ks = min(ks, nk - 1);
        const size_t o = (size_t) ks * GK;
#pragma unroll
        for (int i = 0; i < NA; ++i) ra[q][i] = *(const u32x4_t*) (ap[i] + o);
#pragma unroll
        for (int i = 0; i < NW; ++i) {
            if constexpr (Q8) {
                rw[q][i] = *(const u32x4_t*) (wqp[i] + o);
                rs[q][i] = wsp[i][ks * (GK / 32)];
            } else {
                rw[q][i] = *(const u32x4_t*) (wbp[i] + o);
            }
        }
    };
    auto store = [&](int q, int buf) {
#pragma unroll
        for (int i = 0; i < NA; ++i) *(u32x4_t*) &sA[buf][ar + 32 * i][ak] = ra[q][i];
#pragma unroll
        for (int i = 0; i < NW; ++i) {
            if constexpr (Q8) {
                const float sc = h16_to_f(rs[q][i]);
                *(uint4*) &sW[buf][qr + 64 * i][qk] = q8_quarter_bf16(rw[q][i].x, rw[q][i].y, sc);
                *(uint4*) &sW[buf][qr + 64 * i][qk + 8] = q8_quarter_bf16(rw[q][i].z, rw[q][i].w, sc);
            } else {
                *(u32x4_t*) &sW[buf][ar + 32 * i][ak] = rw[q][i];
            }
        }
    };

    f32x16_t acc[NB][NB];
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    // step ks (in buffer ks % 2): set q held it and takes step ks + DEPTH; step ks + 1 goes to the other buffer
    auto step = [&](int q, int ks) {
        const int buf = SB ? 0 : (ks & 1);
        load(q, ks + DEPTH);
#pragma unroll
        for (int kk = 0; kk < GK / 16; ++kk) {
            bf16x8_t av[NB], bv[NB];
#pragma unroll
            for (int i = 0; i < NB; ++i)
                av[i] = *(const bf16x8_t*) &sA[buf][wm * (GM / 2) + i * 32 + (lane & 31)][kk * 16 + (lane >> 5) * 8];
#pragma unroll
            for (int j = 0; j < NB; ++j)
                bv[j] = *(const bf16x8_t*) &sW[buf][wn * (GN / 2) + j * 32 + (lane & 31)][kk * 16 + (lane >> 5) * 8];
#pragma unroll
            for (int i = 0; i < NB; ++i)
#pragma unroll
                for (int j = 0; j < NB; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[i], bv[j], acc[i][j], 0, 0, 0);
        }
        if constexpr (SB) __syncthreads();                         // every wave is done with the buffer
        store((q + 1) % DEPTH, SB ? 0 : buf ^ 1);
        __syncthreads();
    };
#pragma unroll
    for (int q = 0; q < DEPTH; ++q) load(q, q);
    store(0, 0);
    __syncthreads();
    int ks = 0;
    for (; ks + DEPTH <= nk; ks += DEPTH) {
#pragma unroll
        for (int q = 0; q < DEPTH; ++q) step(q, ks + q);
    }
#pragma unroll
    for (int q = 0; q < DEPTH - 1; ++q)
        if (ks + q < nk) step(q, ks + q);                          // workgroup-uniform
    // acc[i][j][r] = C[row 8*(r/4) + 4*(lane/32) + r%4][col lane%32] of block (i, j)
    if constexpr (UM) {
        // mixed = (sum over streams in order of xn / (1 + exp(-bf16 gate))) / 4, fp32 and bf16
        // (pf_gr_up_mean_fp16, src/wzy_qsa_wmma.cuh:236-252); the xn loads of a 32 x 32 block go first
        // The tile's xn (GM rows x 4 streams x GN/4 positions, bf16) is staged in the GEMM's LDS, whose
        // last use ended at the loop's final barrier: 16-byte coalesced loads instead of 2-byte ones.
        const int D = g.um_d, c = lane & 3, d0 = n0 >> 2;
        uint16_t (*const xs)[XS_LD] = (uint16_t (*)[XS_LD]) sAW;     // [row][stream * GN/4 + position]
#pragma unroll
        for (int i = 0; i < GM * 4 * (GN / 4) / 8 / 256; ++i) {
            constexpr int PS = GN / 32;                              // 16-byte pieces per row and stream
            const int pc = tid + 256 * i, rr = pc / (4 * PS), sc = (pc / PS) & 3, q = pc % PS;
            const int row = min(m0 + rr, g.M - 1);
            *(uint4*) &xs[rr][sc * (GN / 4) + 8 * q] = *(const uint4*) (g.um_xn + (size_t) row * 4 * D + (size_t) sc * D + d0 + 8 * q);
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j) {
                const int d = (n0 + wn * (GN / 2) + j * 32 + (lane & 31)) >> 2;
                float xv[16];
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int rr = wm * (GM / 2) + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                    xv[r] = bf16_to_f(xs[rr][c * (GN / 4) + d - d0]);
                }
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int row = m0 + wm * (GM / 2) + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                    const float gq = bf16_to_f(f_to_bf16(acc[i][j][r]));
                    const float term = xv[r] / (1.0f + __expf(-gq));
                    float sum = 0.f + dpp_f<0x00>(term);             // quad lanes 0..3 = streams 0..3
                    sum += dpp_f<0x55>(term);
                    sum += dpp_f<0xAA>(term);
                    sum += dpp_f<0xFF>(term);
                    const float v = sum * 0.25f;
                    if (c == 0 && row < g.M) {
                        g.um_mixed[(size_t) row * D + d] = v;
                        g.um_xh[(size_t) row * D + d] = f_to_bf16(v);
                    }
                }
            }
        return;
    }
    float* const y = g.y ? g.y + (size_t) ksp * g.M * g.ldy : nullptr;
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            const int col = n0 + wn * (GN / 2) + j * 32 + (lane & 31);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = m0 + wm * (GM / 2) + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                if (row < g.M && col < g.N) {
                    if (y) y[(size_t) row * g.ldy + col] = acc[i][j][r];
                    else g.yb[(size_t) row * g.ldy + col] = f_to_bf16(acc[i][j][r]);
                }
            }
        }
}

// Skinny GEMM for a few bf16 weight rows (N <= 16: the hyper-connection inject, the GDN alpha /
// beta gates), where 128 x 128 MFMA tiles would leave most of the chip idle and read every
// activation row with 128-row tiles on 64 workgroups.  Each thread keeps its 8-value k slices of every
// weight row in registers (k = 2048 j + 8 tid .. +7), walks RB rows, and the block sums its partial
// dots (DPP within a wave, then four wave partials).  fp32 FMAs on the bf16 values.
constexpr int SK_RB = 16;                    // rows per workgroup

template <int NN, int KJ>
__global__ void __launch_bounds__(256) pf_skinny_kernel(PfGemm g) {
    __shared__ float s_red[2][4][NN];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    uint4 wv[NN][KJ];
#pragma unroll
    for (int n = 0; n < NN; ++n)
#pragma unroll
        for (int j = 0; j < KJ; ++j)
            wv[n][j] = *(const uint4*) (g.wb + (size_t) min(n, g.N - 1) * g.K + 2048 * j + 8 * tid);
    const int r0 = blockIdx.x * SK_RB, r1 = min(r0 + SK_RB, g.M);
    uint4 an[KJ];
#pragma unroll
    for (int j = 0; j < KJ; ++j) an[j] = *(const uint4*) (g.a + (size_t) r0 * g.lda + 2048 * j + 8 * tid);
    for (int t = r0; t < r1; ++t) {
        uint4 av[KJ];
#pragma unroll
        for (int j = 0; j < KJ; ++j) av[j] = an[j];
        if (t + 1 < r1) {                            // the next row's loads in flight
#pragma unroll
            for (int j = 0; j < KJ; ++j) an[j] = *(const uint4*) (g.a + (size_t) (t + 1) * g.lda + 2048 * j + 8 * tid);
        }
        float acc[NN];
#pragma unroll
        for (int n = 0; n < NN; ++n) acc[n] = 0.f;
#pragma unroll
        for (int j = 0; j < KJ; ++j) {
            const uint32_t aw[4] = {av[j].x, av[j].y, av[j].z, av[j].w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float x0 = bf16_lo(aw[e]), x1 = bf16_hi(aw[e]);
#pragma unroll
                for (int n = 0; n < NN; ++n) {
                    const uint32_t ww = e == 0 ? wv[n][j].x : e == 1 ? wv[n][j].y : e == 2 ? wv[n][j].z : wv[n][j].w;
                    acc[n] = fmaf(x0, bf16_lo(ww), acc[n]);
                    acc[n] = fmaf(x1, bf16_hi(ww), acc[n]);
                }
            }
        }
        const int pb = t & 1;                        // partials alternate buffers: one barrier per row
#pragma unroll
        for (int n = 0; n < NN; ++n) {
            const float v = wave_sum(acc[n]);
            if (lane == 0) s_red[pb][w][n] = v;
        }
        __syncthreads();
        if (tid < g.N && tid < NN)
            g.y[(size_t) t * g.ldy + tid] = (s_red[pb][0][tid] + s_red[pb][1][tid]) + (s_red[pb][2][tid] + s_red[pb][3][tid]);
    }
}

// ---------------------------------------------------------------------------------------------
// embedding and hyper-connection pieces
// ---------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256) pf_embed_kernel(PfEmb e, const int* __restrict__ toks, float* __restrict__ R,
                                                        int D, int HC) {
    const int t = blockIdx.y, d = blockIdx.x * 256 + threadIdx.x;
    if (d >= D) return;
    const int tok = toks[t];
    float v;
    if (e.emb_q) {                                   // stage_one_emb: out-of-range ids read row 0
        const size_t tk = (tok < 0 || tok >= e.n_vocab) ? 0 : (size_t) tok;
        v = h16_to_f(e.emb_s[(tk * D + d) / 32]) * (float) e.emb_q[tk * D + d];
    } else {
        const size_t tk = (size_t) max(0, min(tok, e.n_vocab - 1));
        v = bf16_to_f(e.emb[tk * D + d]);
    }
    for (int c = 0; c < HC; ++c) R[((size_t) t * HC + c) * D + d] = v;
}

// per (stream c, row t): R += bo * 2 sigmoid(inj_prev / HC) when a block is pending; x = bf16(R *
// rsqrt(mean R^2 + eps) * norm_w)  (pf_gr_norm_fp16, src/wzy_qsa_wmma.cuh:198-234)
// A thread holds NG groups of 4 consecutive values (group tid + 256 i), loaded and stored 16 bytes
// at a time; NG = ceil(D / 1024), D a multiple of 4 and at most 4096.
template <int NG>
__global__ void __launch_bounds__(256) pf_hc_norm_kernel(float* __restrict__ R, const float* __restrict__ bo,
                                                          const float* __restrict__ inj_prev,
                                                          const float* __restrict__ norm_w, uint16_t* __restrict__ xn,
                                                          int D, int HC, float eps) {
    __shared__ float s_red[4];
    const int c = blockIdx.x, t = blockIdx.y, tid = threadIdx.x;
    const int ng = D / 4;
    float4* r = (float4*) (R + ((size_t) t * HC + c) * D);
    const float4* bp = bo ? (const float4*) (bo + (size_t) t * D) : nullptr;
    const float gate = bo ? 2.0f / (1.0f + __expf(-inj_prev[t * HC + c] / (float) HC)) : 0.0f;
    float4 v[NG], bv[NG];
#pragma unroll
    for (int i = 0; i < NG; ++i) {                   // clamped, unconditional loads
        const int gi = min(tid + 256 * i, ng - 1);
        v[i] = r[gi];
        if (bo) bv[i] = bp[gi];
    }
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < NG; ++i) {
        const int gi = tid + 256 * i;
        if (bo) {
            v[i].x = fmaf(bv[i].x, gate, v[i].x);
            v[i].y = fmaf(bv[i].y, gate, v[i].y);
            v[i].z = fmaf(bv[i].z, gate, v[i].z);
            v[i].w = fmaf(bv[i].w, gate, v[i].w);
            if (gi < ng) r[gi] = v[i];
        }
        if (gi >= ng) v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        ss += v[i].x * v[i].x;
        ss += v[i].y * v[i].y;
        ss += v[i].z * v[i].z;
        ss += v[i].w * v[i].w;
    }
    ss = block_sum<4>(ss, s_red);
    const float inv = 1.0f / sqrtf(ss / (float) D + eps);
    const float4* wp = (const float4*) (norm_w + (size_t) c * D);
    uint2* x = (uint2*) (xn + (size_t) t * HC * D + (size_t) c * D);
#pragma unroll
    for (int i = 0; i < NG; ++i) {
        const int gi = tid + 256 * i;
        if (gi < ng) {
            const float4 w = wp[gi];
            x[gi] = make_uint2(pack_bf16(v[i].x * inv * w.x, v[i].y * inv * w.y),
                               pack_bf16(v[i].z * inv * w.z, v[i].w * inv * w.w));
        }
    }
}

__global__ void __launch_bounds__(256) pf_silu_div_kernel(const float* __restrict__ lo, uint16_t* __restrict__ loh,
                                                           size_t n, int nsplit, float inv_hc) {
    const size_t i = (size_t) blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float s = nsplit == 4 ? (lo[i] + lo[n + i]) + (lo[2 * n + i] + lo[3 * n + i]) : lo[i];
    const float v = s * inv_hc;
    loh[i] = f_to_bf16(v / (1.0f + __expf(-v)));
}

// R[t][c][d] += blk[t][d] * 2 sigmoid(inj[t][c] / HC)  (gr_write_multi, src/wzy_kernels_v2.cuh:813-827)
__global__ void __launch_bounds__(256) pf_hc_write_kernel(float* __restrict__ R, const float* __restrict__ blk,
                                                           const float* __restrict__ inj, int D, int HC) {
    const int t = blockIdx.y, i = blockIdx.x * 256 + threadIdx.x;
    if (i >= HC * D) return;
    const int c = i / D, d = i - c * D;
    const float g = 2.0f / (1.0f + __expf(-inj[t * HC + c] / (float) HC));
    float* r = R + (size_t) t * HC * D + i;
    *r = fmaf(blk[(size_t) t * D + d], g, *r);
}

// ---------------------------------------------------------------------------------------------
// GDN
// ---------------------------------------------------------------------------------------------
// decay = exp(softplus(a + dt) * ssm_a), beta = sigmoid(b)  (gdn_ab_act_pf_kernel)
__global__ void __launch_bounds__(256) pf_gdn_ab_kernel(PfGdn g) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= g.B * g.hv) return;
    const int t = i / g.hv, h = i - t * g.hv;
    const float a = g.ab[(size_t) t * 2 * g.hv + h] + g.dt[h];
    const float bv = g.ab[(size_t) t * 2 * g.hv + g.hv + h];
    g.beta[i] = 1.0f / (1.0f + __expf(-bv));
    const float sp = a > 20.0f ? a : log1pf(__expf(a));
    g.decay[i] = __expf(sp * g.ssm_a[h]);
}

// causal depthwise conv (3 history taps + the row) + SiLU, L2 norm of each q / k head; grid
// (QKV/128, B), 128 threads  (pf_gdn_conv_parallel, src/wzy_qsa_wmma.cuh:5-30)
// A thread runs CV_ROWS consecutive rows of its channel with a sliding window in registers, so every
// raw row is read once; the q / k rows' L2 norms span the workgroup's 128 channels (one head).
constexpr int CV_ROWS = 16;
__global__ void __launch_bounds__(128) pf_gdn_conv_kernel(PfGdn g) {
    __shared__ float s_red[2][2];                  // per row parity: one barrier per row
    const int grp = blockIdx.x, t0 = blockIdx.y * CV_ROWS, ch = grp * 128 + threadIdx.x, w = threadIdx.x >> 6;
    const int QKV = (2 * g.hk + g.hv) * 128;
    const float* h = g.conv_hist + (size_t) ch * 3;
    float win[CV_ROWS + 3];                        // rows t0-3 .. t0+CV_ROWS-1 (s < 0: history)
#pragma unroll
    for (int i = 0; i < CV_ROWS + 3; ++i) {
        const int s = t0 - 3 + i;
        win[i] = s < 0 ? h[3 + s] : g.qkv[(size_t) min(s, g.B - 1) * QKV + ch];
    }
    const float* wp = g.conv_w + (size_t) ch * 4;
    const float w0 = wp[0], w1 = wp[1], w2 = wp[2], w3 = wp[3];
    const bool qk = grp < 2 * g.hk;                // workgroup-uniform
#pragma unroll
    for (int r = 0; r < CV_ROWS; ++r) {
        const int t = t0 + r;
        if (t >= g.B) break;                       // workgroup-uniform
        const float sum = win[r] * w0 + win[r + 1] * w1 + win[r + 2] * w2 + win[r + 3] * w3;
        float y = sum / (1.0f + __expf(-sum));
        if (qk) {
            const float ws = wave_sum(y * y);
            if ((threadIdx.x & 63) == 0) s_red[r & 1][w] = ws;
            __syncthreads();
            const float ss = 0.f + s_red[r & 1][0] + s_red[r & 1][1];
            y *= 1.0f / sqrtf(ss + g.eps);
        }
        g.conv_out[(size_t) t * QKV + ch] = y;
    }
}

// conv history <- the last three raw rows (the older history where the chunk is shorter)
__global__ void __launch_bounds__(256) pf_gdn_hist_kernel(PfGdn g) {
    const int QKV = (2 * g.hk + g.hv) * 128;
    const int ch = blockIdx.x * 256 + threadIdx.x;
    if (ch >= QKV) return;
    float* h = g.conv_hist + (size_t) ch * 3;
    float v[3];
    for (int j = 0; j < 3; ++j) {
        const int s = g.B - 3 + j;
        v[j] = s >= 0 ? g.qkv[(size_t) s * QKV + ch] : h[3 + s];
    }
    h[0] = v[0];
    h[1] = v[1];
    h[2] = v[2];
}

// Sums of 32 per-lane values over each 32-lane half, transposed: lane r of the half returns the sum of
// v[r].  Five partner levels, each splitting the values a lane holds in two (16 swaps + 16 adds, then
// reduce_level's 3 operations per value left): about 2.4 operations per value instead of 7.
// (The swap is inline assembly: through the builtin, this compiler hands both results of the swap in
// one register when they feed one add.  The s_nops cover the VALU-write-to-permlane hazard.)
WZY_DEV float sum32_t(const float (&v)[32]) {
    const int lane = threadIdx.x & 63;
    float b[16], c[8], d[4], e[2], f[1];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        uint32_t x = __builtin_bit_cast(uint32_t, v[i]), y = __builtin_bit_cast(uint32_t, v[i + 16]);
        asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(x), "+v"(y));
        b[i] = __builtin_bit_cast(float, x) + __builtin_bit_cast(float, y);
    }
    reduce_level<DPP_ROW_ROR8, 16, 1>(b, c, (lane & 8) != 0);
    reduce_level<DPP_HALF_MIRROR, 8, 1>(c, d, (lane & 4) != 0);
    reduce_level<DPP_XOR2, 4, 1>(d, e, (lane & 2) != 0);
    reduce_level<DPP_XOR1, 2, 1>(e, f, (lane & 1) != 0);
    return f[0];
}

constexpr int GR_LPC = 32;                    // lanes per state column (half a wave)
constexpr int GR_RPL = 128 / GR_LPC;          // state rows per lane (4)
constexpr int GR_CPW = 64 / GR_LPC;           // columns per wave (2)
constexpr int GR_WAVES = 4;
constexpr int GR_COLS = GR_CPW * GR_WAVES;    // columns per workgroup (8)
constexpr int GR_STEPS = 32;                  // rows staged per LDS buffer (= lanes per column: lane r
                                              // stores row r's output)
static_assert(GR_STEPS * GR_COLS == 256, "v staging: one value per thread");
static_assert(GR_RPL == 4, "the row loop holds 4 state rows per lane");
static_assert(GR_STEPS == GR_LPC, "one output row per lane of a column");

// Delta rule over the chunk's rows for one value head and GR_COLS state columns (each column of
// the state evolves independently): per row, S *= decay; kv = S^T k; delta = (v - kv) * beta;
// S += k delta^T; o = S^T q / sqrt(128).  grid (hv * 128 / GR_COLS), 256 threads.  A column's 128
// rows are spread over 32 lanes (4 per lane), so 16 heads put one wave on every SIMD of the chip and a row
// costs what one wave issues, serially from row to row.  Only kv is reduced over the lanes in that chain
// (DPP within each 16-lane row, then a permlane swap); a row's S^T q stays a per-lane partial sum, and 32
// rows of them are reduced together, transposed, when their buffer ends (2.4 operations a row instead of 9,
// and no k . q correction).  k and, per column, v with the row's decay and beta go through LDS 32 rows at a
// time in 16-byte pieces, the next 32 loaded while these run; q stays out of LDS.
// 8,192 rows x 16 heads: 1,050 us with both sums reduced per row and k, q, v through LDS; 861 with the
// transposed sum and reads two rows ahead; about 800 with q in registers (about 32 instructions a row, of which
// 13 form the chain through kv).
// (pf_gdn_recur_kh_kernel, src/wzy_qsa_wmma.cuh:56-195; fused_gdn_step_norm_multi,
// src/wzy_kernels_v2.cuh:908-984)
__global__ void __launch_bounds__(256) pf_gdn_recur_kernel(PfGdn g) {
    __shared__ __align__(16) float sk[2][GR_STEPS][128];
    __shared__ f32x4_t svg[2][GR_STEPS][GR_COLS];               // v, decay, beta, unused
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int h = blockIdx.x / (128 / GR_COLS), cb = blockIdx.x % (128 / GR_COLS);
    const int kh = h % g.hk;
    const int QKV = (2 * g.hk + g.hv) * 128, GV = g.hv * 128;
    const int r8 = lane & (GR_LPC - 1), c8 = lane / GR_LPC;     // row slot, column of the wave
    const int lc = w * GR_CPW + c8, col = cb * GR_COLS + lc;
    float* S = g.state + (size_t) h * 128 * 128;
    float s[GR_RPL];
#pragma unroll
    for (int i = 0; i < GR_RPL; ++i) s[i] = S[(size_t) (r8 * GR_RPL + i) * 128 + col];

    // staging of rows t0 .. t0+GR_STEPS-1.  Row indices are clamped (rows past the chunk are never
    // used), so every load is unconditional.  Thread -> 4 k values of rows tid / 32 + 8 u; v and gates
    // of row tid / 8, column tid % 8.
    constexpr int K_PER = GR_STEPS * 128 / 4 / 256;       // 16-byte pieces per thread (4)
    f32x4_t rk[K_PER];
    f32x4_t rv = {0.f, 0.f, 0.f, 0.f};
    const int k_e = (tid & 31) * 4;
    const float* k_p = g.conv_out + (size_t) (g.hk + kh) * 128 + k_e;
    const float* v_p = g.conv_out + (size_t) 2 * g.hk * 128 + h * 128 + cb * GR_COLS + tid % GR_COLS;
    auto load = [&](int t0) {
#pragma unroll
        for (int u = 0; u < K_PER; ++u) rk[u] = *(const f32x4_t*) (k_p + (size_t) min(t0 + (tid >> 5) + 8 * u, g.B - 1) * QKV);
        const int t = min(t0 + tid / GR_COLS, g.B - 1);
        rv.x = v_p[(size_t) t * QKV];
        rv.y = g.decay[(size_t) t * g.hv + h];
        rv.z = g.beta[(size_t) t * g.hv + h];
    };
    auto store = [&](int bb) {
#pragma unroll
        for (int u = 0; u < K_PER; ++u) *(f32x4_t*) &sk[bb][(tid >> 5) + 8 * u][k_e] = rk[u];
        svg[bb][tid / GR_COLS][tid % GR_COLS] = rv;
    };
    // q does not go through LDS: a lane keeps its 4 q values of the 32 rows in registers and reloads a
    // row's right after its use, 32 rows ahead (four waves reading k and q of every row from LDS kept the
    // LDS busier than the VALU).  A lane's offset counts from the first of 32 rows and stops at the chunk's
    // last row; from the chunk's first row it would pass 32 bits (64 + 64 heads: at 43,691 rows).
    const char* const q_b = (const char*) (g.conv_out + (size_t) kh * 128);
    const uint32_t q_step = (uint32_t) QKV * 4;
    const char* q_w;
    uint32_t q_off, q_end;
    auto q_rows = [&](int r0) {                             // the next 32 rows to load are r0 ..
        r0 = min(r0, g.B - 1);
        q_w = q_b + (size_t) r0 * q_step;
        q_off = r8 * 16;
        q_end = q_off + min(GR_STEPS - 1, g.B - 1 - r0) * q_step;
    };
    f32x4_t q4[GR_STEPS];
    auto next_q = [&]() {
        const f32x4_t v = *(const f32x4_t*) (q_w + q_off);
        q_off = min(q_off + q_step, q_end);
        return v;
    };

    float cp[GR_STEPS];                                     // the buffer's rows: this lane's part of S^T q
    // Row st from its k and gates: kv and the update.  The part of S^T q of the row before (from the
    // state this row starts with), the decayed state and the loads fill the wait states between the
    // dependent lane moves; FENCE keeps them there.
#define FENCE __builtin_amdgcn_sched_barrier(0)
    auto row = [&](int st, const f32x4_t k4, const f32x4_t qp, const f32x3_t vg, auto&& reads) {
        float a = s[0] * k4.x, c = s[0] * qp.x;
        FENCE;
        a = fmaf(s[1], k4.y, a);
        c = fmaf(s[1], qp.y, c);
        FENCE;
        a = fmaf(s[2], k4.z, a);
        c = fmaf(s[2], qp.z, c);
        FENCE;
        a = fmaf(s[3], k4.w, a);
        c = fmaf(s[3], qp.w, c);
        FENCE;
        const float dec = vg.y;
        const float m0 = dec * s[0];
        FENCE;
        a += dpp_f<DPP_XOR1>(a);
        FENCE;
        const float m1 = dec * s[1], m2 = dec * s[2];
        FENCE;
        a += dpp_f<DPP_XOR2>(a);
        FENCE;
        const float m3 = dec * s[3];
        reads(0);
        FENCE;
        a += dpp_f<DPP_HALF_MIRROR>(a);
        FENCE;
        reads(1);
        FENCE;
        uint32_t x = __builtin_bit_cast(uint32_t, a + dpp_f<DPP_MIRROR>(a)), y = x;
        asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(x), "+v"(y));
        a = __builtin_bit_cast(float, x) + __builtin_bit_cast(float, y);
        const float delta = (vg.x - dec * a) * vg.z;
        s[0] = fmaf(k4.x, delta, m0);
        s[1] = fmaf(k4.y, delta, m1);
        s[2] = fmaf(k4.z, delta, m2);
        s[3] = fmaf(k4.w, delta, m3);
        FENCE;
        if (st > 0) cp[st - 1] = c;
    };
    auto last = [&](const f32x4_t qp) {                     // S^T q after a row
        float c = s[0] * qp.x;
        c = fmaf(s[1], qp.y, c);
        c = fmaf(s[2], qp.z, c);
        return fmaf(s[3], qp.w, c);
    };

    const int nfull = g.B / GR_STEPS, rest = g.B - nfull * GR_STEPS;
    q_rows(0);
#pragma unroll
    for (int st = 0; st < GR_STEPS; ++st) q4[st] = next_q();
    load(0);
    store(0);
    // the state has arrived before the loop: without this the wait for it stays inside, behind the
    // prefetch of the next buffer
    asm volatile("" : "+v"(s[0]), "+v"(s[1]), "+v"(s[2]), "+v"(s[3]));
    __syncthreads();
    // k and gates come from LDS two rows ahead, in register sets used in turn; the loop is unrolled over
    // the whole buffer, so every LDS address is a constant offset
    f32x4_t k4[3];
    f32x3_t vg[3];
    auto get = [&](int bb, int st) {
        k4[st % 3] = *(const f32x4_t*) &sk[bb][st][r8 * GR_RPL];
        vg[st % 3] = *(const f32x3_t*) &svg[bb][st][lc];
    };
    float* op = g.o + (size_t) r8 * GV + h * 128 + col;     // lane r8 stores row t0 + r8
    for (int kb = 0; kb < nfull; ++kb) {
        const int bb = kb & 1, t0 = kb * GR_STEPS;
        load(t0 + GR_STEPS);
        q_rows(t0 + GR_STEPS);
        get(bb, 0);
        get(bb, 1);
#pragma unroll
        for (int st = 0; st < GR_STEPS; ++st)
            row(st, k4[st % 3], q4[st > 0 ? st - 1 : 0], vg[st % 3], [&](int part) {
                if (part == 0 && st + 2 < GR_STEPS) get(bb, st + 2);
                if (part == 1 && st > 0) q4[st - 1] = next_q();
            });
        cp[GR_STEPS - 1] = last(q4[GR_STEPS - 1]);
        q4[GR_STEPS - 1] = next_q();
        const float o = sum32_t(cp) * 0.08838834764831845f;
        // the refill first: it waits for this buffer's loads, long arrived; the output store after it
        // is then waited on by nothing before the next buffer's rows
        store(bb ^ 1);
        op[(size_t) t0 * GV] = o;
        __syncthreads();
    }
    if (rest > 0) {
        const int bb = nfull & 1;
#pragma unroll
        for (int st = 0; st < GR_STEPS; ++st) {
            cp[st] = 0.f;
            if (st < rest) {                                 // workgroup-uniform
                get(bb, st);
                row(0, k4[st % 3], k4[st % 3], vg[st % 3], [&](int) {});
                cp[st] = last(q4[st]);
            }
        }
        const float o = sum32_t(cp) * 0.08838834764831845f;
        if (r8 < rest) op[(size_t) nfull * GR_STEPS * GV] = o;
    }
#pragma unroll
    for (int i = 0; i < GR_RPL; ++i) S[(size_t) (r8 * GR_RPL + i) * 128 + col] = s[i];
}
#undef FENCE

// y = bf16(o * rsqrt(mean o^2 + eps) * gamma * sigmoid(z)) per (head, row); grid (hv, B), 128 threads
// (pf_gdn_rmsnorm_gate_parallel, src/wzy_qsa_wmma.cuh:176-195)
__global__ void __launch_bounds__(128) pf_gdn_norm_kernel(PfGdn g) {
    __shared__ float s_red[2];
    const int h = blockIdx.x, t = blockIdx.y, c = threadIdx.x;
    const size_t i = ((size_t) t * g.hv + h) * 128 + c;
    const float o = g.o[i];
    const float ss = block_sum<2>(o * o, s_red);
    const float sc = 1.0f / sqrtf(ss * (1.0f / 128.0f) + g.eps);
    g.y[i] = f_to_bf16(o * sc * g.gamma[c] / (1.0f + __expf(-g.z[i])));
}

// ---------------------------------------------------------------------------------------------
// QSA
// ---------------------------------------------------------------------------------------------
// One wave per (row, head): q heads, kv heads (+ INT8 append), indexer q heads.  Bound by reading and writing
// the heads once (8,192 rows: 0.45 GB); with a workgroup per head and two barriers in each norm the loads of a
// head waited for the one before it (8,191 rows 265 -> 108 us, 1,300 rows 40 -> 24 us; 4.2 TB/s).
__global__ void __launch_bounds__(256) pf_qsa_prep_kernel(PfQsaPrep a, int B) {
    __shared__ float s_rot[4][128];
    const QsaDims& dm = a.dm;
    const int lane = threadIdx.x & 63, roles = dm.qh + dm.kvh + dm.ih;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = blockIdx.x * 4 + w, t = i / roles, role = i % roles;
    if (t >= B) return;                          // wave-uniform; no barrier follows
    const int pos = *a.pos + t, hd = dm.hd, kvd = dm.kvh * dm.hd;
    float y[4];
    if (role < dm.qh) {
        norm_rope_wave(a.qg + (size_t) t * dm.qh * 2 * hd + (size_t) role * 2 * hd, hd, a.q_norm, a.cos_tab, a.sin_tab, pos,
                       dm.n_rot, dm.eps, s_rot[w], y);
    } else if (role < dm.qh + dm.kvh) {
        const int j = role - dm.qh;
        const size_t at = (size_t) t * kvd + (size_t) j * hd;
        float v[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) v[g] = a.vv[at + 64 * g + lane];
        norm_rope_wave(a.kk + at, hd, a.k_norm, a.cos_tab, a.sin_tab, pos, dm.n_rot, dm.eps, s_rot[w], y);
#pragma unroll
        for (int g = 0; g < 4; ++g) qsa_kv_store_group(dm, a.kv, pos, j, g, y[g], v[g]);
    } else {
        const int h = role - dm.qh - dm.kvh;
        norm_rope_wave(a.q_idx + (size_t) t * dm.ih * dm.idim + (size_t) h * dm.idim, dm.idim, a.iq_norm, a.cos_tab,
                       a.sin_tab, pos, dm.n_rot, dm.eps, s_rot[w], y);
    }
}

// One workgroup per indexer event of the chunk [p0, p0 + B): event 0 is position 0 when the chunk
// starts the context (its key doubles as the open-block placeholder "dead"), the others are the
// positions that complete a block.  A block's cells before p0 come from the tail as it was before
// the chunk.  The last event writes the placeholder row after its block (dead, recomputed from row
// 0 when this chunk sets it).  Final state equals B single-row appends (qsa_indexer_append_multi,
// src/wzy_qsa_256k.cuh:147-209).
__global__ void __launch_bounds__(256) pf_idx_append_kernel(PfIdxAppend a, int p0, int B, int has0, int pc0,
                                                             int n_ev) {
    __shared__ float s_vals[256];
    __shared__ float s_red[4];
    const QsaDims& dm = a.dm;
    const int D = dm.idim, BL = dm.iblk, d = threadIdx.x;
    const int e = blockIdx.x;
    const bool last = e == n_ev - 1;
    auto raw = [&](int cell) { return d < D ? round_h16(a.idx_raw[(size_t) (cell - p0) * D + d]) : 0.f; };
    if (has0 && e == 0) {
        const float inc = raw(0);
        const float y = idx_block_key(dm, [&](int) { return inc; }, a.ik_norm, a.cos_tab, a.sin_tab, 0, s_vals, s_red);
        if (d < D) {
            a.ix.dead[d] = y;
            if (p0 + B - 1 < BL - 1) a.ix.pooled[d] = f_to_h16(y);     // block 0 stays open in this chunk
        }
        return;
    }
    const int p = pc0 + (e - has0) * BL, b = p / BL;
    auto cell = [&](int jj) {
        const int c = b * BL + jj;
        return c >= p0 ? raw(c) : (d < D ? a.ix.tail[jj * D + d] : 0.f);
    };
    const float y = idx_block_key(dm, cell, a.ik_norm, a.cos_tab, a.sin_tab, BL * b, s_vals, s_red);
    float dead = 0.f;
    if (last) {
        if (p0 == 0) {
            const float inc = raw(0);
            dead = idx_block_key(dm, [&](int) { return inc; }, a.ik_norm, a.cos_tab, a.sin_tab, 0, s_vals, s_red);
        } else {
            dead = d < D ? a.ix.dead[d] : 0.f;
        }
    }
    if (d < D) {
        a.ix.pooled[(size_t) b * D + d] = f_to_h16(y);
        if (last) a.ix.pooled[(size_t) (b + 1) * D + d] = f_to_h16(dead);
    }
}

// tail slot s <- the last chunk cell at a position with p % iblk == s (s < iblk - 1)
__global__ void __launch_bounds__(128) pf_idx_tail_kernel(PfIdxAppend a, int p0, int B) {
    const int D = a.dm.idim, BL = a.dm.iblk, d = threadIdx.x;
    if (d >= D) return;
    const int pe = p0 + B - 1;
    for (int s = 0; s < BL - 1; ++s) {
        const int c = pe - ((pe % BL) - s + BL) % BL;             // last position <= pe in slot s
        if (c >= p0) a.ix.tail[s * D + d] = round_h16(a.idx_raw[(size_t) (c - p0) * D + d]);
    }
}

// Indexer block scores of the chunk's rows on MFMA: score[t][b] = sum over heads h of
// relu(q_h[t] . key[b]), fp16 queries and keys with fp32 products and sums (v_mfma_f32_32x32x16_f16,
// as the reference's prefill scorer runs on WMMA).  Workgroup = 32 rows x `groups` x 256 blocks, wave w:
// blocks 64w .. 64w+63 of a group as two 32 x 32 tiles, the four heads' accumulators side by side; the queries
// are staged in LDS as fp16, each wave loads its keys' k slices straight into B fragments, one tile ahead.  With
// one group a workgroup staged 64 KB of queries for two tiles a wave and no load was in flight while a tile was
// multiplied (2,048 rows at 33-41 thousand cells 96 -> 53 us, 1,300 at 9-10 thousand 39 -> 23, the open block below included).  Only complete
// blocks of rows whose context exceeds top_k are written; the row group's first workgroup also
// scores the open block against the placeholder key (fp32, +1e9 while the block is partial), as the
// decode scorer does.  (qsa_block_scores_wmma, src/wzy_qsa_wmma.cuh:492-612)
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
constexpr int PS_ROWS = 32, PS_BLOCKS = 256;

__global__ void __launch_bounds__(256, 3) pf_score_kernel(QsaScoreArgs a, int groups) {
    __shared__ __align__(16) _Float16 sQ[4][PS_ROWS][128 + 8];
    const QsaDims& dm = a.dm;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int r0 = blockIdx.y * PS_ROWS, nrows = min(PS_ROWS, a.rows - r0);
    const int base = *a.pos + r0;
    const int B = dm.iblk, IH = dm.ih;
    const int n_kv_max = base + nrows;
    if (n_kv_max <= dm.topk) return;                 // short context: identity selection
    const int b0 = blockIdx.x * groups * PS_BLOCKS;
    const bool tail_wg = blockIdx.x == 0;
    const int b_lim = min(a.max_b, n_kv_max / B);
    if (b0 >= b_lim && !tail_wg) return;
    const float* q_idx = a.q_idx + (size_t) r0 * IH * 128;
    float* scores = a.scores + (size_t) r0 * a.max_b;

    for (int i = tid; i < 4 * PS_ROWS * 32; i += 256) {     // (head, row, 4 k) -> fp16
        const int h = i / (PS_ROWS * 32), r = (i / 32) % PS_ROWS, k4 = i % 32;
        float4 q = make_float4(0.f, 0.f, 0.f, 0.f);
        if (r < nrows && h < IH) q = *(const float4*) (q_idx + (size_t) r * IH * 128 + (size_t) h * 128 + 4 * k4);
        _Float16* d = &sQ[h][r][4 * k4];
        d[0] = (_Float16) q.x; d[1] = (_Float16) q.y; d[2] = (_Float16) q.z; d[3] = (_Float16) q.w;
    }
    __syncthreads();

    if (b0 + 64 * w < b_lim) {
        // one 32-block tile at a time: 64 accumulator registers, so several workgroups share a CU
        const int kb = (lane >> 5) * 8;
        const auto block = [&](int c) { return b0 + (c >> 1) * PS_BLOCKS + 64 * w + 32 * (c & 1) + (lane & 31); };
        const auto key = [&](int c) {                // past the end: the last row again
            return (const _Float16*) a.pooled + (size_t) min(block(c), b_lim - 1) * 128 + kb;
        };
        f16x8_t bv[8];
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) bv[ks] = *(const f16x8_t*) (key(0) + 16 * ks);
        for (int c = 0; c < 2 * groups && block(c) - (lane & 31) < b_lim; ++c) {      // wave-uniform
            const int b = block(c);
            const _Float16* kn = key(c + 1);
            f32x16_t acc[4];
#pragma unroll
            for (int h = 0; h < 4; ++h)
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[h][i] = 0.f;
#pragma unroll
            for (int ks = 0; ks < 8; ++ks) {
#pragma unroll
                for (int h = 0; h < 4; ++h) {
                    if (h >= IH) break;                  // uniform
                    const f16x8_t av = *(const f16x8_t*) &sQ[h][lane & 31][16 * ks + kb];
                    acc[h] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av, bv[ks], acc[h], 0, 0, 0);
                }
                bv[ks] = *(const f16x8_t*) (kn + 16 * ks);           // the next tile's
            }
            // acc[h][i] = q_h[row 8*(i/4) + 4*(lane/32) + i%4] . key[block b, lane%32 of the tile]; the block is
            // complete for rows with n_kv >= (b + 1) B (no division per row)
            const int t_min = max((b + 1) * B, dm.topk + 1) - base - 1;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int t = 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
                float sc = 0.f;
#pragma unroll
                for (int h = 0; h < 4; ++h)
                    if (h < IH) sc += acc[h][i] > 0.f ? acc[h][i] : 0.f;
                if (t >= t_min && t < nrows) scores[(size_t) t * a.max_b + b] = sc;
            }
        }
    }
    // open block: fp32 dot with the placeholder key (wave w handles rows w, w + 4, ...), four rows' loads at a
    // time (a load per row and head, each waited for, kept this workgroup busy after all others had ended)
    if (tail_wg) {
        constexpr int TR = 4;
        const float d0 = a.dead[lane], d1 = a.dead[lane + 64];
        const float* qi = IH > 0 ? q_idx : a.dead;   // without heads any readable row: nothing of it is used
        for (int t0 = w; t0 < nrows; t0 += 4 * TR) {
            float q[TR][4][2];
#pragma unroll
            for (int r = 0; r < TR; ++r)
#pragma unroll
                for (int h = 0; h < 4; ++h) {
                    const float* qp = qi + ((size_t) min(t0 + 4 * r, nrows - 1) * IH + max(0, min(h, IH - 1))) * 128 + lane;
                    q[r][h][0] = qp[0];
                    q[r][h][1] = qp[64];
                }
#pragma unroll
            for (int r = 0; r < TR; ++r) {
                const int t = t0 + 4 * r, n_kv = base + t + 1, nbid = n_kv / B;
                float score = 0.f;
#pragma unroll
                for (int h = 0; h < 4; ++h) {
                    const float p = wave_sum(fmaf(d1, q[r][h][1], fmaf(d0, q[r][h][0], 0.f)));
                    if (h < IH) score += p > 0.f ? p : 0.f;
                }
                if (n_kv % B != 0) score += 1e9f;
                if (lane == 0 && t < nrows && n_kv > dm.topk && nbid < a.max_b) scores[(size_t) t * a.max_b + nbid] = score;
            }
        }
    }
}

// Sparse GQA attention of one row and one KV head (grid (kvh, B), 256 threads): the group's query
// heads (up to 16, columns of a 16 x 16 fp16 MFMA tile) against the selected cells.  Each wave takes
// every fourth 32-cell chunk through a softmax of its own; the four are merged at the end.
//
// Nothing of the loop goes through LDS but the chunk's cell ids.  K and V codes are loaded straight into
// the lanes that feed them to the matrix cores, 16 bytes at a time, and dequantised there:
//   S^T = K Q^T   A = K: lane l holds cell l % 16, its 16-byte pieces at dims 64 u + 16 (l / 16); the sum
//                 over dims may run in any order, so Q^T (B, in registers) takes the same dims.
//   O^T = V^T P^T the accumulator layout of S^T (cells 4 (l / 16) + i of head l % 16) is the B layout of
//                 P^T, so the weights never leave their lane; A = V^T: lane l holds dims 16 (l % 16) + t of
//                 the same eight cells, regrouped from cells x dims to dims x cells by byte permutes.
// Codes become fp16 exactly as 1024 + (code + 128) - 1152 (a byte under the exponent of 1024), then
// code * scale is rounded to fp16 once, two at a time, as a product of fp16 numbers.
// The softmax's reference exponent is the running maximum of the wave's chunks, so the largest weight is 1
// and the weights beside it are rounded to fp16 at the top of its binades: their share of the error against
// 64 bits is 1.5e-4 at scores of spread 1 and 0.65e-4 at spread 2.  (A reference moved only past a factor of
// 2^6 rescales fewer accumulators and has 2.1e-4 and 1.4e-4; one running maximum for all cells, as in the kernel
// before this one, 1.7e-4 and 0.88e-4.  8,192 rows take the same time either way, 1,301 rows 281 us against 286.)
// K of the next chunk is loaded once this chunk's codes are converted, V likewise.  out = acc / max(l,
// 1e-20) * sigmoid(gate), bf16.
// What bounds it: the gather (528 bytes per cell, row and KV head, from the Infinity Cache where a context
// exceeds the L2) and about 480 VALU operations per 32 cells and wave for the conversions.  Against the
// kernel before it, which staged K and a transposed V through LDS with three barriers per 64 cells: 8,192
// rows over 2,048 of 33-41 thousand cells 3,260 -> 1,831 us (9.7 TB/s gathered), 1,300 rows over 2,048 of 9-10
// thousand 530 -> 325 us.
constexpr int AT_C = 32;                      // cells per wave and step
constexpr int AT_OLD = 256 + 4;               // LDS row stride of the partial outputs (floats)
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));

// bytes x0, x1 / x2, x3 of the biased codes w -> 1024 + x, minus 1152: the codes as fp16 pairs
WZY_DEV f16x2_t at_lo(uint32_t w) {
    return __builtin_bit_cast(f16x2_t, __builtin_amdgcn_perm(0x64646464u, w, 0x04010400u)) - (_Float16) 1152.0f;
}
WZY_DEV f16x2_t at_hi(uint32_t w) {
    return __builtin_bit_cast(f16x2_t, __builtin_amdgcn_perm(0x64646464u, w, 0x04030402u)) - (_Float16) 1152.0f;
}
WZY_DEV f16x8_t at_join(f16x2_t a, f16x2_t b, f16x2_t c, f16x2_t d) {
    return f16x8_t{a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y};
}
// eight K codes times their scale
WZY_DEV f16x8_t at_k8(uint32_t a, uint32_t b, f16x2_t sc) {
    a ^= 0x80808080u;
    b ^= 0x80808080u;
    return at_join(at_lo(a) * sc, at_hi(a) * sc, at_lo(b) * sc, at_hi(b) * sc);
}
// maximum / sum over lanes l, l ^ 16, l ^ 32, l ^ 48 (inline assembly as in sum32_t)
template <bool MAX>
WZY_DEV float at_rows(float v) {
    uint32_t x = __builtin_bit_cast(uint32_t, v), y = x;
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(x), "+v"(y));
    const float a = __builtin_bit_cast(float, x), b = __builtin_bit_cast(float, y);
    const float r = MAX ? fmaxf(a, b) : a + b;
    x = y = __builtin_bit_cast(uint32_t, r);
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(x), "+v"(y));
    const float c = __builtin_bit_cast(float, x), d = __builtin_bit_cast(float, y);
    return MAX ? fmaxf(c, d) : c + d;
}

// O32: byte offsets into the code planes fit 32 bits (launch_pf_attn), so a cell's address is the plane's
// base and one register, kept in LDS ready made.
template <bool O32>
__global__ void __launch_bounds__(256, 2) pf_attn_kernel(PfAttn a) {
    typedef typename std::conditional<O32, uint32_t, uint64_t>::type off_t;
    __shared__ __align__(16) float sO[4][16][AT_OLD];
    __shared__ __align__(16) off_t sOff[4][2][AT_C];     // per wave: code offsets of this chunk's cells and the next's
    __shared__ float s_m[4][16], s_l[4][16];
    const QsaDims& dm = a.dm;
    const int j = blockIdx.x, t = blockIdx.y, tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int hd = 256, kvd = dm.kvh * hd, gq = dm.qh / dm.kvh;
    const int n_kv = *a.pos + t + 1;
    const int width = min(n_kv, dm.topk);
    const int* ids = a.sel + (size_t) t * dm.topk;
    const float* qg = a.qg + (size_t) t * dm.qh * 2 * hd;
    const int l16 = lane & 15, g = lane >> 4;

    // Q^T: q[head l16][64 u + 16 g + 8 half .. +7] / 16 for every (u, half)
    f16x8_t qb[8];
#pragma unroll
    for (int uh = 0; uh < 8; ++uh) {
        const float* qp = qg + (size_t) (j * gq + min(l16, gq - 1)) * 2 * hd + 64 * (uh >> 1) + 16 * g + 8 * (uh & 1);
        const f32x4_t x = *(const f32x4_t*) qp, y = *(const f32x4_t*) (qp + 4);
        const float z = l16 < gq ? 0.0625f : 0.f;
        qb[uh] = f16x8_t{(_Float16) (x.x * z), (_Float16) (x.y * z), (_Float16) (x.z * z), (_Float16) (x.w * z),
                         (_Float16) (y.x * z), (_Float16) (y.y * z), (_Float16) (y.z * z), (_Float16) (y.w * z)};
    }
    f32x4_t acc[16];                              // O^T: dims 16 (4 g + i) + t of head l16
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    float m_ref = -1e30f, l_sum = 0.f;            // per head l16; l_sum is this lane's part

    const int nch = (width + AT_C - 1) / AT_C;    // chunks; this wave takes w, w + 4, ...
    // a cell's codes start at its offset, its scales (fp16 per 64 codes) at a 32nd of it
    const char* kb = (const char*) (a.kv.kq + (size_t) j * hd);
    const char* vb = (const char*) (a.kv.vq + (size_t) j * hd);
    const char* ksb = (const char*) (a.kv.ks + (size_t) j * 4);
    const char* vsb = (const char*) (a.kv.vs + (size_t) j * 4);
    const off_t ko = 16 * g, vo = 16 * l16, vso = 2 * (l16 >> 2);
    // cells past the selection repeat its last one: every load is unconditional
    auto read_id = [&](int c) {
        return (off_t) qsa_kv_slot(ids[max(0, min(AT_C * c + (lane & 31), width - 1))], dm) * (off_t) kvd;
    };

    i32x4_t kr[2][4];                             // K codes of cells l16, 16 + l16: pieces u = 0 .. 3
    i32x2_t ksr[2];                               // and their four scales
    i32x4_t vr[8];                                // V codes of cells 4 g + i, 16 + 4 g + i
    uint16_t vsr[8];
#define AT_LOAD_K(slot)                                                                        \
    _Pragma("unroll") for (int c_ = 0; c_ < 2; ++c_) {                                         \
        const off_t p_ = sOff[w][slot][16 * c_ + l16];                                         \
        _Pragma("unroll") for (int u_ = 0; u_ < 4; ++u_)                                       \
            kr[c_][u_] = *(const i32x4_t*) (kb + (off_t) (p_ + ko) + 64 * u_);                 \
        ksr[c_] = *(const i32x2_t*) (ksb + (off_t) (p_ >> 5));                                 \
    }
#define AT_LOAD_V(slot)                                                                        \
    _Pragma("unroll") for (int c_ = 0; c_ < 8; ++c_) {                                         \
        const off_t p_ = sOff[w][slot][16 * (c_ >> 2) + 4 * g + (c_ & 3)];                     \
        vr[c_] = *(const i32x4_t*) (vb + (off_t) (p_ + vo));                                   \
        vsr[c_] = *(const uint16_t*) (vsb + (off_t) ((p_ >> 5) + vso));                        \
    }
    off_t rid = 0;
    if (w < nch) {
        rid = read_id(w);
        if (lane < AT_C) sOff[w][0][lane] = rid;
        wave_lds_sync();
        rid = read_id(w + 4);
        AT_LOAD_K(0)
        AT_LOAD_V(0)
    }
    for (int c = w, it = 0; c < nch; c += 4, ++it) {
        const int nx = (it + 1) & 1;
        if (lane < AT_C) sOff[w][nx][lane] = rid;
        wave_lds_sync();
        rid = read_id(c + 8);
        // S^T of the chunk's two 16-cell tiles
        f32x4_t sc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int u = 0; u < 4; ++u) {
#pragma unroll
            for (int ct = 0; ct < 2; ++ct) {
                const uint32_t sw = (uint32_t) (u < 2 ? ksr[ct].x : ksr[ct].y);
                const uint32_t s2 = __builtin_amdgcn_perm(sw, sw, (u & 1) ? 0x03020302u : 0x01000100u);
                const f16x2_t s = __builtin_bit_cast(f16x2_t, s2);
                const f16x8_t k0 = at_k8((uint32_t) kr[ct][u].x, (uint32_t) kr[ct][u].y, s);
                const f16x8_t k1 = at_k8((uint32_t) kr[ct][u].z, (uint32_t) kr[ct][u].w, s);
                sc[ct] = __builtin_amdgcn_mfma_f32_16x16x32_f16(k0, qb[2 * u], sc[ct], 0, 0, 0);
                sc[ct] = __builtin_amdgcn_mfma_f32_16x16x32_f16(k1, qb[2 * u + 1], sc[ct], 0, 0, 0);
            }
        }
        AT_LOAD_K(nx)
        // softmax weights of this lane's eight cells of head l16, in units of 2^m_ref
        const int left = width - AT_C * c - 4 * g;        // cell (ct, i) is selected iff 16 ct + i < left
        float z[8], mx = -1e30f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            z[e] = sc[e >> 2][e & 3] * 1.44269504f;
            if (16 * (e >> 2) + (e & 3) < left) mx = fmaxf(mx, z[e]);
        }
        mx = at_rows<true>(mx);
        if (__any(mx > m_ref)) {
            const float m_new = fmaxf(m_ref, mx), al = __builtin_amdgcn_exp2f(m_ref - m_new);
            m_ref = m_new;
            l_sum *= al;
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[i] *= al;
        }
        f16x8_t pw;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float p = 16 * (e >> 2) + (e & 3) < left ? __builtin_amdgcn_exp2f(z[e] - m_ref) : 0.f;
            l_sum += p;
            pw[e] = (_Float16) p;
        }
        // O^T: the eight cells of four dims at a time
        f16x2_t vs2[4];
#pragma unroll
        for (int q = 0; q < 4; ++q)
            vs2[q] = f16x2_t{__builtin_bit_cast(_Float16, vsr[2 * q]), __builtin_bit_cast(_Float16, vsr[2 * q + 1])};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint32_t d01[4], d23[4];                      // per cell pair: bytes of dims 4i, 4i+1 / 4i+2, 4i+3
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t x = (uint32_t) vr[2 * q][i] ^ 0x80808080u, y = (uint32_t) vr[2 * q + 1][i] ^ 0x80808080u;
                d01[q] = __builtin_amdgcn_perm(y, x, 0x05010400u);
                d23[q] = __builtin_amdgcn_perm(y, x, 0x07030602u);
            }
            acc[4 * i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                at_join(at_lo(d01[0]) * vs2[0], at_lo(d01[1]) * vs2[1], at_lo(d01[2]) * vs2[2], at_lo(d01[3]) * vs2[3]), pw,
                acc[4 * i], 0, 0, 0);
            acc[4 * i + 1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                at_join(at_hi(d01[0]) * vs2[0], at_hi(d01[1]) * vs2[1], at_hi(d01[2]) * vs2[2], at_hi(d01[3]) * vs2[3]), pw,
                acc[4 * i + 1], 0, 0, 0);
            acc[4 * i + 2] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                at_join(at_lo(d23[0]) * vs2[0], at_lo(d23[1]) * vs2[1], at_lo(d23[2]) * vs2[2], at_lo(d23[3]) * vs2[3]), pw,
                acc[4 * i + 2], 0, 0, 0);
            acc[4 * i + 3] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                at_join(at_hi(d23[0]) * vs2[0], at_hi(d23[1]) * vs2[1], at_hi(d23[2]) * vs2[2], at_hi(d23[3]) * vs2[3]), pw,
                acc[4 * i + 3], 0, 0, 0);
        }
        AT_LOAD_V(nx)
    }
#undef AT_LOAD_K
#undef AT_LOAD_V
    // merge the waves: out[d] = sum_w 2^(m_w - m) acc_w[d] / sum_w 2^(m_w - m) l_w
    l_sum = at_rows<false>(l_sum);
    if (g == 0) {
        s_m[w][l16] = m_ref;
        s_l[w][l16] = l_sum;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q)
            *(f32x4_t*) &sO[w][l16][16 * (4 * g + i) + 4 * q] =
                f32x4_t{acc[4 * q][i], acc[4 * q + 1][i], acc[4 * q + 2][i], acc[4 * q + 3][i]};
    __syncthreads();
    for (int h = 0; h < gq; ++h) {                        // thread = dim
        const float m = fmaxf(fmaxf(s_m[0][h], s_m[1][h]), fmaxf(s_m[2][h], s_m[3][h]));
        float o = 0.f, l = 0.f;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const float f = __builtin_amdgcn_exp2f(s_m[v][h] - m);
            l = fmaf(s_l[v][h], f, l);
            o = fmaf(sO[v][h][tid], f, o);
        }
        const float gate = qg[(size_t) (j * gq + h) * 2 * hd + hd + tid];
        const float y = (o * (1.0f / fmaxf(l, 1e-20f))) / (1.0f + __expf(-gate));
        a.out[(size_t) t * dm.qh * hd + (size_t) (j * gq + h) * hd + tid] = f_to_bf16(y);
    }
}

}  // namespace

// ---------------------------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------------------------
namespace wzy {

// Q8_0 rows -> bf16 (one thread per 8 values): out = bf16(q * fp16 scale), the rounding the GEMM's
// own staging applies (q8_quarter_bf16), so a GEMM on the expanded rows computes the same values.
__global__ void __launch_bounds__(256) pf_q8_to_bf16_kernel(const int8_t* __restrict__ q, const uint16_t* __restrict__ s,
                                                            uint16_t* __restrict__ out, size_t n8) {
    const size_t i = (size_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n8) return;
    const uint2 c = *(const uint2*) (q + 8 * i);
    const float sc = h16_to_f(s[i / 4]);
    const uint4 o0 = q8_quarter_bf16(c.x, c.y, sc);
    *(uint4*) (out + 8 * i) = o0;
}

int launch_pf_gemm(const PfGemm& g0, hipStream_t st) {
    PfGemm g = g0;
    if (g.wq && g.wscratch && g.M >= PF_DEQ_MIN_M && (size_t) g.N * g.K <= g.wscratch_elems && g.K % 32 == 0) {
        // many row tiles read each weight tile: expand the Q8_0 weights to bf16 once
        const size_t n8 = (size_t) g.N * g.K / 8;
        hipLaunchKernelGGL(pf_q8_to_bf16_kernel, dim3((unsigned) ((n8 + 255) / 256)), dim3(256), 0, st, g.wq, g.ws,
                           g.wscratch, n8);
        WZY_LAUNCH_CHECK();
        g.wb = g.wscratch;
        g.wq = nullptr;
        g.ws = nullptr;
    }
    const bool um = g.um_mixed != nullptr;
    const int ksplit = max(g.ksplit, 1);
    WZY_REQUIRE(g.a && (g.wq ? g.ws != nullptr : g.wb != nullptr) && (um ? g.um_xn && g.um_xh : (g.y || g.yb)),
                "pf_gemm: null operand");
    WZY_REQUIRE(g.M >= 1 && g.N >= 1 && g.K >= GK && g.K % GK == 0, "pf_gemm: M %d N %d K %d (K a multiple of %d)",
                g.M, g.N, g.K, GK);
    WZY_REQUIRE(g.lda >= g.K && g.lda % 8 == 0 && (um || g.ldy >= g.N), "pf_gemm: bad leading dimensions");
    WZY_REQUIRE(!um || (g.um_d >= 32 && g.um_d % 32 == 0 && g.N == 4 * g.um_d && ksplit == 1),
                "pf_gemm: stream-mean epilogue needs N = 4 * n_embd (n_embd %d, a multiple of 32), no K split", g.um_d);
    WZY_REQUIRE(ksplit <= 8 && (ksplit == 1 || (g.y && (g.K / GK) % ksplit == 0)),
                "pf_gemm: K split %d needs fp32 output and %d k steps divisible by it", ksplit, g.K / GK);
    if (!um && ksplit == 1 && !g.wq && g.y && g.N <= 16 && g.K % 2048 == 0 && g.K <= 8192 && g.lda % 8 == 0) {
        const int nn = g.N <= 4 ? 4 : g.N <= 8 ? 8 : 16, kj = g.K / 2048;
        // one instantiation per (rows, k slices) whose weight slices fit 64 registers; any other
        // combination takes the MFMA kernel below (a kernel for fewer k slices would drop a K range)
        const dim3 grid((g.M + SK_RB - 1) / SK_RB);
        bool done = true;
        if (nn == 4 && kj == 4) hipLaunchKernelGGL((pf_skinny_kernel<4, 4>), grid, dim3(256), 0, st, g);
        else if (nn == 4 && kj == 3) hipLaunchKernelGGL((pf_skinny_kernel<4, 3>), grid, dim3(256), 0, st, g);
        else if (nn == 4 && kj == 2) hipLaunchKernelGGL((pf_skinny_kernel<4, 2>), grid, dim3(256), 0, st, g);
        else if (nn == 4 && kj == 1) hipLaunchKernelGGL((pf_skinny_kernel<4, 1>), grid, dim3(256), 0, st, g);
        else if (nn == 8 && kj == 2) hipLaunchKernelGGL((pf_skinny_kernel<8, 2>), grid, dim3(256), 0, st, g);
        else if (nn == 8 && kj == 1) hipLaunchKernelGGL((pf_skinny_kernel<8, 1>), grid, dim3(256), 0, st, g);
        else if (nn == 16 && kj == 1) hipLaunchKernelGGL((pf_skinny_kernel<16, 1>), grid, dim3(256), 0, st, g);
        else done = false;
        if (done) {
            WZY_LAUNCH_CHECK();
            return WZY_OK;
        }
    }
    GemmArgs ga;
    ga.g = g;
    auto tiles = [&](int t) { return (long long) ((g.M + t - 1) / t) * ((g.N + t - 1) / t) * ksplit; };
    // 64 x 64 tiles where 128 x 128 ones would leave compute units idle (fewer than 256: Q8_0 250 x 2,048 x
    // 6,144 103 -> 43 us, 1,300 x 2,048 x 2,048 43 -> 29; at 256 tiles bf16 33 us with 128, 40 with 64); from 512
    // of the latter, one LDS buffer and more workgroups a CU.
    const int t = tiles(128) < 256 ? 64 : 128;
    WZY_REQUIRE(tiles(t) < (1LL << 31), "pf_gemm: too many tiles");
    ga.mt = (g.M + t - 1) / t;
    ga.nt = (g.N + t - 1) / t;
    const int grid = (int) tiles(t);
    const bool sb = t == 128 && grid >= 512, q8 = g.wq != nullptr;
#define C_(T, U, S)                                                                                             \
    if (q8) hipLaunchKernelGGL((pf_gemm_kernel<T, U, S, true>), dim3(grid), dim3(256), 0, st, ga);             \
    else hipLaunchKernelGGL((pf_gemm_kernel<T, U, S, false>), dim3(grid), dim3(256), 0, st, ga)
    if (t == 64) {
        if (um) { C_(64, true, false); } else { C_(64, false, false); }
    } else if (sb) {
        if (um) { C_(128, true, true); } else { C_(128, false, true); }
    } else {
        if (um) { C_(128, true, false); } else { C_(128, false, false); }
    }
#undef C_
    WZY_LAUNCH_CHECK();
    return WZY_OK;
}

int launch_pf_embed(const PfEmb& e, const int* toks, float* R, int D, int HC, int B, hipStream_t st) {
    hipLaunchKernelGGL(pf_embed_kernel, dim3((D + 255) / 256, B), dim3(256), 0, st, e, toks, R, D, HC);
    WZY_LAUNCH_CHECK();
    return WZY_OK;
}

int launch_pf_hc_norm(float* R, const float* bo, const float* inj_prev, const float* norm_w, uint16_t* xn, int D,
                      int HC, float eps, int B, hipStream_t st) {
    WZY_REQUIRE(D >= 4 && D <= 4096 && D % 4 == 0, "pf_hc_norm: n_embd %d (a multiple of 4, at most 4096)", D);
    const dim3 grid(HC, B);
    switch ((D + 1023) / 1024) {
        case 1: hipLaunchKernelGGL(pf_hc_norm_kernel<1>, grid, dim3(256), 0, st, R, bo, inj_prev, norm_w, xn, D, HC, eps); break;
        case 2: hipLaunchKernelGGL(pf_hc_norm_kernel<2>, grid, dim3(256), 0, st, R, bo, inj_prev, norm_w, xn, D, HC, eps); break;
        case 3: hipLaunchKernelGGL(pf_hc_norm_kernel<3>, grid, dim3(256), 0, st, R, bo, inj_prev, norm_w, xn, D, HC, eps); break;
        default: hipLaunchKernelGGL(pf_hc_norm_kernel<4>, grid, dim3(256), 0, st, R, bo, inj_prev, norm_w, xn, D, HC, eps); break;
    }
    WZY_LAUNCH_CHECK();
    return WZY_OK;
}

int launch_pf_silu_div(const float* lo, uint16_t* loh, size_t n, int nsplit, float inv_hc, hipStream_t st) {
    WZY_REQUIRE(nsplit == 1 || nsplit == 4, "pf_silu_div: %d partial sums (1 or 4)", nsplit);
    hipLaunchKernelGGL(pf_silu_div_kernel, dim3((unsigned) ((n + 255) / 256)), dim3(256), 0, st, lo, loh, n, nsplit,
                       inv_hc);
    WZY_LAUNCH_CHECK();
    return WZY_OK;
}

int launch_pf_hc_write(float* R, const float* blk, const float* inj, int D, int HC, int B, hipStream_t st) {
    hipLaunchKernelGGL(pf_hc_write_kernel, dim3((HC * D + 255) / 256, B), dim3(256), 0, st, R, blk, inj, D, HC);
    WZY_LAUNCH_CHECK();
    return WZY_OK;
}

int launch_pf_gdn(const PfGdn& g, hipStream_t st) {
    WZY_REQUIRE(g.hk >= 1 && g.hv % g.hk == 0 && g.B >= 1, "pf_gdn: bad heads / rows");
    const int QKV = (2 * g.hk + g.hv) * 128;
    hipLaunchKernelGGL(pf_gdn_ab_kernel, dim3((g.B * g.hv + 255) / 256), dim3(256), 0, st, g);
    hipLaunchKernelGGL(pf_gdn_conv_kernel, dim3(QKV / 128, (g.B + CV_ROWS - 1) / CV_ROWS), dim3(128), 0, st, g);
    hipLaunchKernelGGL(pf_gdn_hist_kernel, dim3((QKV + 255) / 256), dim3(256), 0, st, g);
    hipLaunchKernelGGL(pf_gdn_recur_kernel, dim3(g.hv * 128 / GR_COLS), dim3(256), 0, st, g);
    hipLaunchKernelGGL(pf_gdn_norm_kernel, dim3(g.hv, g.B), dim3(128), 0, st, g);
    WZY_LAUNCH_CHECK();
    return WZY_OK;
}

int launch_pf_qsa_prep(const PfQsaPrep& a, int B, hipStream_t st) {
    WZY_TRY(qsa_check_dims(a.dm));
    const int roles = a.dm.qh + a.dm.kvh + a.dm.ih;
    hipLaunchKernelGGL(pf_qsa_prep_kernel, dim3((unsigned) (((int64_t) roles * B + 3) / 4)), dim3(256), 0, st, a, B);
    WZY_LAUNCH_CHECK();
    return WZY_OK;
}

int launch_pf_idx_append(const PfIdxAppend& a, int p0, int B, hipStream_t st) {
    const int BL = a.dm.iblk;
    WZY_REQUIRE(a.dm.idim <= 128 && BL >= 2 && p0 >= 0 && B >= 1 && p0 + B <= a.dm.ctx_max, "pf_idx_append: bad shape");
    const int has0 = p0 == 0 ? 1 : 0;
    const int pc0 = p0 + ((BL - 1 - p0 % BL) + BL) % BL;          // first position completing a block
    const int pe = p0 + B - 1;
    const int n_comp = pe >= pc0 ? (pe - pc0) / BL + 1 : 0;
    const int n_ev = has0 + n_comp;
    if (n_ev > 0)
        hipLaunchKernelGGL(pf_idx_append_kernel, dim3(n_ev), dim3(256), 0, st, a, p0, B, has0, pc0, n_ev);
    hipLaunchKernelGGL(pf_idx_tail_kernel, dim3(1), dim3(128), 0, st, a, p0, B);
    WZY_LAUNCH_CHECK();
    return WZY_OK;
}

int launch_pf_scores(const QsaScoreArgs& a0, int rows, int max_n_kv, hipStream_t st) {
    WZY_TRY(qsa_check_dims(a0.dm));
    WZY_REQUIRE(a0.dm.idim == 128 && a0.dm.ih <= 4, "pf_scores: indexer layout unsupported");
    WZY_REQUIRE(rows >= 1 && (rows + PS_ROWS - 1) / PS_ROWS <= 65535, "pf_scores: %d rows", rows);
    QsaScoreArgs a = a0;
    a.rows = rows;
    // Groups of 256 blocks per workgroup: as many as leave about two workgroups a CU.  Column 0 also takes the
    // open blocks, so there is always one.
    const int rg = (rows + PS_ROWS - 1) / PS_ROWS;
    const int bg = std::max(1, (std::min(a.max_b, max_n_kv / a.dm.iblk) + PS_BLOCKS - 1) / PS_BLOCKS);
    const int groups = (int) std::max<int64_t>(1, (int64_t) rg * bg / 512);
    hipLaunchKernelGGL(pf_score_kernel, dim3((bg + groups - 1) / groups, rg), dim3(256), 0, st, a, groups);
    WZY_LAUNCH_CHECK();
    return WZY_OK;
}

int launch_pf_attn(const PfAttn& a, int B, hipStream_t st) {
    WZY_TRY(qsa_check_dims(a.dm));
    WZY_REQUIRE(a.dm.hd == 256 && a.dm.qh / a.dm.kvh <= 16 && a.dm.window == 0, "pf_attn: head layout unsupported");
    WZY_REQUIRE(B >= 1 && B <= 65535, "pf_attn: %d rows", B);
    if ((uint64_t) a.dm.ctx_max * a.dm.kvh * a.dm.hd <= UINT32_MAX)
        hipLaunchKernelGGL(pf_attn_kernel<true>, dim3(a.dm.kvh, B), dim3(256), 0, st, a);
    else
        hipLaunchKernelGGL(pf_attn_kernel<false>, dim3(a.dm.kvh, B), dim3(256), 0, st, a);
    WZY_LAUNCH_CHECK();
    return WZY_OK;
}

}  // namespace wzy

// ---------------------------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------------------------
extern "C" int wzy_gemm_bf16(const uint16_t* a, int lda, int M, int K, const int8_t* wq, const uint16_t* ws,
                             const uint16_t* wb, int N, float* y, uint16_t* yb, int ldy, void* stream) {
    WZY_REQUIRE((y == nullptr) != (yb == nullptr), "wzy_gemm_bf16: exactly one of y / yb");
    WZY_REQUIRE((wq == nullptr) != (wb == nullptr), "wzy_gemm_bf16: exactly one of wq / wb");
    PfGemm g{};
    g.a = a; g.lda = lda; g.M = M; g.N = N; g.K = K;
    g.wq = wq; g.ws = ws; g.wb = wb; g.y = y; g.yb = yb; g.ldy = ldy;
    return launch_pf_gemm(g, (hipStream_t) stream);
}
