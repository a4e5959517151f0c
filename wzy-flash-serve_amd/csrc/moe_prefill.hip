// moe_prefill.hip -- NVFP4 mixture-of-experts block for a prefill chunk of N tokens, on MFMA.
//
// Launch sequence of wzy_moe_prefill (N tokens, E experts, top-K):
//   1. pf_cvt      x fp32 -> bf16 (round to nearest even), the A operand of every GEMM
//   2. launch_pf_gemm  router logits [N x E] = x . router^T                  (bf16 weights)
//   3. pf_route    per token, one wave: softmax top-K (the decode routing: probability desc, id asc,
//                  weights renormalised by max(sum, 2^-14)) and the shared-expert gate sg = sgate . x
//   4. pf_hist, pf_tiles, pf_scatter: entries (token, slot) grouped by expert into tiles of up to 64 or
//                  128 (LDS-histogram ranks, one reserving atomic per expert and workgroup, one scan)
//   5. pf_expert<gate|up, Q8_0>  shared expert, dense token blocks, SwiGLU -> sh_act bf16 [N x F]
//   6. pf_expert<down, Q8_0>     shared expert, dense token blocks -> comb = sigmoid(sg) * shared
//   7. pf_expert<gate|up, NVFP4> routed, one expert tile per workgroup, SwiGLU -> act bf16 [N*K x F]
//   8. pf_expert<down, NVFP4>    routed -> y fp32 [N*K x D] per entry; pf_combine: comb[t] +=
//                  sum_k w_k * y[pos(t, k)] in slot order (no float atomics)
// 5 runs in the launch of 7 and 6 in the launch of 8.
// pf_expert: 8 waves, 256 weight rows per workgroup, up to 128 A rows; weights staged through LDS in
// coalesced 64-byte pieces of a row and dequantised by each lane into its v_mfma_f32_32x32x16_bf16 B fragment
// (e2m1 x e4m3 block scale is exact in bf16, the fp32 tensor scale goes onto the accumulators;
// Q8_0 code x fp16 scale is rounded to bf16).
// reference: pf_moe_gu_wmma_kernel, pf_moe_down_wmma_kernel, the tile builder and the shared/router
// prefill GEMMs (src/wzy_prefill_tc.cuh:99-443), with fp16 replaced by bf16.
#include <type_traits>

#include "wzy_device.h"
#include "wzy_host.h"
#include "wzy_moe.h"
#include "wzy_prefill.h"
#include "wzy_route.h"

using namespace wzy;

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef float float2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

namespace {

constexpr int PF_MAX_E = 1024;
constexpr int EK = 64;             // expert GEMM: K step between barriers (four MFMA k16 slices)
constexpr int EA_LD = EK + 8;      // LDS row stride of the staged activations, bf16

struct PfTile {
    int e, off, cnt, pad;          // expert, first entry position, entries (at most the launch's tile size)
};

// Routed-expert GEMM over expert tiles.  Gate|up: A rows = x rows of the entries' tokens, output
// SwiGLU activations per entry; down: A rows = activations per entry, output fp32 per entry.
// Also the dense (shared-expert) GEMMs: tiles = consecutive blocks of `a_rows` token rows, Q8_0
// weights (gate|up: w / w2 rows, down: w rows), outputs per token row.
struct PfExpArgs {
    const uint8_t* experts;
    size_t rec, codes_off, scales_off, tail_off;
    int K;                         // reduction length: n_embd (gate|up) or n_ff (down)
    int F;                         // gate|up: first up row of the plane
    int gx;                        // column blocks per tile
    const PfTile* tiles; const int* n_tiles;   // expert tiles (null: dense blocks of dense_mt of a_rows rows)
    int a_rows, dense_mt;
    const uint16_t* a;
    const int* tok; int topk;      // gate|up: entry position -> token * K + slot
    const int8_t* w; const uint16_t* ws; const int8_t* w2; const uint16_t* ws2;   // Q8_0 weights
    uint16_t* act; float* y; int ld_out;   // outputs per entry position (dense: per token row)
    const float* sg;               // dense down: y = acc * sigmoid(sg[row])
};

WZY_DEV uint16_t f_to_bf16(float f) {                // hardware conversion, round to nearest even
    return __builtin_bit_cast(uint16_t, (__bf16) f);
}
// two of them in one conversion
WZY_DEV uint32_t pack_bf16(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(float2_t{a, b}, bf16x2_t));
}
WZY_DEV uint32_t f_bits(float f) { return __builtin_bit_cast(uint32_t, f); }

// MFMA B fragment (8 consecutive k of one weight row) from one 16-value NVFP4 sub-block: bytes
// w0 (0..3), w1 (4..7), byte i = value i (low nibble) | value i+8 (high nibble).  The lane half
// sa = 0 takes values 0..7, sa = 4 values 8..15: the nibbles are regrouped so that byte i holds
// values i and i+4 of the lane's eight, each converted pair is scaled by the e4m3 block scale (the
// product of a 2-bit and a 4-bit significand: exact in fp32 and in bf16), and the high halves are
// packed in k order.
WZY_DEV bf16x8_t fp4_frag(uint32_t w0, uint32_t w1, uint32_t sa, float sc) {
    const uint32_t d = ((w0 >> sa) & 0x0F0F0F0Fu) | (((w1 >> sa) & 0x0F0F0F0Fu) << 4);
    float2_t p[4];
    p[0] = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(d, 1.0f, 0);
    p[1] = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(d, 1.0f, 1);
    p[2] = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(d, 1.0f, 2);
    p[3] = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(d, 1.0f, 3);
    uint32_t b[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        b[i] = f_bits(p[i].x * sc);            // value i
        b[i + 4] = f_bits(p[i].y * sc);        // value i + 4
    }
    uint4 q;
    q.x = __builtin_amdgcn_perm(b[1], b[0], 0x07060302u);
    q.y = __builtin_amdgcn_perm(b[3], b[2], 0x07060302u);
    q.z = __builtin_amdgcn_perm(b[5], b[4], 0x07060302u);
    q.w = __builtin_amdgcn_perm(b[7], b[6], 0x07060302u);
    return __builtin_bit_cast(bf16x8_t, q);
}

// Two e4m3 block scales (bytes 0 and 1 of s) as fp32: the scaled fp8 -> f32 conversion with unit
// scale decodes OCP e4m3; the sign bit is ignored and code 0x7F (NaN in OCP, 480 in the unsigned
// reading) maps to 480 through the NaN-discarding min.
WZY_DEV float2_t e4m3x2(uint32_t s) {
    const float2_t v = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(s & 0x7F7Fu, 1.0f, false);
    return float2_t{fminf(v.x, 480.0f), fminf(v.y, 480.0f)};
}

constexpr int ECB = 64;            // expert GEMM: code bytes of a weight row per chunk staged through LDS
constexpr int EROWS = 256;         // weight rows per workgroup (8 waves x 32)
constexpr int ETHR = 512;          // threads per expert workgroup
enum { WF_FP4 = 0, WF_Q8 = 1 };    // weight formats of the expert GEMM

// k values of a chunk; 16-byte pieces per thread to stage a chunk's codes, and pieces per row
template <int WF> constexpr int chunk_k() { return WF == WF_FP4 ? 2 * ECB : ECB; }
constexpr int ENP = ECB * EROWS / 16 / ETHR, EPPR = ECB / 16;
static_assert(ENP == 2, "two staging pieces per thread");

struct ExpLane {                   // per-thread view of one expert tile
    const uint8_t* crow0;          // staging: code bytes of the (row, 16-byte piece) slots, chunk 0
    uint32_t crow_d;               // from the first slot's row to the second's (128 local rows on)
    const uint8_t* srow;           // staging: block scales of row tid / 2
    int lr;                        // the lane's weight row (local) = its B fragment column
    int nk, cnt, row0, col, wr, wp;   // wr, wp: staging: LDS row and byte of the first code slot
    uint32_t sa;
    float ts;
};

// MTT: entries per tile; with 64 or 128 of them two workgroups share a CU's 160 KB.  144-byte activation rows
// and code rows whose 16-byte pieces are permuted by the row (code_at) put the 16 rows that one LDS cycle
// reads on different banks.
template <int MTT>
struct ExpLds {
    uint16_t a[2][MTT][EA_LD];                       // activation rows, one K step (64) per buffer
    uint8_t b[2][EROWS][ECB];                        // weight codes, one chunk per buffer
    uint2 s[2][EROWS][2];                            // block scales per weight row, two chunks per buffer
    int row[MTT];                                    // A row of each tile entry
};

// MFMA B fragment from 8 Q8_0 codes (one k16 half) times their fp16 block scale, rounded to bf16
// (code * scale is exact in fp32; the bf16 rounding is the dense reference's dequantisation).
WZY_DEV bf16x8_t q8_frag(uint2 q, float sc) {
    uint32_t b[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t w = i < 2 ? q.x : q.y;
        const float v0 = (float) (int8_t) (w >> (16 * (i & 1))) * sc;
        const float v1 = (float) (int8_t) (w >> (16 * (i & 1) + 8)) * sc;
        b[i] = pack_bf16(v0, v1);
    }
    return __builtin_bit_cast(bf16x8_t, make_uint4(b[0], b[1], b[2], b[3]));
}

// byte `at` of code row `row` in LDS (its 16-byte piece at / 16 lies at piece (at / 16) ^ (row / 4 % 4))
WZY_DEV int code_at(int row, int at) { return at ^ ((row & 12) << 2); }

// Block scales of two chunks (a pair) of a weight row: 16 e4m3 bytes or four fp16.  Threads 2 r and 2 r + 1
// stage row r's halves: read two chunks at a time by two lanes a row, the scales cost an eighth of the cache
// lines they do with one lane a row in every chunk (gate|up of 307 tokens 257 -> 212 us).
template <int WF>
WZY_DEV uint2 get_scales(const uint8_t* row, int pair, int K) {
    const int hb = WF == WF_FP4 ? 8 : 4, half = threadIdx.x & 1;            // bytes per half = per chunk
    const uint8_t* p = row + min((2 * pair + half) * hb, K / (chunk_k<WF>() / hb) - hb);   // an odd last chunk
    if constexpr (WF == WF_FP4) return *(const uint2*) p;
    else return make_uint2(*(const uint32_t*) p, 0u);
}

// staging registers: activation pieces of one K step, codes and scales of one weight chunk
template <int NA>
struct ExpA { u32x4_t v[NA]; };
struct ExpW { u32x4_t q0, q1; };

// K loop and epilogue of one tile with NMB active 32-entry row blocks.  Loads run DEPTH steps (activations)
// and DEPTH chunks (weights) ahead, in register sets used in turn; the activations of a step are requested
// before the weights of a chunk, so that waiting for them leaves the weights in flight.
template <bool DOWN, int WF, int MTT, int NMB>
WZY_DEV void expert_tile(const PfExpArgs& a, const ExpLane c, const uint16_t* const (&ap)[MTT / 64], ExpLds<MTT>& L) {
    constexpr int SPC = chunk_k<WF>() / EK, NA = MTT / 64;          // steps per chunk, activation pieces per thread
    constexpr int DEPTH = MTT == 64 ? 2 : 1;
    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5;
    const int nkc = c.nk / SPC;                                     // weight chunks
    f32x16_t acc[NMB];
#pragma unroll
    for (int mb = 0; mb < NMB; ++mb)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[mb][i] = 0.f;
    ExpA<NA> xa[DEPTH];
    ExpW xw[DEPTH];
    // No load and no staging store of the loop is conditional: past the end the last step's and chunk's
    // values are loaded and stored again, into buffers that nothing reads any more.  (A load under a
    // condition makes the compiler wait for everything in flight wherever it waits at all.)
    auto load_a = [&](ExpA<NA>& x, int ks) {
        const size_t o = (size_t) min(ks, c.nk - 1) * EK;
#pragma unroll
        for (int i = 0; i < NA; ++i) x.v[i] = *(const u32x4_t*) (ap[i] + o);
    };
    auto load_w = [&](ExpW& x, int kc) {                            // coalesced
        kc = min(kc, nkc - 1);
        const size_t o = (size_t) kc * ECB;
        x.q0 = *(const u32x4_t*) (c.crow0 + o);
        x.q1 = *(const u32x4_t*) (c.crow0 + (o + c.crow_d));
    };
    uint2 xs;                                                       // the next pair's scales
    // step 0 and chunk 0 are in LDS; the sets hold steps / chunks 1 .. DEPTH - 1
    if constexpr (DEPTH == 2) {
        load_a(xa[1], 1);
        load_w(xw[1], 1);
    }
    // one chunk; PC = chunk parity, AP = parity of its first step
    auto chunk = [&](auto pc, auto ap, int kc) {
        constexpr int PC = decltype(pc)::value, AP = decltype(ap)::value;
        const uint2 sw = L.s[(kc >> 1) & 1][c.lr][PC];
#pragma unroll
        for (int st = 0; st < SPC; ++st) {
            const int ks = kc * SPC + st;
            const int ab = (AP + st) & 1;
            load_a(xa[DEPTH == 2 ? ab : 0], ks + DEPTH);            // set ab held step ks, stored one step ago
            if (st == 0) load_w(xw[DEPTH == 2 ? PC : 0], kc + DEPTH);
            if (st == 0 && PC == 0) xs = get_scales<WF>(c.srow, (kc >> 1) + 1, a.K);
            const uint32_t sv = st ? sw.y : sw.x;
            float sc[4];                                            // per k16 slice: its block scale
            if constexpr (WF == WF_FP4) {
                const float2_t sc01 = e4m3x2(sv), sc23 = e4m3x2(sv >> 16);
                sc[0] = sc01.x; sc[1] = sc01.y; sc[2] = sc23.x; sc[3] = sc23.y;
            } else {
                sc[0] = sc[1] = h16_to_f((uint16_t) sv);
                sc[2] = sc[3] = h16_to_f((uint16_t) (sv >> 16));
            }
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) {
                // B fragment of the slice: 8 bytes of the row, or this lane's 8 of 16 (Q8_0)
                const uint2 qq = *(const uint2*) &L.b[PC][c.lr][code_at(c.lr, WF == WF_FP4 ? st * 32 + 8 * kk : 16 * kk + 8 * h)];
                const bf16x8_t bv = WF == WF_FP4 ? fp4_frag(qq.x, qq.y, c.sa, sc[kk]) : q8_frag(qq, sc[kk]);
#pragma unroll
                for (int mb = 0; mb < NMB; ++mb) {
                    const bf16x8_t av = *(const bf16x8_t*) &L.a[ab][mb * 32 + (lane & 31)][kk * 16 + h * 8];
                    acc[mb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, bv, acc[mb], 0, 0, 0);
                }
            }
            {
                const ExpA<NA>& x = xa[DEPTH == 2 ? ab ^ 1 : 0];
#pragma unroll
                for (int i = 0; i < NA; ++i) *(u32x4_t*) &L.a[ab ^ 1][(tid >> 3) + 64 * i][(tid & 7) * 8] = x.v[i];
            }
            if (st == SPC - 1) {                                    // the next chunk into the other buffer
                const ExpW& x = xw[DEPTH == 2 ? PC ^ 1 : 0];
                *(u32x4_t*) &L.b[PC ^ 1][c.wr][c.wp] = x.q0;
                *(u32x4_t*) &L.b[PC ^ 1][c.wr + 128][c.wp] = x.q1;
                if (PC == 1) L.s[((kc >> 1) + 1) & 1][tid >> 1][tid & 1] = xs;
            }
            __syncthreads();
        }
    };
    using P0 = std::integral_constant<int, 0>;
    using P1 = std::integral_constant<int, 1>;
    using PS = std::integral_constant<int, SPC & 1>;                // parity of an odd chunk's first step
    int kc = 0;
    for (; kc + 1 < nkc; kc += 2) {
        chunk(P0{}, P0{}, kc);
        chunk(P1{}, PS{}, kc + 1);
    }
    if (kc < nkc) chunk(P0{}, P0{}, kc);

    // acc[mb][i] = C[entry mb*32 + 8*(i/4) + 4*h + i%4][column lane%32 of the wave's weight block]
    const bool gate_lane = (lane & 16) == 0;
#pragma unroll
    for (int mb = 0; mb < NMB; ++mb) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int row = mb * 32 + 8 * (i >> 2) + 4 * h + (i & 3);
            const float v = acc[mb][i] * c.ts;
            if constexpr (DOWN) {
                if (row < c.cnt) {
                    const size_t r = (size_t) (c.row0 + row);
                    a.y[r * a.ld_out + c.col] = a.sg ? v / (1.0f + __expf(-a.sg[r])) : v;
                }
            } else {
                // the matching up value from lane l ^ 16 (swizzle bit-mode: and 0x1F, xor 0x10)
                const float u = __builtin_bit_cast(float, __builtin_amdgcn_ds_swizzle((int) f_bits(v), 0x401F));
                if (gate_lane && row < c.cnt)
                    a.act[(size_t) (c.row0 + row) * a.ld_out + c.col] =
                        f_to_bf16(v * __builtin_amdgcn_rcpf(1.0f + __expf(-v)) * u);
            }
        }
    }
}

// Routed-expert GEMM.  Workgroup = one expert tile (up to MTT entries) x 256 weight rows, 8 waves; wave
// w owns one 32-row weight block (gate|up: 16 gate rows j0+16w.. in columns 0..15 and the matching
// 16 up rows in columns 16..31, paired for SwiGLU across lanes l, l^16; down: rows n0+32w .. +31)
// for all active 32-entry row blocks of the tile (the count selects a specialised loop), so each
// dequantised B fragment feeds up to MTT / 32 MFMAs.  Weight codes move in chunks of 64 bytes a row (128 k
// values of NVFP4, 64 of Q8_0): read as 16-byte pieces by adjacent threads (whole 64-byte segments), one
// chunk ahead, into LDS; each lane then takes its row's bytes per k16 slice from LDS and dequantises them
// into its MFMA B fragment.  The activation rows of the tile are staged in LDS one 64-k step ahead and
// shared by the eight waves.  Workgroups are numbered so that one XCD takes the column blocks of a tile
// back to back, and pairs of consecutive tiles (an expert's tiles share its weights).  The tensor scale is
// applied to the fp32 accumulators.  WF_Q8 with a null tile list runs the dense shared-expert
// GEMMs over consecutive blocks of token rows.  An entry's sums do not depend on its tile or on MTT.
template <bool DOWN, int WF, int MTT>
WZY_DEV void expert_block(const PfExpArgs& a, int bx, ExpLds<MTT>& L) {
    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int jx = bx >> 3, u = jx / a.gx, nb = jx % a.gx;
    const int ti = (u >> 1) * 16 + (bx & 7) * 2 + (u & 1);
    const bool dense = WF == WF_Q8;
    if (ti >= (dense ? (a.a_rows + a.dense_mt - 1) / a.dense_mt : *a.n_tiles)) return;   // workgroup-uniform
    ExpLane c;
    int e = 0;
    if (dense) {
        c.row0 = ti * a.dense_mt;
        c.cnt = min(a.dense_mt, a.a_rows - c.row0);
    } else {
        const PfTile t = a.tiles[ti];
        c.cnt = t.cnt;
        c.row0 = t.off;
        e = t.e;
    }
    if (tid < MTT)
        L.row[tid] = tid < c.cnt ? ((DOWN || dense) ? c.row0 + tid : a.tok[c.row0 + tid] / a.topk) : 0;
    const uint8_t* rec = a.experts + (size_t) e * a.rec;
    // local weight row lr = 32w + column -> weight row: gate|up: columns 0..15 gate rows
    // j0+16w+col, columns 16..31 up rows (plane row F+j0+16w+col-16, or the w2 matrix); down: n0 + lr
    auto wrow = [&](int lr, bool& up) {
        const int wl = lr >> 5, cl = lr & 31;
        up = !DOWN && cl >= 16;
        return DOWN ? nb * EROWS + lr : nb * 128 + wl * 16 + (cl & 15);
    };
    auto code_row = [&](int lr) -> const uint8_t* {
        bool up;
        const int r = wrow(lr, up);
        if constexpr (WF == WF_FP4) return rec + a.codes_off + (size_t) (up ? a.F + r : r) * (a.K / 2);
        else return (const uint8_t*) ((up ? a.w2 : a.w) + (size_t) r * a.K);
    };
    auto scale_row = [&](int lr) -> const uint8_t* {
        bool up;
        const int r = wrow(lr, up);
        if constexpr (WF == WF_FP4) return rec + a.scales_off + (size_t) (up ? a.F + r : r) * (a.K / 16);
        else return (const uint8_t*) ((up ? a.ws2 : a.ws) + (size_t) r * (a.K / 32));
    };
    c.lr = w * 32 + (lane & 31);
    c.col = DOWN ? nb * EROWS + c.lr : nb * 128 + w * 16 + (lane & 15);
    if constexpr (WF == WF_FP4) {
        const float* tail = (const float*) (rec + a.tail_off);
        c.ts = DOWN ? tail[2] : ((lane & 16) ? tail[1] : tail[0]);
    } else {
        c.ts = 1.0f;
    }
    const int pp = (tid % EPPR) * 16;
    c.crow0 = code_row(tid / EPPR) + pp;
    // 128 local rows are four wave blocks: 128 down rows, or 64 rows of the same matrix of gate|up
    c.crow_d = (DOWN ? 128u : 64u) * (uint32_t) (WF == WF_FP4 ? a.K / 2 : a.K);
    c.srow = scale_row(tid >> 1);
    c.nk = a.K / EK;
    c.sa = 4u * h;
    // weight chunk 0
    c.wr = tid / EPPR;
    c.wp = code_at(c.wr, pp);                                       // row wr + 128 has the same permutation
    *(u32x4_t*) &L.b[0][c.wr][c.wp] = *(const u32x4_t*) c.crow0;
    *(u32x4_t*) &L.b[0][c.wr + 128][c.wp] = *(const u32x4_t*) (c.crow0 + c.crow_d);
    L.s[0][tid >> 1][tid & 1] = get_scales<WF>(c.srow, 0, a.K);
    __syncthreads();
    // activation staging: eight lanes read a row's 128 bytes of a step; thread -> rows tid / 8 + 64 i.  Slots
    // past the tile's entries stage row 0 of the operand: their products are never stored.
    constexpr int NA = MTT / 64;
    const uint16_t* ap[NA];
#pragma unroll
    for (int i = 0; i < NA; ++i) {
        const int sr = (tid >> 3) + 64 * i;
        ap[i] = a.a + (size_t) L.row[sr] * a.K + (tid & 7) * 8;
        *(u32x4_t*) &L.a[0][sr][(tid & 7) * 8] = *(const u32x4_t*) ap[i];
    }
    __syncthreads();
    const int nmb = (c.cnt + 31) >> 5;                              // workgroup-uniform
    if constexpr (MTT == 64) {
        if (nmb == 1) expert_tile<DOWN, WF, MTT, 1>(a, c, ap, L);
        else expert_tile<DOWN, WF, MTT, 2>(a, c, ap, L);
    } else {
        switch (nmb) {
            case 1: expert_tile<DOWN, WF, MTT, 1>(a, c, ap, L); break;
            case 2: expert_tile<DOWN, WF, MTT, 2>(a, c, ap, L); break;
            case 3: expert_tile<DOWN, WF, MTT, 3>(a, c, ap, L); break;
            default: expert_tile<DOWN, WF, MTT, 4>(a, c, ap, L); break;
        }
    }
}

// Routed tiles `r`, or dense blocks `d` of the shared expert, or both in one launch (the first nd
// workgroups take the dense blocks): a short chunk's few dense blocks then run beside the routed ones.
template <bool DOWN, int MTT>
__global__ void __launch_bounds__(ETHR, 4) pf_expert_kernel(PfExpArgs r, PfExpArgs d, int nd) {
    __shared__ __align__(16) ExpLds<MTT> L;
    if ((int) blockIdx.x < nd) expert_block<DOWN, WF_Q8, MTT>(d, blockIdx.x, L);
    else expert_block<DOWN, WF_FP4, MTT>(r, blockIdx.x - nd, L);
}

// x fp32 -> bf16; workgroup 0 also clears the per-expert entry cursors
__global__ void __launch_bounds__(256) pf_cvt_kernel(const float* __restrict__ x, uint16_t* __restrict__ xb, size_t n,
                                                     int* __restrict__ cursor, int E) {
    if (blockIdx.x == 0)
        for (int i = threadIdx.x; i < E; i += 256) cursor[i] = 0;
    const size_t i = ((size_t) blockIdx.x * 256 + threadIdx.x) * 4;
    if (i >= n) return;
    const float4 v = *(const float4*) (x + i);
    *(uint2*) (xb + i) = make_uint2(pack_bf16(v.x, v.y), pack_bf16(v.z, v.w));
}

// one wave per token: routing of its logits row and the shared-expert gate
template <int RV>
__global__ void __launch_bounds__(256) pf_route_kernel(const float* __restrict__ logits, const uint16_t* __restrict__ xb,
                                                       const uint16_t* __restrict__ sgate, int N, int E, int K, int D,
                                                       int* __restrict__ ids, float* __restrict__ wts,
                                                       float* __restrict__ sg) {
    __shared__ uint64_t cand[4][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int t = blockIdx.x * 4 + w;
    if (t >= N) return;                                          // wave-uniform
    float p[RV];
#pragma unroll
    for (int i = 0; i < RV; ++i) {
        const int idx = lane + 64 * i;
        const float v = logits[(size_t) t * E + min(idx, E - 1)];
        p[i] = idx < E ? v : -INFINITY;
    }
    float s = 0.f;
    // D a multiple of 256: whole 16-byte pieces; the caller's gate row may start at any bf16
    typedef u32x4_t u32x4_any_t __attribute__((aligned(2)));
    for (int d = lane * 8; d < D; d += 512) {
        const u32x4_t ga = *(const u32x4_any_t*) (sgate + d), xa = *(const u32x4_t*) (xb + (size_t) t * D + d);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            s = fmaf(bf16_lo(ga[i]), bf16_lo(xa[i]), s);
            s = fmaf(bf16_hi(ga[i]), bf16_hi(xa[i]), s);
        }
    }
    s = wave_sum(s);
    if (lane == 0) sg[t] = s;
    int my_id;
    float my_w, wsum;
    route_row<RV>(p, E, K, my_id, my_w, wsum, cand[w]);
    const float sc = fmaxf(wsum, 6.103515625e-05f);
    if (lane < K) {
        ids[(size_t) t * K + lane] = my_id;
        wts[(size_t) t * K + lane] = my_w / sc;
    }
}

constexpr int PF_HCHUNK = 1024;    // entries per histogram workgroup

// entries [g*1024, (g+1)*1024): each entry's rank among the entries of its expert in this workgroup
// (LDS counters), then one atomic add per expert reserves the workgroup's run in the expert's list
// (cursor ends as the expert's entry count)
__global__ void __launch_bounds__(256) pf_hist_kernel(const int* __restrict__ ids, int n_ent, int E,
                                                      int* __restrict__ cursor, int* __restrict__ wg_base,
                                                      int* __restrict__ rank) {
    __shared__ int h[PF_MAX_E];
    const int tid = threadIdx.x, g = blockIdx.x;
    for (int i = tid; i < E; i += 256) h[i] = 0;
    __syncthreads();
    const int i0 = g * PF_HCHUNK, i1 = min(n_ent, i0 + PF_HCHUNK);
    for (int i = i0 + tid; i < i1; i += 256) rank[i] = atomicAdd(&h[ids[i]], 1);
    __syncthreads();
    for (int i = tid; i < E; i += 256) {
        const int c = h[i];
        wg_base[(size_t) g * E + i] = c ? atomicAdd(&cursor[i], c) : 0;
    }
}

// one workgroup: exclusive scans of the entry counts and of the tiles per expert -> each expert's
// first entry position and its tiles of at most mt entries (as many as needed, of equal size rounded up to
// whole 32-entry row blocks)
__global__ void __launch_bounds__(1024) pf_tiles_kernel(const int* __restrict__ cnt, int E, int mt,
                                                        int* __restrict__ exp_off, PfTile* __restrict__ tiles,
                                                        int* __restrict__ n_tiles) {
    __shared__ uint64_t s_w[16];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int c = tid < E ? cnt[tid] : 0;
    const int nt = (c + mt - 1) / mt;
    const uint64_t v = ((uint64_t) c << 24) | (uint64_t) nt;       // both sums in one scan
    uint64_t s = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint64_t o = __shfl_up(s, d);
        if (lane >= d) s += o;
    }
    if (lane == 63) s_w[w] = s;
    __syncthreads();
    uint64_t base = 0;
    for (int i = 0; i < w; ++i) base += s_w[i];
    const uint64_t ex = base + s - v;
    const int off = (int) (ex >> 24), toff = (int) (ex & 0xFFFFFFu);
    if (tid < E) {
        exp_off[tid] = off;
        const int per = nt > 0 ? ((c + nt - 1) / nt + 31) & ~31 : 0;     // <= mt, (nt - 1) * per < c
        for (int q = 0; q < nt; ++q) tiles[toff + q] = PfTile{tid, off + q * per, min(per, c - q * per), 0};
    }
    if (tid == 1023) *n_tiles = (int) ((base + s) & 0xFFFFFFu);
}

// entry i = (token i / K, slot i % K) <-> its position in the expert-sorted list
__global__ void __launch_bounds__(256) pf_scatter_kernel(const int* __restrict__ ids, const int* __restrict__ rank,
                                                         const int* __restrict__ wg_base,
                                                         const int* __restrict__ exp_off, int n_ent, int K, int E,
                                                         int* __restrict__ ent_idx, int* __restrict__ ent_pos) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n_ent) return;
    const int e = ids[i];
    const int pos = exp_off[e] + wg_base[(size_t) (i / PF_HCHUNK) * E + e] + rank[i];
    ent_idx[pos] = i;
    ent_pos[i] = pos;
}

// comb[t] += sum_k w_k * y[pos(t, k)] in slot order (comb holds the gated shared expert). A pass issues the
// row loads of KU slots together; EXACT means K is a multiple of KU, so no slot load is predicated.
template <int KU, bool EXACT>
__global__ void __launch_bounds__(256) pf_combine_kernel(const float* __restrict__ y, const int* __restrict__ ent_pos,
                                                         const float* __restrict__ wts, int K, int D,
                                                         float* __restrict__ comb) {
    const int t = blockIdx.y;
    const int d = (blockIdx.x * 256 + threadIdx.x) * 4;
    if (d >= D) return;
    float4 acc = *(const float4*) (comb + (size_t) t * D + d);
    const int* pt = ent_pos + (size_t) t * K;
    const float* wt = wts + (size_t) t * K;
    for (int k0 = 0; k0 < K; k0 += KU) {
        const int n = EXACT ? KU : min(KU, K - k0);   // uniform over the workgroup
        float4 v[KU];
        float wk[KU];
#pragma unroll
        for (int j = 0; j < KU; ++j) {
            if (EXACT || j < n) {
                wk[j] = wt[k0 + j];
                v[j] = *(const float4*) (y + (size_t) pt[k0 + j] * D + d);
            } else {
                wk[j] = 0.f;
                v[j] = make_float4(0.f, 0.f, 0.f, 0.f);
            }
        }
#pragma unroll
        for (int j = 0; j < KU; ++j) {
            if (EXACT || j < n) {
                acc.x = fmaf(wk[j], v[j].x, acc.x);
                acc.y = fmaf(wk[j], v[j].y, acc.y);
                acc.z = fmaf(wk[j], v[j].z, acc.z);
                acc.w = fmaf(wk[j], v[j].w, acc.w);
            }
        }
    }
    *(float4*) (comb + (size_t) t * D + d) = acc;
}

struct PfWs {
    uint16_t* xb; float* logits; float* sg; int* ids; float* wts;
    int* cursor; int* exp_off; int* wg_base; int* rank; int* ent_idx; int* ent_pos; PfTile* tiles; int* n_tiles;
    uint16_t* act; uint16_t* sh_act; float* y;
    int mt, max_tiles, n_wg;
};

// Entries per expert tile.  Both sizes put two workgroups on a CU, so that one computes while the other waits
// for a K step (one workgroup a CU with 256-entry tiles: 307 tokens 324 + 179 us gate|up + down, now 212 +
// 116; 8,192 tokens 490 + 533, now 483 + 512).  64-entry tiles stage half the rows and load two steps ahead;
// near 60 entries an expert too many experts need two of them.  Whole block with 64 against 128: 512 experts
// top-10, n_embd 2,048, 50 entries 506 and 515 us, 57.5 548 and 549, 62.5 610 and 563; n_embd 2,560, n_ff 640, 50
// entries 741 and 769, 57.5 821 and 807, 62.5 890 and 834; 128 experts top-8, 56 entries 175 and 182, 64 195 and
// 195.  (64 experts of n_embd 512 leave the chip idle either way: 75 entries 57 and 66.)  The 128-entry kernel
// fills its 128 registers; its loops over four row blocks reload one register of routed gate|up every two chunks
// and two of the shared down from scratch, beside 64 and 32 MFMAs.
int pf_tile_entries(size_t n_ent, int E) { return n_ent <= (size_t) 60 * E ? 64 : 128; }

PfWs pf_ws_carve(void* base, size_t cap, int D, int F, int E, int K, int N, size_t* need) {
    Arena a(base, cap);
    PfWs w;
    const size_t n_ent = (size_t) N * K;
    w.mt = pf_tile_entries(n_ent, E);
    w.max_tiles = (int) (n_ent / w.mt + E);
    w.xb = a.take<uint16_t>((size_t) N * D);
    w.logits = a.take<float>((size_t) N * E);
    w.sg = a.take<float>(N);
    w.ids = a.take<int>(n_ent);
    w.wts = a.take<float>(n_ent);
    w.n_wg = (int) ((n_ent + PF_HCHUNK - 1) / PF_HCHUNK);
    w.cursor = a.take<int>(E);
    w.exp_off = a.take<int>(E);
    w.wg_base = a.take<int>((size_t) w.n_wg * E);
    w.rank = a.take<int>(n_ent);
    w.ent_idx = a.take<int>(n_ent);
    w.ent_pos = a.take<int>(n_ent);
    w.tiles = a.take<PfTile>(w.max_tiles);
    w.n_tiles = a.take<int>(1);
    w.act = a.take<uint16_t>(n_ent * F);
    w.sh_act = a.take<uint16_t>((size_t) N * F);
    w.y = a.take<float>(n_ent * D);
    if (need) *need = a.off;
    return w;
}

// workgroups of `tiles` tiles x gx column blocks (whole rounds of 8 XCDs x 2 tiles)
unsigned expert_grid(int tiles, int gx) { return (unsigned) (gx * ((tiles + 15) / 16) * 16); }

// the routed tiles (max_tiles > 0), the dense blocks (d.a_rows > 0), or both in one launch
template <bool DOWN>
void launch_expert(int mt, const PfExpArgs& r, int max_tiles, const PfExpArgs& d, hipStream_t st) {
    const unsigned nd = d.a_rows > 0 ? expert_grid((d.a_rows + d.dense_mt - 1) / d.dense_mt, d.gx) : 0;
    const unsigned n = nd + (max_tiles > 0 ? expert_grid(max_tiles, r.gx) : 0);
    if (mt == 64) hipLaunchKernelGGL((pf_expert_kernel<DOWN, 64>), dim3(n), dim3(ETHR), 0, st, r, d, (int) nd);
    else hipLaunchKernelGGL((pf_expert_kernel<DOWN, 128>), dim3(n), dim3(ETHR), 0, st, r, d, (int) nd);
}

}  // namespace

// ---------------------------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------------------------
extern "C" size_t wzy_moe_prefill_workspace_bytes(int n_embd, int n_ff, int n_exp, int top_k, int n_tok) {
    size_t need = 0;
    pf_ws_carve(nullptr, 0, n_embd, n_ff, n_exp, top_k, n_tok, &need);
    return need + 256;
}

namespace {

constexpr int PF_N_STAGES = 8;     // timing groups of pf_enqueue
int pf_check(const wzy_moe_weights* w, int N) {
    WZY_REQUIRE(w, "wzy_moe_prefill: null weights");
    WZY_REQUIRE(w->router && w->sgate && w->experts && w->sh_gate_q && w->sh_gate_s && w->sh_up_q && w->sh_up_s &&
                    w->sh_down_q && w->sh_down_s,
                "wzy_moe_prefill: null weight pointer");
    const int D = w->n_embd, F = w->n_ff, E = w->n_exp, K = w->top_k;
    WZY_REQUIRE(N >= 1 && (int64_t) N * K <= (1 << 26), "wzy_moe_prefill: n_tok must be in [1, 2^26 / top_k]");
    WZY_REQUIRE(D % 256 == 0 && D >= 256 && F % 128 == 0 && F >= 128,
                "wzy_moe_prefill: n_embd must be a multiple of 256 and n_ff a multiple of 128");
    WZY_REQUIRE(E >= 1 && E <= PF_MAX_E && E % 64 == 0, "wzy_moe_prefill: n_exp must be a multiple of 64 up to %d",
                PF_MAX_E);
    WZY_REQUIRE(K >= 1 && K <= MOE_MAX_K && K <= E, "wzy_moe_prefill: top_k must be in [1, %d]", MOE_MAX_K);
    WZY_REQUIRE((int64_t) (E / 64) * ((N + 63) / 64) * 256 <= INT32_MAX && (int64_t) N * D <= INT32_MAX,
                "wzy_moe_prefill: n_tok x n_embd exceeds the launch grids");
    return WZY_OK;
}

// The launch sequence; with `ev`, event i is recorded before launch group i and event PF_N_STAGES
// after the last one.  The shared expert's dense blocks run in the launches of the routed tiles: beside them
// they cost less than in launches of their own at every length and shape measured (512 experts top-10, n_embd
// 2,048, apart -> together: 2,048 tokens 480 -> 455 us, 8,192 1,143 -> 1,128, 25,600 3,117 -> 3,057; n_embd 2,560
// 8,192 1,680 -> 1,646; 64 experts top-4, n_embd 512, 2,048 tokens 98 -> 70).  Only with `ev` they are launched
// apart, so that each group is timed by itself; the results are the same bits.
int pf_enqueue(const wzy_moe_weights* w, const float* x, int N, float* comb, const PfWs& ws, hipStream_t st,
                hipEvent_t* ev) {
    const int D = w->n_embd, F = w->n_ff, E = w->n_exp, K = w->top_k;
    const int n_ent = N * K;
    const MoeOffsets o = moe_offsets(D, F);
    auto mark = [&](int i) {
        if (ev) (void) hipEventRecord(ev[i], st);
    };
    const size_t nx = (size_t) N * D;
    mark(0);
    hipLaunchKernelGGL(pf_cvt_kernel, dim3((unsigned) ((nx / 4 + 255) / 256)), dim3(256), 0, st, x, ws.xb, nx,
                       ws.cursor, E);
    mark(1);
    {   // router logits, on the dense projections' kernel
        PfGemm g{};
        g.a = ws.xb; g.lda = D; g.M = N; g.N = E; g.K = D; g.wb = w->router; g.y = ws.logits; g.ldy = E;
        WZY_TRY(launch_pf_gemm(g, st));
    }
    mark(2);
    if (E <= 512)
        hipLaunchKernelGGL((pf_route_kernel<8>), dim3((N + 3) / 4), dim3(256), 0, st, ws.logits, ws.xb, w->sgate, N, E, K,
                           D, ws.ids, ws.wts, ws.sg);
    else
        hipLaunchKernelGGL((pf_route_kernel<16>), dim3((N + 3) / 4), dim3(256), 0, st, ws.logits, ws.xb, w->sgate, N, E, K,
                           D, ws.ids, ws.wts, ws.sg);
    mark(3);
    hipLaunchKernelGGL(pf_hist_kernel, dim3((unsigned) ws.n_wg), dim3(256), 0, st, ws.ids, n_ent, E, ws.cursor,
                       ws.wg_base, ws.rank);
    hipLaunchKernelGGL(pf_tiles_kernel, dim3(1), dim3(1024), 0, st, ws.cursor, E, ws.mt, ws.exp_off, ws.tiles, ws.n_tiles);
    hipLaunchKernelGGL(pf_scatter_kernel, dim3((unsigned) ((n_ent + 255) / 256)), dim3(256), 0, st, ws.ids, ws.rank,
                       ws.wg_base, ws.exp_off, n_ent, K, E, ws.ent_idx, ws.ent_pos);
    // shared expert (dense Q8_0 blocks): gate|up + SwiGLU, then down -> comb = sigmoid(sg) * shared; routed
    // experts: gate|up + SwiGLU per tile, down per tile, then the per-token weighted sum
    PfExpArgs sgu{}, sdn{}, rgu{}, rdn{};
    sgu.experts = w->experts; sgu.K = D; sgu.F = F; sgu.gx = F / 128;
    sgu.a_rows = N; sgu.dense_mt = ws.mt; sgu.a = ws.xb;
    sgu.w = (const int8_t*) w->sh_gate_q; sgu.ws = (const uint16_t*) w->sh_gate_s;
    sgu.w2 = (const int8_t*) w->sh_up_q; sgu.ws2 = (const uint16_t*) w->sh_up_s;
    sgu.act = ws.sh_act; sgu.ld_out = F;
    sdn.experts = w->experts; sdn.K = F; sdn.gx = D / EROWS;
    sdn.a_rows = N; sdn.dense_mt = ws.mt; sdn.a = ws.sh_act;
    sdn.w = (const int8_t*) w->sh_down_q; sdn.ws = (const uint16_t*) w->sh_down_s;
    sdn.y = comb; sdn.ld_out = D; sdn.sg = ws.sg;
    rgu.experts = w->experts; rgu.rec = o.rec; rgu.codes_off = o.gu_codes; rgu.scales_off = o.gu_scales;
    rgu.tail_off = o.tail; rgu.K = D; rgu.F = F; rgu.gx = F / 128;
    rgu.tiles = ws.tiles; rgu.n_tiles = ws.n_tiles;
    rgu.a = ws.xb; rgu.tok = ws.ent_idx; rgu.topk = K;
    rgu.act = ws.act; rgu.ld_out = F;
    rdn.experts = w->experts; rdn.rec = o.rec; rdn.codes_off = o.dn_codes; rdn.scales_off = o.dn_scales;
    rdn.tail_off = o.tail; rdn.K = F; rdn.F = 0; rdn.gx = D / EROWS;
    rdn.tiles = ws.tiles; rdn.n_tiles = ws.n_tiles;
    rdn.a = ws.act; rdn.tok = nullptr; rdn.topk = K;
    rdn.y = ws.y; rdn.ld_out = D;
    const bool apart = ev != nullptr;
    const PfExpArgs none{};
    mark(4);
    if (apart) launch_expert<false>(ws.mt, none, 0, sgu, st);
    mark(5);
    if (apart) launch_expert<true>(ws.mt, none, 0, sdn, st);
    mark(6);
    launch_expert<false>(ws.mt, rgu, ws.max_tiles, apart ? none : sgu, st);
    mark(7);
    {
        launch_expert<true>(ws.mt, rdn, ws.max_tiles, apart ? none : sdn, st);
        const dim3 cg((unsigned) ((D / 4 + 255) / 256), (unsigned) N);
        if (K == 10)
            hipLaunchKernelGGL((pf_combine_kernel<10, true>), cg, dim3(256), 0, st, ws.y, ws.ent_pos, ws.wts, K, D, comb);
        else if (K % 8 == 0)
            hipLaunchKernelGGL((pf_combine_kernel<8, true>), cg, dim3(256), 0, st, ws.y, ws.ent_pos, ws.wts, K, D, comb);
        else
            hipLaunchKernelGGL((pf_combine_kernel<8, false>), cg, dim3(256), 0, st, ws.y, ws.ent_pos, ws.wts, K, D, comb);
    }
    mark(8);
    return WZY_OK;
}

PfWs pf_ws_for(const wzy_moe_weights* w, int N, void* workspace, size_t workspace_bytes) {
    char* base = (char*) workspace + (256 - (uintptr_t) workspace % 256) % 256;
    return pf_ws_carve(base, workspace_bytes - 256, w->n_embd, w->n_ff, w->n_exp, w->top_k, N, nullptr);
}

}  // namespace

extern "C" int wzy_moe_prefill(const wzy_moe_weights* w, const float* x, int n_tok, float* comb, int* ids, float* wts,
                               void* workspace, size_t workspace_bytes, void* stream) {
    WZY_REQUIRE(x && comb && workspace, "wzy_moe_prefill: null pointer");
    WZY_TRY(pf_check(w, n_tok));
    const int N = n_tok, K = w->top_k;
    WZY_REQUIRE(workspace_bytes >= wzy_moe_prefill_workspace_bytes(w->n_embd, w->n_ff, w->n_exp, K, N),
                "wzy_moe_prefill: workspace too small");
    hipStream_t st = as_stream(stream);
    const PfWs ws = pf_ws_for(w, N, workspace, workspace_bytes);
    WZY_TRY(pf_enqueue(w, x, N, comb, ws, st, nullptr));
    if (ids) WZY_HIP_TRY(hipMemcpyAsync(ids, ws.ids, (size_t) N * K * sizeof(int), hipMemcpyDeviceToDevice, st));
    if (wts) WZY_HIP_TRY(hipMemcpyAsync(wts, ws.wts, (size_t) N * K * sizeof(float), hipMemcpyDeviceToDevice, st));
    WZY_LAUNCH_CHECK();
    return WZY_OK;
}

extern "C" int wzy_moe_prefill_time(const wzy_moe_weights* w, const float* x, int n_tok, float* comb, void* workspace,
                                    size_t workspace_bytes, int iters, float* us_stages, void* stream) {
    WZY_REQUIRE(x && comb && workspace && us_stages && iters >= 1, "wzy_moe_prefill_time: bad arguments");
    WZY_TRY(pf_check(w, n_tok));
    WZY_REQUIRE(workspace_bytes >= wzy_moe_prefill_workspace_bytes(w->n_embd, w->n_ff, w->n_exp, w->top_k, n_tok),
                "wzy_moe_prefill_time: workspace too small");
    hipStream_t st = as_stream(stream);
    const PfWs ws = pf_ws_for(w, n_tok, workspace, workspace_bytes);
    hipEvent_t ev[PF_N_STAGES + 1];
    for (int i = 0; i <= PF_N_STAGES; ++i) WZY_HIP_TRY(hipEventCreate(&ev[i]));
    double acc[PF_N_STAGES] = {};
    int rc = WZY_OK;
    rc = pf_enqueue(w, x, n_tok, comb, ws, st, nullptr);            // warm-up
    for (int it = 0; it < iters && rc == WZY_OK; ++it) {
        rc = pf_enqueue(w, x, n_tok, comb, ws, st, ev);
        if (rc != WZY_OK) break;
        if (hipEventSynchronize(ev[PF_N_STAGES]) != hipSuccess) { rc = WZY_EHIP; break; }
        for (int i = 0; i < PF_N_STAGES; ++i) {
            float ms = 0.f;
            if (hipEventElapsedTime(&ms, ev[i], ev[i + 1]) != hipSuccess) { rc = WZY_EHIP; break; }
            acc[i] += ms;
        }
    }
    for (int i = 0; i <= PF_N_STAGES; ++i) (void) hipEventDestroy(ev[i]);
    if (rc != WZY_OK) {
        set_error("wzy_moe_prefill_time: event timing failed");
        return rc;
    }
    for (int i = 0; i < PF_N_STAGES; ++i) us_stages[i] = (float) (1000.0 * acc[i] / iters);
    WZY_LAUNCH_CHECK();
    return WZY_OK;
}
