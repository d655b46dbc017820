// Tree-verify / draft decode attention over a bf16 KV cache, split along the context (flash decoding)
// with bf16 MFMA on gfx950, then a wide merge of the chunk partials.
//
// Reference semantics (comfy-mono-decode-xpu): csrc/attn_dpas.sycl:269-342 (contract: rows of one kv
// head attend the committed prefix [0, L) of the cache and, for tree verify, the tree rows their mask
// admits from xk / xv; the softmax is scaled by 1/sqrt(D); P is rounded to bf16 for the P.V product,
// partials merge in fp32; a row with no admitted token writes 0). Tolerance-level parity (fp64 bound),
// as the reference's own kernel is not bit-identical to the chain it replaces.
//
// Query rows of kv head kh: r = (h % groups) * S + s for the heads h of that kv head, 16 rows per
// row tile (rt). Per 32-token step of a query row tile:
//   S^T = K Q^T   v_mfma_f32_16x16x32_bf16, A = 16 K rows (tokens) x 32 dims, B = Q^T held in
//                 registers; the accumulator gives each lane 4 tokens of one query row (lane % 16), so
//                 the online softmax state of a row lives in its lanes;
//   O^T += V^T P^T   A = V^T, its 8 k-slots per lane in the token order the S^T accumulators hold,
//                 B = bf16(P^T) straight from the S^T registers -- no shuffle of P.
// Each work-group stores a chunk partial (m, l, O in fp32); attn_merge_kernel (one work-group of 256 per
// query row) combines the chunks and the tree-row partial and writes bf16. The context split is recomputed
// on the device from seqlen in both launches, so a captured graph replays for any context length.
//
// One work-group per (kv head, chunk) over all of the kv head's row tiles, K/V read once from HBM into an LDS ring (see
// the layout note at stage_k). Head_dim 256 (4 kv heads, 8 rows of 4 heads, ctx 8192): 14.0 us per launch (13.7 without
// the maximum per stage, add_own_max); with K rows straight from HBM as MFMA operands, V transposed through LDS and a
// work-group per (row tile, chunk) it took 23.9 us.
//
// The tree-verify form with the Q/K prep (attn2_kernel<.., PREP>, head_dim 128): the launch also does the
// RoPE/KV kernel's work for these rows (mdx_rope.hpp: per-head RMSNorm, split-half RoPE), so the step
// needs no launch for it. Every work-group computes its kv head's query rows itself (64 rows x 128, into
// LDS) while its first ring stages stream in; the tree work-group also computes the tree rows' k, writes
// them (k_out, and the cache at their positions, which lie past the prefix the chunks read) with the v
// rows, and only then streams them back as its tree stage. Bit-identical to qk_norm_rope_kv + the
// streaming form.
#include <math.h>
#include <stdlib.h>
#include <type_traits>

#include "mdx_common.hpp"
#include "mdx_rope.hpp"

namespace mdx {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

constexpr float LOG2E = 1.4426950408889634f;

struct AttnArgs {
    const uint16_t* q;       // [H, S, D] with strides qh, qs
    int64_t qh, qs;
    const uint16_t* key;     // [Hk, cap, D]
    const uint16_t* value;
    const int32_t* seqlen;   // [1]
    const uint16_t* xk;      // [Hk, S, D] with strides xh, xs (tree rows)
    const uint16_t* xv;
    int64_t xh, xs, vh, vs;
    const int32_t* mask;     // [S] or null (draft row)
    uint16_t* out;           // [S, H, D]
    float* part;             // [Hk][RT][C + 1][2 * 16 + 16 * D]
    int H, Hk, S, cap, groups, rows, RT, C;
    int parts;               // token parts per chunk
    float zscale;            // 1/sqrt(D) * log2(e)
    // the Q/K prep (PREP launches): raw q / k rows [S][H][D] with strides (row, head), the per-head norm
    // weights (null: no norm), the rows' rotation matrices [S][rd / 2][2][2] (row stride fs floats), the
    // caches the tree rows' k / v are written to at pos, k_out = xk [Hk][S][D], q_out [H][S][D] or null
    const uint16_t* rq;
    int64_t rqs, rqh;
    const uint16_t* rk;
    int64_t rks, rkh;
    const uint16_t* wq;
    const uint16_t* wk;
    float epsq, epsk;
    const float* freqs;
    int64_t fs;
    int rd;
    uint16_t* kc;
    uint16_t* vc;
    const int64_t* pos;
    uint16_t* k_out;
    uint16_t* q_out;
    // the merge's output times sigmoid: out <- bf16(out * sig[gate]), gate of (row, head, d) at gate[row * gate_row + 2 D head
    // + D + d] (the gate half of each head's 2 D projection columns); null: no gate
    const uint16_t* gate;
    int64_t gate_row;
    const uint16_t* sig;
};

__device__ __forceinline__ unsigned bf16pair(float a, float b) { return unsigned(f2bf(a)) | (unsigned(f2bf(b)) << 16); }

__device__ __forceinline__ bf16x8 as_bf16x8(u32x4 v) { return __builtin_bit_cast(bf16x8, v); }

__device__ __forceinline__ u32x4 ld16(const uint16_t* p) {
    return *reinterpret_cast<const u32x4*>(p);
}

// ---- The streaming form ----------------------------------------------------------------------------
// One work-group per (kv head, chunk): all of the kv head's query rows (up to 4 row tiles) in one
// work-group, so each K/V byte leaves HBM once and is read from LDS by every row tile. Wave w of NWV
// owns row tile w % RTW and token part w / RTW of the chunk (P = NWV / RTW parts; eight waves, two per
// SIMD, wherever each part still gets two ring stages). A part's K and V stream through its share of
// a 128 KiB LDS ring of 32-token stages by direct-to-LDS loads (1 KiB per wave instruction, the ring's
// stages in flight from the prologue). Per stage a wave reads its S^T and V^T operands from LDS in two
// batches (layouts at stage_k), computes S^T = K Q^T, the online softmax in its lanes, and
// O^T += V^T P^T; the P parts of a row tile merge in LDS. The grid is at most 256 work-groups (one
// round on the chip's 256 CUs: the ring takes most of a CU's LDS).
constexpr int A2_STEP = 32;
constexpr int A2_RING = 128 * 1024;  // K/V ring bytes per work-group
constexpr int A2_MAX_WG = 256;

// LDS layout of a ring stage (32 tokens; no swizzle: every read below covers contiguous bytes)
//   K: [kk < D/32][token 32][g 4][16 B]  -- unit 4 kk + g of each token row; the S^T operand of
//      (16-token tile tt, kk) is one contiguous KiB: lane (c16, g) at kk * 2048 + (16 tt + c16) * 64 + g * 16
//   V: [dt < D/16][token 32][2][16 B]    -- dims 16 dt .. 16 dt + 15 of each token row; a transposing
//      read of (dt, tokens 16 h ..) is 512 contiguous bytes at dt * 1024 + h * 512
// so one base address per lane and immediate offsets reach every operand of the stage. The reads are
// inline asm: the builtins make the compiler wait for every outstanding direct-to-LDS load (vmcnt(0))
// before them, which would drain the ring each stage. Each asm statement ends with its lgkmcnt(0)
// wait, so its results exist (for the compiler) only after the wait. ds_read_b64_tr_b16 (gfx950): in
// each 16-lane group, lane i receives element i % 4 of the 8-byte runs that lanes i / 4 + 4 j point
// at (j = 0..3).
__device__ __forceinline__ uint32_t lds_addr(const unsigned char* p) {
    return uint32_t(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const unsigned char*)p));
}
template <int D>
__device__ __forceinline__ void stage_k(u32x4 (&kf)[2][D / 32], uint32_t base) {
    if constexpr (D == 256) {
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
            asm volatile(
                "ds_read_b128 %0, %8\n\tds_read_b128 %1, %8 offset:2048\n\tds_read_b128 %2, %8 offset:4096\n\t"
                "ds_read_b128 %3, %8 offset:6144\n\tds_read_b128 %4, %8 offset:8192\n\tds_read_b128 %5, %8 offset:10240\n\t"
                "ds_read_b128 %6, %8 offset:12288\n\tds_read_b128 %7, %8 offset:14336\n\ts_waitcnt lgkmcnt(0)"
                : "=&v"(kf[tt][0]), "=&v"(kf[tt][1]), "=&v"(kf[tt][2]), "=&v"(kf[tt][3]), "=&v"(kf[tt][4]), "=&v"(kf[tt][5]),
                  "=&v"(kf[tt][6]), "=&v"(kf[tt][7])
                : "v"(base + tt * 1024));
    } else if constexpr (D == 128) {
        asm volatile(
            "ds_read_b128 %0, %8\n\tds_read_b128 %1, %8 offset:2048\n\tds_read_b128 %2, %8 offset:4096\n\t"
            "ds_read_b128 %3, %8 offset:6144\n\tds_read_b128 %4, %8 offset:1024\n\tds_read_b128 %5, %8 offset:3072\n\t"
            "ds_read_b128 %6, %8 offset:5120\n\tds_read_b128 %7, %8 offset:7168\n\ts_waitcnt lgkmcnt(0)"
            : "=&v"(kf[0][0]), "=&v"(kf[0][1]), "=&v"(kf[0][2]), "=&v"(kf[0][3]), "=&v"(kf[1][0]), "=&v"(kf[1][1]),
              "=&v"(kf[1][2]), "=&v"(kf[1][3])
            : "v"(base));
    } else {
        static_assert(D == 64, "head_dim 64, 128 or 256");
        asm volatile(
            "ds_read_b128 %0, %4\n\tds_read_b128 %1, %4 offset:2048\n\tds_read_b128 %2, %4 offset:1024\n\t"
            "ds_read_b128 %3, %4 offset:3072\n\ts_waitcnt lgkmcnt(0)"
            : "=&v"(kf[0][0]), "=&v"(kf[0][1]), "=&v"(kf[1][0]), "=&v"(kf[1][1])
            : "v"(base));
    }
}
// (dim tiles [8 H, 8 H + 8) of V into va / vb)
template <int H, int DT>
__device__ __forceinline__ void stage_v8(u32x2 (&va)[DT], u32x2 (&vb)[DT], uint32_t base) {
    asm volatile(
        "ds_read_b64_tr_b16 %0, %16\n\tds_read_b64_tr_b16 %1, %16 offset:1024\n\t"
        "ds_read_b64_tr_b16 %2, %16 offset:2048\n\tds_read_b64_tr_b16 %3, %16 offset:3072\n\t"
        "ds_read_b64_tr_b16 %4, %16 offset:4096\n\tds_read_b64_tr_b16 %5, %16 offset:5120\n\t"
        "ds_read_b64_tr_b16 %6, %16 offset:6144\n\tds_read_b64_tr_b16 %7, %16 offset:7168\n\t"
        "ds_read_b64_tr_b16 %8, %16 offset:512\n\tds_read_b64_tr_b16 %9, %16 offset:1536\n\t"
        "ds_read_b64_tr_b16 %10, %16 offset:2560\n\tds_read_b64_tr_b16 %11, %16 offset:3584\n\t"
        "ds_read_b64_tr_b16 %12, %16 offset:4608\n\tds_read_b64_tr_b16 %13, %16 offset:5632\n\t"
        "ds_read_b64_tr_b16 %14, %16 offset:6656\n\tds_read_b64_tr_b16 %15, %16 offset:7680\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(va[8 * H + 0]), "=&v"(va[8 * H + 1]), "=&v"(va[8 * H + 2]), "=&v"(va[8 * H + 3]), "=&v"(va[8 * H + 4]), "=&v"(va[8 * H + 5]), "=&v"(va[8 * H + 6]),
          "=&v"(va[8 * H + 7]), "=&v"(vb[8 * H + 0]), "=&v"(vb[8 * H + 1]), "=&v"(vb[8 * H + 2]), "=&v"(vb[8 * H + 3]), "=&v"(vb[8 * H + 4]), "=&v"(vb[8 * H + 5]),
          "=&v"(vb[8 * H + 6]), "=&v"(vb[8 * H + 7])
        : "v"(base + H * 8192));
}
template <int D>
__device__ __forceinline__ void stage_v(u32x2 (&va)[D / 16], u32x2 (&vb)[D / 16], uint32_t base) {
    if constexpr (D >= 128) {
        stage_v8<0>(va, vb, base);
        if constexpr (D == 256) stage_v8<1>(va, vb, base);
    } else {
        asm volatile(
            "ds_read_b64_tr_b16 %0, %8\n\tds_read_b64_tr_b16 %1, %8 offset:1024\n\t"
            "ds_read_b64_tr_b16 %2, %8 offset:2048\n\tds_read_b64_tr_b16 %3, %8 offset:3072\n\t"
            "ds_read_b64_tr_b16 %4, %8 offset:512\n\tds_read_b64_tr_b16 %5, %8 offset:1536\n\t"
            "ds_read_b64_tr_b16 %6, %8 offset:2560\n\tds_read_b64_tr_b16 %7, %8 offset:3584\n\t"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(va[0]), "=&v"(va[1]), "=&v"(va[2]), "=&v"(va[3]), "=&v"(vb[0]), "=&v"(vb[1]), "=&v"(vb[2]),
              "=&v"(vb[3])
            : "v"(base));
    }
}

// The MFMA operand of P^T: bf16 values in fp32, their top halves.
__device__ __forceinline__ u32x4 p_operand(const float (&p)[2][4]) {
    auto top2 = [](float lo, float hi) { return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u); };
    return u32x4{top2(p[0][0], p[0][1]), top2(p[0][2], p[0][3]), top2(p[1][0], p[1][1]), top2(p[1][2], p[1][3])};
}

// O^T = alpha O^T + beta V^T P of a stage whose P was rounded to bf16 against its own maximum: its products are brought
// to the running maximum in fp32. The weight at the maximum that P is taken against is exactly 1, every other carries
// bf16's rounding, so the error grows with the tokens per maximum: against one running maximum over a part the outputs
// lay up to 2 % further from float64 (head_dim 256, ctx 16000: 1.760e-3, with a maximum per 32 tokens 1.709e-3), against
// one over the whole prefix in the prefill form up to 8 % further than the same rows in chains of 16 (500 rows after 500,
// head_dim 128: 1.862e-3, per stage 1.722e-3 like the chains).
template <int DT>
__device__ __forceinline__ void add_own_max(f32x4 (&acc)[DT], const u32x2 (&va)[DT], const u32x2 (&vb)[DT], const u32x4 pf,
                                            const float alpha, const float beta) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
        const u32x4 vf = {va[dt].x, va[dt].y, vb[dt].x, vb[dt].y};
        const f32x4 o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(vf), as_bf16x8(pf), f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[dt][i] = fmaf(o[i], beta, acc[dt][i] * alpha);
    }
}

// chunk length (tokens, a multiple of 32 P) and active chunk count for context L over C chunks
__device__ __forceinline__ void split2(int L, int C, int P, int& T, int& active) {
    const int per = (L + C - 1) / C, q = A2_STEP * P;
    T = per < 1 ? q : (per + q - 1) / q * q;
    active = L > 0 ? (L + T - 1) / T : 0;
}

template <int D, int RTW, int NWV, bool PREP = false>
__global__ __launch_bounds__(64 * NWV) void attn2_kernel(AttnArgs a) {
    constexpr int P = NWV / RTW;
    constexpr int KK = D / 32, DT = D / 16;
    constexpr int RB = 2 * D;                    // bytes per token row
    constexpr int STAGE = A2_STEP * RB;          // bytes of K (or V) per stage
    constexpr int NS = A2_RING / (2 * STAGE * P);  // ring stages per part
    constexpr int PER = STAGE / 1024 / RTW;      // DMA instructions per wave, stage and matrix
    // A ring of two stages goes out whole in the prologue and refills a slot once every wave has read it (a second
    // barrier per stage): filled one stage ahead, the second stage's load would go out only after the first had landed.
    // Longer rings fill NS - 1 ahead and refill the slot of the stage before at the top of a stage.
    constexpr bool WHOLE = NS == 2;
    // head_dim 256's parts are up to 96 tokens and more long (two parts per chunk): a maximum per stage (add_own_max)
    constexpr bool OWN = D == 256;
    constexpr int AHEAD = WHOLE ? NS : NS - 1;  // stages issued by the prologue
    static_assert(NS >= 2 && PER >= 1 && (AHEAD - 1) * 2 * PER <= 63, "ring geometry");
    extern __shared__ __align__(16) unsigned char smem[];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, g = lane >> 4, c16 = lane & 15;
    const int rt = w % RTW, part = w / RTW;
    const int kh = blockIdx.x / (a.C + 1), cslot = blockIdx.x % (a.C + 1);
    const bool tree = cslot == a.C;
    int L = a.seqlen[0];
    L = L < 0 ? 0 : (L > a.cap ? a.cap : L);
    int T, active;
    split2(L, a.C, P, T, active);
    if (tree ? a.mask == nullptr : cslot >= active) return;  // no tokens: no partial (the merge skips it)
    const int nst = tree ? 1 : T / (A2_STEP * P);  // stages per part

    // this lane's query row
    const int r = rt * 16 + c16;
    const bool rvalid = r < a.rows;
    const int rr = rvalid ? r : 0;
    const int hq = kh * a.groups + rr / a.S, sq = rr % a.S;
    // the tree rows' masks by scalar loads (the tree work-group only): a vector load here would be waited
    // for with vmcnt(0) at its first use, i.e. behind every stage of the ring issued below
    uint32_t rmask = 0u;
    if (tree) {  // (uniform)
        typedef __attribute__((address_space(4))) const int32_t* const_i32p;
        const const_i32p mc = (const_i32p)(a.mask);
        for (int i = 0; i < a.S; ++i) {
            const uint32_t mi = uint32_t(mc[i]);
            rmask = (rvalid && sq == i) ? mi : rmask;
        }
    }

    // the part's tokens and sources (element strides)
    int t_begin, t_end;
    const uint16_t *kb, *vb;
    int64_t ks, vs;
    if (tree) {
        t_begin = 0;
        t_end = part == 0 ? a.S : 0;
        kb = a.xk + kh * a.xh;
        vb = a.xv + kh * a.vh;
        ks = a.xs;
        vs = a.vs;
    } else {
        t_begin = cslot * T + part * (T / P);
        t_end = min(L, t_begin + T / P);
        kb = a.key + int64_t(kh) * a.cap * D;
        vb = a.value + int64_t(kh) * a.cap * D;
        ks = vs = D;
    }
    const int t_last = t_end > t_begin ? t_end - 1 : (tree ? 0 : min(t_begin, L - 1));
    const int t_clamp = t_last < 0 ? 0 : t_last;  // a token every load may read (in bounds)

    // The query rows reach the MFMA operands through LDS, read by inline asm: the compiler waits for every
    // direct-to-LDS load in flight before it uses a vector register that a load wrote, so query rows loaded
    // into registers would drain the ring at every stage. Rows D + 8 elements apart with the Q/K prep
    // (written by asm), D apart otherwise (direct loads of whole rows).
    u32x4 qf[KK];
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) qf[kk] = u32x4{0, 0, 0, 0};
    static_assert(!PREP || (D == 128 && NWV == 8), "the Q/K prep: head_dim 128, eight waves");
    constexpr int QROW = D + (PREP ? 8 : 0);
    __shared__ __align__(16) uint16_t qst[16 * RTW * QROW];
    const uint32_t qbase = lds_addr(reinterpret_cast<const unsigned char*>(qst));
    if constexpr (!PREP) {
        // part 0's wave of each row tile brings the tile's 16 rows (D / 32 loads of 1 KiB, ahead of the ring:
        // the first stage's wait covers them, its barrier every tile's)
        if (part == 0) {
            constexpr int LPR = D / 8, RPI = 64 / LPR;  // lanes per row, rows per load
#pragma unroll
            for (int j = 0; j < D / 32; ++j) {
                const int rr_ = min(rt * 16 + j * RPI + lane / LPR, a.rows - 1);  // (clamped: in bounds)
                const uint16_t* src = a.q + (kh * a.groups + rr_ / a.S) * a.qh + (rr_ % a.S) * a.qs + (lane % LPR) * 8;
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                                 (__attribute__((address_space(3))) void*)(qst + (rt * 16 + j * RPI) * D),
                                                 16, 0, 0);
            }
        }
    }
    auto read_q = [&]() {  // lane (row c16 of tile rt, k-group g): 8 elements at 32 kk + 8 g of its row
        const uint32_t ar = qbase + uint32_t((rvalid ? r : 0) * QROW + 8 * g) * 2;
        if constexpr (KK == 8)
            asm volatile("ds_read_b128 %0, %8\n\tds_read_b128 %1, %8 offset:64\n\tds_read_b128 %2, %8 offset:128\n\t"
                         "ds_read_b128 %3, %8 offset:192\n\tds_read_b128 %4, %8 offset:256\n\tds_read_b128 %5, %8 offset:320\n\t"
                         "ds_read_b128 %6, %8 offset:384\n\tds_read_b128 %7, %8 offset:448\n\ts_waitcnt lgkmcnt(0)"
                         : "=&v"(qf[0]), "=&v"(qf[1]), "=&v"(qf[2]), "=&v"(qf[3]), "=&v"(qf[4]), "=&v"(qf[5]), "=&v"(qf[6]),
                           "=&v"(qf[7])
                         : "v"(ar));
        else if constexpr (KK == 4)
            asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %4 offset:64\n\tds_read_b128 %2, %4 offset:128\n\t"
                         "ds_read_b128 %3, %4 offset:192\n\ts_waitcnt lgkmcnt(0)"
                         : "=&v"(qf[0]), "=&v"(qf[1]), "=&v"(qf[2]), "=&v"(qf[3])
                         : "v"(ar));
        else
            asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %2 offset:64\n\ts_waitcnt lgkmcnt(0)"
                         : "=&v"(qf[0]), "=&v"(qf[1])
                         : "v"(ar));
        if (!rvalid)
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) qf[kk] = u32x4{0, 0, 0, 0};
    };

    // (the tree work-group of a PREP launch writes its one stage itself, into part 0's first slot, which all
    // of its parts read: the other parts have no tokens there)
    unsigned char* ring = smem + ((PREP && tree) ? 0 : part) * NS * 2 * STAGE;
    // stage s of this part into ring slot s % NS: the wave's PER instructions of K and of V (instruction
    // i of a matrix writes LDS bytes [1024 i, 1024 i + 1024) of the stage's block in the layouts above;
    // lane -> (token within the stage, byte offset within the token row)). Byte offsets fit 32 bits
    // (cap * D * 2 < 2^31).
    const unsigned char* kbase = reinterpret_cast<const unsigned char*>(kb);
    const unsigned char* vbase = reinterpret_cast<const unsigned char*>(vb);
    const int ksb = int(ks) * 2, vsb = int(vs) * 2;
    int ktok[PER], kofs[PER], vtok[PER], vofs[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int i = rt * PER + j;
        ktok[j] = 16 * (i & 1) + (lane >> 2);
        kofs[j] = (4 * (i >> 1) + (lane & 3)) * 16;
        vtok[j] = lane >> 1;
        vofs[j] = (2 * i + (lane & 1)) * 16;
    }
    auto issue = [&](int s) {
        unsigned char* kd = ring + (s % NS) * 2 * STAGE;
        const int t0 = t_begin + s * A2_STEP;
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int o0 = (rt * PER + j) * 1024;
            const int tk = min(t0 + ktok[j], t_clamp), tv = min(t0 + vtok[j], t_clamp);
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(kbase + (tk * ksb + kofs[j])),
                                             (__attribute__((address_space(3))) void*)(kd + o0), 16, 0, 0);
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(vbase + (tv * vsb + vofs[j])),
                                             (__attribute__((address_space(3))) void*)(kd + STAGE + o0), 16, 0, 0);
        }
    };

    f32x4 acc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) acc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;

    if constexpr (!PREP) {
        for (int s = 0; s < AHEAD && s < nst; ++s) issue(s);
    } else {
        // The chunk work-groups issue the ring's first round, then the raw query rows (this wave's rows w,
        // w + NWV, ...; lane l: elements l and l + 64), their rotation matrices and norm weights: the wait
        // for these also waits for that round (loads return in order), which the first stage needs
        // anyway. The compiler waits for every direct-to-LDS load before it uses a vector register that a
        // load issued after them wrote, so no loaded register may be live into the stage loop: the query
        // rows go through LDS (inline asm, which the compiler does not track).
        if (!tree)
            for (int s = 0; s < AHEAD && s < nst; ++s) issue(s);
        constexpr int QPW = 64 / NWV;
        float rx0[QPW], rx1[QPW];
        float4 rm[QPW];
        // the rotation pair of element l (a lane past the rotated elements reads pair 0, unused)
        const int jj = lane >= a.rd ? 0 : (lane < a.rd / 2 ? lane : lane - a.rd / 2);
#pragma unroll
        for (int i = 0; i < QPW; ++i) {
            const int rc = min(w + NWV * i, a.rows - 1);  // (clamped: every load in bounds)
            const int s_ = rc % a.S;
            const uint16_t* src = a.rq + s_ * a.rqs + (kh * a.groups + rc / a.S) * a.rqh;
            rx0[i] = bf2f(src[lane]);
            rx1[i] = bf2f(src[lane + 64]);
            rm[i] = *reinterpret_cast<const float4*>(a.freqs + s_ * a.fs + jj * 4);
        }
        const uint16_t* wsrc = a.wq ? a.wq : a.rq;  // (no norm: any valid row, the values unused)
        const float wq0 = bf2f(wsrc[lane]), wq1 = bf2f(wsrc[lane + 64]);
        // the query rows into LDS (rows D + 8 elements apart: no bank conflicts)
        uint16_t qo0[QPW], qo1[QPW];
        qk_rope128_n<QPW>(rx0, rx1, a.wq != nullptr, wq0, wq1, a.epsq, a.rd, rm, lane, qo0, qo1);
#pragma unroll
        for (int i = 0; i < QPW; ++i) {
            const int r_ = w + NWV * i;
            if (r_ < a.rows) {  // (uniform)
                const uint32_t ad = qbase + uint32_t(r_ * QROW + lane) * 2;
                asm volatile("ds_write_b16 %0, %1\n\tds_write_b16 %0, %2 offset:128" ::"v"(ad), "v"(uint32_t(qo0[i])),
                             "v"(uint32_t(qo1[i])));
                if (tree && a.q_out) {
                    uint16_t* qo = a.q_out + ((kh * a.groups + r_ / a.S) * a.S + r_ % a.S) * D;
                    qo[lane] = qo0[i];
                    qo[lane + 64] = qo1[i];
                }
            }
        }
        if (tree) {
            // the tree rows' k (normed, rotated) and v straight into the stage this work-group reads, in the
            // layouts the ring's loads produce (K: block 2 (d / 32) + t / 16, row t % 16, 64 bytes; V: block
            // d / 16, row t, 32 bytes), and to k_out and the caches (stores nothing waits for); the V rows past
            // the tree rows zeroed (their P is 0, which a non-finite V would turn into NaN)
            const uint32_t kl = lds_addr(smem), vl = kl + STAGE;
            if ((threadIdx.x & 63) / 2 >= a.S)
                asm volatile("ds_write_b128 %0, %1" ::"v"(vl + threadIdx.x * 16), "v"(u32x4{0u, 0u, 0u, 0u}));
            for (int s_ = w; s_ < a.S; s_ += NWV) {
                const uint16_t* src = a.rk + s_ * a.rks + kh * a.rkh;
                const uint16_t* vsrc = a.xv + kh * a.vh + s_ * a.vs;
                const float x0 = bf2f(src[lane]), x1 = bf2f(src[lane + 64]);
                const uint16_t v0 = vsrc[lane], v1 = vsrc[lane + 64];
                const float4 m = *reinterpret_cast<const float4*>(a.freqs + s_ * a.fs + jj * 4);
                const float w0 = a.wk ? bf2f(a.wk[lane]) : 1.f, w1 = a.wk ? bf2f(a.wk[lane + 64]) : 1.f;
                uint16_t o0, o1;
                qk_rope128(x0, x1, a.wk != nullptr, w0, w1, a.epsk, a.rd, m, lane, o0, o1);
                asm volatile("ds_write_b16 %0, %1\n\tds_write_b16 %0, %2 offset:4096" ::"v"(
                                 kl + uint32_t((2 * (lane >> 5)) * 1024 + s_ * 64 + (lane & 31) * 2)),
                             "v"(uint32_t(o0)), "v"(uint32_t(o1)));
                asm volatile("ds_write_b16 %0, %1\n\tds_write_b16 %0, %2 offset:4096" ::"v"(
                                 vl + uint32_t((lane >> 4) * 1024 + s_ * 32 + (lane & 15) * 2)),
                             "v"(uint32_t(v0)), "v"(uint32_t(v1)));
                uint16_t* ko = a.k_out + (kh * a.S + s_) * D;
                ko[lane] = o0;
                ko[lane + 64] = o1;
                const int64_t p = a.pos[s_];
                if (p >= 0 && p < a.cap) {  // (a position outside the cache writes nothing)
                    uint16_t* kd = a.kc + (int64_t(kh) * a.cap + p) * D;
                    uint16_t* vd = a.vc + (int64_t(kh) * a.cap + p) * D;
                    kd[lane] = o0;
                    kd[lane + 64] = o1;
                    vd[lane] = v0;
                    vd[lane + 64] = v1;
                }
            }
        }
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this wave's rows are in LDS (the ring stays in flight)
        __builtin_amdgcn_s_barrier();
        read_q();
    }
    for (int s = 0; s < nst; ++s) {
        // stage s landed (this wave's share), then everyone's share and everyone done with stage s - 1 (the
        // PREP tree stage was written to LDS before the barrier that precedes the loop: no wait)
        if (PREP && tree) {
        } else if (s + AHEAD - 1 < nst) {
            constexpr int W = (AHEAD - 1) * 2 * PER;
            __builtin_amdgcn_s_waitcnt((W & 15) | ((W >> 4) << 14) | (7 << 4) | (15 << 8));
        } else {
            __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8));  // vmcnt(0): the ring's tail
        }
        // s_barrier alone: __syncthreads' release fence would wait for the whole ring (vmcnt(0))
        __builtin_amdgcn_s_barrier();
        if constexpr (!PREP)
            if (s == 0) read_q();
        if (!WHOLE && s + NS - 1 < nst) issue(s + NS - 1);
        const unsigned char* kd = ring + (s % NS) * 2 * STAGE;
        const unsigned char* vd = kd + STAGE;
        const int t0 = t_begin + s * A2_STEP;
        // the S^T operands of the stage: lane (token 16 tt + c16, k-group g) reads unit 4 kk + g
        u32x4 kf[2][KK];
        stage_k<D>(kf, lds_addr(kd) + c16 * 64 + g * 16);
        f32x4 st[2];
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) {
            st[tt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kk = 0; kk < KK; ++kk)
                st[tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(kf[tt][kk]), as_bf16x8(qf[kk]), st[tt], 0, 0, 0);
        }
        // V^T operands by transposing reads (issued while the S^T MFMAs run): lane s of group g points at token 4 g + s / 4 (+ 16 for the
        // second read), dims 16 dt + 4 (s % 4) .. + 3, so lane (dim 16 dt + c16, g) receives the 8 tokens
        // of its k-slots (4 g .. 4 g + 3, then 16 + 4 g ..), the order its S^T accumulators give P^T
        u32x2 va[DT], vb2[DT];
        stage_v<D>(va, vb2, lds_addr(vd) + (4 * g + (c16 >> 2)) * 32 + (c16 & 3) * 8);
        if (WHOLE && s + NS < nst) {  // (uniform in the work-group) this slot is read (the reads' asm ended with its wait)
            __builtin_amdgcn_s_barrier();
            issue(s + NS);
        }
        // the stage's admitted tokens (bit j: token t0 + j); whole stages of the prefix skip the mask
        const int nvalid = t_end - t0;
        uint32_t mbits = nvalid >= 32 ? ~0u : (nvalid > 0 ? (1u << nvalid) - 1u : 0u);
        if (tree) mbits &= rmask;
        float z[2][4], mx = -INFINITY;
        if (__builtin_amdgcn_ballot_w64(mbits != ~0u) == 0) {
#pragma unroll
            for (int tt = 0; tt < 2; ++tt)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    z[tt][i] = st[tt][i] * a.zscale;
                    mx = fmaxf(mx, z[tt][i]);
                }
        } else {
            const uint32_t lb = mbits >> (4 * g);
#pragma unroll
            for (int tt = 0; tt < 2; ++tt)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    z[tt][i] = ((lb >> (16 * tt + i)) & 1u) ? st[tt][i] * a.zscale : -INFINITY;
                    mx = fmaxf(mx, z[tt][i]);
                }
        }
        mx = max_x32(max_x16(mx));
        const float mnew = fmaxf(m, mx);
        // v_exp_f32 directly (2^-inf = 0; a result below 2^-126 flushes to 0, far inside the bound);
        // a row with nothing admitted yet subtracts 0, so -inf - -inf never forms
        const float msub = mnew == -INFINITY ? 0.f : mnew;
        const float alpha = __builtin_amdgcn_exp2f(m - msub);
        // the maximum that P is taken against, and the factor from it to the running one (OWN: add_own_max)
        const float pmax = !OWN ? msub : (mx == -INFINITY ? 0.f : mx);
        const float beta = !OWN ? 1.f : __builtin_amdgcn_exp2f(mx - msub);
        float p[2][4], ps = 0.f;
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
#pragma unroll
            for (int i = 0; i < 4; i += 2) {
                p[tt][i] = __builtin_amdgcn_exp2f(z[tt][i] - pmax);
                p[tt][i + 1] = __builtin_amdgcn_exp2f(z[tt][i + 1] - pmax);
                bfround2(p[tt][i], p[tt][i + 1]);
                ps += p[tt][i];
                ps += p[tt][i + 1];
            }
        ps = sum_x32(sum_x16(ps));
        l = l * alpha + (OWN ? ps * beta : ps);
        m = mnew;
        if constexpr (OWN) {
            add_own_max<DT>(acc, va, vb2, p_operand(p), alpha, beta);
        } else {
            // O^T is rescaled only when some row's maximum moved (x * 1 == x: skipping changes no bit)
            if (__builtin_amdgcn_ballot_w64(alpha != 1.f) != 0) {
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) acc[dt] *= alpha;
            }
            const u32x4 pf = p_operand(p);
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                const u32x4 vf = {va[dt].x, va[dt].y, vb2[dt].x, vb2[dt].y};
                acc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(vf), as_bf16x8(pf), acc[dt], 0, 0, 0);
            }
        }
    }

    // the work-group's partial per row tile: (m, l, O) of its rows; P parts merge through LDS first
    float* rec = a.part + (int64_t(kh * a.RT + rt) * (a.C + 1) + cslot) * (32 + 16 * D);
    if (P == 1) {
        if (rt >= a.RT) return;
        if (g == 0) {
            rec[c16] = m;
            rec[16 + c16] = l;
        }
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) *reinterpret_cast<f32x4*>(rec + 32 + c16 * D + 16 * dt + 4 * g) = acc[dt];
        return;
    }
    __syncthreads();  // the ring is free
    // a wave's (m, l, O) in LDS with O's rows D + 4 floats apart (rows D apart would put the 16 rows a
    // store or load instruction touches in the same banks)
    constexpr int OR = D + 4;
    constexpr int WREG = (32 + 16 * OR) * 4;
    float* wr = reinterpret_cast<float*>(smem + w * WREG);
    if (g == 0) {
        wr[c16] = m;
        wr[16 + c16] = l;
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) *reinterpret_cast<f32x4*>(wr + 32 + c16 * OR + 16 * dt + 4 * g) = acc[dt];
    __syncthreads();
    // the row tile's P waves (w = rt + RTW * p) merged in part order by the RTW * 64 threads of part 0
    if (part != 0 || rt >= a.RT) return;
    auto part_reg = [&](int p_) { return reinterpret_cast<const float*>(smem + (rt + RTW * p_) * WREG); };
    float fw[P];
    float M = -INFINITY;
#pragma unroll
    for (int p_ = 0; p_ < P; ++p_) M = fmaxf(M, part_reg(p_)[c16]);
    float sl = 0.f;
#pragma unroll
    for (int p_ = 0; p_ < P; ++p_) {
        const float mv = part_reg(p_)[c16];
        fw[p_] = mv == -INFINITY ? 0.f : exp2f(mv - M);
        sl += part_reg(p_)[16 + c16] * fw[p_];
    }
    if (g == 0) {
        rec[c16] = M;
        rec[16 + c16] = sl;
    }
    // lane (row c16, group g): dims 4g + 16 dt .. + 3 of its row
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
        f32x4 o = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int p_ = 0; p_ < P; ++p_) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(part_reg(p_) + 32 + c16 * OR + 16 * dt + 4 * g);
            o += v * fw[p_];
        }
        *reinterpret_cast<f32x4*>(rec + 32 + c16 * D + 16 * dt + 4 * g) = o;
    }
}

// Merge of the chunk partials and the tree partial: one work-group of 256 per query row. D / 4 threads take a partial's
// O row in 16-byte pieces, so 1024 / D groups walk the partials at once, every load issued beside the maxima (they do not
// depend on the weights): behind the context length, one memory round trip. (One thread per dim over all partials:
// 7.3 us per launch at 54 partials of 256, 4.5 us at 17 of 128.)
constexpr int MERGE_T = 256;

template <int D>
__global__ __launch_bounds__(MERGE_T) void attn_merge_kernel(AttnArgs a) {
    constexpr int TPR = D / 4, G = MERGE_T / TPR, PER = (65 + G - 1) / G;  // (at most 64 chunks and the tree)
    __shared__ float wgt[PER * G];
    __shared__ __align__(16) float osum[G][D];
    const int row = blockIdx.x % 16, rt = (blockIdx.x / 16) % a.RT, kh = blockIdx.x / (16 * a.RT);
    const int r = rt * 16 + row;
    if (r >= a.rows) return;
    int L = a.seqlen[0];
    L = L < 0 ? 0 : (L > a.cap ? a.cap : L);
    int T, active;
    split2(L, a.C, a.parts, T, active);
    const bool use_tree = a.mask != nullptr;
    const int np = active + (use_tree ? 1 : 0);
    const float* base = a.part + int64_t(kh * a.RT + rt) * (a.C + 1) * (32 + 16 * D);
    auto slot = [&](int i) { return i < active ? i : a.C; };
    const int t = threadIdx.x, lane = t % 64, gi = t / TPR, d4 = (t % TPR) * 4;
    float sg = 0.f;  // (the gate's loads go out with the partials')
    if (a.gate) sg = bf2f(a.sig[a.gate[(r % a.S) * a.gate_row + int64_t(kh * a.groups + r / a.S) * 2 * D + D + min(t, D - 1)]]);
    // every wave takes the partials' maxima and sums itself (lane i: partials i and i + 64)
    const int i0 = min(lane, max(np - 1, 0)), i1 = min(lane + 64, max(np - 1, 0));
    float m0 = base[slot(i0) * (32 + 16 * D) + row], m1 = base[slot(i1) * (32 + 16 * D) + row];
    const float l0 = base[slot(i0) * (32 + 16 * D) + 16 + row], l1 = base[slot(i1) * (32 + 16 * D) + 16 + row];
    // (few partials of a small head: a third of the loads; at head_dim 256 the branch costs more than it saves)
    f32x4 ov[PER];
    auto load_o = [&](auto n) {
#pragma unroll
        for (int j = 0; j < decltype(n)::value; ++j)
            ov[j] = *reinterpret_cast<const f32x4*>(base + slot(min(gi + G * j, max(np - 1, 0))) * (32 + 16 * D) + 32 + row * D + d4);
    };
    constexpr int FEW = D == 256 ? PER : (PER + 2) / 3;
    const bool few = np <= FEW * G;  // (uniform)
#pragma unroll
    for (int j = FEW; j < PER; ++j) ov[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (few) load_o(std::integral_constant<int, FEW>{});
    else load_o(std::integral_constant<int, PER>{});
    m0 = lane < np ? m0 : -INFINITY;
    m1 = lane + 64 < np ? m1 : -INFINITY;
    auto ror = [](float v, auto ctl) {
        return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), decltype(ctl)::value, 0xF, 0xF, false));
    };
    using R8 = std::integral_constant<int, 0x128>;
    using R4 = std::integral_constant<int, 0x124>;
    using R2 = std::integral_constant<int, 0x122>;
    using R1 = std::integral_constant<int, 0x121>;
    float M = max_x32(max_x16(fmaxf(m0, m1)));
    M = fmaxf(M, ror(M, R8{}));
    M = fmaxf(M, ror(M, R4{}));
    M = fmaxf(M, ror(M, R2{}));
    M = fmaxf(M, ror(M, R1{}));
    const float w0 = m0 == -INFINITY ? 0.f : exp2f(m0 - M), w1 = m1 == -INFINITY ? 0.f : exp2f(m1 - M);
    // (a partial of weight 0 still counts: its NaN, or the infinity of its values, must reach the row)
    float s = (lane < np ? l0 * w0 : 0.f) + (lane + 64 < np ? l1 * w1 : 0.f);
    s = sum_x32(sum_x16(s));
    s += ror(s, R8{});
    s += ror(s, R4{});
    s += ror(s, R2{});
    s += ror(s, R1{});
    if (t < 64) {  // (weights past the partials are zero)
        wgt[lane] = w0;
        if (lane + 64 < PER * G) wgt[lane + 64] = w1;
    }
    __syncthreads();
    f32x4 o = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const float w = wgt[gi + G * j];
        if (gi + G * j < np) o += ov[j] * w;  // (an unused record may hold anything)
    }
    *reinterpret_cast<f32x4*>(&osum[gi][d4]) = o;
    __syncthreads();
    if (t >= D) return;
    float v = osum[0][t];
#pragma unroll
    for (int g = 1; g < G; ++g) v += osum[g][t];
    const int h = kh * a.groups + r / a.S, sr = r % a.S;
    uint16_t ob = f2bf(s > 0.f ? __fdiv_rn(v, s) : 0.f);
    if (a.gate) ob = f2bf(__fmul_rn(bf2f(ob), sg));  // (uniform)
    a.out[(int64_t(sr) * a.H + h) * D + t] = ob;
}

// ---- The prefill form (head_dim 64 and 128) ------------------------------------------------------
// S consecutive rows of a chain whose K/V rows are in the cache already: row s attends tokens [0, L + s]. A unit of
// work is (kv head, four row tiles of 16 rows in the order [16-row block][head of the group]); a wave owns one tile and
// the four waves share the K/V stages of the streaming form (its layouts, reads and online softmax), four in flight,
// up to the last token any of them attends. Units with the most tokens start first. One launch, no partials.
constexpr int AP_STAGES = 4;

template <int D>
__global__ __launch_bounds__(256) void attn_prefill_kernel(AttnArgs a) {
    constexpr int KK = D / 32, DT = D / 16, STAGE = A2_STEP * 2 * D, PER = STAGE / 1024 / 4;
    extern __shared__ __align__(16) unsigned char smem[];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6), g = lane >> 4, c16 = lane & 15;
    const int tiles = (a.S + 15) / 16 * a.groups, units = (tiles + 3) / 4;
    const int kh = blockIdx.x % a.Hk, unit = units - 1 - int(blockIdx.x) / a.Hk;
    int L = a.seqlen[0];
    L = L < 0 ? 0 : (L > a.cap - a.S ? a.cap - a.S : L);
    const int x = min(unit * 4 + w, tiles - 1);  // (a tile past the last repeats it and stores nothing)
    const bool live = unit * 4 + w < tiles;
    const int head = kh * a.groups + x % a.groups, s0 = x / a.groups * 16;
    const int row = min(s0 + c16, a.S - 1);
    const int wave_end = L + min(s0 + 16, a.S);                                              // tokens of this wave's tile
    const int end = L + min(min(unit * 4 + 3, tiles - 1) / a.groups * 16 + 16, a.S);         // of the unit
    const int nst = (end + A2_STEP - 1) / A2_STEP;
    u32x4 qf[KK];
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) qf[kk] = ld16(a.q + head * a.qh + row * a.qs + 32 * kk + 8 * g);
    // the query rows have arrived before the first direct-to-LDS load goes out (see the streaming form)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) asm volatile("" : "+v"(qf[kk]));
    const unsigned char* kbase = reinterpret_cast<const unsigned char*>(a.key + int64_t(kh) * a.cap * D);
    const unsigned char* vbase = reinterpret_cast<const unsigned char*>(a.value + int64_t(kh) * a.cap * D);
    int ktok[PER], kofs[PER], vofs[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int i = w * PER + j;
        ktok[j] = 16 * (i & 1) + (lane >> 2);
        kofs[j] = (4 * (i >> 1) + (lane & 3)) * 16;
        vofs[j] = (2 * i + (lane & 1)) * 16;
    }
    auto issue = [&](int s_) {
        const int s = min(s_, nst - 1);  // (past the end: the last stage again, into a free slot)
        unsigned char* kd = smem + (s_ % AP_STAGES) * 2 * STAGE;
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int o0 = (w * PER + j) * 1024;
            const int tk = min(s * A2_STEP + ktok[j], end - 1), tv = min(s * A2_STEP + (lane >> 1), end - 1);
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(kbase + (tk * 2 * D + kofs[j])),
                                             (__attribute__((address_space(3))) void*)(kd + o0), 16, 0, 0);
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(vbase + (tv * 2 * D + vofs[j])),
                                             (__attribute__((address_space(3))) void*)(kd + STAGE + o0), 16, 0, 0);
        }
    };
    f32x4 acc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) acc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;
#pragma unroll
    for (int s = 0; s < AP_STAGES - 1; ++s) issue(s);
    for (int s = 0; s < nst; ++s) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((AP_STAGES - 2) * 2 * PER) : "memory");
        __builtin_amdgcn_s_barrier();
        issue(s + AP_STAGES - 1);
        const int t0 = s * A2_STEP;
        if (t0 >= wave_end) continue;  // (uniform in the wave: only the barriers and loads are left)
        const unsigned char* kd = smem + (s % AP_STAGES) * 2 * STAGE;
        u32x4 kf[2][KK];
        stage_k<D>(kf, lds_addr(kd) + c16 * 64 + g * 16);
        f32x4 st[2];
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) {
            st[tt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kk = 0; kk < KK; ++kk)
                st[tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(kf[tt][kk]), as_bf16x8(qf[kk]), st[tt], 0, 0, 0);
        }
        u32x2 va[DT], vb2[DT];
        stage_v<D>(va, vb2, lds_addr(kd + STAGE) + (4 * g + (c16 >> 2)) * 32 + (c16 & 3) * 8);
        const int nvalid = L + row + 1 - t0;  // this row's tokens of the stage
        // a stage whole for every row takes its 32 tokens at once; one on the diagonal as two halves with a maximum each,
        // as a chain of 16 rows takes its own rows apart from the prefix (add_own_max)
        const int parts = __builtin_amdgcn_ballot_w64(nvalid < A2_STEP) == 0 ? 1 : 2;  // (uniform in the wave)
        for (int part = 0; part < parts; ++part) {
            float z[2][4], mx = -INFINITY;
#pragma unroll
            for (int tt = 0; tt < 2; ++tt)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const bool in = parts == 1 || (tt == part && 16 * tt + 4 * g + i < nvalid);
                    z[tt][i] = in ? st[tt][i] * a.zscale : -INFINITY;
                    mx = fmaxf(mx, z[tt][i]);
                }
            mx = max_x32(max_x16(mx));
            const float mnew = fmaxf(m, mx);
            const float msub = mnew == -INFINITY ? 0.f : mnew;
            const float alpha = __builtin_amdgcn_exp2f(m - msub);
            const float pmax = mx == -INFINITY ? 0.f : mx, beta = __builtin_amdgcn_exp2f(mx - msub);
            float p[2][4], ps = 0.f;
#pragma unroll
            for (int tt = 0; tt < 2; ++tt)
#pragma unroll
                for (int i = 0; i < 4; i += 2) {
                    p[tt][i] = __builtin_amdgcn_exp2f(z[tt][i] - pmax);
                    p[tt][i + 1] = __builtin_amdgcn_exp2f(z[tt][i + 1] - pmax);
                    bfround2(p[tt][i], p[tt][i + 1]);
                    ps += p[tt][i];
                    ps += p[tt][i + 1];
                }
            ps = sum_x32(sum_x16(ps));
            l = l * alpha + ps * beta;
            m = mnew;
            add_own_max<DT>(acc, va, vb2, p_operand(p), alpha, beta);
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load into this work-group's LDS may outlive it
    if (!live || s0 + c16 >= a.S) return;
    uint16_t* o = a.out + (int64_t(s0 + c16) * a.H + head) * D + 4 * g;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = l > 0.f ? __fdiv_rn(acc[dt][i], l) : 0.f;
        *reinterpret_cast<uint2*>(o + 16 * dt) = make_uint2(bf16pair(v[0], v[1]), bf16pair(v[2], v[3]));
    }
}

template <int D>
int launch_prefill(const AttnArgs& a, hipStream_t st) {
    constexpr size_t lds = size_t(AP_STAGES) * 2 * A2_STEP * 2 * D;
    const int units = ((a.S + 15) / 16 * a.groups + 3) / 4;
    allow_smem(reinterpret_cast<const void*>(&attn_prefill_kernel<D>), lds);
    hipLaunchKernelGGL(attn_prefill_kernel<D>, dim3(unsigned(units * a.Hk)), dim3(256), lds, st, a);
    MDX_LAUNCHED();
    return MDX_OK;
}

int stream_rtw(int RT) { return RT <= 1 ? 1 : (RT == 2 ? 2 : 4); }
// token parts per chunk (head_dim 256: a stage is 32 KiB, so two parts of two stages, or one of four with four row tiles;
// two waves with one row tile, else four): eight waves per work-group (two per SIMD, so one wave's LDS and MFMA waits
// overlap the other's work) where each part still gets two ring stages, else four waves (head_dim 128
// with one row tile)
int stream_parts(int D, int RT) {
    const int rtw = stream_rtw(RT);
    if (D == 256) return rtw == 4 ? 1 : 2;
    if (D == 128) return rtw == 4 ? 2 : 4;
    return 8 / rtw;
}
// chunks per kv head of the streaming form: one work-group per (kv head, chunk) plus the tree
// work-group within one round of 256, at least 32 tokens per part, at most 64 chunks (the merge)
int plan_chunks2(int Hk, int RT, int D, int cap, int hint) {
    const int P = stream_parts(D, RT);
    int c = A2_MAX_WG / Hk - 1;
    const int by_cap = (cap + A2_STEP * P - 1) / (A2_STEP * P);
    c = c > by_cap ? by_cap : c;
    if (hint > 0 && c > hint) c = hint;
    return c < 1 ? 1 : (c > 64 ? 64 : c);
}

size_t workspace_bytes(int Hk, int RT, int C, int D) {
    return 256 + size_t(Hk) * RT * (C + 1) * (32 + 16 * size_t(D)) * sizeof(float);
}

template <int D, int RTW, int NWV, bool PREP = false>
int launch2(const AttnArgs& a, hipStream_t st) {
    allow_smem(reinterpret_cast<const void*>(&attn2_kernel<D, RTW, NWV, PREP>), A2_RING);
    hipLaunchKernelGGL((attn2_kernel<D, RTW, NWV, PREP>), dim3(a.Hk * (a.C + 1)), dim3(64 * NWV), A2_RING, st, a);
    MDX_LAUNCHED();
    hipLaunchKernelGGL(attn_merge_kernel<D>, dim3(a.Hk * a.RT * 16), dim3(MERGE_T), 0, st, a);
    MDX_LAUNCHED();
    return MDX_OK;
}

template <int D>
int launch(const AttnArgs& a, hipStream_t st) {
    const int rtw = stream_rtw(a.RT);
    if constexpr (D == 256) {
        if (rtw == 1) return launch2<D, 1, 2>(a, st);
        if (rtw == 2) return launch2<D, 2, 4>(a, st);
        return launch2<D, 4, 4>(a, st);
    } else {
        if (rtw == 1) return launch2<D, 1, (D == 128 ? 4 : 8)>(a, st);
        if (rtw == 2) return launch2<D, 2, 8>(a, st);
        return launch2<D, 4, 8>(a, st);
    }
}

}  // namespace
}  // namespace mdx

using namespace mdx;

extern "C" size_t mdx_attn_workspace(int64_t H, int64_t Hk, int64_t S, int64_t D, int64_t cap, int64_t chunks_hint) {
    if (Hk <= 0 || H % Hk != 0 || S <= 0) return 0;
    const int RT = int((H / Hk * S + 15) / 16);
    const int C = plan_chunks2(int(Hk), RT, int(D), int(cap), int(chunks_hint));
    return workspace_bytes(int(Hk), RT, C, int(D));
}

namespace {

int attn_decode_run(const uint16_t* q, int64_t q_head_stride, int64_t q_row_stride, const uint16_t* key, const uint16_t* value,
                    const int32_t* seqlen, const uint16_t* xk, int64_t xk_head_stride, int64_t xk_row_stride,
                    const uint16_t* xv, int64_t xv_head_stride, int64_t xv_row_stride, const int32_t* mask, uint16_t* out,
                    int64_t H, int64_t Hk, int64_t S, int64_t D, int64_t cap, int64_t chunks_hint, const uint16_t* gate,
                    int64_t gate_row, const uint16_t* sig, void* workspace, size_t workspace_bytes_, void* stream) {
    MDX_CHECK(q && key && value && seqlen && xk && xv && out, "null pointer");
    MDX_CHECK(D == 64 || D == 128 || D == 256, "head_dim must be 64, 128 or 256");
    MDX_CHECK(Hk >= 1 && H % Hk == 0 && S >= 1 && S <= 16, "heads / 1..16 rows");
    MDX_CHECK(mask || S == 1, "a draft (no mask) has one row");
    MDX_CHECK(H / Hk * S <= 64, "at most 64 query rows per kv head");
    MDX_CHECK(cap >= 1 && cap < (int64_t(1) << 30) / D, "cache capacity");
    MDX_CHECK(aligned(q, 16) && aligned(key, 16) && aligned(value, 16) && aligned(xk, 16) && aligned(xv, 16) &&
                  q_head_stride % 8 == 0 && q_row_stride % 8 == 0 && xk_head_stride % 8 == 0 &&
                  xk_row_stride % 8 == 0 && xv_head_stride % 8 == 0 && xv_row_stride % 8 == 0,
              "16-byte aligned rows");
    const int RT = int((H / Hk * S + 15) / 16);
    const int C = plan_chunks2(int(Hk), RT, int(D), int(cap), int(chunks_hint));
    MDX_CHECK(workspace && aligned(workspace, 256) && workspace_bytes_ >= workspace_bytes(int(Hk), RT, C, int(D)),
              "workspace: %zu bytes, 256-byte aligned, zeroed once", workspace_bytes(int(Hk), RT, C, int(D)));
    AttnArgs a{};
    a.q = q;
    a.qh = q_head_stride;
    a.qs = q_row_stride;
    a.key = key;
    a.value = value;
    a.seqlen = seqlen;
    a.xk = xk;
    a.xv = xv;
    a.xh = xk_head_stride;
    a.xs = xk_row_stride;
    a.vh = xv_head_stride;
    a.vs = xv_row_stride;
    a.mask = mask;
    a.out = out;
    a.gate = gate;
    a.gate_row = gate_row;
    a.sig = sig;
    a.part = reinterpret_cast<float*>(static_cast<char*>(workspace) + 256);
    a.H = int(H);
    a.Hk = int(Hk);
    a.S = int(S);
    a.cap = int(cap);
    a.groups = int(H / Hk);
    a.rows = int(H / Hk * S);
    a.RT = RT;
    a.C = C;
    a.parts = stream_parts(int(D), RT);
    a.zscale = float(1.0 / sqrt(double(D)) * 1.4426950408889634);
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (D == 64) return launch<64>(a, st);
    if (D == 128) return launch<128>(a, st);
    return launch<256>(a, st);
}

}  // namespace

extern "C" int mdx_attn_decode(const uint16_t* q, int64_t q_head_stride, int64_t q_row_stride, const uint16_t* key,
                               const uint16_t* value, const int32_t* seqlen, const uint16_t* xk, int64_t xk_head_stride,
                               int64_t xk_row_stride, const uint16_t* xv, int64_t xv_head_stride, int64_t xv_row_stride,
                               const int32_t* mask, uint16_t* out,
                               int64_t H, int64_t Hk, int64_t S, int64_t D, int64_t cap, int64_t chunks_hint,
                               void* workspace, size_t workspace_bytes_, void* stream) {
    return attn_decode_run(q, q_head_stride, q_row_stride, key, value, seqlen, xk, xk_head_stride, xk_row_stride, xv, xv_head_stride,
                           xv_row_stride, mask, out, H, Hk, S, D, cap, chunks_hint, nullptr, 0, nullptr, workspace,
                           workspace_bytes_, stream);
}

extern "C" int mdx_attn_decode_gated(const uint16_t* q, int64_t q_head_stride, int64_t q_row_stride, const uint16_t* key,
                               const uint16_t* value, const int32_t* seqlen, const uint16_t* xk, int64_t xk_head_stride,
                               int64_t xk_row_stride, const uint16_t* xv, int64_t xv_head_stride, int64_t xv_row_stride,
                               const int32_t* mask, uint16_t* out,
                               int64_t H, int64_t Hk, int64_t S, int64_t D, int64_t cap, int64_t chunks_hint,
                               const uint16_t* gate, int64_t gate_row_stride, const uint16_t* sig_lut,
                               void* workspace, size_t workspace_bytes_, void* stream) {
    MDX_CHECK(gate && sig_lut && gate_row_stride >= 2 * H * D, "gate rows [S, >= 2 H D] and a sigmoid table");
    return attn_decode_run(q, q_head_stride, q_row_stride, key, value, seqlen, xk, xk_head_stride, xk_row_stride, xv, xv_head_stride,
                           xv_row_stride, mask, out, H, Hk, S, D, cap, chunks_hint, gate, gate_row_stride, sig_lut, workspace,
                           workspace_bytes_, stream);
}

// Tree-verify attention with the RoPE/KV kernel's Q/K prep in the same launch: see the note at the top of
// this file. Raw rows as mdx_qk_norm_rope_kv takes them, the cache written at position[s] as it writes it,
// k_out [Hk, S, D] (also the tree rows' k the launch attends), q_out [H, S, D] optional.
extern "C" int mdx_attn_decode_rope(const uint16_t* q, int64_t q_row_stride, int64_t q_head_stride, const uint16_t* k,
                                    int64_t k_row_stride, int64_t k_head_stride, const uint16_t* v, int64_t v_row_stride,
                                    int64_t v_head_stride, const uint16_t* weight_q, const uint16_t* weight_k, float eps_q,
                                    float eps_k, const float* freqs, int64_t freqs_row_stride, int64_t rd, uint16_t* key,
                                    uint16_t* value, const int64_t* position, const int32_t* seqlen, const int32_t* mask,
                                    uint16_t* k_out, uint16_t* q_out, uint16_t* out, int64_t H, int64_t Hk, int64_t S,
                                    int64_t D, int64_t cap, int64_t chunks_hint, void* workspace, size_t workspace_bytes_,
                                    void* stream) {
    MDX_CHECK(q && k && v && freqs && key && value && position && seqlen && mask && k_out && out, "null pointer");
    MDX_CHECK((weight_q == nullptr) == (weight_k == nullptr), "norm weights: both or neither");
    MDX_CHECK(D == 128, "the Q/K prep form: head_dim 128");
    MDX_CHECK(rd == 32 || rd == 64 || rd == 128, "rotary dimension 32, 64 or 128");
    MDX_CHECK(Hk >= 1 && H % Hk == 0 && S >= 1 && S <= 16, "heads / 1..16 rows");
    const int64_t rows = H / Hk * S;
    MDX_CHECK(rows > 16 && rows <= 64, "17..64 query rows per kv head (fewer: the separate launches)");
    MDX_CHECK(cap >= 1 && cap < (int64_t(1) << 30) / D, "cache capacity");
    MDX_CHECK(aligned(key, 16) && aligned(value, 16) && aligned(k_out, 16) && aligned(v, 16) && aligned(freqs, 16) &&
                  v_row_stride % 8 == 0 && v_head_stride % 8 == 0 && freqs_row_stride % 4 == 0,
              "16-byte aligned cache, k_out, v rows and rotation rows");
    const int RT = int((rows + 15) / 16);
    const int C = plan_chunks2(int(Hk), RT, int(D), int(cap), int(chunks_hint));
    MDX_CHECK(workspace && aligned(workspace, 256) && workspace_bytes_ >= workspace_bytes(int(Hk), RT, C, int(D)),
              "workspace: %zu bytes, 256-byte aligned, zeroed once", workspace_bytes(int(Hk), RT, C, int(D)));
    AttnArgs a{};
    a.key = key;
    a.value = value;
    a.seqlen = seqlen;
    a.xk = k_out;
    a.xh = S * D;
    a.xs = D;
    a.xv = v;
    a.vh = v_head_stride;
    a.vs = v_row_stride;
    a.mask = mask;
    a.out = out;
    a.part = reinterpret_cast<float*>(static_cast<char*>(workspace) + 256);
    a.H = int(H);
    a.Hk = int(Hk);
    a.S = int(S);
    a.cap = int(cap);
    a.groups = int(H / Hk);
    a.rows = int(rows);
    a.RT = RT;
    a.C = C;
    a.parts = stream_parts(int(D), RT);
    a.zscale = float(1.0 / sqrt(double(D)) * 1.4426950408889634);
    a.rq = q;
    a.rqs = q_row_stride;
    a.rqh = q_head_stride;
    a.rk = k;
    a.rks = k_row_stride;
    a.rkh = k_head_stride;
    a.wq = weight_q;
    a.wk = weight_k;
    a.epsq = eps_q;
    a.epsk = eps_k;
    a.freqs = freqs;
    a.fs = freqs_row_stride;
    a.rd = int(rd);
    a.kc = key;
    a.vc = value;
    a.pos = position;
    a.k_out = k_out;
    a.q_out = q_out;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (stream_rtw(RT) == 2) return launch2<128, 2, 8, true>(a, st);
    return launch2<128, 4, 8, true>(a, st);
}

extern "C" int mdx_attn_prefill(const uint16_t* q, int64_t q_head_stride, int64_t q_row_stride, const uint16_t* key,
                                const uint16_t* value, const int32_t* seqlen, uint16_t* out, int64_t H, int64_t Hk,
                                int64_t S, int64_t D, int64_t cap, void* stream) {
    MDX_CHECK(q && key && value && seqlen && out, "null pointer");
    MDX_CHECK(D == 64 || D == 128, "head_dim must be 64 or 128");
    MDX_CHECK(Hk >= 1 && H % Hk == 0 && S >= 1 && S <= cap, "heads / rows within the cache");
    MDX_CHECK(cap >= 1 && cap < (int64_t(1) << 30) / D, "cache capacity");
    MDX_CHECK(aligned(q, 16) && aligned(key, 16) && aligned(value, 16) && aligned(out, 8) && q_head_stride % 8 == 0 &&
                  q_row_stride % 8 == 0,
              "16-byte aligned rows");
    AttnArgs a{};
    a.q = q;
    a.qh = q_head_stride;
    a.qs = q_row_stride;
    a.key = key;
    a.value = value;
    a.seqlen = seqlen;
    a.out = out;
    a.H = int(H);
    a.Hk = int(Hk);
    a.S = int(S);
    a.cap = int(cap);
    a.groups = int(H / Hk);
    a.zscale = float(1.0 / sqrt(double(D)) * 1.4426950408889634);
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (D == 64) return launch_prefill<64>(a, st);
    return launch_prefill<128>(a, st);
}
