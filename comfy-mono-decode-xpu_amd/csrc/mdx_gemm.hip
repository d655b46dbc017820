// Many-row linears of the prompt prefill: W4A8 (the GEMV engine's contract, mdx_gemv.hip) and bf16, for any row count.
//
// The decode kernels stream every weight once per 16 rows; a prompt of a thousand tokens would stream them 63 times.
// Here a work-group of four waves computes RT x 16 rows by 4 x NT x 16 columns: a wave owns NT tiles of 16 columns
// for all of the work-group's rows, so a weight is decoded once per work-group, in registers, straight into its
// MFMA operand. The activation rows go through LDS (shared by the waves), 128 bytes of K per stage; the waves' codes
// and scales go through LDS regions of their own, so that every load of the loop is a direct-to-LDS one and a ring of
// three stages hides the memory latency behind the products.
//
// The loads are issued by inline asm: the compiler, which does not see them, schedules the LDS reads, the decode and
// the MFMAs of a stage freely (with the builtin it waits for every direct-to-LDS load in flight before any LDS
// read, which drains the ring at each stage). The kernel waits itself: s_waitcnt vmcnt, then s_barrier, per stage.
//
// Bound by a stage's parts one after another (operand reads, the decode of about 75 VALU per 16 x 128 codes, 32 MFMAs of
// a wave) behind one barrier: no single part taken out gains more than a fifth (gate/up 140 us; without the decode 127,
// without 7/8 of the MFMAs 115, without operand reads 140, without loads 132). 1000 rows, K = 4096: gate/up 2 x 12288
// columns 140 us (1.44 POP/s), 12288 columns 87 us; 4096 columns with two waves per SIMD (KSP) 32 us against 41 us with one. The same 1000 rows through the decode kernels: 63 x 16 rows,
// 1.0 ms for the gate/up pair.
//
// Products: v_mfma_i32_16x16x64_i8 (exact int32 sums: the bits are the GEMV's) or v_mfma_f32_16x16x32_bf16, A = 16
// weight columns, B = 16 rows; lane l holds row l % 16, columns 4 (l / 16) .. + 3 of its tile's outputs.
#include <algorithm>
#include <stdlib.h>
#include <type_traits>

#include "mdx_common.hpp"
#include "mdx_w4.hpp"

namespace mdx {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// the weights of a launch: W4 with fp16 scales (groups of at least one 128-k chunk), W4 with fp8 e4m3 scales (any
// group), bf16 (tile-major)
enum Mode : int { M_F16 = 0, M_FP8 = 1, M_BF16 = 2 };

struct GMat {
    const uint8_t* q;
    const uint8_t* s;
    const float* sch;
    int n, tiles;
};

struct GemmArgs {
    GMat m[3];
    int nm, pair;        // pair: gate / up interleaved tile by tile (nm == 2)
    int total;           // column tiles of 16
    int steps;           // K / 128 (W4) or K / 64 (bf16): 128 bytes of an activation row each
    int kb;              // bytes per activation row
    int lgG, ng;         // log2(group size), groups per row
    const float* cb;     // codebook or null (code - 8)
    const uint8_t* x;    // rows [M][kb]
    const float* xs;     // row scales [M] (W4)
    int M, MB, NB;       // rows, row blocks, column blocks
    void* out[3];
    const void* res[3];
    const uint16_t* lut; // pair: SiLU table
    int slice;           // bf16: stages per K slice
};

constexpr int STAGES = 3;

template <int MODE, int RT, int NT, int KSP>
struct Geo {
    static constexpr int A_STAGE = RT * 2048;                          // RT x 16 rows x 128 B
    static constexpr int W_TILE = MODE == M_BF16 ? 2048 : 1024;        // a tile's weights per stage
    static constexpr int S_STAGE = MODE == M_BF16 ? 0 : 256;           // a wave's scales per stage
    static constexpr int W_OFF = STAGES * A_STAGE;                     // (a K half's ring)
    static constexpr int S_OFF = W_OFF + STAGES * 4 * NT * W_TILE;
    static constexpr int RING = S_OFF + STAGES * 4 * S_STAGE;
    static constexpr int T_OFF = KSP * RING;
    static constexpr int LDS = T_OFF + (MODE == M_FP8 ? 4096 : 0);     // fp8: the tables of the 256 scale bytes
    static_assert(KSP == 1 || 4 * NT * RT * 1024 <= RING * KSP, "the halves' sums fit the rings");
    static constexpr int LOADS = RT / 2 + NT * (W_TILE / 1024) + (MODE == M_BF16 ? 0 : 1);  // per wave and stage
};

__device__ __forceinline__ uint32_t lds_u32(const void* p) {
    return uint32_t(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const unsigned char*)p));
}
// one direct-to-LDS load: 16 (4) bytes per lane from base + off (ptr) to LDS bytes dst + 16 (4) lane
__device__ __forceinline__ void dma16(uint32_t dst, const uint8_t* base, uint32_t off) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(off), "s"(base)
                 : "memory", "m0");
}
__device__ __forceinline__ void dma4(uint32_t dst, const uint8_t* ptr) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" ::"s"(dst), "v"(ptr) : "memory", "m0");
}

__device__ __forceinline__ int gmat(const GemmArgs& a, int g, int& tile) {
    if (a.pair) {
        tile = g >> 1;
        return g & 1;
    }
    tile = g;
    if (a.nm < 2 || tile < a.m[0].tiles) return 0;
    tile -= a.m[0].tiles;
    if (a.nm < 3 || tile < a.m[1].tiles) return 1;
    tile -= a.m[1].tiles;
    return 2;
}

template <int MODE, int RT, int NT, int KSP>
__global__ __launch_bounds__(256 * KSP, 2) void gemm_kernel(GemmArgs a) {
    using G = Geo<MODE, RT, NT, KSP>;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
    const int wave = wv & 3, half = wv >> 2;  // (half: 0 with KSP == 1)
    const int c = lane & 15, kq = lane >> 4;
    // work-group -> (column block, row block): the row blocks of a column block run one after another on one XCD
    // (ids go round the 8 XCDs), which re-reads the block's weights from its L2
    const int xcd = blockIdx.x & 7, loc = blockIdx.x >> 3;
    const int nb = (loc / a.MB) * 8 + xcd, m0 = (loc % a.MB) * RT * 16;
    if (nb >= a.NB) return;  // (uniform)
    // this wave's column tiles (a tile past the last repeats tile 0 and is not stored)
    int mi[NT], tile[NT];
    bool live[NT];
    const uint8_t* wq[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        const int g = (nb * 4 + wave) * NT + i;
        live[i] = g < a.total;
        mi[i] = gmat(a, live[i] ? g : 0, tile[i]);
        const uint8_t* q = mi[i] == 0 ? a.m[0].q : (mi[i] == 1 ? a.m[1].q : a.m[2].q);
        wq[i] = q + size_t(tile[i]) * a.steps * G::W_TILE;
    }
    uint8_t* ring = lds + half * G::RING;
    const uint32_t l0 = lds_u32(ring);
    // activation pieces: load j of this wave brings rows 8 (wave RT / 2 + j) .. + 7; 16-byte piece p of row r lies
    // at position p ^ (r / 2 % 8) of the row's 128 bytes, so that the 16 rows an operand read touches fall in
    // distinct banks
    uint32_t aoff[RT / 2];
#pragma unroll
    for (int j = 0; j < RT / 2; ++j) {
        const int r = (wave * (RT / 2) + j) * 8 + (lane >> 3);
        aoff[j] = uint32_t(min(m0 + r, a.M - 1)) * uint32_t(a.kb) + (((lane & 7) ^ ((r >> 1) & 7)) << 4);
    }
    // scales: fp16, one dword (two groups) per column: lane 16 i + c loads tile i's; fp8, an 8-byte window per column:
    // lane 32 i + 2 c + d loads dword d of tile i's
    const uint8_t* sp = nullptr;
    if constexpr (MODE != M_BF16) {
        static_assert(NT <= 2, "a wave's scales are one load per stage");
        const int ti = MODE == M_F16 ? (lane >> 4) % NT : (lane >> 5) % NT, sc = MODE == M_F16 ? c : (lane >> 1) & 15;
        const uint8_t* sb = nullptr;
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            const uint8_t* s = mi[i] == 0 ? a.m[0].s : (mi[i] == 1 ? a.m[1].s : a.m[2].s);
            s += size_t(tile[i]) * 16 * a.ng * (MODE == M_F16 ? 2 : 1);
            if (ti == i) sb = s;
        }
        sp = sb + size_t(sc) * a.ng * (MODE == M_F16 ? 2 : 1) + (MODE == M_FP8 ? 4 * (lane & 1) : 0);
    }
    auto issue = [&](int t_, int b) {
        const int s = min(t_ * KSP + half, a.steps - 1);  // (past the end: the last stage again, never used)
#pragma unroll
        for (int j = 0; j < RT / 2; ++j)
            dma16(l0 + b * G::A_STAGE + (wave * (RT / 2) + j) * 1024, a.x + size_t(s) * 128, aoff[j]);
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int h = 0; h < G::W_TILE / 1024; ++h)
                dma16(l0 + G::W_OFF + ((b * 4 + wave) * NT + i) * G::W_TILE + h * 1024, wq[i] + size_t(s) * G::W_TILE + h * 1024,
                      uint32_t(lane) * 16);
        if constexpr (MODE == M_F16) dma4(l0 + G::S_OFF + (b * 4 + wave) * 256, sp + ((s >> (a.lgG - 7)) & ~1) * 2);
        if constexpr (MODE == M_FP8) dma4(l0 + G::S_OFF + (b * 4 + wave) * 256, sp + (((s * 128) >> a.lgG) & ~7));
    };
    issue(0, 0);
    issue(1, 1);
    uint4* tbl = reinterpret_cast<uint4*>(lds + G::T_OFF);
    if constexpr (MODE == M_FP8) {
        float cb[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) cb[i] = a.cb ? a.cb[i] : float(i - 8);
        const float s = fp8_to_f32(uint8_t(threadIdx.x));
        const Lut L = a.cb ? make_lut(s, cb) : make_lut_c8(s);
        if (threadIdx.x < 256) tbl[threadIdx.x] = make_uint4(L.w[0], L.w[1], L.w[2], L.w[3]);
    }
    typedef typename std::conditional<MODE == M_BF16, v4f, v4i>::type Acc;
    Acc acc[NT][RT];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int r = 0; r < RT; ++r) acc[i][r] = Acc{};
    // operand reads: row c of a row tile, the lane's 16-byte pieces of the stage (W4: 2 kq, 2 kq + 1, the lane's 32 k in
    // code order; bf16: kq, 4 + kq, its 8 k of each 32)
    const int sw = (c >> 1) & 7;
    const int p0 = (MODE == M_BF16 ? kq : 2 * kq) ^ sw, p1 = (MODE == M_BF16 ? 4 + kq : 2 * kq + 1) ^ sw;
    int b = 0;
    const int turns = (a.steps + KSP - 1) / KSP;
    [[maybe_unused]] Acc tot[MODE == M_BF16 ? NT : 1][MODE == M_BF16 ? RT : 1] = {};
    for (int t = 0; t < turns; ++t) {
        const int s = t * KSP + half;  // this half's stage
        // the stage landed (this wave's loads: the next stage's may stay in flight) and this wave is done reading the one
        // before; then everyone's, and that one's slot takes the stage after next
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(G::LOADS) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const uint8_t* ab = ring + b * G::A_STAGE + c * 128;
        const uint8_t* wb = ring + G::W_OFF + (b * 4 + wave) * NT * G::W_TILE + lane * 16;
        const uint8_t* sb = ring + G::S_OFF + (b * 4 + wave) * 256;
        // every LDS read of the stage first: the row operands arrive while the codes are decoded
        uint4 cw[NT][G::W_TILE / 1024];
        uint32_t sc[NT][2];
#pragma unroll
        for (int i = 0; i < NT; ++i) {
#pragma unroll
            for (int h = 0; h < G::W_TILE / 1024; ++h) cw[i][h] = *reinterpret_cast<const uint4*>(wb + i * G::W_TILE + h * 1024);
            if constexpr (MODE == M_F16) sc[i][0] = *reinterpret_cast<const uint16_t*>(sb + (16 * i + c) * 4 + ((s >> (a.lgG - 7)) & 1) * 2);
            if constexpr (MODE == M_FP8) {
                const uint8_t* sp8 = sb + 128 * i + 8 * c - (((min(s, a.steps - 1) * 128) >> a.lgG) & ~7);
                sc[i][0] = sp8[(min(s, a.steps - 1) * 128 + 32 * kq) >> a.lgG];
                sc[i][1] = sp8[(min(s, a.steps - 1) * 128 + 32 * kq + 16) >> a.lgG];
            }
        }
        uint4 f[RT][2];
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            f[r][0] = *reinterpret_cast<const uint4*>(ab + r * 2048 + p0 * 16);
            f[r][1] = *reinterpret_cast<const uint4*>(ab + r * 2048 + p1 * 16);
        }
        __builtin_amdgcn_sched_barrier(0);
        issue(t + 2, b == 0 ? 2 : b - 1);
        uint4 w[NT][2];
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            if constexpr (MODE == M_BF16) {
                w[i][0] = cw[i][0];
                w[i][1] = cw[i][1];
            } else {
                uint32_t lo[4], hi[4];
                if constexpr (MODE == M_F16) {
                    const uint32_t sh = sc[i][0];
                    Lut L;
                    if (a.cb == nullptr && __builtin_amdgcn_ballot_w64((sh & 0x7FFFu) > F16_FAST_MAX) == 0) {
                        const uint2 q8 = make_q8_f16(sh);
                        L = lut_from_q8(q8.x, q8.y);
                    } else if (a.cb == nullptr) {
                        L = make_lut_c8(fp16_to_f32(uint16_t(sh)));
                    } else {
                        L = make_lut(fp16_to_f32(uint16_t(sh)), a.cb);
                    }
                    decode_tb<false>(cw[i][0], make_uint4(L.w[0], L.w[1], L.w[2], L.w[3]), lo, hi);
                } else {
                    decode_tb2(cw[i][0], tbl[sc[i][0]], tbl[sc[i][1]], lo, hi);
                }
                w[i][0] = make_uint4(lo[0], hi[0], lo[1], hi[1]);
                w[i][1] = make_uint4(lo[2], hi[2], lo[3], hi[3]);
            }
        }
        if (KSP == 1 || s < a.steps) {  // (uniform; past the end with an odd stage count)
#pragma unroll
            for (int r = 0; r < RT; ++r)
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int i = 0; i < NT; ++i) {
                        if constexpr (MODE == M_BF16)
                            acc[i][r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w[i][h]),
                                                                                __builtin_bit_cast(bf16x8, f[r][h]), acc[i][r], 0, 0, 0);
                        else
                            acc[i][r] = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(v4i, w[i][h]),
                                                                              __builtin_bit_cast(v4i, f[r][h]), acc[i][r], 0, 0, 0);
                    }
        }
        if constexpr (MODE == M_BF16) {
            // fp32 sums in mdx_bf16_linear's order: per K slice, the slices added in order
            if ((t + 1) % a.slice == 0) {  // (uniform)
#pragma unroll
                for (int i = 0; i < NT; ++i)
#pragma unroll
                    for (int r = 0; r < RT; ++r) {
                        tot[i][r] = t + 1 == a.slice ? acc[i][r] : tot[i][r] + acc[i][r];
                        acc[i][r] = Acc{};
                    }
            }
        }
        b = b == STAGES - 1 ? 0 : b + 1;
    }
    // no load into this work-group's LDS may outlive it
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if constexpr (MODE == M_BF16)
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int r = 0; r < RT; ++r) acc[i][r] = tot[i][r];
    if constexpr (KSP == 2) {
        // the halves exchange row tiles through the rings (free now): half h keeps tiles h RT / 2 .. + RT / 2 - 1
        __syncthreads();
        Acc* ex = reinterpret_cast<Acc*>(lds);
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int r = 0; r < RT; ++r)
                if (r / (RT / 2) != half) ex[((wave * NT + i) * RT + r) * 64 + lane] = acc[i][r];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int r = 0; r < RT; ++r)
                if (r / (RT / 2) == half) acc[i][r] += ex[((wave * NT + i) * RT + r) * 64 + lane];
    }
    auto mine = [&](int r) { return KSP == 1 || r / (RT / 2) == half; };  // (uniform)
    // epilogue: lane (row c of row tile r, columns 4 kq .. + 3 of each tile)
    auto sch4 = [&](int i, float (&f)[4]) {
        const float* s = mi[i] == 0 ? a.m[0].sch : (mi[i] == 1 ? a.m[1].sch : a.m[2].sch);
        const float4 v = *reinterpret_cast<const float4*>(s + tile[i] * 16 + 4 * kq);
        f[0] = v.x, f[1] = v.y, f[2] = v.z, f[3] = v.w;
    };
    auto pack = [](const uint16_t (&v)[4]) {
        return make_uint2(uint32_t(v[0]) | (uint32_t(v[1]) << 16), uint32_t(v[2]) | (uint32_t(v[3]) << 16));
    };
    if constexpr (MODE != M_BF16) {
        if (a.pair) {  // (uniform; NT == 2: tile 0 gate, tile 1 up)
            if (!live[0]) return;
            float sg[4], su[4];
            sch4(0, sg);
            sch4(1, su);
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                const int m = m0 + r * 16 + c;
                if (!mine(r) || m >= a.M) continue;
                const float xs = a.xs[m];
                uint16_t v[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint16_t g = f2bf(scaleback(acc[0][r][j], xs, sg[j])), u = f2bf(scaleback(acc[1][r][j], xs, su[j]));
                    v[j] = f2bf(__fmul_rn(bf2f(a.lut[g]), bf2f(u)));
                }
                *reinterpret_cast<uint2*>(static_cast<uint16_t*>(a.out[0]) + size_t(m) * a.m[0].n + tile[0] * 16 + 4 * kq) = pack(v);
            }
            return;
        }
    }
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        if (!live[i]) continue;
        float sc[4] = {0.f, 0.f, 0.f, 0.f};
        if constexpr (MODE != M_BF16) sch4(i, sc);
        const int n = mi[i] == 0 ? a.m[0].n : (mi[i] == 1 ? a.m[1].n : a.m[2].n);
        uint16_t* out = static_cast<uint16_t*>(mi[i] == 0 ? a.out[0] : (mi[i] == 1 ? a.out[1] : a.out[2]));
        const uint16_t* res = static_cast<const uint16_t*>(mi[i] == 0 ? a.res[0] : (mi[i] == 1 ? a.res[1] : a.res[2]));
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const int m = m0 + r * 16 + c;
            if (!mine(r) || m >= a.M) continue;
            const size_t o = size_t(m) * n + tile[i] * 16 + 4 * kq;
            uint16_t v[4];
            if constexpr (MODE == M_BF16) {
#pragma unroll
                for (int j = 0; j < 4; ++j) v[j] = f2bf(acc[i][r][j]);
            } else {
                const float xs = a.xs[m];
#pragma unroll
                for (int j = 0; j < 4; ++j) v[j] = f2bf(scaleback(acc[i][r][j], xs, sc[j]));
            }
            if (res) {
                const uint2 rv = *reinterpret_cast<const uint2*>(res + o);
                const uint16_t rb[4] = {uint16_t(rv.x), uint16_t(rv.x >> 16), uint16_t(rv.y), uint16_t(rv.y >> 16)};
#pragma unroll
                for (int j = 0; j < 4; ++j) v[j] = f2bf(__fadd_rn(bf2f(rb[j]), bf2f(v[j])));
            }
            *reinterpret_cast<uint2*>(out + o) = pack(v);
        }
    }
}

template <int MODE, int RT, int KSP>
int launch_gemm(GemmArgs& a, hipStream_t st) {
    constexpr int NT = 2;
    const void* fn = reinterpret_cast<const void*>(&gemm_kernel<MODE, RT, NT, KSP>);
    allow_smem(fn, Geo<MODE, RT, NT, KSP>::LDS);
    hipLaunchKernelGGL((gemm_kernel<MODE, RT, NT, KSP>), dim3(unsigned((a.NB + 7) / 8 * 8 * a.MB)), dim3(256 * KSP),
                       (Geo<MODE, RT, NT, KSP>::LDS), st, a);
    MDX_LAUNCHED();
    return MDX_OK;
}

template <int MODE>
int launch_rows(GemmArgs& a, hipStream_t st) {
    // 128 rows per work-group (each decodes its weights for all of its rows), 64 where that is all there are
    const int rt = a.M <= 64 ? 4 : 8;
    a.MB = (a.M + rt * 16 - 1) / (rt * 16);
    a.NB = (a.total + 7) / 8;
    if constexpr (MODE != M_BF16) {
        // at most one work-group per CU: a second set of four waves takes every other stage (two waves per SIMD, so the
        // decode of one overlaps the products of the other)
        if (a.MB * a.NB <= 256) return rt == 4 ? launch_gemm<MODE, 4, 2>(a, st) : launch_gemm<MODE, 8, 2>(a, st);
    }
    return rt == 4 ? launch_gemm<MODE, 4, 1>(a, st) : launch_gemm<MODE, 8, 1>(a, st);
}

int lg2(int64_t v) {
    int l = 0;
    while ((int64_t(1) << l) < v) ++l;
    return l;
}

bool w4_fits(const mdx_w4& w) {
    if (w.layout != MDX_LAYOUT_TILE || w.n <= 0 || w.n % 16 || w.k <= 0 || w.k % 128 || w.k > 65536 ||
        w.n * w.k / 2 >= (int64_t(1) << 31) || w.group_size < 16 || (w.group_size & (w.group_size - 1)) || w.k % w.group_size)
        return false;
    if (!aligned(w.q, 16) || !aligned(w.s_rel, 16) || !aligned(w.s_channel, 16)) return false;
    const int64_t ng = w.k / w.group_size;
    if (w.s_dtype == MDX_DT_F16) return w.group_size >= 128 && ng % 2 == 0;
    return w.s_dtype == MDX_DT_FP8E4M3 && ng % 8 == 0;
}

}  // namespace
}  // namespace mdx

using namespace mdx;

extern "C" int32_t mdx_w4a8_gemm_fits(const mdx_w4* w) { return w && w4_fits(*w) ? 1 : 0; }

extern "C" int mdx_w4a8_gemm(const int8_t* x, const float* x_scale, const mdx_w4* const* mats, int32_t nmats,
                             int32_t gate_up, uint16_t* const* outs, const uint16_t* const* residuals,
                             const uint16_t* silu_lut, int64_t rows, void* stream) {
    MDX_CHECK(x && x_scale && mats && outs, "null pointer");
    MDX_CHECK(nmats >= 1 && nmats <= 3, "1..3 matrices");
    MDX_CHECK(rows >= 1 && rows <= 65535, "rows must be in 1..65535");
    MDX_CHECK(!gate_up || (nmats == 2 && silu_lut && mats[0] && mats[1] && mats[0]->n == mats[1]->n && !residuals),
              "gate/up needs 2 matrices of one N, a SiLU table and no residual");
    GemmArgs a{};
    a.nm = nmats;
    a.pair = gate_up != 0;
    for (int i = 0; i < 3; ++i) {
        const mdx_w4* w = mats[i < nmats ? i : 0];
        MDX_CHECK(w && w->q && w->s_rel && w->s_channel && w4_fits(*w),
                  "weights: 16-byte aligned, tile-major codes, fp16 scales in groups >= 128 (an even count) or fp8 ones (a multiple of 8)");
        const mdx_w4* w0 = mats[0];
        MDX_CHECK(w->k == w0->k && w->group_size == w0->group_size && w->s_dtype == w0->s_dtype && w->codebook == w0->codebook,
                  "fused matrices must share K, group size, scale dtype and codebook");
        a.m[i] = GMat{reinterpret_cast<const uint8_t*>(w->q), reinterpret_cast<const uint8_t*>(w->s_rel), w->s_channel,
                      int(w->n), int(w->n / 16)};
        a.out[i] = outs[gate_up ? 0 : (i < nmats ? i : 0)];
        a.res[i] = residuals ? residuals[i < nmats ? i : 0] : nullptr;
        MDX_CHECK(a.out[i] && aligned(a.out[i], 8) && aligned(a.res[i], 8), "outputs / residuals: 8-byte aligned");
        if (i < nmats) a.total += int(w->n / 16);
    }
    const mdx_w4& w = *mats[0];
    MDX_CHECK(aligned(x, 16) && rows * w.k < (int64_t(1) << 31), "x: 16-byte aligned, below 2 GiB");
    a.steps = int(w.k / 128);
    a.kb = int(w.k);
    a.lgG = lg2(w.group_size);
    a.ng = int(w.k / w.group_size);
    a.cb = w.codebook;
    a.x = reinterpret_cast<const uint8_t*>(x);
    a.xs = x_scale;
    a.M = int(rows);
    a.lut = silu_lut;
    const hipStream_t st = static_cast<hipStream_t>(stream);
    return w.s_dtype == MDX_DT_F16 ? launch_rows<M_F16>(a, st) : launch_rows<M_FP8>(a, st);
}

extern "C" int mdx_bf16_gemm(const uint16_t* x, const uint16_t* w, uint16_t* out, int64_t rows, int64_t N, int64_t n0,
                             int64_t n1, int64_t K, void* stream) {
    MDX_CHECK(x && w && out, "null pointer");
    MDX_CHECK(rows >= 1 && rows <= 65535 && N % 16 == 0 && n0 % 16 == 0 && n1 % 16 == 0 && n0 >= 0 && n0 < n1 && n1 <= N &&
                  N < (int64_t(1) << 31) && K >= 64 && K % 64 == 0 && K <= 65536,
              "rows in 1..65535, columns [n0, n1) of N in steps of 16, K % 64 == 0");
    MDX_CHECK(aligned(x, 16) && aligned(w, 16) && aligned(out, 8) && rows * K < (int64_t(1) << 30),
              "16-byte aligned x / w, 8-byte aligned out, x below 2 GiB");
    GemmArgs a{};
    a.nm = 1;
    a.total = int((n1 - n0) / 16);
    for (int i = 0; i < 3; ++i) {
        a.m[i] = GMat{reinterpret_cast<const uint8_t*>(w + n0 * K), nullptr, nullptr, int(n1 - n0), a.total};
        a.out[i] = out;
    }
    a.steps = int(K / 64);
    // mdx_bf16_linear's K slices, so that the same rows give the same bits (slices of an odd number of 32-k chunks, which
    // no stage boundary meets: one sum over K)
    const int NC = int(K / 32), KS = bf16_kslices(int(N / 16), NC);
    a.slice = NC / KS % 2 == 0 ? NC / KS / 2 : a.steps;
    a.kb = int(K * 2);
    a.x = reinterpret_cast<const uint8_t*>(x);
    a.M = int(rows);
    return launch_rows<M_BF16>(a, static_cast<hipStream_t>(stream));
}
