// The Gated-DeltaNet core of a prompt prefill: the conv, the gates and the delta rule over a whole run of committed
// rows (a chain: each row's parent is the row before it), where the decode core (mdx_gdn.hip) takes at most 16 rows and
// replays them in the next step. Arithmetic and orders are the decode core's, so the state after the run and every
// output row are the bits that the same rows give it in chains of 16.
//
// Reference semantics (comfy-mono-decode-xpu): csrc/mono_gdn.sycl:313-374 (conv), :424-450 (gates), :398-571 (delta
// rule); buffers as in mdx_gdn.hip. The rows still pending from a decode step (ctl) are taken first: the conv history
// is shifted by them, the delta rule replays them. The run's own last rows may be left pending the same way: their
// outputs are computed, the states stop before them, and gdn_run_tail_kernel leaves their buffers for the next step.
#include "mdx_common.hpp"
#include "mdx_gdn_ops.hpp"

namespace mdx {
namespace {

constexpr int DH = GDN_DH, CW = GDN_CW;

struct RunArgs {
    const uint16_t* proj;    // [M, C] this run's projections
    const uint16_t* xn;      // [M, K]
    const uint16_t* wa;      // [HV, K]
    const uint16_t* wb;
    int K;
    const uint16_t* conv_w;  // [C, 4]
    uint16_t* conv_state;    // [C, 3]
    uint16_t* pb;            // [2][slots][C]: the pending rows before the run, the tail's after it
    uint16_t* qb;
    float* old_gates;        // [2][slots][HV][2]
    const int32_t* ctl;      // pending, parity, accepted slots ..
    const float* dt_bias;
    const float* g_decay;
    uint16_t* qkv;           // [M, C] conv outputs
    float* gates;            // [M, HV, 2]
    float* rec;              // [HV][128][128]
    uint16_t* core;          // [M, HV * 128]
    float qscale;
    int M, HK, HV, C, slots, nconv;
    int commit, tail_parity; // rows whose state is kept (the rest: the tail), the tail's buffers
};

// The control words that a launch takes (uniform in the wave, by every lane's loads): the pending rows' count and parity,
// and each pending row's slot. One rule for the three kernels, so that invalid words leave every output alone.
__device__ __forceinline__ bool run_ctl_ok(const RunArgs& a) {
    const int pending = a.ctl[0], lane = threadIdx.x & 63;
    if (!gdn_ctl_ok(pending, a.ctl[1], a.slots)) return false;
    const int sl = lane < pending ? a.ctl[2 + lane] : 0;
    return __builtin_amdgcn_ballot_w64(sl < 0 || sl >= a.slots) == 0;
}

constexpr int CR = 16;  // rows per conv work-group (their taps reach 3 rows back)
constexpr int GR = 16;  // rows per gate wave

// Work-groups [0, nconv): 512 channels x CR rows of the conv, two channels per thread. The others: four waves, each
// the gates of one head for GR rows, the head's a / b weights held in registers (gdn_gate_row's sums in its order).
__global__ __launch_bounds__(256) void gdn_run_prep_kernel(RunArgs a) {
    const int t = threadIdx.x;
    if (!run_ctl_ok(a)) return;  // (uniform)
    if (int(blockIdx.x) < a.nconv) {
        const int cb = a.C / 512, c = (blockIdx.x % cb) * 512 + 2 * t, r0 = (blockIdx.x / cb) * CR;
        const int pending = a.ctl[0], p = a.ctl[1], S = a.slots;
        auto row = [&](int r) { return *reinterpret_cast<const uint32_t*>(a.proj + size_t(r) * a.C + c); };
        uint32_t tap[CW];  // the rows before r0, oldest first
        if (r0 == 0) {
            // the history: conv_state shifted by the pending rows
#pragma unroll
            for (int i = 0; i < CW; ++i) {
                const int j = pending + i;
                const int slot = a.ctl[2 + (j < CW ? 0 : j - CW)];
                if (j < CW)
                    tap[i] = uint32_t(a.conv_state[c * CW + j]) | (uint32_t(a.conv_state[(c + 1) * CW + j]) << 16);
                else
                    tap[i] = *reinterpret_cast<const uint32_t*>(a.pb + size_t((1 - p) * S + slot) * a.C + c);
            }
        } else {
#pragma unroll
            for (int i = 0; i < CW; ++i) tap[i] = row(r0 - CW + i);
        }
        float w[2][CW + 1];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int d = 0; d <= CW; ++d) w[h][d] = bf2f(a.conv_w[(c + h) * (CW + 1) + d]);
        uint32_t in[CR];
#pragma unroll
        for (int i = 0; i < CR; ++i) in[i] = row(min(r0 + i, a.M - 1));
#pragma unroll
        for (int i = 0; i < CR; ++i) {
            if (r0 + i >= a.M) break;
            uint32_t o = 0;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                auto val = [&](uint32_t v) { return __uint_as_float(h ? (v & 0xFFFF0000u) : (v << 16)); };
                float sum = fmaf(val(in[i]), w[h][CW], 0.f);
#pragma unroll
                for (int d = 1; d <= CW; ++d) sum = fmaf(val(i >= d ? in[i >= d ? i - d : 0] : tap[CW + i - d < 0 ? 0 : (CW + i - d) % CW]), w[h][CW - d], sum);
                const float y = bfround(sum);
                o |= uint32_t(f2bf(__fdiv_rn(y, __fadd_rn(1.f, expf(-y))))) << (16 * h);
            }
            *reinterpret_cast<uint32_t*>(a.qkv + size_t(r0 + i) * a.C + c) = o;
        }
        return;
    }
    const int lane = t & 63, id = (int(blockIdx.x) - a.nconv) * 4 + (t >> 6);
    const int h = id % a.HV, r0 = (id / a.HV) * GR;
    if (r0 >= a.M) return;
    const int nb = a.K / 8;
    uint4 av[8], bv[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int b = lane + 64 * j < nb ? lane + 64 * j : 0;
        av[j] = *reinterpret_cast<const uint4*>(a.wa + size_t(h) * a.K + 8 * b);
        bv[j] = *reinterpret_cast<const uint4*>(a.wb + size_t(h) * a.K + 8 * b);
    }
    const float dt = a.dt_bias[h], gd = a.g_decay[h];
    for (int r = r0; r < min(r0 + GR, a.M); ++r) {
        uint4 xv[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)
            xv[j] = *reinterpret_cast<const uint4*>(a.xn + size_t(r) * a.K + 8 * (lane + 64 * j < nb ? lane + 64 * j : 0));
        float pa = 0.f, pb = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            if (lane + 64 * j >= nb) continue;
            const uint32_t xw[4] = {xv[j].x, xv[j].y, xv[j].z, xv[j].w}, aw[4] = {av[j].x, av[j].y, av[j].z, av[j].w},
                           bw[4] = {bv[j].x, bv[j].y, bv[j].z, bv[j].w};
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                auto val = [&](uint32_t v) { return __uint_as_float((e & 1) ? (v & 0xFFFF0000u) : (v << 16)); };
                const float xe = val(xw[e >> 1]);
                pa = fmaf(xe, val(aw[e >> 1]), pa);
                pb = fmaf(xe, val(bw[e >> 1]), pb);
            }
        }
        pa = tree_sum64(pa);
        pb = tree_sum64(pb);
        const float avv = __fadd_rn(bfround(pa), dt);
        const float sp = avv > 20.f ? avv : log1pf(expf(avv));
        const float decay = expf(__fmul_rn(gd, sp));
        const float beta = bfround(__fdiv_rn(1.f, __fadd_rn(1.f, expf(-bfround(pb)))));
        if (lane == 0) *reinterpret_cast<float2*>(a.gates + (size_t(r) * a.HV + h) * 2) = make_float2(decay, beta);
    }
}

// The delta rule over the run: work-group (value head h, 16 state columns), thread (row group rg, column) as in
// gdn_head_kernel. The rows come in blocks of 16: thread t holds piece t % 16 (8 elements) of row t / 16's k and q, so
// the norms and k . q are sums over 16 lanes (halving trees) and the scaled rows go to LDS, double-buffered: the block
// after next is in flight from memory while the waves walk one. Bound by the serial walk, 0.27 us a row
// (1000 rows 274 us).
constexpr int SC = 16, RG = 8, EB = 16;

__device__ __forceinline__ float ror4_sum(float v) {
    return __fadd_rn(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x124, 0xF, 0xF, false)));
}
__device__ __forceinline__ float column_sum(float v) { return sum_x32(sum_x16(ror4_sum(sum_x8(v)))); }
__device__ __forceinline__ float tree16(float v) {
#pragma unroll
    for (int d = 8; d >= 1; d >>= 1) v = __fadd_rn(v, __shfl_xor(v, d, 16));
    return v;
}

__global__ __launch_bounds__(256) void gdn_run_delta_kernel(RunArgs a) {
    __shared__ __align__(16) float kvec[2][EB][DH], qvec[2][EB][DH];
    __shared__ float vvec[2][EB][SC];
    __shared__ float4 scal[2][EB];  // decay, beta, k . q
    const int t = threadIdx.x, lane = t & 63, h = blockIdx.x / (DH / SC), cs = blockIdx.x % (DH / SC);
    const int S = a.slots, KD = a.HK * DH, kh = h / (a.HV / a.HK);
    const int pending = a.ctl[0], p = a.ctl[1];
    if (!run_ctl_ok(a)) return;  // (uniform)
    const int col = (t >> 6) * 4 + (lane & 3), rg = lane >> 2;
    float st[RG];
    float* rs = a.rec + (size_t(h) * DH + rg * RG) * DH + cs * SC + col;
#pragma unroll
    for (int r = 0; r < RG; ++r) st[r] = rs[r * DH];
    // the conv history after the run: its last three committed rows (the conv kernel of this run has read the old one)
    if (int(blockIdx.x) * 256 + t < a.C) {
        const int c = blockIdx.x * 256 + t;
#pragma unroll
        for (int i = 0; i < CW; ++i) a.conv_state[c * CW + i] = a.proj[size_t(a.commit - CW + i) * a.C + c];
    }
    // blocks: the pending rows, the committed ones, the tail
    const int nr = pending > 0 ? 1 : 0, nc = (a.commit + EB - 1) / EB, nblk = nr + nc + (a.M - a.commit + EB - 1) / EB;
    struct Raw {
        uint4 k, q, v;
        float2 g;
    };
    auto row0 = [&](int b) { return b - nr < nc ? (b - nr) * EB : a.commit + (b - nr - nc) * EB; };
    auto rows_of = [&](int b) { return b < nr ? pending : min(EB, (b - nr < nc ? a.commit : a.M) - row0(b)); };
    auto load = [&](int b, Raw& w) {
        const int n = rows_of(b), e = min(t >> 4, n - 1), e2 = min(t >> 1, n - 1);
        auto base = [&](int e_) {
            return b < nr ? a.qb + size_t((1 - p) * S + a.ctl[2 + e_]) * a.C : a.qkv + size_t(row0(b) + e_) * a.C;
        };
        const uint16_t* row = base(e) + kh * DH + (t & 15) * 8;
        w.q = *reinterpret_cast<const uint4*>(row);
        w.k = *reinterpret_cast<const uint4*>(row + KD);
        const bool vt = t < 2 * EB;  // (the first lanes: 2 pieces of the 16 columns per row)
        w.v = vt ? *reinterpret_cast<const uint4*>(base(e2) + 2 * KD + h * DH + cs * SC + (t & 1) * 8) : make_uint4(0u, 0u, 0u, 0u);
        const float* gt = b < nr ? a.old_gates + (size_t((1 - p) * S + a.ctl[2 + e]) * a.HV + h) * 2
                                 : a.gates + (size_t(row0(b) + e) * a.HV + h) * 2;
        w.g = *reinterpret_cast<const float2*>(gt);
    };
    auto prep = [&](int buf, const Raw& w) {
        auto el = [](const uint4& v, int i) {
            const uint32_t u[4] = {v.x, v.y, v.z, v.w};
            return __uint_as_float((i & 1) ? (u[i >> 1] & 0xFFFF0000u) : (u[i >> 1] << 16));
        };
        float kk = 0.f, qq = 0.f, kq = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            kk = fmaf(el(w.k, i), el(w.k, i), kk);
            qq = fmaf(el(w.q, i), el(w.q, i), qq);
            kq = fmaf(el(w.k, i), el(w.q, i), kq);
        }
        kk = tree16(kk);
        qq = tree16(qq);
        kq = tree16(kq);
        const float ki = __fdiv_rn(1.f, fmaxf(sqrt_rn(kk), 1e-12f)), qi = __fdiv_rn(1.f, fmaxf(sqrt_rn(qq), 1e-12f));
        const int e = t >> 4, d0 = (t & 15) * 8;
        float4 ko[2], qo[2];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            reinterpret_cast<float*>(ko)[i] = __fmul_rn(el(w.k, i), ki);
            reinterpret_cast<float*>(qo)[i] = __fmul_rn(__fmul_rn(el(w.q, i), a.qscale), qi);
        }
        float4* kd = reinterpret_cast<float4*>(&kvec[buf][e][d0]);
        float4* qd = reinterpret_cast<float4*>(&qvec[buf][e][d0]);
        kd[0] = ko[0], kd[1] = ko[1];
        qd[0] = qo[0], qd[1] = qo[1];
        if ((t & 15) == 0) scal[buf][e] = make_float4(w.g.x, w.g.y, __fmul_rn(__fmul_rn(kq, ki), __fmul_rn(a.qscale, qi)), 0.f);
        if (t < 2 * EB)
#pragma unroll
            for (int i = 0; i < 8; ++i) vvec[buf][t >> 1][(t & 1) * 8 + i] = el(w.v, i);
    };
    auto load8 = [&](const float* src, float (&r8)[RG]) {
        const float4* p4 = reinterpret_cast<const float4*>(src + rg * RG);
        const float4 x0 = p4[0], x1 = p4[1];
        r8[0] = x0.x, r8[1] = x0.y, r8[2] = x0.z, r8[3] = x0.w, r8[4] = x1.x, r8[5] = x1.y, r8[6] = x1.z, r8[7] = x1.w;
    };
    auto dot_col = [&](const float (&r8)[RG]) {
        float m4[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) m4[r] = __fmul_rn(st[r], r8[r]);
#pragma unroll
        for (int r = 4; r < RG; ++r) m4[r & 3] = fmaf(st[r], r8[r], m4[r & 3]);
        return column_sum(__fadd_rn(__fadd_rn(m4[0], m4[1]), __fadd_rn(m4[2], m4[3])));
    };
    Raw raw;
    load(0, raw);
    prep(0, raw);
    load(min(1, nblk - 1), raw);
    __syncthreads();
    for (int b = 0; b < nblk; ++b) {
        const int buf = b & 1, n = rows_of(b);
        if (b == nr + nc)  // (uniform) the tail follows: the state to keep
#pragma unroll
            for (int r = 0; r < RG; ++r) rs[r * DH] = st[r];
        prep(buf ^ 1, raw);                // block b + 1 (its buffer was last read before the barrier)
        load(min(b + 2, nblk - 1), raw);
        float held = 0.f;
        float kA[RG], kB[RG], qA[RG], qB[RG], vv;
        float4 g;
        load8(kvec[buf][0], kA);
        load8(qvec[buf][0], qA);
        vv = vvec[buf][0][col], g = scal[buf][0];
        auto entry = [&](int e, const float (&kc)[RG], const float (&qc)[RG], float (&kn)[RG], float (&qn)[RG]) {
            const int en = min(e + 1, n - 1);
            load8(kvec[buf][en], kn);
            load8(qvec[buf][en], qn);
            const float vn = vvec[buf][en][col];
            const float4 gn = scal[buf][en];
            const float ks = dot_col(kc), qs = dot_col(qc);
            const float delta = __fmul_rn(__fsub_rn(vv, __fmul_rn(g.x, ks)), g.y);
            const float o = fmaf(delta, g.z, __fmul_rn(g.x, qs));
            held = e == rg ? o : held;
#pragma unroll
            for (int r = 0; r < RG; ++r) st[r] = fmaf(kc[r], delta, __fmul_rn(st[r], g.x));
            vv = vn, g = gn;
        };
        for (int e = 0; e < n; e += 2) {
            entry(e, kA, qA, kB, qB);
            if (e + 1 < n) entry(e + 1, kB, qB, kA, qA);
        }
        // row e's output of the column is held by row group e
        if (b >= nr && rg < n) a.core[(size_t(row0(b) + rg) * a.HV + h) * DH + cs * SC + col] = f2bf(held);
        __syncthreads();
    }
    if (nblk == nr + nc)
#pragma unroll
        for (int r = 0; r < RG; ++r) rs[r * DH] = st[r];
}

// The tail rows' projections, conv outputs and gates into the buffers of their parity, zeros past them (a launch of its
// own: the delta rule's replay may still read the same parity).
__global__ __launch_bounds__(256) void gdn_run_tail_kernel(RunArgs a) {
    const int tail = a.M - a.commit, S = a.slots, p = a.tail_parity;
    if (!run_ctl_ok(a)) return;  // (uniform)
    const int ng = a.HV * 2, per = a.C / 8;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < S * per; i += gridDim.x * 256) {
        const int r = i / per, c = (i % per) * 8;
        const uint4 z = make_uint4(0u, 0u, 0u, 0u);
        const size_t src = size_t(a.commit + r) * a.C + c, dst = size_t(p * S + r) * a.C + c;
        *reinterpret_cast<uint4*>(a.pb + dst) = r < tail ? *reinterpret_cast<const uint4*>(a.proj + src) : z;
        *reinterpret_cast<uint4*>(a.qb + dst) = r < tail ? *reinterpret_cast<const uint4*>(a.qkv + src) : z;
    }
    for (int i = blockIdx.x * 256 + threadIdx.x; i < S * ng; i += gridDim.x * 256)
        a.old_gates[p * S * ng + i] = i < tail * ng ? a.gates[size_t(a.commit) * ng + i] : 0.f;
}

}  // namespace
}  // namespace mdx

using namespace mdx;

extern "C" int mdx_gdn_run(const uint16_t* proj, const uint16_t* xn, const uint16_t* wa, const uint16_t* wb, int64_t K,
                           const uint16_t* conv_w, uint16_t* conv_state, uint16_t* proj_buf, uint16_t* qkv_buf,
                           float* gates_buf, const int32_t* ctl, const float* dt_bias, const float* g_decay,
                           float* rec_state, float qscale, uint16_t* qkv, float* gates, uint16_t* core, int64_t rows,
                           int64_t tail, int32_t tail_parity, int64_t HK, int64_t HV, int64_t slots, void* stream) {
    MDX_CHECK(proj && xn && wa && wb && conv_w && conv_state && proj_buf && qkv_buf && gates_buf && ctl && dt_bias &&
                  g_decay && rec_state && qkv && gates && core,
              "null pointer");
    MDX_CHECK(slots == 8 || slots == 16, "slots must be 8 or 16");
    MDX_CHECK(tail >= 0 && tail <= slots && (tail_parity == 0 || tail_parity == 1) && rows - tail >= GDN_CW && rows <= 65535,
              "at least 3 committed rows, at most slots pending ones, 65535 in all");
    MDX_CHECK(HK >= 1 && HV >= HK && HV % HK == 0 && HV <= 128 && (2 * HK + HV) % 4 == 0, "heads (2 HK + HV a multiple of 4, HV <= 128)");
    MDX_CHECK(K >= 512 && K <= 4096 && K % 512 == 0 && aligned(xn, 16) && aligned(wa, 16) && aligned(wb, 16) &&
                  aligned(proj, 16) && aligned(qkv, 16) && aligned(proj_buf, 16) && aligned(qkv_buf, 16) && aligned(gates, 8) &&
                  aligned(gates_buf, 8),
              "a / b input: K % 512 == 0, K <= 4096, 16-byte aligned rows");
    RunArgs a{};
    a.proj = proj;
    a.xn = xn;
    a.wa = wa;
    a.wb = wb;
    a.K = int(K);
    a.conv_w = conv_w;
    a.conv_state = conv_state;
    a.pb = proj_buf;
    a.qb = qkv_buf;
    a.old_gates = gates_buf;
    a.ctl = ctl;
    a.dt_bias = dt_bias;
    a.g_decay = g_decay;
    a.qkv = qkv;
    a.gates = gates;
    a.rec = rec_state;
    a.core = core;
    a.qscale = qscale;
    a.M = int(rows);
    a.commit = int(rows - tail);
    a.tail_parity = tail_parity;
    a.HK = int(HK);
    a.HV = int(HV);
    a.C = int((2 * HK + HV) * GDN_DH);
    a.slots = int(slots);
    a.nconv = (a.C / 512) * ((a.M + CR - 1) / CR);
    const int ngate = (a.HV * ((a.M + GR - 1) / GR) + 3) / 4;
    const hipStream_t st = static_cast<hipStream_t>(stream);
    hipLaunchKernelGGL(gdn_run_prep_kernel, dim3(unsigned(a.nconv + ngate)), dim3(256), 0, st, a);
    MDX_LAUNCHED();
    hipLaunchKernelGGL(gdn_run_delta_kernel, dim3(unsigned(a.HV * (DH / SC))), dim3(256), 0, st, a);
    MDX_LAUNCHED();
    if (tail > 0) {
        hipLaunchKernelGGL(gdn_run_tail_kernel, dim3(unsigned((a.slots * (a.C / 8) + 255) / 256)), dim3(256), 0, st, a);
        MDX_LAUNCHED();
    }
    return MDX_OK;
}
