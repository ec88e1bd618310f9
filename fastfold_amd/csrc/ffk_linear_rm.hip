// Weights-in-registers variant of the fused linear layer for row-major operands (see ffk_fused_linear in include/ffk.h),
// bf16, K = 64, 128 or 256: the projections of the MSA, pair, extra-MSA and template stacks and of their backward passes.
//
// A workgroup keeps the MFMA fragments of its weight units (32 output rows each, one or two per wave) in registers; rows of A
// stream through a double-buffered slab in LDS: global -> registers -> (LayerNorm in registers) -> LDS, the loads of slab i + 1
// in flight while slab i is multiplied.  Each wave multiplies 32-row groups of the slab against its own units and finishes the
// 32 x 32 blocks straight from the accumulators - bias, activation, GLU, row mask, gate, residual - and stores them:
//   by rows  (plain [row][channel] outputs, q / k / gate tiles): product W . A^T, a lane owns one row and 16 channels
//   by cols  (v tiles, channel-major outputs): product A . W^T, a lane owns one channel and 16 rows
//
// What bounds it: a 32 x 32 block costs K / 16 matrix instructions of 32 cycles, and a vector instruction costs a SIMD 4 cycles
// that no matrix instruction of it overlaps with.  So the loop is arranged for few vector instructions per block: the position
// of a group in its output is scalar arithmetic (a multiplication by a reciprocal) and a store takes a scalar base and a 32-bit
// lane offset fixed for the launch; what a unit's epilogue needs fits 48 bytes, so that of both units of a wave stays in scalar
// registers; two units of a wave share the fragments of a row group (K <= 128), which are requested one step ahead.
#include "ffk_common.h"
#include <type_traits>

namespace {

typedef bf16_t T;

constexpr int RM_MAX_SLOTS = 32;

// Per-K geometry: a slab is as many rows as the threads fetch with NP 16-byte loads each.
template <int K, int WAVES, int NP> struct RmGeo {
    static constexpr int THREADS = 64 * WAVES;
    static constexpr int KS = K / 16;                // MFMA K steps
    static constexpr int AP = K * 2 + 16;            // LDS row pitch in bytes
    static constexpr int LPR = K / 8;                // lanes (16-byte vectors) per row
    static constexpr int RPP = THREADS / LPR;        // rows fetched per pass
    static constexpr int BM = NP * RPP;              // rows per slab
    static constexpr int RG = BM / 32;               // 32-row groups per slab
    static constexpr int STAGE = WAVES * 32 * (K < 128 ? K : 128) * 2;
    static constexpr int SLABS = 2 * BM * AP > STAGE ? 2 * BM * AP : STAGE;    // bytes of the double-buffered slab, first the staging area of the weights
};

// Exact quotients of 32-bit numbers by a fixed divisor: n / d = (mulhi(n, mul) + n) >> shift for n < 2^31.
struct RmDiv {
    unsigned mul, shift, d;
};

// A weight slot: 32 rows of the weights and what their epilogue needs; channel offsets of the unit are folded into the pointers.
struct RmSlot {
    T* out;
    const T* bias;           // of the slot's 32 rows, or nullptr
    int s_o, s_i, s_d;
    int wrow;                // first weight row of the slot, -1 = unused
    int ncols_left;          // valid channels from the slot's first output channel on
    float scale;
    signed char kind, act;
    signed char glu;         // 0 plain, 1 value half of a GLU unit (gate half in the next slot), 2 gate half
    unsigned char flags;     // RM_*
    int pad;
};
enum { RM_MASKED = 1, RM_BIAS = 2, RM_ROWS = 4, RM_TAU = 8, RM_SIG = 16 };
struct RmRes {               // operands of the residual epilogues
    const T* resid;
    const T* gate;
    int8_t* xtail;           // tail bytes of resid / out as an extended residual stream, or nullptr
    int gate_ld;
    int gate_periodic;       // the gate's row is m % gate_rows
    RmDiv gate_rows;
    int pad;
};

struct RmCommon {
    const T* a;
    const T* w;
    const T* ln_gamma;
    const T* ln_beta;
    const T* rowmask;        // row mask of the launch (all masked tiles share it), or nullptr
    int a_so, a_si;
    int m_so, m_si;
    int M;
    RmDiv a_div;             // rows of A per outer step
    RmDiv inner;             // rows per outer step of all outputs
    int a_flat, flat;        // every row lies in the first outer step
    float ln_eps;
    int row_perm;            // rows of a group are read through tau (launch has channel-major tiles)
    int rg_step;             // a wave takes the row groups (wave / (WAVES / rg_step)) + i * rg_step of a slab
    // trailing FFK_TILE_BIAS tile (<= 4 heads, K = 128), pb_heads = 0: none.  It takes no weight slot - its few dot products per row
    // are 16 x 16 x 32 MFMAs on the slab in LDS
    int pb_heads, pb_wrow;
    unsigned pb_inner;
    T* pb_out;
    int pb_so, pb_sh;
    float pb_scale;
};
template <bool RES> struct RmArgs : RmCommon {
    RmSlot slot[RM_MAX_SLOTS];       // [column group][wave][slot]
};
template <> struct RmArgs<true> : RmCommon {
    RmSlot slot[RM_MAX_SLOTS];
    RmRes res[RM_MAX_SLOTS];
};
static_assert(sizeof(RmArgs<true>) <= 4096, "kernel arguments");

__device__ __forceinline__ unsigned rm_quot(const RmDiv& q, unsigned n) { return (__umulhi(n, q.mul) + n) >> q.shift; }

// sigmoid(acc + b) with the bias table entry pre-multiplied:  bs = -log2(e) * b
__device__ __forceinline__ float rm_sigmoid_pre(float acc, float bs) {
    return fast_rcp(1.0f + fast_exp2(__builtin_fmaf(acc, -1.4426950408889634f, bs)));
}

__host__ __device__ __forceinline__ bool rm_by_rows(const ffk_tile& t) {
    return t.kind == FFK_TILE_QK || t.kind == FFK_TILE_ACC || (t.kind == FFK_TILE_STRIDED && t.s_d == 1);
}

__device__ __forceinline__ uint32_t rm_pack2(float a, float b) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    const bf16x2 v = {(T)a, (T)b};
    return __builtin_bit_cast(uint32_t, v);
}
__device__ __forceinline__ float rm_lo(uint32_t v) { return __builtin_bit_cast(float, v << 16); }
__device__ __forceinline__ float rm_hi(uint32_t v) { return __builtin_bit_cast(float, v & 0xFFFF0000u); }

// ---- accumulators -> sixteen rounded values of a lane, packed in eight words ------------------------------------------
// Every combination of bias / activation / scale is its own straight-line path to the packed words: fp32 intermediates that
// outlive a branch make the compiler copy sixteen registers where the paths join, and the time of these kernels follows their
// vector instruction count.
// sb: this slot's 32 (GLU: and its gate's) bias values in LDS (fp32).
// by rows: registers hold channels 16 half + v (STRIDED, weight rows through tau) or 8a + 4 half + b (ACC, QK)
template <bool GLU>
__device__ __forceinline__ void rm_value_rows(const RmSlot& t, const f32x16& acc, const f32x16& accg, const float* sb, float rmask,
                                              int half, u32x4 (&y)[2]) {
    const bool scaled = (t.flags & RM_MASKED) || t.scale != 1.0f;
    const float scl = t.scale * rmask;
    const float* sl = sb + ((t.flags & RM_TAU) ? 16 * half : 4 * half);
    const int step = (t.flags & RM_TAU) ? 4 : 8;
    auto emit = [&](auto value) __attribute__((always_inline)) {        // value(v, bias of v, gate bias of v)
        if (scaled) {
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                const f32x4 b = *reinterpret_cast<const f32x4*>(sl + a * step), g = GLU ? *reinterpret_cast<const f32x4*>(sl + 32 + a * step) : b;
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    y[a >> 1][2 * (a & 1) + j] = rm_pack2(value(4 * a + 2 * j, b[2 * j], g[2 * j]) * scl, value(4 * a + 2 * j + 1, b[2 * j + 1], g[2 * j + 1]) * scl);
            }
        } else {
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                const f32x4 b = *reinterpret_cast<const f32x4*>(sl + a * step), g = GLU ? *reinterpret_cast<const f32x4*>(sl + 32 + a * step) : b;
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    y[a >> 1][2 * (a & 1) + j] = rm_pack2(value(4 * a + 2 * j, b[2 * j], g[2 * j]), value(4 * a + 2 * j + 1, b[2 * j + 1], g[2 * j + 1]));
            }
        }
    };
    if (GLU) emit([&](int v, float b, float g) { return (acc[v] + b) * rm_sigmoid_pre(accg[v], g); });
    else if (t.act == FFK_ACT_SIGMOID) emit([&](int v, float b, float) { return rm_sigmoid_pre(acc[v], b); });
    else if (t.act == FFK_ACT_RELU) emit([&](int v, float b, float) { return relu_f(acc[v] + b); });
    else if (t.flags & RM_BIAS) emit([&](int v, float b, float) { return acc[v] + b; });
    else emit([&](int v, float, float) { return acc[v]; });
}
// by cols: a lane's channel is l32; registers hold rows 8a + 4 half + b of the group (V) or 16 half + v (rows through tau).
// sm: mask values (fp32, LDS) of the group's 32 rows, or nullptr.
template <bool GLU>
__device__ __forceinline__ void rm_value_cols(const RmSlot& t, const f32x16& acc, const f32x16& accg, const float* sb, const float* sm,
                                              int l32, int half, u32x4 (&y)[2]) {
    const float b = sb[l32], g = GLU ? sb[32 + l32] : 0.0f;
    // the mask multiply is skipped for row groups without a masked row (the common case); V tiles have no mask here: their rows
    // lie in another order, and carrying both costs every variant five to ten more spilled scalar registers
    const bool masked = sm && __builtin_amdgcn_ballot_w64(sm[l32] != 1.0f) != 0;
    auto emit = [&](auto value) __attribute__((always_inline)) {
        if (masked || t.scale != 1.0f) {
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                f32x4 k = {1.0f, 1.0f, 1.0f, 1.0f};
                if (masked) k = *reinterpret_cast<const f32x4*>(sm + 16 * half + 4 * a);
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    y[a >> 1][2 * (a & 1) + j] = rm_pack2(value(4 * a + 2 * j) * k[2 * j] * t.scale, value(4 * a + 2 * j + 1) * k[2 * j + 1] * t.scale);
            }
        } else {
#pragma unroll
            for (int v = 0; v < 16; v += 2) y[v >> 3][(v >> 1) & 3] = rm_pack2(value(v), value(v + 1));
        }
    };
    if (GLU) emit([&](int v) { return (acc[v] + b) * rm_sigmoid_pre(accg[v], g); });
    else if (t.act == FFK_ACT_SIGMOID) emit([&](int v) { return rm_sigmoid_pre(acc[v], b); });
    else if (t.act == FFK_ACT_RELU) emit([&](int v) { return relu_f(acc[v] + b); });
    else emit([&](int v) { return acc[v] + b; });
}

constexpr bool rm_takes_bias(int K, bool res, bool uni) { return !res && K == 128 && uni; }

// UNI: 32-row groups lie inside one outer step of the outputs (inner % 32 == 0, or one step only)
template <int K, int NS, int WAVES, int NP, bool RES, bool XT, bool UNI, int OCC>
__global__ __launch_bounds__(64 * WAVES, OCC) void linear_rm_kernel(const RmArgs<RES> args) {
    typedef Mma<T> MM;
    typedef RmGeo<K, WAVES, NP> G;
    constexpr int KS = G::KS, AP = G::AP, BM = G::BM, RG = G::RG, LPR = G::LPR, RPP = G::RPP, THREADS = G::THREADS;
    constexpr int CH = K == 256 && NS == 2 ? 2 : 4;              // fragments are taken in chunks of CH
    constexpr int KC = KS / CH;
    constexpr bool PB = rm_takes_bias(K, RES, UNI);              // variants that take a trailing pair-bias tile
    constexpr bool SHARE = K <= 128;                             // two slots at a time; at K = 256 their weights leave no room for it
    const RmArgs<RES>& d = args;
    extern __shared__ __align__(16) unsigned char smem[];
    unsigned char* s_a = smem;                                                  // [2][BM][AP]
    float* s_mask = reinterpret_cast<float*>(smem + G::SLABS);                  // [2][BM]
    float* s_bias = s_mask + 2 * BM;                                            // [WAVES][NS][32]
    T* s_wb = reinterpret_cast<T*>(s_bias + WAVES * NS * 32);                   // PB: [4][K] head weights
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    const int M = d.M;
    const T* A = d.a;
    const T* W = d.w;

    RmSlot sp[NS];
    bf16x8 wf[NS][KS];
    const int slot0 = ((int)blockIdx.y * WAVES + wave) * NS;
#pragma unroll
    for (int s = 0; s < NS; ++s) sp[s] = args.slot[slot0 + s];
    const int n32 = d.row_perm ? ffk_tau(l32) : l32;

    // ---- slab streaming: thread -> (row tid / LPR + RPP * i, 8 channels starting at 8 * (tid % LPR)) ----
    const int c8 = tid % LPR, r0 = tid / LPR;
    const bool ln = d.ln_gamma != nullptr;
    const T* rm = d.rowmask;
    Vec16<T> pre[NP];
    T pm = (T)1.0f;
    auto fetch = [&](int slab) __attribute__((always_inline)) {                         // rows past the end are clamped: never stored
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            int m = slab * BM + r0 + RPP * i;
            m = m < M ? m : M - 1;
            const unsigned hi = d.a_flat ? 0u : rm_quot(d.a_div, (unsigned)m), lo = (unsigned)m - hi * d.a_div.d;
            pre[i] = ld16(A + (long)hi * d.a_so + (long)lo * d.a_si + c8 * 8);
        }
        if (rm && tid < BM) {
            int m = slab * BM + tid;
            m = m < M ? m : M - 1;
            const unsigned mh = d.flat ? 0u : rm_quot(d.inner, (unsigned)m), ml = (unsigned)m - mh * d.inner.d;
            pm = rm[(long)mh * d.m_so + (long)ml * d.m_si];
        }
    };
    const int nslabs = (M + BM - 1) / BM;
    int slab = blockIdx.x;                               // grid.x <= nslabs
    fetch(slab);                                         // the first slab travels while the weights are fetched

    // ---- weights: every wave reads the 32 rows of its slots as whole lines (a lane's fragments are 16-byte pieces 32 bytes
    // apart in one row, 32 rows per request: fetched that way every request touches 32 lines and uses a quarter of each) and
    // re-orders them through a private piece of the slab buffer, which is idle until the first commit.  A piece is 32 rows x PW
    // channels; its 16-byte chunks are stored at chunk ^ (row % LR) so that the fragment reads spread over the banks.
    Vec16<T> gam, bet;
    {
        constexpr int PW = K < 128 ? K : 128;            // channels per piece
        constexpr int LR = PW / 8;                       // 16-byte chunks (lanes) per row of a piece
        constexpr int NI = 32 / (64 / LR);               // requests per piece = K steps per piece
        constexpr int NPC = K / PW;                      // pieces per slot
        static_assert(NI * NPC == KS, "piece geometry");
        static_assert(WAVES * 32 * PW * 2 <= G::SLABS, "the staging area is the slab buffer");
        unsigned char* stage = s_a + wave * (32 * PW * 2);
        const int lrow = lane / LR, lcol = lane % LR;
#pragma unroll
        for (int sl = 0; sl < NS; ++sl) {
            const T* wp = W + (long)(sp[sl].wrow >= 0 ? sp[sl].wrow : 0) * K + lrow * K + lcol * 8;
#pragma unroll
            for (int pc = 0; pc < NPC; ++pc)
#pragma unroll
                for (int i = 0; i < NI; ++i) wf[sl][pc * NI + i] = MM::ld(wp + i * (64 / LR) * K + pc * PW);
        }
        float tb[NS];
#pragma unroll
        for (int sl = 0; sl < NS; ++sl) tb[sl] = sp[sl].wrow >= 0 && sp[sl].bias ? (float)sp[sl].bias[l32] : 0.0f;
        if (ln) {
            gam = ld16(d.ln_gamma + c8 * 8);
            bet = ld16(d.ln_beta + c8 * 8);
        }
        constexpr int NW = PB ? 4 * K / THREADS : 1;     // head weights per thread
        T tw[NW];
#pragma unroll
        for (int i = 0; i < NW; ++i) {
            tw[i] = (T)0.0f;
            if (PB && tid + i * THREADS < d.pb_heads * K) tw[i] = W[(long)d.pb_wrow * K + tid + i * THREADS];
        }
#pragma unroll
        for (int sl = 0; sl < NS; ++sl)
#pragma unroll
            for (int pc = 0; pc < NPC; ++pc) {
#pragma unroll
                for (int i = 0; i < NI; ++i) {
                    const int row = i * (64 / LR) + lrow;
                    *reinterpret_cast<bf16x8*>(stage + row * (PW * 2) + ((lcol ^ (row & (LR - 1))) * 16)) = wf[sl][pc * NI + i];
                }
                // [row][channel] tiles take their weight rows through tau (16 consecutive channels per lane)
                const int wl = (sp[sl].flags & RM_TAU) ? ffk_tau(l32) : l32;
#pragma unroll
                for (int k = 0; k < NI; ++k)
                    wf[sl][pc * NI + k] = *reinterpret_cast<const bf16x8*>(stage + wl * (PW * 2) + (((2 * k + half) ^ (wl & (LR - 1))) * 16));
            }
        if (half == 0) {
#pragma unroll
            for (int sl = 0; sl < NS; ++sl)
                s_bias[(wave * NS + sl) * 32 + l32] = (sp[sl].flags & RM_SIG) ? -1.4426950408889634f * tb[sl] : tb[sl];
        }
        if (PB && d.pb_heads) {
#pragma unroll
            for (int i = 0; i < NW; ++i) s_wb[tid + i * THREADS] = tw[i];
        }
    }

    auto commit = [&](int buf) __attribute__((always_inline)) {
        unsigned char* sa = s_a + buf * (BM * AP);
        u32x4 gw = *reinterpret_cast<const u32x4*>(&gam), bw = *reinterpret_cast<const u32x4*>(&bet);
        if (NS * K >= 256 || OCC > 2) asm volatile("" : "+v"(gw), "+v"(bw));      // opaque: kept packed between the slabs
        const Vec16<T> gam = *reinterpret_cast<const Vec16<T>*>(&gw), bet = *reinterpret_cast<const Vec16<T>*>(&bw);
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            Vec16<T> x = pre[i];
            if (ln) {
                float f[8], s = 0.0f;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    f[e] = (float)x.e[e];
                    s += f[e];
                }
                const float mu = group_sum(s, LPR) * (1.0f / K);
                float q = 0.0f;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    f[e] -= mu;
                    q += f[e] * f[e];
                }
                const float rs = rsqrtf(group_sum(q, LPR) * (1.0f / K) + d.ln_eps);
#pragma unroll
                for (int e = 0; e < 8; ++e) x.e[e] = (T)(f[e] * rs * (float)gam.e[e] + (float)bet.e[e]);
            }
            *reinterpret_cast<Vec16<T>*>(sa + (r0 + RPP * i) * AP + c8 * 16) = x;
        }
        if (rm && tid < BM) s_mask[buf * BM + tid] = (float)pm;
    };

    // ---- fixed lane offsets of the slots' stores (bytes) ----
    unsigned voff[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const RmSlot& t = sp[s];
        voff[s] = t.kind == FFK_TILE_ACC  ? (unsigned)((half * 32 + n32) << 5)
                  : t.kind == FFK_TILE_V  ? (unsigned)((half * 32 + l32) << 5)
                  : t.kind == FFK_TILE_QK ? (unsigned)(n32 * 32 + 8 * half)
                  : (t.flags & RM_ROWS)   ? (unsigned)(n32 * t.s_i + 16 * half) * 2u
                                          : (unsigned)(l32 * t.s_d + 16 * half) * 2u;
    }

    // ---- operands of the residual epilogues, requested one row group ahead ----
    struct Ahead {
        u32x4 r0, r1, t;
    };
    [[maybe_unused]] Ahead ahead[RES ? NS : 1];
    const int rg_first = wave / (WAVES / d.rg_step);
    // element offset of this lane's first channel of a strided by-rows slot, for row group m0g (rows past the end: the last row)
    auto row_off = [&](const RmSlot& t, int m0g, int row) __attribute__((always_inline)) -> long {
        if (UNI) {
            const unsigned hi = d.flat ? 0u : rm_quot(d.inner, (unsigned)m0g), lo = (unsigned)m0g - hi * d.inner.d;
            return (long)hi * t.s_o + (long)lo * t.s_i + (long)(row - m0g) * t.s_i + 16 * half;
        }
        const unsigned hi = rm_quot(d.inner, (unsigned)row), lo = (unsigned)row - hi * d.inner.d;
        return (long)hi * t.s_o + (long)lo * t.s_i + 16 * half;
    };
    [[maybe_unused]] auto ahead_load = [&](auto s_tag, int m0g) __attribute__((always_inline)) {
        if constexpr (RES) {
            constexpr int s = decltype(s_tag)::value;
            const RmSlot& t = sp[s];
            const RmRes& q = args.res[slot0 + s];
            if (!q.resid) return;
            if (UNI && m0g + 32 <= M) {                  // scalar base, lane offset of the launch
                const unsigned hi = d.flat ? 0u : rm_quot(d.inner, (unsigned)m0g), lo = (unsigned)m0g - hi * d.inner.d;
                const long base = (long)hi * t.s_o + (long)lo * t.s_i;
                const char* rp = reinterpret_cast<const char*>(q.resid + base);
                if (16 * half + 8 <= t.ncols_left) ahead[s].r0 = *reinterpret_cast<const u32x4*>(rp + voff[s]);
                if (16 * half + 16 <= t.ncols_left) {
                    ahead[s].r1 = *reinterpret_cast<const u32x4*>(rp + voff[s] + 16);
                    if (XT && q.xtail) ahead[s].t = *reinterpret_cast<const u32x4*>(reinterpret_cast<const char*>(q.xtail + base) + (voff[s] >> 1));
                }
                return;
            }
            const int row = m0g + n32 < M ? m0g + n32 : M - 1;
            const long off = row_off(t, m0g, row);
            if (16 * half + 8 <= t.ncols_left) ahead[s].r0 = *reinterpret_cast<const u32x4*>(q.resid + off);
            if (16 * half + 16 <= t.ncols_left) {
                ahead[s].r1 = *reinterpret_cast<const u32x4*>(q.resid + off + 8);
                if (XT && q.xtail) ahead[s].t = *reinterpret_cast<const u32x4*>(q.xtail + off);
            }
        }
    };
    if constexpr (RES) {
        auto first = [&](auto s_tag) __attribute__((always_inline)) {
            constexpr int s = decltype(s_tag)::value;
            ahead[s].r0 = ahead[s].r1 = ahead[s].t = u32x4{0, 0, 0, 0};
            if (sp[s].wrow >= 0 && slab * BM + rg_first * 32 < M) ahead_load(s_tag, slab * BM + rg_first * 32);
        };
        first(std::integral_constant<int, 0>());
        if constexpr (NS > 1) first(std::integral_constant<int, 1>());
    }

    lds_barrier();                                       // every wave is done with the staging area
    commit(0);
    lds_barrier();
    int buf = 0;
    bf16x8 af[KC > 1 ? 2 : 1][CH];
    for (; slab < nslabs; slab += gridDim.x) {
        const bool more = slab + (int)gridDim.x < nslabs;
        if (more) fetch(slab + (int)gridDim.x);          // in flight during the products below
        const unsigned char* sa = s_a + buf * (BM * AP);
        if (PB && d.pb_heads && blockIdx.y == 0 && wave * 16 < BM) {
            // pair bias of this slab on the matrix pipe: wave w takes the rows 16 w .. 16 w + 15 as the N operand of
            // four 16 x 16 x 32 products against the (at most four) head weight rows, zero rows up to 16 (M operand).
            // The rows are the operand as the other products see it (normalised, rounded to bf16), so the value
            // equals a further output column group of four channels.  Result layout: lane = row, register v = head
            // (4 * (lane / 16) + v: only the first sixteen lanes hold real heads).
            const int r16 = lane & 15, kq = lane >> 4;
            const unsigned char* xr = sa + (wave * 16 + r16) * AP + kq * 16;
            const T* wr = s_wb + (r16 & 3) * K + kq * 8;
            f32x4 pacc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int ks = 0; ks < K / 32; ++ks) {
                const bf16x8 xv = *reinterpret_cast<const bf16x8*>(xr + ks * 64);
                bf16x8 wv = *reinterpret_cast<const bf16x8*>(wr + ks * 32);
                if (r16 >= 4) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) wv[e] = (T)0.0f;
                }
                pacc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv, xv, pacc, 0, 0, 0);
            }
            const int pr = slab * BM + wave * 16 + r16;
            if (kq == 0 && pr < M) {
                const unsigned hi = (unsigned)pr / d.pb_inner, lo = (unsigned)pr - hi * d.pb_inner;
                T* po = d.pb_out + (long)(int)(hi >> 5) * d.pb_so + (long)(lo >> 5) * 1024 + qk_tile_off((int)(lo & 31), (int)(hi & 31));
#pragma unroll
                for (int hd = 0; hd < 4; ++hd)
                    if (hd < d.pb_heads) po[(long)hd * d.pb_sh] = (T)(pacc[hd] * d.pb_scale);
            }
        }
        auto lda = [&](int b, const unsigned char* ap, int c) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < CH; ++i) af[b][i] = *reinterpret_cast<const bf16x8*>(ap + (c * CH + i) * 32);
        };
        const unsigned char* ap = sa + (rg_first * 32 + n32) * AP + half * 16;
        lda(0, ap, 0);
        for (int rg = rg_first; rg < RG; rg += d.rg_step) {
            const int m0g = slab * BM + rg * 32;
            if (m0g >= M) break;
            const bool valid = m0g + n32 < M;
            const unsigned hi = d.flat ? 0u : rm_quot(d.inner, (unsigned)m0g), lo = (unsigned)m0g - hi * d.inner.d;
            const float* smk = s_mask + buf * BM + rg * 32;
            const unsigned char* ap_next = rg + d.rg_step < RG ? ap + d.rg_step * 32 * AP : ap;
            const int m0g_next = rg + d.rg_step < RG && m0g + d.rg_step * 32 < M ? m0g + d.rg_step * 32
                                 : more                                         ? (slab + (int)gridDim.x) * BM + rg_first * 32
                                                                                : M;

            // the finished block of slot s to its tile
            auto store = [&](auto s_tag, const f32x16& acc, const f32x16& accg, auto rows_tag, auto glu_tag) __attribute__((always_inline)) {
                constexpr int s = decltype(s_tag)::value;
                constexpr bool ROWS = decltype(rows_tag)::value, GLU = decltype(glu_tag)::value;
                const RmSlot& t = sp[s];
                const float* sb = s_bias + (wave * NS + s) * 32;
                u32x4 y[2];
                if constexpr (ROWS) {
                    const float rmask = (t.flags & RM_MASKED) ? smk[n32] : 1.0f;
                    rm_value_rows<GLU>(t, acc, accg, sb, rmask, half, y);
                } else {
                    rm_value_cols<GLU>(t, acc, accg, sb, (t.flags & RM_MASKED) ? smk : nullptr, l32, half, y);
                }
                const u32x4 &y0 = y[0], &y1 = y[1];
                if constexpr (!ROWS) {
                    if (UNI || t.kind == FFK_TILE_V) {
                        // the group is one whole key tile (V), or sixteen consecutive rows per lane of one outer step
                        const long base = (long)hi * t.s_o + (t.kind == FFK_TILE_V ? (long)(lo >> 5) * 1024 : (long)lo);
                        char* p = reinterpret_cast<char*>(t.out + base);
                        const bool ok = t.kind == FFK_TILE_V ? t.ncols_left >= 32 : l32 < t.ncols_left && m0g + 16 * half < M;
                        if (ok) {
                            *reinterpret_cast<u32x4*>(p + voff[s]) = y0;
                            *reinterpret_cast<u32x4*>(p + voff[s] + 16) = y1;
                        }
                    } else {                             // inner % 16 == 0: each half of the group lies in one outer step
                        const int mr = m0g + 16 * half;
                        const unsigned h = rm_quot(d.inner, (unsigned)(mr < M ? mr : 0)), l = (unsigned)(mr < M ? mr : 0) - h * d.inner.d;
                        if (mr < M && l32 < t.ncols_left) {
                            T* p = t.out + (long)h * t.s_o + l + (long)l32 * t.s_d;
                            *reinterpret_cast<u32x4*>(p) = y0;
                            *reinterpret_cast<u32x4*>(p + 8) = y1;
                        }
                    }
                    return;
                } else {
                    if (t.kind == FFK_TILE_ACC || t.kind == FFK_TILE_QK) {
                        if (UNI) {
                            char* p = reinterpret_cast<char*>(t.out + (long)hi * t.s_o + (long)(lo >> 5) * 1024);
                            if (valid && t.ncols_left >= 32) {
                                if (t.kind == FFK_TILE_ACC) {
                                    *reinterpret_cast<u32x4*>(p + voff[s]) = y0;
                                    *reinterpret_cast<u32x4*>(p + voff[s] + 16) = y1;
                                } else {
#pragma unroll
                                    for (int a = 0; a < 4; ++a)      // d = 8a + 4 half + b  ->  (d >> 4) * 512 + n * 16 + (d & 15)
                                        *reinterpret_cast<u32x2*>(p + voff[s] + (a >> 1) * 1024 + (a & 1) * 16) = u32x2{y[a >> 1][2 * (a & 1)], y[a >> 1][2 * (a & 1) + 1]};
                                }
                            }
                        } else if (valid && t.ncols_left >= 32) {
                            const unsigned h = rm_quot(d.inner, (unsigned)(m0g + n32)), l = (unsigned)(m0g + n32) - h * d.inner.d;
                            T* p = t.out + (long)h * t.s_o + (long)(l >> 5) * 1024;
                            if (t.kind == FFK_TILE_ACC) {
                                p += (half * 32 + (l & 31)) << 4;
                                *reinterpret_cast<u32x4*>(p) = y0;
                                *reinterpret_cast<u32x4*>(p + 8) = y1;
                            } else {
                                p += (l & 31) * 16 + 4 * half;
#pragma unroll
                                for (int a = 0; a < 4; ++a)
                                    *reinterpret_cast<u32x2*>(p + (a >> 1) * 512 + (a & 1) * 8) = u32x2{y[a >> 1][2 * (a & 1)], y[a >> 1][2 * (a & 1) + 1]};
                            }
                        }
                        return;
                    }
                    const int cl = 16 * half;            // this lane's 16 channels, relative to the slot
                    const bool ok0 = valid && cl + 8 <= t.ncols_left, ok1 = valid && cl + 16 <= t.ncols_left;
                    char* p;                             // UNI: scalar; else this lane's first channel
                    unsigned vo;
                    long off = 0;
                    if (UNI) {
                        off = (long)hi * t.s_o + (long)lo * t.s_i;
                        vo = voff[s];
                    } else {
                        off = row_off(t, m0g, valid ? m0g + n32 : M - 1);
                        vo = 0;
                    }
                    p = reinterpret_cast<char*>(t.out + off);
                    u32x4 o0 = y0, o1 = y1;
                    if constexpr (RES) {
                        const RmRes& q = args.res[slot0 + s];
                        const bool gated = q.gate != nullptr;
                        u32x4 g0, g1;
                        if (gated) {
                            const unsigned mc = (unsigned)(valid ? m0g + n32 : M - 1);
                            const unsigned gr = q.gate_periodic ? mc - rm_quot(q.gate_rows, mc) * q.gate_rows.d : mc;
                            const T* gp = q.gate + (long)gr * q.gate_ld + cl;
                            if (ok0) g0 = *reinterpret_cast<const u32x4*>(gp);
                            if (ok1) g1 = *reinterpret_cast<const u32x4*>(gp + 8);
                        }
                        const Ahead cur = ahead[s];
                        if (m0g_next < M) ahead_load(s_tag, m0g_next);
                        if (gated) {
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                o0[e] = rm_pack2(rm_lo(o0[e]) * gate_factor(rm_lo(g0[e]), t.act), rm_hi(o0[e]) * gate_factor(rm_hi(g0[e]), t.act));
                                o1[e] = rm_pack2(rm_lo(o1[e]) * gate_factor(rm_lo(g1[e]), t.act), rm_hi(o1[e]) * gate_factor(rm_hi(g1[e]), t.act));
                            }
                        }
                        if (XT && q.xtail) {             // extended residual stream (whole 16-channel runs: ncols % 16 == 0)
                            float f[16];
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                f[2 * e] = rm_lo(o0[e]);
                                f[2 * e + 1] = rm_hi(o0[e]);
                                f[8 + 2 * e] = rm_lo(o1[e]);
                                f[9 + 2 * e] = rm_hi(o1[e]);
                            }
                            u32x4 tn;
                            xs_update16(f, cur.r0, cur.r1, cur.t, o0, o1, tn);
                            if (ok1) {
                                *reinterpret_cast<u32x4*>(p + vo) = o0;
                                *reinterpret_cast<u32x4*>(p + vo + 16) = o1;
                                *reinterpret_cast<u32x4*>(reinterpret_cast<char*>(q.xtail + off) + (vo >> 1)) = tn;
                            }
                            return;
                        }
                        if (q.resid) {
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                o0[e] = rm_pack2(rm_lo(o0[e]) + rm_lo(cur.r0[e]), rm_hi(o0[e]) + rm_hi(cur.r0[e]));
                                o1[e] = rm_pack2(rm_lo(o1[e]) + rm_lo(cur.r1[e]), rm_hi(o1[e]) + rm_hi(cur.r1[e]));
                            }
                        }
                    }
                    if (ok0) *reinterpret_cast<u32x4*>(p + vo) = o0;
                    if (ok1) *reinterpret_cast<u32x4*>(p + vo + 16) = o1;
                }
            };

            // products of slots S0 (and S0 + 1) with this row group; `nx`: where the following products' rows start
            auto products = [&](auto s0_tag, auto two_tag, auto rows_tag, f32x16& acc0, f32x16& acc1, const unsigned char* nx) __attribute__((always_inline)) {
                constexpr int S0 = decltype(s0_tag)::value;
                constexpr bool TWO = decltype(two_tag)::value, ROWS = decltype(rows_tag)::value;
                constexpr int S1 = TWO ? S0 + 1 : S0;
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    acc0[v] = 0.0f;
                    if (TWO) acc1[v] = 0.0f;
                }
#pragma unroll
                for (int c = 0; c < KC; ++c) {
                    const int b = KC > 1 ? (c & 1) : 0;
                    if (KC > 1) {
                        if (c + 1 < KC) lda(b ^ 1, ap, c + 1);
                        else lda(b ^ 1, nx, 0);
                        __builtin_amdgcn_sched_barrier(0);
                    }
#pragma unroll
                    for (int i = 0; i < CH; ++i) {
                        if (ROWS) MM::mma(acc0, wf[S0][c * CH + i], af[b][i]);
                        else MM::mma(acc0, af[b][i], wf[S0][c * CH + i]);
                    }
                    if (TWO) {
#pragma unroll
                        for (int i = 0; i < CH; ++i) {
                            if (ROWS) MM::mma(acc1, wf[S1][c * CH + i], af[b][i]);
                            else MM::mma(acc1, af[b][i], wf[S1][c * CH + i]);
                        }
                    }
                    if (KC == 1) lda(0, nx, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            };
            typedef std::integral_constant<bool, true> Yes;
            typedef std::integral_constant<bool, false> No;
            // slots S0 and S0 + 1 (if the wave has it)
            auto pair = [&](auto s0_tag) __attribute__((always_inline)) {
                constexpr int S0 = decltype(s0_tag)::value;
                constexpr bool HAS1 = S0 + 1 < NS;
                constexpr int S1 = HAS1 ? S0 + 1 : S0;
                constexpr std::integral_constant<int, S1> s1_tag{};
                if (sp[S0].wrow < 0) return;
                const bool rows = sp[S0].flags & RM_ROWS;
                const unsigned char* nx = ap_next;
                f32x16 acc0, acc1;
                if constexpr (HAS1) {
                    if (SHARE && sp[S1].wrow >= 0 && rows == (bool)(sp[S1].flags & RM_ROWS)) {
                        if (!RES && sp[S0].glu == 1) {
                            if constexpr (!RES) {
                                if (rows) {
                                    products(s0_tag, Yes(), Yes(), acc0, acc1, nx);
                                    store(s0_tag, acc0, acc1, Yes(), Yes());
                                } else {
                                    products(s0_tag, Yes(), No(), acc0, acc1, nx);
                                    store(s0_tag, acc0, acc1, No(), Yes());
                                }
                            }
                        } else if (rows) {
                            products(s0_tag, Yes(), Yes(), acc0, acc1, nx);
                            store(s0_tag, acc0, acc0, Yes(), No());
                            store(s1_tag, acc1, acc1, Yes(), No());
                        } else if constexpr (!RES) {
                            products(s0_tag, Yes(), No(), acc0, acc1, nx);
                            store(s0_tag, acc0, acc0, No(), No());
                            store(s1_tag, acc1, acc1, No(), No());
                        }
                        return;
                    }
                }
                auto single = [&](auto s_tag, const unsigned char* nxt) __attribute__((always_inline)) {
                    constexpr int S = decltype(s_tag)::value;
                    if (sp[S].flags & RM_ROWS) {
                        products(s_tag, No(), Yes(), acc0, acc1, nxt);
                        store(s_tag, acc0, acc0, Yes(), No());
                    } else if constexpr (!RES) {
                        products(s_tag, No(), No(), acc0, acc1, nxt);
                        store(s_tag, acc0, acc0, No(), No());
                    }
                };
                if constexpr (HAS1) {
                    if (sp[S1].wrow >= 0) {
                        single(s0_tag, ap);
                        single(std::integral_constant<int, S1>(), nx);
                        return;
                    }
                }
                single(s0_tag, nx);
            };
            pair(std::integral_constant<int, 0>());
            ap = ap_next;
        }
        if (!more) break;                                // nothing left to commit: the stores drain on their own
        commit(buf ^ 1);
        lds_barrier();
        buf ^= 1;
    }
}

}  // namespace
// ------------------------------------------------------------------------------------------------------ host ----
namespace {

RmDiv rm_div(unsigned d) {
    unsigned l = 0;
    while ((1ull << l) < d) ++l;
    const unsigned long long mul = ((1ull << 32) * ((1ull << l) - d)) / d + 1;
    return RmDiv{(unsigned)mul, l, d};
}

struct RmUnit { int tile, chan, wrow; bool glu, rows; };
// How a launch is laid out: workgroups of `waves` waves whose slabs hold np 16-byte loads per thread, `ns` slots per wave; R waves
// hold the same units and take every R-th row group each; `groups` sets of workgroups (blockIdx.y), each with units of its own.
struct RmCfg { int waves, ns, np, R, groups; };

constexpr int rm_occ(int K, int waves, int ns, int np, bool res) {      // waves per SIMD: three where 168 registers hold a variant
    return waves == 4 && ns == 1 && np * 64 * 4 / (K / 8) <= (K == 64 ? 64 : 32) && K <= 128 && !res ? 3 : 2;
}

// The variants built per K, and the layout a launch of M rows takes among them: the one with the least
//     start + rounds * (time of a slab)
// in microseconds.  start: 3 for the dispatch, 1 more for eight waves, and the weights of a CU at 50 KB/us; rounds: slabs per
// workgroup that fits on the chip at the same time, rounded up (at 128 x 192 rows a grid of 256 eight-wave workgroups runs a second
// round for an eighth of them: 25.7 us against 20.5); a slab: the bytes its CU reads and writes for it - the rows again for every
// group - or its blocks at 0.25 us per wave of a SIMD.  Rates of a CU measured at full grids: 15.8 KB/us with eight waves (13.2 for
// two units of K = 256 each), 17 with four, 20 with three such workgroups per CU.  Measured, 128 -> 512 in operand tiles, eight
// waves x two units / four waves x two / four waves x one over 32 rows: 1 024 rows 12.8 / 7.9 / 4.5 us, 9 216 rows 14.2 / 10.2 / 8.6,
// 65 536 rows 28.1 / 29.1 / 32.0, 1 048 576 rows 315 / 345 / 560.
struct RmVariant { int K, waves, ns, np; bool res; };
constexpr RmVariant RM_VARIANTS[] = {
    {64, 8, 2, 4, false},  {64, 4, 1, 2, false},  {64, 4, 2, 2, false},  {64, 8, 1, 4, true},  {64, 4, 1, 2, true},
    {128, 8, 1, 4, false}, {128, 8, 2, 4, false}, {128, 4, 1, 2, false}, {128, 4, 2, 2, false}, {128, 4, 2, 4, false},
    {128, 8, 1, 4, true},  {128, 4, 1, 2, true},  {128, 4, 1, 4, true},
    {256, 8, 1, 4, false}, {256, 8, 2, 4, false}, {256, 4, 1, 4, false}, {256, 8, 1, 4, true},  {256, 4, 1, 4, true},
};

RmCfg rm_layout(int K, int M, const RmUnit* u, int nu, bool res, bool tails, bool uni, bool one_group) {
    RmCfg best{0, 0, 0, 0, 0};
    double least = 1e30;
    bool glu = false;
    for (int i = 0; i < nu; ++i) glu = glu || u[i].glu;
    for (const RmVariant& v : RM_VARIANTS) {
        if (v.K != K || v.res != res || (glu && v.ns == 1) || (!uni && (v.waves != 8 || v.ns != (res ? 1 : 2)))) continue;
        int items = 0;                                   // what a slot (or a pair of slots) takes
        for (int k = 0; k < nu; ++items) k += v.ns == 1 || u[k].glu || k + 1 >= nu || u[k + 1].glu || u[k + 1].rows != u[k].rows ? 1 : 2;
        const int bm = v.np * 64 * v.waves / (K / 8), rg = bm / 32, slabs = ffk_cdiv(M, bm);
        for (int R = 1; R <= rg && R <= v.waves; R *= 2) {
            const int G = v.waves / R, groups = items > G ? ffk_cdiv(items, G) : 1;
            if (groups * v.waves * v.ns > RM_MAX_SLOTS || (one_group && groups > 1)) continue;
            const int per_cu = 4 * rm_occ(K, v.waves, v.ns, v.np, res) / v.waves, grid = 256 * per_cu / groups;
            const int on = ffk_cdiv((long)(slabs < grid ? slabs : grid) * groups, 256);         // workgroups of a CU
            const double rounds = ffk_cdiv(slabs, grid), wk = on * v.waves * v.ns * K / 16.0;   // KB of weights
            const int sets = items < 1 ? 1 : G < items ? G : items;
            const double out = (double)nu / groups * 64 * (glu ? 0.5 : 1.0) * (res ? (tails ? 3 : 2) : 1);
            const double rate = v.waves == 8 ? (K == 256 && v.ns == 2 ? 13.2 : 15.8) : per_cu == 3 ? 20.0 : 17.0;
            const double bytes = on * bm * (2.0 * K + out) / 1024 / rate;
            const double blocks = on * (v.waves / 4) * ffk_cdiv(ffk_cdiv(items, groups), sets) * v.ns * (rg / R) * 0.25 * (K / 128.0 > 1 ? 1.5 : 1.0);
            const double cost = 3.0 + (v.waves == 8 ? 1.0 : 0.0) + wk / 50 + rounds * (bytes > blocks ? bytes : blocks);
            if (cost < least) {
                least = cost;
                best = RmCfg{v.waves, v.ns, v.np, R, groups};
            }
        }
    }
    return best;
}

bool rm_tile_ok(const ffk_linear_desc& d, const ffk_tile& t) {
    auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    auto lane32 = [](int64_t s) { return s >= 0 && s <= (1 << 26); };     // 31 rows or channels fit a 32-bit byte offset
    if (t.inner <= 0 || t.ncols <= 0 || !al16(t.out)) return false;
    if (rm_by_rows(t)) {
        if (t.kind == FFK_TILE_STRIDED) {
            if (t.ncols % 8 != 0 || t.s_o % 8 || t.s_i % 8 || t.s_h % 8 || !lane32(t.s_i)) return false;
            if (t.resid && !al16(t.resid)) return false;
            if (t.gate && (!al16(t.gate) || t.gate_ld % 8)) return false;
            if (t.xtail && (!t.resid || t.ncols % 16 != 0 || t.s_o % 16 || t.s_i % 16 || t.s_h % 16)) return false;
        } else {
            if (t.ncols % 32 != 0 || t.resid || t.gate || t.xtail || t.s_o % 8 || t.s_h % 8) return false;
        }
        return true;
    }
    if (t.resid || t.gate || t.xtail) return false;
    if (t.kind == FFK_TILE_V)        // stored by whole key tiles
        return !t.rowmask && d.M % 32 == 0 && t.inner % 32 == 0 && t.ncols % 32 == 0 && t.s_o % 8 == 0 && t.s_h % 8 == 0;
    if (t.kind != FFK_TILE_STRIDED) return false;
    return d.M % 16 == 0 && t.inner % 16 == 0 && t.s_i == 1 && t.s_o % 8 == 0 && t.s_h % 8 == 0 && t.s_d % 8 == 0 && lane32(t.s_d);
}

template <bool RES>
void rm_fill(RmArgs<RES>& p, const ffk_linear_desc& d, const RmUnit* u, int nu, const RmCfg& c, int inner) {
    for (auto& q : p.slot) {
        q = RmSlot{};
        q.wrow = -1;
    }
    if constexpr (RES)
        for (auto& q : p.res) q = RmRes{};
    const int G = c.waves / c.R, sets = G * c.groups;
    const bool pairs = c.ns > 1;                         // slots are dealt two at a time: GLU units, or two units of one store order
    int i = 0;
    for (int set = 0; set < sets; ++set) {
        // an even share of what is left
        int take = 0;
        if (pairs) {
            int items = 0;
            for (int k = i; k < nu; ++items) k += u[k].glu || k + 1 >= nu || u[k + 1].glu || u[k + 1].rows != u[k].rows ? 1 : 2;
            take = ffk_cdiv(items, sets - set);
        } else {
            take = ffk_cdiv(nu - i, sets - set);
        }
        for (int s = 0; take > 0 && i < nu; --take) {
            auto put = [&](const RmUnit& q, int sl, int half, int glu) {
                const ffk_tile& t = d.tiles[q.tile];
                RmSlot r{};
                const long coff = (long)(q.chan >> 5) * t.s_h;
                r.out = (T*)t.out + coff;
                r.wrow = q.wrow + 32 * half;
                r.bias = t.bias ? (const T*)t.bias + (r.wrow & 127) : nullptr;
                r.s_i = (int)t.s_i;
                r.s_o = (int)t.s_o;
                if (t.inner >= d.M && inner < d.M)       // one outer step, seen in steps of the launch
                    r.s_o = t.kind == FFK_TILE_STRIDED ? (int)(inner * t.s_i) : inner / 32 * 1024;
                r.s_d = (int)t.s_d;
                r.ncols_left = t.ncols - q.chan;
                r.scale = t.scale;
                r.kind = (signed char)t.kind;
                r.act = (signed char)t.act;
                r.glu = (signed char)glu;
                const bool sig = t.glu ? glu == 2 : t.act == FFK_ACT_SIGMOID;
                r.flags = (unsigned char)((t.rowmask ? RM_MASKED : 0) | (t.bias ? RM_BIAS : 0) | (q.rows ? RM_ROWS : 0) |
                                          (t.kind == FFK_TILE_STRIDED && t.s_d == 1 ? RM_TAU : 0) | (sig ? RM_SIG : 0));
                for (int w = set % G; w < c.waves; w += G) {
                    const int at = ((set / G) * c.waves + w) * c.ns + sl;
                    p.slot[at] = r;
                    if constexpr (RES) {
                        RmRes& e = p.res[at];
                        e.resid = t.resid ? (const T*)t.resid + coff : nullptr;
                        e.gate = t.gate ? (const T*)t.gate + q.chan : nullptr;
                        e.xtail = t.xtail ? (int8_t*)t.xtail + coff : nullptr;
                        e.gate_ld = (int)t.gate_ld;
                        e.gate_periodic = t.gate_rows > 0;
                        e.gate_rows = rm_div(t.gate_rows > 0 ? (unsigned)t.gate_rows : 1u);
                    }
                }
            };
            if (u[i].glu) {
                put(u[i], s, 0, 1);
                put(u[i], s + 1, 1, 2);
                ++i;
                s += 2;
            } else {
                put(u[i], s, 0, 0);
                const bool two = pairs && i + 1 < nu && !u[i + 1].glu && u[i + 1].rows == u[i].rows;
                if (two) put(u[i + 1], s + 1, 0, 0);
                i += two ? 2 : 1;
                s += pairs ? 2 : 1;
            }
        }
    }
}

template <int K, int NS, int WAVES, int NP, bool RES, bool XT, bool UNI>
int rm_launch_one(const RmArgs<RES>& a, const RmCfg& c, hipStream_t st) {
    typedef RmGeo<K, WAVES, NP> G;
    constexpr int OCC = rm_occ(K, WAVES, NS, NP, RES);
    const size_t smem = G::SLABS + (2 * G::BM + WAVES * NS * 32) * sizeof(float) + (rm_takes_bias(K, RES, UNI) ? 4 * K * sizeof(T) : 0);
    static FfkLdsReservation lds_reserved;
    const int rc = ffk_reserve_lds(lds_reserved, (const void*)linear_rm_kernel<K, NS, WAVES, NP, RES, XT, UNI, OCC>, smem, "ffk_fused_linear");
    if (rc != FFK_OK) return rc;
    const int nslabs = ffk_cdiv(a.M, G::BM), most = 256 * (4 * OCC / WAVES) / c.groups;
    linear_rm_kernel<K, NS, WAVES, NP, RES, XT, UNI, OCC><<<dim3(nslabs < most ? nslabs : most, c.groups), G::THREADS, smem, st>>>(a);
    return ffk_check_launch("ffk_fused_linear");
}
template <int K, bool RES, bool XT, bool UNI, int I = 0>
int rm_launch(const RmArgs<RES>& a, const RmCfg& c, hipStream_t st) {
    if constexpr (I < (int)(sizeof(RM_VARIANTS) / sizeof(RM_VARIANTS[0]))) {
        constexpr RmVariant v = RM_VARIANTS[I];
        if constexpr (v.K == K && v.res == RES && (UNI || (v.waves == 8 && v.ns == (RES ? 1 : 2))))
            if (c.waves == v.waves && c.ns == v.ns && c.np == v.np) return rm_launch_one<K, v.ns, v.waves, v.np, RES, XT, UNI>(a, c, st);
        return rm_launch<K, RES, XT, UNI, I + 1>(a, c, st);
    }
    return ffk_fail(FFK_ERR_UNSUPPORTED, "ffk_fused_linear: no kernel for this layout");
}

}  // namespace

// Launches this kernel if it can take this (already validated) descriptor and returns 1 with the launch status in *status;
// returns 0 if the caller has to use another variant.
int ffk_linear_rm_try(const ffk_linear_desc* d, hipStream_t st, int* status) {
    if (d->dtype != FFK_BF16 || (d->K != 64 && d->K != 128 && d->K != 256)) return 0;
    if (d->ln_folded || d->a2 || d->a_chanmajor || d->variant == FFK_LINEAR_STAGED) return 0;
    if (!ffk_aligned16(d->ln_gamma) || !ffk_aligned16(d->ln_beta)) return 0;
    auto i32 = [](int64_t v) { return v >= -0x7fffffffL && v <= 0x7fffffffL; };      // the kernel's strides have 32 bits
    if (!i32(d->a_so) || !i32(d->a_si)) return 0;
    // a trailing pair-bias tile (score-operand tiles of <= 4 heads) rides on the launch without a weight slot; it may be
    // the only tile (a chunked attention computes its bias before the first slab, with the bits of the riding one)
    int n = d->n_tiles;
    const ffk_tile* bias_tile = nullptr;
    if (d->tiles[n - 1].kind == FFK_TILE_BIAS) {
        const ffk_tile& t = d->tiles[n - 1];
        if (d->K != 128 || t.ncols < 1 || t.ncols > 4 || t.bias || t.resid || t.gate || t.rowmask || t.xtail || t.glu ||
            t.act != FFK_ACT_NONE || t.inner <= 0 || !t.out || !ffk_aligned16(t.out))
            return 0;
        bias_tile = &t;
        --n;
    }
    bool chan_major = false, v_tiles = false, tails = false, res = false, cols = false, glu = false;
    int mask_tile = -1, inner = 0x7fffffff;
    const char* a0 = (const char*)d->a;
    bool over_input = false;
    for (int i = 0; i < d->n_tiles; ++i) {
        const ffk_tile& t = d->tiles[i];
        if (!i32(t.s_o) || !i32(t.s_i) || !i32(t.s_d) || !i32(t.s_h) || !i32(t.gate_ld) || !i32(t.m_so) || !i32(t.m_si)) return 0;
        const char* o = (const char*)t.out;
        over_input = over_input || (o >= a0 && o < a0 + (size_t)d->M * d->K * sizeof(T));
    }
    for (int i = 0; i < n; ++i) {
        const ffk_tile& t = d->tiles[i];
        if (t.kind == FFK_TILE_BIAS || !rm_tile_ok(*d, t)) return 0;
        tails = tails || t.xtail;
        res = res || t.resid || t.gate;
        cols = cols || !rm_by_rows(t);
        glu = glu || t.glu;
        chan_major = chan_major || (!rm_by_rows(t) && t.kind == FFK_TILE_STRIDED);
        v_tiles = v_tiles || t.kind == FFK_TILE_V;
        if (t.inner < d->M) {
            if (inner != 0x7fffffff && inner != t.inner) return 0;
            inner = t.inner;
        }
        if (t.rowmask) {
            if (mask_tile < 0) mask_tile = i;
            const ffk_tile& f = d->tiles[mask_tile];         // one mask per launch
            if (t.rowmask != f.rowmask || t.inner != f.inner || t.m_so != f.m_so || t.m_si != f.m_si) return 0;
        }
    }
    if (chan_major && v_tiles) return 0;                     // they need different row orders within a group
    if (glu && d->K == 256) return 0;                        // GLU units are built for K = 64 and 128
    if (res && (cols || glu || bias_tile)) return 0;         // residual epilogues are built for [row][channel] launches
    const bool flat = inner == 0x7fffffff, uni = flat || inner % 32 == 0;
    if (flat) inner = d->M;
    if (mask_tile >= 0 && d->tiles[mask_tile].inner >= d->M && !flat) return 0;
    if (bias_tile && !uni) return 0;
    for (int i = 0; i < n; ++i) {
        const ffk_tile& t = d->tiles[i];
        if (!flat && t.inner >= d->M && (t.kind == FFK_TILE_STRIDED ? !i32((int64_t)inner * t.s_i) : inner % 32 != 0)) return 0;
        if (res && t.kind != FFK_TILE_STRIDED) return 0;
    }
    // units, those stored by rows first
    RmUnit units[FFK_MAX_TILES * 4];
    int nu = 0;
    for (int pass = 0; pass < 2; ++pass)
        for (int i = 0; i < n; ++i) {
            const ffk_tile& t = d->tiles[i];
            if (rm_by_rows(t) != (pass == 0)) continue;
            for (int c = 0; c < t.ncols; c += 32) units[nu++] = {i, c, i * 128 + (t.glu ? 2 * c : c), t.glu != 0, pass == 0};
        }
    if (nu > RM_MAX_SLOTS) return 0;
    // a launch over its own input: one group, whose workgroups have read the rows of a slab before they store any of it
    const RmCfg c = rm_layout(d->K, d->M, units, nu, res, tails, uni, over_input);
    if (c.waves == 0) return 0;
    RmCommon k{};
    k.a = (const T*)d->a;
    k.w = (const T*)d->w;
    k.ln_gamma = (const T*)d->ln_gamma;
    k.ln_beta = (const T*)d->ln_beta;
    k.a_so = (int)d->a_so;
    k.a_si = (int)d->a_si;
    k.M = d->M;
    k.a_div = rm_div((unsigned)d->a_inner);
    k.a_flat = d->a_inner >= d->M;
    k.inner = rm_div((unsigned)inner);
    k.flat = flat;
    k.ln_eps = d->ln_eps;
    k.row_perm = chan_major;
    k.rg_step = c.R;
    if (mask_tile >= 0) {
        const ffk_tile& t = d->tiles[mask_tile];
        k.rowmask = (const T*)t.rowmask;
        k.m_so = (int)t.m_so;
        k.m_si = (int)t.m_si;
    }
    if (bias_tile) {
        k.pb_heads = bias_tile->ncols;
        k.pb_wrow = (d->n_tiles - 1) * 128;
        k.pb_inner = (unsigned)bias_tile->inner;
        k.pb_out = (T*)bias_tile->out;
        k.pb_so = (int)bias_tile->s_o;
        k.pb_sh = (int)bias_tile->s_h;
        k.pb_scale = bias_tile->scale;
    }
    auto go = [&](auto res_tag, auto tail_tag) {
        constexpr bool R = decltype(res_tag)::value, X = decltype(tail_tag)::value;
        RmArgs<R> a;
        static_cast<RmCommon&>(a) = k;
        rm_fill<R>(a, *d, units, nu, c, inner);
        if (!uni) {
            if (d->K == 64) return rm_launch<64, R, X, false>(a, c, st);
            if (d->K == 128) return rm_launch<128, R, X, false>(a, c, st);
            return rm_launch<256, R, X, false>(a, c, st);
        }
        if (d->K == 64) return rm_launch<64, R, X, true>(a, c, st);
        if (d->K == 128) return rm_launch<128, R, X, true>(a, c, st);
        return rm_launch<256, R, X, true>(a, c, st);
    };
    typedef std::integral_constant<bool, true> Yes;
    typedef std::integral_constant<bool, false> No;
    *status = !res ? go(No(), No()) : tails ? go(Yes(), Yes()) : go(Yes(), No());
    return 1;
}
