// Weights-stationary variant of the fused linear layer in fp32 (see ffk_fused_linear in include/ffk.h), K = 128 or 256.
//
// Products are six bf16 products of the operands' parts (split4): 196 cycles for a 32 x 32 block and a K step of 16, where
// v_mfma_f32_32x32x2_f32 takes 512 and no vector instruction of another wave runs beside it.  Rows are cut once, behind their
// LayerNorm and on the way to LDS, for up to eight weight units of 32 rows; weights stay in registers, at K = 128 as parts (96
// registers a unit), else (GLU units, K = 256) as they are and cut for every use, one step ahead of the products where the registers
// allow.  Against the fp32 instructions, us: 65 536 rows, 128 -> 1 024 173 -> 135, 128 -> 512 91 -> 70, 128 -> 128 34 -> 26, GLU 256 + 128
// channels 134 -> 100; 32 768 rows, 256 -> 1 024 161 -> 122, 256 -> 256 52 -> 36; 4 096 rows, 128 -> 512 12.4 -> 10.4.  A launch of
// 65 536 rows, 128 -> 512, is 35 us of memory traffic, 23 us of products and as many of vector instructions, which overlap in part:
// without its stores it takes 52 us, without its products 55.  Stores go through LDS, 128 bytes of eight lanes side by side (by a lane's own
// 16-byte pieces: 91 us), and the upper four waves prepare the next slab ahead of their products, the lower four behind them (all
// behind: 2 to 4 % more).
//
// Persistent workgroups of eight waves, one per CU: the units of a launch are dealt to groups (blockIdx.y), each with workgroups of
// its own over all rows; unit i of a group goes to wave i % 8, or, in a group of up to four with slabs of 64 rows, to waves i and i + 4,
// which take one half of the slab each - so the SIMDs have equal shares of any multiple of four units.  Few rows, GLU units and
// channel-major rows take workgroups of four waves with one slab and one unit per wave (ONE): what few rows wait for is the weights, which
// come as whole lines while the rows are normalised, and the residual, which is requested before the products.
//   by rows   (plain, q / k tiles, pair-bias tiles): product W . A^T, a lane owns one row and 16 consecutive channels
//             (64 bytes; weight rows are taken through tau, except for accumulator-order tiles)
//   by columns (v tiles, channel-major outputs): A . W^T, a lane owns one channel and 16 rows
#include "ffk_common.h"
#include <algorithm>
#include <type_traits>

namespace {

constexpr int W3_MAXU = FFK_MAX_TILES * 4, W3_CUS = 256;

// ONE: every workgroup has one slab of BM rows; else workgroups are persistent and the slab is double-buffered (32 rows at K = 256, else 64)
template <int K, bool GLU, bool ONE, int BM_> struct W3Geo {
    static constexpr int WAVES = ONE ? 4 : 8, THREADS = 64 * WAVES, BM = BM_, RG = BM / 32;
    static constexpr int KF = K / 8;                     // 16-byte pieces per unit and lane, two to a K step of 16
    static constexpr int AP = K * 6 + 16;                // LDS row pitch in bytes: [K step of 16][part][16] (see split4)
    static constexpr int OP = 65 * 64 + 64 * 8;          // LDS of a wave's outputs
    static constexpr int LPR = K / 4;                    // lanes per row
    static constexpr int RPP = THREADS / LPR;            // rows fetched per pass
    static constexpr int NP = BM / RPP;                  // passes: 4, 8 or 16
    static constexpr int SLOTS = GLU ? 2 : 1;            // weight units in a wave's registers
    static constexpr bool CUT = K == 128 && !GLU;        // the weights' parts in the registers, not the weights
    static constexpr int NBUF = ONE ? 1 : 2;
};

struct W3Args {
    ffk_linear_desc d;
    signed char unit[W3_MAXU];                           // first 32-row block of the weights (4 per tile) of every unit
    int n_units, per_group;                              // units of the launch; of a group (the last one may have fewer)
    int row_perm;                                        // rows of a group through tau (launches with channel-major tiles)
    int mask_tile;                                       // tile whose row mask the launch uses, -1: none
};

__host__ __device__ __forceinline__ bool w3_by_rows(const ffk_tile& t) {
    return t.kind == FFK_TILE_QK || t.kind == FFK_TILE_ACC || t.kind == FFK_TILE_BIAS || (t.kind == FFK_TILE_STRIDED && t.s_d == 1);
}

// 32-channel block of the output that unit u of its tile makes
template <bool GLU> __device__ __forceinline__ int w3_sub(const ffk_tile& t, int u) { return GLU && t.glu ? (u & 3) >> 1 : u & 3; }

// GLU: the launch has GLU tiles; the slots of a wave are then value and gate of one unit (a plain unit leaves the second empty)
// CM: element (m, k) of the operand at a + k * a_cs + rowoffset(m) (ONE only)
template <int K, bool GLU, bool ONE, int BM, bool CM>
__global__ __launch_bounds__(ONE ? 256 : 512, K == 128 && !GLU && BM == 32 ? 3 : 2) void linear_ws32_kernel(const W3Args args) {
    typedef W3Geo<K, GLU, ONE, BM> G;
    constexpr int NS = G::SLOTS, KF = G::KF, AP = G::AP, LPR = G::LPR, RPP = G::RPP, NP = G::NP;
    constexpr int W3_WAVES = G::WAVES, W3_RG = G::RG;
    const ffk_linear_desc& d = args.d;
    extern __shared__ __align__(16) unsigned char smem[];
    unsigned char* s_a = smem;                                                  // [NBUF][BM][AP]
    unsigned char* s_out = smem + G::NBUF * BM * AP;                            // [wave][OP]
    float* s_mask = reinterpret_cast<float*>(s_out + G::WAVES * G::OP);         // [parity of the slab][BM]
    float* s_bias = s_mask + 2 * BM;                                            // [wave][slot][32]
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    const int M = d.M;
    const float* A = (const float*)d.a;
    const float* W = (const float*)d.w;

    const int c4 = tid % LPR, r0 = tid / LPR;
    const bool ln = d.ln_gamma != nullptr;
    const int mt = args.mask_tile;
    const float* rm = mt >= 0 ? (const float*)d.tiles[mt].rowmask : nullptr;
    const bool a_flat = d.a_inner >= M;
    f32x4 pre[NP];                                       // CM: a row's channels tid / BM + (THREADS / BM) * i, i < 4 NP
    float pm = 1.0f;
    auto fetch = [&](int slab) __attribute__((always_inline)) {                         // rows past the end are clamped: never stored
        if constexpr (CM) {                              // consecutive lanes, consecutive rows: no alignment to keep
            const int m = slab * BM + (tid & (BM - 1)), mc = m < M ? m : M - 1;
            const unsigned hi = a_flat ? 0u : (unsigned)mc / (unsigned)d.a_inner, lo = (unsigned)mc - hi * (unsigned)d.a_inner;
            const float* p = A + (long)hi * d.a_so + (long)lo * d.a_si + (long)(tid / BM) * d.a_cs;
#pragma unroll
            for (int i = 0; i < 4 * NP; ++i) pre[i >> 2][i & 3] = p[(long)(i * (G::THREADS / BM)) * d.a_cs];
        } else if (a_flat) {
#pragma unroll
            for (int i = 0; i < NP; ++i) {
                const int m = slab * BM + r0 + RPP * i;
                pre[i] = *reinterpret_cast<const f32x4*>(A + (long)(m < M ? m : M - 1) * d.a_si + c4 * 4);
            }
        } else {
#pragma unroll
            for (int i = 0; i < NP; ++i) {
                const int m = slab * BM + r0 + RPP * i, mc = m < M ? m : M - 1;
                const unsigned hi = (unsigned)mc / (unsigned)d.a_inner, lo = (unsigned)mc - hi * (unsigned)d.a_inner;
                pre[i] = *reinterpret_cast<const f32x4*>(A + (long)hi * d.a_so + (long)lo * d.a_si + c4 * 4);
            }
        }
        if (rm) {
            const ffk_tile& t = d.tiles[mt];
            const int m = slab * BM + (tid & (BM - 1)), mc = m < M ? m : M - 1;
            const unsigned mh = (unsigned)mc / (unsigned)t.inner, ml = (unsigned)mc - mh * (unsigned)t.inner;
            pm = rm[(long)mh * t.m_so + (long)ml * t.m_si];
        }
    };
    f32x4 gam = {0, 0, 0, 0}, bet = gam;
    if (ONE) {                                           // the rows first: the products start with the weights that have come by then
        fetch(blockIdx.x);
        if (ln) {
            gam = *reinterpret_cast<const f32x4*>((const float*)d.ln_gamma + c4 * 4);
            bet = *reinterpret_cast<const f32x4*>((const float*)d.ln_beta + c4 * 4);
        }
    }

    const int u0 = blockIdx.y * args.per_group, n_u = args.n_units - u0 < args.per_group ? args.n_units - u0 : args.per_group;
    const bool halves = n_u <= W3_WAVES / W3_RG;         // two waves per unit
    int units[NS];                                       // -1: none
    // Weights: every wave reads the 32 rows of its units as whole lines (a lane's fragments are 16-byte pieces 32 bytes apart in 32
    // rows: fetched that way a request costs the address unit 64 cycles instead of 16, 3.5 us of a launch at K = 256) and re-orders
    // them through 4 KB of the slab buffer, 32 channels at a time.
    f32x4 wf[NS][KF];
    float tb[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int i = halves ? wave % (W3_WAVES / W3_RG) : wave;
        int u = i < n_u ? args.unit[u0 + i] : -1;
        if (GLU && s) u = u >= 0 && d.tiles[u >> 2].glu ? u + 1 : -1;
        units[s] = u;
        const ffk_tile& t = d.tiles[u >= 0 ? u >> 2 : 0];
        const float* wp = W + (long)((u >= 0 ? u : 0) * 32 + (lane >> 3)) * K + 4 * (lane & 7);
#pragma unroll
        for (int f = 0; f < KF; ++f) wf[s][f] = *reinterpret_cast<const f32x4*>(wp + (f & 3) * 8 * K + 32 * (f >> 2));
        tb[s] = u >= 0 && t.bias ? ((const float*)t.bias)[(u & 3) * 32 + l32] : 0.0f;
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const ffk_tile& t = d.tiles[units[s] >= 0 ? units[s] >> 2 : 0];
        const int wl = w3_by_rows(t) && t.kind != FFK_TILE_ACC ? ffk_tau(l32) : l32;
        unsigned char* stage = s_a + wave * 4096;
#pragma unroll
        for (int p = 0; p < KF; p += 4) {
#pragma unroll
            for (int i = 0; i < 4; ++i)                  // row i * 8 + lane / 8 of the piece, its 16-byte chunk lane % 8
                *reinterpret_cast<f32x4*>(stage + i * 1024 + (lane >> 3) * 128 + (((lane & 7) ^ (lane >> 3)) * 16)) = wf[s][p + i];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                wf[s][p + i] = *reinterpret_cast<const f32x4*>(stage + wl * 128 + (((4 * (i >> 1) + 2 * half + (i & 1)) ^ (wl & 7)) * 16));
        }
        if (half == 0) s_bias[(wave * NS + s) * 32 + l32] = tb[s];
    }
    bf16x8 wp[G::CUT ? KF / 2 : 1][3];
    if constexpr (G::CUT) {
#pragma unroll
        for (int g = 0; g < KF / 2; ++g) {
            const Split4 a = split4<false, true>(wf[0][2 * g]), b = split4<false, true>(wf[0][2 * g + 1]);
#pragma unroll
            for (int p = 0; p < 3; ++p) wp[g][p] = split_frag(a, b, p);
        }
    }
    lds_barrier();                                       // every wave is done with the staging area
    const int n32 = args.row_perm ? ffk_tau(l32) : l32;

    // ---- slab streaming ----
    if (!ONE && ln) {
        gam = *reinterpret_cast<const f32x4*>((const float*)d.ln_gamma + c4 * 4);
        bet = *reinterpret_cast<const f32x4*>((const float*)d.ln_beta + c4 * 4);
    }
    auto commit = [&](int buf) __attribute__((always_inline)) {        // buf: parity of the slab
        unsigned char* sa = s_a + (G::NBUF == 2 ? buf : 0) * (BM * AP);
        if constexpr (CM) {                              // transposed through LDS; rows are whole only there
#pragma unroll
            for (int i = 0; i < 4 * NP; ++i)
                *reinterpret_cast<float*>(sa + (tid & (BM - 1)) * AP + (tid / BM + i * (G::THREADS / BM)) * 4) = pre[i >> 2][i & 3];
            lds_barrier();
#pragma unroll
            for (int i = 0; i < NP; ++i) pre[i] = *reinterpret_cast<const f32x4*>(sa + (r0 + RPP * i) * AP + c4 * 16);
            lds_barrier();
        }
#pragma unroll
        for (int i = 0; i < NP; i += 4) {
            if (ln) ffk_ln_rows4<LPR>(pre + i, gam, bet, d.ln_eps);
#pragma unroll
            for (int j = i; j < i + 4; ++j) {
                const Split4 x = split4<false, true>(pre[j]);
#pragma unroll
                for (int p = 0; p < 3; ++p) *reinterpret_cast<u32x2*>(sa + (r0 + RPP * j) * AP + (c4 >> 2) * 96 + p * 32 + (c4 & 3) * 8) = x.p[p];
            }
        }
        if (rm && tid < BM) s_mask[buf * BM + tid] = pm;
    };

    // the sixteen values of one lane to their tile; u: unit, bias: of its 32 rows (GLU: and of its gate's)
    auto store = [&](int u, const float* bias, const f32x16& acc, const f32x16& accg, int m0g, const float* sm, [[maybe_unused]] const f32x4 (&rv)[4]) __attribute__((always_inline)) {
        const ffk_tile& t = d.tiles[u >> 2];
        const bool by_rows = w3_by_rows(t), glu = GLU && t.glu != 0;
        const int sub = w3_sub<GLU>(t, u), left = t.ncols - 32 * sub;      // channels left
        // channels of this lane: by rows 16 half + v (through tau) or 8 a + 4 half + b (ACC); by columns l32
        const bool nat = t.kind == FFK_TILE_ACC;
        const float* bp = bias + (by_rows ? (nat ? 4 : 16) * half : l32);
        float x[16];
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            f32x4 b, g;
            if (by_rows) {
                b = *reinterpret_cast<const f32x4*>(bp + a * (nat ? 8 : 4));
                if (glu) g = *reinterpret_cast<const f32x4*>(bp + 32 + a * (nat ? 8 : 4));
            } else {
                b = f32x4{bp[0], bp[0], bp[0], bp[0]};
                if (glu) g = f32x4{bp[32], bp[32], bp[32], bp[32]};
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                x[4 * a + e] = acc[4 * a + e] + b[e];
                if (glu) x[4 * a + e] *= sigmoid_f(accg[4 * a + e] + g[e]);
            }
        }
        if (!glu && t.act == FFK_ACT_RELU) {
#pragma unroll
            for (int v = 0; v < 16; ++v) x[v] = relu_f(x[v]);
        }
        if (!glu && t.act == FFK_ACT_SIGMOID) {
#pragma unroll
            for (int v = 0; v < 16; ++v) x[v] = sigmoid_f(x[v]);
        }
        if (t.scale != 1.0f) {
#pragma unroll
            for (int v = 0; v < 16; ++v) x[v] *= t.scale;
        }
        const unsigned inner = (unsigned)t.inner;
        if (t.rowmask) {
            if (by_rows) {
                const float k = sm[n32];
#pragma unroll
                for (int v = 0; v < 16; ++v) x[v] *= k;
            } else {
                const float* p = sm + (t.kind == FFK_TILE_V ? 4 : 16) * half;
#pragma unroll
                for (int v = 0; v < 16; ++v) x[v] *= p[t.kind == FFK_TILE_V ? 8 * (v >> 2) + (v & 3) : v];
            }
        }
        float* out = (float*)t.out + (long)sub * t.s_h;
        if (t.kind == FFK_TILE_V && (inner % 32 != 0 || (M & 31))) {         // the rows of a group may lie in two key tiles, or end in one
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int mrow = m0g + 8 * (v >> 2) + 4 * half + (v & 3);
                if (mrow >= M) continue;
                const unsigned hi = (unsigned)mrow / inner, lo = (unsigned)mrow - hi * inner;
                out[(long)hi * t.s_o + (long)(lo >> 5) * 1024 + acc_tile_off((int)(lo & 31), l32)] = x[v];
            }
            return;
        }
        if (t.kind == FFK_TILE_STRIDED && !by_rows && (inner % 16 != 0 || (M & 15))) {       // sixteen rows of a channel, wherever they end
            if (l32 >= left) return;
            int mrow = m0g + 16 * half;
            unsigned hi = t.inner < M ? (unsigned)mrow / inner : 0u, lo = (unsigned)mrow - hi * inner;
            float* p = out + (long)hi * t.s_o + (long)l32 * t.s_d;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                if (mrow + v < M) p[lo] = x[v];
                if (++lo == inner) {
                    lo = 0;
                    p += t.s_o;
                }
            }
            return;
        }
        // row of this lane (by rows), of its key tile (V) or first of its sixteen (channel-major: they never straddle `inner`)
        const int mrow = m0g + (by_rows ? n32 : t.kind == FFK_TILE_V ? 0 : 16 * half);
        unsigned hi = 0, lo = (unsigned)mrow;
        if (t.inner < M) {
            hi = lo / inner;
            lo -= hi * inner;
        }
        // The 64 bytes of every lane (null: none), four lanes side by side: by a lane's own 16-byte pieces every 64 bytes are four
        // requests to L2, and they, not the products, bound the launch.
        auto put = [&](float* p) __attribute__((always_inline)) {
            unsigned char* to = s_out + wave * G::OP;
#pragma unroll
            for (int a = 0; a < 4; ++a)
                *reinterpret_cast<f32x4*>(to + (lane + half) * 64 + ((a ^ (lane >> 2)) & 3) * 16) = f32x4{x[4 * a], x[4 * a + 1], x[4 * a + 2], x[4 * a + 3]};
            *reinterpret_cast<float**>(to + 65 * 64 + lane * 8) = p;
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int j = 0; j < 4; ++j) {                // rows (channels) 8 j .. 8 j + 7 and their other sixteen values
                const int h = lane >> 2 & 1, from = 8 * j + (lane >> 3) + 32 * h;
                const f32x4 y = *reinterpret_cast<const f32x4*>(to + (from + h) * 64 + ((lane ^ (from >> 2)) & 3) * 16);
                float* q = *reinterpret_cast<float* const*>(to + 65 * 64 + from * 8);
                if (q) *reinterpret_cast<f32x4*>(q + 4 * (lane & 3)) = y;
            }
            __builtin_amdgcn_wave_barrier();
        };
        if (t.kind == FFK_TILE_BIAS) {
            float* p = out + (long)(hi >> 5) * t.s_o + (long)(lo >> 5) * 1024 + qk_tile_off((int)(lo & 31), (int)(hi & 31));
            if (half == 0 && mrow < M) {
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    if (v < t.ncols) p[(long)v * t.s_h] = x[v];
            }
            return;
        }
        out += (long)hi * t.s_o;
        if (t.kind != FFK_TILE_STRIDED) {
            put(mrow >= M ? nullptr : out + (long)(lo >> 5) * 1024 + (t.kind == FFK_TILE_QK ? half * 512 + (int)(lo & 31) * 16 : (half * 32 + (by_rows ? (int)(lo & 31) : l32)) * 16));
            return;
        }
        if (!by_rows) {
            put(l32 < left && mrow < M ? out + lo + (long)l32 * t.s_d : nullptr);
            return;
        }
        const long off = (long)lo * t.s_i + 16 * half;
        if (t.gate && mrow < M) {
            const float* gate = (const float*)t.gate + (long)(t.gate_rows > 0 ? mrow % t.gate_rows : mrow) * t.gate_ld + 32 * sub + 16 * half;
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                if (16 * half + 4 * a >= left) break;
                const f32x4 g = *reinterpret_cast<const f32x4*>(gate + 4 * a);
#pragma unroll
                for (int e = 0; e < 4; ++e) x[4 * a + e] *= gate_factor(g[e], t.act);
            }
        }
        if (t.resid && mrow < M) {
            [[maybe_unused]] const float* r = (const float*)t.resid + (out - (float*)t.out) + off;
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                if (16 * half + 4 * a >= left) break;
                f32x4 y;
                if constexpr (ONE) y = rv[a];
                else y = *reinterpret_cast<const f32x4*>(r + 4 * a);
#pragma unroll
                for (int e = 0; e < 4; ++e) x[4 * a + e] += y[e];
            }
        }
        if (left >= 32) {
            put(mrow < M ? out + off : nullptr);
            return;
        }
        if (mrow >= M) return;
#pragma unroll
        for (int a = 0; a < 4; ++a) {                    // ncols is a multiple of 4
            if (16 * half + 4 * a >= left) break;
            *reinterpret_cast<f32x4*>(out + off + 4 * a) = f32x4{x[4 * a], x[4 * a + 1], x[4 * a + 2], x[4 * a + 3]};
        }
    };

    // products of R row groups with the first N slots, rows: W . A^T.  The weights are cut into their parts as they are used.
    auto products = [&](f32x16* acc, const unsigned char* ap, auto rows, auto n, auto rt) __attribute__((always_inline)) {
        constexpr int N = decltype(n)::value, R = decltype(rt)::value;
#pragma unroll
        for (int s = 0; s < N * R; ++s)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[s][v] = 0.0f;
        constexpr bool AHEAD = N * R == 1;     // the next step's operands are read and cut beside this step's products
        bf16x8 xf[2][R][3], w[2][N][3];
        auto rows_at = [&](int g) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < R; ++i)
#pragma unroll
                for (int p = 0; p < 3; ++p) xf[g & 1][i][p] = *reinterpret_cast<const bf16x8*>(ap + i * 32 * AP + g * 96 + p * 32);
        };
        auto weights_at = [&](int g) __attribute__((always_inline)) {
#pragma unroll
            for (int s = 0; s < N; ++s) {
                if constexpr (G::CUT) {
#pragma unroll
                    for (int p = 0; p < 3; ++p) w[g & 1][s][p] = wp[g][p];
                    continue;
                }
                const Split4 a = split4<true>(wf[s][2 * g]), b = split4<true>(wf[s][2 * g + 1]);     // all ahead of the loop over slabs they would not fit
#pragma unroll
                for (int p = 0; p < 3; ++p) w[g & 1][s][p] = split_frag(a, b, p);
            }
        };
        if (AHEAD) {
            rows_at(0);
            weights_at(0);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int g = 0; g < K / 16; ++g) {
            if (!AHEAD) {
                rows_at(g);
                weights_at(g);
            } else if (g + 1 < K / 16) {
                rows_at(g + 1);
                __builtin_amdgcn_sched_barrier(0);
                weights_at(g + 1);
            }
#pragma unroll
            for (int t = 0; t < 6; ++t)
#pragma unroll
                for (int s = 0; s < N; ++s)
#pragma unroll
                    for (int i = 0; i < R; ++i) {
                        if constexpr (rows.value) Mma<bf16_t>::mma(acc[s * R + i], w[g & 1][s][SPLIT_A[t]], xf[g & 1][i][SPLIT_B[t]]);
                        else Mma<bf16_t>::mma(acc[s * R + i], xf[g & 1][i][SPLIT_B[t]], w[g & 1][s][SPLIT_A[t]]);
                        if (AHEAD && !G::CUT) {
                            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(0x002, 8, 0);
                        }
                    }
            __builtin_amdgcn_sched_barrier(0);
        }
        // infinite operands, whose parts make NaN of every product: those sums with the fp32 instructions, the others keep their bits
        float sum = acc[0][0];
#pragma unroll
        for (int v = 1; v < 16 * N * R; ++v) sum += acc[v >> 4][v & 15];
        if (__builtin_expect(__any(sum - sum != 0.0f), 0)) {
#pragma unroll
            for (int s = 0; s < N; ++s)
#pragma unroll
                for (int i = 0; i < R; ++i) {
                    f32x16& y = acc[s * R + i];
                    int l = lane;
                    asm volatile("" : "+v"(l));              // no address of it kept in registers on the way here
                    f32x4* const kept = reinterpret_cast<f32x4*>(s_out + wave * G::OP) + l;         // free between this wave's stores
#pragma unroll
                    for (int a = 0; a < 4; ++a) kept[a * 64] = f32x4{y[4 * a], y[4 * a + 1], y[4 * a + 2], y[4 * a + 3]};
#pragma unroll
                    for (int v = 0; v < 16; ++v) y[v] = 0.0f;
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int g = 0; g < K / 16; ++g) {
                        const unsigned char* xp = ap + i * 32 * AP + g * 96;
                        [[maybe_unused]] bf16x8 wq[3];
                        if constexpr (G::CUT) {
#pragma unroll
                            for (int p = 0; p < 3; ++p) {
                                u32x4 q = __builtin_bit_cast(u32x4, wp[g][p]);
                                asm volatile("" : "+v"(q));      // whatever is made of it stays here
                                wq[p] = __builtin_bit_cast(bf16x8, q);
                            }
                        }
#pragma unroll
                        for (int e = 0; e < 8; ++e) {
                            const float x = split_sum(reinterpret_cast<const bf16_t*>(xp)[e], reinterpret_cast<const bf16_t*>(xp + 32)[e], reinterpret_cast<const bf16_t*>(xp + 64)[e]);
                            float w;
                            if constexpr (G::CUT) w = split_sum(wq[0][e], wq[1][e], wq[2][e]);
                            else w = wf[s][2 * g + (e >> 2)][e & 3];
                            if constexpr (rows.value) y = __builtin_amdgcn_mfma_f32_32x32x2f32(w, x, y, 0, 0, 0);
                            else y = __builtin_amdgcn_mfma_f32_32x32x2f32(x, w, y, 0, 0, 0);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
#pragma unroll
                    for (int a = 0; a < 4; ++a) {
                        const f32x4 k = kept[a * 64];
#pragma unroll
                        for (int e = 0; e < 4; ++e) y[4 * a + e] = k[e] == k[e] ? k[e] : y[4 * a + e];
                    }
                }
        }
    };
    const int nslabs = (M + BM - 1) / BM;
    const bool early = !ONE && wave >= G::WAVES / 2;
    // R row groups against one unit.  With the last ones of a slab the next slab comes: its loads are issued before the products
    // and normalised and written to LDS after them, ahead of this block's stores - a wait for loads is a wait for the stores
    // issued before them.  The waves of `early` do that ahead of the products, with loads of the iteration before, so that the two
    // waves of a SIMD are not at their vector instructions at the same time.
    auto block = [&](int u, const unsigned char* ap, int m0g, const float* sm, auto n, auto rt, int next, int nbuf) __attribute__((always_inline)) {
        constexpr int N = decltype(n)::value, R = decltype(rt)::value;
        f32x16 acc[N * R];
        f32x4 rv[R][4];
        if constexpr (ONE) {                             // the residual arrives behind the products
            const ffk_tile& t = d.tiles[u >> 2];
            const int sub = w3_sub<GLU>(t, u), left = t.ncols - 32 * sub;
#pragma unroll
            for (int i = 0; i < R; ++i) {
                const int mrow = m0g + 32 * i + n32;
                if (t.resid && mrow < M) {
                    const unsigned hi = t.inner < M ? (unsigned)mrow / (unsigned)t.inner : 0u, lo = (unsigned)mrow - hi * (unsigned)t.inner;
                    const float* r = (const float*)t.resid + (long)sub * t.s_h + (long)hi * t.s_o + (long)lo * t.s_i + 16 * half;
#pragma unroll
                    for (int a = 0; a < 4; ++a)
                        if (16 * half + 4 * a < left) rv[i][a] = *reinterpret_cast<const f32x4*>(r + 4 * a);
                }
            }
        }
        if (next >= 0) {
            if (early) commit(nbuf);
            const int n2 = early ? next + (int)gridDim.x : next;
            if (n2 < nslabs) fetch(n2);
        }
        if (w3_by_rows(d.tiles[u >> 2])) products(acc, ap, std::true_type{}, n, rt);
        else products(acc, ap, std::false_type{}, n, rt);
        if (next >= 0 && !early) commit(nbuf);
#pragma unroll
        for (int i = 0; i < R; ++i)
            if (i == 0 || m0g + 32 * i < M)
                store(u, s_bias + (wave * NS) * 32, acc[i], acc[(N - 1) * R + i], m0g + 32 * i, sm + 32 * i, rv[i]);
    };

    int slab = blockIdx.x;                               // grid.x <= nslabs
    if (!ONE) fetch(slab);
    commit(0);
    if (!ONE) __builtin_amdgcn_s_waitcnt(0x0f70);        // vmcnt(0): the products of the loop wait for no weights
    if (early && slab + (int)gridDim.x < nslabs) fetch(slab + gridDim.x);
    lds_barrier();
    int buf = 0;
    typedef std::integral_constant<int, 1> I1;
    constexpr int PAIR = GLU ? 1 : W3_RG;                // row groups multiplied together
    typedef std::integral_constant<int, PAIR> IR;
    for (; slab < nslabs; slab += gridDim.x) {
        const int next = !ONE && slab + (int)gridDim.x < nslabs ? slab + (int)gridDim.x : -1;
        const int nbuf = buf ^ 1;
        if (units[0] < 0 && next >= 0) {
            if (!early) fetch(next);
            commit(nbuf);
            if (early && next + (int)gridDim.x < nslabs) fetch(next + (int)gridDim.x);
        }
        const int m0 = slab * BM;
        auto rows_of = [&](int rg) { return s_a + (G::NBUF == 2 ? buf : 0) * (BM * AP) + (rg * 32 + n32) * AP + half * 16; };
        const float* sm = s_mask + buf * BM;
        const int rg = halves ? wave / (W3_WAVES / W3_RG) : 0;
        if (units[0] < 0) {
        } else if (halves && W3_RG > 1) {                // this wave's half of the slab
            if (m0 + rg * 32 < M) {
                if (NS == 2 && units[NS - 1] >= 0) block(units[0], rows_of(rg), m0 + rg * 32, sm + rg * 32, std::integral_constant<int, NS>{}, I1{}, next, nbuf);
                else block(units[0], rows_of(rg), m0 + rg * 32, sm + rg * 32, I1{}, I1{}, next, nbuf);
            }
        } else {
#pragma unroll
            for (int g = 0; g < W3_RG; g += PAIR) {
                if (m0 + g * 32 >= M) break;             // in the last slab only
                const int nx = g + PAIR == W3_RG ? next : -1;
                if (NS == 2 && units[NS - 1] >= 0) block(units[0], rows_of(g), m0 + g * 32, sm + g * 32, std::integral_constant<int, NS>{}, IR{}, nx, nbuf);
                else block(units[0], rows_of(g), m0 + g * 32, sm + g * 32, I1{}, IR{}, nx, nbuf);
            }
        }
        if (next < 0) break;
        lds_barrier();
        buf = nbuf;
    }
}

bool w3_tile_ok(const ffk_linear_desc& d, const ffk_tile& t) {
    auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    if (t.inner <= 0 || t.ncols <= 0 || !al16(t.out) || t.xtail) return false;
    if (t.kind == FFK_TILE_BIAS) return t.ncols <= 16 && !t.resid && !t.gate && !t.glu;
    if (t.kind == FFK_TILE_STRIDED && t.s_d == 1) {
        if (t.ncols % 4 || t.s_o % 4 || t.s_i % 4 || t.s_h % 4) return false;
        return (!t.resid || al16(t.resid)) && (!t.gate || (al16(t.gate) && t.gate_ld % 4 == 0));
    }
    if (t.resid || t.gate || t.s_o % 4 || t.s_h % 4) return false;
    if (t.kind != FFK_TILE_STRIDED) return t.ncols % 32 == 0 && !t.glu;
    return t.s_i == 1 && t.s_d % 4 == 0;
}

template <int K, bool GLU, bool ONE, int BM, bool CM = false>
int w3_launch(const W3Args& a, int gx, int groups, hipStream_t st) {
    typedef W3Geo<K, GLU, ONE, BM> G;
    const size_t smem = G::NBUF * (size_t)BM * G::AP + G::WAVES * G::OP + (2 * BM + G::WAVES * G::SLOTS * 32) * sizeof(float);
    static FfkLdsReservation lds_reserved;
    const int rc = ffk_reserve_lds(lds_reserved, (const void*)linear_ws32_kernel<K, GLU, ONE, BM, CM>, smem, "ffk_fused_linear");
    if (rc != FFK_OK) return rc;
    linear_ws32_kernel<K, GLU, ONE, BM, CM><<<dim3(gx, groups), G::THREADS, smem, st>>>(a);
    return ffk_check_launch("ffk_fused_linear");
}

}  // namespace

// Launches the fp32 weights-stationary kernel if it can take this (already validated) descriptor and returns 1 with the launch
// status in *status; returns 0 if the caller has to use the staged kernel.
int ffk_linear_ws32_try(const ffk_linear_desc* d, hipStream_t st, int* status) {
    if (d->dtype != FFK_F32 || (d->K != 128 && d->K != 256) || (d->a_chanmajor && d->K != 128) || d->a2 || d->ln_folded || d->variant == FFK_LINEAR_STAGED)
        return 0;
    if ((reinterpret_cast<uintptr_t>(d->ln_gamma) & 15) || (reinterpret_cast<uintptr_t>(d->ln_beta) & 15)) return 0;
    bool chan_major = false, v_tiles = false, glu = false;
    W3Args a;
    a.mask_tile = -1;
    a.n_units = 0;
    const char* a0 = (const char*)d->a;
    for (int i = 0; i < d->n_tiles; ++i) {
        const ffk_tile& t = d->tiles[i];
        if (!w3_tile_ok(*d, t) || (t.glu && d->K != 128)) return 0;
        // groups of workgroups read the rows at different times: a launch over its own input is not for this kernel
        const char* o = (const char*)t.out;
        if (o >= a0 && o < a0 + (size_t)d->M * d->K * 4) return 0;
        chan_major = chan_major || !(w3_by_rows(t) || t.kind == FFK_TILE_V);
        v_tiles = v_tiles || t.kind == FFK_TILE_V;
        glu = glu || t.glu;
        if (t.rowmask) {
            if (a.mask_tile < 0) a.mask_tile = i;
            const ffk_tile& f = d->tiles[a.mask_tile];
            if (t.rowmask != f.rowmask || t.inner != f.inner || t.m_so != f.m_so || t.m_si != f.m_si) return 0;
        }
        const int n = t.kind == FFK_TILE_BIAS ? 1 : (t.ncols + 31) / 32;
        for (int u = 0; u < n; ++u) a.unit[a.n_units++] = (signed char)(4 * i + (t.glu ? 2 * u : u));
    }
    if (d->a_chanmajor && glu) return 0;
    if (chan_major && v_tiles) return 0;                 // they need different row orders within a group
    a.row_perm = chan_major ? 1 : 0;
    a.d = *d;
    // Persistent workgroups of eight waves, or one slab per workgroup of four waves with a unit each (two or three workgroups per CU):
    // the latter starts sooner, spreads few rows over more CUs and is alone built for channel-major operands and for GLU units.  In
    // microseconds, with a round = one workgroup per CU:
    //   one slab of 32 rows: K = 128 4 + 3.4 per round (GLU 5 + 5), K = 256 3 + 5.7; of 64 rows (K = 128): 5 + 5.5 per round (GLU
    //     4 + 7.8), 0.6 of it with fewer units than waves;
    //   persistent: 8 to 8.5, then per slab (64 rows at K = 128, 32 at K = 256) 1.6 (0.7) and 3.0 (3.2) for every four units: one per SIMD.
    // Measured, one slab of 32 / of 64 rows / persistent, K = 128: 65 536 rows, 1 024 channels 220 / 179 / 130 us, 512 111 / 91 / 68, 128
    // 30.7 / 26.6 / 25.9, 32 23.2 / 18.3 / 22.7; 36 864 rows, 512 channels 66 / 54 / 45; 13 689 28.3 / 27.0 / 22.4; 8 192 17.6 / 14.7 / 15.9;
    // 4 096 10.4 / 11.5 / 12.1; GLU 256 + 128 channels, 65 536 rows 127 / 99 / 146, 8 192 19.8 / 17.8 / 24.8, 4 096 12.5 / 15.3 / 18.2.
    // K = 256, 1 024 channels: 32 768 rows 186 / - / 122, 8 192 49.5 / - / 36.5, 4 096 26.3 / - / 21.7, 2 048 14.3 / - / 16.1; 256 channels:
    // 32 768 46.9 / - / 35.2, 8 192 13.4 / - / 14.8.
    const int quads = ffk_cdiv(a.n_units, 4), sl32 = ffk_cdiv(d->M, 32), sl64 = ffk_cdiv(d->M, 64);
    const long r32 = ffk_cdiv((long)sl32 * quads, W3_CUS), r64 = ffk_cdiv((long)sl64 * quads, W3_CUS);
    const double few = a.n_units < 4 ? 0.6 : 1.0;
    const double c32 = d->K == 256 ? 3 + 5.7 * r32 : glu ? 5 + 5.0 * r32 : 4 + 3.4 * r32;
    const double c64 = d->K == 256 ? 1e30 : glu ? std::max(15.0, 4 + 7.8 * r64) : std::max(11.0, 5 + 5.5 * few * r64);
    int gx = 1, groups = 1;
    double best = 1e30;
    if (!glu && !d->a_chanmajor) {
        const int nslabs = d->K == 256 ? sl32 : sl64;
        for (int per = 8; per >= 4; per -= 4) {
            const int g = ffk_cdiv(a.n_units, per), each = ffk_cdiv(a.n_units, g);
            int x = W3_CUS / g;
            x = x < nslabs ? x : nslabs;
            const double grain = ffk_cdiv(each, 4), cost = d->K == 256 ? 8.5 + ffk_cdiv(nslabs, x) * (0.7 + 3.2 * grain) : 8 + ffk_cdiv(nslabs, x) * (1.6 + 3.0 * grain);
            if (cost < best) {
                best = cost;
                gx = x;
                groups = ffk_cdiv(a.n_units, each);
                a.per_group = each;
            }
        }
    }
    if (c32 <= best || c64 <= best) {
        a.per_group = 4;
        const bool small = c32 <= c64;
        gx = small ? sl32 : sl64;
        if (d->a_chanmajor) *status = small ? w3_launch<128, false, true, 32, true>(a, gx, quads, st) : w3_launch<128, false, true, 64, true>(a, gx, quads, st);
        else if (d->K == 256) *status = w3_launch<256, false, true, 32>(a, gx, quads, st);
        else if (glu) *status = small ? w3_launch<128, true, true, 32>(a, gx, quads, st) : w3_launch<128, true, true, 64>(a, gx, quads, st);
        else *status = small ? w3_launch<128, false, true, 32>(a, gx, quads, st) : w3_launch<128, false, true, 64>(a, gx, quads, st);
        return 1;
    }
    *status = d->K == 256 ? w3_launch<256, false, false, 32>(a, gx, groups, st) : w3_launch<128, false, false, 64>(a, gx, groups, st);
    return 1;
}
