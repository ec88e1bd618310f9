// Weights-stationary variant of the fused linear layer in fp32 (see ffk_fused_linear in include/ffk.h), K = 128 or 256.
//
// v_mfma_f32_32x32x2_f32 does 64 multiply-adds per cycle and SIMD, and it does not overlap with vector instructions of other
// waves (a SIMD given 491 us of one and 617 us of the other takes 1 050 us; with bf16 products they hide each other).  So what
// bounds a launch is products plus vector instructions, and the kernel is arranged to need few of the latter per product: a
// row is normalised once for up to 16 weight units of 32 rows, weights stay in registers (two units per wave at K = 128, value
// and gate of a GLU unit, one at K = 256), activations stream through a double-buffered slab of 64 rows in LDS whose 16-byte
// fragments feed four products each, and a wave stores its blocks straight from registers (exchanging pieces between lanes
// for wider stores cost 30 % of the launch).  Measured against the LDS-staged kernel: 32 768 rows, 256 -> 1 024: 263 -> 168 us
// (102 TFLOP/s); 65 536 rows, 128 -> 1 024: 234 -> 181 us; 128 -> 128: 42.5 -> 39.7 us.
//
// Persistent workgroups of eight waves, one per CU: the units of a launch are dealt to groups (blockIdx.y), each with workgroups of
// its own over all rows; unit i of a group goes to wave i % 8, or, in a group of up to four, to waves i and i + 4, which take one
// half of the slab each - so the SIMDs have equal shares of any multiple of four units.  Few rows take workgroups of four waves
// with one slab and one unit per wave (ONE): what such a launch waits for is the weights, which come as whole lines while the rows
// are normalised, and the residual, which is requested before the products.  1 024 rows, 256 -> 256: 21.5 us on the staged
// kernel, 10.8 us; 4 096 rows, 128 -> 128 from channel-major rows: 20.6 -> 9.7 us.
//   by rows   (plain, q / k tiles, pair-bias tiles): product W . A^T, a lane owns one row and 16 consecutive channels
//             (64 bytes; weight rows are taken through tau, except for accumulator-order tiles)
//   by columns (v tiles, channel-major outputs): A . W^T, a lane owns one channel and 16 rows
#include "ffk_common.h"
#include <type_traits>

namespace {

constexpr int W3_MAXU = FFK_MAX_TILES * 4, W3_CUS = 256;

// ONE: every workgroup has one slab of BM rows; else workgroups are persistent and the slab is double-buffered
template <int K, bool GLU, bool ONE, int BM_> struct W3Geo {
    static constexpr int WAVES = ONE ? 4 : 8, THREADS = 64 * WAVES, BM = BM_, RG = BM / 32;
    static constexpr int KF = K / 8;                     // fragments (four MFMAs each) per unit
    static constexpr int AP = K * 4 + 16;                // LDS row pitch in bytes
    static constexpr int LPR = K / 4;                    // lanes per row
    static constexpr int RPP = THREADS / LPR;            // rows fetched per pass
    static constexpr int NP = BM / RPP;                  // passes: 4, 8 or 16
    static constexpr int SLOTS = K == 128 && (GLU || !ONE) ? 2 : 1;       // weight units in a wave's registers
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
__global__ __launch_bounds__(ONE ? 256 : 512, 2) void linear_ws32_kernel(const W3Args args) {
    typedef W3Geo<K, GLU, ONE, BM> G;
    constexpr int NS = G::SLOTS, KF = G::KF, AP = G::AP, LPR = G::LPR, RPP = G::RPP, NP = G::NP, PF = 3;
    constexpr int W3_WAVES = G::WAVES, W3_RG = G::RG;
    const ffk_linear_desc& d = args.d;
    extern __shared__ __align__(16) unsigned char smem[];
    unsigned char* s_a = smem;                                                  // [NBUF][BM][AP]
    float* s_mask = reinterpret_cast<float*>(smem + G::NBUF * BM * AP);         // [NBUF][BM]
    float* s_bias = s_mask + G::NBUF * BM;                                            // [wave][slot][32]
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
        const int i = halves ? wave % (W3_WAVES / W3_RG) : wave + (GLU ? 0 : s * W3_WAVES);
        int u = i < n_u && !(halves && s && !GLU) ? args.unit[u0 + i] : -1;
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
                wf[s][p + i] = *reinterpret_cast<const f32x4*>(stage + wl * 128 + (((2 * i + half) ^ (wl & 7)) * 16));
        }
        if (half == 0) s_bias[(wave * NS + s) * 32 + l32] = tb[s];
    }
    lds_barrier();                                       // every wave is done with the staging area
    const int n32 = args.row_perm ? ffk_tau(l32) : l32;

    // ---- slab streaming ----
    if (!ONE && ln) {
        gam = *reinterpret_cast<const f32x4*>((const float*)d.ln_gamma + c4 * 4);
        bet = *reinterpret_cast<const f32x4*>((const float*)d.ln_beta + c4 * 4);
    }
    auto commit = [&](int buf) __attribute__((always_inline)) {
        unsigned char* sa = s_a + buf * (BM * AP);
        if constexpr (CM) {                              // transposed through LDS; rows are whole only there
#pragma unroll
            for (int i = 0; i < 4 * NP; ++i)
                *reinterpret_cast<float*>(sa + (tid & (BM - 1)) * AP + (tid / BM + i * (G::THREADS / BM)) * 4) = pre[i >> 2][i & 3];
            if (rm && tid < BM) s_mask[buf * BM + tid] = pm;
            if (!ln) return;
            lds_barrier();
#pragma unroll
            for (int i = 0; i < NP; ++i) pre[i] = *reinterpret_cast<const f32x4*>(sa + (r0 + RPP * i) * AP + c4 * 16);
        }
#pragma unroll
        for (int i = 0; i < NP; i += 4) {
            if (ln) ffk_ln_rows4<LPR>(pre + i, gam, bet, d.ln_eps);
#pragma unroll
            for (int j = i; j < i + 4; ++j) *reinterpret_cast<f32x4*>(sa + (r0 + RPP * j) * AP + c4 * 16) = pre[j];
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
        if (mrow >= M) return;
        unsigned hi = 0, lo = (unsigned)mrow;
        if (t.inner < M) {
            hi = lo / inner;
            lo -= hi * inner;
        }
        auto put = [&](float* p) __attribute__((always_inline)) {
#pragma unroll
            for (int a = 0; a < 4; ++a) *reinterpret_cast<f32x4*>(p + 4 * a) = f32x4{x[4 * a], x[4 * a + 1], x[4 * a + 2], x[4 * a + 3]};
        };
        if (t.kind == FFK_TILE_BIAS) {
            float* p = out + (long)(hi >> 5) * t.s_o + (long)(lo >> 5) * 1024 + qk_tile_off((int)(lo & 31), (int)(hi & 31));
            if (half == 0) {
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    if (v < t.ncols) p[(long)v * t.s_h] = x[v];
            }
            return;
        }
        out += (long)hi * t.s_o;
        if (t.kind != FFK_TILE_STRIDED) {
            put(out + (long)(lo >> 5) * 1024 + (t.kind == FFK_TILE_QK ? half * 512 + (int)(lo & 31) * 16 : (half * 32 + (by_rows ? (int)(lo & 31) : l32)) * 16));
            return;
        }
        if (!by_rows) {
            if (l32 < left) put(out + lo + (long)l32 * t.s_d);
            return;
        }
        const long off = (long)lo * t.s_i + 16 * half;
        if (t.gate) {
            const float* gate = (const float*)t.gate + (long)(t.gate_rows > 0 ? mrow % t.gate_rows : mrow) * t.gate_ld + 32 * sub + 16 * half;
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                if (16 * half + 4 * a >= left) break;
                const f32x4 g = *reinterpret_cast<const f32x4*>(gate + 4 * a);
#pragma unroll
                for (int e = 0; e < 4; ++e) x[4 * a + e] *= gate_factor(g[e], t.act);
            }
        }
        if (t.resid) {
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
            put(out + off);
            return;
        }
#pragma unroll
        for (int a = 0; a < 4; ++a) {                    // ncols is a multiple of 4
            if (16 * half + 4 * a >= left) break;
            *reinterpret_cast<f32x4*>(out + off + 4 * a) = f32x4{x[4 * a], x[4 * a + 1], x[4 * a + 2], x[4 * a + 3]};
        }
    };

    // products of one row group with slots S0 .. S0 + N - 1, rows: W . A^T
    auto products = [&](f32x16* acc, const unsigned char* ap, auto rows, auto s0, auto n) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < n.value; ++s)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[s][v] = 0.0f;
        f32x4 af[PF];                                    // fragments in flight
#pragma unroll
        for (int f = 0; f < PF; ++f) af[f] = *reinterpret_cast<const f32x4*>(ap + f * 32);
        __builtin_amdgcn_sched_group_barrier(0x100, PF, 0);
#pragma unroll
        for (int f = 0; f < KF; ++f) {
            const f32x4 x = af[f % PF];
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int s = 0; s < n.value; ++s) {
                    const float w = wf[s0.value + s][f][e];
                    if constexpr (rows.value) acc[s] = __builtin_amdgcn_mfma_f32_32x32x2f32(w, x[e], acc[s], 0, 0, 0);
                    else acc[s] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[e], w, acc[s], 0, 0, 0);
                }
            __builtin_amdgcn_sched_group_barrier(0x008, 4 * n.value, 0);
            if (f + PF < KF) {
                af[f % PF] = *reinterpret_cast<const f32x4*>(ap + (f + PF) * 32);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            }
        }
    };
    // One row group against one unit.  With the last one of a slab the next slab comes: its loads are issued before the products
    // and normalised and written to LDS after them, ahead of this block's stores - a wait for loads is a wait for the stores
    // issued after them.
    auto block = [&](int u, const unsigned char* ap, int m0g, const float* sm, auto s0, auto n, int next, int nbuf) __attribute__((always_inline)) {
        f32x16 acc[n.value];
        f32x4 rv[4];
        if constexpr (ONE) {                             // the residual arrives behind the products
            const ffk_tile& t = d.tiles[u >> 2];
            const int sub = w3_sub<GLU>(t, u), mrow = m0g + n32, left = t.ncols - 32 * sub;
            if (t.resid && mrow < M) {
                const unsigned hi = t.inner < M ? (unsigned)mrow / (unsigned)t.inner : 0u, lo = (unsigned)mrow - hi * (unsigned)t.inner;
                const float* r = (const float*)t.resid + (long)sub * t.s_h + (long)hi * t.s_o + (long)lo * t.s_i + 16 * half;
#pragma unroll
                for (int a = 0; a < 4; ++a)
                    if (16 * half + 4 * a < left) rv[a] = *reinterpret_cast<const f32x4*>(r + 4 * a);
            }
        }
        if (next >= 0) fetch(next);
        if (w3_by_rows(d.tiles[u >> 2])) products(acc, ap, std::true_type{}, s0, n);
        else products(acc, ap, std::false_type{}, s0, n);
        if (next >= 0) commit(nbuf);
        store(u, s_bias + (wave * NS + s0.value) * 32, acc[0], acc[n.value - 1], m0g, sm, rv);
    };

    const int nslabs = (M + BM - 1) / BM;
    int slab = blockIdx.x;                               // grid.x <= nslabs
    if (!ONE) fetch(slab);
    commit(0);
    if (!ONE) __builtin_amdgcn_s_waitcnt(0x0f70);        // vmcnt(0): the products of the loop wait for no weights
    lds_barrier();
    int buf = 0;
    typedef std::integral_constant<int, 0> I0;
    typedef std::integral_constant<int, 1> I1;
    for (; slab < nslabs; slab += gridDim.x) {
        const int next = !ONE && slab + (int)gridDim.x < nslabs ? slab + (int)gridDim.x : -1;
        if (units[0] < 0 && next >= 0) {
            fetch(next);
            commit(buf ^ 1);
        }
        const int rg_end = halves && wave < W3_WAVES / W3_RG ? 1 : W3_RG;
        for (int rg = halves ? wave / (W3_WAVES / W3_RG) : 0; rg < rg_end && units[0] >= 0; ++rg) {
            const int m0g = slab * BM + rg * 32;
            if (m0g >= M) break;                         // in the last slab only
            const int nx = rg + 1 == rg_end ? next : -1;
            const unsigned char* ap = s_a + buf * (BM * AP) + (rg * 32 + n32) * AP + half * 16;
            const float* sm = s_mask + buf * BM + rg * 32;
            if constexpr (GLU) {
                if (units[NS - 1] >= 0) block(units[0], ap, m0g, sm, I0{}, std::integral_constant<int, NS>{}, nx, buf ^ 1);
                else block(units[0], ap, m0g, sm, I0{}, I1{}, nx, buf ^ 1);
            } else {
                block(units[0], ap, m0g, sm, I0{}, I1{}, units[NS - 1] >= 0 && NS == 2 ? -1 : nx, buf ^ 1);
                if constexpr (NS == 2)
                    if (units[1] >= 0) block(units[1], ap, m0g, sm, I1{}, I1{}, nx, buf ^ 1);
            }
        }
        if (next < 0) break;
        lds_barrier();
        buf ^= 1;
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
    const size_t smem = G::NBUF * (size_t)BM * G::AP + (G::NBUF * BM + G::WAVES * G::SLOTS * 32) * sizeof(float);
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
    // Persistent workgroups of eight waves, or one slab per workgroup of four waves with a unit each (two to four workgroups per CU):
    // the latter starts sooner, spreads few rows over more CUs and is alone built for channel-major operands.  In microseconds:
    //   one slab: a start of 2 to 6.5, then for every workgroup of a CU about twice its products, which take 2 048 cycles per 32 x 32
    //     block of K = 64 (2.05 x for 32 rows, 1.9 x for 64, 1.6 x for 64 rows of GLU units, whose products are twice as many)
    //   persistent: a start of 7 to 10, then at 1 800 cycles per us, per slab, 2 x 2 048 per 64 x 32 block of K = 64 with four units (one
    //     per SIMD) as the grain, LayerNorm and staging 12 per row and K = 64, and 3 000 for what is in flight at the slab's
    //     barrier; fewer groups normalise the rows less often, more groups spread few rows over the CUs.
    // Measured, staged kernel before / one slab of 32 / of 64 rows / persistent: 2 048 rows, 256 -> 1 024: 28.3 / 18.0 / 19.7 / 19.8 us;
    // 256 -> 256: 22.5 / 11.2 / 16.3 / 17.2; 4 096 rows, 128 -> 512: 16.9 / 11.8 / 12.9 / 15.2; 36 864 rows 89.6 / 65.0 / 65.9 / 65.5;
    // 65 536 rows, GLU 256 + 128 channels: - / 166 / 134 / 147; 128 -> 512: - / 102.8 / 108.6 / 95.2.
    const int nslabs = ffk_cdiv(d->M, 64), kk = d->K / 64;
    constexpr double US_PER_BLOCK = 2048.0 / 2350;
    const int quads = ffk_cdiv(a.n_units, 4);
    const double blk = US_PER_BLOCK * kk * (glu ? 2 : 1);
    const double c32 = (glu ? 2.0 : 3.5) + ffk_cdiv((long)ffk_cdiv(d->M, 32) * quads, W3_CUS) * blk * 2.05;
    const double c64 = (glu ? 6.5 : 4.0) + ffk_cdiv((long)nslabs * quads, W3_CUS) * blk * 2 * (glu ? 1.6 : 1.9);
    const int cap = 8 * (glu || d->K == 256 ? 1 : 2);
    int gx = 1, groups = 1;
    double best = 1e30;
    for (int per = cap; per >= 4; per -= 4) {
        const int g = ffk_cdiv(a.n_units, per), each = ffk_cdiv(a.n_units, g);
        int x = W3_CUS / g;
        x = x < nslabs ? x : nslabs;
        const double cost = (d->K == 128 ? 10.0 : 7.0) + ffk_cdiv(nslabs, x) * (ffk_cdiv(each, 4) * 4096.0 * kk * (glu ? 2 : 1) + 64 * 12.0 * kk + 3000.0) / 1800;
        if (cost < best) {
            best = cost;
            gx = x;
            groups = ffk_cdiv(a.n_units, each);
            a.per_group = each;
        }
    }
    if (d->a_chanmajor || c32 <= best || c64 <= best) {
        a.per_group = 4;
        const bool small = c32 <= c64;
        gx = ffk_cdiv(d->M, small ? 32 : 64);
        if (d->a_chanmajor) *status = small ? w3_launch<128, false, true, 32, true>(a, gx, quads, st) : w3_launch<128, false, true, 64, true>(a, gx, quads, st);
        else if (d->K == 256) *status = small ? w3_launch<256, false, true, 32>(a, gx, quads, st) : w3_launch<256, false, true, 64>(a, gx, quads, st);
        else if (glu) *status = small ? w3_launch<128, true, true, 32>(a, gx, quads, st) : w3_launch<128, true, true, 64>(a, gx, quads, st);
        else *status = small ? w3_launch<128, false, true, 32>(a, gx, quads, st) : w3_launch<128, false, true, 64>(a, gx, quads, st);
        return 1;
    }
    if (d->K == 256) *status = w3_launch<256, false, false, 64>(a, gx, groups, st);
    else *status = glu ? w3_launch<128, true, false, 64>(a, gx, groups, st) : w3_launch<128, false, false, 64>(a, gx, groups, st);
    return 1;
}
