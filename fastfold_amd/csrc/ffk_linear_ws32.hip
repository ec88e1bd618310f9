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
// One persistent workgroup of eight waves per CU.  The units of a launch are dealt to groups (blockIdx.y), each with workgroups
// of its own over all rows; unit i of a group goes to wave i % 8, or, in a group of up to four, to waves i and i + 4, which
// take one half of the slab each - so the SIMDs have equal shares of any multiple of four units.
//   by rows   (plain, q / k tiles, pair-bias tiles): product W . A^T, a lane owns one row and 16 consecutive channels
//             (64 bytes; weight rows are taken through tau, except for accumulator-order tiles)
//   by columns (v tiles, channel-major outputs): A . W^T, a lane owns one channel and 16 rows
#include "ffk_common.h"
#include <type_traits>

namespace {

constexpr int W3_BM = 64, W3_RG = 2, W3_WAVES = 8, W3_THREADS = 512, W3_MAXU = FFK_MAX_TILES * 4, W3_CUS = 256;

template <int K> struct W3Geo {
    static constexpr int KF = K / 8;                     // fragments (four MFMAs each) per unit
    static constexpr int AP = K * 4 + 16;                // LDS row pitch in bytes
    static constexpr int LPR = K / 4;                    // lanes per row
    static constexpr int RPP = W3_THREADS / LPR;         // rows fetched per pass
    static constexpr int NP = W3_BM / RPP;               // passes: 4 or 8
    static constexpr int SLOTS = K == 128 ? 2 : 1;       // weight units in a wave's registers
};

struct W3Args {
    ffk_linear_desc d;
    signed char unit[W3_MAXU];                           // first 32-row block of the weights (4 per tile) of every unit
    int n_units, per_group;                              // units of the launch; of a group (the last one may have fewer)
    int row_perm;                                        // rows of a group through tau (launches with channel-major tiles)
    int mask_tile;                                       // tile whose row mask the launch uses, -1: none
};

__device__ __forceinline__ int w3_tau(int i) { return ((i >> 2) & 1) * 16 + (i >> 3) * 4 + (i & 3); }

__host__ __device__ __forceinline__ bool w3_by_rows(const ffk_tile& t) {
    return t.kind == FFK_TILE_QK || t.kind == FFK_TILE_ACC || t.kind == FFK_TILE_BIAS || (t.kind == FFK_TILE_STRIDED && t.s_d == 1);
}

// GLU: the launch has GLU tiles; the slots of a wave are then value and gate of one unit (a plain unit leaves the second empty)
template <int K, bool GLU>
__global__ __launch_bounds__(W3_THREADS, 2) void linear_ws32_kernel(const W3Args args) {
    typedef W3Geo<K> G;
    constexpr int NS = G::SLOTS, KF = G::KF, AP = G::AP, LPR = G::LPR, RPP = G::RPP, NP = G::NP, BM = W3_BM, PF = 3;
    const ffk_linear_desc& d = args.d;
    extern __shared__ __align__(16) unsigned char smem[];
    unsigned char* s_a = smem;                                                  // [2][BM][AP]
    float* s_mask = reinterpret_cast<float*>(smem + 2 * BM * AP);               // [2][BM]
    float* s_bias = s_mask + 2 * BM;                                            // [wave][slot][32]
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    const int M = d.M;
    const float* A = (const float*)d.a;
    const float* W = (const float*)d.w;

    const int u0 = blockIdx.y * args.per_group, n_u = args.n_units - u0 < args.per_group ? args.n_units - u0 : args.per_group;
    const bool halves = n_u <= W3_WAVES / W3_RG;         // two waves per unit
    int units[NS];                                       // -1: none
    f32x4 wf[NS][KF];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int i = halves ? wave % (W3_WAVES / W3_RG) : wave + (GLU ? 0 : s * W3_WAVES);
        int u = i < n_u && !(halves && s && !GLU) ? args.unit[u0 + i] : -1;
        if (GLU && s) u = u >= 0 && d.tiles[u >> 2].glu ? u + 1 : -1;
        units[s] = u;
        const ffk_tile& t = d.tiles[u >= 0 ? u >> 2 : 0];
        const float* wp = W + (long)((u >= 0 ? u : 0) * 32 + (w3_by_rows(t) && t.kind != FFK_TILE_ACC ? w3_tau(l32) : l32)) * K + 4 * half;
#pragma unroll
        for (int f = 0; f < KF; ++f) wf[s][f] = *reinterpret_cast<const f32x4*>(wp + 8 * f);
        if (half == 0) s_bias[(wave * NS + s) * 32 + l32] = u >= 0 && t.bias ? ((const float*)t.bias)[(u & 3) * 32 + l32] : 0.0f;
    }
    const int n32 = args.row_perm ? w3_tau(l32) : l32;

    // ---- slab streaming ----
    const int c4 = tid % LPR, r0 = tid / LPR;
    const bool ln = d.ln_gamma != nullptr;
    f32x4 gam = {0, 0, 0, 0}, bet = gam;
    if (ln) {
        gam = *reinterpret_cast<const f32x4*>((const float*)d.ln_gamma + c4 * 4);
        bet = *reinterpret_cast<const f32x4*>((const float*)d.ln_beta + c4 * 4);
    }
    const int mt = args.mask_tile;
    const float* rm = mt >= 0 ? (const float*)d.tiles[mt].rowmask : nullptr;
    const bool a_flat = d.a_inner >= M;
    f32x4 pre[NP];
    float pm = 1.0f;
    auto fetch = [&](int slab) {                         // rows past the end are clamped: never stored
        if (a_flat) {
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
    auto commit = [&](int buf) {
        unsigned char* sa = s_a + buf * (BM * AP);
#pragma unroll
        for (int i = 0; i < NP; i += 4) {
            if (ln) ffk_ln_rows4<LPR>(pre + i, gam, bet, d.ln_eps);
#pragma unroll
            for (int j = i; j < i + 4; ++j) *reinterpret_cast<f32x4*>(sa + (r0 + RPP * j) * AP + c4 * 16) = pre[j];
        }
        if (rm && tid < BM) s_mask[buf * BM + tid] = pm;
    };

    // the sixteen values of one lane to their tile; u: unit, bias: of its 32 rows (GLU: and of its gate's)
    auto store = [&](int u, const float* bias, const f32x16& acc, const f32x16& accg, int m0g, const float* sm) {
        const ffk_tile& t = d.tiles[u >> 2];
        const bool by_rows = w3_by_rows(t), glu = GLU && t.glu != 0;
        const int sub = glu ? (u & 3) >> 1 : u & 3, left = t.ncols - 32 * sub;        // 32-channel block of the output, channels left
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
        if (t.kind == FFK_TILE_V && inner % 32 != 0) {   // the rows of a group may lie in two key tiles
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int mrow = m0g + 8 * (v >> 2) + 4 * half + (v & 3);
                if (mrow >= M) continue;
                const unsigned hi = (unsigned)mrow / inner, lo = (unsigned)mrow - hi * inner;
                out[(long)hi * t.s_o + (long)(lo >> 5) * 1024 + acc_tile_off((int)(lo & 31), l32)] = x[v];
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
        auto put = [&](float* p) {
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
            const float* r = (const float*)t.resid + (out - (float*)t.out) + off;
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                if (16 * half + 4 * a >= left) break;
                const f32x4 y = *reinterpret_cast<const f32x4*>(r + 4 * a);
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
    auto products = [&](f32x16* acc, const unsigned char* ap, auto rows, auto s0, auto n) {
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
    auto block = [&](int u, const unsigned char* ap, int m0g, const float* sm, auto s0, auto n, int next, int nbuf) {
        f32x16 acc[n.value];
        if (next >= 0) fetch(next);
        if (w3_by_rows(d.tiles[u >> 2])) products(acc, ap, std::true_type{}, s0, n);
        else products(acc, ap, std::false_type{}, s0, n);
        if (next >= 0) commit(nbuf);
        store(u, s_bias + (wave * NS + s0.value) * 32, acc[0], acc[n.value - 1], m0g, sm);
    };

    const int nslabs = (M + BM - 1) / BM;
    int slab = blockIdx.x;                               // grid.x <= nslabs
    fetch(slab);
    commit(0);
    __builtin_amdgcn_s_waitcnt(0x0f70);                  // vmcnt(0): the products of the loop wait for no weights
    lds_barrier();
    int buf = 0;
    typedef std::integral_constant<int, 0> I0;
    typedef std::integral_constant<int, 1> I1;
    for (; slab < nslabs; slab += gridDim.x) {
        const int next = slab + (int)gridDim.x < nslabs ? slab + (int)gridDim.x : -1;
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
    return d.M % 16 == 0 && t.inner % 16 == 0 && t.s_i == 1 && t.s_d % 4 == 0;
}

template <int K, bool GLU>
int w3_launch(const W3Args& a, int gx, int groups, hipStream_t st) {
    const size_t smem = 2 * (size_t)W3_BM * W3Geo<K>::AP + (2 * W3_BM + W3_WAVES * W3Geo<K>::SLOTS * 32) * sizeof(float);
    static FfkLdsReservation lds_reserved;
    const int rc = ffk_reserve_lds(lds_reserved, (const void*)linear_ws32_kernel<K, GLU>, smem, "ffk_fused_linear");
    if (rc != FFK_OK) return rc;
    linear_ws32_kernel<K, GLU><<<dim3(gx, groups), W3_THREADS, smem, st>>>(a);
    return ffk_check_launch("ffk_fused_linear");
}

}  // namespace

// Launches the fp32 weights-stationary kernel if it can take this (already validated) descriptor and returns 1 with the launch
// status in *status; returns 0 if the caller has to use the staged kernel.
int ffk_linear_ws32_try(const ffk_linear_desc* d, hipStream_t st, int* status) {
    if (d->dtype != FFK_F32 || (d->K != 128 && d->K != 256) || d->a_chanmajor || d->a2 || d->ln_folded || d->variant == FFK_LINEAR_STAGED)
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
    if (chan_major && v_tiles) return 0;                 // they need different row orders within a group
    // Short launches stay with the staged kernel, which has more workgroups to hide the latencies of loading weights and rows:
    // 8 192 rows, 128 -> 512: 22.1 us there, 23.5 us here; 128 -> 1 024: 35.6 and 34.0 us; 4 096 rows, 256 -> 1 024: 45.6 and 32.6 us.
    const int nslabs = ffk_cdiv(d->M, W3_BM), kk = d->K / 64;
    if ((long)nslabs * a.n_units * kk < 8192) return 0;
    a.row_perm = chan_major ? 1 : 0;
    a.d = *d;
    // Units per group: fewer groups normalise the rows less often, more groups spread few rows over the CUs.  Estimated in
    // cycles of a SIMD per slab: 2 x 2 048 per 64 x 32 block of K = 64, LayerNorm and staging 12 per row and K = 64, and
    // 3 000 for what is in flight at the slab's barrier; four units (one per SIMD) are the grain of the first part.
    const int cap = W3_WAVES * (glu || d->K == 256 ? 1 : 2);
    int gx = 1, groups = 1;
    double best = 1e30;
    for (int per = cap; per >= 4; per -= 4) {
        const int g = ffk_cdiv(a.n_units, per), each = ffk_cdiv(a.n_units, g);
        int x = W3_CUS / g;
        x = x < nslabs ? x : nslabs;
        const double cost = (double)ffk_cdiv(nslabs, x) * (ffk_cdiv(each, 4) * 4096.0 * kk * (glu ? 2 : 1) + W3_BM * 12.0 * kk + 3000.0);
        if (cost < best) {
            best = cost;
            gx = x;
            groups = ffk_cdiv(a.n_units, each);
            a.per_group = each;
        }
    }
    if (d->K == 256) *status = w3_launch<256, false>(a, gx, groups, st);
    else *status = glu ? w3_launch<128, true>(a, gx, groups, st) : w3_launch<128, false>(a, gx, groups, st);
    return 1;
}
