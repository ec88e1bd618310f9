// Weights-stationary fused linear layer for channel-major operands (see ffk_fused_linear in include/ffk.h), bf16, K = 64 or
// 128: the output stage of the triangle multiplications, whose operand is the result of the contraction.
//
// Two persistent workgroups of four wavefronts per CU, so that one loads, normalises or waits at a barrier while the other
// multiplies (one workgroup of eight waves over slabs of twice the rows, output stage of the triangle multiplication with the gate
// in place: 9 216 rows 12.7 -> 9.7 us, 65 536 rows 29.1 -> 27.8, 102 400 rows 49.2 -> 39.3, 1 048 576 rows 327 -> 310).  The
// weight matrix is split into "slots" of 32 output rows; every wave keeps the MFMA fragments of two slots in registers for the
// whole kernel, so weights are read from memory exactly once per workgroup.  Rows of A stream through a double-buffered
// slab in LDS (64 rows at K = 128), transposed on the way (global -> registers -> LayerNorm -> LDS),
// the loads of slab i+1 being in flight while slab i is multiplied.  Each wave multiplies every 32-row group of the slab
// against its own slots and finishes the resulting 32x32 blocks straight from the accumulator registers - bias, activation,
// GLU, gate and residual - and stores them without LDS staging:
//   * tiles that are contiguous along channels (plain [row][channel] outputs, q / k / gate tiles)
//     use the product W . A^T, so a lane owns one row and 4 x 4 consecutive channels;
//   * tiles that are contiguous along rows (v tiles, channel-major outputs) use A . W^T, so a
//     lane owns one channel and 4 x 4 consecutive rows.
#include "ffk_common.h"
#include <type_traits>

namespace {

constexpr int WS_WAVES = 4;
constexpr int WS_THREADS = 64 * WS_WAVES;
constexpr int WS_NS = 2;                 // weight slots per wave
constexpr int WS_MAX_GRID = 512;         // two workgroups per CU
// Per-K geometry: a slab is as many rows as 256 threads fetch with four 16-byte loads each.
template <int K> struct WsGeo {
    static constexpr int KS = K / 16;                // MFMA K steps
    static constexpr int AP = K * 2 + 16;            // LDS row pitch in bytes
    static constexpr int LPR = K / 8;                // lanes (16-byte vectors) per row
    static constexpr int RPP = WS_THREADS / LPR;     // rows fetched per pass
    static constexpr int BM = 4 * RPP;               // rows per slab: 64 (K = 128) or 128 (K = 64)
    static constexpr int RG = BM / 32;               // 32-row groups per slab
};

typedef bf16_t T;

// A weight slot: 32 rows of the weights and everything its epilogue needs, laid out by the host so that a wave reads it in
// one piece (a chain of scalar loads - plan, tile, pointers - cost a launch 0.8 us per link before the first row was requested).
// Channel offsets of the slot's unit are folded into the pointers.
struct WsSlot {
    T* out;
    const T* resid;
    const T* gate;
    const T* bias;           // of the slot's 32 rows, or nullptr
    int8_t* xtail;           // tail bytes of resid / out as an extended residual stream, or nullptr
    long s_o, s_i, s_d, gate_ld;
    unsigned inner;
    unsigned gate_rows;      // 0, or the period of the gate's row index
    int ncols_left;          // valid channels from the unit's first channel on
    int wrow;                // first weight row of the slot, -1 = unused
    float scale;
    signed char kind, act;
    signed char glu;         // 0 plain, 1 value half of a GLU unit (gate half in the next slot), 2 gate half
    bool has_bias, by_rows;
    signed char rg_first, rg_mask;   // row groups of a slab this wave takes for the slot: those with rg & rg_mask == rg_first
    bool tau;                // weight rows through ffk_tau
    bool sig;                // bias pre-multiplied for ws_sigmoid_pre
};

struct WsArgs {
    const T* a;
    const T* w;
    const T* a2;
    const void* ln_gamma;
    const void* ln_beta;
    int a_so, a_si, a_cs, a2_so, a2_si;
    int M, n_tiles, a_inner, a2_inner;
    float ln_eps;
    int row_perm;                // 1: rows of a group are read through tau (launch has channel-major tiles)
    int resid_a2;                // 1: every residual is the second operand itself (same rows): taken from its LDS slab
    WsSlot slot[WS_WAVES * WS_NS];   // [wave][slot]
};
static_assert(sizeof(WsArgs) <= 4096, "kernel arguments");

// sigmoid(acc + b) with the bias table entry pre-multiplied:  bs = -log2(e) * b
__device__ __forceinline__ float ws_sigmoid_pre(float acc, float bs) {
    return fast_rcp(1.0f + fast_exp2(__builtin_fmaf(acc, -1.4426950408889634f, bs)));
}

// tiles stored with channels contiguous (lane = row) vs rows contiguous (lane = channel)
__host__ __device__ __forceinline__ bool ws_by_rows(const ffk_tile& t) {
    return t.kind == FFK_TILE_QK || t.kind == FFK_TILE_ACC || (t.kind == FFK_TILE_STRIDED && t.s_d == 1);
}

// ---- lane = row (n32 = its row within the group), registers = channels -----------------------
// STRIDED tiles: weight rows were loaded through tau, registers hold channels 16*half + v.
// ACC / QK tiles: natural weight order, registers hold channels 8a + 4*half + b.
// sb: this slot's 32 (GLU: 64) bias values in LDS (fp32).
template <bool GLU>
__device__ __forceinline__ void ws_store_rows(const WsSlot& t, const f32x16& acc, const f32x16& accg, const float* sb,
                                              bool valid, unsigned mc, unsigned hi, unsigned lo, int half) {
    const bool strided = t.kind == FFK_TILE_STRIDED;
    float x[16];
    {
        f32x4 bv[4], bg[4];
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const int o = strided ? 16 * half + 4 * a : 4 * half + 8 * a;
            bv[a] = *reinterpret_cast<const f32x4*>(sb + o);
            if (GLU) bg[a] = *reinterpret_cast<const f32x4*>(sb + 32 + o);
        }
        if (GLU) {
#pragma unroll
            for (int v = 0; v < 16; ++v) x[v] = (acc[v] + bv[v >> 2][v & 3]) * ws_sigmoid_pre(accg[v], bg[v >> 2][v & 3]);
        } else if (t.act == FFK_ACT_SIGMOID) {
#pragma unroll
            for (int v = 0; v < 16; ++v) x[v] = ws_sigmoid_pre(acc[v], bv[v >> 2][v & 3]);
        } else if (t.has_bias) {
#pragma unroll
            for (int v = 0; v < 16; ++v) x[v] = acc[v] + bv[v >> 2][v & 3];
        } else {
#pragma unroll
            for (int v = 0; v < 16; ++v) x[v] = acc[v];
        }
    }
    if (!GLU && t.act == FFK_ACT_RELU) {
#pragma unroll
        for (int v = 0; v < 16; ++v) x[v] = relu_f(x[v]);
    }
    T y[16];
    if (t.scale != 1.0f) {
        const float scl = t.scale;
#pragma unroll
        for (int v = 0; v < 16; ++v) y[v] = (T)(x[v] * scl);
    } else {
#pragma unroll
        for (int v = 0; v < 16; ++v) y[v] = (T)x[v];
    }

    T* out = t.out;
    if (t.kind == FFK_TILE_ACC) {
        if (valid && t.ncols_left >= 32) {
            T* p = out + (long)hi * t.s_o + (long)(lo >> 5) * 1024 + ((half * 32 + (lo & 31)) << 4);
            *reinterpret_cast<u32x4*>(p) = *reinterpret_cast<const u32x4*>(&y[0]);
            *reinterpret_cast<u32x4*>(p + 8) = *reinterpret_cast<const u32x4*>(&y[8]);
        }
    } else if (t.kind == FFK_TILE_QK) {
        if (valid && t.ncols_left >= 32) {
            T* p = out + (long)hi * t.s_o + (long)(lo >> 5) * 1024 + (lo & 31) * 16 + 4 * half;
#pragma unroll
            for (int a = 0; a < 4; ++a)      // d = 8a + 4 half + b  ->  (d >> 4) * 512 + n * 16 + (d & 15)
                *reinterpret_cast<u32x2*>(p + (a >> 1) * 512 + (a & 1) * 8) = *reinterpret_cast<const u32x2*>(&y[4 * a]);
        }
    } else {
        const int cl = 16 * half;                        // this lane's 16 channels, relative to the unit
        const long off = (long)hi * t.s_o + (long)lo * t.s_i + cl;
        const bool ok0 = valid && cl + 8 <= t.ncols_left, ok1 = valid && cl + 16 <= t.ncols_left;
        if (t.gate || t.resid) {
            // every load first (clamped, unconditional), then combine and store
            u32x4 gv[2], rv[2];
            const T* gate = t.gate ? t.gate + (long)(int)(t.gate_rows ? mc % t.gate_rows : mc) * t.gate_ld + cl : nullptr;
            const T* resid = t.resid ? t.resid + off : nullptr;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int cj = cl + 8 * j + 8 <= t.ncols_left ? 8 * j : (cl + 8 <= t.ncols_left ? 0 : -cl);
                if (gate) gv[j] = *reinterpret_cast<const u32x4*>(gate + cj);
                if (resid) rv[j] = *reinterpret_cast<const u32x4*>(resid + cj);
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const T* gh = reinterpret_cast<const T*>(&gv[j]);
                const T* rh = reinterpret_cast<const T*>(&rv[j]);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    float f = (float)y[8 * j + e];
                    if (gate) f = (float)(T)(f * gate_factor((float)gh[e], t.act));
                    if (resid) f += (float)rh[e];
                    y[8 * j + e] = (T)f;
                }
            }
        }
        if (ok0) *reinterpret_cast<u32x4*>(out + off) = *reinterpret_cast<const u32x4*>(&y[0]);
        if (ok1) *reinterpret_cast<u32x4*>(out + off + 8) = *reinterpret_cast<const u32x4*>(&y[8]);
    }
}

// ---- lane = channel, registers = rows ----------------------------------------------------------
// V tiles: natural row order (registers hold rows 8a + 4*half + b of the group).
// STRIDED (channel-major) tiles: the A fragments were loaded through tau, registers hold rows
// 16*half + v: sixteen consecutive rows, which never straddle `inner` (inner % 16 == 0, M % 16 == 0).
template <bool GLU>
__device__ __forceinline__ void ws_store_cols(const WsSlot& t, const f32x16& acc, const f32x16& accg, const float* sb,
                                              long m0g, int M, int l32, int half) {
    const float bv = sb[l32], bg = GLU ? sb[32 + l32] : 0.0f;
    float x[16];
    if (GLU) {
#pragma unroll
        for (int v = 0; v < 16; ++v) x[v] = (acc[v] + bv) * ws_sigmoid_pre(accg[v], bg);
    } else if (t.act == FFK_ACT_SIGMOID) {
#pragma unroll
        for (int v = 0; v < 16; ++v) x[v] = ws_sigmoid_pre(acc[v], bv);
    } else {
#pragma unroll
        for (int v = 0; v < 16; ++v) x[v] = acc[v] + bv;
        if (t.act == FFK_ACT_RELU) {
#pragma unroll
            for (int v = 0; v < 16; ++v) x[v] = relu_f(x[v]);
        }
    }

    T* out = t.out;
    const bool vt = t.kind == FFK_TILE_V;
    const long mr = vt ? m0g : m0g + 16 * half;          // V: the group is one whole key tile (inner % 32 == 0)
    const bool ok = mr < M;
    const unsigned mc = (unsigned)(ok ? mr : 0);
    unsigned hi = 0, lo = mc;
    if (t.inner < (unsigned)M) {
        hi = mc / t.inner;
        lo = mc - hi * t.inner;
    }
    T y[16];
    if (t.scale != 1.0f) {
#pragma unroll
        for (int v = 0; v < 16; ++v) y[v] = (T)(x[v] * t.scale);
    } else {
#pragma unroll
        for (int v = 0; v < 16; ++v) y[v] = (T)x[v];
    }
    if (vt) {
        if (ok && t.ncols_left >= 32) {
            T* p = out + (long)hi * t.s_o + (long)(lo >> 5) * 1024 + ((half * 32 + l32) << 4);
            *reinterpret_cast<u32x4*>(p) = *reinterpret_cast<const u32x4*>(&y[0]);
            *reinterpret_cast<u32x4*>(p + 8) = *reinterpret_cast<const u32x4*>(&y[8]);
        }
    } else if (ok && l32 < t.ncols_left) {
        T* p = out + (long)hi * t.s_o + lo + (long)l32 * t.s_d;
        *reinterpret_cast<u32x4*>(p) = *reinterpret_cast<const u32x4*>(&y[0]);
        *reinterpret_cast<u32x4*>(p + 8) = *reinterpret_cast<const u32x4*>(&y[8]);
    }
}

// GLU unit of a [row][channel] tile of a second-operand launch, where both LayerNorms are folded into the
// weights (see a2 in include/ffk.h): with W' = W * gamma the normalised product is
//     W LN(x) + b = rstd * (W' x - mean * c1) + c2,   c1[n] = sum_k W'[n][k],  c2[n] = sum_k W[n][k] beta[k] + b[n],
// so the slab needs no normalisation pass at all: mean and rstd of the lane's row come from the fragments the
// products use, c2 sits in the bias table, c1 in a table of its own; the gate half does the same with the
// second operand's row.  out = resid + value * sigmoid(gate), rounded once.  sb / sc1: this unit's 64 bias
// values / 64 row sums in LDS (fp32), value half first.
template <bool XT>
__device__ __forceinline__ void ws_store_rows_folded(const WsSlot& t, const f32x16& acc, const f32x16& accg, const float* sb,
                                                     const float* sc1, float rstd, float nmr, float rstd_g, float nmr_g,
                                                     bool valid, unsigned hi, unsigned lo, int half,
                                                     const unsigned char* a2row, int a2vec, int a2swz) {
    // rstd_g / nmr_g (the second operand's statistics) arrive multiplied by -log2(e), as the gate's bias table is
    // a2row: this lane's row of the second operand's LDS slab when that operand is also the residual (the triangle
    // multiplication's output stage: gate input and residual are both z), else nullptr; a2vec: the 16-byte vector
    // of the row this lane's 16 channels start at; a2swz: the row's swizzle (vector v lives at v ^ a2swz)
    const int cl = 16 * half;
    const long off = (long)hi * t.s_o + (long)lo * t.s_i + cl;
    u32x4 rv[2];
    if (t.resid) {
        if (a2row) {
            rv[0] = *reinterpret_cast<const u32x4*>(a2row + ((a2vec ^ a2swz) << 4));
            rv[1] = *reinterpret_cast<const u32x4*>(a2row + (((a2vec + 1) ^ a2swz) << 4));
        } else {
            rv[0] = *reinterpret_cast<const u32x4*>(t.resid + off);
            rv[1] = *reinterpret_cast<const u32x4*>(t.resid + off + 8);
        }
    }
    if (XT && t.xtail) {       // extended residual stream: the update is added at 24 bits, eight channels at a time
        const u32x4 tv = *reinterpret_cast<const u32x4*>(t.xtail + off);
        u32x4 tn;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            f32x4 bv[2], bg[2], cv[2], cg[2];      // the tables of these eight channels only (register budget)
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                const int o = cl + 8 * j + 4 * a;
                bv[a] = *reinterpret_cast<const f32x4*>(sb + o);
                bg[a] = *reinterpret_cast<const f32x4*>(sb + 32 + o);
                cv[a] = *reinterpret_cast<const f32x4*>(sc1 + o);
                cg[a] = *reinterpret_cast<const f32x4*>(sc1 + 32 + o);
            }
            float f[8];
            xs_decode8(rv[j], tv[2 * j], tv[2 * j + 1], f);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int v = 8 * j + e;
                const float val = __builtin_fmaf(acc[v], rstd, __builtin_fmaf(cv[e >> 2][e & 3], nmr, bv[e >> 2][e & 3]));
                const float garg = __builtin_fmaf(accg[v], rstd_g, __builtin_fmaf(cg[e >> 2][e & 3], nmr_g, bg[e >> 2][e & 3]));
                f[e] += (float)(T)(val * fast_rcp(1.0f + fast_exp2(garg)));
            }
            u32x4 hv;
            uint32_t ta, tb;
            xs_encode8(f, hv, ta, tb);
            tn[2 * j] = ta;
            tn[2 * j + 1] = tb;
            if (valid) *reinterpret_cast<u32x4*>(t.out + off + 8 * j) = hv;
        }
        if (valid) *reinterpret_cast<u32x4*>(t.xtail + off) = tn;
        return;
    }
    f32x4 bv[4], bg[4], cv[4], cg[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        const int o = 16 * half + 4 * a;
        bv[a] = *reinterpret_cast<const f32x4*>(sb + o);
        bg[a] = *reinterpret_cast<const f32x4*>(sb + 32 + o);
        cv[a] = *reinterpret_cast<const f32x4*>(sc1 + o);
        cg[a] = *reinterpret_cast<const f32x4*>(sc1 + 32 + o);
    }
    T y[16];
    const T* rh = reinterpret_cast<const T*>(&rv[0]);
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        const float val = __builtin_fmaf(acc[v], rstd, __builtin_fmaf(cv[v >> 2][v & 3], nmr, bv[v >> 2][v & 3]));
        const float garg = __builtin_fmaf(accg[v], rstd_g, __builtin_fmaf(cg[v >> 2][v & 3], nmr_g, bg[v >> 2][v & 3]));
        float x = val * fast_rcp(1.0f + fast_exp2(garg));
        if (t.resid) x += (float)rh[v];
        y[v] = (T)x;
    }
    if (valid) {
        *reinterpret_cast<u32x4*>(t.out + off) = *reinterpret_cast<const u32x4*>(&y[0]);
        *reinterpret_cast<u32x4*>(t.out + off + 8) = *reinterpret_cast<const u32x4*>(&y[8]);
    }
}

// DUAL: the gate halves of the GLU units multiply a second operand (row-major rows, own LayerNorm).  Its
// slab goes from global memory straight into LDS (unpadded 256-byte rows, 16-byte columns XOR-swizzled
// with the row index) one slab ahead and is normalised in place by the threads that requested it.
// XT (with DUAL): the launch has tiles with a residual tail (extended residual stream); only that instantiation carries its code
template <int WS_K, bool DUAL, bool XT>
__global__ __launch_bounds__(WS_THREADS, 2) void linear_ws_kernel(const WsArgs args) {
    typedef Mma<T> MM;
    typedef WsGeo<WS_K> G;
    constexpr int WS_KS = G::KS, WS_AP = G::AP, WS_BM = G::BM, WS_RG = G::RG;
    constexpr int NS = WS_NS, AFC = WS_K == 128 ? 8 : 4;   // AFC: A fragments held at a time (register budget)
    const WsArgs& d = args;
    extern __shared__ __align__(16) unsigned char smem[];
    unsigned char* s_a = smem;                                                 // [2][WS_BM][WS_AP]
    float* s_bias = reinterpret_cast<float*>(smem + 2 * WS_BM * WS_AP);        // [n_tiles][128]
    unsigned char* s_a2 = reinterpret_cast<unsigned char*>(s_bias + FFK_MAX_TILES * 128);   // DUAL: [2][WS_BM][256 B]
    static_assert(!DUAL || WS_K == 128, "the second operand is built for K = 128");
    // LayerNorm parameters that are only needed when a slab is committed wait in LDS, not in registers
    float* s_ln = reinterpret_cast<float*>(s_a2 + (DUAL ? 2 * WS_BM * 256 : 0));            // gamma[128], beta[128] (fp32)
    T* s_ln2 = reinterpret_cast<T*>(s_ln + 256);                               // DUAL: gamma2[128], beta2[128]
    float* s_c1 = reinterpret_cast<float*>(s_ln2 + (DUAL ? 256 : 0));                       // DUAL: folded LayerNorm row sums
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    const int M = d.M;
    const T* A = d.a;
    const T* W = d.w;

    // ---- this wave's weight slots, resident in registers ----
    WsSlot sp[NS];
    bf16x8 wf[NS][WS_KS];
#pragma unroll
    for (int s = 0; s < NS; ++s) sp[s] = args.slot[wave * NS + s];
    // launches with channel-major tiles read the rows of a group through tau (16 consecutive rows per lane)
    const int n32 = args.row_perm ? ffk_tau(l32) : l32;

    // ---- slab streaming ----
    // DUAL launches carry both LayerNorms folded into the weights: ln_gamma is the fp32 table of row sums and
    // both slabs are used as they arrive (see ws_store_rows_folded)
    const bool folded = DUAL;
    const bool ln = d.ln_gamma != nullptr && !folded;
    // plain row-major operands (inner >= M) need no division per fetched vector
    const bool a_flat = d.a_inner >= M, a2_flat = DUAL && d.a2_inner >= M;
    Vec16<T> pre[4];
    // Channel-major A (element (m, k) at a + k * a_cs + rowoffset(m), K = 128 or 64): a thread fetches eight
    // consecutive rows of channel k = lane % 32 + 32 cb (cb < K / 32); the two half-waves of wave w own the row
    // groups 2w and 2w + 1 of each 64-row pass of the slab (one pass at K = 128, two at K = 64), so the LayerNorm
    // reduction over k stays inside 32 lanes.  The slab is transposed on its way into LDS (2-byte stores,
    // consecutive lanes -> consecutive k of one row).
    constexpr int CMI = WS_K / 32;                       // channel blocks per thread
    static_assert(WS_K == 128 || WS_K == 64, "channel-major operands are built for K = 128 and 64");
    const int cm_k = lane & 31, cm_mg = 2 * wave + (lane >> 5);
    // second operand: vector v = i * 256 + tid of a slab is row v / 16, LDS column v % 16, which holds
    // global column (v % 16) ^ (row % 16); the 16 lanes of a row are adjacent, as the LayerNorm wants them
    const int a2_col = (tid & 15) ^ ((tid >> 4) & 15);
    const unsigned lds_a2 = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)s_a2;
    auto fetch = [&](int slab, int tobuf) {
        if (DUAL) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                long m = (long)slab * WS_BM + i * (WS_THREADS / 16) + (tid >> 4);
                m = m < M ? m : M - 1;
                const unsigned hi = a2_flat ? 0u : (unsigned)m / (unsigned)d.a2_inner, lo = (unsigned)m - hi * (unsigned)d.a2_inner;
                const T* gp = d.a2 + (long)hi * d.a2_so + (long)lo * d.a2_si + a2_col * 8;
                const unsigned dst = lds_a2 + tobuf * (WS_BM * 256) + (i * WS_THREADS + wave * 64) * 16;
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
                asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(gp), "s"(dst) : "memory", "m0");
#pragma clang diagnostic pop
            }
        }
#pragma unroll
        for (int rp = 0; rp < 4 / CMI; ++rp) {
            long m = (long)slab * WS_BM + (cm_mg + 2 * WS_WAVES * rp) * 8;
            m = m < M ? m : M - 8;                       // M % 8 == 0; clamped groups are never stored
            const unsigned hi = a_flat ? 0u : (unsigned)m / (unsigned)d.a_inner, lo = (unsigned)m - hi * (unsigned)d.a_inner;
            const T* base = A + (long)hi * d.a_so + lo;  // a_si == 1
#pragma unroll
            for (int cb = 0; cb < CMI; ++cb) pre[rp * CMI + cb] = ld16(base + (long)(cm_k + 32 * cb) * d.a_cs);
        }
    };
    auto commit = [&](int buf) {
        unsigned char* sa = s_a + buf * (WS_BM * WS_AP);
        if (DUAL) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this thread's vectors of the second operand have landed
        if (!ln) {       // nothing to normalise here: the transposition is a plain copy
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    *reinterpret_cast<T*>(sa + ((cm_mg + 2 * WS_WAVES * (i / CMI)) * 8 + j) * WS_AP + (cm_k + 32 * (i % CMI)) * 2) = pre[i].e[j];
            return;
        }
        float f[4][8];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 8; ++j) f[i][j] = (float)pre[i].e[j];
        {
            float cm_g[CMI], cm_b[CMI];              // gamma / beta of this lane's channels
#pragma unroll
            for (int cb = 0; cb < CMI; ++cb) {
                cm_g[cb] = s_ln[(lane & 31) + 32 * cb];
                cm_b[cb] = s_ln[WS_K + (lane & 31) + 32 * cb];
            }
#pragma unroll
            for (int rp = 0; rp < 4 / CMI; ++rp)
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    float su = 0.0f;
                    if (CMI == 4) {
                        su = (f[0][j] + f[1][j]) + (f[2][j] + f[3][j]);
                    } else {
#pragma unroll
                        for (int cb = 0; cb < CMI; ++cb) su += f[rp * CMI + cb][j];
                    }
                    const float mu = group_sum(su, 32) * (1.0f / WS_K);
                    float q = 0.0f;
#pragma unroll
                    for (int cb = 0; cb < CMI; ++cb) {
                        f[rp * CMI + cb][j] -= mu;
                        q += f[rp * CMI + cb][j] * f[rp * CMI + cb][j];
                    }
                    const float rs = rsqrtf(group_sum(q, 32) * (1.0f / WS_K) + d.ln_eps);
#pragma unroll
                    for (int cb = 0; cb < CMI; ++cb)
                        f[rp * CMI + cb][j] = f[rp * CMI + cb][j] * rs * cm_g[cb] + cm_b[cb];
                }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 8; ++j)
                *reinterpret_cast<T*>(sa + ((cm_mg + 2 * WS_WAVES * (i / CMI)) * 8 + j) * WS_AP + (cm_k + 32 * (i % CMI)) * 2) = (T)f[i][j];
    };

    const int nslabs = (M + WS_BM - 1) / WS_BM;
    int slab = blockIdx.x;                               // grid <= nslabs
    fetch(slab, 0);                                      // the first slab travels while the weights are fetched
    // ---- weights: every wave reads the 32 rows of its slots as whole lines (a lane's fragments are 16-byte pieces
    // 32 bytes apart in one row, 32 rows per request: fetched that way every request touches 32 lines and uses a
    // quarter of each, and a workgroup's 128 .. 256 KB of weights do not stay in the first-level cache between the
    // K steps) and re-orders them through a private piece of the slab buffer, which is idle until the first commit.
    // A piece is 32 rows x PW channels; its 16-byte chunks are stored at chunk ^ (row % LR) so that the fragment
    // reads (one row per lane) spread over the banks.
    {
        constexpr int PW = WS_K < 128 ? WS_K : 128;      // channels per piece
        constexpr int LR = PW / 8;                       // 16-byte chunks (lanes) per row of a piece
        constexpr int NI = 32 / (64 / LR);               // requests per piece = K steps per piece
        constexpr int NP = WS_K / PW;                    // pieces per slot
        static_assert(NI * NP == WS_KS, "piece geometry");
        static_assert(WS_WAVES * 32 * PW * 2 <= 2 * WS_BM * WS_AP, "the staging area is the slab buffer");
        unsigned char* stage = s_a + wave * (32 * PW * 2);
        const int lrow = lane / LR, lcol = lane % LR;
#pragma unroll
        for (int sl = 0; sl < NS; ++sl)
#pragma unroll
            for (int pc = 0; pc < NP; ++pc)
#pragma unroll
                for (int i = 0; i < NI; ++i)
                    wf[sl][pc * NI + i] = MM::ld(W + (long)((sp[sl].wrow >= 0 ? sp[sl].wrow : 0) + i * (64 / LR) + lrow) * WS_K + pc * PW + lcol * 8);
        // tables the epilogues and the commits read from LDS (no global loads there); the barrier in front of the first
        // commit publishes them.  All are requested together with the weights and stored when these have arrived.
        float tb[NS], tc[2];
        T tg[2] = {(T)0.0f, (T)0.0f};
#pragma unroll
        for (int sl = 0; sl < NS; ++sl) tb[sl] = sp[sl].wrow >= 0 && sp[sl].bias ? (float)sp[sl].bias[l32] : 0.0f;
        if (ln && tid < WS_K) {
            tg[0] = ((const T*)d.ln_gamma)[tid];
            tg[1] = ((const T*)d.ln_beta)[tid];
        }
        if (folded) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
                tc[i] = tid + i * WS_THREADS < d.n_tiles * 128 ? ((const float*)d.ln_gamma)[tid + i * WS_THREADS] : 0.0f;
        }
#pragma unroll
        for (int sl = 0; sl < NS; ++sl)
#pragma unroll
            for (int pc = 0; pc < NP; ++pc) {
#pragma unroll
                for (int i = 0; i < NI; ++i) {
                    const int row = i * (64 / LR) + lrow;
                    *reinterpret_cast<bf16x8*>(stage + row * (PW * 2) + ((lcol ^ (row & (LR - 1))) * 16)) = wf[sl][pc * NI + i];
                }
                // [row][channel] tiles take their weight rows through tau (16 consecutive channels per lane)
                const int wl = sp[sl].tau ? ffk_tau(l32) : l32;
#pragma unroll
                for (int k = 0; k < NI; ++k)
                    wf[sl][pc * NI + k] = *reinterpret_cast<const bf16x8*>(
                        stage + wl * (PW * 2) + (((2 * k + half) ^ (wl & (LR - 1))) * 16));
            }
#pragma unroll
        for (int sl = 0; sl < NS; ++sl)                   // (waves of a group write the same values)
            if (half == 0 && sp[sl].wrow >= 0) s_bias[sp[sl].wrow + l32] = sp[sl].sig ? -1.4426950408889634f * tb[sl] : tb[sl];
        if (ln && tid < WS_K) {
            s_ln[tid] = (float)tg[0];
            s_ln[WS_K + tid] = (float)tg[1];
        }
        if (folded) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
                if (tid + i * WS_THREADS < FFK_MAX_TILES * 128) s_c1[tid + i * WS_THREADS] = tc[i];
            for (int i = tid + 2 * WS_THREADS; i < d.n_tiles * 128; i += WS_THREADS) s_c1[i] = ((const float*)d.ln_gamma)[i];
        }
    }
    lds_barrier();                                       // every wave is done with the staging area
    commit(0);
    lds_barrier();
    int buf = 0;
    for (; slab < nslabs; slab += gridDim.x) {
        const bool more = slab + (int)gridDim.x < nslabs;
        if (more) fetch(slab + (int)gridDim.x, buf ^ 1);  // in flight during the products below
        const unsigned char* sa = s_a + buf * (WS_BM * WS_AP);
        int rg_by = 1;
        asm volatile("" : "+s"(rg_by));                    // opaque: a known trip count makes the compiler keep addresses it spills for
        for (int rg = 0; rg < WS_RG; rg += rg_by) {
            const long m0g = (long)slab * WS_BM + rg * 32;
            if (m0g >= M) break;
            const unsigned char* ap = sa + (rg * 32 + n32) * WS_AP + half * 16;
            // position of this lane's row for the [row][channel] tiles; the division is redone only
            // when a slot's tile has another `inner`
            const long mrow = m0g + n32;
            const bool valid = mrow < M;
            const unsigned mc = (unsigned)(valid ? mrow : M - 1);
            unsigned c_inner = 0, c_hi = 0, c_lo = mc;
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                if (sp[s].wrow < 0 || sp[s].glu == 2 || (rg & sp[s].rg_mask) != sp[s].rg_first) continue;
                const WsSlot& t = sp[s];
                const bool glu = sp[s].glu == 1;
                const int sg = s + 1 < NS ? s + 1 : s;             // gate slot of a GLU unit (constant after unrolling)
                const float* sb = s_bias + sp[s].wrow;
                // The A fragments are re-read from LDS for every slot: keeping them across the epilogue of
                // the previous slot costs 32 registers, and a single spilled register puts a scratch
                // reload with a full vector-memory wait into every epilogue.
                int reread = 0;
                asm volatile("" : "+v"(reread));                   // opaque zero: keeps the compiler from reusing the loads
                f32x16 acc, accg;
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[v] = accg[v] = 0.0f;
                float st1 = 0.0f, st2 = 0.0f, su1 = 0.0f, su2 = 0.0f;   // row statistics of the two operands (DUAL)
                const bool rows = sp[s].by_rows;
                if (DUAL && glu) {
                    // gate half: fragments of the second operand's row (row % 16 == l32 % 16 picks the swizzle)
                    const unsigned a2row = (unsigned)(buf * (WS_BM * 256) + (rg * 32 + n32) * 256 + ((half ^ (n32 & 15)) << 4));
#pragma unroll
                    for (int k0 = 0; k0 < WS_KS; k0 += AFC) {
                        bf16x8 af[AFC];
#pragma unroll
                        for (int ks = 0; ks < AFC; ++ks)
                            af[ks] = *reinterpret_cast<const bf16x8*>(s_a2 + ((a2row + reread) ^ (unsigned)((k0 + ks) * 32)));
                        {
                            typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
                            const bf16x2 ones = {(bf16_t)1.0f, (bf16_t)1.0f};
#pragma unroll
                            for (int ks = 0; ks < AFC; ++ks)
#pragma unroll
                                for (int e = 0; e < 4; ++e) {
                                    const bf16x2 pr = {af[ks][2 * e], af[ks][2 * e + 1]};
                                    su1 = __builtin_amdgcn_fdot2_f32_bf16(pr, ones, su1, false);
                                    su2 = __builtin_amdgcn_fdot2_f32_bf16(pr, pr, su2, false);
                                }
                        }
#pragma unroll
                        for (int ks = 0; ks < AFC; ++ks) MM::mma(accg, wf[sg][k0 + ks], af[ks]);
                    }
                }
#pragma unroll
                for (int k0 = 0; k0 < WS_KS; k0 += AFC) {          // AFC K steps of A in registers at a time
                    bf16x8 af[AFC];
#pragma unroll
                    for (int ks = 0; ks < AFC; ++ks) af[ks] = *reinterpret_cast<const bf16x8*>(ap + reread + (k0 + ks) * 32);
                    if (DUAL && folded) {
                        // sum and sum of squares of this lane's half of its row, from the fragments themselves
                        typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
                        const bf16x2 ones = {(bf16_t)1.0f, (bf16_t)1.0f};
#pragma unroll
                        for (int ks = 0; ks < AFC; ++ks)
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                const bf16x2 pr = {af[ks][2 * e], af[ks][2 * e + 1]};
                                st1 = __builtin_amdgcn_fdot2_f32_bf16(pr, ones, st1, false);
                                st2 = __builtin_amdgcn_fdot2_f32_bf16(pr, pr, st2, false);
                            }
                    }
                    if (rows) {
#pragma unroll
                        for (int ks = 0; ks < AFC; ++ks) MM::mma(acc, wf[s][k0 + ks], af[ks]);
                        if (!DUAL && glu) {
#pragma unroll
                            for (int ks = 0; ks < AFC; ++ks) MM::mma(accg, wf[sg][k0 + ks], af[ks]);
                        }
                    } else {
#pragma unroll
                        for (int ks = 0; ks < AFC; ++ks) MM::mma(acc, af[ks], wf[s][k0 + ks]);
                        if (glu) {
#pragma unroll
                            for (int ks = 0; ks < AFC; ++ks) MM::mma(accg, af[ks], wf[sg][k0 + ks]);
                        }
                    }
                }
                if (rows) {
                    if (t.inner != c_inner) {
                        c_inner = t.inner;
                        if (c_inner < (unsigned)M) {
                            c_hi = mc / c_inner;
                            c_lo = mc - c_hi * c_inner;
                        } else {
                            c_hi = 0;
                            c_lo = mc;
                        }
                    }
                    if (DUAL && folded) {
                        st1 += lane_xor<32>(st1);
                        st2 += lane_xor<32>(st2);
                        const float mean = st1 * (1.0f / WS_K);
                        const float rstd = rsqrtf(fmaxf(st2 * (1.0f / WS_K) - mean * mean, 0.0f) + d.ln_eps);
                        su1 += lane_xor<32>(su1);
                        su2 += lane_xor<32>(su2);
                        const float mean_g = su1 * (1.0f / WS_K);
                        const float rstd_g = -1.4426950408889634f * rsqrtf(fmaxf(su2 * (1.0f / WS_K) - mean_g * mean_g, 0.0f) + d.ln_eps);
                        const unsigned char* a2r = nullptr;
                        int a2v = 0;
                        if (args.resid_a2 && t.resid) {
                            a2r = s_a2 + buf * (WS_BM * 256) + (rg * 32 + n32) * 256;
                            a2v = (int)(t.resid - d.a2) / 8 + 2 * half;
                        }
                        ws_store_rows_folded<XT>(t, acc, accg, sb, s_c1 + sp[s].wrow, rstd, -rstd * mean, rstd_g, -rstd_g * mean_g,
                                             valid, c_hi, c_lo, half, a2r, a2v, n32 & 15);
                    } else if (glu) ws_store_rows<true>(t, acc, accg, sb, valid, mc, c_hi, c_lo, half);
                    else ws_store_rows<false>(t, acc, accg, sb, valid, mc, c_hi, c_lo, half);
                } else {
                    if (glu) ws_store_cols<true>(t, acc, accg, sb, m0g, M, l32, half);
                    else ws_store_cols<false>(t, acc, accg, sb, m0g, M, l32, half);
                }
            }
        }
        if (!more) break;                                // nothing left to commit: the stores drain on their own
        commit(buf ^ 1);
        lds_barrier();
        buf ^= 1;
    }
}

// tiles stored with channels contiguous (lane = row) vs rows contiguous (lane = channel): host side
bool ws_tile_ok(const ffk_linear_desc& d, const ffk_tile& t) {
    auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    if (t.inner <= 0 || t.ncols <= 0 || !al16(t.out)) return false;
    if (ws_by_rows(t)) {
        if (t.kind == FFK_TILE_STRIDED) {
            if (t.ncols % 8 != 0 || t.s_o % 8 || t.s_i % 8 || t.s_h % 8) return false;
            if (t.resid && !al16(t.resid)) return false;
            if (t.gate && (!al16(t.gate) || t.gate_ld % 8)) return false;
            if (t.xtail && (!t.resid || t.ncols % 16 != 0 || t.s_o % 16 || t.s_i % 16 || t.s_h % 16)) return false;
        } else {
            if (t.ncols % 32 != 0 || t.resid || t.gate || t.xtail || t.s_o % 8 || t.s_h % 8) return false;
        }
        return true;
    }
    if (t.resid || t.gate || t.xtail) return false;
    if (t.kind == FFK_TILE_V) return d.M % 32 == 0 && t.inner % 32 == 0 && t.ncols % 32 == 0 && t.s_o % 8 == 0 && t.s_h % 8 == 0;
    if (t.kind != FFK_TILE_STRIDED) return false;
    return d.M % 16 == 0 && t.inner % 16 == 0 && t.s_i == 1 && t.s_o % 8 == 0 && t.s_h % 8 == 0 && t.s_d % 8 == 0;
}

WsSlot ws_slot(const ffk_linear_desc& d, int tile, int chan, int wrow, int glu, int rg_first, int rg_step) {
    const ffk_tile& t = d.tiles[tile];
    const long coff = (long)(chan >> 5) * t.s_h;
    WsSlot q{};
    q.wrow = wrow;
    q.glu = (signed char)glu;
    q.out = (T*)t.out + coff;
    q.resid = t.resid ? (const T*)t.resid + coff : nullptr;
    q.gate = t.gate ? (const T*)t.gate + chan : nullptr;
    q.bias = t.bias ? (const T*)t.bias + (wrow & 127) : nullptr;
    q.xtail = t.xtail ? (int8_t*)t.xtail + coff : nullptr;
    q.s_o = t.s_o;
    q.s_i = t.s_i;
    q.s_d = t.s_d;
    q.gate_ld = t.gate_ld;
    q.inner = (unsigned)t.inner;
    q.gate_rows = (unsigned)t.gate_rows;
    q.ncols_left = t.ncols - chan;
    q.scale = t.scale;
    q.kind = (signed char)t.kind;
    q.act = (signed char)t.act;
    q.has_bias = t.bias != nullptr;
    q.by_rows = ws_by_rows(t);
    q.tau = t.kind == FFK_TILE_STRIDED && t.s_d == 1;
    q.sig = t.glu ? glu == 2 : t.act == FFK_ACT_SIGMOID;     // gate halves of a GLU unit and sigmoid tiles
    q.rg_first = (signed char)rg_first;
    q.rg_mask = (signed char)(rg_step - 1);
    return q;
}

// Distributes the 32-row weight units over the waves, GLU units (two slots) first; false if they do not fit.  The waves form
// G = WS_WAVES / R groups; the R waves of a group hold the same units and take every R-th row group (R as large as the units allow).
bool ws_make_plan(const ffk_linear_desc& d, WsArgs& p, int rg_per_slab) {
    struct Unit { int tile, chan, wrow, slots; };
    Unit units[FFK_MAX_TILES * 4];
    int nu = 0;
    for (int i = 0; i < d.n_tiles; ++i) {
        const ffk_tile& t = d.tiles[i];
        const int n = (t.ncols + 31) / 32;
        for (int u = 0; u < n; ++u) units[nu++] = {i, u * 32, i * 128 + (t.glu ? u * 64 : u * 32), t.glu ? 2 : 1};
    }
    for (auto& q : p.slot) {
        q = WsSlot{};
        q.wrow = -1;
    }
    int assign[WS_WAVES][WS_NS];
    int G = 0, R = 0;
    for (R = rg_per_slab < WS_WAVES ? rg_per_slab : WS_WAVES; R >= 1; R >>= 1) {
        G = WS_WAVES / R;
        int load[WS_WAVES] = {0};
        for (int g = 0; g < G; ++g)
            for (int s = 0; s < WS_NS; ++s) assign[g][s] = -1;
        bool fits = true;
        for (int pass = 2; pass >= 1 && fits; --pass) {
            for (int i = 0; i < nu && fits; ++i) {
                if (units[i].slots != pass) continue;
                int best = -1;
                for (int g = 0; g < G; ++g)
                    if (load[g] + pass <= WS_NS && (best < 0 || load[g] < load[best])) best = g;
                if (best < 0) {
                    fits = false;
                    break;
                }
                assign[best][load[best]] = i;
                if (pass == 2) assign[best][load[best] + 1] = -2 - i;   // gate half of unit i
                load[best] += pass;
            }
        }
        if (fits) break;
    }
    if (R < 1) return false;
    for (int w = 0; w < WS_WAVES; ++w)
        for (int sl = 0; sl < WS_NS; ++sl) {
            const int a = assign[w % G][sl];
            if (a == -1) continue;
            const Unit& u = units[a >= 0 ? a : -2 - a];
            p.slot[w * WS_NS + sl] = ws_slot(d, u.tile, u.chan, u.wrow + (a >= 0 ? 0 : 32), a < 0 ? 2 : u.slots == 2 ? 1 : 0, w / G, R);
        }
    return true;
}

template <int K, bool DUAL = false, bool XT = false>
int ws_launch(const WsArgs& args, hipStream_t st) {
    constexpr int WS_BM = WsGeo<K>::BM;
    const size_t smem = 2 * (size_t)WS_BM * WsGeo<K>::AP + FFK_MAX_TILES * 128 * sizeof(float) + 256 * sizeof(float) +
                        (DUAL ? 2 * (size_t)WS_BM * 256 + 256 * sizeof(T) + FFK_MAX_TILES * 128 * sizeof(float) : 0);
    static FfkLdsReservation lds_reserved;
    {
        const int rc_lds = ffk_reserve_lds(lds_reserved, (const void*)linear_ws_kernel<K, DUAL, XT>, smem, "ffk_fused_linear");
        if (rc_lds != FFK_OK) return rc_lds;
    }
    const int nslabs = ffk_cdiv(args.M, WS_BM);
    linear_ws_kernel<K, DUAL, XT><<<nslabs < WS_MAX_GRID ? nslabs : WS_MAX_GRID, WS_THREADS, smem, st>>>(args);
    return ffk_check_launch("ffk_fused_linear");
}

}  // namespace

// Launches the weights-stationary kernel if it can take this (already validated) descriptor and
// returns 1 with the launch status in *status; returns 0 if the caller has to use another variant.
int ffk_linear_ws_try(const ffk_linear_desc* d, hipStream_t st, int* status) {
    if (d->dtype != FFK_BF16 || !d->a_chanmajor || (d->K != 64 && d->K != 128) || d->variant == FFK_LINEAR_STAGED) return 0;
    if ((d->ln_folded != 0) != (d->a2 != nullptr)) return 0;    // folded LayerNorms and the second operand go together
    if (d->a_si != 1 || d->a_inner % 8 || d->a_so % 8 || d->a_cs % 8 || d->M % 8) return 0;
    if (d->a2 && (d->K != 128 || d->a2_si % 8 || d->a2_so % 8)) return 0;    // the second operand is built for K = 128
    auto i32 = [](int64_t v) { return v >= -0x7fffffffL && v <= 0x7fffffffL; };      // the kernel's strides have 32 bits
    if (!i32(d->a_so) || !i32(d->a_si) || !i32(d->a_cs) || !i32(d->a2_so) || !i32(d->a2_si)) return 0;
    bool chan_major = false, v_tiles = false, tails = false, resid_a2 = true;
    for (int i = 0; i < d->n_tiles; ++i) {
        const ffk_tile& t = d->tiles[i];
        if (!i32(t.s_o) || !i32(t.s_i) || !i32(t.s_d) || !i32(t.s_h) || !i32(t.gate_ld)) return 0;
        if (t.kind == FFK_TILE_BIAS || t.rowmask || !ws_tile_ok(*d, t)) return 0;
        tails = tails || t.xtail != nullptr;
        chan_major = chan_major || (!ws_by_rows(t) && t.kind == FFK_TILE_STRIDED);
        v_tiles = v_tiles || t.kind == FFK_TILE_V;
        if (!d->a2) continue;
        // second operand: every unit must be a plain residual GLU unit of 64 channels stored [row][channel]
        if (!t.glu || t.kind != FFK_TILE_STRIDED || t.s_d != 1 || t.gate || t.scale != 1.0f || t.ncols != 64) return 0;
        // whether the residual is the second operand itself: same rows, channels [c0, c0 + 64) of its 128
        const long c0 = (const T*)t.resid - (const T*)d->a2;
        if (!t.resid || c0 < 0 || c0 + t.ncols > 128 || c0 % 32 || t.s_o != d->a2_so || t.s_i != d->a2_si ||
            t.inner != d->a2_inner || t.s_h != 32)
            resid_a2 = false;
    }
    if (chan_major && v_tiles) return 0;          // they need different row orders within a group
    if (tails && !d->a2) return 0;                // residual tails: built for the launches with a second operand
    WsArgs args;
    if (!ws_make_plan(*d, args, d->K == 64 ? WsGeo<64>::RG : WsGeo<128>::RG)) return 0;
    args.a = (const T*)d->a;
    args.w = (const T*)d->w;
    args.a2 = (const T*)d->a2;
    args.ln_gamma = d->ln_gamma;
    args.ln_beta = d->ln_beta;
    args.a_so = (int)d->a_so;
    args.a_si = (int)d->a_si;
    args.a_cs = (int)d->a_cs;
    args.a2_so = (int)d->a2_so;
    args.a2_si = (int)d->a2_si;
    args.M = d->M;
    args.n_tiles = d->n_tiles;
    args.a_inner = d->a_inner;
    args.a2_inner = d->a2_inner;
    args.ln_eps = d->ln_eps;
    args.row_perm = chan_major ? 1 : 0;
    args.resid_a2 = resid_a2 ? 1 : 0;
    if (d->a2) *status = tails ? ws_launch<128, true, true>(args, st) : ws_launch<128, true, false>(args, st);
    else *status = d->K == 64 ? ws_launch<64>(args, st) : ws_launch<128>(args, st);
    return 1;
}
