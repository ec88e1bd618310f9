// Weights-stationary variant of the fused linear layer (see ffk_fused_linear in include/ffk.h),
// bf16, K = 64, 128 or 256: the projections of the pair and MSA stacks (and of the extra-MSA and
// template stacks at 64 channels), where M is 10^5 .. 10^6 rows and the whole weight matrix is a few
// hundred KB.
//
// One persistent workgroup of 8 wavefronts per CU.  The weight matrix is split into "slots" of 32
// output rows; every wave keeps the MFMA fragments of up to three slots in registers for the whole
// kernel, so weights are read from memory exactly once per workgroup.  Rows of A stream through a
// double-buffered 128-row slab in LDS: global -> registers -> (LayerNorm in registers, 16 lanes
// per row) -> LDS, the loads of slab i+1 being in flight while slab i is multiplied.  Each wave
// multiplies every 32-row group of the slab against its own slots and finishes the resulting
// 32x32 blocks straight from the accumulator registers - bias, activation, GLU, row mask, gate
// and residual - and stores them without LDS staging:
//   * tiles that are contiguous along channels (plain [row][channel] outputs, q / k / gate tiles)
//     use the product W . A^T, so a lane owns one row and 4 x 4 consecutive channels;
//   * tiles that are contiguous along rows (v tiles, channel-major outputs) use A . W^T, so a
//     lane owns one channel and 4 x 4 consecutive rows.
// Attention operand tiles are written as 32 contiguous bytes per lane, the order in which the
// attention kernel loads them.
#include "ffk_common.h"
#include <stdlib.h>
#include <type_traits>

namespace {

constexpr int WS_WAVES = 8;
constexpr int WS_THREADS = 64 * WS_WAVES;
constexpr int WS_NS = 4;                 // weight slots per wave: up to 4 (K = 64), 3 (K = 128), 2 (K = 256, 64 registers a slot)
constexpr int WS_MAX_GRID = 256;         // one workgroup per CU
// Per-K geometry: a slab is as many rows as 512 threads fetch with four 16-byte loads each.
template <int K> struct WsGeo {
    static constexpr int KS = K / 16;                // MFMA K steps
    static constexpr int AP = K * 2 + 16;            // LDS row pitch in bytes
    static constexpr int LPR = K / 8;                // lanes (16-byte vectors) per row
    static constexpr int RPP = WS_THREADS / LPR;     // rows fetched per pass
    static constexpr int BM = 4 * RPP;               // rows per slab: 128 (K = 128) or 64 (K = 256)
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
    bool masked, has_bias, by_rows;
    signed char rg_first, rg_mask;   // row groups of a slab this wave takes for the slot: those with rg & rg_mask == rg_first
    bool tau;                // weight rows through ws_tau
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
    int col_groups;              // sets of workgroups (blockIdx.y), each with slots of its own over all rows
    int row_perm;                // 1: rows of a group are read through tau (launch has channel-major tiles)
    int max_slots;               // largest number of slots any wave holds
    int resid_a2;                // 1: every residual is the second operand itself (same rows): taken from its LDS slab
    // row mask of the launch (all masked tiles share it), or nullptr
    const T* rowmask;
    int m_so, m_si;
    unsigned m_inner;
    // trailing FFK_TILE_BIAS tile (<= 4 heads, K = 128), pb_heads = 0: none.  It takes no weight slot - its few dot products per row
    // are 16 x 16 x 32 MFMAs on the slab in LDS
    int pb_heads, pb_wrow;
    unsigned pb_inner;
    T* pb_out;
    int pb_so, pb_sh;
    float pb_scale;
    WsSlot slot[WS_WAVES * WS_NS];   // [column group][wave][slot]
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

__device__ __forceinline__ void unpack4(const T* p, float (&f)[4]) {
    u32x2 raw = *reinterpret_cast<const u32x2*>(p);
    const T* h = reinterpret_cast<const T*>(&raw);
#pragma unroll
    for (int e = 0; e < 4; ++e) f[e] = (float)h[e];
}

// Index permutation tau(8a + 4h + b) = 16h + 4a + b.  An MFMA accumulator register v = 4a + b of
// half-wave h holds row 8a + 4h + b of the M operand; loading M-operand row i from source row tau(i)
// therefore leaves source rows 16h .. 16h + 15 in registers 0 .. 15: sixteen consecutive channels
// (or rows) per lane, i.e. 32 contiguous bytes to store.
__device__ __forceinline__ int ws_tau(int i) { return ((i >> 2) & 1) * 16 + (i >> 3) * 4 + (i & 3); }

__device__ __forceinline__ void unpack8(const T* p, float* f) {
    u32x4 raw = *reinterpret_cast<const u32x4*>(p);
    const T* h = reinterpret_cast<const T*>(&raw);
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] = (float)h[e];
}

// Two forms of each epilogue.  The "compact" one funnels every bias / activation / scale combination
// through one intermediate array; the other gives each combination its own straight-line path from the
// accumulators to the rounded outputs, which executes about 30 vector instructions fewer per 32x32 block
// (no register copies where paths join, no cleared gate accumulator for plain units) but needs more
// registers.  The kernel variants with three or four weight slots or K = 256 have no registers to spare -
// there the second form spills, and a spill costs far more than it saves - so they keep the compact form.
// ---- lane = row (n32 = its row within the group), registers = channels -----------------------
// STRIDED tiles: weight rows were loaded through tau, registers hold channels 16*half + v.
// ACC / QK tiles: natural weight order, registers hold channels 8a + 4*half + b.
// sb: this slot's 32 (GLU: 64) bias values in LDS (fp32); rmask: the row's mask value.
template <bool GLU, bool XT, bool POS>
__device__ __forceinline__ void ws_store_rows_compact(const WsSlot& t, const f32x16& acc, const f32x16& accg, const float* sb,
                                              bool valid, unsigned mc, unsigned hi, unsigned lo, float rmask, int half) {
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
    if (t.masked || t.scale != 1.0f) {
        const float scl = t.scale * rmask;
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
            if (XT && t.xtail) {     // extended residual stream (whole 16-channel runs: ncols % 16 == 0 with a tail)
                const u32x4 tv = *reinterpret_cast<const u32x4*>(t.xtail + (ok1 ? off : off - cl));
                u32x4 tn;
#pragma unroll
                for (int j = 0; j < 2; ++j) {       // eight channels at a time (register budget)
                    float f[8];
                    xs_decode8(rv[j], tv[2 * j], tv[2 * j + 1], f);
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        float u = (float)y[8 * j + e];
                        if (gate) u = (float)(T)(u * gate_factor((float)reinterpret_cast<const T*>(&gv[j])[e], POS ? t.act : FFK_ACT_NONE));
                        f[e] += u;
                    }
                    u32x4 hv;
                    uint32_t ta, tb;
                    xs_encode8(f, hv, ta, tb);
                    tn[2 * j] = ta;
                    tn[2 * j + 1] = tb;
                    if (ok1) *reinterpret_cast<u32x4*>(out + off + 8 * j) = hv;
                }
                if (ok1) *reinterpret_cast<u32x4*>(t.xtail + off) = tn;
                return;
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const T* gh = reinterpret_cast<const T*>(&gv[j]);
                const T* rh = reinterpret_cast<const T*>(&rv[j]);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    float f = (float)y[8 * j + e];
                    if (gate) f = (float)(T)(f * gate_factor((float)gh[e], POS ? t.act : FFK_ACT_NONE));
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
// sm: mask values (fp32, LDS) of the group's 32 rows, or nullptr.
template <bool GLU>
__device__ __forceinline__ void ws_store_cols_compact(const WsSlot& t, const f32x16& acc, const f32x16& accg, const float* sb,
                                              const float* sm, long m0g, int M, int l32, int half) {
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
    // the mask multiply is skipped for row groups without a masked row (the common case)
    if (sm && !vt && __builtin_amdgcn_ballot_w64(sm[l32] != 1.0f) != 0) {
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const f32x4 mk = *reinterpret_cast<const f32x4*>(sm + 16 * half + 4 * a);
#pragma unroll
            for (int b = 0; b < 4; ++b) x[4 * a + b] *= mk[b];
        }
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

// ---- lane = row (n32 = its row within the group), registers = channels -----------------------
// STRIDED tiles: weight rows were loaded through tau, registers hold channels 16*half + v.
// ACC / QK tiles: natural weight order, registers hold channels 8a + 4*half + b.
// sb: this slot's 32 (GLU: 64) bias values in LDS (fp32); rmask: the row's mask value.
template <bool GLU, bool XT>
__device__ __forceinline__ void ws_store_rows(const WsSlot& t, const f32x16& acc, const f32x16& accg, const float* sb,
                                              bool valid, unsigned mc, unsigned hi, unsigned lo, float rmask, int half) {
    const bool strided = t.kind == FFK_TILE_STRIDED;
    // Every combination of bias / activation / scale is its own straight-line path from the accumulators
    // to the rounded outputs: a shared intermediate array makes the compiler copy the 16 registers where
    // the paths join, and the vector instruction count is what this kernel's time follows.
    T y[16];
    const bool scaled = t.masked || t.scale != 1.0f;
    const float scl = t.scale * rmask;
    auto emit = [&](auto value) {
        if (scaled) {
#pragma unroll
            for (int v = 0; v < 16; ++v) y[v] = (T)(value(v) * scl);
        } else {
#pragma unroll
            for (int v = 0; v < 16; ++v) y[v] = (T)value(v);
        }
    };
    if (GLU || t.has_bias || t.act == FFK_ACT_SIGMOID) {
        f32x4 bv[4], bg[4];
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const int o = strided ? 16 * half + 4 * a : 4 * half + 8 * a;
            bv[a] = *reinterpret_cast<const f32x4*>(sb + o);
            if (GLU) bg[a] = *reinterpret_cast<const f32x4*>(sb + 32 + o);
        }
        if (GLU) {
            emit([&](int v) { return (acc[v] + bv[v >> 2][v & 3]) * ws_sigmoid_pre(accg[v], bg[v >> 2][v & 3]); });
        } else if (t.act == FFK_ACT_SIGMOID) {
            emit([&](int v) { return ws_sigmoid_pre(acc[v], bv[v >> 2][v & 3]); });
        } else if (t.act == FFK_ACT_RELU) {
            emit([&](int v) { return relu_f(acc[v] + bv[v >> 2][v & 3]); });
        } else {
            emit([&](int v) { return acc[v] + bv[v >> 2][v & 3]; });
        }
    } else if (t.act == FFK_ACT_RELU) {
        emit([&](int v) { return relu_f(acc[v]); });
    } else {
        emit([&](int v) { return acc[v]; });
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
            if (XT && t.xtail) {     // extended residual stream (whole 16-channel runs: ncols % 16 == 0 with a tail)
                const u32x4 tv = *reinterpret_cast<const u32x4*>(t.xtail + (ok1 ? off : off - cl));
                u32x4 tn;
#pragma unroll
                for (int j = 0; j < 2; ++j) {       // eight channels at a time (register budget)
                    float f[8];
                    xs_decode8(rv[j], tv[2 * j], tv[2 * j + 1], f);
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        float u = (float)y[8 * j + e];
                        if (gate) u = (float)(T)(u * gate_factor((float)reinterpret_cast<const T*>(&gv[j])[e], t.act));
                        f[e] += u;
                    }
                    u32x4 hv;
                    uint32_t ta, tb;
                    xs_encode8(f, hv, ta, tb);
                    tn[2 * j] = ta;
                    tn[2 * j + 1] = tb;
                    if (ok1) *reinterpret_cast<u32x4*>(out + off + 8 * j) = hv;
                }
                if (ok1) *reinterpret_cast<u32x4*>(t.xtail + off) = tn;
                return;
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
// sm: mask values (fp32, LDS) of the group's 32 rows, or nullptr.
template <bool GLU>
__device__ __forceinline__ void ws_store_cols(const WsSlot& t, const f32x16& acc, const f32x16& accg, const float* sb,
                                              const float* sm, long m0g, int M, int l32, int half) {
    const float bv = sb[l32], bg = GLU ? sb[32 + l32] : 0.0f;
    float x[16];
    if (GLU) {
#pragma unroll
        for (int v = 0; v < 16; ++v) x[v] = (acc[v] + bv) * ws_sigmoid_pre(accg[v], bg);
    } else if (t.act == FFK_ACT_SIGMOID) {
#pragma unroll
        for (int v = 0; v < 16; ++v) x[v] = ws_sigmoid_pre(acc[v], bv);
    } else if (t.act == FFK_ACT_RELU) {
#pragma unroll
        for (int v = 0; v < 16; ++v) x[v] = relu_f(acc[v] + bv);
    } else if (t.has_bias) {
#pragma unroll
        for (int v = 0; v < 16; ++v) x[v] = acc[v] + bv;
    } else {
#pragma unroll
        for (int v = 0; v < 16; ++v) x[v] = acc[v];
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
    // the mask multiply is skipped for row groups without a masked row (the common case)
    if (sm && !vt && __builtin_amdgcn_ballot_w64(sm[l32] != 1.0f) != 0) {
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const f32x4 mk = *reinterpret_cast<const f32x4*>(sm + 16 * half + 4 * a);
#pragma unroll
            for (int b = 0; b < 4; ++b) x[4 * a + b] *= mk[b];
        }
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
// XT: the launch has tiles with a residual tail (extended residual stream); only those instantiations carry its code
template <int NS, int WS_K, bool CM, bool DUAL, bool XT>
__global__ __launch_bounds__(WS_THREADS, 2) void linear_ws_kernel(const WsArgs args) {
    typedef Mma<T> MM;
    typedef WsGeo<WS_K> G;
    constexpr int WS_KS = G::KS, WS_AP = G::AP, WS_BM = G::BM, WS_RG = G::RG, LPR = G::LPR, RPP = G::RPP;
    constexpr bool ALLOW_GLU = NS >= 2 && WS_K <= 128;
    constexpr bool LEAN = NS == 2 && WS_K <= 128 && !DUAL;   // straight-line epilogues where the registers allow them
    constexpr bool POS = NS == 2 && !XT;                   // variants that take FFK_ACT_GATE_POS (the others have no register for it)
    constexpr int AFC = WS_K == 128 ? 8 : 4;               // A fragments held at a time (register budget)
    const WsArgs& d = args;
    extern __shared__ __align__(16) unsigned char smem[];
    unsigned char* s_a = smem;                                                 // [2][WS_BM][WS_AP]
    float* s_mask = reinterpret_cast<float*>(smem + 2 * WS_BM * WS_AP);        // [2][WS_BM]
    float* s_bias = s_mask + 2 * WS_BM;                                        // [n_tiles][128]
    unsigned char* s_a2 = reinterpret_cast<unsigned char*>(s_bias + FFK_MAX_TILES * 128);   // DUAL: [2][WS_BM][256 B]
    static_assert(!DUAL || (WS_K == 128 && WS_BM == 128), "the second operand is built for K = 128");
    // LayerNorm parameters that are only needed when a slab is committed wait in LDS, not in registers
    float* s_cmln = reinterpret_cast<float*>(s_a2 + (DUAL ? 2 * WS_BM * 256 : 0));          // CM: gamma[128], beta[128] (fp32)
    T* s_ln2 = reinterpret_cast<T*>(s_cmln + (CM ? 256 : 0));                               // DUAL: gamma2[128], beta2[128]
    T* s_ln1 = s_ln2 + (DUAL ? 256 : 0);                                                    // !CM: gamma[K], beta[K]
    float* s_c1 = reinterpret_cast<float*>(s_ln1 + (CM ? 0 : 2 * WS_K));                    // DUAL: folded LayerNorm row sums
    constexpr bool PB = !CM && !DUAL && !XT && WS_K == 128;    // variants that take a trailing pair-bias tile
    T* s_wb = reinterpret_cast<T*>(s_c1);                                                   // PB: [4][WS_K] head weights
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
    for (int s = 0; s < NS; ++s) sp[s] = args.slot[((int)blockIdx.y * WS_WAVES + wave) * NS + s];
    // launches with channel-major tiles read the rows of a group through tau (16 consecutive rows per lane)
    const int n32 = args.row_perm ? ws_tau(l32) : l32;

    // ---- slab streaming: thread -> (row tid / LPR + RPP * i, 8 channels starting at 8 * (tid % LPR)) ----
    const int c8 = tid % LPR, r0 = tid / LPR;
    // DUAL launches carry both LayerNorms folded into the weights: ln_gamma is the fp32 table of row sums and
    // both slabs are used as they arrive (see ws_store_rows_folded)
    const bool folded = DUAL;
    const bool ln = d.ln_gamma != nullptr && !folded;
    // row mask of the launch (all masked tiles share it): fetched with the slab, kept in LDS as fp32
    const T* rm = args.rowmask;
    const unsigned m_inner = args.m_inner;
    const int m_so = args.m_so, m_si = args.m_si;
    // plain row-major operands (inner >= M) need no division per fetched vector
    const bool a_flat = d.a_inner >= M, a2_flat = DUAL && d.a2_inner >= M, m_flat = m_inner >= (unsigned)M;
    Vec16<T> pre[4];
    T pm[4];
    // Channel-major A (element (m, k) at a + k * a_cs + rowoffset(m), K = 128 or 64): a thread fetches eight
    // consecutive rows of channel k = lane % 32 + 32 cb (cb < K / 32); the two half-waves of wave w own the row
    // groups 2w and 2w + 1 of each 128-row pass of the slab (one pass at K = 128, two at K = 64), so the LayerNorm
    // reduction over k stays inside 32 lanes.  The slab is transposed on its way into LDS (2-byte stores,
    // consecutive lanes -> consecutive k of one row).
    constexpr int CMI = CM ? WS_K / 32 : 4;              // channel blocks per thread
    static_assert(!CM || WS_K == 128 || WS_K == 64, "channel-major operands are built for K = 128 and 64");
    const int cm_k = lane & 31, cm_mg = 2 * wave + (lane >> 5);
    // second operand: vector v = i * 512 + tid of a slab is row v / 16, LDS column v % 16, which holds
    // global column (v % 16) ^ (row % 16); the 16 lanes of a row are adjacent, as the LayerNorm wants them
    const int a2_col = (tid & 15) ^ ((tid >> 4) & 15);
    const unsigned lds_a2 = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)s_a2;
    auto fetch = [&](int slab, int tobuf) {
        if (DUAL) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                long m = (long)slab * WS_BM + i * 32 + (tid >> 4);
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
        if (CM) {
#pragma unroll
            for (int rp = 0; rp < 4 / CMI; ++rp) {
                long m = (long)slab * WS_BM + (cm_mg + 16 * rp) * 8;
                m = m < M ? m : M - 8;                   // M % 8 == 0; clamped groups are never stored
                const unsigned hi = a_flat ? 0u : (unsigned)m / (unsigned)d.a_inner, lo = (unsigned)m - hi * (unsigned)d.a_inner;
                const T* base = A + (long)hi * d.a_so + lo;  // a_si == 1
#pragma unroll
                for (int cb = 0; cb < CMI; ++cb) pre[rp * CMI + cb] = ld16(base + (long)(cm_k + 32 * cb) * d.a_cs);
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            long m = (long)slab * WS_BM + r0 + RPP * i;
            m = m < M ? m : M - 1;                       // clamped: rows past the end are never stored
            const unsigned hi = a_flat ? 0u : (unsigned)m / (unsigned)d.a_inner, lo = (unsigned)m - hi * (unsigned)d.a_inner;
            pre[i] = ld16(A + (long)hi * d.a_so + (long)lo * d.a_si + c8 * 8);
            if (rm) {
                const unsigned mh = m_flat ? 0u : (unsigned)m / m_inner, ml = (unsigned)m - mh * m_inner;
                pm[i] = rm[(long)mh * m_so + (long)ml * m_si];
            }
        }
    };
    auto commit = [&](int buf) {
        unsigned char* sa = s_a + buf * (WS_BM * WS_AP);
        if (DUAL) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this thread's vectors of the second operand have landed
        if (CM) {
            if (!ln) {       // nothing to normalise here: the transposition is a plain copy
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int j = 0; j < 8; ++j)
                        *reinterpret_cast<T*>(sa + ((cm_mg + 16 * (i / CMI)) * 8 + j) * WS_AP + (cm_k + 32 * (i % CMI)) * 2) = pre[i].e[j];
                return;
            }
            float f[4][8];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 8; ++j) f[i][j] = (float)pre[i].e[j];
            if (ln) {
                float cm_g[CMI], cm_b[CMI];              // gamma / beta of this lane's channels
#pragma unroll
                for (int cb = 0; cb < CMI; ++cb) {
                    cm_g[cb] = s_cmln[(lane & 31) + 32 * cb];
                    cm_b[cb] = s_cmln[WS_K + (lane & 31) + 32 * cb];
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
                    *reinterpret_cast<T*>(sa + ((cm_mg + 16 * (i / CMI)) * 8 + j) * WS_AP + (cm_k + 32 * (i % CMI)) * 2) = (T)f[i][j];
            return;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            Vec16<T> x = pre[i];
            if (ln) {
                const Vec16<T> gam = *reinterpret_cast<const Vec16<T>*>(s_ln1 + c8 * 8);
                const Vec16<T> bet = *reinterpret_cast<const Vec16<T>*>(s_ln1 + WS_K + c8 * 8);
                float f[8], s = 0.0f;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    f[e] = (float)x.e[e];
                    s += f[e];
                }
                const float mu = group_sum(s, LPR) * (1.0f / WS_K);
                float q = 0.0f;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    f[e] -= mu;
                    q += f[e] * f[e];
                }
                const float rs = rsqrtf(group_sum(q, LPR) * (1.0f / WS_K) + d.ln_eps);
#pragma unroll
                for (int e = 0; e < 8; ++e) x.e[e] = (T)(f[e] * rs * (float)gam.e[e] + (float)bet.e[e]);
            }
            *reinterpret_cast<Vec16<T>*>(sa + (r0 + RPP * i) * WS_AP + c8 * 16) = x;
            if (rm && c8 == 0) s_mask[buf * WS_BM + r0 + RPP * i] = (float)pm[i];
        }
    };

    const int nslabs = (M + WS_BM - 1) / WS_BM;
    int slab = blockIdx.x;                               // grid <= nslabs
    const int pb_heads = PB ? args.pb_heads : 0;
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
        T tg[2] = {(T)0.0f, (T)0.0f}, tw = (T)0.0f;
#pragma unroll
        for (int sl = 0; sl < NS; ++sl) tb[sl] = sp[sl].wrow >= 0 && sp[sl].bias ? (float)sp[sl].bias[l32] : 0.0f;
        if (ln && tid < WS_K) {
            tg[0] = ((const T*)d.ln_gamma)[tid];
            tg[1] = ((const T*)d.ln_beta)[tid];
        }
        if (PB && pb_heads && tid < pb_heads * WS_K) tw = W[(long)args.pb_wrow * WS_K + tid];     // 4 * WS_K == WS_THREADS
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
                const int wl = sp[sl].tau ? ws_tau(l32) : l32;
#pragma unroll
                for (int k = 0; k < NI; ++k)
                    wf[sl][pc * NI + k] = *reinterpret_cast<const bf16x8*>(
                        stage + wl * (PW * 2) + (((2 * k + half) ^ (wl & (LR - 1))) * 16));
            }
#pragma unroll
        for (int sl = 0; sl < NS; ++sl)                   // (waves of a group write the same values)
            if (half == 0 && sp[sl].wrow >= 0) s_bias[sp[sl].wrow + l32] = sp[sl].sig ? -1.4426950408889634f * tb[sl] : tb[sl];
        if (ln && tid < WS_K) {
            if (CM) {
                s_cmln[tid] = (float)tg[0];
                s_cmln[WS_K + tid] = (float)tg[1];
            } else {
                s_ln1[tid] = tg[0];
                s_ln1[WS_K + tid] = tg[1];
            }
        }
        if (PB && pb_heads && tid < 4 * WS_K) s_wb[tid] = tw;
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
        if (PB && pb_heads && blockIdx.y == 0) {
            // pair bias of this slab on the matrix pipe: wave w takes the rows 16 w .. 16 w + 15 as the N operand of
            // four 16 x 16 x 32 products against the (at most four) head weight rows, zero rows up to 16 (M operand).
            // The rows are the operand as the other products see it (normalised, rounded to bf16), so the value
            // equals a further output column group of four channels.  Result layout: lane = row, register v = head
            // (4 * (lane / 16) + v: only the first sixteen lanes hold real heads).
            const int r16 = lane & 15, kq = lane >> 4;
            const unsigned char* xr = sa + (wave * 16 + r16) * WS_AP + kq * 16;
            const T* wr = s_wb + (r16 & 3) * WS_K + kq * 8;
            f32x4 pacc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int ks = 0; ks < WS_K / 32; ++ks) {
                const bf16x8 xv = *reinterpret_cast<const bf16x8*>(xr + ks * 64);
                bf16x8 wv = *reinterpret_cast<const bf16x8*>(wr + ks * 32);
                if (r16 >= 4) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) wv[e] = (T)0.0f;
                }
                pacc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv, xv, pacc, 0, 0, 0);
            }
            const long pm = (long)slab * WS_BM + wave * 16 + r16;
            if (kq == 0 && pm < M) {
                const unsigned hi = (unsigned)pm / args.pb_inner, lo = (unsigned)pm - hi * args.pb_inner;
                T* po = args.pb_out + (long)(int)(hi >> 5) * args.pb_so + (long)(lo >> 5) * 1024 + qk_tile_off((int)(lo & 31), (int)(hi & 31));
#pragma unroll
                for (int hd = 0; hd < 4; ++hd)
                    if (hd < pb_heads) po[(long)hd * args.pb_sh] = (T)(pacc[hd] * args.pb_scale);
            }
        }
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
            const float* smk = s_mask + buf * WS_BM + rg * 32;
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
                if constexpr (LEAN) {
                    const bool rows = sp[s].by_rows;
                    // One straight-line body per (store order, GLU or not): the gate accumulator only exists
                    // where it is used, and no accumulator has to be copied or cleared where paths would join.
                    auto slot_body = [&](auto rows_tag, auto glu_tag) {
                        constexpr bool ROWS = decltype(rows_tag)::value, G = decltype(glu_tag)::value;
                        f32x16 acc, accg;
#pragma unroll
                        for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
                        if (G) {
#pragma unroll
                            for (int v = 0; v < 16; ++v) accg[v] = 0.0f;
                        }
                        if (DUAL && G) {
                            // gate half: fragments of the second operand's row (row % 16 == l32 % 16 picks the swizzle)
                            const unsigned a2row = (unsigned)(buf * (WS_BM * 256) + (rg * 32 + n32) * 256 + ((half ^ (n32 & 15)) << 4));
#pragma unroll
                            for (int k0 = 0; k0 < WS_KS; k0 += AFC) {
                                bf16x8 af[AFC];
#pragma unroll
                                for (int ks = 0; ks < AFC; ++ks)
                                    af[ks] = *reinterpret_cast<const bf16x8*>(s_a2 + ((a2row + reread) ^ (unsigned)((k0 + ks) * 32)));
#pragma unroll
                                for (int ks = 0; ks < AFC; ++ks) MM::mma(accg, wf[sg][k0 + ks], af[ks]);
                            }
                        }
#pragma unroll
                        for (int k0 = 0; k0 < WS_KS; k0 += AFC) {          // AFC K steps of A in registers at a time
                            bf16x8 af[AFC];
#pragma unroll
                            for (int ks = 0; ks < AFC; ++ks) af[ks] = *reinterpret_cast<const bf16x8*>(ap + reread + (k0 + ks) * 32);
                            if (ROWS) {
#pragma unroll
                                for (int ks = 0; ks < AFC; ++ks) MM::mma(acc, wf[s][k0 + ks], af[ks]);
                                if (!DUAL && G) {
#pragma unroll
                                    for (int ks = 0; ks < AFC; ++ks) MM::mma(accg, wf[sg][k0 + ks], af[ks]);
                                }
                            } else {
#pragma unroll
                                for (int ks = 0; ks < AFC; ++ks) MM::mma(acc, af[ks], wf[s][k0 + ks]);
                                if (G) {
#pragma unroll
                                    for (int ks = 0; ks < AFC; ++ks) MM::mma(accg, af[ks], wf[sg][k0 + ks]);
                                }
                            }
                        }
                        if (ROWS) {
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
                            const float rmask = t.masked ? smk[n32] : 1.0f;
                            ws_store_rows<G, XT>(t, acc, G ? accg : acc, sb, valid, mc, c_hi, c_lo, rmask, half);
                        } else {
                            const float* sm = t.masked ? smk : nullptr;
                            ws_store_cols<G>(t, acc, G ? accg : acc, sb, sm, m0g, M, l32, half);
                        }
                    };
                    typedef std::integral_constant<bool, true> Yes;
                    typedef std::integral_constant<bool, false> No;
                    if (ALLOW_GLU && glu) {
                        if (rows) slot_body(Yes(), Yes());
                        else slot_body(No(), Yes());
                    } else {
                        if (rows) slot_body(Yes(), No());
                        else slot_body(No(), No());
                    }
                } else {
                    f32x16 acc, accg;
#pragma unroll
                    for (int v = 0; v < 16; ++v) acc[v] = accg[v] = 0.0f;
                    float st1 = 0.0f, st2 = 0.0f, su1 = 0.0f, su2 = 0.0f;   // row statistics of the two operands (DUAL)
                    const bool rows = sp[s].by_rows;
                    if (DUAL && ALLOW_GLU && glu) {
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
                            if (!DUAL && ALLOW_GLU && glu) {
#pragma unroll
                                for (int ks = 0; ks < AFC; ++ks) MM::mma(accg, wf[sg][k0 + ks], af[ks]);
                            }
                        } else {
#pragma unroll
                            for (int ks = 0; ks < AFC; ++ks) MM::mma(acc, af[ks], wf[s][k0 + ks]);
                            if (ALLOW_GLU && glu) {
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
                        const float rmask = t.masked ? smk[n32] : 1.0f;
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
                        } else if (ALLOW_GLU && glu) ws_store_rows_compact<true, XT, POS>(t, acc, accg, sb, valid, mc, c_hi, c_lo, rmask, half);
                        else ws_store_rows_compact<false, XT, POS>(t, acc, accg, sb, valid, mc, c_hi, c_lo, rmask, half);
                    } else {
                        const float* sm = t.masked ? smk : nullptr;
                        if (ALLOW_GLU && glu) ws_store_cols_compact<true>(t, acc, accg, sb, sm, m0g, M, l32, half);
                        else ws_store_cols_compact<false>(t, acc, accg, sb, sm, m0g, M, l32, half);
                    }
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
    if (t.kind == FFK_TILE_V) return t.inner % 32 == 0 && t.ncols % 32 == 0 && t.s_o % 8 == 0 && t.s_h % 8 == 0;
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
    q.masked = t.rowmask != nullptr;
    q.has_bias = t.bias != nullptr;
    q.by_rows = ws_by_rows(t);
    q.tau = t.kind == FFK_TILE_STRIDED && t.s_d == 1;
    q.sig = t.glu ? glu == 2 : t.act == FFK_ACT_SIGMOID;     // gate halves of a GLU unit and sigmoid tiles
    q.rg_first = (signed char)rg_first;
    q.rg_mask = (signed char)(rg_step - 1);
    return q;
}

// Distributes the 32-row weight units over the waves; false if they do not fit.  Plain units, up to 16 of them: unit i goes to
// wave i % 8 as its first or second slot; a round of at most four units is given to two or more waves each, which take every
// second (or fourth ..) row group of a slab, so that any multiple of four units loads the waves equally.  Up to 32 plain units
// are two column groups of 16: one launch pays for its start (6 .. 7 us) once.  Otherwise (GLU units) the waves form G = 8 / R
// groups; the R waves of a group hold the same units and take every R-th row group (R as large as the units allow).
bool ws_make_plan(const ffk_linear_desc& d, int n_tiles, WsArgs& p, int rg_per_slab, int max_ns) {
    struct Unit { int tile, chan, wrow, slots; };
    Unit units[FFK_MAX_TILES * 4];
    int nu = 0;
    bool plain = true;
    for (int i = 0; i < n_tiles; ++i) {
        const ffk_tile& t = d.tiles[i];
        const int n = (t.ncols + 31) / 32;
        plain = plain && !t.glu;
        for (int u = 0; u < n; ++u) units[nu++] = {i, u * 32, i * 128 + (t.glu ? u * 64 : u * 32), t.glu ? 2 : 1};
    }
    for (auto& q : p.slot) {
        q = WsSlot{};
        q.wrow = -1;
    }
    p.col_groups = 1;
    if (plain && nu <= 32) {
        p.max_slots = 2;
        p.col_groups = nu <= 16 ? 1 : 2;
        const int per = (nu + p.col_groups - 1) / p.col_groups;
        for (int cg = 0; cg < p.col_groups; ++cg)
            for (int sl = 0; sl < 2; ++sl) {
                const int first = cg * per + 8 * sl;
                int n = (cg + 1) * per < nu ? (cg + 1) * per - first : nu - first;
                n = n > 8 ? 8 : n;
                int R = 1;
                while (n > 0 && 2 * R * n <= WS_WAVES && 2 * R <= rg_per_slab) R *= 2;
                for (int w = 0; w < n * R; ++w) {
                    const Unit& u = units[first + w % n];
                    p.slot[(cg * WS_WAVES + w) * 2 + sl] = ws_slot(d, u.tile, u.chan, u.wrow, 0, w / n, R);
                }
            }
        return true;
    }
    int assign[WS_WAVES][WS_NS];
    int G = 0, R = 0;
    for (R = rg_per_slab; R >= 1; R >>= 1) {
        G = WS_WAVES / R;
        int load[WS_WAVES] = {0};
        for (int g = 0; g < G; ++g)
            for (int s = 0; s < WS_NS; ++s) assign[g][s] = -1;
        bool fits = true;
        for (int pass = 2; pass >= 1 && fits; --pass) {            // two-slot (GLU) units first
            for (int i = 0; i < nu && fits; ++i) {
                if (units[i].slots != pass) continue;
                int best = -1;
                for (int g = 0; g < G; ++g)
                    if (load[g] + pass <= max_ns && (best < 0 || load[g] < load[best])) best = g;
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
    p.max_slots = 2;
    for (int g = 0; g < G; ++g) {
        int n = 0;
        for (int sl = 0; sl < WS_NS; ++sl) n += assign[g][sl] != -1;
        p.max_slots = n > p.max_slots ? n : p.max_slots;
    }
    if (p.max_slots > 2) p.max_slots = max_ns;                     // the slots a wave of the launched kernel has
    for (int w = 0; w < WS_WAVES; ++w)
        for (int sl = 0; sl < p.max_slots; ++sl) {
            const int a = assign[w % G][sl];
            if (a == -1) continue;
            const Unit& u = units[a >= 0 ? a : -2 - a];
            p.slot[w * p.max_slots + sl] = ws_slot(d, u.tile, u.chan, u.wrow + (a >= 0 ? 0 : 32), a < 0 ? 2 : u.slots == 2 ? 1 : 0, w / G, R);
        }
    return true;
}

template <int NS, int K, bool CM, bool DUAL = false, bool XT = false>
int ws_launch(const WsArgs& args, hipStream_t st) {
    constexpr int WS_BM = WsGeo<K>::BM;
    const size_t smem = 2 * (size_t)WS_BM * WsGeo<K>::AP + 2 * WS_BM * sizeof(float) + FFK_MAX_TILES * 128 * sizeof(float) +
                        (DUAL ? 2 * (size_t)WS_BM * 256 + 256 * sizeof(T) + FFK_MAX_TILES * 128 * sizeof(float) : 0) +
                        (CM ? 256 * sizeof(float) : 2 * K * sizeof(T)) +
                        (!CM && !DUAL && !XT && K == 128 ? 4 * K * sizeof(T) : 0);      // head weights of a pair-bias tile
    static FfkLdsReservation lds_reserved;
    {
        const int rc_lds = ffk_reserve_lds(lds_reserved, (const void*)linear_ws_kernel<NS, K, CM, DUAL, XT>, smem, "ffk_fused_linear");
        if (rc_lds != FFK_OK) return rc_lds;
    }
    const int nslabs = ffk_cdiv(args.M, WS_BM), most = WS_MAX_GRID / args.col_groups;
    linear_ws_kernel<NS, K, CM, DUAL, XT><<<dim3(nslabs < most ? nslabs : most, args.col_groups), WS_THREADS, smem, st>>>(args);
    return ffk_check_launch("ffk_fused_linear");
}

}  // namespace

// Launches the weights-stationary kernel if it can take this (already validated) descriptor and
// returns 1 with the launch status in *status; returns 0 if the caller has to use another variant.
int ffk_linear_ws_try(const ffk_linear_desc* d, hipStream_t st, int* status) {
    if (d->dtype != FFK_BF16 || (d->K != 64 && d->K != 128 && d->K != 256)) return 0;
    if ((d->ln_folded != 0) != (d->a2 != nullptr)) return 0;    // folded LayerNorms and the second operand go together
    if (d->a_chanmajor && ((d->K != 128 && d->K != 64) || d->a_si != 1 || d->a_inner % 8 || d->a_so % 8 || d->a_cs % 8 || d->M % 8)) return 0;
    if (d->a2 && d->K != 128) return 0;                          // the second operand is built for K = 128
    const bool k256 = d->K == 256;
    if (d->variant == FFK_LINEAR_STAGED) return 0;
    auto i32 = [](int64_t v) { return v >= -0x7fffffffL && v <= 0x7fffffffL; };      // the kernel's strides have 32 bits
    if (!i32(d->a_so) || !i32(d->a_si) || !i32(d->a_cs) || !i32(d->a2_so) || !i32(d->a2_si)) return 0;
    for (int i = 0; i < d->n_tiles; ++i) {
        const ffk_tile& t = d->tiles[i];
        if (!i32(t.s_o) || !i32(t.s_i) || !i32(t.s_d) || !i32(t.s_h) || !i32(t.gate_ld) || !i32(t.m_so) || !i32(t.m_si)) return 0;
    }
    bool chan_major = false, v_tiles = false, tails = false;
    int mask_tile = -1;
    // a trailing pair-bias tile (score-operand tiles of <= 4 heads) rides on the launch without a weight slot; it may be
    // the only tile (a chunked attention computes its bias before the first slab, with the bits of the riding one)
    int n_slot_tiles = d->n_tiles, bias_tile = -1;
    if (d->tiles[d->n_tiles - 1].kind == FFK_TILE_BIAS) {
        const ffk_tile& t = d->tiles[d->n_tiles - 1];
        auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
        if (d->K != 128 || d->a_chanmajor || d->a2 || t.ncols < 1 || t.ncols > 4 || t.bias || t.resid || t.gate || t.rowmask ||
            t.xtail || t.glu || t.act != FFK_ACT_NONE || t.inner <= 0 || !t.out || !al16(t.out))
            return 0;
        bias_tile = d->n_tiles - 1;
        n_slot_tiles = d->n_tiles - 1;
    }
    for (int i = 0; i < n_slot_tiles; ++i) {
        const ffk_tile& t = d->tiles[i];
        if (t.kind == FFK_TILE_BIAS) return 0;
        if (!ws_tile_ok(*d, t)) return 0;
        tails = tails || t.xtail != nullptr;
        chan_major = chan_major || (!ws_by_rows(t) && t.kind == FFK_TILE_STRIDED);
        v_tiles = v_tiles || t.kind == FFK_TILE_V;
        if (t.rowmask) {
            if (mask_tile < 0) {
                mask_tile = i;
            } else {
                const ffk_tile& f = d->tiles[mask_tile];     // one mask per launch
                if (t.rowmask != f.rowmask || t.inner != f.inner || t.m_so != f.m_so || t.m_si != f.m_si) return 0;
            }
        }
    }
    if (chan_major && v_tiles) return 0;          // they need different row orders within a group
    WsArgs args;
    const bool k64 = d->K == 64;
    if (!ws_make_plan(*d, n_slot_tiles, args, k256 ? WsGeo<256>::RG : (k64 ? WsGeo<64>::RG : WsGeo<128>::RG), k256 ? 2 : (k64 ? 4 : 3)))
        return 0;
    if (bias_tile >= 0 && (tails || chan_major)) return 0;   // built into the plain K = 128 variants only
    for (int i = 0; i < n_slot_tiles; ++i)
        if (d->tiles[i].act == FFK_ACT_GATE_POS && (tails || args.max_slots > 2)) return 0;
    if (k256) {
        for (int i = 0; i < d->n_tiles; ++i)
            if (d->tiles[i].glu) return 0;                   // GLU units are only built for K = 128
    }
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
    args.resid_a2 = 0;
    args.rowmask = nullptr;
    args.m_so = args.m_si = 0;
    args.m_inner = 1;
    if (mask_tile >= 0) {
        const ffk_tile& t = d->tiles[mask_tile];
        args.rowmask = (const T*)t.rowmask;
        args.m_so = (int)t.m_so;
        args.m_si = (int)t.m_si;
        args.m_inner = (unsigned)t.inner;
    }
    args.pb_heads = 0;
    if (bias_tile >= 0) {
        const ffk_tile& t = d->tiles[bias_tile];
        args.pb_heads = t.ncols;
        args.pb_wrow = bias_tile * 128;
        args.pb_inner = (unsigned)t.inner;
        args.pb_out = (T*)t.out;
        args.pb_so = (int)t.s_o;
        args.pb_sh = (int)t.s_h;
        args.pb_scale = t.scale;
    }
    if (d->a2) {
        // second operand: every unit must be a GLU unit stored [row][channel], first operand channel-major
        if (!d->a_chanmajor || args.max_slots > 2 || mask_tile >= 0 || d->a2_si % 8 || d->a2_so % 8) return 0;
        bool resid_a2 = true;
        for (int i = 0; i < d->n_tiles; ++i) {
            const ffk_tile& t = d->tiles[i];
            if (!t.glu || !ws_by_rows(t)) return 0;
            // plain residual GLU tiles of 64 channels only
            if (t.kind != FFK_TILE_STRIDED || t.gate || t.rowmask || t.scale != 1.0f || t.ncols != 64) return 0;
            // the residual is the second operand itself: same rows, channels [c0, c0 + 64) of its 128
            const long c0 = (const T*)t.resid - (const T*)d->a2;
            if (!t.resid || c0 < 0 || c0 + t.ncols > 128 || c0 % 32 || t.s_o != d->a2_so || t.s_i != d->a2_si ||
                t.inner != d->a2_inner || t.s_h != 32 || t.s_d != 1)
                resid_a2 = false;
        }
        args.resid_a2 = resid_a2 ? 1 : 0;
        *status = tails ? ws_launch<2, 128, true, true, true>(args, st) : ws_launch<2, 128, true, true>(args, st);
    } else if (tails) {
        // residual tails: built for the output projections of the attentions (one plain tile group, two slots)
        if (d->a_chanmajor || args.max_slots > 2 || k64) return 0;
        *status = k256 ? ws_launch<2, 256, false, false, true>(args, st) : ws_launch<2, 128, false, false, true>(args, st);
    } else if (d->a_chanmajor) {
        if (args.max_slots > 2 || mask_tile >= 0) return 0;
        *status = k64 ? ws_launch<2, 64, true>(args, st) : ws_launch<2, 128, true>(args, st);
    } else if (k256) {
        *status = ws_launch<2, 256, false>(args, st);
    } else if (k64) {
        *status = args.max_slots <= 2 ? ws_launch<2, 64, false>(args, st) : ws_launch<4, 64, false>(args, st);
    } else {
        *status = args.max_slots <= 2 ? ws_launch<2, 128, false>(args, st) : ws_launch<3, 128, false>(args, st);
    }
    return 1;
}
