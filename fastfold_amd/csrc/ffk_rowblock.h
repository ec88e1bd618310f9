// Kernels that take a block of rows from x to the updated rows (ffk_attention_block.hip, ffk_transition_block.hip): eight waves, the
// rows and the update in LDS, row by row, so that every access to memory is of whole rows.
#pragma once
#include "ffk_common.h"

namespace {

typedef bf16_t T;
typedef Mma<T> MM;

struct RbRows {
    T* out;
    const T* x;
    int8_t* xtail;           // tail bytes of x / out as an extended residual stream, or nullptr
    const T *gamma, *beta;
    const T* drop;           // [n][C] multipliers of the update, or nullptr
    long s_tok;              // elements from row to row
    int n;                   // rows of the block
    float eps;
};

// The lane number anew, so that the addresses made from it are not kept in registers from one end of a kernel to the other.
__device__ __forceinline__ int rb_lane(int lane) {
    asm volatile("" : "+v"(lane));
    return lane;
}
// Computed here: the compiler would otherwise move the packing to the value's use and keep the unpacked numbers in twice the registers.
__device__ __forceinline__ void rb_pin(bf16x8& f) { asm volatile("" : "+v"(*reinterpret_cast<u32x4*>(&f))); }

__device__ __forceinline__ bf16x8 rb_pack8(const f32x16& a, int v0, float scale) {
    bf16x8 r;
#pragma unroll
    for (int t = 0; t < 8; ++t) r[t] = (T)(a[v0 + t] * scale);
    return r;
}

// What the rows take: eight waves, C / 8 lanes to a row, so that a request of a wave is 1 KB of whole rows.
template <int C, int NT_MAX> struct RbGeo {
    static constexpr int LPR = C / 8, RPI = 64 / LPR, NI = NT_MAX * 32 / (8 * RPI), XP = C * 2 + 16;
    // rows i of all waves lie before row 32 NT, or none (half of them: 64 channels and an odd NT)
    static __device__ __forceinline__ bool past(int i, int NT) { return i * 8 * RPI >= NT * 32; }
    static __device__ __forceinline__ int row(int i, int wave, int lane) { return (i * 8 + wave) * RPI + lane / LPR; }
};

// Rows of the batch row -> LayerNorm -> LDS (row-major, 16 bytes of padding); rows past the end repeat the last one.
template <int C, int NT_MAX>
__device__ __forceinline__ void rb_normalise(const RbRows& a, const T* xrow, unsigned char* s_x, int NT, int wave, int lane) {
    typedef RbGeo<C, NT_MAX> R;
    const int c8 = lane % R::LPR;
    const Vec16<T> g = ld16(a.gamma + c8 * 8), b = ld16(a.beta + c8 * 8);
    Vec16<T> r[R::NI];
#pragma unroll
    for (int i = 0; i < R::NI; ++i) {
        if (R::past(i, NT)) break;
        const int tok = R::row(i, wave, lane);
        r[i] = ld16(xrow + (long)(tok < a.n ? tok : a.n - 1) * a.s_tok + c8 * 8);
    }
#pragma unroll
    for (int i = 0; i < R::NI; ++i) {
        if (R::past(i, NT)) break;
        float f[8], s = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            f[e] = (float)r[i].e[e];
            s += f[e];
        }
        const float q = centre8(f, group_sum(s, R::LPR) * (1.0f / C));
        const float rs = rsqrtf(group_sum(q, R::LPR) * (1.0f / C) + a.eps);
        bf16x8 y;
#pragma unroll
        for (int e = 0; e < 8; ++e) y[e] = (T)__builtin_fmaf(f[e] * rs, (float)g.e[e], (float)b.e[e]);
        const int row = R::row(i, wave, lane);
        if (row < NT * 32) *reinterpret_cast<bf16x8*>(s_x + row * R::XP + c8 * 16) = y;
    }
}

// The update of a 32 x 32 block (lane: token l32, channels 16 half ..), rounded, to its place in the rows of updates in LDS.
__device__ __forceinline__ void rb_put(unsigned char* p, f32x16& acc, const T* bo) {
    if (bo) {
        const Vec16<T> b0 = ld16(bo), b1 = ld16(bo + 8);
#pragma unroll
        for (int v = 0; v < 8; ++v) {
            acc[v] += (float)b0.e[v];
            acc[8 + v] += (float)b1.e[v];
        }
    }
    *reinterpret_cast<bf16x8*>(p) = rb_pack8(acc, 0, 1.0f);
    *reinterpret_cast<bf16x8*>(p + 16) = rb_pack8(acc, 8, 1.0f);
}

// out = x + update (times its dropout multipliers).  The rows are requested (`fetch`) before the barrier that completes the updates:
// a lane with a token's 16 channels, as the accumulators have them, would touch 32 lines per request and the epilogue take twice as long.
template <int C, int NT_MAX> struct RbUpdate {
    typedef RbGeo<C, NT_MAX> R;
    u32x4 h[R::NI];
    u32x2 t[R::NI];
    __device__ __forceinline__ void fetch(const RbRows& a, long row_off, int NT, int wave, int lane) {
#pragma unroll
        for (int i = 0; i < R::NI; ++i) {
            if (R::past(i, NT)) break;
            const int tok = R::row(i, wave, lane);
            const long off = row_off + (long)(tok < a.n ? tok : a.n - 1) * a.s_tok + (lane % R::LPR) * 8;
            h[i] = *reinterpret_cast<const u32x4*>(a.x + off);
            if (a.xtail) t[i] = *reinterpret_cast<const u32x2*>(a.xtail + off);
        }
    }
    __device__ __forceinline__ void store(const RbRows& a, const unsigned char* s_u, long row_off, int NT, int wave, int lane) const {
        const int c8 = lane % R::LPR;
#pragma unroll
        for (int i = 0; i < R::NI; ++i) {
            if (R::past(i, NT)) break;
            const int tok = R::row(i, wave, lane);
            if (tok >= a.n) continue;
            const bf16x8 u = *reinterpret_cast<const bf16x8*>(s_u + tok * R::XP + c8 * 16);
            float upd[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) upd[e] = (float)u[e];
            if (a.drop) {
                const Vec16<T> d = ld16(a.drop + (long)tok * C + c8 * 8);
#pragma unroll
                for (int e = 0; e < 8; ++e) upd[e] = (float)(T)(upd[e] * (float)d.e[e]);
            }
            const long off = row_off + (long)tok * a.s_tok + c8 * 8;
            u32x4 hn;
            if (a.xtail) {
                float f[8];
                u32x2 tn;
                xs_decode8(h[i], t[i][0], t[i][1], f);
#pragma unroll
                for (int e = 0; e < 8; ++e) f[e] += upd[e];
                xs_encode8(f, hn, tn);
                *reinterpret_cast<u32x2*>(a.xtail + off) = tn;
            } else {
                const bf16x8 x = __builtin_bit_cast(bf16x8, h[i]);
                bf16x8 y;
#pragma unroll
                for (int e = 0; e < 8; ++e) y[e] = (T)(upd[e] + (float)x[e]);
                hn = __builtin_bit_cast(u32x4, y);
            }
            *reinterpret_cast<u32x4*>(a.out + off) = hn;
        }
    }
};

}  // namespace
