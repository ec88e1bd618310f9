// Backward of the attention core for head dimensions 32, 64 and 128 (see ffk_attention_bwd and ffk_attention_bwd_rows in
// include/ffk.h).
// A head wider than 32 is cut into DP = D / 32 parts of 32 channels, each with operand tiles of its own (part-major:
// part p of a tensor lies p * part elements behind part 0): scores and dP are sums over the parts, dq / dk / dv have one
// accumulator tile per part.
//
// Like the forward kernel it never forms the [B2, H, Nq, Nk] logits in memory: all three kernels recompute the
// 32 x 32 score tiles from q and k on the matrix pipe.  With  s = q.k / sqrt(d) + bias  (masked keys very
// negative),  P = softmax_k(s),  o = P v  and the incoming gradient  do:
//     D[q]  = sum_d do[q, d] o[q, d]
//     dP    = do . v^T                 dS = P (dP - D)         (gradient w.r.t. the logits s)
//     dq    = dS . k / sqrt(d)         dk = dS^T . q / sqrt(d)
//     dv    = P^T . do                 dbias[h, q, k] = sum_b2 dS
//   attention_bwd_dq_kernel   one wave per (b2, head, NT tiles of 32 queries): a walk over the key tiles accumulates dq^T = k^T . dS^T,
//                             the score tile transposed (keys along the MFMA rows) exactly as in the forward kernel,
//                             so that dS^T is the N operand of that product as it stands.  Row log-sum-exp and D come
//                             from the forward pass and the re-tiling (ffk_attention_bwd_rows) or from a walk before
//                             it (ffk_attention_bwd, log2 domain), which leaves them for the other two kernels.
//   attention_bwd_dkv_kernel  one wave per (b2, head, NT tiles of 32 keys): walks the query tiles with the score tile the other
//                             way round (queries along the MFMA rows, one key per lane), so that P and dS are the N
//                             operands of  dv^T = do^T . P  and  dk^T = q^T . dS.
//   attention_bwd_dbias_kernel  one wave per (head, query tile, NT key tiles, slice of the batch rows): recomputes dS of
//                             its tiles for every batch row of the slice and sums in registers; the slices (what fills
//                             the chip when H * QT * KT alone is a few hundred tiles) are left as partial sums the
//                             caller adds up (ffk_attention_bwd_rows) or added with one fp32 atomic per element.
// They take the pair bias from the same operand tiles as the forward kernel: added to the scores by a product with
// an identity operand, in the last two with the roles of the two operands exchanged (rows = queries); in fp32 dq and
// dk / dv read its values in the order of the scores and add them.
// Every operand arrives in the tile order its role needs.  Waves load their tiles straight from global memory, each
// operand of the next step requested as soon as its registers are free, and no LDS is used: what bounds the kernels is
// the latency of that chain and the exponentials, with three waves per SIMD to cover it, or two of two tiles each (NT = 2:
// the operands of the walk are read once for both).  128 x 8 heads of 256 x 256 logits, bf16, one tile per wave and loads
// that waited for each other, requested in time, two tiles per wave: dq 39.6, 38.8, 35.0 us, dk / dv 56.5, 56.2, 46.1,
// d bias 41.5, 40.5, 32.1; fp32, the first two: dq 198, 173, dk / dv 232, 229, d bias 127, 121.
#include "ffk_common.h"
#include <initializer_list>
#include <type_traits>

namespace {

constexpr float REF_FLOOR = -1.0e4f;          // as in the forward kernel: rows whose every score lies below are all-masked
constexpr float NO_ROW = 3.0e38f;             // log-sum-exp of a row without a valid key: exp2(s - NO_ROW) = 0

template <typename T> struct Tile16 {         // the 16 elements one lane owns of a 1024-element tile
    static constexpr int NV = 16 / DT<T>::VEC;
    Vec16<T> v[NV];
    __device__ __forceinline__ void load(const T* p) {
#pragma unroll
        for (int i = 0; i < NV; ++i) v[i] = ld16(p + i * DT<T>::VEC);
    }
    // Both operands of a product over the tiles' minor index may take that index in any common order: access i of the lanes of
    // row `row` covers elements 16 i' + VEC (2 i'' + half) .. of it (bf16: i' = i, so that one access of the wave is a
    // contiguous KB; in the order of load() it is every other 16 bytes of two).  p: the tile + row * 16.
    __device__ __forceinline__ void load_rows(const T* p, int half) {
        constexpr int PER = NV / 2;
#pragma unroll
        for (int i = 0; i < NV; ++i) v[i] = ld16(p + (i / PER) * 512 + ((i % PER) * 2 + half) * DT<T>::VEC);
    }
    __device__ __forceinline__ float f(int j) const { return DT<T>::to_f(v[j / DT<T>::VEC].e[j % DT<T>::VEC]); }
    __device__ __forceinline__ typename Mma<T>::Frag frag(int i) const {
        return *reinterpret_cast<const typename Mma<T>::Frag*>(
            reinterpret_cast<const unsigned char*>(&v[0]) + i * sizeof(typename Mma<T>::Frag));
    }
};

// Requests above this point are issued above it: without it the compiler moves loads of the next step behind the branch back, in
// front of their first use, to save registers, and every step waits for them (117 x 4 heads of 117 x 117: d bias 18.1 us, 14.4 with
// it; dk / dv are left as they are by the compiler, and d bias in pairs, 32.1 us at 128 x 8 heads of 256, is 34.0 with it).
template <bool HERE> __device__ __forceinline__ void issue_here() {
    if (HERE) asm volatile("" ::: "memory");
}

// fragments (N operand) of 16 fp32 values held in accumulator order, rounded to the operand type
template <typename T> struct NFrag;
template <> struct NFrag<bf16_t> {
    static __device__ __forceinline__ bf16x8 make(const float* p) {
        bf16x8 r;
#pragma unroll
        for (int t = 0; t < 8; ++t) r[t] = (bf16_t)p[t];
        return r;
    }
};
template <> struct NFrag<float> {
    static __device__ __forceinline__ f32x4 make(const float* p) {
        f32x4 r;
#pragma unroll
        for (int t = 0; t < 4; ++t) r[t] = p[t];
        return r;
    }
};

template <typename T>
__device__ __forceinline__ typename Mma<T>::Frag identity_frag(int i, int l32, int half) {
    constexpr int PER = 8 / Mma<T>::KLANE;                      // the order of Tile16::load_rows
    typename Mma<T>::Frag f;
#pragma unroll
    for (int t = 0; t < Mma<T>::KLANE; ++t) f[t] = (T)((16 * (i / PER) + ((i % PER) * 2 + half) * Mma<T>::KLANE + t) == l32 ? 1.0f : 0.0f);
    return f;
}

// fp32: the bias is added to the scores; through the matrix pipe, as in bf16, it was a product of 16 x 64 cycles beside the three (four)
// that the walk is made of (128 x 8 heads of 256 x 256: dq 173 -> 150, dk / dv 229 -> 195 us).
template <typename T> constexpr bool bias_add = sizeof(T) == 4;

// Workgroup -> logical block.  The hardware hands consecutive workgroup ids to the eight XCDs in turn, each with its own
// L2; the launches round their grids up to a multiple of eight and every XCD takes a contiguous eighth of the logical
// order, so that the waves that walk the same k / v (or q / do) tiles run behind one L2.
__device__ __forceinline__ long bwd_logical_block() {
    const unsigned per_xcd = gridDim.x >> 3;
    return (long)(blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
}

// Where a gradient goes: element (b2, head, token, d) at b2 * s_b + head * s_h + token * s_n + d.
struct OutMap {
    long s_b, s_h, s_n;
};

template <typename T>
__device__ __forceinline__ void store4(T* o, const float* f) {          // four consecutive elements, 4-element aligned
    T r[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) r[e] = DT<T>::from_f(f[e]);
    if (sizeof(T) == 2) *reinterpret_cast<u32x2*>(o) = *reinterpret_cast<const u32x2*>(r);
    else *reinterpret_cast<u32x4*>(o) = *reinterpret_cast<const u32x4*>(r);
}

// ------------------------------------------------------------------------------ dq ----
// STATS: the row statistics are computed here (a walk over the keys of its own) and written for the other kernels; otherwise
// the forward pass has left the log-sum-exp and the gate's backward kernel sum_d do o.
template <typename T, int DP, int NT, bool HAS_BIAS, bool STATS>
__global__ __launch_bounds__(256, DP == 1 && sizeof(T) == 2 ? (NT == 1 ? 3 : 2) : 1) void attention_bwd_dq_kernel(
    T* __restrict__ dq, float* __restrict__ lse, float* __restrict__ dsum, const T* __restrict__ q_qk,
    const T* __restrict__ k_qk, const T* __restrict__ k_acc, const T* __restrict__ v_qk, const T* __restrict__ bias_t,
    const float* __restrict__ keybias, const T* __restrict__ do_qk, const T* __restrict__ o_qk, int B2, int H, int Nq,
    int Nk, float dq_scale, long part_q, long part_k, OutMap om, int bias_pad) {
    typedef Mma<T> MM;
    typedef typename MM::Frag Frag;
    constexpr bool BIAS_ADD = bias_add<T>;
    constexpr int NF = 16 / MM::KLANE;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int l32 = lane & 31, half = lane >> 5;
    const int QT = (Nq + 31) >> 5, KT = (Nk + 31) >> 5;
    static_assert(NT == 1 || !STATS, "statistics: one query tile per wave");
    const int QP = (QT + NT - 1) / NT;
    const long item = bwd_logical_block() * 4 + wave;
    if (item >= (long)B2 * H * QP) return;
    const int qt0 = (int)(item % QP) * NT;
    const long bh = item / QP;
    const int h = (int)(bh % H), b2 = (int)(bh / H);
    auto qtile = [&](int t) { return NT == 1 || qt0 + t < QT ? qt0 + t : QT - 1; };   // a tile past the last one is the last one again, not stored
    const int qt = qt0;

    Tile16<T> qf[NT][DP], dof[NT][DP];
    float dpart = 0.0f;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int p = 0; p < DP; ++p) {
            const long off = p * part_q + ((bh * QT + qtile(t)) << 10) + l32 * 16;
            qf[t][p].load_rows(q_qk + off, half);
            dof[t][p].load_rows(do_qk + off, half);
            if (STATS) {
                Tile16<T> of;
                of.load_rows(o_qk + off, half);
#pragma unroll
                for (int j = 0; j < 16; ++j) dpart += dof[t][p].f(j) * of.f(j);
            }
        }
    float D[NT];                                               // this lane's queries: sum_d do o
#pragma unroll
    for (int t = 0; t < NT; ++t) D[t] = STATS ? dpart + lane_xor<32>(dpart) : dsum[(bh * QT + qtile(t)) * 32 + l32];
    const float* mp = keybias + (long)b2 * KT * 32 + 4 * half;

    Frag ident[NF];
    if (HAS_BIAS) {
#pragma unroll
        for (int i = 0; i < NF; ++i) ident[i] = identity_frag<T>(i, l32, half);
    }
    // S^T tile kt (rows: keys, columns: queries), log2 domain, key bias included
    auto score = [&](int kt, f32x16& s) {
#pragma unroll
        for (int v = 0; v < 16; ++v) s[v] = 0.0f;
#pragma unroll
        for (int p = 0; p < DP; ++p) {
            Tile16<T> kc;
            kc.load_rows(k_qk + p * part_k + ((bh * KT + kt) << 10) + l32 * 16, half);
#pragma unroll
            for (int i = 0; i < NF; ++i) MM::mma(s, kc.frag(i), qf[0][p].frag(i));
        }
        if (HAS_BIAS) {
            Tile16<T> bc;
            bc.load_rows(bias_t + ((((long)h * QT + qt) * (KT + bias_pad) + kt) << 10) + l32 * 16, half);
#pragma unroll
            for (int i = 0; i < NF; ++i) MM::mma(s, bc.frag(i), ident[i]);
        }
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const f32x4 mk = *reinterpret_cast<const f32x4*>(mp + kt * 32 + 8 * g);
#pragma unroll
            for (int e = 0; e < 4; ++e) s[4 * g + e] += mk[e];
        }
    };

    float L[NT];
    if (STATS) {
        // first walk: row maximum and sum
        float m_run = REF_FLOOR, l_run = 0.0f;
        for (int kt = 0; kt < KT; ++kt) {
            f32x16 s;
            score(kt, s);
            float mt = fmaxf(s[0], s[1]);
#pragma unroll
            for (int v = 2; v < 16; ++v) mt = fmaxf(mt, s[v]);
            mt = fmaxf(mt, lane_xor<32>(mt));
            const float m_new = fmaxf(m_run, mt);
            float ts = 0.0f;
#pragma unroll
            for (int v = 0; v < 16; ++v) ts += fast_exp2(s[v] - m_new);
            l_run = l_run * fast_exp2(m_run - m_new) + ts;
            m_run = m_new;
        }
        const float l_tot = l_run + lane_xor<32>(l_run);
        L[0] = l_tot > 0.0f ? m_run + __builtin_amdgcn_logf(l_tot) : NO_ROW;   // v_log_f32 is log2
        if (half == 0) {
            lse[(bh * QT + qt) * 32 + l32] = L[0];
            dsum[(bh * QT + qt) * 32 + l32] = D[0];
        }
    } else {
#pragma unroll
        for (int t = 0; t < NT; ++t) L[t] = lse[(bh * QT + qtile(t)) * 32 + l32];
    }

    // second walk: dq^T += k^T . dS^T.  What a step reads is requested for the next step as soon as its registers are free
    // (a step later it is there; waiting for each tile where it is used took 57 us, NT = 1, at 128 x 8 heads of 256 x 256 logits).
    // The scores start at key bias - log-sum-exp and dP at -D, so that the products leave the exponent and dP - D themselves.
    f32x16 acc[NT][DP];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int p = 0; p < DP; ++p)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[t][p][v] = 0.0f;
    Tile16<T> kc[DP], vq[DP], ka[DP], bc[NT];
    f32x4 mk[4];
    const T* bias_row[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
        bias_row[t] = HAS_BIAS ? bias_t + ((((long)h * QT + qtile(t)) * (KT + bias_pad)) << 10) + l32 * 16 : nullptr;
    const T* bias_tile = HAS_BIAS ? bias_t + ((((long)h * QT + qt) * (KT + bias_pad)) << 10) + (4 * half + 32 * (l32 >> 4)) * 16 + (l32 & 15) : nullptr;
    float ba[HAS_BIAS && BIAS_ADD ? 16 : 1];
    const long krow = (bh * KT) << 10;
    auto load_mask = [&](int kt) {
#pragma unroll
        for (int g = 0; g < 4; ++g) mk[g] = *reinterpret_cast<const f32x4*>(mp + kt * 32 + 8 * g);
    };
    auto load_scores = [&](int kt) {
#pragma unroll
        for (int p = 0; p < DP; ++p) {
            kc[p].load_rows(k_qk + p * part_k + krow + ((long)kt << 10) + l32 * 16, half);
            vq[p].load_rows(v_qk + p * part_k + krow + ((long)kt << 10) + l32 * 16, half);
        }
        if constexpr (HAS_BIAS && BIAS_ADD) {                  // keys 8 g + 4 half + e of this lane's query
            const T* bp = bias_tile + ((long)kt << 10);
#pragma unroll
            for (int v = 0; v < 16; ++v) ba[v] = (float)bp[(8 * (v >> 2) + (v & 3)) * 16];
        } else if (HAS_BIAS) {
#pragma unroll
            for (int t = 0; t < NT; ++t) bc[t].load_rows(bias_row[t] + ((long)kt << 10), half);
        }
    };
    auto load_acc = [&](int kt) {
#pragma unroll
        for (int p = 0; p < DP; ++p) ka[p].load(k_acc + p * part_k + krow + ((long)kt << 10) + lane * 16);
    };
    load_mask(0);
    load_scores(0);
    load_acc(0);
    for (int kt = 0; kt < KT; ++kt) {
        const int next = kt + 1 < KT ? kt + 1 : kt;
        f32x16 s[NT], dp[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                s[t][v] = mk[v >> 2][v & 3] - L[t];
                dp[t][v] = -D[t];
            }
#pragma unroll
            for (int p = 0; p < DP; ++p) {
#pragma unroll
                for (int i = 0; i < NF; ++i) MM::mma(s[t], kc[p].frag(i), qf[t][p].frag(i));
#pragma unroll
                for (int i = 0; i < NF; ++i) MM::mma(dp[t], vq[p].frag(i), dof[t][p].frag(i));   // dP^T[key, q] = v[key] . do[q]
            }
            if constexpr (HAS_BIAS && BIAS_ADD) {
#pragma unroll
                for (int v = 0; v < 16; ++v) s[t][v] += ba[v];
            } else if (HAS_BIAS) {
#pragma unroll
                for (int i = 0; i < NF; ++i) MM::mma(s[t], bc[t].frag(i), ident[i]);
            }
        }
        load_scores(next);
        issue_here<DP == 1>();
        Frag dsf[NT][NF];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            float ds[16];
#pragma unroll
            for (int v = 0; v < 16; ++v) ds[v] = fast_exp2(s[t][v]) * dp[t][v];
#pragma unroll
            for (int i = 0; i < NF; ++i) dsf[t][i] = NFrag<T>::make(ds + i * MM::KLANE);
        }
        load_mask(next);                                       // late: the registers are those of the scores
        issue_here<DP == 1>();
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int p = 0; p < DP; ++p)
#pragma unroll
                for (int i = 0; i < NF; ++i) MM::mma(acc[t][p], ka[p].frag(i), dsf[t][i]);
        load_acc(next);
        issue_here<DP == 1>();
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int q = (qt0 + t) * 32 + l32;
        if (q >= Nq) continue;
        T* o = dq + (long)b2 * om.s_b + (long)h * om.s_h + (long)q * om.s_n + 4 * half;
#pragma unroll
        for (int p = 0; p < DP; ++p)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                float f[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) f[e] = acc[t][p][4 * g + e] * dq_scale;
                store4(o + 32 * p + 8 * g, f);
            }
    }
}

// ------------------------------------------------------------------------- dk, dv ----
template <typename T, int DP, int NT>
__global__ __launch_bounds__(256, DP == 1 && sizeof(T) == 2 ? (NT == 1 ? 3 : 2) : 1) void attention_bwd_dkv_kernel(
    T* __restrict__ dk, T* __restrict__ dv, const T* __restrict__ q_qk,
    const T* __restrict__ q_acc, const T* __restrict__ k_qk, const T* __restrict__ v_qk, const T* __restrict__ bias_t,
    const float* __restrict__ keybias, const T* __restrict__ do_qk, const T* __restrict__ do_acc,
    const float* __restrict__ lse, const float* __restrict__ dsum, int B2, int H, int Nq, int Nk, float dk_scale,
    long part_q, long part_k, OutMap om, int bias_pad) {
    typedef Mma<T> MM;
    typedef typename MM::Frag Frag;
    constexpr bool BIAS_ADD = bias_add<T>;
    constexpr int NF = 16 / MM::KLANE;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int l32 = lane & 31, half = lane >> 5;
    const int QT = (Nq + 31) >> 5, KT = (Nk + 31) >> 5;
    const int KP = (KT + NT - 1) / NT;
    const long item = bwd_logical_block() * 4 + wave;
    if (item >= (long)B2 * H * KP) return;
    const int kt0 = (int)(item % KP) * NT;
    const long bh = item / KP;
    const int h = (int)(bh % H), b2 = (int)(bh / H);
    auto ktile = [&](int t) { return NT == 1 || kt0 + t < KT ? kt0 + t : KT - 1; };   // a tile past the last one is the last one again, not stored

    Tile16<T> kf[NT][DP], vf[NT][DP];              // this lane's keys (column l32): k and v rows as N operands
    float kb[NT];                                  // 0, masked (-1e9 log2e) or padding (hugely negative)
#pragma unroll
    for (int t = 0; t < NT; ++t) {
#pragma unroll
        for (int p = 0; p < DP; ++p) {
            kf[t][p].load_rows(k_qk + p * part_k + ((bh * KT + ktile(t)) << 10) + l32 * 16, half);
            vf[t][p].load_rows(v_qk + p * part_k + ((bh * KT + ktile(t)) << 10) + l32 * 16, half);
        }
        kb[t] = keybias[((long)b2 * KT + ktile(t)) * 32 + l32];
    }
    Frag ident[NF];
    if (bias_t) {
#pragma unroll
        for (int i = 0; i < NF; ++i) ident[i] = identity_frag<T>(i, l32, half);
    }

    f32x16 acc_k[NT][DP], acc_v[NT][DP];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int p = 0; p < DP; ++p)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc_k[t][p][v] = acc_v[t][p][v] = 0.0f;
    // as in the dq kernel: each operand is requested for the next step once its registers are free
    Tile16<T> qc[DP], doc[DP], qa[DP], doa[DP], bc[NT];
    f32x4 L4[4], D4[4];
    const long qrow = (bh * QT) << 10;
    const float* lp = lse + bh * QT * 32 + 4 * half;
    const float* dpz = dsum + bh * QT * 32 + 4 * half;
    const T* bias_col[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) bias_col[t] = bias_t ? bias_t + ((((long)h * QT) * (KT + bias_pad) + ktile(t)) << 10) + l32 * 16 : nullptr;
    auto load_rows = [&](int qt) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            L4[g] = *reinterpret_cast<const f32x4*>(lp + qt * 32 + 8 * g);
            D4[g] = *reinterpret_cast<const f32x4*>(dpz + qt * 32 + 8 * g);
        }
    };
    auto load_scores = [&](int qt) {
#pragma unroll
        for (int p = 0; p < DP; ++p) {
            qc[p].load_rows(q_qk + p * part_q + qrow + ((long)qt << 10) + l32 * 16, half);
            doc[p].load_rows(do_qk + p * part_q + qrow + ((long)qt << 10) + l32 * 16, half);
        }
        if (bias_t) {
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const T* bp = bias_col[t] + (((long)qt * (KT + bias_pad)) << 10);
                if constexpr (BIAS_ADD) {                      // queries 8 g + 4 half .. of this lane's key
#pragma unroll
                    for (int g = 0; g < 4; ++g) bc[t].v[g] = ld16(bp + (g >> 1) * 512 + 8 * (g & 1) + 4 * half);
                } else {
                    bc[t].load_rows(bp, half);
                }
            }
        }
    };
    auto load_acc = [&](int qt) {
#pragma unroll
        for (int p = 0; p < DP; ++p) {
            qa[p].load(q_acc + p * part_q + qrow + ((long)qt << 10) + lane * 16);
            doa[p].load(do_acc + p * part_q + qrow + ((long)qt << 10) + lane * 16);
        }
    };
    load_rows(0);
    load_scores(0);
    load_acc(0);
    for (int qt = 0; qt < QT; ++qt) {
        const int next = qt + 1 < QT ? qt + 1 : qt;
        f32x16 s[NT], dp[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                s[t][v] = kb[t] - L4[v >> 2][v & 3];
                dp[t][v] = -D4[v >> 2][v & 3];
            }
#pragma unroll
            for (int p = 0; p < DP; ++p) {
#pragma unroll
                for (int i = 0; i < NF; ++i) MM::mma(s[t], qc[p].frag(i), kf[t][p].frag(i));       // S[q, key], log2 domain
#pragma unroll
                for (int i = 0; i < NF; ++i) MM::mma(dp[t], doc[p].frag(i), vf[t][p].frag(i));     // dP[q, key] = do[q] . v[key]
            }
            if (bias_t) {                                                           // S += bias; bf16: I . bias (rows = queries)
                if constexpr (BIAS_ADD) {
#pragma unroll
                    for (int v = 0; v < 16; ++v) s[t][v] += bc[t].f(v);
                } else {
#pragma unroll
                    for (int i = 0; i < NF; ++i) MM::mma(s[t], ident[i], bc[t].frag(i));
                }
            }
        }
        load_scores(next);
        Frag pfr[NT][NF], dsf[NT][NF];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            float p[16], ds[16];
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                p[v] = fast_exp2(s[t][v]);
                ds[v] = p[v] * dp[t][v];
            }
#pragma unroll
            for (int i = 0; i < NF; ++i) {
                pfr[t][i] = NFrag<T>::make(p + i * MM::KLANE);
                dsf[t][i] = NFrag<T>::make(ds + i * MM::KLANE);
            }
        }
        load_rows(next);                                   // late: the 32 registers are those of the scores
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int pp = 0; pp < DP; ++pp) {
#pragma unroll
                for (int i = 0; i < NF; ++i) MM::mma(acc_v[t][pp], doa[pp].frag(i), pfr[t][i]);   // dv^T += do^T . P
#pragma unroll
                for (int i = 0; i < NF; ++i) MM::mma(acc_k[t][pp], qa[pp].frag(i), dsf[t][i]);    // dk^T += q^T . dS
            }
        load_acc(next);
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int key = (kt0 + t) * 32 + l32;
        if (key >= Nk) continue;
        const long o = (long)b2 * om.s_b + (long)h * om.s_h + (long)key * om.s_n + 4 * half;
#pragma unroll
        for (int pp = 0; pp < DP; ++pp)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                float fk[4], fv[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    fk[e] = acc_k[t][pp][4 * g + e] * dk_scale;
                    fv[e] = acc_v[t][pp][4 * g + e];
                }
                store4(dk + o + 32 * pp + 8 * g, fk);
                store4(dv + o + 32 * pp + 8 * g, fv);
            }
    }
}

// ---------------------------------------------------------------------------- dbias ----
// dbias[h, q, key] += sum over the batch rows b2 = slice, slice + NS, ... of dS[b2, h, q, key].
template <typename T, int DP, int NT>
__global__ __launch_bounds__(256, DP == 1 && sizeof(T) == 2 ? (NT == 1 ? 3 : 2) : 1) void attention_bwd_dbias_kernel(
    float* __restrict__ dbias, const T* __restrict__ q_qk, const T* __restrict__ k_qk, const T* __restrict__ v_qk,
    const T* __restrict__ bias_t, const float* __restrict__ keybias, const T* __restrict__ do_qk,
    const float* __restrict__ lse, const float* __restrict__ dsum, int B2, int H, int Nq, int Nk, int NS,
    long part_q, long part_k, int bias_pad, int partial) {
    typedef Mma<T> MM;
    constexpr int NF = 16 / MM::KLANE;
    constexpr bool PIN = DP == 1 && (sizeof(T) == 4 || NT == 1);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int l32 = lane & 31, half = lane >> 5;
    const int QT = (Nq + 31) >> 5, KT = (Nk + 31) >> 5;
    const int KP = (KT + NT - 1) / NT;
    const long item = bwd_logical_block() * 4 + wave;          // key tile fastest: a block's waves share q and do
    if (item >= (long)NS * H * QT * KP) return;
    const int kt0 = (int)(item % KP) * NT;
    const int qt = (int)((item / KP) % QT);
    const int h = (int)((item / ((long)KP * QT)) % H);
    const int slice = (int)(item / ((long)KP * QT * H));
    auto ktile = [&](int t) { return NT == 1 || kt0 + t < KT ? kt0 + t : KT - 1; };   // a tile past the last one is the last one again, not stored

    f32x16 sb[NT], acc[NT];                                     // the bias tile in accumulator order, once; the sums
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        Tile16<T> bc;
        bc.load_rows(bias_t + ((((long)h * QT + qt) * (KT + bias_pad) + ktile(t)) << 10) + l32 * 16, half);
#pragma unroll
        for (int v = 0; v < 16; ++v) sb[t][v] = acc[t][v] = 0.0f;
#pragma unroll
        for (int i = 0; i < NF; ++i) MM::mma(sb[t], identity_frag<T>(i, l32, half), bc.frag(i));
    }
    // as in the dq kernel: each operand is requested for the next batch row once its registers are free
    Tile16<T> qc[DP], doc[DP], kf[NT][DP], vf[NT][DP];
    f32x4 L4[4], D4[4];
    float kb[NT];
    auto load_rows = [&](int b2) {
        const long bh = (long)b2 * H + h;
#pragma unroll
        for (int t = 0; t < NT; ++t) kb[t] = keybias[((long)b2 * KT + ktile(t)) * 32 + l32];
        const float* lp = lse + (bh * QT + qt) * 32 + 4 * half;
        const float* dpz = dsum + (bh * QT + qt) * 32 + 4 * half;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            L4[g] = *reinterpret_cast<const f32x4*>(lp + 8 * g);
            D4[g] = *reinterpret_cast<const f32x4*>(dpz + 8 * g);
        }
    };
    auto load_scores = [&](int b2) {
        const long bh = (long)b2 * H + h;
#pragma unroll
        for (int p = 0; p < DP; ++p) {
            qc[p].load_rows(q_qk + p * part_q + ((bh * QT + qt) << 10) + l32 * 16, half);
#pragma unroll
            for (int t = 0; t < NT; ++t) kf[t][p].load_rows(k_qk + p * part_k + ((bh * KT + ktile(t)) << 10) + l32 * 16, half);
            doc[p].load_rows(do_qk + p * part_q + ((bh * QT + qt) << 10) + l32 * 16, half);
#pragma unroll
            for (int t = 0; t < NT; ++t) vf[t][p].load_rows(v_qk + p * part_k + ((bh * KT + ktile(t)) << 10) + l32 * 16, half);
        }
    };
    load_rows(slice);                                          // slice < NS <= B2
    load_scores(slice);
    for (int b2 = slice; b2 < B2; b2 += NS) {
        const int next = b2 + NS < B2 ? b2 + NS : b2;
        f32x16 s[NT], dp[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                s[t][v] = sb[t][v] + (kb[t] - L4[v >> 2][v & 3]);
                dp[t][v] = -D4[v >> 2][v & 3];
            }
        load_rows(next);
        issue_here<PIN>();
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int p = 0; p < DP; ++p) {
#pragma unroll
                for (int i = 0; i < NF; ++i) MM::mma(s[t], qc[p].frag(i), kf[t][p].frag(i));
#pragma unroll
                for (int i = 0; i < NF; ++i) MM::mma(dp[t], doc[p].frag(i), vf[t][p].frag(i));
            }
        load_scores(next);
        issue_here<PIN>();
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[t][v] += fast_exp2(s[t][v]) * dp[t][v];
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int key = (kt0 + t) * 32 + l32;
        if (key >= Nk) continue;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int qrow = qt * 32 + acc_row(v, lane);
            if (qrow >= Nq) continue;
            if (partial) dbias[(((long)slice * H + h) * Nq + qrow) * Nk + key] = acc[t][v];
            else atomicAdd(dbias + ((long)h * Nq + qrow) * Nk + key, acc[t][v]);
        }
    }
}

// Slices of the batch rows of the pair-bias gradient: enough for ~ 8 waves per SIMD, at least 8 rows each.
long dbias_slices(long B2, long H, long QT, long KT) {
    const long tiles = H * QT * KT;
    long ns = (8L * 1024 + tiles - 1) / tiles;
    if (ns > (B2 + 7) / 8) ns = (B2 + 7) / 8;
    return ns < 1 ? 1 : ns;
}

template <typename T, int DP, bool STATS>
int launch_bwd(void* dq, void* dk, void* dv, float* dbias, float* lse, float* dsum, const void* q_qk, const void* q_acc,
               const void* k_qk, const void* k_acc, const void* v_qk, const void* bias_t,
               const float* keybias, const void* do_qk, const void* do_acc, const void* o_qk, long B2, long H, long Nq,
               long Nk, float dq_scale, float dk_scale, OutMap mq, OutMap mk, int bias_pad, long dbias_parts, hipStream_t st) {
    const long QT = (Nq + 31) / 32, KT = (Nk + 31) / 32;
    const long part_q = B2 * H * QT * 1024, part_k = B2 * H * KT * 1024;
    constexpr bool PAIRS = DP == 1 && sizeof(T) == 2;
    auto blocks = [](long waves) { return 8 * ((waves + 31) / 32); };                       // of four waves, a multiple of 8
    const long ns = !dbias ? 0 : (dbias_parts > 0 ? dbias_parts : dbias_slices(B2, H, QT, KT));
    FFK_REQUIRE(blocks(B2 * H * QT) < (1L << 31) && blocks(B2 * H * KT) < (1L << 31) && blocks(ns * H * QT * KT) < (1L << 31), FFK_ERR_SHAPE,
                "ffk_attention_bwd: too many tiles for one launch");
    typedef std::integral_constant<int, 1> One;
    typedef std::integral_constant<int, PAIRS ? 2 : 1> Two;
    auto run_dq = [&](auto nt_c) {
        constexpr int NT = decltype(nt_c)::value;
        const unsigned g = (unsigned)blocks(B2 * H * ((QT + NT - 1) / NT));
        if (bias_t)
            attention_bwd_dq_kernel<T, DP, NT, true, STATS><<<g, 256, 0, st>>>((T*)dq, lse, dsum, (const T*)q_qk, (const T*)k_qk, (const T*)k_acc,
                                                                             (const T*)v_qk, (const T*)bias_t, keybias, (const T*)do_qk,
                                                                             (const T*)o_qk, (int)B2, (int)H, (int)Nq, (int)Nk, dq_scale, part_q,
                                                                             part_k, mq, bias_pad);
        else
            attention_bwd_dq_kernel<T, DP, NT, false, STATS><<<g, 256, 0, st>>>((T*)dq, lse, dsum, (const T*)q_qk, (const T*)k_qk, (const T*)k_acc,
                                                                              (const T*)v_qk, nullptr, keybias, (const T*)do_qk, (const T*)o_qk,
                                                                              (int)B2, (int)H, (int)Nq, (int)Nk, dq_scale, part_q, part_k, mq, 0);
        return ffk_check_launch("ffk_attention_bwd");
    };
    auto run_dkv = [&](auto nt_c) {
        constexpr int NT = decltype(nt_c)::value;
        attention_bwd_dkv_kernel<T, DP, NT><<<(unsigned)blocks(B2 * H * ((KT + NT - 1) / NT)), 256, 0, st>>>(
            (T*)dk, (T*)dv, (const T*)q_qk, (const T*)q_acc, (const T*)k_qk, (const T*)v_qk, (const T*)bias_t, keybias, (const T*)do_qk,
            (const T*)do_acc, lse, dsum, (int)B2, (int)H, (int)Nq, (int)Nk, dk_scale, part_q, part_k, mk, bias_pad);
        return ffk_check_launch("ffk_attention_bwd");
    };
    auto run_dbias = [&](auto nt_c) {
        constexpr int NT = decltype(nt_c)::value;
        attention_bwd_dbias_kernel<T, DP, NT><<<(unsigned)blocks(ns * H * QT * ((KT + NT - 1) / NT)), 256, 0, st>>>(
            dbias, (const T*)q_qk, (const T*)k_qk, (const T*)v_qk, (const T*)bias_t, keybias, (const T*)do_qk, lse, dsum, (int)B2, (int)H,
            (int)Nq, (int)Nk, (int)ns, part_q, part_k, bias_pad, dbias_parts > 0 ? 1 : 0);
        return ffk_check_launch("ffk_attention_bwd");
    };
    // Two tiles per wave (bf16, 32 channels) read what a step shares once for both and are two chains that cover each other, in
    // registers for two waves per SIMD instead of three.  A launch takes about as long as the rounds of one wave on every SIMD that
    // it is, and a round of pairs 1.4 (d bias, dk / dv) or 1.7 (dq) rounds of single tiles.  us, single tiles and pairs, 4 heads:
    //   d bias  784 tiles 14.2, 19.3   1 536 20.3, 20.3   1 960 (seven a row) 22.0, 28.5   4 096 40.5, 31.8   8 192 76.7, 59.8
    //   dk / dv 768 5.2, 6.6   1 280 8.1, 7.1   2 560 15.4, 15.5   4 096 29.5, 23.0   8 192 56.2, 45.6   16 384 121.4, 91.6
    //   dq      2 560 18.5, 19.1   3 072 16.5, 17.5   3 584 19.1, 16.8   5 120 25.2, 26.3   6 144 30.4, 27.4   8 192 38.8, 34.7
    auto rounds = [](long waves) { return (waves + 1023) / 1024; };
    const bool pq = 4 * rounds(B2 * H * QT) >= 7 * rounds(B2 * H * ((QT + 1) / 2));
    const bool pk = 2 * rounds(B2 * H * KT) >= 3 * rounds(B2 * H * ((KT + 1) / 2));
    const bool pb = 2 * rounds(ns * H * QT * KT) >= 3 * rounds(ns * H * QT * ((KT + 1) / 2));
    int rc;
    if constexpr (STATS) rc = run_dq(One());
    else rc = pq ? run_dq(Two()) : run_dq(One());
    if (rc != FFK_OK) return rc;
    rc = pk ? run_dkv(Two()) : run_dkv(One());
    if (rc != FFK_OK || !dbias) return rc;
    return pb ? run_dbias(Two()) : run_dbias(One());
}

}  // namespace

extern "C" int ffk_attention_bwd(void* dq, void* dk, void* dv, float* dbias, float* lse, float* dsum, const void* q_qk,
                                 const void* q_acc, const void* k_qk, const void* k_acc, const void* v_qk, const void* bias_t,
                                 const float* keybias, const void* do_qk, const void* do_acc,
                                 const void* o_qk, int64_t B2, int64_t H, int64_t Nq, int64_t Nk, int64_t D, float dq_scale,
                                 float dk_scale, int dtype, void* stream) {
    FFK_REQUIRE(D == 32 || D == 64 || D == 128, FFK_ERR_SHAPE,
                "ffk_attention_bwd: head dimension %ld (32, 64 or 128; narrower heads arrive zero-padded to 32)", (long)D);
    FFK_REQUIRE(dq && dk && dv && lse && dsum && q_qk && q_acc && k_qk && k_acc && v_qk && keybias && do_qk && do_acc && o_qk,
                FFK_ERR_NULL, "ffk_attention_bwd: null pointer");
    FFK_REQUIRE(!dbias || bias_t, FFK_ERR_NULL, "ffk_attention_bwd: dbias needs bias_t");
    FFK_REQUIRE(B2 > 0 && B2 < 131072 && H > 0 && H < 65536 && Nq > 0 && Nk > 0 && Nq < (1 << 24) && Nk < (1 << 24),
                FFK_ERR_SHAPE, "ffk_attention_bwd: bad shape B2=%ld H=%ld Nq=%ld Nk=%ld", (long)B2, (long)H, (long)Nq, (long)Nk);
    FFK_REQUIRE(ffk_aligned16(dq) && ffk_aligned16(dk) && ffk_aligned16(dv) && ffk_aligned16(lse) && ffk_aligned16(dsum) &&
                    ffk_aligned16(q_qk) && ffk_aligned16(q_acc) && ffk_aligned16(k_qk) && ffk_aligned16(k_acc) &&
                    ffk_aligned16(v_qk) && ffk_aligned16(keybias) && ffk_aligned16(do_qk) && ffk_aligned16(do_acc) &&
                    ffk_aligned16(o_qk) && (!bias_t || ffk_aligned16(bias_t)),
                FFK_ERR_ALIGN, "ffk_attention_bwd: buffers must be 16-byte aligned");
    hipStream_t st = (hipStream_t)stream;
    const OutMap mq = {H * Nq * D, Nq * D, D}, mk = {H * Nk * D, Nk * D, D};
#define FFK_BWD_ARGS dq, dk, dv, dbias, lse, dsum, q_qk, q_acc, k_qk, k_acc, v_qk, bias_t, keybias, do_qk, do_acc, o_qk, \
                     B2, H, Nq, Nk, dq_scale, dk_scale, mq, mk, 0, 0, st
    switch (dtype) {
        case FFK_BF16:
            // D = 32 with the statistics found here is for callers of the library; this package has them from the forward pass
            return D == 32 ? launch_bwd<bf16_t, 1, true>(FFK_BWD_ARGS)
                           : (D == 64 ? launch_bwd<bf16_t, 2, true>(FFK_BWD_ARGS) : launch_bwd<bf16_t, 4, true>(FFK_BWD_ARGS));
        case FFK_F32:
            return D == 32 ? launch_bwd<float, 1, true>(FFK_BWD_ARGS)
                           : (D == 64 ? launch_bwd<float, 2, true>(FFK_BWD_ARGS) : launch_bwd<float, 4, true>(FFK_BWD_ARGS));
        default: return ffk_fail(FFK_ERR_DTYPE, "ffk_attention_bwd: unsupported dtype tag %d", dtype);
    }
#undef FFK_BWD_ARGS
}

extern "C" int ffk_attention_bwd_rows(void* dq, void* dk, void* dv, float* dbias, int64_t dbias_parts, const float* lse,
                                      const float* dsum, const void* q_t, const void* q_v, const void* k_t, const void* k_v,
                                      const void* v_t, const void* bias_t, const float* keybias, const void* do_t, const void* do_v,
                                      int64_t B2, int64_t H, int64_t N, int64_t s_b, int64_t s_h, int64_t s_n, float dq_scale,
                                      float dk_scale, int flags, int dtype, void* stream) {
    FFK_REQUIRE(dq && dk && dv && lse && dsum && q_t && q_v && k_t && k_v && v_t && keybias && do_t && do_v, FFK_ERR_NULL,
                "ffk_attention_bwd_rows: null pointer");
    FFK_REQUIRE(!dbias || (bias_t && dbias_parts > 0 && dbias_parts <= B2), FFK_ERR_NULL,
                "ffk_attention_bwd_rows: dbias needs bias_t and a number of partial sums between 1 and B2");
    FFK_REQUIRE(B2 > 0 && B2 < 131072 && H > 0 && H < 65536 && N > 0 && N < (1 << 24), FFK_ERR_SHAPE,
                "ffk_attention_bwd_rows: bad shape B2=%ld H=%ld N=%ld", (long)B2, (long)H, (long)N);
    for (const void* p : {(const void*)dq, (const void*)dk, (const void*)dv, (const void*)lse, (const void*)dsum, q_t, q_v, k_t, k_v,
                          v_t, bias_t, (const void*)keybias, do_t, do_v})
        FFK_REQUIRE(ffk_aligned16(p), FFK_ERR_ALIGN, "ffk_attention_bwd_rows: buffers must be 16-byte aligned");
    FFK_REQUIRE(s_b % 4 == 0 && s_h % 4 == 0 && s_n % 4 == 0, FFK_ERR_ALIGN, "ffk_attention_bwd_rows: strides must be multiples of 4 elements");
    const OutMap om = {s_b, s_h, s_n};
    const int pad = (flags & FFK_ATT_BIAS_PADDED) ? 1 : 0;
    hipStream_t st = (hipStream_t)stream;
    // with the statistics given neither is written
    switch (dtype) {
        case FFK_BF16: return launch_bwd<bf16_t, 1, false>(dq, dk, dv, dbias, (float*)lse, (float*)dsum, q_t, q_v, k_t, k_v, v_t, bias_t,
                                                           keybias, do_t, do_v, nullptr, B2, H, N, N, dq_scale, dk_scale, om, om, pad, dbias_parts, st);
        case FFK_F32: return launch_bwd<float, 1, false>(dq, dk, dv, dbias, (float*)lse, (float*)dsum, q_t, q_v, k_t, k_v, v_t, bias_t,
                                                         keybias, do_t, do_v, nullptr, B2, H, N, N, dq_scale, dk_scale, om, om, pad, dbias_parts, st);
        default: return ffk_fail(FFK_ERR_DTYPE, "ffk_attention_bwd_rows: unsupported dtype tag %d", dtype);
    }
}
