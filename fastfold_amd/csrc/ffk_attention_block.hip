// A whole gated attention sub-module in one kernel (see ffk_attention_block in include/ffk.h), bf16, as many hidden as input channels:
//     out = x + Wo . ( sigmoid( Wg . y + bg ) * softmax( q . k^T + bias ) v ) + bo,     q, k, v = Wq y, Wk y, Wv y,  y = LayerNorm(x)
//
// A workgroup of eight waves owns one batch row - the N tokens that attend to each other - from the rows of x to the updated rows.
// A wave owns a head (or a block of 32 channels: two heads of 16) of some or all of the tiles of 32 tokens, so that a weight fragment
// is fetched once for several products: with a wave per token tile, every wave fetching all the weights, the projections of 256 rows of
// 128 tokens at 256 channels took 42 us of a launch of 86, as many bytes out of the second-level cache as it delivers.  The phases:
//   rows -> LayerNorm -> LDS;  barrier
//   q, k, v and the gate of the wave's tiles in registers, packed as the MFMA operands they are next (the gate of 128 channels in fp32)
//   attention over the key tiles (k, v of all tokens in LDS, or in registers where one wave has all of a head's)
//   gated outputs -> LDS;  barrier;  output projection, a wave 32 output channels;  updates -> LDS;  barrier;  rows updated
// Nothing is transposed on the way: the accumulator of Wk y^T is the score product's A operand as it stands, that of Wq y^T its B
// operand, that of y Wv^T the A operand of the weighted sum, and the gated outputs are the B operand of the output projection, whose
// weight columns are packed in the accumulator's order.
//
// What bounds it: the matrix and vector instructions of a SIMD, which do not overlap (ffk_attention.hip), at two waves per SIMD.  At
// 256 rows of 256 tokens, 128 channels, of 37 us: rows and LayerNorm 4, projections 6, attention 15 (240 ns per wave and 32 x 32 scores;
// its instructions take 230 at the 2 GHz the clock falls to), barriers and exchanges 7, output projection and update 4.
// What it replaces moves q, k, v, the gate and the heads' outputs through memory and fills and drains the chip three times.
// us per sub-module, launches of their own -> here (both with the launch that computes the pair bias):
//   128 channels in 4 heads, N rows of N tokens:  N = 64 17.7 -> 15.0, 96 24.6 -> 19.6, 128 29.4 -> 22.8, 192 49 -> 33.5, 256 62 -> 48
//     (the gate in fp32 until it multiplies: no slower with a fourth tile's in LDS, 48.1 -> 54.3 with registers spilled for it; relative
//     error of the update against float64, launches of their own / gate in bf16 / in fp32: 5.00e-3 / 4.96e-3 / 4.77e-3)
//   64 channels in 4 heads:  N = 64 18.6 -> 11.1, 128 26.0 -> 15.0, 256 50.5 -> 32, 320 79 -> 77, 512 184 -> 171
//     (row sums of the probabilities as the matrix product's idle rows instead of eight dot instructions a tile: 320 77 -> 71, 512 171 -> 157)
//   64 channels in 8 heads, 1 024 rows of N tokens:  N = 64 68 -> 39, 160 147 -> 96, 256 196 -> 157, 384 376 -> 320
//     (more than 384 tokens: four tiles a wave with four heads each do not fit the registers, 512 593 -> 2 583)
//   256 channels in 8 heads, rows of 128 tokens, no bias:  64 rows 33.5 -> 27.8, 256 69 -> 34, 416 109 -> 59, 1 024 266 -> 125
//                            with a pair bias:  128 rows of 96 tokens 45 -> 29, of 128 tokens 51 -> 36
//   the same to the gated heads, output projection apart (k and v of four heads of 256 tokens fill the LDS: two workgroups to a row):
//                            128 rows of 160 tokens 67 -> 49, 192 74 -> 53, 256 87 -> 72;  512 rows of 256 296 -> 228
// Other numbers of rows: attention_block_tokens in model/fastnn/_fused.py.  Longer rows do not fit: at 128 channels, k and v of more than
// 256 tokens go into LDS in two passes only (heads two by two, rows normalised twice), which was built and is slower (288 tokens 122 us against 92, 416 235 against 189).
#include "ffk_rowblock.h"
#include <type_traits>

namespace {

struct AbArgs : RbRows {
    const T* w;              // [5][C / 32][C / 16][64][8]: q, k, v, gate, output projection
    const T *bg, *bo;
    const T* bias_t;         // [H][NT][bias_pitch] key x query tiles
    const float* keybias;    // [B2][32 NT]
    const int* flags;        // [B2][NT]
    long s_row;
    int B2, bias_pitch;
    float qscale;
};

// Geometry: eight waves, WB blocks of 32 channels (one head of 32, two of 16, four of 8) to a workgroup, 8 / WB waves to a block, each with every
// (8 / WB)-th tile of 32 tokens, at most TPW of them.  64 and 128 channels: all blocks.  256 channels: half of them, k and v of more
// would not fit; the output projection, which needs all heads, is a launch of its own (HEADS: `out` takes the gated outputs).
template <int C, int D, int TPW> struct AbGeo {
    static constexpr bool HEADS = C == 256;
    static constexpr int KS = C / 16;               // K steps of a projection
    static constexpr int NB = C / 32;               // 32-channel blocks
    static constexpr int WB = HEADS ? NB / 2 : NB;  // ... of a workgroup
    static constexpr int HPB = 32 / D;              // heads per block
    static constexpr int WPB = 8 / WB;              // waves per block
    static constexpr int NT_MAX = WPB * TPW;
    static constexpr int XP = C * 2 + 16;           // pitch of the normalised rows (bytes)
    static constexpr int HP = WB * 64 + 16;         // HEADS: pitch of the gated outputs
    static constexpr bool ONES = D < 32;            // row sums through the weighted sum's product (see attend)
    static constexpr bool GATE32 = C == 128;        // the gate stays in fp32 until it multiplies, as in ffk_gated_out_fused,
    static constexpr bool GATE_LDS = GATE32 && TPW == 4;       // that of a wave's fourth tile in LDS, behind k and v
    static constexpr size_t smem(long NT) {         // rows, then k and v (and a tile of ones or of the gate), then the gated outputs (and the updates)
        const size_t rows = (size_t)NT * 32 * XP, kv = (size_t)NT * WB * 4096 + (ONES ? 2048 : 0) + (GATE_LDS ? 32768 : 0),
                     end = HEADS ? 0 : rows + (size_t)NT * NB * 2048;
        return rows > kv ? (rows > end ? rows : end) : (kv > end ? kv : end);
    }
};

template <int C, int D, int TPW>
__global__ __launch_bounds__(512, 2) void attention_block_kernel(const AbArgs a) {
    typedef AbGeo<C, D, TPW> G;
    constexpr int KS = G::KS, NB = G::NB, WB = G::WB, HPB = G::HPB, WPB = G::WPB, XP = G::XP, PARTS = NB / WB;
    constexpr float NEG_FLOOR = -1.0e4f;             // reference of a row that has met no key (see ffk_attention.hip)
    extern __shared__ __align__(16) unsigned char ab_smem[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    const int NT = (a.n + 31) >> 5;
    // consecutive workgroup ids go to the eight XCDs in turn: each takes a contiguous eighth of the batch rows
    const unsigned per_xcd = (unsigned)(a.B2 * PARTS + 7) >> 3;
    const unsigned item = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (item >= (unsigned)a.B2 * PARTS) return;      // whole workgroup
    const unsigned b2 = item / PARTS;
    const int wb = wave % WB, t_first = wave / WB;   // block within the workgroup, first tile of this wave
    const int blk = (int)(item % PARTS) * WB + wb;   // block of hidden (at the end: output) channels
    unsigned char* s_x = ab_smem;                    // [32 NT][XP]
    T* s_k = reinterpret_cast<T*>(ab_smem);          // [WB][NT][2][64][8]
    T* s_v = s_k + (size_t)WB * NT * 1024;           // the same
    T* s_one = s_v + (size_t)WB * NT * 1024;         // ONES: a tile of ones
    T* s_o = s_k;                                    // [NT][NB][2][64][8]
    const T* xrow = a.x + (long)b2 * a.s_row;

    // key tiles with a masked key; trailing tiles without a valid one are left out
    const int fl = lane < NT ? a.flags[(long)b2 * NT + lane] : 2;
    const unsigned long long m_some = __builtin_amdgcn_ballot_w64(fl != 0), m_live = __builtin_amdgcn_ballot_w64(fl != 2);
    const int kt_end = m_live ? 64 - __builtin_clzll(m_live) : 1;
    const float* kb = a.keybias + (long)b2 * NT * 32 + 4 * half;

    bf16x8 ident[2];                                 // identity as B operand of the bias (see ffk_attention.hip)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 8; ++e) ident[i][e] = (T)(16 * half + 8 * i + e == l32 ? 1.0f : 0.0f);

    // weight fragments of block b of weight `which` (0 q, 1 k, 2 v, 3 gate, 4 output)
    auto wptr = [&](int which, int b) { return a.w + ((long)which * NB + b) * (KS * 512) + lane * 8; };
    // tile i of this wave; past the end the last tile again, whose products nobody uses
    auto tile = [&](int i) { return t_first + WPB * i < NT ? t_first + WPB * i : NT - 1; };
    // acc = W y^T (or y W^T) over this wave's tiles; fragments of `next` are requested on the way
    bf16x8 w[KS];
    auto request = [&](const T* p) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < KS; ++i) w[i] = MM::ld(p + i * 512);
    };
    auto project = [&](auto swap, const T* next, f32x16 (&acc)[TPW]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < TPW; ++i)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][v] = 0.0f;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const bf16x8 c = w[ks];
#pragma unroll
            for (int i = 0; i < TPW; ++i) {
                const bf16x8 x = *reinterpret_cast<const bf16x8*>(s_x + (tile(i) * 32 + l32) * XP + ks * 32 + half * 16);
                if (decltype(swap)::value) MM::mma(acc[i], x, c);
                else MM::mma(acc[i], c, x);
            }
            if (next) w[ks] = MM::ld(next + ks * 512);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // ---- one head of one query tile over all key tiles; o: its D normalised channels, in accumulator order.  bias: tiles 0 and 1
    // have been requested; those of the next call (bp_next) are requested in the last two steps ----
    bf16x8 bias[2][2];
    auto bias_load = [&](const T* p, bf16x8 (&b)[2]) __attribute__((always_inline)) {
        b[0] = MM::ld(p);
        b[1] = MM::ld(p + 8);
    };
    auto attend = [&](int sub, const T* bp, const T* bp_next, const bf16x8& q0, const bf16x8& q1, f32x16& acc, float& inv) __attribute__((always_inline)) {
        const T* kp = s_k + (size_t)wb * NT * 1024 + lane * 8;
        // D < 32: what v's tile holds of other heads is read as ones, so that the product's other rows are the row sums of the
        // probabilities, in every lane for all keys
        const bool own = !G::ONES || l32 / D == sub;
        const T* vp = (own ? s_v + (size_t)wb * NT * 1024 : s_one) + lane * 8;
        const int vstep = own ? 1024 : 0;
        constexpr int REGS = D / 2;                  // accumulator registers of a head
        const int lreg = sub == 0 ? REGS & 15 : 0;
        bf16x8 qs = q0;                              // D < 32: the fragment with the head's channels, the others' cleared
        if (sub * REGS >= 8) qs = q1;
        if (D == 8) {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if ((e >> 2) != (sub & 1)) qs[e] = (T)0.0f;
        }
        f32x16 negm, s;
        float l_run;
        auto bias_req = [&](int kt, bf16x8 (&b)[2]) __attribute__((always_inline)) {
            const int past = kt - kt_end < kt_end ? kt - kt_end : 0;
            bias_load(kt < kt_end ? bp + (long)kt * 1024 : bp_next + (long)past * 1024, b);
        };
        bf16x8 kf[2], vf[2], p[2];
        auto k_req = [&](int kt) __attribute__((always_inline)) {
            const T* q = kp + (kt < kt_end ? kt : kt_end - 1) * 1024;
            if (D == 32) {
                kf[0] = MM::ld(q);
                kf[1] = MM::ld(q + 512);
            } else {
                kf[0] = MM::ld(q + sub * REGS / 8 * 512);
            }
        };
        auto v_req = [&](int kt) __attribute__((always_inline)) {
            const T* q = vp + kt * vstep;
            vf[0] = MM::ld(q);
            vf[1] = MM::ld(q + 512);
        };
        auto score = [&](int kt, const bf16x8 (&b)[2]) __attribute__((always_inline)) {
            s = negm;
            if (D == 32) {
                MM::mma(s, kf[0], q0);
                MM::mma(s, kf[1], q1);
            } else {
                MM::mma(s, kf[0], qs);
            }
            MM::mma(s, b[0], ident[0]);
            MM::mma(s, b[1], ident[1]);
            if ((m_some >> kt) & 1) {
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const f32x4 mk = *reinterpret_cast<const f32x4*>(kb + kt * 32 + 8 * g);
#pragma unroll
                    for (int e = 0; e < 4; ++e) s[4 * g + e] += mk[e];
                }
            }
        };
        auto prob = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int t = 0; t < 8; ++t) p[i][t] = (T)fast_exp2(s[8 * i + t]);
        };
        auto row_sum = [&]() __attribute__((always_inline)) -> float {         // of this lane's keys
            typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
            const bf16x2 ones = {(T)1.0f, (T)1.0f};
            float sum = 0.0f;
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const bf16x2 pr = {p[i][2 * t], p[i][2 * t + 1]};
                    sum = __builtin_amdgcn_fdot2_f32_bf16(pr, ones, sum, false);
                }
            return sum;
        };
        auto weigh = [&]() __attribute__((always_inline)) {
            MM::mma(acc, vf[0], p[0]);
            MM::mma(acc, vf[1], p[1]);
        };
        // The reference is set by the first tile; a second walk moves it where a row sum shows that a later score lay far above it
        // (see ffk_attention.hip).
        for (int careful = 0; careful < 2; ++careful) {
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[v] = negm[v] = 0.0f;
            if (careful) {
                bias_req(0, bias[0]);
                bias_req(1, bias[1]);
            }
            k_req(0);
            score(0, bias[0]);
            bias_req(2, bias[0]);
            v_req(0);
            k_req(1);
            asm volatile("" ::: "memory");           // requested here, not at their first use
            float mt = fmaxf(s[0], s[1]);
#pragma unroll
            for (int v = 2; v < 16; ++v) mt = fmaxf(mt, s[v]);
            const float m0 = fmaxf(fmaxf(mt, lane_xor<32>(mt)), NEG_FLOOR);
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                s[v] -= m0;
                negm[v] = -m0;
            }
            prob();
            l_run = G::ONES ? 0.0f : row_sum();
            weigh();
            auto step = [&](int kt, bf16x8 (&b)[2]) __attribute__((always_inline)) {
                v_req(kt);
                score(kt, b);
                if (!careful) {
                    k_req(kt + 1);
                    bias_req(kt + 2, b);
                }
                asm volatile("" ::: "memory");
                prob();
                float sum = G::ONES ? 0.0f : row_sum();
                if (careful) {
                    if (G::ONES) sum = row_sum();
                    if (__builtin_amdgcn_ballot_w64(!(sum <= 1048576.0f)) != 0) {
                        const bool fresh = negm[0] == -NEG_FLOOR;
                        if (fresh) {
#pragma unroll
                            for (int v = 0; v < 16; ++v) negm[v] = 0.0f;
                        }
                        score(kt, b);
                        float mx = fmaxf(s[0], s[1]);
#pragma unroll
                        for (int v = 2; v < 16; ++v) mx = fmaxf(mx, s[v]);
                        const float delta = fmaxf(fmaxf(mx, lane_xor<32>(mx)), fresh ? NEG_FLOOR : 0.0f);
                        const float alpha = fast_exp2((fresh ? NEG_FLOOR : 0.0f) - delta);
#pragma unroll
                        for (int v = 0; v < 16; ++v) {
                            s[v] -= delta;
                            negm[v] -= delta;
                            acc[v] *= alpha;
                        }
                        l_run *= alpha;
                        prob();
                        sum = row_sum();
                    }
                    k_req(kt + 1);
                    bias_req(kt + 2, b);
                }
                if (!G::ONES) l_run += sum;
                weigh();
            };
            int kt = 1;
            for (; kt + 1 < kt_end; kt += 2) {
                step(kt, bias[1]);
                step(kt + 1, bias[0]);
            }
            if (kt < kt_end) step(kt, bias[1]);
            if (G::ONES) l_run = acc[lreg];
            // probabilities are not negative: a finite sum shows that none overflowed
            if (careful || __builtin_amdgcn_ballot_w64(!(l_run <= 1.8446744e19f)) == 0) break;
        }
        if (kt_end == 1) {                           // nothing of the next call has been requested in place
            bias_load(bp_next, bias[0]);
        } else if (kt_end & 1) {                     // the next call's tiles 0 and 1 lie in the other order
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const bf16x8 t = bias[0][i];
                bias[0][i] = bias[1][i];
                bias[1][i] = t;
            }
        }
        const float l_tot = G::ONES ? l_run : l_run + lane_xor<32>(l_run);
        inv = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;              // all keys masked: zero
    };

    bf16x8 of[TPW][2];                       // gate (but for GATE32), then gated outputs
    f32x16 gate[G::GATE32 ? TPW : 1];
    f32x4* const s_gate = reinterpret_cast<f32x4*>(ab_smem + (size_t)NT * WB * 4096) + tid;        // [4][512], each lane its own
    request(wptr(1, blk));
    rb_normalise<C, G::NT_MAX>(a, xrow, s_x, NT, wave, lane);
    lds_barrier();
    // ---- projections of this wave's tiles ----
    bf16x8 qf[TPW][2];
    {
        bf16x8 kf[TPW][2], vf[TPW][2];
        f32x16 acc[TPW];
        project(std::false_type(), wptr(2, blk), acc);
#pragma unroll
        for (int i = 0; i < TPW; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                kf[i][j] = rb_pack8(acc[i], 8 * j, 1.0f);
                rb_pin(kf[i][j]);
            }
        project(std::true_type(), wptr(0, blk), acc);
#pragma unroll
        for (int i = 0; i < TPW; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                vf[i][j] = rb_pack8(acc[i], 8 * j, 1.0f);
                rb_pin(vf[i][j]);
            }
        project(std::false_type(), wptr(3, blk), acc);
#pragma unroll
        for (int i = 0; i < TPW; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                qf[i][j] = rb_pack8(acc[i], 8 * j, a.qscale);
                rb_pin(qf[i][j]);
            }
        bf16x4 bg[4];
#pragma unroll
        for (int g = 0; g < 4; ++g)
            bg[g] = __builtin_bit_cast(bf16x4, *reinterpret_cast<const u32x2*>(a.bg + blk * 32 + 4 * half + 8 * g));
        project(std::false_type(), (const T*)nullptr, acc);
#pragma unroll
        for (int i = 0; i < TPW; ++i) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float y = sigmoid_f(acc[i][8 * j + e] + (float)bg[2 * j + (e >> 2)][e & 3]);
                    if (G::GATE32) gate[i][8 * j + e] = y;
                    else of[i][j][e] = (T)y;
                }
                if (!G::GATE32) rb_pin(of[i][j]);
            }
            if constexpr (G::GATE32) asm volatile("" : "+v"(gate[i]));        // one tile after the other
            if constexpr (G::GATE_LDS)
                if (i == 3) {
#pragma unroll
                    for (int v = 0; v < 4; ++v) s_gate[v * 512] = f32x4{gate[i][4 * v], gate[i][4 * v + 1], gate[i][4 * v + 2], gate[i][4 * v + 3]};
                }
        }
        lds_barrier();                           // nobody reads the rows any more
        if (G::ONES && tid < 128) *reinterpret_cast<u32x4*>(s_one + tid * 8) = u32x4{0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};
#pragma unroll
        for (int i = 0; i < TPW; ++i) {
            if (t_first + WPB * i < NT) {
                T* d = s_k + ((size_t)wb * NT + t_first + WPB * i) * 1024 + lane * 8;
                T* e = s_v + ((size_t)wb * NT + t_first + WPB * i) * 1024 + lane * 8;
                *reinterpret_cast<bf16x8*>(d) = kf[i][0];
                *reinterpret_cast<bf16x8*>(d + 512) = kf[i][1];
                *reinterpret_cast<bf16x8*>(e) = vf[i][0];
                *reinterpret_cast<bf16x8*>(e + 512) = vf[i][1];
            }
        }
    }
    auto bias_row = [&](int i, int sub) {        // bias tiles of a call: tile i, head sub of the block
        return a.bias_t + ((long)(blk * HPB + sub) * NT + tile(i)) * a.bias_pitch * 1024 + lane * 16;
    };
    bias_load(bias_row(0, 0), bias[0]);
    bias_load(bias_row(0, 0) + (kt_end > 1 ? 1024 : 0), bias[1]);
    lds_barrier();
    // ---- attention ----
#pragma unroll
    for (int i = 0; i < TPW; ++i) {
        if (t_first + WPB * i < NT) {
#pragma unroll
            for (int sub = 0; sub < HPB; ++sub) {
                f32x16 acc;
                float inv;
                const T* next = sub + 1 < HPB ? bias_row(i, sub + 1) : bias_row(i + 1 < TPW ? i + 1 : i, 0);
                attend(sub, bias_row(i, sub), next, qf[i][0], qf[i][1], acc, inv);
                if constexpr (G::GATE_LDS)
                    if (i == 3) {
#pragma unroll
                        for (int v = 0; v < 4; ++v) {
                            const f32x4 y = s_gate[v * 512];
#pragma unroll
                            for (int e = 0; e < 4; ++e) gate[i][4 * v + e] = y[e];
                        }
                    }
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    if (8 * j + 7 < sub * (D / 2) || 8 * j >= (sub + 1) * (D / 2)) continue;
#pragma unroll
                    for (int e = 0; e < 8; ++e)      // the head's registers
                        if ((8 * j + e) / (D / 2) == sub) of[i][j][e] = (T)(acc[8 * j + e] * inv * (G::GATE32 ? gate[i][8 * j + e] : (float)of[i][j][e]));
                    rb_pin(of[i][j]);
                }
            }
        }
    }
    lds_barrier();                               // nobody reads k and v any more

    if constexpr (G::HEADS) {                        // gated outputs -> LDS -> their rows, WB * 64 bytes at a time
        constexpr int LPR = WB * 4, RPI = 64 / LPR;
#pragma unroll
        for (int i = 0; i < TPW; ++i) {
            if (t_first + WPB * i < NT) {
                unsigned char* p = ab_smem + ((t_first + WPB * i) * 32 + l32) * G::HP + wb * 64 + half * 8;
#pragma unroll
                for (int j = 0; j < 4; ++j) {        // channels 8 j + 4 half ..
                    const u32x4 y = *reinterpret_cast<const u32x4*>(&of[i][j >> 1]);
                    *reinterpret_cast<u32x2*>(p + j * 16) = u32x2{y[2 * (j & 1)], y[2 * (j & 1) + 1]};
                }
            }
        }
        lds_barrier();
        T* orow = a.out + (long)b2 * a.n * C + (item % PARTS) * (WB * 32) + (lane % LPR) * 8;
        for (int tok = wave * RPI + lane / LPR; tok < a.n; tok += 8 * RPI)
            st16(orow + (long)tok * C, *reinterpret_cast<const Vec16<T>*>(ab_smem + tok * G::HP + (lane % LPR) * 16));
        return;
    }

    // ---- gated outputs to LDS; output projection: 32 channels of the wave's tiles ----
    request(wptr(4, blk));
#pragma unroll
    for (int i = 0; i < TPW; ++i) {
        if (t_first + WPB * i < NT) {
            T* d = s_o + ((size_t)(t_first + WPB * i) * NB + blk) * 1024 + lane * 8;
            *reinterpret_cast<bf16x8*>(d) = of[i][0];
            *reinterpret_cast<bf16x8*>(d + 512) = of[i][1];
        }
    }
    unsigned char* s_u = ab_smem + (size_t)NT * NB * 2048;         // [32 NT][XP]
    RbUpdate<C, G::NT_MAX> rows;
    rows.fetch(a, (long)b2 * a.s_row, NT, wave, rb_lane(lane));
    lds_barrier();
    const T* bo = a.bo ? a.bo + blk * 32 + 16 * half : nullptr;
    f32x16 acc[TPW];
#pragma unroll
    for (int i = 0; i < TPW; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][v] = 0.0f;
#pragma unroll
    for (int f = 0; f < KS; ++f)
#pragma unroll
        for (int i = 0; i < TPW; ++i) MM::mma(acc[i], w[f], MM::ld(s_o + ((size_t)tile(i) * KS + f) * 512 + lane * 8));
#pragma unroll
    for (int i = 0; i < TPW; ++i)                    // past the end: the last tile's update once more
        rb_put(s_u + (tile(i) * 32 + l32) * XP + blk * 64 + half * 32, acc[i], bo);
    lds_barrier();
    rows.store(a, s_u, (long)b2 * a.s_row, NT, wave, rb_lane(lane));
}

// 256 channels in eight heads, rows of at most 128 tokens: a wave owns a head, its q, k, v and gate of all NT token tiles stay in its
// registers, and no weight is read by two waves.  The normalised rows lie in LDS (row-major, 16 bytes of padding), the gated outputs
// of the heads beside them, in the order of the output projection's fragments; there a wave owns 32 output channels of all tokens.
constexpr int AW_C = 256, AW_KS = 16, AW_XP = AW_C * 2 + 16;
template <int NT> constexpr size_t aw_smem() { return (size_t)NT * 32 * AW_XP + (size_t)NT * 8 * 2048; }

template <int NT, bool BIAS>
__global__ __launch_bounds__(512, 2) void attention_block_wide_kernel(const AbArgs a) {
    constexpr int C = AW_C, KS = AW_KS, XP = AW_XP;
    constexpr int AHEAD = 4;                         // weight fragments requested ahead, of each of two weights
    extern __shared__ __align__(16) unsigned char ab_smem[];
    unsigned char* s_x = ab_smem;                    // [32 NT][XP]
    T* s_o = reinterpret_cast<T*>(ab_smem + NT * 32 * XP);   // [NT][8 heads][2][64][8]

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    const unsigned per_xcd = (unsigned)(a.B2 + 7) >> 3;      // see attention_block_kernel
    const unsigned b2 = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (b2 >= (unsigned)a.B2) return;
    const T* xrow = a.x + (long)b2 * a.s_row;
    const T* wbase = a.w + (long)wave * KS * 512 + lane * 8;         // this head's block (output: this wave's channels)
    auto wptr = [&](int which) { return wbase + (long)which * 8 * KS * 512; };
    bf16x8 f0[AHEAD], f1[AHEAD];
    auto request = [&](const T* w0, const T* w1) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
            f0[i] = MM::ld(w0 + i * 512);
            f1[i] = MM::ld(w1 + i * 512);
        }
    };
    request(wptr(0), wptr(1));
    rb_normalise<C, NT>(a, xrow, s_x, NT, wave, lane);
    const unsigned char* xp = s_x + l32 * XP + half * 16;

    // two weights at a time over all tokens, their first fragments requested: acc[0] = W0 y^T, acc[1] = W1 y^T or (V1) y W1^T
    auto project2 = [&](const T* w0, const T* w1, auto v1, f32x16 (&acc)[2][NT]) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[0][t][v] = acc[1][t][v] = 0.0f;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const bf16x8 c0 = f0[ks % AHEAD], c1 = f1[ks % AHEAD];
            if (ks + AHEAD < KS) {
                f0[ks % AHEAD] = MM::ld(w0 + (ks + AHEAD) * 512);
                f1[ks % AHEAD] = MM::ld(w1 + (ks + AHEAD) * 512);
            }
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const bf16x8 x = *reinterpret_cast<const bf16x8*>(xp + t * 32 * XP + ks * 32);
                MM::mma(acc[0][t], c0, x);
                if (decltype(v1)::value) MM::mma(acc[1][t], x, c1);
                else MM::mma(acc[1][t], c1, x);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    bf16x8 qf[NT][2], kf[NT][2], vf[NT][2], gf[NT][2];
    lds_barrier();
    {
        f32x16 acc[2][NT];
        project2(wptr(0), wptr(1), std::false_type(), acc);
        request(wptr(3), wptr(2));
#pragma unroll
        for (int t = 0; t < NT; ++t) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                qf[t][i] = rb_pack8(acc[0][t], 8 * i, a.qscale);
                kf[t][i] = rb_pack8(acc[1][t], 8 * i, 1.0f);
                rb_pin(qf[t][i]);
                rb_pin(kf[t][i]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        project2(wptr(3), wptr(2), std::true_type(), acc);
        bf16x4 bg[4];
#pragma unroll
        for (int g = 0; g < 4; ++g)
            bg[g] = __builtin_bit_cast(bf16x4, *reinterpret_cast<const u32x2*>(a.bg + wave * 32 + 4 * half + 8 * g));
#pragma unroll
        for (int t = 0; t < NT; ++t) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                vf[t][i] = rb_pack8(acc[1][t], 8 * i, 1.0f);
#pragma unroll
                for (int e = 0; e < 8; ++e) gf[t][i][e] = (T)sigmoid_f(acc[0][t][8 * i + e] + (float)bg[2 * i + (e >> 2)][e & 3]);
                rb_pin(vf[t][i]);
                rb_pin(gf[t][i]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    // ---- the head's attention: the scores of a query tile with all keys fit the registers ----
    const int fl = lane < NT ? a.flags[(long)b2 * NT + lane] : 0;
    const unsigned some = (unsigned)__builtin_amdgcn_ballot_w64(fl != 0);
    const float* kb = a.keybias + (long)b2 * NT * 32 + 4 * half;
    bf16x8 ident[2];
    if (BIAS) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int e = 0; e < 8; ++e) ident[i][e] = (T)(16 * half + 8 * i + e == l32 ? 1.0f : 0.0f);
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        f32x16 s[NT];
        float m = -1.0e4f;                           // a row without a key: every probability zero
        bf16x8 bias[NT][2];
        if (BIAS) {
            const T* bp = a.bias_t + ((long)wave * NT + t) * a.bias_pitch * 1024 + lane * 16;
#pragma unroll
            for (int kt = 0; kt < NT; ++kt) {
                bias[kt][0] = MM::ld(bp + kt * 1024);
                bias[kt][1] = MM::ld(bp + kt * 1024 + 8);
            }
        }
#pragma unroll
        for (int kt = 0; kt < NT; ++kt) {
#pragma unroll
            for (int v = 0; v < 16; ++v) s[kt][v] = 0.0f;
            MM::mma(s[kt], kf[kt][0], qf[t][0]);
            MM::mma(s[kt], kf[kt][1], qf[t][1]);
            if (BIAS) {
                MM::mma(s[kt], bias[kt][0], ident[0]);
                MM::mma(s[kt], bias[kt][1], ident[1]);
            }
        }
        if (some) {                                  // some key of the row is masked or padding
#pragma unroll
            for (int kt = 0; kt < NT; ++kt)
                if ((some >> kt) & 1) {
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const f32x4 mk = *reinterpret_cast<const f32x4*>(kb + kt * 32 + 8 * g);
#pragma unroll
                        for (int e = 0; e < 4; ++e) s[kt][4 * g + e] += mk[e];
                    }
                }
        }
#pragma unroll
        for (int kt = 0; kt < NT; ++kt)
#pragma unroll
            for (int v = 0; v < 16; ++v) m = fmaxf(m, s[kt][v]);
        m = fmaxf(m, lane_xor<32>(m));
        float l = 0.0f;
        f32x16 o;
#pragma unroll
        for (int v = 0; v < 16; ++v) o[v] = 0.0f;
#pragma unroll
        for (int kt = 0; kt < NT; ++kt) {
            typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
            const bf16x2 ones = {(T)1.0f, (T)1.0f};
            bf16x8 p[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
#pragma unroll
                for (int e = 0; e < 8; ++e) p[i][e] = (T)fast_exp2(s[kt][8 * i + e] - m);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const bf16x2 pr = {p[i][2 * e], p[i][2 * e + 1]};
                    l = __builtin_amdgcn_fdot2_f32_bf16(pr, ones, l, false);
                }
                MM::mma(o, vf[kt][i], p[i]);
            }
        }
        l += lane_xor<32>(l);
        const float inv = l > 0.0f ? 1.0f / l : 0.0f;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            bf16x8 y;
#pragma unroll
            for (int e = 0; e < 8; ++e) y[e] = (T)(o[8 * i + e] * inv * (float)gf[t][i][e]);
            *reinterpret_cast<bf16x8*>(s_o + ((t * 8 + wave) * 2 + i) * 512 + lane * 8) = y;
        }
        __builtin_amdgcn_sched_barrier(0);
    }

    // ---- output projection: 32 channels of all tokens ----
    const T* wo = wptr(4);
    bf16x8 w[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) w[i] = MM::ld(wo + i * 512);
    RbUpdate<C, NT> rows;
    rows.fetch(a, (long)b2 * a.s_row, NT, wave, rb_lane(lane));
    lds_barrier();
    f32x16 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[t][v] = 0.0f;
#pragma unroll
    for (int f = 0; f < KS; ++f) {
        const bf16x8 c = w[f % 8];
        if (f + 8 < KS) w[f % 8] = MM::ld(wo + (f + 8) * 512);
#pragma unroll
        for (int t = 0; t < NT; ++t) MM::mma(acc[t], c, MM::ld(s_o + (t * KS + f) * 512 + lane * 8));
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int t = 0; t < NT; ++t)                     // the normalised rows are not read any more
        rb_put(s_x + (t * 32 + l32) * XP + wave * 64 + half * 32, acc[t], a.bo ? a.bo + wave * 32 + 16 * half : nullptr);
    lds_barrier();
    rows.store(a, s_x, (long)b2 * a.s_row, NT, wave, rb_lane(lane));
}

template <int C, int D, int TPW> int ab_launch(const AbArgs& a, long NT, hipStream_t st) {
    typedef AbGeo<C, D, TPW> G;
    static FfkLdsReservation lds_reserved;
    const int rc = ffk_reserve_lds(lds_reserved, (const void*)attention_block_kernel<C, D, TPW>, G::smem(G::NT_MAX), "ffk_attention_block");
    if (rc != FFK_OK) return rc;
    attention_block_kernel<C, D, TPW><<<dim3(8u * ffk_cdiv((long)a.B2 * (G::NB / G::WB), 8)), 512, G::smem(NT), st>>>(a);
    return ffk_check_launch("ffk_attention_block");
}
template <int NT, bool BIAS> int aw_launch(const AbArgs& a, hipStream_t st) {
    static FfkLdsReservation lds_reserved;
    const int rc = ffk_reserve_lds(lds_reserved, (const void*)attention_block_wide_kernel<NT, BIAS>, aw_smem<NT>(), "ffk_attention_block");
    if (rc != FFK_OK) return rc;
    attention_block_wide_kernel<NT, BIAS><<<dim3(8u * ffk_cdiv(a.B2, 8)), 512, aw_smem<NT>(), st>>>(a);
    return ffk_check_launch("ffk_attention_block");
}
template <bool BIAS> int aw_launch_nt(const AbArgs& a, long NT, hipStream_t st) {
    switch (NT) {
        case 1: return aw_launch<1, BIAS>(a, st);
        case 2: return aw_launch<2, BIAS>(a, st);
        case 3: return aw_launch<3, BIAS>(a, st);
        default: return aw_launch<4, BIAS>(a, st);
    }
}

}  // namespace

extern "C" int ffk_attention_block(void* out, const void* x, void* xtail, const void* gamma, const void* beta, const void* w,
                                   const void* bg, const void* bo, const void* bias_t, const float* keybias,
                                   const int32_t* tileflags, const void* drop, int64_t B2, int64_t N, int64_t C, int64_t D,
                                   int64_t s_row, int64_t s_tok, int64_t bias_pitch, float eps, int dtype, void* stream) {
    FFK_REQUIRE(out && x && gamma && beta && w && bg && keybias && tileflags, FFK_ERR_NULL, "ffk_attention_block: null pointer");
    FFK_REQUIRE(dtype == FFK_BF16, FFK_ERR_DTYPE, "ffk_attention_block: bf16 only (dtype tag %d)", dtype);
    FFK_REQUIRE((C == 128 && D == 32) || (C == 64 && (D == 16 || D == 8)) || (C == 256 && D == 32), FFK_ERR_UNSUPPORTED,
                "ffk_attention_block: built for 128 or 256 channels in heads of 32 and 64 in heads of 16 or 8, got %ld / %ld", (long)C, (long)D);
    FFK_REQUIRE(C == 256 || bias_t, FFK_ERR_UNSUPPORTED, "ffk_attention_block: built with a pair bias for 64 and 128 channels");
    FFK_REQUIRE(B2 > 0 && B2 < (1L << 31) - 64 && N > 0, FFK_ERR_SHAPE, "ffk_attention_block: bad shape B2=%ld N=%ld", (long)B2, (long)N);
    FFK_REQUIRE(s_row % 16 == 0 && s_tok % 16 == 0, FFK_ERR_ALIGN, "ffk_attention_block: row strides must be multiples of 16 elements");
    FFK_REQUIRE(ffk_aligned16(out) && ffk_aligned16(x) && ffk_aligned16(xtail) && ffk_aligned16(gamma) && ffk_aligned16(beta) &&
                    ffk_aligned16(w) && ffk_aligned16(bg) && ffk_aligned16(bo) && ffk_aligned16(bias_t) && ffk_aligned16(keybias) &&
                    ffk_aligned16(drop),
                FFK_ERR_ALIGN, "ffk_attention_block: buffers must be 16-byte aligned");
    const long NT = (N + 31) / 32;
    FFK_REQUIRE(NT <= (C == 256 ? 4 : C == 128 ? 8 : D == 16 ? 16 : 12), FFK_ERR_UNSUPPORTED,
                "ffk_attention_block: rows of %ld tokens are too long for %ld channels", (long)N, (long)C);
    FFK_REQUIRE(!bias_t || bias_pitch >= NT, FFK_ERR_SHAPE, "ffk_attention_block: bias rows of %ld tiles, %ld needed", (long)bias_pitch, NT);
    const AbArgs a = {{(T*)out, (const T*)x, (int8_t*)xtail, (const T*)gamma, (const T*)beta, (const T*)drop, (long)s_tok, (int)N, eps},
                      (const T*)w, (const T*)bg, (const T*)bo, (const T*)bias_t, keybias, (const int*)tileflags, (long)s_row, (int)B2,
                      (int)bias_pitch, 1.4426950408889634f / sqrtf((float)D)};
    hipStream_t st = (hipStream_t)stream;
    if (C == 256) return bias_t ? aw_launch_nt<true>(a, NT, st) : aw_launch_nt<false>(a, NT, st);
    if (C == 64 && D == 8) {
        switch ((NT + 3) / 4) {
            case 1: return ab_launch<64, 8, 1>(a, NT, st);
            case 2: return ab_launch<64, 8, 2>(a, NT, st);
            default: return ab_launch<64, 8, 3>(a, NT, st);
        }
    }
    if (C == 64) {
        switch ((NT + 3) / 4) {
            case 1: return ab_launch<64, 16, 1>(a, NT, st);
            case 2: return ab_launch<64, 16, 2>(a, NT, st);
            case 3: return ab_launch<64, 16, 3>(a, NT, st);
            default: return ab_launch<64, 16, 4>(a, NT, st);
        }
    }
    switch ((NT + 1) / 2) {
        case 1: return ab_launch<128, 32, 1>(a, NT, st);
        case 2: return ab_launch<128, 32, 2>(a, NT, st);
        case 3: return ab_launch<128, 32, 3>(a, NT, st);
        default: return ab_launch<128, 32, 4>(a, NT, st);
    }
}

extern "C" int ffk_attention_heads(void* o, const void* x, const void* gamma, const void* beta, const void* w, const void* bg,
                                   const void* bias_t, const float* keybias, const int32_t* tileflags, int64_t B2, int64_t N,
                                   int64_t C, int64_t D, int64_t s_row, int64_t s_tok, int64_t bias_pitch, float eps, int dtype,
                                   void* stream) {
    FFK_REQUIRE(o && x && gamma && beta && w && bg && bias_t && keybias && tileflags, FFK_ERR_NULL, "ffk_attention_heads: null pointer");
    FFK_REQUIRE(dtype == FFK_BF16, FFK_ERR_DTYPE, "ffk_attention_heads: bf16 only (dtype tag %d)", dtype);
    FFK_REQUIRE(C == 256 && D == 32, FFK_ERR_UNSUPPORTED, "ffk_attention_heads: built for 256 channels in heads of 32, got %ld / %ld", (long)C, (long)D);
    FFK_REQUIRE(B2 > 0 && B2 < (1L << 30) - 64 && N > 0, FFK_ERR_SHAPE, "ffk_attention_heads: bad shape B2=%ld N=%ld", (long)B2, (long)N);
    FFK_REQUIRE(N <= 256, FFK_ERR_UNSUPPORTED, "ffk_attention_heads: rows of %ld tokens are too long", (long)N);
    FFK_REQUIRE(s_row % 8 == 0 && s_tok % 8 == 0, FFK_ERR_ALIGN, "ffk_attention_heads: row strides must be multiples of 8 elements");
    FFK_REQUIRE(ffk_aligned16(o) && ffk_aligned16(x) && ffk_aligned16(gamma) && ffk_aligned16(beta) && ffk_aligned16(w) &&
                    ffk_aligned16(bg) && ffk_aligned16(bias_t) && ffk_aligned16(keybias),
                FFK_ERR_ALIGN, "ffk_attention_heads: buffers must be 16-byte aligned");
    const long NT = (N + 31) / 32;
    FFK_REQUIRE(bias_pitch >= NT, FFK_ERR_SHAPE, "ffk_attention_heads: bias rows of %ld tiles, %ld needed", (long)bias_pitch, NT);
    const AbArgs a = {{(T*)o, (const T*)x, nullptr, (const T*)gamma, (const T*)beta, nullptr, (long)s_tok, (int)N, eps},
                      (const T*)w, (const T*)bg, nullptr, (const T*)bias_t, keybias, (const int*)tileflags, (long)s_row, (int)B2,
                      (int)bias_pitch, 1.4426950408889634f / sqrtf((float)D)};
    hipStream_t st = (hipStream_t)stream;
    switch ((NT + 1) / 2) {
        case 1: return ab_launch<256, 32, 1>(a, NT, st);
        case 2: return ab_launch<256, 32, 2>(a, NT, st);
        case 3: return ab_launch<256, 32, 3>(a, NT, st);
        default: return ab_launch<256, 32, 4>(a, NT, st);
    }
}
