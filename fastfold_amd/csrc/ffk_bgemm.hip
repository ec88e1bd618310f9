// Batched NT GEMM with a K loop (see ffk_bgemm_nt in include/ffk.h).
//
// A workgroup's 4 wavefronts compute one output tile.  K-chunks of A and B stream through a double-buffered LDS ring with
// register prefetch.  As in the fused linear kernel the MFMA computes C^T (rows of B are the M-operand) so that a lane holds
// 4 consecutive n of one row m, and the tile is staged through LDS for 16-byte stores.  Three tiles (see launch_tile):
//   128 x 128, chunks of 128 bytes, 64 x 64 per wave       (four 32 x 32 products per two fragments of each operand)
//    64 x  64, chunks of 256 bytes, 32 x 32 per wave
//    32 x  32, chunks of 4 x 128 bytes, each wave takes one piece of K in four (fp32, K >= 512)
// fp32 products are six bf16 products of the operands' parts (split4), which are cut on the way to LDS, one slot of it.  Against the
// fp32 instructions, us: 128 products of 256 x 256 x 256 48 -> 35, of 384 x 384 x 384 169 -> 108; 65 536 x 128, K = 1 024 149 -> 110,
// K = 512 80 -> 56; 32 768 x 256, K = 1 024 147 -> 97; 8 192 x 8 192, K = 128 193 -> 141; 4 096 x 128, K = 1 024, where the launch waits for one
// chunk after the other and cutting lengthens that chain, 17.7 -> 19.1.
// Every tile gives the same bits (callers cut their rows into pieces as memory allows, and pieces take other tiles): products are
// added in ascending order of K, for fp32 and K >= 512 within pieces of K (quarters up to K = 1 024, then 256), the pieces as
// ((p0 + p1) + p2) + p3 ..  The bf16 instructions cut off what the sum has no room for, towards minus infinity: in long chains, of
// numbers of one sign above all, that would add up to more than the roundings (K = 8 192 in four pieces 3.3e-6 of the sum), so a
// piece ends after 256 and every other one has its sign turned.
#include "ffk_common.h"
#include <algorithm>
#include <type_traits>

namespace {

constexpr int THREADS = 256;
constexpr int BG_PIECES = 512;                   // K from which fp32 products are added in pieces of K

template <typename T, typename OT, int BT>
__global__ __launch_bounds__(THREADS, 2) void bgemm_nt_kernel(const ffk_bgemm_desc d) {
    typedef Mma<T> MM;
    constexpr int VEC = DT<T>::VEC;
    constexpr int ES = sizeof(T);
    constexpr int OES = sizeof(OT);
    constexpr int OVEC = 16 / OES;
    constexpr bool XS_OK = std::is_same<OT, bf16_t>::value;     // outputs that may carry a residual tail
    constexpr int WT = BT == 128 ? 2 : 1;          // 32 x 32 blocks per wave and dimension
    constexpr bool KSPLIT = BT == 32;
    constexpr bool PIECES = std::is_same<T, float>::value;    // sums in pieces of K possible
    constexpr int BKB = 128 * 128 / BT;            // bytes of K per row and chunk
    constexpr int BK = BKB / ES;
    // fp32: operands lie in LDS as their three bf16 parts (see split4), [K step of 16][part][16] per row, one slot of each
    constexpr bool SPLIT = std::is_same<T, float>::value;
    constexpr int NSLOT = SPLIT ? 1 : 2;
    constexpr int P = (SPLIT ? BKB / 2 * 3 : BKB) + 16;        // row pitch of a slot (bytes)
    constexpr int SLOT = BT * P;
    constexpr int CP = BT * OES + 16;              // staged C pitch [m][n]
    constexpr int NV = BT * (BK / VEC) / THREADS;  // 16-byte vectors per thread per operand chunk (= 4)

    extern __shared__ __align__(16) unsigned char smem[];
    unsigned char* sA = smem;                      // NSLOT slots
    unsigned char* sB = smem + NSLOT * SLOT;       // NSLOT slots
    unsigned char* sC = smem;                      // aliases the ring after the K loop

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = KSPLIT ? 0 : wave >> 1, wn = KSPLIT ? 0 : wave & 1;
    const int l32 = lane & 31, half = lane >> 5;
    const int M = d.M, N = d.N, K = d.K;
    // Workgroup -> tile.  Consecutive workgroup ids go to the eight XCDs in turn, each with its own L2.
    // With at least eight batches every XCD takes a contiguous eighth of the (batch, n-tile, m-tile)
    // order, so that all tiles of one batch matrix pair run behind one L2 and A / B are fetched from
    // HBM once instead of once per XCD.  With fewer batches the plain order is kept: tiles that run
    // together then share their operand panels across the XCDs' row / column residues.
    const unsigned tiles_m = (M + BT - 1) / BT, tiles_n = (N + BT - 1) / BT;
    unsigned item = blockIdx.x;
    if (d.batch >= 8) {
        const unsigned total = tiles_m * tiles_n * (unsigned)d.batch, per_xcd = (total + 7) >> 3;
        item = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
        if (item >= total) return;
    }
    const long m0 = (long)(item % tiles_m) * BT, n0 = (long)((item / tiles_m) % tiles_n) * BT;
    const int bz = (item / tiles_m) / tiles_n;
    const T* A = (const T*)d.a + (long)bz * d.a_bs;
    const T* B = (const T*)d.b + (long)bz * d.b_bs;

    const int kq = PIECES && K >= BG_PIECES ? (K > 1024 ? 256 : (K + 255) / 256 * 64) : K;     // length of a piece (whole chunks)
    auto round_of = [&](int kc) { return K > 1024 ? kc >> 3 : 0; };
    auto k_of = [&](int kc, int c) {               // K index of vector c of a chunk row
        if (!KSPLIT) return kc * BK + c * VEC;
        const int round = round_of(kc);            // four pieces at a time
        return (4 * round + c / (BK / VEC / 4)) * kq + (kc - 8 * round) * (BK / 4) + c % (BK / VEC / 4) * VEC;
    };
    int piece = 0;                               // finished pieces
    Vec16<T> ra[NV], rb[NV];
    auto fetch = [&](int kc) {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int v = tid + THREADS * i;
            const int r = v / (BK / VEC), c = v % (BK / VEC);
            const int k = k_of(kc, c);
            long ma = m0 + r;
            if (ma >= M) ma = M - 1;
            long nb = n0 + r;
            if (nb >= N) nb = N - 1;
            // branch-free: clamp the K offset to the last full vector; the K tail is zeroed when the
            // registers are committed to LDS (touching them here would serialise the loads)
            const int kk = k < K ? k : K - VEC;
            ra[i] = ld16(A + ma * d.lda + kk);
            rb[i] = ld16(B + nb * d.ldb + kk);
        }
    };
    auto commit = [&](int slot, int kc) {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int v = tid + THREADS * i;
            const int r = v / (BK / VEC), c = v % (BK / VEC);
            const bool tail = k_of(kc, c) >= K;
            Vec16<T> xa = ra[i], xb = rb[i];
            if (tail) {
#pragma unroll
                for (int e = 0; e < VEC; ++e) xa.e[e] = xb.e[e] = DT<T>::from_f(0.0f);
            }
            if constexpr (SPLIT) {
                const int o = r * P + (c >> 2) * 96 + (c & 3) * 8;
                const uint32_t sign = K >= BG_PIECES ? (uint32_t)(KSPLIT ? c / (BK / VEC / 4) : piece) << 31 : 0u;
                u32x4& bits = *reinterpret_cast<u32x4*>(&xa);
#pragma unroll
                for (int e = 0; e < 4; ++e) bits[e] ^= sign;
                const Split4 a3 = split4(*reinterpret_cast<const f32x4*>(&xa)), b3 = split4(*reinterpret_cast<const f32x4*>(&xb));
#pragma unroll
                for (int p = 0; p < 3; ++p) {
                    *reinterpret_cast<u32x2*>(sA + o + p * 32) = a3.p[p];
                    *reinterpret_cast<u32x2*>(sB + o + p * 32) = b3.p[p];
                }
            } else {
                *reinterpret_cast<Vec16<T>*>(sA + slot * SLOT + r * P + c * 16) = xa;
                *reinterpret_cast<Vec16<T>*>(sB + slot * SLOT + r * P + c * 16) = xb;
            }
        }
    };

    f32x16 acc[WT][WT];   // [ni][mi]
#pragma unroll
    for (int a = 0; a < WT; ++a)
#pragma unroll
        for (int b = 0; b < WT; ++b)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[a][b][v] = 0.0f;

    f32x16 sum[PIECES ? WT : 1][PIECES ? WT : 1];       // of the finished pieces
    auto end_piece = [&]() {
#pragma unroll
        for (int a = 0; a < WT; ++a)
#pragma unroll
            for (int b = 0; b < WT; ++b)
#pragma unroll
                for (int v = 0; v < 16; ++v) sum[a][b][v] = piece == 0 ? acc[a][b][v] : piece & 1 ? sum[a][b][v] - acc[a][b][v] : sum[a][b][v] + acc[a][b][v];
        ++piece;
    };
    // KSPLIT: wave 0 adds the four pieces
    [[maybe_unused]] auto end_round = [&]() {
        float* red = reinterpret_cast<float*>(smem);
        if (wave) {
#pragma unroll
            for (int v = 0; v < 16; ++v) red[((wave - 1) * 16 + v) * 64 + lane] = acc[0][0][v];
        }
        lds_barrier();
        if (wave == 0) {
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const float p0 = piece ? sum[0][0][v] + acc[0][0][v] : acc[0][0][v];
                sum[0][0][v] = ((p0 - red[v * 64 + lane]) + red[(16 + v) * 64 + lane]) - red[(32 + v) * 64 + lane];
            }
        }
        lds_barrier();
        piece = 1;
    };
    const int kchunks = KSPLIT ? (K + 4 * kq - 1) / (4 * kq) * (kq / (BK / 4)) : (K + BK - 1) / BK;
    fetch(0);
    for (int kc = 0; kc < kchunks; ++kc) {
        if constexpr (PIECES && !KSPLIT) {
            if (kc * BK == (piece + 1) * kq) {
                end_piece();
#pragma unroll
                for (int a = 0; a < WT; ++a)
#pragma unroll
                    for (int b = 0; b < WT; ++b)
#pragma unroll
                        for (int v = 0; v < 16; ++v) acc[a][b][v] = 0.0f;
            }
        }
        const int slot = kc & (NSLOT - 1);
        if (SPLIT && kc) lds_barrier();            // nobody reads the chunk before any more
        if constexpr (KSPLIT) {
            if (kc && kc == 8 * round_of(kc)) {
                end_round();
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[0][0][v] = 0.0f;
            }
        }
        commit(slot, kc);
        lds_barrier();
        if (kc + 1 < kchunks) fetch(kc + 1);
        if constexpr (SPLIT) {
            constexpr int STEPS = BK / 16 / (KSPLIT ? 4 : 1);
            const unsigned char* pa = sA + (wm * WT * 32 + l32) * P + (KSPLIT ? wave * STEPS * 96 : 0) + half * 16;
            const unsigned char* pb = sB + (wn * WT * 32 + l32) * P + (KSPLIT ? wave * STEPS * 96 : 0) + half * 16;
            constexpr int FB = WT == 1 ? 2 : 1;    // fragments a step ahead, where the registers hold them
            bf16x8 fa[FB][WT][3], fb[FB][WT][3];
            auto frags = [&](int ks, bf16x8 (&fa)[WT][3], bf16x8 (&fb)[WT][3]) __attribute__((always_inline)) {
#pragma unroll
                for (int i = 0; i < WT; ++i)
#pragma unroll
                    for (int p = 0; p < 3; ++p) {
                        fa[i][p] = *reinterpret_cast<const bf16x8*>(pa + i * 32 * P + ks * 96 + p * 32);
                        fb[i][p] = *reinterpret_cast<const bf16x8*>(pb + i * 32 * P + ks * 96 + p * 32);
                    }
            };
            frags(0, fa[0], fb[0]);
#pragma unroll
            for (int ks = 0; ks < STEPS; ++ks) {
                if (FB == 2) {
                    if (ks + 1 < STEPS) frags(ks + 1, fa[(ks + 1) % FB], fb[(ks + 1) % FB]);
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int t = 0; t < 6; ++t)
#pragma unroll
                    for (int ni = 0; ni < WT; ++ni)
#pragma unroll
                        for (int mi = 0; mi < WT; ++mi)
                            Mma<bf16_t>::mma(acc[ni][mi], fb[ks % FB][ni][SPLIT_B[t]], fa[ks % FB][mi][SPLIT_A[t]]);
                if (FB == 1 && ks + 1 < STEPS) frags(ks + 1, fa[0], fb[0]);
                if (FB == 2) __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            const unsigned char* pa = sA + slot * SLOT + (wm * WT * 32 + l32) * P + half * (MM::KLANE * ES);
            const unsigned char* pb = sB + slot * SLOT + (wn * WT * 32 + l32) * P + half * (MM::KLANE * ES);
#pragma unroll
            for (int k0 = 0; k0 < BK / MM::KSTEP / (KSPLIT ? 4 : 1); ++k0) {
                const int ks = KSPLIT ? wave * (BK / MM::KSTEP / 4) + k0 : k0;
                typename MM::Frag fa[WT], fb[WT];
#pragma unroll
                for (int i = 0; i < WT; ++i) {
                    fa[i] = *reinterpret_cast<const typename MM::Frag*>(pa + i * 32 * P + ks * MM::KSTEP * ES);
                    fb[i] = *reinterpret_cast<const typename MM::Frag*>(pb + i * 32 * P + ks * MM::KSTEP * ES);
                }
#pragma unroll
                for (int ni = 0; ni < WT; ++ni)
#pragma unroll
                    for (int mi = 0; mi < WT; ++mi) MM::mma(acc[ni][mi], fb[ni], fa[mi]);
            }
        }
    }
    if constexpr (PIECES && !KSPLIT) {
        if (piece) {
            end_piece();
#pragma unroll
            for (int a = 0; a < WT; ++a)
#pragma unroll
                for (int b = 0; b < WT; ++b) acc[a][b] = sum[a][b];
        }
    }
    lds_barrier();
    if constexpr (KSPLIT) {
        end_round();
        if (wave == 0) acc[0][0] = sum[0][0];
    }

    // infinite operands, whose parts make NaN of every product: those sums by the fp32 instructions, the others keep their bits; and sums of
    // fewer products than make up for the six roundings of one (one product 2.6e-8 -> 3.5e-8, two 3.1e-8 -> 3.4e-8, four 4.0e-8 -> 3.3e-8)
    if constexpr (SPLIT) {
        const bool few = K <= 4;
#pragma unroll
        for (int ni = 0; ni < WT; ++ni)
#pragma unroll
            for (int mi = 0; mi < WT; ++mi) {
                if (KSPLIT && wave) continue;          // wave 0 has the sums
                float x = acc[ni][mi][0];
#pragma unroll
                for (int v = 1; v < 16; ++v) x += acc[ni][mi][v];
                if (__builtin_expect(!few && !__any(x - x != 0.0f), 1)) continue;
                const long m = m0 + wm * WT * 32 + mi * 32 + l32, n = n0 + wn * WT * 32 + ni * 32 + l32;
                const T* pa = A + (m < M ? m : M - 1) * d.lda;
                const T* pb = B + (n < N ? n : N - 1) * d.ldb;
                f32x16 y;
#pragma unroll
                for (int v = 0; v < 16; ++v) y[v] = 0.0f;
#pragma unroll 1
                for (int k = 4 * half; k - 4 * half < K; k += 8) {
                    typename MM::Frag fa = {0, 0, 0, 0}, fb = {0, 0, 0, 0};
                    if (k < K) {
                        fa = *reinterpret_cast<const typename MM::Frag*>(pa + k);
                        fb = *reinterpret_cast<const typename MM::Frag*>(pb + k);
                    }
                    MM::mma(y, fb, fa);
                }
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[ni][mi][v] = !few && acc[ni][mi][v] == acc[ni][mi][v] ? acc[ni][mi][v] : y[v];
            }
    }

    // row offsets of this tile, one integer division per row (kept in LDS for phase 2)
    __shared__ long s_off[BT];
    if (tid < BT) {
        long m = m0 + tid;
        if (m >= M) m = M - 1;
        const unsigned hi = (unsigned)m / (unsigned)d.inner;
        const unsigned lo = (unsigned)m - hi * (unsigned)d.inner;
        s_off[tid] = (long)hi * d.s_o + (long)lo * d.s_i;
    }

    // ---- phase 1: registers -> staged tile [m][n] (values after bias / act / scale / rowdiv) ----
    // (bias / rowdiv are fetched with clamped indices, i.e. without per-lane branches, so the loads
    // are issued back to back; out-of-range values are computed but never stored)
    const T* bias = (const T*)d.bias;
    if (!KSPLIT || wave == 0) {
        float bv[WT][4][4];
#pragma unroll
        for (int ni = 0; ni < WT; ++ni)
#pragma unroll
            for (int g = 0; g < 4; ++g)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    long n = n0 + wn * WT * 32 + ni * 32 + 8 * g + 4 * half + e;
                    n = n < N ? n : N - 1;
                    bv[ni][g][e] = bias ? DT<T>::to_f(bias[n]) : 0.0f;
                }
#pragma unroll
        for (int mi = 0; mi < WT; ++mi) {
            const int mr = wm * WT * 32 + mi * 32 + l32;
            long m = m0 + mr;
            m = m < M ? m : M - 1;
            float rdiv = 1.0f;
            if (d.rowdiv) rdiv = 1.0f / (d.rowdiv[(long)bz * M + m] + d.div_eps);
#pragma unroll
            for (int ni = 0; ni < WT; ++ni) {
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const int nc = wn * WT * 32 + ni * 32 + 8 * g + 4 * half;
                    OT* dst = reinterpret_cast<OT*>(sC + mr * CP + nc * OES);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        float x = acc[ni][mi][4 * g + e] + bv[ni][g][e];
                        if (d.act == FFK_ACT_RELU) x = relu_f(x);
                        else if (d.act == FFK_ACT_SIGMOID) x = sigmoid_f(x);
                        dst[e] = DT<OT>::from_f(x * d.scale * rdiv);
                    }
                }
            }
        }
    }
    lds_barrier();

    // ---- phase 2: staged tile -> global ----
    OT* out = (OT*)d.out + (long)bz * d.o_bs;
    const OT* resid = d.resid ? (const OT*)d.resid + (long)bz * d.o_bs : nullptr;
    // extended residual stream (bf16 output with a residual, s_d == 1): the update is added at 24 bits
    int8_t* xtail = nullptr;
    if constexpr (XS_OK) xtail = d.xtail ? (int8_t*)d.xtail + (long)bz * d.o_bs : nullptr;
    if (d.s_d == 1) {
        constexpr int VPR = BT / OVEC;
        constexpr int N_V = BT * VPR, N_IT = (N_V + THREADS - 1) / THREADS, NB = N_IT < 4 ? N_IT : 4;
        // vector path when every row pitch / base keeps 16-byte alignment and N is a multiple of the vector
        const bool vec_ok = (N % OVEC) == 0 && (reinterpret_cast<uintptr_t>(out) & 15u) == 0 &&
                            (!resid || (reinterpret_cast<uintptr_t>(resid) & 15u) == 0) && (d.s_o % OVEC) == 0 &&
                            (d.s_i % OVEC) == 0 && (d.s_h % OVEC) == 0;
        if (vec_ok) {
            const long n_last = N - OVEC;
            const bool live = N_V >= THREADS || tid < N_V;
#pragma unroll 1
            for (int i0 = 0; i0 < N_IT; i0 += NB) {
                Vec16<OT> x[NB], rv[NB];
                u32x2 tv[NB];
                long o[NB];
#pragma unroll
                for (int j = 0; j < NB; ++j) {
                    const int v = N_V >= THREADS ? tid + THREADS * (i0 + j) : tid % N_V;       // the repetitions store nothing
                    const int r = v / VPR, c = (v % VPR) * OVEC;
                    long n = n0 + c;
                    n = n <= n_last ? n : n_last;
                    o[j] = s_off[r] + (n >> 5) * d.s_h + (n & 31);
                    x[j] = *reinterpret_cast<const Vec16<OT>*>(sC + r * CP + c * OES);
                    if (resid) rv[j] = ld16(resid + o[j]);
                    if (xtail) tv[j] = *reinterpret_cast<const u32x2*>(xtail + o[j]);
                }
#pragma unroll
                for (int j = 0; j < NB; ++j) {
                    const int v = N_V >= THREADS ? tid + THREADS * (i0 + j) : tid % N_V;       // the repetitions store nothing
                    const int r = v / VPR, c = (v % VPR) * OVEC;
                    if constexpr (XS_OK) {
                        if (xtail) {
                            float f[8];
                            xs_decode8(*reinterpret_cast<const u32x4*>(&rv[j]), tv[j][0], tv[j][1], f);
#pragma unroll
                            for (int e = 0; e < 8; ++e) f[e] += (float)x[j].e[e];
                            u32x4 hv;
                            u32x2 tn;
                            xs_encode8(f, hv, tn);
                            if (live && m0 + r < M && n0 + c < N) {
                                *reinterpret_cast<u32x4*>(out + o[j]) = hv;
                                *reinterpret_cast<u32x2*>(xtail + o[j]) = tn;
                            }
                            continue;
                        }
                    }
                    if (resid) {
#pragma unroll
                        for (int e = 0; e < OVEC; ++e)
                            x[j].e[e] = DT<OT>::from_f(DT<OT>::to_f(x[j].e[e]) + DT<OT>::to_f(rv[j].e[e]));
                    }
                    if (live && m0 + r < M && n0 + c < N) st16(out + o[j], x[j]);
                }
            }
        } else {
            for (int v = tid; v < BT * BT; v += THREADS) {
                const int r = v / BT, c = v % BT;
                const long m = m0 + r, n = n0 + c;
                if (m >= M || n >= N) continue;
                const long o = s_off[r] + (n >> 5) * d.s_h + (n & 31);
                float y = DT<OT>::to_f(*reinterpret_cast<const OT*>(sC + r * CP + c * OES));
                if constexpr (XS_OK) {
                    if (xtail) {
                        xs_round(y + xs_value(resid[o], xtail[o]), &out[o], &xtail[o]);
                        continue;
                    }
                }
                if (resid) y += DT<OT>::to_f(resid[o]);
                out[o] = DT<OT>::from_f(y);
            }
        }
    } else {
        for (int v = tid; v < BT * BT; v += THREADS) {
            const int c = v / BT, r = v % BT;           // consecutive threads -> consecutive rows m
            const long m = m0 + r, n = n0 + c;
            if (m >= M || n >= N) continue;
            const long o = s_off[r] + (n >> 5) * d.s_h + (n & 31) * d.s_d;
            float y = DT<OT>::to_f(*reinterpret_cast<const OT*>(sC + r * CP + c * OES));
            if (resid) y += DT<OT>::to_f(resid[o]);
            out[o] = DT<OT>::from_f(y);
        }
    }
}

template <typename T, typename OT, int BT>
int launch_tile(const ffk_bgemm_desc& d, hipStream_t st) {
    const size_t ring = sizeof(T) == 4 ? 2 * (size_t)BT * (128 * 192 / BT + 16) : 4 * (size_t)BT * (128 * 128 / BT + 16);
    size_t ct = (size_t)BT * (BT * sizeof(OT) + 16);
    const size_t smem = ring > ct ? ring : ct;
    static FfkLdsReservation lds_reserved;
    {
        const int rc_lds = ffk_reserve_lds(lds_reserved, (const void*)bgemm_nt_kernel<T, OT, BT>, smem, "ffk_bgemm_nt");
        if (rc_lds != FFK_OK) return rc_lds;
    }
    const long tiles = (long)ffk_cdiv(d.M, BT) * ffk_cdiv(d.N, BT) * d.batch;
    FFK_REQUIRE(tiles < (1L << 31) - 8, FFK_ERR_SHAPE, "ffk_bgemm_nt: %ld output tiles exceed the grid limit", tiles);
    dim3 grid((unsigned)(d.batch >= 8 ? 8 * ffk_cdiv(tiles, 8) : tiles));
    bgemm_nt_kernel<T, OT, BT><<<grid, THREADS, smem, st>>>(d);
    return ffk_check_launch("ffk_bgemm_nt");
}

// Which tile: the launch takes about  start + rounds * (each + per_k * K)  microseconds, rounds = tiles / 256 CUs.  The constants are
// fitted to measured launches of 32 .. 65 536 rows, 32 .. 8 192 columns and K = 16 .. 1 024: a small tile pays its latencies over less
// work, but a large one leaves CUs without a tile or works on padding.  bf16, rounds rounded up: 2 048 x 256, K = 1 024 14.0 us with 16
// tiles of 256 x 128, 9.8 us with 128 of 64.  fp32, where the start grows with K and two or three of the smaller tiles share a CU (128 /
// 64 / 32, us): 4 096 x 128, K = 1 024 75 / 30 / 20.7; 9 000 rows 76 / 37 / 40; 13 689 76 / 41 / 56; 65 536 114 / 148 / 219; K = 512, 4 096 rows
// 41 / 17.6 / 12.5, 16 384 44 / 24.5 / 34, 65 536 59 / 77 / 121; 128 products of K = 64, 64 x 64: 12.2 / 5.7 / -, of 256 x 256 x 256
// 36 / 45 / -.  0: the large tiles of the other kernel, if it takes the launch.
int pick_tile(const ffk_bgemm_desc& d, bool large) {
    auto tiles = [&](int bm, int bn) { return (long)ffk_cdiv(d.M, bm) * ffk_cdiv(d.N, bn) * d.batch; };
    if (d.dtype == FFK_F32) {
        auto rounds = [&](int t) { return std::max(1.0, tiles(t, t) / 256.0); };
        const double c128 = 8.0 + 0.0245 * d.K + ffk_cdiv(tiles(128, 128), 256) * (2.0 + 0.04 * d.K);
        const double c64 = 3.0 + 0.009 * d.K + rounds(64) * (0.5 + 0.0165 * d.K);
        const double c32 = 3.0 + 0.005 * d.K + rounds(32) * (0.6 + 0.0059 * d.K);
        return d.K >= BG_PIECES && c32 < c64 && c32 < c128 ? 32 : c64 < c128 ? 64 : 128;
    }
    auto cost = [&](int bm, int bn, double start, double each, double per_k) {
        return start + ffk_cdiv(tiles(bm, bn), 256) * (each + per_k * d.K);
    };
    const double c128 = cost(128, 128, 3.5, 5.0, 0.0060), c64 = cost(64, 64, 3.0, 1.9, 0.0035);
    if (large && (c64 >= c128 || c64 >= cost(256, d.N <= 128 ? 128 : 256, 4.7, 0.0, 0.0095))) return 0;
    return c64 < c128 ? 64 : 128;
}

template <typename T, typename OT>
int launch_bgemm(const ffk_bgemm_desc& d, int tile, hipStream_t st) {
    if constexpr (sizeof(T) == 4) {
        if (tile == 32) return launch_tile<T, OT, 32>(d, st);
    }
    return tile == 64 ? launch_tile<T, OT, 64>(d, st) : launch_tile<T, OT, 128>(d, st);
}

}  // namespace

extern "C" int ffk_bgemm_nt(const ffk_bgemm_desc* d, void* stream) {
    FFK_REQUIRE(d, FFK_ERR_NULL, "ffk_bgemm_nt: null descriptor");
    FFK_REQUIRE(d->a && d->b && d->out, FFK_ERR_NULL, "ffk_bgemm_nt: null operand");
    FFK_REQUIRE(!d->xtail || (d->dtype == FFK_BF16 && !d->out_f32 && d->resid && d->s_d == 1 && d->N % 16 == 0),
                FFK_ERR_UNSUPPORTED, "ffk_bgemm_nt: a residual tail needs bf16 output, a residual, s_d == 1 and N %% 16 == 0");
    FFK_REQUIRE(ffk_aligned16(d->xtail) && (!d->xtail || (d->o_bs % 16 == 0 && d->s_o % 8 == 0 && d->s_i % 8 == 0 && d->s_h % 8 == 0)),
                FFK_ERR_ALIGN, "ffk_bgemm_nt: residual tail rows must be 16-byte aligned");
    const int es = d->dtype == FFK_F32 ? 4 : 2;
    const int vec = 16 / es;
    FFK_REQUIRE(d->M > 0 && d->N > 0 && d->K > 0 && d->batch > 0 && d->batch < 65536 && d->inner > 0, FFK_ERR_SHAPE,
                "ffk_bgemm_nt: bad shape M=%d N=%d K=%d batch=%d inner=%d", d->M, d->N, d->K, d->batch, d->inner);
    FFK_REQUIRE(d->K % vec == 0, FFK_ERR_SHAPE, "ffk_bgemm_nt: K=%d must be a multiple of %d", d->K, vec);
    FFK_REQUIRE(ffk_aligned16(d->a) && ffk_aligned16(d->b) && d->lda % vec == 0 && d->ldb % vec == 0 &&
                    d->a_bs % vec == 0 && d->b_bs % vec == 0,
                FFK_ERR_ALIGN, "ffk_bgemm_nt: operand rows must be 16-byte aligned");
    hipStream_t st = (hipStream_t)stream;
    int tile = pick_tile(*d, d->dtype == FFK_BF16);
    if (tile == 0) {
        int status = FFK_OK;
        if (ffk_bgemm_big_try(d, st, &status)) return status;
        tile = pick_tile(*d, false);
    }
    if (d->dtype == FFK_BF16) {
        return d->out_f32 ? launch_bgemm<bf16_t, float>(*d, tile, st) : launch_bgemm<bf16_t, bf16_t>(*d, tile, st);
    } else if (d->dtype == FFK_F32) {
        return launch_bgemm<float, float>(*d, tile, st);
    }
    return ffk_fail(FFK_ERR_DTYPE, "ffk_bgemm_nt: unsupported dtype tag %d", d->dtype);
}
