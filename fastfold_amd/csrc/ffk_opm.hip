// Fused outer-product-mean core (see ffk_opm_fused in include/ffk.h):
//     out[i, j, c] = resid[i, j, c] + ( sum_{d,e} O_ij[d, e] * W[c, d, e] + bias[c] ) / (norm[i, j] + eps),
//     O_ij[d, e]   = sum_s a[s, i, d] * b[s, j, e]                       (32 x 32 per residue pair)
// without ever writing the [r, r, 1024] outer product to memory.
//
// A workgroup owns TI i x 32 j residue pairs, TI = 8 or 4 (8 wavefronts) or 2 (4), and walks the 32 values of e in 16
// chunks of two.  Per chunk (TI = 8):
//   phase A  (outer product)  wave w multiplies its own i = i0 + w: rows (d) x columns (j, e in chunk),
//            K = s.  Its a-fragments stay in registers for the whole tile; the b rows of the chunk come
//            from LDS.  The 32 x 32 results are rounded to bf16 and written to LDS as rows of
//            A2[pair][k2 = (e, d)] - exactly the operand layout of the second product.
//   phase B  (projection)     out[pair, c] += A2[pair, chunk] . W2[c, chunk]: 8 x 4 MFMA tiles, each
//            wave owns 2 x 2 of them; accumulators live in registers across all chunks.
// b and W2 chunks arrive by direct global -> LDS loads (XOR-swizzled unpadded rows) one iteration
// ahead; phase B of chunk q - 1 and phase A of chunk q run between the same pair of barriers, so there
// is one barrier per chunk.  With TI = 4 or 2 two waves share an i (one column tile each) and a wave owns 1 x 2 output tiles: less
// work per chunk and more workgroups, for launches that leave CUs empty (see ffk_opm_fused).  The weight is expected pre-permuted
// to k2 = e * 32 + d order.
// What bounds it is the chain of a step: LDS reads, products, rounding, LDS writes, barrier (matrix pipe busy 45 % at r = 1 024
// when each of them waited for the one before).  Operands requested a group ahead, the outer products rounded between the products
// of the projection, and loads to LDS issued where the compiler does not order LDS reads behind them: r = 1 024, 128 sequences
// 576 -> 536 us, 416 104 -> 99 us, 256 39.0 -> 37.0 us.
#include "ffk_common.h"
#include <type_traits>

namespace {

typedef bf16_t T;
constexpr int OP_TJ = 32;                        // pairs per workgroup: TI i x 32 j
constexpr int OP_EC = 2;                         // values of e per chunk
constexpr int OP_NCHUNK = 32 / OP_EC;            // 16
constexpr int OP_K2C = OP_EC * 32;               // k2 elements per chunk (64)
constexpr int OP_PA = OP_K2C * 2 + 16;           // A2 row pitch in bytes (padded: written by ds_write)
constexpr int OP_W2SLOT = 128 * OP_K2C * 2;      // W2 chunk: 128 rows of 128 bytes (16 KB)

template <int KS1, int OP_TI, int WAVES>   // KS1: MFMA K steps of the outer product, spad / 16 (4 or 8)
__global__ __launch_bounds__(64 * WAVES, WAVES / 4) void opm_fused_kernel(T* __restrict__ out, const T* __restrict__ resid, int8_t* __restrict__ xtail,
                                                                 const T* __restrict__ at, const T* __restrict__ bt,
                                                                 const T* __restrict__ w2p, const T* __restrict__ bias,
                                                                 const float* __restrict__ norm, int r, float eps) {
    typedef Mma<T> MM;
    constexpr int OP_A2 = OP_TI * OP_TJ * OP_PA;         // one A2 buffer
    constexpr int OP_THREADS = 64 * WAVES, WM = WAVES / 2, WLD = OP_W2SLOT / 16 / OP_THREADS;
    constexpr int MT = OP_TI / WM, WI = WAVES / OP_TI, NCT = 2 / WI;    // m-tiles per wave (phase B), waves per i, column tiles per wave (phase A)
    constexpr int SPAD = KS1 * 16;                       // K of the outer product
    constexpr int BROW = SPAD * 2;                       // bytes per b row (128 or 256)
    constexpr int BCOLS = BROW / 16;                     // 16-byte columns per b row (8 or 16)
    constexpr int BSLOT = OP_TJ * OP_EC * BROW;          // b chunk: 64 rows
    constexpr int BLD = BSLOT / 16 / OP_THREADS;         // loads per thread per b chunk (1 or 2)
    extern __shared__ __align__(16) unsigned char smem[];
    unsigned char* s_a2 = smem;                          // [2][256][OP_PA]
    unsigned char* s_w2 = smem + 2 * OP_A2;              // [3][128][128 B]
    unsigned char* s_b = s_w2 + 3 * OP_W2SLOT;           // [2][64][BROW]

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    const int tiles_j = r / OP_TJ;
    const int i0 = (blockIdx.x / tiles_j) * OP_TI, j0 = (blockIdx.x % tiles_j) * OP_TJ;

    const int iw = wave / WI, ctw = (wave % WI) * NCT;   // phase A: this wave's i and first column tile
    // ---- a fragments of this wave's i (rows d through tau: registers of the result hold d = 16 half + v) ----
    bf16x8 af[KS1];
    {
        const T* ap = at + ((long)(i0 + iw) * 32 + ffk_tau(l32)) * SPAD + half * 8;
#pragma unroll
        for (int ks = 0; ks < KS1; ++ks) af[ks] = MM::ld(ap + ks * 16);
    }

    // ---- chunk loaders (direct to LDS; lane L of a wave lands at dst + 16 L) ----
    // b chunk: LDS row rho = j_local * 2 + ee, column c holds global column c ^ swz(rho)
    const T* bsrc[BLD];
#pragma unroll
    for (int i = 0; i < BLD; ++i) {
        const int v = i * OP_THREADS + tid, rho = v / BCOLS, c = v % BCOLS;
        const int swz = BCOLS == 16 ? (rho & 15) : ((rho >> 1) & 7);
        bsrc[i] = bt + ((long)(j0 + (rho >> 1)) * 32 + (rho & 1)) * SPAD + ((c ^ swz) * 8);
    }
    // W2 chunk: LDS row rho (0..127) holds weight row 32 * (rho / 32) + tau(rho % 32); 8 columns of 16 bytes
    const T* wsrc[WLD];
#pragma unroll
    for (int i = 0; i < WLD; ++i) {
        const int v = i * OP_THREADS + tid, rho = v >> 3, c = v & 7;
        wsrc[i] = w2p + (long)((rho & ~31) + ffk_tau(rho & 31)) * 1024 + ((c ^ ((rho >> 1) & 7)) * 8);
    }
    const unsigned lds_base = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)smem;
    // asm: with loads to LDS that it knows of the compiler waits for every LDS read of the wave in front of each group of products
    auto dma = [&](const T* src, unsigned dst) __attribute__((always_inline)) {
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(lds_base + dst) : "memory", "m0");
#pragma clang diagnostic pop
    };
    auto fetch = [&](int q) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < BLD; ++i)
            dma(bsrc[i] + (long)q * OP_EC * SPAD, 2 * OP_A2 + 3 * OP_W2SLOT + (q & 1) * BSLOT + (i * OP_THREADS + wave * 64) * 16);
#pragma unroll
        for (int i = 0; i < WLD; ++i) dma(wsrc[i] + q * OP_K2C, 2 * OP_A2 + (q % 3) * OP_W2SLOT + (i * OP_THREADS + wave * 64) * 16);
    };

    // ---- phase B roles: m-tiles MT * (wave % WM) .., c-tiles 2 * (wave / WM) + {0, 1} ----
    const int mt0 = MT * (wave % WM), ct0 = 2 * (wave / WM);
    f32x16 acc2[MT][2];   // [m][c]
#pragma unroll
    for (int a = 0; a < MT; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc2[a][b][v] = 0.0f;

    // per-lane LDS offsets
    int boff[KS1];                                       // b fragment of column-tile 0: row l32, column 2 ks + half
#pragma unroll
    for (int ks = 0; ks < KS1; ++ks) {
        const int swz = BCOLS == 16 ? (l32 & 15) : ((l32 >> 1) & 7);
        boff[ks] = l32 * BROW + (((2 * ks + half) ^ swz) << 4);
    }
    // (column tile 1 = rows 32..63: same swizzle since 32 is a multiple of 16)
    int woff[4];                                         // W2 fragment of c-tile 0: row l32, column 2 ks + half
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) woff[ks] = l32 * 128 + (((2 * ks + half) ^ ((l32 >> 1) & 7)) << 4);
    // A2 write position of phase A: pair (iw, 16 ct + l32 / 2), k2 = (l32 & 1) * 32 + 16 half
    const int a2w = (iw * 32 + (l32 >> 1)) * OP_PA + ((l32 & 1) * 32 + 16 * half) * 2;
    // A2 fragment of phase B: pair row mt * 32 + l32, k2 = 16 ks + 8 half
    const int a2r = l32 * OP_PA + half * 16;

    // The epilogue's operands (residual, its tail, the normaliser) are requested during the third chunk, not in the
    // epilogue: with one workgroup per CU (154 KB of LDS) nothing else would cover their latency - four dependent round
    // trips took 8 of a workgroup's 42 microseconds.  The wait at the top of the next chunk covers them.
    u32x4 e_rv[MT][2][2], e_tv[MT][2];
    float e_norm[MT];
    const int pf_q = 2 + (int)((blockIdx.x >> 3) % 12u);   // spread over the chunks: the workgroups of a launch run in step
    // A step: the outer products of chunk q (A) and the projection of chunk q - 1 (B).  All operands come through one ring of two
    // groups of up to four fragments, requested a group ahead; the outer products are rounded and written between the products of
    // the projection, so that neither an LDS latency nor the rounding stands alone between two barriers.
    constexpr int AG = KS1 / 4, NA = NCT * AG;           // groups of the outer product
    bf16x8 ring[2][4];
    auto step = [&](int q, auto do_a, auto do_b) __attribute__((always_inline)) {
        constexpr bool A = decltype(do_a)::value, B = decltype(do_b)::value;
        constexpr int G0 = A ? 0 : NA, G1 = B ? NA + 4 : NA;
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");    // chunk q has landed (this wave's part), its A2 rows are written
        __builtin_amdgcn_s_barrier();                        // ... everyone's; A2 of chunk q - 1 is complete
        asm volatile("" ::: "memory");
        if (q + 1 < OP_NCHUNK) fetch(q + 1);
        if (q == pf_q) {
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const long pr = (long)(i0 + mt0 + m) * r + j0 + l32;
                e_norm[m] = norm[pr];
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    const long o = pr * 128 + (ct0 + c) * 32 + 16 * half;
                    e_rv[m][c][0] = *reinterpret_cast<const u32x4*>(resid + o);
                    e_rv[m][c][1] = *reinterpret_cast<const u32x4*>(resid + o + 8);
                    if (xtail) e_tv[m][c] = *reinterpret_cast<const u32x4*>(xtail + o);
                }
            }
        }
        const unsigned char* bs = s_b + (q & 1) * BSLOT + ctw * 32 * BROW;
        const unsigned char* a2 = s_a2 + ((q + 1) & 1) * OP_A2 + mt0 * 32 * OP_PA + a2r;
        const unsigned char* w2 = s_w2 + ((q + 2) % 3) * OP_W2SLOT + ct0 * 32 * 128;
        unsigned char* a2n = s_a2 + (q & 1) * OP_A2 + a2w + ctw * 16 * OP_PA;
        f32x16 o[NCT];
        auto request = [&](int g) __attribute__((always_inline)) {
            bf16x8* f = ring[g & 1];
            if (g < NA) {
#pragma unroll
                for (int i = 0; i < 4; ++i) f[i] = *reinterpret_cast<const bf16x8*>(bs + g / AG * 32 * BROW + boff[g % AG * 4 + i]);
            } else {
#pragma unroll
                for (int m = 0; m < MT; ++m) f[m] = *reinterpret_cast<const bf16x8*>(a2 + m * 32 * OP_PA + (g - NA) * 32);
#pragma unroll
                for (int c = 0; c < 2; ++c) f[2 + c] = *reinterpret_cast<const bf16x8*>(w2 + c * 32 * 128 + woff[g - NA]);
            }
        };
        // eight values of a column tile's result
        auto hand_over = [&](int piece) __attribute__((always_inline)) {
            typedef float f32x2 __attribute__((ext_vector_type(2)));
            typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
            u32x4 y;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const f32x2 pr = {o[piece >> 1][8 * (piece & 1) + 2 * t], o[piece >> 1][8 * (piece & 1) + 2 * t + 1]};
                y[t] = __builtin_bit_cast(uint32_t, __builtin_convertvector(pr, bf16x2));
            }
            *reinterpret_cast<u32x4*>(a2n + (piece >> 1) * 16 * OP_PA + (piece & 1) * 16) = y;
        };
        if (A) {
#pragma unroll
            for (int c = 0; c < NCT; ++c)
#pragma unroll
                for (int v = 0; v < 16; ++v) o[c][v] = 0.0f;
        }
        request(G0);
#pragma unroll
        for (int g = G0; g < G1; ++g) {
            if (g + 1 < G1) request(g + 1);
            __builtin_amdgcn_sched_barrier(0);
            const bf16x8* f = ring[g & 1];
            if (g < NA) {
#pragma unroll
                for (int i = 0; i < 4; ++i) MM::mma(o[g / AG], af[g % AG * 4 + i], f[i]);
            } else {
                if (A && g - NA < 2 * NCT) hand_over(g - NA);
#pragma unroll
                for (int m = 0; m < MT; ++m)
#pragma unroll
                    for (int c = 0; c < 2; ++c) MM::mma(acc2[m][c], f[2 + c], f[m]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (A && !B) {
#pragma unroll
            for (int p = 0; p < 2 * NCT; ++p) hand_over(p);
        }
    };
    typedef std::integral_constant<bool, true> Yes;
    typedef std::integral_constant<bool, false> No;
    fetch(0);
    step(0, Yes(), No());
    // Kernel arguments that only the epilogue reads would count as outstanding at the head of the loop, where a wait for a fragment
    // would then be one for every LDS read of the wave
    __builtin_amdgcn_s_waitcnt(0xc07f);                  // lgkmcnt(0)
    for (int q = 1; q < OP_NCHUNK; ++q) step(q, Yes(), Yes());
    step(OP_NCHUNK, No(), Yes());

    // ---- epilogue: lane = pair, registers = 16 consecutive channels ----
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const long pr = (long)(i0 + mt0 + m) * r + j0 + l32;
        const float inv = 1.0f / (e_norm[m] + eps);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int ch = (ct0 + c) * 32 + 16 * half;
            const long o = pr * 128 + ch;
            u32x4 bv[2], rv[2];
            bv[0] = *reinterpret_cast<const u32x4*>(bias + ch);
            bv[1] = *reinterpret_cast<const u32x4*>(bias + ch + 8);
            rv[0] = e_rv[m][c][0];
            rv[1] = e_rv[m][c][1];
            if (xtail) {       // extended residual stream: the update is added at 24 bits
                const u32x4 tv = e_tv[m][c];
                float upd[16];
#pragma unroll
                for (int v = 0; v < 16; ++v) upd[v] = (float)(T)((acc2[m][c][v] + (float)reinterpret_cast<const T*>(&bv[v >> 3])[v & 7]) * inv);
                u32x4 h0, h1, tn;
                xs_update16(upd, rv[0], rv[1], tv, h0, h1, tn);
                *reinterpret_cast<u32x4*>(out + o) = h0;
                *reinterpret_cast<u32x4*>(out + o + 8) = h1;
                *reinterpret_cast<u32x4*>(xtail + o) = tn;
                continue;
            }
            T y[16];
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const float x = (acc2[m][c][v] + (float)reinterpret_cast<const T*>(&bv[v >> 3])[v & 7]) * inv;
                y[v] = (T)((float)(T)x + (float)reinterpret_cast<const T*>(&rv[v >> 3])[v & 7]);
            }
            *reinterpret_cast<u32x4*>(out + o) = *reinterpret_cast<const u32x4*>(&y[0]);
            *reinterpret_cast<u32x4*>(out + o + 8) = *reinterpret_cast<const u32x4*>(&y[8]);
        }
    }
}

template <int KS1, int OP_TI, int WAVES>
int opm_launch(T* out, const T* resid, int8_t* xtail, const T* at, const T* bt, const T* w2p, const T* bias, const float* norm, int r,
               float eps, hipStream_t st) {
    const size_t smem = 2 * (size_t)(OP_TI * OP_TJ * OP_PA) + 3 * OP_W2SLOT + 2 * (size_t)(OP_TJ * OP_EC * KS1 * 32);
    static FfkLdsReservation lds_reserved;
    {
        const int rc_lds = ffk_reserve_lds(lds_reserved, (const void*)opm_fused_kernel<KS1, OP_TI, WAVES>, smem, "ffk_opm_fused");
        if (rc_lds != FFK_OK) return rc_lds;
    }
    const unsigned grid = (unsigned)((r / OP_TI) * (r / OP_TJ));
    opm_fused_kernel<KS1, OP_TI, WAVES><<<grid, 64 * WAVES, smem, st>>>(out, resid, xtail, at, bt, w2p, bias, norm, r, eps);
    return ffk_check_launch("ffk_opm_fused");
}

}  // namespace

extern "C" int ffk_opm_fused(void* out, const void* resid, void* xtail, const void* a_t, const void* b_t, const void* w2p, const void* bias,
                             const float* norm, int64_t r, int64_t spad, float eps, int dtype, void* stream) {
    FFK_REQUIRE(out && resid && a_t && b_t && w2p && bias && norm, FFK_ERR_NULL, "ffk_opm_fused: null pointer");
    FFK_REQUIRE(dtype == FFK_BF16, FFK_ERR_DTYPE, "ffk_opm_fused: bf16 only (dtype tag %d)", dtype);
    FFK_REQUIRE(r > 0 && r % 32 == 0 && r <= 32768, FFK_ERR_SHAPE, "ffk_opm_fused: r=%ld must be a positive multiple of 32", (long)r);
    FFK_REQUIRE(spad == 64 || spad == 128, FFK_ERR_UNSUPPORTED, "ffk_opm_fused: padded sequence count %ld must be 64 or 128", (long)spad);
    FFK_REQUIRE(ffk_aligned16(out) && ffk_aligned16(resid) && ffk_aligned16(a_t) && ffk_aligned16(b_t) && ffk_aligned16(w2p) &&
                    ffk_aligned16(bias) && ffk_aligned16(xtail),
                FFK_ERR_ALIGN, "ffk_opm_fused: buffers must be 16-byte aligned");
    hipStream_t st = (hipStream_t)stream;
    // Two i and four waves per workgroup while no CU has two of these, then four i and eight waves, then eight i: a workgroup's time is
    // mostly its 17 steps (0.65 us each with one wave per SIMD, 0.9 with two, 1.4 with twice the rows), so more and smaller workgroups
    // win until they come in rounds.  128 sequences, TI = 2 / 4 / 8: r = 96 16.5 / 19.6 / 28.6 us, 128 17.9 / 20.9 / 29.3, 160
    // 30.9 / 22.3 / 29.9, 192 45.2 / 38.6 / 30.5, 256 61 / 42.8 / 36.9.
    const long tj = r / OP_TJ;
    const int ti = (r / 2) * tj <= 256 ? 2 : (r / 4) * tj <= 256 ? 4 : 8;
#define FFK_OPM(KS1, TI, W) opm_launch<KS1, TI, W>((T*)out, (const T*)resid, (int8_t*)xtail, (const T*)a_t, (const T*)b_t, (const T*)w2p, (const T*)bias, norm, (int)r, eps, st)
    if (spad == 128) return ti == 2 ? FFK_OPM(8, 2, 4) : ti == 4 ? FFK_OPM(8, 4, 8) : FFK_OPM(8, 8, 8);
    return ti == 2 ? FFK_OPM(4, 2, 4) : ti == 4 ? FFK_OPM(4, 4, 8) : FFK_OPM(4, 8, 8);
#undef FFK_OPM
}
