// Fused transition (see ffk_transition_fused in include/ffk.h):
//     out = x + W2 . relu( W1 . LayerNorm(x) + b1 ) + b2        (C -> 4C -> C channels, C = 128 or 256, bf16)
// with the hidden activation never leaving the chip: two kernels, chosen by width and rows at the end of this file.
//
// transition_fused_kernel (many rows of 128 channels): a workgroup (4 wavefronts) owns 128 rows, a wavefront 32 of
// them from start to end.  Set-up: the rows are fetched once, normalised in registers (16 lanes per row) and passed through LDS into the MFMA
// fragments of their wave, where they stay.  The hidden layer is walked in chunks of 32 channels
// (16 chunks); per chunk and wave
//   first GEMM   H^T[hidden, rows] = W1[chunk] . x^T  (+ b1, relu): one tile of 32 hidden channels; lane =
//                row, registers = hidden channels;
//   second GEMM  out^T[c, rows] += W2[c, chunk] . H^T: the rounded accumulators of the first GEMM are the
//                N operand as they stand.  A lane holds hidden channels 8a + 4h + b of a tile (h = its
//                half-wave) in registers 4a + b, and an MFMA K step wants 8 consecutive K per half-wave,
//                so the first GEMM's M-operand row i is loaded from weight row sigma(i) such that
//                registers 8j .. 8j + 7 of half-wave h are hidden channels 16j + 8h .. 16j + 8h + 7.
// Only the weights go through LDS: W1 / W2 chunks arrive by direct global -> LDS loads (XOR-swizzled
// unpadded rows) one chunk ahead, shared by the four waves; one barrier per chunk.  A workgroup spends about
// a third of its life fetching its rows and storing its results (measured with wall-clock stamps: 3.5 us set-up,
// 14 us in the chunk loop, 5 us in the epilogue at C = 128 with residual tails), so as many workgroups as fit share
// a CU and cover each other's waits: with 32-channel chunks the rings take 32 KB (C = 128; the row buffer of the
// set-up, 34 KB, is then the larger) and the kernel 149 registers: three workgroups per CU.
#include "ffk_common.h"
#include <type_traits>

namespace {

typedef bf16_t T;
constexpr int TR_THREADS = 256;
constexpr int TR_BM = 128;                     // rows per workgroup
// The weights are the same for every workgroup and new to the chip (a stack's blocks have weights of their own): the workgroups of
// an XCD ask for the same chunk at the same time, so each chunk costs all of them the latency of the memory behind the XCD's L2,
// and a CU's misses in flight allow it 30 bytes per ns where hits allow 60.  So every workgroup of an XCD (they are dealt round
// robin) first touches its share of the lines, one word each, while its rows are on their way: 16 384 rows of 256 channels 31.6 ->
// 28.1 us, of 128 channels 11.3 -> 10.8 us.
__device__ __forceinline__ uint32_t tr_touch(const T* w1, const T* w2, int lines, int threads) {
    const int share = (blockIdx.x >> 3) * threads + threadIdx.x, step = ((gridDim.x + 7 - (blockIdx.x & 7)) >> 3) * threads;
    uint32_t x = 0;
    for (int i = share; i < 2 * lines; i += step)
        x ^= *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(i < lines ? w1 : w2) + (long)(i < lines ? i : i - lines) * 128);
    return x;
}

constexpr int TR_C = 128, TR_H = 4 * TR_C;
template <int NS> struct TrGeo {
    static constexpr int C = TR_C, H = TR_H;
    static constexpr int HC = 32;                   // hidden channels per chunk
    static constexpr int NCHUNK = H / HC;
    static constexpr int W1SLOT = HC * C * 2;       // HC rows of 2 C bytes (8 KB)
    static constexpr int W2SLOT = C * HC * 2;       // C rows of 2 HC bytes (8 KB)
    static constexpr int XP = C * 2 + 16;           // pitch of the normalised rows (set-up only)
    static constexpr int NC1 = C / 8;               // 16-byte columns of a W1 row
    static constexpr int NC2 = HC / 8;              // 16-byte columns of a W2 row
    static constexpr int RP2 = 256 / (HC * 2);      // W2 rows per 256 bytes of LDS: the swizzle period
    static constexpr int KS1 = C / 16, KS2 = HC / 16, CT = C / 32;
    static constexpr size_t SMEM_RINGS = NS * (size_t)W1SLOT + NS * W2SLOT + H * sizeof(float);
    static constexpr size_t SMEM_ROWS = (size_t)TR_BM * XP;
    static constexpr int NLD = W1SLOT / 16 / TR_THREADS;   // 16-byte requests per thread and ring slot
    static_assert(W1SLOT == W2SLOT, "ring slots of one size");
    static constexpr size_t SMEM = SMEM_RINGS > SMEM_ROWS ? SMEM_RINGS : SMEM_ROWS;
};

// i = 8a + 4h + b  ->  16 (a / 2) + 8h + 4 (a % 2) + b
__device__ __forceinline__ int tr_sigma(int i) { return (i >> 4) * 16 + ((i >> 2) & 1) * 8 + ((i >> 3) & 1) * 4 + (i & 3); }

__device__ __forceinline__ void tr_load_lds(const T* src, unsigned char* dst_wave) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                     (__attribute__((address_space(3))) void*)dst_wave, 16, 0, 0);
}

// NS: slots of the weight rings.  Two slots (one chunk in flight) when three workgroups share a CU and cover each
// other's waits; four when the launch has at most one workgroup per CU and the chunk stream has to hide the whole
// memory latency by itself (a chunk is multiplied in less than half a microsecond).
template <int NS>
__global__ __launch_bounds__(TR_THREADS, NS == 4 ? 1 : 3) void transition_fused_kernel(T* __restrict__ out, const T* __restrict__ x, int8_t* __restrict__ xtail,
                                                                        const T* __restrict__ gamma, const T* __restrict__ beta,
                                                                        const T* __restrict__ w1, const T* __restrict__ b1,
                                                                        const T* __restrict__ w2, const T* __restrict__ b2,
                                                                        long M, float eps) {
    typedef Mma<T> MM;
    typedef TrGeo<NS> G;
    constexpr int NLD = G::NLD;
    constexpr int TR_HC = G::HC, TR_NCHUNK = G::NCHUNK, TR_W1SLOT = G::W1SLOT, TR_W2SLOT = G::W2SLOT, TR_XP = G::XP;
    extern __shared__ __align__(16) unsigned char smem[];
    unsigned char* s_w1 = smem;                           // [NS][HC][2 C bytes]
    unsigned char* s_w2 = smem + NS * TR_W1SLOT;          // [NS][C][2 HC bytes]
    float* s_b1 = reinterpret_cast<float*>(s_w2 + NS * TR_W2SLOT);  // [H]
    unsigned char* s_x = smem;                            // [128][TR_XP], set-up only (aliases the rings)

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    const long m0 = (long)blockIdx.x * TR_BM;

    // ---- set-up: rows -> LayerNorm in registers -> LDS -> this wave's fragments ----
    {
        constexpr int LPR = TR_C / 8, RPP = TR_THREADS / LPR, NPASS = TR_BM / RPP;   // lanes per row, rows per pass
        const int c8 = tid % LPR, r0 = tid / LPR;
        const Vec16<T> g = ld16(gamma + c8 * 8), b = ld16(beta + c8 * 8);
        Vec16<T> v[NPASS];
#pragma unroll
        for (int i = 0; i < NPASS; ++i) {
            long m = m0 + r0 + RPP * i;
            m = m < M ? m : M - 1;                        // clamped: rows past the end are never stored
            v[i] = ld16(x + m * TR_C + c8 * 8);
        }
#pragma unroll
        for (int i = 0; i < NPASS; ++i) {
            float f[8], s = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                f[e] = (float)v[i].e[e];
                s += f[e];
            }
            const float q = centre8(f, group_sum(s, LPR) * (1.0f / TR_C));
            const float rs = rsqrtf(group_sum(q, LPR) * (1.0f / TR_C) + eps);
            Vec16<T> y;
#pragma unroll
            for (int e = 0; e < 8; ++e) y.e[e] = (T)__builtin_fmaf(f[e] * rs, (float)g.e[e], (float)b.e[e]);
            *reinterpret_cast<Vec16<T>*>(s_x + (r0 + RPP * i) * TR_XP + c8 * 16) = y;
        }
    }
    lds_barrier();
    bf16x8 xf[G::KS1];                                     // rows 32 wave + l32, all of K = C
#pragma unroll
    for (int ks = 0; ks < G::KS1; ++ks)
        xf[ks] = *reinterpret_cast<const bf16x8*>(s_x + (wave * 32 + l32) * TR_XP + ks * 32 + half * 16);
    lds_barrier();                                         // the row buffer is free: the rings may overwrite it
    for (int i = tid; i < TR_H; i += TR_THREADS) s_b1[i] = (float)b1[i];

    // ---- chunk loaders (direct to LDS; lane L of a wave lands at dst + 16 L) ----
    // W1 chunk: LDS row rho (0..31) holds weight row sigma(rho) of the chunk; 16 columns
    const T* w1src[NLD];
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
        const int v = i * TR_THREADS + tid, rho = v / G::NC1, c = v % G::NC1;
        w1src[i] = w1 + (long)tr_sigma(rho) * TR_C + ((c ^ (rho & 15)) * 8);
    }
    // W2 chunk: LDS row rho (0..127) holds weight row 32 * (rho / 32) + tau(rho % 32); 4 columns
    const T* w2src[NLD];
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
        const int v = i * TR_THREADS + tid, rho = v / G::NC2, c = v % G::NC2;
        w2src[i] = w2 + (long)((rho & ~31) + ffk_tau(rho & 31)) * TR_H + ((c ^ ((rho / G::RP2) & (G::NC2 - 1))) * 8);
    }
    auto fetch = [&](int q) {                              // past the last chunk it is fetched again (into a free slot)
        const int qc = q < TR_NCHUNK ? q : TR_NCHUNK - 1;
        unsigned char* d1 = s_w1 + (q % NS) * TR_W1SLOT + wave * 1024;
#pragma unroll
        for (int i = 0; i < NLD; ++i) tr_load_lds(w1src[i] + (long)qc * TR_HC * TR_C, d1 + i * (TR_THREADS * 16));
        unsigned char* d2 = s_w2 + (q % NS) * TR_W2SLOT + wave * 1024;
#pragma unroll
        for (int i = 0; i < NLD; ++i) tr_load_lds(w2src[i] + qc * TR_HC, d2 + i * (TR_THREADS * 16));
    };

    f32x16 acc2[G::CT];                                    // out^T tiles: channels 32 ct + 16 half + v, row l32
#pragma unroll
    for (int c = 0; c < G::CT; ++c) {                      // start from b2: the epilogue has no bias to add
        const Vec16<T> b0 = ld16(b2 + c * 32 + 16 * half), b1v = ld16(b2 + c * 32 + 16 * half + 8);
#pragma unroll
        for (int v = 0; v < 8; ++v) {
            acc2[c][v] = (float)b0.e[v];
            acc2[c][8 + v] = (float)b1v.e[v];
        }
    }

    int w1off[G::KS1];                                     // W1 fragment: row l32, column 2 ks + half
#pragma unroll
    for (int ks = 0; ks < G::KS1; ++ks) w1off[ks] = l32 * (TR_C * 2) + (((2 * ks + half) ^ (l32 & 15)) << 4);
    int w2off[G::KS2];                                     // W2 fragment of c-tile 0: row l32, column 2 ks + half
#pragma unroll
    for (int ks = 0; ks < G::KS2; ++ks) w2off[ks] = l32 * (TR_HC * 2) + (((2 * ks + half) ^ ((l32 / G::RP2) & (G::NC2 - 1))) << 4);

#pragma unroll
    for (int q = 0; q < NS - 1; ++q) fetch(q);
    for (int q = 0; q < TR_NCHUNK; ++q) {
        // chunk q has landed (this wave's part) once only the NS - 2 younger chunks (8 loads each) are outstanding
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NLD * (NS - 2)) : "memory");
        __builtin_amdgcn_s_barrier();                        // ... everyone's; nobody still reads the slot of chunk q - 1
        fetch(q + NS - 1);
        const unsigned char* wa = s_w1 + (q % NS) * TR_W1SLOT;
        const unsigned char* wb = s_w2 + (q % NS) * TR_W2SLOT;
        f32x16 h;
        // registers 0..7: hidden 8 half + 0..7 of the chunk, registers 8..15: 16 + 8 half + 0..7
        const float* bp = s_b1 + q * TR_HC + 8 * half;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const f32x4 b4 = *reinterpret_cast<const f32x4*>(bp + (a >> 1) * 16 + (a & 1) * 4);
#pragma unroll
            for (int b = 0; b < 4; ++b) h[4 * a + b] = b4[b];
        }
#pragma unroll
        for (int ks = 0; ks < G::KS1; ++ks) MM::mma(h, *reinterpret_cast<const bf16x8*>(wa + w1off[ks]), xf[ks]);
        // relu after the rounding, on the packed bf16 bit patterns: a negative bf16 is a negative 16-bit integer, so
        // one packed integer max per pair replaces one clamp per value (rounding is monotonic: same bits)
        bf16x8 hf[2];                                      // [K step]: the chunk's N operand
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            typedef float f32x2 __attribute__((ext_vector_type(2)));
            typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
            typedef short s16x2 __attribute__((ext_vector_type(2)));
            const s16x2 zero = {0, 0};
            u32x4 w;
#pragma unroll
            for (int t = 0; t < 4; ++t) {                  // one packed conversion and one packed max per pair
                const f32x2 pr = {h[8 * j + 2 * t], h[8 * j + 2 * t + 1]};
                const bf16x2 r = __builtin_convertvector(pr, bf16x2);
                w[t] = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(s16x2, r), zero));
            }
            hf[j] = __builtin_bit_cast(bf16x8, w);
        }
#pragma unroll
        for (int ks = 0; ks < G::KS2; ++ks)
#pragma unroll
            for (int c = 0; c < G::CT; ++c)
                MM::mma(acc2[c], *reinterpret_cast<const bf16x8*>(wb + c * 32 * (TR_HC * 2) + w2off[ks]), hf[ks]);
    }

    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");         // the re-fetches past the last chunk

    // ---- epilogue: lane = row, registers = 16 consecutive channels ----
    const long row = m0 + wave * 32 + l32;
    const bool ok = row < M;
    const long rc = ok ? row : M - 1;
#pragma unroll
    for (int c = 0; c < G::CT; ++c) {
        const int ch = c * 32 + 16 * half;
        const long o = rc * TR_C + ch;
        u32x4 rv[2];
        rv[0] = *reinterpret_cast<const u32x4*>(x + o);
        rv[1] = *reinterpret_cast<const u32x4*>(x + o + 8);
        if (xtail) {           // extended residual stream: the update is added at 24 bits
            const u32x4 tv = *reinterpret_cast<const u32x4*>(xtail + o);
            float upd[16];
#pragma unroll
            for (int v = 0; v < 16; ++v) upd[v] = (float)(T)acc2[c][v];
            u32x4 h0, h1, tn;
            xs_update16(upd, rv[0], rv[1], tv, h0, h1, tn);
            if (ok) {
                *reinterpret_cast<u32x4*>(out + o) = h0;
                *reinterpret_cast<u32x4*>(out + o + 8) = h1;
                *reinterpret_cast<u32x4*>(xtail + o) = tn;
            }
            continue;
        }
        T y[16];
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            y[v] = (T)((float)(T)acc2[c][v] + (float)reinterpret_cast<const T*>(&rv[v >> 3])[v & 7]);
        }
        if (ok) {
            *reinterpret_cast<u32x4*>(out + o) = *reinterpret_cast<const u32x4*>(&y[0]);
            *reinterpret_cast<u32x4*>(out + o + 8) = *reinterpret_cast<const u32x4*>(&y[8]);
        }
    }
}

// (Modules: 128 channels from 16 385 to 32 768 rows.  256 channels and fewer rows of 128 are theirs in ffk_transition_block, with weights
// in fragment order; here they serve callers with plain weights.)
// The same computation, to the bit, with the two layers on different waves and 64 rows per wave: every launch of 256 channels, and
// those of 128 that leave a CU at most two workgroups.  A fragment of the weights read from LDS feeds two products instead of one:
// with 32 rows per wave the four SIMDs ask LDS for a kilobyte per product each, which is all it delivers.  A workgroup has RP row
// pairs: of its 4 RP waves the first half multiply W1 (row pair, hidden tile w % 2 of a chunk of 64), the other half W2 one or two
// chunks behind (row pair, half of the output channels).  RP = 2 gives every SIMD one wave of either kind; RP = 1 puts one wave
// on every SIMD, twice as many CUs to work, and leaves a wave 512 registers at 256 channels, enough to round the hidden values of
// a chunk between the products of the next.  Hidden values go through LDS in the order the second product reads.  LDS is full at
// C = 256 (two slots of 32 KB for either matrix), so the first layer's bias, which a lane keeps in registers, enters
// through a product with ones.  What is left: the latency of a step (LDS reads, products, barrier: 1.2 us per chunk at RP = 1 for
// 0.45 us of products) and, above one workgroup per CU, the rows and the epilogue, which nothing covers.
// us per launch, with residual tails, one kernel of four (two) waves of each kind over 128 rows before, RP = 1, RP = 2:
//   256 channels: 4 096 rows 35.9, 24.4, 33.1; 12 288 rows 37.0, 25.9, 34.0; 16 384 rows 42.6, 28.1, 35.8; 20 480 rows 44.3, 49.0, 36.9;
//     32 768 rows 51.3, 52.0, 42.1; (transition_fused_kernel:) 65 536 rows 87.6, 98, 82.2; 131 072 rows 167, 192, 155
//   128 channels: 4 096 rows 16.4, 9.3, 12.3; 16 384 rows 17.6, 10.8, 13.2; 32 768 rows 21.7, 17.0, 16.2; (fused:) 65 536 rows 30.5, 30.5, 30.0;
//     1 048 576 rows 359, 420, 400
constexpr int TW_HC = 64;                              // hidden channels per chunk
constexpr int tw_occ(int C, int RP) { return C == 128 ? 2 : RP; }     // waves per SIMD
template <int C, int RP> struct TwGeo {                // RP: row pairs (of 64 rows) of a workgroup
    static constexpr int THREADS = 256 * RP, BM = 64 * RP, H = 4 * C, NCH = H / TW_HC;
    static constexpr int SLOT = TW_HC * C * 2;         // a chunk of either matrix: 32 or 16 KB
    static constexpr int XP = C * 2 + 16;
    static constexpr int HBUF = BM * TW_HC * 2;        // [row pair][row group][K step][lane] 16 bytes
    static constexpr size_t SMEM = 4 * (size_t)SLOT + 2 * HBUF;
    static_assert(2 * SLOT + BM * XP <= SMEM, "the rows of the set-up lie behind the first layer's slots");
    // hidden values rounded between the next chunk's products, where the registers hold two chunks' sums
    static constexpr bool PIPE = C == 128 || RP == 1;
};

template <int C, int RP>
__global__ __launch_bounds__(256 * RP, tw_occ(C, RP)) void transition_wide_kernel(T* out, const T* x, int8_t* xtail, const T* __restrict__ gamma,
                                                                    const T* __restrict__ beta, const T* __restrict__ w1, const T* __restrict__ b1,
                                                                    const T* __restrict__ w2, const T* __restrict__ b2, long M, float eps, int use_touch) {
    typedef Mma<T> MM;
    typedef TwGeo<C, RP> W;
    constexpr int KS1 = C / 16, CT = C / 64, TW_C = C, TW_H = W::H, TW_NCH = W::NCH, TW_SLOT = W::SLOT, TW_XP = W::XP, TW_THREADS = W::THREADS,
                  TW_HBUF = W::HBUF, NLD = TW_SLOT / 16 / TW_THREADS;
    constexpr int NC1 = C / 8, RPR = TW_THREADS / NC1;    // 16-byte columns of a row of W1 (and of x), rows per request of a workgroup
    constexpr bool PIPE = W::PIPE;
    constexpr int LAG = PIPE ? 2 : 1;                     // chunks the second layer is behind
    extern __shared__ __align__(16) unsigned char smem[];
    unsigned char* s_w1 = smem;                           // [2][64 hidden][512 bytes]
    unsigned char* s_w2 = smem + 2 * TW_SLOT;             // [2][256 channels][128 bytes]
    unsigned char* s_h = smem + 4 * TW_SLOT;              // [2][TW_HBUF]
    unsigned char* s_x = s_w2;                            // [128][TW_XP], set-up only
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool first = wave < 2 * RP;
    const int rp = (wave >> 1) & (RP - 1), sub = wave & 1;
    const int l32 = lane & 31, half = lane >> 5;
    const long m0 = (long)blockIdx.x * W::BM;

    // ---- chunk loaders (direct to LDS; lane L of a wave lands at dst + 16 L) ----
    // W1: LDS row rho holds weight row sigma(rho % 32) of its tile, 32 columns of 16 bytes; W2: row tau(rho % 32), 8 columns; columns
    // swizzled within 256 bytes of LDS
    // (request i of a thread: a multiple of 16, or of 32, rows further, where either permutation and swizzle repeat up to tau)
    constexpr int W1P = RPR == 8 ? 2 : 1;                 // eight rows a request: even and odd requests differ
    const T* w1src[W1P];
#pragma unroll
    for (int i = 0; i < W1P; ++i) {
        const int r = tid / NC1 + i * RPR;
        w1src[i] = w1 + (long)tr_sigma(r) * TW_C + (((tid % NC1) ^ (r & 15)) * 8);
    }
    const T* w2src = w2 + (long)((tid / 8 & ~31) + ffk_tau(tid / 8 & 31)) * TW_H + (((tid % 8) ^ ((tid / 16) & 7)) * 8);
    const unsigned lds_base = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)smem;
    // asm: the compiler would order every later LDS read behind these loads
    auto dma = [&](const T* src, unsigned dst) __attribute__((always_inline)) {
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(lds_base + dst) : "memory", "m0");
#pragma clang diagnostic pop
    };
    auto fetch1 = [&](int q) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NLD; ++i) dma(w1src[i % W1P] + ((long)q * TW_HC + i / W1P * W1P * RPR) * TW_C, (q & 1) * TW_SLOT + (i * TW_THREADS + wave * 64) * 16);
    };
    auto fetch2 = [&](int q) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NLD; ++i) dma(w2src + (long)i * (TW_THREADS / 8) * TW_H + q * TW_HC, (2 + (q & 1)) * TW_SLOT + (i * TW_THREADS + wave * 64) * 16);
    };

    // ---- set-up: rows -> LayerNorm in registers -> LDS -> fragments of the first layer's waves ----
    {
        constexpr int NP = W::BM / RPR;
        const int c8 = tid % NC1, r0 = tid / NC1;
        Vec16<T> v[NP];
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            long m = m0 + r0 + RPR * i;
            m = m < M ? m : M - 1;                        // clamped: rows past the end are never stored
            v[i] = ld16(x + m * TW_C + c8 * 8);
        }
        const uint32_t touched = use_touch ? tr_touch(w1, w2, TW_H * TW_C * 2 / 128, TW_THREADS) : 0;
        const Vec16<T> g = ld16(gamma + c8 * 8), b = ld16(beta + c8 * 8);
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            float f[8], s = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                f[e] = (float)v[i].e[e];
                s += f[e];
            }
            const float q = centre8(f, group_sum(s, NC1) * (1.0f / TW_C));
            const float rs = rsqrtf(group_sum(q, NC1) * (1.0f / TW_C) + eps);
            Vec16<T> y;
#pragma unroll
            for (int e = 0; e < 8; ++e) y.e[e] = (T)__builtin_fmaf(f[e] * rs, (float)g.e[e], (float)b.e[e]);
            *reinterpret_cast<Vec16<T>*>(s_x + (r0 + RPR * i) * TW_XP + c8 * 16) = y;
        }
        asm volatile("" ::"v"(touched));
    }
    // The step of chunk q: what this wave asked for has landed, everyone's after the barrier, which also publishes the hidden chunk
    // q - 1 and frees the slots of the step before
    auto step = [&](int q) __attribute__((always_inline)) {
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (q + 1 < TW_NCH) fetch1(q + 1);
        const int k = q + 1 - LAG;                        // read in the step after this one
        if (k >= 0 && k < TW_NCH) fetch2(k);
    };
    // residual (and tail) of four output tiles of one row group, and a finished tile
    const int rg_out = first ? 1 : 0;                     // the row group of the pair this wave finishes
    const long row = m0 + rp * 64 + rg_out * 32 + l32;
    const bool ok = row < M;
    const long o0 = (ok ? row : M - 1) * TW_C + sub * (C / 2) + 16 * half;
    u32x4 rv[CT][2], tv[CT];
    auto request = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < CT; ++c) {
            rv[c][0] = *reinterpret_cast<const u32x4*>(x + o0 + c * 32);
            rv[c][1] = *reinterpret_cast<const u32x4*>(x + o0 + c * 32 + 8);
            if (xtail) tv[c] = *reinterpret_cast<const u32x4*>(xtail + o0 + c * 32);
        }
    };
    auto finish = [&](const f32x16& acc, int c) __attribute__((always_inline)) {
        const long o = o0 + c * 32;
        if (xtail) {           // extended residual stream: the update is added at 24 bits
            float upd[16];
#pragma unroll
            for (int v = 0; v < 16; ++v) upd[v] = (float)(T)acc[v];
            u32x4 h0, h1, tn;
            xs_update16(upd, rv[c][0], rv[c][1], tv[c], h0, h1, tn);
            if (ok) {
                *reinterpret_cast<u32x4*>(out + o) = h0;
                *reinterpret_cast<u32x4*>(out + o + 8) = h1;
                *reinterpret_cast<u32x4*>(xtail + o) = tn;
            }
            return;
        }
        T y[16];
#pragma unroll
        for (int v = 0; v < 16; ++v) y[v] = (T)((float)(T)acc[v] + (float)reinterpret_cast<const T*>(&rv[c][v >> 3])[v & 7]);
        if (ok) {
            *reinterpret_cast<u32x4*>(out + o) = *reinterpret_cast<const u32x4*>(&y[0]);
            *reinterpret_cast<u32x4*>(out + o + 8) = *reinterpret_cast<const u32x4*>(&y[8]);
        }
    };
    unsigned char* xch = smem + (wave & (2 * RP - 1)) * (CT * 4096) + lane * 16;          // sums handed over: [row pair, half][tile][a][lane] 16 bytes

    if (first) {
        // ---- first layer: hidden tile sub of a chunk, rows 64 rp .. 64 rp + 63 ----
        uint32_t bw[TW_NCH / 2];                          // bias of this lane's weight row, two chunks a word
        {
            const uint16_t* bp = reinterpret_cast<const uint16_t*>(b1) + sub * 32 + tr_sigma(l32);
#pragma unroll
            for (int i = 0; i < TW_NCH / 2; ++i) bw[i] = (uint32_t)bp[2 * i * TW_HC] | ((uint32_t)bp[(2 * i + 1) * TW_HC] << 16);
        }
        lds_barrier();                                    // the rows are there
        fetch1(0);
        bf16x8 xf[2][KS1];
#pragma unroll
        for (int rg = 0; rg < 2; ++rg)
#pragma unroll
            for (int ks = 0; ks < KS1; ++ks)
                xf[rg][ks] = *reinterpret_cast<const bf16x8*>(s_x + (rp * 64 + rg * 32 + l32) * TW_XP + ks * 32 + half * 16);
        int w1off[8];
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) w1off[ks] = (sub * 32 + l32) * (2 * C) + (((2 * ks + half) ^ (l32 & 15)) << 4);
        u32x4 onew = {half == 0 ? 0x3F80u : 0u, 0, 0, 0};  // one in the first K of the step
        const bf16x8 one = *reinterpret_cast<const bf16x8*>(&onew);
        // products of chunk q into h; between them the hidden values of chunk q - 1 (old) are rounded and handed over
        auto convert = [&](const f32x16& v, int q, int rg, int j) __attribute__((always_inline)) {
            typedef float f32x2 __attribute__((ext_vector_type(2)));
            typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
            typedef short s16x2 __attribute__((ext_vector_type(2)));
            const s16x2 zero = {0, 0};                    // relu on the packed bf16 patterns (see above)
            u32x4 w;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const f32x2 pr = {v[8 * j + 2 * t], v[8 * j + 2 * t + 1]};
                const bf16x2 r = __builtin_convertvector(pr, bf16x2);
                w[t] = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(s16x2, r), zero));
            }
            *reinterpret_cast<u32x4*>(s_h + (q & 1) * TW_HBUF + (rp * 8 + sub * 2 + rg * 4 + j) * 1024 + lane * 16) = w;
        };
        auto chunk = [&](int q, uint32_t bias, f32x16 (&h)[2], const f32x16 (&old)[2], bool has_old) __attribute__((always_inline)) {
            step(q);
            const unsigned char* wa = s_w1 + (q & 1) * TW_SLOT;
            u32x4 biasw = {half == 0 ? bias & 0xFFFFu : 0u, 0, 0, 0};
            bf16x8 wf[2][2];
#pragma unroll
            for (int i = 0; i < 2; ++i) wf[0][i] = *reinterpret_cast<const bf16x8*>(wa + w1off[i]);
#pragma unroll
            for (int rg = 0; rg < 2; ++rg) {
#pragma unroll
                for (int v = 0; v < 16; ++v) h[rg][v] = 0.0f;
                MM::mma(h[rg], *reinterpret_cast<const bf16x8*>(&biasw), one);
            }
#pragma unroll
            for (int g = 0; g < KS1 / 2; ++g) {
                if (g + 1 < KS1 / 2) {
#pragma unroll
                    for (int i = 0; i < 2; ++i) wf[(g + 1) & 1][i] = *reinterpret_cast<const bf16x8*>(wa + w1off[(2 * g + 2 + i) & 7] + ((g + 1) >> 2) * 256);
                }
                __builtin_amdgcn_sched_barrier(0);
                if (has_old && (KS1 == 8 || !(g & 1))) convert(old[KS1 == 8 ? g >> 1 : g >> 2], q - 1, KS1 == 8 ? g >> 1 : g >> 2, KS1 == 8 ? g & 1 : (g >> 1) & 1);
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    MM::mma(h[0], wf[g & 1][i], xf[0][2 * g + i]);
                    MM::mma(h[1], wf[g & 1][i], xf[1][2 * g + i]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        f32x16 ha[2], hb[2];
        auto hand_over = [&](const f32x16 (&h)[2], int q) __attribute__((always_inline)) {
#pragma unroll
            for (int g = 0; g < 4; ++g) convert(h[g >> 1], q, g >> 1, g & 1);
        };
        if constexpr (PIPE) {
            chunk(0, bw[0], ha, hb, false);
            for (int q = 1; q < TW_NCH - 1; q += 2) {
                chunk(q, bw[0] >> 16, hb, ha, true);
#pragma unroll
                for (int i = 0; i + 1 < TW_NCH / 2; ++i) bw[i] = bw[i + 1];
                chunk(q + 1, bw[0], ha, hb, true);
            }
            chunk(TW_NCH - 1, bw[0] >> 16, hb, ha, true);
            step(TW_NCH);
            hand_over(hb, TW_NCH - 1);
        } else {
            for (int q = 0; q < TW_NCH; q += 2) {
                const uint32_t b = bw[0];
#pragma unroll
                for (int i = 0; i + 1 < TW_NCH / 2; ++i) bw[i] = bw[i + 1];
                chunk(q, b, ha, ha, false);
                hand_over(ha, q);
                chunk(q + 1, b >> 16, ha, ha, false);
                hand_over(ha, q + 1);
            }
        }
        step(TW_NCH + LAG - 1);
        request();                                        // arrives behind the second layer's last chunk
        lds_barrier();                                    // the slots are free: nobody reads them, no request is on its way
        lds_barrier();                                    // the sums are there
#pragma unroll
        for (int c = 0; c < CT; ++c) {
            f32x16 acc;
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                const f32x4 p = *reinterpret_cast<const f32x4*>(xch + (c * 4 + a) * 1024);
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[4 * a + e] = p[e];
            }
            finish(acc, c);
        }
    } else {
        // ---- second layer: output tiles 4 sub .. 4 sub + 3 ----
        f32x16 acc[2][CT];                                // out^T tiles: channels 32 c + 16 half + v, row l32
#pragma unroll
        for (int c = 0; c < CT; ++c) {                     // start from b2: the epilogue has no bias to add
            const T* bp = b2 + sub * (C / 2) + c * 32 + 16 * half;
            const Vec16<T> v0 = ld16(bp), v1 = ld16(bp + 8);
#pragma unroll
            for (int v = 0; v < 8; ++v) {
                acc[0][c][v] = acc[1][c][v] = (float)v0.e[v];
                acc[0][c][8 + v] = acc[1][c][8 + v] = (float)v1.e[v];
            }
        }
        int w2off[4];
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) w2off[ks] = (sub * (C / 2) + l32) * 128 + (((2 * ks + half) ^ ((l32 >> 1) & 7)) << 4);
        lds_barrier();
        fetch1(0);
        step(0);
        if (PIPE) step(1);
        auto chunk = [&](int q) __attribute__((always_inline)) {
            step(q);
            const unsigned char* wb = s_w2 + ((q - LAG) & 1) * TW_SLOT;
            const unsigned char* hs = s_h + ((q - LAG) & 1) * TW_HBUF + rp * 8192 + lane * 16;
            bf16x8 hf[2][4], wf[2][CT];
#pragma unroll
            for (int c = 0; c < CT; ++c) wf[0][c] = *reinterpret_cast<const bf16x8*>(wb + c * 4096 + w2off[0]);
#pragma unroll
            for (int ks = 0; ks < 4; ++ks)
#pragma unroll
                for (int rg = 0; rg < 2; ++rg) hf[rg][ks] = *reinterpret_cast<const bf16x8*>(hs + (rg * 4 + ks) * 1024);
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                if (ks + 1 < 4) {
#pragma unroll
                    for (int c = 0; c < CT; ++c) wf[(ks + 1) & 1][c] = *reinterpret_cast<const bf16x8*>(wb + c * 4096 + w2off[ks + 1]);
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int c = 0; c < CT; ++c) {
                    MM::mma(acc[0][c], wf[ks & 1][c], hf[0][ks]);
                    MM::mma(acc[1][c], wf[ks & 1][c], hf[1][ks]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        for (int q = LAG; q < TW_NCH + LAG; ++q) chunk(q);
        request();
        lds_barrier();
#pragma unroll
        for (int c = 0; c < CT; ++c)
#pragma unroll
            for (int a = 0; a < 4; ++a)
                *reinterpret_cast<f32x4*>(xch + (c * 4 + a) * 1024) = f32x4{acc[1][c][4 * a], acc[1][c][4 * a + 1], acc[1][c][4 * a + 2], acc[1][c][4 * a + 3]};
        lds_barrier();
#pragma unroll
        for (int c = 0; c < CT; ++c) finish(acc[0][c], c);
    }
}

}  // namespace

extern "C" int ffk_transition_fused(void* out, const void* x, void* xtail, const void* gamma, const void* beta, const void* w1,
                                    const void* b1, const void* w2, const void* b2, int64_t M, int64_t C, int64_t hidden,
                                    float eps, int dtype, void* stream) {
    FFK_REQUIRE(out && x && gamma && beta && w1 && b1 && w2 && b2, FFK_ERR_NULL, "ffk_transition_fused: null pointer");
    FFK_REQUIRE(dtype == FFK_BF16, FFK_ERR_DTYPE, "ffk_transition_fused: bf16 only (dtype tag %d)", dtype);
    FFK_REQUIRE((C == 128 || C == 256) && hidden == 4 * C, FFK_ERR_UNSUPPORTED,
                "ffk_transition_fused: built for 128 -> 512 -> 128 and 256 -> 1024 -> 256, got %ld -> %ld", (long)C, (long)hidden);
    FFK_REQUIRE(M > 0 && M < (1L << 31) * (long)TR_BM, FFK_ERR_SHAPE, "ffk_transition_fused: bad row count %ld", (long)M);
    FFK_REQUIRE(ffk_aligned16(out) && ffk_aligned16(x) && ffk_aligned16(gamma) && ffk_aligned16(beta) && ffk_aligned16(w1) &&
                    ffk_aligned16(w2) && ffk_aligned16(b2) && ffk_aligned16(xtail),
                FFK_ERR_ALIGN, "ffk_transition_fused: buffers must be 16-byte aligned");
    // 256 channels: one row pair per workgroup up to one workgroup per CU, two from there on.  128 channels the same, and above
    // 32 768 rows the kernel with three workgroups per CU.  The lines of the weights are touched first where enough workgroups share
    // the work (with one workgroup per XCD it costs 4 us) and more than the first round of them gains by it.
    typedef std::integral_constant<int, 1> One;
    typedef std::integral_constant<int, 2> Two;
    typedef std::integral_constant<int, 128> C128;
    typedef std::integral_constant<int, 256> C256;
    auto wide = [&](auto c, auto rp) {
        constexpr int CC = decltype(c)::value, RP = decltype(rp)::value;
        typedef TwGeo<CC, RP> W;
        static FfkLdsReservation lds_reserved;
        const int rc = ffk_reserve_lds(lds_reserved, (const void*)transition_wide_kernel<CC, RP>, W::SMEM, "ffk_transition_fused");
        if (rc != FFK_OK) return rc;
        const unsigned grid = (unsigned)ffk_cdiv(M, W::BM);
        transition_wide_kernel<CC, RP><<<grid, W::THREADS, W::SMEM, (hipStream_t)stream>>>(
            (T*)out, (const T*)x, (int8_t*)xtail, (const T*)gamma, (const T*)beta, (const T*)w1, (const T*)b1, (const T*)w2, (const T*)b2,
            (long)M, eps, RP == 1 ? grid >= 64 : grid > 256);
        return ffk_check_launch("ffk_transition_fused");
    };
    if (C == 256) return M <= 64 * 256 ? wide(C256(), One()) : wide(C256(), Two());
    if (M <= 64 * 256) return wide(C128(), One());
    if (M <= 128 * 256) return wide(C128(), Two());
    const unsigned grid = (unsigned)ffk_cdiv(M, TR_BM);
    const bool deep = grid <= 256 + 128;                     // at most ~one workgroup on most CUs: four-slot rings
    auto fused = [&](auto slots) {
        constexpr int NS = decltype(slots)::value;
        static FfkLdsReservation lds_reserved;
        const int rc = ffk_reserve_lds(lds_reserved, (const void*)transition_fused_kernel<NS>, TrGeo<NS>::SMEM, "ffk_transition_fused");
        if (rc != FFK_OK) return rc;
        transition_fused_kernel<NS><<<grid, TR_THREADS, TrGeo<NS>::SMEM, (hipStream_t)stream>>>(
            (T*)out, (const T*)x, (int8_t*)xtail, (const T*)gamma, (const T*)beta, (const T*)w1, (const T*)b1, (const T*)w2, (const T*)b2,
            (long)M, eps);
        return ffk_check_launch("ffk_transition_fused");
    };
    return deep ? fused(std::integral_constant<int, 4>()) : fused(Two());
}
