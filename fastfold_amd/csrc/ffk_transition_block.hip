// Fused transition with the weights in fragment order (see ffk_transition_block in include/ffk.h):
//     out = x + W2 . relu( W1 . LayerNorm(x) + b1 ) + b2        (C -> F C -> C channels, bf16)
//
// A workgroup of eight waves owns 32 RT rows: normalised once into LDS, the hidden layer in chunks of (at most) 256 channels, the update
// through LDS back to the rows.  In the first layer a wave owns a block of 32 hidden channels, in the second one of 32 output channels;
// where there are fewer blocks than waves, several waves own one and divide the row tiles.  A weight fragment goes from the cache into
// the registers of the wave that multiplies by it, requested a layer of a chunk ahead (16 KB a wave, 128 KB a CU in flight); only
// the rows and the hidden chunk are read from LDS.  The accumulators of the first layer are the second's operand as they stand (the
// rows of W1 are packed so that a lane's are consecutive hidden channels), so the hidden values cross LDS in whole fragments.  Sums are
// begun and added as in ffk_transition_fused, to the bit: a caller may cut its rows anywhere, whichever kernel a piece goes to.
//
// What bounds it: at 256 channels the weights - 1 MB a workgroup, which a CU gets at 60 KB/us where the second-level cache has them and at
// half that where it does not; 64 rows are multiplied by them in 8 us, 128 in 16.  At 64 channels, memory (393 216 rows: 151 MB with
// the residual in 53 us).  us a launch, ffk_transition_fused (64 channels: projection and product with the hidden layer in memory) -> here:
//   256 channels: 2 048 rows 22.6 -> 16.9, 12 288 24.2 -> 19.7, 32 768 41.0 -> 40.7, 131 072 157 -> 152; between the launches of a
//     stack, its weights new to the cache: 12 288 29.2 -> 22.8, 32 768 43.0 -> 40.2, 131 072 168 -> 158
//   128 channels: 1 024 rows 8.6 -> 7.4, 9 216 9.5 -> 8.3, 16 384 10.0 -> 9.0; but 110 592 45 -> 50, 1 048 576 376 -> 430: three
//     workgroups of the other kernel share a CU there and cover each other's waits
//   64 channels, 4 x: 8 192 rows 11.7 -> 5.4, 98 304 42 -> 15.5, 393 216 133 -> 53;  2 x: 25 600 16.5 -> 5.1, 102 400 33 -> 11.8
#include "ffk_rowblock.h"

namespace {

struct TbArgs : RbRows {
    const T* w1;             // [F C / 32][C / 16][64][8]
    const T* b1;             // [F C]
    const T* w2;             // [C / 32][F C / 16][64][8]
    const T* b2;             // [C]
    long M;
};

template <int C, int F, int RT> struct TbGeo {
    static constexpr int H = F * C, HB = H / 32, NB = C / 32;
    static constexpr int CB = HB < 8 ? HB : 8;       // hidden blocks of a chunk
    static constexpr int NCH = HB / CB;              // chunks
    static constexpr int WH = 8 / CB, T1 = RT / WH;  // waves per hidden block, row tiles of each
    static constexpr int WO = 8 / NB, T2 = RT / WO;  // waves per output block, row tiles of each
    static constexpr int KS1 = C / 16, KS2 = 2 * CB; // K steps of the first layer, of the second per chunk
    static constexpr int XP = C * 2 + 16;
    static constexpr size_t ROWS = (size_t)RT * 32 * XP, HID = (size_t)RT * CB * 2048;
    static constexpr bool TWICE = NCH > 1 && ROWS + 2 * HID + 4 * H <= 160 * 1024;      // two buffers for hidden chunks
    static constexpr size_t SMEM = ROWS + (TWICE ? 2 : 1) * HID + 4 * H;
    static_assert(T1 >= 1 && T2 >= 1 && RT % WH == 0 && RT % WO == 0 && SMEM <= 160 * 1024, "geometry");
};

template <int C, int F, int RT, int OCC>
__global__ __launch_bounds__(512, OCC) void transition_block_kernel(TbArgs a) {
    typedef TbGeo<C, F, RT> G;
    constexpr int KS1 = G::KS1, KS2 = G::KS2, T1 = G::T1, T2 = G::T2, NCH = G::NCH, CB = G::CB, XP = G::XP;
    extern __shared__ __align__(16) unsigned char tb_smem[];
    unsigned char* s_x = tb_smem;                    // [32 RT][XP]; at the end the updates
    T* s_h = reinterpret_cast<T*>(tb_smem + G::ROWS);        // [1 or 2][RT][KS2][64][8]
    float* s_b1 = reinterpret_cast<float*>(tb_smem + G::SMEM - 4 * G::H);

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    const int hb = wave % CB, t1 = wave / CB * T1;   // hidden block within a chunk and first row tile, first layer
    const int ob = wave % G::NB, t2 = wave / G::NB * T2;     // output block and first row tile, second layer
    const long m0 = (long)blockIdx.x * (32 * RT);
    a.n = a.M - m0 < 32 * RT ? (int)(a.M - m0) : 32 * RT;

    const T* p1 = a.w1 + ((long)hb * KS1) * 512 + lane * 8;                  // chunk q: + q CB KS1 512
    const T* p2 = a.w2 + ((long)ob * (G::H / 16)) * 512 + lane * 8;          // chunk q: + q KS2 512
    bf16x8 w1[KS1], w2[KS2];
#pragma unroll
    for (int i = 0; i < KS1; ++i) w1[i] = MM::ld(p1 + i * 512);
    for (int i = tid; i < G::H; i += 512) s_b1[i] = (float)a.b1[i];
    rb_normalise<C, RT>(a, a.x + m0 * C, s_x, RT, wave, lane);
    lds_barrier();

    f32x16 acc2[T2];                                 // from b2 on
    {
        const Vec16<T> v0 = ld16(a.b2 + ob * 32 + 16 * half), v1 = ld16(a.b2 + ob * 32 + 16 * half + 8);
#pragma unroll
        for (int t = 0; t < T2; ++t)
#pragma unroll
            for (int v = 0; v < 8; ++v) {
                acc2[t][v] = (float)v0.e[v];
                acc2[t][8 + v] = (float)v1.e[v];
            }
    }
    const unsigned char* xp = s_x + (t1 * 32 + l32) * XP + half * 16;
#pragma unroll
    for (int q = 0; q < NCH; ++q) {
        // ---- first layer; the second layer's fragments are requested meanwhile ----
        f32x16 h[T1];
        {
            // registers 0 .. 7: hidden 8 half + 0 .. 7 of the block, registers 8 .. 15: 16 + 8 half + 0 .. 7
            const float* bp = s_b1 + (q * CB + hb) * 32 + 8 * half;
            f32x16 bias;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const f32x4 b = *reinterpret_cast<const f32x4*>(bp + (g >> 1) * 16 + (g & 1) * 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) bias[4 * g + e] = b[e];
            }
#pragma unroll
            for (int t = 0; t < T1; ++t) h[t] = bias;
        }
        constexpr int R2 = (KS2 + KS1 - 1) / KS1;    // requests per step
#pragma unroll
        for (int ks = 0; ks < KS1; ++ks) {
            const bf16x8 c = w1[ks];
#pragma unroll
            for (int i = ks * R2; i < (ks + 1) * R2 && i < KS2; ++i) w2[i] = MM::ld(p2 + (long)(q * KS2 + i) * 512);
#pragma unroll
            for (int t = 0; t < T1; ++t) MM::mma(h[t], c, *reinterpret_cast<const bf16x8*>(xp + t * 32 * XP + ks * 32));
            __builtin_amdgcn_sched_barrier(0);
        }
        T* hd = s_h + (G::TWICE ? (q & 1) * (RT * KS2 * 512) : 0);
        u32x4 hw[T1][2];
#pragma unroll
        for (int t = 0; t < T1; ++t)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                typedef float f32x2 __attribute__((ext_vector_type(2)));
                typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
                typedef short s16x2 __attribute__((ext_vector_type(2)));
                const s16x2 zero = {0, 0};            // relu on the packed bf16 patterns: negative numbers are negative integers
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const f32x2 pr = {h[t][8 * j + 2 * e], h[t][8 * j + 2 * e + 1]};
                    hw[t][j][e] = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(
                        __builtin_bit_cast(s16x2, __builtin_convertvector(pr, bf16x2)), zero));
                }
            }
        if (!G::TWICE && q > 0) lds_barrier();       // nobody reads the chunk before any more
#pragma unroll
        for (int t = 0; t < T1; ++t)
#pragma unroll
            for (int j = 0; j < 2; ++j) *reinterpret_cast<u32x4*>(hd + ((t1 + t) * KS2 + 2 * hb + j) * 512 + lane * 8) = hw[t][j];
        lds_barrier();
        // ---- second layer; the next chunk's first-layer fragments are requested meanwhile ----
        constexpr int R1 = (KS1 + KS2 - 1) / KS2;
#pragma unroll
        for (int f = 0; f < KS2; ++f) {
            const bf16x8 c = w2[f];
            if (q + 1 < NCH) {
#pragma unroll
                for (int i = f * R1; i < (f + 1) * R1 && i < KS1; ++i) w1[i] = MM::ld(p1 + ((long)(q + 1) * CB * KS1 + i) * 512);
            }
#pragma unroll
            for (int t = 0; t < T2; ++t) MM::mma(acc2[t], c, MM::ld(hd + ((t2 + t) * KS2 + f) * 512 + lane * 8));
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    RbUpdate<C, RT> rows;
    rows.fetch(a, m0 * C, RT, wave, rb_lane(lane));
#pragma unroll
    for (int t = 0; t < T2; ++t) rb_put(s_x + ((t2 + t) * 32 + l32) * XP + ob * 64 + half * 32, acc2[t], nullptr);
    lds_barrier();
    rows.store(a, s_x, m0 * C, RT, wave, rb_lane(lane));
}

template <int C, int F, int RT, int OCC> int tb_launch(const TbArgs& a, hipStream_t st) {
    typedef TbGeo<C, F, RT> G;
    static FfkLdsReservation lds_reserved;
    const int rc = ffk_reserve_lds(lds_reserved, (const void*)transition_block_kernel<C, F, RT, OCC>, G::SMEM, "ffk_transition_block");
    if (rc != FFK_OK) return rc;
    transition_block_kernel<C, F, RT, OCC><<<dim3((unsigned)ffk_cdiv(a.M, 32 * RT)), 512, G::SMEM, st>>>(a);
    return ffk_check_launch("ffk_transition_block");
}

}  // namespace

extern "C" int ffk_transition_block(void* out, const void* x, void* xtail, const void* gamma, const void* beta, const void* w1,
                                    const void* b1, const void* w2, const void* b2, int64_t M, int64_t C, int64_t hidden, float eps,
                                    int dtype, void* stream) {
    FFK_REQUIRE(out && x && gamma && beta && w1 && b1 && w2 && b2, FFK_ERR_NULL, "ffk_transition_block: null pointer");
    FFK_REQUIRE(dtype == FFK_BF16, FFK_ERR_DTYPE, "ffk_transition_block: bf16 only (dtype tag %d)", dtype);
    FFK_REQUIRE(((C == 64 || C == 128 || C == 256) && hidden == 4 * C) || (C == 64 && hidden == 128), FFK_ERR_UNSUPPORTED,
                "ffk_transition_block: built for 64, 128 and 256 channels with four times as many hidden ones and 64 -> 128, got %ld -> %ld",
                (long)C, (long)hidden);
    FFK_REQUIRE(M > 0 && M < (1L << 36), FFK_ERR_SHAPE, "ffk_transition_block: bad row count %ld", (long)M);
    FFK_REQUIRE(ffk_aligned16(out) && ffk_aligned16(x) && ffk_aligned16(xtail) && ffk_aligned16(gamma) && ffk_aligned16(beta) &&
                    ffk_aligned16(w1) && ffk_aligned16(b1) && ffk_aligned16(w2) && ffk_aligned16(b2),
                FFK_ERR_ALIGN, "ffk_transition_block: buffers must be 16-byte aligned");
    const TbArgs a = {{(T*)out, (const T*)x, (int8_t*)xtail, (const T*)gamma, (const T*)beta, nullptr, (long)C, 0, eps},
                      (const T*)w1, (const T*)b1, (const T*)w2, (const T*)b2, (long)M};
    hipStream_t st = (hipStream_t)stream;
    // 64 rows a workgroup as long as every one has a CU, 128 from there on (fewer weights per row).  The modules send more than 16 384 rows
    // of 128 channels to ffk_transition_fused (figures above); a caller that holds only these weights is served as well
    if (C == 256) return M <= 64 * 256 ? tb_launch<256, 4, 2, 2>(a, st) : tb_launch<256, 4, 4, 2>(a, st);
    if (C == 128) return M <= 64 * 256 ? tb_launch<128, 4, 2, 2>(a, st) : tb_launch<128, 4, 4, 2>(a, st);
    return hidden == 256 ? tb_launch<64, 4, 4, 2>(a, st) : tb_launch<64, 2, 4, 4>(a, st);
}
