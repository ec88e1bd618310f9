// Re-tiling of a strided [B2, H, N, D <= 32] tensor into the 32 x 32 operand tiles of the attention kernels
// (FFK_TILE_QK or FFK_TILE_V order, see ffk_common.h), in one pass: rows past N and channels past D become zero,
// and an optional factor (the log2(e) / sqrt(d) of the q operand) is applied in fp32 before the rounding.  It serves
// the stand-alone attention operator and its backward pass, whose operands come as plain tensors; inside the
// inference block the projection kernel writes these tiles itself.
#include "ffk_common.h"

namespace {

template <typename T>
__global__ __launch_bounds__(256) void tile_pack_kernel(T* __restrict__ dst, const T* __restrict__ src, long tiles,
                                                       int H, int NT, int N, int D, long s_b, long s_h, long s_n,
                                                       float scale, int kind, int vec_ok) {
    constexpr int VEC = DT<T>::VEC;
    constexpr int NV = 16 / VEC;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const long item = (long)blockIdx.x * 4 + wave;
    if (item >= tiles) return;
    const int nt = (int)(item % NT);
    const long bh = item / NT;
    const int h = (int)(bh % H);
    const long b = bh / H;
    const T* base = src + b * s_b + (long)h * s_h;
    T* out = dst + (item << 10) + lane * 16;
    Vec16<T> o[NV];
    if (kind == FFK_TILE_QK) {
        // lane (n = lane / 2 ... ) of the tile: element (n32, d) at (d / 16) * 512 + n32 * 16 + d % 16, so the lane
        // that owns elements [lane * 16, lane * 16 + 16) holds channels 16 * (lane / 32) .. + 15 of row lane % 32
        const int n = nt * 32 + (lane & 31);
        const int d0 = (lane >> 5) * 16;
        const T* p = base + (long)n * s_n + d0;
        if (vec_ok && n < N && d0 + 16 <= D) {
#pragma unroll
            for (int i = 0; i < NV; ++i) o[i] = ld16_nt(p + i * VEC);
            if (scale != 1.0f) {
#pragma unroll
                for (int i = 0; i < NV; ++i)
#pragma unroll
                    for (int e = 0; e < VEC; ++e) o[i].e[e] = DT<T>::from_f(DT<T>::to_f(o[i].e[e]) * scale);
            }
        } else {
#pragma unroll
            for (int i = 0; i < NV; ++i)
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    const int d = d0 + i * VEC + e;
                    o[i].e[e] = DT<T>::from_f((n < N && d < D) ? DT<T>::to_f(p[i * VEC + e]) * scale : 0.0f);
                }
        }
    } else {
        // accumulator order: lane (kg = lane / 32, col = lane % 32) holds rows 8a + 4kg + b, a, b = 0..3, at 4a + b
        const int col = lane & 31, kg = lane >> 5;
#pragma unroll
        for (int i = 0; i < NV; ++i)
#pragma unroll
            for (int e = 0; e < VEC; ++e) {
                const int idx = i * VEC + e;
                const int n = nt * 32 + 8 * (idx >> 2) + 4 * kg + (idx & 3);
                o[i].e[e] = DT<T>::from_f((n < N && col < D) ? DT<T>::to_f(base[(long)n * s_n + col]) * scale : 0.0f);
            }
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) st16_nt(out + i * VEC, o[i]);
}

template <typename T>
int tile_pack_launch(void* dst, const void* src, long B2, long H, long N, long D, long s_b, long s_h, long s_n,
                     float scale, int kind, hipStream_t st) {
    const long NT = (N + 31) / 32;
    const long tiles = B2 * H * NT;
    const long grid = (tiles + 3) / 4;
    FFK_REQUIRE(grid < (1L << 31), FFK_ERR_SHAPE, "ffk_tile_pack: too many tiles for one launch");
    constexpr int VEC = DT<T>::VEC;
    const int vec_ok = ffk_aligned16(src) && s_b % VEC == 0 && s_h % VEC == 0 && s_n % VEC == 0;
    tile_pack_kernel<T><<<(unsigned)grid, 256, 0, st>>>((T*)dst, (const T*)src, tiles, (int)H, (int)NT, (int)N, (int)D,
                                                       s_b, s_h, s_n, scale, kind, vec_ok);
    return ffk_check_launch("ffk_tile_pack");
}


// ------------------------------------------------------------------------- all operands of an attention in one launch ----
// Every source tile is read once, 32 contiguous bytes per lane, and written in the order(s) asked for: FFK_TILE_QK is how the
// lanes hold it, FFK_TILE_V its transpose through a wave's own LDS tile.  blockIdx.y is the operand; the last one may be the
// pair bias.  Bound by the bytes: seven tiles of 16.8 MB from five at [128, 8, 256, 32] bf16 (a launch per tile order took
// 12.6 us each, the FFK_TILE_V ones on sixteen two-byte loads per lane).
constexpr int PACK_PITCH_BYTES = 16;            // LDS row: 32 elements + 16 bytes, keeps 16-byte writes aligned

template <typename T>
__global__ __launch_bounds__(256) void attention_pack_kernel(const ffk_pack_desc d, int NT, int vec_mask) {
    constexpr int VEC = DT<T>::VEC, NV = 16 / VEC, PITCH = 32 + PACK_PITCH_BYTES / (int)sizeof(T);
    __shared__ __align__(16) T lds[4][32 * PITCH];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l32 = lane & 31, half = lane >> 5;
    const long item = (long)blockIdx.x * 4 + wave;
    const int job = blockIdx.y;
    const int H = d.H, N = d.N, D = d.D;
    if (job == d.n) {                           // pair bias: element (k, q) at [q / 16][k][q % 16], from rows of keys
        if (item >= (long)H * NT * NT) return;
        const int kt = (int)(item % NT), qt = (int)((item / NT) % NT), h = (int)(item / ((long)NT * NT));
        const T* p = (const T*)d.bias + ((long)h * N + qt * 32 + 16 * half) * N + kt * 32 + l32;
        T* out = (T*)d.bias_t + (item << 10) + lane * 16;
        const int rows = N - qt * 32 - 16 * half;
        const bool in = kt * 32 + l32 < N;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            Vec16<T> o;
#pragma unroll
            for (int e = 0; e < VEC; ++e) {
                const int q = i * VEC + e;
                o.e[e] = DT<T>::from_f(in && q < rows ? DT<T>::to_f(p[(long)q * N]) * d.bias_scale : 0.0f);
            }
            st16(out + i * VEC, o);
        }
        return;
    }
    if (item >= (long)d.B2 * H * NT) return;
    const ffk_pack_job& j = d.job[job];
    const int nt = (int)(item % NT), n = nt * 32 + l32, d0 = 16 * half;
    const long bh = item / NT;
    const int h = (int)(bh % H);
    const long b = bh / H;
    auto load = [&](const void* src, long s_b, long s_h, long s_n, bool vec, Vec16<T>* o) {
        const T* p = (const T*)src + b * s_b + (long)h * s_h + (long)n * s_n + d0;
        if (vec && n < N && d0 + 16 <= D) {
#pragma unroll
            for (int i = 0; i < NV; ++i) o[i] = ld16_nt(p + i * VEC);
        } else {
#pragma unroll
            for (int i = 0; i < NV; ++i)
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    const bool in = n < N && d0 + i * VEC + e < D;
                    o[i].e[e] = in ? p[i * VEC + e] : DT<T>::from_f(0.0f);
                }
        }
    };
    Vec16<T> v[NV];
    if (j.tiled) {                              // already in FFK_TILE_QK order
#pragma unroll
        for (int i = 0; i < NV; ++i) v[i] = ld16_nt((const T*)j.src + (item << 10) + lane * 16 + i * VEC);
    } else {
        load(j.src, j.s_b, j.s_h, j.s_n, (vec_mask >> job) & 1, v);
    }
    if (j.dsum) {                               // sum over the channels of this operand times another
        Vec16<T> o[NV];
        load(j.other, j.o_sb, j.o_sh, j.o_sn, (vec_mask >> (8 + job)) & 1, o);
        float t = 0.0f;
#pragma unroll
        for (int i = 0; i < NV; ++i)
#pragma unroll
            for (int e = 0; e < VEC; ++e) t += DT<T>::to_f(v[i].e[e]) * DT<T>::to_f(o[i].e[e]);
        t += lane_xor<32>(t);
        if (half == 0) j.dsum[item * 32 + l32] = t;
    }
    if (j.scale != 1.0f) {
#pragma unroll
        for (int i = 0; i < NV; ++i)
#pragma unroll
            for (int e = 0; e < VEC; ++e) v[i].e[e] = DT<T>::from_f(DT<T>::to_f(v[i].e[e]) * j.scale);
    }
    if (j.qk) {
#pragma unroll
        for (int i = 0; i < NV; ++i) st16((T*)j.qk + (item << 10) + lane * 16 + i * VEC, v[i]);
    }
    if (j.acc) {
        T* t = lds[wave];                       // the wave's own tile: its LDS operations complete in order, no barrier
#pragma unroll
        for (int i = 0; i < NV; ++i) *reinterpret_cast<Vec16<T>*>(t + l32 * PITCH + d0 + i * VEC) = v[i];
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            Vec16<T> o;
#pragma unroll
            for (int e = 0; e < VEC; ++e) {
                const int idx = i * VEC + e;
                o.e[e] = t[(8 * (idx >> 2) + 4 * half + (idx & 3)) * PITCH + l32];
            }
            st16((T*)j.acc + (item << 10) + lane * 16 + i * VEC, o);
        }
    }
}

template <typename T>
int attention_pack_launch(const ffk_pack_desc& d, hipStream_t st) {
    const long NT = (d.N + 31) / 32;
    const long tiles = (long)d.B2 * d.H * NT, btiles = d.bias ? d.H * NT * NT : 0;
    const long grid = ((tiles > btiles ? tiles : btiles) + 3) / 4;
    FFK_REQUIRE(grid < (1L << 31), FFK_ERR_SHAPE, "ffk_attention_pack: too many tiles for one launch");
    constexpr int VEC = DT<T>::VEC;
    int vec = 0;
    for (int i = 0; i < d.n; ++i) {
        const ffk_pack_job& j = d.job[i];
        if (ffk_aligned16(j.src) && j.s_b % VEC == 0 && j.s_h % VEC == 0 && j.s_n % VEC == 0) vec |= 1 << i;
        if (ffk_aligned16(j.other) && j.o_sb % VEC == 0 && j.o_sh % VEC == 0 && j.o_sn % VEC == 0) vec |= 256 << i;
    }
    attention_pack_kernel<T><<<dim3((unsigned)grid, (unsigned)(d.n + (d.bias ? 1 : 0))), 256, 0, st>>>(d, (int)NT, vec);
    return ffk_check_launch("ffk_attention_pack");
}

}  // namespace

extern "C" int ffk_tile_pack(void* dst, const void* src, int64_t B2, int64_t H, int64_t N, int64_t D, int64_t s_b,
                             int64_t s_h, int64_t s_n, float scale, int kind, int dtype, void* stream) {
    FFK_REQUIRE(dst && src, FFK_ERR_NULL, "ffk_tile_pack: null pointer");
    FFK_REQUIRE(B2 > 0 && H > 0 && H < 65536 && N > 0 && N < (1 << 24) && D > 0 && D <= 32, FFK_ERR_SHAPE,
                "ffk_tile_pack: bad shape B2=%ld H=%ld N=%ld D=%ld", (long)B2, (long)H, (long)N, (long)D);
    FFK_REQUIRE(kind == FFK_TILE_QK || kind == FFK_TILE_V, FFK_ERR_UNSUPPORTED,
                "ffk_tile_pack: tile kind %d (FFK_TILE_QK and FFK_TILE_V are built)", kind);
    FFK_REQUIRE(ffk_aligned16(dst), FFK_ERR_ALIGN, "ffk_tile_pack: dst must be 16-byte aligned");
    hipStream_t st = (hipStream_t)stream;
    switch (dtype) {
        case FFK_BF16: return tile_pack_launch<bf16_t>(dst, src, B2, H, N, D, s_b, s_h, s_n, scale, kind, st);
        case FFK_F16: return tile_pack_launch<f16_t>(dst, src, B2, H, N, D, s_b, s_h, s_n, scale, kind, st);
        case FFK_F32: return tile_pack_launch<float>(dst, src, B2, H, N, D, s_b, s_h, s_n, scale, kind, st);
        default: return ffk_fail(FFK_ERR_DTYPE, "ffk_tile_pack: unsupported dtype tag %d", dtype);
    }
}

extern "C" int ffk_attention_pack(const ffk_pack_desc* desc, void* stream) {
    FFK_REQUIRE(desc, FFK_ERR_NULL, "ffk_attention_pack: null pointer");
    const ffk_pack_desc& d = *desc;
    FFK_REQUIRE(d.n > 0 && d.n <= FFK_PACK_JOBS && d.B2 > 0 && d.H > 0 && d.H < 65536 && d.N > 0 && d.N < (1 << 24) && d.D > 0 && d.D <= 32,
                FFK_ERR_SHAPE, "ffk_attention_pack: bad shape n=%d B2=%d H=%d N=%d D=%d", d.n, d.B2, d.H, d.N, d.D);
    FFK_REQUIRE(!d.bias || d.bias_t, FFK_ERR_NULL, "ffk_attention_pack: null pointer");
    FFK_REQUIRE(ffk_aligned16(d.bias_t), FFK_ERR_ALIGN, "ffk_attention_pack: tiles must be 16-byte aligned");
    for (int i = 0; i < d.n; ++i) {
        const ffk_pack_job& j = d.job[i];
        FFK_REQUIRE(j.src && (j.qk || j.acc || j.dsum) && (!j.dsum || j.other), FFK_ERR_NULL, "ffk_attention_pack: null pointer");
        FFK_REQUIRE(ffk_aligned16(j.qk) && ffk_aligned16(j.acc) && (!j.tiled || ffk_aligned16(j.src)), FFK_ERR_ALIGN,
                    "ffk_attention_pack: tiles must be 16-byte aligned");
    }
    switch (d.dtype) {
        case FFK_BF16: return attention_pack_launch<bf16_t>(d, (hipStream_t)stream);
        case FFK_F32: return attention_pack_launch<float>(d, (hipStream_t)stream);
        default: return ffk_fail(FFK_ERR_DTYPE, "ffk_attention_pack: unsupported dtype tag %d", d.dtype);
    }
}
