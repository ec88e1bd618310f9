// Weight gradients (see ffk_weight_grad in include/ffk.h):  out[n][k] = sum_m y[m][n] x[m][k]  and the column sums of y,
// for activations of 10^4 .. 10^6 rows and weights of a few hundred rows and columns.
//
// The product contracts over the rows of two row-major operands, and its output alone (a few 128 x 128 tiles) cannot fill
// the chip: the rows are cut into slices, one workgroup multiplies one slice for one output tile into fp32 accumulators and
// leaves them in a workspace, and a second launch adds the slices in a fixed order (no atomics: the same gradients every
// time) and rounds once.  Workgroups are ordered slice by slice and each XCD takes a contiguous part of that order, so the
// tiles that read the same rows run behind one L2.
//
//   bf16   v_mfma_f32_32x32x16_bf16 wants eight consecutive rows of one column per lane.  A thread fetches an 8 x 8 block
//          (eight 16-byte loads, whole 256-byte row pieces per 16 lanes), transposes it in registers (32 byte permutes) and
//          stores eight columns of eight rows; in LDS a column is 64 rows = 128 bytes, its eight 16-byte chunks XOR-swizzled
//          with the column index so that neither the stores (columns 8 apart) nor the fragment reads (adjacent columns) meet
//          in one bank group.  The permutes cost a fifth of the MFMA time.
//   fp32   rows stay as they are; a lane reads eight rows of its column and cuts them into bf16 parts (split4) for six bf16 products.
//          Against the fp32 instructions, which the matrix pipe bounded, with
//          the sums over the slices: 13 689 rows, 640 x 128 42 -> 34 us, 14 976 rows, 1 024 x 256 92 -> 73, 65 536 rows, 512 x 128 95 -> 77.
// Bound: the reads of y and x (from HBM or the last-level cache), in bf16; the vector instructions of the cuts in fp32.  The rows of a step are requested
// before the products of the step before it and nothing looks at them in between: the rows past the end of a slice, which have to be
// zeroed, are a step of their own behind the loop (as conditions of every load they made each step wait for its rows).
// 65 536 rows, us of the first launch, before and after: 640 x 128 36.9, 26.1, 512 x 128 27.9, 23.5; 32 768 rows, 1 032 x 256 50.7,
// 35.4; fp32 126.8, 113.3, 93.0, 86.3, 208, 187; the sums over the slices 5 .. 7 us.
#include "ffk_common.h"
#include <type_traits>

namespace {

constexpr int WG_THREADS = 256;
constexpr int WG_T = 128;                   // output tile: 128 columns of y by 128 columns of x

struct WgArgs {
    const void* y;
    const void* x;
    float* part;                            // [slices][N * K]
    float* csum;                            // [slices][N], or nullptr
    long y_so, y_si, x_so, x_si;
    unsigned y_inner, x_inner;
    int M, N, K, slices, rows_per_slice;    // rows_per_slice: a multiple of 64
};

__device__ __forceinline__ long wg_row(unsigned m, unsigned inner, long so, long si, bool flat) {
    const unsigned hi = flat ? 0u : m / inner;
    return (long)hi * so + (long)(m - hi * inner) * si;
}

// The rows m, m + RS, m + 2 RS .. of an operand that a thread fetches, a group every MB rows: no division and no multiplication per
// row - the offset moves by a step the launch fixes, and by another one where the inner index wraps (FLAT: it never does; a kernel of
// its own, because a branch between the two makes the compiler wait for the loads it merges).
template <typename T, int RS, int MB, bool FLAT> struct RowWalk {
    const T* p;                             // this thread's column in row 0
    long off, row_inc, group_inc, wrap;     // of the group's first row; per row; per group; where lo passes inner
    unsigned lo, inner, row_lo, group_lo;
    __device__ __forceinline__ void init(const T* base, unsigned m, unsigned inner_, unsigned M, long so, long si) {
        p = base;
        inner = inner_ < M ? inner_ : 0x80000000u;          // rows and steps together stay below: no wrap
        const unsigned hi = FLAT ? 0u : m / inner;
        lo = m - hi * inner;
        off = (long)hi * so + (long)lo * si;
        row_lo = RS % inner;
        group_lo = MB % inner;
        row_inc = FLAT ? RS * si : (long)(RS / inner) * so + (long)row_lo * si;
        group_inc = FLAT ? MB * si : (long)(MB / inner) * so + (long)group_lo * si;
        wrap = so - (long)inner * si;
    }
    template <int N> __device__ __forceinline__ void fetch(Vec16<T>* v) {          // N rows of the group, on to the next group
        long o = off;
        unsigned l = lo;
#pragma unroll
        for (int e = 0; e < N; ++e) {
            v[e] = ld16(p + (FLAT ? off + e * row_inc : o));
            if (!FLAT) {
                o += row_inc;
                l += row_lo;
                if (l >= inner) {
                    l -= inner;
                    o += wrap;
                }
            }
        }
        off += group_inc;
        if (!FLAT) {
            lo += group_lo;
            if (lo >= inner) {
                lo -= inner;
                off += wrap;
            }
        }
    }
};

template <typename T, bool FLAT>
__global__ __launch_bounds__(WG_THREADS, 2) void weight_grad_kernel(const WgArgs a) {
    constexpr bool BF = std::is_same<T, bf16_t>::value;
    constexpr int MB = BF ? 64 : 32;                       // rows per step
    constexpr int BUF = BF ? WG_T * 128 : MB * 640;        // bytes of one operand's buffer
    constexpr int NP = BF ? 8 : 4;                         // 16-byte loads per thread, operand and step
    extern __shared__ __align__(16) unsigned char smem[];  // [2 buffers][y | x]
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    const int tn = (a.N + WG_T - 1) / WG_T, tk = (a.K + WG_T - 1) / WG_T;
    const unsigned per_xcd = gridDim.x >> 3;
    const unsigned item = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (item >= (unsigned)(tn * tk) * (unsigned)a.slices) return;
    const int n0 = (int)(item % tn) * WG_T, k0 = (int)((item / tn) % tk) * WG_T, slice = (int)(item / (tn * tk));
    const int m_begin = slice * a.rows_per_slice;
    const int m_end = m_begin + a.rows_per_slice < a.M ? m_begin + a.rows_per_slice : a.M;

    // bf16: waves 0 and 1 fetch y, 2 and 3 x, an 8 x 8 block per thread.  fp32: every thread half of its vectors from each.
    const int bt = BF ? (tid & 127) : tid;
    const int cb = BF ? (bt & 15) : (bt & 31);             // column block (8 or 4 columns)
    const int rb = BF ? (bt >> 4) : (bt >> 5);             // row block
    const bool is_x = BF && wave >= 2;                     // of the whole wave
    constexpr int VEC = DT<T>::VEC, RS = BF ? 1 : 8;       // row e of a thread: first row + RS e
    const unsigned r0 = BF ? rb * 8 : rb;
    RowWalk<T, RS, MB, FLAT> wy, wx;                             // bf16: wy is the walk of the thread's one operand
    auto column = [&](int first, int cols) {               // clamped columns are never stored
        const int c = first + cb * VEC;
        return c < cols ? c : cols - VEC;
    };
    auto start = [&]() __attribute__((always_inline)) {
        if (is_x) wy.init((const T*)a.x + column(k0, a.K), m_begin + r0, a.x_inner, a.M, a.x_so, a.x_si);
        else wy.init((const T*)a.y + column(n0, a.N), m_begin + r0, a.y_inner, a.M, a.y_so, a.y_si);
        if (!BF) wx.init((const T*)a.x + column(k0, a.K), m_begin + r0, a.x_inner, a.M, a.x_so, a.x_si);
    };
    auto fetch_rows = [&](Vec16<T>* pre) __attribute__((always_inline)) {      // a whole step: requests only, nothing waits for them here
        wy.template fetch<NP>(pre);
        if (!BF) wx.template fetch<NP>(pre + (BF ? 0 : NP));
    };
    auto fetch_tail = [&](Vec16<T>* pre, int m0) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < NP; ++e) {                     // the last rows: clamped, and those past the end add nothing
            const int m = m0 + r0 + RS * e;
            const unsigned mc = (unsigned)(m < m_end ? m : m_end - 1);
            if (BF) {
                pre[e] = ld16(wy.p + (is_x ? wg_row(mc, a.x_inner, a.x_so, a.x_si, FLAT || a.x_inner >= (unsigned)a.M) : wg_row(mc, a.y_inner, a.y_so, a.y_si, FLAT || a.y_inner >= (unsigned)a.M)));
                if (m >= m_end && !is_x) pre[e] = Vec16<T>{};
            } else {
                pre[e] = ld16(wy.p + wg_row(mc, a.y_inner, a.y_so, a.y_si, FLAT || a.y_inner >= (unsigned)a.M));
                pre[(BF ? 0 : NP) + e] = ld16(wx.p + wg_row(mc, a.x_inner, a.x_so, a.x_si, FLAT || a.x_inner >= (unsigned)a.M));
                if (m >= m_end) pre[e] = Vec16<T>{};
            }
        }
    };
    [[maybe_unused]] uint32_t sign = (uint32_t)slice << 31;       // fp32: of the piece the next commit belongs to
    auto commit = [&](const Vec16<T>* pre, int buf) __attribute__((always_inline)) {
        unsigned char* sb = smem + buf * 2 * BUF;
        if constexpr (BF) {
            unsigned char* so = sb + (is_x ? BUF : 0);
#pragma unroll
            for (int d = 0; d < 4; ++d) {                  // columns 2 d and 2 d + 1 of the block
                u32x4 lo, hi;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint32_t w0 = reinterpret_cast<const u32x4*>(&pre[2 * j])[0][d], w1 = reinterpret_cast<const u32x4*>(&pre[2 * j + 1])[0][d];
                    lo[j] = __builtin_amdgcn_perm(w1, w0, 0x05040100u);
                    hi[j] = __builtin_amdgcn_perm(w1, w0, 0x07060302u);
                }
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int n = cb * 8 + 2 * d + h;
                    *reinterpret_cast<u32x4*>(so + n * 128 + (((rb ^ n ^ (n >> 3)) & 7) << 4)) = h ? hi : lo;
                }
            }
        } else {
#pragma unroll
            for (int e = 0; e < NP; ++e) {
                u32x4 y = *reinterpret_cast<const u32x4*>(&pre[e]);
#pragma unroll
                for (int j = 0; j < 4; ++j) y[j] ^= sign;
                *reinterpret_cast<u32x4*>(sb + (rb + 8 * e) * 640 + cb * 16) = y;
                *reinterpret_cast<Vec16<T>*>(sb + BUF + (rb + 8 * e) * 640 + cb * 16) = pre[(BF ? 0 : NP) + e];
            }
        }
    };

    const int wn = wave >> 1, wk = wave & 1;               // the wave's 64 x 64 quarter of the tile
    const bool sums = a.csum != nullptr && k0 == 0 && wk == 0;
    float cs[2] = {0.0f, 0.0f};
    [[maybe_unused]] float turn = slice & 1 ? -1.0f : 1.0f;        // fp32: sign of the products of this piece
    // fp32: one or two rows by the fp32 instructions (one row 2.6e-8 -> 3.5e-8 by parts, two 3.1e-8 -> 3.4e-8, four 4.0e-8 -> 3.1e-8)
    [[maybe_unused]] const bool few = m_end - m_begin <= 2;
    f32x16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

    // The products of a step.  The fragments of a K step are requested one K step ahead.
    auto products = [&](const unsigned char* sy, [[maybe_unused]] auto plain) __attribute__((always_inline)) {
        const unsigned char* sx = sy + BUF;
        if constexpr (BF) {
            bf16x8 fy[2][2], fx[2][2];
            auto read = [&](int ks) __attribute__((always_inline)) {
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const int n = wn * 64 + i * 32 + l32, k = wk * 64 + i * 32 + l32;
                    fy[ks & 1][i] = *reinterpret_cast<const bf16x8*>(sy + n * 128 + ((((2 * ks + half) ^ n ^ (n >> 3)) & 7) << 4));
                    fx[ks & 1][i] = *reinterpret_cast<const bf16x8*>(sx + k * 128 + ((((2 * ks + half) ^ k ^ (k >> 3)) & 7) << 4));
                }
            };
            read(0);
#pragma unroll
            for (int ks = 0; ks < MB / 16; ++ks) {
                if (ks + 1 < MB / 16) read(ks + 1);
                const bf16x8* y2 = fy[ks & 1];
                const bf16x8* x2 = fx[ks & 1];
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j) Mma<bf16_t>::mma(acc[i][j], y2[i], x2[j]);
                if (sums) {
                    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
                    const bf16x2 ones = {(bf16_t)1.0f, (bf16_t)1.0f};
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const bf16x2 pr = {y2[i][2 * e], y2[i][2 * e + 1]};
                            cs[i] = __builtin_amdgcn_fdot2_f32_bf16(pr, ones, cs[i], false);
                        }
                }
            }
        } else if constexpr (!plain.value) {
#pragma unroll
            for (int ks = 0; ks < MB / 16; ++ks) {         // rows 16 ks + 8 half .. + 7 of a column per lane
                bf16x8 fy[2][3];
                auto cut = [&](bf16x8 (&f)[3], const unsigned char* p, float* c) __attribute__((always_inline)) {
                    f32x4 x[2];
#pragma unroll
                    for (int e = 0; e < 8; ++e) x[e >> 2][e & 3] = *reinterpret_cast<const float*>(p + (16 * ks + 8 * half + e) * 640);
                    const Split4 lo = split4(x[0]), hi = split4(x[1]);
#pragma unroll
                    for (int t = 0; t < 3; ++t) f[t] = split_frag(lo, hi, t);
                    if (c) *c += turn * (((x[0][0] + x[0][1]) + (x[0][2] + x[0][3])) + ((x[1][0] + x[1][1]) + (x[1][2] + x[1][3])));
                };
#pragma unroll
                for (int i = 0; i < 2; ++i) cut(fy[i], sy + (wn * 64 + i * 32 + l32) * 4, sums ? &cs[i] : nullptr);
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    bf16x8 fx[3];
                    cut(fx, sx + (wk * 64 + j * 32 + l32) * 4, nullptr);
#pragma unroll
                    for (int t = 0; t < 6; ++t)
#pragma unroll
                        for (int i = 0; i < 2; ++i) Mma<bf16_t>::mma(acc[i][j], fy[i][SPLIT_A[t]], fx[SPLIT_B[t]]);
                }
            }
        } else {
#pragma unroll 1
            for (int ks = 0; ks < MB / 2; ++ks) {
                float fy[2], fx[2];
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    fy[i] = *reinterpret_cast<const float*>(sy + (2 * ks + half) * 640 + (wn * 64 + i * 32 + l32) * 4);
                    fx[i] = *reinterpret_cast<const float*>(sx + (2 * ks + half) * 640 + (wk * 64 + i * 32 + l32) * 4);
                }
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fy[i], fx[j], acc[i][j], 0, 0, 0);
                if (few && sums) {
#pragma unroll
                    for (int i = 0; i < 2; ++i) cs[i] += fy[i];
                }
            }
        }
    };

    constexpr int NV = NP * (BF ? 1 : 2);
    const int whole = (m_end - m_begin) / MB;
    const bool tail = (m_end - m_begin) % MB != 0;
    // fp32: the sums of every PIECE steps (256 rows) by themselves, and y's sign turned for every other piece and every other slice: the
    // bf16 instructions cut off towards minus infinity, which in a long chain or the sum of many is more than its roundings.  Relative
    // error (2-norm), fp32 instructions -> one chain per slice, no turns -> this: 65 536 rows in 64 slices 5.8e-7 -> 6.4e-7 -> 2.6e-7, in 256
    // 3.2e-7 -> 3.7e-7 -> 2.8e-7.
    constexpr int PIECE = 8;
    f32x16 sum[BF ? 1 : 2][BF ? 1 : 2];
#pragma unroll
    for (auto& s : sum)
#pragma unroll
        for (f32x16& t : s) t = acc[0][0];
    [[maybe_unused]] auto end_piece = [&]() __attribute__((always_inline)) {
        if constexpr (!BF) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        sum[i][j][v] = fmaf(turn, acc[i][j][v], sum[i][j][v]);
                        acc[i][j][v] = 0.0f;
                    }
            turn = -turn;
        }
    };
    auto walk = [&](auto plain) __attribute__((always_inline)) {
        start();
        {
            Vec16<T> pre[NV];
            if (whole > 0) fetch_rows(pre);
            else fetch_tail(pre, m_begin);
            commit(pre, 0);
        }
        lds_barrier();
        int buf = 0, steps = 1;                            // committed steps
        auto step = [&](auto tail_c) __attribute__((always_inline)) {      // products of one buffer while the rows of the next are on their way
            Vec16<T> pre[NV];
            if constexpr (decltype(tail_c)::value) fetch_tail(pre, m_begin + whole * MB);
            else fetch_rows(pre);
            products(smem + buf * 2 * BUF, plain);
            if (!BF && !plain.value && steps % PIECE == 0) {
                end_piece();
                sign ^= 0x80000000u;
            }
            ++steps;
            commit(pre, buf ^ 1);                          // its last readers passed the barrier below
            lds_barrier();
            buf ^= 1;
        };
        for (int i = 1; i < whole; ++i) step(std::false_type());
        if (tail && whole > 0) step(std::true_type());
        products(smem + buf * 2 * BUF, plain);
        if (!BF && !plain.value) end_piece();
    };
    if constexpr (BF) walk(std::false_type());
    else {
        int* bad = reinterpret_cast<int*>(smem);
        if (!few) {
            walk(std::false_type());
            float t = 0.0f;
#pragma unroll
            for (int v = 0; v < 64; ++v) t += sum[v >> 5][(v >> 4) & 1][v & 15];
            lds_barrier();
            if (lane == 0) bad[wave] = 0;
            if (t - t != 0.0f) bad[wave] = 1;
            lds_barrier();
        }
        // infinite operands, whose parts make NaN of every product: those sums by the fp32 instructions, the others keep their bits
        const bool again = few || (bad[0] | bad[1] | bad[2] | bad[3]);
        if (__builtin_expect(again, 0)) {
            lds_barrier();
            sign = 0;
            walk(std::true_type());
#pragma unroll
            for (int v = 0; v < 64; ++v) {
                const float y = sum[v >> 5][(v >> 4) & 1][v & 15];
                if (!few && y == y) acc[v >> 5][(v >> 4) & 1][v & 15] = y;
            }
        } else {
#pragma unroll
            for (int v = 0; v < 64; ++v) acc[v >> 5][(v >> 4) & 1][v & 15] = sum[v >> 5][(v >> 4) & 1][v & 15];
        }
    }
    float* part = a.part + (long)slice * a.N * a.K;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int k = k0 + wk * 64 + j * 32 + l32;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int n = n0 + wn * 64 + i * 32 + acc_row(v, lane);
                if (n < a.N && k < a.K) part[(long)n * a.K + k] = acc[i][j][v];
            }
        }
    if (sums) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const float s = cs[i] + lane_xor<32>(cs[i]);
            const int n = n0 + wn * 64 + i * 32 + l32;
            if (half == 0 && n < a.N) a.csum[(long)slice * a.N + n] = s;
        }
    }
}

// One sum over slices: of part[s][i] over s, plus acc[i] if READ: to acc[i] if WRITE, else to out.  Element i = (row n, column k) of
// out is at (n / inner) * o_so + (n % inner) * o_si + k * o_sk.
struct SliceSum {
    void* out;
    const float* part;
    float* acc;
    long n, pitch, o_so, o_si, o_sk;
    int K;
    unsigned inner, blocks;                              // workgroups of 256 values
};

// Four adjacent values per lane, the slices spread over the four waves.  The matrix and its column sums go in one launch (a
// launch of its own took the few hundred column sums 5 us): workgroups from a.blocks on belong to b.
template <typename OT>
__global__ __launch_bounds__(256) void slice_sum_kernel(const SliceSum a, const SliceSum b, int flags, int slices) {
    __shared__ f32x4 red[3][64];
    const bool second = blockIdx.x >= a.blocks;
    const SliceSum& q = second ? b : a;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const long i = ((long)(blockIdx.x - (second ? a.blocks : 0u)) * 64 + lane) * 4;
    f32x4 s = {0.0f, 0.0f, 0.0f, 0.0f};
    if (i < q.n) {
        const float* p = q.part + i;
        const long pitch = q.pitch;
#pragma unroll 8
        for (int sl = wave; sl < slices; sl += 4) s += *reinterpret_cast<const f32x4*>(p + (long)sl * pitch);
    }
    if (wave) red[wave - 1][lane] = s;
    __syncthreads();
    if (wave || i >= q.n) return;
    s = (s + red[0][lane]) + (red[1][lane] + red[2][lane]);
    if (flags & FFK_WGRAD_READ) s += *reinterpret_cast<const f32x4*>(q.acc + i);
    if (flags & FFK_WGRAD_WRITE) {
        *reinterpret_cast<f32x4*>(q.acc + i) = s;
        return;
    }
    const unsigned row = (unsigned)(i / q.K), k = (unsigned)(i - (long)row * q.K), hi = row / q.inner;      // K % 4 == 0
    OT* o = (OT*)q.out + (long)hi * q.o_so + (long)(row - hi * q.inner) * q.o_si + (long)k * q.o_sk;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e * q.o_sk] = DT<OT>::from_f(s[e]);
}

SliceSum slice_sum(void* out, const float* part, float* acc, long n, int K, long inner, long so, long si, long sk, long pitch) {
    return SliceSum{out, part, acc, n, pitch, so, si, sk, K, (unsigned)inner, (unsigned)((n + 255) / 256)};
}

template <typename T>
int slice_sum_launch(const SliceSum& a, const SliceSum& b, int flags, long slices, hipStream_t st) {
    slice_sum_kernel<T><<<a.blocks + b.blocks, 256, 0, st>>>(a, b, flags, (int)slices);
    return ffk_check_launch("ffk_weight_grad");
}

template <typename T>
int launch_weight_grad(const WgArgs& a, void* out, long n_out, void* colsum, long cs_first, long cs_count, float* acc, long o_inner, long o_so, long o_si, long o_sk, int flags,
                       hipStream_t st) {
    const size_t smem = std::is_same<T, bf16_t>::value ? 4 * (size_t)WG_T * 128 : 4 * (size_t)32 * 640;
    const long items = (long)ffk_cdiv(a.N, WG_T) * ffk_cdiv(a.K, WG_T) * a.slices;
    FFK_REQUIRE(items < (1L << 31) - 8, FFK_ERR_SHAPE, "ffk_weight_grad: %ld workgroups exceed the grid limit", items);
    auto launch = [&](auto flat_c) {
        constexpr bool FLAT = decltype(flat_c)::value;
        static FfkLdsReservation lds_reserved;
        const int rc_lds = ffk_reserve_lds(lds_reserved, (const void*)weight_grad_kernel<T, FLAT>, smem, "ffk_weight_grad");
        if (rc_lds != FFK_OK) return rc_lds;
        weight_grad_kernel<T, FLAT><<<(unsigned)(8 * ffk_cdiv(items, 8)), WG_THREADS, smem, st>>>(a);
        return ffk_check_launch("ffk_weight_grad");
    };
    const bool flat = a.y_inner >= (unsigned)a.M && a.x_inner >= (unsigned)a.M;
    const int rc = flat ? launch(std::true_type()) : launch(std::false_type());
    if (rc != FFK_OK) return rc;
    const long nk = (long)a.N * a.K;
    const SliceSum m = slice_sum(out, a.part, acc, n_out * a.K, a.K, o_inner, o_so, o_si, o_sk, nk);
    SliceSum c{};
    if (a.csum) c = slice_sum(colsum, a.csum + cs_first, acc ? acc + n_out * a.K : nullptr, cs_count, (int)cs_count, 1, 0, 0, 1, a.N);
    return slice_sum_launch<T>(m, c, flags, a.slices, st);
}

}  // namespace

extern "C" int ffk_weight_grad(void* out, int64_t n_out, void* colsum, int64_t cs_first, int64_t cs_count, float* acc, float* ws,
                               const void* y, const void* x, int64_t M, int64_t N, int64_t K, int64_t slices, int64_t y_inner, int64_t y_so, int64_t y_si, int64_t x_inner, int64_t x_so,
                               int64_t x_si, int64_t o_inner, int64_t o_so, int64_t o_si, int64_t o_sk, int flags, int dtype,
                               void* stream) {
    FFK_REQUIRE(out && ws && y && x && (acc || flags == 0), FFK_ERR_NULL, "ffk_weight_grad: null pointer");
    FFK_REQUIRE(M > 0 && M < (1L << 31) - 128 && N > 0 && N % 8 == 0 && K > 0 && K % 8 == 0 && N < (1 << 20) && K < (1 << 20) &&
                    slices > 0 && slices <= 65536 && y_inner > 0 && x_inner > 0 && o_inner > 0 && N * K < (1L << 32),
                FFK_ERR_SHAPE, "ffk_weight_grad: bad shape M=%ld N=%ld K=%ld slices=%ld", (long)M, (long)N, (long)K, (long)slices);
    FFK_REQUIRE(n_out > 0 && n_out <= N && (!colsum || (cs_first >= 0 && cs_first % 4 == 0 && cs_count > 0 && cs_count % 4 == 0 && cs_first + cs_count <= N)),
                FFK_ERR_SHAPE, "ffk_weight_grad: rows %ld and column sums [%ld, +%ld) of %ld", (long)n_out, (long)cs_first, (long)cs_count, (long)N);
    const int vec = dtype == FFK_F32 ? 4 : 8;
    FFK_REQUIRE(ffk_aligned16(ws) && ffk_aligned16(acc) && ffk_aligned16(y) && ffk_aligned16(x) && y_so % vec == 0 && y_si % vec == 0 && x_so % vec == 0 &&
                    x_si % vec == 0,
                FFK_ERR_ALIGN, "ffk_weight_grad: operand rows must be 16-byte aligned");
    WgArgs a;
    a.y = y;
    a.x = x;
    a.part = ws;
    a.csum = colsum ? ws + slices * N * K : nullptr;
    a.y_so = y_so;
    a.y_si = y_si;
    a.x_so = x_so;
    a.x_si = x_si;
    a.y_inner = (unsigned)(y_inner < M ? y_inner : M);
    a.x_inner = (unsigned)(x_inner < M ? x_inner : M);
    a.M = (int)M;
    a.N = (int)N;
    a.K = (int)K;
    a.slices = (int)slices;
    a.rows_per_slice = (int)(((M + slices - 1) / slices + 63) / 64 * 64);
    FFK_REQUIRE((slices - 1) * (int64_t)a.rows_per_slice < M, FFK_ERR_SHAPE,
                "ffk_weight_grad: %ld slices of 64-row steps leave empty slices of %ld rows", (long)slices, (long)M);
    hipStream_t st = (hipStream_t)stream;
    switch (dtype) {
        case FFK_BF16: return launch_weight_grad<bf16_t>(a, out, n_out, colsum, cs_first, cs_count, acc, o_inner, o_so, o_si, o_sk, flags, st);
        case FFK_F32: return launch_weight_grad<float>(a, out, n_out, colsum, cs_first, cs_count, acc, o_inner, o_so, o_si, o_sk, flags, st);
        default: return ffk_fail(FFK_ERR_DTYPE, "ffk_weight_grad: unsupported dtype tag %d", dtype);
    }
}

extern "C" int ffk_slice_sum(void* out, const float* part, int64_t slices, int64_t N, int64_t K, int64_t o_inner, int64_t o_so,
                             int64_t o_si, int64_t o_sk, int dtype, void* stream) {
    FFK_REQUIRE(out && part, FFK_ERR_NULL, "ffk_slice_sum: null pointer");
    FFK_REQUIRE(slices > 0 && slices <= 65536 && N > 0 && K > 0 && K % 4 == 0 && N < (1L << 31) && K < (1L << 31) && o_inner > 0 &&
                    N * K < (1L << 38),
                FFK_ERR_SHAPE, "ffk_slice_sum: bad shape slices=%ld N=%ld K=%ld", (long)slices, (long)N, (long)K);
    FFK_REQUIRE(ffk_aligned16(part), FFK_ERR_ALIGN, "ffk_slice_sum: the partial sums must be 16-byte aligned");
    hipStream_t st = (hipStream_t)stream;
    const SliceSum q = slice_sum(out, part, nullptr, N * K, (int)K, o_inner < N ? o_inner : N, o_so, o_si, o_sk, N * K);
    switch (dtype) {
        case FFK_BF16: return slice_sum_launch<bf16_t>(q, SliceSum{}, 0, slices, st);
        case FFK_F32: return slice_sum_launch<float>(q, SliceSum{}, 0, slices, st);
        default: return ffk_fail(FFK_ERR_DTYPE, "ffk_slice_sum: unsupported dtype tag %d", dtype);
    }
}
