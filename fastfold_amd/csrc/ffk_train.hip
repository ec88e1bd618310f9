// Row kernels of the block's backward pass (see the section "backward pass of a block" in include/ffk.h).  All of them stream
// activations once: what bounds them is the bytes they read and write (16-byte accesses, a few rows in flight per wave).
#include "ffk_common.h"
#include <initializer_list>

namespace {

constexpr int TR_THREADS = 256;
constexpr int LN_BLOCKS = FFK_LN_BWD_BLOCKS;

template <typename T> __device__ __forceinline__ void unpack(const Vec16<T>& v, float* f) {
#pragma unroll
    for (int e = 0; e < DT<T>::VEC; ++e) f[e] = DT<T>::to_f(v.e[e]);
}
template <typename T> __device__ __forceinline__ Vec16<T> pack(const float* f) {
    Vec16<T> v;
#pragma unroll
    for (int e = 0; e < DT<T>::VEC; ++e) v.e[e] = DT<T>::from_f(f[e]);
    return v;
}

// ---------------------------------------------------------------------------------------------- LayerNorm ----
// dx = resid + LayerNorm'(x)^T dy and, optionally, xn = LayerNorm(x) for the weight gradient behind it.  A row is LPR = C / VEC
// adjacent lanes with one 16-byte vector each; mean and rstd are recomputed from the row (it is read anyway, and nothing has
// to be kept from the forward pass).  A thread sums its columns of dgamma / dbeta over the rows it sees; the workgroup adds
// them in LDS and leaves one partial row per workgroup, which ln_finish_kernel adds up: no
// atomics, the same result every time.
template <typename T, int C>
__global__ __launch_bounds__(TR_THREADS) void ln_bwd_rows_kernel(T* dx, T* __restrict__ xn, float* __restrict__ part,
                                                               const T* dy, const T* __restrict__ x, const T* __restrict__ gamma,
                                                               const T* __restrict__ beta, const T* resid, long rows, float eps) {
    constexpr int V = DT<T>::VEC, LPR = C / V, RPB = TR_THREADS / LPR;
    __shared__ float red[2 * C * 4];                            // one partial row per wave
    const int tid = threadIdx.x, c = (tid % LPR) * V;
    const int wave = tid >> 6;
    float g[V], b[V], dg[V], db[V];
    unpack<T>(ld16(gamma + c), g);
    if (xn) unpack<T>(ld16(beta + c), b);
#pragma unroll
    for (int e = 0; e < V; ++e) dg[e] = db[e] = 0.0f;
    // RU rows per thread at a time: their loads go out together, and the reductions - a chain of two, the statistics of the
    // gradient need only the centred row - run side by side
    constexpr int RU = 2;
    for (long r0 = (long)blockIdx.x * RPB; r0 < rows; r0 += (long)gridDim.x * RPB * RU) {
        Vec16<T> vx[RU], vd[RU], vr[RU];
        bool ok[RU];
        long o[RU];
#pragma unroll
        for (int u = 0; u < RU; ++u) {
            const long r = r0 + (long)u * gridDim.x * RPB + tid / LPR;
            ok[u] = r < rows;
            o[u] = (ok[u] ? r : rows - 1) * C + c;
            vx[u] = ld16(x + o[u]);
            vd[u] = ld16(dy + o[u]);
            vr[u] = Vec16<T>{};
            if (resid) vr[u] = ld16(resid + o[u]);
        }
        float mu[RU], rs[RU], s1[RU], s2[RU];
#pragma unroll
        for (int u = 0; u < RU; ++u) {
            float xv[V], s = 0.0f;
            unpack<T>(vx[u], xv);
#pragma unroll
            for (int e = 0; e < V; ++e) s += xv[e];
            mu[u] = s;
        }
#pragma unroll
        for (int u = 0; u < RU; ++u) mu[u] = group_sum(mu[u], LPR) * (1.0f / C);
#pragma unroll
        for (int u = 0; u < RU; ++u) {
            float xv[V], dv[V], q = 0.0f, t1 = 0.0f, t2 = 0.0f;
            unpack<T>(vx[u], xv);
            unpack<T>(vd[u], dv);
#pragma unroll
            for (int e = 0; e < V; ++e) {
                const float xc = xv[e] - mu[u], t = dv[e] * g[e];
                q += xc * xc;
                t1 += t;
                t2 += t * xc;
            }
            rs[u] = q;
            s1[u] = t1;
            s2[u] = t2;
        }
#pragma unroll
        for (int u = 0; u < RU; ++u) {
            rs[u] = rsqrtf(group_sum(rs[u], LPR) * (1.0f / C) + eps);
            s1[u] = group_sum(s1[u], LPR) * (1.0f / C);
            s2[u] = group_sum(s2[u], LPR) * rs[u] * (1.0f / C);
        }
#pragma unroll
        for (int u = 0; u < RU; ++u) {
            float xv[V], dv[V], rv[V], out[V], xo[V];
            unpack<T>(vx[u], xv);
            unpack<T>(vd[u], dv);
            unpack<T>(vr[u], rv);
#pragma unroll
            for (int e = 0; e < V; ++e) {
                const float xh = (xv[e] - mu[u]) * rs[u];
                out[e] = rv[e] + rs[u] * (dv[e] * g[e] - s1[u] - xh * s2[u]);
                xo[e] = xh * g[e] + (xn ? b[e] : 0.0f);
                if (ok[u]) {
                    dg[e] += dv[e] * xh;
                    db[e] += dv[e];
                }
            }
            if (ok[u]) {
                st16(dx + o[u], pack<T>(out));
                if (xn) st16(xn + o[u], pack<T>(xo));
            }
        }
    }
    // lanes of a wave that own the same columns: LPR .. 64 apart
#pragma unroll
    for (int e = 0; e < V; ++e) {
#pragma unroll
        for (int w = LPR; w < 64; w <<= 1) {
            dg[e] += __shfl_xor(dg[e], w, 64);
            db[e] += __shfl_xor(db[e], w, 64);
        }
    }
    if ((tid & 63) < LPR) {
#pragma unroll
        for (int e = 0; e < V; ++e) {
            red[wave * 2 * C + c + e] = dg[e];
            red[wave * 2 * C + C + c + e] = db[e];
        }
    }
    __syncthreads();
    // LPR <= 64: every wave holds whole rows
    for (int i = tid; i < 2 * C; i += TR_THREADS)
        part[(long)blockIdx.x * 2 * C + i] = (red[i] + red[2 * C + i]) + (red[4 * C + i] + red[6 * C + i]);
}

// dgamma[c] / dbeta[c] = sum of the partial rows: a workgroup per 16 columns, 64 groups of four lanes over the partial rows (a
// workgroup per 32 columns with eight groups walked 128 rows one load after the other: 34 us at C = 256, now 4.6)
template <typename T>
__global__ __launch_bounds__(256) void ln_finish_kernel(T* __restrict__ dgamma, T* __restrict__ dbeta, const float* __restrict__ part,
                                                        int blocks, int C) {
    __shared__ f32x4 red[256];
    const int tid = threadIdx.x, col = blockIdx.x * 16 + (tid & 3) * 4;
    f32x4 s = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 4
    for (int b = tid >> 2; b < blocks; b += 64) s += *reinterpret_cast<const f32x4*>(part + (long)b * 2 * C + col);
    red[tid] = s;
    __syncthreads();
    if (tid < 64) {
        s = (red[tid] + red[tid + 64]) + (red[tid + 128] + red[tid + 192]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float v = s[e];
#pragma unroll
            for (int w = 4; w < 64; w <<= 1) v += __shfl_xor(v, w, 64);
            s[e] = v;
        }
        if (tid < 4) {
            T* out = col < C ? dgamma + col : dbeta + (col - C);
#pragma unroll
            for (int e = 0; e < 4; ++e) out[e] = DT<T>::from_f(s[e]);
        }
    }
}

// --------------------------------------------------------------------------------------------- row scaling ----
// out[m][c] = x[m][c] * mul(m, c).  MODE 0: a vector of C multipliers per row; 1: one multiplier per row; 2: one fp32 divisor
// per row, out = x / (mul + eps).  The multiplier of row m lies at (m / inner) * m_so + (m % inner) * m_si.
template <typename T, int MODE>
__global__ __launch_bounds__(TR_THREADS) void scale_rows_kernel(T* out, const T* x, const void* __restrict__ mul, long rows, int C,
                                                              unsigned inner, long m_so, long m_si, float eps) {
    constexpr int V = DT<T>::VEC;
    const int vpr = C / V;
    const long n = rows * vpr;
    for (long i = (long)blockIdx.x * TR_THREADS + threadIdx.x; i < n; i += (long)gridDim.x * TR_THREADS) {
        const unsigned m = (unsigned)(i / vpr);
        const int c = (int)(i - (long)m * vpr) * V;
        const unsigned hi = m / inner;
        const long mo = (long)hi * m_so + (long)(m - hi * inner) * m_si;
        float f[V];
        unpack<T>(ld16(x + i * V), f);
        if constexpr (MODE == 0) {
            float g[V];
            unpack<T>(ld16((const T*)mul + mo + c), g);
#pragma unroll
            for (int e = 0; e < V; ++e) f[e] *= g[e];
        } else {
            const float s = MODE == 1 ? DT<T>::to_f(((const T*)mul)[mo]) : 1.0f / (((const float*)mul)[mo] + eps);
#pragma unroll
            for (int e = 0; e < V; ++e) f[e] *= s;
        }
        st16(out + i * V, pack<T>(f));
    }
}

// -------------------------------------------------------------------------------- gate of an attention ----
// One wave per (batch row, 32 tokens, head): with s = sigmoid(gpre + gbias),
//     go = s o,   do = dgo s,   dgpre = dgo o s (1 - s),   dsum[token] = sum_d do o,
// do written as the two operand tiles the attention backward reads (accumulator order of the rows, accumulator order of the
// keys); the second one wants tokens along registers and is transposed through a 32 x 33 piece of LDS.
template <typename T>
__global__ __launch_bounds__(TR_THREADS) void att_gate_bwd_kernel(T* __restrict__ go, T* __restrict__ dgpre, T* __restrict__ do_t,
                                                                T* __restrict__ do_v, float* __restrict__ dsum,
                                                                const T* __restrict__ dgo, const T* __restrict__ gpre,
                                                                const T* __restrict__ gbias, const T* __restrict__ o, long B2, int N,
                                                                int H, long g_ld, long dg_ld) {
    constexpr int V = DT<T>::VEC, NV = 16 / V;
    __shared__ float tr[4][32 * 33];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l32 = lane & 31, half = lane >> 5;
    const int NT = (N + 31) >> 5, HC = H * 32;
    const long item = (long)blockIdx.x * 4 + wave;
    if (item >= B2 * NT * H) return;                   // no barrier below: the LDS piece belongs to the wave
    const int h = (int)(item % H);
    const long bt = item / H;
    const int t = (int)(bt % NT);
    const long b = bt / NT;
    const int n = t * 32 + l32;
    const bool ok = n < N;
    const long m = b * N + (ok ? n : N - 1);
    const int c = h * 32 + 16 * half;
    float fd[16], fg[16], fb[16], fo[16];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        unpack<T>(ld16(dgo + m * HC + c + i * V), fd + i * V);
        unpack<T>(ld16(gpre + m * g_ld + c + i * V), fg + i * V);
        unpack<T>(ld16(gbias + c + i * V), fb + i * V);
        unpack<T>(ld16(o + m * HC + c + i * V), fo + i * V);
    }
    float vgo[16], vdg[16], vdo[16], ds = 0.0f;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const float s = sigmoid_f(fg[e] + fb[e]);
        vgo[e] = s * fo[e];
        vdo[e] = ok ? fd[e] * s : 0.0f;                // rows past the end are zero in the operand tiles
        vdg[e] = fd[e] * fo[e] * s * (1.0f - s);
        vdo[e] = DT<T>::to_f(DT<T>::from_f(vdo[e]));   // as the products will see it
        ds += vdo[e] * fo[e];
    }
    ds += lane_xor<32>(ds);
    const long bh = b * H + h;
    if (half == 0) dsum[(bh * NT + t) * 32 + l32] = ds;
    if (ok) {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            st16(go + m * HC + c + i * V, pack<T>(vgo + i * V));
            st16(dgpre + m * dg_ld + c + i * V, pack<T>(vdg + i * V));
        }
    }
    // token order (FFK_TILE_ACC): channel d of token l32 at ((d / 4 % 2) * 32 + l32) * 16 + 4 * (d / 8) + d % 4; this lane holds
    // d = 16 half + 8 a + 4 hh + e
    T* pt = do_t + ((bh * NT + t) << 10);
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
        float w[8];
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int e = 0; e < 4; ++e) w[4 * a + e] = vdo[8 * a + 4 * hh + e];
        T* p = pt + ((hh * 32 + l32) << 4) + 8 * half;
#pragma unroll
        for (int i = 0; i < 8 / V; ++i) st16(p + i * V, pack<T>(w + i * V));
    }
    // key order (FFK_TILE_V): channel l32 over tokens 8 a + 4 half + e
    float* w = tr[wave];
#pragma unroll
    for (int e = 0; e < 16; ++e) w[l32 * 33 + 16 * half + e] = vdo[e];
    __builtin_amdgcn_wave_barrier();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    float y[16];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int e = 0; e < 4; ++e) y[4 * a + e] = w[(8 * a + 4 * half + e) * 33 + l32];
    T* pv = do_v + ((bh * NT + t) << 10) + lane * 16;
#pragma unroll
    for (int i = 0; i < NV; ++i) st16(pv + i * V, pack<T>(y + i * V));
}

// ------------------------------------------------------------------- triangle multiplication, output gate ----
// With s = sigmoid(gpre) and d = dz * drop[m % period]:  dab = d s,  dgpre = d ab s (1 - s).
template <typename T>
__global__ __launch_bounds__(TR_THREADS) void trimul_gate_bwd_kernel(T* __restrict__ dab, T* __restrict__ dgpre, const T* __restrict__ dz,
                                                                   const T* __restrict__ drop, unsigned period,
                                                                   const T* __restrict__ ab, const T* __restrict__ gpre, long rows, int C,
                                                                   long g_ld, long dg_ld) {
    constexpr int V = DT<T>::VEC;
    const int vpr = C / V;
    const long n = rows * vpr;
    for (long i = (long)blockIdx.x * TR_THREADS + threadIdx.x; i < n; i += (long)gridDim.x * TR_THREADS) {
        const long m = i / vpr;
        const int c = (int)(i - m * vpr) * V;
        float fd[V], fa[V], fg[V], o1[V], o2[V];
        unpack<T>(ld16(dz + i * V), fd);
        unpack<T>(ld16(ab + i * V), fa);
        unpack<T>(ld16(gpre + m * g_ld + c), fg);
        if (drop) {
            float fm[V];
            unpack<T>(ld16(drop + (long)((unsigned)m % period) * C + c), fm);
#pragma unroll
            for (int e = 0; e < V; ++e) fd[e] *= fm[e];
        }
#pragma unroll
        for (int e = 0; e < V; ++e) {
            const float s = sigmoid_f(fg[e]);
            o1[e] = fd[e] * s;
            o2[e] = fd[e] * fa[e] * s * (1.0f - s);
        }
        st16(dab + i * V, pack<T>(o1));
        st16(dgpre + m * dg_ld + c, pack<T>(o2));
    }
}

// ------------------------------------------------------------ triangle multiplication, gated projections ----
// The projections of one side are  l = mask proj sigmoid(gate)  (channel-major [c][i][k]); from dl and l and the gate's
// pre-activation rows:   dproj = dl mask s,   dgate = dl l (1 - s),   s = sigmoid(gate).
// A workgroup takes 64 k x 64 channels of one i: dl and l arrive along k, leave along the channels, transposed through LDS.
// Row (i, k) of the outputs and of the gate is i * r_i + k * r_k rows in (the incoming multiplication exchanges the two).
template <typename T>
__global__ __launch_bounds__(TR_THREADS) void glu_bwd_kernel(T* __restrict__ dproj, T* __restrict__ dgate, const T* __restrict__ dl,
                                                           const T* __restrict__ l, const T* __restrict__ gate,
                                                           const T* __restrict__ mask, int R, int C, long cs, int kpad, long d_ld,
                                                           long g_ld, long r_i, long r_k) {
    constexpr int V = DT<T>::VEC, CH = 64 / V;
    __shared__ __align__(16) float t_d[64 * 65], t_l[64 * 65];
    const int kt = (R + 63) / 64;
    const int k0 = (int)(blockIdx.x % kt) * 64, i = (int)(blockIdx.x / kt), c0 = (int)blockIdx.y * 64;
    for (int v = threadIdx.x; v < 64 * CH; v += TR_THREADS) {
        const int c = v / CH, k = (v % CH) * V;
        float a[V], b[V];
#pragma unroll
        for (int e = 0; e < V; ++e) a[e] = b[e] = 0.0f;
        if (k0 + k < kpad) {                                    // rows of the channel planes are whole 16-byte vectors
            const long o = (long)(c0 + c) * cs + (long)i * kpad + k0 + k;
            unpack<T>(ld16(dl + o), a);
            unpack<T>(ld16(l + o), b);
        }
#pragma unroll
        for (int e = 0; e < V; ++e) {
            t_d[(k + e) * 65 + c] = a[e];
            t_l[(k + e) * 65 + c] = b[e];
        }
    }
    __syncthreads();
    for (int v = threadIdx.x; v < 64 * CH; v += TR_THREADS) {
        const int k = v / CH, c = (v % CH) * V;
        if (k0 + k >= R) continue;
        const long row = (long)i * r_i + (long)(k0 + k) * r_k;
        float g[V], o1[V], o2[V];
        unpack<T>(ld16(gate + row * g_ld + c0 + c), g);
        const float mk = DT<T>::to_f(mask[row]);
#pragma unroll
        for (int e = 0; e < V; ++e) {
            const float d = t_d[k * 65 + c + e], s = sigmoid_f(g[e]);
            o1[e] = d * mk * s;
            o2[e] = d * t_l[k * 65 + c + e] * (1.0f - s);
        }
        st16(dproj + row * d_ld + c0 + c, pack<T>(o1));
        st16(dgate + row * d_ld + c0 + c, pack<T>(o2));
    }
}

// -------------------------------------------------------------------------- pair-bias gradient as columns ----
// out[m][0 .. 32): the sum over the parts of dbias[part][h][m] for h < H, zero behind (the columns a product over them pads
// with).  A workgroup takes 32 rows; its eight groups of 32 lanes one head at a time.
template <typename T>
__global__ __launch_bounds__(TR_THREADS) void bias_cols_kernel(T* __restrict__ out, const float* __restrict__ dbias, int parts, long rows,
                                                             int H, long ld) {
    __shared__ float t[32 * 33];
    const int l = threadIdx.x & 31;
    const long m0 = (long)blockIdx.x * 32, m = m0 + l < rows ? m0 + l : rows - 1;
    for (int h = threadIdx.x >> 5; h < 32; h += 8) {
        float s = 0.0f;
        if (h < H) {
#pragma unroll 4
            for (int p = 0; p < parts; ++p) s += dbias[((long)p * H + h) * rows + m];
        }
        t[l * 33 + h] = s;
    }
    __syncthreads();
    constexpr int V = DT<T>::VEC;
    for (int i = threadIdx.x; i < 32 * 32 / V; i += TR_THREADS) {
        const int r = i / (32 / V), c = (i % (32 / V)) * V;
        if (m0 + r >= rows) continue;
        float f[V];
#pragma unroll
        for (int e = 0; e < V; ++e) f[e] = t[r * 33 + c + e];
        st16(out + (m0 + r) * ld + c, pack<T>(f));
    }
}

inline unsigned tr_grid(long items) {
    const long b = (items + TR_THREADS - 1) / TR_THREADS;
    return (unsigned)(b < 1 ? 1 : (b < 256L * 32 ? b : 256L * 32));
}

template <typename T>
int ln_bwd_launch(T* dx, T* xn, T* dgamma, T* dbeta, float* ws, const T* dy, const T* x, const T* gamma, const T* beta,
                  const T* resid, long rows, int C, float eps, hipStream_t st) {
    const int rpb = TR_THREADS / (C / DT<T>::VEC);
    const long want = (rows + rpb - 1) / rpb;
    const int blocks = (int)(want < LN_BLOCKS ? want : LN_BLOCKS);
#define FFK_LN_BWD(CC)                                                                                                        \
    ln_bwd_rows_kernel<T, CC><<<blocks, TR_THREADS, 0, st>>>(dx, xn, ws, dy, x, gamma, beta, resid, rows, eps)
    switch (C) {
        case 64: FFK_LN_BWD(64); break;
        case 128: FFK_LN_BWD(128); break;
        case 256: FFK_LN_BWD(256); break;
        default: return ffk_fail(FFK_ERR_SHAPE, "ffk_layernorm_bwd_rows: C=%d (64, 128 or 256)", C);
    }
#undef FFK_LN_BWD
    int rc = ffk_check_launch("ffk_layernorm_bwd_rows");
    if (rc != FFK_OK) return rc;
    ln_finish_kernel<T><<<2 * C / 16, 256, 0, st>>>(dgamma, dbeta, ws, blocks, C);
    return ffk_check_launch("ffk_layernorm_bwd_rows");
}

template <typename T>
int scale_rows_launch(T* out, const T* x, const void* mul, long rows, int C, unsigned inner, long m_so, long m_si, int mode,
                      float eps, hipStream_t st) {
    const unsigned grid = tr_grid(rows * (C / DT<T>::VEC));
    if (mode == 0) scale_rows_kernel<T, 0><<<grid, TR_THREADS, 0, st>>>(out, x, mul, rows, C, inner, m_so, m_si, eps);
    else if (mode == 1) scale_rows_kernel<T, 1><<<grid, TR_THREADS, 0, st>>>(out, x, mul, rows, C, inner, m_so, m_si, eps);
    else scale_rows_kernel<T, 2><<<grid, TR_THREADS, 0, st>>>(out, x, mul, rows, C, inner, m_so, m_si, eps);
    return ffk_check_launch("ffk_scale_rows");
}

}  // namespace

#define FFK_TR_DISPATCH(name, CALL)                                                                     \
    switch (dtype) {                                                                                    \
        case FFK_BF16: { typedef bf16_t T; CALL; }                                                      \
        case FFK_F32: { typedef float T; CALL; }                                                        \
        default: return ffk_fail(FFK_ERR_DTYPE, name ": unsupported dtype tag %d", dtype);              \
    }

static bool tr_al(int dtype, std::initializer_list<const void*> ps, std::initializer_list<int64_t> strides) {
    for (const void* p : ps)
        if (!ffk_aligned16(p)) return false;
    for (int64_t s : strides)
        if (s % (dtype == FFK_F32 ? 4 : 8)) return false;
    return true;
}

extern "C" int ffk_layernorm_bwd_rows(void* dx, void* xn, void* dgamma, void* dbeta, float* ws, const void* dy, const void* x,
                                      const void* gamma, const void* beta, const void* resid, int64_t rows, int64_t C, float eps,
                                      int dtype, void* stream) {
    FFK_REQUIRE(dx && dgamma && dbeta && ws && dy && x && gamma && (beta || !xn), FFK_ERR_NULL, "ffk_layernorm_bwd_rows: null pointer");
    FFK_REQUIRE(rows > 0 && rows < (1L << 40), FFK_ERR_SHAPE, "ffk_layernorm_bwd_rows: bad shape [%ld,%ld]", (long)rows, (long)C);
    FFK_REQUIRE(tr_al(dtype, {dx, xn, dy, x, gamma, beta, resid}, {}), FFK_ERR_ALIGN, "ffk_layernorm_bwd_rows: buffers must be 16-byte aligned");
    FFK_TR_DISPATCH("ffk_layernorm_bwd_rows",
                    return ln_bwd_launch<T>((T*)dx, (T*)xn, (T*)dgamma, (T*)dbeta, ws, (const T*)dy, (const T*)x, (const T*)gamma,
                                            (const T*)beta, (const T*)resid, rows, (int)C, eps, (hipStream_t)stream))
}

extern "C" int ffk_scale_rows(void* out, const void* x, const void* mul, int64_t rows, int64_t C, int64_t inner, int64_t m_so,
                              int64_t m_si, int mode, float eps, int dtype, void* stream) {
    FFK_REQUIRE(out && x && mul, FFK_ERR_NULL, "ffk_scale_rows: null pointer");
    FFK_REQUIRE(rows > 0 && rows < (1L << 31) && C > 0 && C % 8 == 0 && inner > 0 && mode >= 0 && mode <= 2, FFK_ERR_SHAPE,
                "ffk_scale_rows: bad shape [%ld,%ld], inner %ld, mode %d", (long)rows, (long)C, (long)inner, mode);
    FFK_REQUIRE(tr_al(dtype, {out, x}, {}) && (mode != 0 || tr_al(dtype, {mul}, {m_so, m_si})), FFK_ERR_ALIGN,
                "ffk_scale_rows: rows must be 16-byte aligned");
    FFK_TR_DISPATCH("ffk_scale_rows", return scale_rows_launch<T>((T*)out, (const T*)x, mul, rows, (int)C,
                                                                  (unsigned)(inner < rows ? inner : rows), m_so, m_si, mode, eps,
                                                                  (hipStream_t)stream))
}

extern "C" int ffk_att_gate_bwd(void* go, void* dgpre, void* do_t, void* do_v, float* dsum, const void* dgo, const void* gpre,
                                const void* gbias, const void* o, int64_t B2, int64_t N, int64_t H, int64_t g_ld, int64_t dg_ld,
                                int dtype, void* stream) {
    FFK_REQUIRE(go && dgpre && do_t && do_v && dsum && dgo && gpre && gbias && o, FFK_ERR_NULL, "ffk_att_gate_bwd: null pointer");
    FFK_REQUIRE(B2 > 0 && N > 0 && H > 0 && B2 < (1 << 24) && N < (1 << 24) && H < 1024, FFK_ERR_SHAPE,
                "ffk_att_gate_bwd: bad shape B2=%ld N=%ld H=%ld", (long)B2, (long)N, (long)H);
    FFK_REQUIRE(tr_al(dtype, {go, dgpre, do_t, do_v, dgo, gpre, gbias, o}, {g_ld, dg_ld}), FFK_ERR_ALIGN,
                "ffk_att_gate_bwd: rows must be 16-byte aligned");
    const long items = B2 * ((N + 31) / 32) * H;
    FFK_REQUIRE(items < (1L << 32), FFK_ERR_SHAPE, "ffk_att_gate_bwd: too many tiles for one launch");
    FFK_TR_DISPATCH("ffk_att_gate_bwd",
                    (att_gate_bwd_kernel<T><<<(unsigned)((items + 3) / 4), TR_THREADS, 0, (hipStream_t)stream>>>(
                        (T*)go, (T*)dgpre, (T*)do_t, (T*)do_v, dsum, (const T*)dgo, (const T*)gpre, (const T*)gbias, (const T*)o, B2,
                        (int)N, (int)H, g_ld, dg_ld));
                    return ffk_check_launch("ffk_att_gate_bwd"))
}

extern "C" int ffk_trimul_gate_bwd(void* dab, void* dgpre, const void* dz, const void* drop, const void* ab, const void* gpre,
                                   int64_t rows, int64_t C, int64_t period, int64_t g_ld, int64_t dg_ld, int dtype, void* stream) {
    FFK_REQUIRE(dab && dgpre && dz && ab && gpre, FFK_ERR_NULL, "ffk_trimul_gate_bwd: null pointer");
    FFK_REQUIRE(rows > 0 && rows < (1L << 31) && C > 0 && C % 8 == 0 && period > 0 && period <= rows, FFK_ERR_SHAPE,
                "ffk_trimul_gate_bwd: bad shape [%ld,%ld], period %ld", (long)rows, (long)C, (long)period);
    FFK_REQUIRE(tr_al(dtype, {dab, dgpre, dz, drop, ab, gpre}, {g_ld, dg_ld}), FFK_ERR_ALIGN, "ffk_trimul_gate_bwd: rows must be 16-byte aligned");
    FFK_TR_DISPATCH("ffk_trimul_gate_bwd",
                    (trimul_gate_bwd_kernel<T><<<tr_grid(rows * C / DT<T>::VEC), TR_THREADS, 0, (hipStream_t)stream>>>(
                        (T*)dab, (T*)dgpre, (const T*)dz, (const T*)drop, (unsigned)period, (const T*)ab, (const T*)gpre, rows, (int)C,
                        g_ld, dg_ld));
                    return ffk_check_launch("ffk_trimul_gate_bwd"))
}

extern "C" int ffk_glu_bwd(void* dproj, void* dgate, const void* dl, const void* l, const void* gate, const void* mask, int64_t R,
                           int64_t C, int64_t cs, int64_t kpad, int64_t d_ld, int64_t g_ld, int64_t r_i, int64_t r_k, int dtype,
                           void* stream) {
    FFK_REQUIRE(dproj && dgate && dl && l && gate && mask, FFK_ERR_NULL, "ffk_glu_bwd: null pointer");
    FFK_REQUIRE(R > 0 && R < (1 << 20) && C > 0 && C % 64 == 0 && C < (1 << 20) && kpad >= R, FFK_ERR_SHAPE,
                "ffk_glu_bwd: bad shape R=%ld C=%ld kpad=%ld", (long)R, (long)C, (long)kpad);
    FFK_REQUIRE(tr_al(dtype, {dproj, dgate, dl, l, gate}, {cs, kpad, d_ld, g_ld}), FFK_ERR_ALIGN, "ffk_glu_bwd: rows must be 16-byte aligned");
    const dim3 grid((unsigned)(((R + 63) / 64) * R), (unsigned)(C / 64));
    FFK_TR_DISPATCH("ffk_glu_bwd",
                    (glu_bwd_kernel<T><<<grid, TR_THREADS, 0, (hipStream_t)stream>>>(
                        (T*)dproj, (T*)dgate, (const T*)dl, (const T*)l, (const T*)gate, (const T*)mask, (int)R, (int)C, cs, (int)kpad,
                        d_ld, g_ld, r_i, r_k));
                    return ffk_check_launch("ffk_glu_bwd"))
}

extern "C" int ffk_bias_cols(void* out, const float* dbias, int64_t parts, int64_t rows, int64_t H, int64_t ld, int dtype, void* stream) {
    FFK_REQUIRE(out && dbias, FFK_ERR_NULL, "ffk_bias_cols: null pointer");
    FFK_REQUIRE(parts > 0 && rows > 0 && rows < (1L << 36) && H > 0 && H <= 32, FFK_ERR_SHAPE, "ffk_bias_cols: bad shape rows=%ld H=%ld", (long)rows, (long)H);
    FFK_REQUIRE(tr_al(dtype, {out}, {ld}), FFK_ERR_ALIGN, "ffk_bias_cols: rows must be 16-byte aligned");
    FFK_TR_DISPATCH("ffk_bias_cols",
                    (bias_cols_kernel<T><<<(unsigned)((rows + 31) / 32), TR_THREADS, 0, (hipStream_t)stream>>>((T*)out, dbias, (int)parts, rows,
                                                                                             (int)H, ld));
                    return ffk_check_launch("ffk_bias_cols"))
}
