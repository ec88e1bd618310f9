// Flash-style attention for head dimension 32 (see ffk_attention_fwd in include/ffk.h).
//
// One wavefront owns 32 queries of one (b2, head) and walks the keys 32 at a time.  Every
// operand is stored in HBM in exactly the order a wave consumes it (1024-element tiles, 16
// contiguous elements per lane); the eight waves of a workgroup share their operand tiles
// through a double-buffered LDS stage (see attention_kernel).
//
// The score tile is computed transposed, S^T = K . Q^T (rows = keys, columns = queries):
// a lane then holds 16 keys of ONE query, so the running max / sum are per-lane scalars
// (one cross-half shuffle per tile), and exp2(S^T - max) is already in the operand layout
// of the second MFMA  O^T += V^T . P^T  - no transpose of P.  The additive bias tile is
// stored as an MFMA operand (keys x queries) and added to S^T by one more MFMA against the
// identity: the matrix pipe has slack here (head dim 32 makes the kernel VALU / exp bound), the
// vector pipe has none.  Per-tile flags skip the key-mask add for tiles without masked keys and
// drop trailing fully-masked tiles; the running output is rescaled only when a row maximum moves.
#include "ffk_common.h"
#include <type_traits>

namespace {

constexpr float NEG_BIG = -3.0e38f;

template <typename T> struct Ops16 {   // the 16 elements one lane owns of a 1024-element tile
    static constexpr int NV = 16 / DT<T>::VEC;
    Vec16<T> v[NV];
    __device__ __forceinline__ void load(const T* p) {
#pragma unroll
        for (int i = 0; i < NV; ++i) v[i] = ld16(p + i * DT<T>::VEC);
    }
    // the same 16 elements from a tile kept in LDS vector-interleaved: vector i of lane l at (i * 64 + l)
    // * 16 bytes, so that the 64 lanes of one read touch 1 KB of consecutive addresses (the tile's own
    // order, 32 or 64 bytes from lane to lane, makes every 16-byte read a two- or four-way bank conflict)
    __device__ __forceinline__ void load_lds(const T* tile, int lane) {
#pragma unroll
        for (int i = 0; i < NV; ++i) v[i] = ld16(tile + (i * 64 + lane) * DT<T>::VEC);
    }
    __device__ __forceinline__ float f(int j) const { return DT<T>::to_f(v[j / DT<T>::VEC].e[j % DT<T>::VEC]); }
    // MFMA fragment number i (KLANE elements each)
    __device__ __forceinline__ typename Mma<T>::Frag frag(int i) const {
        return *reinterpret_cast<const typename Mma<T>::Frag*>(&v[i]);
    }
};

template <typename T> struct PFrag;
template <> struct PFrag<bf16_t> {
    static __device__ __forceinline__ bf16x8 make(const float* p) {
        bf16x8 r;
#pragma unroll
        for (int t = 0; t < 8; ++t) r[t] = (bf16_t)p[t];
        return r;
    }
    // acc + sum of the eight rounded probabilities (the values the PV product really uses), two
    // per instruction
    static __device__ __forceinline__ float add_sum(const bf16x8& f, float acc) {
        typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
        const bf16x2 ones = {(bf16_t)1.0f, (bf16_t)1.0f};
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const bf16x2 pr = {f[2 * t], f[2 * t + 1]};
            acc = __builtin_amdgcn_fdot2_f32_bf16(pr, ones, acc, false);
        }
        return acc;
    }
};
template <> struct PFrag<float> {
    static __device__ __forceinline__ f32x4 make(const float* p) {
        f32x4 r;
#pragma unroll
        for (int t = 0; t < 4; ++t) r[t] = p[t];
        return r;
    }
    static __device__ __forceinline__ float add_sum(const f32x4& f, float acc) {
        return acc + ((f[0] + f[1]) + (f[2] + f[3]));
    }
};

// One-hot fragments of the 32x32 identity in N-operand layout: lane (column q = l & 31, K-group
// kg = l >> 5) holds rows j = 16 * kg + i * KLANE + t; the entry is 1 where j == q.  Multiplying a
// bias tile stored in M-operand order by it adds the tile to the score accumulator on the matrix
// pipe, with no conversion or VALU work.
template <typename T>
__device__ __forceinline__ typename Mma<T>::Frag identity_frag(int i, int l32, int half) {
    typename Mma<T>::Frag f;
#pragma unroll
    for (int t = 0; t < Mma<T>::KLANE; ++t) f[t] = (T)((16 * half + i * Mma<T>::KLANE + t) == l32 ? 1.0f : 0.0f);
    return f;
}

// Workgroup = 8 wavefronts = 2 batch rows x 4 query tiles of one head.  Per 32-key step the
// workgroup needs the K and V tiles of its two batch rows and the bias tiles of its four query
// tiles: 8 operand tiles, each consumed by 4 (K, V) or 2 (bias) waves.  They are fetched from
// global memory once per workgroup (two 16-byte loads per thread), double-buffered in LDS, and read
// from there by the waves in exactly the lane order of the MFMA operands, which divides the
// traffic through the vector memory path by three compared with per-wave global loads.
constexpr int ATT_WAVES = 8;
constexpr int ATT_THREADS = 64 * ATT_WAVES;

// HD < 32: heads of 16 or 8 channels, packed two or four to an operand tile (head h is channels HD * (h % G) .. of tile h / G).
// A wave takes its head's share of the packed tiles: the one fragment of k its channels lie in (for HD = 8 with the other head's
// half of q zeroed), and the accumulator registers of its channels from the product with v, whose other rows it drops - the
// kernel is bound by exp2 and by what it reads, and padding such heads to 32 channels made q, k, v and the gate two to four
// times as large (extra-MSA row attention, 1 024 x 384, 8 heads of 8, padded -> packed: projection 185 -> 67 us, core 347 ->
// 259 .. 279 us, output projection 85 -> 43 us).
template <typename T, bool HAS_BIAS, int HD>
__global__ __launch_bounds__(ATT_THREADS, sizeof(T) == 2 ? 4 : 2) void attention_kernel(
    T* __restrict__ out, const T* __restrict__ q_t, const T* __restrict__ k_t, const T* __restrict__ v_t,
    const T* __restrict__ bias_t, const float* __restrict__ keybias, const int* __restrict__ tileflags,
    const T* __restrict__ gate, float* __restrict__ lse, int B2, int H, int Nq, int Nk, int flags) {
    typedef Mma<T> MM;
    typedef typename MM::Frag Frag;
    constexpr int NF = 16 / MM::KLANE;            // fragments per 16-element lane slice (bf16 2, fp32 4)
    constexpr int VEC = DT<T>::VEC;
    constexpr int NTILES = HAS_BIAS ? 8 : 4;      // operand tiles per key step: K0 K1 V0 V1 [B0 B1 B2 B3]
    constexpr int TILE_VECS = 1024 / VEC;         // 16-byte vectors per tile
    constexpr int NVL = (NTILES * TILE_VECS + ATT_THREADS - 1) / ATT_THREADS;   // vectors per thread per step
    extern __shared__ __align__(16) unsigned char att_smem[];
    constexpr int NSLOT = 3;                      // operand ring: the tile in use and two in flight behind it
    // fp32: the bias is added to the scores as it is read (16 LDS reads and additions a lane and tile).  Through the matrix pipe, as
    // in bf16, where it costs two products of 32 cycles, it was a third of all products: 16 of 64 cycles.  128 x 8 heads of 256 x 256:
    // 121.8 -> 97.3 us, 391 x 391 355 -> 274.  Its tiles lie [query][key] transposed to what a lane needs (16 keys of one query); the 16-byte pieces of a tile go
    // to LDS permuted, so that the lanes of a read - four adjacent queries to a piece - meet 16 pieces in 16 bank groups.
    constexpr bool BIAS_ADD = HAS_BIAS && sizeof(T) == 4;
    T* lds = reinterpret_cast<T*>(att_smem);      // [NSLOT][NTILES][1024] operand slots, then [ATT_THREADS][16] gate values

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // wave-uniform: everything derived from it stays scalar
    const int l32 = lane & 31, half = lane >> 5;
    const int bsel = wave >> 2, qsel = wave & 3;
    const int QT = (Nq + 31) >> 5, KT = (Nk + 31) >> 5;
    // Workgroup -> work mapping.  The hardware hands consecutive workgroup ids to the eight XCDs in
    // turn, and each XCD has its own L2.  Logical work items are ordered (head, batch-row pair,
    // query group) and every XCD takes one contiguous eighth of that order, so that the query groups
    // that share a K / V pair and the batch rows that share a head's bias run behind the same L2.
    const int NQG = (QT + 3) >> 2, NZ = (B2 + 1) >> 1;
    const unsigned total = (unsigned)NQG * H * NZ, per_xcd = (total + 7) >> 3;
    const unsigned item = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (item >= total) return;                    // whole workgroup leaves together
    constexpr int G = 32 / HD;                    // heads per operand tile; those of one tile and batch-row pair run together
    const int wg_q = item % NQG, rest = item / NQG;
    const int wg_z = (rest / G) % NZ;
    const int ht = (rest / G) / NZ, Ht = H / G, h = ht * G + rest % G;
    const int c0 = HD * (rest % G);               // first channel of the head in its tile
    const int b2_raw = wg_z * 2 + bsel, qt_raw = wg_q * 4 + qsel;
    const bool live = b2_raw < B2 && qt_raw < QT;      // dead waves still help loading and keep the barriers
    const int b2 = b2_raw < B2 ? b2_raw : B2 - 1;
    const int qt = qt_raw < QT ? qt_raw : QT - 1;
    const long bh = (long)b2 * Ht + ht;

    Ops16<T> qf;
    qf.load(q_t + ((bh * QT + qt) << 10) + lane * 16);
    if constexpr (HD < 32) {                      // v[0]: the fragment with the head's channels
        if (c0 >= 16) qf.v[0] = qf.v[1];
        if constexpr (HD == 8) {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if ((e >> 2) != ((c0 >> 3) & 1)) qf.v[0].e[e] = DT<T>::from_f(0.0f);
        }
    }
    const float* mp = keybias + (long)b2 * KT * 32 + 4 * half;
    const int* fl = tileflags + (long)b2 * KT;

    // cooperative operand fetch: vector slot v = tid + i * ATT_THREADS -> (tile, vector in tile).  The
    // 16-byte vectors go from global memory straight into LDS (no staging registers); the hardware places
    // the 64 vectors of a request at  base + 16 * lane,  while the source address is per lane: a request
    // gathers vector c of each lane's 16 elements (stride 16 * NV bytes), which leaves the tile in LDS
    // vector-interleaved (see Ops16::load_lds).
    static_assert(NVL * ATT_THREADS == NTILES * TILE_VECS, "every thread fetches the same number of vectors");
    const T* src[NVL];                            // wave-uniform: start of the wave's 64 vectors in key tile 0
#pragma unroll
    for (int i = 0; i < NVL; ++i) {
        const int v = wave * 64 + i * ATT_THREADS;
        const int tile = v / TILE_VECS, wv = v % TILE_VECS;
        const T* base;
        if (tile < 4) {
            int bb = wg_z * 2 + (tile & 1);
            bb = bb < B2 ? bb : B2 - 1;
            base = (tile < 2 ? k_t : v_t) + ((((long)bb * Ht + ht) * KT) << 10);
        } else {
            int qq = wg_q * 4 + (tile - 4);
            qq = qq < QT ? qq : QT - 1;
            // FFK_ATT_BIAS_PADDED: one unused tile after the KT tiles of each query-tile row
            base = bias_t + ((((long)h * QT + qq) * (KT + ((flags >> 1) & 1))) << 10);
        }
        // the wave's 64 vectors of this request: vector number wv / 64 of every lane's 16 elements
        src[i] = base + (wv / 64) * VEC;
    }

    // gate values of this lane's 16 outputs, fetched now so that their latency is hidden by the loop
    const int q = qt * 32 + l32;
    const int qc = q < Nq ? q : Nq - 1;
    const long rowo = ((long)b2 * Nq + qc) * (H * HD) + ht * 32 + 4 * half;
    // They wait in LDS (each lane's own 16 values), not in registers.
    T* gate_lds = lds + NSLOT * NTILES * 1024 + tid * 16;
    if (gate) {
        T gv[4][4];
        if (flags & FFK_ATT_GATE_TILED) {
            // accumulator-order tile: this lane's 16 values are contiguous
            const T* gp = gate + ((bh * QT + qt) << 10) + lane * 16;
            if (sizeof(T) == 2) {
                *reinterpret_cast<u32x4*>(&gv[0][0]) = *reinterpret_cast<const u32x4*>(gp);
                *reinterpret_cast<u32x4*>(&gv[2][0]) = *reinterpret_cast<const u32x4*>(gp + 8);
            } else {
#pragma unroll
                for (int g = 0; g < 4; ++g) *reinterpret_cast<u32x4*>(&gv[g][0]) = *reinterpret_cast<const u32x4*>(gp + 4 * g);
            }
        } else {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                if (sizeof(T) == 2) {
                    *reinterpret_cast<u32x2*>(&gv[g][0]) = *reinterpret_cast<const u32x2*>(gate + rowo + 8 * g);
                } else {
                    *reinterpret_cast<u32x4*>(&gv[g][0]) = *reinterpret_cast<const u32x4*>(gate + rowo + 8 * g);
                }
            }
        }
#pragma unroll
        for (int i = 0; i < 16 / VEC; ++i)
            *reinterpret_cast<u32x4*>(gate_lds + i * VEC) = *reinterpret_cast<const u32x4*>(&gv[0][0] + i * VEC);
    }

    // trailing key tiles that are completely masked in both batch rows contribute exactly zero
    int kt_end = KT;
    {
        const int* f0 = tileflags + (long)(wg_z * 2 < B2 ? wg_z * 2 : B2 - 1) * KT;
        const int* f1 = tileflags + (long)(wg_z * 2 + 1 < B2 ? wg_z * 2 + 1 : B2 - 1) * KT;
        while (kt_end > 1 && f0[kt_end - 1] == 2 && f1[kt_end - 1] == 2) --kt_end;
    }

    Frag ident[NF];
    if (HAS_BIAS && !BIAS_ADD) {
#pragma unroll
        for (int i = 0; i < NF; ++i) ident[i] = identity_frag<T>(i, l32, half);
    }

    // Online softmax with a lazily updated reference.  Instead of subtracting the running row maximum
    // from every score on the vector pipe, the negated reference  -m_ref[q]  is the C operand of the
    // first MFMA of each tile, so the accumulator already holds  s - m_ref  and exp2 is applied to it
    // directly.  m_ref is only moved (and O / l rescaled) when the probabilities of a tile show that
    // a score lies more than REF_SLACK above it, which bounds  p = exp2(s - m_ref) <= 2^REF_SLACK
    // in everything that is accumulated;  the first tile always sets it.
    constexpr float REF_LIMIT = 1048576.0f;       // 2^REF_SLACK, REF_SLACK = 20
    constexpr float REF_FLOOR = -1.0e4f;          // keeps m_ref small when the first tile is fully masked
    f32x16 o_acc, negm;
#pragma unroll
    for (int v = 0; v < 16; ++v) o_acc[v] = negm[v] = 0.0f;
    float l_run = 0.0f;                           // partial row sum of this lane's 16 keys per tile
    bool first = true;

    // The loads are issued from an asm statement on purpose: the compiler orders every later LDS read
    // after all outstanding loads of this kind it knows of (a full s_waitcnt vmcnt(0) right behind
    // the issue), while here the slot being filled is never the slot being read.  The explicit wait
    // at the top of the loop is what orders them.
    const unsigned lds_base = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)att_smem;
    const unsigned lane_off = lane * 16 * Ops16<T>::NV;   // byte offset of this lane's 16 elements; the base address is scalar
    // piece c of lane L's 16 elements (key L % 32, queries 16 (L / 32) + 4 c ..) goes to place L ^ (c + 8 (L / 32)); a wave fetches one c
    const unsigned bias_off = BIAS_ADD ? (lane ^ ((wave & 3) | half << 3)) * 16 * Ops16<T>::NV : lane_off;
    static_assert(!BIAS_ADD || (TILE_VECS == 256 && ATT_THREADS == 512), "vectors of a wave's requests: number wave % 4 of every lane");
    const int bq = (l32 & 15) >> 2, bhi = l32 >> 4;            // this lane's query: piece and half of the bias tile's rows
    const T* bias_lane = lds + (4 + qsel) * 1024 + (bq * 64 + bhi * 32 + half * 4) * 4 + (l32 & 3);
    auto fetch = [&](int kt, int slot) {
#pragma unroll
        for (int i = 0; i < NVL; ++i) {
            const T* gp = src[i] + ((long)kt << 10);
            const unsigned dst = lds_base + (slot * NTILES * TILE_VECS + wave * 64 + i * ATT_THREADS) * 16;
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
            asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(BIAS_ADD && i * ATT_THREADS >= 4 * TILE_VECS ? bias_off : lane_off), "s"(gp), "s"(dst)
                         : "memory", "m0");
#pragma clang diagnostic pop
        }
    };

    // Every load the compiler knows of (q fragments, gate) is made to complete here: a wait it would
    // otherwise place at the first use inside the loop would also wait for the operand loads issued
    // just before that use.
#pragma unroll
    for (int i = 0; i < Ops16<T>::NV; ++i) asm volatile("" : "+v"(*reinterpret_cast<u32x4*>(&qf.v[i])));
    // The walk over the key tiles.  CAREFUL = false is the common case: the first tile sets the reference and no
    // later tile looks at its probabilities - the row sum is tested once, after the walk (see below).
    auto walk = [&](auto careful_c) {
    constexpr bool CAREFUL = decltype(careful_c)::value;
    fetch(0, 0);
    fetch(kt_end > 1 ? 1 : 0, 1);
    int flag_nxt = fl[0];
    int slot = 0;                                 // ring slot of tile kt
    for (int kt = 0; kt < kt_end; ++kt) {
        // Tile kt was requested two steps ago: wait until only the newest request (tile kt + 1) of this
        // thread is still in flight, then the barrier publishes tile kt and retires the slot of tile kt - 1.
        if (NVL == 1) asm volatile("s_waitcnt vmcnt(1)" ::: "memory");
        else if (NVL == 2) asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
        const int flag = __builtin_amdgcn_readfirstlane(flag_nxt);
        lds_barrier();
        const int nxt = kt + 1 < kt_end ? kt + 1 : kt;
        const int nxt2 = kt + 2 < kt_end ? kt + 2 : kt_end - 1;
        fetch(nxt2, slot == 0 ? 2 : slot - 1);    // (slot + 2) % 3: the slot tile kt - 1 was read from
        flag_nxt = fl[nxt];
        const T* buf = lds + slot * NTILES * 1024;
        slot = slot == 2 ? 0 : slot + 1;
        Ops16<T> vc;
        vc.load_lds(buf + (2 + bsel) * 1024, lane);

        // S^T - m_ref = K . Q^T + Bias^T . I + (-m_ref)   (rows: keys, columns: queries)
        f32x16 s;
        auto score_tile = [&]() {
            Ops16<T> kc, bc;
            if constexpr (HD == 32) kc.load_lds(buf + bsel * 1024, lane);
            else kc.v[0] = ld16(buf + bsel * 1024 + ((c0 >> 4) * 64 + lane) * VEC);
            if (HAS_BIAS && !BIAS_ADD) bc.load_lds(buf + (4 + qsel) * 1024, lane);
            float ba[BIAS_ADD ? 16 : 1];
            if constexpr (BIAS_ADD) {                          // key 8 g + 4 half + e of the tile, at place key ^ (bq + 8 bhi)
                const T* bp = bias_lane + (buf - lds);
#pragma unroll
                for (int g = 0; g < 4; ++g)
#pragma unroll
                    for (int e = 0; e < 4; ++e) ba[4 * g + e] = (float)bp[((8 * g ^ 8 * bhi) + (e ^ bq)) * 4];
            }
            s = negm;
            // FFK_ATT_HALF_K: elements 8 .. 15 of every lane's sixteen are zero padding in q and k (narrow heads): the
            // second half of the score product adds nothing and is skipped
#pragma unroll
            for (int i = 0; i < NF / 2; ++i) MM::mma(s, kc.frag(i), qf.frag(i));
            if (HD == 32 && !(flags & FFK_ATT_HALF_K)) {
#pragma unroll
                for (int i = NF / 2; i < NF; ++i) MM::mma(s, kc.frag(i), qf.frag(i));
            }
            if constexpr (BIAS_ADD) {
#pragma unroll
                for (int v = 0; v < 16; ++v) s[v] += ba[v];
            } else if (HAS_BIAS) {
#pragma unroll
                for (int i = 0; i < NF; ++i) MM::mma(s, bc.frag(i), ident[i]);
            }
            if (flag != 0) {         // some key of this tile is masked or padding: add the key bias
                f32x4 mk[4];
#pragma unroll
                for (int g = 0; g < 4; ++g) mk[g] = *reinterpret_cast<const f32x4*>(mp + kt * 32 + 8 * g);
#pragma unroll
                for (int g = 0; g < 4; ++g)
#pragma unroll
                    for (int e = 0; e < 4; ++e) s[4 * g + e] += mk[g][e];
            }
        };
        // P^T = exp2(S^T - m_ref) rounded to the operand type, and the sum of this lane's 16 rounded values
        Frag pf[NF];
        float tsum;
        auto prob_tile = [&]() {
            float p[16];
#pragma unroll
            for (int v = 0; v < 16; ++v) p[v] = fast_exp2(s[v]);
            tsum = 0.0f;
#pragma unroll
            for (int i = 0; i < NF; ++i) {
                pf[i] = PFrag<T>::make(p + i * MM::KLANE);
                tsum = PFrag<T>::add_sum(pf[i], tsum);
            }
        };
        // No maximum is taken on the common path: probabilities are non-negative, so a partial row sum
        // within 2^REF_SLACK proves that no score of the tile is more than REF_SLACK above the reference.
        // Only when some lane's sum exceeds that (or on the first tile, which sets the reference) is
        // the tile recomputed from its LDS slot, the reference moved to the row maximum and O / l rescaled.
        score_tile();
        bool move_ref = first, fresh = first;
        if (!first) {
            prob_tile();
            if (CAREFUL) {
                move_ref = __builtin_amdgcn_ballot_w64(!(tsum <= REF_LIMIT)) != 0;
                if (move_ref) {
                    // A row that has met no key so far stands at the floor, beside which a score keeps three decimals: its
                    // scores are taken again without a reference.
                    fresh = negm[0] == -REF_FLOOR;
                    if (fresh) {
#pragma unroll
                        for (int v = 0; v < 16; ++v) negm[v] = 0.0f;
                    }
                    score_tile();
                }
            }
        }
        if (move_ref) {
            float mt = fmaxf(s[0], s[1]);
#pragma unroll
            for (int v = 2; v < 16; ++v) mt = fmaxf(mt, s[v]);
            const float mfull = fmaxf(mt, lane_xor<32>(mt));
            const float delta = fmaxf(mfull, fresh ? REF_FLOOR : 0.0f);
            const float alpha = first ? 1.0f : fast_exp2((fresh ? REF_FLOOR : 0.0f) - delta);   // nothing accumulated before the first tile
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                s[v] -= delta;
                negm[v] -= delta;
                o_acc[v] *= alpha;
            }
            l_run *= alpha;
            first = false;
            prob_tile();
        }
        l_run += tsum;
        // O^T += V^T . P^T   (rows: head dim, columns: queries)
#pragma unroll
        for (int i = 0; i < NF; ++i) MM::mma(o_acc, vc.frag(i), pf[i]);

    }
    // the requests past the last tile must have landed before the ring is reused or handed on
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    };

    // Optimistic walk first.  Probabilities are non-negative, so a finite row sum within 2^OPT_SLACK proves that
    // no score of the row lay more than OPT_SLACK (log2 units) above the first tile's maximum: nothing overflowed,
    // and fp32 accumulation keeps its relative precision at any such scale.  Otherwise (steeply rising scores, a
    // first tile that is completely masked) the whole workgroup walks again with the reference moved tile by tile.
    walk(std::false_type());
    {
        constexpr float OPT_LIMIT = 1.8446744e19f;    // 2^64
        int* redo = reinterpret_cast<int*>(lds + NSLOT * NTILES * 1024 + ATT_THREADS * 16);
        if (tid == 0) *redo = 0;
        lds_barrier();
        const bool bad = __builtin_amdgcn_ballot_w64(!(l_run <= OPT_LIMIT)) != 0;
        if (bad && lane == 0) *redo = 1;
        lds_barrier();
        if (*redo != 0) {                              // workgroup-uniform
            lds_barrier();
#pragma unroll
            for (int v = 0; v < 16; ++v) o_acc[v] = negm[v] = 0.0f;
            l_run = 0.0f;
            first = true;
            walk(std::true_type());
        }
    }

    // rows whose keys are all masked have l == 0 and produce zeros
    const float l_tot = l_run + lane_xor<32>(l_run);
    const float inv = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
    // log-sum-exp of the row (log2 domain) for the backward kernels; an all-masked row's makes every exp2(s - lse) zero
    if (lse && live && half == 0)
        lse[(bh * QT + qt) * 32 + l32] = l_tot > 0.0f ? __builtin_amdgcn_logf(l_tot) - negm[0] : 3.0e38f;
    if (live && q < Nq) {
        T gv[4][4];
        if (gate) {
#pragma unroll
            for (int i = 0; i < 16 / VEC; ++i)
                *reinterpret_cast<u32x4*>(&gv[0][0] + i * VEC) = *reinterpret_cast<const u32x4*>(gate_lds + i * VEC);
        }
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            if (HD < 32 && (8 * g < c0 || 8 * g >= c0 + HD)) continue;        // another head's channels
            T r4[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float x = o_acc[4 * g + e] * inv;
                if (gate) x *= DT<T>::to_f(gv[g][e]);
                r4[e] = DT<T>::from_f(x);
            }
            if (sizeof(T) == 2) {
                *reinterpret_cast<u32x2*>(out + rowo + 8 * g) = *reinterpret_cast<const u32x2*>(r4);
            } else {
                *reinterpret_cast<u32x4*>(out + rowo + 8 * g) = *reinterpret_cast<const u32x4*>(r4);
            }
        }
    }
}

constexpr int PAIR_THREADS = 256;

// bf16 heads of 32 channels with a bias: a wave owns 32 queries of one head in TWO batch rows, two waves per SIMD.  The kernel above
// takes the sum of its matrix and vector instructions (its waves leave a barrier together and then all wait for scores, all for
// exp2), although one hides the other where both are at hand: six products, 18 exp2 and 24 other vector instructions of a wave in
// turns take 133 ns, one kind after the other 203.  So here the scores of step kt + 1 are made while step kt is exponentiated, one
// row's products beside the other row's exponentials, in an order that is written down; K and the bias of a step are read a step
// ahead of V (four ring slots), and products go first where two waves ask (s_setprio: 2 %).  The bias tile is multiplied by the
// identity once for both rows: its accumulator is the C operand of their scores (five products per tile, not six), which leaves no
// place for a row's reference, so the reference is zero.  Sums of exp2 within OPT_LOW .. OPT_HIGH prove that no probability over- or
// underflowed, weighted sums that are numbers and, where the row's sum is below one, not all below OUT_LOW that no product with v did
// (large v beside a large sum, small v beside a small one); a workgroup with queries that lack that proof walks again with a running
// maximum, for them alone.
// Before -> after, us: 64 rows x 4 heads of 4 096 queries 888 -> 780, 1 024 x 4 of 1 024 984 -> 920, 391 x 4 of 391 99 -> 94, 320 x 4 of 320
// 53.0 -> 49.0.  Of the 190 ns a tile takes at 4 096 queries its instructions take 148, LDS 14, the barrier 7 and
// the ring's requests the rest.  Without a bias (212 -> 213 us, 128 x 8 of 1 024) the kernel above stays.  Workgroup = 2 batch rows x 4
// query tiles, two per CU (one of 4 x 4 leaves the CU idle at its start and end: 985 us at 1 024 queries).
__global__ __launch_bounds__(PAIR_THREADS, 2) void attention_pair_kernel(
    bf16_t* __restrict__ out, const bf16_t* __restrict__ q_t, const bf16_t* __restrict__ k_t, const bf16_t* __restrict__ v_t,
    const bf16_t* __restrict__ bias_t, const float* __restrict__ keybias, const int* __restrict__ tileflags,
    const bf16_t* __restrict__ gate, int B2, int H, int Nq, int Nk, int flags) {
    typedef Mma<bf16_t> MM;
    constexpr int NTILES = 8;                     // operand tiles per key step: K0 K1 V0 V1 B0 .. B3
    constexpr int NVL = 4, NSLOT = 4;             // 16-byte vectors per thread and step
    constexpr float OPT_HIGH = 1.2676506e30f, OPT_LOW = 8.2718061e-25f;        // 2^100, 2^-80
    constexpr unsigned OUT_LOW = 27u << 23;       // 2^-100
    constexpr float REF_FLOOR = -1.0e4f;
    extern __shared__ __align__(16) unsigned char att_smem[];
    bf16_t* lds = reinterpret_cast<bf16_t*>(att_smem);       // [NSLOT][NTILES][1024]

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    const int QT = (Nq + 31) >> 5, KT = (Nk + 31) >> 5;
    const int NQG = (QT + 3) >> 2, NZ = (B2 + 1) >> 1;
    const unsigned total = (unsigned)NQG * H * NZ, per_xcd = (total + 7) >> 3;
    const unsigned item = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);      // as above
    if (item >= total) return;                    // whole workgroup leaves together
    // (head, eight query groups, row pair, query group): the 64 workgroups an XCD holds share the bias of eight groups and the keys of
    // eight pairs.  With all query groups of a pair first, 4 096 queries read their bias anew for every two pairs.
    const int h = item / (NQG * NZ), in_head = item - h * (NQG * NZ), qb = in_head / (8 * NZ) * 8, in_block = in_head - qb * NZ;
    const int width = NQG - qb < 8 ? NQG - qb : 8, wg_z = in_block / width, wg_q = qb + in_block - wg_z * width;
    const int qt_raw = wg_q * 4 + wave, qt = qt_raw < QT ? qt_raw : QT - 1;
    const int q = qt * 32 + l32, qc = q < Nq ? q : Nq - 1;
    int b2[2];
    bool live[2];                                 // of the wave; dead ones still help loading and keep the barriers
    long bh[2], rowo[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const int raw = wg_z * 2 + r;
        live[r] = raw < B2 && qt_raw < QT;
        b2[r] = raw < B2 ? raw : B2 - 1;
        bh[r] = (long)b2[r] * H + h;
        rowo[r] = ((long)b2[r] * Nq + qc) * (H * 32) + h * 32 + 4 * half;
    }

    const bf16_t* src[NVL];                       // wave-uniform: start of the wave's 64 vectors in key tile 0 (see above)
#pragma unroll
    for (int i = 0; i < NVL; ++i) {
        const int v = wave * 64 + i * PAIR_THREADS, tile = v >> 7, wv = v & 127;
        const bf16_t* base;
        if (tile < 4) {
            int bb = wg_z * 2 + (tile & 1);
            bb = bb < B2 ? bb : B2 - 1;
            base = (tile < 2 ? k_t : v_t) + ((((long)bb * H + h) * KT) << 10);
        } else {
            int qq = wg_q * 4 + (tile - 4);
            qq = qq < QT ? qq : QT - 1;
            base = bias_t + ((((long)h * QT + qq) * (KT + ((flags >> 1) & 1))) << 10);
        }
        src[i] = base + (wv >> 6) * 512;
    }

    // from an asm statement for the reason given above
    const unsigned lds_base = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)att_smem;
    // A request fetches 1 KB, and sixteen lanes 256 bytes of it side by side (by 16-byte pieces 32 bytes apart, as above, every line is
    // asked for twice).  Of a lane's two pieces one lies in the first half of its sixteen places, the other in the second, the other
    // way round in every other group of eight lanes: the sixteen lanes of a read meet sixteen places in sixteen bank groups.
    const unsigned lane_off = ((lane >> 4) * 8 + (lane & 7)) * 32 + ((lane >> 3 ^ lane >> 4) & 1) * 16;
    const int piece0 = (lane >> 5) * 512 + ((lane >> 3 & 3) * 16 + (lane & 7) + 8 * (lane >> 3 & 1)) * 8, piece1 = piece0 ^ 64;
    auto operand = [&](const bf16_t* tile) __attribute__((always_inline)) {
        Ops16<bf16_t> o;
        o.v[0] = ld16(tile + piece0);
        o.v[1] = ld16(tile + piece1);
        return o;
    };
    auto fetch = [&](int kt, int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NVL; ++i) {
            const bf16_t* gp = src[i] + ((long)kt << 10);
            const unsigned dst = lds_base + (slot * NTILES * 128 + wave * 64 + i * PAIR_THREADS) * 16;
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
            asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(lane_off), "s"(gp), "s"(dst)
                         : "memory", "m0");
#pragma clang diagnostic pop
        }
    };
    // the first steps (all masked or not), then what the wave itself needs
    fetch(0, 0);
    fetch(KT > 1 ? 1 : 0, 1);
    fetch(KT > 2 ? 2 : KT - 1, 2);

    Ops16<bf16_t> qf[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) qf[r].load(q_t + ((bh[r] * QT + qt) << 10) + lane * 16);

    bf16_t gv[2][4][4];                           // this lane's gate values, fetched now
    if (gate) {
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            if (flags & FFK_ATT_GATE_TILED) {
                const bf16_t* gp = gate + ((bh[r] * QT + qt) << 10) + lane * 16;
                *reinterpret_cast<u32x4*>(&gv[r][0][0]) = *reinterpret_cast<const u32x4*>(gp);
                *reinterpret_cast<u32x4*>(&gv[r][2][0]) = *reinterpret_cast<const u32x4*>(gp + 8);
            } else {
#pragma unroll
                for (int g = 0; g < 4; ++g) *reinterpret_cast<u32x2*>(&gv[r][g][0]) = *reinterpret_cast<const u32x2*>(gate + rowo[r] + 8 * g);
            }
        }
    }

    // trailing key tiles that are completely masked in all batch rows contribute exactly zero
    int kt_end = KT;
    {
        auto masked = [&](int kt) {
            bool m = true;
#pragma unroll
            for (int r = 0; r < 2; ++r) m = m && tileflags[(long)b2[r] * KT + kt] == 2;
            return m;
        };
        while (kt_end > 1 && masked(kt_end - 1)) --kt_end;
    }
    const int* fl0 = tileflags + (long)b2[0] * KT;
    const int* fl1 = tileflags + (long)b2[1] * KT;
    int first_flag = KT;                          // from here on some key may be masked or padding
    for (int k0 = 0; k0 < KT; k0 += 64) {
        const int k = k0 + lane < KT ? k0 + lane : KT - 1;
        const unsigned long long f = __builtin_amdgcn_ballot_w64((fl0[k] | fl1[k]) != 0);
        if (f) {
            first_flag = k0 + __builtin_ctzll(f);
            break;
        }
    }

    bf16x8 ident[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) ident[i] = identity_frag<bf16_t>(i, l32, half);
    f32x16 o_acc[2];
    float l_run[2] = {0.0f, 0.0f}, ref[2] = {0.0f, 0.0f};
#pragma unroll
    for (int v = 0; v < 16; ++v) o_acc[0][v] = o_acc[1][v] = 0.0f;

    auto landed = [&](auto steps) __attribute__((always_inline)) {             // all but the newest `steps` requests of this thread
        static_assert(NVL == 4);
        if constexpr (decltype(steps)::value == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        else if constexpr (decltype(steps)::value == 1) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
        lds_barrier();
    };
    typedef std::integral_constant<int, 0> I0;
    typedef std::integral_constant<int, 1> I1;
    typedef std::integral_constant<int, 2> I2;
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int i = 0; i < 2; ++i) asm volatile("" : "+v"(*reinterpret_cast<u32x4*>(&qf[r].v[i])));

    auto bias_tile = [&](const bf16_t* buf) __attribute__((always_inline)) {
        f32x16 c;
#pragma unroll
        for (int v = 0; v < 16; ++v) c[v] = 0.0f;
        const Ops16<bf16_t> bc = operand(buf + (4 + wave) * 1024);
#pragma unroll
        for (int i = 0; i < 2; ++i) MM::mma(c, bc.frag(i), ident[i]);
        return c;
    };
    auto scores = [&](const bf16_t* buf, int r, const f32x16& c) __attribute__((always_inline)) {
        const Ops16<bf16_t> kc = operand(buf + r * 1024);
        f32x16 s = c;
#pragma unroll
        for (int i = 0; i < 2; ++i) MM::mma(s, kc.frag(i), qf[r].frag(i));
        return s;
    };
    auto add_keybias = [&](f32x16 (&s)[2], int kt) __attribute__((always_inline)) {          // some key of this tile is masked or padding
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const float* mp = keybias + ((long)b2[r] * KT + kt) * 32 + 4 * half;
            f32x4 mk[4];
#pragma unroll
            for (int g = 0; g < 4; ++g) mk[g] = *reinterpret_cast<const f32x4*>(mp + 8 * g);
#pragma unroll
            for (int g = 0; g < 4; ++g)
#pragma unroll
                for (int e = 0; e < 4; ++e) s[r][4 * g + e] += mk[g][e];
        }
    };
    auto exponentiate = [&](const f32x16& s, bf16x8 (&pf)[2]) __attribute__((always_inline)) {        // and the sum of the rounded values
        float p[16], t = 0.0f;
#pragma unroll
        for (int v = 0; v < 16; ++v) p[v] = fast_exp2(s[v]);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            pf[i] = PFrag<bf16_t>::make(p + i * 8);
            t = PFrag<bf16_t>::add_sum(pf[i], t);
        }
        return t;
    };

    {
        const int last = kt_end - 1;
        landed(I2{});
        f32x16 s[2], n[2];
        {
            const f32x16 c = bias_tile(lds);
#pragma unroll
            for (int r = 0; r < 2; ++r) s[r] = scores(lds, r, c);
            if (first_flag == 0) add_keybias(s, 0);
        }
        int slot = 0;
        auto step = [&](int kt, f32x16 (&s)[2], f32x16 (&n)[2]) __attribute__((always_inline)) {
            landed(I1{});                         // step kt + 1; and everyone is done with step kt - 1
            fetch(kt + 3 < kt_end ? kt + 3 : last, (slot + 3) & 3);
            const bf16_t* buf = lds + slot * NTILES * 1024;
            slot = (slot + 1) & 3;
            const bf16_t* ahead = lds + slot * NTILES * 1024;
            // everything is read at once; then a product to every four exponentials, in this order
            Ops16<bf16_t> kc[2], vc[2], bc;
            bc = operand(ahead + (4 + wave) * 1024);
#pragma unroll
            for (int r = 0; r < 2; ++r) kc[r] = operand(ahead + r * 1024);
#pragma unroll
            for (int r = 0; r < 2; ++r) vc[r] = operand(buf + (2 + r) * 1024);
            __builtin_amdgcn_sched_barrier(0);
            f32x16 c;
#pragma unroll
            for (int v = 0; v < 16; ++v) c[v] = 0.0f;
            float p[2][16], t[2] = {0.0f, 0.0f};
            bf16x8 pf[2][2];
            auto e4 = [&](int r, int g) __attribute__((always_inline)) {
#pragma unroll
                for (int e = 0; e < 4; ++e) p[r][4 * g + e] = fast_exp2(s[r][4 * g + e]);
                if (g & 1) pf[r][g >> 1] = PFrag<bf16_t>::make(p[r] + 8 * (g >> 1));
                __builtin_amdgcn_sched_barrier(0);
            };
            auto score = [&](int r, int i) __attribute__((always_inline)) {
                if (i == 0) n[r] = c;
                __builtin_amdgcn_s_setprio(1);
                MM::mma(n[r], kc[r].frag(i), qf[r].frag(i));
                __builtin_amdgcn_s_setprio(0);
                __builtin_amdgcn_sched_barrier(0);
            };
            auto value = [&](int r, int i) __attribute__((always_inline)) {
                __builtin_amdgcn_s_setprio(1);
                MM::mma(o_acc[r], vc[r].frag(i), pf[r][i]);
                __builtin_amdgcn_s_setprio(0);
                t[r] = PFrag<bf16_t>::add_sum(pf[r][i], t[r]);
                __builtin_amdgcn_sched_barrier(0);
            };
            auto bias = [&](int i) __attribute__((always_inline)) {
                MM::mma(c, bc.frag(i), ident[i]);
                __builtin_amdgcn_sched_barrier(0);
            };
            e4(0, 0);
            bias(0);
            e4(0, 1);
            bias(1);
            e4(0, 2);
            value(0, 0);
            e4(0, 3);
            score(0, 0);
            e4(1, 0);
            value(0, 1);
            e4(1, 1);
            score(0, 1);
            e4(1, 2);
            score(1, 0);
            value(1, 0);
            e4(1, 3);
            score(1, 1);
            value(1, 1);
            l_run[0] += t[0];
            l_run[1] += t[1];
            if (kt + 1 >= first_flag && kt < last) add_keybias(n, kt + 1);
        };
        int kt = 0;
#pragma unroll 1
        for (; kt < last; kt += 2) {
            step(kt, s, n);
            step(kt + 1, n, s);
        }
        if (kt == last) step(kt, s, n);
        landed(I0{});
    }

    float l_tot[2];
    {
        int* redo = reinterpret_cast<int*>(lds + NSLOT * NTILES * 1024);
        bool bad = false, again[2];               // some query of the wave, this lane's query: to be walked again
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            l_tot[r] = l_run[r] + lane_xor<32>(l_run[r]);
            unsigned big = 0;                     // largest magnitude of the lane's outputs; infinities and NaN above all numbers
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const unsigned m = __builtin_bit_cast(unsigned, o_acc[r][v]) & 0x7FFFFFFFu;
                big = big > m ? big : m;
            }
            const bool sound = l_tot[r] <= OPT_HIGH && l_tot[r] >= OPT_LOW && big < 0x7F800000u && (l_tot[r] >= 1.0f || big >= OUT_LOW);
            const bool out_of_range = live[r] && q < Nq && !sound;
            unsigned long long which = __builtin_amdgcn_ballot_w64(out_of_range);
            which |= which >> 32 | which << 32;   // both halves of a query
            again[r] = false;
            if (which != 0) {
                bool any = false;                 // a row without keys has a sum of zero, and zeros for its result
                for (int kt = 0; kt < KT; ++kt) any = any || (r ? fl1 : fl0)[kt] != 2;
                bad = bad || any;
                again[r] = any && (which >> lane & 1);
            }
        }
        if (tid == 0) *redo = 0;
        lds_barrier();
        if (bad && lane == 0) *redo = 1;
        lds_barrier();
        if (*redo != 0) {                         // workgroup-uniform
            // What the first walk has proven is kept, in the ring's other slots: a query's bits are its own
            f32x4* const kept = reinterpret_cast<f32x4*>(lds + NTILES * 1024) + tid;
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                l_run[r] = 0.0f;
                ref[r] = REF_FLOOR;
#pragma unroll
                for (int a = 0; a < 4; ++a)
                    kept[(4 * r + a) * PAIR_THREADS] = f32x4{o_acc[r][4 * a], o_acc[r][4 * a + 1], o_acc[r][4 * a + 2], o_acc[r][4 * a + 3]};
#pragma unroll
                for (int v = 0; v < 16; ++v) o_acc[r][v] = 0.0f;
            }
#pragma unroll 1
            for (int kt = 0; kt < kt_end; ++kt) {
                lds_barrier();
                fetch(kt, 0);
                landed(I0{});
                const f32x16 c = bias_tile(lds);
                f32x16 sc[2];
#pragma unroll
                for (int r = 0; r < 2; ++r) sc[r] = scores(lds, r, c);
                if (kt >= first_flag) add_keybias(sc, kt);
#pragma unroll
                for (int r = 0; r < 2; ++r) {
                    f32x16& s = sc[r];
                    float m = s[0];
#pragma unroll
                    for (int v = 1; v < 16; ++v) m = fmaxf(m, s[v]);
                    m = fmaxf(m, lane_xor<32>(m));
                    m = fmaxf(m, ref[r]);
                    const float alpha = fast_exp2(ref[r] - m);
                    ref[r] = m;
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        s[v] -= m;
                        o_acc[r][v] *= alpha;
                    }
                    bf16x8 pf[2];
                    l_run[r] = l_run[r] * alpha + exponentiate(s, pf);
                    const Ops16<bf16_t> vc = operand(lds + (2 + r) * 1024);
#pragma unroll
                    for (int i = 0; i < 2; ++i) MM::mma(o_acc[r], vc.frag(i), pf[i]);
                }
            }
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                const float l = l_run[r] + lane_xor<32>(l_run[r]);
                l_tot[r] = again[r] ? l : l_tot[r];
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    const f32x4 k = kept[(4 * r + a) * PAIR_THREADS];
#pragma unroll
                    for (int e = 0; e < 4; ++e) o_acc[r][4 * a + e] = again[r] ? o_acc[r][4 * a + e] : k[e];
                }
            }
        }
    }

#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const float inv = l_tot[r] > 0.0f ? 1.0f / l_tot[r] : 0.0f;
        if (!live[r] || q >= Nq) continue;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            bf16_t r4[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float x = o_acc[r][4 * g + e] * inv;
                if (gate) x *= (float)gv[r][g][e];
                r4[e] = (bf16_t)x;
            }
            *reinterpret_cast<u32x2*>(out + rowo[r] + 8 * g) = *reinterpret_cast<const u32x2*>(r4);
        }
    }
}

// Head dimensions 64 and 128 (the widths the reference's attention core also accepts; no module of the Evoformer
// uses them): the head is cut into DP = D / 32 parts of 32 channels, each part an operand tile of its own
// (part-major: part p of every tensor lies p * part elements behind part 0), so a score tile is the sum of DP
// products and the output DP accumulator tiles.  One wave per (batch row, head, 32 queries), operands straight
// from global memory, the classic running-maximum walk: this instantiation serves the stand-alone operator, not
// the inference block, and is not tuned beyond that.
template <typename T, int DP, bool HAS_BIAS>
__global__ __launch_bounds__(256) void attention_wide_kernel(
    T* __restrict__ out, const T* __restrict__ q_t, const T* __restrict__ k_t, const T* __restrict__ v_t,
    const T* __restrict__ bias_t, const float* __restrict__ keybias, const int* __restrict__ tileflags,
    int B2, int H, int Nq, int Nk, long part_q, long part_k) {
    typedef Mma<T> MM;
    typedef typename MM::Frag Frag;
    constexpr int NF = 16 / MM::KLANE;
    constexpr float REF_FLOOR = -1.0e4f;          // rows whose every score lies below are all-masked: they give zeros
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int l32 = lane & 31, half = lane >> 5;
    const int QT = (Nq + 31) >> 5, KT = (Nk + 31) >> 5;
    const long item = (long)blockIdx.x * 4 + wave;
    if (item >= (long)B2 * H * QT) return;
    const int qt = (int)(item % QT);
    const long bh = item / QT;
    const int h = (int)(bh % H), b2 = (int)(bh / H);

    Ops16<T> qf[DP];
#pragma unroll
    for (int p = 0; p < DP; ++p) qf[p].load(q_t + p * part_q + ((bh * QT + qt) << 10) + lane * 16);
    const float* mp = keybias + (long)b2 * KT * 32 + 4 * half;
    const int* fl = tileflags + (long)b2 * KT;
    Frag ident[NF];
    if (HAS_BIAS) {
#pragma unroll
        for (int i = 0; i < NF; ++i) ident[i] = identity_frag<T>(i, l32, half);
    }
    f32x16 o_acc[DP];
#pragma unroll
    for (int p = 0; p < DP; ++p)
#pragma unroll
        for (int v = 0; v < 16; ++v) o_acc[p][v] = 0.0f;
    float m_run = REF_FLOOR, l_run = 0.0f;
    for (int kt = 0; kt < KT; ++kt) {
        if (fl[kt] == 2) continue;                 // every key masked or padding: contributes exactly zero
        f32x16 s;
#pragma unroll
        for (int v = 0; v < 16; ++v) s[v] = 0.0f;
#pragma unroll
        for (int p = 0; p < DP; ++p) {
            Ops16<T> kc;
            kc.load(k_t + p * part_k + ((bh * KT + kt) << 10) + lane * 16);
#pragma unroll
            for (int i = 0; i < NF; ++i) MM::mma(s, kc.frag(i), qf[p].frag(i));
        }
        if (HAS_BIAS) {
            Ops16<T> bc;
            bc.load(bias_t + ((((long)h * QT + qt) * KT + kt) << 10) + lane * 16);
#pragma unroll
            for (int i = 0; i < NF; ++i) MM::mma(s, bc.frag(i), ident[i]);
        }
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const f32x4 mk = *reinterpret_cast<const f32x4*>(mp + kt * 32 + 8 * g);
#pragma unroll
            for (int e = 0; e < 4; ++e) s[4 * g + e] += mk[e];
        }
        float mt = fmaxf(s[0], s[1]);
#pragma unroll
        for (int v = 2; v < 16; ++v) mt = fmaxf(mt, s[v]);
        mt = fmaxf(mt, lane_xor<32>(mt));
        const float m_new = fmaxf(m_run, mt);
        const float alpha = fast_exp2(m_run - m_new);
        m_run = m_new;
        float pr[16];
#pragma unroll
        for (int v = 0; v < 16; ++v) pr[v] = fast_exp2(s[v] - m_new);
        Frag pf[NF];
        float tsum = 0.0f;
#pragma unroll
        for (int i = 0; i < NF; ++i) {
            pf[i] = PFrag<T>::make(pr + i * MM::KLANE);
            tsum = PFrag<T>::add_sum(pf[i], tsum);
        }
        l_run = l_run * alpha + tsum;
#pragma unroll
        for (int p = 0; p < DP; ++p) {
            Ops16<T> vc;
            vc.load(v_t + p * part_k + ((bh * KT + kt) << 10) + lane * 16);
#pragma unroll
            for (int v = 0; v < 16; ++v) o_acc[p][v] *= alpha;
#pragma unroll
            for (int i = 0; i < NF; ++i) MM::mma(o_acc[p], vc.frag(i), pf[i]);
        }
    }
    const float l_tot = l_run + lane_xor<32>(l_run);
    const float inv = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
    const int q = qt * 32 + l32;
    if (q < Nq) {
        T* o = out + ((long)b2 * Nq + q) * ((long)H * DP * 32) + (long)h * DP * 32 + 4 * half;
#pragma unroll
        for (int p = 0; p < DP; ++p)
#pragma unroll
            for (int g = 0; g < 4; ++g)
#pragma unroll
                for (int e = 0; e < 4; ++e) o[p * 32 + 8 * g + e] = DT<T>::from_f(o_acc[p][4 * g + e] * inv);
    }
}

template <typename T, int DP>
int launch_attention_wide(void* out, const void* q, const void* k, const void* v, const void* bias, const float* kb,
                          const int* flags, long B2, long H, long Nq, long Nk, hipStream_t st) {
    const long QT = (Nq + 31) / 32, KT = (Nk + 31) / 32;
    const long grid = (B2 * H * QT + 3) / 4;
    FFK_REQUIRE(grid < (1L << 31), FFK_ERR_SHAPE, "ffk_attention_fwd: too many tiles for one launch");
    const long part_q = B2 * H * QT * 1024, part_k = B2 * H * KT * 1024;
    if (bias)
        attention_wide_kernel<T, DP, true><<<(unsigned)grid, 256, 0, st>>>((T*)out, (const T*)q, (const T*)k, (const T*)v,
                                                                         (const T*)bias, kb, flags, (int)B2, (int)H,
                                                                         (int)Nq, (int)Nk, part_q, part_k);
    else
        attention_wide_kernel<T, DP, false><<<(unsigned)grid, 256, 0, st>>>((T*)out, (const T*)q, (const T*)k, (const T*)v,
                                                                          nullptr, kb, flags, (int)B2, (int)H, (int)Nq,
                                                                          (int)Nk, part_q, part_k);
    return ffk_check_launch("ffk_attention_fwd");
}

// One thread block per batch row: writes the additive key bias and, per 32-key tile, a flag
// (0: all keys valid, 1: some masked / padding, 2: every key masked or padding).
template <typename T>
__global__ void key_bias_kernel(float* kb, int* flags, const T* mask, long N, long Npad, long sb, long sn) {
    const long b = blockIdx.x;
    for (long t0 = 0; t0 < Npad; t0 += blockDim.x) {
        const long k = t0 + threadIdx.x;           // blockDim.x is a multiple of 64, Npad of 32
        float v = 0.0f;
        if (k < Npad) {
            if (k >= N) v = NEG_BIG;
            else if (mask && DT<T>::to_f(mask[b * sb + k * sn]) == 0.0f) v = -1e9f * 1.4426950408889634f;
            kb[b * Npad + k] = v;
        }
        const unsigned long long bad = __builtin_amdgcn_ballot_w64(k < Npad && v != 0.0f);
        const int half = (threadIdx.x & 63) >> 5;
        const unsigned part = half ? (unsigned)(bad >> 32) : (unsigned)bad;
        if ((threadIdx.x & 31) == 0 && k < Npad) flags[b * (Npad >> 5) + (k >> 5)] = part == 0 ? 0 : (part == 0xffffffffu ? 2 : 1);
    }
}

template <typename T, bool HAS_BIAS, int HD>
int launch_attention_b(void* out, const void* q, const void* k, const void* v, const void* bias, const float* kb,
                       const int* flags, const void* gate, float* lse, long B2, long H, long Nq, long Nk, int aflags,
                       hipStream_t st) {
    const size_t smem = (3 * (size_t)(HAS_BIAS ? 8 : 4) * 1024 + ATT_THREADS * 16) * sizeof(T) + 16;   // operand ring + gate + redo flag
    static FfkLdsReservation lds_reserved;
    {
        const int rc_lds = ffk_reserve_lds(lds_reserved, (const void*)attention_kernel<T, HAS_BIAS, HD>, smem, "ffk_attention_fwd");
        if (rc_lds != FFK_OK) return rc_lds;
    }
    const long items = (long)ffk_cdiv((Nq + 31) / 32, 4) * H * ffk_cdiv(B2, 2);
    FFK_REQUIRE(items < (1L << 31) - 8, FFK_ERR_SHAPE, "ffk_attention_fwd: %ld workgroups exceed the grid limit", items);
    dim3 grid((unsigned)(8 * ffk_cdiv(items, 8)));
    attention_kernel<T, HAS_BIAS, HD><<<grid, ATT_THREADS, smem, st>>>((T*)out, (const T*)q, (const T*)k, (const T*)v,
                                                                  (const T*)bias, kb, flags, (const T*)gate, lse, (int)B2,
                                                                  (int)H, (int)Nq, (int)Nk, aflags);
    return ffk_check_launch("ffk_attention_fwd");
}

int launch_attention_pair(void* out, const void* q, const void* k, const void* v, const void* bias, const float* kb, const int* flags,
                          const void* gate, long B2, long H, long Nq, long Nk, int aflags, hipStream_t st) {
    const size_t smem = 4 * (size_t)8 * 2048 + 16;             // operand ring + redo flag
    static FfkLdsReservation lds_reserved;
    const int rc_lds = ffk_reserve_lds(lds_reserved, (const void*)attention_pair_kernel, smem, "ffk_attention_fwd");
    if (rc_lds != FFK_OK) return rc_lds;
    const long items = (long)ffk_cdiv((Nq + 31) / 32, 4) * H * ffk_cdiv(B2, 2);
    FFK_REQUIRE(items < (1L << 31) - 8, FFK_ERR_SHAPE, "ffk_attention_fwd: %ld workgroups exceed the grid limit", items);
    attention_pair_kernel<<<dim3((unsigned)(8 * ffk_cdiv(items, 8))), PAIR_THREADS, smem, st>>>(
        (bf16_t*)out, (const bf16_t*)q, (const bf16_t*)k, (const bf16_t*)v, (const bf16_t*)bias, kb, flags, (const bf16_t*)gate, (int)B2,
        (int)H, (int)Nq, (int)Nk, aflags);
    return ffk_check_launch("ffk_attention_fwd");
}

template <typename T, int HD = 32>
int launch_attention(void* out, const void* q, const void* k, const void* v, const void* bias, const float* kb,
                     const int* flags, const void* gate, float* lse, long B2, long H, long Nq, long Nk, int aflags,
                     hipStream_t st) {
    return bias ? launch_attention_b<T, true, HD>(out, q, k, v, bias, kb, flags, gate, lse, B2, H, Nq, Nk, aflags, st)
                : launch_attention_b<T, false, HD>(out, q, k, v, nullptr, kb, flags, gate, lse, B2, H, Nq, Nk, aflags, st);
}

}  // namespace

extern "C" int ffk_attention_fwd(void* out, const void* q_t, const void* k_t, const void* v_t, const void* bias_t,
                                 const float* keybias, const int32_t* tileflags, const void* gate, int64_t B2, int64_t H, int64_t Nq,
                                 int64_t Nk, int64_t D, int flags, int dtype, void* stream) {
    return ffk_attention_fwd_lse(out, nullptr, q_t, k_t, v_t, bias_t, keybias, tileflags, gate, B2, H, Nq, Nk, D, flags, dtype, stream);
}

extern "C" int ffk_attention_fwd_lse(void* out, float* lse, const void* q_t, const void* k_t, const void* v_t, const void* bias_t,
                                     const float* keybias, const int32_t* tileflags, const void* gate, int64_t B2, int64_t H,
                                     int64_t Nq, int64_t Nk, int64_t D, int flags, int dtype, void* stream) {
    FFK_REQUIRE(out && q_t && k_t && v_t && keybias && tileflags, FFK_ERR_NULL, "ffk_attention_fwd: null pointer");
    FFK_REQUIRE(B2 > 0 && B2 < 131072 && H > 0 && H < 65536 && Nq > 0 && Nk > 0 && Nq < (1 << 24) && Nk < (1 << 24),
                FFK_ERR_SHAPE, "ffk_attention_fwd: bad shape B2=%ld H=%ld Nq=%ld Nk=%ld", (long)B2, (long)H, (long)Nq,
                (long)Nk);
    FFK_REQUIRE(ffk_aligned16(out) && ffk_aligned16(q_t) && ffk_aligned16(k_t) && ffk_aligned16(v_t) &&
                    ffk_aligned16(keybias) && (!bias_t || ffk_aligned16(bias_t)) && (!gate || ffk_aligned16(gate)),
                FFK_ERR_ALIGN, "ffk_attention_fwd: buffers must be 16-byte aligned");
    FFK_REQUIRE(D == 8 || D == 16 || D == 32 || D == 64 || D == 128, FFK_ERR_SHAPE,
                "ffk_attention_fwd: head dimension %ld (8 and 16 packed into 32-channel tiles, 32, 64 or 128)", (long)D);
    hipStream_t st = (hipStream_t)stream;
    if (D < 32) {
        FFK_REQUIRE(dtype == FFK_BF16 && H * D % 32 == 0 && !lse && (!gate || (flags & FFK_ATT_GATE_TILED)) && !(flags & FFK_ATT_HALF_K),
                    FFK_ERR_UNSUPPORTED, "ffk_attention_fwd: packed heads need bf16, whole tiles, a tiled gate or none, and no log-sum-exp");
        return D == 16 ? launch_attention<bf16_t, 16>(out, q_t, k_t, v_t, bias_t, keybias, tileflags, gate, lse, B2, H, Nq, Nk, flags, st)
                       : launch_attention<bf16_t, 8>(out, q_t, k_t, v_t, bias_t, keybias, tileflags, gate, lse, B2, H, Nq, Nk, flags, st);
    }
    if (D != 32) {
        FFK_REQUIRE(!gate && !lse && !(flags & (FFK_ATT_BIAS_PADDED | FFK_ATT_HALF_K)), FFK_ERR_UNSUPPORTED,
                    "ffk_attention_fwd: the gate, the log-sum-exp, padded bias rows and the narrow-head flag are built for head dimension 32 only");
        if (dtype == FFK_BF16)
            return D == 64 ? launch_attention_wide<bf16_t, 2>(out, q_t, k_t, v_t, bias_t, keybias, tileflags, B2, H, Nq, Nk, st)
                           : launch_attention_wide<bf16_t, 4>(out, q_t, k_t, v_t, bias_t, keybias, tileflags, B2, H, Nq, Nk, st);
        if (dtype == FFK_F32)
            return D == 64 ? launch_attention_wide<float, 2>(out, q_t, k_t, v_t, bias_t, keybias, tileflags, B2, H, Nq, Nk, st)
                           : launch_attention_wide<float, 4>(out, q_t, k_t, v_t, bias_t, keybias, tileflags, B2, H, Nq, Nk, st);
        return ffk_fail(FFK_ERR_DTYPE, "ffk_attention_fwd: unsupported dtype tag %d", dtype);
    }
    switch (dtype) {
        case FFK_BF16:
            // Two rows per wave (FFK_ATT_HALF_K or not: the padding adds nothing) for a bias and more than 256 keys, one row / two, us:
            // 256 x 4 heads of 256 queries 26.8 / 28.0, 320 x 4 of 320 53.0 / 49.0, 128 x 4 of 512 41 / 38, and see there.  Few rows (the
            // one-row kernel with its log-sum-exp), 1 / 8 / 32 / 64 x 4 of 288: 8.1 / 8.0, 8.6 / 8.6, 9.1 / 9.0, 12.7 / 12.6; of 512: 11.4 / 10.8,
            // 11.8 / 11.6, 13.0 / 12.8, 19.2 / 20.0; of 1 024: 19.2 / 17.6, 19.7 / 18.8, 31.2 / 31.3, 59 / 58; of 2 048: 34 / 32, 36 / 35, 110 / 105,
            // 217 / 204.  With the
            // log-sum-exp, from sums of probabilities that were not rounded against a zero reference, 256 x 4 of 256 27.0 / 29.3,
            // 391 x 4 of 391 102 / 102: one row.
            if (bias_t && !lse && Nk > 256) return launch_attention_pair(out, q_t, k_t, v_t, bias_t, keybias, tileflags, gate, B2, H, Nq, Nk, flags, st);
            return launch_attention<bf16_t>(out, q_t, k_t, v_t, bias_t, keybias, tileflags, gate, lse, B2, H, Nq, Nk, flags, st);
        case FFK_F32: return launch_attention<float>(out, q_t, k_t, v_t, bias_t, keybias, tileflags, gate, lse, B2, H, Nq, Nk, flags, st);
        default: return ffk_fail(FFK_ERR_DTYPE, "ffk_attention_fwd: unsupported dtype tag %d", dtype);
    }
}

extern "C" int ffk_key_bias(float* keybias, int32_t* tileflags, const void* mask, int64_t B, int64_t N,
                            int64_t mask_sb, int64_t mask_sn, int dtype, void* stream) {
    FFK_REQUIRE(keybias && tileflags, FFK_ERR_NULL, "ffk_key_bias: null pointer");
    FFK_REQUIRE(B > 0 && N > 0 && B < (1L << 31), FFK_ERR_SHAPE, "ffk_key_bias: bad shape B=%ld N=%ld", (long)B, (long)N);
    const long Npad = (N + 31) / 32 * 32;
    hipStream_t st = (hipStream_t)stream;
    dim3 grid((unsigned)B);
    switch (dtype) {
        case FFK_BF16: key_bias_kernel<bf16_t><<<grid, 256, 0, st>>>(keybias, tileflags, (const bf16_t*)mask, N, Npad, mask_sb, mask_sn); break;
        case FFK_F32: key_bias_kernel<float><<<grid, 256, 0, st>>>(keybias, tileflags, (const float*)mask, N, Npad, mask_sb, mask_sn); break;
        case FFK_F16: key_bias_kernel<f16_t><<<grid, 256, 0, st>>>(keybias, tileflags, (const f16_t*)mask, N, Npad, mask_sb, mask_sn); break;
        default: return ffk_fail(FFK_ERR_DTYPE, "ffk_key_bias: unsupported dtype tag %d", dtype);
    }
    return ffk_check_launch("ffk_key_bias");
}
