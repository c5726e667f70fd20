// Stage (a)+(b): query generation and sparse-signal evaluation on gfx950.
//
// For every query m of a coset {M_c l + d_p mod q : l in Z_q^b} the signal
// x(m) = sum_s a_s w^{<m, k_s>} (w = e^{2 pi i / q}) is evaluated the way the
// reference's SyntheticSubsampledSignal.subsample does
// (synt_exp/synt_src/synthetic_signal.py:97-118), with the phase exponent
// <m, k_s> computed exactly:
//
//   * one wave owns 16 queries; each lane builds 16 (or 32/48/64) query digits
//     of one query in registers (stage (a): exact integer work, never stored);
//   * per block of 16 supports, v_mfma_i32_16x16x64_i8 forms E = m . k^T over
//     the digit axis (int8 x int8 -> int32, exact: E <= n (q-1)^2);
//   * each lane reduces its 4 entries of E mod q, reads w^e from an LDS table
//     and accumulates a_s w^e in FP32 or FP64 (the VALU part that bounds the
//     kernel);
//   * the 16 lanes that share a query row are reduced with xor-shuffles.
//
// MFMA fragment layout (16x16x64 int8): lane L supplies row L%16 of A and
// column L%16 of B, each as 16 consecutive k-bytes of k-group L/16; the
// int32 result D[i][j] sits in lane j + 16*(i/4), register i%4. A and B use
// the same lane/k mapping, so any fixed digit order inside a 64-digit block
// gives the same dot product.
#include "qsft_common.h"

namespace qsft {

typedef int v4i __attribute__((ext_vector_type(4)));

template <typename T>
__device__ __forceinline__ void fill_wtable(cplx_t<T>* tab, int q) {
    for (int r = threadIdx.x; r < q; r += blockDim.x) {
        double s, c;
        sincospi(2.0 * (double)r / (double)q, &s, &c);
        tab[r].x = (T)c;
        tab[r].y = (T)s;
    }
}

// Pack 16 digits (values < 128) into a 16-byte MFMA fragment.
__device__ __forceinline__ v4i pack16(const int (&d)[16]) {
    v4i r;
#pragma unroll
    for (int w = 0; w < 4; ++w)
        r[w] = (d[4 * w] & 0xFF) | ((d[4 * w + 1] & 0xFF) << 8) | ((d[4 * w + 2] & 0xFF) << 16) |
               ((d[4 * w + 3] & 0xFF) << 24);
    return r;
}

__device__ __forceinline__ int byte_of(const v4i& v, int j) {
    return (v[j >> 2] >> (8 * (j & 3))) & 0xFF;
}

// Accumulate sum_s a_s w^{E mod q} for the wave's 16 queries over all S
// supports; afrag holds this lane's query digits. Returns this lane's 4
// partial sums (rows 4*(lane/16)+v, the column of this lane).
template <typename T, bool POW2, int NKB>
__device__ __forceinline__ void accumulate(const v4i (&afrag)[NKB], const int8_t* __restrict__ K,
                                           const cplx_t<T>* __restrict__ a, int S, int n_pad,
                                           const cplx_t<T>* tab, ModQ mq, uint32_t qmask,
                                           cplx_t<T> (&acc)[4]) {
    const int lane = threadIdx.x & 63;
    const int g = lane >> 4, r16 = lane & 15;
#pragma unroll
    for (int v = 0; v < 4; ++v) acc[v].x = acc[v].y = (T)0;
    for (int s0 = 0; s0 < S; s0 += 16) {
        const int s = s0 + r16;
        const bool ok = s < S;
        v4i e = {0, 0, 0, 0};
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb) {
            v4i bf = {0, 0, 0, 0};
            if (ok) bf = *reinterpret_cast<const v4i*>(K + (size_t)s * n_pad + 64 * kb + 16 * g);
            e = __builtin_amdgcn_mfma_i32_16x16x64_i8(afrag[kb], bf, e, 0, 0, 0);
        }
        cplx_t<T> as;
        as.x = as.y = (T)0;
        if (ok) as = a[s];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const uint32_t r = POW2 ? ((uint32_t)e[v] & qmask) : mq((uint32_t)e[v]);
            const cplx_t<T> w = tab[r];
            acc[v].x += as.x * w.x - as.y * w.y;
            acc[v].y += as.x * w.y + as.y * w.x;
        }
    }
    // reduce over the 16 lanes (columns) that share the same 4 rows
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            acc[v].x += __shfl_xor(acc[v].x, off);
            acc[v].y += __shfl_xor(acc[v].y, off);
        }
    }
}

template <typename T>
__device__ __forceinline__ cplx_t<T> pick4(const cplx_t<T> (&acc)[4], int v) {
    cplx_t<T> r = acc[0];
    if (v == 1) r = acc[1];
    if (v == 2) r = acc[2];
    if (v == 3) r = acc[3];
    return r;
}

template <typename T, bool POW2, int NKB>
__global__ __launch_bounds__(256) void k_eval_cosets(const qsft_eval_desc* __restrict__ descs,
                                                     const int32_t* __restrict__ pre, int n_inst) {
    using C2 = cplx_t<T>;
    __shared__ C2 tab[QSFT_MAX_Q];
    const int inst = find_inst(pre, n_inst, blockIdx.x);
    const qsft_eval_desc& d = descs[inst];
    const int q = d.q, b = d.b, n_pad = d.n_pad;
    const int Q = ipow(q, b);
    const int tiles = (Q + 63) >> 6;
    const int local = blockIdx.x - pre[inst];
    const int row = local / tiles;               // c * P + p
    const int tile = local - row * tiles;
    const int c = row / d.P;
    fill_wtable<T>(tab, q);
    __syncthreads();

    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int g = lane >> 4, r16 = lane & 15;
    const int lq0 = tile * 64 + wave * 16;
    const int l = lq0 + r16;                     // this lane's query (A row)
    const ModQ mq((uint32_t)q);
    const int8_t* __restrict__ Mt = d.Mt + (size_t)c * b * n_pad;
    const int8_t* __restrict__ drow = d.D + (size_t)row * n_pad;

    v4i afrag[NKB];
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb) {
        const int i0 = 64 * kb + 16 * g;         // first digit of this lane's slice
        const v4i dv = *reinterpret_cast<const v4i*>(drow + i0);
        int acc[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[j] = byte_of(dv, j);
        int rem = l, pw = Q;
        for (int t = 0; t < b; ++t) {            // digit l_t of l, MSB first
            pw /= q;
            const int lt = rem / pw;
            rem -= lt * pw;
            const v4i mv = *reinterpret_cast<const v4i*>(Mt + (size_t)t * n_pad + i0);
#pragma unroll
            for (int j = 0; j < 16; ++j) acc[j] += lt * byte_of(mv, j);
        }
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[j] = (int)mq((uint32_t)acc[j]);
        afrag[kb] = pack16(acc);
    }

    C2 sum[4];
    accumulate<T, POW2, NKB>(afrag, in_global(d.K), in_global(reinterpret_cast<const C2*>(d.a)), d.S, n_pad, tab, mq,
                             (uint32_t)(q - 1), sum);
    if (r16 < 4) {
        const int ql = lq0 + 4 * g + r16;
        if (ql < Q) in_global(reinterpret_cast<C2*>(d.x))[(size_t)row * Q + ql] = pick4<T>(sum, r16);
    }
}

// Terms of one 64-query block by the w-table, four waves of 16 queries.
template <typename T, bool POW2, int NKB>
__device__ __forceinline__ void points_by_table(const qsft_eval_points_desc& d, int64_t local, cplx_t<T>* tab) {
    using C2 = cplx_t<T>;
    const int q = d.q, n_pad = d.n_pad;
    fill_wtable<T>(tab, q);
    __syncthreads();
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int g = lane >> 4, r16 = lane & 15;
    const int64_t lq0 = local * 64 + wave * 16;
    const int64_t l = lq0 + r16;
    const ModQ mq((uint32_t)q);
    v4i afrag[NKB];
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb) {
        v4i z = {0, 0, 0, 0};
        if (l < d.N) z = *reinterpret_cast<const v4i*>(in_global(d.m) + (size_t)l * n_pad + 64 * kb + 16 * g);
        afrag[kb] = z;
    }
    C2 sum[4];
    accumulate<T, POW2, NKB>(afrag, in_global(d.K), in_global(reinterpret_cast<const C2*>(d.a)), d.S, n_pad, tab, mq,
                             (uint32_t)(q - 1), sum);
    if (r16 < 4) {
        const int64_t ql = lq0 + 4 * g + r16;
        if (ql < d.N) in_global(reinterpret_cast<C2*>(d.x))[ql] = pick4<T>(sum, r16);
    }
}

template <typename T, bool POW2, int NKB>
__global__ __launch_bounds__(256) void k_eval_points(const qsft_eval_points_desc* __restrict__ descs,
                                                     const int32_t* __restrict__ pre, int n_inst) {
    __shared__ cplx_t<T> tab[QSFT_MAX_Q];
    const int inst = find_inst(pre, n_inst, blockIdx.x);
    points_by_table<T, POW2, NKB>(descs[inst], blockIdx.x - pre[inst], tab);
}

// Transposes the 4 x 4 bytes of four neighbouring lanes: byte i of lane v
// becomes byte v of lane i.
__device__ __forceinline__ uint32_t quad_transpose(uint32_t x, int lane) {
    uint32_t y = (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0xB1, 0xF, 0xF, true);     // lane ^ 1
    x = __builtin_amdgcn_perm(x, y, lane & 1 ? 0x07030501u : 0x02060004u);
    y = (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x4E, 0xF, 0xF, true);              // lane ^ 2
    return __builtin_amdgcn_perm(x, y, lane & 2 ? 0x07060302u : 0x01000504u);
}

// q in {2, 3, 4}: cosine and sine of every phase are small integers (q = 3: of
// 2 cos and sin / (sqrt(3)/2)), so the sum over the support is a contraction of
// an int8 matrix with the coefficients, and runs on the matrix cores without a
// rounding: each component of a coefficient is an integer of a common unit, in
// 62-bit limbs of eight signed base-256 digits; [cos | sin] (16 queries x 64
// supports) times [re | im digits] (64 x 16) per limb accumulates exactly in
// int32 (S < 2^23), and the digit sums meet in a wide integer once per query.
//
// The unit is one that every component is a whole multiple of, so nothing is
// lost on the way in: one limb where the largest component is below 2^62 units,
// two up to 2^124 (FP64 components of random phases: 53 bits and a spread of
// about log2 S more), four, two after the other, up to 2^248, the table form
// beyond that and where a coefficient is not finite. For q = 2 the real and the imaginary parts never meet and have units
// of their own. The result is the exact sum rounded once for q = 2 and 4; for
// q = 3 the two sums are carried to about 2^-96 and sqrt(3)/2 to 2^-107, so
// that the last rounding is the only one that shows.
//
// The phases come from the MFMA with the support along its rows: a lane then
// holds 4 supports of one query per tile, and four tiles are the 16 bytes of
// the A fragment of the second product, in the order 4 t + v that the digit
// fragments are laid out in, so nothing crosses lanes. The four waves take the
// support's 64-blocks in turn for the same 64 queries (one read of the support
// per workgroup, every wave busy also for few queries) and add their integer
// sums in LDS, in any order.
//
// The table form is bound by its VALU and LDS reads (one 16 B entry and six
// FP64 operations per term); this one by the conversion and packing (about 1.5
// operations per term) and, as a launch of 100k queries is one and a half
// rounds of the four waves per SIMD, by its last round. Fetching the next
// block's support ahead costs the registers of a wave; digits of the queries
// stay in LDS for the same reason. Table and this form, FP64 strengths of 53
// bits (two limbs): S = 1000, n = 50, q = 4, 100003 queries 53 and 32 us (one
// limb, strengths of 24 bits: 23), 1000 queries 23 and 11; S = 4000, n = 100,
// 50000 queries 249 and 126 (70); q = 3, 100003 queries 58 and 43 (35); S = 10,
// 100000 queries 22 and 11.
constexpr int kPointTiles = 4;                    // query tiles of 16 per workgroup
constexpr int kSumPitch = 36;                     // rows 4 g + v of one column in 64 distinct banks

template <int NKB>
struct PointsLds {
    int32_t sum[2][64][kSumPitch];                // [cos | sin][query][re, im digits of a limb | of the next]
    int8_t dig[4][2][16][64];                     // [wave][limb][digit column][support of the block]
    int8_t query[64][64 * NKB + 16];              // digits of the queries
};

// The magnitude of sum_i g[i] 2^(32 i), |g[i]| < 2^62, as m 2^e with m in
// [2^63, 2^64) (or 0), the 32 bits below m, and whether any bit follows those.
template <int N>
struct WideInt {
    uint64_t m;
    uint32_t next;
    int e;
    bool neg, more;
    __device__ __forceinline__ explicit WideInt(int64_t (&g)[N]) {
        uint32_t w[N - 1];                        // the words below the top, carries passed up
#pragma unroll
        for (int i = 0; i < N - 1; ++i) {
            w[i] = (uint32_t)g[i];
            g[i + 1] += g[i] >> 32;
        }
        neg = g[N - 1] < 0;
        m = (uint64_t)g[N - 1];
        if (neg) {                                // two's complement
            uint64_t carry = 1;
#pragma unroll
            for (int i = 0; i < N - 1; ++i) {
                carry += (uint32_t)~w[i];
                w[i] = (uint32_t)carry;
                carry >>= 32;
            }
            m = ~m + carry;
        }
        e = 32 * (N - 1);
        next = 0;
        more = false;
        bool full = false;                        // m has 33 bits or more and `next` is taken
#pragma unroll
        for (int i = N - 2; i >= 0; --i) {
            if (full) {
                more |= w[i] != 0;
            } else if (m >> 32) {
                next = w[i];
                full = true;
            } else {
                m = m << 32 | w[i];
                e -= 32;
            }
        }
        const int lz = m ? (int)__builtin_clzll(m) : 0;            // (above 31 only without a next word)
        m = m << lz | ((uint64_t)next << (lz & 31)) >> 32;
        next = lz < 32 ? next << lz : 0;
        e -= lz;
    }
    // rounded to nearest, in units of 2^e
    template <typename T>
    __device__ __forceinline__ T rounded() const {
        const T v = (T)(m | (next != 0 || more ? 1u : 0u));
        return neg ? -v : v;
    }
    // hi + lo to about 2^-96 of it, times 2^e
    __device__ __forceinline__ double2 pair() const {
        double hi = (double)(m & ~0x7FFull), lo = (double)(m & 0x7FFull) + (double)next * 0x1p-32;
        if (neg) {
            hi = -hi;
            lo = -lo;
        }
        return make_double2(ldexp(hi, e), ldexp(lo, e));
    }
};

// Limb `first` (and the next, where H = 2) of v, a whole number of units 2^unit
// below 2^(62 LIMBS) of them: v is the sum of limb h times 2^(62 h), each rounded
// to nearest from the top (|limb| <= 2^61 below the highest; a remainder has no
// more bits than v, so every step is exact). Byte i of a word is the limb's
// signed base-256 digit i: (x + b) ^ b with b = 0x80 in every byte turns the
// bytes of a two's complement number into them.
template <int LIMBS, int H>
__device__ __forceinline__ void signed_digits(double v, int unit, int first, uint64_t (&w)[H]) {
    constexpr uint64_t bias = 0x8080808080808080ull;
    double r = ldexp(v, -unit), limb[H];
#pragma unroll
    for (int h = LIMBS - 1; h >= 0; --h) {
        double t = r;
        if (h > 0) {
            t = rint(ldexp(r, -62 * h));
            r = fma(-t, __builtin_bit_cast(double, (uint64_t)(1023 + 62 * h) << 52), r);
        }
        if (LIMBS == H || (h & ~(H - 1)) == first) limb[h & (H - 1)] = t;
    }
#pragma unroll
    for (int h = 0; h < H; ++h) w[h] = ((uint64_t)__double2ll_rn(limb[h]) + bias) ^ bias;
}

template <typename T, int NKB, int LIMBS>
__device__ __forceinline__ void points_exact(const qsft_eval_points_desc& d, int64_t local, PointsLds<NKB>& sh,
                                             const int (&unit)[2]) {
    using C2 = cplx_t<T>;
    constexpr int kHeld = LIMBS < 2 ? LIMBS : 2;  // limbs at once
    // query tiles at once: with two limbs and two digit blocks the accumulators of all four do not fit the
    // registers of four waves per SIMD
    constexpr int kTiles = kHeld == 2 && NKB > 1 ? 2 : kPointTiles;
    const int q = d.q, S = d.S, n_pad = d.n_pad;
    const C2* __restrict__ a = in_global(reinterpret_cast<const C2*>(d.a));
    const int8_t* __restrict__ K = in_global(d.K);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int g = lane >> 4, r16 = lane & 15;
    const uint32_t cosine = q == 4 ? 0x00FF0001u : q == 2 ? 0x0000FF01u : 0x00FFFF02u;
    const uint32_t sine = q == 4 ? 0xFF000100u : q == 2 ? 0u : 0x00FF0100u;
    const uint32_t mask = q == 4 ? 0x03030303u : q == 2 ? 0x01010101u : 0xFFFFFFFFu;

    const int qi = threadIdx.x >> 1, part = threadIdx.x & 1;      // query, re or im
    const int64_t ql = local * 64 + qi;
    int64_t c[2 * LIMBS], z[2 * LIMBS];           // four digits each, of the two sums
#pragma unroll 1
    for (int first = 0; first < LIMBS; first += kHeld) {
#pragma unroll 1
        for (int t0 = 0; t0 < kPointTiles; t0 += kTiles) {
            v4i csum[kHeld][kTiles], ssum[kHeld][kTiles];
#pragma unroll
            for (int h = 0; h < kHeld; ++h) {
#pragma unroll
                for (int t = 0; t < kTiles; ++t) {
                    csum[h][t] = v4i{0, 0, 0, 0};
                    ssum[h][t] = v4i{0, 0, 0, 0};
                }
            }
            for (int s0 = 64 * wave; s0 < S; s0 += 256) {
                v4i kfrag[4][NKB];
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const int s = s0 + 16 * t + r16;
#pragma unroll
                    for (int kb = 0; kb < NKB; ++kb) {
                        v4i z = {0, 0, 0, 0};
                        if (s < S) z = *reinterpret_cast<const v4i*>(K + (size_t)s * n_pad + 64 * kb + 16 * g);
                        kfrag[t][kb] = z;
                    }
                }
                C2 as;
                as.x = as.y = (T)0;
                if (s0 + lane < S) as = a[s0 + lane];
                // digits of this lane's support, at its place in the fragments' order:
                // support 16 t + 4 g + v is byte 16 g + 4 t + v, so four neighbouring
                // lanes hold the four bytes of a word of each digit's row
                uint64_t word[2][kHeld];
                signed_digits<LIMBS>((double)as.x, unit[0], first, word[0]);
                signed_digits<LIMBS>((double)as.y, unit[1], first, word[1]);
                const int pos = 16 * ((lane >> 2) & 3) + 4 * (lane >> 4);
#pragma unroll
                for (int h = 0; h < kHeld; ++h) {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        *reinterpret_cast<uint32_t*>(&sh.dig[wave][h][4 * j + (lane & 3)][pos]) =
                            quad_transpose((uint32_t)(word[j >> 1][h] >> (32 * (j & 1))), lane);
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
                v4i bfrag[kHeld];
#pragma unroll
                for (int h = 0; h < kHeld; ++h) bfrag[h] = *reinterpret_cast<const v4i*>(&sh.dig[wave][h][r16][16 * g]);
#pragma unroll
                for (int t = 0; t < kTiles; ++t) {
                    v4i qfrag[NKB], cf, sf;
#pragma unroll
                    for (int kb = 0; kb < NKB; ++kb)
                        qfrag[kb] = *reinterpret_cast<const v4i*>(&sh.query[16 * (t0 + t) + r16][64 * kb + 16 * g]);
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        v4i p = {0, 0, 0, 0};
#pragma unroll
                        for (int kb = 0; kb < NKB; ++kb)
                            p = __builtin_amdgcn_mfma_i32_16x16x64_i8(kfrag[u][kb], qfrag[kb], p, 0, 0, 0);
                        if (q == 3) {
                            // p - 3 floor((p + 1/2) / 3) in FP32: p < 2^22, so the quotient is off by less than 0.09
                            // of the 1/6 that it may be
#pragma unroll
                            for (int w = 0; w < 4; ++w)
                                p[w] -= 3 * (int)fmaf((float)p[w], 1.0f / 3.0f, 1.0f / 6.0f);
                        }
                        const uint32_t lo = __builtin_amdgcn_perm((uint32_t)p[1], (uint32_t)p[0], 0x0C0C0400u);
                        const uint32_t up = __builtin_amdgcn_perm((uint32_t)p[3], (uint32_t)p[2], 0x04000C0Cu);
                        const uint32_t r = (lo | up) & mask;
                        cf[u] = (int)__builtin_amdgcn_perm(0u, cosine, r);
                        sf[u] = (int)__builtin_amdgcn_perm(0u, sine, r);
                    }
#pragma unroll
                    for (int h = 0; h < kHeld; ++h) {
                        csum[h][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(cf, bfrag[h], csum[h][t], 0, 0, 0);
                        ssum[h][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(sf, bfrag[h], ssum[h][t], 0, 0, 0);
                    }
                }
                __builtin_amdgcn_wave_barrier();      // the fragments are read before the next block's digits
            }
#pragma unroll
            for (int h = 0; h < kHeld; ++h) {
#pragma unroll
                for (int t = 0; t < kTiles; ++t) {
#pragma unroll
                    for (int w = 0; w < 4; ++w) {
                        atomicAdd(&sh.sum[0][16 * (t0 + t) + 4 * g + w][16 * h + r16], csum[h][t][w]);
                        atomicAdd(&sh.sum[1][16 * (t0 + t) + 4 * g + w][16 * h + r16], ssum[h][t][w]);
                    }
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 2 * kHeld; ++i) {
            const int at = 16 * (i >> 1) + 4 * (i & 1);
            int64_t cv = 0, zv = 0;
            if (qi < 64) {
#pragma unroll
                for (int j = 3; j >= 0; --j) {
                    cv = cv * 256 + sh.sum[0][qi][at + 8 * part + j];
                    zv = zv * 256 + sh.sum[1][qi][at + 8 * (1 - part) + j];
                }
            }
            // limb h counts 2^(62 h) units = 2^(64 h) 4^(LIMBS - 1 - h) quarters of them, LIMBS - 1 times over
            const int up = 2 * (LIMBS - 1 - first - (i >> 1));
            c[2 * first + i] = cv << up;
            z[2 * first + i] = (part ? zv : -zv) << up;            // re: cos re - sin im; im: cos im + sin re
        }
        if (first + kHeld < LIMBS) {
            __syncthreads();                      // the sums are read
            for (int i = threadIdx.x; i < 2 * 64 * kSumPitch; i += 256) (&sh.sum[0][0][0])[i] = 0;
            __syncthreads();
        }
    }
    if (qi >= 64 || ql >= d.N) return;
    T x;
    if (q == 3) {                                 // c / 2 + sqrt(3)/2 z
#pragma clang fp contract(off)
        const double h0 = 0.8660254037844386, h1 = 5.0175421109034514e-17;
        const double2 cs = WideInt<2 * LIMBS>(c).pair(), zs = WideInt<2 * LIMBS>(z).pair();
        const double p = h0 * zs.x, a0 = 0.5 * cs.x, s = a0 + p;
        const double bb = s - a0, err = (a0 - (s - bb)) + (p - bb);                   // s + err = a0 + p
        const double rest = fma(h0, zs.x, -p) + fma(h0, zs.y, fma(h1, zs.x, 0.5 * cs.y));
        x = (T)ldexp(s + (err + rest), unit[part] - 2 * (LIMBS - 1));
    } else {
#pragma unroll
        for (int i = 0; i < 2 * LIMBS; ++i) c[i] += z[i];
        const WideInt<2 * LIMBS> w(c);
        x = ldexp(w.template rounded<T>(), w.e + unit[part] - 2 * (LIMBS - 1));
    }
    in_global(reinterpret_cast<T*>(d.x))[2 * ql + part] = x;
}

// Bits of one component: the exponent that it stays below, and that of its
// lowest set bit.
__device__ __forceinline__ void component_range(double v, int& top, int& low) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v) & ~(1ull << 63);
    if (b == 0) return;
    const int f = (int)(b >> 52);
    const uint64_t mant = (b & ((1ull << 52) - 1)) | (f ? 1ull << 52 : 0ull);
    top = max(top, max(f, 1) - 1022);
    low = min(low, max(f, 1) - 1075 + (int)__builtin_ctzll(mant));
}

template <typename T, int NKB>
__global__ __launch_bounds__(256, NKB <= 2 ? 4 : 1) void k_eval_points_int(const qsft_eval_points_desc* __restrict__ descs,
                                                         const int32_t* __restrict__ pre, int n_inst) {
    using C2 = cplx_t<T>;
    constexpr int kNotFinite = 0x7FF - 1022;
    __shared__ union {
        PointsLds<NKB> s;
        C2 tab[QSFT_MAX_Q];
    } sh;
    __shared__ int range[2][2];                   // [re | im][top, low]
    const int inst = find_inst(pre, n_inst, blockIdx.x);
    const qsft_eval_points_desc& d = descs[inst];
    const int64_t local = blockIdx.x - pre[inst];
    const int q = d.q, S = d.S, n_pad = d.n_pad;
    const C2* __restrict__ a = in_global(reinterpret_cast<const C2*>(d.a));
    const int lane = threadIdx.x & 63;
    constexpr int kNone = 4096;                   // beyond every exponent
    if (threadIdx.x < 2) {
        range[threadIdx.x][0] = -kNone;
        range[threadIdx.x][1] = kNone;
    }
#pragma unroll
    for (int k = 0; k < NKB; ++k) {
        const int i = threadIdx.x + 256 * k, row = i / (4 * NKB), col = 16 * (i - row * (4 * NKB));
        v4i z = {0, 0, 0, 0};
        if (local * 64 + row < d.N) z = *reinterpret_cast<const v4i*>(in_global(d.m) + (size_t)(local * 64 + row) * n_pad + col);
        *reinterpret_cast<v4i*>(&sh.s.query[row][col]) = z;
    }
    for (int i = threadIdx.x; i < 2 * 64 * kSumPitch; i += 256) (&sh.s.sum[0][0][0])[i] = 0;
    int top[2] = {-kNone, -kNone}, low[2] = {kNone, kNone};
    for (int s = threadIdx.x; s < S; s += 256) {
        const C2 v = a[s];
        component_range((double)v.x, top[0], low[0]);
        component_range((double)v.y, top[1], low[1]);
    }
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            top[p] = max(top[p], __shfl_xor(top[p], off));
            low[p] = min(low[p], __shfl_xor(low[p], off));
        }
    }
    __syncthreads();
    if (lane == 0) {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            atomicMax(&range[p][0], top[p]);
            atomicMin(&range[p][1], low[p]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int p = 0; p < 2; ++p) {                 // (the same words in all threads)
        top[p] = __builtin_amdgcn_readfirstlane(range[p][0]);
        low[p] = __builtin_amdgcn_readfirstlane(range[p][1]);
    }
    if (q != 2) {
        top[0] = top[1] = max(top[0], top[1]);
        low[0] = low[1] = min(low[0], low[1]);
    }
    const int bits = max(top[0] - low[0], top[1] - low[1]);       // (negative where all are zero)
    if (bits <= 62 && top[0] < kNotFinite && top[1] < kNotFinite) {
        const int unit[2] = {low[0] < kNone ? top[0] - 62 : 0, low[1] < kNone ? top[1] - 62 : 0};
        points_exact<T, NKB, 1>(d, local, sh.s, unit);
    } else if (bits <= 124 && top[0] < kNotFinite && top[1] < kNotFinite) {
        const int unit[2] = {low[0] < kNone ? top[0] - 124 : 0, low[1] < kNone ? top[1] - 124 : 0};
        points_exact<T, NKB, 2>(d, local, sh.s, unit);
    } else if (bits <= 248 && top[0] < kNotFinite && top[1] < kNotFinite) {
        const int unit[2] = {low[0] < kNone ? top[0] - 248 : 0, low[1] < kNone ? top[1] - 248 : 0};
        points_exact<T, NKB, 4>(d, local, sh.s, unit);
    } else {
        __syncthreads();
        points_by_table<T, false, NKB>(d, local, sh.tab);
    }
}


// Stage (a) alone: write the digits of every query (M_c l + d_p) mod q as
// int8 [C][P][Q][n_pad] (for user callbacks that need the indices).
__global__ __launch_bounds__(256) void k_query_digits(const qsft_eval_desc* __restrict__ descs,
                                                      const int32_t* __restrict__ pre, int n_inst) {
    const int inst = find_inst(pre, n_inst, blockIdx.x);
    const qsft_eval_desc& d = descs[inst];
    const int q = d.q, b = d.b, n = d.n, n_pad = d.n_pad;
    const int Q = ipow(q, b);
    const int tiles = (Q + 255) >> 8;
    const int local = blockIdx.x - pre[inst];
    const int row = local / tiles;
    const int l = (local - row * tiles) * 256 + threadIdx.x;
    if (l >= Q) return;
    const int c = row / d.P;
    const ModQ mq((uint32_t)q);
    const int8_t* __restrict__ Mt = d.Mt + (size_t)c * b * n_pad;
    const int8_t* __restrict__ drow = d.D + (size_t)row * n_pad;
    int8_t* __restrict__ out = reinterpret_cast<int8_t*>(d.x) + ((size_t)row * Q + l) * n_pad;
    for (int i = 0; i < n_pad; ++i) {
        uint32_t acc = 0;
        if (i < n) {
            acc = (uint32_t)drow[i];
            int rem = l, pw = Q;
            for (int t = 0; t < b; ++t) {
                pw /= q;
                const int lt = rem / pw;
                rem -= lt * pw;
                acc += (uint32_t)(lt * Mt[(size_t)t * n_pad + i]);
            }
            acc = mq(acc);
        }
        out[i] = (int8_t)acc;
    }
}

}  // namespace qsft

using namespace qsft;

namespace {

template <template <typename, bool, int> class Dummy>
struct unused {};

template <typename T, bool POW2>
hipError_t launch_cosets(int nkb, const qsft_eval_desc* d, const int32_t* pre, int n_inst, int blocks,
                         hipStream_t st) {
    switch (nkb) {
        case 1: hipLaunchKernelGGL((k_eval_cosets<T, POW2, 1>), dim3(blocks), dim3(256), 0, st, d, pre, n_inst); break;
        case 2: hipLaunchKernelGGL((k_eval_cosets<T, POW2, 2>), dim3(blocks), dim3(256), 0, st, d, pre, n_inst); break;
        case 3: hipLaunchKernelGGL((k_eval_cosets<T, POW2, 3>), dim3(blocks), dim3(256), 0, st, d, pre, n_inst); break;
        default: hipLaunchKernelGGL((k_eval_cosets<T, POW2, 4>), dim3(blocks), dim3(256), 0, st, d, pre, n_inst); break;
    }
    return hipGetLastError();
}

template <typename T, bool POW2>
hipError_t launch_points(int nkb, const qsft_eval_points_desc* d, const int32_t* pre, int n_inst,
                         int blocks, hipStream_t st) {
    switch (nkb) {
        case 1: hipLaunchKernelGGL((k_eval_points<T, POW2, 1>), dim3(blocks), dim3(256), 0, st, d, pre, n_inst); break;
        case 2: hipLaunchKernelGGL((k_eval_points<T, POW2, 2>), dim3(blocks), dim3(256), 0, st, d, pre, n_inst); break;
        case 3: hipLaunchKernelGGL((k_eval_points<T, POW2, 3>), dim3(blocks), dim3(256), 0, st, d, pre, n_inst); break;
        default: hipLaunchKernelGGL((k_eval_points<T, POW2, 4>), dim3(blocks), dim3(256), 0, st, d, pre, n_inst); break;
    }
    return hipGetLastError();
}

template <typename T>
hipError_t launch_points_int(int nkb, const qsft_eval_points_desc* d, const int32_t* pre, int n_inst, int blocks,
                             hipStream_t st) {
    switch (nkb) {
        case 1: hipLaunchKernelGGL((k_eval_points_int<T, 1>), dim3(blocks), dim3(256), 0, st, d, pre, n_inst); break;
        case 2: hipLaunchKernelGGL((k_eval_points_int<T, 2>), dim3(blocks), dim3(256), 0, st, d, pre, n_inst); break;
        case 3: hipLaunchKernelGGL((k_eval_points_int<T, 3>), dim3(blocks), dim3(256), 0, st, d, pre, n_inst); break;
        default: hipLaunchKernelGGL((k_eval_points_int<T, 4>), dim3(blocks), dim3(256), 0, st, d, pre, n_inst); break;
    }
    return hipGetLastError();
}

}  // namespace

// implemented in abi.cpp
extern "C" void qsft_set_error(const char* msg);
extern "C" int qsft_hip_status(hipError_t e, const char* where);

// A launch covers instances that share q's power-of-two class and the digit
// block count; the binding groups instances accordingly (one launch per key).
extern "C" int qsft_eval_blocks(const qsft_eval_desc* h) {
    if (!h || h->q < 2 || h->q > QSFT_MAX_Q || h->b < 1 || h->b > QSFT_MAX_B || h->n < 1 ||
        h->n > h->n_pad || h->n_pad % 64 || h->n_pad > QSFT_MAX_N || h->C < 1 || h->P < 1 || h->S < 0)
        return -1;
    const long long Q = (long long)ipow(h->q, h->b);
    const long long blocks = (long long)h->C * h->P * ((Q + 63) / 64);
    return blocks > 0x7FFFFFFF ? -1 : (int)blocks;
}

extern "C" int qsft_eval_points_blocks(const qsft_eval_points_desc* h) {
    if (!h || h->q < 2 || h->q > QSFT_MAX_Q || h->n < 1 || h->n > h->n_pad || h->n_pad % 64 ||
        h->n_pad > QSFT_MAX_N || h->N < 0 || h->S < 0)
        return -1;
    const long long blocks = (h->N + 63) / 64;
    return blocks > 0x7FFFFFFF ? -1 : (int)blocks;
}

// Integer sums for q whose cosines and sines are one constant times small
// integers, up to the S that int32 digit sums hold (2^23 digits of at most 2^7).
// They win at every size measured, from S = 10 or 1000 queries up (above). What
// the coefficients allow is found by the kernel.
extern "C" int qsft_eval_points_int(const qsft_eval_points_desc* h) {
    return h && h->q >= 2 && h->q <= 4 && h->S < (1 << 23);
}

// `precision` selects the accumulation type; bit 8 marks power-of-two q for
// every instance in the launch; bits 4..7 give the 64-digit block count (1..4);
// bit 9, for explicit points, that qsft_eval_points_int holds for every one.
extern "C" int qsft_eval_cosets(const qsft_eval_desc* d, const int32_t* pre, int n_inst, int blocks,
                                int precision, void* stream) {
    if (!d || !pre || n_inst < 1 || blocks < 0) { qsft_set_error("qsft_eval_cosets: bad arguments"); return QSFT_ERR_ARG; }
    if (blocks == 0) return QSFT_OK;
    const int prec = precision & 0xF;
    const int nkb = (precision >> 4) & 0xF;
    const bool pow2 = (precision >> 8) & 1;
    if (nkb < 1 || nkb > 4 || (prec != QSFT_F32 && prec != QSFT_F64)) {
        qsft_set_error("qsft_eval_cosets: bad precision word");
        return QSFT_ERR_ARG;
    }
    hipStream_t st = (hipStream_t)stream;
    hipError_t e;
    if (prec == QSFT_F32) e = pow2 ? launch_cosets<float, true>(nkb, d, pre, n_inst, blocks, st)
                                   : launch_cosets<float, false>(nkb, d, pre, n_inst, blocks, st);
    else e = pow2 ? launch_cosets<double, true>(nkb, d, pre, n_inst, blocks, st)
                  : launch_cosets<double, false>(nkb, d, pre, n_inst, blocks, st);
    return qsft_hip_status(e, "qsft_eval_cosets");
}

extern "C" int qsft_eval_points(const qsft_eval_points_desc* d, const int32_t* pre, int n_inst, int blocks,
                                int precision, void* stream) {
    if (!d || !pre || n_inst < 1 || blocks < 0) { qsft_set_error("qsft_eval_points: bad arguments"); return QSFT_ERR_ARG; }
    if (blocks == 0) return QSFT_OK;
    const int prec = precision & 0xF;
    const int nkb = (precision >> 4) & 0xF;
    const bool pow2 = (precision >> 8) & 1;
    if (nkb < 1 || nkb > 4 || (prec != QSFT_F32 && prec != QSFT_F64)) {
        qsft_set_error("qsft_eval_points: bad precision word");
        return QSFT_ERR_ARG;
    }
    hipStream_t st = (hipStream_t)stream;
    hipError_t e;
    if ((precision >> 9) & 1)
        e = prec == QSFT_F32 ? launch_points_int<float>(nkb, d, pre, n_inst, blocks, st)
                             : launch_points_int<double>(nkb, d, pre, n_inst, blocks, st);
    else if (prec == QSFT_F32) e = pow2 ? launch_points<float, true>(nkb, d, pre, n_inst, blocks, st)
                                   : launch_points<float, false>(nkb, d, pre, n_inst, blocks, st);
    else e = pow2 ? launch_points<double, true>(nkb, d, pre, n_inst, blocks, st)
                  : launch_points<double, false>(nkb, d, pre, n_inst, blocks, st);
    return qsft_hip_status(e, "qsft_eval_points");
}

extern "C" int qsft_query_digits_blocks(const qsft_eval_desc* h) {
    if (qsft_eval_blocks(h) < 0) return -1;
    const long long Q = (long long)ipow(h->q, h->b);
    const long long blocks = (long long)h->C * h->P * ((Q + 255) / 256);
    return blocks > 0x7FFFFFFF ? -1 : (int)blocks;
}

extern "C" int qsft_query_digits(const qsft_eval_desc* d, const int32_t* pre, int n_inst, int blocks, void* stream) {
    if (!d || !pre || n_inst < 1 || blocks < 0) { qsft_set_error("qsft_query_digits: bad arguments"); return QSFT_ERR_ARG; }
    if (blocks == 0) return QSFT_OK;
    hipLaunchKernelGGL(k_query_digits, dim3(blocks), dim3(256), 0, (hipStream_t)stream, d, pre, n_inst);
    return qsft_hip_status(hipGetLastError(), "qsft_query_digits");
}
