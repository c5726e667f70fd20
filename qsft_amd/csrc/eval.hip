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
// rounding: each coefficient, as a fixed-point number of 63 bits below the
// largest one, is eight signed base-256 digits; [cos | sin] (16 queries x 64
// supports) times [re | im digits] (64 x 16) accumulates exactly in int32 (S <
// 2^23), and the digit sums meet in int64 once per query. The error is the
// final rounding and 2^-64 of the largest coefficient per term, less than a
// sum in FP64 makes. A coefficient that is not finite sends the workgroup to
// the table form, which carries it through as before.
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
// rounds of the four waves per SIMD, by its last round. S = 1000, n = 50, q = 4,
// FP64: 100003 queries 53 -> 20 us, 1000 queries 23 -> 7.5 us; S = 4000, n =
// 100, 50000 queries 250 -> 65 us; q = 3, 100003 queries 58 -> 30 us; S = 10,
// 100000 queries 22 -> 8 us. Fetching the next block's support ahead costs the
// registers of a wave (20 us); eight waves per workgroup 24 us. Digits of the
// queries stay in LDS for the same reason (n = 100: 110 us in registers).
template <typename T, int NKB>
__global__ __launch_bounds__(256, NKB <= 2 ? 4 : 1) void k_eval_points_int(const qsft_eval_points_desc* __restrict__ descs,
                                                         const int32_t* __restrict__ pre, int n_inst) {
    using C2 = cplx_t<T>;
    constexpr int kTiles = 4;                     // query tiles of 16
    constexpr int kSumPitch = 20;                 // rows 4 g + v of one column in 64 distinct banks
    __shared__ union {
        struct {
            int32_t sum[2][64][kSumPitch];        // [cos | sin][query][re, im digits]
            int8_t dig[4][16][64];                // [wave][digit column][support of the block]
            int8_t query[64][64 * NKB + 16];      // digits of the queries
        } s;
        C2 tab[QSFT_MAX_Q];
    } sh;
    __shared__ uint32_t top;
    const int inst = find_inst(pre, n_inst, blockIdx.x);
    const qsft_eval_points_desc& d = descs[inst];
    const int64_t local = blockIdx.x - pre[inst];
    const int q = d.q, S = d.S, n_pad = d.n_pad;
    const C2* __restrict__ a = in_global(reinterpret_cast<const C2*>(d.a));
    const int8_t* __restrict__ K = in_global(d.K);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int g = lane >> 4, r16 = lane & 15;

    // exponent of the largest |re|, |im|
    if (threadIdx.x == 0) top = 0;
#pragma unroll
    for (int k = 0; k < NKB; ++k) {
        const int i = threadIdx.x + 256 * k, row = i / (4 * NKB), col = 16 * (i - row * (4 * NKB));
        v4i z = {0, 0, 0, 0};
        if (local * 64 + row < d.N) z = *reinterpret_cast<const v4i*>(in_global(d.m) + (size_t)(local * 64 + row) * n_pad + col);
        *reinterpret_cast<v4i*>(&sh.s.query[row][col]) = z;
    }
    for (int i = threadIdx.x; i < 2 * 64 * kSumPitch; i += 256) (&sh.s.sum[0][0][0])[i] = 0;
    uint32_t hi = 0;
    for (int s = threadIdx.x; s < S; s += 256) {
        const C2 v = a[s];
        hi = max(hi, max((uint32_t)__double2hiint((double)v.x) & 0x7FFFFFFFu,
                         (uint32_t)__double2hiint((double)v.y) & 0x7FFFFFFFu));
    }
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) hi = max(hi, (uint32_t)__shfl_xor((int)hi, off));
    __syncthreads();
    if (lane == 0) atomicMax(&top, hi);
    __syncthreads();
    const int field = (int)(top >> 20);
    if (field == 0x7FF) {                         // infinity or NaN (the same word in all threads)
        __syncthreads();
        points_by_table<T, false, NKB>(d, local, sh.tab);
        return;
    }
    const int e = max(field, 1) - 1022;           // largest component < 2^e
    const uint32_t cosine = q == 4 ? 0x00FF0001u : q == 2 ? 0x0000FF01u : 0x00FFFF02u;
    const uint32_t sine = q == 4 ? 0xFF000100u : q == 2 ? 0u : 0x00FF0100u;
    const uint32_t mask = q == 4 ? 0x03030303u : q == 2 ? 0x01010101u : 0xFFFFFFFFu;

    v4i csum[kTiles], ssum[kTiles];
#pragma unroll
    for (int t = 0; t < kTiles; ++t) {
        csum[t] = v4i{0, 0, 0, 0};
        ssum[t] = v4i{0, 0, 0, 0};
    }
    int8_t(*dig)[64] = sh.s.dig[wave];
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
        const uint64_t bias = 0x8080808080808080ull;
        const uint64_t re = ((uint64_t)__double2ll_rn(ldexp((double)as.x, 62 - e)) + bias) ^ bias;
        const uint64_t im = ((uint64_t)__double2ll_rn(ldexp((double)as.y, 62 - e)) + bias) ^ bias;
        const uint32_t word[4] = {(uint32_t)re, (uint32_t)(re >> 32), (uint32_t)im, (uint32_t)(im >> 32)};
        const int pos = 16 * ((lane >> 2) & 3) + 4 * (lane >> 4);
#pragma unroll
        for (int j = 0; j < 4; ++j)
            *reinterpret_cast<uint32_t*>(&dig[4 * j + (lane & 3)][pos]) = quad_transpose(word[j], lane);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        const v4i bfrag = *reinterpret_cast<const v4i*>(&dig[r16][16 * g]);
#pragma unroll
        for (int t = 0; t < kTiles; ++t) {
            v4i qfrag[NKB], cf, sf;
#pragma unroll
            for (int kb = 0; kb < NKB; ++kb)
                qfrag[kb] = *reinterpret_cast<const v4i*>(&sh.s.query[16 * t + r16][64 * kb + 16 * g]);
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
                    for (int v = 0; v < 4; ++v)
                        p[v] -= 3 * (int)fmaf((float)p[v], 1.0f / 3.0f, 1.0f / 6.0f);
                }
                const uint32_t lo = __builtin_amdgcn_perm((uint32_t)p[1], (uint32_t)p[0], 0x0C0C0400u);
                const uint32_t up = __builtin_amdgcn_perm((uint32_t)p[3], (uint32_t)p[2], 0x04000C0Cu);
                const uint32_t r = (lo | up) & mask;
                cf[u] = (int)__builtin_amdgcn_perm(0u, cosine, r);
                sf[u] = (int)__builtin_amdgcn_perm(0u, sine, r);
            }
            csum[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(cf, bfrag, csum[t], 0, 0, 0);
            ssum[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(sf, bfrag, ssum[t], 0, 0, 0);
        }
        __builtin_amdgcn_wave_barrier();          // the fragment is read before the next block's digits
    }
#pragma unroll
    for (int t = 0; t < kTiles; ++t) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            atomicAdd(&sh.s.sum[0][16 * t + 4 * g + v][r16], csum[t][v]);
            atomicAdd(&sh.s.sum[1][16 * t + 4 * g + v][r16], ssum[t][v]);
        }
    }
    __syncthreads();
    const int qi = threadIdx.x >> 1, part = threadIdx.x & 1;      // query, re or im
    const int64_t ql = local * 64 + qi;
    if (qi >= 64 || ql >= d.N) return;
    int64_t c0 = 0, c1 = 0, z0 = 0, z1 = 0;       // low and high four digits of the two sums
#pragma unroll
    for (int j = 3; j >= 0; --j) {
        c0 = c0 * 256 + sh.s.sum[0][qi][8 * part + j];
        c1 = c1 * 256 + sh.s.sum[0][qi][8 * part + 4 + j];
        z0 = z0 * 256 + sh.s.sum[1][qi][8 * (1 - part) + j];
        z1 = z1 * 256 + sh.s.sum[1][qi][8 * (1 - part) + 4 + j];
    }
    if (!part) {                                  // re: cos re - sin im; im: cos im + sin re
        z0 = -z0;
        z1 = -z1;
    }
    double x;
    if (q == 3) {
        const double cs = fma((double)c1, 4294967296.0, (double)c0);
        const double zs = fma((double)z1, 4294967296.0, (double)z0);
        x = fma(0.86602540378443864676, zs, 0.5 * cs);
    } else {
        x = fma((double)(c1 + z1), 4294967296.0, (double)(c0 + z0));
    }
    in_global(reinterpret_cast<T*>(d.x))[2 * ql + part] = (T)ldexp(x, e - 62);
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
// They win at every size measured, from S = 10 or 1000 queries up (above).
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
