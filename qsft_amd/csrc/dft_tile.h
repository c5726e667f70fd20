// The sub-DFT building blocks shared by the forward passes (dft.hip) and the
// inverse ones of the coset evaluation (fold.hip): q-point pencils in LDS and
// registers, and the axis loop over a staged tile.
#pragma once
#include "qsft_common.h"

namespace qsft {

// Workgroups of the tile kernels by their LDS: 256 threads up to 32 KiB (four
// and more per CU), 512 up to 64 KiB (two per CU; a strided pass, bound by its
// loads, stays at 256: 134 against 149 us on a serving mix's q = 20, b = 4
// rows), and for whole rows beyond that, at most 144 of the 160 KiB of a CU, as
// many as the registers allow. q = 20, b = 3: the samples of 102 rows in FP32
// (64 KiB) 19.6 us with 256 threads, 13.4 with 512; their FP64 sub-DFT 29 us in
// two passes, 17 as whole rows of 128 KiB.
constexpr int kDftThreads = 256;
constexpr int kDftMidBytes = 32768;
constexpr int kDftMidThreads = 512;
constexpr int kDftLdsBytes = 65536;
constexpr int kRowLdsBytes = 147456;
template <typename T> constexpr int row_threads() { return sizeof(T) == 8 ? 512 : 1024; }

template <typename T>
__device__ __forceinline__ cplx_t<T> cmul(cplx_t<T> a, cplx_t<T> b) {
    cplx_t<T> r;
    r.x = a.x * b.x - a.y * b.y;
    r.y = a.x * b.y + a.y * b.x;
    return r;
}

// x / d for x d < 2^32 by one multiply-high (m = floor(2^32 / d) + 1; the
// error term x / 2^32 < 1 / d cannot cross the next integer).
struct FastDiv {
    uint32_t d, m;
    __device__ explicit FastDiv(uint32_t d_) : d(d_), m(d_ > 1 ? (uint32_t)(0xFFFFFFFFull / d_) + 1u : 0u) {}
    __device__ __forceinline__ uint32_t div(uint32_t x) const { return d == 1 ? x : __umulhi(x, m); }
};

template <typename T>
__device__ __forceinline__ void dft4_reg(cplx_t<T>& x0, cplx_t<T>& x1, cplx_t<T>& x2, cplx_t<T>& x3) {
    using C2 = cplx_t<T>;
    const C2 s02{x0.x + x2.x, x0.y + x2.y}, d02{x0.x - x2.x, x0.y - x2.y};
    const C2 s13{x1.x + x3.x, x1.y + x3.y}, d13{x1.x - x3.x, x1.y - x3.y};
    x0 = C2{s02.x + s13.x, s02.y + s13.y};
    x2 = C2{s02.x - s13.x, s02.y - s13.y};
    x1 = C2{d02.x + d13.y, d02.y - d13.x};                        // d02 + (-i) d13
    x3 = C2{d02.x - d13.y, d02.y + d13.x};
}

// Five-point forward DFT in registers: with a1 = x1 + x4, a2 = x2 + x3,
// b1 = x1 - x4, b2 = x2 - x3, c_k = cos(2 pi k / 5), s_k = sin(2 pi k / 5):
// X1,4 = x0 + c1 a1 + c2 a2 -/+ i (s1 b1 + s2 b2), X2,3 = x0 + c2 a1 + c1 a2 -/+ i (s2 b1 - s1 b2).
template <typename T>
__device__ __forceinline__ void dft5_reg(cplx_t<T>& x0, cplx_t<T>& x1, cplx_t<T>& x2, cplx_t<T>& x3,
                                         cplx_t<T>& x4) {
    using C2 = cplx_t<T>;
    const T c1 = (T)0.30901699437494742410, c2 = (T)-0.80901699437494742410;
    const T s1 = (T)0.95105651629515357212, s2 = (T)0.58778525229247312917;
    const C2 a1{x1.x + x4.x, x1.y + x4.y}, a2{x2.x + x3.x, x2.y + x3.y};
    const C2 b1{x1.x - x4.x, x1.y - x4.y}, b2{x2.x - x3.x, x2.y - x3.y};
    const C2 t1{x0.x + c1 * a1.x + c2 * a2.x, x0.y + c1 * a1.y + c2 * a2.y};
    const C2 t2{x0.x + c2 * a1.x + c1 * a2.x, x0.y + c2 * a1.y + c1 * a2.y};
    const C2 u1{s1 * b1.x + s2 * b2.x, s1 * b1.y + s2 * b2.y};
    const C2 u2{s2 * b1.x - s1 * b2.x, s2 * b1.y - s1 * b2.y};
    x0 = C2{x0.x + a1.x + a2.x, x0.y + a1.y + a2.y};
    x1 = C2{t1.x + u1.y, t1.y - u1.x};                            // t1 - i u1
    x4 = C2{t1.x - u1.y, t1.y + u1.x};
    x2 = C2{t2.x + u2.y, t2.y - u2.x};
    x3 = C2{t2.x - u2.y, t2.y + u2.x};
}

// In-place q-point forward DFT of the pencil v[0], v[st], ..., v[(q-1) st].
template <typename T, int QR>
__device__ __forceinline__ void pencil(cplx_t<T>* v, int st, const cplx_t<T>* tw) {
    using C2 = cplx_t<T>;
    if constexpr (QR == 2) {
        const C2 a = v[0], b = v[st];
        v[0] = C2{a.x + b.x, a.y + b.y};
        v[st] = C2{a.x - b.x, a.y - b.y};
    } else if constexpr (QR == 3) {
        const T h = (T)0.86602540378443864676;                    // sin(2 pi / 3)
        const C2 x0 = v[0], x1 = v[st], x2 = v[2 * st];
        const C2 a{x1.x + x2.x, x1.y + x2.y}, d{x1.x - x2.x, x1.y - x2.y};
        const C2 t{x0.x - (T)0.5 * a.x, x0.y - (T)0.5 * a.y};
        v[0] = C2{x0.x + a.x, x0.y + a.y};
        v[st] = C2{t.x + h * d.y, t.y - h * d.x};                 // t - i h d
        v[2 * st] = C2{t.x - h * d.y, t.y + h * d.x};
    } else if constexpr (QR == 4) {
        C2 x0 = v[0], x1 = v[st], x2 = v[2 * st], x3 = v[3 * st];
        dft4_reg<T>(x0, x1, x2, x3);
        v[0] = x0;
        v[st] = x1;
        v[2 * st] = x2;
        v[3 * st] = x3;
    } else if constexpr (QR == 5) {
        C2 x0 = v[0], x1 = v[st], x2 = v[2 * st], x3 = v[3 * st], x4 = v[4 * st];
        dft5_reg<T>(x0, x1, x2, x3, x4);
        v[0] = x0;
        v[st] = x1;
        v[2 * st] = x2;
        v[3 * st] = x3;
        v[4 * st] = x4;
    } else if constexpr (QR == 20) {
        // prime-factor 4 x 5: y[n1][n2] = x[(5 n1 + 4 n2) mod 20]
        C2 y[4][5];
#pragma unroll
        for (int n1 = 0; n1 < 4; ++n1)
#pragma unroll
            for (int n2 = 0; n2 < 5; ++n2) y[n1][n2] = v[((5 * n1 + 4 * n2) % 20) * st];
#pragma unroll
        for (int n2 = 0; n2 < 5; ++n2) dft4_reg<T>(y[0][n2], y[1][n2], y[2][n2], y[3][n2]);
#pragma unroll
        for (int k1 = 0; k1 < 4; ++k1) dft5_reg<T>(y[k1][0], y[k1][1], y[k1][2], y[k1][3], y[k1][4]);
#pragma unroll
        for (int k1 = 0; k1 < 4; ++k1)
#pragma unroll
            for (int k2 = 0; k2 < 5; ++k2) v[((5 * k1 + 16 * k2) % 20) * st] = y[k1][k2];
    } else {
        C2 x[QR];
#pragma unroll
        for (int r = 0; r < QR; ++r) x[r] = v[r * st];
#pragma unroll
        for (int k = 0; k < QR; ++k) {
            C2 acc = x[0];
#pragma unroll
            for (int r = 1; r < QR; ++r) {
                const C2 w = tw[(r * k) % QR];
                acc.x += x[r].x * w.x - x[r].y * w.y;
                acc.y += x[r].x * w.y + x[r].y * w.x;
            }
            v[k * st] = acc;
        }
    }
}

// Generic q (not compiled for a fixed radix): one axis (stride G) of a tile of
// E elements, out of place through a second LDS buffer, N outputs of q terms
// per thread: a pencil per thread left a workgroup three quarters idle behind
// q^2 terms one after the other (33 rows of q = 64, b = 2, the samples of S =
// 10: 690 us a call in FP32, now 42; 710 in FP64, now 62). Bound by its LDS
// reads, a term and a root of unity for every product: four outputs share their
// terms where the axis has enough of them (FP64, q = 64: 70 us with one).
template <typename T, int N>
__device__ __forceinline__ void axis_generic_by(const cplx_t<T>* src, cplx_t<T>* dst, int E, int q, int G,
                                                const cplx_t<T>* tw) {
    constexpr int kUnroll = N > 1 ? 2 : 4;
    const int nk = (q + N - 1) / N;                                // a thread's outputs are nk apart
    const FastDiv fg((uint32_t)G), fk((uint32_t)nk);
    const int items = E / q * nk;
    for (int i = threadIdx.x; i < items; i += blockDim.x) {
        const int a = (int)fg.div((uint32_t)i), X = (int)fk.div((uint32_t)a), k = a - X * nk;
        const int p0 = X * q * G + (i - a * G);
        const cplx_t<T>* v = src + p0;
        cplx_t<T> acc[N];
        int rk[N], kn[N];                                          // r k mod q
#pragma unroll
        for (int n = 0; n < N; ++n) {
            kn[n] = k + n * nk < q ? k + n * nk : 0;               // (past the last output: not stored)
            rk[n] = 0;
            acc[n] = v[0];
        }
#pragma unroll kUnroll
        for (int r = 1; r < q; ++r) {
            const cplx_t<T> x = v[r * G];
#pragma unroll
            for (int n = 0; n < N; ++n) {
                rk[n] += kn[n];
                if (rk[n] >= q) rk[n] -= q;
                const cplx_t<T> w = tw[rk[n]];
                acc[n].x += x.x * w.x - x.y * w.y;
                acc[n].y += x.x * w.y + x.y * w.x;
            }
        }
#pragma unroll
        for (int n = 0; n < N; ++n)
            if (k + n * nk < q) dst[p0 + (k + n * nk) * G] = acc[n];
    }
}
template <typename T>
__device__ __forceinline__ void axis_generic(const cplx_t<T>* src, cplx_t<T>* dst, int E, int q, int G,
                                             const cplx_t<T>* tw) {
    if (q >= 16) axis_generic_by<T, 4>(src, dst, E, q, G, tw);
    else axis_generic_by<T, 1>(src, dst, E, q, G, tw);
}

__host__ __device__ __forceinline__ bool radix_compiled(int q) {
    return q == 2 || q == 3 || q == 4 || q == 5 || q == 20;
}

// A tile of E elements into LDS, get(e) being the global load of element e:
// kTileLoads loads of a thread are in flight together (one at a time, each
// waited for before the next was issued, a 64 KiB tile of 256 threads spent 31
// memory latencies on its way in).
// A tile of at most two elements per thread moves without the other six steps'
// conditions (q = 20, b = 2, 1347 rows in FP64: 20.2 -> 16.6 us back to back).
constexpr int kTileLoads = 8;
template <int N, typename C2, typename G>
__device__ __forceinline__ void tile_load_steps(C2* lds, int E, G get) {
    for (int e0 = threadIdx.x; e0 < E; e0 += N * blockDim.x) {
        C2 v[N];
#pragma unroll
        for (int k = 0; k < N; ++k) {
            const int e = e0 + k * blockDim.x;
            if (e < E) v[k] = get(e);
        }
#pragma unroll
        for (int k = 0; k < N; ++k) {
            const int e = e0 + k * blockDim.x;
            if (e < E) lds[e] = v[k];
        }
    }
}
template <typename C2, typename G>
__device__ __forceinline__ void tile_load(C2* lds, int E, G get) {
    if (E <= 2 * (int)blockDim.x) tile_load_steps<2>(lds, E, get);
    else tile_load_steps<kTileLoads>(lds, E, get);
}

// And out again: put(e, value).
template <int N, typename C2, typename F>
__device__ __forceinline__ void tile_store_steps(const C2* lds, int E, F put) {
    for (int e0 = threadIdx.x; e0 < E; e0 += N * blockDim.x) {
        C2 v[N];
#pragma unroll
        for (int k = 0; k < N; ++k) {
            const int e = e0 + k * blockDim.x;
            if (e < E) v[k] = lds[e];
        }
#pragma unroll
        for (int k = 0; k < N; ++k) {
            const int e = e0 + k * blockDim.x;
            if (e < E) put(e, v[k]);
        }
    }
}
template <typename C2, typename F>
__device__ __forceinline__ void tile_store(const C2* lds, int E, F put) {
    if (E <= 2 * (int)blockDim.x) tile_store_steps<2>(lds, E, put);
    else tile_store_steps<kTileLoads>(lds, E, put);
}

// The axis transforms of a tile of E elements, [.., q^mb, ti] with its mb axes
// innermost first, or outermost first (axis t has stride q^(mb-1-t) ti in the
// tile), by the whole workgroup, which has synchronised after filling `cur`.
// The generic radix is out of place (`alt`, E more elements). Returns the
// buffer that holds the result; the workgroup is synchronised.
template <typename T, int QR>
__device__ __forceinline__ cplx_t<T>* tile_axes(cplx_t<T>* cur, cplx_t<T>* alt, int E, int q, int mb, int ti,
                                                const cplx_t<T>* tw, bool outermost_first = false) {
    const int pencils = E / q;
    for (int t = 0; t < mb; ++t) {
        const int G = ti * ipow(q, outermost_first ? mb - 1 - t : t);
        if constexpr (QR > 0) {
            const FastDiv fd((uint32_t)G);
            for (int pc = threadIdx.x; pc < pencils; pc += blockDim.x) {
                const int X = (int)fd.div((uint32_t)pc);
                pencil<T, QR>(cur + X * q * G + (pc - X * G), G, tw);
            }
        } else {
            axis_generic<T>(cur, alt, E, q, G, tw);
            cplx_t<T>* tmp = cur;
            cur = alt;
            alt = tmp;
        }
        __syncthreads();
    }
    return cur;
}

// Q = q^b: the forward scale of the last pass (a division in FP64, like numpy's
// / q**n; a multiply by the rounded reciprocal in FP32)
template <typename T>
__device__ __forceinline__ cplx_t<T> dft_scaled(cplx_t<T> v, int Q) {
    if constexpr (sizeof(T) == 8) return cplx_t<T>{v.x / (double)Q, v.y / (double)Q};
    const T sc = (T)(1.0 / (double)Q);
    return cplx_t<T>{v.x * sc, v.y * sc};
}

// q = 4, whole rows held 16 samples a thread: element index of register j when
// the thread holds digits w, w + 1 (base-4 digit t at bits 2t, 2t + 1)
__device__ __forceinline__ int dft4_index(int w, int tid, int j) {
    const int lo = 2 * w;
    return ((tid >> lo) << (lo + 4)) | (j << lo) | (tid & ((1 << lo) - 1));
}
__device__ __forceinline__ int dft4_pad(int i) { return i + (i >> 4); }
// dft4_pad(dft4_index(w, tid, j)) = dft4_lds_base(w, tid) + j dft4_lds_step(w) for
// w = 0 or w >= 2: one address per window, the 16 elements at immediate offsets
__device__ __forceinline__ int dft4_lds_base(int w, int tid) { return dft4_pad(dft4_index(w, tid, 0)); }
__device__ __forceinline__ constexpr int dft4_lds_step(int w) { return w == 0 ? 1 : 17 << (2 * w - 4); }

}  // namespace qsft
