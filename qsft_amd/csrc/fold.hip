// Stage (a)+(b), coset evaluation through the folded spectrum.
//
// Every query of group c is m = (M_c l + d_p) mod q, and mod q is a ring
// homomorphism, so its phase against a support vector splits exactly:
//   <m, k_s> = <l, M_c^T k_s> + <d_p, k_s>   (mod q).
// The first product depends on k_s only through its bin j_s = M_c^T k_s mod q,
// so the q^b samples of a coset are
//   x[c][p][l] = sum_j w^{<l, j>} F[c][p][j],
//   F[c][p][j] = sum over j_s = j of a_s w^{<d_p, k_s>},
// the unscaled inverse [q]*b transform of the S terms folded into their bins:
// S + Q b (q - 1) operations a row where the sum over every support at every
// query takes S Q. Every sample is still the whole sum of a_s w^{<m, k_s>};
// terms and bin sums are formed in FP64 and rounded once.
//
//   * k_fold_phase: the int8 contraction K . [D; M]^T on
//     v_mfma_i32_16x16x64_i8 (exact int32), then mod q: the phases
//     E[p][s] = <d_p, k_s> as bytes, and the bins j_s of every group from the
//     b products with M_c^T.
//   * k_fold_rank: per group the supports sorted by (bin, s), each at its rank,
//     counted against LDS tiles of the bins: the terms of a bin are adjacent
//     and always summed in one order (a scan over blocks of 64 sorted
//     positions), so the sums have the same bits on every run. Also the first sorted position of every tile of the row
//     kernel. Many supports are ranked in two steps: within chunks of 2048
//     (k_fold_chunk), then by a binary search in every other chunk.
//   * k_fold_pass / k_fold4_rows: a workgroup clears a tile of bins of one row
//     in LDS, adds the tile's terms and runs the
//     inverse transform over the tile's axes; k_fold4_rows (q = 4, b = 4
//     .. 7) does the whole row, two digits at a time in registers. Rows
//     larger than a tile take further k_fold_pass passes in place.
//
// The inverse transform is the forward one with the real and imaginary parts
// swapped on the way in and out, so it shares the forward radix kernels: the
// fold stores swapped terms and the last pass swaps back.
//
// HBM is all that it cannot do without: a row is written once (8 or 16 bytes a
// sample) where it fits one tile; nothing else of that order is read. One
// instance is bound by three dependent launches, many by the VALU (see
// k_fold4_rows). Measured against the sums over every support that these
// kernels replaced: one q = 4, n = 50, S = 1000, b = 6, 306-row signal in FP64
// 463 -> 23 us a call, 64 of them in FP32 in one launch 0.91 -> 0.26 ms; q = 20,
// S = 2000, b = 3, FP32 570 -> 27 us. FP32 against FP64, of the samples' size:
// 6e-8 to 1.3e-7 for every S (the direct sums 5e-8 at S = 10, 1e-7 at 300, 3e-7
// at 5000; generic radices up to 2e-7).
#include <algorithm>

#include "dft_tile.h"

namespace qsft {

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int kPhaseThreads = 256;   // four waves, 16 supports each
constexpr int kPhaseTiles = 4;       // 16-row tiles of [D; M] per workgroup
constexpr int kRankThreads = 1024;
constexpr int kRankTileKeys = 2048;
// Supports up to which every one is compared with every other, S^2 comparisons a
// group; beyond, S / 2048 searches of twelve steps each. A call of few samples,
// C = 3, one step / two: S = 8000 111 us / -, 10000 129 / 107, 30000 600 / 295,
// 100000 4720 / 1004, 300000 36400 / 4320.
constexpr int kRankDirect = 8192;

__host__ __device__ __forceinline__ int fold_sp(int S) { return (S + 15) / 16 * 16; }
// chunks of kRankTileKeys supports that are ranked by themselves first; 0: one step
__host__ __device__ __forceinline__ int fold_chunks(int S) {
    return S > kRankDirect ? (S + kRankTileKeys - 1) / kRankTileKeys : 0;
}
// tile boundaries ranked with the supports: none where a row is one tile
__host__ __device__ __forceinline__ int fold_bounds(int tiles) { return tiles > 1 ? tiles + 1 : 0; }

// tab[r] = w^r, exact for q in {2, 4}
__device__ __forceinline__ void fold_wtable(double2* tab, int q) {
    for (int r = threadIdx.x; r < q; r += blockDim.x) {
        double s, c;
        if (q == 4) {
            c = (double)((r == 0) - (r == 2));
            s = (double)((r == 1) - (r == 3));
        } else {
            sincospi(2.0 * (double)r / (double)q, &s, &c);
        }
        tab[r] = make_double2(c, s);
    }
}

// Phases and bins. A workgroup owns 64 supports (one 16-support block per
// wave) and kPhaseTiles of the instance's 16-row tiles: first the delay-row
// tiles (of every group that has its own), then one M^T tile per group. The
// support digits are the A operand (lane 16 g + r: row r, digits 16 g .. +15),
// the rows the B operand; lane 16 g + r then holds column r, supports
// 4 g .. 4 g + 3.
template <typename SRC>
__global__ __launch_bounds__(kPhaseThreads) void k_fold_phase(const SRC src) {
    int local;
    const qsft_fold_desc& d = src.at(blockIdx.x, local);
    const int q = d.q, b = d.b, C = d.C, P = d.P, S = d.S, n_pad = d.n_pad;
    const int Sp = fold_sp(S);
    const int sgroups = (S + 63) / 64;
    const int tg = local / sgroups, sg = local - tg * sgroups;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int g = lane >> 4, r16 = lane & 15;
    const int s0 = sg * 64 + wave * 16;
    if (local == 0 && threadIdx.x == 0) in_global(d.bad)[0] = 0;   // (counted by k_fold_rank)
    if (s0 >= S) return;
    const int ptiles = (P + 15) / 16;
    const int dtiles = (d.shared_d ? 1 : C) * ptiles;
    const ModQ mq((uint32_t)q);
    const int8_t* __restrict__ krow = in_global(d.K) + (size_t)min(s0 + r16, S - 1) * n_pad + 16 * g;
    v4i kf[QSFT_MAX_N / 64];
#pragma unroll
    for (int kb = 0; kb < QSFT_MAX_N / 64; ++kb)
        kf[kb] = (64 * kb < n_pad) ? *reinterpret_cast<const v4i*>(krow + 64 * kb) : v4i{0, 0, 0, 0};
    for (int tile = tg * kPhaseTiles; tile < min((tg + 1) * kPhaseTiles, dtiles + C); ++tile) {
        const bool bins = tile >= dtiles;
        const int c = bins ? tile - dtiles : tile / ptiles;
        const int p = (bins ? 0 : 16 * (tile - c * ptiles)) + r16;
        const int rows = bins ? b : P;
        const int8_t* __restrict__ row =
            (bins ? d.Mt : d.D) + ((size_t)c * rows + min(p, rows - 1)) * n_pad + 16 * g;
        v4i e = {0, 0, 0, 0};
#pragma unroll
        for (int kb = 0; kb < QSFT_MAX_N / 64; ++kb) {
            if (64 * kb < n_pad)
                e = __builtin_amdgcn_mfma_i32_16x16x64_i8(kf[kb], *reinterpret_cast<const v4i*>(row + 64 * kb), e, 0,
                                                          0, 0);
        }
        if (!bins) {
            uint32_t w = 0;
#pragma unroll
            for (int v = 0; v < 4; ++v) w |= mq((uint32_t)e[v]) << (8 * v);
            if (p < P) *reinterpret_cast<uint32_t*>(in_global(d.E) + ((size_t)c * P + p) * Sp + s0 + 4 * g) = w;
        } else {
            int place = 0;                                         // q^(b - 1 - r16)
            if (r16 < b) {
                place = 1;
                for (int t = r16 + 1; t < b; ++t) place *= q;
            }
            int j[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) j[v] = row_sum_i((int)mq((uint32_t)e[v]) * place);
            const int mine = r16 == 0 ? j[0] : r16 == 1 ? j[1] : r16 == 2 ? j[2] : j[3];
            if (r16 < 4 && s0 + 4 * g + r16 < S) in_global(d.J)[(size_t)c * S + s0 + 4 * g + r16] = (uint32_t)mine;
        }
    }
}

__device__ __forceinline__ bool finite2(double2 a) {
    return __builtin_isfinite(a.x) && __builtin_isfinite(a.y);
}

// The keys of one LDS tile (the supports from t0, tn of them, then padding that
// counts nowhere) below bin j, or of bin j and a support before `upto`: this
// wave's sixteenth of them.
__device__ __forceinline__ uint32_t rank_in_tile(const uint32_t* keys, int t0, int tn, uint32_t j, int upto, int wave) {
    constexpr int kWaves = kRankThreads / 64;
    const int share = ((tn + kWaves - 1) / kWaves + 3) & ~3;
    const int z = min(tn, (wave + 1) * share);
    uint32_t rank = 0;
#pragma unroll 4
    for (int t = wave * share; t < z; t += 4) {
        const uint4 k = *reinterpret_cast<const uint4*>(keys + t);
        const int at = t0 + t;
        rank += k.x < j + (at < upto ? 1u : 0u) ? 1u : 0u;
        rank += k.y < j + (at + 1 < upto ? 1u : 0u) ? 1u : 0u;
        rank += k.z < j + (at + 2 < upto ? 1u : 0u) ? 1u : 0u;
        rank += k.w < j + (at + 3 < upto ? 1u : 0u) ? 1u : 0u;
    }
    return rank;
}

// First step of many supports, 64 of one chunk per workgroup: their ranks in the
// chunk, and the chunk's bins in that order.
template <typename SRC>
__global__ __launch_bounds__(kRankThreads) void k_fold_chunk(const SRC src) {
    constexpr int kWaves = kRankThreads / 64;
    __shared__ __align__(16) uint32_t keys[kRankTileKeys];
    __shared__ uint32_t part[kWaves][64];
    int local;
    const qsft_fold_desc& d = src.at(blockIdx.x, local);
    if (!d.chunk) return;
    const int S = d.S, S64 = (S + 63) / 64 * 64;
    const int per_c = (S64 + fold_bounds(d.tiles) + 63) / 64;
    const int c = local / per_c, first = (local - c * per_c) * 64;
    if (first >= S) return;                                        // tile boundaries
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, item = first + lane;
    const uint32_t* __restrict__ J = in_global(d.J) + (size_t)c * S;
    const int t0 = first / kRankTileKeys * kRankTileKeys, tn = min(kRankTileKeys, S - t0);
    for (int t = threadIdx.x; t < kRankTileKeys; t += kRankThreads) keys[t] = t < tn ? J[t0 + t] : 0xFFFFFFFFu;
    __syncthreads();
    const uint32_t j = item < S ? keys[item - t0] : 0;
    part[wave][lane] = rank_in_tile(keys, t0, tn, j, item, wave);
    __syncthreads();
    if (wave != 0 || item >= S) return;
    uint32_t rank = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) rank += part[w][lane];
    uint32_t* __restrict__ out = in_global(d.chunk) + (size_t)c * S;
    out[t0 + rank] = j;
    out[(size_t)d.C * S + item] = rank;
}

// Keys below j among the chunks (in order) of one group, those of bin j too in
// the chunks before `own`, whose own count is left out: this wave's share of the
// chunks, four searches at once.
__device__ __forceinline__ uint32_t rank_in_chunks(const uint32_t* __restrict__ sorted, int S, int chunks, uint32_t j,
                                                   int own, int wave) {
    constexpr int kWaves = kRankThreads / 64, kAtOnce = 4;
    uint32_t rank = 0;
    for (int c0 = wave * kAtOnce; c0 < chunks; c0 += kWaves * kAtOnce) {
        int pos[kAtOnce];
#pragma unroll
        for (int i = 0; i < kAtOnce; ++i) pos[i] = 0;
        for (int step = kRankTileKeys; step > 0; step >>= 1) {
#pragma unroll
            for (int i = 0; i < kAtOnce; ++i) {
                const int ch = c0 + i, t0 = ch * kRankTileKeys;
                const int tn = ch < chunks && ch != own ? min(kRankTileKeys, S - t0) : 0;
                if (pos[i] + step <= tn && sorted[t0 + pos[i] + step - 1] < j + (ch < own ? 1u : 0u)) pos[i] += step;
            }
        }
#pragma unroll
        for (int i = 0; i < kAtOnce; ++i) rank += (uint32_t)pos[i];
    }
    return rank;
}

// Items of one group: its S supports, then (from the next multiple of 64) the
// tiles + 1 tile boundaries. An item's rank among the supports by (bin, s) is
// its sorted position, where its key and strength are written; a boundary's is
// the number of supports in lower bins. A workgroup ranks 64 items, one per
// lane; its 16 waves each count a sixteenth of every LDS tile of bins (the
// scan is a chain of LDS reads: one wave counting all 1000 supports of the
// headline size took 27 us, sixteen take 5).
template <typename SRC>
__global__ __launch_bounds__(kRankThreads) void k_fold_rank(const SRC src) {
    constexpr int kWaves = kRankThreads / 64;
    __shared__ __align__(16) uint32_t keys[kRankTileKeys];
    __shared__ uint32_t part[kWaves][64];
    int local;
    const qsft_fold_desc& d = src.at(blockIdx.x, local);
    const int S = d.S, S64 = (S + 63) / 64 * 64;
    const int per_c = (S64 + fold_bounds(d.tiles) + 63) / 64;
    const int c = local / per_c;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int item = (local - c * per_c) * 64 + lane;
    const bool support = item < S, bound = item >= S64 && item - S64 < fold_bounds(d.tiles);
    const uint32_t* __restrict__ J = in_global(d.J) + (size_t)c * S;
    uint32_t j = 0;
    if (support) j = J[item];
    if (bound) j = (uint32_t)(item - S64) * (uint32_t)d.tile_bins;
    const int upto = item < S64 ? item : 0;                        // equal bins count before this index
    uint32_t rank = 0;
    if (d.chunk) {                                                 // (block-uniform)
        const uint32_t* __restrict__ sorted = in_global(d.chunk) + (size_t)c * S;
        const int own = support ? item / kRankTileKeys : -1;
        rank = rank_in_chunks(sorted, S, fold_chunks(S), j, own, wave);
        if (wave == 0 && support) rank += sorted[(size_t)d.C * S + item];
    } else {
        for (int t0 = 0; t0 < S; t0 += kRankTileKeys) {
            const int tn = min(kRankTileKeys, S - t0);
            __syncthreads();                                       // the previous tile is consumed
            for (int t = threadIdx.x; t < kRankTileKeys; t += kRankThreads) keys[t] = t < tn ? J[t0 + t] : 0xFFFFFFFFu;
            __syncthreads();
            rank += rank_in_tile(keys, t0, tn, j, upto, wave);
        }
    }
    part[wave][lane] = rank;
    __syncthreads();
    if (wave != 0) return;
    rank = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) rank += part[w][lane];
    if (support) {
        in_global(d.key)[(size_t)c * S + rank] = ((uint64_t)j << 32) | (uint32_t)item;
        double2 a;
        if (d.a_prec == QSFT_F32) {
            const float2 f = reinterpret_cast<const float2*>(d.a)[item];
            a = make_double2(f.x, f.y);
        } else {
            a = reinterpret_cast<const double2*>(d.a)[item];
        }
        if (!finite2(a)) {
            if (d.fwd) {
                a = make_double2(__builtin_nan(""), __builtin_nan(""));
            } else {
                if (c == 0) in_global(d.bad)[1 + atomicAdd(in_global(d.bad), 1u)] = (uint32_t)item;
                a = make_double2(0.0, 0.0);
            }
        }
        reinterpret_cast<double2*>(d.as)[(size_t)c * S + rank] = a;
    }
    if (bound) in_global(d.start)[(size_t)c * (d.tiles + 1) + (item - S64)] = (int32_t)rank;
}

// The terms of one row are added to their bins in LDS by the waves of a
// workgroup. Wave `wave` of `waves` takes an equal share of the blocks of 64
// sorted positions that hold [lo, hi) of the group, moved to the ends of runs
// (the terms of one bin), so no two waves touch a bin and none waits for
// another. A block at a time: each lane forms one term, a segmented scan over
// the run (as many steps as the longest run in the block needs) leaves a run's
// sum in its last lane, which stores it, or hands it on to the next block in
// FP64 registers where the run goes on there: a bin is rounded once, however
// many terms it has. Equal shares keep a row's time even where terms crowd in a
// few bins, down to one wave's for a single bin. The blocks are the same for
// every tile and workgroup size, so the order of a sum depends on the sorted
// positions only.
//
// What a lane needs of its position, the same for every row of the group:
struct Term {
    uint32_t j, s;       // bin and support
    gd2 a;               // strength
    int flags;           // kTermLive | kTermEmit | kTermOpen | kTermOn | lanes back to the run's first live lane
};
constexpr int kTermDepth = 63;       // mask of the distance
constexpr int kTermLive = 64;        // a term of this wave
constexpr int kTermEmit = 128;       // last term of the run
constexpr int kTermOpen = 256;       // lane 63 of a run that goes on in the next block
constexpr int kTermOn = 512;         // a run that began in an earlier block

struct TermShare {
    int lo, hi, first, last;
    bool started;        // a run that began before `first` is another wave's
    __device__ __forceinline__ TermShare(int lo_, int hi_, int wave, int waves) : lo(lo_), hi(hi_) {
        const int b0 = lo >> 6, nb = hi > lo ? ((hi + 63) >> 6) - b0 : 0;
        first = (b0 + (int)((int64_t)nb * wave / waves)) << 6;
        last = (b0 + (int)((int64_t)nb * (wave + 1) / waves)) << 6;
        started = first <= lo;
    }
    // Loads the block of 64 positions from i0; false once the share has ended.
    __device__ __forceinline__ bool load(const qsft_fold_desc& d, int c, int i0, Term& t) {
        const int lane = threadIdx.x & 63;
        t.flags = 0;
        t.j = t.s = 0;
        t.a = gd2{0.0, 0.0};
        if (i0 >= hi || first >= last) return false;
        const QSFT_GLOBAL uint64_t* __restrict__ key = gptr(d.key) + (size_t)c * d.S;
        const QSFT_GLOBAL gd2* __restrict__ as =
            reinterpret_cast<const QSFT_GLOBAL gd2*>(gptr(d.as)) + (size_t)c * d.S;
        const int i = i0 + lane;
        const bool in = i >= lo && i < hi;
        const uint64_t k = in ? key[i] : ~0ull;
        const uint32_t kp = (in && i > lo) ? (uint32_t)(key[i - 1] >> 32) : 0xFFFFFFFFu;
        const uint32_t kn = (in && i + 1 < hi) ? (uint32_t)(key[i + 1] >> 32) : 0xFFFFFFFFu;
        if (in) t.a = as[i];
        t.j = (uint32_t)(k >> 32);
        t.s = (uint32_t)k;
        const bool begins = in && t.j != kp;                       // first term of its bin
        const uint64_t bm = __ballot(begins);
        const uint64_t past = __ballot(begins && i >= last);       // the runs of the next share
        int from = max(0, lo - i0), to = min(64, hi - i0);
        if (!started) from = bm ? __builtin_ctzll(bm) : 64;
        if (past) to = min(to, (int)__builtin_ctzll(past));
        if (from < to) {
            started = true;
            if (lane >= from && lane < to) {
                const uint64_t before = bm & (~0ull >> (63 - lane));
                t.flags = kTermLive | (lane - max(before ? 63 - (int)__builtin_clzll(before) : 0, from));
                if (t.j != kn) t.flags |= kTermEmit;
                else if (lane == 63) t.flags |= kTermOpen;
                if (!before) t.flags |= kTermOn;
            }
        }
        return past == 0;
    }
};

// The value one lane below (lane 0: unspecified), on the VALU.
__device__ __forceinline__ double lane_below(double v) {
    return dpp_f64<0x138>(v);                                      // wave_shr:1
}

// FP64 value of lane 63 in all lanes.
__device__ __forceinline__ double lane63(double v) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, 63);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), 63);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// Sums of one block's runs: term(t, sx, sy) forms a live lane's term,
// put(t, sx, sy) takes the sum of a run in its last lane. cx, cy: the sum so
// far of the run that the block before left open.
template <typename TM, typename F>
__device__ __forceinline__ void term_add(const Term& t, double& cx, double& cy, TM term, F put) {
    if (!__ballot(t.flags & kTermLive)) return;
    double sx = 0.0, sy = 0.0;
    if (t.flags & kTermLive) term(t, sx, sy);
    const int depth = t.flags & kTermDepth;
    if (__ballot(depth >= 1)) {
        const double px = lane_below(sx), py = lane_below(sy);
        if (depth >= 1) {
            sx += px;
            sy += py;
        }
        for (int off = 2; __ballot(depth >= off); off <<= 1) {
            const double qx = __shfl_up(sx, off), qy = __shfl_up(sy, off);
            if (depth >= off) {
                sx += qx;
                sy += qy;
            }
        }
    }
    if (t.flags & kTermOn) {
        sx += cx;
        sy += cy;
    }
    if (t.flags & kTermEmit) put(t, sx, sy);
    if (__ballot(t.flags & kTermOpen)) {
        cx = lane63(sx);
        cy = lane63(sy);
    }
}

template <typename TM, typename F>
__device__ __forceinline__ void fold_terms(const qsft_fold_desc& d, int c, int lo, int hi, int wave, int waves,
                                           TM term, F put) {
    TermShare sh(lo, hi, wave, waves);
    Term t;
    bool more = true;
    double cx = 0.0, cy = 0.0;
    for (int i0 = sh.first; more; i0 += 64) {
        more = sh.load(d, c, i0, t);
        term_add(t, cx, cy, term, put);
    }
}

// Phases of row p of group c.
__device__ __forceinline__ const QSFT_GLOBAL uint8_t* phase_row(const qsft_fold_desc& d, int c, int p) {
    return gptr(d.E) + ((size_t)(d.shared_d ? 0 : c) * d.P + p) * fold_sp(d.S);
}

// Strengths that are not finite stay out of the transforms, whose butterflies
// would meet infinities of both signs and, for q = 4, never the product with a
// zero cosine or sine: k_fold_rank lists them and takes zero, and here their
// terms a w^{<m, k>} are added to the finished samples of row p of group c, the
// elements at(e) for e < E, as the sum over every support has them: an infinity
// of the right sign or a NaN. (Sub-transforms are sums over all samples of a
// row, which then are NaN: fwd descriptors take NaN for such a strength.)
template <typename T, typename G>
__device__ __forceinline__ void add_not_finite(const qsft_fold_desc& d, uint32_t count, int c, int p,
                                               cplx_t<T>* __restrict__ x, int E, G at) {
    const QSFT_GLOBAL uint8_t* ph = phase_row(d, c, p);
    __syncthreads();                                               // the row's samples are written
    for (int e = threadIdx.x; e < E; e += blockDim.x) {
        const int64_t l = at(e);
        cplx_t<T> v = x[l];
        for (uint32_t i = 0; i < count; ++i) {
            const uint32_t s = gptr(d.bad)[1 + i];
            uint32_t r = ph[s], j = gptr(d.J)[(size_t)c * d.S + s], m = (uint32_t)l;
            for (int t = 0; t < d.b; ++t, j /= d.q, m /= d.q) r += (j % d.q) * (m % d.q);
            double sn, cs, ax, ay;
            sincospi(2.0 * (double)(r % d.q) / (double)d.q, &sn, &cs);
            if (d.a_prec == QSFT_F32) {
                ax = reinterpret_cast<const float2*>(d.a)[s].x;
                ay = reinterpret_cast<const float2*>(d.a)[s].y;
            } else {
                ax = reinterpret_cast<const double2*>(d.a)[s].x;
                ay = reinterpret_cast<const double2*>(d.a)[s].y;
            }
            v.x += (T)(ax * cs - ay * sn);
            v.y += (T)(ax * sn + ay * cs);
        }
        x[l] = v;
    }
}

// One pass over the axes [d0, d1) of every row (dft.hip's tile scheme). The
// first pass (FIRST: the innermost axes, so a tile is a contiguous run of
// bins) folds its terms into the tile; later passes read x. Between passes x
// holds the swapped parts; the last pass swaps back.
template <typename T, int QR, bool FIRST, int TH, typename SRC>
__global__ __launch_bounds__(TH) void k_fold_pass(const SRC src, int pass, int lds_bytes) {
    using C2 = cplx_t<T>;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ double2 tab[QSFT_MAX_Q];
    C2* lds = reinterpret_cast<C2*>(smem_raw);
    int local;
    const qsft_fold_desc& d = src.at(blockIdx.x, local);
    if (pass >= d.n_pass) return;
    const int q = (QR > 0) ? QR : d.q;
    const int b = d.b;
    const int d0 = d.pass_d0[pass], d1 = d.pass_d1[pass], ti = d.pass_ti[pass], ta = d.pass_ta[pass];
    const int mb = d1 - d0;
    const int Q = ipow(q, b);
    const int A = ipow(q, d0), M = ipow(q, mb), I = ipow(q, b - d1);
    const bool contiguous = ti == I;
    const int ichunks = I / ti;
    const int tiles_per_row = (A / ta) * ichunks;
    const int row = local / tiles_per_row;
    const int rt = local - row * tiles_per_row;
    const int ac = rt / ichunks;
    const int64_t base = (int64_t)ac * ta * M * I + (rt - ac * ichunks) * ti;
    const int E = ta * M * ti;
    C2* tw = lds + (QR > 0 ? E : 2 * E);
    if ((int)(((QR > 0 ? E : 2 * E) + (QR > 0 ? 0 : q)) * sizeof(C2)) > lds_bytes) return;   // launch sized too small
    const FastDiv fti((uint32_t)ti);
    if constexpr (QR == 0) {
        for (int r = threadIdx.x; r < q; r += blockDim.x) {
            double s, c;
            sincospi(-2.0 * (double)r / (double)q, &s, &c);
            tw[r].x = (T)c;
            tw[r].y = (T)s;
        }
    }
    auto goff = [&](int e) -> int64_t {
        if (contiguous) return base + e;
        const int m = (int)fti.div((uint32_t)e);
        return base + (int64_t)m * I + (e - m * ti);
    };
    C2* __restrict__ x = in_global(reinterpret_cast<C2*>(d.x)) + (int64_t)row * Q;
    if constexpr (FIRST) {
        const int c = row / d.P;
        fold_wtable(tab, q);
        for (int e = threadIdx.x; e < E; e += blockDim.x) lds[e] = C2{(T)0, (T)0};
        __syncthreads();
        int lo = 0, hi = d.S;
        if (d.tiles > 1 && d.S > 0) {
            const QSFT_GLOBAL int32_t* st = gptr(d.start) + (size_t)c * (d.tiles + 1) + ac;
            lo = st[0];
            hi = st[1];
        }
        const QSFT_GLOBAL uint8_t* ph = phase_row(d, c, row - c * d.P);
        fold_terms(d, c, lo, hi, threadIdx.x >> 6, TH / 64,
                   [&](const Term& t, double& sx, double& sy) {
                       const double2 w = tab[ph[t.s]];
                       sx = t.a.x * w.x - t.a.y * w.y;
                       sy = t.a.x * w.y + t.a.y * w.x;
                   },
                   [&](const Term& t, double sx, double sy) { lds[t.j - (uint32_t)base] = C2{(T)sy, (T)sx}; });   // swapped
    } else {
        tile_load(lds, E, [&](int e) { return x[goff(e)]; });
    }
    __syncthreads();
    C2* cur = tile_axes<T, QR>(lds, lds + E, E, q, mb, ti, tw);
    if (d.fwd && pass == d.n_pass - 1) {
        // the tile now holds samples: back along the same axes, the outermost first
        // as over all passes (the order of the axes, and with it the bits, do not
        // follow from how they are grouped), scaled by q^-b as k_dft_pass scales
        // it if these are all (else its last pass does that)
        for (int e = threadIdx.x; e < E; e += blockDim.x) cur[e] = C2{cur[e].y, cur[e].x};
        __syncthreads();
        cur = tile_axes<T, QR>(cur, cur == lds ? lds + E : lds, E, q, mb, ti, tw, true);
        if (FIRST) tile_store(cur, E, [&](int e, C2 v) { x[goff(e)] = dft_scaled<T>(v, Q); });
        else tile_store(cur, E, [&](int e, C2 v) { x[goff(e)] = v; });
    } else if (pass == d.n_pass - 1) {
        tile_store(cur, E, [&](int e, C2 v) { x[goff(e)] = C2{v.y, v.x}; });
        if (const uint32_t bad = d.S > 0 ? cptr(d.bad)[0] : 0)
            add_not_finite<T>(d, bad, row / d.P, row % d.P, x, E, goff);
    } else {
        tile_store(cur, E, [&](int e, C2 v) { x[goff(e)] = v; });
    }
}

// q = 4, whole rows of 4^B samples (k_dft4_rows' register scheme): 4^B / 16
// threads a row, kRows rows at a time, d.rpw times over for the rows of one
// group, so that what the rows share (positions, strengths, run structure) is
// loaded into registers once and the next row's phases arrive while this one
// is transformed: a row alone spent most of its time in three dependent loads
// before its first LDS write. Terms that do not fit the registers, or phases
// their LDS buffer, are read per row.
//
// A thread's 16 samples differ in the two digits of a window. The inverse
// transform runs through the windows 0, 2, 4 (two digits each), an odd B ends
// with the window of its two top digits, of which only the last is left. With
// d.fwd the row's samples are transformed back to its sub-transform before
// they leave the registers (the last window first, which needs no exchange,
// then the others upwards, so that the stores are 128-byte segments), and x
// receives that.
// 64 instances of q = 4, S = 1000, b = 6, P = 102 in FP32: 0.227 ms for the
// samples and 0.268 ms for k_dft4_rows as two launches, 0.23 ms in one (2.8
// TB/s of writes). Bound by its VALU, 70 % busy, between the chain of exchanges
// (LDS 43 %) at four waves per SIMD, all that 34 KiB of LDS a row allow.
typedef float gf2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void store_c2(QSFT_GLOBAL float2* p, float2 v) {
    *reinterpret_cast<QSFT_GLOBAL gf2*>(p) = gf2{v.x, v.y};
}
__device__ __forceinline__ void store_c2(QSFT_GLOBAL double2* p, double2 v) {
    *reinterpret_cast<QSFT_GLOBAL gd2*>(p) = gd2{v.x, v.y};
}

template <int B>
constexpr int fold4_rows() { return B <= 5 ? 4 : 1; }             // rows of 16 (b = 4) or 64 threads at a time
template <int B>
constexpr int fold4_threads() { return fold4_rows<B>() << (2 * B - 4); }
template <int B>
constexpr int fold4_phases() { return B == 6 ? 4096 : B == 7 ? 8192 : 0; }   // phases of one row in LDS
constexpr int kTermBlocks = 4;       // blocks of 64 terms a wave keeps in registers
// window k of the inverse transform: its lower digit
template <int B>
__device__ __forceinline__ constexpr int fold4_window(int k) { return 2 * k < B - 1 ? 2 * k : B - 2; }

template <typename T, int B, bool FWD, typename SRC>
__global__ __launch_bounds__(fold4_threads<B>()) __attribute__((
    amdgpu_waves_per_eu(sizeof(T) == 4 ? 4 : 2))) void k_fold4_rows(const SRC src) {
    using C2 = cplx_t<T>;
    constexpr int Q = 1 << (2 * B), kTpr = Q / 16, kRows = fold4_rows<B>(), kThreads = kRows * kTpr;
    constexpr int kPhases = fold4_phases<B>(), kWindows = (B + 1) / 2;
    static_assert(B >= 4 && B <= 7, "16 samples a thread, at most 1024 threads a row");
    __shared__ __align__(16) C2 lds_all[kRows][Q + Q / 16];
    __shared__ __align__(16) uint8_t phl[kPhases ? kPhases : 16];
    int local;
    const qsft_fold_desc& d = src.at(blockIdx.x, local);
    if (d.q != 4 || d.b != B || (d.fwd != 0) != FWD) return;       // launched for other shapes
    const int P = d.P, Sp = fold_sp(d.S), per = d.rpw * kRows, wpg = (P + per - 1) / per;
    const int c = local / wpg, p0 = (local - c * wpg) * per, p1 = min(P, p0 + per);
    const int sub = threadIdx.x / kTpr, tid = threadIdx.x % kTpr, wave = threadIdx.x >> 6;
    C2* lds = lds_all[sub];
    const bool phases_staged = Sp <= kPhases;
    gu4 ph_next = {0, 0, 0, 0};                                    // the next row's phases, 16 per thread
    auto fetch = [&](int p) {
        if (phases_staged && 16 * (int)threadIdx.x < Sp)
            ph_next = *reinterpret_cast<const QSFT_GLOBAL gu4*>(phase_row(d, c, p) + 16 * threadIdx.x);
    };
    fetch(p0);
    Term kept[kTermBlocks];
    TermShare share(0, d.S, wave, kThreads / 64);
    bool more = true;
#pragma unroll
    for (int i = 0; i < kTermBlocks; ++i) {
        kept[i].flags = 0;
        if (more) more = share.load(d, c, share.first + 64 * i, kept[i]);
    }
    more = more && share.first < share.last && share.first + 64 * kTermBlocks < d.S;   // terms beyond the registers
    for (int p = p0; p < p1; p += kRows) {
        __syncthreads();                                           // the last row's reads are done
        if (phases_staged && 16 * (int)threadIdx.x < Sp) reinterpret_cast<gu4*>(phl)[threadIdx.x] = ph_next;
        for (int e = threadIdx.x; e < (int)(sizeof(lds_all) / 16); e += kThreads)
            reinterpret_cast<gu4*>(lds_all)[e] = gu4{0, 0, 0, 0};
        __syncthreads();
        if (p + kRows < p1) fetch(p + kRows);
#pragma unroll 1
        for (int r = 0; r < kRows; ++r) {                          // the workgroup folds one row after the other
            if (p + r >= p1) break;
            const QSFT_GLOBAL uint8_t* ph = phase_row(d, c, p + r);
            auto term = [&](const Term& t, double& sx, double& sy) {
                // a w^e, w^e in {1, i, -1, -i}: parts exchanged for odd e, signs from e
                const uint32_t e = phases_staged ? phl[t.s] : ph[t.s];
                const bool odd = e & 1;
                sx = odd ? -t.a.y : t.a.x;
                sy = odd ? t.a.x : t.a.y;
                if (e & 2) {
                    sx = -sx;
                    sy = -sy;
                }
            };
            auto put = [&](const Term& t, double sx, double sy) {
                lds_all[r][dft4_pad((int)t.j)] = C2{(T)sy, (T)sx};    // swapped parts
            };
            double cx = 0.0, cy = 0.0;
#pragma unroll
            for (int i = 0; i < kTermBlocks; ++i) {
                Term t = kept[i];
                __asm__ volatile("" : "+v"(t.flags));              // or every step's run masks are kept across rows
                term_add(t, cx, cy, term, put);
            }
            if (more) {
                TermShare rest = share;
                Term t;
                bool go = true;
                for (int i0 = share.first + 64 * kTermBlocks; go; i0 += 64) {
                    go = rest.load(d, c, i0, t);
                    term_add(t, cx, cy, term, put);
                }
            }
        }
        __syncthreads();
        C2 v[16];
        auto exchange = [&](int from, int to) {                     // registers hold window `from`, then `to`
            if (from >= 0) {
                __syncthreads();                                   // the previous reads of lds are done
                C2* w = lds + dft4_lds_base(from, tid);
#pragma unroll
                for (int j = 0; j < 16; ++j) w[j * dft4_lds_step(from)] = v[j];
                __syncthreads();
            }
            const C2* r = lds + dft4_lds_base(to, tid);
#pragma unroll
            for (int j = 0; j < 16; ++j) v[j] = r[j * dft4_lds_step(to)];
        };
        // the transforms along the digits of the window that are its own
        auto digits = [&](int w) {
            if (w % 2 == 0) {
#pragma unroll
                for (int a = 0; a < 4; ++a) dft4_reg<T>(v[4 * a], v[4 * a + 1], v[4 * a + 2], v[4 * a + 3]);
            }
#pragma unroll
            for (int a = 0; a < 4; ++a) dft4_reg<T>(v[a], v[a + 4], v[a + 8], v[a + 12]);
        };
#pragma unroll
        for (int k = 0; k < kWindows; ++k) {
            exchange(k ? fold4_window<B>(k - 1) : -1, fold4_window<B>(k));
            digits(fold4_window<B>(k));
        }
        int row = c * P + p;
        __asm__ volatile("" : "+s"(row));                          // not an induction variable per store address
        QSFT_GLOBAL C2* x = gptr(reinterpret_cast<C2*>(d.x)) + (int64_t)row * Q;
        const bool live = p + sub < p1;
        const uint32_t xo = (uint32_t)sub * Q;
        if constexpr (FWD) {
#pragma unroll
            for (int j = 0; j < 16; ++j) v[j] = C2{v[j].y, v[j].x};   // the samples
            digits(B - 2);                                         // the last window, still in registers
#pragma unroll
            for (int k = 0; k < kWindows - 1; ++k) {
                exchange(k ? fold4_window<B>(k - 1) : B - 2, fold4_window<B>(k));
                digits(fold4_window<B>(k));
            }
            if (live) {
                constexpr int w = fold4_window<B>(kWindows - 2);
#pragma unroll
                for (int j = 0; j < 16; ++j)
                    store_c2(x + (xo + dft4_index(w, tid, 0) + (j << (2 * w))), dft_scaled<T>(v[j], Q));
            }
        } else if (live) {
#pragma unroll
            for (int j = 0; j < 16; ++j) store_c2(x + (xo + tid + j * kTpr), C2{v[j].y, v[j].x});   // (window B - 2)
        }
    }
    if constexpr (!FWD) {
        if (const uint32_t bad = d.S > 0 ? cptr(d.bad)[0] : 0) {
            for (int p = p0; p < p1; ++p)
                add_not_finite<T>(d, bad, c, p, in_global(reinterpret_cast<C2*>(d.x)) + ((int64_t)c * P + p) * Q, Q,
                                  [](int e) { return (int64_t)e; });
        }
    }
}

}  // namespace qsft

using namespace qsft;

extern "C" void qsft_set_error(const char* msg);
extern "C" int qsft_hip_status(hipError_t e, const char* where);

namespace {

size_t al256(size_t x) { return (x + 255) & ~(size_t)255; }

// rows that k_fold4_rows takes: q = 4, b = 4..6, and in FP32 b = 7 (144 KiB of LDS)
bool fold_rows4(int q, int b, int precision) { return q == 4 && b >= 4 && b <= (precision == QSFT_F32 ? 7 : 6); }

// Whether the whole-row kernel takes an instance of such rows. Its workgroups of
// b = 4 and 5 fold their four rows one after the other with one wave and with
// four, which pays only while the terms are few: the tile kernel (a workgroup
// a row) takes more. The line depends on the instance alone, so that a request
// has the same bits in every batch. Rows of 64 instances of C = 3, P = 62,
// FP32, as sub-transforms, whole-row / tile kernel: b = 4, S = 200 49 / 68 us,
// S = 400 99 / 75, S = 5000 1820 / 307; b = 5, S = 1000 91 / 124, S = 2000
// 189 / 167, S = 5000 531 / 304; one such instance, S = 5000: 331 / 30 and 90 / 28.
bool fold_rows4_takes(int q, int b, int S, int precision) {
    return fold_rows4(q, b, precision) && S <= (b == 4 ? 256 : b == 5 ? 1600 : 0x7FFFFFFF);
}

bool fold_shape_ok(int q, int n, int b, int C, int P, int S, int n_pad) {
    if (q < 2 || q > QSFT_MAX_Q || b < 1 || b > QSFT_MAX_B || n < 1 || n > n_pad || n_pad % 64 || n_pad > QSFT_MAX_N ||
        C < 1 || P < 1 || S < 0)
        return false;
    long long Q = 1;
    for (int i = 0; i < b; ++i) {
        Q *= q;
        if (Q > 0x7FFFFFFF) return false;                          // 32-bit bins
    }
    return (long long)C * P <= 0x7FFFFFFF && (long long)S + Q + 4 * kRankThreads <= 0x7FFFFFFF;
}

}  // namespace

// Phases (groups x P x 16-padded S bytes), sorted strengths and keys, bins (C x S), the
// strengths that are not finite (a count and at most S), tile starts (a first-pass tile
// holds at least q bins), sorted bins of chunks and ranks in them (C x S each).
extern "C" size_t qsft_fold_workspace_bytes(int q, int b, int C, int P, int S, int shared_d) {
    if (!fold_shape_ok(q, 1, b, C, P, S, 64)) return 0;
    return al256((size_t)(shared_d ? 1 : C) * P * fold_sp(S)) + al256((size_t)C * S * 16) +
           al256((size_t)C * S * 8) + al256((size_t)C * S * 4) + al256(((size_t)S + 1) * 4) +
           al256((size_t)C * (ipow(q, b) / std::min(q, 32) + 2) * 4) + (fold_chunks(S) ? al256((size_t)C * S * 8) : 0);
}

extern "C" int qsft_fold_whole_rows(int q, int b, int precision) {
    if (!fold_shape_ok(q, 1, b, 1, 1, 0, 64) || (precision != QSFT_F32 && precision != QSFT_F64)) return 0;
    const long long elem = precision == QSFT_F32 ? 8 : 16, Q = ipow(q, b);
    return fold_rows4(q, b, precision) || (radix_compiled(q) ? Q * elem : (2 * Q + q) * elem) <= kRowLdsBytes;
}

extern "C" int qsft_fold_bind(qsft_fold_desc* h, int q, int n, int b, int C, int P, int S, int n_pad, int shared_d,
                              int precision, int a_precision, int transform, int launch_rows, const int8_t* Mt,
                              const int8_t* D, const int8_t* K, const void* a, void* x, void* ws, size_t ws_bytes) {
    if (!h || !fold_shape_ok(q, n, b, C, P, S, n_pad) || (shared_d != 0 && shared_d != 1) ||
        (precision != QSFT_F32 && precision != QSFT_F64) || (a_precision != QSFT_F32 && a_precision != QSFT_F64) ||
        (((uintptr_t)Mt | (uintptr_t)D | (uintptr_t)K | (uintptr_t)a) & 15) || ((uintptr_t)ws & 255)) {
        qsft_set_error("qsft_fold_bind: bad shape or alignment (Mt, D, K, a 16-byte, workspace 256-byte aligned)");
        return QSFT_ERR_ARG;
    }
    if (!ws || ws_bytes < qsft_fold_workspace_bytes(q, b, C, P, S, shared_d)) {
        qsft_set_error("qsft_fold_bind: workspace too small");
        return QSFT_ERR_ARG;
    }
    qsft_fold_desc d{};
    d.q = q; d.n = n; d.b = b; d.C = C; d.P = P; d.S = S; d.n_pad = n_pad;
    d.shared_d = shared_d; d.a_prec = a_precision;
    d.Mt = Mt; d.D = D; d.K = K; d.a = a; d.x = x;
    char* w = static_cast<char*>(ws);
    d.E = reinterpret_cast<uint8_t*>(w);
    w += al256((size_t)(shared_d ? 1 : C) * P * fold_sp(S));
    d.as = reinterpret_cast<double*>(w);
    w += al256((size_t)C * S * 16);
    d.key = reinterpret_cast<uint64_t*>(w);
    w += al256((size_t)C * S * 8);
    d.J = reinterpret_cast<uint32_t*>(w);
    w += al256((size_t)C * S * 4);
    d.bad = reinterpret_cast<uint32_t*>(w);
    w += al256(((size_t)S + 1) * 4);
    d.start = reinterpret_cast<int32_t*>(w);
    w += al256((size_t)C * (ipow(q, b) / std::min(q, 32) + 2) * 4);
    if ((transform & QSFT_FOLD_CHUNKS) && fold_chunks(S)) d.chunk = reinterpret_cast<uint32_t*>(w);
    const int Q = ipow(q, b);
    if (fold_rows4_takes(q, b, S, precision)) {
        // rows of a group per workgroup: one where the launch has fewer rows than
        // the chip holds (256 CUs x 4 workgroups), up to four where it has many
        d.rpw = launch_rows >= 8192 ? 4 : launch_rows >= 4096 ? 2 : 1;
        const int per = d.rpw * (b <= 5 ? fold4_rows<4>() : fold4_rows<6>());
        d.n_pass = 1;
        d.pass_d1[0] = b;
        d.pass_ti[0] = 1;
        d.pass_ta[0] = 1;
        d.pass_blocks[0] = C * ((P + per - 1) / per);
        d.pass_lds[0] = 16;
        d.tiles = 1;
        d.tile_bins = Q;
    } else {
        // whole rows where they fit the LDS, else the sub-DFT planner's schedule,
        // measured or modelled, innermost first. A measured forward transform says
        // nothing about whole rows here: one pass writes a row once, where two
        // write it, read it and write it again, and two more follow for a
        // sub-transform.
        qsft_dft_desc s{};
        s.q = q; s.b = b; s.rows = C * P; s.in_stride = 1; s.in_row_stride = Q;
        if (qsft_fold_whole_rows(q, b, precision)) {
            s.n_pass = 1;
            s.pass_d1[0] = b;
            s.pass_ti[0] = s.pass_ta[0] = 1;
            s.pass_blocks[0] = C * P;
        } else {
            const int rc = qsft_dft_plan(&s, precision);
            if (rc != QSFT_OK) return rc;
        }
        d.n_pass = s.n_pass;
        for (int p = 0; p < s.n_pass; ++p) {
            d.pass_d0[p] = s.pass_d0[p];
            d.pass_d1[p] = s.pass_d1[p];
            d.pass_ti[p] = s.pass_ti[p];
            d.pass_ta[p] = s.pass_ta[p];
            d.pass_blocks[p] = s.pass_blocks[p];
            d.pass_lds[p] = qsft_dft_lds_bytes(&s, p, precision);
            if (d.pass_lds[p] < 0) {
                qsft_set_error("qsft_fold_bind: tile does not fit the LDS");
                return QSFT_ERR_ARG;
            }
        }
        d.tile_bins = ipow(q, b - s.pass_d0[0]) * s.pass_ta[0];   // whole innermost axes: contiguous bins
        d.tiles = Q / d.tile_bins;
    }
    d.fwd = (transform & ~QSFT_FOLD_CHUNKS) != 0;
    *h = d;
    return QSFT_OK;
}

// The forward passes a fwd descriptor's launches leave: those over the axes of
// every pass but the last, in place on x and from the outermost group inwards
// (n_pass 0: none).
extern "C" int qsft_fold_rest(const qsft_fold_desc* h, qsft_dft_desc* out) {
    if (!h || !out || !h->fwd || h->n_pass < 1) {
        qsft_set_error("qsft_fold_rest: a descriptor bound with transform is needed");
        return QSFT_ERR_ARG;
    }
    qsft_dft_desc r{};
    r.q = h->q;
    r.b = h->b;
    r.rows = h->C * h->P;
    r.in_stride = 1;
    r.in_row_stride = ipow(h->q, h->b);
    r.in = h->x;
    r.out = h->x;
    r.n_pass = h->n_pass - 1;
    r.order = 1;
    for (int p = 0; p < r.n_pass; ++p) {
        const int f = r.n_pass - 1 - p;
        r.pass_d0[p] = h->pass_d0[f];
        r.pass_d1[p] = h->pass_d1[f];
        r.pass_ti[p] = h->pass_ti[f];
        r.pass_ta[p] = h->pass_ta[f];
        r.pass_blocks[p] = h->pass_blocks[f];
    }
    *out = r;
    return QSFT_OK;
}

extern "C" int qsft_fold_blocks(const qsft_fold_desc* h, int* phase_blocks, int* rank_blocks) {
    if (!h || !phase_blocks || !rank_blocks || !fold_shape_ok(h->q, h->n, h->b, h->C, h->P, h->S, h->n_pad) ||
        h->tiles < 1)
        return -1;
    const long long tiles = (long long)(h->shared_d ? 1 : h->C) * ((h->P + 15) / 16) + h->C;
    const long long ph = ((h->S + 63) / 64) * ((tiles + kPhaseTiles - 1) / kPhaseTiles);
    const long long S64 = (h->S + 63) / 64 * 64;
    const long long rk = h->S == 0 ? 0 : h->C * ((S64 + fold_bounds(h->tiles) + 63) / 64);
    if (ph > 0x7FFFFFFF || rk > 0x7FFFFFFF) return -1;
    *phase_blocks = (int)ph;
    *rank_blocks = (int)rk;
    return 0;
}

namespace {

using FoldBatch = DescBatch<qsft_fold_desc>;
using FoldOne = DescOne<qsft_fold_desc>;

template <typename SRC>
int launch_chunks(const SRC& src, int rank_blocks, hipStream_t st) {
    if (rank_blocks > 0) hipLaunchKernelGGL(k_fold_chunk<SRC>, dim3(rank_blocks), dim3(kRankThreads), 0, st, src);
    return qsft_hip_status(hipGetLastError(), "qsft_fold(chunks)");
}

template <typename SRC>
int launch_prep(const SRC& src, int phase_blocks, int rank_blocks, hipStream_t st) {
    if (phase_blocks > 0) {
        hipLaunchKernelGGL(k_fold_phase<SRC>, dim3(phase_blocks), dim3(kPhaseThreads), 0, st, src);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return qsft_hip_status(e, "qsft_fold(phases)");
    }
    if (rank_blocks > 0) {
        hipLaunchKernelGGL(k_fold_rank<SRC>, dim3(rank_blocks), dim3(kRankThreads), 0, st, src);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return qsft_hip_status(e, "qsft_fold(ranks)");
    }
    return QSFT_OK;
}

template <typename T, int QR, typename SRC>
void launch_pass(const SRC& src, int blocks, int pass, int lds, hipStream_t st) {
    const dim3 g(blocks), th(kDftThreads), mid(kDftMidThreads), big(row_threads<T>());
    const size_t sh = (size_t)lds;
    if (lds > kDftLdsBytes)                                        // whole rows: the first pass is the only one
        hipLaunchKernelGGL((k_fold_pass<T, QR, true, row_threads<T>(), SRC>), g, big, sh, st, src, pass, lds);
    else if (pass == 0 && lds > kDftMidBytes)
        hipLaunchKernelGGL((k_fold_pass<T, QR, true, kDftMidThreads, SRC>), g, mid, sh, st, src, pass, lds);
    else if (pass == 0)
        hipLaunchKernelGGL((k_fold_pass<T, QR, true, kDftThreads, SRC>), g, th, sh, st, src, pass, lds);
    else
        hipLaunchKernelGGL((k_fold_pass<T, QR, false, kDftThreads, SRC>), g, th, sh, st, src, pass, lds);
}

template <typename T, int B, typename SRC>
void launch_rows4(bool fwd, const SRC& src, int blocks, hipStream_t st) {
    if (fwd) hipLaunchKernelGGL((k_fold4_rows<T, B, true, SRC>), dim3(blocks), dim3(fold4_threads<B>()), 0, st, src);
    else hipLaunchKernelGGL((k_fold4_rows<T, B, false, SRC>), dim3(blocks), dim3(fold4_threads<B>()), 0, st, src);
}

template <typename T, typename SRC>
int launch_rows(int q, int b, bool fwd, const SRC& src, int blocks, int pass, int lds, hipStream_t st) {
    if (blocks == 0) return QSFT_OK;
    if (fold_rows4(q, b, sizeof(T) == 4 ? QSFT_F32 : QSFT_F64)) {
        switch (b) {
            case 4: launch_rows4<T, 4>(fwd, src, blocks, st); break;
            case 5: launch_rows4<T, 5>(fwd, src, blocks, st); break;
            case 6: launch_rows4<T, 6>(fwd, src, blocks, st); break;
            default:
                if constexpr (sizeof(T) == 4) launch_rows4<T, 7>(fwd, src, blocks, st);
        }
    } else {
        switch (q) {
            case 2: launch_pass<T, 2>(src, blocks, pass, lds, st); break;
            case 3: launch_pass<T, 3>(src, blocks, pass, lds, st); break;
            case 4: launch_pass<T, 4>(src, blocks, pass, lds, st); break;
            case 5: launch_pass<T, 5>(src, blocks, pass, lds, st); break;
            case 20: launch_pass<T, 20>(src, blocks, pass, lds, st); break;
            default: launch_pass<T, 0>(src, blocks, pass, lds, st); break;
        }
    }
    return qsft_hip_status(hipGetLastError(), "qsft_fold(rows)");
}

}  // namespace

extern "C" int qsft_fold_chunks(const qsft_fold_desc* d, const int32_t* pre_rank, int n_inst, int rank_blocks,
                                void* stream) {
    if (!d || !pre_rank || n_inst < 1 || rank_blocks < 0) {
        qsft_set_error("qsft_fold_chunks: bad arguments");
        return QSFT_ERR_ARG;
    }
    return launch_chunks(FoldBatch{d, pre_rank, n_inst}, rank_blocks, (hipStream_t)stream);
}

extern "C" int qsft_fold_prep(const qsft_fold_desc* d, const int32_t* pre_phase, const int32_t* pre_rank, int n_inst,
                              int phase_blocks, int rank_blocks, void* stream) {
    if (!d || !pre_phase || !pre_rank || n_inst < 1 || phase_blocks < 0 || rank_blocks < 0) {
        qsft_set_error("qsft_fold_prep: bad arguments");
        return QSFT_ERR_ARG;
    }
    const int rc = launch_prep(FoldBatch{d, pre_phase, n_inst}, phase_blocks, 0, (hipStream_t)stream);
    return rc != QSFT_OK ? rc : launch_prep(FoldBatch{d, pre_rank, n_inst}, 0, rank_blocks, (hipStream_t)stream);
}

extern "C" int qsft_fold_rows(const qsft_fold_desc* d, const int32_t* pre, int n_inst, int blocks, int pass, int word,
                              int lds_bytes, void* stream) {
    const int prec = word & 0xF, q = (word >> 8) & 0xFF, b = (word >> 16) & 0xFF;
    const bool fwd = (word >> 24) & 1;
    if (!d || !pre || n_inst < 1 || blocks < 0 || pass < 0 || pass >= QSFT_DFT_MAX_PASSES || lds_bytes < 16 ||
        lds_bytes > kRowLdsBytes || (lds_bytes > kDftLdsBytes && pass != 0) || (prec != QSFT_F32 && prec != QSFT_F64) || q < 2 || q > QSFT_MAX_Q ||
        (fold_rows4(q, b, prec) && pass != 0)) {
        qsft_set_error("qsft_fold_rows: bad arguments");
        return QSFT_ERR_ARG;
    }
    const FoldBatch src{d, pre, n_inst};
    return prec == QSFT_F32 ? launch_rows<float>(q, b, fwd, src, blocks, pass, lds_bytes, (hipStream_t)stream)
                            : launch_rows<double>(q, b, fwd, src, blocks, pass, lds_bytes, (hipStream_t)stream);
}

extern "C" int qsft_fold_one(int q, int n, int b, int C, int P, int S, int n_pad, int shared_d, int precision,
                             int a_precision, const int8_t* Mt, const int8_t* D, const int8_t* K, const void* a,
                             void* x, void* ws, size_t ws_bytes, void* stream) {
    FoldOne src;
    int rc = qsft_fold_bind(&src.d, q, n, b, C, P, S, n_pad, shared_d, precision, a_precision, QSFT_FOLD_CHUNKS, C * P,
                            Mt, D, K, a, x, ws, ws_bytes);
    if (rc != QSFT_OK) return rc;
    int pb = 0, rb = 0;
    if (qsft_fold_blocks(&src.d, &pb, &rb) != 0) {
        qsft_set_error("qsft_fold_one: launch too large");
        return QSFT_ERR_ARG;
    }
    hipStream_t st = (hipStream_t)stream;
    const int rows4 = src.d.rpw ? b : 0;
    rc = launch_prep(src, pb, 0, st);
    if (rc == QSFT_OK && src.d.chunk) rc = launch_chunks(src, rb, st);
    if (rc == QSFT_OK) rc = launch_prep(src, 0, rb, st);
    for (int p = 0; rc == QSFT_OK && p < src.d.n_pass; ++p)
        rc = precision == QSFT_F32 ? launch_rows<float>(q, rows4, src.d.fwd, src, src.d.pass_blocks[p], p, src.d.pass_lds[p], st)
                                   : launch_rows<double>(q, rows4, src.d.fwd, src, src.d.pass_blocks[p], p, src.d.pass_lds[p], st);
    return rc;
}
