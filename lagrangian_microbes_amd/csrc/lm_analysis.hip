// On-device reductions for long runs: the species count of every recorded
// step (analysis.py:31-35 counts species == ROCK / PAPER / SCISSORS per
// time) and the histogram of all pairwise great-circle distances
// (sandbox/pairwise_distance_histogram_gpu.jl:14-43,
// sandbox/pairwise_distance_histogram_distributed.jl:49-55).
//
// Distance histogram: for every unordered pair i < j, the haversine term
//   a = sin^2(dlat / 2) + cos(lat_i) cos(lat_j) sin^2(dlon / 2)
// (degrees, float32 positions widened to double; sin and cos of degree
// arguments as the fma-Horner polynomials every liblm unit shares, so the
// oracle reproduces a bit for bit) is binned against increasing thresholds:
// bin = number of thresholds <= a.  The caller derives the thresholds from
// distance edges (d = 2 R asin(sqrt(a))), so the bins are distance bins and
// the counts are exact integers.
//
// A float32 value of a decides nearly every pair: its error is bounded (see
// kHistTol), so a pair farther than that from every threshold lands in the
// bin the float64 value lands in, and only the others (about 2 in 100,000 at
// ten bins per decade) evaluate the float64 term.
#include "lm_common.h"

#include <cfloat>
#include <cmath>

namespace lm {

constexpr int kHistTile = 256;
constexpr int kHistMaxBins = 256;

// Bytes of one row per workgroup: 8 vectors of 16 bytes per lane, all in
// flight.  Reading a byte per lane and load moved 326 GB/s (1082 us for 720
// rows of 490,000); 16 bytes per load move 5.6 TB/s (63 us), HBM's rate.  Rows
// of up to 4 KB take one vector per lane: 10,000 rows of 100 bytes 28 us, 41
// through the eight.
constexpr int kCountVecs = 8;
constexpr int64_t kCountBytes = 16ll * kCountVecs * kBlock;

// Adds the bytes equal to 1, 2, 3 of a word to c[0..2].  Codes 0..3 take two
// bits: popcounts of their combinations; a word with any other code is
// counted byte by byte.
__device__ __forceinline__ void count_word(uint32_t w, uint32_t (&c)[3]) {
    if ((w & 0xfcfcfcfcu) == 0u) {
        const uint32_t lo = w & 0x01010101u, hi = (w >> 1) & 0x01010101u;
        c[0] += __popc(lo & ~hi);
        c[1] += __popc(hi & ~lo);
        c[2] += __popc(lo & hi);
    } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t v = (w >> (8 * q)) & 0xffu;
            c[0] += v == 1u;
            c[1] += v == 2u;
            c[2] += v == 3u;
        }
    }
}

__device__ __forceinline__ void count_vec(const uint4& q, uint32_t (&c)[3]) {
    count_word(q.x, c);
    count_word(q.y, c);
    count_word(q.z, c);
    count_word(q.w, c);
}

// Rows may start at any byte: the aligned 16-byte vectors in between are
// shared out over blockIdx.x, and the row's first block takes the bytes
// before and after them.
__global__ void __launch_bounds__(kBlock)
species_count_kernel(const int8_t* __restrict__ rec, int64_t n, int64_t stride,
                     unsigned long long* __restrict__ counts) {
    __shared__ uint32_t part[kBlock / 64][4];
    const int64_t s = blockIdx.y;
    const int8_t* row = rec + s * stride;
    const int64_t head0 = (int64_t)((16u - (unsigned)((uintptr_t)row & 15u)) & 15u);
    const int64_t head = head0 < n ? head0 : n;
    const int64_t nv = (n - head) / 16;
    const uint4* vec = reinterpret_cast<const uint4*>(row + head);
    uint32_t c[3] = {0, 0, 0}, seen = 0;
    for (int64_t v0 = (int64_t)blockIdx.x * kCountVecs * kBlock; v0 < nv; v0 += (int64_t)gridDim.x * kCountVecs * kBlock) {
        if (nv - v0 <= kBlock) {  // uniform: the rest is a vector per lane
            if (v0 + threadIdx.x < nv) {
                count_vec(vec[v0 + threadIdx.x], c);
                seen += 16;
            }
            break;
        }
        uint4 q[kCountVecs];
#pragma unroll
        for (int k = 0; k < kCountVecs; ++k) {
            const int64_t v = v0 + k * kBlock + threadIdx.x;
            q[k] = make_uint4(0u, 0u, 0u, 0u);
            if (v < nv) {
                q[k] = vec[v];
                seen += 16;
            }
        }
#pragma unroll
        for (int k = 0; k < kCountVecs; ++k) count_vec(q[k], c);
    }
    if (blockIdx.x == 0) {
        const int64_t t = threadIdx.x, tail = n - head - 16 * nv;  // head, tail < 16
        int64_t at = -1;
        if (t < head) at = t;
        else if (t >= 16 && t - 16 < tail) at = head + 16 * nv + (t - 16);
        if (at >= 0) {
            const int v = row[at];
            c[0] += v == 1;
            c[1] += v == 2;
            c[2] += v == 3;
            seen += 1;
        }
    }
    uint32_t all[4] = {seen - c[0] - c[1] - c[2], c[0], c[1], c[2]};
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        uint32_t x = all[k];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) x += __shfl_down(x, off, 64);
        if (lane == 0) part[wave][k] = x;
    }
    __syncthreads();
    if (threadIdx.x < 4) {
        uint32_t t = 0;
        for (int w = 0; w < kBlock / 64; ++w) t += part[w][threadIdx.x];
        if (t) atomicAdd(counts + s * 4 + threadIdx.x, (unsigned long long)t);
    }
}

// ---------------------------------------------------------------------------
// distance histogram
// ---------------------------------------------------------------------------
// The float32 term, for |dlon|, |dlat| <= 30 (WIDE: 180) degrees and
// latitudes in [-90, 90]: sin^2(d / 2) = z (1 - z / 3 + 2 z^2 / 45 - ...) in
// z = (d / 2)^2 rad^2, so both summands are products without cancellation.
// With u = 2^-24: the difference of two float32 positions is within u
// (relative), z within 3 u, the narrow polynomial within 2.2 u (its later
// terms are below 0.023 of the first; truncation 3e-9), cos cos within 3 u,
// the sum within 11 u.  The wide polynomial's terms cancel to 0.4 of 2.1 at 90
// degrees: within 30 u in all.  kHistTol (67 u) covers both.
constexpr float kHistTol = 4e-6f;
constexpr float kHistNarrow = 30.0f, kHistWide = 180.0f;

constexpr double half_deg_rad2() { return 0.25 * LM_DEG2RAD * LM_DEG2RAD; }

// Coefficient m (from 1) of sin^2 x = sum_m c_m x^(2m): (-1)^(m+1) 2^(2m-1) / (2m)!.
constexpr double sin2_coef(int m) {
    double c = 1.0;  // m = 1: 2 / 2!
    for (int k = 2; k <= m; ++k) c *= -4.0 / ((2.0 * k) * (2.0 * k - 1.0));
    return c;
}

template <bool WIDE>
__device__ __forceinline__ float sin2_half(float d) {
    if constexpr (WIDE) {
        const float t = d * (float)(0.5 * LM_DEG2RAD);
        const float z = t * t;
        float p = (float)sin2_coef(12);
#pragma unroll
        for (int m = 11; m >= 1; --m) p = fmaf(p, z, (float)sin2_coef(m));
        return z * p;
    } else {
        // in degrees: the scale is in the coefficients
        constexpr double r = half_deg_rad2();
        const float z = d * d;
        float p = (float)(sin2_coef(4) * r * r * r * r);
        p = fmaf(p, z, (float)(sin2_coef(3) * r * r * r));
        p = fmaf(p, z, (float)(sin2_coef(2) * r * r));
        p = fmaf(p, z, (float)(sin2_coef(1) * r));
        return z * p;
    }
}

// Table over the float32 values of a in [2^-60, 2): cells of 1/16 octave,
// found from the value's top bits.  A cell holds the number of thresholds
// below it (less the tolerance) and the one threshold that may lie in it
// (FLT_MAX: none); more than one, and values outside the table, have a NaN
// threshold, on which no comparison decides.
constexpr int kLutShift = 19;
constexpr uint32_t kLutBase = (127u - 60u) << (23 - kLutShift);
constexpr uint32_t kLutCells = 61u << (23 - kLutShift);

// Number of increasing edges e[0 .. m) with e * scale <= v.
__device__ __forceinline__ int edges_below(const double* e, int m, double scale, double v) {
    int lo = 0, hi = m;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (e[mid] * scale <= v) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// A pair's bin from its float64 term.
__device__ __forceinline__ int exact_bin(const double* e, int m, float xi, float yi, float xj, float yj) {
    const double s1 = sin_deg(0.5 * ((double)yj - (double)yi));
    const double s2 = sin_deg(0.5 * ((double)xj - (double)xi));
    const double a = s1 * s1 + (cos_deg((double)yi) * cos_deg((double)yj)) * (s2 * s2);
    return edges_below(e, m, 1.0, a);
}

// A workgroup takes a tile of 512 points i (two per lane) against `per`
// tiles of 256 points j (staged in LDS, read by all lanes at once), from the
// diagonal on.  Counters: a column per lane, [bin][lane], shared by the
// wavefronts: neighbouring lanes' pairs mostly share a bin, and adds to one
// counter would go one after the other (the first version, one counter per
// wavefront and bin, and FP64 sines and a binary search for every pair, took
// 16.2 ms for 98,587 points; this one takes 3.2 ms, bound by VALU issue, ~30
// instructions per pair).
constexpr int kHistI = 2;

struct HistShared {
    float4 pj[kHistTile];             // x, y, cos(lat)
    double cj[kHistTile];             // cos(lat)
    float2 lut[kLutCells + 1];        // threshold, bin below it
    double edges[kHistMaxBins];
    float box[4][kHistTile / 64];
    uint32_t turn;                    // (float bits) below every threshold that is less than the one before it
};

template <bool WIDE>
__device__ __forceinline__ void hist_tile(const HistShared& S, uint32_t* __restrict__ h, int jend, const float (&xi)[kHistI],
                                          const float (&yi)[kHistI], const float (&ci)[kHistI],
                                          const int (&after)[kHistI], int nedges, uint32_t cols, uint32_t col) {
    for (int k0 = 0; k0 < jend; k0 += 32) {
        const int m = min(32, jend - k0);
        uint32_t amb[kHistI] = {};  // pairs the float32 term does not decide
#pragma unroll 4
        for (int kk = 0; kk < m; ++kk) {
            const float4 p = S.pj[k0 + kk];
#pragma unroll
            for (int u = 0; u < kHistI; ++u) {
                const float a = fmaf(ci[u] * p.z, sin2_half<WIDE>(p.x - xi[u]), sin2_half<WIDE>(p.y - yi[u]));
                // out of the table (0, tiny, above 2, negative, NaN): the last entry
                const uint32_t cell = min((__float_as_uint(a) >> kLutShift) - kLutBase, kLutCells);
                const float2 e = S.lut[cell];
                const bool above = a > e.x * (1.0f + kHistTol), below = a < e.x * (1.0f - kHistTol);
                const bool ok = k0 + kk > after[u], clear = above | below;
                const uint32_t bin = __float_as_uint(e.y) + (above ? 1u : 0u);
                atomicAdd(&h[bin * cols + col], (ok & clear) ? 1u : 0u);
                amb[u] |= ((ok & !clear) ? 1u : 0u) << kk;
            }
        }
#pragma unroll
        for (int u = 0; u < kHistI; ++u)
            while (amb[u]) {
                const float4 p = S.pj[k0 + __ffs(amb[u]) - 1];
                amb[u] &= amb[u] - 1u;
                atomicAdd(&h[(uint32_t)exact_bin(S.edges, nedges, xi[u], yi[u], p.x, p.y) * cols + col], 1u);
            }
    }
}

// A tile that the float32 term does not cover (points more than kHistWide
// apart, past the poles, or not finite): the float64 term of every pair, whose
// bin the table gives too, but for terms within the tolerance of a threshold
// (the term's rounding to float32 is far less).  20,000 points over the globe
// take 470 us; 996 with the cosines taken per pair and a binary search for
// each, 854 with the search alone.
__device__ __forceinline__ void hist_tile_f64(const HistShared& S, uint32_t* __restrict__ h, int jend,
                                              const float (&xi)[kHistI], const float (&yi)[kHistI],
                                              const int (&after)[kHistI], int nedges, uint32_t cols, uint32_t col) {
    double ci[kHistI];
#pragma unroll
    for (int u = 0; u < kHistI; ++u) ci[u] = cos_deg((double)yi[u]);
    for (int k = 0; k < jend; ++k) {
        const float4 p = S.pj[k];
        const double cj = S.cj[k];
#pragma unroll
        for (int u = 0; u < kHistI; ++u) {
            const double s1 = sin_deg(0.5 * ((double)p.y - (double)yi[u]));
            const double s2 = sin_deg(0.5 * ((double)p.x - (double)xi[u]));
            const double a = s1 * s1 + (ci[u] * cj) * (s2 * s2);
            const float af = (float)a;
            const uint32_t cell = min((__float_as_uint(af) >> kLutShift) - kLutBase, kLutCells);
            const float2 e = S.lut[cell];
            const bool above = af > e.x * (1.0f + kHistTol), below = af < e.x * (1.0f - kHistTol);
            uint32_t bin = __float_as_uint(e.y) + (above ? 1u : 0u);
            if (!(above | below)) bin = a == a ? (uint32_t)edges_below(S.edges, nedges, 1.0, a) : 0u;
            if (k > after[u]) atomicAdd(&h[bin * cols + col], 1u);
        }
    }
}

__global__ void __launch_bounds__(kHistTile)
dist_hist_kernel(int64_t n, const float* __restrict__ lon, const float* __restrict__ lat, int nbins,
                 const double* __restrict__ edges, unsigned long long* __restrict__ hist, int per, uint32_t cols) {
    extern __shared__ uint32_t h[];  // [nbins][cols]
    __shared__ HistShared S;
    const int64_t i0 = (int64_t)blockIdx.x * (kHistTile * kHistI);
    const int64_t jt0 = (int64_t)blockIdx.x * kHistI + (int64_t)blockIdx.y * per;  // first j tile
    if (jt0 * kHistTile >= n) return;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const uint32_t col = (uint32_t)lane & (cols - 1u);
    const int nedges = nbins - 1;
    for (uint32_t b = t; b < (uint32_t)nbins * cols; b += kHistTile) h[b] = 0u;
    for (int b = t; b < nedges; b += kHistTile) S.edges[b] = edges[b];
    float xi[kHistI], yi[kHistI], ci[kHistI];
    // extents of the i tile; a position that is not finite, or a latitude
    // past the poles, leaves it unbounded and so every pair to the float64 term
    float lo_x = INFINITY, hi_x = -INFINITY, lo_y = INFINITY, hi_y = -INFINITY;
#pragma unroll
    for (int u = 0; u < kHistI; ++u) {
        const int64_t i = i0 + u * kHistTile + t;
        const bool in = i < n;
        xi[u] = in ? lon[i] : 0.0f;
        yi[u] = in ? lat[i] : 0.0f;
        ci[u] = (float)cos_deg((double)yi[u]);
        if (in) {
            const bool fine = fabsf(xi[u]) < 1e6f && fabsf(yi[u]) <= 90.0f;
            lo_x = fine ? fminf(lo_x, xi[u]) : -INFINITY;
            hi_x = fine ? fmaxf(hi_x, xi[u]) : INFINITY;
            lo_y = fine ? fminf(lo_y, yi[u]) : -INFINITY;
            hi_y = fine ? fmaxf(hi_y, yi[u]) : INFINITY;
        }
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        lo_x = fminf(lo_x, __shfl_xor(lo_x, d, 64));
        hi_x = fmaxf(hi_x, __shfl_xor(hi_x, d, 64));
        lo_y = fminf(lo_y, __shfl_xor(lo_y, d, 64));
        hi_y = fmaxf(hi_y, __shfl_xor(hi_y, d, 64));
    }
    if (t == 0) S.turn = __float_as_uint(FLT_MAX);
    if (lane == 0) {
        S.box[0][wave] = lo_x;
        S.box[1][wave] = hi_x;
        S.box[2][wave] = lo_y;
        S.box[3][wave] = hi_y;
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kHistTile / 64; ++w) {
        lo_x = fminf(lo_x, S.box[0][w]);
        hi_x = fmaxf(hi_x, S.box[1][w]);
        lo_y = fminf(lo_y, S.box[2][w]);
        hi_y = fmaxf(hi_y, S.box[3][w]);
    }
    // thresholds past the antipodes turn back (a = sin^2): cells from the
    // lowest such one on are left to the binary search, as for every pair before
    for (int b = t + 1; b < nedges; b += kHistTile)
        if (!(S.edges[b] >= S.edges[b - 1]))
            atomicMin(&S.turn, __float_as_uint(fmaxf((float)S.edges[b] * (1.0f - kHistTol), 0.0f)));
    __syncthreads();
    const float turn = __uint_as_float(S.turn);
    for (uint32_t c = t; c <= kLutCells; c += kHistTile) {
        const float from = __uint_as_float((c + kLutBase) << kLutShift);
        const float to = __uint_as_float((c + 1u + kLutBase) << kLutShift);
        const int b0 = edges_below(S.edges, nedges, 1.0 + (double)kHistTol, (double)from);
        // how many of the thresholds from b0 on may lie below the cell's end: none, one, more
        const double first = b0 < nedges ? S.edges[b0] : INFINITY, second = b0 + 1 < nedges ? S.edges[b0 + 1] : INFINITY;
        float e = first * (1.0 - (double)kHistTol) < (double)to ? (float)first : FLT_MAX;
        if (c == kLutCells || to >= turn || second * (1.0 - (double)kHistTol) < (double)to) e = NAN;
        S.lut[c] = make_float2(e, __uint_as_float((uint32_t)b0));
    }
    for (int q = 0; q < per; ++q) {
        const int64_t j0 = (jt0 + q) * kHistTile;
        if (j0 >= n) break;  // uniform over the block
        const bool in = j0 + t < n;
        const float x = in ? lon[j0 + t] : 0.0f, y = in ? lat[j0 + t] : 0.0f;
        const float far = fmaxf(fmaxf(x - lo_x, hi_x - x), fmaxf(y - lo_y, hi_y - y));
        const bool fine = fabsf(x) < 1e6f && fabsf(y) <= 90.0f;
        __syncthreads();  // the tile before has been read
        S.cj[t] = cos_deg((double)y);
        S.pj[t] = make_float4(x, y, (float)S.cj[t], 0.0f);
        const bool narrow = __syncthreads_and(!in || (fine && far <= kHistNarrow));
        const bool wide = __syncthreads_and(!in || (fine && far <= kHistWide));
        const int jend = (int)(n - j0 < kHistTile ? n - j0 : kHistTile);
        int after[kHistI];  // pairs (i, j0 + k) with k > after
#pragma unroll
        for (int u = 0; u < kHistI; ++u) {
            const int64_t i = i0 + u * kHistTile + t;
            after[u] = i >= n ? jend : i < j0 ? -1 : (int)(i - j0);
        }
        if (narrow) {
            hist_tile<false>(S, h, jend, xi, yi, ci, after, nedges, cols, col);
        } else if (wide) {
            hist_tile<true>(S, h, jend, xi, yi, ci, after, nedges, cols, col);
        } else {
            hist_tile_f64(S, h, jend, xi, yi, after, nedges, cols, col);
        }
    }
    __syncthreads();
    for (int b = wave; b < nbins; b += kHistTile / 64) {
        uint32_t v = lane < (int)cols ? h[(uint32_t)b * cols + lane] : 0u;
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
        if (lane == 0 && v) atomicAdd(hist + b, (unsigned long long)v);
    }
}

}  // namespace lm

extern "C" {

int lm_species_counts(const int8_t* species, int64_t n, int32_t nsteps, int64_t stride, uint64_t* counts,
                      void* stream) {
    LM_REQUIRE(n >= 0 && nsteps >= 0, LM_ERR_ARG, "negative size");
    LM_REQUIRE(nsteps <= 65535, LM_ERR_ARG, "at most 65535 steps per call");
    LM_REQUIRE(nsteps <= 1 || stride >= n, LM_ERR_ARG, "stride < n");
    if (n == 0 || nsteps == 0) return LM_OK;
    LM_REQUIRE(species && counts, LM_ERR_ARG, "NULL pointer");
    unsigned gx = (unsigned)((n + lm::kCountBytes - 1) / lm::kCountBytes < 1024 ? (n + lm::kCountBytes - 1) / lm::kCountBytes : 1024);
    LM_LAUNCH(lm::K_SPECIES_COUNT, lm::species_count_kernel, dim3(gx, (unsigned)nsteps), dim3(lm::kBlock), 0,
              (hipStream_t)stream, species, n, nsteps <= 1 ? n : stride,
              reinterpret_cast<unsigned long long*>(counts));
    LM_LAUNCH_CHECK();
    return LM_OK;
}

int lm_distance_histogram(int64_t n, const float* lon, const float* lat, int32_t nbins, const double* edges,
                          uint64_t* hist, void* stream) {
    LM_REQUIRE(n >= 0, LM_ERR_ARG, "negative size");
    LM_REQUIRE(nbins >= 1 && nbins <= lm::kHistMaxBins, LM_ERR_ARG, "nbins must be in 1..%d", lm::kHistMaxBins);
    const int64_t ntiles = (n + lm::kHistTile - 1) / lm::kHistTile;
    LM_REQUIRE(ntiles <= 65535, LM_ERR_ARG, "at most %lld points", (long long)65535 * lm::kHistTile);
    if (n < 2) return LM_OK;
    LM_REQUIRE(lon && lat && hist && (nbins == 1 || edges), LM_ERR_ARG, "NULL pointer");
    const int64_t itiles = (n + lm::kHistTile * lm::kHistI - 1) / (lm::kHistTile * lm::kHistI);
    // j tiles per workgroup: as many as leave 4096 workgroups (16 per CU), at
    // most 16, so that the table each one builds is a few percent of its work
    int64_t per = itiles * ntiles / 2 / 4096;
    per = per < 1 ? 1 : per > 16 ? 16 : per;
    // a counter column per lane while the counters take at most 32 KB
    const uint32_t cols = nbins <= 128 ? 64u : 32u;
    LM_LAUNCH(lm::K_DIST_HIST, lm::dist_hist_kernel, dim3((unsigned)itiles, (unsigned)((ntiles + per - 1) / per)),
              dim3(lm::kHistTile), (unsigned)(sizeof(uint32_t) * nbins * cols), (hipStream_t)stream, n, lon, lat,
              (int)nbins, edges, reinterpret_cast<unsigned long long*>(hist), (int)per, cols);
    LM_LAUNCH_CHECK();
    return LM_OK;
}

}  // extern "C"
