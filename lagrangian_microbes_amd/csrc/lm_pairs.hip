// Fixed-radius pair search in lon/lat degree space, for one or many steps.
//
// Cell list with cells of side h >= radius over a fixed box, stored as a sort
// of the particles by bucket over T = 2^k buckets (bucket = dense cell id mod
// T, so the three cells of a stencil row are three consecutive buckets; when
// the box has fewer than T cells the table is dense and nothing aliases):
//   1. bin_keys     : each particle's bucket
//   2. partition    : one radix pass on the bucket's high bits (super-
//                     buckets; no order inside one is needed)
//   3. bin_table    : bucket starts (every bucket between two neighbouring
//                     sorted keys starts at the later one) and records
//                     {x, y, index} in bucket order
//   4. pair_count   : per particle i, the neighbours j > i within radius over
//                     the 3x3 cell stencil (run in bucket order for locality);
//                     up to kNbr of them are kept in a scratch row
//   5. scan         : row offsets and the pair count P
//   6. pair_emit    : per particle, its neighbours sorted ascending, written at
//                     its row offset; rows with more than kNbr neighbours are
//                     re-searched kNbr at a time.  The result is the (i, j)
//                     lexicographic pair list.
// A batch of S steps (S position snapshots) runs every phase once with
// blockIdx.y = step, each step with its own tables and pair region, so a
// launch carries S times the parallelism of one step.  No global atomics.
// Ensembles: with a run id per particle (independent runs sharing the index
// range), the bucket is (run * cells + cell) mod T and the record carries the
// run, so a stencil visits the cells of its own run and candidates of other
// runs whose cells alias into the same buckets are dropped: pairs never cross
// runs.
// Small populations (kSmallMax particles, no runs) take two launches instead,
// whose workgroups bin a whole step in LDS (see "small populations" below).
// Distances use the float32 positions widened to double, with the same
// operations cKDTree applies: dx*dx + dy*dy <= r*r for p = 2, evaluated as
// written (the library is built without FMA contraction).  For positions of
// similar magnitude the double difference of two floats is exact and so is
// its square.
#include "lm_common.h"
#include "lm_scan.h"
#include "lm_small.h"
#include "lm_sort.h"

#include <cmath>
#include <cstdint>
#include <type_traits>

namespace lm {

constexpr int kNbr = 8;  // neighbours kept per particle before the selection path

struct CellGrid {
    double x0, y0, inv_h;
    int32_t nx, ny;
    uint32_t mask;   // T - 1
    uint32_t T;
    uint32_t cells;  // nx * ny (mod 2^32): the key distance between runs
};

enum MetricKind { kL2 = 0, kL1 = 1, kLinf = 2, kLp = 3 };

struct Metric {
    int kind;
    double r;    // radius
    double r2;   // radius*radius (p = 2) or radius^p (general p)
    double p;
    float box;   // float32 bound above the radius: |dx| or |dy| beyond it rules a pair out
    // p = 2: a float32 dx*dx + dy*dy at or below sure_in is within the radius,
    // above sure_out beyond it, whatever the float64 test rounds (-inf / +inf:
    // every candidate takes the float64 test)
    float sure_in, sure_out;
};

// Per-step strides of a batch (elements).
struct Strides {
    int64_t pos;    // between position snapshots
    int64_t tab;    // bucket tables (>= T + 1, multiple of 4)
    int64_t rec;    // bucket-ordered records and sort buffers
    int64_t row;    // per-particle counts / offsets (>= n + 1, multiple of 4)
    int64_t nbr;    // neighbour scratch rows
    int64_t pair;   // pair list capacity per step
};

__device__ __forceinline__ void cell_of(const CellGrid& g, float xf, float yf, int* cx, int* cy) {
    const double fx = ((double)xf - g.x0) * g.inv_h;
    const double fy = ((double)yf - g.y0) * g.inv_h;
    int ix = 0, iy = 0;
    if (fx >= 1.0) ix = fx >= (double)(g.nx - 1) ? g.nx - 1 : (int)fx;
    if (fy >= 1.0) iy = fy >= (double)(g.ny - 1) ? g.ny - 1 : (int)fy;
    *cx = ix;
    *cy = iy;
}

__device__ __forceinline__ uint32_t bucket_of(const CellGrid& g, int cx, int cy, uint32_t run) {
    return (run * g.cells + (uint32_t)cy * (uint32_t)g.nx + (uint32_t)cx) & g.mask;
}

// The metric is a template argument of the kernels that test candidates, so
// each instance holds only its own test (the general-p form inlines pow).
template <int KIND>
__device__ __forceinline__ bool within(const Metric& m, float xa, float ya, float xb, float yb) {
    const double dx = (double)xb - (double)xa;
    const double dy = (double)yb - (double)ya;
    if constexpr (KIND == kL2) return dx * dx + dy * dy <= m.r2;
    else if constexpr (KIND == kL1) return fabs(dx) + fabs(dy) <= m.r;
    else if constexpr (KIND == kLinf) return fmax(fabs(dx), fabs(dy)) <= m.r;
    else return pow(fabs(dx), m.p) + pow(fabs(dy), m.p) <= m.r2;
}

// The same decision, mostly in float32, for a candidate (cand) or false.
template <int KIND>
__device__ __forceinline__ bool pair_hit(const Metric& m, bool cand, float xa, float ya, float xb, float yb) {
    if constexpr (KIND == kL2) {
        // A float32 difference of two float32 positions is within one
        // rounding (relative 2^-24) of the exact one, so the float32
        // dx*dx + dy*dy is within 2.4e-7 (relative) of the exact sum of
        // squares, and the float64 test within 2^-52: outside r^2 (1 -/+
        // 1e-6) both decide alike.  Only candidates in that band take
        // the float64 test (a branch almost never taken).
        const float dx = xb - xa, dy = yb - ya;
        const float d2 = fmaf(dx, dx, dy * dy);
        bool hit = cand & (d2 <= m.sure_in);
        if (cand & !(d2 <= m.sure_in) & !(d2 > m.sure_out)) hit = within<KIND>(m, xa, ya, xb, yb);
        return hit;
    } else {
        // |dx| <= r and |dy| <= r hold for every p >= 1; a float32
        // difference is within one rounding (relative 2^-24) of the exact
        // one and m.box lies above r by more than that, so the prefilter
        // only drops pairs the exact test drops.
        const float ax = fabsf(xb - xa), ay = fabsf(yb - ya);
        return cand & (ax <= m.box) & (ay <= m.box) & within<KIND>(m, xa, ya, xb, yb);
    }
}

// Visit the record slots of the (up to) 3x3 cells around (cx, cy).  Slot
// ranges are clamped to nrec so that even inconsistent bucket starts cannot
// index past the records.
template <typename F>
__device__ __forceinline__ void for_stencil(const CellGrid& g, const uint32_t* __restrict__ start,
                                            uint32_t nrec, int cx, int cy, uint32_t run, F&& visit) {
    const int c0 = cx > 0 ? cx - 1 : 0;
    const int c1 = cx < g.nx - 1 ? cx + 1 : g.nx - 1;
#pragma unroll
    for (int dyc = -1; dyc <= 1; ++dyc) {
        const int row = cy + dyc;
        if (row < 0 || row >= g.ny) continue;
        const uint32_t b0 = bucket_of(g, c0, row, run);
        const uint32_t b1 = bucket_of(g, c1, row, run);
        if (b0 <= b1) {
            const uint32_t e = min(start[b1 + 1], nrec);
            for (uint32_t s = start[b0]; s < e; ++s) visit(s);
        } else {  // the row wraps around the bucket table
            const uint32_t e0 = min(start[g.T], nrec);
            for (uint32_t s = start[b0]; s < e0; ++s) visit(s);
            const uint32_t e1 = min(start[b1 + 1], nrec);
            for (uint32_t s = start[0]; s < e1; ++s) visit(s);
        }
    }
}

__global__ void __launch_bounds__(kBlock)
bin_keys_kernel(int64_t n, const float* __restrict__ x, const float* __restrict__ y,
                const uint16_t* __restrict__ run, CellGrid g, Strides st, uint32_t* __restrict__ keys,
                uint32_t* __restrict__ vals, float2* __restrict__ xy) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const int64_t s = blockIdx.y;
    const float xf = x[s * st.pos + i], yf = y[s * st.pos + i];
    int cx, cy;
    cell_of(g, xf, yf, &cx, &cy);
    keys[s * st.rec + i] = bucket_of(g, cx, cy, run ? (uint32_t)run[i] : 0u);
    if (vals) vals[s * st.rec + i] = (uint32_t)i;  // NULL when the radix pass generates the indices
    // interleaved copy: the binning gathers a particle's position with one 8-byte load
    xy[s * st.rec + i] = make_float2(xf, yf);
}

// Second level of the binning: one block per super-bucket (the particles
// whose bucket has the same high bits, made contiguous by one radix pass),
// counting its `fine` buckets in LDS.  It writes their starts (a contiguous
// slice of the table; the last super-bucket also the end, start[T] = n) and
// places the records {x, y, index} of its particles in bucket order (the
// order inside a bucket is free: the pair list is sorted later).  FINE_MAX
// buckets per block: 4096 up to 2^22 buckets, 8192 up to 2^23.
constexpr uint32_t kFineMax = 4096;
constexpr int kPlace = 8;  // particles per thread in flight when placing records
constexpr uint32_t kFineMaxWide = 8192;

template <uint32_t FINE_MAX>
__global__ void __launch_bounds__(kBlock)
bin_table_kernel(int64_t n, const float2* __restrict__ xy, const uint16_t* __restrict__ run, CellGrid g, Strides st,
                 const uint32_t* __restrict__ keys_all,
                 const uint32_t* __restrict__ vals_all, const uint32_t* __restrict__ dstart, int64_t drow,
                 int64_t dstride, uint32_t fine, uint32_t* __restrict__ start_all, float4* __restrict__ recs_all) {
    uint32_t bx, by;
    xcd_block(&bx, &by);  // an XCD works through a contiguous range of steps: one step's arrays in its L2
    __shared__ uint32_t cnt[FINE_MAX];
    __shared__ uint32_t scan_lds[kBlock / 64];
    const uint32_t d = bx, nsuper = gridDim.x, t = threadIdx.x;
    const int64_t s = by;
    const uint32_t* keys = keys_all + s * st.rec;
    const uint32_t* vals = vals_all + s * st.rec;
    uint32_t* start = start_all + s * st.tab;
    const uint32_t nn = (uint32_t)n;
    uint32_t a = 0, b = nn;
    if (dstart != nullptr) {
        a = min(dstart[s * drow + (int64_t)d * dstride], nn);
        b = d + 1 < nsuper ? min(dstart[s * drow + (int64_t)(d + 1) * dstride], nn) : nn;
        b = max(a, b);
    }
    const uint32_t fmask = fine - 1u;
    for (uint32_t f = t; f < fine; f += kBlock) cnt[f] = 0;
    __syncthreads();
    // kPlace keys per thread in flight at once (indices clamped into the
    // super-bucket, loads pinned ahead of the atomics)
    for (uint32_t e0 = a + t; e0 < b; e0 += kBlock * kPlace) {
        uint32_t kk[kPlace];
#pragma unroll
        for (int u = 0; u < kPlace; ++u) kk[u] = keys[min(e0 + (uint32_t)u * kBlock, b - 1u)];
#pragma unroll
        for (int u = 0; u < kPlace; ++u) lm_pin(kk[u]);
#pragma unroll
        for (int u = 0; u < kPlace; ++u)
            if (e0 + (uint32_t)u * kBlock < b) atomicAdd(&cnt[kk[u] & fmask], 1u);
    }
    __syncthreads();
    // exclusive offsets: thread t owns `per` consecutive buckets
    const uint32_t per = (fine + kBlock - 1) / kBlock;
    const uint32_t f0 = min(t * per, fine), f1 = min(f0 + per, fine);
    uint32_t sum = 0;
    for (uint32_t f = f0; f < f1; ++f) sum += cnt[f];
    uint32_t all;
    uint32_t acc = block_exclusive_scan(sum, scan_lds, &all);
    for (uint32_t f = f0; f < f1; ++f) {
        const uint32_t c = cnt[f];
        cnt[f] = acc;
        acc += c;
    }
    __syncthreads();
    const uint64_t base = (uint64_t)d * fine;
    for (uint32_t f = t; f < fine; f += kBlock)
        if (base + f < (uint64_t)g.T) start[base + f] = a + cnt[f];
    if (d + 1 == nsuper && t == 0) start[g.T] = nn;
    __syncthreads();
    // kPlace particles per thread at once, so their position gathers (random
    // lines) are in flight together
    // two rounds of loads per kPlace particles, each issued at once (indices
    // clamped, loads pinned ahead of their uses): indices and keys, then the
    // positions the indices point at
    for (uint32_t e0 = a + t; e0 < b; e0 += kBlock * kPlace) {
        uint32_t ii[kPlace], kk[kPlace], pp[kPlace];
#pragma unroll
        for (int u = 0; u < kPlace; ++u) {
            const uint32_t e = min(e0 + (uint32_t)u * kBlock, b - 1u);
            ii[u] = vals[e];
            kk[u] = keys[e];
        }
#pragma unroll
        for (int u = 0; u < kPlace; ++u) lm_pin(ii[u], kk[u]);
#pragma unroll
        for (int u = 0; u < kPlace; ++u) {
            const bool live = e0 + (uint32_t)u * kBlock < b && ii[u] < nn;
            pp[u] = live ? a + atomicAdd(&cnt[kk[u] & fmask], 1u) : b;
        }
        float2 pv[kPlace];
#pragma unroll
        for (int u = 0; u < kPlace; ++u) pv[u] = xy[s * st.rec + (ii[u] < nn ? ii[u] : 0u)];
        uint32_t rr[kPlace];
#pragma unroll
        for (int u = 0; u < kPlace; ++u) rr[u] = run ? (uint32_t)run[ii[u] < nn ? ii[u] : 0u] : 0u;
#pragma unroll
        for (int u = 0; u < kPlace; ++u)
            if (pp[u] < b)
                recs_all[s * st.rec + pp[u]] = make_float4(pv[u].x, pv[u].y, __uint_as_float(ii[u]),
                                                           __uint_as_float(rr[u]));
    }
}

// The (up to) six record ranges of the 3x3 stencil around (cx, cy): a row of
// three cells is one bucket range, or two when it wraps around the table.
// All bucket starts are loaded at once.  Ranges are clamped to nrec.
__device__ __forceinline__ void stencil_ranges(const CellGrid& g, const uint32_t* __restrict__ start, uint32_t nrec,
                                               int cx, int cy, uint32_t run, uint32_t (&rb)[6], uint32_t (&re)[6]) {
    const int c0 = cx > 0 ? cx - 1 : 0;
    const int c1 = cx < g.nx - 1 ? cx + 1 : g.nx - 1;
    uint32_t lo[6], hi[6];
    bool on[6];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        const int row = cy + r - 1;
        const bool valid = row >= 0 && row < g.ny;
        const uint32_t b0 = valid ? bucket_of(g, c0, row, run) : 0u;
        const uint32_t b1 = valid ? bucket_of(g, c1, row, run) : 0u;
        const bool wrap = b0 > b1;
        // first segment [b0, wrap ? T : b1 + 1), second [0, b1 + 1) if wrapped
        lo[2 * r] = b0;
        hi[2 * r] = wrap ? g.T : b1 + 1u;
        on[2 * r] = valid;
        lo[2 * r + 1] = 0u;
        hi[2 * r + 1] = b1 + 1u;
        on[2 * r + 1] = valid && wrap;
    }
    uint32_t sb[6], se[6];
    // the three main segments load unconditionally (index 0 for a row off the
    // grid, then discarded); the wrapped second segments are rare
#pragma unroll
    for (int r = 0; r < 6; r += 2) {
        sb[r] = start[on[r] ? lo[r] : 0u];
        se[r] = start[on[r] ? hi[r] : 0u];
        sb[r] = on[r] ? sb[r] : 0u;
        se[r] = on[r] ? se[r] : 0u;
    }
#pragma unroll
    for (int r = 1; r < 6; r += 2) {
        sb[r] = on[r] ? start[lo[r]] : 0u;
        se[r] = on[r] ? start[hi[r]] : 0u;
    }
#pragma unroll
    for (int r = 0; r < 6; ++r) {
        re[r] = min(se[r], nrec);
        rb[r] = min(sb[r], re[r]);
    }
}

constexpr int kCand = 8;  // candidate records in flight per thread

template <int KIND>
__global__ void __launch_bounds__(kBlock)
pair_count_kernel(int64_t n, CellGrid g, Metric m, Strides st, const uint32_t* __restrict__ start_all,
                  const float4* __restrict__ recs_all, uint32_t* __restrict__ nbr_cnt,
                  uint32_t* __restrict__ nbr) {
    uint32_t bx, by;
    xcd_block(&bx, &by);  // a particle's stencil rows lie a few blocks away in bucket order
    const int64_t s0 = (int64_t)bx * kBlock + threadIdx.x;
    if (s0 >= n) return;
    const int64_t s = by;
    const uint32_t* start = start_all + s * st.tab;
    const float4* recs = recs_all + s * st.rec;
    const float4 me = recs[s0];
    uint32_t i = __float_as_uint(me.z), my_run = __float_as_uint(me.w);
    lm_pin(i, my_run);  // the whole record in one load, not split around the branch
    if (i >= (uint64_t)n) return;
    int cx, cy;
    cell_of(g, me.x, me.y, &cx, &cy);
    uint32_t rb[6], re[6];
    stencil_ranges(g, start, (uint32_t)n, cx, cy, my_run, rb, re);
    // the ranges as one sequence: candidate t lies in range r when
    // pre[r] <= t < pre[r + 1], at slot t + dlt[r]
    uint32_t pre[6], dlt[6];
    pre[0] = 0;
#pragma unroll
    for (int r = 0; r < 6; ++r) {
        dlt[r] = rb[r] - pre[r];  // mod 2^32
        if (r < 5) pre[r + 1] = pre[r] + (re[r] - rb[r]);
    }
    const uint32_t total = pre[5] + (re[5] - rb[5]);
    uint32_t cnt = 0;
    uint32_t* row = nbr + s * st.nbr + (int64_t)i * kNbr;
    for (uint32_t t0 = 0; t0 < total; t0 += kCand) {
        float4 o[kCand];
#pragma unroll
        for (int u = 0; u < kCand; ++u) {
            // past the end the lane is masked off (no address-unit work) and
            // the candidate is discarded below
            const uint32_t t = t0 + u;
            uint32_t d = dlt[0];
#pragma unroll
            for (int r = 1; r < 6; ++r) d = t >= pre[r] ? dlt[r] : d;
            o[u] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (t < total) o[u] = recs[t + d];
        }
        // every load of the batch is issued before any use of the first: the
        // scheduler would otherwise start testing candidate 0 early and wait
        // for it before issuing the rest
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < kCand; ++u) {
            const uint32_t j = __float_as_uint(o[u].z);
            const bool cand = (t0 + u < total) & (j > i) & (__float_as_uint(o[u].w) == my_run);
            const bool hit = pair_hit<KIND>(m, cand, me.x, me.y, o[u].x, o[u].y);
            if (hit & (cnt < kNbr)) row[cnt] = j;
            cnt += hit ? 1u : 0u;
        }
    }
    nbr_cnt[s * st.row + i] = cnt;
}

// Sort the first c (<= K) entries of a scratch row in registers and write
// them as row o.. of the pair list.
template <int K>
__device__ __forceinline__ void emit_sorted(const uint32_t* row, uint32_t c, uint32_t i, uint32_t o,
                                            int32_t* __restrict__ pair_i, int32_t* __restrict__ pair_j) {
    uint32_t v[K];
#pragma unroll
    for (int t = 0; t < K; ++t) v[t] = (uint32_t)t < c ? row[t] : 0xffffffffu;
#pragma unroll
    for (int a = 1; a < K; ++a)
#pragma unroll
        for (int b = a; b > 0; --b) {
            const uint32_t lo = min(v[b - 1], v[b]), hi = max(v[b - 1], v[b]);
            v[b - 1] = lo;
            v[b] = hi;
        }
#pragma unroll
    for (int t = 0; t < K; ++t)
        if ((uint32_t)t < c) {
            pair_i[o + t] = (int32_t)i;
            pair_j[o + t] = (int32_t)v[t];
        }
}

template <int KIND>
__global__ void __launch_bounds__(kBlock)
pair_emit_kernel(int64_t n, const float* __restrict__ x_all, const float* __restrict__ y_all,
                 const uint16_t* __restrict__ run, CellGrid g, Metric m, Strides st, const uint32_t* __restrict__ start_all, const float4* __restrict__ recs_all,
                 const uint32_t* __restrict__ nbr_cnt_all, const uint32_t* __restrict__ nbr_all,
                 const uint32_t* __restrict__ row_off_all, int32_t* __restrict__ pair_i_all,
                 int32_t* __restrict__ pair_j_all) {
    uint32_t bx, by;
    xcd_block(&bx, &by);  // an XCD works through a contiguous range of steps: one step's arrays in its L2
    const int64_t i64 = (int64_t)bx * kBlock + threadIdx.x;
    if (i64 >= n) return;
    const int64_t s = by;
    const uint32_t* row_off = row_off_all + s * st.row;
    const uint32_t i = (uint32_t)i64;
    // the step's total, this row's count and offset and its first two
    // partners (read whatever the count, then used as it says) load
    // together, before any branch on them
    const uint32_t total = row_off[n];
    const uint32_t* row = nbr_all + s * st.nbr + (int64_t)i * kNbr;
    uint32_t c = nbr_cnt_all[s * st.row + i], o = row_off[i];
    const uint2 ab = *reinterpret_cast<const uint2*>(row);  // rows are 32-byte aligned
    uint32_t r0 = ab.x, r1 = ab.y;
    lm_pin(c, o, r0, r1);
    if ((int64_t)total > st.pair) return;  // caller enlarges and calls again
    if (c == 0) return;
    int32_t* pair_i = pair_i_all + s * st.pair;
    int32_t* pair_j = pair_j_all + s * st.pair;
    if (c <= 2) {
        const uint32_t a = r0, b = c == 2 ? r1 : 0xffffffffu;
        pair_i[o] = (int32_t)i;
        pair_j[o] = (int32_t)min(a, b);
        if (c == 2) {
            pair_i[o + 1] = (int32_t)i;
            pair_j[o + 1] = (int32_t)max(a, b);
        }
        return;
    }
    if (c <= 4) return emit_sorted<4>(row, c, i, o, pair_i, pair_j);
    if (c <= (uint32_t)kNbr) return emit_sorted<kNbr>(row, c, i, o, pair_i, pair_j);
    // Dense neighbourhood: emit in ascending order, 16 at a time, each pass
    // keeping the 16 smallest partners above the last one written.
    constexpr int kSel = 16;
    const uint32_t* start = start_all + s * st.tab;
    const float4* recs = recs_all + s * st.rec;
    const float xf = x_all[s * st.pos + i], yf = y_all[s * st.pos + i];
    const uint32_t my_run = run ? (uint32_t)run[i] : 0u;
    int cx, cy;
    cell_of(g, xf, yf, &cx, &cy);
    uint32_t last = i;
    for (uint32_t t = 0; t < c;) {
        uint32_t v[kSel];
#pragma unroll
        for (int q = 0; q < kSel; ++q) v[q] = 0xffffffffu;
        for_stencil(g, start, (uint32_t)n, cx, cy, my_run, [&](uint32_t q0) {
            const float4 rec = recs[q0];
            uint32_t j = __float_as_uint(rec.z);
            if (j > last && j < v[kSel - 1] && __float_as_uint(rec.w) == my_run && within<KIND>(m, xf, yf, rec.x, rec.y)) {
#pragma unroll
                for (int q = 0; q < kSel; ++q) {  // insert into the sorted register array
                    const uint32_t lo = min(v[q], j), hi = max(v[q], j);
                    v[q] = lo;
                    j = hi;
                }
            }
        });
        const uint32_t take = min((uint32_t)kSel, c - t);
#pragma unroll
        for (int q = 0; q < kSel; ++q)
            if ((uint32_t)q < take) {
                pair_i[o + t + q] = (int32_t)i;
                pair_j[o + t + q] = (int32_t)v[q];
                last = v[q];
            }
        t += take;
    }
}

// ---------------------------------------------------------------------------
// small populations
// ---------------------------------------------------------------------------
// Two launches.  Launch latency was the cost of these sizes: the search of
// 2,500 particles took ten launches of 3 to 9 us each, 42 us in all, and takes
// 13.4 us with these two (8 and 4.5 us); twelve steps of 10,000 took 107 us
// and take 28.  The line is where a step's particles still fit one LDS.
//   count  workgroups of 1024 lanes, each binning the whole step into its LDS
//          (positions and indices in bucket order, behind one bucket table)
//          and searching its own 1024 / LPP particles, LPP lanes each (with
//          4, three lanes take a stencil row each): partners above each
//          particle, counted, the first kSmallNbr kept
//   emit   every workgroup sums the counts before its ROWS rows, scans its
//          own and writes them sorted; its rows of more than kSmallNbr
//          partners are found again by a wavefront each, from the bucket order
//          that the count left in memory, or, with hundreds of partners,
//          among all particles in index order
// The cells wrap onto a torus of 2^LWX x 2^LWY buckets (a stencil's nine cells
// always fall into nine buckets: the sides are at least 64; cells further
// apart may share one, and the distance test drops what the stencil does not
// reach), so the table fits LDS whatever the box.
constexpr int kSmallNbr = 16;  // 16-bit partners kept per particle, in the bytes of kNbr 32-bit ones
constexpr int64_t kSmallTable = 4096;  // particles up to which the table has 2^12 buckets (2^13 above)
// Entries per step, in memory, of a table of 2^bits buckets.
constexpr int64_t small_tab(int bits) { return ((int64_t)1 << bits) + 4; }

// A crowded row's partners are gathered from its buckets and ranked against
// each other (the work grows with their square) up to 128 + n / 48 of them, and
// found among all particles in index order (the work grows with n, and there
// is nothing to rank) above.  2,500 particles with a mean of 150 partners: 514
// us with the line at 512, 294 at 180; 12,288 with 200: 899 at 384, 1,042 at 256.
constexpr uint32_t kSmallGather = 128 + (uint32_t)kSmallMax / 48;

__device__ __forceinline__ uint32_t lane_of(uint32_t v, int lane) {  // lane: uniform
    return (uint32_t)__builtin_amdgcn_readlane((int)v, lane);
}
__device__ __forceinline__ float lane_of(float v, int lane) {
    return __uint_as_float(lane_of(__float_as_uint(v), lane));
}

template <int LWX, int LWY, typename F>
__device__ __forceinline__ void small_row(const uint32_t* start, const CellGrid& g, int cx, int row, F&& visit) {
    constexpr uint32_t WX = 1u << LWX, WY = 1u << LWY;
    if (row < 0 || row >= g.ny) return;
    const uint32_t a = (uint32_t)(cx > 0 ? cx - 1 : 0) & (WX - 1u);
    const uint32_t b = (uint32_t)(cx < g.nx - 1 ? cx + 1 : g.nx - 1) & (WX - 1u);
    const uint32_t base = ((uint32_t)row & (WY - 1u)) << LWX;
    // one bucket range, or two when the row wraps
    const uint32_t e0 = start[base + (a <= b ? b + 1u : WX)];
    for (uint32_t s = start[base + a]; s < e0; ++s) visit(s);
    if (a > b) {
        const uint32_t e1 = start[base + b + 1u];
        for (uint32_t s = start[base]; s < e1; ++s) visit(s);
    }
}

template <int KIND, int NMAX, int LWX, int LWY, int LPP>
__global__ void __launch_bounds__(kSmallBlock)
pair_small_count_kernel(int n, const float* __restrict__ x_all, const float* __restrict__ y_all, CellGrid g, Metric m,
                        Strides st, uint32_t* __restrict__ cnt_all, uint16_t* __restrict__ nbr_all,
                        uint32_t* __restrict__ tab_all, uint32_t* __restrict__ order_all) {
    constexpr int kItems = NMAX / kSmallBlock;
    constexpr uint32_t T = 1u << (LWX + LWY);
    static_assert(NMAX % kSmallBlock == 0 && NMAX <= 65536, "16-bit indices, whole items");
    static_assert(LPP == 1 || LPP == 4, "a lane per particle, or one per stencil row");
    __shared__ float2 pos[NMAX];  // in bucket order
    __shared__ __align__(4) uint16_t idx[NMAX];
    __shared__ uint32_t start[T + 1];
    __shared__ uint32_t scan_lds[kSmallBlock / 64];
    const int64_t s = blockIdx.y;
    const float* x = x_all + s * st.pos;
    const float* y = y_all + s * st.pos;
    const int t = threadIdx.x;
    float px[kItems], py[kItems];
    uint32_t bucket[kItems], slot[kItems];
#pragma unroll
    for (int q = 0; q < kItems; ++q) {
        const int i = q * kSmallBlock + t;
        px[q] = i < n ? x[i] : 0.0f;
        py[q] = i < n ? y[i] : 0.0f;
    }
    for (uint32_t b = t; b <= T; b += kSmallBlock) start[b] = 0u;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kItems; ++q) {
        bucket[q] = slot[q] = 0u;
        if (q * kSmallBlock + t < n) {
            int cx, cy;
            cell_of(g, px[q], py[q], &cx, &cy);
            bucket[q] = (((uint32_t)cy & ((1u << LWY) - 1u)) << LWX) | ((uint32_t)cx & ((1u << LWX) - 1u));
            slot[q] = atomicAdd(&start[bucket[q]], 1u);
        }
    }
    __syncthreads();
    small_scan_array(start, T, scan_lds);
    if (t == 0) start[T] = (uint32_t)n;
#pragma unroll
    for (int q = 0; q < kItems; ++q) {
        const int i = q * kSmallBlock + t;
        if (i < n) {
            const uint32_t at = start[bucket[q]] + slot[q];
            pos[at] = make_float2(px[q], py[q]);
            idx[at] = (uint16_t)i;
        }
    }
    __syncthreads();
    if (blockIdx.x == 0) {  // for the rows that the emit finds again
        for (uint32_t b = t; b <= T; b += kSmallBlock) tab_all[s * small_tab(LWX + LWY) + b] = start[b];
        for (int k = t; k < (n + 1) / 2; k += kSmallBlock)
            order_all[s * st.rec + k] = reinterpret_cast<const uint32_t*>(idx)[k];
    }
    const int sub = t % LPP;
    for (int i = (int)blockIdx.x * (kSmallBlock / LPP) + t / LPP; i < n; i += (int)gridDim.x * (kSmallBlock / LPP)) {
        // (all lanes of a particle take the loop and its exits together)
        const float xi = x[i], yi = y[i];
        int cx, cy;
        cell_of(g, xi, yi, &cx, &cy);
        auto search = [&](auto&& visit) {
            if constexpr (LPP == 4) {
                if (sub < 3) small_row<LWX, LWY>(start, g, cx, cy + sub - 1, visit);
            } else {
                for (int r = -1; r <= 1; ++r) small_row<LWX, LWY>(start, g, cx, cy + r, visit);
            }
        };
        uint32_t c = 0;
        search([&](uint32_t k) {
            const float2 o = pos[k];
            c += pair_hit<KIND>(m, (int)idx[k] > i, xi, yi, o.x, o.y) ? 1u : 0u;
        });
        uint32_t at = 0, all = c;
        if constexpr (LPP == 4) {  // the particle's lanes add up
            const uint32_t up1 = __shfl_up(c, 1, 4), up2 = __shfl_up(c, 2, 4);
            at = (sub > 0 ? up1 : 0u) + (sub > 1 ? up2 : 0u);
            all = __shfl(at + c, 2, 4);
        }
        if (sub == 0) cnt_all[s * st.row + i] = all;
        if (c == 0 || all > (uint32_t)kSmallNbr) continue;
        uint16_t* row = nbr_all + 2 * s * st.nbr + (int64_t)i * kSmallNbr;
        search([&](uint32_t k) {
            const float2 o = pos[k];
            if (pair_hit<KIND>(m, (int)idx[k] > i, xi, yi, o.x, o.y)) {
                row[at] = idx[k];
                ++at;
            }
        });
    }
}

// LDS accesses of a wavefront's lanes before and after keep their order: the
// hardware's is that of the instructions, which the fence makes the compiler keep.
__device__ __forceinline__ void wave_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// One crowded row by a wavefront, from its buckets: rc <= kSmallGather partners
// (found: kSmallGather 16-bit slots of LDS), written sorted to [at, at + rc).
// from[0 .. 6), len: the row's candidates, as ranges of the bucket order.
template <int KIND>
__device__ __forceinline__ void small_gather_row(int n, const float* __restrict__ x, const float* __restrict__ y,
                                                 const Metric& m, const uint16_t* __restrict__ order, int r, float xr,
                                                 float yr, const uint32_t (&from)[6], const uint32_t (&len)[6],
                                                 uint32_t rc, uint32_t at, uint16_t* found, int32_t* __restrict__ pair_i,
                                                 int32_t* __restrict__ pair_j) {
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t total = 0;
#pragma unroll
    for (int q = 0; q < 6; ++q) total += len[q];
    uint32_t have = 0;
    for (uint32_t c0 = 0; c0 < total; c0 += 64) {
        uint32_t c = c0 + lane, k = 0;
        const bool cand = c < total;
#pragma unroll
        for (int q = 0; q < 6; ++q) {  // the range that holds candidate c
            k = c < len[q] ? from[q] + c : k;
            c = c < len[q] ? 0xffffffffu : c - len[q];
        }
        const int j = cand ? (int)order[k] : 0;
        const bool hit = pair_hit<KIND>(m, cand && j > r && j < n, xr, yr, x[j], y[j]);
        const uint64_t hits = __ballot(hit);
        const uint32_t slot = have + (uint32_t)__popcll(hits & ((1ull << lane) - 1ull));
        if (hit && slot < rc) found[slot] = (uint16_t)j;
        have += (uint32_t)__popcll(hits);
    }
    have = min(have, rc);
    // the slots after the last one, read eight at a time below
    if (lane < 8 && have + lane < kSmallGather) found[have + lane] = 0xffffu;
    wave_order();
    for (uint32_t v0 = 0; v0 < have; v0 += 64) {
        const bool mine = v0 + lane < have;
        const uint32_t v = mine ? found[v0 + lane] : 0u;
        uint32_t rank = 0;
        for (uint32_t q = 0; q < have; q += 8) {
            const uint4 o = *reinterpret_cast<const uint4*>(found + q);
            rank += ((o.x & 0xffffu) < v) + ((o.x >> 16) < v) + ((o.y & 0xffffu) < v) + ((o.y >> 16) < v) +
                    ((o.z & 0xffffu) < v) + ((o.z >> 16) < v) + ((o.w & 0xffffu) < v) + ((o.w >> 16) < v);
        }
        if (mine) {
            pair_i[at + rank] = r;
            pair_j[at + rank] = (int32_t)v;
        }
    }
    wave_order();
}

template <int KIND, int LWX, int LWY, int ROWS>
__global__ void __launch_bounds__(kSmallBlock)
pair_small_emit_kernel(int n, const float* __restrict__ x_all, const float* __restrict__ y_all, CellGrid g, Metric m,
                       Strides st, const uint32_t* __restrict__ cnt_all, const uint16_t* __restrict__ nbr_all,
                       const uint32_t* __restrict__ tab_all, const uint16_t* __restrict__ order_all,
                       int32_t* __restrict__ pair_i_all, int32_t* __restrict__ pair_j_all,
                       int64_t* __restrict__ npairs) {
    constexpr uint32_t WX = 1u << LWX, WY = 1u << LWY;
    __shared__ uint32_t sums[3][kSmallBlock / 64], crowded;  // per wavefront: before, own, after
    __shared__ uint32_t who[ROWS], count[ROWS], place[ROWS];  // the crowded rows
    __shared__ __align__(16) uint16_t found[kSmallBlock / 64][kSmallGather];
    const int64_t s = blockIdx.y;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, i0 = (int)blockIdx.x * ROWS, i = i0 + t;
    const bool own = t < ROWS && i < n;
    const uint32_t* cnt = cnt_all + s * st.row;
    const uint16_t* row = nbr_all + 2 * s * st.nbr + (int64_t)(own ? i : 0) * kSmallNbr;
    // this row's count and partners (read whatever the count) and the counts
    // before and after the workgroup's rows load together
    uint32_t c = own ? cnt[i] : 0u;
    const uint4 lo = reinterpret_cast<const uint4*>(row)[0], hi = reinterpret_cast<const uint4*>(row)[1];
    uint32_t before = 0, after = 0;
#pragma unroll
    for (int q = 0; q < (int)(kSmallMax / kSmallBlock); ++q) {
        const int k = q * kSmallBlock + t;
        const uint32_t v = k < n && (k < i0 || k >= i0 + ROWS) ? cnt[k] : 0u;
        before += k < i0 ? v : 0u;
        after += k < i0 ? 0u : v;
    }
    if (t == 0) crowded = 0u;
    const uint32_t inc = wave_inclusive_scan(c);
    before = wave_sum(before);
    after = wave_sum(after);
    if (lane == 63) {
        sums[0][wave] = before;
        sums[1][wave] = inc;
        sums[2][wave] = after;
    }
    __syncthreads();
    uint32_t o = inc - c, total = 0;
#pragma unroll
    for (int w = 0; w < kSmallBlock / 64; ++w) {
        const uint32_t own_w = sums[1][w];
        o += sums[0][w] + (w < wave ? own_w : 0u);
        total += sums[0][w] + own_w + sums[2][w];
    }
    if (blockIdx.x == 0 && t == 0) npairs[s] = (int64_t)total;
    if ((int64_t)total > st.pair) return;  // caller enlarges and calls again
    int32_t* pair_i = pair_i_all + s * st.pair;
    int32_t* pair_j = pair_j_all + s * st.pair;
    if (c > 0 && c <= (uint32_t)kSmallNbr) {
        const uint32_t w[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
        uint32_t v[kSmallNbr];
#pragma unroll
        for (int k = 0; k < kSmallNbr; ++k) v[k] = (uint32_t)k < c ? (w[k >> 1] >> (16 * (k & 1))) & 0xffffu : 0xffffffffu;
        auto sort = [&](auto K) {
            constexpr int N = decltype(K)::value;
#pragma unroll
            for (int a = 1; a < N; ++a)
#pragma unroll
                for (int b = a; b > 0; --b) {
                    const uint32_t x = min(v[b - 1], v[b]), y = max(v[b - 1], v[b]);
                    v[b - 1] = x;
                    v[b] = y;
                }
        };
        if (c <= 4) sort(std::integral_constant<int, 4>{});
        else sort(std::integral_constant<int, kSmallNbr>{});
#pragma unroll
        for (int k = 0; k < kSmallNbr; ++k)
            if ((uint32_t)k < c) {
                pair_i[o + k] = i;
                pair_j[o + k] = (int32_t)v[k];
            }
    }
    if (c > (uint32_t)kSmallNbr) {
        const uint32_t q = atomicAdd(&crowded, 1u);
        who[q] = (uint32_t)i;
        count[q] = c;
        place[q] = o;
    }
    __syncthreads();
    // the crowded rows, shared out over the wavefronts: lane q of a wavefront
    // looks up the buckets of its q-th row
    static_assert(ROWS <= 64 * (kSmallBlock / 64), "a lane per row of a wavefront");
    if (crowded == 0u) return;  // uniform
    const float* x = x_all + s * st.pos;
    const float* y = y_all + s * st.pos;
    const uint32_t* tab = tab_all + s * small_tab(LWX + LWY);
    const uint16_t* order = order_all + 2 * s * st.rec;
    const uint32_t entry = (uint32_t)lane * (kSmallBlock / 64) + (uint32_t)wave, e = min(entry, crowded - 1u);
    const uint32_t rows = crowded > (uint32_t)wave ? (crowded - (uint32_t)wave + kSmallBlock / 64 - 1) / (kSmallBlock / 64) : 0u;
    const uint32_t my_r = who[e], my_c = count[e], my_o = place[e];
    const float my_x = x[my_r], my_y = y[my_r];
    uint32_t my_from[6], my_len[6];
    int cx, cy;
    cell_of(g, my_x, my_y, &cx, &cy);
    const uint32_t a = (uint32_t)(cx > 0 ? cx - 1 : 0) & (WX - 1u);
    const uint32_t b = (uint32_t)(cx < g.nx - 1 ? cx + 1 : g.nx - 1) & (WX - 1u);
#pragma unroll
    for (int q = 0; q < 3; ++q) {  // as small_row
        const int cr = cy + q - 1;
        const bool ok = cr >= 0 && cr < g.ny, wraps = a > b;
        const uint32_t base = ((uint32_t)cr & (WY - 1u)) << LWX;
        const uint32_t s0 = tab[base + a], e0 = tab[base + (wraps ? WX : b + 1u)];
        const uint32_t s1 = tab[base], e1 = tab[base + b + 1u];
        my_from[2 * q] = s0;
        my_len[2 * q] = ok ? e0 - s0 : 0u;
        my_from[2 * q + 1] = s1;
        my_len[2 * q + 1] = ok && wraps ? e1 - s1 : 0u;
    }
    for (uint32_t q = 0; q < rows; ++q) {
        const int r = (int)lane_of(my_r, (int)q);
        const uint32_t rc = lane_of(my_c, (int)q);
        uint32_t at = lane_of(my_o, (int)q);
        const float xr = lane_of(my_x, (int)q), yr = lane_of(my_y, (int)q);
        if (rc <= 128u + (uint32_t)n / 48u) {
            uint32_t from[6], len[6];
#pragma unroll
            for (int w = 0; w < 6; ++w) {
                from[w] = lane_of(my_from[w], (int)q);
                len[w] = lane_of(my_len[w], (int)q);
            }
            small_gather_row<KIND>(n, x, y, m, order, r, xr, yr, from, len, rc, at, found[wave], pair_i, pair_j);
            continue;
        }
        const uint32_t end = at + rc;
        for (int j0 = r + 1; j0 < n && at < end; j0 += 64) {
            const int j = j0 + lane;
            const float xj = j < n ? x[j] : 0.0f, yj = j < n ? y[j] : 0.0f;
            const bool hit = pair_hit<KIND>(m, j < n, xr, yr, xj, yj);
            const uint64_t hits = __ballot(hit);
            if (hit) {
                const uint32_t k = at + (uint32_t)__popcll(hits & ((1ull << lane) - 1ull));
                if (k < end) {
                    pair_i[k] = r;
                    pair_j[k] = j;
                }
            }
            at += (uint32_t)__popcll(hits);
        }
    }
}

__global__ void zero_i64_kernel(int64_t* p, int64_t count) {
    for (int64_t k = threadIdx.x; k < count; k += blockDim.x) p[k] = 0;
}

}  // namespace lm

struct lm_pairs_ws {
    int64_t n_max = 0;
    int32_t steps_max = 0;
    double max_radius = 0.0;
    lm::CellGrid grid{};
    int64_t tab_stride = 0, row_stride = 0;
    uint32_t* keys[2] = {nullptr, nullptr};  // [steps][n_max] sort buffers
    uint32_t* vals[2] = {nullptr, nullptr};
    lm::SortScratch sort{};
    int key_bits = 0;              // log2(T)
    uint32_t* start = nullptr;     // [steps][tab]
    uint32_t* scan_tmp = nullptr;  // block sums
    float4* recs = nullptr;        // [steps][n_max]
    float2* xy = nullptr;          // [steps][n_max] positions interleaved, in index order
    uint32_t* nbr_cnt = nullptr;   // [steps][row]
    uint32_t* nbr = nullptr;       // [steps][n_max * kNbr]
    uint32_t* row_off = nullptr;   // [steps][row]
    uint32_t* small_tab = nullptr; // [steps][small_tab] bucket starts of a small population (its order: vals[0])
    int64_t bytes = 0;
};

static void pairs_ws_free(lm_pairs_ws* w) {
    if (!w) return;
    for (int q = 0; q < 2; ++q) {
        (void)hipFree(w->keys[q]);
        (void)hipFree(w->vals[q]);
    }
    lm::sort_scratch_free(&w->sort);
    (void)hipFree(w->start);
    (void)hipFree(w->scan_tmp);
    (void)hipFree(w->recs);
    (void)hipFree(w->xy);
    (void)hipFree(w->nbr_cnt);
    (void)hipFree(w->nbr);
    (void)hipFree(w->row_off);
    (void)hipFree(w->small_tab);
    delete w;
}

template <typename T>
static int ws_alloc(T** p, int64_t count, int64_t* bytes) {
    const size_t b = (size_t)(count < 1 ? 1 : count) * sizeof(T);
    hipError_t e = hipMalloc((void**)p, b);
    if (e != hipSuccess) {
        lm::set_error("hipMalloc(%zu) failed: %s", b, hipGetErrorString(e));
        return LM_ERR_NOMEM;
    }
    *bytes += (int64_t)b;
    return LM_OK;
}

static uint32_t next_pow2_u32(uint64_t v) {
    uint64_t p = 1;
    while (p < v) p <<= 1;
    return (uint32_t)p;
}

namespace lm {

// Phases 4-6 with the distance test of metric KIND.
template <int KIND>
static int count_and_emit(lm_pairs_ws* ws, int32_t nsteps, int64_t n, const float* lon, const float* lat,
                          const uint16_t* run, const CellGrid& g, const Metric& m, const Strides& st, int64_t* npairs,
                          int32_t* pair_i, int32_t* pair_j, hipStream_t s) {
    const dim3 grid(grid_for(n), (unsigned)nsteps);
    LM_LAUNCH(K_PAIR_COUNT, pair_count_kernel<KIND>, grid, dim3(kBlock), 0, s, n, g, m, st,
              (const uint32_t*)ws->start, (const float4*)ws->recs, ws->nbr_cnt, ws->nbr);
    LM_LAUNCH_CHECK();
    const int rc = exclusive_scan_u32_batched(ws->nbr_cnt, n, st.row, ws->row_off, st.row, nsteps, ws->scan_tmp,
                                              npairs, s);
    if (rc) return rc;
    LM_LAUNCH(K_PAIR_EMIT, pair_emit_kernel<KIND>, grid, dim3(kBlock), 0, s, n, lon, lat, run, g, m, st,
              (const uint32_t*)ws->start, (const float4*)ws->recs, (const uint32_t*)ws->nbr_cnt,
              (const uint32_t*)ws->nbr, (const uint32_t*)ws->row_off, pair_i, pair_j);
    LM_LAUNCH_CHECK();
    return LM_OK;
}

// Turns of 1,024 particles that a workgroup of the count takes, of the `blocks`
// of a step: binning the step again costs a workgroup about 12 us, a turn 10
// (12,288 particles), and kSmallFit workgroups run at once, one per CU.
constexpr int kSmallFit = 256;

static int small_turns(int64_t nsteps, int blocks) {
    int best = 1;
    int64_t least = INT64_MAX;
    for (int turns = 1; turns <= blocks; ++turns) {
        const int64_t rounds = (nsteps * ((blocks + turns - 1) / turns) + kSmallFit - 1) / kSmallFit;
        const int64_t cost = rounds * (6 + 5 * turns);
        if (cost < least) {
            least = cost;
            best = turns;
        }
    }
    return best;
}

// The search of a small population.  A table of 64 x 64 buckets up to 4,096
// particles, 128 x 64 above: about one particle in each.  Four lanes per
// particle while the workgroups they take still run at once (one fills a
// CU's LDS), else one; and as long as that holds, an emit of 256 rows per
// workgroup, which finds crowded rows four times as many at a time.  With one
// lane per particle and above 4,096 particles, where binning a step is as much
// work as searching for 1,024 of them, a step's workgroups each take several
// turns (see small_turns), and whole multiples of kSmallFit steps, a workgroup
// each, go out before the rest: 256 steps of 12,288 particles take 213 us, with
// a workgroup for every 1,024 particles 305 (the general kernels 236); 300
// steps 269, 363 (268); 64 steps 79, 95 (102).  4,096 particles, 300 steps: 104
// us with a workgroup per 1,024, 125 in turns.
template <int KIND, int NMAX, int LWX, int LWY>
static int search_small_table(lm_pairs_ws* ws, int32_t nsteps, int64_t n, const float* lon, const float* lat,
                              const CellGrid& g, const Metric& m, const Strides& st, int64_t* npairs, int32_t* pair_i,
                              int32_t* pair_j, hipStream_t s) {
    uint16_t* nbr = reinterpret_cast<uint16_t*>(ws->nbr);
    const bool wide = (n + kSmallBlock / 4 - 1) / (kSmallBlock / 4) * nsteps <= 256;
    const unsigned blocks = grid_for(n, wide ? kSmallBlock / 4 : kSmallBlock);
    const dim3 block(kSmallBlock);
    // steps [s0, s0 + ns), gx workgroups each
    auto count = [&](auto kernel, int32_t s0, int32_t ns, unsigned gx) {
        LM_LAUNCH(K_PAIR_SMALL, kernel, dim3(gx, (unsigned)ns), block, 0, s, (int)n, lon + s0 * st.pos,
                  lat + s0 * st.pos, g, m, st, ws->nbr_cnt + s0 * st.row, nbr + 2 * s0 * st.nbr,
                  ws->small_tab + s0 * small_tab(LWX + LWY), ws->vals[0] + s0 * st.rec);
    };
    auto emit = [&](auto kernel) {
        LM_LAUNCH(K_EMIT_SMALL, kernel, dim3(blocks, (unsigned)nsteps), block, 0, s, (int)n, lon, lat, g, m, st,
                  (const uint32_t*)ws->nbr_cnt, (const uint16_t*)nbr, (const uint32_t*)ws->small_tab,
                  (const uint16_t*)ws->vals[0], pair_i, pair_j, npairs);
    };
    if (wide) {
        count(pair_small_count_kernel<KIND, NMAX, LWX, LWY, 4>, 0, nsteps, blocks);
        LM_LAUNCH_CHECK();
        emit(pair_small_emit_kernel<KIND, LWX, LWY, kSmallBlock / 4>);
    } else {
        const bool in_turns = NMAX > kSmallTable;
        const int32_t even = in_turns ? nsteps / kSmallFit * kSmallFit : 0, rest = nsteps - even;
        if (even > 0) {
            count(pair_small_count_kernel<KIND, NMAX, LWX, LWY, 1>, 0, even, 1);
            LM_LAUNCH_CHECK();
        }
        if (rest > 0) {
            const unsigned turns = in_turns ? (unsigned)small_turns(rest, (int)blocks) : 1u;
            count(pair_small_count_kernel<KIND, NMAX, LWX, LWY, 1>, even, rest, (blocks + turns - 1) / turns);
            LM_LAUNCH_CHECK();
        }
        emit(pair_small_emit_kernel<KIND, LWX, LWY, kSmallBlock>);
    }
    LM_LAUNCH_CHECK();
    return LM_OK;
}

template <int KIND>
static int search_small(lm_pairs_ws* ws, int32_t nsteps, int64_t n, const float* lon, const float* lat,
                        const CellGrid& g, const Metric& m, const Strides& st, int64_t* npairs, int32_t* pair_i,
                        int32_t* pair_j, hipStream_t s) {
    if (n <= kSmallTable)
        return search_small_table<KIND, (int)kSmallTable, 6, 6>(ws, nsteps, n, lon, lat, g, m, st, npairs, pair_i, pair_j, s);
    return search_small_table<KIND, (int)kSmallMax, 7, 6>(ws, nsteps, n, lon, lat, g, m, st, npairs, pair_i, pair_j, s);
}

}  // namespace lm

extern "C" {

int lm_pairs_ws_create(int64_t n_max, int32_t steps_max, double lon_min, double lon_max, double lat_min,
                       double lat_max, double max_radius, lm_pairs_ws** out) {
    return lm_pairs_ws_create_ex(n_max, steps_max, lon_min, lon_max, lat_min, lat_max, max_radius, 1.0, out);
}

int lm_pairs_ws_create_ex(int64_t n_max, int32_t steps_max, double lon_min, double lon_max, double lat_min,
                          double lat_max, double max_radius, double cell_scale, lm_pairs_ws** out) {
    LM_REQUIRE(out != nullptr, LM_ERR_ARG, "out is NULL");
    *out = nullptr;
    LM_REQUIRE(n_max >= 0 && n_max < (int64_t)0x7fffffff, LM_ERR_ARG, "n_max out of range");
    LM_REQUIRE(steps_max >= 1 && steps_max <= 65535, LM_ERR_ARG, "steps_max must be in 1..65535");
    LM_REQUIRE(std::isfinite(lon_min) && std::isfinite(lon_max) && std::isfinite(lat_min) &&
                   std::isfinite(lat_max) && lon_max >= lon_min && lat_max >= lat_min,
               LM_ERR_ARG, "invalid bounding box");
    LM_REQUIRE(std::isfinite(max_radius) && max_radius > 0.0, LM_ERR_ARG, "max_radius must be > 0");
    LM_REQUIRE(std::isfinite(cell_scale) && cell_scale >= 1.0 && cell_scale <= 16.0, LM_ERR_ARG,
               "cell_scale must be in [1, 16]");

    lm_pairs_ws* w = new lm_pairs_ws();
    w->n_max = n_max;
    w->steps_max = steps_max;
    w->max_radius = max_radius;
    // cells strictly larger than the radius so rounding in the cell index can
    // never separate two points within the radius by more than one cell
    double h = max_radius * cell_scale * (1.0 + 1e-6);
    const double ext = (lon_max - lon_min) > (lat_max - lat_min) ? (lon_max - lon_min) : (lat_max - lat_min);
    if (ext / h > 30000.0) h = ext / 30000.0;
    lm::CellGrid& g = w->grid;
    g.inv_h = 1.0 / h;
    g.x0 = lon_min - h;
    g.y0 = lat_min - h;
    g.nx = (int32_t)std::floor((lon_max - lon_min) * g.inv_h) + 3;
    g.ny = (int32_t)std::floor((lat_max - lat_min) * g.inv_h) + 3;
    const uint64_t cells = (uint64_t)g.nx * (uint64_t)g.ny;
    // about two buckets per particle: fewer cells alias into a stencil's buckets
    uint64_t want = 2ull * (uint64_t)n_max;
    if (want < 4ull * (uint64_t)g.nx + 4) want = 4ull * (uint64_t)g.nx + 4;
    if (want < 1024) want = 1024;
    uint32_t T = next_pow2_u32(want);
    if ((uint64_t)T >= cells) T = next_pow2_u32(cells);
    if (T < 1024) T = 1024;
    // the binning splits a bucket key into at most 13 bits counted in LDS and one radix pass of at
    // most kMaxDigitBits: at most 2^23 buckets
    const uint32_t t_max = 1u << (13 + lm::kMaxDigitBits);
    if (T > t_max) T = t_max;
    g.T = T;
    g.mask = T - 1;
    g.cells = (uint32_t)((uint64_t)g.nx * (uint64_t)g.ny);
    w->tab_stride = lm::scan_row_stride((int64_t)T);
    w->row_stride = lm::scan_row_stride(n_max);

    const int64_t S = steps_max;
    int64_t nb = lm::scan_num_blocks((int64_t)T);
    const int64_t nb2 = lm::scan_num_blocks(n_max);
    if (nb2 > nb) nb = nb2;
    int rc = LM_OK;
    if ((rc = ws_alloc(&w->keys[0], S * n_max, &w->bytes)) || (rc = ws_alloc(&w->keys[1], S * n_max, &w->bytes)) ||
        (rc = ws_alloc(&w->vals[0], S * n_max, &w->bytes)) || (rc = ws_alloc(&w->vals[1], S * n_max, &w->bytes)) ||
        (rc = lm::sort_scratch_alloc(&w->sort, n_max, steps_max)) ||
        (rc = ws_alloc(&w->start, S * w->tab_stride, &w->bytes)) ||
        (rc = ws_alloc(&w->scan_tmp, S * nb, &w->bytes)) || (rc = ws_alloc(&w->recs, S * n_max, &w->bytes)) ||
        (rc = ws_alloc(&w->xy, S * n_max, &w->bytes)) ||
        (rc = ws_alloc(&w->nbr_cnt, S * w->row_stride, &w->bytes)) ||
        (rc = ws_alloc(&w->nbr, S * n_max * lm::kNbr, &w->bytes)) ||
        (rc = ws_alloc(&w->row_off, S * w->row_stride, &w->bytes)) ||
        (rc = ws_alloc(&w->small_tab, S * lm::small_tab(n_max <= lm::kSmallTable ? 12 : 13), &w->bytes))) {
        pairs_ws_free(w);
        return rc;
    }
    w->bytes += w->sort.bytes;
    while (((uint32_t)1 << w->key_bits) < T) ++w->key_bits;
    *out = w;
    return LM_OK;
}

void lm_pairs_ws_destroy(lm_pairs_ws* ws) { pairs_ws_free(ws); }

int64_t lm_pairs_ws_bytes(const lm_pairs_ws* ws) { return ws ? ws->bytes : 0; }

int64_t lm_pairs_ws_buckets(const lm_pairs_ws* ws) { return ws ? (int64_t)ws->grid.T : 0; }

int lm_query_pairs_batch(lm_pairs_ws* ws, int32_t nsteps, int64_t n, const float* lon, const float* lat,
                         int64_t pos_stride, double radius, double p, int32_t* pair_i, int32_t* pair_j,
                         int64_t pair_stride, int64_t* npairs, void* stream) {
    return lm_query_pairs_runs(ws, nsteps, n, lon, lat, pos_stride, nullptr, radius, p, pair_i, pair_j, pair_stride,
                               npairs, stream);
}

int lm_query_pairs_runs(lm_pairs_ws* ws, int32_t nsteps, int64_t n, const float* lon, const float* lat,
                        int64_t pos_stride, const uint16_t* run, double radius, double p, int32_t* pair_i,
                        int32_t* pair_j, int64_t pair_stride, int64_t* npairs, void* stream) {
    LM_REQUIRE(ws != nullptr, LM_ERR_ARG, "workspace is NULL");
    LM_REQUIRE(npairs != nullptr, LM_ERR_ARG, "npairs is NULL");
    LM_REQUIRE(nsteps >= 0 && nsteps <= ws->steps_max, LM_ERR_ARG, "nsteps=%d outside 0..%d of the workspace",
               nsteps, ws->steps_max);
    LM_REQUIRE(n >= 0 && n <= ws->n_max, LM_ERR_ARG, "n=%lld exceeds the workspace (n_max=%lld)",
               (long long)n, (long long)ws->n_max);
    LM_REQUIRE(radius >= 0.0 && radius <= ws->max_radius, LM_ERR_ARG,
               "radius %g outside [0, %g] of the workspace", radius, ws->max_radius);
    LM_REQUIRE(p >= 1.0, LM_ERR_ARG, "Minkowski p must be >= 1 (got %g)", p);
    LM_REQUIRE(pair_stride >= 0, LM_ERR_ARG, "negative pair capacity");
    LM_REQUIRE(nsteps <= 1 || pos_stride >= n, LM_ERR_ARG, "position stride < n");
    hipStream_t s = (hipStream_t)stream;
    if (nsteps == 0) return LM_OK;
    if (n == 0) {
        hipLaunchKernelGGL(lm::zero_i64_kernel, dim3(1), dim3(64), 0, s, npairs, (int64_t)nsteps);
        LM_LAUNCH_CHECK();
        return LM_OK;
    }
    LM_REQUIRE(lon && lat, LM_ERR_ARG, "NULL positions");
    LM_REQUIRE(pair_stride == 0 || (pair_i && pair_j), LM_ERR_ARG, "NULL pair buffers");

    lm::Metric m;
    m.r = radius;
    m.p = p;
    // above r by more than float32 rounding of a difference (2^-24 relative)
    m.box = std::nextafter((float)(radius * (1.0 + 1e-6)), INFINITY);
    m.sure_in = -INFINITY;
    m.sure_out = INFINITY;
    if (p == 2.0) {
        m.kind = lm::kL2;
        m.r2 = radius * radius;
        // far from float32 underflow and overflow, the float32 bounds of the
        // band around r^2 in which candidates take the float64 test
        if (m.r2 >= 1e-30 && m.r2 <= 1e30) {
            m.sure_in = std::nextafter((float)(m.r2 * (1.0 - 1e-6)), -INFINITY);
            m.sure_out = std::nextafter((float)(m.r2 * (1.0 + 1e-6)), INFINITY);
        }
    } else if (p == 1.0) {
        m.kind = lm::kL1;
        m.r2 = radius;
    } else if (std::isinf(p)) {
        m.kind = lm::kLinf;
        m.r2 = radius;
    } else {
        m.kind = lm::kLp;
        m.r2 = std::pow(radius, p);
    }
    const lm::CellGrid& g = ws->grid;
    lm::Strides st;
    st.pos = pos_stride;
    st.tab = ws->tab_stride;
    st.rec = ws->n_max;
    st.row = ws->row_stride;
    st.nbr = ws->n_max * lm::kNbr;
    st.pair = pair_stride;
    if (n <= lm::kSmallMax && run == nullptr) {
        switch (m.kind) {
            case lm::kL2: return lm::search_small<lm::kL2>(ws, nsteps, n, lon, lat, g, m, st, npairs, pair_i, pair_j, s);
            case lm::kL1: return lm::search_small<lm::kL1>(ws, nsteps, n, lon, lat, g, m, st, npairs, pair_i, pair_j, s);
            case lm::kLinf: return lm::search_small<lm::kLinf>(ws, nsteps, n, lon, lat, g, m, st, npairs, pair_i, pair_j, s);
            default: return lm::search_small<lm::kLp>(ws, nsteps, n, lon, lat, g, m, st, npairs, pair_i, pair_j, s);
        }
    }
    // two-level binning: one radix pass on the high bits of the bucket, then
    // a block per super-bucket sorts its fine buckets in LDS
    // 12 fine bits in LDS (13 above 2^22 buckets), the rest in one radix pass
    const int fine_bits = ws->key_bits <= 12 ? ws->key_bits : ws->key_bits <= 22 ? 12 : ws->key_bits - lm::kMaxDigitBits;
    const int super_bits = ws->key_bits - fine_bits;
    const dim3 grid(lm::grid_for(n), (unsigned)nsteps);
    // the particle indices are written only when no radix pass generates them
    LM_LAUNCH(lm::K_BIN_KEYS, lm::bin_keys_kernel, grid, dim3(lm::kBlock), 0, s, n, lon, lat, run, g, st,
              ws->keys[0], super_bits > 0 ? nullptr : ws->vals[0], ws->xy);
    LM_LAUNCH_CHECK();
    const uint32_t* dstart = nullptr;
    int64_t dstride = 0;
    int rc = LM_OK;
    int res = 0;
    if (super_bits > 0) {
        // unstable: the binning places a bucket's records in any order (the
        // pair list is sorted later), so no ranking of equal digits is needed
        rc = lm::radix_partition_u32(ws->keys, ws->vals, st.rec, nsteps, n, fine_bits, super_bits, &ws->sort, s,
                                     &dstart, &dstride, true, false);
        if (rc) return rc;
        res = 1;
    }
    if (fine_bits <= 12) {
        LM_LAUNCH(lm::K_BIN_TABLE, lm::bin_table_kernel<lm::kFineMax>, dim3(1u << super_bits, (unsigned)nsteps),
                  dim3(lm::kBlock), 0, s, n, (const float2*)ws->xy, run, g, st, (const uint32_t*)ws->keys[res],
                  (const uint32_t*)ws->vals[res], dstart, ws->sort.row, dstride, 1u << fine_bits, ws->start, ws->recs);
    } else {
        LM_LAUNCH(lm::K_BIN_TABLE, lm::bin_table_kernel<lm::kFineMaxWide>, dim3(1u << super_bits, (unsigned)nsteps),
                  dim3(lm::kBlock), 0, s, n, (const float2*)ws->xy, run, g, st, (const uint32_t*)ws->keys[res],
                  (const uint32_t*)ws->vals[res], dstart, ws->sort.row, dstride, 1u << fine_bits, ws->start, ws->recs);
    }
    LM_LAUNCH_CHECK();
    switch (m.kind) {
        case lm::kL2: rc = lm::count_and_emit<lm::kL2>(ws, nsteps, n, lon, lat, run, g, m, st, npairs, pair_i, pair_j, s); break;
        case lm::kL1: rc = lm::count_and_emit<lm::kL1>(ws, nsteps, n, lon, lat, run, g, m, st, npairs, pair_i, pair_j, s); break;
        case lm::kLinf:
            rc = lm::count_and_emit<lm::kLinf>(ws, nsteps, n, lon, lat, run, g, m, st, npairs, pair_i, pair_j, s);
            break;
        default: rc = lm::count_and_emit<lm::kLp>(ws, nsteps, n, lon, lat, run, g, m, st, npairs, pair_i, pair_j, s); break;
    }
    return rc;
}

int lm_query_pairs(lm_pairs_ws* ws, int64_t n, const float* lon, const float* lat, double radius, double p,
                   int32_t* pair_i, int32_t* pair_j, int64_t capacity, int64_t* npairs, void* stream) {
    return lm_query_pairs_batch(ws, 1, n, lon, lat, n, radius, p, pair_i, pair_j, capacity, npairs, stream);
}

}  // extern "C"
