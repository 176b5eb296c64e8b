// rg_line.hip -- weights along one axis: conservative 1-D and multilinear 1-D.
//
// Conservative 1-D (regridding/_weights/_weights_conservative_1d/
// _weights_conservative_1d.py:57-318): the sweep of the input vertices across
// the output vertices of each element (one line of the orthogonal stack).  A
// counting pass gives every (element, input cell) its number of triples;
// after a scan the emitting pass writes each triple straight to its position
// in the coalesced order (sorted by (input, output); every pair occurs once).
//
// Where both grids of an element are strictly monotonic, the sweep's state at
// every input vertex follows from one search of the output vertices, and all
// input cells are independent (k_line_count, k_line_emit, one thread per
// cell).  Any other element (repeated or unordered vertices, NaN) goes
// through the reference's state machine, replayed by one thread per element
// (sweep_1d), including its first-point search, and so do elements of a few
// vertices (short_elements).  Both reverse descending
// grids and emit the wraparound (negative) indices as the reference does.
// The state machine alone is a serial chain of one memory round trip per
// step on as many lanes as there are elements: 2048 elements of 2049 -> 1537
// vertices took 2.0 ms to count and 4.4 ms to emit.
//
// Multilinear 1-D (regridding/_weights/_weights_multilinear.py:148-206): two
// weights per output vertex from the searchsorted index, clamped and marked
// outside as in :95-118, in the reference's storage order.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "rg_internal.hpp"

namespace rg {

namespace {

// The grid of one element viewed ascending (the reference reverses
// descending grids, :88-102).
struct Axis {
    const double* x;
    int64_t n;
    bool rev;
    __device__ double operator()(int64_t k) const { return rev ? x[n - 1 - k] : x[k]; }
};

// _grids.py:40-73 index_of_point: bisection returning the right index.
__device__ int64_t index_of_point(double p, const Axis& g)
{
    int64_t lo = 0, hi = g.n;
    while (hi - lo > 1) {
        const int64_t mid = (lo + hi) / 2;
        if (g(mid) > p) hi = mid;
        else lo = mid;
    }
    return hi;
}

// numpy / numba wraparound of a negative index into an array of length n
__device__ inline int64_t wrap(int64_t i, int64_t n) { return i < 0 ? i + n : i; }

constexpr int64_t OUTSIDE = INT64_MAX;  // sys.maxsize

// The sweep of one element (_weights_conservative_1d.py:78-190).  Calls
// sink(index_input, index_output, ratio, piece) for every triple in the
// reference's order; `piece` counts the triples of the current input cell.
template <class Sink>
__device__ void sweep_1d(const double* xin, int64_t n, const double* xout, int64_t m,
                         const double* wi, Sink& sink)
{
    const Axis xs{xin, n, !(xin[0] < xin[n - 1])};
    const Axis xt{xout, m, !(xout[0] < xout[m - 1])};
    int64_t index_sweep = 0, k;
    double p1 = xs(0);
    bool outside;
    const double t_left = xt(0), t_right = xt(m - 1);
    if (t_left == p1) {
        outside = false;
        k = 0;
    } else if (t_left < p1 && p1 < t_right) {
        outside = false;
        k = index_of_point(p1, xt) - 1;
    } else {
        outside = true;
        k = OUTSIDE;
    }
    int64_t piece = 0, last_cell = -1;
    while (index_sweep < n - 1) {
        double p2 = xs(index_sweep + 1);
        if (outside) {  // _step_outside_static, :193-240
            const double ps = xt(0);
            if (p1 < ps && ps < p2) {
                k = 0;
                p2 = ps;
            } else if (ps == p2) {
                index_sweep++;
                k = 0;
            } else {
                index_sweep++;
            }
            if (k < OUTSIDE) outside = false;
        } else {  // _step_inside_static, :243-318
            int64_t index_input = xs.rev ? ~index_sweep : index_sweep;
            int64_t index_output = xt.rev ? ~k : k;
            const double ps = xt(k + 1);
            if (p1 < ps && ps < p2) {
                k++;
                p2 = ps;
            } else if (ps == p2) {
                k++;
                index_sweep++;
            } else {
                index_sweep++;
            }
            const double length = p2 - p1;
            // length_input comes from the ascending view (:112), indexed
            // with the emitted (possibly negative) input index
            const int64_t li = wrap(index_input, n - 1);
            double ratio = length / (xs(li + 1) - xs(li));
            if (wi) ratio = ratio * wi[li];
            if (li != last_cell) {
                last_cell = li;
                piece = 0;
            }
            sink(index_input, index_output, ratio, li, piece++);
            if (!(0 <= k && k < m - 1)) break;
        }
        p1 = p2;
    }
}

struct CountSink {
    int32_t* cnt;  // per input cell of the element
    __device__ void operator()(int64_t, int64_t, double, int64_t li, int64_t)
    {
        cnt[li]++;
    }
};

struct EmitSink {
    const int64_t* off;  // per input cell: first position (coalesced order)
    const int32_t* cnt;
    bool rev_out;
    int64_t* ii;
    int64_t* io;
    double* w;
    __device__ void operator()(int64_t in, int64_t out, double v, int64_t li,
                               int64_t piece)
    {
        // within an input cell the output index falls when the output grid
        // is descending (the emitted index is ~k): reverse the cell's run
        const int64_t p = off[li] + (rev_out ? cnt[li] - 1 - piece : piece);
        ii[p] = in;
        io[p] = out;
        w[p] = v;
    }
};

// ---- strictly monotonic elements, one thread per input cell ----------------
//
// A block takes LINE_CELLS input cells of one element and keeps the part of
// the output vertices they meet in LDS (LINE_OUT of them at most, otherwise
// they are searched in memory), so the searches, a chain of log2 steps each,
// wait on LDS only: first every 16th vertex in the whole part, then the others
// between their neighbours'.  The vertices' results are shared between the two
// cells of a vertex through LDS.  Each pass then moves little more than its
// arrays: count 2.0 ms -> 31 us, emit 4.4 ms -> 85 us at 2048
// elements of 2049 -> 1537 vertices (7.3 M triples).
constexpr int LINE_BLOCK = 256;
constexpr int LINE_CELLS = 1024;
constexpr int LINE_PER = LINE_CELLS / LINE_BLOCK;  // cells per thread
constexpr int LINE_COARSE = 16;
// 16 KiB, with the 4 KiB of results seven blocks per CU (five in the emit pass,
// whose entries take 8 KiB); an output grid of up
// to this size is staged whole, without a search for the part the block meets
// (two dependent memory round trips)
constexpr int LINE_OUT = 2048;

struct LineLds {
    double out[LINE_OUT];
    int32_t u[LINE_CELLS + 1];
    int32_t coarse[LINE_CELLS / LINE_COARSE + 1];
    int64_t range[2];
};

// #{k : xt(k) <= v} of ascending vertices by a whole wavefront: 64 of them
// compared per step.  (The state is a start and a length: written with two
// ends, both selected from 64-bit comparisons, the start came out selected by
// the other comparison's result.)
__device__ inline int64_t wave_upper_bound(double v, int64_t len, const Axis& xt)
{
    const int lane = threadIdx.x & 63;
    int64_t lo = 0, left = len;  // the answer is in [lo, lo + left]
    while (left > 0) {
        const int64_t step = (left + 63) / 64, q = (lane + 1) * step - 1;
        const bool below = q < left && xt(lo + (q < left ? q : left - 1)) <= v;
        const int64_t at = __popcll(__ballot(below)) * step;
        lo += at;
        left = left - at < step - 1 ? left - at : step - 1;
    }
    return lo;
}

// The output vertices of one block's cells: in LDS, or in memory.
struct OutRange {
    Axis g;
    const double* s;  // LDS copy of [base, base + len)
    int64_t base, len;
    bool staged;
    __device__ double operator()(int64_t k) const
    {
        const int64_t q = k - base;
        return staged && q >= 0 && q < len ? s[q] : g(k);
    }
};

// Shared start of both passes: the block's element and cells, the output
// vertices they meet, and for each of the cells' vertices 2 (u - base) + e
// with u = #{xt <= vertex} and e = 1 when a vertex of the output equals it.
// A vertex out of order (or NaN) in the element flags it for sweep_1d (where
// there are flags).
struct LineBlock {
    int64_t d, i0;  // element, first cell (ascending)
    int ncell;
    Axis xs;
    OutRange xt;

    // uniform over the block; every thread of the block takes part
    __device__ LineBlock(const double* xin, int64_t n, const double* xout, int64_t m,
                         int64_t nseg, int64_t block, int32_t* bad, LineLds& S)
    {
        const int tid = threadIdx.x;
        d = block / nseg;
        const int64_t seg = block - d * nseg;
        i0 = seg * LINE_CELLS;
        ncell = n - 1 - i0 < LINE_CELLS ? (int)(n - 1 - i0) : LINE_CELLS;
        const double* a = xin + d * n;
        const double* b = xout + d * m;
        xs = Axis{a, n, !(a[0] < a[n - 1])};
        const Axis g{b, m, !(b[0] < b[m - 1])};
        int64_t base = 0, end = m;
        if (m > LINE_OUT) {  // the part the cells meet, found by the first two wavefronts
            if (tid < 128) {
                const int64_t u = wave_upper_bound(xs(tid < 64 ? i0 : i0 + ncell), m, g);
                if ((tid & 63) == 0) S.range[tid >> 6] = u;
            }
            __syncthreads();
            // (an element out of order may give any range within [0, m])
            base = S.range[0] > 0 ? S.range[0] - 1 : 0;
            end = S.range[1] + 1 < m ? S.range[1] + 1 : m;
            if (end < base) end = base;
        }
        // (a range too long for the 32-bit results goes the serial way too)
        bool ok = end - base < ((int64_t)1 << 30);
        if (!ok) end = base;
        xt = OutRange{g, S.out, base, end - base, end - base <= LINE_OUT};
        const int len = (int)xt.len;
        // every load of the block in flight together
        double v[LINE_PER], r[LINE_PER], o[LINE_OUT / LINE_BLOCK], vc = 0;
#pragma unroll
        for (int t = 0; t < LINE_PER; t++) {
            const int q = tid + t * LINE_BLOCK;
            v[t] = r[t] = 0;
            if (q < ncell) {
                v[t] = xs(i0 + q);
                r[t] = xs(i0 + q + 1);
            }
        }
        const int qc = tid * LINE_COARSE < ncell ? tid * LINE_COARSE : ncell;
        if (tid <= LINE_CELLS / LINE_COARSE) vc = xs(i0 + qc);
        if (xt.staged) {
#pragma unroll
            for (int t = 0; t < LINE_OUT / LINE_BLOCK; t++)
                if (tid + t * LINE_BLOCK < len) o[t] = g(base + tid + t * LINE_BLOCK);
#pragma unroll
            for (int t = 0; t < LINE_OUT / LINE_BLOCK; t++)
                if (tid + t * LINE_BLOCK < len) S.out[tid + t * LINE_BLOCK] = o[t];
        }
        __syncthreads();
        // the order of the block's own input vertices, and of the output
        // vertices: all of them where they are staged whole, otherwise the
        // block's share of the element's
#pragma unroll
        for (int t = 0; t < LINE_PER; t++)
            if (tid + t * LINE_BLOCK < ncell) ok = ok && v[t] < r[t];
        if (m <= LINE_OUT) {
            for (int k = tid; k < len - 1; k += LINE_BLOCK) ok = ok && S.out[k] < S.out[k + 1];
        } else {
            const int64_t share = (m - 1 + nseg - 1) / nseg, k1 = (seg + 1) * share;
            for (int64_t k = seg * share + tid; k < k1 && k < m - 1; k += LINE_BLOCK)
                ok = ok && g(k) < g(k + 1);
        }
        if (!ok && bad) bad[d] = 1;
        const auto count = [&](double x, int lo, int hi) {  // #{xt <= x} in [lo, hi]
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if ((xt.staged ? S.out[mid] : g(base + mid)) <= x) lo = mid + 1;
                else hi = mid;
            }
            return lo;
        };
        if (tid <= LINE_CELLS / LINE_COARSE) S.coarse[tid] = count(vc, 0, len);
        __syncthreads();
        const auto vertex = [&](int q, double x, int next) {
            const int c = q / LINE_COARSE;
            int lo = S.coarse[c], hi = S.coarse[c + next];
            if (lo > hi) lo = hi;  // out of order
            const int u = count(x, lo, hi);
            S.u[q] = 2 * u + (u > 0 && (xt.staged ? S.out[u - 1] : g(base + u - 1)) == x ? 1 : 0);
        };
#pragma unroll
        for (int t = 0; t < LINE_PER; t++) {
            const int q = tid + t * LINE_BLOCK;
            if (q < ncell) vertex(q, v[t], 1);
            if (q == ncell - 1) {  // the last vertex: its own coarse entry, or past the cells'
                const int c = ncell / LINE_COARSE;
                const int u = ncell % LINE_COARSE ? S.coarse[c + 1] : S.coarse[c];
                S.u[ncell] = 2 * u + (u > 0 && (xt.staged ? S.out[u - 1] : g(base + u - 1)) == r[t]
                                          ? 1 : 0);
            }
        }
        __syncthreads();
    }

    // Pieces of cell q of the block: the output cells from the one that holds
    // its left end (*k0; the first one when it lies left of them all) to the
    // one that holds its right end.
    __device__ int64_t pieces(const LineLds& S, int q, int64_t m, int64_t* k0) const
    {
        const int64_t u0 = xt.base + (S.u[q] >> 1);
        const int64_t l1 = xt.base + (S.u[q + 1] >> 1) - (S.u[q + 1] & 1);  // #{xt < right end}
        *k0 = u0 > 0 ? u0 - 1 : 0;
        const int64_t last = l1 < m - 1 ? l1 : m - 1;
        return last > *k0 ? last - *k0 : 0;
    }
};

__global__ __launch_bounds__(LINE_BLOCK) void k_line_count(
    const double* __restrict__ xin, int64_t n, const double* __restrict__ xout, int64_t m,
    int64_t nseg, int64_t block0, int32_t* __restrict__ bad, int32_t* __restrict__ cnt)
{
    __shared__ LineLds S;
    const LineBlock L(xin, n, xout, m, nseg, block0 + blockIdx.x, bad, S);
    int32_t* c = cnt + L.d * (n - 1);
#pragma unroll
    for (int t = 0; t < LINE_PER; t++) {
        const int q = threadIdx.x + t * LINE_BLOCK;
        if (q >= L.ncell) break;
        int64_t k0;
        const int64_t i = L.i0 + q;
        c[L.xs.rev ? n - 2 - i : i] = (int32_t)L.pieces(S, q, m, &k0);
    }
}

// The block's cells hold one range of the entries.  A thread for each entry,
// LINE_ENTRIES at a time, finds its cell in LDS, so that entries are computed
// once each whatever their cells' counts (a wavefront of cells took the most
// of 64, three steps where the mean is 1.7) and each array is written by
// consecutive threads at consecutive entries, nontemporal: 99 -> 85 us at 2048
// elements of 2049 -> 1537 vertices (105 us with ordinary stores), of which 30
// are what the count pass takes too; it writes 175 MB, 2.1 TB/s.  Entries four at a time or
// starting at cache lines, and blocks of 512 cells or threads, measure the
// same.
constexpr int LINE_ENTRIES = 2 * LINE_CELLS;

__global__ __launch_bounds__(LINE_BLOCK) void k_line_emit(
    const double* __restrict__ xin, int64_t n, const double* __restrict__ xout, int64_t m,
    int64_t nseg, int64_t block0, int32_t* __restrict__ bad, const double* __restrict__ wi,
    const int64_t* __restrict__ off, int64_t* __restrict__ ii, int64_t* __restrict__ io,
    double* __restrict__ w)
{
    __shared__ LineLds S;
    __shared__ int32_t first[LINE_CELLS + 1];   // of each cell's entries, in storage order
    __shared__ uint16_t owner[LINE_ENTRIES];    // cell of each entry
    const LineBlock L(xin, n, xout, m, nseg, block0 + blockIdx.x, bad, S);
    const int64_t row = L.d * (n - 1);
    const int64_t l0 = row + (L.xs.rev ? n - 1 - L.i0 - L.ncell : L.i0);
    const int64_t e0 = off[l0];
#pragma unroll
    for (int t = 0; t <= LINE_PER; t++) {
        const int j = threadIdx.x + t * LINE_BLOCK;
        // (more entries than this only in an element out of order, which
        // sweep_1d writes again)
        if (j <= L.ncell) first[j] = (int32_t)min(off[l0 + j] - e0, (int64_t)INT32_MAX);
    }
    __syncthreads();
    const int32_t total = first[L.ncell];
    for (int64_t w0 = 0; w0 < total; w0 += LINE_ENTRIES) {
        const int32_t in_window = (int32_t)min(total - w0, (int64_t)LINE_ENTRIES);
#pragma unroll
        for (int t = 0; t < LINE_PER; t++) {
            const int j = threadIdx.x + t * LINE_BLOCK;
            if (j >= L.ncell) break;
            const int32_t a = (int32_t)max(first[j] - w0, (int64_t)0);
            const int32_t b = (int32_t)min(first[j + 1] - w0, (int64_t)in_window);
            for (int32_t e = a; e < b; e++) owner[e] = (uint16_t)j;
        }
        __syncthreads();
        for (int32_t e = threadIdx.x; e < in_window; e += LINE_BLOCK) {
            const int j = owner[e], q = L.xs.rev ? L.ncell - 1 - j : j;
            const int64_t i = L.i0 + q, at = w0 + e - first[j];
            int64_t k0;
            int64_t c = L.pieces(S, q, m, &k0);
            // (an element out of order stays in its counted range)
            if (c > first[j + 1] - first[j]) c = first[j + 1] - first[j];
            if (at >= c) continue;
            const int64_t k = L.xt.g.rev ? c - 1 - at : at;
            const double xl = L.xs(i), xr = L.xs(i + 1);
            // the reference divides by the ascending view's cell at the
            // emitted (wrapped) index
            const int64_t li = n - 2 - i;
            const double size = L.xs.rev ? L.xs(li + 1) - L.xs(li) : xr - xl;
            const bool leftmost = k == 0 && L.xt.base + (S.u[q] >> 1) > 0;
            const double p1 = leftmost ? xl : L.xt(k0 + k);
            const double ps = L.xt(k0 + k + 1);
            const double p2 = ps < xr ? ps : xr;
            double ratio = (p2 - p1) / size;
            if (wi) ratio = ratio * wi[l0 + j];
            const int64_t p = e0 + w0 + e;
            __builtin_nontemporal_store(L.xs.rev ? ~i : i, &ii[p]);
            __builtin_nontemporal_store(L.xt.g.rev ? ~(k0 + k) : k0 + k, &io[p]);
            __builtin_nontemporal_store(ratio, &w[p]);
        }
        __syncthreads();
    }
}

// ---- any other element (all of them, without flags) --------------------------

__global__ void k_cons1d_count(const double* __restrict__ xin, int64_t n,
                               const double* __restrict__ xout, int64_t m,
                               int64_t D, const int32_t* __restrict__ bad,
                               int32_t* __restrict__ cnt)
{
    const int64_t d = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (d >= D || (bad && !bad[d])) return;
    int32_t* c = cnt + d * (n - 1);
    for (int64_t i = 0; i < n - 1; i++) c[i] = 0;
    CountSink sink{c};
    sweep_1d(xin + d * n, n, xout + d * m, m, nullptr, sink);
}

__global__ void k_cons1d_emit(const double* __restrict__ xin, int64_t n,
                              const double* __restrict__ xout, int64_t m,
                              int64_t D, const int32_t* __restrict__ bad,
                              const double* __restrict__ wi,
                              const int64_t* __restrict__ off,
                              const int32_t* __restrict__ cnt,
                              int64_t* __restrict__ ii, int64_t* __restrict__ io,
                              double* __restrict__ w)
{
    const int64_t d = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (d >= D || (bad && !bad[d])) return;
    const double* xo = xout + d * m;
    EmitSink sink{off + d * (n - 1), cnt + d * (n - 1), !(xo[0] < xo[m - 1]), ii, io, w};
    sweep_1d(xin + d * n, n, xo, m, wi ? wi + d * (n - 1) : nullptr, sink);
}

// The same without flags, a block per element that looks its vertices over
// itself: for an emit under stream capture, whose replays find nothing of the
// call's own memory.
__global__ __launch_bounds__(LINE_BLOCK) void k_cons1d_emit_unordered(
    const double* __restrict__ xin, int64_t n, const double* __restrict__ xout, int64_t m,
    int64_t d0, const double* __restrict__ wi, const int64_t* __restrict__ off,
    const int32_t* __restrict__ cnt, int64_t* __restrict__ ii, int64_t* __restrict__ io,
    double* __restrict__ w)
{
    const int64_t d = d0 + blockIdx.x;
    const double* xi = xin + d * n;
    const double* xo = xout + d * m;
    const Axis a{xi, n, !(xi[0] < xi[n - 1])}, b{xo, m, !(xo[0] < xo[m - 1])};
    bool ok = m < ((int64_t)1 << 30);
    for (int64_t k = threadIdx.x; k < n - 1; k += LINE_BLOCK) ok = ok && a(k) < a(k + 1);
    for (int64_t k = threadIdx.x; k < m - 1; k += LINE_BLOCK) ok = ok && b(k) < b(k + 1);
    if (__syncthreads_and(ok) || threadIdx.x != 0) return;
    EmitSink sink{off + d * (n - 1), cnt + d * (n - 1), b.rev, ii, io, w};
    sweep_1d(xi, n, xo, m, wi ? wi + d * (n - 1) : nullptr, sink);
}

__global__ void k_multilinear_1d(const double* __restrict__ xin, int64_t n,
                                 const double* __restrict__ xout, int64_t m,
                                 int64_t D, const int64_t* __restrict__ index,
                                 const double* __restrict__ wi, int32_t bounds_nan,
                                 int64_t* __restrict__ ii, int64_t* __restrict__ io,
                                 double* __restrict__ w,
                                 unsigned long long* __restrict__ n_outside)
{
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (t >= D * m) return;
    const int64_t d = t / m, i = t - d * m;
    const double* x_in = xin + d * n;
    const double x = xout[t];
    const int64_t index_max = n - 2;
    const int64_t raw = index[t];
    const bool outside = raw < 0 || raw > index_max;
    if (outside) atomicAdd(n_outside, 1ull);
    const bool below = x < x_in[0];
    const int64_t i0 = below ? 0 : (raw < 0 ? 0 : (raw > index_max ? index_max : raw));
    const int64_t i1 = i0 + 1;
    const double x0 = x_in[i0], x1 = x_in[i1];
    double w1 = (x - x0) / (x1 - x0);
    double w0 = 1.0 - w1;
    if (wi) {
        w0 = w0 * wi[d * n + i0];
        w1 = w1 * wi[d * n + i1];
    }
    if (outside && bounds_nan) {
        w0 = __builtin_nan("");
        w1 = __builtin_nan("");
    }
    const int64_t base = d * 2 * m + 2 * i;
    ii[base] = i0;
    io[base] = i;
    w[base] = w0;
    ii[base + 1] = i1;
    io[base + 1] = i;
    w[base + 1] = w1;
}

// _weights_conservative_1d/_grids.py:11-37 cell_length, per element
__global__ void k_cell_length(const double* __restrict__ x, int64_t n, int64_t D,
                              double* __restrict__ out)
{
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (t >= D * (n - 1)) return;
    const int64_t d = t / (n - 1), i = t - d * (n - 1);
    out[t] = x[d * n + i + 1] - x[d * n + i];
}

__global__ void k_zero_flags(int32_t* __restrict__ p, int64_t n)
{
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

// Elements that one thread each sweeps sooner than a block each finds their
// cells: few vertices, more of them where the elements are many (a block costs
// 5.5 ns, what a thread's first 30 us are to 5000 elements), until the sweeps'
// scattered reads and writes outgrow the caches.  us for both passes, serial /
// by cells, D elements of n -> m vertices:
//   300: 9 -> 7 42 / 75, 17 -> 13 58 / 74, 33 -> 5 65 / 65, 33 -> 25 86 / 72
//   10^4: 33 -> 25 89 / 98, 2 -> 100 108 / 105, 17 -> 60 109 / 106, 60 -> 3 109 / 95
//   45000: 2 -> 100 159 / 318, 33 -> 25 224 / 295, 2 -> 200 291 / 340, 49 -> 37 332 / 312
//   10^5: 2 -> 200 561 / 692, 5 -> 60 360 / 644, 17 -> 13 316 / 581, 33 -> 5 384 / 552,
//     33 -> 25 784 / 605
//   10^6: 2 -> 50 1796 / 6062, 9 -> 50 6616 / 6439, 17 -> 13 4000 / 5840, 25 -> 19
//     6780 / 6096, 33 -> 25 9500 / 6199
bool short_elements(int64_t n, int64_t m, int64_t D)
{
    return D < 50000 ? 2 * n + m <= std::min<int64_t>(50 + D / 250, 150)
                     : (n + m) * std::min<int64_t>(n, 12) <= 600;
}

constexpr int64_t LINE_GRID = LAUNCH_THREADS / LINE_BLOCK;  // blocks per launch

int check_line(const double* xin, int64_t n, const double* xout, int64_t m, int64_t D)
{
    if (D < 0) return fail(RG_ERR_ARGUMENT, "negative element count");
    if (D > 0 && (!xin || !xout)) return fail(RG_ERR_ARGUMENT, "coordinate pointer is NULL");
    if (n < 2 || m < 2) return fail(RG_ERR_ARGUMENT, "each grid needs at least 2 vertices");
    return RG_OK;
}

}  // namespace

}  // namespace rg

using namespace rg;

extern "C" {

int rg_conservative_1d_count(const double* x_input, int64_t n_input,
                             const double* x_output, int64_t n_output, int64_t D,
                             int32_t* counts, int64_t* offsets, int64_t* total,
                             void* stream)
{
    RG_TRY(check_line(x_input, n_input, x_output, n_output, D));
    if (!counts || !offsets || !total) return fail(RG_ERR_ARGUMENT, "NULL output");
    hipStream_t s = (hipStream_t)stream;
    *total = 0;
    const int64_t cells = D * (n_input - 1);
    if (cells == 0) return RG_OK;
    DevBuf<int32_t> bad;
    if (!short_elements(n_input, n_output, D)) {
        const int64_t nseg = (n_input - 1 + LINE_CELLS - 1) / LINE_CELLS, blocks = D * nseg;
        RG_TRY(bad.alloc(D, s));
        k_zero_flags<<<grid_for(D, 256), 256, 0, s>>>(bad.p, D);
        for (int64_t b = 0; b < blocks; b += LINE_GRID)
            k_line_count<<<(unsigned)std::min(blocks - b, LINE_GRID), LINE_BLOCK, 0, s>>>(
                x_input, n_input, x_output, n_output, nseg, b, bad.p, counts);
    }
    k_cons1d_count<<<grid_for(D, 64), 64, 0, s>>>(x_input, n_input, x_output,
                                                   n_output, D, bad.p, counts);
    RG_HIP(hipGetLastError());
    RG_TRY(scan_i32_to_i64(counts, offsets, cells, s));
    RG_TRY(read_scalars(offsets + cells, total, sizeof(int64_t), s));
    return RG_OK;
}

int rg_conservative_1d_emit(const double* x_input, int64_t n_input,
                            const double* x_output, int64_t n_output, int64_t D,
                            const double* weights_input, const int32_t* counts,
                            const int64_t* offsets, int64_t* indices_input,
                            int64_t* indices_output, double* values, void* stream)
{
    RG_TRY(check_line(x_input, n_input, x_output, n_output, D));
    if (D == 0) return RG_OK;
    if (!counts || !offsets || !indices_input || !indices_output || !values)
        return fail(RG_ERR_ARGUMENT, "NULL array");
    hipStream_t s = (hipStream_t)stream;
    DevBuf<int32_t> bad;
    const bool by_cells = !short_elements(n_input, n_output, D);
    if (by_cells) {
        const int64_t nseg = (n_input - 1 + LINE_CELLS - 1) / LINE_CELLS, blocks = D * nseg;
        if (!capturing(s)) {
            RG_TRY(bad.alloc(D, s));
            k_zero_flags<<<grid_for(D, 256), 256, 0, s>>>(bad.p, D);
        }
        for (int64_t b = 0; b < blocks; b += LINE_GRID)
            k_line_emit<<<(unsigned)std::min(blocks - b, LINE_GRID), LINE_BLOCK, 0, s>>>(
                x_input, n_input, x_output, n_output, nseg, b, bad.p, weights_input, offsets,
                indices_input, indices_output, values);
    }
    if (by_cells && !bad.p)
        for (int64_t d = 0; d < D; d += LINE_GRID)
            k_cons1d_emit_unordered<<<(unsigned)std::min(D - d, LINE_GRID), LINE_BLOCK, 0, s>>>(
                x_input, n_input, x_output, n_output, d, weights_input, offsets, counts,
                indices_input, indices_output, values);
    else
        k_cons1d_emit<<<grid_for(D, 64), 64, 0, s>>>(x_input, n_input, x_output, n_output,
                                                      D, bad.p, weights_input, offsets, counts,
                                                      indices_input, indices_output, values);
    RG_HIP(hipGetLastError());
    return RG_OK;
}

int rg_cell_length_1d(const double* x, int64_t n, int64_t D, double* length,
                      void* stream)
{
    if (D < 0 || n < 2) return fail(RG_ERR_ARGUMENT, "need D >= 0 elements of >= 2 vertices");
    if (D == 0) return RG_OK;
    if (!x || !length) return fail(RG_ERR_ARGUMENT, "NULL array");
    hipStream_t s = (hipStream_t)stream;
    k_cell_length<<<grid_for(D * (n - 1), 256), 256, 0, s>>>(x, n, D, length);
    RG_HIP(hipGetLastError());
    return RG_OK;
}

int rg_multilinear_1d(const double* x_input, int64_t n_input, const double* x_output,
                      int64_t n_output, int64_t D, const int64_t* indices,
                      const double* weights_input, int32_t bounds_nan,
                      int64_t* indices_input, int64_t* indices_output, double* values,
                      int64_t* n_outside, void* stream)
{
    RG_TRY(check_line(x_input, n_input, x_output, n_output, D));
    if (!n_outside) return fail(RG_ERR_ARGUMENT, "n_outside is NULL");
    *n_outside = 0;
    const int64_t total = D * n_output;
    if (total == 0) return RG_OK;
    if (!indices || !indices_input || !indices_output || !values)
        return fail(RG_ERR_ARGUMENT, "NULL array");
    hipStream_t s = (hipStream_t)stream;
    DevBuf<unsigned long long> cnt;
    RG_TRY(cnt.alloc(1, s));
    RG_HIP(hipMemsetAsync(cnt.p, 0, sizeof(unsigned long long), s));
    k_multilinear_1d<<<grid_for(total, 256), 256, 0, s>>>(
        x_input, n_input, x_output, n_output, D, indices, weights_input, bounds_nan,
        indices_input, indices_output, values, cnt.p);
    RG_HIP(hipGetLastError());
    unsigned long long h = 0;
    RG_TRY(read_scalars(cnt.p, &h, sizeof(h), s));
    *n_outside = (int64_t)h;
    return RG_OK;
}

}  // extern "C"
