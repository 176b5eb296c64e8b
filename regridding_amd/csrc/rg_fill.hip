// rg_fill.hip -- the reference's companions of the regrid: filling missing
// values by red-black Gauss-Seidel relaxation and linear interpolation of an
// array at fractional indices.
//
// Red-black Gauss-Seidel (regridding/_fill/_gauss_seidel.py:83-139).  The
// reference sweeps each colour row-major with periodic neighbours.  Within
// one colour a cell's neighbours have the other colour -- except across the
// periodic wrap when a dimension is odd: cells (j, 0) and (j, nx-1) then
// share a colour (likewise (0, i) and (ny-1, i)), and the sequential sweep
// updates the later one from the already-updated earlier one.  Every such
// pair has exactly one "late" member (last column for odd nx, last row for
// odd ny), so a colour is applied in steps that give the sequential sweep's
// result exactly:
//   1. every non-late cell of the colour, in parallel: a same-colour
//      neighbour of one is late, and still holds its old value in the
//      sequential sweep too;
//   2. every late cell but the corner (ny-1, nx-1), in parallel: their
//      same-colour neighbours are non-late (already new, as in the sweep)
//      or the corner (still old, as in the sweep);
//   3. the corner, when both dimensions are odd: its same-colour neighbours
//      (0, nx-1) and (ny-1, 0) are late and already new.
// Only the masked cells change, so a workgroup lists those of its part, by
// colour and step, and keeps each thread's share of the lists in registers.
// A slice of up to GS_LDS_CELLS cells runs every iteration in one workgroup
// in LDS (k_gs_lds).  A larger one runs GS_ITER iterations per launch in
// tiles with a halo (k_gs_tile); thin slices too large for the LDS, and calls
// under stream capture or without room for the second buffer, take one launch
// per step (k_gs_color, k_gs_late).
//
// Linear interpolation (regridding/_interp_ndarray.py:172-269): one lane per
// output point, clamped linear / bilinear weights.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "rg_internal.hpp"

namespace rg {

namespace {

struct GsCoef {
    double dxxinv, dyyinv, dcent;
};

// _gauss_seidel.py:110-122
GsCoef gs_coef(int64_t nx, int64_t ny)
{
    const double xmin = -1, xmax = 1, ymin = -1, ymax = 1;
    const double dx = (xmax - xmin) / (double)(nx - 1);
    const double dy = (ymax - ymin) / (double)(ny - 1);
    GsCoef c;
    c.dxxinv = 1 / (dx * dx);
    c.dyyinv = 1 / (dy * dy);
    c.dcent = 1 / (2 * (c.dxxinv + c.dyyinv));
    return c;
}

// _gauss_seidel.py:124-139: one cell
__device__ inline void gs_cell(double* __restrict__ a, int64_t nx, int64_t ny,
                               int64_t j, int64_t i, GsCoef c)
{
    const int64_t i9 = (i - 1 + nx) % nx, i1 = (i + 1) % nx;
    const int64_t j9 = (j - 1 + ny) % ny, j1 = (j + 1) % ny;
    const double xterm = c.dxxinv * (a[j * nx + i9] + a[j * nx + i1]);
    const double yterm = c.dyyinv * (a[j9 * nx + i] + a[j1 * nx + i]);
    a[j * nx + i] = (xterm + yterm) * c.dcent;
}

__device__ inline bool late_cell(int64_t j, int64_t i, int64_t nx, int64_t ny)
{
    return ((nx & 1) && i == nx - 1) || ((ny & 1) && j == ny - 1);
}

__global__ void k_gs_color(double* __restrict__ a, const uint8_t* __restrict__ where,
                           int64_t T, int64_t ny, int64_t nx, int parity, GsCoef c)
{
    const int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (q >= T * ny * nx) return;
    const int64_t t = q / (ny * nx), r = q - t * ny * nx;
    const int64_t j = r / nx, i = r - j * nx;
    if (((i + j) & 1) != parity || !where[q] || late_cell(j, i, nx, ny)) return;
    gs_cell(a + t * ny * nx, nx, ny, j, i, c);
}

// number of late cells other than the corner: the last column (odd nx),
// the last row (odd ny); the corner is counted separately when both are odd
__host__ __device__ inline int64_t n_late(int64_t ny, int64_t nx)
{
    const int64_t lx = nx & 1, ly = ny & 1;
    return lx * (ny - ly) + ly * (nx - lx);
}

__device__ inline void late_cell_at(int64_t q, int64_t ny, int64_t nx, int64_t& j, int64_t& i)
{
    const int64_t lx = nx & 1, ly = ny & 1;
    const int64_t ncol = lx * (ny - ly);
    if (q < ncol) {
        j = q;
        i = nx - 1;
    } else {
        j = ny - 1;
        i = q - ncol;
    }
}

// steps 2 and 3 for one slice per workgroup
__global__ void k_gs_late(double* __restrict__ a, const uint8_t* __restrict__ where,
                          int64_t ny, int64_t nx, int parity, GsCoef c)
{
    double* at = a + blockIdx.x * ny * nx;
    const uint8_t* wt = where + blockIdx.x * ny * nx;
    const int64_t nl = n_late(ny, nx);
    for (int64_t q = threadIdx.x; q < nl; q += blockDim.x) {
        int64_t j, i;
        late_cell_at(q, ny, nx, j, i);
        if (((i + j) & 1) == parity && wt[j * nx + i]) gs_cell(at, nx, ny, j, i, c);
    }
    if ((nx & 1) && (ny & 1)) {
        __syncthreads();
        const int64_t j = ny - 1, i = nx - 1;
        if (threadIdx.x == 0 && ((i + j) & 1) == parity && wt[j * nx + i])
            gs_cell(at, nx, ny, j, i, c);
    }
}

constexpr int GS_BLOCK = 512;

// The step of a cell within its colour: 0, 1 or 2 (steps 1-3 above).
__device__ inline int gs_step(int j, int i, int nx, int ny)
{
    return ((nx & 1) && i == nx - 1 ? 1 : 0) + ((ny & 1) && j == ny - 1 ? 1 : 0);
}

// Appends `entry` to list[0 .. *n) (LDS) from the lanes with `take`: one
// atomic per wavefront.
template <class E>
__device__ inline void gs_append(E* list, int32_t* n, bool take, E entry, int lane)
{
    const uint64_t m = __ballot(take);
    if (m == 0) return;
    int32_t at = 0;
    if (lane == 0) at = atomicAdd(n, __popcll(m));
    at = __shfl(at, 0, 64);
    if (take) list[at + __popcll(m & (((uint64_t)1 << lane) - 1))] = entry;
}

// ---- whole slices in LDS ---------------------------------------------------
//
// The lists are made in the LDS that the values take afterwards (the thread's
// share waits in registers), so a slice holds 8 bytes of LDS per cell.  An
// entry is the cell (13 bits) and which of its neighbours lie across the
// periodic wrap (4 bits).  Every thread visiting every cell of both colours,
// with 64-bit remainders for its neighbours, 100 iterations of 3 slices of 58
// x 43 took 692 us (4 % masked) and 752 (all); now 84 and 120.  Slices of one row
// or column (their cells are their own neighbours across it, and all late) fit
// the same lists: one of 1 x 1000 72 us, 1.5 ms in a launch per step.
constexpr int GS_LDS_CELLS = 8192;
constexpr int GS_LDS_PER = GS_LDS_CELLS / 2 / GS_BLOCK;  // cells per thread and colour
// Slices of up to GS_SMALL_CELLS take a wavefront each, whose steps need no
// barrier across wavefronts: 10^5 slices of 8 x 8 0.78 ms (7.1 in blocks of 512),
// of 16 x 16 all masked 1.42 (7.6); one of 16 x 16 45 us (37).
constexpr int GS_SMALL_BLOCK = 64, GS_SMALL_CELLS = 256;
static_assert(GS_SMALL_CELLS / 2 <= GS_SMALL_BLOCK * GS_LDS_PER, "a thread's cells");

// every cell of one slice of ny x nx <= GS_LDS_CELLS
template <int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_gs_lds(double* __restrict__ a,
                                                  const uint8_t* __restrict__ where, int ny,
                                                  int nx, int64_t num_iterations, GsCoef c)
{
    extern __shared__ double s[];
    __shared__ int32_t cnt[3];
    const int cells = ny * nx, tid = threadIdx.x, lane = tid & 63;
    uint32_t* list = reinterpret_cast<uint32_t*>(s);          // colour 0 from the front,
    uint32_t* list1 = list + cells;                           // colour 1 from the middle
    uint32_t* late = reinterpret_cast<uint32_t*>(s + cells);  // past the values
    double* at = a + (int64_t)blockIdx.x * cells;
    const uint8_t* wt = where + (int64_t)blockIdx.x * cells;
    if (tid < 3) cnt[tid] = 0;
    __syncthreads();
    for (int q0 = 0; q0 < cells; q0 += BLOCK) {  // uniform
        const int q = q0 + tid;
        const int j = (unsigned)q / (unsigned)nx, i = q - j * nx;
        const bool in = q < cells && wt[q];
        const int step = in ? gs_step(j, i, nx, ny) : 0;
        const uint32_t e = (uint32_t)q | (i == 0 ? 1u << 13 : 0) | (i == nx - 1 ? 1u << 14 : 0) |
                           (j == 0 ? 1u << 15 : 0) | (j == ny - 1 ? 1u << 16 : 0);
        const int colour = (i + j) & 1;
        gs_append(list, &cnt[0], in && step == 0 && colour == 0, e, lane);
        gs_append(list1, &cnt[1], in && step == 0 && colour == 1, e, lane);
        gs_append(late, &cnt[2], in && step > 0,
                  e | (uint32_t)colour << 17 | (uint32_t)step << 18, lane);
    }
    __syncthreads();
    const int n0 = cnt[0], n1 = cnt[1], nl = cnt[2];
    if (n0 + n1 + nl == 0) return;  // uniform
    uint32_t e0[GS_LDS_PER], e1[GS_LDS_PER];
#pragma unroll
    for (int t = 0; t < GS_LDS_PER; t++) {
        const int k = tid + t * BLOCK;
        e0[t] = k < n0 ? list[k] : 0;
        e1[t] = k < n1 ? list1[k] : 0;
    }
    __syncthreads();
    for (int q = tid; q < cells; q += BLOCK) s[q] = at[q];
    __syncthreads();
    const auto update = [&](uint32_t e) {
        const int q = e & 8191;
        const double xterm = c.dxxinv * (s[e >> 13 & 1 ? q + nx - 1 : q - 1] +
                                         s[e >> 14 & 1 ? q - nx + 1 : q + 1]);
        const double yterm = c.dyyinv * (s[e >> 15 & 1 ? q + cells - nx : q - nx] +
                                         s[e >> 16 & 1 ? q - cells + nx : q + nx]);
        s[q] = (xterm + yterm) * c.dcent;
    };
    const int steps = nl ? (nx & 1) + (ny & 1) : 0;
    for (int64_t k = 0; k < num_iterations; k++) {
#pragma unroll
        for (int colour = 0; colour < 2; colour++) {
            const int n = colour ? n1 : n0;
#pragma unroll
            for (int t = 0; t < GS_LDS_PER; t++)
                if (tid + t * BLOCK < n) update(colour ? e1[t] : e0[t]);
            __syncthreads();
            for (int step = 1; step <= steps; step++) {
                for (int q = tid; q < nl; q += BLOCK)
                    if (late[q] >> 17 == (uint32_t)(colour | step << 1)) update(late[q]);
                __syncthreads();
            }
        }
    }
    for (int q = tid; q < cells; q += BLOCK) at[q] = s[q];
}

// ---- tiles -------------------------------------------------------------------
//
// A workgroup holds a tile of GS_H x GS_W cells (periodic) in LDS and runs up
// to GS_ITER iterations on it.  A colour reaches one cell, and one more where
// it crosses an odd edge (a late cell reads a cell of its own colour there;
// with at least GS_MIN cells an axis the halo crosses at most two edges), so
// after k iterations what the tile's rim lacks has come 2 k + 2 cells in at
// most: the halo.  The interior is written to a second buffer; the number of
// launches is even, so the last one writes the caller's.  The first launch
// makes the tiles' lists and writes every cell, the others read the lists and
// write the masked cells; a tile without any ends at once.
//
// One launch per colour and step (k_gs_color, k_gs_late) read the whole array
// and its mask 200 times for 100 iterations, with 64-bit divisions per cell.
// 100 iterations on 4 slices: 768 x 1001, 4 % masked, 3.46 -> 0.44 ms; 768 x
// 1000 all masked 2.76 -> 0.78 ms; one slice of 400 x 401 1.31 -> 0.16 ms.
// What bounds a launch now is reading the tiles (25 us of about 29 at 768 x
// 1000; two workgroups per CU, one's loads beside the other's steps).  Tiles
// twice as high with 13 iterations a launch (one workgroup per CU) took
// 0.45-0.57 ms where these took 0.52-0.62, and 0.90 against 0.89 all masked,
// before the lists were kept; 96 x 96 tiles 0.68 ms (divisions by 96).
constexpr int GS_W = 128, GS_H = 72;  // columns, rows
constexpr int GS_ITER = 8;
constexpr int GS_HALO = 2 * GS_ITER + 2;
constexpr int GS_IN_W = GS_W - 2 * GS_HALO, GS_IN_H = GS_H - 2 * GS_HALO;
constexpr int GS_MIN = 16;
constexpr int GS_CELLS = GS_W * GS_H;
constexpr int GS_WAVES = GS_BLOCK / 64;
constexpr int GS_ROWS = GS_H / GS_WAVES;         // rows loaded per wavefront
constexpr int GS_OWN = 2 * GS_ROWS;              // cells loaded per thread
constexpr int GS_PER = GS_CELLS / 2 / GS_BLOCK;  // cells updated per thread and colour
// late cells of a tile: an odd edge comes every 17 cells at least
constexpr int GS_LATE = GS_H * (GS_W / (GS_MIN + 1) + 1) + GS_W * (GS_H / (GS_MIN + 1) + 1);
constexpr int GS_HALF = GS_W / 2, GS_PLANE = GS_CELLS / 2;
static_assert(GS_W == 128 && GS_H % GS_WAVES == 0, "two cells of a row per lane");
static_assert(GS_CELLS % (2 * GS_BLOCK) == 0 && GS_CELLS <= 1 << 14, "lists and their entries");

struct GsTileLds {
    double v[GS_CELLS];  // (first the lists are made here)
    uint32_t late[GS_LATE];
    uint32_t wave[GS_WAVES];  // list entries of each wavefront
    int32_t late_n;
};
static_assert(2 * sizeof(GsTileLds) <= 160 * 1024, "two workgroups per CU");

// Cell (r, k) of a tile: the cells of each colour of the tile sit together,
// row by row, so that the lanes of an update, which take every other cell of
// a row, read consecutive words (in a row-major tile two lanes share a bank).
__device__ inline int gs_place(int r, int k)
{
    return ((r + k) & 1) * GS_PLANE + r * GS_HALF + (k >> 1);
}

// A list entry of a tile: the place (14 bits) and the column's parity; a late
// cell's has its colour and step at bit 17.
__device__ inline uint32_t gs_entry(int r, int k)
{
    return (uint32_t)gs_place(r, k) | (uint32_t)(k & 1) << 14;
}

__device__ inline void gs_update(double* v, uint32_t e, GsCoef c)
{
    const int q = e & 0x3fff;
    const int o = q < GS_PLANE ? q + GS_PLANE : q - GS_PLANE;  // the same place, other colour
    const int l = o - 1 + (int)(e >> 14 & 1);
    const double xterm = c.dxxinv * (v[l] + v[l + 1]);
    const double yterm = c.dyyinv * (v[o - GS_HALF] + v[o + GS_HALF]);
    v[q] = (xterm + yterm) * c.dcent;
}

__device__ inline int gs_wrap(int i, int n)
{
    i %= n;
    return i < 0 ? i + n : i;
}

// The lists of a tile, kept for the launches after the first: colour 0 from
// the front of `cell`, colour 1 from its end.
struct GsTileLists {
    uint16_t cell[GS_CELLS];
    uint32_t late[GS_LATE];
    int32_t n0, n1, nl;
};

// `first`: makes the tile's lists, writes every cell of the interior to dst.
// Otherwise the lists are there, and only the masked cells are written.
// (two workgroups of eight wavefronts per CU: at most 128 registers)
template <bool first>
__global__ __launch_bounds__(GS_BLOCK, 4) void k_gs_tile(
    const double* __restrict__ src, double* __restrict__ dst, const uint8_t* __restrict__ where,
    GsTileLists* __restrict__ lists, int ny, int nx, int ntx, int nty, int iterations, GsCoef c)
{
    extern __shared__ double gs_lds[];
    GsTileLds& S = *reinterpret_cast<GsTileLds*>(gs_lds);
    // wavefront w takes rows w, w + 8, ... of the tile, lane l their columns
    // l and l + 64
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    GsTileLists& L = lists[blockIdx.x];
    int n0 = 0, n1 = 0, nl = 0;
    if (!first) {
        n0 = L.n0;
        n1 = L.n1;
        nl = L.nl;
        if (n0 + n1 + nl == 0) return;  // uniform; dst holds the tile already
    }
    const unsigned per = (unsigned)(ntx * nty);
    const int64_t t = blockIdx.x / per;
    const int tile = (int)(blockIdx.x - t * per), ty = tile / ntx, tx = tile - ty * ntx;
    const int64_t base = t * ny * nx;
    const int j0 = ty * GS_IN_H, i0 = tx * GS_IN_W;  // the interior's first cell
    const int ci[2] = {gs_wrap(i0 - GS_HALO + lane, nx), gs_wrap(i0 - GS_HALO + lane + 64, nx)};
    // the tile's values and its mask or lists, all loads in flight together
    double v[GS_OWN];
    uint8_t w8[GS_OWN];
    uint32_t e0[GS_PER], e1[GS_PER];
    int rj[GS_ROWS];  // the rows in the slice (wave-uniform)
#pragma unroll
    for (int u = 0; u < GS_ROWS; u++) {
        rj[u] = gs_wrap(j0 - GS_HALO + wave + u * GS_WAVES, ny);
        if (!first) continue;
#pragma unroll
        for (int h = 0; h < 2; h++) w8[2 * u + h] = where[base + (int64_t)rj[u] * nx + ci[h]];
    }
#pragma unroll
    for (int u = 0; u < GS_ROWS; u++)
#pragma unroll
        for (int h = 0; h < 2; h++) v[2 * u + h] = src[base + (int64_t)rj[u] * nx + ci[h]];
    if (!first) {
#pragma unroll
        for (int u = 0; u < GS_PER; u++) {
            const int k = tid + u * GS_BLOCK;
            e0[u] = k < n0 ? L.cell[k] : 0;
            e1[u] = k < n1 ? L.cell[GS_CELLS - 1 - k] : 0;
        }
        for (int k = tid; k < nl; k += GS_BLOCK) S.late[k] = L.late[k];
    } else {
        if (tid == 0) S.late_n = 0;
        __syncthreads();
        // which of the thread's cells are masked and not on the rim, and
        // which of those are of colour 1; the few late cells are listed apart
        uint32_t in = 0, second = 0;
        const bool rim_h[2] = {lane == 0, lane == 63};
#pragma unroll
        for (int u = 0; u < GS_ROWS; u++) {
            const int r = wave + u * GS_WAVES;
            const bool rim_r = r == 0 || r == GS_H - 1;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int b = 2 * u + h, colour = (rj[u] + ci[h]) & 1;
                bool take = w8[b] != 0 && !rim_r && !rim_h[h];
                const int step = gs_step(rj[u], ci[h], nx, ny);
                if (take && step > 0) {
                    take = false;
                    S.late[atomicAdd(&S.late_n, 1)] = gs_entry(r, lane + 64 * h) |
                                                      (uint32_t)colour << 17 |
                                                      (uint32_t)step << 18;
                }
                in |= (uint32_t)take << b;
                second |= (uint32_t)(take && colour) << b;
                n0 += __popcll(__ballot(take && !colour));
                n1 += __popcll(__ballot(take && colour));
            }
        }
        if (lane == 0) S.wave[wave] = (uint32_t)n0 | (uint32_t)n1 << 16;
        __syncthreads();
        uint32_t before = 0, all = 0;
#pragma unroll
        for (int w = 0; w < GS_WAVES; w++) {
            const uint32_t x = S.wave[w];
            before += w < wave ? x : 0;
            all += x;
        }
        n0 = all & 0xffff;
        n1 = all >> 16;
        nl = S.late_n;
        // each wavefront's cells in order (listed thread by thread,
        // neighbours in a list would be rows apart and collide in the banks)
        int p0 = before & 0xffff, p1 = before >> 16;
        const uint64_t lower = ((uint64_t)1 << lane) - 1;
        uint16_t* list = reinterpret_cast<uint16_t*>(S.v);
#pragma unroll
        for (int b = 0; b < GS_OWN; b++) {
            const uint16_t e =
                (uint16_t)gs_entry(wave + (b >> 1) * GS_WAVES, lane + 64 * (b & 1));
            const bool y = second >> b & 1, x = (in >> b & 1) && !y;
            const uint64_t m0 = __ballot(x), m1 = __ballot(y);
            if (x) list[p0 + __popcll(m0 & lower)] = e;
            if (y) list[GS_CELLS - 1 - p1 - __popcll(m1 & lower)] = e;
            p0 += __popcll(m0);
            p1 += __popcll(m1);
        }
        if (tid == 0) {
            L.n0 = n0;
            L.n1 = n1;
            L.nl = nl;
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < GS_PER; u++) {
            const int k = tid + u * GS_BLOCK;
            e0[u] = k < n0 ? list[k] : 0;
            e1[u] = k < n1 ? list[GS_CELLS - 1 - k] : 0;
            if (k < n0) L.cell[k] = (uint16_t)e0[u];
            if (k < n1) L.cell[GS_CELLS - 1 - k] = (uint16_t)e1[u];
        }
        for (int k = tid; k < nl; k += GS_BLOCK) L.late[k] = S.late[k];
        __syncthreads();
    }
#pragma unroll
    for (int b = 0; b < GS_OWN; b++)
        S.v[gs_place(wave + (b >> 1) * GS_WAVES, lane + 64 * (b & 1))] = v[b];
    __syncthreads();
    const int steps = nl ? (nx & 1) + (ny & 1) : 0;
    for (int it = 0; it < iterations; it++) {
#pragma unroll
        for (int colour = 0; colour < 2; colour++) {
            const int n = colour ? n1 : n0;
#pragma unroll
            for (int u = 0; u < GS_PER; u++)
                if (tid + u * GS_BLOCK < n) gs_update(S.v, colour ? e1[u] : e0[u], c);
            __syncthreads();
            for (int step = 1; step <= steps; step++) {
                for (int k = tid; k < nl; k += GS_BLOCK)
                    if (S.late[k] >> 17 == (uint32_t)(colour | step << 1))
                        gs_update(S.v, S.late[k], c);
                __syncthreads();
            }
        }
    }
    const int hj = ny - j0 < GS_IN_H ? ny - j0 : GS_IN_H, hi = nx - i0 < GS_IN_W ? nx - i0 : GS_IN_W;
    double* db = dst + base + (int64_t)j0 * nx + i0;
    const auto store = [&](int r, int k, double x) {
        const int y = r - GS_HALO, z = k - GS_HALO;
        if (y >= 0 && y < hj && z >= 0 && z < hi) db[(int64_t)y * nx + z] = x;
    };
    if (first) {
#pragma unroll
        for (int b = 0; b < GS_OWN; b++) {
            const int r = wave + (b >> 1) * GS_WAVES, k = lane + 64 * (b & 1);
            store(r, k, S.v[gs_place(r, k)]);
        }
        return;
    }
    const auto store_entry = [&](uint32_t e) {
        const int q = e & 0x3fff, h = q < GS_PLANE ? q : q - GS_PLANE;
        store(h / GS_HALF, 2 * (h % GS_HALF) + (int)(e >> 14 & 1), S.v[q]);
    };
#pragma unroll
    for (int u = 0; u < GS_PER; u++) {
        if (tid + u * GS_BLOCK < n0) store_entry(e0[u]);
        if (tid + u * GS_BLOCK < n1) store_entry(e1[u]);
    }
    for (int k = tid; k < nl; k += GS_BLOCK) store_entry(S.late[k]);
}

// _interp_ndarray.py:208-224 _linear_interpolation
__global__ void k_interp_1d(const double* __restrict__ a, int64_t n,
                            const double* __restrict__ x, int64_t m, int64_t D,
                            double* __restrict__ out)
{
    const int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (q >= D * m) return;
    const int64_t d = q / m;
    const double xv = x[q];
    int64_t x0 = (int64_t)floor(xv);
    if (x0 < 0) x0 = 0;
    else if (x0 > n - 2) x0 = n - 2;
    const double a0 = a[d * n + x0], a1 = a[d * n + x0 + 1];
    const double dx = xv - (double)x0;
    out[q] = a0 * (1 - dx) + a1 * dx;
}

// _interp_ndarray.py:227-269 _bilinear_interpolation
__global__ void k_interp_2d(const double* __restrict__ a, int64_t nx, int64_t ny,
                            const double* __restrict__ x, const double* __restrict__ y,
                            int64_t m, int64_t D, double* __restrict__ out)
{
    const int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (q >= D * m) return;
    const int64_t d = q / m;
    const double xv = x[q], yv = y[q];
    int64_t x00 = (int64_t)floor(xv), y00 = (int64_t)floor(yv);
    if (x00 < 0) x00 = 0;
    else if (x00 > nx - 2) x00 = nx - 2;
    if (y00 < 0) y00 = 0;
    else if (y00 > ny - 2) y00 = ny - 2;
    const double* ad = a + d * nx * ny;
    const double a00 = ad[x00 * ny + y00];
    const double a01 = ad[x00 * ny + y00 + 1];
    const double a10 = ad[(x00 + 1) * ny + y00];
    const double a11 = ad[(x00 + 1) * ny + y00 + 1];
    const double dx = xv - (double)x00, dy = yv - (double)y00;
    const double w00 = (1 - dx) * (1 - dy);
    const double w01 = (1 - dx) * dy;
    const double w10 = dx * (1 - dy);
    const double w11 = dx * dy;
    out[q] = (a00 * w00) + (a01 * w01) + (a10 * w10) + (a11 * w11);
}

int64_t gs_tiles(int64_t n, int64_t in) { return (n + in - 1) / in; }

// Below this many iterations the launches per colour are as fast: at 3, 17.5
// us both ways for a slice of 24 x 1000 (at 2, 12 against 17), 53 against 82
// for 4 of 768 x 1000 (at 2, 51 against 55).
constexpr int64_t GS_FEW = 3;

// Whether a call takes the tiles: both axes long enough for the halo, enough
// iterations, 32-bit cell indices, and no stream capture (the second buffer
// and the lists are allocated).
bool tiles_apply(int64_t T, int64_t ny, int64_t nx, int64_t iterations, hipStream_t s)
{
    if (ny < GS_MIN || nx < GS_MIN || iterations < GS_FEW || ny * nx >= INT32_MAX) return false;
    if (T * gs_tiles(ny, GS_IN_H) * gs_tiles(nx, GS_IN_W) >= INT32_MAX) return false;
    return !capturing(s);
}

int fill_tiles(double* a, double* other, const uint8_t* where, GsTileLists* lists, int64_t T,
               int64_t ny, int64_t nx, int64_t iterations, GsCoef c, hipStream_t s)
{
    const int ntx = (int)gs_tiles(nx, GS_IN_W), nty = (int)gs_tiles(ny, GS_IN_H);
    const unsigned grid = (unsigned)(T * ntx * nty);
    const int64_t launches = 2 * ((iterations + 2 * GS_ITER - 1) / (2 * GS_ITER));
    int64_t done = 0;
    for (int64_t k = 0; k < launches; k++) {
        const int64_t upto = iterations * (k + 1) / launches;
        const int n = (int)(upto - done);
        if (k == 0)
            k_gs_tile<true><<<grid, GS_BLOCK, sizeof(GsTileLds), s>>>(
                a, other, where, lists, (int)ny, (int)nx, ntx, nty, n, c);
        else
            k_gs_tile<false><<<grid, GS_BLOCK, sizeof(GsTileLds), s>>>(
                k % 2 ? other : a, k % 2 ? a : other, where, lists, (int)ny, (int)nx, ntx, nty, n,
                c);
        done = upto;
    }
    RG_HIP(hipGetLastError());
    return RG_OK;
}

// T slices, each launch of them within LAUNCH_THREADS
int fill_slices(double* a, const uint8_t* where, int64_t T, int64_t ny, int64_t nx,
                int64_t num_iterations, GsCoef c, hipStream_t s)
{
    if (ny * nx <= GS_LDS_CELLS) {
        const size_t lds = 8 * ny * nx + 4 * (n_late(ny, nx) + 1);
        if (ny * nx <= GS_SMALL_CELLS)
            k_gs_lds<GS_SMALL_BLOCK><<<(unsigned)T, GS_SMALL_BLOCK, lds, s>>>(
                a, where, (int)ny, (int)nx, num_iterations, c);
        else
            k_gs_lds<GS_BLOCK><<<(unsigned)T, GS_BLOCK, lds, s>>>(a, where, (int)ny, (int)nx,
                                                                  num_iterations, c);
        RG_HIP(hipGetLastError());
        return RG_OK;
    }
    if (tiles_apply(T, ny, nx, num_iterations, s)) {
        DevBuf<double> other;
        DevBuf<GsTileLists> lists;
        if (other.alloc(T * ny * nx, s) == RG_OK &&
            lists.alloc(T * gs_tiles(ny, GS_IN_H) * gs_tiles(nx, GS_IN_W), s) == RG_OK)
            return fill_tiles(a, other.p, where, lists.p, T, ny, nx, num_iterations, c, s);
    }
    const int64_t cells = T * ny * nx;
    const bool late = (nx & 1) || (ny & 1);
    for (int64_t k = 0; k < num_iterations; k++) {
        for (int parity = 0; parity < 2; parity++) {
            k_gs_color<<<grid_for(cells, 256), 256, 0, s>>>(a, where, T, ny, nx, parity, c);
            if (late) k_gs_late<<<(unsigned)T, 256, 0, s>>>(a, where, ny, nx, parity, c);
        }
    }
    RG_HIP(hipGetLastError());
    return RG_OK;
}

}  // namespace

}  // namespace rg

using namespace rg;

extern "C" {

int rg_fill_gauss_seidel_2d(double* a, const uint8_t* where, int64_t T, int64_t ny,
                            int64_t nx, int64_t num_iterations, void* stream)
{
    if (T < 0 || ny < 1 || nx < 1 || num_iterations < 0 || T > 0xffffffffLL)
        return fail(RG_ERR_ARGUMENT, "invalid fill shape or iteration count");
    if (T == 0 || num_iterations == 0) return RG_OK;
    if (!a || !where) return fail(RG_ERR_ARGUMENT, "NULL array");
    const GsCoef c = gs_coef(nx, ny);
    const int64_t cells = ny * nx;
    const int64_t threads =  // of a slice, on the way that takes the most
        std::max(cells, GS_BLOCK * gs_tiles(ny, GS_IN_H) * gs_tiles(nx, GS_IN_W));
    const int64_t most = std::max<int64_t>(1, (LAUNCH_THREADS - GS_BLOCK) / threads);
    for (int64_t t = 0; t < T; t += most)
        RG_TRY(fill_slices(a + t * cells, where + t * cells, std::min(T - t, most), ny, nx,
                           num_iterations, c, (hipStream_t)stream));
    return RG_OK;
}

int rg_interp_linear_1d(const double* a, int64_t n, const double* x, int64_t m,
                        int64_t D, double* out, void* stream)
{
    if (D < 0 || n < 2 || m < 0) return fail(RG_ERR_ARGUMENT, "invalid interpolation shape");
    if (D == 0 || m == 0) return RG_OK;
    if (!a || !x || !out) return fail(RG_ERR_ARGUMENT, "NULL array");
    k_interp_1d<<<grid_for(D * m, 256), 256, 0, (hipStream_t)stream>>>(a, n, x, m, D, out);
    RG_HIP(hipGetLastError());
    return RG_OK;
}

int rg_interp_linear_2d(const double* a, int64_t nx, int64_t ny, const double* x,
                        const double* y, int64_t m, int64_t D, double* out, void* stream)
{
    if (D < 0 || nx < 2 || ny < 2 || m < 0)
        return fail(RG_ERR_ARGUMENT, "invalid interpolation shape");
    if (D == 0 || m == 0) return RG_OK;
    if (!a || !x || !y || !out) return fail(RG_ERR_ARGUMENT, "NULL array");
    k_interp_2d<<<grid_for(D * m, 256), 256, 0, (hipStream_t)stream>>>(a, nx, ny, x, y, m, D,
                                                                        out);
    RG_HIP(hipGetLastError());
    return RG_OK;
}

}  // extern "C"
