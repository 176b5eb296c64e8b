// rg_search.hip -- point location: the 2-D cell search used by the build
// (index_of_point_secant, _weights_conservative_2d/_grids.py:356-463) as a
// standalone vectorised entry point, the 1-D find_indices searches
// (_find_indices_brute.py:24-51, _find_indices_searchsorted.py:24-62) and
// the cell-area entry point.
#include <hip/hip_runtime.h>

#include <string>

#include "rg_internal.hpp"
#include "rg_wave.hpp"

namespace rg {

int launch_area(const double* x, const double* y, int64_t nx, int64_t ny,
                double* out, hipStream_t s);

constexpr int CELLS_BLOCK = 128;

// One lane per point: the secant iteration of the reference, its cell written
// as (i, j) or (INT64_MAX, INT64_MAX).  Points the reference would hand to
// the exhaustive search are marked RG_SEARCH_BRUTE in their own row for
// k_cells_brute.
// 2.36 M points in a 1025^2 vertex grid: 228 us reading every vertex where it
// is used, 154 reading it once (secant_search).
__global__ __launch_bounds__(CELLS_BLOCK) void k_cells_secant(
    const double* __restrict__ x, const double* __restrict__ y, int64_t nx, int64_t ny,
    const double* __restrict__ px, const double* __restrict__ py, int64_t n,
    int64_t* __restrict__ ij)
{
    const int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (q >= n) return;
    int64_t ci = INT64_MAX, cj = INT64_MAX;
    const int64_t r = secant_search(VertexArrays{x, y}, nx, ny, px[q], py[q], &ci, &cj);
    ij[2 * q] = r == RG_SEARCH_BRUTE ? RG_SEARCH_BRUTE : ci;
    ij[2 * q + 1] = cj;
}

// The exhaustive lowest-index search for the marked points, one at a time over
// a wavefront (a pass over the grid each).  A block looks at BRUTE_WAVES * per
// points, lists the marked ones and has its wavefronts take them in turn: one
// point a wavefront while that many wavefronts fill the chip, up to 64 of a long
// list (2.36 M points, none marked: a wavefront each took 217 us, 64 each 6).
// Marked points tend to lie together (a masked region), so a block's points are
// not consecutive: it takes a cache line of rows at a time, BRUTE_LINE points,
// every gridDim.x lines.  400000 points in 257^2 vertices, the 10000 NaN ones in
// a row: 2.1 ms a wavefront each, 22 in 64 consecutive ones, now 2.1.
constexpr int BRUTE_WAVES = 8, BRUTE_LINE = 8;
constexpr int BRUTE_BLOCK = 64 * BRUTE_WAVES;

__global__ __launch_bounds__(BRUTE_BLOCK) void k_cells_brute(
    const double* __restrict__ x, const double* __restrict__ y, int64_t nx, int64_t ny,
    const double* __restrict__ px, const double* __restrict__ py, int64_t n, int per,
    int64_t* __restrict__ ij)
{
    __shared__ int32_t list[BRUTE_BLOCK];
    __shared__ int32_t marked;
    const int tid = threadIdx.x, lane = tid & 63;
    const auto point = [&](int t) {  // the block's t-th
        return (blockIdx.x + (int64_t)(t / BRUTE_LINE) * gridDim.x) * BRUTE_LINE +
               t % BRUTE_LINE;
    };
    if (tid == 0) marked = 0;
    __syncthreads();
    const int64_t own = point(tid);
    if (tid < BRUTE_WAVES * per && own < n && ij[2 * own] == RG_SEARCH_BRUTE)
        list[atomicAdd(&marked, 1)] = tid;
    __syncthreads();
    const int32_t nm = marked;
    for (int32_t k = block_wave(); k < nm; k += BRUTE_WAVES) {  // uniform per wavefront
        const int64_t q = point(__builtin_amdgcn_readfirstlane(list[k]));
        const int64_t c = wave_brute(x, y, nx, ny, px[q], py[q], lane);
        if (lane == 0) {
            ij[2 * q] = c >= 0 ? c / (ny - 1) : INT64_MAX;
            ij[2 * q + 1] = c >= 0 ? c % (ny - 1) : INT64_MAX;
        }
    }
}

// _find_indices_brute.py:42-49: first m with x[m] <= v <= x[m+1].
__global__ void k_find_brute_1d(const double* __restrict__ xin, int64_t m,
                                const double* __restrict__ xout, int64_t n,
                                int64_t batch, int64_t fill,
                                int64_t* __restrict__ res)
{
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (t >= n * batch) return;
    const int64_t d = t / n;
    const double* a = xin + d * m;
    const double v = xout[t];
    int64_t r = fill;
    for (int64_t q = 0; q < m - 1; q++)
        if (a[q] <= v && v <= a[q + 1]) {
            r = q;
            break;
        }
    res[t] = r;
}

// numpy's searchsorted order: NaN sorts after every number.
__device__ inline bool np_less(double a, double b)
{
    return a < b || (b != b && a == a);
}

// _find_indices_searchsorted.py:38-60 with np.searchsorted(side="left").
__global__ void k_find_sorted_1d(const double* __restrict__ xin, int64_t m,
                                 const double* __restrict__ xout, int64_t n,
                                 int64_t batch, int64_t fill,
                                 int64_t* __restrict__ res)
{
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (t >= n * batch) return;
    const int64_t d = t / n;
    const double* a = xin + d * m;
    const double v = xout[t];
    int64_t lo = 0, hi = m;
    while (lo < hi) {
        int64_t mid = lo + (hi - lo) / 2;
        if (np_less(a[mid], v)) lo = mid + 1;
        else hi = mid;
    }
    int64_t r = lo - 1;
    if (v == a[0]) r = 0;
    else if (r < 0) r = fill;
    else if (r > m - 2) r = fill;
    res[t] = r;
}

namespace {

int check_find_cells(const double* x, const double* y, int64_t nx, int64_t ny,
                     const double* px, const double* py, int64_t* cell_ij)
{
    if (!x || !y || !px || !py || !cell_ij)
        return fail(RG_ERR_ARGUMENT, "NULL argument");
    if (nx < 2 || ny < 2)
        return fail(RG_ERR_ARGUMENT, "grid needs at least 2x2 vertices");
    return RG_OK;
}

int launch_find_cells(const double* x, const double* y, int64_t nx, int64_t ny,
                      const double* px, const double* py, int64_t n,
                      int64_t* cell_ij, hipStream_t s)
{
    k_cells_secant<<<grid_for(n, CELLS_BLOCK), CELLS_BLOCK, 0, s>>>(x, y, nx, ny, px, py, n,
                                                                    cell_ij);
    int per = 1;
    while (per < 64 && n / (2 * per) >= 16384) per *= 2;
    const int64_t lines = (n + BRUTE_LINE - 1) / BRUTE_LINE;
    static_assert(BRUTE_WAVES == BRUTE_LINE, "a block of BRUTE_WAVES * per points is per lines");
    k_cells_brute<<<grid_for(lines, per), BRUTE_BLOCK, 0, s>>>(x, y, nx, ny, px, py, n, per,
                                                               cell_ij);
    RG_HIP(hipGetLastError());
    return RG_OK;
}

}  // namespace

}  // namespace rg

using namespace rg;

extern "C" {

int rg_cell_area_2d(const double* x, const double* y, int64_t nx, int64_t ny,
                    double* area, void* stream)
{
    if (nx < 2 || ny < 2) return RG_OK;  // no cells
    if (!x || !y || !area) return fail(RG_ERR_ARGUMENT, "NULL argument");
    return launch_area(x, y, nx, ny, area, (hipStream_t)stream);
}

int rg_find_cells_2d(const double* x, const double* y, int64_t nx, int64_t ny,
                     const double* px, const double* py, int64_t n,
                     int64_t* cell_ij, void* stream)
{
    if (n == 0) return RG_OK;
    RG_TRY(check_find_cells(x, y, nx, ny, px, py, cell_ij));
    return launch_find_cells(x, y, nx, ny, px, py, n, cell_ij, (hipStream_t)stream);
}

int rg_find_cells_2d_noalloc(const double* x, const double* y, int64_t nx,
                             int64_t ny, const double* px, const double* py,
                             int64_t n, int64_t* cell_ij, void* stream)
{
    if (n == 0) return RG_OK;
    RG_TRY(check_find_cells(x, y, nx, ny, px, py, cell_ij));
    // (the size that its scratch had when there was one)
    if (n < 0 || n > RG_FIND_CELLS_NOALLOC_MAX)
        return fail(RG_ERR_ARGUMENT,
                    "rg_find_cells_2d_noalloc: " + std::to_string(n) +
                        " points exceed its fixed scratch size of " +
                        std::to_string((long long)RG_FIND_CELLS_NOALLOC_MAX) +
                        " points per call; search them in slices");
    return launch_find_cells(x, y, nx, ny, px, py, n, cell_ij, (hipStream_t)stream);
}

int rg_find_indices_1d(const double* x_input, int64_t m,
                       const double* x_output, int64_t n, int64_t batch,
                       int method, int64_t fill_value, int64_t* result,
                       void* stream)
{
    if (n == 0 || batch == 0) return RG_OK;
    if (!x_input || !x_output || !result)
        return fail(RG_ERR_ARGUMENT, "NULL argument");
    if (m < 1) return fail(RG_ERR_ARGUMENT, "empty input grid");
    hipStream_t s = (hipStream_t)stream;
    const int64_t tot = n * batch;
    if (method == RG_FIND_BRUTE)
        k_find_brute_1d<<<grid_for(tot, 256), 256, 0, s>>>(
            x_input, m, x_output, n, batch, fill_value, result);
    else if (method == RG_FIND_SEARCHSORTED)
        k_find_sorted_1d<<<grid_for(tot, 256), 256, 0, s>>>(
            x_input, m, x_output, n, batch, fill_value, result);
    else
        return fail(RG_ERR_ARGUMENT, "unknown method");
    RG_HIP(hipGetLastError());
    return RG_OK;
}

}  // extern "C"
