// rg_geometry.hpp -- FP64 geometry primitives of the conservative sweep.
//
// Every function here is __host__ __device__ so that the GPU kernels and the
// CPU emulation harness (tests/emu) execute the same instructions.  The build
// uses -ffp-contract=off and no fast-math: each product and each quotient is
// rounded separately, in the order the reference writes the expression, so
// the discrete decisions of the sweep (hit / no hit, t ordering) and the
// emitted weights are bit-identical to an exact-order run of the reference.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#define RG_HD __host__ __device__ __forceinline__

namespace rg {

// Element i of an array in device global memory.  A pointer read from a
// table in device memory (the grids of a Build) carries no address space,
// so plain loads through it are flat loads, whose completion is also counted
// on the LDS / scalar-load counter: every wait for one then waits for both
// kinds.  On the device the load names the global address space; the host
// twin serves the CPU emulation of the same functions.
template <class T, class I>
__device__ __forceinline__ T gload(const T* p, I i)
{
    return ((const __attribute__((address_space(1))) T*)p)[i];
}
template <class T, class I>
__host__ __forceinline__ T gload(const T* p, I i)
{
    return p[i];
}

// geometry.py:153-284 bounding_boxes_intersect_2d: inclusive (touching
// boxes intersect); each box is given by two corner points in any order.
RG_HD bool bbox_overlap(double xp1, double yp1, double xp2, double yp2,
                        double xq1, double yq1, double xq2, double yq2)
{
    double pxl = xp1 > xp2 ? xp2 : xp1, pxh = xp1 > xp2 ? xp1 : xp2;
    double qxl = xq1 > xq2 ? xq2 : xq1, qxh = xq1 > xq2 ? xq1 : xq2;
    if (!(pxl <= qxh && qxl <= pxh)) return false;
    double pyl = yp1 > yp2 ? yp2 : yp1, pyh = yp1 > yp2 ? yp1 : yp2;
    double qyl = yq1 > yq2 ? yq2 : yq1, qyh = yq1 > yq2 ? yq1 : yq2;
    if (!(pyl <= qyh && qyl <= pyh)) return false;
    return true;
}

// Intersection parameters of segments p1->p2 and q1->q2
// (geometry.py:370-445): t along p, u along q.  Disjoint bounding boxes give
// (inf, inf); parallel segments give inf/NaN through the division.
struct TU {
    double t, u;
};

RG_HD TU seg_params(double x1, double y1, double x2, double y2, double x3,
                    double y3, double x4, double y4)
{
    TU r;
    if (!bbox_overlap(x1, y1, x2, y2, x3, y3, x4, y4)) {
        r.t = __builtin_huge_val();
        r.u = __builtin_huge_val();
        return r;
    }
    double tdet = (x1 - x3) * (y3 - y4) - (y1 - y3) * (x3 - x4);
    double udet = (x1 - x2) * (y1 - y3) - (y1 - y2) * (x1 - x3);
    double det = (x1 - x2) * (y3 - y4) - (y1 - y2) * (x3 - x4);
    r.t = tdet / det;
    r.u = -udet / det;
    return r;
}

// geometry.py:448-475: hit iff 0 <= t < 1 and 0 <= u < 1.
RG_HD bool seg_hit(TU p)
{
    return (0 <= p.t && p.t < 1) && (0 <= p.u && p.u < 1);
}

// geometry.py:968-995 signed area of the triangle (origin, v1, v2).
RG_HD double area_tri(double x1, double y1, double x2, double y2)
{
    return (x1 * y2 - x2 * y1) / 2;
}

// Contribution of polygon edge (vx0,vy0)->(vx1,vy1) to the extended winding
// number of point (x, y) (geometry.py:775-829).  The total is a sum of
// +-1 and +-0.5 terms, so it is exact in any summation order, which lets a
// wavefront split the edges between its lanes.
RG_HD double winding_term(double x, double y, double vx0, double vy0,
                          double vx1, double vy1)
{
    double x0 = vx0 - x, y0 = vy0 - y;
    double x1 = vx1 - x, y1 = vy1 - y;
    if (y0 * y1 < 0) {
        double r = x0 + y0 * (x1 - x0) / (y0 - y1);
        if (r > 0) return y0 < 0 ? 1.0 : -1.0;
        return y0 < 0 ? -1.0 : 1.0;
    }
    if (y0 == 0) {
        if (x0 > 0) {
            if (y1 > 0) return 0.5;
            if (y1 < 0) return -0.5;
        } else if (x0 < 0) {
            if (y1 < 0) return 0.5;
            if (y1 > 0) return -0.5;
        }
        return 0.0;
    }
    if (y1 == 0) {
        if (x1 > 0) {
            if (y0 < 0) return 0.5;
            if (y0 > 0) return -0.5;
        } else if (x1 < 0) {
            if (y0 > 0) return 0.5;
            if (y0 < 0) return -0.5;
        }
    }
    return 0.0;
}

// point_is_inside_polygon for the quadrilateral cell (i, j) of a vertex grid
// with ny vertices per row; vertex order (i,j) (i+1,j) (i+1,j+1) (i,j+1) as in
// _grids.py:256-269.  The polygon loop starts with the closing edge
// v3 -> v0 (python index -1), exactly like geometry.py:775.
RG_HD bool cell_contains(const double* __restrict__ x,
                         const double* __restrict__ y, int64_t ny, int64_t i,
                         int64_t j, double px, double py)
{
    int64_t a = i * ny + j, b = (i + 1) * ny + j;
    double vx0 = x[a], vy0 = y[a];
    double vx1 = x[b], vy1 = y[b];
    double vx2 = x[b + 1], vy2 = y[b + 1];
    double vx3 = x[a + 1], vy3 = y[a + 1];
    double w = 0;
    w += winding_term(px, py, vx3, vy3, vx0, vy0);
    w += winding_term(px, py, vx0, vy0, vx1, vy1);
    w += winding_term(px, py, vx1, vy1, vx2, vy2);
    w += winding_term(px, py, vx2, vy2, vx3, vy3);
    return w != 0;
}

// floor(v) as int64, saturating where numba's int(math.floor(v)) would be
// undefined (NaN, beyond int64).
RG_HD int64_t floor_i64(double v)
{
    double f = __builtin_floor(v);
    if (!(f > -4.0e18)) return -4000000000000000000LL;
    if (!(f < 4.0e18)) return 4000000000000000000LL;
    return (int64_t)f;
}

// _interp_ndarray.py:226-269 _bilinear_interpolation: the lower-left corner
// is clamped into the grid, the fractional offsets are not.
RG_HD double bilinear(const double* __restrict__ a, int64_t nx, int64_t ny,
                      double x, double y)
{
    int64_t x0 = floor_i64(x), y0 = floor_i64(y);
    if (x0 < 0) x0 = 0;
    else if (x0 > nx - 2) x0 = nx - 2;
    if (y0 < 0) y0 = 0;
    else if (y0 > ny - 2) y0 = ny - 2;
    double a00 = a[x0 * ny + y0];
    double a01 = a[x0 * ny + y0 + 1];
    double a10 = a[(x0 + 1) * ny + y0];
    double a11 = a[(x0 + 1) * ny + y0 + 1];
    double dx = x - (double)x0;
    double dy = y - (double)y0;
    double w00 = (1 - dx) * (1 - dy);
    double w01 = (1 - dx) * dy;
    double w10 = dx * (1 - dy);
    double w11 = dx * dy;
    return (a00 * w00) + (a01 * w01) + (a10 * w10) + (a11 * w11);
}

// _grids.py:286-349 _index_of_point_local: lowest-index cell of the 3x3
// block around (i0, j0) containing the point; -1 when none does.
RG_HD int64_t index_local(const double* __restrict__ x,
                          const double* __restrict__ y, int64_t nx, int64_t ny,
                          int64_t i0, int64_t j0, double px, double py)
{
    int64_t ncx = nx - 1, ncy = ny - 1;
    int64_t ia = i0 - 1 > 0 ? i0 - 1 : 0, ib = i0 + 2 < ncx ? i0 + 2 : ncx;
    int64_t ja = j0 - 1 > 0 ? j0 - 1 : 0, jb = j0 + 2 < ncy ? j0 + 2 : ncy;
    for (int64_t ii = ia; ii < ib; ii++)
        for (int64_t jj = ja; jj < jb; jj++)
            if (cell_contains(x, y, ny, ii, jj, px, py)) return ii * ncy + jj;
    return -1;
}

// Result codes of the secant search.
enum : int64_t {
    RG_SEARCH_OUTSIDE = -1,  // sys.maxsize in the reference
    RG_SEARCH_BRUTE = -2,    // the reference falls back to index_of_point_brute
};

// _grids.py:356-463 index_of_point_secant without its brute-force fallback,
// statement by statement (what secant_search below is checked against):
// returns the flat cell index, RG_SEARCH_OUTSIDE, or RG_SEARCH_BRUTE when
// the reference would scan every cell (singular Jacobian or 100 iterations
// without a decision).  The caller runs the exhaustive search cooperatively.
RG_HD int64_t index_secant(const double* __restrict__ x,
                           const double* __restrict__ y, int64_t nx, int64_t ny,
                           double px, double py)
{
    const double h = 1e-3;
    int64_t ncx = nx - 1, ncy = ny - 1;
    double i = (double)nx / 2;
    double j = (double)ny / 2;
    for (int it = 0; it < 100; it++) {
        double xv = bilinear(x, nx, ny, i, j);
        double yv = bilinear(y, nx, ny, i, j);
        int64_t i0 = floor_i64(i), j0 = floor_i64(j);
        double ex = xv - px;
        double ey = yv - py;
        if (i0 >= 0 && j0 >= 0 && i0 < ncx && j0 < ncy &&
            cell_contains(x, y, ny, i0, j0, px, py)) {
            int64_t c = index_local(x, y, nx, ny, i0, j0, px, py);
            return c >= 0 ? c : RG_SEARCH_OUTSIDE;
        }
        if (__builtin_fabs(ex) < 1e-10 && __builtin_fabs(ey) < 1e-10) {
            int64_t c = index_local(x, y, nx, ny, i0, j0, px, py);
            return c >= 0 ? c : RG_SEARCH_OUTSIDE;
        }
        double dx_di = (bilinear(x, nx, ny, i + h, j) - xv) / h;
        double dx_dj = (bilinear(x, nx, ny, i, j + h) - xv) / h;
        double dy_di = (bilinear(y, nx, ny, i + h, j) - yv) / h;
        double dy_dj = (bilinear(y, nx, ny, i, j + h) - yv) / h;
        double det = dx_di * dy_dj - dx_dj * dy_di;
        if (det == 0) return RG_SEARCH_BRUTE;
        double di = (+dy_dj * ex - dx_dj * ey) / det;
        double dj = (-dy_di * ex + dx_di * ey) / det;
        i -= di;
        j -= dj;
    }
    return RG_SEARCH_BRUTE;
}

// ---- the same search, reading each vertex once -------------------------------
//
// index_secant above evaluates the bilinear map three times per iteration
// and the cell test from memory, 32 loads in three dependent round trips, and
// tests the 3 x 3 block cell by cell.  secant_search returns the same answer
// from the same arithmetic: an iteration loads its cell's four corners once
// for the map, its two differences (which leave the cell only near its
// edge) and the cell test, and the block's vertices are requested together.

// Vertex access: index -> (x, y).
struct VertexXY {  // interleaved vertices
    const double2* xy;
    RG_HD double2 operator()(int64_t i) const { return gload(xy, i); }
};
struct VertexArrays {
    const double* x;
    const double* y;
    RG_HD double2 operator()(int64_t i) const
    {
        double2 v;
        v.x = gload(x, i);
        v.y = gload(y, i);
        return v;
    }
};

// The cell (i, j) with corners c0..c3 = (i, j) (i + 1, j) (i + 1, j + 1)
// (i, j + 1) contains the point: the sum of cell_contains.
//
// Most cells asked about lie clearly beside the point, and then the sum is
// zero: every term is zero where all corners lie strictly above or all
// strictly below it; with all corners strictly on one side in x, each edge
// across the point's height counts by its direction alone and the closed
// polygon's directions cancel.  (An edge's side is computed from its
// intersection, so x must clear the point by more than the rounding; whether
// it crosses from a product of the heights, which must not vanish; neither
// may overflow.)
RG_HD bool quad_contains(double2 c0, double2 c1, double2 c2, double2 c3, double px, double py)
{
    const double b0 = c0.y - py, b1 = c1.y - py, b2 = c2.y - py, b3 = c3.y - py;
    if ((b0 > 0 && b1 > 0 && b2 > 0 && b3 > 0) || (b0 < 0 && b1 < 0 && b2 < 0 && b3 < 0))
        return false;
    const double h0 = __builtin_fabs(b0), h1 = __builtin_fabs(b1);
    const double h2 = __builtin_fabs(b2), h3 = __builtin_fabs(b3);
    const double tiny = 1e-150, huge = 1e150;
    if (h0 > tiny && h1 > tiny && h2 > tiny && h3 > tiny && (h0 + h1) + (h2 + h3) < huge) {
        const double a0 = c0.x - px, a1 = c1.x - px, a2 = c2.x - px, a3 = c3.x - px;
        const double lo = fmin(fmin(a0, a1), fmin(a2, a3)), hi = fmax(fmax(a0, a1), fmax(a2, a3));
        // (fmin and fmax pass over a NaN; the sum does not)
        if (__builtin_fabs((a0 + a1) + (a2 + a3)) < huge &&
            ((lo > 0 && lo > 1e-6 * hi) || (hi < 0 && hi < 1e-6 * lo)))
            return false;
    }
    double w = 0;
    w += winding_term(px, py, c3.x, c3.y, c0.x, c0.y);
    w += winding_term(px, py, c0.x, c0.y, c1.x, c1.y);
    w += winding_term(px, py, c1.x, c1.y, c2.x, c2.y);
    w += winding_term(px, py, c2.x, c2.y, c3.x, c3.y);
    return w != 0;
}

// index_secant with the result as a row and a column: 0 and (*ci, *cj), or
// RG_SEARCH_OUTSIDE, or RG_SEARCH_BRUTE.
template <class V>
RG_HD int64_t secant_search(const V& vtx, int64_t nx, int64_t ny, double px, double py,
                            int64_t* ci, int64_t* cj)
{
    const double h = 1e-3;
    const int64_t ncx = nx - 1, ncy = ny - 1;
    const double last_x = (double)(nx - 2), last_y = (double)(ny - 2);
    double i = (double)nx / 2;
    double j = (double)ny / 2;
    for (int it = 0; it < 100; it++) {
        // the cell of (i, j), clamped into the grid (NaN: the first one)
        const double fi = __builtin_floor(i), fj = __builtin_floor(j);
        const double x0 = !(fi > 0) ? 0 : (fi > last_x ? last_x : fi);
        const double y0 = !(fj > 0) ? 0 : (fj > last_y ? last_y : fj);
        const int64_t a = (int64_t)x0 * ny + (int64_t)y0;
        const double2 c00 = vtx(a), c01 = vtx(a + 1), c10 = vtx(a + ny), c11 = vtx(a + ny + 1);
        const auto blend = [](double2 v00, double2 v01, double2 v10, double2 v11, double dx,
                              double dy) {
            const double w00 = (1 - dx) * (1 - dy);
            const double w01 = (1 - dx) * dy;
            const double w10 = dx * (1 - dy);
            const double w11 = dx * dy;
            double2 r;
            r.x = (v00.x * w00) + (v01.x * w01) + (v10.x * w10) + (v11.x * w11);
            r.y = (v00.y * w00) + (v01.y * w01) + (v10.y * w10) + (v11.y * w11);
            return r;
        };
        // the map at (u, v), from the corners at hand where that is the same cell
        const auto map = [&](double u, double v) {
            const double fu = __builtin_floor(u), fv = __builtin_floor(v);
            const double u0 = !(fu > 0) ? 0 : (fu > last_x ? last_x : fu);
            const double v0 = !(fv > 0) ? 0 : (fv > last_y ? last_y : fv);
            if (u0 == x0 && v0 == y0) return blend(c00, c01, c10, c11, u - x0, v - y0);
            const int64_t b = (int64_t)u0 * ny + (int64_t)v0;
            return blend(vtx(b), vtx(b + 1), vtx(b + ny), vtx(b + ny + 1), u - u0, v - v0);
        };
        const double2 v = blend(c00, c01, c10, c11, i - x0, j - y0);
        const double xv = v.x, yv = v.y;
        const double ex = xv - px;
        const double ey = yv - py;
        const bool in = fi >= 0 && fj >= 0 && fi < (double)ncx && fj < (double)ncy &&
                        quad_contains(c00, c10, c11, c01, px, py);
        if (in || (__builtin_fabs(ex) < 1e-10 && __builtin_fabs(ey) < 1e-10)) {
            // the lowest-index cell of the 3 x 3 block around (fi, fj) that
            // contains the point: its 4 x 4 vertices row by row, clamped
            // into the grid (cells outside it are passed over).  (A point
            // the cell itself contains needs only the cells before it.)
            if (!(fi >= -2 && fj >= -2 && fi <= (double)ncx && fj <= (double)ncy))
                return RG_SEARCH_OUTSIDE;  // no cell of the block is in the grid
            const int64_t i0 = (int64_t)fi, j0 = (int64_t)fj;
            double2 lo[4], hi[4];
            const auto row = [&](int64_t r, double2* to) {
                const int64_t rr = r < 0 ? 0 : (r > nx - 1 ? nx - 1 : r);
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int64_t cc = j0 - 1 + q;
                    to[q] = vtx(rr * ny + (cc < 0 ? 0 : (cc > ny - 1 ? ny - 1 : cc)));
                }
            };
            row(i0 - 1, lo);
            row(i0, hi);
#pragma unroll
            for (int r = 0; r < 3; r++) {
                const int64_t ii = i0 - 1 + r;
#pragma unroll
                for (int q = 0; q < 3; q++) {
                    const int64_t jj = j0 - 1 + q;
                    if (in && r == 1 && q == 1) {
                        *ci = i0;
                        *cj = j0;
                        return 0;
                    }
                    if (ii >= 0 && ii < ncx && jj >= 0 && jj < ncy &&
                        quad_contains(lo[q], hi[q], hi[q + 1], lo[q + 1], px, py)) {
                        *ci = ii;
                        *cj = jj;
                        return 0;
                    }
                }
                if (r == 2) break;
#pragma unroll
                for (int q = 0; q < 4; q++) lo[q] = hi[q];
                row(i0 + 1 + r, hi);
            }
            return RG_SEARCH_OUTSIDE;
        }
        const double2 vi = map(i + h, j);
        const double2 vj = map(i, j + h);
        double dx_di = (vi.x - xv) / h;
        double dx_dj = (vj.x - xv) / h;
        double dy_di = (vi.y - yv) / h;
        double dy_dj = (vj.y - yv) / h;
        double det = dx_di * dy_dj - dx_dj * dy_di;
        if (det == 0) return RG_SEARCH_BRUTE;
        double di = (+dy_dj * ex - dx_dj * ey) / det;
        double dj = (-dy_di * ex + dx_di * ey) / det;
        i -= di;
        j -= dj;
    }
    return RG_SEARCH_BRUTE;
}

// secant_search over interleaved vertices, with index_secant's result.
RG_HD int64_t index_secant_xy(const double2* __restrict__ xy, int64_t nx, int64_t ny,
                              double px, double py)
{
    int64_t ci = 0, cj = 0;
    const int64_t r = secant_search(VertexXY{xy}, nx, ny, px, py, &ci, &cj);
    return r == 0 ? ci * (ny - 1) + cj : r;
}

}  // namespace rg
