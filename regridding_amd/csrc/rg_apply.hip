// rg_apply.hip -- application of device-resident weights (the hot loop of
// _regrid/_regrid_from_weights.py:172-182) and its adjoint.
//
// The reference scatters out[i_out] += w * in[i_in] over the triples in
// storage order (sorted by (input, output)).  Each output therefore receives
// its terms in ascending input order, one rounded multiply and one rounded
// add at a time, starting from +0.0.  The GPU gathers instead: one lane owns
// one output cell and adds up its CSR row (columns ascending) in exactly that
// order, which reproduces the reference bit for bit without atomics.
//
// One image, small weights and batched jobs read the entries as they lie and
// gather from global memory (k_apply, k_apply_jobs), long rows a wavefront
// each (long_rows).  Several images of large weights stage patches of the
// input in LDS, DB images at a time, which takes a plan (k_apply_rounds).
//
// The adjoint (transpose=1) is the same gather over the CSR by input, whose
// rows hold the outputs in ascending order: exactly the order in which the
// reference applies regrid_from_weights(*transpose_weights(w)).
//
// Launch layout.  The rows of a CSR are the cells of a 2-D grid.  A block
// of 256 lanes owns a tile of output cells (with a plan tile_w wide along the
// grid's last axis and 256 / tile_w tall, otherwise 64 and 4), so the input
// cells it gathers form one compact patch (a linear run of rows would be a thin
// band tilted across the input grid, re-fetched by every neighbouring run).  Blocks are
// renumbered so each of the 8 XCDs of the MI355X (blocks arrive
// round-robin) sweeps one contiguous band of tiles, keeping the patches of
// neighbouring tiles in that XCD's L2.
//
// The results are stored nontemporal, except where a tile's rows end inside
// 64-byte pieces that the caches can merge (planned_shape): each is written once
// and not read back by the launch, so written through the caches they would
// only evict the input patches that neighbouring tiles share (at 2049^2 ->
// 1537^2 and 16 images: FP64 0.239 -> 0.232 ms, FP32 0.164 -> 0.150 ms, FP64
// adjoint 0.301 -> 0.286 ms, FP32 adjoint 0.212 -> 0.115 ms).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <mutex>
#include <vector>

#include "rg_internal.hpp"

namespace rg {

constexpr int APPLY_BLOCK = 256;
constexpr int NUM_XCD = 8;

struct ApplyGrid {
    int64_t gx, gy;       // rows of the CSR as a gx x gy grid of cells
    int64_t tw, th;       // tile shape (tw * th = APPLY_BLOCK)
    int64_t ntx, ntiles;  // tiles along gy, tiles in total
};

// Stores a result: nontemporal, or (MERGE) through the caches.  (A template,
// since the compiler joins the two stores of a branch into an ordinary one.)
template <bool MERGE, class T>
__device__ inline void store_result(T* y, T v)
{
    if constexpr (MERGE)
        *y = v;
    else
        __builtin_nontemporal_store(v, y);
}

// ---- the apply without a plan ----------------------------------------------
//
// A lane that walks its own row reads col and w at a stride of one row (about
// five entries): every load instruction of the wavefront touches 20 to 30
// cache lines, and the next entry's the same lines again, which bounds it far
// below the memory's rate.  Here the wavefront reads the entries of its 64
// rows as they lie, 64 at a time, gathers x for each (neighbouring lanes hold
// neighbouring columns), and puts the rounded products into LDS; a lane then
// adds up its own row's in entry order: the same roundings in the same order.
// One image of FP64, plain pairs: 1025^2 -> 769^2 21.9 -> 12.4 us, 2049^2 ->
// 1537^2 74 -> 31 us (6.9 TB/s), its adjoint 62 -> 38 us, adjoint of 1025^2
// -> 1500^2 83 -> 23 us; eight views of a 1024^2 image, 134 -> 95 us.
// The wavefronts need no barrier; a block is four of them only so that
// neighbouring rows share the L1.
//
// Entries per lane at a time: 6 (a wavefront's 345 entries at output cells a
// third larger than the input's are one chunk) at 54 registers; 8 are 66 and
// 10 are 78 registers and lose 5 % to 10 % where the rows are short, and gain
// 15 % only where they hold nine or more.
constexpr int ENTRIES_U = 6;
constexpr int PROD_SLOTS = 64 * ENTRIES_U + 1;  // the last one is 0
// Launches of fewer tiles than this split the images over more blocks: 8
// images of 129^2 -> 101^2 take 7.6 us in 40 blocks, 4.6 us in 320 (any
// limit from 512 to 4096 measures the same).
constexpr int64_t SPLIT_TILES = 1024;
// Long rows.  Where a row is a good part of a chunk, a few of the 64 lanes add
// up products one after another, an entry at a time taking the LDS's latency.
// Rows of 64 entries on average, or of LONG_FEW in few rows (long_rows), get a
// wavefront each, which is as many chains at once as there are rows and, with
// several images, images (apply_long_row).  A wavefront of 64 rows that holds
// more than LONG_ENTRIES a row (weights of a small input on a large output grid)
// takes its rows one after another like that where there are several images
// (four pairs of 2049^2 -> 1025^2, ten times as wide, 3 / 8 images: 2489 / 6060
// us by a lane per row from memory, 3786 / 10063 by chunks of 128, 1395 / 2882
// so); with one image its sums are pipelined.  us for 1 / 8 images of FP64, a
// lane per row from memory -> rows in chunks only -> this:
//   1025^2 -> 65^2 (239 a row)     90 / 737 -> 423 / 345 -> 12 / 25
//   2049^2 -> 9^2 (53045)          17456 / 79939 -> 80365 / 89562 -> 1350 / 980
//   eight of 257^2 -> 17^2 (239)   73 / 645 -> 409 / 3226 -> 15 / 23
//   513^2 -> 513^2, twenty times as wide (426 a row in 26^2 cells of the output)
//                                  128 / 1665 -> 201 / 1664 -> 103 / 1660
//   513^2 -> 86^2 (43), chunks     21 / 129 -> 21 / 20 (a wavefront a row 12 / 13,
//     but 51 where chunks take 29 for eight such pairs of 1 image)
constexpr int32_t LONG_ENTRIES = 64;
constexpr int64_t LONG_FEW_ROWS = 4096, LONG_FEW_ONE = 40, LONG_FEW = 28;
constexpr int LONG_IMAGES = 5;
static_assert((LONG_IMAGES - 1) * 65 + 64 <= PROD_SLOTS, "the products of a long row's images");

// acc + prod[s] + ... + prod[e - 1], one after another.  The last steps of four
// read the zero past the products, which changes no sum (none is -0, as it
// starts from +0).  PIPELINE: a long run's next eight are read while the last
// eight are added, where an entry takes the LDS's latency otherwise.
template <bool PIPELINE, class T>
__device__ inline T add_products(const T* __restrict__ prod, int32_t s, int32_t e, T acc)
{
    if (PIPELINE && e - s >= 16) {
        T p[8];
#pragma unroll
        for (int u = 0; u < 8; u++) p[u] = prod[s + u];
#pragma unroll 1
        for (; s + 16 <= e; s += 8) {
            T n[8];
#pragma unroll
            for (int u = 0; u < 8; u++) n[u] = prod[s + 8 + u];
#pragma unroll
            for (int u = 0; u < 8; u++) acc = acc + p[u];
#pragma unroll
            for (int u = 0; u < 8; u++) p[u] = n[u];
        }
#pragma unroll
        for (int u = 0; u < 8; u++) acc = acc + p[u];
        s += 8;
    }
    for (int32_t q = s; q < e; q += 4) {
        T p[4];
#pragma unroll
        for (int u = 0; u < 4; u++) p[u] = prod[q + u < e ? q + u : PROD_SLOTS - 1];
#pragma unroll
        for (int u = 0; u < 4; u++) acc = acc + p[u];
    }
    return acc;
}

// Entries [c0, c0 + 64 * U) of the wavefront's `total` for `images` images:
// the products go to LDS in entry order, and each lane adds up those of its
// row, entries [s, e), to y (from 0 where c0 is 0).
template <bool MERGE, bool PIPELINE, class T, int U>
__device__ inline void apply_entries(const int32_t* __restrict__ col, const T* __restrict__ w,
                                     const T* __restrict__ x, T* __restrict__ y, int64_t nrows,
                                     int64_t ncols, int32_t images, int32_t c0, int32_t total,
                                     int32_t s, int32_t e, bool has_row,
                                     T* __restrict__ prod)
{
    const int32_t lane = threadIdx.x & 63;
    uint32_t c[U];
    T wq[U], xv[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
        const uint32_t t = min(c0 + u * 64 + lane, total - 1);
        c[u] = (uint32_t)col[t];
        wq[u] = w[t];
    }
    s = max(s - c0, 0);
    e = min(e - c0, 64 * U);
    const bool stores = c0 ? s < e : has_row;
    for (int32_t m = 0; m < images; m++) {
#pragma unroll
        for (int u = 0; u < U; u++) xv[u] = x[c[u]];
        __builtin_amdgcn_wave_barrier();  // the last image's products are read
#pragma unroll
        for (int u = 0; u < U; u++) prod[u * 64 + lane] = wq[u] * xv[u];
        x += ncols;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (stores) {
            const T acc = add_products<PIPELINE>(prod, s, e, c0 ? *y : T(0));
            store_result<MERGE>(y, acc);
        }
        y += nrows;
    }
}

// One row of `total` entries for up to LONG_IMAGES images, by a wavefront: 64
// entries at a time, their products for every image in LDS, added up by one
// lane per image (image m's are at 65 m, so that the lanes' reads fall in
// different banks).  The next entries are requested before the sums.
template <bool MERGE, class T>
__device__ inline void apply_long_row(const int32_t* __restrict__ col, const T* __restrict__ w,
                                      const T* __restrict__ x, T* __restrict__ y, int64_t nrows,
                                      int64_t ncols, int32_t images, int32_t total,
                                      T* __restrict__ prod)
{
    const int32_t lane = threadIdx.x & 63;
    uint32_t c = 0;
    T wq = T(0), acc = T(0);
    const auto request = [&](int32_t c0) {
        const uint32_t t = min(c0 + lane, total - 1);
        c = (uint32_t)col[t];
        wq = w[t];
    };
    if (total > 0) request(0);
    for (int32_t c0 = 0; c0 < total; c0 += 64) {
        T xv[LONG_IMAGES];
#pragma unroll
        for (int m = 0; m < LONG_IMAGES; m++)
            if (m < images) xv[m] = x[m * ncols + c];
        __builtin_amdgcn_wave_barrier();  // the last products are read
#pragma unroll
        for (int m = 0; m < LONG_IMAGES; m++)
            if (m < images) prod[m * 65 + lane] = wq * xv[m];
        if (c0 + 64 < total) request(c0 + 64);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (lane < images) {
            const T* const p = prod + lane * 65;
            const int32_t n = min(64, total - c0);
            int32_t k = 0;
            for (; k + 8 <= n; k += 8) {
                T v[8];
#pragma unroll
                for (int u = 0; u < 8; u++) v[u] = p[k + u];
#pragma unroll
                for (int u = 0; u < 8; u++) acc = acc + v[u];
            }
            for (; k < n; k++) acc = acc + p[k];
        }
    }
    if (lane < images) store_result<MERGE>(y + lane * nrows, acc);
}

// Applies the CSR to one tile and `images` images, a wavefront for each 64
// consecutive rows and by itself.  A tile is 64 columns of APPLY_BLOCK / 64
// grid rows at (ib, jb); APPLY_BLOCK rows of one long row (`th` 1); or, of a
// grid one column wide, APPLY_BLOCK / 64 rows, a wavefront each.
template <bool MERGE, class T>
__device__ inline void apply_rows(const int32_t* __restrict__ rowptr,
                                  const int32_t* __restrict__ col, const T* __restrict__ w,
                                  const T* __restrict__ x, T* __restrict__ y, int64_t nrows,
                                  int64_t ncols, int32_t images, int64_t gy, int64_t ib,
                                  int64_t jb, int64_t th, T* __restrict__ prod)
{
    const int32_t lane = threadIdx.x & 63;
    const int32_t wave = __builtin_amdgcn_readfirstlane((int32_t)threadIdx.x / 64);
    const bool flat = th == 1;
    const int64_t i = ib + (flat ? 0 : wave), j = jb + (flat ? wave * 64 : 0);
    const int64_t r0 = i * gy + j;
    if (r0 >= nrows || j >= gy) return;
    const int32_t rows = gy - j < 64 ? (int32_t)(gy - j) : 64;
    // lanes past the last row take that row's end: no entries
    const int64_t r = r0 + min(lane, rows - 1);
    int32_t s = rowptr[r];
    int32_t e = rowptr[r + 1];
    const bool valid = lane < rows;
    if (!valid) s = e;
    const int32_t first = __builtin_amdgcn_readlane(s, 0);
    const int32_t total = __builtin_amdgcn_readlane(e, 63) - first;
    s -= first;
    e -= first;
    col += first;
    w += first;
    T* const y0 = y + r0;
    y += r;
    if (lane == 0) prod[PROD_SLOTS - 1] = T(0);
    if (total == 0) {
        if (valid)
            for (int32_t m = 0; m < images; m++) y[m * nrows] = T(0);
        return;
    }
    if (images > 1 && (rows == 1 || total > LONG_ENTRIES * rows)) {
        // (eight images in two passes of four)
        const int32_t step = images <= LONG_IMAGES ? images : (images + 1) / 2;
        static_assert(JOB_DB <= 2 * LONG_IMAGES, "two passes");
        for (int32_t q = 0; q < rows; q++) {
            const int32_t at = __builtin_amdgcn_readlane(s, q);
            const int32_t n = __builtin_amdgcn_readlane(e, q) - at;
            for (int32_t m = 0; m < images; m += step)
                apply_long_row<MERGE, T>(col + at, w + at, x + m * ncols, y0 + q + m * nrows,
                                         nrows, ncols, min(step, images - m), n, prod);
        }
        return;
    }
    if (total <= 64 * (ENTRIES_U / 2)) {
        apply_entries<MERGE, false, T, ENTRIES_U / 2>(col, w, x, y, nrows, ncols, images, 0, total,
                                                      s, e, valid, prod);
    } else if (images == 1) {
        for (int32_t c0 = 0; c0 < total; c0 += 64 * ENTRIES_U)
            apply_entries<MERGE, true, T, ENTRIES_U>(col, w, x, y, nrows, ncols, 1, c0, total, s,
                                                     e, valid, prod);
    } else {
        for (int32_t c0 = 0; c0 < total; c0 += 64 * ENTRIES_U)
            apply_entries<MERGE, false, T, ENTRIES_U>(col, w, x, y, nrows, ncols, images, c0,
                                                      total, s, e, valid, prod);
    }
}

template <class T, bool MERGE>
__global__ __launch_bounds__(APPLY_BLOCK) void k_apply(
    const int32_t* __restrict__ rowptr, const int32_t* __restrict__ col,
    const T* __restrict__ w, const T* __restrict__ x, T* __restrict__ y,
    int64_t nrows, int64_t ncols, int64_t batch, int32_t db, ApplyGrid G)
{
    __shared__ T prod[APPLY_BLOCK / 64][PROD_SLOTS];
    const uint32_t nb = gridDim.x;  // a multiple of NUM_XCD
    const uint32_t b = blockIdx.x;
    const uint32_t tile = (b % NUM_XCD) * (nb / NUM_XCD) + b / NUM_XCD;
    if (tile >= G.ntiles) return;
    const uint32_t ntx = (uint32_t)G.ntx, ti = tile / ntx, tj = tile % ntx;
    const int64_t d0 = (int64_t)blockIdx.y * db;
    const int64_t nd = batch - d0 < db ? batch - d0 : db;
    apply_rows<MERGE, T>(rowptr, col, w, x + d0 * ncols, y + d0 * nrows, nrows, ncols, (int32_t)nd, G.gy,
                  ti * G.th, tj * G.tw, G.th, prod[threadIdx.x / 64]);
}

// ---- the apply plan -------------------------------------------------------
//
// With many images per pass, one tile's gathered footprint (patch cells x
// images x 8 B) outgrows the L1, and the tiles in flight on an XCD outgrow
// its L2: a cache line of the input is evicted before the neighbouring cells
// it also holds are used, and comes back from HBM several times.  The plan
// removes the dependence on cache luck.  Made once per handle and direction
// (the weights are static; every later apply reuses it), it stores for every
// tile the bounding box (i0, j0, rows, cols) of the input cells its rows
// gather, and for every CSR entry the entry's offset inside that box.  The
// planned apply then stages the box of DB images in LDS with one coalesced
// row load per box row, and gathers from LDS.

constexpr int LDS_BYTES = 64 * 1024;  // staged patch per block
constexpr int64_t PLAN_MIN_ROWS = 65536;

// a / b from a float reciprocal and one correction step (the float quotient
// is off by at most one).  Exact for 0 <= a <= 65536 and 1 <= b <= 16384,
// checked exhaustively; a staged patch holds at most 16384 cells.
__device__ inline int32_t fast_div(int32_t a, int32_t b, float inv_b)
{
    int32_t q = (int32_t)((float)a * inv_b);
    const int32_t r = a - q * b;
    if (r < 0) q--;
    else if (r >= b) q++;
    return q;
}

// One input cell of a staged patch: its values in the DB images of the pass,
// side by side.  The patch is cell-major, so a gather reads one entry's DB
// values with one or a few wide LDS loads at one address; an image-major
// patch needs a load and an address computation per image (the FP32 apply
// was bound by that arithmetic).  Images past the pass's count hold 0.
template <class T, int DB>
struct alignas(DB * sizeof(T) >= 16 ? 16 : DB * sizeof(T)) CellVals {
    T v[DB];
};

// Cells each thread stages per step (their DB loads in flight together).
template <class T, int DB>
constexpr int stage_cells_per_step()
{
    return DB >= 16 ? 1 : 16 / DB;
}

// Stages the (rows x cols) box of nd images at xb (image stride ncols, row
// stride src_gy) into `patch`, cell (ii, jj) at ii * cols + jj.  Consecutive
// threads take consecutive cells, so each image's loads are coalesced.
template <class T, int DB>
__device__ inline void stage_cells(CellVals<T, DB>* __restrict__ patch,
                                   const T* __restrict__ xb, int64_t ncols, int64_t src_gy,
                                   int32_t rows, int32_t cols, int32_t nd)
{
    constexpr int SU = stage_cells_per_step<T, DB>();
    const int32_t ncell = rows * cols;
    const float inv_cols = 1.0f / (float)cols;
    for (int32_t c0 = threadIdx.x; c0 < ncell; c0 += APPLY_BLOCK * SU) {
        CellVals<T, DB> cv[SU];
#pragma unroll
        for (int u = 0; u < SU; u++) {
            const int32_t c = c0 + u * APPLY_BLOCK;
            if (c < ncell) {
                const int32_t ii = fast_div(c, cols, inv_cols);
                const T* xc = xb + (int64_t)ii * src_gy + (c - ii * cols);
#pragma unroll
                for (int m = 0; m < DB; m++) cv[u].v[m] = m < nd ? xc[m * ncols] : T(0);
            }
        }
#pragma unroll
        for (int u = 0; u < SU; u++) {
            const int32_t c = c0 + u * APPLY_BLOCK;
            if (c < ncell) patch[c] = cv[u];
        }
    }
}

__global__ __launch_bounds__(APPLY_BLOCK) void k_plan(
    const int32_t* __restrict__ rowptr, const int32_t* __restrict__ col,
    ApplyGrid G, int64_t src_gy, int32_t* __restrict__ box,
    uint16_t* __restrict__ off)
{
    __shared__ int32_t lo_i, hi_i, lo_j, hi_j;
    if (threadIdx.x == 0) {
        lo_i = INT32_MAX; hi_i = INT32_MIN; lo_j = INT32_MAX; hi_j = INT32_MIN;
    }
    __syncthreads();
    const int64_t tile = blockIdx.x;
    const int64_t ti = tile / G.ntx, tj = tile % G.ntx;
    const int64_t i = ti * G.th + threadIdx.x / G.tw;
    const int64_t j = tj * G.tw + threadIdx.x % G.tw;
    const bool valid = i < G.gx && j < G.gy;
    const int64_t r = i * G.gy + j;
    int32_t s = 0, e = 0;
    if (valid) {
        s = rowptr[r];
        e = rowptr[r + 1];
    }
    // The row's first PLAN_E entries are loaded once, all at once, and kept
    // for both passes (a row holds about five at the usual grid ratios);
    // columns and the row length fit 32 bits, so the divisions are 32-bit.
    constexpr int PLAN_E = 8;
    const uint32_t gy = (uint32_t)src_gy;
    uint32_t cr[PLAN_E];
#pragma unroll
    for (int u = 0; u < PLAN_E; u++) cr[u] = s + u < e ? (uint32_t)col[s + u] : 0u;
    int32_t a0 = INT32_MAX, a1 = INT32_MIN, b0 = INT32_MAX, b1 = INT32_MIN;
#pragma unroll
    for (int u = 0; u < PLAN_E; u++)
        if (s + u < e) {
            const int32_t ci = (int32_t)(cr[u] / gy), cj = (int32_t)(cr[u] - (uint32_t)ci * gy);
            a0 = min(a0, ci); a1 = max(a1, ci);
            b0 = min(b0, cj); b1 = max(b1, cj);
        }
    for (int32_t q = s + PLAN_E; q < e; q++) {
        const uint32_t c = (uint32_t)col[q];
        const int32_t ci = (int32_t)(c / gy), cj = (int32_t)(c - (uint32_t)ci * gy);
        a0 = min(a0, ci); a1 = max(a1, ci);
        b0 = min(b0, cj); b1 = max(b1, cj);
    }
    // the wavefront's extremes first (shuffles), then one LDS atomic per
    // wavefront and bound: 256 threads' atomics on the same four words
    // serialize in the LDS and made this kernel (a row without entries holds
    // the neutral values)
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        a0 = min(a0, __shfl_xor(a0, o, 64)); a1 = max(a1, __shfl_xor(a1, o, 64));
        b0 = min(b0, __shfl_xor(b0, o, 64)); b1 = max(b1, __shfl_xor(b1, o, 64));
    }
    if ((threadIdx.x & 63) == 0 && a0 <= a1) {
        atomicMin(&lo_i, a0); atomicMax(&hi_i, a1);
        atomicMin(&lo_j, b0); atomicMax(&hi_j, b1);
    }
    __syncthreads();
    const bool empty = lo_i > hi_i;
    const int32_t rows = empty ? 0 : hi_i - lo_i + 1;
    const int32_t cols = empty ? 0 : hi_j - lo_j + 1;
    if (threadIdx.x == 0) {
        box[4 * tile + 0] = empty ? 0 : lo_i;
        box[4 * tile + 1] = empty ? 0 : lo_j;
        box[4 * tile + 2] = rows;
        box[4 * tile + 3] = cols;
    }
    // offsets are only read for patches that fit the LDS (< 2^16 cells)
    const int64_t cells = (int64_t)rows * cols;
#pragma unroll
    for (int u = 0; u < PLAN_E; u++)
        if (s + u < e) {
            const int32_t ci = (int32_t)(cr[u] / gy), cj = (int32_t)(cr[u] - (uint32_t)ci * gy);
            const int64_t o = (int64_t)(ci - lo_i) * cols + (cj - lo_j);
            off[s + u] = cells < 65536 ? (uint16_t)o : (uint16_t)0;
        }
    for (int32_t q = s + PLAN_E; q < e; q++) {
        const uint32_t c = (uint32_t)col[q];
        const int32_t ci = (int32_t)(c / gy), cj = (int32_t)(c - (uint32_t)ci * gy);
        const int64_t o = (int64_t)(ci - lo_i) * cols + (cj - lo_j);
        off[q] = cells < 65536 ? (uint16_t)o : (uint16_t)0;
    }
}

// One block of PLAN_MAX_BLOCK threads: the largest patch over all tiles
// (each thread's share of the tiles is loaded four at a time).
constexpr int PLAN_MAX_BLOCK = 1024;

__global__ __launch_bounds__(PLAN_MAX_BLOCK) void k_plan_max(const int32_t* __restrict__ box,
                                                             int64_t ntiles,
                                                             int64_t* __restrict__ out)
{
    int64_t m = 0;
    for (int64_t t0 = threadIdx.x; t0 < ntiles; t0 += 4 * PLAN_MAX_BLOCK) {
        int64_t c[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int64_t t = t0 + u * PLAN_MAX_BLOCK;
            c[u] = t < ntiles ? (int64_t)box[4 * t + 2] * box[4 * t + 3] : 0;
        }
#pragma unroll
        for (int u = 0; u < 4; u++) m = c[u] > m ? c[u] : m;
    }
    __shared__ int64_t sh[PLAN_MAX_BLOCK];
    sh[threadIdx.x] = m;
    __syncthreads();
    for (int o = PLAN_MAX_BLOCK / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o && sh[threadIdx.x + o] > sh[threadIdx.x])
            sh[threadIdx.x] = sh[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = sh[0];
}

// lds_bytes: the dynamic LDS of the launch; a tile whose patch for the
// block's images does not fit gathers from global memory instead.
template <class T, int DB>
__global__ __launch_bounds__(APPLY_BLOCK) void k_apply_planned(
    const int32_t* __restrict__ rowptr, const int32_t* __restrict__ col,
    const uint16_t* __restrict__ off, const int32_t* __restrict__ box,
    const T* __restrict__ w, const T* __restrict__ x, T* __restrict__ y,
    int64_t nrows, int64_t ncols, int64_t src_gy, int64_t batch, ApplyGrid G,
    int64_t lds_bytes)
{
    extern __shared__ __align__(16) unsigned char lds_raw[];
    CellVals<T, DB>* patch = reinterpret_cast<CellVals<T, DB>*>(lds_raw);
    const int64_t nb = gridDim.x;  // a multiple of NUM_XCD
    const int64_t b = blockIdx.x;
    const int64_t tile = (b % NUM_XCD) * (nb / NUM_XCD) + b / NUM_XCD;
    if (tile >= G.ntiles) return;  // uniform per block
    const int32_t i0 = box[4 * tile + 0], j0 = box[4 * tile + 1];
    const int32_t rows = box[4 * tile + 2], cols = box[4 * tile + 3];
    const int64_t cells = (int64_t)rows * cols;
    const int64_t d0 = (int64_t)blockIdx.y * DB;
    const int32_t nd = (int32_t)(batch - d0 < DB ? batch - d0 : DB);
    const bool staged = cells > 0 && cells * DB * (int64_t)sizeof(T) <= lds_bytes;
    if (staged) {
        stage_cells<T, DB>(patch, x + d0 * ncols + (int64_t)i0 * src_gy + j0, ncols, src_gy,
                           rows, cols, nd);
        __syncthreads();
    }
    const int32_t ti = (int32_t)(tile / G.ntx), tj = (int32_t)(tile - (int64_t)ti * G.ntx);
    const int32_t tw = (int32_t)G.tw;
    const int64_t i = (int64_t)ti * G.th + (int32_t)threadIdx.x / tw;
    const int64_t j = (int64_t)tj * G.tw + (int32_t)threadIdx.x % tw;
    if (i >= G.gx || j >= G.gy) return;
    const int64_t r = i * G.gy + j;
    const int32_t s = rowptr[r], e = rowptr[r + 1];
    T acc[DB];
#pragma unroll
    for (int m = 0; m < DB; m++) acc[m] = T(0);
    if (staged) {
        int32_t q = s;
        // four entries' loads in flight at once; the terms are still added
        // one at a time in column order
        for (; q + 4 <= e; q += 4) {
            int32_t o[4];
            T wq[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                o[u] = off[q + u];
                wq[u] = w[q + u];
            }
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const CellVals<T, DB> cv = patch[o[u]];
#pragma unroll
                for (int m = 0; m < DB; m++) acc[m] = acc[m] + wq[u] * cv.v[m];
            }
        }
        for (; q < e; q++) {
            const CellVals<T, DB> cv = patch[off[q]];
            const T wq = w[q];
#pragma unroll
            for (int m = 0; m < DB; m++) acc[m] = acc[m] + wq * cv.v[m];
        }
    } else {
        const T* xb = x + d0 * ncols;
        for (int32_t q = s; q < e; q++) {
            const int64_t c = col[q];
            const T wq = w[q];
#pragma unroll
            for (int m = 0; m < DB; m++)
                if (m < nd) acc[m] = acc[m] + wq * xb[m * ncols + c];
        }
    }
    T* yb = y + d0 * nrows + r;
#pragma unroll
    for (int m = 0; m < DB; m++)
        if (m < nd) store_result<false>(&yb[m * nrows], acc[m]);
}

// The planned apply with all images in one block: the lane's CSR entries
// (up to MAXE) are loaded once into registers, then for each group of DB
// images the block stages the input patch in LDS and gathers from it.  The
// entries and row pointers are read once per launch instead of once per
// image group, and the blocks (one per tile) stay resident longer.
template <class T, int DB, int MAXE, bool MERGE>
__global__ __launch_bounds__(APPLY_BLOCK) void k_apply_rounds(
    const int32_t* __restrict__ rowptr, const int32_t* __restrict__ col,
    const uint16_t* __restrict__ off, const int32_t* __restrict__ box,
    const T* __restrict__ w, const T* __restrict__ x, T* __restrict__ y,
    int64_t nrows, int64_t ncols, int64_t src_gy, int64_t batch, ApplyGrid G,
    int64_t lds_bytes)
{
    extern __shared__ __align__(16) unsigned char lds_raw[];
    CellVals<T, DB>* patch = reinterpret_cast<CellVals<T, DB>*>(lds_raw);
    const int64_t nb = gridDim.x;  // a multiple of NUM_XCD
    const int64_t b = blockIdx.x;
    const int64_t tile = (b % NUM_XCD) * (nb / NUM_XCD) + b / NUM_XCD;
    if (tile >= G.ntiles) return;  // uniform per block
    const int32_t i0 = box[4 * tile + 0], j0 = box[4 * tile + 1];
    const int32_t rows = box[4 * tile + 2], cols = box[4 * tile + 3];
    const int32_t ncell = rows * cols;
    const int32_t ti = (int32_t)(tile / G.ntx), tj = (int32_t)(tile - (int64_t)ti * G.ntx);
    const int32_t tw = (int32_t)G.tw;
    const int64_t i = (int64_t)ti * G.th + (int32_t)threadIdx.x / tw;
    const int64_t j = (int64_t)tj * G.tw + (int32_t)threadIdx.x % tw;
    const bool valid = i < G.gx && j < G.gy;
    const int64_t r = valid ? i * G.gy + j : 0;
    int32_t s = 0, e = 0;
    if (valid) {
        s = rowptr[r];
        e = rowptr[r + 1];
    }
    const int32_t cnt = e - s;
    int32_t ro[MAXE];
    T rw[MAXE];
#pragma unroll
    for (int q = 0; q < MAXE; q++) {
        if (q < cnt) {
            ro[q] = off[s + q];
            rw[q] = w[s + q];
        }
    }
    const bool fits = ncell > 0 && (int64_t)ncell * DB * (int64_t)sizeof(T) <= lds_bytes;
    for (int64_t d0 = 0; d0 < batch; d0 += DB) {
        const int32_t nd = (int32_t)(batch - d0 < DB ? batch - d0 : DB);
        if (fits) {
            stage_cells<T, DB>(patch, x + d0 * ncols + (int64_t)i0 * src_gy + j0, ncols, src_gy,
                               rows, cols, nd);
            __syncthreads();
        }
        if (valid) {
            T acc[DB];
#pragma unroll
            for (int m = 0; m < DB; m++) acc[m] = T(0);
            if (fits) {
                // (the accumulators of images past nd add 0 and are not stored)
#pragma unroll
                for (int q = 0; q < MAXE; q++) {
                    if (q < cnt) {
                        const CellVals<T, DB> cv = patch[ro[q]];
#pragma unroll
                        for (int m = 0; m < DB; m++) acc[m] = acc[m] + rw[q] * cv.v[m];
                    }
                }
                for (int32_t q = s + MAXE; q < e; q++) {
                    const CellVals<T, DB> cv = patch[off[q]];
                    const T wq = w[q];
#pragma unroll
                    for (int m = 0; m < DB; m++) acc[m] = acc[m] + wq * cv.v[m];
                }
            } else {
                const T* xg = x + d0 * ncols;
                for (int32_t q = s; q < e; q++) {
                    const int64_t c = col[q];
                    const T wq = w[q];
#pragma unroll
                    for (int m = 0; m < DB; m++)
                        if (m < nd) acc[m] = acc[m] + wq * xg[m * ncols + c];
                }
            }
            T* yb = y + d0 * nrows + r;
#pragma unroll
            for (int m = 0; m < DB; m++)
                if (m < nd) store_result<MERGE>(&yb[m * nrows], acc[m]);
        }
        if (fits) __syncthreads();  // the next group overwrites the patch
    }
}

__global__ void k_to_f32(const double* __restrict__ a, float* __restrict__ b,
                         int64_t n)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        b[i] = (float)a[i];
}

// ---- batched apply ---------------------------------------------------------
//
// Many applies, each with its own weights, in one launch.  Jobs are cut into
// blocks of one tile of output rows x JOB_DB images; block b finds its job in
// the jobs' block prefix.  The tiles and the accumulation per output are
// those of k_apply.
//
// Blocks are renumbered so each of the 8 XCDs takes one contiguous range of
// the blocks (blocks arrive round-robin over the XCDs): neighbouring tiles
// of a job gather overlapping inputs, which then stay in one XCD's L2
// instead of being fetched by all eight.
template <class T>
__global__ __launch_bounds__(APPLY_BLOCK) void k_apply_jobs(
    const JobDesc* __restrict__ jobs, const int64_t* __restrict__ block_prefix,
    int njobs, int64_t first, int64_t nblocks, const int32_t* __restrict__ abort_flag)
{
    __shared__ T prod[APPLY_BLOCK / 64][PROD_SLOTS];
    if (abort_flag && *abort_flag) return;  // uniform: one word for the grid
    const int64_t ng = gridDim.x;  // a multiple of NUM_XCD
    const int64_t b = first + (blockIdx.x % NUM_XCD) * (ng / NUM_XCD) + blockIdx.x / NUM_XCD;
    if (b >= nblocks) return;
    const JobDesc& J = jobs[seg_of(block_prefix, njobs, b)];
    const uint32_t lt = (uint32_t)(b - J.block_base), nrt = (uint32_t)J.nrt;
    const uint32_t ntx = (uint32_t)J.ntx, grp = lt / nrt, tile = lt - grp * nrt;
    const int64_t ti = tile / ntx, tj = tile % ntx;
    const int64_t d0 = (int64_t)grp * JOB_DB;
    const int64_t nd = J.batch - d0 < JOB_DB ? J.batch - d0 : JOB_DB;
    apply_rows<false, T>(J.rowptr, J.col, (const T*)J.w, (const T*)J.x + d0 * J.ncols,
                  (T*)J.y + d0 * J.nrows, J.nrows, J.ncols, (int32_t)nd, J.gy, ti * J.th,
                  tj * J.tw, J.th, prod[threadIdx.x / 64]);
}

namespace {

// Tile width, and how results are stored, for the apply with a plan.
//
// A nontemporal store sends what it holds of a 64-byte piece to memory by
// itself.  Where the output's rows are whole pieces, so are a tile's, and its
// results are stored nontemporal.  Elsewhere a tile's row ends in two pieces that
// the neighbouring tiles also write: while the images fit the Infinity Cache with
// room to spare, they are stored through the caches, which merge the parts;
// beyond that, tiles are two or four times as wide (fewer parts), the less the
// more input cells there are to an output, as a wider tile's patch leaves fewer
// images per pass; and up to FEW_BYTES the parts cost less than the caches' way
// (or are left to the wider tiles).  FP32 tiles are 32 wide, 128 bytes, unless the
// input is the finer grid or, with the parts merged, the images take several
// passes (5 of 1202 x 1501 -> 1000 x 1334 24-26 us 16 wide, 22-25 32 wide, the
// adjoint 25-28 and 25-28).  us, 16 wide nontemporal /
// 32 wide nontemporal / 16 wide merged / 64 wide nontemporal, 16 images unless
// given, where the grids' angles make a range:
//   whole pieces
//     2049^2 -> 1537^2 FP64 192-234 / 185-284 / 200-242, its adjoint 231-287 /
//       212-324 / 231-302; FP32 144-150 / 109-151 / 138-166
//     1401^2 -> 1001^2 adjoint FP64 72-89 / 70-99 / 119-165
//     1501^2 -> 2001^2 FP32 81-103 / 76-109 / 149-184 / 77-152 (62.5 lines a row)
//   others
//     803^2 -> 642^2 adjoint FP64, 2 images 9.6-12.7 / 9.6-12.6 / 10.5-12.7 (17 MB);
//       FP32 37 / 26-29 / 19-24 (67 MB)
//     701^2 -> 1400^2 FP64 155-164 / 103-110 / 105-118 / 79-86 (313 MB); FP32
//       109-117 / 70-79 / 37-40 / 49-59 (157 MB)
//     1204^2 -> 903^2 FP64 74-78 / 56-84 / 79-91 (289 MB)
//     1530^2 -> 1161^2 adjoint FP32 157-161 / 106-117 / 99-107 / 75-118 (236 MB)
// (A tile as wide as it can be without its patch growing depends on the angle of
// the grids, which is not known here.)
constexpr int64_t LINE = 128, PIECE = 64;
constexpr double FEW_BYTES = 50e6, MERGE_BYTES_8 = 130e6, MERGE_BYTES_4 = 190e6;

struct PlannedShape {
    int widen;   // tiles g_tile_w << widen
    bool merge;  // results stored through the caches
};

PlannedShape planned_shape(int64_t row_bytes, int64_t value_bytes, double bytes, double c,
                           int64_t images)
{
    const bool lines = row_bytes % LINE == 0, pieces = row_bytes % PIECE == 0;
    const bool few = bytes <= FEW_BYTES;
    const bool small = bytes <= (value_bytes < 8 ? MERGE_BYTES_4 : MERGE_BYTES_8);
    if (value_bytes >= 8) {
        if (pieces) return {!lines && !small && c <= 1.75, false};
        const bool merge = small && !few;
        return {!merge && c <= 1.9, merge};
    }
    if (lines) return {c <= 2.2, false};
    if (few && c <= 2.2) return {1, false};
    if (small) return {(!pieces && c <= 0.75) || (images <= JOB_DB && c <= 1.5), true};
    return {c <= 0.75 && !pieces ? 2 : c <= 2.2, false};
}

int g_tile_w = 16;
int g_images_per_pass = 8;
// staged patch per block above which fewer images are staged per pass: at
// 32 KiB the FP64 forward apply of the plain 2049^2 -> 1537^2 pair stages 4
// images per pass and holds four blocks per CU instead of three (5 % faster);
// FP32 and the adjoints stage 8 either way
int64_t g_lds_limit = 32 * 1024;
bool g_use_plan = true;
bool g_rounds = true;  // one block per tile looping over image groups
std::mutex g_plan_mu;
std::mutex g_use_mu;

// Waits for the applies of W queued on streams other than its own.
void wait_uses(rg_weights* W)
{
    std::lock_guard<std::mutex> lk(g_use_mu);
    for (auto& u : W->uses)
        if (hipEventSynchronize(u.second) != hipSuccess)
            (void)hipGetLastError();  // (recorded in a capture: nothing to wait for)
}

ApplyGrid make_grid(const int64_t* shape, int64_t nrows, int64_t tile_w)
{
    ApplyGrid G;
    G.gx = shape[0];
    G.gy = shape[1];
    if (G.gx * G.gy != nrows) {  // shape unknown: one long row
        G.gx = 1;
        G.gy = nrows;
    }
    G.tw = tile_w;
    if (G.gx == 1 || G.tw > G.gy) G.tw = APPLY_BLOCK;
    G.th = APPLY_BLOCK / G.tw;
    G.ntx = (G.gy + G.tw - 1) / G.tw;
    G.ntiles = G.ntx * ((G.gx + G.th - 1) / G.th);
    return G;
}

// Whether an apply without a plan gives every row a wavefront: us of chunks /
// of a wavefront a row, 1 image, 31 to 69 entries a row: 2601 rows 15 / 11, 1764
// 22 / 11, 7225 21 / 12, 42025 12 / 23, 28900 18 / 18, 16384 42 / 14; eight
// images 12 / 11, 19 / 11, 20 / 13, 31 / 50, 30 / 38, 38 / 38; eight jobs of 1764
// rows and 1, 3 and 8 images 29 / 19, 62 / 18, 167 / 26, of 7225 rows 29 / 51, 60 /
// 48, 143 / 71, of 2601 rows 18 / 22, 34 / 21, 94 / 31.
bool long_rows(int64_t nrows, int64_t nnz, int64_t images)
{
    return nnz >= LONG_ENTRIES * nrows ||
           (nrows <= LONG_FEW_ROWS && nnz >= (images > 1 ? LONG_FEW : LONG_FEW_ONE) * nrows);
}

// Tiles of an apply without a plan: 64 columns of four grid rows (16 or 32
// columns of more rows measure the same).  Grids of narrow rows are taken as
// one long row, where a block's consecutive rows are a compact patch too; so
// are rows of unknown shape.  Long rows are a grid one column wide.
ApplyGrid gather_grid(const int64_t* shape, int64_t nrows, int64_t nnz, int64_t images)
{
    ApplyGrid G;
    if (long_rows(nrows, nnz, images)) {
        G.gx = nrows;
        G.gy = G.tw = G.ntx = 1;
        G.th = APPLY_BLOCK / 64;
        G.ntiles = (nrows + G.th - 1) / G.th;
        return G;
    }
    G.gx = shape[0];
    G.gy = shape[1];
    G.tw = 64;
    // (grids of narrow rows as well: a block's consecutive rows are a compact
    // patch there)
    if (G.gx * G.gy != nrows || G.gy < 64) {
        G.gx = 1;
        G.gy = nrows;
        G.tw = APPLY_BLOCK;
    }
    G.th = APPLY_BLOCK / G.tw;
    G.ntx = (G.gy + G.tw - 1) / G.tw;
    G.ntiles = G.ntx * ((G.gx + G.th - 1) / G.th);
    return G;
}

bool plan_fits(const rg_weights::Plan& P, const ApplyGrid& G, int64_t src_gy)
{
    return P.tile_w == G.tw && P.gx == G.gx && P.gy == G.gy && P.src_gy == src_gy;
}

// The plan of one direction for tiles g_tile_w << widen of the output grid
// (made on first use on stream s; later applies on other streams must be
// ordered after it), and the tiles.  A plan cannot be made under capture (it
// ends in a host read): there, any plan the direction has serves, and without
// one the apply goes without.
int ensure_plan(rg_weights* W, int dir, int widen, const int32_t* rowptr,
                const int32_t* col, const int64_t* shape, int64_t nrows, int64_t src_gy,
                int64_t batch, hipStream_t s, rg_weights::Plan** out, ApplyGrid* tiles)
{
    *out = nullptr;
    const auto grid = [&](int wide) {
        return make_grid(shape, nrows, std::min(g_tile_w << wide, APPLY_BLOCK));
    };
    ApplyGrid G = grid(widen);
    // below PLAN_MIN_ROWS outputs the gathered input stays in L2 anyway and
    // a plan (two kernels and a host wait) would only add latency; one image
    // is faster without (2049^2 -> 1537^2 FP64 31 against 37 us, FP32 25
    // against 30, their adjoints 38 against 49 and 29 against 42; two images
    // are even, and from four on the plan is faster)
    if (!g_use_plan || batch == 1 || G.gx == 1 || W->nnz == 0 || G.gx * G.gy < PLAN_MIN_ROWS)
        return RG_OK;
    std::lock_guard<std::mutex> lk(g_plan_mu);
    if (!plan_fits(W->plan[dir][widen], G, src_gy) && capturing(s)) {
        widen = -1;
        for (int k = 0; k < 3; k++)
            if (plan_fits(W->plan[dir][k], grid(k), src_gy)) widen = k;
        if (widen < 0) return RG_OK;
        G = grid(widen);
    }
    rg_weights::Plan& P = W->plan[dir][widen];
    if (!plan_fits(P, G, src_gy)) {
        // (a plan that is replaced may still be read by applies on other streams)
        if (P.box) wait_uses(W);
        dev_free(P.box);
        dev_free(P.off);
        P.box = nullptr;
        P.off = nullptr;
        P.tile_w = 0;
        if (s != W->home) W->off_home = true;
        int st = dev_alloc((void**)&P.box, 4 * sizeof(int32_t) * G.ntiles, s);
        if (st == RG_OK) st = dev_alloc((void**)&P.off, sizeof(uint16_t) * W->nnz, s);
        if (st == RG_ERR_MEMORY) {  // the apply works without
            dev_free(P.box);
            P.box = nullptr;
            return RG_OK;
        }
        RG_TRY(st);
        k_plan<<<(unsigned)G.ntiles, APPLY_BLOCK, 0, s>>>(rowptr, col, G, src_gy,
                                                        P.box, P.off);
        DevBuf<int64_t> mx;
        RG_TRY(mx.alloc(1, s));
        k_plan_max<<<1, PLAN_MAX_BLOCK, 0, s>>>(P.box, G.ntiles, mx.p);
        RG_HIP(hipGetLastError());
        RG_TRY(read_scalars(mx.p, &P.max_cells, sizeof(int64_t), s));
        P.tile_w = G.tw;
        P.gx = G.gx;
        P.gy = G.gy;
        P.src_gy = src_gy;
    }
    *out = &P;
    *tiles = G;
    return RG_OK;
}

template <class T>
int launch_apply(rg_weights* W, int dir, const int32_t* rowptr,
                 const int32_t* col, const T* w, const T* x, T* y,
                 int64_t nrows, int64_t ncols, const int64_t* shape,
                 int64_t src_gy, int64_t batch, hipStream_t s)
{
    if (nrows == 0 || batch == 0) return RG_OK;
    const double bytes = (double)batch * (nrows + ncols) * sizeof(T);
    // (a shape that is not known has no plan)
    const PlannedShape planned = planned_shape(shape[1] * (int64_t)sizeof(T), sizeof(T), bytes,
                                               (double)ncols / (double)nrows, batch);
    ApplyGrid G;
    rg_weights::Plan* P = nullptr;
    RG_TRY(ensure_plan(W, dir, planned.widen, rowptr, col, shape, nrows, src_gy, batch, s, &P, &G));
    int32_t sb = 0;
    if (!P) {
        G = gather_grid(shape, nrows, W->nnz, batch);
        sb = (int32_t)std::min<int64_t>(batch, JOB_DB);
        while (sb > 1 && G.ntiles * ((batch + sb - 1) / sb) < SPLIT_TILES) sb = (sb + 1) / 2;
    }
    const int64_t nb = (G.ntiles + NUM_XCD - 1) / NUM_XCD * NUM_XCD;
    int db = g_images_per_pass;
    while (db > 1 && db > batch) db >>= 1;
    // staged patches: stage fewer images per pass rather than fall back to
    // the direct gather for the largest tiles
    while (P && db > 1 && P->max_cells * db * (int64_t)sizeof(T) > g_lds_limit) db >>= 1;
    dim3 g((unsigned)nb, (unsigned)((batch + db - 1) / db)), bl(APPLY_BLOCK);
    if (P && g_rounds) {
        int64_t lds = P->max_cells * db * (int64_t)sizeof(T);
        lds = (lds + 255) / 256 * 256;
        if (lds > LDS_BYTES) lds = LDS_BYTES;
        dim3 g1((unsigned)nb);
        // rows of more than 8 entries would read the rest once per image
        // group: the adjoint of 1025^2 -> 1500^2 (7.6 a row where there are
        // any, at most 12), 16 images: FP64 265 -> 195 us, FP32 121 -> 93; at
        // three or four a row the longer row costs 8 % in FP32, at five 1 or 2 %;
        // in FP64 it gains 0 to 8 % from 4.5 a row on
        const bool long_rows = 2 * W->nnz >= (sizeof(T) < 8 ? 11 : 9) * nrows;
        const bool merge = planned.merge;
#define RG_ROUNDS_K(D, E, M)                                                           \
    k_apply_rounds<T, D, E, M><<<g1, bl, (size_t)lds, s>>>(                            \
        rowptr, col, P->off, P->box, w, x, y, nrows, ncols, src_gy, batch, G, lds)
#define RG_ROUNDS(D)                                                                   \
    do {                                                                               \
        if (long_rows && merge) RG_ROUNDS_K(D, 12, true);                              \
        else if (long_rows) RG_ROUNDS_K(D, 12, false);                                 \
        else if (merge) RG_ROUNDS_K(D, 8, true);                                       \
        else RG_ROUNDS_K(D, 8, false);                                                 \
    } while (0)
        switch (db) {
        case 16: RG_ROUNDS(16); break;
        case 8: RG_ROUNDS(8); break;
        case 4: RG_ROUNDS(4); break;
        case 2: RG_ROUNDS(2); break;
        default: RG_ROUNDS(1); break;
        }
#undef RG_ROUNDS
#undef RG_ROUNDS_K
    } else if (P) {
        int64_t lds = P->max_cells * db * (int64_t)sizeof(T);
        lds = (lds + 255) / 256 * 256;
        if (lds > LDS_BYTES) lds = LDS_BYTES;
#define RG_PLANNED(D)                                                                  \
    k_apply_planned<T, D><<<g, bl, (size_t)lds, s>>>(                                  \
        rowptr, col, P->off, P->box, w, x, y, nrows, ncols, src_gy, batch, G, lds)
        switch (db) {
        case 16: RG_PLANNED(16); break;
        case 8: RG_PLANNED(8); break;
        case 4: RG_PLANNED(4); break;
        case 2: RG_PLANNED(2); break;
        default: RG_PLANNED(1); break;
        }
#undef RG_PLANNED
    } else {
        const dim3 gs((unsigned)nb, (unsigned)((batch + sb - 1) / sb));
        // (a wavefront stores 64 values of a row: ends at whole lines, or merged
        // where the images fit the cache)
        const bool lines = shape[0] * shape[1] == nrows &&
                           shape[1] * (int64_t)sizeof(T) % LINE == 0;
        if (!lines && bytes <= (sizeof(T) < 8 ? MERGE_BYTES_4 : MERGE_BYTES_8))
            k_apply<T, true><<<gs, bl, 0, s>>>(rowptr, col, w, x, y, nrows, ncols, batch, sb, G);
        else
            k_apply<T, false><<<gs, bl, 0, s>>>(rowptr, col, w, x, y, nrows, ncols, batch, sb, G);
    }
    RG_HIP(hipGetLastError());
    return RG_OK;
}

std::mutex g_f32_mu;

int ensure_f32(rg_weights* W, hipStream_t s)
{
    std::lock_guard<std::mutex> lk(g_f32_mu);
    if (W->val_out_f32 || W->nnz == 0) return RG_OK;
    float *a = nullptr, *b = nullptr;
    if (s != W->home) W->off_home = true;
    RG_TRY(dev_alloc((void**)&a, W->nnz * sizeof(float), s));
    int st = dev_alloc((void**)&b, W->nnz * sizeof(float), s);
    if (st != RG_OK) {
        dev_free(a);
        return st;
    }
    unsigned gs = grid_for(W->nnz, 256);
    if (gs > 8192) gs = 8192;
    k_to_f32<<<gs, 256, 0, s>>>(W->val_in, a, W->nnz);
    k_to_f32<<<gs, 256, 0, s>>>(W->val_out, b, W->nnz);
    RG_HIP(hipGetLastError());
    // other streams may use the copies as soon as they are published
    RG_HIP(hipStreamSynchronize(s));
    W->val_in_f32 = a;
    W->val_out_f32 = b;
    return RG_OK;
}

}  // namespace

int note_use(rg_weights* W, hipStream_t s)
{
    if (s == W->home && !W->off_home) return RG_OK;
    std::lock_guard<std::mutex> lk(g_use_mu);
    hipEvent_t ev = nullptr;
    for (auto& u : W->uses)
        if (u.first == s) ev = u.second;
    if (!ev) {
        RG_HIP(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
        W->uses.emplace_back(s, ev);
    }
    RG_HIP(hipEventRecord(ev, s));
    return RG_OK;
}

namespace {

int check_apply(rg_weights* W, const void* vin, void* vout, int64_t batch)
{
    if (!W) return fail(RG_ERR_ARGUMENT, "weights handle is NULL");
    if (batch < 0) return fail(RG_ERR_ARGUMENT, "negative batch");
    if (batch > 0 && (!vin || !vout))
        return fail(RG_ERR_ARGUMENT, "values pointer is NULL");
    if (injected_failure("apply"))
        return fail(RG_ERR_INJECTED, "injected apply failure");
    return RG_OK;
}

// Pinned staging of a batched apply's job table, one per host thread; the
// event marks when the previous upload from it has been consumed.
struct JobUpload {
    void* buf = nullptr;
    size_t cap = 0;
    hipEvent_t done = nullptr;
    int device = -1;  // the device `done` belongs to
    bool recorded = false;
};

// The blocks of a job table, in launches within LAUNCH_THREADS.
template <class T>
int launch_jobs(const JobDesc* jobs, const int64_t* prefix, int njobs, int64_t nblocks,
                const int32_t* abort_flag, hipStream_t s)
{
    constexpr int64_t MOST = LAUNCH_THREADS / APPLY_BLOCK / NUM_XCD * NUM_XCD;
    for (int64_t b = 0; b < nblocks; b += MOST) {
        const int64_t n = std::min(MOST, (nblocks - b + NUM_XCD - 1) / NUM_XCD * NUM_XCD);
        k_apply_jobs<T><<<(unsigned)n, APPLY_BLOCK, 0, s>>>(jobs, prefix, njobs, b, nblocks,
                                                            abort_flag);
    }
    RG_HIP(hipGetLastError());
    return RG_OK;
}

int launch_jobs_common(const rg_apply_job* jobs, int64_t njobs, bool f32,
                       hipStream_t s)
{
    if (njobs < 0) return fail(RG_ERR_ARGUMENT, "negative job count");
    if (njobs > 0 && !jobs) return fail(RG_ERR_ARGUMENT, "jobs is NULL");
    std::vector<JobDesc> table;
    std::vector<int64_t> prefix;
    table.reserve(njobs);
    int64_t nblocks = 0;
    for (int64_t k = 0; k < njobs; k++) {
        const rg_apply_job& jb = jobs[k];
        rg_weights* W = jb.weights;
        RG_TRY(check_apply(W, jb.values_input, jb.values_output, jb.batch));
        if (f32) RG_TRY(ensure_f32(W, s));
        JobDesc d;
        if (jb.transpose) {
            d.rowptr = W->rowptr_in;
            d.col = W->col_in;
            d.w = f32 ? (const void*)W->val_in_f32 : (const void*)W->val_in;
            d.nrows = W->n_in;
            d.ncols = W->n_out;
        } else {
            d.rowptr = W->rowptr_out;
            d.col = W->col_out;
            d.w = f32 ? (const void*)W->val_out_f32 : (const void*)W->val_out;
            d.nrows = W->n_out;
            d.ncols = W->n_in;
        }
        d.x = jb.values_input;
        d.y = jb.values_output;
        d.batch = jb.batch;
        if (d.nrows == 0 || d.batch == 0) continue;
        const int64_t* shape = jb.transpose ? W->shape_in : W->shape_out;
        job_tiles(d, shape[0], shape[1], W->nnz);
        d.block_base = nblocks;
        prefix.push_back(nblocks);
        nblocks += d.nrt * ((d.batch + JOB_DB - 1) / JOB_DB);
        table.push_back(d);
    }
    if (table.empty()) return RG_OK;
    if (nblocks >= INT32_MAX) return fail(RG_ERR_ARGUMENT, "batched apply too large");
    const size_t tbytes = table.size() * sizeof(JobDesc);
    const size_t pbytes = prefix.size() * sizeof(int64_t);
    const size_t poff = (tbytes + 255) / 256 * 256, bytes = poff + pbytes;
    static thread_local JobUpload up;
    if (up.recorded) RG_HIP(hipEventSynchronize(up.done));
    if (bytes > up.cap) {
        if (up.buf) (void)hipHostFree(up.buf);
        up.buf = nullptr;
        up.cap = 0;
        const size_t sz = std::max<size_t>(bytes, 1 << 16);
        RG_HIP(hipHostMalloc(&up.buf, sz, hipHostMallocDefault));
        up.cap = sz;
    }
    int device = 0;
    RG_HIP(hipGetDevice(&device));
    if (up.done && up.device != device) {  // an event records on its own device only
        (void)hipEventDestroy(up.done);
        up.done = nullptr;
    }
    if (!up.done) {
        RG_HIP(hipEventCreateWithFlags(&up.done, hipEventDisableTiming));
        up.device = device;
    }
    std::memcpy(up.buf, table.data(), tbytes);
    std::memcpy((char*)up.buf + poff, prefix.data(), pbytes);
    DevBuf<unsigned char> dt;
    RG_TRY(dt.alloc(bytes, s));
    RG_HIP(hipMemcpyAsync(dt.p, up.buf, bytes, hipMemcpyHostToDevice, s));
    RG_HIP(hipEventRecord(up.done, s));
    up.recorded = true;
    const JobDesc* d_jobs = (const JobDesc*)dt.p;
    const int64_t* d_prefix = (const int64_t*)(dt.p + poff);
    if (f32)
        RG_TRY(launch_jobs<float>(d_jobs, d_prefix, (int)table.size(), nblocks, nullptr, s));
    else
        RG_TRY(launch_jobs<double>(d_jobs, d_prefix, (int)table.size(), nblocks, nullptr, s));
    for (int64_t k = 0; k < njobs; k++) RG_TRY(note_use(jobs[k].weights, s));
    return RG_OK;  // dt returns to the stream's pool after the kernel
}

}  // namespace

int apply_jobs_device(const JobDesc* jobs, const int64_t* prefix, int njobs, int64_t nblocks,
                      const int32_t* abort_flag, hipStream_t s)
{
    if (njobs == 0 || nblocks == 0) return RG_OK;
    if (nblocks >= INT32_MAX) return fail(RG_ERR_ARGUMENT, "batched apply too large");
    return launch_jobs<double>(jobs, prefix, njobs, nblocks, abort_flag, s);
}

void job_tiles(JobDesc& d, int64_t gx, int64_t gy, int64_t nnz)
{
    const int64_t shape[2] = {gx, gy};
    const ApplyGrid G = gather_grid(shape, d.nrows, nnz, d.batch);
    d.tw = (int32_t)G.tw;
    d.th = (int32_t)G.th;
    d.gy = G.gy;
    d.ntx = G.ntx;
    d.nrt = G.ntiles;
}

}  // namespace rg

using namespace rg;

extern "C" {

int rg_apply_f64(rg_weights_t w, int transpose, const double* values_input,
                 double* values_output, int64_t batch, void* stream)
{
    RG_TRY(check_apply(w, values_input, values_output, batch));
    hipStream_t s = (hipStream_t)stream;
    if (transpose)
        RG_TRY(launch_apply<double>(w, 1, w->rowptr_in, w->col_in, w->val_in,
                                    values_input, values_output, w->n_in,
                                    w->n_out, w->shape_in, w->shape_out[1],
                                    batch, s));
    else
        RG_TRY(launch_apply<double>(w, 0, w->rowptr_out, w->col_out, w->val_out,
                                    values_input, values_output, w->n_out, w->n_in,
                                    w->shape_out, w->shape_in[1], batch, s));
    return note_use(w, s);
}

int rg_apply_f32(rg_weights_t w, int transpose, const float* values_input,
                 float* values_output, int64_t batch, void* stream)
{
    RG_TRY(check_apply(w, values_input, values_output, batch));
    hipStream_t s = (hipStream_t)stream;
    RG_TRY(ensure_f32(w, s));
    if (transpose)
        RG_TRY(launch_apply<float>(w, 1, w->rowptr_in, w->col_in, w->val_in_f32,
                                   values_input, values_output, w->n_in,
                                   w->n_out, w->shape_in, w->shape_out[1],
                                   batch, s));
    else
        RG_TRY(launch_apply<float>(w, 0, w->rowptr_out, w->col_out, w->val_out_f32,
                                   values_input, values_output, w->n_out, w->n_in,
                                   w->shape_out, w->shape_in[1], batch, s));
    return note_use(w, s);
}

int rg_apply_batched_f64(const rg_apply_job* jobs, int64_t njobs, void* stream)
{
    return launch_jobs_common(jobs, njobs, false, (hipStream_t)stream);
}

int rg_apply_batched_f32(const rg_apply_job* jobs, int64_t njobs, void* stream)
{
    return launch_jobs_common(jobs, njobs, true, (hipStream_t)stream);
}

int rg_set_apply_tuning(int tile_w, int images_per_pass, int lds_kib, int rounds)
{
    if (rounds >= 0) g_rounds = rounds != 0;
    // negative tile_w: keep the tile width, turn the staged (planned) apply
    // off; the direct-gather kernel computes the same bits
    if (tile_w < 0) {
        g_use_plan = false;
        tile_w = -tile_w;
    } else if (tile_w > 0) {
        g_use_plan = true;
    }
    if (tile_w) {
        if (tile_w < 1 || tile_w > APPLY_BLOCK || APPLY_BLOCK % tile_w)
            return fail(RG_ERR_ARGUMENT, "tile_w must divide 256");
        g_tile_w = tile_w;
    }
    if (images_per_pass) {
        if (images_per_pass != 1 && images_per_pass != 2 && images_per_pass != 4 &&
            images_per_pass != 8 && images_per_pass != 16)
            return fail(RG_ERR_ARGUMENT, "images_per_pass must be 1, 2, 4, 8 or 16");
        g_images_per_pass = images_per_pass;
    }
    if (lds_kib) {
        if (lds_kib < 1 || lds_kib > LDS_BYTES / 1024)
            return fail(RG_ERR_ARGUMENT, "lds_kib must be in 1..64");
        g_lds_limit = (int64_t)lds_kib * 1024;
    }
    return RG_OK;
}

}  // extern "C"
