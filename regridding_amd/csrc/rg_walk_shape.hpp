// rg_walk_shape.hpp -- how a build's sweep rows are split among walk threads
// and how many triples each thread stages (host code).
#pragma once

#include <stdint.h>

#include <algorithm>
#include <cmath>

#include "../../include/regridding_amd.h"
#include "rg_sweep.hpp"

namespace rg {

// The split of the sweep rows into chunks, one walk thread each, and the
// triples staged per thread.
//
// A chunk is a serial chain of dependent loads and divisions, whose time grows
// with its triples (t of them), and costs a start search, whose time grows
// with the number of chunks (all triples W / t): their sum is least at a t
// that grows as sqrt(W).  A pass's edges emit about 2 (1 + c) triples each
// when they cross c static cell edges, c from the grids' cell counts (they
// are taken to cover each other, at a mean angle), and a pass's chunk is as
// many edges as make t.  Build times, 16 edges for every pass -> this rule:
//   67 x 190 -> 81 x 125 vertices   813 -> 389 us (the walk alone 469 -> 68)
//   129^2 -> 101^2                  721 -> 322
//   257^2 -> 193^2                  610 -> 354 (2 edges 359)
//   513^2 -> 385^2                  692 -> 485 (2 edges 483, 4 edges 478)
//   1025^2 -> 769^2                1013 -> 930 (4 edges 939, 8 edges 922)
// (below ONE_EDGE_WORK triples, about 270^2 -> 200^2, every chunk is one edge)
// and from about 2000^2 on t is at its bound, MAX_TRIPLES, and the chunks
// are the 16 edges they were.  Each pass stages 1.8 times its own chunks'
// expected triples: with 8 per edge for every pass, chunks of coarse sweeps
// over fine static grids overflowed and walked twice (64 mixed pairs of 33 to
// 1025 vertices per axis: the build 6.84 -> 5.56 ms), and with the most of any
// pass for all, one coarse pass among many fine ones made every thread stage
// as much as its own (9^2 -> 400^2 vertices 734 MB, now 83).
//
// An explicit edges_per_lane or stage_per_edge applies to every pass as given
// (a missing one of the two is 16 edges, or 8 triples).
struct WalkShape {
    static constexpr double MAX_TRIPLES = 72, ONE_EDGE_WORK = 1e6;
    static constexpr int64_t MAX_EDGES = 32, MIN_CAP = 16, MAX_CAP = 128;
    int64_t K;           // edges per chunk of every pass; 0: by expected work
    double target = 1;   // expected triples of a chunk
    int64_t cap = 0;     // triples staged per walk thread of every pass; 0: by pass

    struct Dims {
        int64_t rows, edges;  // sweep rows, edges per row
        double per_edge;      // expected triples per edge
    };

    static Dims dims(const rg_pair_desc& d, int p)
    {
        const bool in = p >= 2;
        const int64_t nxs = in ? d.nxi : d.nxo, nys = in ? d.nyi : d.nyo;
        const int64_t nxt = in ? d.nxo : d.nxi, nyt = in ? d.nyo : d.nyi;
        Dims q;
        q.rows = (p & 1) ? nxs : nys;
        q.edges = ((p & 1) ? nys : nxs) - 1;
        // 2 / pi: the mean of |cos| and |sin| over the angle
        const double c = 0.64 * (double)(nxt - 1 + nyt - 1) / (double)q.edges;
        q.per_edge = 2 * (1 + c);
        return q;
    }

    // Expected triples of a pair.
    static double triples(const rg_pair_desc& d)
    {
        double t = 0;
        for (int p = 0; p < 4; p++) {
            const Dims q = dims(d, p);
            t += (double)q.rows * (double)q.edges * q.per_edge;
        }
        return t;
    }

    WalkShape(const rg_pair_desc* pairs, int64_t npairs, int64_t edges, int64_t per_edge)
    {
        if (edges > 0 || per_edge > 0) {
            K = edges > 0 ? edges : 16;
            cap = K * (per_edge > 0 ? per_edge : 8);
            return;
        }
        K = 0;
        double work = 0;
        for (int64_t k = 0; k < npairs; k++) work += triples(pairs[k]);
        target = work < ONE_EDGE_WORK ? 1 : std::min(std::sqrt(work) / 105, MAX_TRIPLES);
    }

    // Edges per chunk of pass p of a pair: the target's, spread evenly over
    // the chunks of a row.
    int64_t edges_per_chunk(const rg_pair_desc& d, int p) const
    {
        if (K > 0) return K;
        const Dims q = dims(d, p);
        int64_t e = (int64_t)(target / q.per_edge + 0.5);
        e = std::max<int64_t>(1, std::min({e, MAX_EDGES, q.edges}));
        const int64_t chunks = (q.edges + e - 1) / e;
        return (q.edges + chunks - 1) / chunks;
    }

    // Triples staged per walk thread of pass p of a pair.
    int64_t staged(const rg_pair_desc& d, int p) const
    {
        if (cap > 0) return cap;
        const double expected = (double)edges_per_chunk(d, p) * dims(d, p).per_edge;
        return (int64_t)std::min((double)MAX_CAP, std::max((double)MIN_CAP, 1.8 * expected + 1));
    }

    // Walk threads of pass p of a pair.
    int64_t threads(const rg_pair_desc& d, int p) const
    {
        const Dims q = dims(d, p);
        const int64_t e = edges_per_chunk(d, p);
        return threads_of_pass(q.rows, (q.edges + e - 1) / e);
    }
};

// Device bytes of the working set of a pair's build, alone or as part of a
// batch: the staging and what overflows it, about 48 bytes a triple (records,
// their reduction, both CSR layouts) and about 100 a sweep edge (chunk, cell
// and row tables).  The chunks of a batch are no shorter than the pair's own,
// so they stage no more per edge, except that a row's edges divide less evenly
// into them (by 4/3 at most, three edges in chunks of two).
inline int64_t build_bytes(const rg_pair_desc& d)
{
    const WalkShape shape(&d, 1, 0, 0);
    double b = 0;
    for (int p = 0; p < 4; p++) {
        const WalkShape::Dims q = WalkShape::dims(d, p);
        const double chunk = (double)shape.edges_per_chunk(d, p) * q.per_edge;
        const double over = std::max(0.0, chunk - (double)shape.staged(d, p));
        b += 4.0 / 3 * 16 * (double)shape.threads(d, p) * ((double)shape.staged(d, p) + over);
        b += 100.0 * (double)q.rows * (double)q.edges;
    }
    return (int64_t)(b + 48 * WalkShape::triples(d));
}

}  // namespace rg
