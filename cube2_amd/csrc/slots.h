// Slot-parallel walks over an image's particles.
//
// The particles of a coarse cell are one contiguous run of slots, and an
// image's cells hold from none to 10^5 of them.  A wavefront per cell leaves
// the whole device waiting for the few that own a clump (C1's densest cell,
// 115,201 particles: 1800 dependent steps of one wavefront, 2-5 ms whatever
// the kernel).  Instead a block takes a fixed number of consecutive slots
// and finds the cells they lie in from the exclusive scan of the cell counts.
#pragma once
#include <algorithm>
#include <climits>

#include "common.h"

namespace cube2 {

constexpr int kSlotThreads = 256;
constexpr int kSlotChunk = 1024;  // slots a block takes at a time
constexpr int kSlotWin = 1024;    // cell starts staged in LDS at a time, at most

// n / d for n < 2^31 by a multiply (Granlund and Montgomery's round-up
// method: m = floor(2^32 (2^l - d) / d) + 1, l = ceil(log2 d)).
struct FastDiv {
    uint32_t d, m, l;
};
inline FastDiv make_fastdiv(uint32_t d) {
    uint32_t l = 0;
    while (((uint64_t)1 << l) < d) l++;
    const uint64_t m = (((uint64_t)1 << 32) * (((uint64_t)1 << l) - d)) / d + 1;
    return FastDiv{d, (uint32_t)m, l};
}
__device__ inline uint32_t fdiv(uint32_t n, const FastDiv& f) {
    return (__umulhi(n, f.m) + n) >> f.l;
}

// An image's geometry for cell index arithmetic.
struct SlotGeom {
    FastDiv nte, nnt, nc;
    int nt, ncb;
    uint32_t ncells;
};
inline SlotGeom make_slotgeom(const Geom& g) {
    SlotGeom s;
    s.nte = make_fastdiv((uint32_t)g.nte);
    s.nnt = make_fastdiv((uint32_t)g.p.nnt);
    s.nc = make_fastdiv((uint32_t)g.nc);
    s.nt = g.nt;
    s.ncb = g.ncb;
    s.ncells = (uint32_t)((int64_t)g.ntile * g.nte * g.nte * g.nte);
    return s;
}

// Extended cell q: its row (tile, k, j), and its coordinates.
struct CellPos {
    uint32_t row, tile;
    int i, j, k;
};
__device__ inline CellPos cell_pos(const SlotGeom& G, uint32_t q) {
    CellPos c;
    c.row = fdiv(q, G.nte);
    c.i = (int)(q - c.row * G.nte.d);
    const uint32_t p = fdiv(c.row, G.nte);
    c.j = (int)(c.row - p * G.nte.d);
    c.tile = fdiv(p, G.nte);
    c.k = (int)(p - c.tile * G.nte.d);
    return c;
}
__device__ inline void tile_pos(const SlotGeom& G, uint32_t t, int& tx, int& ty, int& tz) {
    const uint32_t a = fdiv(t, G.nnt), b = fdiv(a, G.nnt);
    tx = (int)(t - a * G.nnt.d);
    ty = (int)(a - b * G.nnt.d);
    tz = (int)b;
}

// The image coordinate of extended coordinate c of a tile (periodic).
__device__ inline int image_coord(const SlotGeom& G, int tile_c, int c) {
    const int nc = (int)G.nc.d;
    int g = tile_c * G.nt + c - G.ncb;
    // a halo may be wider than the image: g + nc * ncb >= 0
    uint32_t u = (uint32_t)(g + nc * G.ncb);
    return (int)(u - fdiv(u, G.nc) * (uint32_t)nc);
}

// Block-wide: the last q in [0, n) with start[q] <= v, for start ascending
// with start[0] <= v (the cell that holds v, empty cells before it skipped):
// 256 probes a round.
__device__ inline uint32_t block_last_le(const long long* __restrict__ start, uint32_t n, int64_t v) {
    uint32_t lo = 0, hi = n;
    while (hi - lo > 1) {
        const uint32_t step = (hi - lo + kSlotThreads - 1) / kSlotThreads;
        const uint64_t p = (uint64_t)lo + (uint64_t)threadIdx.x * step;
        const int k = __syncthreads_count(p < hi && start[p] <= v);
        lo += (uint32_t)max(k - 1, 0) * step;
        hi = min(hi, lo + step);
    }
    return lo;
}

// Block-wide walk of the n <= kSlotChunk slots from v0 on of the running slot
// count `start` [ncells + 1] (win: kSlotWin + 1 ints of LDS).  For each window
// of cells, body(begin, end, cell_of) with the slots [begin, end) it covers,
// counted from v0 in 32 bits (an image may have 2^31 slots and more);
// cell_of(v, s0, s1) gives slot v's cell and the cell's slot range, counted
// alike: a range may begin before v0 (by less than 2^31, the largest count),
// and one that ends 2^31 or more past v0 is cut there.  body is called
// block-uniformly and may synchronise.
template <class Body>
__device__ inline void walk_slots(const long long* __restrict__ start, uint32_t ncells, int64_t v0,
                                  int n, int* win, Body&& body) {
    for (int v = 0; v < n;) {
        const uint32_t q0 = block_last_le(start, ncells, v0 + v);
        // (as few as reach the end, where a cell holds several slots)
        int nw = (int)min((uint32_t)kSlotThreads, ncells - q0);
        if (start[q0 + nw] < v0 + n) nw = (int)min((uint32_t)kSlotWin, ncells - q0);
        for (int a = threadIdx.x; a <= nw; a += kSlotThreads)
            win[a] = (int)min(start[q0 + a] - (long long)v0, (long long)INT_MAX);
        __syncthreads();
        const int end = min(n, max(win[nw], v + 1));
        body(v, end, [&](int s, int& s0, int& s1) {
            int lo = 0, hi = nw;
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (win[mid] <= s) lo = mid;
                else hi = mid;
            }
            s0 = win[lo];
            s1 = win[lo + 1];
            return q0 + (uint32_t)lo;
        });
        __syncthreads();  // win is rewritten by the next window
        v = end;
    }
}

// Blocks of walk_all_slots over about n slots.
inline unsigned slot_blocks(int64_t n) {
    return std::min(ceil_div((size_t)std::max<int64_t>(n, 1), kSlotChunk), 1u << 20);
}

// Slots of the chunk at v0 of `total`.
__device__ inline int block_slots(int64_t total, int64_t v0) {
    return (int)min((long long)kSlotChunk, max((long long)(total - v0), 0ll));
}

// walk_slots over all `total` slots: body(v0, begin, end, cell_of) with slots
// counted from v0.
template <class Body>
__device__ inline void walk_all_slots(const long long* __restrict__ start, uint32_t ncells,
                                      int64_t total, int* win, Body&& body) {
    for (int64_t v0 = (int64_t)blockIdx.x * kSlotChunk; v0 < total; v0 += (int64_t)gridDim.x * kSlotChunk)
        walk_slots(start, ncells, v0, block_slots(total, v0), win,
                   [&](int b, int e, auto cell_of) { body(v0, b, e, cell_of); });
}

// Running slot counts of the cells (scan.hip: negative counts as 0) and,
// per row, what to add to a running count to get a slot: idx_b_r of the row
// less the running count at its end (0 where idx_b_r is the running total,
// as spine_image leaves it).
__device__ inline int64_t row_shift(const long long* __restrict__ start, const int64_t* __restrict__ idx_b_r,
                                    uint32_t row, uint32_t nte) {
    return idx_b_r[row] - start[(size_t)(row + 1) * nte];
}

}  // namespace cube2
