// The image layout on the device: the kick path's inputs rhoc, idx_b_r, xp,
// vp built from particle positions in HBM, as buffer_grid and spine_image
// produce them for one periodic image (buffer_grid.f90:13-155,
// variables.f90:146-216), halo copies included (the buffer_x copies of
// buffer_particle.f90:23-345 for a single image):
//   encode   global coarse cell and 16-bit in-cell position of every particle
//            (FP64, parameters.f90:87-88);
//   sort     stable radix sort (sort.hip) of (coarse cell, particle index): the order of
//            the particles of one cell is their input order;
//   starts   first sorted position of every coarse cell (binary search);
//   rhoc     particles per coarse cell of every tile's extended region (the
//            periodic neighbour's cell for halo cells);
//   slots    exclusive scan of rhoc: slot ranges per cell, idx_b_r = row ends;
//   gather   codes and velocities into sorted order;
//   fill     every slot copies its particle's code and velocity, a block per
//            1024 slots (slots.h).
#include <algorithm>
#include <cstring>

#include "common.h"
#include "engine.h"
#include "profile.h"
#include "scan.h"
#include "slots.h"
#include "sort.h"

namespace cube2 {

struct LayoutState {
    DevBuf gid, gid_sorted, idx, idx_sorted, code, code_sorted, vel_sorted, cnt, slot, sort_tmp,
        scan_tmp, red;
};
static LayoutState g_lay;

// Global coarse cell (z-major) and int16 code of each position, in the same
// FP64 operations as the host layout builder: p = pos mod ng (sign of the
// divisor), pc = p / ratio_cs, c = clamp(floor(pc)), u = clamp(floor((pc - c)
// * 65536)) stored as the int16 with the same bits.
__global__ void k_layout_encode(const double* __restrict__ pos, int64_t n, int ng, int ratio_cs,
                                int nc, uint32_t* __restrict__ gid, uint32_t* __restrict__ idx,
                                int16_t* __restrict__ code) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int g[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        double p = fmod(pos[3 * i + d], (double)ng);
        if (p != 0.0 && p < 0.0) p += (double)ng;
        const double pc = p / (double)ratio_cs;
        int c = (int)floor(pc);
        c = min(max(c, 0), nc - 1);
        const double frac = pc - (double)c;
        double u = floor(frac * 65536.0);
        u = fmin(fmax(u, 0.0), 65535.0);
        code[3 * i + d] = (int16_t)(uint16_t)u;
        g[d] = c;
    }
    gid[i] = (uint32_t)((g[2] * nc + g[1]) * nc + g[0]);
    idx[i] = (uint32_t)i;
}

// gstart[b] = first sorted position of a cell id >= b (b <= nbin): the
// cell starts straight from the sorted ids, by binary search.
__global__ void k_layout_starts(const uint32_t* __restrict__ gid_sorted, int64_t n, int64_t nbin,
                                int* __restrict__ gstart) {
    const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b > nbin) return;
    int64_t lo = 0, hi = n;
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if ((int64_t)gid_sorted[mid] < b) lo = mid + 1;
        else hi = mid;
    }
    gstart[b] = (int)lo;
}

// Global coarse cell of extended cell (i, j, k) of tile t (periodic).
__device__ inline int ext_global(int64_t q, int nt, int ncb, int nte, int nnt, int nc) {
    const int i = (int)(q % nte), j = (int)((q / nte) % nte), k = (int)((q / ((int64_t)nte * nte)) % nte);
    const int t = (int)(q / ((int64_t)nte * nte * nte));
    const int tx = t % nnt, ty = (t / nnt) % nnt, tz = t / (nnt * nnt);
    const int gx = ((tx * nt + i - ncb) % nc + nc) % nc;
    const int gy = ((ty * nt + j - ncb) % nc + nc) % nc;
    const int gz = ((tz * nt + k - ncb) % nc + nc) % nc;
    return (gz * nc + gy) * nc + gx;
}

__global__ void k_layout_rhoc(const int* __restrict__ gstart, int64_t ncells, int nt, int ncb,
                              int nte, int nnt, int nc, int* __restrict__ rhoc) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= ncells) return;
    const int g = ext_global(q, nt, ncb, nte, nnt, nc);
    rhoc[q] = gstart[g + 1] - gstart[g];
}

__global__ void k_layout_rows(const long long* __restrict__ slot, int64_t nrows, int nte,
                              int64_t* __restrict__ idx_b_r) {
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r < nrows) idx_b_r[r] = slot[(r + 1) * nte];  // exclusive start of the next row
}

// Codes and velocities in sorted (cell) order, so that the fill below copies
// runs instead of gathering every particle once per tile that holds it.
__global__ void k_layout_gather(const uint32_t* __restrict__ src, int64_t n,
                                const int16_t* __restrict__ code, const float* __restrict__ vel,
                                int16_t* __restrict__ code_s, float* __restrict__ vel_s) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const int64_t s = src[p];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        code_s[3 * p + d] = code[3 * s + d];
        vel_s[3 * p + d] = vel ? vel[3 * s + d] : 0.0f;
    }
}

// A block per kSlotChunk slots: each slot's particle from its cell's run of
// the sorted arrays.  Bound by its stores (18 bytes a slot): 90 M slots at
// 256^3 in 0.85 ms, and 0.25 ms for the gather before it; a wavefront per
// cell that gathered every copy took 5.6 ms.
__global__ __launch_bounds__(kSlotThreads) void k_layout_fill(
    SlotGeom G, const int* __restrict__ gstart, const long long* __restrict__ slot, int64_t total,
    const int16_t* __restrict__ code_s, const float* __restrict__ vel_s, int16_t* __restrict__ xp,
    float* __restrict__ vp) {
    __shared__ int win[kSlotWin + 1];
    const int64_t v0 = (int64_t)blockIdx.x * kSlotChunk;
    walk_slots(slot, G.ncells, v0, block_slots(total, v0), win, [&](int b, int e, auto cell_of) {
        for (int v = b + (int)threadIdx.x; v < e; v += kSlotThreads) {
            int s0, s1;
            const CellPos c = cell_pos(G, cell_of(v, s0, s1));
            int tx, ty, tz;
            tile_pos(G, c.tile, tx, ty, tz);
            const int nc = (int)G.nc.d;
            const int g = (image_coord(G, tz, c.k) * nc + image_coord(G, ty, c.j)) * nc +
                          image_coord(G, tx, c.i);
            const int64_t p = (int64_t)gstart[g] + (v - s0), d = v0 + v;
#pragma unroll
            for (int k = 0; k < 3; k++) {
                xp[3 * d + k] = code_s[3 * p + k];
                vp[3 * d + k] = vel_s[3 * p + k];
            }
        }
    });
}

int layout_build(const double* d_pos, const float* d_vel, int64_t n, int* d_rhoc,
                 int64_t* d_idx_b_r, int16_t* d_xp, float* d_vp, int64_t cap, int64_t* n_used) {
    ensure_params();
    Context& C = ctx();
    const Geom& g = C.g;
    if ((!d_pos && n > 0) || !d_rhoc || !d_idx_b_r || !n_used || n < 0 || n >= ((int64_t)1 << 31) ||
        (int64_t)g.nc * g.nc * g.nc >= ((int64_t)1 << 31)) {
        set_error("layout: null argument or size out of range");
        return CUBE2_ERR_ARG;
    }
    C2_TRY(ensure_init());
    hipStream_t s = C.stream;
    const int64_t nbin = (int64_t)g.nc * g.nc * g.nc;
    const int64_t ncells = (int64_t)g.ntile * g.nte * g.nte * g.nte;
    if (ncells >= ((int64_t)1 << 31)) {
        set_error("layout: more than 2^31 cells with the halos");
        return CUBE2_ERR_CAPACITY;
    }
    const int64_t nrows = (int64_t)g.ntile * g.nte * g.nte;
    const size_t nn = (size_t)std::max<int64_t>(n, 1);
    C2_TRY(g_lay.gid.reserve(nn * 4));
    C2_TRY(g_lay.gid_sorted.reserve(nn * 4));
    C2_TRY(g_lay.idx.reserve(nn * 4));
    C2_TRY(g_lay.idx_sorted.reserve(nn * 4));
    C2_TRY(g_lay.code.reserve(nn * 6));
    C2_TRY(g_lay.code_sorted.reserve(nn * 6));
    C2_TRY(g_lay.vel_sorted.reserve(nn * 12));
    C2_TRY(g_lay.cnt.reserve((nbin + 1) * sizeof(int)));
    C2_TRY(g_lay.slot.reserve((ncells + 1) * sizeof(long long)));
    C2_TRY(g_lay.scan_tmp.reserve(scan_tmp_ints(std::max(nbin, ncells)) * sizeof(int)));
    int end_bit = 1;
    while (((int64_t)1 << end_bit) < nbin) end_bit++;
    {
        Stage st("layout_encode", (double)n * (24 + 14));
        if (n) {
            k_layout_encode<<<ceil_div(n, 256), 256, 0, s>>>(d_pos, n, g.p.ng, g.p.ratio_cs, g.nc,
                                                            g_lay.gid.as<uint32_t>(),
                                                            g_lay.idx.as<uint32_t>(),
                                                            g_lay.code.as<int16_t>());
            C2_HIP(hipGetLastError());
        }
    }
    {
        Stage st("layout_sort", (double)n * 16);
        C2_TRY(radix_sort_pairs_u32(g_lay.gid.as<uint32_t>(), g_lay.gid_sorted.as<uint32_t>(),
                                    g_lay.idx.as<uint32_t>(), g_lay.idx_sorted.as<uint32_t>(), n,
                                    end_bit, g_lay.sort_tmp, g_lay.scan_tmp, s));
    }
    int* cnt = g_lay.cnt.as<int>();
    long long* slot = g_lay.slot.as<long long>();
    {
        Stage st("layout_cells", (double)n * 8 + (double)ncells * 16);
        k_layout_starts<<<ceil_div(nbin + 1, 256), 256, 0, s>>>(g_lay.gid_sorted.as<uint32_t>(), n,
                                                                nbin, cnt);  // total at [nbin]
        C2_HIP(hipGetLastError());
        k_layout_rhoc<<<ceil_div(ncells, 256), 256, 0, s>>>(cnt, ncells, g.nt, g.ncb, g.nte,
                                                            g.p.nnt, g.nc, d_rhoc);
        C2_HIP(hipGetLastError());
        C2_TRY(exclusive_scan_counts(d_rhoc, slot, ncells, g_lay.scan_tmp, s));
        k_layout_rows<<<ceil_div(nrows, 256), 256, 0, s>>>(slot, nrows, g.nte, d_idx_b_r);
        C2_HIP(hipGetLastError());
    }
    long long total = 0;
    C2_HIP(hipMemcpyAsync(&total, slot + ncells, sizeof(total), hipMemcpyDeviceToHost, s));
    C2_HIP(hipStreamSynchronize(s));
    *n_used = total;
    if (total >= (1ll << 31)) {
        set_error("layout: more than 2^31 particle slots");
        return CUBE2_ERR_CAPACITY;
    }
    if (total > cap || !d_xp || !d_vp) {
        set_error("layout: %lld slots needed, capacity %lld", total, (long long)cap);
        return CUBE2_ERR_CAPACITY;
    }
    {
        Stage st("layout_fill", (double)n * (4 + 2 * (6 + 12)) + (double)total * (6 + 12) * 2);
        if (n) {
            k_layout_gather<<<ceil_div(n, 256), 256, 0, s>>>(
                g_lay.idx_sorted.as<uint32_t>(), n, g_lay.code.as<int16_t>(), d_vel,
                g_lay.code_sorted.as<int16_t>(), g_lay.vel_sorted.as<float>());
            C2_HIP(hipGetLastError());
        }
        if (total) {
            k_layout_fill<<<ceil_div(total, kSlotChunk), kSlotThreads, 0, s>>>(
                make_slotgeom(g), cnt, slot, total, g_lay.code_sorted.as<int16_t>(),
                g_lay.vel_sorted.as<float>(), d_xp, d_vp);
            C2_HIP(hipGetLastError());
        }
    }
    return sync_and_flush();
}

// buffer_v for one image (buffer_particle.f90:11-21 through buffer_xvp,
// :23-345): the velocities of every halo cell's slots from the periodic
// source cell's slots, which hold the same particles in the same order.  A
// block per kSlotChunk slots; those of physical cells are left alone.  90 M
// slots at 256^3: 0.71 ms (a wavefront per cell: 4.25 ms).
// err: 1 a halo cell and its source differ, or slots outside [0, n_used).
__global__ __launch_bounds__(kSlotThreads) void k_halo_vp(SlotGeom G, const int* __restrict__ rhoc,
                                                          const long long* __restrict__ start,
                                                          const int64_t* __restrict__ idx_b_r,
                                                          float* __restrict__ vp, int64_t n_used,
                                                          int* __restrict__ err) {
    __shared__ int win[kSlotWin + 1];
    const int nte = (int)G.nte.d;
    int bad = 0;
    // (more than n_used slots where rows share theirs)
    walk_all_slots(start, G.ncells, start[G.ncells], win, [&](int64_t v0, int b, int e, auto cell_of) {
        for (int v = b + (int)threadIdx.x; v < e; v += kSlotThreads) {
            int s0, s1;
            const CellPos c = cell_pos(G, cell_of(v, s0, s1));
            const int cc[3] = {c.i, c.j, c.k};
            bool halo = false;
#pragma unroll
            for (int d = 0; d < 3; d++) halo |= cc[d] < G.ncb || cc[d] >= G.ncb + G.nt;
            if (!halo) continue;
            // source: the physical cell of the periodic image holding this cell
            int tc[3], st[3], sc[3];
            tile_pos(G, c.tile, tc[0], tc[1], tc[2]);
#pragma unroll
            for (int d = 0; d < 3; d++) {
                const int gcell = image_coord(G, tc[d], cc[d]);
                st[d] = gcell / G.nt;
                sc[d] = gcell - st[d] * G.nt + G.ncb;
            }
            const uint32_t ts = (uint32_t)((st[2] * (int)G.nnt.d + st[1]) * (int)G.nnt.d + st[0]);
            const uint32_t rs = (ts * nte + sc[2]) * nte + sc[1], qs = rs * nte + sc[0];
            const int64_t u0 = start[qs];
            const int64_t np = s1 < INT_MAX ? (int64_t)s1 - s0 : rhoc[c.row * nte + c.i];
            const int64_t h0 = row_shift(start, idx_b_r, c.row, nte) + v0;
            const int64_t h1 = row_shift(start, idx_b_r, rs, nte);
            const int64_t d0 = v + h0, d1 = u0 + (v - s0) + h1;
            if (start[qs + 1] - u0 != np || d0 < 0 || d1 < 0 || d0 >= n_used ||
                d1 >= n_used) {
                bad = 1;
                continue;
            }
            const float a0 = vp[3 * d1], a1 = vp[3 * d1 + 1], a2 = vp[3 * d1 + 2];
            vp[3 * d0] = a0;
            vp[3 * d0 + 1] = a1;
            vp[3 * d0 + 2] = a2;
        }
    });
    if (bad) atomicOr(err, 1);
}

int halo_velocities(const int* d_rhoc, const int64_t* d_idx_b_r, float* d_vp, int64_t n_used) {
    ensure_params();
    Context& C = ctx();
    const Geom& g = C.g;
    if (!d_rhoc || !d_idx_b_r || n_used < 0 || (n_used > 0 && !d_vp)) {
        set_error("halo velocities: null argument");
        return CUBE2_ERR_ARG;
    }
    C2_TRY(ensure_init());
    hipStream_t s = C.stream;
    C2_TRY(g_lay.red.reserve(sizeof(int)));
    int* err = g_lay.red.as<int>();
    C2_TRY(fill_zero(err, sizeof(int), s));
    const int64_t ncells = (int64_t)g.ntile * g.nte * g.nte * g.nte;
    if (ncells >= ((int64_t)1 << 31)) {
        set_error("halo velocities: more than 2^31 cells");
        return CUBE2_ERR_CAPACITY;
    }
    C2_TRY(g_lay.slot.reserve((ncells + 1) * sizeof(long long)));
    {
        Stage st("halo_vp", (double)n_used * 24);
        long long* start = g_lay.slot.as<long long>();
        C2_TRY(exclusive_scan_counts(d_rhoc, start, ncells, g_lay.scan_tmp, s));
        k_halo_vp<<<slot_blocks(n_used), kSlotThreads, 0, s>>>(
            make_slotgeom(g), d_rhoc, start, d_idx_b_r, d_vp, n_used, err);
        C2_HIP(hipGetLastError());
    }
    int h = 0;
    C2_HIP(hipMemcpyAsync(&h, err, sizeof(int), hipMemcpyDeviceToHost, s));
    C2_TRY(sync_and_flush());
    if (h) {
        set_error("halo velocities: a halo cell and its source cell differ (not one image's layout)");
        return CUBE2_ERR_ARG;
    }
    return CUBE2_OK;
}

void layout_release() {
    LayoutState& L = g_lay;
    for (DevBuf* b : {&L.gid, &L.gid_sorted, &L.idx, &L.idx_sorted, &L.code, &L.code_sorted,
                      &L.vel_sorted, &L.cnt, &L.slot,
                      &L.sort_tmp, &L.scan_tmp, &L.red})
        b->release();
}

}  // namespace cube2
