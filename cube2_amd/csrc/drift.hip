// Drift of one image on the device (drift.f90:1-158, spine_image of
// variables.f90:146-216): from the image with halo copies to the new
// physical-only image.
//   keys     every slot moves by dt_mid*vp (the reference's FP32/FP64 mix):
//            target cell ceiling(xq + deltax), new int16 code xp +
//            nint(dt_mid*vp / (x_resolution*ratio_cs)) (wrapping).  Of the
//            slots (halo copies included) only those whose target is a
//            physical cell of the same tile stay, a fifth of them at 256^3:
//            a first pass counts them per block of 1024 slots (slots.h), a
//            second one writes, in slot order, their key (tile, cell, layer
//            of the source z), slot and new code;
//   sort     stable radix sort (sort.hip) of (key, entry): within a target cell the
//            particles come by source layer, then in slot order (source z,
//            y, x, slot), the arrival order of the layered loop
//            drift.f90:36-62, 90-122 (one source z per layer can reach a
//            cell when |dz| <= (nlayer-2)/2, which the kernel checks);
//   counts   run boundaries of the sorted cells give the new rhoc (halo
//            cells 0), a row scan gives idx_b_r;
//   gather   codes and velocities of the kept slots in sorted order.
// At 256^3 (90 M slots, 16.7 M kept) the two key passes take 0.64 and 0.31 ms
// (18 bytes a slot: 2.4 TB/s) and the sort 0.9 ms; a wavefront per cell that
// wrote and sorted every slot took 5.9 and 3.3 ms.
#include <algorithm>
#include <cstring>

#include "common.h"
#include "engine.h"
#include "profile.h"
#include "scan.h"
#include "slots.h"
#include "sort.h"

namespace cube2 {

struct DriftState {
    DevBuf start, kept, key, key_sorted, val, val_sorted, slot, xpn, sort_tmp, bounds, rows,
        scan_tmp, red;
    HostBuf h_red;
};
static DriftState g_dr;

struct DriftArgs {
    SlotGeom G;
    const long long* start;  // running slot counts of the extended cells
    const int64_t* idx_b_r;
    const int16_t* xp;
    const float* vp;
    int64_t n_used;
    int ratio_cs, nlayer;
    float dt_mid;
};

// err bits: 1 slot range, 2 moved beyond ncb cells, 4 |dz| beyond the layer
// spacing.  kEmit false: kept[block] = the block's kept slots, and the
// checks.  kEmit true: kept[] holds the exclusive scan of those counts; the
// kept slots' keys, entry numbers, slots and codes are written in slot order
// (a wavefront takes 256 consecutive slots; blocks that keep none, most of
// the halo, end at once).  kPow2: ratio_cs is a power of two, so that its
// divisions are multiplications by the exact reciprocal (the same real
// number, the same rounding).
template <bool kEmit, bool kPow2>
__global__ __launch_bounds__(kSlotThreads) void k_drift_keys(
    DriftArgs A, int* __restrict__ kept, uint32_t* __restrict__ key, uint32_t* __restrict__ val,
    uint32_t* __restrict__ slot, int16_t* __restrict__ xpn, unsigned* __restrict__ err) {
#pragma clang fp contract(off)
    __shared__ int win[kSlotWin + 1];
    __shared__ int wsum[kSlotThreads / 64];
    const SlotGeom& G = A.G;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int64_t total = A.start[G.ncells];
    if (total > A.n_used) {
        if (!kEmit && threadIdx.x == 0) {
            kept[blockIdx.x] = 0;
            if (blockIdx.x == 0) atomicOr(err, 1u);
        }
        return;
    }
    int out = 0;
    if (kEmit) {
        out = kept[blockIdx.x];
        if (kept[blockIdx.x + 1] == out) return;
    }
    const int64_t v0 = (int64_t)blockIdx.x * kSlotChunk;
    const int dmax = (A.nlayer - 2) / 2;
    const float rf = (float)A.ratio_cs, irf = 1.0f / rf;
    const double rd = 1.0 / 65536.0 * (double)A.ratio_cs, ird = 1.0 / rd;
    unsigned bad = 0;
    int mine = 0;  // kept slots of the wavefront's windows
    constexpr int kIt = kSlotChunk / kSlotThreads;
    walk_slots(A.start, G.ncells, v0, block_slots(total, v0), win, [&](int b, int e, auto cell_of) {
        uint32_t kk[kIt], ss[kIt];
        int16_t code[kIt][3];
        uint64_t km[kIt];
        int n = 0;
#pragma unroll
        for (int it = 0; it < kIt; it++) {
            const int v = b + (wave * kIt + it) * 64 + lane;
            bool keep = false;
            if (v < e) {
                int s0, s1;
                const CellPos c = cell_pos(G, cell_of(v, s0, s1));
                const int64_t ip = v + v0 + row_shift(A.start, A.idx_b_r, c.row, G.nte.d);
                if (ip < 0 || ip >= A.n_used) {
                    bad |= 1u;
                } else {
                    const int src[3] = {c.i, c.j, c.k};
                    int ig[3];
                    float f[3];
                    int16_t x[3];
#pragma unroll
                    for (int d = 0; d < 3; d++) {
                        x[d] = A.xp[3 * ip + d];
                        f[d] = A.dt_mid * A.vp[3 * ip + d];  // FP32 product
                    }
                    keep = true;
#pragma unroll
                    for (int d = 0; d < 3; d++) {
                        const double xq = (double)(src[d] - G.ncb) + frac16(x[d]);  // (cell - 1) + frac
                        const double deltax = (double)(kPow2 ? f[d] * irf : f[d] / rf);  // FP32 quotient
                        ig[d] = (int)ceil(xq + deltax) - 1;  // 0-based physical target cell
                        const int moved = ig[d] - (src[d] - G.ncb);
                        if (moved > G.ncb || moved < -G.ncb) bad |= 2u;
                        if (d == 2 && (moved > dmax || moved < -dmax)) bad |= 4u;
                        keep &= ig[d] >= 0 && ig[d] < G.nt;
                    }
                    if (kEmit && keep) {
                        const uint32_t cell =
                            (uint32_t)(((int64_t)c.tile * G.nt + ig[2]) * G.nt + ig[1]) * G.nt + ig[0];
                        kk[it] = cell * (uint32_t)A.nlayer + (uint32_t)(c.k % A.nlayer);
                        ss[it] = (uint32_t)ip;
#pragma unroll
                        for (int d = 0; d < 3; d++) {
                            const double m = kPow2 ? (double)f[d] * ird : (double)f[d] / rd;
                            code[it][d] = (int16_t)(uint16_t)(uint32_t)((long long)x[d] + llround(m));
                        }
                    }
                }
            }
            km[it] = __ballot(keep);
            n += __popcll(km[it]);
        }
        if (!kEmit) {
            mine += n;
        } else {
            if (lane == 0) wsum[wave] = n;
            __syncthreads();
            int o = out;
            for (int w = 0; w < kSlotThreads / 64; w++) {
                if (w < wave) o += wsum[w];
                out += wsum[w];
            }
            const uint64_t lt = lane ? (~0ull >> (64 - lane)) : 0ull;
#pragma unroll
            for (int it = 0; it < kIt; it++) {
                if (km[it] >> lane & 1) {
                    const int64_t p = o + __popcll(km[it] & lt);
                    key[p] = kk[it];
                    val[p] = (uint32_t)p;
                    slot[p] = ss[it];
#pragma unroll
                    for (int d = 0; d < 3; d++) xpn[3 * p + d] = code[it][d];
                }
                o += __popcll(km[it]);
            }
        }
    });
    if (!kEmit) {
        if (lane == 0) wsum[wave] = mine;
        __syncthreads();
        if (threadIdx.x == 0) kept[blockIdx.x] = wsum[0] + wsum[1] + wsum[2] + wsum[3];
        if (bad) atomicOr(err, bad);
    }
}

// Positions (standard cells, FP64, wrapped into [0, ng)) of every slot of
// the image: a block per kSlotChunk slots (16.7 M slots without halo copies:
// 0.19 ms; a wavefront per cell 1.85 ms).
__global__ __launch_bounds__(kSlotThreads) void k_slot_positions(
    SlotGeom G, const long long* __restrict__ start, const int64_t* __restrict__ idx_b_r,
    const int16_t* __restrict__ xp, int64_t n_used, int ratio_cs, double* __restrict__ pos,
    unsigned* __restrict__ err) {
    __shared__ int win[kSlotWin + 1];
    unsigned bad = 0;
    // (more than n_used slots where rows share theirs)
    walk_all_slots(start, G.ncells, start[G.ncells], win, [&](int64_t v0, int b, int e, auto cell_of) {
        for (int v = b + (int)threadIdx.x; v < e; v += kSlotThreads) {
            int s0, s1;
            const CellPos c = cell_pos(G, cell_of(v, s0, s1));
            const int64_t ip = v + v0 + row_shift(start, idx_b_r, c.row, G.nte.d);
            if (ip < 0 || ip >= n_used) {
                bad = 1u;
                continue;
            }
            int tx, ty, tz;
            tile_pos(G, c.tile, tx, ty, tz);
            const int gc[3] = {image_coord(G, tx, c.i), image_coord(G, ty, c.j),
                               image_coord(G, tz, c.k)};
#pragma unroll
            for (int d = 0; d < 3; d++)
                pos[3 * ip + d] = ((double)gc[d] + frac16(xp[3 * ip + d])) * (double)ratio_cs;
        }
    });
    if (bad) atomicOr(err, bad);
}

// bounds[2c] / bounds[2c+1]: first / past-last sorted position of cell c.
__global__ void k_drift_bounds(const uint32_t* __restrict__ ks, int64_t n_kept, int nlayer,
                               int* __restrict__ bounds) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n_kept) return;
    const uint32_t c = ks[p] / (uint32_t)nlayer;
    if (p == 0 || ks[p - 1] / (uint32_t)nlayer != c) bounds[2 * (int64_t)c] = (int)p;
    if (p == n_kept - 1 || ks[p + 1] / (uint32_t)nlayer != c) bounds[2 * (int64_t)c + 1] = (int)(p + 1);
}

// New rhoc over every extended cell (halo cells 0) and its row sums.
__global__ void k_drift_rhoc(const int* __restrict__ bounds, int nt, int ncb, int nte, int ntile,
                             int* __restrict__ rhoc_out, int* __restrict__ rows) {
    const int64_t row = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;  // (t, k, j)
    const int64_t nrows = (int64_t)ntile * nte * nte;
    if (row >= nrows) return;
    const int t = (int)(row / ((int64_t)nte * nte));
    const int rr = (int)(row - (int64_t)t * nte * nte);
    const int k = rr / nte - ncb, j = rr % nte - ncb;  // physical indices
    int* out = rhoc_out + row * nte;
    int sum = 0;
    const bool phys_row = k >= 0 && k < nt && j >= 0 && j < nt;
    for (int i = 0; i < nte; i++) {
        int c = 0;
        const int pi = i - ncb;
        if (phys_row && pi >= 0 && pi < nt) {
            const int64_t cell = (((int64_t)t * nt + k) * nt + j) * nt + pi;
            c = bounds[2 * cell + 1] - bounds[2 * cell];
        }
        out[i] = c;
        sum += c;
    }
    rows[row] = sum;
}

__global__ void k_drift_rows(const int* __restrict__ rows, int64_t nrows, int64_t* __restrict__ idx_out) {
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r < nrows) idx_out[r] = (int64_t)rows[r + 1];  // running total through row r
}

__global__ void k_drift_gather(const uint32_t* __restrict__ vs, int64_t n_kept,
                               const uint32_t* __restrict__ slot,
                               const int16_t* __restrict__ xpn, const float* __restrict__ vp,
                               int16_t* __restrict__ xp_out, float* __restrict__ vp_out) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n_kept) return;
    const int64_t e = vs[p], s = slot[e];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        xp_out[3 * p + d] = xpn[3 * e + d];
        vp_out[3 * p + d] = vp[3 * s + d];
    }
}

int drift(const int* d_rhoc, const int64_t* d_idx_b_r, const int16_t* d_xp, const float* d_vp,
          int64_t n_used, float dt_mid, float vz_max, int* d_rhoc_out, int64_t* d_idx_out,
          int16_t* d_xp_out, float* d_vp_out, int64_t cap, int64_t* n_out) {
    ensure_params();
    Context& C = ctx();
    const Geom& g = C.g;
    if (!d_rhoc || !d_idx_b_r || !d_rhoc_out || !d_idx_out || !n_out || n_used < 0 ||
        n_used >= ((int64_t)1 << 31) || (n_used > 0 && (!d_xp || !d_vp)) || !(dt_mid >= 0.0f) ||
        !(vz_max >= 0.0f)) {
        set_error("drift: null argument or value out of range");
        return CUBE2_ERR_ARG;
    }
    // nlayer = 2*ceiling(dt_mid*vz_max/ratio_cs)+2 (drift.f90:26), FP32
    volatile float qv = dt_mid * vz_max;
    const float qf = qv / (float)g.p.ratio_cs;
    if (!(qf <= (float)g.ncb + 1.0f)) {
        set_error("drift: dt_mid*vz_max/ratio_cs = %g exceeds the halo depth %d", (double)qf, g.ncb);
        return CUBE2_ERR_ARG;
    }
    const int nlayer = 2 * (int)std::ceil(qf) + 2;
    const int64_t ncell_phys = (int64_t)g.ntile * g.nt * g.nt * g.nt;
    if (ncell_phys * nlayer + 1 >= ((int64_t)1 << 32) || ncell_phys >= ((int64_t)1 << 30)) {
        set_error("drift: image too large for 32-bit keys");
        return CUBE2_ERR_CAPACITY;
    }
    C2_TRY(ensure_init());
    hipStream_t s = C.stream;
    const int64_t ncells = (int64_t)g.nte * g.nte * g.nte * g.ntile;
    if (ncells >= ((int64_t)1 << 31)) {
        set_error("drift: image too large for 32-bit cells");
        return CUBE2_ERR_CAPACITY;
    }
    const int64_t nrows = (int64_t)g.ntile * g.nte * g.nte;
    const int64_t nblk = std::max<int64_t>(1, (n_used + kSlotChunk - 1) / kSlotChunk);
    C2_TRY(g_dr.start.reserve((size_t)(ncells + 1) * sizeof(long long)));
    C2_TRY(g_dr.kept.reserve((size_t)(nblk + 1) * sizeof(int)));
    C2_TRY(g_dr.bounds.reserve((size_t)(2 * ncell_phys) * sizeof(int)));
    C2_TRY(g_dr.rows.reserve((size_t)(nrows + 1) * sizeof(int)));
    C2_TRY(g_dr.red.reserve(sizeof(unsigned)));
    C2_TRY(g_dr.h_red.reserve(2 * sizeof(int)));
    const uint32_t key_none = (uint32_t)(ncell_phys * nlayer);  // past every key
    unsigned end_bit = 1;
    while (end_bit < 32 && ((uint64_t)1 << end_bit) < key_none) end_bit++;
    unsigned* err = g_dr.red.as<unsigned>();
    C2_TRY(fill_zero(err, sizeof(unsigned), s));
    DriftArgs A;
    A.G = make_slotgeom(g);
    A.start = g_dr.start.as<long long>();
    A.idx_b_r = d_idx_b_r;
    A.xp = d_xp;
    A.vp = d_vp;
    A.n_used = n_used;
    A.ratio_cs = g.p.ratio_cs;
    A.nlayer = nlayer;
    A.dt_mid = dt_mid;
    const bool pow2 = (g.p.ratio_cs & (g.p.ratio_cs - 1)) == 0;
    int* kept = g_dr.kept.as<int>();
    int* h = g_dr.h_red.as<int>();
    {
        Stage st("drift_keys", (double)n_used * (6 + 12));
        C2_TRY(exclusive_scan_counts(d_rhoc, g_dr.start.as<long long>(), ncells, g_dr.scan_tmp, s));
        auto kern = pow2 ? k_drift_keys<false, true> : k_drift_keys<false, false>;
        kern<<<(unsigned)nblk, kSlotThreads, 0, s>>>(A, kept, nullptr, nullptr, nullptr, nullptr, err);
        C2_HIP(hipGetLastError());
        C2_TRY(exclusive_scan(kept, nblk, g_dr.scan_tmp, s));
        C2_HIP(hipMemcpyAsync(h, kept + nblk, sizeof(int), hipMemcpyDeviceToHost, s));
        C2_HIP(hipMemcpyAsync(h + 1, err, sizeof(int), hipMemcpyDeviceToHost, s));
    }
    C2_HIP(hipStreamSynchronize(s));
    if (h[1]) {
        set_error(h[1] & 1 ? "drift: rhoc and idx_b_r describe slots outside [0, n_used)"
                  : h[1] & 2 ? "drift: a particle moved more than ncb coarse cells"
                             : "drift: a particle moved further in z than vz_max allows");
        return CUBE2_ERR_ARG;
    }
    const int64_t n_kept = (int64_t)h[0];
    *n_out = n_kept;
    if (n_kept > cap || (n_kept > 0 && (!d_xp_out || !d_vp_out))) {
        set_error("drift: %lld particles kept, capacity %lld", (long long)n_kept, (long long)cap);
        return CUBE2_ERR_CAPACITY;
    }
    const size_t nn = (size_t)std::max<int64_t>(n_kept, 1);
    C2_TRY(g_dr.key.reserve(nn * 4));
    C2_TRY(g_dr.key_sorted.reserve(nn * 4));
    C2_TRY(g_dr.val.reserve(nn * 4));
    C2_TRY(g_dr.val_sorted.reserve(nn * 4));
    C2_TRY(g_dr.slot.reserve(nn * 4));
    C2_TRY(g_dr.xpn.reserve(nn * 6));
    if (n_kept) {
        Stage st("drift_emit", (double)n_kept * (2 * (6 + 4) + 12 + 4));
        auto kern = pow2 ? k_drift_keys<true, true> : k_drift_keys<true, false>;
        kern<<<(unsigned)nblk, kSlotThreads, 0, s>>>(A, kept, g_dr.key.as<uint32_t>(),
                                                     g_dr.val.as<uint32_t>(),
                                                     g_dr.slot.as<uint32_t>(),
                                                     g_dr.xpn.as<int16_t>(), err);
        C2_HIP(hipGetLastError());
    }
    {
        Stage st("drift_sort", (double)n_kept * 16);
        C2_TRY(radix_sort_pairs_u32(g_dr.key.as<uint32_t>(), g_dr.key_sorted.as<uint32_t>(),
                                    g_dr.val.as<uint32_t>(), g_dr.val_sorted.as<uint32_t>(),
                                    n_kept, (int)end_bit, g_dr.sort_tmp, g_dr.scan_tmp, s));
    }
    {
        Stage st("drift_cells", (double)n_kept * 4 + (double)ncells * 8);
        int* bounds = g_dr.bounds.as<int>();
        C2_TRY(fill_zero(bounds, (size_t)(2 * ncell_phys) * sizeof(int), s));
        if (n_kept) {
            k_drift_bounds<<<ceil_div(n_kept, 256), 256, 0, s>>>(g_dr.key_sorted.as<uint32_t>(),
                                                                 n_kept, nlayer, bounds);
            C2_HIP(hipGetLastError());
        }
        int* rows = g_dr.rows.as<int>();
        k_drift_rhoc<<<ceil_div(nrows, 256), 256, 0, s>>>(bounds, g.nt, g.ncb, g.nte, g.ntile,
                                                          d_rhoc_out, rows);
        C2_HIP(hipGetLastError());
        C2_TRY(exclusive_scan(rows, nrows, g_dr.scan_tmp, s));
        k_drift_rows<<<ceil_div(nrows, 256), 256, 0, s>>>(rows, nrows, d_idx_out);
        C2_HIP(hipGetLastError());
    }
    if (n_kept) {
        Stage st("drift_gather", (double)n_kept * (4 + 2 * (6 + 12)));
        k_drift_gather<<<ceil_div(n_kept, 256), 256, 0, s>>>(g_dr.val_sorted.as<uint32_t>(),
                                                             n_kept, g_dr.slot.as<uint32_t>(),
                                                             g_dr.xpn.as<int16_t>(), d_vp,
                                                             d_xp_out, d_vp_out);
        C2_HIP(hipGetLastError());
    }
    return sync_and_flush();
}

int slot_positions(const int* d_rhoc, const int64_t* d_idx_b_r, const int16_t* d_xp,
                   int64_t n_used, double* d_pos) {
    ensure_params();
    Context& C = ctx();
    const Geom& g = C.g;
    if (!d_rhoc || !d_idx_b_r || n_used < 0 || (n_used > 0 && (!d_xp || !d_pos))) {
        set_error("positions: null argument");
        return CUBE2_ERR_ARG;
    }
    C2_TRY(ensure_init());
    hipStream_t s = C.stream;
    const int64_t ncells = (int64_t)g.nte * g.nte * g.nte * g.ntile;
    if (ncells >= ((int64_t)1 << 31)) {
        set_error("positions: image too large for 32-bit cells");
        return CUBE2_ERR_CAPACITY;
    }
    C2_TRY(g_dr.red.reserve(sizeof(unsigned)));
    C2_TRY(g_dr.h_red.reserve(2 * sizeof(int)));
    C2_TRY(g_dr.start.reserve((size_t)(ncells + 1) * sizeof(long long)));
    unsigned* err = g_dr.red.as<unsigned>();
    C2_TRY(fill_zero(err, sizeof(unsigned), s));
    long long* start = g_dr.start.as<long long>();
    C2_TRY(exclusive_scan_counts(d_rhoc, start, ncells, g_dr.scan_tmp, s));
    k_slot_positions<<<slot_blocks(n_used), kSlotThreads, 0, s>>>(
        make_slotgeom(g), start, d_idx_b_r, d_xp, n_used, g.p.ratio_cs, d_pos, err);
    C2_HIP(hipGetLastError());
    int* h = g_dr.h_red.as<int>();
    C2_HIP(hipMemcpyAsync(h, err, sizeof(int), hipMemcpyDeviceToHost, s));
    C2_TRY(sync_and_flush());
    if (h[0]) {
        set_error("positions: rhoc and idx_b_r describe slots outside [0, n_used)");
        return CUBE2_ERR_ARG;
    }
    return CUBE2_OK;
}

void drift_release() {
    DriftState& D = g_dr;
    for (DevBuf* b : {&D.start, &D.kept, &D.slot, &D.key, &D.key_sorted, &D.val, &D.val_sorted, &D.xpn, &D.sort_tmp,
                      &D.bounds, &D.rows, &D.scan_tmp, &D.red})
        b->release();
    D.h_red.release();
}

}  // namespace cube2
