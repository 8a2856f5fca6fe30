// Pairs-once pass: the particles of PP cells of at most `small` particles.
//
// The PP grid of a tile follows its densest subtile, so that in the sparse
// subtiles beside a clump a PP cell holds one particle or none while its
// stencil has up to 13^2 rows.  Taken as chunks of the pair kernel, a chunk
// per cell, these particles (64% of C1's, 2.5% of its accepted pairs) cost
// 11.1 M chunks of 25 to 169 rows each: half of that kernel's instructions
// and most of its memory traffic (cell starts, and registers spilled around
// each chunk).
//
// Here a wavefront takes part of a coarse cell: it lists the particles of its
// small cells, up to 64 at a time, and walks the cells within R of any of them once
// for all, each row of cells being read once instead of once per particle.  Every j of that
// region is tested against every i (lane (i, s) takes j slot t + s); whether
// j's cell lies in i's stencil, for the count of candidates, is one packed
// comparison of cell coordinates.  Accepted pairs are queued in LDS and their
// forces evaluated 64 at a time, summed per i as 64-bit fixed point (integer
// LDS atomics; float ones cost ~190 cycles an instruction on gfx950) at a scale
// for the 512 pairs of 8 such steps, and in FP64 over the steps: the pass's
// scale, for as many pairs as there are slots, rounds each pair to 2^-12 where
// the softening is small.  These particles evaluate all their pairs themselves
// and nothing else adds to them (k_chunk_flags marks them), so their sums are
// stored, not added, unless their j are split; what the pass's scale cannot hold
// of them goes to `low`.
// Bound by the chains of row and batch loads of each region: 0.16 VALU and 0.14
// scalar instructions per SIMD cycle, half of the wavefronts' time waiting, 1.3
// TB/s (7.3-8.0 ms alone at 256^3).  The particles beside a clump cost
// the most by far, one batch of them up to 1 ms, and the kernel waits for the
// last: k_sparse_items shares a coarse cell among wavefronts and lists the
// costly ones first.  REF, clustered, ms at 256^3 / 128^3 / 120^3 in level-6
// cells: a wavefront per coarse cell 12.1 / 3.8 / 2.3, eight 7.9 / 2.0 / 1.1,
// with j split too 8.1 / 1.1 / 0.94 (128^3 drop-in call 14.7 -> 13.7).
#include <algorithm>

#include "common.h"
#include "engine.h"
#include "pp_kernels.h"
#include "pp_law.h"
#include "profile.h"
#include "reduce.h"

namespace cube2 {

constexpr unsigned kOnes = 1u | 1u << 10 | 1u << 20;  // one in each packed coordinate
constexpr unsigned kTop = 512u * kOnes;

struct SparseLDS {
    float4 q[kQ];             // accepted pairs (dx, dy, dz, r^2)
    unsigned char qi[kQ];     // and their i slot
    unsigned long long acc[64][3];
    float4 jb[64];            // a batch of j (w: packed cell), far-away ones past it
    int list[128];            // sorted indices of small cells' particles
    unsigned lcell[128];      // their cells (packed, in the coarse cell) and
    unsigned short lblk[128]; // blocks
    int rs[64], rp[64];       // row group: j = v + rs[k] for rp[k-1] <= v < rp[k]
    unsigned rc[64];          // packed cell of a j of row k, less its cell id
};

template <int kMode>
__device__ inline void sparse_flush(SparseLDS& L, int lane, int begin, int count, const FraK& Ka,
                                    const FraK& Kr, float scale) {
    if (lane < count) {
        const int s = (begin + lane) & (kQ - 1);
        const float4 e = L.q[s];
        const int ii = L.qi[s];
        float f[3];
        pair_force<kMode>(e, Ka, Kr, f[0], f[1], f[2]);
#pragma unroll
        for (int c = 0; c < 3; c++) atomicAdd(&L.acc[ii][c], to_fixed(f[c], scale));
    }
    wave_lds_sync();
}

// The sums of the last steps, of the lane's i slot, into FP64.
__device__ inline void sparse_drain(SparseLDS& L, int lane, double (&sum)[3], double inv_scale) {
    wave_lds_sync();
#pragma unroll
    for (int c = 0; c < 3; c++) {
        sum[c] += (double)(long long)L.acc[lane][c] * inv_scale;
        L.acc[lane][c] = 0ull;
    }
    wave_lds_sync();
}

// n / d as the high word of n * recip(d), exact for n d < 2^32.
__device__ inline unsigned recip_u32(unsigned d) { return 0xffffffffu / d + 1u; }
__device__ inline int quot(int n, unsigned recip) { return (int)__umulhi((unsigned)n, recip); }

// Pairs between two drains (a multiple of 64).
constexpr int kDrainPairs = 512;

// Mean particles of a block (below): small blocks walk less that only one of
// their particles needs, large ones read rows less often (at 256^3 with one
// wavefront per coarse cell 4: 17.1 ms, 8: 13.0, 16: 12.1, 32: 13.2).
constexpr float kBlockCount = 16.0f;
// Items of a coarse cell: its blocks in kParts, each once per kItemCount
// particles of the 27 coarse cells (at most kMaxSplit), the j of the regions
// split among the latter (ms as above: 4096: 8.6 / 1.15 / 0.84, 16384: 8.1 /
// 1.1 / 0.94, 65536: 7.7 / 1.45 / 1.1).
constexpr int kParts = 8, kItemCount = 16384, kMaxSplit = 16;

// The items of every coarse cell that holds particles: x = the cell, y = part,
// split, splits and blocks per side.  Those of split cells go to the front of
// the list (count[0]) and are taken first, the others to its end
// (count[kRunPad]).
__global__ __launch_bounds__(256) void k_sparse_items(const int* __restrict__ rhoc, int nt, int ncb,
                                                      int ncoarse, const PPTile* __restrict__ tiles,
                                                      const int* __restrict__ err, int cap,
                                                      int2* __restrict__ items, int* __restrict__ count) {
    const int w = blockIdx.x * blockDim.x + threadIdx.x, lane = threadIdx.x & 63;
    __shared__ int wsum[2][4], first[2];
    int nitem = 0, parts = 0, splits = 1, nb1 = 1;
    if (w < ncoarse && *err == 0) {
        const int t = w / (nt * nt * nt), wr = w - t * nt * nt * nt, nte = nt + 2 * ncb;
        const int x = wr % nt + ncb, y = wr / nt % nt + ncb, z = wr / (nt * nt) + ncb;
        const int* c0 = rhoc + (((size_t)t * nte + z) * nte + y) * nte + x;
        if (*c0 > 0) {
            long long n27 = 0;
            for (int dz = -1; dz <= 1; dz++)
                for (int dy = -1; dy <= 1; dy++)
                    for (int dx = -1; dx <= 1; dx++)
                        n27 += max(c0[((long long)dz * nte + dy) * nte + dx], 0);
            const int rcp = tiles[t].rcp;
            const float mean = (float)n27 * (1.0f / 27.0f);
            nb1 = min(rcp, max(1, (int)ceilf(cbrtf(mean * (1.0f / kBlockCount)))));
            const int Bs = (rcp + nb1 - 1) / nb1, nbl = (rcp + Bs - 1) / Bs;
            parts = min(kParts, nbl * nbl * nbl);
            splits = (int)min(1 + n27 / kItemCount, (long long)kMaxSplit);
            nitem = parts * splits;
        }
    }
#pragma unroll
    for (int heavy = 0; heavy < 2; heavy++) {
        const int mine = (splits > 1) == (heavy == 1) ? nitem : 0;
        int inc = mine;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int u = __shfl_up(inc, o, 64);
            if (lane >= o) inc += u;
        }
        if (lane == 63) wsum[heavy][threadIdx.x >> 6] = inc;
        __syncthreads();
        if (threadIdx.x == 0) {  // one atomic per block
            int tot = 0;
            for (int v = 0; v < 4; v++) {
                const int n = wsum[heavy][v];
                wsum[heavy][v] = tot;
                tot += n;
            }
            first[heavy] = tot ? atomicAdd(&count[heavy ? 0 : kRunPad], tot) : 0;
        }
        __syncthreads();
        int at = first[heavy] + wsum[heavy][threadIdx.x >> 6] + inc - mine;
        for (int k = 0; k < mine; k++, at++)
            if (at < cap)
                items[heavy ? at : cap - 1 - at] =
                    make_int2(w, k % parts | parts << 4 | k / parts << 8 | splits << 16 | nb1 << 24);
    }
}

template <int kMode>
__global__ __launch_bounds__(256, 5) void k_pp_sparse(PPArgs A, const int2* __restrict__ items, int cap,
                                                      const int* __restrict__ count, int nt, int small,
                                                      float scale, double inv_scale) {
    __shared__ SparseLDS lds[4];
    const int wave = uni((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    SparseLDS& L = lds[wave];
    const uint64_t lt = lane ? (~0ull >> (64 - lane)) : 0ull;
    const FraK Ka = uni(make_frak(A.app));
    unsigned long long pc = 0, pa = 0;  // (wavefront-uniform)
    // the split cells' items by all blocks alike; neighbouring coarse cells
    // share most of their j: one XCD takes a run of the others
    const int nheavy = min(count[0], cap), nlight = min(count[kRunPad], cap - nheavy);
    bool heavy = true;
    int w = (int)blockIdx.x * 4 + wave;
    for (;; w += gridDim.x * 4) {
        if (heavy && w >= nheavy) {
            heavy = false;
            w = (int)xcd_remap(blockIdx.x, gridDim.x) * 4 + wave;
        }
        if (!heavy && w >= nlight) break;
        const int2 item = items[heavy ? w : cap - 1 - w];
        const int cw = uni(item.x), code = uni(item.y);
        const int part = code & 15, parts = code >> 4 & 15, sp = code >> 8 & 255, splits = code >> 16 & 255;
        const int t = cw / (nt * nt * nt), wr = cw - t * nt * nt * nt;
        const PPTile T = A.tiles[t];
        const int S = T.S, rcp = T.rcp;
        const int bx = (wr % nt + 1) * rcp, by = (wr / nt % nt + 1) * rcp, bz = (wr / (nt * nt) + 1) * rcp;
        const unsigned off = (unsigned)T.cell_off;
        const int nb1 = code >> 24;  // (from the mean count of the 27 coarse cells around)
        const int Bs = uni((rcp + nb1 - 1) / nb1), nbl = (rcp + Bs - 1) / Bs;  // blocks of Bs^3 cells
        const int nblk = nbl * nbl * nbl, cblk = Bs * Bs * Bs;  // blocks, cells of one
        const int ncell = nblk * (part + 1) / parts * cblk;
        const unsigned i1 = recip_u32(Bs), i2 = recip_u32(Bs * Bs), i3 = recip_u32(Bs * Bs * Bs);
        const unsigned k1 = recip_u32(nbl), k2 = recip_u32(nbl * nbl);
        const unsigned long long pc0 = pc, pa0 = pa;
        int c0 = nblk * part / parts * cblk, depth = 0, n = 0, first = 0, blk = 0, head = 0, tail = 0;
        unsigned cpk = 0;
        float range = 0.0f;
        FraK Kr = Ka;
        int R = 0;
        float pp2 = 0.0f;
        for (;;) {
            // list the small cells' particles, the depth-th of 64 cells at a time
            while (tail - head < 64 && c0 < ncell) {
                if (depth == 0) {
                    n = 0;
                    const int c = c0 + lane;
                    if (c < ncell) {
                        // (block, cell in it) -> cell of the coarse cell
                        blk = Bs > 1 ? quot(c, i3) : c;
                        const int r = c - blk * Bs * Bs * Bs;
                        const int kz = nbl > 1 ? quot(blk, k2) : blk, kzy = nbl > 1 ? quot(blk, k1) : blk;
                        const int rz = Bs > 1 ? quot(r, i2) : r, rzy = Bs > 1 ? quot(r, i1) : r;
                        const int z = kz * Bs + rz, y = (kzy - kz * nbl) * Bs + rzy - rz * Bs,
                                  x = (blk - kzy * nbl) * Bs + r - rzy * Bs;
                        if (z < rcp && y < rcp && x < rcp) {
                            const unsigned cell = off + ((unsigned)(bz + z) * S + by + y) * S + bx + x;
                            first = A.cell_start[cell];
                            n = A.cell_start[cell + 1] - first;
                            if (n > small) n = 0;
                            cpk = (unsigned)z << 20 | (unsigned)y << 10 | (unsigned)x;
                        }
                    }
                }
                const uint64_t m = __ballot(n > depth);
                if (n > depth) {
                    const int at = (tail + __popcll(m & lt)) & 127;
                    L.list[at] = first + depth;
                    L.lcell[at] = cpk;
                    L.lblk[at] = (unsigned short)blk;
                }
                tail += __popcll(m);
                depth++;
                if (!__ballot(n > depth)) {
                    depth = 0;
                    c0 += 64;
                }
            }
            wave_lds_sync();
            if (tail == head) break;
            // the batch: the listed particles of the first one's block
            const int b0 = uni((int)L.lblk[head & 127]);
            const uint64_t same = __ballot(head + lane < tail && L.lblk[(head + lane) & 127] == b0);
            const int ni = ~same ? __ffsll((unsigned long long)~same) - 1 : 64;
            int lgI = 0;
            while ((1 << lgI) < ni) lgI++;
            const int I = 1 << lgI, J = 64 >> lgI;
            const int islot = lane & (I - 1), jslot = lane >> lgI;
            const bool vi = islot < ni;
            const int at = (head + (vi ? islot : 0)) & 127, ia = L.list[at];
            const unsigned cell = L.lcell[at];
            head += ni;
            const float4 p = A.pos4[ia];
            if (range == 0.0f) {  // one subtile per coarse cell: one range
                range = fabsf(uni(p.w));
                if (range == 0.0f || (A.learned_occ && range == A.learned_range)) break;
                R = (int)ceilf(__fmul_rn(range, (float)rcp) / (float)A.ratio_cs);
                pp2 = __fmul_rn(range, range);
                Kr = uni(make_frak(range));
            }
            // cells relative to the origin (bx, by, bz) - R; j's cell is in i's
            // stencil iff each coordinate of (j - i + R) and of (i - j + R) is
            // not negative: with 512 added to each, iff its top bit stays
            // (|j - i| + R < 512)
            const int X0 = bx - R, Y0 = by - R, Z0 = bz - R;
            const unsigned lo = cell - kTop, hi = cell + 2u * (unsigned)R * kOnes + kTop;
            // the region: the block's cells and R around them
            const int kz = b0 / (nbl * nbl), ky = b0 / nbl % nbl, kx = b0 % nbl;
            const int xa = max(X0 + kx * Bs, 0), xb = min(bx + min(kx * Bs + Bs, rcp) - 1 + R, S - 1);
            const int ya = max(Y0 + ky * Bs, 0), yb = min(by + min(ky * Bs + Bs, rcp) - 1 + R, S - 1);
            const int za = max(Z0 + kz * Bs, 0), zb = min(bz + min(kz * Bs + Bs, rcp) - 1 + R, S - 1);
            const int ny = yb - ya + 1, nrows = ny * (zb - za + 1);
            const unsigned inv_ny = recip_u32(ny);
            const uint64_t vim = __ballot(vi);
            const float pix = vi ? p.x : -kFar, piy = vi ? p.y : -kFar, piz = vi ? p.z : -kFar;
            for (int q = lane; q < 64 * 3; q += 64) (&L.acc[0][0])[q] = 0ull;
            int qhead = 0, qtail = 0;
            double sum[3] = {0.0, 0.0, 0.0};  // of i slot `lane`
            for (int rg = 0; rg < nrows; rg += 64) {
                int js = 0, cnt = 0;
                const int r = rg + lane;
                if (r < nrows) {
                    const int rz = ny > 1 ? quot(r, inv_ny) : r;
                    const int zz = za + rz, yy = ya + r - rz * ny;
                    const unsigned row = off + ((unsigned)zz * S + yy) * S;
                    js = A.cell_start[row + xa];
                    cnt = A.cell_start[row + xb + 1] - js;
                    L.rc[lane] = ((unsigned)(zz - Z0) << 20 | (unsigned)(yy - Y0) << 10) - row - (unsigned)X0;
                }
                int inc = cnt;
#pragma unroll
                for (int o = 1; o < 64; o <<= 1) {
                    const int u = __shfl_up(inc, o, 64);
                    if (lane >= o) inc += u;
                }
                const int M0 = uni(__shfl(inc, 63, 64));
                // this split's candidates [v0, M) of the group's
                const int v0 = (int)((long long)M0 * sp / splits), M = (int)((long long)M0 * (sp + 1) / splits);
                L.rs[lane] = js - (inc - cnt);
                L.rp[lane] = inc;
                wave_lds_sync();
                int frow = 0;  // (a lane's candidates only grow: its row walks forward)
                unsigned rc = 0, jc = 0;
                auto fetch = [&](int vb) {
                    const int v = vb + lane;
                    float4 q4 = make_float4(0.f, 0.f, 0.f, 0.f);
                    if (v < M) {
                        while (L.rp[frow] <= v) frow++;
                        const int jx = v + L.rs[frow];
                        q4 = A.pos4[jx];
                        jc = A.cellid[jx];
                        rc = L.rc[frow];
                    }
                    return q4;
                };
                float4 qc = fetch(v0);
                for (int vb = v0; vb < M; vb += 64) {
                    const int nb = min(64, M - vb);
                    qc.w = __uint_as_float(rc + jc);
                    // past the batch: far away and in no stencil
                    if (lane >= nb) qc = make_float4(kFar, kFar, kFar, __uint_as_float(511u * kOnes));
                    L.jb[lane] = qc;
                    wave_lds_sync();
                    if (vb + 64 < M) qc = fetch(vb + 64);
                    // lane's pair with the j at slot u: its vector, r^2, whether
                    // it pairs; candidates counted
                    auto test = [&](const float4& qj, float4& e) {
#pragma clang fp contract(off)
                        e.x = qj.x - pix;
                        e.y = qj.y - piy;
                        e.z = qj.z - piz;
                        e.w = e.x * e.x + e.y * e.y + e.z * e.z;
                        const unsigned jk = __float_as_uint(qj.w);
                        pc += __popcll(__ballot(((jk - lo) & (hi - jk) & kTop) == kTop) & vim);
                        return (e.w > 0.0f) & (e.w < pp2);
                    };
                    auto append = [&](bool ok, const float4& e) {
                        const uint64_t m = __ballot(ok);
                        if (!m) return;
                        if (ok) {
                            const int s = (qtail + __popcll(m & lt)) & (kQ - 1);
                            L.q[s] = e;
                            L.qi[s] = (unsigned char)islot;
                        }
                        qtail += __popcll(m);
                        if (qtail - qhead >= 64) {
                            wave_lds_sync();
                            sparse_flush<kMode>(L, lane, qhead, 64, Ka, Kr, scale);
                            qhead += 64;
                            if (qhead % kDrainPairs == 0) sparse_drain(L, lane, sum, inv_scale);
                        }
                    };
                    if (J <= 16) {  // (4 J divides 64: no slot past them)
                        for (int u = 0; u < nb; u += 4 * J) {
                            float4 qj[4], e[4];
                            bool ok[4];
#pragma unroll
                            for (int k = 0; k < 4; k++) qj[k] = L.jb[u + k * J + jslot];
#pragma unroll
                            for (int k = 0; k < 4; k++) ok[k] = test(qj[k], e[k]);
#pragma unroll
                            for (int k = 0; k < 4; k++) append(ok[k], e[k]);
                        }
                    } else {
                        for (int u = 0; u < nb; u += J) {
                            float4 e;
                            const bool ok = test(L.jb[u + jslot], e);
                            append(ok, e);
                        }
                    }
                    wave_lds_sync();  // jb is rewritten by the next batch
                }
            }
            wave_lds_sync();
            if (qtail > qhead) sparse_flush<kMode>(L, lane, qhead, qtail - qhead, Ka, Kr, scale);
            sparse_drain(L, lane, sum, inv_scale);
            pa += (unsigned)qtail;
            if (sp == 0) pc -= (unsigned)ni;  // the particles themselves
            if (vi && jslot == 0) {  // (lane = islot)
                int4 lo;
                int* const l = &lo.x;
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    unsigned long long* d = A.react + c * (size_t)A.cap + ia;
                    const double v = sum[c] * (double)A.react_scale, hi = rint(v);
                    l[c] = (int)rint((v - hi) * kLowScale);
                    if (splits > 1) {
                        atomicAdd(d, (unsigned long long)(long long)hi);
                        atomicAdd(&A.low[ia].x + c, l[c]);
                    } else {
                        *d = (unsigned long long)(long long)hi;
                    }
                }
                lo.w = 0;
                if (splits == 1) A.low[ia] = lo;
            }
            wave_lds_sync();  // acc, the queue and the list are reused
        }
        if (A.tile_pairs && lane == 0) {  // per-tile counts (on request only)
            atomicAdd(&A.tile_pairs[2 * t], pc - pc0);
            atomicAdd(&A.tile_pairs[2 * t + 1], pa - pa0);
        }
    }
    const unsigned long long sm[2] = {lane == 0 ? pc : 0ull, lane == 0 ? pa : 0ull};
    block_sum_to<2>(&A.red->p_cand, sm);
}

// Largest stencil radius and PP cells per coarse cell whose packed cell
// coordinates fit (rcp + 3 R < 512); beyond it the pass is not pairs-once.
bool pp_sparse_fits(int rcp, float range, int ratio_cs) {
    const double R = std::ceil((double)range * rcp / ratio_cs) + 1.0;
    return R < 512.0 && rcp + 3.0 * R < 512.0;
}

// Scale of the LDS sums: a component of a pair's force is below 10 / app^2 (as
// in pp_prepare) and kDrainPairs of them stay below 2^62.
float pp_sparse_scale(double app) {
    return std::ldexp(1.0f, (int)std::floor(62.0 - std::log2(10.0 / (app * app) * kDrainPairs)));
}

// A coarse cell has up to kParts items and kParts more per kItemCount particles
// around it; a slot is around 27 coarse cells.
size_t pp_sparse_items(int64_t ncoarse, int64_t n_used) {
    return (size_t)(ncoarse * kParts + n_used * 27 * kParts / kItemCount + 1);
}

int launch_pp_sparse(const PPArgs& a, const int* rhoc, int nt, int ncb, int ncoarse, int2* items,
                     size_t cap, int small, int mode, hipStream_t s) {
    const float scale = pp_sparse_scale(ctx().g.p.app);
    const double inv = 1.0 / (double)scale;
    if (ncoarse <= 0) return CUBE2_OK;
    Stage st("pp_pairs_sparse");
    int dev = 0, ncu = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        ncu = 256;
    // as the pair kernel's: far more blocks than are resident, so that the
    // hardware balances their uneven costs
    const unsigned blocks = (unsigned)std::min(ceil_div((size_t)ncoarse * kParts, 4), (unsigned)std::max(1, ncu) * 64u);
    int* count = a.taken + kPartRuns * kRunPad;
    k_sparse_items<<<ceil_div((size_t)ncoarse, 256), 256, 0, s>>>(rhoc, nt, ncb, ncoarse, a.tiles, &a.red->err,
                                                                  (int)cap, items, count);
    C2_HIP(hipGetLastError());
    if (mode == CUBE2_PP_REF) k_pp_sparse<kModeRef><<<blocks, 256, 0, s>>>(a, items, (int)cap, count, nt, small, scale, inv);
    else k_pp_sparse<kModeFast><<<blocks, 256, 0, s>>>(a, items, (int)cap, count, nt, small, scale, inv);
    C2_HIP(hipGetLastError());
    return CUBE2_OK;
}

}  // namespace cube2
