// PP pair kernel of the pairs-once pass (REF and FAST): a pair of two active
// particles of one range is evaluated once and its force added to both.
//
// The pair force is exactly antisymmetric (RN(a - b) = -RN(b - a)).  Of two
// active particles of one tile and range in cells of more than `small`
// particles, the one with the lower sorted index evaluates the pair; other j
// (halo copies, other levels, particles of small cells) act on i alone, and
// the small cells' particles evaluate all their pairs themselves
// (pp_sparse.hip).  Sums are kept as signed 64-bit fixed point per particle
// (integer adds commute: the result does not depend on the order of the
// atomics).
//
// A chunk is physical particles of one PP cell: the whole cell if it holds
// fewer than 64, else 2^dense_lg at a time (32 built in) in the Morton sub-cell
// order of k_pp_subsort, so that a chunk is spatially compact.  A chunk of many
// candidates is split into parts of about 2048 of them (k_chunk_flags), any
// wavefront taking any part: whole chunks took 0.3 ms on average but up to 29
// ms in a clump, and the kernel waited for the last of them (the chunks' times
// at 256^3 summed to 19.5 ms of all wavefronts' time, the kernel took 32; at
// 128^3 1.9 and 3.9).  Wavefronts take parts from counters, one for each of
// kPartRuns runs of the list (one counter for all serialised them, 15 ns a
// part: a 64^3 lattice 0.50 ms, with runs 0.15), so that a second launch on
// another stream can join at any time: beside PM3 the kernel runs at half its
// occupancy, which leaves registers for the mesh kernels, and PM3's stream
// helps once it is done.  The j of the
// (2R+1)^2 neighbour rows are contiguous runs of the sorted particles; a
// wavefront concatenates them into one candidate list, fetches it 64 at a
// time (one coalesced load, a batch ahead) and keeps the j within the range
// of the chunk's bounding box.  Each 64 kept j then meet the I particles of
// the chunk (rounded up to a power of two) in I steps: at step s, lane l
// takes j (l + s) mod 64 and i = l mod I, so that each j meets I consecutive
// lanes, every i once, and its reaction moves along with it, rotated by one
// lane per step in the DPP operand of the add that sums it: one pair per lane
// and three additions a step (summing a j's reaction over the lanes of one
// step took 18 instructions more).  The forces on i are summed in FP32 over
// one such block and in FP64 over the blocks.
//
// Bound by VALU issue (about 95 instructions per step; 0.36 a SIMD cycle at 42 of
// 64 lanes, 0.54 TB/s) and, in clumps, the reactions' atomics: they are laid out by component, so that the 64 lanes'
// atomics of one instruction fall into a few cache lines (by particle, three
// times as many: 64^3 lattice 0.154 -> 0.115 ms).  REF at 256^3 (16.7 M
// particles, clustered): 28 ms of the kick's 85, beside 7.9 ms for the small
// cells (57.8 ms in one kernel with a chunk for every cell, the kick 104.2;
// 60.9 and 109.7 with each j's reaction summed over the lanes at each step);
// at 128^3 3.0 ms, 512 uneven tiles 5.3, 120^3 in level-6 cells 4.2 (whole
// chunks by a static stride 3.9, 5.4, 8.2).
#include <algorithm>
#include <climits>

#include "pp_kernels.h"
#include "pp_law.h"
#include "profile.h"
#include "reduce.h"

namespace cube2 {

static_assert(kPartRuns == 64, "one lane per run");

constexpr int kJBlock = 96;  // a block of 64 j and its first 32 again

struct NewtonLDS {
    float4 jb[2 * kJBlock];  // two blocks of kept j (w: sorted index, INT_MAX: acts on i alone)
    double acc[3][64];       // per lane force sums
    int rs[64], rp[64];      // row group: j = v + rs[k] for rp[k-1] <= v < rp[k]
};

// x from the next higher lane, lane 63 from lane 0 (DPP, folded into the add
// that uses it).  Every lane must be active.
__device__ inline float wave_rol1(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x134, 0xf, 0xf, true));
}

// First of the candidates [0, m) that part p of np takes.
__device__ inline int part_of(int m, int p, int np) { return (int)((long long)m * p / np); }

template <int kMode, int kJB>
__global__ __launch_bounds__(256, 6) void k_pp_newton(PPArgs A, const int* __restrict__ chunks,
                                                      const int* __restrict__ first, int small,
                                                      int dense_lg) {
    static_assert(kJB == 64 || kJB == 128, "j batch of 64 or 128");
    constexpr int kH = kJB / 64;  // fetched float4 per lane per batch
    __shared__ NewtonLDS lds[4];
    const int wave = uni((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    NewtonLDS& L = lds[wave];
    const int nparts = uni(first[A.cap]);
    const uint64_t lt = lane ? (~0ull >> (64 - lane)) : 0ull;
    const FraK Ka = uni(make_frak(A.app));
    unsigned long long pc = 0, pa = 0;  // (wavefront-uniform)
    // run r of the list: parts [r len, (r + 1) len)
    const int len = (nparts + kPartRuns - 1) / kPartRuns;
    int run = (int)(blockIdx.x % kPartRuns);
    auto take = [&]() { return lane == 0 ? atomicAdd(&A.taken[run * kRunPad], 1) : 0; };
    int got = uni(take());
    for (;;) {
        if (got >= len || run * len + got >= nparts) {  // run done: the next one that is not
            const int have = __hip_atomic_load(&A.taken[lane * kRunPad], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            uint64_t open = __ballot(have < len && lane * len + have < nparts);
            if (!open) break;
            const uint64_t after = run == 63 ? 0ull : open & (~0ull << (run + 1));
            run = __ffsll((unsigned long long)(after ? after : open)) - 1;
            got = uni(take());
            continue;
        }
        const int ck = run * len + got;
        const int nxt = take();  // (in flight during the part)
        const int k = A.order ? uni(A.order[ck]) : ck, a0 = uni(chunks[k]);
        // the part of the chunk, and the chunk's parts
        const int f0 = uni(first[a0]), np = uni(first[a0 + 1]) - f0, part = k - f0;
        const uint32_t cid = (uint32_t)uni((int)A.cellid[a0]);
        const int cend = uni(A.cell_start[cid + 1]), cbeg = uni(A.cell_start[cid]);
        const bool grouped = cend - cbeg >= 64;
        const int ni = min(grouped ? 1 << dense_lg : 64, cend - a0);
        int lgI = 0;
        while ((1 << lgI) < ni) lgI++;
        const int I = 1 << lgI;
        const int islot = lane & (I - 1);
        const bool vi = islot < ni;
        const int ia = a0 + (vi ? islot : 0);
        const float4 p = A.pos4[ia];
        const int ti = uni(pp_find_tile(A.tiles, A.ntile, cid));
        const PPTile T = A.tiles[ti];
        const unsigned long long pc0 = pc, pa0 = pa;
        const int S = T.S;
        const unsigned key = cid - (unsigned)T.cell_off;
        const int z = (int)(key / ((unsigned)S * S)), y = (int)(key / S % S), x = (int)(key % S);
        const float range = fabsf(uni(p.w));  // one subtile per PP cell: one range
        const int R = (int)ceilf(__fmul_rn(range, (float)T.rcp) / (float)A.ratio_cs);
        const float pp2 = __fmul_rn(range, range);
        const FraK Kr = uni(make_frak(range));
        // A chunk whose stencil lies inside its own subtile meets only j of
        // its own range, so it skips the rows and cells before its own.
        bool interior;
        {
            const int cps = A.ntt * T.rcp, span = S - 2 * T.rcp;
            auto inside = [&](int c) {
                const int lo = c - R - T.rcp, hi = c + R - T.rcp;
                return lo >= 0 && hi < span && lo / cps == hi / cps;
            };
            interior = inside(x) && inside(y) && inside(z);
        }
        // bounding box of the chunk's i; a j farther than the range from it
        // cannot pair with any of them (the 1e-4 relative margin keeps every
        // j the per-pair test could accept)
        float bx0 = p.x, bx1 = p.x, by0 = p.y, by1 = p.y, bz0 = p.z, bz1 = p.z;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            bx0 = fminf(bx0, __shfl_xor(bx0, o, 64));
            bx1 = fmaxf(bx1, __shfl_xor(bx1, o, 64));
            by0 = fminf(by0, __shfl_xor(by0, o, 64));
            by1 = fmaxf(by1, __shfl_xor(by1, o, 64));
            bz0 = fminf(bz0, __shfl_xor(bz0, o, 64));
            bz1 = fmaxf(bz1, __shfl_xor(bz1, o, 64));
        }
        bx0 = uni(bx0);
        bx1 = uni(bx1);
        by0 = uni(by0);
        by1 = uni(by1);
        bz0 = uni(bz0);
        bz1 = uni(bz1);
        const float pp2m = pp2 * 1.0001f;
        // the pair tests' i position: a far-away one for lanes past the chunk
        const float pix = vi ? p.x : -kFar, piy = vi ? p.y : -kFar, piz = vi ? p.z : -kFar;
#pragma unroll
        for (int c = 0; c < 3; c++) L.acc[c][lane] = 0.0;
        unsigned npa = 0, ncand = 0;
        int jhead = 0, jtail = 0;  // kept j taken and staged
        const int xlo = max(x - R, 0), xhi = min(x + R, S - 1);
        const int W = 2 * R + 1, nrows = W * W;
        // neighbour rows in groups of 64: a group's runs form one virtual
        // list of M candidates
        for (int rg = 0; rg < nrows; rg += 64) {
            int js = 0, cnt = 0, cfull = 0;
            const int r = rg + lane;
            if (r < nrows) {
                const int zz = z + r / W - R, yy = y + r % W - R;
                if (zz >= 0 && zz < S && yy >= 0 && yy < S) {
                    const unsigned row = (unsigned)T.cell_off + ((unsigned)zz * S + yy) * S;
                    js = A.cell_start[row + xlo];
                    cnt = A.cell_start[row + xhi + 1] - js;
                    cfull = cnt;
                    if (interior && zz * S + yy <= z * S + y) {
                        // rows before the chunk's: none; its own row: from its
                        // first i -- unless a small cell (in the learned kick
                        // one of the network's) lies there, whose j act on
                        // this chunk's i only from here
                        const bool own = zz * S + yy == z * S + y;
                        const int xe = own ? x : xhi + 1;
                        bool has_small = false;
                        const int marked = range == A.learned_range ? max(small, A.learned_occ - 1) : small;
                        if (marked > 0) {
                            int c0 = js;
                            for (int xc = xlo; xc < xe; xc++) {
                                const int c1 = A.cell_start[row + xc + 1];
                                has_small |= c1 - c0 > 0 && c1 - c0 <= marked;
                                c0 = c1;
                            }
                        }
                        if (!has_small) {
                            const int j0 = own ? a0 : js + cnt;
                            cnt -= j0 - js;
                            js = j0;
                        }
                    }
                }
            }
            // the candidates counted: the whole stencil, for each i
            int sf = cfull;
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) sf += __shfl_xor(sf, o, 64);
            if (part == 0) ncand += (unsigned)uni(sf);
            int inc = cnt;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int t = __shfl_up(inc, o, 64);
                if (lane >= o) inc += t;
            }
            const int M0 = uni(__shfl(inc, 63, 64));
            // the part's candidates [v0, M) of the group's
            const int v0 = part_of(M0, part, np), M = part_of(M0, part + 1, np);
            L.rs[lane] = js - (inc - cnt);
            L.rp[lane] = inc;
            wave_lds_sync();
            // a lane's candidates v = vb + lane only grow, so its row (the
            // first with rp > v) is found by walking forward from the last
            // one: rp of the rows past the group is M > v, so the walk stops
            // inside the group
            int frow = 0;  // (rp of the last row is the group's M0 >= M)
            auto fetch = [&](int vb, int& jx) {
                const int v = vb + lane;
                float4 q4 = make_float4(0.f, 0.f, 0.f, 0.f);
                if (v < M) {
                    while (L.rp[frow] <= v) frow++;
                    jx = v + L.rs[frow];
                    q4 = A.pos4[jx];
                }
                return q4;
            };
            float4 qcur[kH];
            int jcur[kH] = {};
#pragma unroll
            for (int h = 0; h < kH; h++) qcur[h] = fetch(v0 + 64 * h, jcur[h]);
            // (a last step without candidates takes the j left over)
            const bool last = rg + 64 >= nrows;
            const int vend = last ? v0 + (M - v0 + kJB - 1) / kJB * kJB + kJB : M;
            for (int vb = v0; vb < vend; vb += kJB) {
#pragma unroll
                for (int h = 0; h < kH; h++) {
                    float4 qh = qcur[h];
                    const int jx = qh.w == range ? jcur[h] : INT_MAX;
                    qh.w = __int_as_float(jx);
                    const float ex = fmaxf(fmaxf(bx0 - qh.x, qh.x - bx1), 0.0f);
                    const float ey = fmaxf(fmaxf(by0 - qh.y, qh.y - by1), 0.0f);
                    const float ez = fmaxf(fmaxf(bz0 - qh.z, qh.z - bz1), 0.0f);
                    // (a j of the chunk's range before its first i evaluates
                    // the pair itself)
                    const bool keep = (vb + 64 * h + lane < M) & (jx >= a0) &
                                      (ex * ex + ey * ey + ez * ez < pp2m);
                    const uint64_t km = __ballot(keep);
                    if (keep) {
                        const int t = jtail + __popcll(km & lt);
                        const int at = (t >> 6 & 1) * kJBlock + (t & 63);
                        L.jb[at] = qh;
                        if ((t & 63) < 32) L.jb[at + 64] = qh;
                    }
                    jtail += __popcll(km);
                    if (h == kH - 1) {
#pragma unroll
                        for (int k = 0; k < kH; k++)
                            if (vb + kJB + 64 * k < M) qcur[k] = fetch(vb + kJB + 64 * k, jcur[k]);
                    }
                    const bool rest = last && vb + kJB >= vend && h == kH - 1;
                    if (jtail - jhead < 64 && !(rest && jtail > jhead)) continue;
                    const int bb = (jhead >> 6 & 1) * kJBlock;
                    if (rest && lane >= jtail - jhead) {  // far-away j to the block's end
                        const float4 far4 = make_float4(kFar, kFar, kFar, __int_as_float(INT_MAX));
                        L.jb[bb + lane] = far4;
                        if (lane < 32) L.jb[bb + lane + 64] = far4;
                    }
                    wave_lds_sync();
                    float rx = 0.0f, ry = 0.0f, rz = 0.0f, dx = 0.0f, dy = 0.0f, dz = 0.0f;
                    for (int s0 = 0; s0 < I; s0 += 32) {
                        const float4* jp = &L.jb[bb + ((lane + s0) & 63)];
                        const int ns = uni(min(32, I - s0));
                        for (int s = 0; s < ns; s++, jp++) {
#pragma clang fp contract(off)
                            const float4 qj = *jp;
                            const int jw = __float_as_int(qj.w);
                            float4 e;
                            e.x = qj.x - pix;
                            e.y = qj.y - piy;
                            e.z = qj.z - piz;
                            e.w = e.x * e.x + e.y * e.y + e.z * e.z;
                            const bool ok = (e.w > 0.0f) & (e.w < pp2) & (jw > ia);
                            const uint64_t okm = __ballot(ok);
                            npa += 2 * __popcll(okm) - __popcll(okm & __ballot(jw == INT_MAX));
                            float fx = 0.0f, fy = 0.0f, fz = 0.0f;
                            if (ok) {
                                pair_force<kMode>(e, Ka, Kr, fx, fy, fz);
                                dx += fx;
                                dy += fy;
                                dz += fz;
                            }
                            rx = wave_rol1(rx) + fx;
                            ry = wave_rol1(ry) + fy;
                            rz = wave_rol1(rz) + fz;
                        }
                    }
                    L.acc[0][lane] += (double)dx;
                    L.acc[1][lane] += (double)dy;
                    L.acc[2][lane] += (double)dz;
                    // lane l now holds the reaction of j (l + I - 1) mod 64
                    const int jw = __float_as_int(L.jb[bb + ((lane + I - 1) & 63)].w);
                    if (jw != INT_MAX) {
                        unsigned long long* d = A.react + jw;
                        fixed_add(d, -rx, A.react_scale);
                        fixed_add(d + A.cap, -ry, A.react_scale);
                        fixed_add(d + 2 * (size_t)A.cap, -rz, A.react_scale);
                    }
                    jhead += 64;
                    wave_lds_sync();
                }
            }
        }
        // the i's own sums (their 64 / I lanes added) join their reactions;
        // k_pp_newton_terms forms the velocity term once every chunk has
        // added to it
        if (vi && lane < I) {
#pragma unroll
            for (int c = 0; c < 3; c++) {
                double v = 0.0;
                for (int q = lane; q < 64; q += I) v += L.acc[c][q];
                fixed_add(A.react + c * (size_t)A.cap + ia, v, A.react_scale);
            }
        }
        // (each i once for the chunk, and not with itself)
        if (part == 0) pc += (unsigned long long)(ncand - 1u) * (unsigned)ni;
        pa += npa;
        if (A.tile_pairs && lane == 0) {  // per-tile counts (on request only)
            atomicAdd(&A.tile_pairs[2 * ti], pc - pc0);
            atomicAdd(&A.tile_pairs[2 * ti + 1], pa - pa0);
        }
        wave_lds_sync();  // acc and the blocks are reused by the next chunk
        got = uni(nxt);
    }
    const unsigned long long sm[2] = {lane == 0 ? pc : 0ull, lane == 0 ? pa : 0ull};
    block_sum_to<2>(&A.red->p_cand, sm);
}

int launch_pp_newton(const PPArgs& a, const int* chunks, const int* first, int grid, int small,
                     int mode, bool help, hipStream_t s) {
    Stage st(help ? "pp_pairs_help" : mode == CUBE2_PP_REF ? "pp_pairs_ref" : "pp_pairs_fastq");
    const unsigned blocks = (unsigned)std::max(1, grid);
    const int dl = pp_dense_lg(true);
    if (mode == CUBE2_PP_REF && pp_jbatch() == 128)
        k_pp_newton<kModeRef, 128><<<blocks, 256, 0, s>>>(a, chunks, first, small, dl);
    else if (mode == CUBE2_PP_REF)
        k_pp_newton<kModeRef, 64><<<blocks, 256, 0, s>>>(a, chunks, first, small, dl);
    else if (pp_jbatch() == 128)
        k_pp_newton<kModeFast, 128><<<blocks, 256, 0, s>>>(a, chunks, first, small, dl);
    else
        k_pp_newton<kModeFast, 64><<<blocks, 256, 0, s>>>(a, chunks, first, small, dl);
    C2_HIP(hipGetLastError());
    return CUBE2_OK;
}

}  // namespace cube2
