// Kernels of the learned PP stand-in: a 3-D CNN of 3^3 valid convolutions
// in channels-last layout (activation [patch][z][y][x][channel], FP32),
// convolved on the matrix cores (k_conv3); for grids larger than training
// patches (those: cnn_bwd.hip) the backward is im2col (BF16) and a BF16 GEMM
// with FP32 accumulation on transposed operands.
//
// GEMM: C[m][n] (+)= sum_k A(m,k) B(k,n), A(m,k) = A[m*sam + k*sak],
// B(k,n) = B[k*sbk + n*sbn], C row-major with leading dimension ldc.  One
// wavefront owns a 32 x 32 tile of C as 2 x 2 v_mfma_f32_16x16x16_bf16
// tiles; operand lanes: A row m0 + (lane % 16), K values 4 (lane / 16) +
// 0..3; B column n0 + (lane % 16), the same K values; result lane holds rows
// 4 (lane / 16) + 0..3 of column lane % 16.  Out-of-range operands are
// zeros, so any M, N, K work.
#include <algorithm>
#include <type_traits>

#include "adam.h"
#include "common.h"
#include "engine.h"

namespace cube2 {

typedef short v4s __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

// FP32 -> BF16, round to nearest even (finite inputs).
__device__ inline uint16_t to_bf16(float f) {
    const uint32_t u = __float_as_uint(f);
    return (uint16_t)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
}

// Split K: block z of gridDim.z takes k in [z*kc, (z+1)*kc) and stores its
// partial product to C + z*zs (the partials are then summed in order).
__global__ __launch_bounds__(256) void k_gemm_bf16(const uint16_t* __restrict__ A, int64_t sam,
                                                   int64_t sak, const uint16_t* __restrict__ B,
                                                   int64_t sbk, int64_t sbn, float* __restrict__ C,
                                                   int64_t ldc, int M, int N, int K, int acc,
                                                   int kc, int64_t zs) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int kbeg = blockIdx.z * kc, kend = min(K, kbeg + kc);
    A += (int64_t)kbeg * sak;
    B += (int64_t)kbeg * sbk;
    K = kend - kbeg;
    C += blockIdx.z * zs;
    const int m0 = blockIdx.y * 64 + (wave >> 1) * 32, n0 = blockIdx.x * 64 + (wave & 1) * 32;
    const int r16 = lane & 15, kq = (lane >> 4) * 4;
    v4f d[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) d[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
    // A rows contiguous in k and 8-byte aligned: one 8-byte load per lane
    const bool avec = sak == 1 && (sam & 3) == 0 && ((uintptr_t)A & 7) == 0;
    for (int k0 = 0; k0 < K; k0 += 16) {
        v4s a[2], b[2];
        const bool kfull = k0 + 16 <= K;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int m = m0 + i * 16 + r16, n = n0 + i * 16 + r16;
            if (avec && kfull) {
                a[i] = m < M ? *reinterpret_cast<const v4s*>(A + (int64_t)m * sam + k0 + kq)
                             : v4s{0, 0, 0, 0};
            } else {
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int k = k0 + kq + q;
                    a[i][q] = (m < M && k < K) ? (short)A[(int64_t)m * sam + (int64_t)k * sak]
                                               : (short)0;
                }
            }
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int k = k0 + kq + q;
                b[i][q] = (n < N && k < K) ? (short)B[(int64_t)k * sbk + (int64_t)n * sbn] : (short)0;
            }
        }
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
                d[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[i], b[j], d[i][j], 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int m = m0 + i * 16 + kq + q, n = n0 + j * 16 + r16;
                if (m < M && n < N) {
                    float* c = C + (int64_t)m * ldc + n;
                    *c = acc ? *c + d[i][j][q] : d[i][j][q];
                }
            }
}

// C[m][n] (+)= sum over the S split-K partials P[s][m][n], in order.
__global__ void k_sum_partials(const float* __restrict__ P, float* __restrict__ C, int64_t ldc,
                               int M, int N, int S, int acc) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (int64_t)M * N) return;
    const int m = (int)(e / N), n = (int)(e % N);
    float v = 0.f;
    for (int s = 0; s < S; s++) v += P[(int64_t)s * M * N + e];
    float* c = C + (int64_t)m * ldc + n;
    *c = acc ? *c + v : v;
}

// col[(p, z, y, x)][((dz*3 + dy)*3 + dx)*Cin + c] = X[p][z+dz][y+dy][x+dx][c]
// for the (D-2)^3 output positions of a D^3 input.
__global__ void k_im2col3(const float* __restrict__ X, uint16_t* __restrict__ col, int B, int D,
                          int Cin) {
    const int P = D - 2, Kd = 27 * Cin;
    const int64_t tot = (int64_t)B * P * P * P * Kd;
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= tot) return;
    const int k = (int)(e % Kd);
    int64_t r = e / Kd;
    const int x = (int)(r % P), y = (int)((r / P) % P), z = (int)((r / ((int64_t)P * P)) % P);
    const int64_t p = r / ((int64_t)P * P * P);
    const int c = k % Cin, o = k / Cin, dx = o % 3, dy = (o / 3) % 3, dz = o / 9;
    col[e] = to_bf16(X[(((p * D + z + dz) * D + y + dy) * D + x + dx) * Cin + c]);
}

// dX[p][iz][iy][ix][c] = sum over the offsets (dz, dy, dx) whose output
// position (iz-dz, iy-dy, ix-dx) exists of dcol[that position][offset, c].
__global__ void k_col2im3(const float* __restrict__ dcol, float* __restrict__ dX, int B, int D,
                          int Cin) {
    const int P = D - 2, Kd = 27 * Cin;
    const int64_t tot = (int64_t)B * D * D * D * Cin;
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= tot) return;
    const int c = (int)(e % Cin);
    int64_t r = e / Cin;
    const int ix = (int)(r % D), iy = (int)((r / D) % D), iz = (int)((r / ((int64_t)D * D)) % D);
    const int64_t p = r / ((int64_t)D * D * D);
    float s = 0.f;
    for (int dz = 0; dz < 3; dz++) {
        const int z = iz - dz;
        if (z < 0 || z >= P) continue;
        for (int dy = 0; dy < 3; dy++) {
            const int y = iy - dy;
            if (y < 0 || y >= P) continue;
            for (int dx = 0; dx < 3; dx++) {
                const int x = ix - dx;
                if (x < 0 || x >= P) continue;
                const int64_t row = ((p * P + z) * P + y) * P + x;
                s += dcol[row * Kd + ((dz * 3 + dy) * 3 + dx) * Cin + c];
            }
        }
    }
    dX[e] = s;
}

__global__ void k_bias_act(float* __restrict__ Y, const float* __restrict__ bias, int64_t n, int C,
                           int relu) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    float v = Y[e] + bias[e % C];
    Y[e] = relu ? fmaxf(v, 0.f) : v;
}

// dY *= (Y > 0) for a ReLU layer; dY as BF16 for the GEMMs.
__global__ void k_act_bwd(const float* __restrict__ Y, float* __restrict__ dY,
                          uint16_t* __restrict__ dYb, int64_t n, int relu) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    float g = dY[e];
    if (relu && !(Y[e] > 0.f)) g = 0.f;
    dY[e] = g;
    dYb[e] = to_bf16(g);
}

// dbias[c] = sum over rows of dY[row][c]: one block per channel, fixed order.
__global__ __launch_bounds__(256) void k_colsum(const float* __restrict__ dY, float* __restrict__ db,
                                                int64_t rows, int C) {
    __shared__ float red[256];
    const int c = blockIdx.x;
    float s = 0.f;
    for (int64_t r = threadIdx.x; r < rows; r += blockDim.x) s += dY[r * C + c];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) db[c] = red[0];
}

__global__ void k_to_bf16(const float* __restrict__ x, uint16_t* __restrict__ y, int64_t n) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e < n) y[e] = to_bf16(x[e]);
}

// Adam on FP32 master weights (bias-corrected step t >= 1); refreshes the
// BF16 copy the GEMMs read when wb is given.
__global__ void k_adam(float* __restrict__ w, const float* __restrict__ g, float* __restrict__ m,
                       float* __restrict__ v, uint16_t* __restrict__ wb, int64_t n, float lr,
                       float b1, float b2, float eps, float c1, float c2) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    float mi = m[e], vi = v[e];
    const float wi = adam_update(w[e], g[e], mi, vi, lr, b1, b2, eps, c1, c2);
    m[e] = mi;
    v[e] = vi;
    w[e] = wi;
    if (wb) wb[e] = to_bf16(wi);
}

// Mean squared error over n values and its gradient 2 (out - t) / n.
__global__ __launch_bounds__(256) void k_mse(const float* __restrict__ out,
                                             const float* __restrict__ t, float* __restrict__ d,
                                             float* __restrict__ loss, int64_t n) {
    __shared__ float red[256];
    float s = 0.f;
    for (int64_t e = threadIdx.x; e < n; e += blockDim.x) {
        const float r = out[e] - t[e];
        d[e] = 2.f * r / (float)n;
        s += r * r;
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) *loss = red[0] / (float)n;
}

// ------------------------------------------------------ 3^3 convolution
// Y[b][z][y][x][o] = act(bias[o] + sum over taps t = (dz, dy, dx) and input
// channels c of X[b][z+dz][y+dy][x+dx][c] * W[t*CIN + c][o]) for the
// P^3 = (D-2)^3 outputs of each of B inputs of D^3 x CIN cells
// (channels-last), on v_mfma_f32_16x16x32_bf16 (BF16 operands, FP32
// accumulation) with no materialised im2col.
//
// MFMA operands: lane l holds row (output channel) l % 16 of A and column
// (position) l % 16 of B with K indices 8 (l / 16) + 0..7; the result lane
// holds channels 4 (l / 16) + 0..3 of position l % 16, so that its store is
// one 16-byte (BF16: 8-byte) access.  K runs over (tap, channel) with the
// channel fastest: for CIN = 32 one K step is one tap; for CIN = 4 a step is
// 8 taps (taps 27..31 are zeros).
//
// The 16 positions of a tile are tx (16, 8 or 4) consecutive x of 16 / tx
// grids, whichever wastes the fewest positions (conv_tile): subtile grids of
// 72^3 outputs divide by 8, training patches have 8^3, 6^3, 4^3 and 2^3.
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v4bf __attribute__((ext_vector_type(4)));
// The same in memory, at any address of their elements (one 16-byte access
// wherever it begins): activations are a caller's, views among them.
typedef v8bf v8bf_at __attribute__((aligned(2)));
typedef float v4f_at __attribute__((ext_vector_type(4), aligned(4)));

struct ConvTile {
    int tx;   // consecutive x of a tile (16, 8, 4); 16 / tx grids side by side
    int nx, ny, nz, nb;  // tiles along x, rows of tiles, z chunks, groups of grids
    int zc;   // output planes of a z chunk
};

// 16 bytes of BF16 channels from 8 values of the input.
__device__ inline v8bf load_bf16x8(const uint16_t* p) { return *reinterpret_cast<const v8bf_at*>(p); }
__device__ inline v8bf load_bf16x8(const float* p) {
    const v4f a = reinterpret_cast<const v4f_at*>(p)[0], b = reinterpret_cast<const v4f_at*>(p)[1];
    return v8bf{(__bf16)a[0], (__bf16)a[1], (__bf16)a[2], (__bf16)a[3],
                (__bf16)b[0], (__bf16)b[1], (__bf16)b[2], (__bf16)b[3]};
}

// The output channel in MFMA row r (0..15) of row tile ct.  BF16 outputs: a
// lane's two result tiles are then 8 consecutive channels, 16 bytes.
template <class TOut>
__device__ inline int conv_channel(int ct, int r) {
    return sizeof(TOut) == 2 ? 8 * (r >> 2) + 4 * ct + (r & 3) : ct * 16 + r;
}

// Stores a lane's two result tiles at its position's channels.
__device__ inline void store32(uint16_t* row, int kq, const v4f& u, const v4f& v) {
    *reinterpret_cast<v8bf_at*>(row + 8 * kq) =
        v8bf{(__bf16)u[0], (__bf16)u[1], (__bf16)u[2], (__bf16)u[3],
             (__bf16)v[0], (__bf16)v[1], (__bf16)v[2], (__bf16)v[3]};
}
__device__ inline void store32(float* row, int kq, const v4f& u, const v4f& v) {
    *reinterpret_cast<v4f_at*>(row + 4 * kq) = u;
    *reinterpret_cast<v4f_at*>(row + 16 + 4 * kq) = v;
}

// 32 input channels.  A wavefront owns 4 rows of tiles (4 y of tx x) and
// marches along a chunk of z: the input plane's 6 rows are read into
// registers once for the 27 taps and 4 output rows that use them, against
// accumulators of the three output planes in progress.  Weights (55 KB) are in
// LDS for the workgroup's life, a fragment read there feeds 4 MFMAs (half
// of LDS's rate); the next plane's cells are fetched during this plane's
// MFMAs, converted, and put into the wavefront's own LDS buffer, so that
// wavefronts never wait for each other.  LDS rows of 64 bytes are swizzled
// in 16-byte units by (row / 4) % 4: the 16 rows a quarter wavefront reads lie
// in distinct banks.  Each accumulator takes its taps in the order 0..26.
// 8 wavefronts of up to 256 VGPRs fill a CU.  8 grids of 72^3 FP32 inputs:
// 235 and 205 us for the two 32 -> 32 layers (0.73 and 0.67 GB, 3.2 TB/s; 670
// TFLOP/s) and 111 us for 32 -> 3; a workgroup with one staged block of 4 x 4 x
// 8 outputs, every fragment read from LDS for each 2 MFMAs, took 666, 536 and
// 318 us.
constexpr int kConvWaves = 8;
constexpr int kConvRows = 4;                   // output rows of a wavefront
constexpr int kConvIn = kConvRows + 2;         // staged rows of a wavefront
constexpr int kConvRow = 32 * 4;               // a staged row: 32 cells of 4 16-byte parts
constexpr int kConvItems = kConvIn + 3;        // 16-byte items a lane stages

// In 16-byte units: part kq of weight row (channel) r, and of cell x of grid
// g of a staged row (16 / tx grids of tx + 2 cells; gs cells from one to the
// next).
__device__ inline int conv_w_addr(int r, int kq) { return r * 4 + (kq ^ ((r >> 2) & 3)); }
__device__ inline int conv_x_addr(int tx, int g, int x, int kq) {
    const int gs = tx == 8 ? 16 : 8, turn = tx == 8 ? 2 * g : g;  // (tx 16: g = 0)
    return (g * gs + x) * 4 + (kq ^ (((x >> 2) + turn) & 3));
}

template <int NT>
constexpr size_t conv_lds_bytes() {
    return (size_t)27 * NT * 16 * 64 + (size_t)kConvWaves * kConvIn * kConvRow * 16;
}

template <int NT, class TIn, class TOut>
__global__ __launch_bounds__(kConvWaves * 64) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_conv3(
    const TIn* __restrict__ X, const uint16_t* __restrict__ Wp, const float* __restrict__ bias,
    TOut* __restrict__ Y, int B, int D, int cout, int relu, ConvTile T) {
    extern __shared__ __align__(16) uint4 conv_lds[];
    uint4* wl = conv_lds;  // [tap][NT*16 channels][32], swizzled
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    uint4* xl = conv_lds + 27 * NT * 64 + wave * kConvIn * kConvRow;
    for (int i = tid; i < 27 * NT * 64; i += kConvWaves * 64) {
        const int r = i >> 2, row = r % (NT * 16);
        wl[conv_w_addr(r, i & 3)] = reinterpret_cast<const uint4*>(
            Wp)[(r - row + conv_channel<TOut>(row >> 4, row & 15)) * 4 + (i & 3)];
    }
    __syncthreads();
    const int P = D - 2, r16 = lane & 15, kq = lane >> 4;
    const int ng = 16 / T.tx, rs = T.tx + 2;
    const int xs = r16 % T.tx, gi = r16 / T.tx;  // the lane's position
    int xa[3];                                   // its cells' addresses in a staged row
#pragma unroll
    for (int dx = 0; dx < 3; dx++) xa[dx] = conv_x_addr(T.tx, gi, xs + dx, kq);
    const int wa = conv_w_addr(r16, kq);
    // A row is ng * rs * 4 items of 16 bytes (72, 80 or 96): the first 64 are
    // one per lane, the rest of the 6 rows fill up to three more steps.
    const int rest = ng * rs * 4 - 64;
    int scell[4], srow[4], dst[4];  // [0]: the main step (row added per row)
#pragma unroll
    for (int m = 0; m < 4; m++) {
        const int e = (m - 1) * 64 + lane;
        srow[m] = m ? min(e / rest, kConvIn - 1) : 0;
        const int i = m ? 64 + e % rest : lane;
        const int g = (i >> 2) / rs, x = (i >> 2) - g * rs;
        scell[m] = g * 64 + x;  // (x < 18)
        dst[m] = srow[m] * kConvRow + conv_x_addr(T.tx, g, x, i & 3);
    }
    const uint32_t items = (uint32_t)T.nb * T.nx * T.ny * T.nz;
    // (neighbouring items share input rows: one XCD takes a run of them)
    for (uint32_t it = xcd_remap(blockIdx.x, gridDim.x) * kConvWaves + wave; it < items;
         it += gridDim.x * kConvWaves) {
        uint32_t q = it;
        const int ix = (int)(q % T.nx);
        q /= T.nx;
        const int iy = (int)(q % T.ny);
        q /= T.ny;
        const int iz = (int)(q % T.nz), b0 = (int)(q / T.nz) * ng;
        const int x0 = ix * T.tx, y0 = iy * kConvRows, z0 = iz * T.zc;
        const int nz = min(T.zc, P - z0);  // output planes of the chunk
        // staged items' places in the input plane (cells past the grid repeat
        // its last ones; they reach only positions that are not stored)
        int src[4];
#pragma unroll
        for (int m = 0; m < 4; m++) {
            const int gb = min(scell[m] >> 6, B - 1 - b0), gx = min(x0 + (scell[m] & 63), D - 1);
            const int gy = m ? min(y0 + srow[m], D - 1) : 0;
            src[m] = ((gb * D * D + gy) * D + gx) * 32 + (lane & 3) * 8;
        }
        const TIn* Xp = X + ((int64_t)b0 * D + z0) * D * D * 32;
        auto item = [&](int k) {
            if (k < kConvIn) return load_bf16x8(Xp + (int64_t)min(y0 + k, D - 1) * D * 32 + src[0]);
            return load_bf16x8(Xp + src[k - kConvIn + 1]);
        };
        v4f acc[3][kConvRows][NT];
        v8bf nxt[kConvItems];
        auto stage = [&]() {
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int k = 0; k < kConvItems; k++)
                *reinterpret_cast<v8bf*>(xl + (k < kConvIn ? k * kConvRow + dst[0] : dst[k - kConvIn + 1])) = nxt[k];
            __builtin_amdgcn_wave_barrier();
        };
#pragma unroll
        for (int k = 0; k < kConvItems; k++) nxt[k] = item(k);
        stage();
        // Input plane zz of the chunk (R = zz % 3): tap plane dz of output
        // plane zz - dz, accumulated in slot (R - dz) mod 3.
        auto plane = [&](auto r_c, int zz) {
            constexpr int R = decltype(r_c)::value;
            Xp += (int64_t)D * D * 32;
            const bool more = zz + 1 < nz + 2;
#pragma unroll
            for (int y = 0; y < kConvRows; y++)
#pragma unroll
                for (int ct = 0; ct < NT; ct++) acc[R][y][ct] = v4f{0.f, 0.f, 0.f, 0.f};
            v8bf a[kConvRows + 2][3];
            auto row = [&](int y) {
#pragma unroll
                for (int dx = 0; dx < 3; dx++)
                    a[y][dx] = *reinterpret_cast<const v8bf*>(xl + y * kConvRow + xa[dx]);
            };
#pragma unroll
            for (int y = 0; y < kConvRows - 1; y++) row(y);
#pragma unroll
            for (int dy = 0; dy < 3; dy++) {
                row(kConvRows - 1 + dy);
                if (more) {  // a third of the next plane's items
#pragma unroll
                    for (int k = dy * kConvItems / 3; k < (dy + 1) * kConvItems / 3; k++)
                        nxt[k] = item(k);
                }
#pragma unroll
                for (int dz = 0; dz < 3; dz++) {
                    const int o = zz - dz;
                    if (o < 0 || o >= nz) continue;
#pragma unroll
                    for (int dx = 0; dx < 3; dx++) {
                        const int t = dz * 9 + dy * 3 + dx;
                        v8bf w[NT];
#pragma unroll
                        for (int ct = 0; ct < NT; ct++)
                            w[ct] = *reinterpret_cast<const v8bf*>(
                                wl + (t * NT + ct) * 64 + wa);
#pragma unroll
                        for (int y = 0; y < kConvRows; y++)
#pragma unroll
                            for (int ct = 0; ct < NT; ct++)
                                acc[(R - dz + 3) % 3][y][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                    w[ct], a[y + dy][dx], acc[(R - dz + 3) % 3][y][ct], 0, 0, 0);
                    }
                }
            }
            // The next plane goes to LDS before this one's stores: a wavefront's
            // loads and stores complete in one order, so that waiting for
            // loads after the stores would wait for the stores too.
            if (more) stage();
            if (zz >= 2) {  // output plane zz - 2 is complete
                const int gz = z0 + zz - 2, gx = x0 + xs;
                if (gx < P && b0 + gi < B) {
#pragma unroll
                    for (int y = 0; y < kConvRows; y++) {
                        if (y0 + y >= P) continue;
                        if (NT == 1 && kq > 0) continue;  // 3 channels
                        TOut* out = Y + ((((int64_t)(b0 + gi) * P + gz) * P + y0 + y) * P + gx) * cout;
                        v4f v[NT];
#pragma unroll
                        for (int ct = 0; ct < NT; ct++)
#pragma unroll
                            for (int i = 0; i < 4; i++) {
                                const int o = conv_channel<TOut>(ct, 4 * kq + i);
                                v[ct][i] = acc[(R + 1) % 3][y][ct][i];
                                if (NT == 2 || i < 3) v[ct][i] += bias[o];
                                if (relu) v[ct][i] = fmaxf(v[ct][i], 0.f);
                            }
                        if constexpr (NT == 2) {
                            store32(out, kq, v[0], v[1]);
                        } else {
                            out[0] = v[0][0];
                            out[1] = v[0][1];
                            out[2] = v[0][2];
                        }
                    }
                }
            }
        };
        for (int zz = 0; zz < nz + 2; zz += 3) {
            plane(std::integral_constant<int, 0>{}, zz);
            if (zz + 1 < nz + 2) plane(std::integral_constant<int, 1>{}, zz + 1);
            if (zz + 2 < nz + 2) plane(std::integral_constant<int, 2>{}, zz + 2);
        }
    }
}

// 4 input channels (FP32): a wavefront takes tiles (one row of 16 positions,
// all 32 channels: 8 MFMAs) along kC4Rows rows of y, its weights in
// registers.  The 3 x (kC4Rows + 2) input rows of the item are fetched at
// once, converted and kept in the wavefront's own LDS; a lane reads its two
// taps of a K step from there.  Bound by the stores of the 32 output channels
// and the loads that queue behind them: 8 grids of 72^3 outputs (FP32, 382 MB)
// take 140 us, 79 without the stores and 85 without the loads.  Rows of 8 and
// the next item's loads ahead of the stores (more registers, fewer
// wavefronts): 150 and 174 us; taps straight from the grid, eight scattered
// loads a tile: 172.
constexpr int kC4Rows = 4;
constexpr int kC4Row = 24;                                  // staged cells of a row, at most
constexpr int kC4Items = (3 * (kC4Rows + 2) * kC4Row + 63) / 64;  // cells a lane stages

template <class TOut>
__global__ __launch_bounds__(256, 4) void k_conv3_c4(const float* __restrict__ X,
                                                  const uint16_t* __restrict__ Wp,
                                                  const float* __restrict__ bias,
                                                  TOut* __restrict__ Y, int B, int D, int relu,
                                                  ConvTile T) {
    __shared__ v4bf lds[4][kC4Items * 64];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    v4bf* xl = lds[wave];
    const int P = D - 2, r16 = lane & 15, kq = lane >> 4;
    const int xs = r16 % T.tx, gi = r16 / T.tx, ng = 16 / T.tx;
    const int rs = T.tx + 2, rc = ng * rs;  // cells of a grid's row, of a staged row
    v8bf w[4][2];
    int off[4][2];  // the lane's taps in the staged rows [dz][y][grid][x]
#pragma unroll
    for (int s = 0; s < 4; s++) {
#pragma unroll
        for (int ct = 0; ct < 2; ct++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const v4bf q = *reinterpret_cast<const v4bf*>(
                    Wp + ((8 * s + 2 * kq + h) * 32 + conv_channel<TOut>(ct, r16)) * 4);
#pragma unroll
                for (int j = 0; j < 4; j++) w[s][ct][4 * h + j] = q[j];
            }
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int t = min(8 * s + 2 * kq + h, 26);
            off[s][h] = (t / 9 * (kC4Rows + 2) + t / 3 % 3) * rc + gi * rs + xs + t % 3;
        }
    }
    float bs[2][4];
#pragma unroll
    for (int ct = 0; ct < 2; ct++)
#pragma unroll
        for (int i = 0; i < 4; i++) bs[ct][i] = bias[conv_channel<TOut>(ct, 4 * kq + i)];
    int cell[kC4Items];  // staged cell: dz << 20 | y << 16 | grid << 8 | x
#pragma unroll
    for (int k = 0; k < kC4Items; k++) {
        const int e = k * 64 + lane, row = min(e / rc, 3 * (kC4Rows + 2) - 1), c = e % rc;
        const int dz = row / (kC4Rows + 2);
        cell[k] = dz << 20 | (row - dz * (kC4Rows + 2)) << 16 | c / rs << 8 | c % rs;
    }
    // (an item is 128 output positions or more: the count fits 32 bits)
    const uint32_t nyc = (uint32_t)(P + kC4Rows - 1) / kC4Rows;
    const uint32_t items = (uint32_t)T.nb * P * T.nx * nyc;
    for (uint32_t it = xcd_remap(blockIdx.x, gridDim.x) * 4 + wave; it < items; it += gridDim.x * 4) {
        uint32_t q = it;
        const int x0 = (int)(q % T.nx) * T.tx;
        q /= T.nx;
        const int y0 = (int)(q % nyc) * kC4Rows;
        q /= nyc;
        const int gz = (int)(q % P), b0 = (int)(q / P) * ng;
        const v4f_at* Xi = reinterpret_cast<const v4f_at*>(X) + ((int64_t)b0 * D + gz) * D * D;
        v4f v[kC4Items];
#pragma unroll
        for (int k = 0; k < kC4Items; k++) {
            const int dz = cell[k] >> 20, y = min(y0 + (cell[k] >> 16 & 15), D - 1),
                      g = min(cell[k] >> 8 & 255, B - 1 - b0), x = min(x0 + (cell[k] & 255), D - 1);
            v[k] = Xi[((int64_t)(g * D + dz) * D + y) * D + x];
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int k = 0; k < kC4Items; k++)
            xl[k * 64 + lane] = v4bf{(__bf16)v[k][0], (__bf16)v[k][1], (__bf16)v[k][2], (__bf16)v[k][3]};
        __builtin_amdgcn_wave_barrier();
        const int gx = x0 + xs, gb = b0 + gi, ny = min(kC4Rows, P - y0);
        TOut* out = Y + ((((int64_t)gb * P + gz) * P + y0) * P + gx) * 32;
        const bool valid = gx < P && gb < B;
        for (int y = 0; y < ny; y++, out += (int64_t)P * 32) {
            v4f acc[2] = {v4f{0.f, 0.f, 0.f, 0.f}, v4f{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
            for (int s = 0; s < 4; s++) {
                v4bf e = xl[y * rc + off[s][0]], f = xl[y * rc + off[s][1]];
                // taps 27..31: their weights are zeros, an infinity times one is not
                if (s == 3 && kq > 1) e = v4bf{};
                if (s == 3 && kq > 0) f = v4bf{};
                const v8bf a = {e[0], e[1], e[2], e[3], f[0], f[1], f[2], f[3]};
#pragma unroll
                for (int ct = 0; ct < 2; ct++)
                    acc[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[s][ct], a, acc[ct], 0, 0, 0);
            }
            if (!valid) continue;
#pragma unroll
            for (int ct = 0; ct < 2; ct++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    acc[ct][i] += bs[ct][i];
                    if (relu) acc[ct][i] = fmaxf(acc[ct][i], 0.f);
                }
            store32(out, kq, acc[0], acc[1]);
        }
    }
}

// Wp[t][o][c] = BF16(W[t*cin + c][o]) for t < 27, o < cout, zero elsewhere
// ([taps_padded][coutp][cin]).
__global__ void k_conv_pack(const float* __restrict__ W, uint16_t* __restrict__ Wp, int cin,
                            int cout, int taps, int coutp) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= taps * coutp * cin) return;
    const int c = e % cin, o = (e / cin) % coutp, t = e / (cin * coutp);
    Wp[e] = (t < 27 && o < cout) ? to_bf16(W[(t * cin + c) * cout + o]) : (uint16_t)0;
}

// Cloud-in-cell combination of the 2^3 output cells of each sample with its
// fractions f (pred = sum over corners of prod_d (f_d or 1 - f_d) out), the
// mean squared error against target over n*3 values and its gradient with
// respect to the 2^3 outputs.  One block.
__global__ __launch_bounds__(256) void k_cic_mse(const float* __restrict__ out8,
                                                 const float* __restrict__ frac,
                                                 const float* __restrict__ target, int n,
                                                 float* __restrict__ pred,
                                                 float* __restrict__ dout8,
                                                 float* __restrict__ loss) {
    __shared__ float red[256];
    float s = 0.f;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const float f0 = frac[3 * i], f1 = frac[3 * i + 1], f2 = frac[3 * i + 2];
        float w[8];
#pragma unroll
        for (int c = 0; c < 8; c++)
            w[c] = ((c & 1) ? f0 : 1.f - f0) * ((c & 2) ? f1 : 1.f - f1) * ((c & 4) ? f2 : 1.f - f2);
#pragma unroll
        for (int d = 0; d < 3; d++) {
            float p = 0.f;
#pragma unroll
            for (int c = 0; c < 8; c++) p += w[c] * out8[(8 * i + c) * 3 + d];
            if (pred) pred[3 * i + d] = p;
            const float r = p - target[3 * i + d];
            s += r * r;
            const float g = 2.f * r / (3.f * (float)n);
#pragma unroll
            for (int c = 0; c < 8; c++) dout8[(8 * i + c) * 3 + d] = w[c] * g;
        }
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) *loss = red[0] / (3.f * (float)n);
}

static int cnn_check(bool ok, const char* what) {
    if (ok) return CUBE2_OK;
    set_error("cnn: bad arguments to %s", what);
    return CUBE2_ERR_ARG;
}

static unsigned blocks_for(int64_t n) { return (unsigned)((n + 255) / 256); }

// Split-K schedule of a product: S partial products over K ranges of kc
// (a multiple of 16); S = 1 for no split.  Few output tiles and a long K
// (the weight gradients, K = rows) are split over blocks, and the partials
// summed in a fixed order.  S * M * N <= 2^21 for every split shape (tiles
// >= M N / 4096 and S <= 512 / tiles).
static void gemm_split(int M, int N, int K, int* S_out, int* kc_out) {
    const int64_t tiles = (int64_t)((N + 63) / 64) * ((M + 63) / 64);
    int S = 1;
    if (tiles < 256 && K >= 4096) S = (int)std::min<int64_t>(std::min<int64_t>(512 / tiles, K / 2048), 64);
    int kc = K;
    if (S > 1) {
        kc = (int)(((K + S - 1) / S + 15) / 16 * 16);
        S = (K + kc - 1) / kc;
    }
    *S_out = S;
    *kc_out = kc;
}

// The product on stream s, split-K partials (S > 1) in part[S * M * N].
static int gemm_launch(const uint16_t* A, int64_t sam, int64_t sak, const uint16_t* B, int64_t sbk,
                       int64_t sbn, float* C, int64_t ldc, int M, int N, int K, int acc, int S,
                       int kc, float* part, hipStream_t s) {
    dim3 grid((unsigned)((N + 63) / 64), (unsigned)((M + 63) / 64));
    if (S <= 1) {
        k_gemm_bf16<<<grid, 256, 0, s>>>(A, sam, sak, B, sbk, sbn, C, ldc, M, N, K, acc, K, 0);
        C2_HIP(hipGetLastError());
        return CUBE2_OK;
    }
    grid.z = (unsigned)S;
    k_gemm_bf16<<<grid, 256, 0, s>>>(A, sam, sak, B, sbk, sbn, part, N, M, N, K, 0, kc,
                                     (int64_t)M * N);
    C2_HIP(hipGetLastError());
    k_sum_partials<<<blocks_for((int64_t)M * N), 256, 0, s>>>(part, C, ldc, M, N, S, acc);
    C2_HIP(hipGetLastError());
    return CUBE2_OK;
}

static DevBuf g_partials;  // split-K partials of cnn_gemm (released by the finalizer)

int cnn_gemm(const uint16_t* A, int64_t sam, int64_t sak, const uint16_t* B, int64_t sbk,
             int64_t sbn, float* C, int64_t ldc, int M, int N, int K, int acc) {
    C2_TRY(cnn_check(A && B && C && M >= 0 && N >= 0 && K >= 0 && ldc >= N, "gemm"));
    C2_TRY(ensure_init());
    if (M == 0 || N == 0) return CUBE2_OK;
    int S, kc;
    gemm_split(M, N, K, &S, &kc);
    if (S > 1) C2_TRY(g_partials.reserve((size_t)S * M * N * sizeof(float)));
    return gemm_launch(A, sam, sak, B, sbk, sbn, C, ldc, M, N, K, acc, S, kc, g_partials.as<float>(),
                       ctx().stream);
}

// ------------------------------------------------ allocation-free product
// cube2_gemm_bf16_noalloc_dev keeps its split-K partials in this file-scope
// device array (4 MiB; every GPU the library runs on holds its own copy
// until the process ends).  Host code never passes the array's name to a
// kernel: in host code it is a stand-in, not a device address.  The device
// address comes from hipGetSymbolAddress, once per device with that device
// current, and is kept per device.  Calls that overlap on one GPU share the
// array and race; the partials need no clearing (every call writes all
// S * M * N of them before they are summed).
constexpr size_t kScratchFloats = (size_t)1 << 20;
static __device__ __align__(256) float scratch[kScratchFloats];
constexpr int kMaxDevices = 64;
static float* g_scratch_ptr[kMaxDevices] = {};

static int scratch_address(float** out) {
    int dev = 0;
    C2_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) {
        set_error("device %d outside the scratch table", dev);
        return CUBE2_ERR_STATE;
    }
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        C2_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        g_scratch_ptr[dev] = static_cast<float*>(p);
    }
    *out = g_scratch_ptr[dev];
    return CUBE2_OK;
}

int cnn_gemm_noalloc(const uint16_t* A, int64_t sam, int64_t sak, const uint16_t* B, int64_t sbk,
                     int64_t sbn, float* C, int64_t ldc, int M, int N, int K, int acc) {
    C2_TRY(cnn_check(A && B && C && M >= 0 && N >= 0 && K >= 0 && ldc >= N, "gemm_noalloc"));
    C2_TRY(ensure_init());
    float* part = nullptr;
    C2_TRY(scratch_address(&part));
    if (M == 0 || N == 0) return CUBE2_OK;
    int S, kc;
    gemm_split(M, N, K, &S, &kc);
    if (S > 1 && (size_t)S * M * N > kScratchFloats) {
        set_error("gemm_noalloc: M=%d N=%d K=%d needs %zu bytes of split-K scratch; the static "
                  "scratch holds %zu", M, N, K, (size_t)S * M * N * sizeof(float),
                  kScratchFloats * sizeof(float));
        return CUBE2_ERR_CAPACITY;
    }
    return gemm_launch(A, sam, sak, B, sbk, sbn, C, ldc, M, N, K, acc, S, kc, part, ctx().stream);
}

void cnn_release() { g_partials.release(); }

// ---------------------------------------------------------- convolution
int cnn_conv_pack(const float* W, uint16_t* Wp, int cin, int cout, hipStream_t s) {
    C2_TRY(cnn_check(W && Wp && (cin == 4 || cin == 32) && (cout == 32 || (cout == 3 && cin == 32)),
                     "conv_pack"));
    const int taps = cin == 32 ? 27 : 32, coutp = cout == 3 ? 16 : 32;
    const int n = taps * coutp * cin;
    k_conv_pack<<<blocks_for(n), 256, 0, s>>>(W, Wp, cin, cout, taps, coutp);
    C2_HIP(hipGetLastError());
    return CUBE2_OK;
}

size_t cnn_conv_packed_count(int cin, int cout) {
    return (size_t)(cin == 32 ? 27 : 32) * (cout == 3 ? 16 : 32) * cin;
}

// Tile shape of a convolution over B grids of P^3 outputs: the x width with
// the fewest positions computed, counting padding in x and in the groups of
// 16 / tx grids (the wider one where equal), and as many z chunks as fill the
// given wavefronts evenly.  A chunk costs its planes and about one more (the
// halo planes' loads and the start of the pipeline).
static ConvTile conv_tile(int B, int P, int64_t waves) {
    ConvTile T{};
    int64_t best = -1;
    for (int tx : {16, 8, 4}) {
        const int g = 16 / tx;
        const int64_t n = (int64_t)((P + tx - 1) / tx) * ((B + g - 1) / g);
        // (offsets within a group of grids are 32-bit)
        const bool fits = g == 1 || (int64_t)g * (P + 2) * (P + 2) * (P + 2) * 32 < ((int64_t)1 << 31);
        if (best < 0 || (fits && n < best)) {
            best = n;
            T.tx = tx;
            T.nx = (P + tx - 1) / tx;
            T.nb = (B + g - 1) / g;
        }
    }
    T.ny = (P + kConvRows - 1) / kConvRows;
    const int64_t cols = (int64_t)T.nx * T.ny * T.nb;
    double cost = 0.0;
    for (int zc = P; zc >= 1; zc--) {
        const int nz = (P + zc - 1) / zc;
        const double c = (double)((cols * nz + waves - 1) / waves) * (zc + 1.0);
        if (T.nz == 0 || c < cost) {
            cost = c;
            T.nz = nz;
            T.zc = zc;
        }
    }
    return T;
}

static int device_cus() {
    int dev = 0, ncu = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        ncu = 256;
    return std::max(1, ncu);
}

template <int NT, class TIn, class TOut>
static int conv_launch(const void* X, const uint16_t* Wp, const float* bias, void* Y, int B, int D,
                       int cout, int relu, hipStream_t s) {
    auto kern = k_conv3<NT, TIn, TOut>;
    const size_t lds = conv_lds_bytes<NT>();
    static bool attr = false;  // (one value per instantiation)
    if (!attr) {
        C2_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)lds));
        attr = true;
    }
    const int ncu = device_cus();
    const ConvTile T = conv_tile(B, D - 2, (int64_t)ncu * kConvWaves);
    const int64_t items = (int64_t)T.nb * T.nx * T.ny * T.nz;
    const unsigned grid = (unsigned)std::min<int64_t>((items + kConvWaves - 1) / kConvWaves, ncu);
    kern<<<grid, kConvWaves * 64, lds, s>>>(static_cast<const TIn*>(X), Wp, bias,
                                            static_cast<TOut*>(Y), B, D, cout, relu, T);
    C2_HIP(hipGetLastError());
    return CUBE2_OK;
}

template <class TOut>
static int conv_c4_launch(const void* X, const uint16_t* Wp, const float* bias, void* Y, int B,
                          int D, int relu, hipStream_t s) {
    const int ncu = device_cus();
    const ConvTile T = conv_tile(B, D - 2, (int64_t)ncu * 16);
    const int64_t items = (int64_t)T.nb * T.nx * (D - 2) * ((D - 2 + kC4Rows - 1) / kC4Rows);
    const unsigned grid = (unsigned)std::min<int64_t>((items + 3) / 4, (int64_t)ncu * 16);
    k_conv3_c4<TOut><<<grid, 256, 0, s>>>(static_cast<const float*>(X), Wp, bias,
                                          static_cast<TOut*>(Y), B, D, relu, T);
    C2_HIP(hipGetLastError());
    return CUBE2_OK;
}

// x_bf16 / y_bf16: activations stored as BF16 (else FP32).
int cnn_conv3(const void* X, int x_bf16, const uint16_t* Wp, const float* bias, void* Y, int y_bf16,
              int B, int D, int cin, int cout, int relu, hipStream_t s) {
    C2_TRY(cnn_check(X && Wp && bias && Y && B >= 0 && D >= 3, "conv3"));
    if (B == 0) return CUBE2_OK;
    if (cin == 4 && cout == 32 && !x_bf16)
        return y_bf16 ? conv_c4_launch<uint16_t>(X, Wp, bias, Y, B, D, relu, s)
                      : conv_c4_launch<float>(X, Wp, bias, Y, B, D, relu, s);
    if (cin == 32 && cout == 32)
        return x_bf16 ? (y_bf16 ? conv_launch<2, uint16_t, uint16_t>(X, Wp, bias, Y, B, D, cout, relu, s)
                                : conv_launch<2, uint16_t, float>(X, Wp, bias, Y, B, D, cout, relu, s))
                      : (y_bf16 ? conv_launch<2, float, uint16_t>(X, Wp, bias, Y, B, D, cout, relu, s)
                                : conv_launch<2, float, float>(X, Wp, bias, Y, B, D, cout, relu, s));
    if (cin == 32 && cout == 3 && !y_bf16)
        return x_bf16 ? conv_launch<1, uint16_t, float>(X, Wp, bias, Y, B, D, cout, relu, s)
                      : conv_launch<1, float, float>(X, Wp, bias, Y, B, D, cout, relu, s);
    set_error("conv3: no kernel for %d -> %d channels (x %s, y %s)", cin, cout,
              x_bf16 ? "bf16" : "f32", y_bf16 ? "bf16" : "f32");
    return CUBE2_ERR_ARG;
}

int cnn_im2col(const float* X, uint16_t* col, int B, int D, int Cin) {
    C2_TRY(cnn_check(X && col && B >= 0 && D >= 3 && Cin >= 1, "im2col"));
    C2_TRY(ensure_init());
    const int64_t P = D - 2, tot = (int64_t)B * P * P * P * 27 * Cin;
    if (tot) k_im2col3<<<blocks_for(tot), 256, 0, ctx().stream>>>(X, col, B, D, Cin);
    C2_HIP(hipGetLastError());
    return CUBE2_OK;
}

int cnn_col2im(const float* dcol, float* dX, int B, int D, int Cin) {
    C2_TRY(cnn_check(dcol && dX && B >= 0 && D >= 3 && Cin >= 1, "col2im"));
    C2_TRY(ensure_init());
    const int64_t tot = (int64_t)B * D * D * D * Cin;
    if (tot) k_col2im3<<<blocks_for(tot), 256, 0, ctx().stream>>>(dcol, dX, B, D, Cin);
    C2_HIP(hipGetLastError());
    return CUBE2_OK;
}

int cnn_bias_act(float* Y, const float* bias, int64_t rows, int C, int relu) {
    C2_TRY(cnn_check(Y && bias && rows >= 0 && C >= 1, "bias_act"));
    C2_TRY(ensure_init());
    const int64_t n = rows * C;
    if (n) k_bias_act<<<blocks_for(n), 256, 0, ctx().stream>>>(Y, bias, n, C, relu);
    C2_HIP(hipGetLastError());
    return CUBE2_OK;
}

int cnn_act_bwd(const float* Y, float* dY, uint16_t* dYb, float* dbias, int64_t rows, int C,
                int relu) {
    C2_TRY(cnn_check(Y && dY && dYb && dbias && rows >= 0 && C >= 1, "act_bwd"));
    C2_TRY(ensure_init());
    const int64_t n = rows * C;
    hipStream_t s = ctx().stream;
    if (n) k_act_bwd<<<blocks_for(n), 256, 0, s>>>(Y, dY, dYb, n, relu);
    k_colsum<<<C, 256, 0, s>>>(dY, dbias, rows, C);
    C2_HIP(hipGetLastError());
    return CUBE2_OK;
}

int cnn_to_bf16(const float* x, uint16_t* y, int64_t n) {
    C2_TRY(cnn_check(x && y && n >= 0, "to_bf16"));
    C2_TRY(ensure_init());
    if (n) k_to_bf16<<<blocks_for(n), 256, 0, ctx().stream>>>(x, y, n);
    C2_HIP(hipGetLastError());
    return CUBE2_OK;
}

int cnn_adam(float* w, const float* g, float* m, float* v, uint16_t* wb, int64_t n, float lr,
             float b1, float b2, float eps, int t) {
    C2_TRY(cnn_check(w && g && m && v && n >= 0 && t >= 1, "adam"));
    C2_TRY(ensure_init());
    const float c1 = 1.f - powf(b1, (float)t), c2 = 1.f - powf(b2, (float)t);
    if (n) k_adam<<<blocks_for(n), 256, 0, ctx().stream>>>(w, g, m, v, wb, n, lr, b1, b2, eps, c1, c2);
    C2_HIP(hipGetLastError());
    return CUBE2_OK;
}

int cnn_cic_mse(const float* out8, const float* frac, const float* target, int n, float* pred,
                float* dout8, float* loss) {
    C2_TRY(cnn_check(out8 && frac && target && dout8 && loss && n >= 1, "cic_mse"));
    C2_TRY(ensure_init());
    k_cic_mse<<<1, 256, 0, ctx().stream>>>(out8, frac, target, n, pred, dout8, loss);
    C2_HIP(hipGetLastError());
    return CUBE2_OK;
}

int cnn_mse(const float* out, const float* target, float* dout, float* loss, int64_t n) {
    C2_TRY(cnn_check(out && target && dout && loss && n >= 1, "mse"));
    C2_TRY(ensure_init());
    k_mse<<<1, 256, 0, ctx().stream>>>(out, target, dout, loss, n);
    C2_HIP(hipGetLastError());
    return CUBE2_OK;
}

}  // namespace cube2
