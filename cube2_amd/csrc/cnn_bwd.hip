// Backward pass and optimiser step of the learned stand-in's network on
// training patches (at most 10^3 inputs: 8^3, 6^3, 4^3 and 2^3 outputs of the
// four layers), with no im2col and one product kernel per gradient:
//   k_bwd_dw   dW[t][c][o] = sum over patches and positions of X[p + t][c]
//              dY[p][o], and the bias gradients;
//   k_bwd_dx   dX[p][c] = sum over taps of dY[p - t] W[t]^T;
//   k_bwd_sum  the workgroups' weight gradients summed, all layers at once;
//   k_net_adam one Adam step of every tensor, its BF16 copy and its packed
//              form for the convolution.
// dY passes a ReLU where it is read (dY if Y > 0).  BF16 operands, FP32
// accumulation, as in the im2col products (cnn.hip), which remain for larger
// grids: their operands do not fit LDS.  256 patches of 10^3: the four layers'
// backward takes 150 us in 8 launches (im2col, GEMMs, col2im and column sums
// 1480 us in 24), a training step with its host calls 431 us (2182).
#include <algorithm>

#include "adam.h"
#include "common.h"
#include "engine.h"

namespace cube2 {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef short v4s __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kBwdMaxD = 10;       // largest input side
constexpr int kDwThreads = 576;    // 9 wavefronts, one per (dz, dy)
constexpr int kDxThreads = 512;
constexpr int kDwGroups = 256;     // workgroups (partial gradients) of a layer: one per CU

// --- weight gradients.  The contraction runs over positions: a K step of 32
// is 4 rows (y) of 8 (x), rows and positions past the outputs zero.  LDS
// holds the patch transposed, channel-major, as 16-byte rows of 8 x: dY once,
// X three times, shifted by dx, so that the fragments of every tap are
// aligned 16-byte reads (the channels' strides are odd multiples of 16 bytes:
// the 16 rows a quarter wavefront reads lie in distinct banks).  Wavefront
// (dz, dy) keeps its three taps' products in registers over all its patches.
// Bound by the staging (a patch's loads and transpose); the products are a
// tenth of it.  One workgroup per CU: 128 of them with two patches each took
// 116 us for the four layers against 74, their sum 8 against 14.
template <int CIN, int COUT>
struct DwShape {
    static constexpr int kCT = CIN == 32 ? 2 : 1;   // row tiles per tap (CIN 4: one for the three)
    static constexpr int kAT = CIN == 32 ? 6 : 1;   // row tiles of a wavefront
    static constexpr int kOT = COUT == 32 ? 2 : 1;  // column tiles
    static constexpr int kN = 27 * CIN * COUT + COUT;
};
__host__ __device__ inline int dw_groups(int P) { return (P + 3) / 4; }       // row groups per plane
__host__ __device__ inline int dw_xrows(int P) {                              // rows of a channel of X
    return ((P + 2) * (4 * dw_groups(P) + 2)) | 1;
}
__host__ __device__ inline int dw_yrows(int P) { return (P * 4 * dw_groups(P)) | 1; }
template <int CIN, int COUT>
size_t dw_lds_bytes(int P) {
    return 16 * ((size_t)3 * CIN * dw_xrows(P) + (size_t)COUT * dw_yrows(P));
}

template <int CIN, int COUT>
__global__ __launch_bounds__(kDwThreads) void k_bwd_dw(const float* __restrict__ X,
                                                       const float* __restrict__ Y,
                                                       const float* __restrict__ dY, int B, int D,
                                                       int relu, float* __restrict__ part) {
    using S = DwShape<CIN, COUT>;
    extern __shared__ __align__(16) v8bf dw_lds[];
    __shared__ float red[kDwThreads];
    const int P = D - 2, G4 = dw_groups(P), YR = 4 * G4 + 2;
    const int RX = dw_xrows(P), RY = dw_yrows(P);
    v8bf* xt = dw_lds;                  // [dx][c][z][y]
    v8bf* yt = dw_lds + 3 * CIN * RX;   // [o][z][y]
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, r16 = lane & 15, kq = lane >> 4;
    const int dz = wave / 3, dy = wave % 3;
    v4f acc[S::kAT][S::kOT];
#pragma unroll
    for (int a = 0; a < S::kAT; a++)
#pragma unroll
        for (int o = 0; o < S::kOT; o++) acc[a][o] = v4f{0.f, 0.f, 0.f, 0.f};
    float bsum = 0.0f;
    for (int b = blockIdx.x; b < B; b += gridDim.x) {
        __syncthreads();  // the previous patch's reads are done
        {
            const int c = tid % CIN;
            for (int r = tid / CIN; r < D * YR; r += kDwThreads / CIN) {
                const int z = r / YR, y = r - z * YR;
                float v[kBwdMaxD];
                const float* src = X + ((((int64_t)b * D + z) * D + min(y, D - 1)) * D) * CIN + c;
#pragma unroll
                for (int x = 0; x < kBwdMaxD; x++) v[x] = x < D && y < D ? src[x * CIN] : 0.0f;
#pragma unroll
                for (int dx = 0; dx < 3; dx++) {
                    v8bf w;
#pragma unroll
                    for (int x = 0; x < 8; x++) w[x] = (__bf16)(x < P ? v[x + dx] : 0.0f);
                    xt[(dx * CIN + c) * RX + r] = w;
                }
            }
        }
        {
            const int o = tid % COUT;
            for (int r = tid / COUT; r < P * 4 * G4; r += kDwThreads / COUT) {
                const int z = r / (4 * G4), y = r - z * 4 * G4;
                const int64_t at = ((((int64_t)b * P + z) * P + min(y, P - 1)) * P) * COUT + o;
                v8bf w;
#pragma unroll
                for (int x = 0; x < 8; x++) {
                    float g = 0.0f;
                    if (x < P && y < P) {
                        g = dY[at + x * COUT];
                        if (relu && !(Y[at + x * COUT] > 0.f)) g = 0.0f;
                    }
                    bsum += g;
                    w[x] = (__bf16)g;
                }
                yt[o * RY + r] = w;
            }
        }
        __syncthreads();
        for (int z = 0; z < P; z++)
            for (int g = 0; g < G4; g++) {
                v8bf bm[S::kOT];
#pragma unroll
                for (int o = 0; o < S::kOT; o++)  // (COUT 3: the columns past it repeat, unused)
                    bm[o] = yt[min(o * 16 + r16, COUT - 1) * RY + (z * G4 + g) * 4 + kq];
                const int row = (z + dz) * YR + g * 4 + kq + dy;
#pragma unroll
                for (int a = 0; a < S::kAT; a++) {
                    // CIN 32: tap dx = a / 2, channels 16 (a % 2)..; CIN 4:
                    // row r16 = (dx, c), dx = 3 repeats 2, unused
                    const int ch = CIN == 32 ? (a >> 1) * CIN + (a & 1) * 16 + r16
                                             : min(r16 >> 2, 2) * CIN + (r16 & 3);
                    v8bf am = xt[ch * RX + row];
                    // (a row past the outputs: dY is zero, an infinite X times it is not)
                    if (g * 4 + 4 > P && g * 4 + kq >= P) am = v8bf{};
#pragma unroll
                    for (int o = 0; o < S::kOT; o++)
                        acc[a][o] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(am, bm[o], acc[a][o], 0, 0, 0);
                }
            }
    }
    float* out = part + (size_t)blockIdx.x * S::kN;
#pragma unroll
    for (int a = 0; a < S::kAT; a++)
#pragma unroll
        for (int o = 0; o < S::kOT; o++) {
            const int col = o * 16 + r16;
            if (col >= COUT) continue;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int row = 4 * kq + i;  // of the tile
                const int dx = CIN == 32 ? a >> 1 : row >> 2;
                const int c = CIN == 32 ? (a & 1) * 16 + row : row & 3;
                if (dx < 3) out[((wave * 3 + dx) * CIN + c) * COUT + col] = acc[a][o][i];
            }
        }
    red[tid] = bsum;
    __syncthreads();
    if (tid < COUT) {
        float s = 0.0f;
        for (int q = tid; q < kDwThreads; q += COUT) s += red[q];
        out[27 * CIN * COUT + tid] = s;
    }
}

// --- input gradients (32 input channels): a workgroup per patch.  LDS holds
// dY (BF16) with a border of two zero cells and the layer's weights; a
// wavefront takes four tiles of 16 positions and adds, tap by tap in the
// order 0..26, each tap's product (two 16x16x16 MFMAs) to its sum: the same
// products and the same additions as the im2col GEMM and its col2im, so the
// same bits (the next layer rounds them to BF16, where a last-bit change of
// a sum would flip roundings).  Rows of LDS are padded by 8 bytes (conflict-
// free 8-byte reads).  Bound by the dependent MFMA and add chain of a tap.
template <int COUT>
struct DxShape {
    static constexpr int KP = COUT == 32 ? 32 : 16, KH = KP / 16, ST = KP + 4;  // (BF16 elements)
};

// A tile of 16 positions, its lane's p, tap by tap within the outputs.
template <int COUT>
__device__ inline void dx_tile_bounded(const uint16_t* wl, const uint16_t* yl, int p, int kq, int D,
                                       float* __restrict__ dX) {
    using S = DxShape<COUT>;
    const int P = D - 2, E = P + 4, r16 = threadIdx.x & 15;
    const int pc = min(p, D * D * D - 1), z = pc / (D * D), y = pc / D % D, x = pc % D;
    v4f s[2] = {v4f{0.f, 0.f, 0.f, 0.f}, v4f{0.f, 0.f, 0.f, 0.f}};
#pragma unroll 1
    for (int t = 0; t < 27; t++) {
        const int oz = z - t / 9, oy = y - t / 3 % 3, ox = x - t % 3;
        const bool in = (unsigned)oz < (unsigned)P && (unsigned)oy < (unsigned)P && (unsigned)ox < (unsigned)P;
        const uint16_t* cell = yl + (((oz + 2) * E + oy + 2) * E + ox + 2) * S::ST + kq * 4;
#pragma unroll
        for (int ct = 0; ct < 2; ct++) {
            v4f d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int h = 0; h < S::KH; h++)
                d = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(
                    *reinterpret_cast<const v4s*>(wl + (t * 32 + ct * 16 + r16) * S::ST + h * 16 + kq * 4),
                    *reinterpret_cast<const v4s*>(cell + h * 16), d, 0, 0, 0);
            if (in) s[ct] += d;
        }
    }
    if (p >= D * D * D) return;
#pragma unroll
    for (int ct = 0; ct < 2; ct++) *reinterpret_cast<v4f*>(dX + (int64_t)p * 32 + 4 * kq + ct * 16) = s[ct];
}

template <int COUT>
__global__ __launch_bounds__(kDxThreads) void k_bwd_dx(const float* __restrict__ Y,
                                                       const float* __restrict__ dY,
                                                       const uint16_t* __restrict__ Wb, int B,
                                                       int D, int relu, float* __restrict__ dX) {
    constexpr int KP = DxShape<COUT>::KP, KH = DxShape<COUT>::KH, ST = DxShape<COUT>::ST;
    extern __shared__ __align__(16) uint16_t dx_lds[];
    uint16_t* wl = dx_lds;                // [27 * 32][ST]
    uint16_t* yl = dx_lds + 27 * 32 * ST;  // [(P + 4)^3][ST]
    const int P = D - 2, E = P + 4, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int r16 = lane & 15, kq = lane >> 4;
    for (int e = tid; e < 27 * 32 * KP; e += kDxThreads) {
        const int r = e / KP, o = e % KP;
        wl[r * ST + o] = o < COUT ? Wb[r * COUT + o] : (uint16_t)0;
    }
    for (int e = tid; e < E * E * E * ST / 2; e += kDxThreads) reinterpret_cast<uint32_t*>(yl)[e] = 0u;
    const int ntile = (D * D * D + 15) / 16;
    for (int b = blockIdx.x; b < B; b += gridDim.x) {
        __syncthreads();
        for (int e = tid; e < P * P * P * COUT; e += kDxThreads) {
            const int o = e % COUT, p = e / COUT;
            const int64_t at = (int64_t)b * P * P * P * COUT + e;
            float g = dY[at];
            if (relu && !(Y[at] > 0.f)) g = 0.0f;
            const int cell = ((p / (P * P) + 2) * E + p / P % P + 2) * E + p % P + 2;
            reinterpret_cast<__bf16*>(yl)[cell * ST + o] = (__bf16)g;
        }
        __syncthreads();
        for (int t0 = wave * 4; t0 < ntile; t0 += kDxThreads / 64 * 4) {
            int cell[4];
            v4f s[4][2];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int p = min((t0 + q) * 16 + r16, D * D * D - 1);
                cell[q] = (((p / (D * D) + 2) * E + p / D % D + 2) * E + p % D + 2) * ST + kq * 4;
                s[q][0] = s[q][1] = v4f{0.f, 0.f, 0.f, 0.f};
            }
            for (int zy = 0; zy < 9; zy++) {
#pragma unroll
                for (int dx = 0; dx < 3; dx++) {
                    const int t = zy * 3 + dx, back = ((zy / 3 * E + zy % 3) * E + dx) * ST;
                    v4s w[2][KH];
#pragma unroll
                    for (int ct = 0; ct < 2; ct++)
#pragma unroll
                        for (int h = 0; h < KH; h++)
                            w[ct][h] = *reinterpret_cast<const v4s*>(
                                wl + (t * 32 + ct * 16 + r16) * ST + h * 16 + kq * 4);
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        v4s y[KH];
#pragma unroll
                        for (int h = 0; h < KH; h++)
                            y[h] = *reinterpret_cast<const v4s*>(yl + cell[q] - back + h * 16);
#pragma unroll
                        for (int ct = 0; ct < 2; ct++) {
                            v4f d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                            for (int h = 0; h < KH; h++)
                                d = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(w[ct][h], y[h], d, 0, 0, 0);
                            s[q][ct] += d;
                        }
                    }
                }
            }
            // A zero of the border times an infinite weight is no zero: where a sum
            // is not finite, the tiles again with each tap only where it reaches an
            // output.
            float any = 0.0f;
#pragma unroll
            for (int q = 0; q < 4; q++)
#pragma unroll
                for (int k = 0; k < 8; k++) any += s[q][k >> 2][k & 3];
            if (__ballot(!(fabsf(any) < INFINITY))) {
#pragma unroll 1
                for (int q = 0; q < 4; q++)
                    dx_tile_bounded<COUT>(wl, yl, (t0 + q) * 16 + r16, kq, D, dX + (int64_t)b * D * D * D * 32);
                continue;
            }
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int p = (t0 + q) * 16 + r16;
                if (p >= D * D * D) continue;
                float* out = dX + ((int64_t)b * D * D * D + p) * 32 + 4 * kq;
#pragma unroll
                for (int ct = 0; ct < 2; ct++) *reinterpret_cast<v4f*>(out + ct * 16) = s[q][ct];
            }
        }
    }
}

struct SumArgs {
    const float* part[4];
    float* dW[4];
    float* db[4];
    int nW[4], n[4];
    int groups;
};
__global__ __launch_bounds__(256) void k_bwd_sum(SumArgs A) {
    int e = blockIdx.x * blockDim.x + threadIdx.x, l = 0;
    while (l < 4 && e >= A.n[l]) e -= A.n[l++];
    if (l == 4) return;
    const float* p = A.part[l] + e;
    float s = 0.0f;
#pragma unroll 8
    for (int g = 0; g < A.groups; g++) s += p[(size_t)g * A.n[l]];
    if (e < A.nW[l]) A.dW[l][e] = s;
    else A.db[l][e - A.nW[l]] = s;
}

struct AdamArgs {
    float* w[8];        // W of the four layers, then b
    const float* g[8];
    float* m[8];
    float* v[8];
    uint16_t* wb[4];
    uint16_t* wp[4];
    int n[8], cin[4], cout[4];
    float lr, b1, b2, eps, c1, c2;
};
__global__ __launch_bounds__(256) void k_net_adam(AdamArgs A) {
    int e = blockIdx.x * blockDim.x + threadIdx.x, l = 0;
    while (l < 8 && e >= A.n[l]) e -= A.n[l++];
    if (l == 8) return;
    float mi = A.m[l][e], vi = A.v[l][e];
    const float wi = adam_update(A.w[l][e], A.g[l][e], mi, vi, A.lr, A.b1, A.b2, A.eps, A.c1, A.c2);
    A.m[l][e] = mi;
    A.v[l][e] = vi;
    A.w[l][e] = wi;
    if (l < 4) {
        const __bf16 h = (__bf16)wi;
        const uint16_t bits = __builtin_bit_cast(uint16_t, h);
        A.wb[l][e] = bits;
        const int o = e % A.cout[l], r = e / A.cout[l], c = r % A.cin[l], t = r / A.cin[l];
        A.wp[l][(t * (A.cout[l] == 3 ? 16 : 32) + o) * A.cin[l] + c] = bits;
    }
}

// ------------------------------------------------------------------ host
static DevBuf g_part, g_dx[2];  // workspaces, grow-only (released by the finalizer)
void cnn_bwd_release() {
    g_part.release();
    g_dx[0].release();
    g_dx[1].release();
}

constexpr int kNetC[5] = {4, 32, 32, 32, 3};

template <int CIN, int COUT>
static int launch_dw(const float* X, const float* Y, const float* dY, int B, int D, int relu,
                     int groups, float* part, hipStream_t s) {
    const size_t lds = dw_lds_bytes<CIN, COUT>(D - 2);
    static bool attr = false;
    if (!attr) {
        C2_HIP(hipFuncSetAttribute((const void*)k_bwd_dw<CIN, COUT>,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, 156 * 1024));
        attr = true;
    }
    k_bwd_dw<CIN, COUT><<<groups, kDwThreads, lds, s>>>(X, Y, dY, B, D, relu, part);
    C2_HIP(hipGetLastError());
    return CUBE2_OK;
}

template <int COUT>
static int launch_dx(const float* Y, const float* dY, const uint16_t* Wb, int B, int D, int relu,
                     float* dX, hipStream_t s) {
    constexpr int st = (COUT == 32 ? 32 : 16) + 4;
    const int E = D + 2;
    const size_t lds = (size_t)2 * st * (27 * 32 + E * E * E);
    static bool attr = false;
    if (!attr) {
        C2_HIP(hipFuncSetAttribute((const void*)k_bwd_dx<COUT>,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, 156 * 1024));
        attr = true;
    }
    k_bwd_dx<COUT><<<std::min(B, 256), kDxThreads, lds, s>>>(Y, dY, Wb, B, D, relu, dX);
    C2_HIP(hipGetLastError());
    return CUBE2_OK;
}

// acts[0..4]: the input [B][D^3][4] and the layers' outputs, FP32; dout the
// gradient of acts[4].
int cnn_net_backward(const float* const* acts, const uint16_t* const* Wb, const float* dout, int B,
                     int D, float* const* dW, float* const* db, hipStream_t s) {
    const int groups = std::min(B, kDwGroups);
    SumArgs A;
    size_t off[4], tot = 0;
    int sum = 0;
    for (int l = 0; l < 4; l++) {
        A.nW[l] = 27 * kNetC[l] * kNetC[l + 1];
        A.n[l] = A.nW[l] + kNetC[l + 1];
        A.dW[l] = dW[l];
        A.db[l] = db[l];
        off[l] = tot;
        tot += (size_t)groups * A.n[l];
        sum += A.n[l];
    }
    A.groups = groups;
    C2_TRY(g_part.reserve(tot * sizeof(float)));
    for (int q = 0; q < 2; q++) {  // dX of layers 3 and 1 (the largest), of layer 2
        const int d = D - (q ? 4 : 2);
        C2_TRY(g_dx[q].reserve((size_t)B * d * d * d * 32 * sizeof(float)));
    }
    const float* g = dout;
    for (int l = 3; l >= 0; l--) {
        const int d = D - 2 * l;
        float* part = g_part.as<float>() + off[l];
        A.part[l] = part;
        if (l == 3) C2_TRY((launch_dw<32, 3>(acts[3], acts[4], g, B, d, 0, groups, part, s)));
        else if (l > 0) C2_TRY((launch_dw<32, 32>(acts[l], acts[l + 1], g, B, d, 1, groups, part, s)));
        else C2_TRY((launch_dw<4, 32>(acts[0], acts[1], g, B, d, 1, groups, part, s)));
        if (l > 0) {
            float* dx = g_dx[l & 1 ? 0 : 1].as<float>();
            if (l == 3) C2_TRY(launch_dx<3>(acts[4], g, Wb[3], B, d, 0, dx, s));
            else C2_TRY(launch_dx<32>(acts[l + 1], g, Wb[l], B, d, 1, dx, s));
            g = dx;
        }
    }
    k_bwd_sum<<<ceil_div(sum, 256), 256, 0, s>>>(A);
    C2_HIP(hipGetLastError());
    return CUBE2_OK;
}

bool cnn_net_backward_fits(int D) { return D >= 9 && D <= kBwdMaxD; }

int cnn_net_adam(float* const* w, const float* const* g, float* const* m, float* const* v,
                 uint16_t* const* wb, uint16_t* const* wp, float lr, float b1, float b2, float eps,
                 int t, hipStream_t s) {
    AdamArgs A;
    int sum = 0;
    for (int l = 0; l < 8; l++) {
        A.w[l] = w[l];
        A.g[l] = g[l];
        A.m[l] = m[l];
        A.v[l] = v[l];
        A.n[l] = l < 4 ? 27 * kNetC[l] * kNetC[l + 1] : kNetC[l - 3];
        sum += A.n[l];
        if (l < 4) {
            A.wb[l] = wb[l];
            A.wp[l] = wp[l];
            A.cin[l] = kNetC[l];
            A.cout[l] = kNetC[l + 1];
        }
    }
    A.lr = lr;
    A.b1 = b1;
    A.b2 = b2;
    A.eps = eps;
    A.c1 = 1.f - powf(b1, (float)t);
    A.c2 = 1.f - powf(b2, (float)t);
    k_net_adam<<<ceil_div(sum, 256), 256, 0, s>>>(A);
    C2_HIP(hipGetLastError());
    return CUBE2_OK;
}

}  // namespace cube2
