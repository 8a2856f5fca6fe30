// Device-wide exclusive prefix sum of int32 counts (cell lists), in 32 or 64
// bits.
#include <limits>

#include "common.h"
#include "scan.h"

namespace cube2 {

constexpr int kScanThreads = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kScanThreads * kScanItems;

template <class T>
__device__ inline T wave_inclusive_scan(T x) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        T y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    return x;
}

// Block-wide exclusive scan of one value per thread; returns the block total.
template <class T>
__device__ inline T block_exclusive_scan(T v, T* total) {
    __shared__ T wsum[kScanThreads / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    T inc = wave_inclusive_scan(v);
    if (lane == 63) wsum[wave] = inc;
    __syncthreads();
    T off = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < kScanThreads / 64; w++) {
        T s = wsum[w];
        if (w < wave) off += s;
        tot += s;
    }
    __syncthreads();
    *total = tot;
    return off + inc - v;
}

// lo: values below it count as lo (0 for counts from a caller, the type's lowest
// for none)
template <class S, class T>
__global__ __launch_bounds__(kScanThreads) void k_block_sums(const S* __restrict__ d, int64_t n,
                                                             S lo, T* __restrict__ sums) {
    int64_t base = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanItems;
    T s = 0;
#pragma unroll
    for (int q = 0; q < kScanItems; q++)
        if (base + q < n) s += max(d[base + q], lo);
    T tot;
    (void)block_exclusive_scan(s, &tot);
    if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}

// Exclusive scan of each tile of src into d (may be src), offset by
// offs[blockIdx.x] (nullptr: 0); writes the grand total to d[n] from the last
// block.
template <class S, class T>
__global__ __launch_bounds__(kScanThreads) void k_scan_tiles(const S* src, T* d, int64_t n, S lo,
                                                             const T* __restrict__ offs) {
    int64_t base = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanItems;
    T v[kScanItems];
    T s = 0;
#pragma unroll
    for (int q = 0; q < kScanItems; q++) {
        v[q] = base + q < n ? max(src[base + q], lo) : 0;
        s += v[q];
    }
    T tot;
    T excl = block_exclusive_scan(s, &tot);
    const T o = offs ? offs[blockIdx.x] : 0;
    T run = o + excl;
#pragma unroll
    for (int q = 0; q < kScanItems; q++) {
        if (base + q < n) d[base + q] = run;
        run += v[q];
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == kScanThreads - 1) d[n] = o + tot;
}

// The whole scan by one block, for counts that fill only a few tiles: one launch
// of about 6 us instead of three of 3 to 4 us each and the gaps between them
// (a kick of 3600 particles has two such scans).
constexpr int64_t kScanOneMax = 32768;
template <class S, class T>
__global__ __launch_bounds__(1024) void k_scan_one(const S* src, T* d, int n, S lo) {
    __shared__ T wsum[1024 / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    T carry = 0;
    for (int b = 0; b < n; b += 1024 * kScanItems) {
        const int base = b + (int)threadIdx.x * kScanItems;
        T v[kScanItems], s = 0;
#pragma unroll
        for (int q = 0; q < kScanItems; q++) {
            v[q] = base + q < n ? max(src[base + q], lo) : 0;
            s += v[q];
        }
        const T inc = wave_inclusive_scan(s);
        if (lane == 63) wsum[wave] = inc;
        __syncthreads();
        T run = carry + inc - s;
#pragma unroll
        for (int w = 0; w < 1024 / 64; w++) {
            run += w < wave ? wsum[w] : 0;
            carry += wsum[w];
        }
#pragma unroll
        for (int q = 0; q < kScanItems; q++) {
            if (base + q < n) d[base + q] = run;
            run += v[q];
        }
        __syncthreads();  // wsum is rewritten
    }
    if (threadIdx.x == 0) d[n] = carry;
}

template <class S, class T>
static int scan_rec(const S* src, T* d, int64_t n, S lo, T* tmp, hipStream_t s) {
    const int64_t nb = (n + kScanTile - 1) / kScanTile;
    if (nb <= 1) {
        k_scan_tiles<S, T><<<1, kScanThreads, 0, s>>>(src, d, n, lo, nullptr);
        C2_HIP(hipGetLastError());
        return CUBE2_OK;
    }
    if (n <= kScanOneMax) {
        k_scan_one<S, T><<<1, 1024, 0, s>>>(src, d, (int)n, lo);
        C2_HIP(hipGetLastError());
        return CUBE2_OK;
    }
    T* sums = tmp;
    k_block_sums<S, T><<<(unsigned)nb, kScanThreads, 0, s>>>(src, n, lo, sums);
    C2_HIP(hipGetLastError());
    C2_TRY((scan_rec<T, T>(sums, sums, nb, std::numeric_limits<T>::lowest(), tmp + nb + 1, s)));
    k_scan_tiles<S, T><<<(unsigned)nb, kScanThreads, 0, s>>>(src, d, n, lo, sums);
    C2_HIP(hipGetLastError());
    return CUBE2_OK;
}

size_t scan_tmp_ints(int64_t n) {
    size_t t = 0;
    int64_t m = n;
    while (m > kScanTile) {
        m = (m + kScanTile - 1) / kScanTile;
        t += (size_t)m + 1;
    }
    return t + 16;
}

__global__ void k_fill_zero(uint32_t* __restrict__ d, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) d[i] = 0u;
}

// Zeroes bytes (a multiple of 4) with a kernel: recordable into HIP graphs,
// where memset nodes are avoided.
int fill_zero(void* d, size_t bytes, hipStream_t s) {
    const size_t n = bytes / 4;
    if (!n) return CUBE2_OK;
    k_fill_zero<<<ceil_div(n, 256), 256, 0, s>>>(static_cast<uint32_t*>(d), n);
    C2_HIP(hipGetLastError());
    return CUBE2_OK;
}

int exclusive_scan(int* d, int64_t n, DevBuf& tmp, hipStream_t s) {
    if (n <= 0) return fill_zero(d, sizeof(int), s);
    C2_TRY(tmp.reserve(scan_tmp_ints(n) * sizeof(int)));
    return scan_rec<int, int>(d, d, n, std::numeric_limits<int>::lowest(), tmp.as<int>(), s);
}

int exclusive_scan_counts(const int* counts, long long* d, int64_t n, DevBuf& tmp, hipStream_t s) {
    if (n <= 0) return fill_zero(d, sizeof(long long), s);
    C2_TRY(tmp.reserve(scan_tmp_ints(n) * sizeof(long long)));
    return scan_rec<int, long long>(counts, d, n, 0, tmp.as<long long>(), s);
}

}  // namespace cube2
