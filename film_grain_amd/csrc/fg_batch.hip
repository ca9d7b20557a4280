// fg_batch.hip -- device helpers of the batched persistent renderer.
//
// Everything here is a plain kernel (no library calls, no memsets), so the
// whole batch pipeline can be captured in a HIP graph and replayed: the bin
// scan, the work of each (plane, tile) item, the heaviest-first item order,
// counter fills and the grain-capacity check.
#include <algorithm>

#include "fg_device.h"
#include "fg_pixelwise_hbm.h"
#include "fg_region.h"

namespace fg {

constexpr int kScanItems = 4;                       // elements per thread
constexpr int kScanTile = kBlock * kScanItems;      // elements per workgroup

size_t scan_partials(long long n) { return (size_t)((n + kScanTile - 1) / kScanTile) + 1; }

// Workgroup sums of kScanTile-element tiles.
__global__ __launch_bounds__(kBlock) void scan_tile_sums(const uint32_t *in, long long n, uint32_t *partials)
{
    __shared__ uint32_t s_wave[kBlock / 64];
    const long long base = (long long)blockIdx.x * kScanTile + (long long)threadIdx.x * kScanItems;
    uint32_t v = 0;
    for (int i = 0; i < kScanItems; ++i)
        if (base + i < n) v += in[base + i];
    uint32_t total;
    (void)block_exclusive_scan(v, s_wave, total);
    if (threadIdx.x == 0) partials[blockIdx.x] = total;
}

// Exclusive scan of the tile sums in place (one workgroup, any count).
__global__ __launch_bounds__(kBlock) void scan_tile_prefix(uint32_t *partials, long long m)
{
    __shared__ uint32_t s_wave[kBlock / 64];
    __shared__ uint32_t s_carry;
    if (threadIdx.x == 0) s_carry = 0;
    __syncthreads();
    for (long long b = 0; b < m; b += kBlock) {
        const long long i = b + threadIdx.x;
        const uint32_t v = i < m ? partials[i] : 0u;
        uint32_t total;
        const uint32_t ex = block_exclusive_scan(v, s_wave, total);
        const uint32_t carry = s_carry;
        if (i < m) partials[i] = carry + ex;
        __syncthreads();
        if (threadIdx.x == 0) s_carry = carry + total;
        __syncthreads();
    }
    if (threadIdx.x == 0) partials[m] = s_carry;
}

// out[i] = tile prefix + exclusive prefix within the tile; out[n] = total.
__global__ __launch_bounds__(kBlock) void scan_tile_apply(const uint32_t *in, uint32_t *out, long long n,
                                                          const uint32_t *partials, long long m)
{
    __shared__ uint32_t s_wave[kBlock / 64];
    const long long base = (long long)blockIdx.x * kScanTile + (long long)threadIdx.x * kScanItems;
    uint32_t v[kScanItems], sum = 0;
    for (int i = 0; i < kScanItems; ++i) {
        v[i] = base + i < n ? in[base + i] : 0u;
        sum += v[i];
    }
    uint32_t total;
    uint32_t run = partials[blockIdx.x] + block_exclusive_scan(sum, s_wave, total);
    for (int i = 0; i < kScanItems; ++i) {
        if (base + i < n) out[base + i] = run;
        run += v[i];
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) out[n] = partials[m];
}

hipError_t launch_scan_u32(const uint32_t *in, uint32_t *out, long long n, uint32_t *partials, hipStream_t s)
{
    const long long m = (n + kScanTile - 1) / kScanTile;
    if (m > 0) {
        hipLaunchKernelGGL(scan_tile_sums, dim3((unsigned)m), dim3(kBlock), 0, s, in, n, partials);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(scan_tile_prefix, dim3(1), dim3(kBlock), 0, s, partials, m);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(scan_tile_apply, dim3((unsigned)std::max<long long>(m, 1)), dim3(kBlock), 0, s, in, out, n,
                       partials, m);
    return hipGetLastError();
}

// ---- the bins of a plane, or of a frame's planes, in one set of launches ----
// As above with 64-bit sums (a plane's total may reach 2^32: the host refuses
// it then), the starts truncated to 32 bits, and each plane's total published
// to the host.  A workgroup takes kBinScanTile bins; up to kBinScanSmall bins
// one workgroup a plane does everything.
constexpr int kBinScanThreads = 1024;
constexpr int kBinScanItems = 4;
constexpr int kBinScanTile = kBinScanThreads * kBinScanItems;
constexpr long long kBinScanSmall = 4 * kBinScanTile;

size_t bin_scan_partials(long long n) { return (size_t)((n + kBinScanTile - 1) / kBinScanTile) + 1; }

// Exclusive prefix of v over the workgroup, and its total, in 64 bits (values
// below 2^26 by the 32-bit wave sum).
__device__ __forceinline__ unsigned long long bin_scan_prefix(unsigned long long v, unsigned long long *s_wave,
                                                              unsigned long long &total)
{
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    unsigned long long x = v;
    if (__ballot(v >= (1ull << 26)) == 0ull) {
        x = wave_inclusive_sum((uint32_t)v);
    } else {
        for (int o = 1; o < 64; o <<= 1) {
            const unsigned long long y = __shfl_up(x, o, 64);
            if (lane >= o) x += y;
        }
    }
    if (lane == 63) s_wave[wid] = x;
    __syncthreads();
    unsigned long long before = 0;
    total = 0;
    for (int w = 0; w < kBinScanThreads / 64; ++w) {
        const unsigned long long t = s_wave[w];
        before += w < wid ? t : 0ull;
        total += t;
    }
    __syncthreads();
    return before + x - v;
}

// A plane's total to the host (one thread), then its flag.
__device__ __forceinline__ void publish_total(HostPublish *pub, uint32_t seq, int plane, unsigned long long total)
{
    __hip_atomic_store(&pub->total[plane], total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(&pub->total_seq[plane], seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

__device__ __forceinline__ unsigned long long bin_scan_load(const uint32_t *in, long long base, long long n,
                                                            uint32_t v[kBinScanItems])
{
    unsigned long long sum = 0;
    for (int i = 0; i < kBinScanItems; ++i) {
        v[i] = base + i < n ? in[base + i] : 0u;
        sum += v[i];
    }
    return sum;
}

__global__ __launch_bounds__(kBinScanThreads) void bin_scan_sums_kernel(BinScan b)
{
    __shared__ unsigned long long s_wave[kBinScanThreads / 64];
    const int p = blockIdx.y;
    uint32_t v[kBinScanItems];
    unsigned long long total;
    const long long base = (long long)blockIdx.x * kBinScanTile + (long long)threadIdx.x * kBinScanItems;
    (void)bin_scan_prefix(bin_scan_load(b.in[p], base, b.n, v), s_wave, total);
    if (threadIdx.x == 0) b.partials[p][blockIdx.x] = total;
}

__global__ __launch_bounds__(kBinScanThreads) void bin_scan_prefix_kernel(BinScan b, long long m)
{
    __shared__ unsigned long long s_wave[kBinScanThreads / 64];
    const int p = blockIdx.x;
    unsigned long long carry = 0;
    for (long long i0 = 0; i0 < m; i0 += kBinScanThreads) {
        const long long i = i0 + threadIdx.x;
        const unsigned long long v = i < m ? b.partials[p][i] : 0ull;
        unsigned long long total;
        const unsigned long long ex = bin_scan_prefix(v, s_wave, total);
        if (i < m) b.partials[p][i] = carry + ex;
        carry += total;
    }
    if (threadIdx.x == 0) {
        b.out[p][b.n] = (uint32_t)carry;
        publish_total(b.pub, b.seq, p, carry);
    }
}

__global__ __launch_bounds__(kBinScanThreads) void bin_scan_apply_kernel(BinScan b)
{
    __shared__ unsigned long long s_wave[kBinScanThreads / 64];
    const int p = blockIdx.y;
    uint32_t v[kBinScanItems];
    unsigned long long total;
    const long long base = (long long)blockIdx.x * kBinScanTile + (long long)threadIdx.x * kBinScanItems;
    uint32_t run = (uint32_t)(b.partials[p][blockIdx.x] +
                              bin_scan_prefix(bin_scan_load(b.in[p], base, b.n, v), s_wave, total));
    for (int i = 0; i < kBinScanItems; ++i) {
        if (base + i < b.n) b.out[p][base + i] = run;
        run += v[i];
    }
}

__global__ __launch_bounds__(kBinScanThreads) void bin_scan_small_kernel(BinScan b)
{
    __shared__ unsigned long long s_wave[kBinScanThreads / 64];
    const int p = blockIdx.x;
    unsigned long long carry = 0;
    for (long long i0 = 0; i0 < b.n; i0 += kBinScanTile) {
        uint32_t v[kBinScanItems];
        unsigned long long total;
        const long long base = i0 + (long long)threadIdx.x * kBinScanItems;
        uint32_t run = (uint32_t)(carry + bin_scan_prefix(bin_scan_load(b.in[p], base, b.n, v), s_wave, total));
        for (int i = 0; i < kBinScanItems; ++i) {
            if (base + i < b.n) b.out[p][base + i] = run;
            run += v[i];
        }
        carry += total;
    }
    if (threadIdx.x == 0) {
        b.out[p][b.n] = (uint32_t)carry;
        publish_total(b.pub, b.seq, p, carry);
    }
}

hipError_t launch_bin_scan(const BinScan &b, hipStream_t s)
{
    if (b.planes < 1 || b.planes > kFramePlanes || b.n < 1) return hipErrorInvalidValue;
    if (b.n <= kBinScanSmall) {
        hipLaunchKernelGGL(bin_scan_small_kernel, dim3((unsigned)b.planes), dim3(kBinScanThreads), 0, s, b);
        return hipGetLastError();
    }
    const long long m = (b.n + kBinScanTile - 1) / kBinScanTile;
    hipLaunchKernelGGL(bin_scan_sums_kernel, dim3((unsigned)m, (unsigned)b.planes), dim3(kBinScanThreads), 0, s, b);
    hipLaunchKernelGGL(bin_scan_prefix_kernel, dim3((unsigned)b.planes), dim3(kBinScanThreads), 0, s, b, m);
    hipLaunchKernelGGL(bin_scan_apply_kernel, dim3((unsigned)m, (unsigned)b.planes), dim3(kBinScanThreads), 0, s, b);
    return hipGetLastError();
}

__global__ __launch_bounds__(kBlock) void fill_u32_kernel(uint32_t *p, long long n, uint32_t v)
{
    for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n; i += (long long)gridDim.x * kBlock)
        p[i] = v;
}

hipError_t launch_fill_u32(uint32_t *p, long long n, uint32_t v, hipStream_t s)
{
    const long long blocks = std::max<long long>(1, std::min<long long>((n + kBlock - 1) / kBlock, 4096));
    hipLaunchKernelGGL(fill_u32_kernel, dim3((unsigned)blocks), dim3(kBlock), 0, s, p, n, v);
    return hipGetLastError();
}

// The plane of batch item `item` (planes sorted by item_base).
__device__ __forceinline__ int plane_of(const BatchPlane *planes, int n_planes, long long item)
{
    int lo = 0, hi = n_planes - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (planes[mid].item_base <= item)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

__global__ __launch_bounds__(kBlock) void batch_weights_kernel(const BatchPlane *planes, int n_planes, uint32_t *w,
                                                               int n_items)
{
    const int item = blockIdx.x * kBlock + threadIdx.x;
    if (item >= n_items) return;
    const int pl = plane_of(planes, n_planes, item);
    w[item] = tile_weight(planes[pl].a, planes[pl].geo, planes[pl].bin_start, (int)(item - planes[pl].item_base));
}

hipError_t launch_batch_weights(const BatchPlane *planes, int n_planes, uint32_t *w, int n_items, hipStream_t s)
{
    if (n_items <= 0) return hipSuccess;
    hipLaunchKernelGGL(batch_weights_kernel, dim3((unsigned)((n_items + kBlock - 1) / kBlock)), dim3(kBlock), 0, s,
                       planes, n_planes, w, n_items);
    return hipGetLastError();
}

// Counting sort of the items by bucket floor(log2(w + 1)), heaviest bucket
// first (one workgroup; the order inside a bucket is whatever the atomics
// give, which changes no result, only the schedule).
__device__ __forceinline__ int weight_bucket(uint32_t w)
{
    return 32 - __clz(w == 0xFFFFFFFFu ? w : w + 1u);  // 1..32
}

__global__ __launch_bounds__(1024) void batch_order_kernel(const BatchPlane *planes, int n_planes, const uint32_t *w,
                                                           int n_items, int2 *items)
{
    __shared__ uint32_t s_count[64], s_pos[64];
    if (threadIdx.x < 64) s_count[threadIdx.x] = 0;
    __syncthreads();
    for (int i = threadIdx.x; i < n_items; i += 1024) atomicAdd(&s_count[weight_bucket(w[i])], 1u);
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t run = 0;
        for (int b = 63; b >= 0; --b) {
            s_pos[b] = run;
            run += s_count[b];
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < n_items; i += 1024) {
        const uint32_t pos = atomicAdd(&s_pos[weight_bucket(w[i])], 1u);
        const int pl = plane_of(planes, n_planes, i);
        items[pos] = make_int2(pl, (int)(i - planes[pl].item_base));
    }
}

hipError_t launch_batch_order(const BatchPlane *planes, int n_planes, const uint32_t *w, int n_items, int2 *items,
                              uint32_t *scratch, hipStream_t s)
{
    (void)scratch;
    if (n_items <= 0) return hipSuccess;
    hipLaunchKernelGGL(batch_order_kernel, dim3(1), dim3(1024), 0, s, planes, n_planes, w, n_items, items);
    return hipGetLastError();
}

// Heaviest-first order of one plane's tiles in one workgroup: a counting sort
// by sixteenth octaves of the weight.  Up to kOrderFused tiles compute their
// weights here as well (w null): 5 to 8 us.  More have too many scattered
// reads for one workgroup (4080 tiles: 63 us) and take a launch of their own
// (10 us and 6 here).  A radix sort takes two to five launches, 13 to 28 us;
// beyond kOrderTiles it is the shorter.
__global__ __launch_bounds__(1024) void tile_order_kernel(PixelArgs a, PixGeom geo, const uint32_t *bin_start,
                                                          const uint32_t *w, int n, int *order)
{
    constexpr int kPer = kOrderTiles / 1024, kBuckets = 512, kBucketsLane = kBuckets / 64;
    __shared__ uint32_t s_count[kBuckets], s_pos[kBuckets];
    if (threadIdx.x < kBuckets) s_count[threadIdx.x] = 0;
    __syncthreads();
    uint32_t bucket[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int tile = j * 1024 + (int)threadIdx.x;
        bucket[j] = 0;
        if (tile >= n) continue;
        const uint32_t v = w ? w[tile] : tile_weight(a, geo, bin_start, tile);
        // 16 log2(v + 1) by the float's exponent and four mantissa bits
        bucket[j] = min(kBuckets - 1u, (__float_as_uint((float)v + 1.0f) >> 19) - (127u << 4));
        atomicAdd(&s_count[bucket[j]], 1u);
    }
    __syncthreads();
    if (threadIdx.x < 64) {  // first position of each bucket, heaviest first
        const int b = kBuckets - 1 - kBucketsLane * (int)threadIdx.x;
        uint32_t sum = 0;
        for (int j = 0; j < kBucketsLane; ++j) sum += s_count[b - j];
        uint32_t pos = wave_inclusive_sum(sum) - sum;
        for (int j = 0; j < kBucketsLane; ++j) {
            s_pos[b - j] = pos;
            pos += s_count[b - j];
        }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int tile = j * 1024 + (int)threadIdx.x;
        if (tile < n) order[atomicAdd(&s_pos[bucket[j]], 1u)] = tile;
    }
}

hipError_t launch_tile_order(const PixelArgs &a, const PixGeom &g, const uint32_t *bin_start, int *order, hipStream_t s)
{
    if (a.n_tiles > kOrderFused) return hipErrorInvalidValue;
    hipLaunchKernelGGL(tile_order_kernel, dim3(1), dim3(1024), 0, s, a, g, bin_start, nullptr, a.n_tiles, order);
    return hipGetLastError();
}

hipError_t launch_weight_order(const uint32_t *w, int n, int *order, hipStream_t s)
{
    if (n > kOrderTiles) return hipErrorInvalidValue;
    hipLaunchKernelGGL(tile_order_kernel, dim3(1), dim3(1024), 0, s, PixelArgs{}, PixGeom{}, nullptr, w, n, order);
    return hipGetLastError();
}

// *out += the sum of n u32 values in 64 bits (one atomic per workgroup).
__global__ __launch_bounds__(kBlock) void sum_u64_kernel(const uint32_t *in, long long n, unsigned long long *out)
{
    __shared__ unsigned long long s_part[kBlock / 64];
    unsigned long long acc = 0;
    for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n; i += (long long)gridDim.x * kBlock)
        acc += in[i];
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
    if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long t = 0;
        for (int w = 0; w < kBlock / 64; ++w) t += s_part[w];
        if (t) atomicAdd(out, t);
    }
}

hipError_t launch_sum_u64(const uint32_t *in, long long n, unsigned long long *out, hipStream_t s)
{
    const long long blocks = std::max<long long>(1, std::min<long long>((n + kBlock - 1) / kBlock, 512));
    hipLaunchKernelGGL(sum_u64_kernel, dim3((unsigned)blocks), dim3(kBlock), 0, s, in, n, out);
    return hipGetLastError();
}

__global__ void capacity_check_kernel(const unsigned long long *total, uint32_t cap, int *status)
{
    if (*total > cap) atomicOr(status, kStatusCapacity);
}

hipError_t launch_capacity_check(const unsigned long long *total, uint32_t cap, int *status, hipStream_t s)
{
    hipLaunchKernelGGL(capacity_check_kernel, dim3(1), dim3(1), 0, s, total, cap, status);
    return hipGetLastError();
}

}  // namespace fg
