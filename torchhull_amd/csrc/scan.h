// Device-wide exclusive prefix sums over 32-bit counts, written for 64-lane
// wavefronts: a tile of 256 threads x 16 items per block, wave prefix sums by
// lane shuffles, one LDS slot per wave, and a three-kernel reduce / scan /
// down-sweep that needs no inter-block waiting.
//
// Counts are read through a loader functor `L`, `uint32_t L::operator()(uint64_t i)`,
// so callers scan derived quantities (popcounts, table lookups) without a
// staging pass.
#pragma once

#include "common.h"
#include "kernels.h" // launch_fill_u32

namespace thull
{

constexpr int kScanThreads = 256;
constexpr int kScanItems = 16;
constexpr int kScanTile = kScanThreads * kScanItems;

// Inclusive prefix sum across the 64 lanes of a wavefront.
__device__ __forceinline__ uint32_t
wave_inclusive_sum(uint32_t v)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1)
    {
        uint32_t o = __shfl_up(v, d, 64);
        if (lane >= d)
            v += o;
    }
    return v;
}

// Exclusive prefix of v over the block (blockDim.x == kScanThreads); returns
// the block total in `total`.  `lds` holds kScanThreads / 64 entries.
__device__ __forceinline__ uint32_t
block_exclusive_sum(uint32_t v, uint32_t* lds, uint32_t& total)
{
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    uint32_t inc = wave_inclusive_sum(v);
    if (lane == 63)
        lds[wave] = inc;
    __syncthreads();
    uint32_t wave_off = 0;
    total = 0;
#pragma unroll
    for (int w = 0; w < kScanThreads / 64; ++w)
    {
        uint32_t s = lds[w];
        if (w < wave)
            wave_off += s;
        total += s;
    }
    __syncthreads();
    return wave_off + inc - v;
}

template <typename L>
__global__ __launch_bounds__(kScanThreads) void
scan_reduce_kernel(L load, uint64_t n, uint32_t* block_sums)
{
    __shared__ uint32_t lds[kScanThreads / 64];
    const uint64_t base = uint64_t(blockIdx.x) * kScanTile + uint64_t(threadIdx.x) * kScanItems;
    uint32_t s = 0;
    if (base + kScanItems <= n)
    {
        // full run of items: unconditional consecutive reads the compiler merges into wide loads
#pragma unroll
        for (int k = 0; k < kScanItems; ++k)
            s += load(base + k);
    }
    else
    {
#pragma unroll
        for (int k = 0; k < kScanItems; ++k)
        {
            uint64_t i = base + k;
            if (i < n)
                s += load(i);
        }
    }
    uint32_t total;
    block_exclusive_sum(s, lds, total);
    if (threadIdx.x == 0)
        block_sums[blockIdx.x] = total;
}

// Host notification of a scan's total: `slot` (3 words of coherent pinned
// host memory, device address) receives the total and a copy of *extra (0
// without it), then `seq` with a system-scope release store, so a host that
// sees seq in slot[2] reads the two words written before it.
struct ScanNotify
{
    unsigned long long* slot = nullptr;
    const unsigned long long* extra = nullptr;
    unsigned long long seq = 0;
};

// Clamp of a scan's total to a capacity: a larger total sets *overflow and is
// stored as `cap` (the prefixes themselves are not changed).
struct ScanGuard
{
    unsigned long long cap = ~0ull;
    uint32_t* overflow = nullptr;
};

// Group k of 4 sums with the entries past n as zeros.
__device__ __forceinline__ uint4
load_sums4(const uint4* v, uint32_t k, uint32_t n)
{
    uint4 u = v[k];
    u.y = 4 * k + 1 < n ? u.y : 0u;
    u.z = 4 * k + 2 < n ? u.z : 0u;
    u.w = 4 * k + 3 < n ? u.w : 0u;
    return u;
}

// Single-block exclusive scan of the block sums (16-byte aligned, room for nblocks rounded up to 4); writes the grand
// total (64-bit).  A thread takes a run of whole 16-byte groups (the three scans of a level-11 hull, the largest of
// 70 000 sums: 167 -> 39 us).
template <typename Tag = void>
__global__ __launch_bounds__(1024) void
scan_block_sums_kernel(uint32_t* sums, uint32_t nblocks, unsigned long long* total_out, ScanNotify note = {},
                       ScanGuard guard = {})
{
    __shared__ unsigned long long lds[1024 / 64];
    const uint32_t groups = (nblocks + 3) / 4, per = (groups + 1023) / 1024;
    const uint32_t begin = threadIdx.x * per, end = min(begin + per, groups);
    uint4* const v = reinterpret_cast<uint4*>(sums);
    unsigned long long local = 0;
#pragma unroll 4
    for (uint32_t k = begin; k < end; ++k)
    {
        const uint4 u = load_sums4(v, k, nblocks);
        local += (unsigned long long)u.x + u.y + u.z + u.w;
    }
    // block scan of 64-bit partial sums
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    unsigned long long inc = local;
    for (int d = 1; d < 64; d <<= 1)
    {
        unsigned long long o = __shfl_up(inc, d, 64);
        if (lane >= d)
            inc += o;
    }
    if (lane == 63)
        lds[wave] = inc;
    __syncthreads();
    unsigned long long off = 0, total = 0;
    for (int w = 0; w < 1024 / 64; ++w)
    {
        if (w < wave)
            off += lds[w];
        total += lds[w];
    }
    if (threadIdx.x == 0)
    {
        unsigned long long t = total;
        if (guard.overflow != nullptr && t > guard.cap)
        {
            *guard.overflow = 1u;
            t = guard.cap;
        }
        *total_out = t;
        if (note.slot != nullptr)
        {
            note.slot[0] = t;
            note.slot[1] = note.extra != nullptr ? *note.extra : 0ull;
            __hip_atomic_store(note.slot + 2, note.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
    unsigned long long run = off + inc - local;
#pragma unroll 4
    for (uint32_t k = begin; k < end; ++k)
    {
        const uint4 u = load_sums4(v, k, nblocks);
        v[k] = make_uint4(uint32_t(run), uint32_t(run + u.x), uint32_t(run + u.x + u.y),
                          uint32_t(run + u.x + u.y + u.z));
        run += (unsigned long long)u.x + u.y + u.z + u.w;
    }
}

// As scan_block_sums_kernel for two arrays of n sums at once (16-byte aligned, room for n rounded up to 4);
// the host is sent both totals (`note.extra` unused).  A thread takes a run of whole 16-byte groups.
template <typename Tag = void>
__global__ __launch_bounds__(1024) void
scan_block_sums2_kernel(uint32_t* a, uint32_t* b, uint32_t n, unsigned long long* totals, ScanNotify note)
{
    __shared__ unsigned long long lds[2][1024 / 64];
    const uint32_t groups = (n + 3) / 4, per = (groups + 1023) / 1024;
    const uint32_t begin = threadIdx.x * per, end = min(begin + per, groups);
    uint4* const v[2] = { reinterpret_cast<uint4*>(a), reinterpret_cast<uint4*>(b) };
    unsigned long long sum[2] = { 0, 0 };
    for (uint32_t k = begin; k < end; ++k)
#pragma unroll
        for (int q = 0; q < 2; ++q)
        {
            const uint4 u = load_sums4(v[q], k, n);
            sum[q] += (unsigned long long)u.x + u.y + u.z + u.w;
        }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    unsigned long long inc[2] = { sum[0], sum[1] };
    for (int d = 1; d < 64; d <<= 1)
#pragma unroll
        for (int q = 0; q < 2; ++q)
        {
            const unsigned long long o = __shfl_up(inc[q], d, 64);
            if (lane >= d)
                inc[q] += o;
        }
    if (lane == 63)
    {
        lds[0][wave] = inc[0];
        lds[1][wave] = inc[1];
    }
    __syncthreads();
    unsigned long long run[2], total[2] = { 0, 0 };
#pragma unroll
    for (int q = 0; q < 2; ++q)
    {
        unsigned long long off = 0;
        for (int w = 0; w < 1024 / 64; ++w)
        {
            if (w < wave)
                off += lds[q][w];
            total[q] += lds[q][w];
        }
        run[q] = off + inc[q] - sum[q];
    }
    if (threadIdx.x == 0)
    {
        totals[0] = total[0];
        totals[1] = total[1];
        note.slot[0] = total[0];
        note.slot[1] = total[1];
        __hip_atomic_store(note.slot + 2, note.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    for (uint32_t k = begin; k < end; ++k)
#pragma unroll
        for (int q = 0; q < 2; ++q)
        {
            const uint4 u = load_sums4(v[q], k, n);
            const unsigned long long r = run[q];
            v[q][k] = make_uint4(uint32_t(r), uint32_t(r + u.x), uint32_t(r + u.x + u.y),
                                 uint32_t(r + u.x + u.y + u.z));
            run[q] = r + u.x + u.y + u.z + u.w;
        }
}

template <typename L>
__global__ __launch_bounds__(kScanThreads) void
scan_downsweep_kernel(L load, uint64_t n, const uint32_t* block_offsets, uint32_t* out)
{
    __shared__ uint32_t lds[kScanThreads / 64];
    const uint64_t base = uint64_t(blockIdx.x) * kScanTile + uint64_t(threadIdx.x) * kScanItems;
    uint32_t v[kScanItems];
    uint32_t s = 0;
    const bool full = base + kScanItems <= n;
    if (full)
    {
#pragma unroll
        for (int k = 0; k < kScanItems; ++k)
        {
            v[k] = load(base + k);
            s += v[k];
        }
    }
    else
    {
#pragma unroll
        for (int k = 0; k < kScanItems; ++k)
        {
            uint64_t i = base + k;
            v[k] = (i < n) ? load(i) : 0u;
            s += v[k];
        }
    }
    uint32_t total;
    uint32_t run = block_offsets[blockIdx.x] + block_exclusive_sum(s, lds, total);
    if (full)
    {
#pragma unroll
        for (int k = 0; k < kScanItems; ++k)
        {
            out[base + k] = run;
            run += v[k];
        }
    }
    else
    {
#pragma unroll
        for (int k = 0; k < kScanItems; ++k)
        {
            uint64_t i = base + k;
            if (i < n)
                out[i] = run;
            run += v[k];
        }
    }
}

// Exclusive scan of up to kSmallScan values in one launch of one block: each
// thread holds a contiguous run of up to kSmallItems inputs in registers (all
// reads in flight together), the block scans the 64-bit run sums, and each
// thread writes its run's prefixes.  Writes the total like
// scan_block_sums_kernel, notification included.
constexpr int kSmallItems = 32;
constexpr uint64_t kSmallScan = 1024 * kSmallItems;

template <typename L>
__global__ __launch_bounds__(1024) void
scan_small_kernel(L load, uint32_t n, uint32_t* out, unsigned long long* total_out, ScanNotify note = {},
                  ScanGuard guard = {})
{
    __shared__ unsigned long long lds[1024 / 64];
    const uint32_t per = (n + 1023) / 1024; // <= kSmallItems
    const uint32_t begin = threadIdx.x * per;
    uint32_t v[kSmallItems];
#pragma unroll
    for (int k = 0; k < kSmallItems; ++k)
        v[k] = (uint32_t(k) < per && begin + k < n) ? load(begin + k) : 0u;
    unsigned long long local = 0;
#pragma unroll
    for (int k = 0; k < kSmallItems; ++k)
        local += v[k];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    unsigned long long inc = local;
    for (int d = 1; d < 64; d <<= 1)
    {
        unsigned long long o = __shfl_up(inc, d, 64);
        if (lane >= d)
            inc += o;
    }
    if (lane == 63)
        lds[wave] = inc;
    __syncthreads();
    unsigned long long off = 0, total = 0;
    for (int w = 0; w < 1024 / 64; ++w)
    {
        if (w < wave)
            off += lds[w];
        total += lds[w];
    }
    unsigned long long run = off + inc - local;
#pragma unroll
    for (int k = 0; k < kSmallItems; ++k)
    {
        if (uint32_t(k) < per && begin + k < n)
            out[begin + k] = uint32_t(run);
        run += v[k];
    }
    if (threadIdx.x == 0)
    {
        if (guard.overflow != nullptr && total > guard.cap)
        {
            *guard.overflow = 1u;
            total = guard.cap;
        }
        *total_out = total;
        if (note.slot != nullptr)
        {
            note.slot[0] = total;
            note.slot[1] = note.extra != nullptr ? *note.extra : 0ull;
            __hip_atomic_store(note.slot + 2, note.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
}

// Exclusive scan of load(i), i in [0, n), into out[0, n).  `block_sums` must
// hold scan_sums_room(n) entries, 16-byte aligned; the 64-bit total lands in *total_dev.
inline uint32_t
scan_blocks(uint64_t n)
{
    return uint32_t((n + kScanTile - 1) / kScanTile);
}

// Entries of an array of block sums: at least one group of 4, whole groups.
inline uint32_t
scan_sums_room(uint64_t n)
{
    return std::max((scan_blocks(n) + 3u) & ~3u, 4u);
}

// `note` (optional, n > 0) also sends the total to the host; `guard` (optional) clamps it.  Every
// step is a kernel, so that the scan can sit in a captured graph.
template <typename L>
void
exclusive_scan(L load, uint64_t n, uint32_t* out, uint32_t* block_sums, unsigned long long* total_dev, hipStream_t st,
               ScanNotify note = {}, ScanGuard guard = {})
{
    const uint32_t nb = scan_blocks(n);
    if (nb == 0)
    {
        THULL_CHECK(note.slot == nullptr, "scan notification of an empty scan");
        launch_fill_u32(reinterpret_cast<uint32_t*>(total_dev), 2, 0u, st);
        return;
    }
    if (n <= kSmallScan)
    {
        scan_small_kernel<<<1, 1024, 0, st>>>(load, uint32_t(n), out, total_dev, note, guard);
        THULL_LAUNCH_CHECK();
        return;
    }
    scan_reduce_kernel<<<nb, kScanThreads, 0, st>>>(load, n, block_sums);
    THULL_LAUNCH_CHECK();
    scan_block_sums_kernel<><<<1, 1024, 0, st>>>(block_sums, nb, total_dev, note, guard);
    THULL_LAUNCH_CHECK();
    scan_downsweep_kernel<<<nb, kScanThreads, 0, st>>>(load, n, block_sums, out);
    THULL_LAUNCH_CHECK();
}

struct LoadU32
{
    const uint32_t* p;
    __device__ uint32_t operator()(uint64_t i) const { return p[i]; }
};

} // namespace thull
