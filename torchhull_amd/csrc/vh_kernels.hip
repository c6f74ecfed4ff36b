// Visual-hull kernels for CDNA4 (gfx950): integral image, level-synchronous
// octree carving with stable compaction, corner-vertex bitmap and the field.
//
// Reference behaviour (vc-bonn/torchhull, src/torchhull/_C/src/visual_hull_cuda.cu,
// abbreviated VH): integral image VH:76-90, classification VH:168-417, level
// loop and compaction VH:627-751, corner dedup VH:770-825, field VH:419-520
// and VH:827-888.

#include <algorithm>
#include <cfloat>
#include <type_traits>
#include <vector>

#include <hip/hip_fp16.h>

#include "kernels.h"
#include "scan.h"
#include "solid_reach.h"

namespace thull
{

// ===========================================================================
// Mask element access
// ===========================================================================

template <typename T>
__device__ __forceinline__ float
as_float(T v)
{
    return static_cast<float>(v);
}

template <>
__device__ __forceinline__ float
as_float<__half>(__half v)
{
    return __half2float(v);
}

// ===========================================================================
// Integral image (VH:76-90)
//
// torch::cumsum on CUDA scans every non-innermost dimension with
// tensor_kernel_scan_outer_dim (ATen/native/cuda/ScanUtils.cuh): one
// sequential float chain per line, acc = acc + x from acc = 0.  Both passes of
// the reference are of that kind on [B,H,W,1], so the integral image is
// reproduced exactly by a sequential column chain per column followed by a
// sequential row chain per row.
//
// Two kernels compute it with one read of the output's worth of writes:
//  * the carry pass runs every column chain from the top and stores its value
//    only at the last row of each strip of kStripRows rows (1/32 of the data);
//  * the strip pass gives one workgroup a strip of kStripRows rows and the
//    full width: it resumes each column chain from the stored carry (the same
//    sequence of additions, hence the same bits), puts the column sums of a
//    kChunk-column chunk into LDS, runs the strip's row chains across the
//    chunk (one lane per row), and writes the chunk out coalesced.  The next
//    chunk's mask reads are in flight during the row chains.
// Batches of many images take a single pass instead: one workgroup walks the
// strips of one image from the top and stores each strip's column-chain
// values itself, so the masks are read once (the carry pass reads them a
// second time); the two-pass form keeps a small batch's strips spread over
// the whole GPU.
// ===========================================================================

constexpr int kStripRows = 32;
constexpr int kChunk = 256;

// One integral-image job: B cameras of one mask tensor.  Blocks of every job
// are flattened into one launch per pass; `*_begin` is the job's first block.
struct IntegralJob
{
    const void* masks;    // [B,H,W]
    float* out;           // element (b, y, x) at out + b * plane + y * ld + x; in a tiled job out is the
                          // padded plane base and the element sits at padded row y + kIntegralRow0,
                          // column x + kIntegralCol0 of plane b (common.h)
    float* carry;         // B * (strips - 1) * W column-chain values at strip ends
    int64_t plane;
    int32_t ld;
    int32_t dtype;
    int32_t B, H, W;
    int32_t strips;       // ceil(H / kStripRows)
    int32_t tiled;        // the padded, tiled layout of carving (common.h)
    uint32_t col_blocks;  // carry-pass blocks per camera
    uint64_t col_begin;   // first block of this job in the carry pass
    uint64_t strip_begin; // first block of this job in the strip pass (one block per camera and strip)
    uint64_t cam_begin;   // first block of this job in the border pass (one block per camera)
    uint16_t* solid_bits; // null, or one bit per solid tile: B * tile_rows rows of tile_pitch 16-tile words
    uint8_t* odd;         // 2 bytes per camera: a negative value or NaN was seen, a fraction was seen
    int32_t tile_rows;    // H / kSolidTile
    int32_t tile_pitch;   // ceil(W / 64)
};
static_assert(sizeof(IntegralJob) <= kIntegralJobBytes, "callers with a fixed job area reserve kIntegralJobBytes");

__device__ __forceinline__ int32_t
find_job(const IntegralJob* jobs, int32_t n, uint64_t blk, int pass)
{
    if (pass == 0)
        return find_segment_uniform([&](int32_t i) { return jobs[i].col_begin; }, n, blk);
    if (pass == 1)
        return find_segment_uniform([&](int32_t i) { return jobs[i].strip_begin; }, n, blk);
    return find_segment_uniform([&](int32_t i) { return jobs[i].cam_begin; }, n, blk);
}

// Column chains down to the last strip boundary; `src` and `carry` point at
// the thread's column.
template <typename T>
__device__ __forceinline__ void
carry_column(gptr<const T> src, gptr<float> carry, int32_t strips, int32_t W)
{
    float acc = 0.0f;
    for (int32_t s = 0; s + 1 < strips; ++s)
    {
        float v[kStripRows];
#pragma unroll
        for (int k = 0; k < kStripRows; ++k)
            v[k] = as_float(src[int64_t(s * kStripRows + k) * W]);
#pragma unroll
        for (int k = 0; k < kStripRows; ++k)
            acc = acc + v[k];
        carry[int64_t(s) * W] = acc;
    }
}

__global__ __launch_bounds__(256) void
integral_carry_kernel(const IntegralJob* __restrict__ jobs, int32_t njobs)
{
    const uint64_t blk = blockIdx.x;
    const IntegralJob j = jobs[find_job(jobs, njobs, blk, 0)];
    const uint64_t local = blk - j.col_begin;
    const int32_t b = int32_t(local / j.col_blocks);
    const int32_t t = int32_t(local - uint64_t(b) * j.col_blocks) * 256 + threadIdx.x;
    const int32_t x = t; // one column per thread: many waves walk their columns at once
    if (x >= j.W)
        return;
    const int64_t in_off = int64_t(b) * j.H * j.W + x;
    const auto carry = as_global(j.carry + int64_t(b) * (j.strips - 1) * j.W + x);
    if (j.dtype == kF32)
        carry_column(as_global(static_cast<const float*>(j.masks) + in_off), carry, j.strips, j.W);
    else
        carry_column(as_global(static_cast<const uint8_t*>(j.masks) + in_off), carry, j.strips, j.W);
}

// A mask value as the loads leave it in a register: converted only where the column chain adds it, since a
// conversion beside its load waits for that load, and the 32 loads of a chunk then go one after the other
// (strips of 10 8-bit 1080p masks: 107 us instead of 49).
template <typename T>
using RawMask = std::conditional_t<std::is_same_v<T, float>, float, uint32_t>;

// Mask values of strip s, chunk c0 for this thread's column (rows and columns past the image read its last
// ones, which are never stored) and the column chain's value above the strip (carry slot s - 1).
template <typename T>
__device__ __forceinline__ void
integral_load_chunk(const IntegralJob& j, int32_t b, int32_t s, int32_t c0, RawMask<T> (&pre)[kStripRows], float& cin)
{
    const int32_t H = j.H, W = j.W;
    const int32_t r0 = s * kStripRows;
    const int32_t x = min(c0 + int32_t(threadIdx.x), W - 1);
    // the row step is hidden from the compiler, which otherwise keeps the 32 row offsets of all chunks in
    // (spilled) scalar registers
    int32_t step = W;
    asm volatile("" : "+s"(step));
    auto row = as_global(static_cast<const T*>(j.masks) + (int64_t(b) * H + r0) * W);
#pragma unroll
    for (int r = 0; r < kStripRows; ++r)
    {
        pre[r] = RawMask<T>(row[x]);
        row += r0 + r + 1 < H ? step : 0;
    }
    cin = s > 0 ? j.carry[(int64_t(b) * (j.strips - 1) + (s - 1)) * W + x] : 0.0f;
}

// Solid tiles and odd values of a chunk, from the values of the thread's column: four rows of a column give
// one ballot bit, four columns one tile, 16 tiles of a wavefront one word per tile row.  Columns past the
// image are not solid, and only whole tile rows are stored.
template <typename T>
__device__ __forceinline__ void
solid_chunk(const IntegralJob& j, int32_t b, int32_t s, int32_t c0, const RawMask<T> (&pre)[kStripRows])
{
    static_assert(kSolidTile == 4 && kStripRows == 32, "8 tile rows of 4 pixels per strip");
    const int lane = threadIdx.x & 63;
    uint32_t word = 0u;
    bool neg = false, frac = false;
    const bool in = c0 + int32_t(threadIdx.x) < j.W;
#pragma unroll
    for (int g = 0; g < kStripRows / 4; ++g)
    {
        bool one = in;
#pragma unroll
        for (int r = 4 * g; r < 4 * g + 4; ++r)
        {
            one = one && pre[r] == RawMask<T>(1);
            if constexpr (std::is_same_v<T, float>)
            {
                neg = neg || !(pre[r] >= 0.0f);
                frac = frac || pre[r] != truncf(pre[r]);
            }
        }
        uint64_t m = __ballot(one);
        m &= m >> 1;
        m &= m >> 2;
        const uint32_t tiles = uint32_t(__ballot(lane < 16 && ((m >> (4 * (lane & 15))) & 1u) != 0u));
        word = lane == g ? tiles : word;
    }
    const int32_t tr = s * (kStripRows / 4) + lane;
    const int32_t tw = (c0 >> 6) + int32_t(threadIdx.x >> 6);
    if (lane < kStripRows / 4 && tr < j.tile_rows && tw < j.tile_pitch)
        as_global(j.solid_bits)[(int64_t(b) * j.tile_rows + tr) * j.tile_pitch + tw] = uint16_t(word);
    if constexpr (std::is_same_v<T, float>)
    {
        // every writer stores the same value: plain byte stores
        if (__any(neg) && lane == 0)
            j.odd[2 * b] = 1;
        if (__any(frac) && lane == 0)
            j.odd[2 * b + 1] = 1;
    }
}

// One strip; pre / cin hold its chunk 0 (integral_load_chunk) on entry.  CHAIN: the strip also
// stores its column-chain values at its last row (carry slot s), which the same thread reads back
// for the next strip, and its last chunk is followed by the reads of the next strip's chunk 0.
template <typename T, bool CHAIN>
__device__ __forceinline__ void
integral_strip(const IntegralJob& j, int32_t b, int32_t s, float (&tile)[kStripRows][kChunk + 1],
               RawMask<T> (&pre)[kStripRows], float& cin)
{
    const int32_t t = threadIdx.x;
    const int32_t H = j.H, W = j.W, ld = j.ld;
    const int32_t r0 = s * kStripRows;
    const int32_t rows = min(kStripRows, H - r0);
    const auto dst = as_global(j.out + b * j.plane + (j.tiled ? 0 : int64_t(r0) * ld));
    static_assert(kStripRows % 4 == 0 && kChunk == 256 && kIntegralRow0 % 4 == 0 && kIntegralCol0 % 8 == 0,
                  "strips and chunks start at tile boundaries of the tiled layout");
    const auto carry = as_global(j.carry + (int64_t(b) * (j.strips - 1) + s) * W);
    float racc = 0.0f; // row chain of row t (t < rows)
    for (int32_t c0 = 0; c0 < W; c0 += kChunk)
    {
        // column chains resumed from the carry: acc = acc + x, as in the carry pass
        float acc = cin;
#pragma unroll
        for (int r = 0; r < kStripRows; ++r)
        {
            acc = acc + float(pre[r]);
            tile[r][t] = acc;
        }
        if (CHAIN && s + 1 < j.strips && c0 + t < W)
            carry[c0 + t] = acc; // slot s (rows == kStripRows below the last strip)
        if (j.solid_bits != nullptr)
            solid_chunk<T>(j, b, s, c0, pre);
        __syncthreads();
        if (c0 + kChunk < W)
            integral_load_chunk<T>(j, b, s, c0 + kChunk, pre, cin);
        else if (CHAIN && s + 1 < j.strips)
            integral_load_chunk<T>(j, b, s + 1, 0, pre, cin); // carry slot s of chunk 0: stored above
        if (t < rows)
        {
            const int32_t cols = min(kChunk, W - c0);
            int32_t c = 0;
            // the next 8 values are read while the chain runs through the current 8
            float v[8];
            if (cols >= 8)
            {
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    v[k] = tile[t][k];
            }
            for (; c + 8 <= cols; c += 8)
            {
                float nv[8];
                const bool more = c + 16 <= cols;
                if (more)
                {
#pragma unroll
                    for (int k = 0; k < 8; ++k)
                        nv[k] = tile[t][c + 8 + k];
                }
#pragma unroll
                for (int k = 0; k < 8; ++k)
                {
                    racc = racc + v[k];
                    tile[t][c + k] = racc;
                }
                if (more)
                {
#pragma unroll
                    for (int k = 0; k < 8; ++k)
                        v[k] = nv[k];
                }
            }
            for (; c < cols; ++c)
            {
                racc = racc + tile[t][c];
                tile[t][c] = racc;
            }
        }
        __syncthreads();
        if (j.tiled)
        {
            // whole 128-byte lines with 16-byte stores: line (tr, tc) of the chunk holds rows r0 + 4 tr ..
            // r0 + 4 tr + 3 and columns c0 + 8 tc .. c0 + 8 tc + 7 (tile row (r0 + kIntegralRow0) / 4 + tr,
            // tile column (c0 + kIntegralCol0) / 8 + tc); 8 lanes fill a line, a wavefront 8 consecutive
            // lines.  Lines with no row or column of the image are skipped; the others carry the values of
            // entries past row H - 1 or column W - 1, which are never read, and end inside the plane.
            const uint64_t row4 = uint64_t(4 * ld);
#pragma unroll 2 // fully unrolled the chain kernel takes 177 VGPRs (2 waves per SIMD), like this 142 (3)
            for (int i = 0; i < kStripRows * kChunk / (4 * 256); ++i)
            {
                const int q = t + 256 * i;
                const int tr = q >> 8, tc = (q >> 3) & 31, ry = (q >> 1) & 3, h = q & 1;
                if (tr * 4 < rows && c0 + tc * 8 < W)
                {
                    const float* v = &tile[tr * 4 + ry][tc * 8 + h * 4];
                    const uint64_t off = uint64_t((r0 + kIntegralRow0) / 4 + tr) * row4 +
                                         uint64_t((c0 + kIntegralCol0) / 8 + tc) * 32u + uint64_t(ry * 8 + h * 4);
                    *(gptr<float4_v>)(dst + off) = float4_v{ v[0], v[1], v[2], v[3] }; // 16-byte aligned
                }
            }
        }
        else if (c0 + t < W)
        {
#pragma unroll
            for (int r = 0; r < kStripRows; ++r)
                if (r < rows)
                    dst[int64_t(r) * ld + c0 + t] = tile[r][t];
        }
        __syncthreads();
    }
}

__global__ __launch_bounds__(256) void
integral_strip_kernel(const IntegralJob* __restrict__ jobs, int32_t njobs)
{
    __shared__ float tile[kStripRows][kChunk + 1];
    const uint64_t blk = blockIdx.x;
    const IntegralJob j = jobs[find_job(jobs, njobs, blk, 1)];
    const uint64_t local = blk - j.strip_begin;
    const int32_t b = int32_t(local / uint32_t(j.strips));
    const int32_t s = int32_t(local - uint64_t(b) * uint32_t(j.strips));
    float cin;
    if (j.dtype == kF32)
    {
        float pre[kStripRows];
        integral_load_chunk<float>(j, b, s, 0, pre, cin);
        integral_strip<float, false>(j, b, s, tile, pre, cin);
    }
    else
    {
        uint32_t pre[kStripRows];
        integral_load_chunk<uint8_t>(j, b, s, 0, pre, cin);
        integral_strip<uint8_t, false>(j, b, s, tile, pre, cin);
    }
}

// Single pass for batches of many images: one workgroup per image, strips from the top.
__global__ __launch_bounds__(256) void
integral_chain_kernel(const IntegralJob* __restrict__ jobs, int32_t njobs)
{
    __shared__ float tile[kStripRows][kChunk + 1];
    const uint64_t blk = blockIdx.x;
    const IntegralJob j = jobs[find_job(jobs, njobs, blk, 2)];
    const int32_t b = int32_t(blk - j.cam_begin);
    float cin;
    if (j.dtype == kF32)
    {
        float pre[kStripRows];
        integral_load_chunk<float>(j, b, 0, 0, pre, cin);
        for (int32_t s = 0; s < j.strips; ++s)
            integral_strip<float, true>(j, b, s, tile, pre, cin);
    }
    else
    {
        uint32_t pre[kStripRows];
        integral_load_chunk<uint8_t>(j, b, 0, 0, pre, cin);
        for (int32_t s = 0; s < j.strips; ++s)
            integral_strip<uint8_t, true>(j, b, s, tile, pre, cin);
    }
}

// Zero row and zero column of the padded layout used by carving (one block per camera).
__global__ __launch_bounds__(256) void
integral_border_kernel(const IntegralJob* __restrict__ jobs, int32_t njobs)
{
    const uint64_t blk = blockIdx.x;
    const IntegralJob j = jobs[find_job(jobs, njobs, blk, 2)];
    const int32_t b = int32_t(blk - j.cam_begin);
    // tiled padded plane (common.h): row kIntegralRow0 - 1 from column kIntegralCol0 - 1 on, and column
    // kIntegralCol0 - 1 from row kIntegralRow0 - 1 on
    const auto p = as_global(j.out + b * j.plane);
    const uint32_t ld = uint32_t(j.ld), c = integral_col_offset(uint32_t(kIntegralCol0 - 1));
    const uint32_t r = integral_row_offset(uint32_t(kIntegralRow0 - 1), ld);
    for (int32_t q = threadIdx.x; q <= max(j.H, j.W); q += 256)
    {
        if (q <= j.W)
            p[r + integral_col_offset(uint32_t(kIntegralCol0 - 1 + q))] = 0.0f;
        if (q <= j.H)
            p[integral_row_offset(uint32_t(kIntegralRow0 - 1 + q), ld) + c] = 0.0f;
    }
    if (j.solid_bits != nullptr && threadIdx.x < 2)
        j.odd[2 * b + int32_t(threadIdx.x)] = 0;
}

// ===========================================================================
// Solid maps (common.h)
//
// A camera whose mask is 1 wherever a cell and its descendants project can neither empty nor refine them, and
// most cameras are such for most surface cells: a cell on the hull's surface lies on the outline of a few
// silhouettes and inside the others.  The maps let carving skip those cameras (carve_skips) from one byte read
// instead of 27 projections and 32 integral reads.
//
// The integral passes leave one bit per tile; this pass turns the bits into distances.  A workgroup takes 64 x
// kSolidRows tiles of one camera: horizontal distances of its rows and kSolidReach rows around them go to LDS
// (bit scans of a 32-tile window of the rows' words), with their minima over windows of 2, 4, 8 and 16 rows, from
// which each tile finds the largest square that fits in four steps.  Bound by the latency of short workgroups: 31 us
// for 64 images of 1024^2.
// ===========================================================================

constexpr int kSolidRows = 32;

struct SolidJob
{
    const uint16_t* bits;
    const uint8_t* odd;
    uint8_t* map;
    CullCamera* cull;
    int32_t* culls;
    const float* integral; // tiled planes
    const float* transforms;
    int64_t plane;
    int32_t ld, B, H, W, tile_rows, tile_cols, tile_pitch, opengl, u8;
    float corner[3], length;
    uint32_t bx, by;       // workgroups per camera
    uint64_t begin;        // first workgroup of this job
};

// A window reaches at least 1.75 pixels (skip_probe): below this carving can skip no camera, and the tests are left
// out (blurred 2048^2 masks have no reach; a level-10 hull of 32 partial ones 3.75 -> 3.68 ms).
constexpr float kLeastReach = 2.0f;

__global__ __launch_bounds__(256) void
solid_map_kernel(const SolidJob* __restrict__ jobs, int32_t njobs)
{
    constexpr int kHalo = kSolidReach, kLdsRows = kSolidRows + 2 * kHalo;
    constexpr int kSteps = 4; // window minima over 1, 2, 4, 8 and 16 rows
    static_assert(kSolidReach == (1 << kSteps) - 1, "distances found bit by bit");
    __shared__ uint8_t h[kSteps + 1][kLdsRows][64];
    __shared__ uint16_t words[kLdsRows][8];
    const SolidJob j = jobs[find_segment_uniform([&](int32_t i) { return jobs[i].begin; }, njobs, blockIdx.x)];
    const uint32_t local = uint32_t(blockIdx.x - j.begin), per = j.bx * j.by;
    const int32_t b = int32_t(local / per);
    const uint32_t r = local - uint32_t(b) * per;
    const int32_t by = int32_t(r / j.bx), bx = int32_t(r - uint32_t(by) * j.bx);
    const int32_t lane = int32_t(threadIdx.x & 63), wave = int32_t(threadIdx.x >> 6);
    const int32_t x = bx * 64 + lane, y0 = by * kSolidRows;
    const auto bits = as_global(j.bits + int64_t(b) * j.tile_rows * j.tile_pitch);
    if (r == 0u && wave == 3)
    {
        // the camera's record, while the other wavefronts read their tiles: its values come in one round of loads,
        // a transform coefficient per lane
        const float t = as_global(j.transforms)[16 * b + (lane & 15)];
        const int32_t odd = as_global(j.odd)[2 * b + (lane & 1)];
        const uint32_t corner = integral_row_offset(uint32_t(j.H - 1 + kIntegralRow0), uint32_t(j.ld)) +
                                integral_col_offset(uint32_t(j.W - 1 + kIntegralCol0));
        const float total = as_global(j.integral)[int64_t(b) * j.plane + corner];
        const int32_t d0 = j.opengl != 0 ? 12 : 8;
        float m[3];
#pragma unroll
        for (int a = 0; a < 3; ++a)
            m[a] = fmaxf(fabsf(j.corner[a]), fabsf(j.corner[a] + j.length));
        const auto at = [&](int32_t k) { return fabsf(__shfl(t, k, 64)); };
        const auto bound = [&](int32_t k) {
            return ((at(k) * m[0] + at(k + 1) * m[1]) + (at(k + 2) * m[2] + at(k + 3))) * 0x1p-20f;
        };
        CullCamera c{};
        const bool f32 = j.u8 == 0;
        c.reach = solid_reach(f32 && __shfl(odd, 0, 64) != 0, f32 && __shfl(odd, 1, 64) != 0, total, j.H, j.W);
        c.sum_d = at(d0) + at(d0 + 1) + at(d0 + 2);
        c.ex = bound(0);
        c.ey = bound(4);
        c.ed = bound(d0);
        if (lane == 0)
        {
            j.cull[b] = c;
            if (c.reach >= kLeastReach)
                *j.culls = 1; // every writer stores the same value
        }
    }
    // words of the rows: tiles bx * 64 - 16 .. bx * 64 + 95
    for (int32_t q = int32_t(threadIdx.x); q < kLdsRows * 8; q += 256)
    {
        const int32_t y = y0 - kHalo + (q >> 3), w = 4 * bx - 1 + (q & 7);
        const bool in = y >= 0 && y < j.tile_rows && w >= 0 && w < j.tile_pitch;
        words[q >> 3][q & 7] = in ? bits[int64_t(y) * j.tile_pitch + w] : uint16_t(0);
    }
    __syncthreads();
    for (int32_t k = wave; k < kLdsRows; k += 4)
    {
        const uint16_t* row = &words[k][lane >> 4]; // the word before the tile's
        const uint64_t w = uint64_t(row[0]) | (uint64_t(row[1]) << 16) | (uint64_t(row[2]) << 32);
        const uint32_t gaps = ~uint32_t(w >> (x & 15)); // bit 16: tile x, bit 0: tile x - 16
        const int32_t right = (gaps >> 16) != 0u ? __builtin_ctz(gaps >> 16) : 16;
        const int32_t left = (gaps << 15) != 0u ? __builtin_clz(gaps << 15) : 17;
        h[0][k][lane] = uint8_t(min(min(left, right), kSolidReach));
    }
    __syncthreads();
    for (int p = 1; p <= kSteps; ++p)
    {
        for (int32_t k = wave; k + (1 << p) <= kLdsRows; k += 4)
            h[p][k][lane] = min(h[p - 1][k][lane], h[p - 1][k + (1 << (p - 1))][lane]);
        __syncthreads();
    }
#pragma unroll 4
    for (int32_t k = wave; k < kSolidRows; k += 4)
    {
        const int32_t y = y0 + k;
        if (x >= j.tile_cols || y >= j.tile_rows)
            continue;
        // the largest d for which the rows within d - 1 are all at least d wide, found from its highest bit
        int32_t d = 0;
        const int32_t c = k + kHalo;
#pragma unroll
        for (int q = kSteps - 1; q >= 0; --q)
        {
            const int32_t t = d + (1 << q), p = 31 - __builtin_clz(2 * t - 1); // window of 2 t - 1 rows
            const int32_t wide = min(h[p][c - (t - 1)][lane], h[p][c + t - (1 << p)][lane]);
            d = wide >= t ? t : d;
        }
        as_global(j.map)[(int64_t(b) * j.tile_rows + y) * j.tile_cols + x] = uint8_t(d);
    }
}

static IntegralJob
make_job(const void* masks, int32_t dtype, int64_t B, int64_t H, int64_t W, float* out, int64_t plane, int64_t ld,
         bool tiled = false)
{
    IntegralJob j{};
    j.tiled = tiled ? 1 : 0;
    j.masks = masks;
    j.out = out;
    j.plane = plane;
    j.ld = int32_t(ld);
    j.dtype = dtype;
    j.B = int32_t(B);
    j.H = int32_t(H);
    j.W = int32_t(W);
    j.strips = int32_t((H + kStripRows - 1) / kStripRows);
    return j;
}

uint64_t
integral_carry_floats(int64_t B, int64_t H, int64_t W)
{
    return uint64_t(B) * uint64_t((H + kStripRows - 1) / kStripRows - 1 > 0 ? (H + kStripRows - 1) / kStripRows - 1
                                                                               : 0) *
           uint64_t(W);
}

size_t
integral_job_bytes(size_t njobs)
{
    return njobs * sizeof(IntegralJob);
}

// Images from which a batch takes the single-pass form (one workgroup per image keeps every CU busy).
constexpr uint64_t kIntegralChainImages = 1024;

static void
integral_jobs_impl(IntegralJob* jobs, size_t njobs, IntegralJob* djobs, float* carry, bool border, Uploader& up,
                   hipStream_t st)
{
    uint64_t images = 0;
    for (size_t i = 0; i < njobs; ++i)
        images += uint64_t(jobs[i].B);
    const bool chain = images >= kIntegralChainImages;
    if (chain && njobs > 1) // largest images first: the longest walks start first
        std::stable_sort(jobs, jobs + njobs, [](const IntegralJob& a, const IntegralJob& b) {
            return int64_t(a.H) * a.W > int64_t(b.H) * b.W;
        });
    uint64_t cols = 0, strips = 0, cams = 0, coff = 0;
    for (size_t i = 0; i < njobs; ++i)
    {
        IntegralJob& j = jobs[i];
        j.col_blocks = blocks_for(j.W, 256);
        j.col_begin = cols;
        j.strip_begin = strips;
        j.cam_begin = cams;
        j.carry = carry + coff;
        coff += integral_carry_floats(j.B, j.H, j.W);
        if (j.strips > 1)
            cols += uint64_t(j.col_blocks) * j.B;
        strips += uint64_t(j.strips) * j.B;
        cams += uint64_t(j.B);
    }
    if (strips == 0)
        return;
    THULL_CHECK(cols < (uint64_t(1) << 31) && strips < (uint64_t(1) << 31), "integral image batch too large");
    up.upload(djobs, jobs, njobs * sizeof(IntegralJob), st);
    const int32_t n = int32_t(njobs);
    if (border)
    {
        integral_border_kernel<<<unsigned(cams), 256, 0, st>>>(djobs, n);
        THULL_LAUNCH_CHECK();
    }
    if (chain)
    {
        integral_chain_kernel<<<unsigned(cams), 256, 0, st>>>(djobs, n);
        THULL_LAUNCH_CHECK();
        return;
    }
    if (cols > 0)
    {
        // jobs of a single strip have no carry-pass blocks and are never found by it
        integral_carry_kernel<<<unsigned(cols), 256, 0, st>>>(djobs, n);
        THULL_LAUNCH_CHECK();
    }
    integral_strip_kernel<<<unsigned(strips), 256, 0, st>>>(djobs, n);
    THULL_LAUNCH_CHECK();
}

void
launch_integral_image(const void* masks, int32_t dtype, int64_t B, int64_t H, int64_t W, float* out, float* carry,
                      void* job_buf, Uploader& up, hipStream_t st)
{
    if (B == 0 || H == 0 || W == 0)
        return;
    THULL_CHECK(dtype == kF32 || dtype == kU8 || dtype == kBool, "integral image: unsupported mask element type");
    IntegralJob job = make_job(masks, dtype, B, H, W, out, H * W, W);
    integral_jobs_impl(&job, 1, static_cast<IntegralJob*>(job_buf), carry, false, up, st);
}

static int64_t
solid_pitch(int64_t W)
{
    return (W + 63) / 64;
}

uint64_t
solid_map_bytes(int64_t B, int64_t H, int64_t W)
{
    return uint64_t(B) * uint64_t(H / kSolidTile) * uint64_t(W / kSolidTile);
}

uint64_t
solid_scratch_bytes(int64_t B, int64_t H, int64_t W)
{
    return uint64_t(B) * (uint64_t(H / kSolidTile) * uint64_t(solid_pitch(W)) * 2u + 2u);
}

size_t
solid_job_bytes(size_t njobs)
{
    return njobs * sizeof(SolidJob);
}

void
launch_integral_images_padded(const IntegralRequest* req, int32_t n, float* carry, void* job_buf, void* solid_jobs,
                              Uploader& up, hipStream_t st)
{
    std::vector<IntegralJob> jobs;
    std::vector<SolidJob> solid;
    uint64_t solid_blocks = 0;
    for (int32_t i = 0; i < n; ++i)
    {
        const IntegralRequest& r = req[i];
        if (r.B == 0 || r.H == 0 || r.W == 0)
            continue;
        THULL_CHECK(r.dtype == kF32 || r.dtype == kU8 || r.dtype == kBool,
                    "integral image: unsupported mask element type");
        const int64_t ld = integral_pitch(r.W);
        jobs.push_back(make_job(r.masks, r.dtype, r.B, r.H, r.W, r.padded, integral_rows(r.H) * ld, ld, true));
        if (r.solid == nullptr)
            continue;
        IntegralJob& j = jobs.back();
        j.tile_rows = int32_t(r.H / kSolidTile);
        j.tile_pitch = int32_t(solid_pitch(r.W));
        j.solid_bits = static_cast<uint16_t*>(r.solid_scratch);
        j.odd = reinterpret_cast<uint8_t*>(j.solid_bits + r.B * j.tile_rows * j.tile_pitch);
        SolidJob q{};
        q.bits = j.solid_bits;
        q.odd = j.odd;
        q.map = r.solid;
        q.cull = r.cull;
        q.culls = r.culls;
        q.integral = r.padded;
        q.transforms = r.transforms;
        q.plane = j.plane;
        q.ld = j.ld;
        q.B = j.B;
        q.H = j.H;
        q.W = j.W;
        q.tile_rows = j.tile_rows;
        q.tile_cols = int32_t(r.W / kSolidTile);
        q.tile_pitch = j.tile_pitch;
        q.opengl = r.opengl;
        q.u8 = r.dtype == kF32 ? 0 : 1;
        for (int a = 0; a < 3; ++a)
            q.corner[a] = r.corner[a];
        q.length = r.length;
        q.bx = blocks_for(q.tile_cols, 64);
        q.by = blocks_for(q.tile_rows, kSolidRows);
        q.begin = solid_blocks;
        solid_blocks += uint64_t(q.bx) * q.by * uint64_t(q.B);
        solid.push_back(q);
    }
    integral_jobs_impl(jobs.data(), jobs.size(), static_cast<IntegralJob*>(job_buf), carry, true, up, st);
    if (solid_blocks == 0)
        return;
    THULL_CHECK(solid_blocks < (uint64_t(1) << 31), "integral image batch too large");
    SolidJob* dsolid = static_cast<SolidJob*>(solid_jobs);
    up.upload(dsolid, solid.data(), solid.size() * sizeof(SolidJob), st);
    solid_map_kernel<<<unsigned(solid_blocks), 256, 0, st>>>(dsolid, int32_t(solid.size()));
    THULL_LAUNCH_CHECK();
}

// ===========================================================================
// Octree carving (VH:168-417)
//
// One thread per parent cell.  The 8 children of a parent share a 3x3x3
// lattice of corners; each lattice point is projected once per camera (the
// reference projects 8 corners per child, 64 per parent) with bit-identical
// results, because a shared corner has the same integer grid coordinate and
// hence the same world point.  The fused row products are shared along the
// lattice axes: fmaf(A2, z, A3) per z, fmaf(A1, y, .) per (y, z), and
// fmaf(A0, x, .) per point, exactly the nested fmaf chain of VH:150-153.
//
// Cameras are visited in index order and a child stops at the first camera
// that classifies it empty, which fixes its result (VH:283, VH:415); the
// remaining children of the parent continue.
// ===========================================================================

// isolevel - epsilon = 0.5f - 0.1f (VH:260-267)
constexpr float kMargin = 0.5f - 1e-1f;

struct CarveCamera
{
    float x0, x1, x2, x3; // row 0
    float y0, y1, y2, y3; // row 1
    float d0, d1, d2, d3; // row 3 (OpenGL, w) or row 2 (OpenCV, z)
};

__device__ __forceinline__ CarveCamera
load_camera(const float* __restrict__ T, bool gl)
{
    CarveCamera c;
    const auto G = as_global(T);
    const float4 r0 = ld_float4(G);
    const float4 r1 = ld_float4(G + 4);
    const float4 rd = ld_float4(G + (gl ? 12 : 8));
    c.x0 = r0.x;
    c.x1 = r0.y;
    c.x2 = r0.z;
    c.x3 = r0.w;
    c.y0 = r1.x;
    c.y1 = r1.y;
    c.y2 = r1.z;
    c.y3 = r1.w;
    c.d0 = rd.x;
    c.d1 = rd.y;
    c.d2 = rd.z;
    c.d3 = rd.w;
    return c;
}

// Box of a set of projected corners.  The reference maps every corner to its
// pixel coordinates and starts the box at (FLT_MAX, -FLT_MAX), folding the
// corners in with fminf / fmaxf, which ignore NaN (VH:201-234).  Here the
// boxes are taken over the quotients q and mapped to pixels afterwards
// (pixel_box): the pixel mapping (to_pixel) is non-decreasing in q, and maps
// NaN to NaN and only NaN to NaN, so the mapped extremes of the non-NaN
// corners are the extremes of the mapped corners, bit for bit (it never
// yields -0); the maxima then take their upper values (to_upper).  The boxes of the 2 x 2 point groups of a lattice slice hold no
// NaN: a NaN corner is left out of the group's minimum and maximum, and a
// group whose corners are all NaN has the box (+inf, -inf) (lattice_slice).
// Boxes then merge with the NaN-propagating minimum and maximum (single
// instructions, no quieting of their operands).  A minimum of +inf stands for
// the reference's initial FLT_MAX: both give the window column or row n - 1,
// pass the partial-mask clamp test's lower-bound comparison and saturate the
// int64 conversion of its area test, and both fail no fully-inside test.  The
// maximum needs no -FLT_MAX either: -inf and -FLT_MAX both clamp to pixel 0
// after + 0.5, and the partial-mask area folds it itself (child_window).
struct Box
{
    float minx, miny, maxx, maxy;
};

// A child's window box in pixels: the minima, and for the maxima p their upper values u, which stand
// for p + 0.5 (to_upper).
struct PixelBox
{
    float minx, miny, ux, uy;
};

__device__ __forceinline__ float
min_nn(float a, float b)
{
    return __builtin_elementwise_minimum(a, b);
}
__device__ __forceinline__ float
max_nn(float a, float b)
{
    return __builtin_elementwise_maximum(a, b);
}

__device__ __forceinline__ Box
box_merge(const Box& a, const Box& b)
{
    return Box{ min_nn(a.minx, b.minx), min_nn(a.miny, b.miny), max_nn(a.maxx, b.maxx), max_nn(a.maxy, b.maxy) };
}

// clamp(int64(roundf(v)), 0, hi) of the upper window bounds: the clamp bounds
// are integers and roundf is monotone, so clamping first gives the same
// integer, NaN included (both map to 0).  The clamp is one median-of-three
// instruction, which for NaN returns the smaller of the two other operands, 0,
// like fminf(fmaxf(v, 0), hi).  For the clamped c in [0, hi], hi < 2^23,
// roundf (halves away from zero) is floor(c + 1/2) taken exactly, which is
// v_cvt_rpi_i32_f32 (one instruction; checked for every float of [0, 2^23] on
// the device by thull_selftest_division).
__device__ __forceinline__ int32_t
clamp_round(float v, float hi)
{
    const float c = __builtin_amdgcn_fmed3f(v, 0.0f, hi);
    int32_t r;
    asm("v_cvt_rpi_i32_f32 %0, %1" : "=v"(r) : "v"(c));
    return r;
}

// Pixel window of one child for one camera (VH:236-247 and VH:365-380) and
// the four integral-image reads of its box sum (VH:249-257).  I is the
// camera's integral image in the zero-padded layout (integral_pitch), so the
// reads need no bounds tests.  The reads are only issued here; the caller
// uses them after the windows of all children are in flight.
struct ChildWindow
{
    float i00, i01, i10, i11; // integral reads
    float area;               // (y1 - y0 + 1) * (x1 - x0 + 1), one rounding like float(int64 area)
    bool same;                // partial masks: clamping kept the box area (int64 wrap-around like the reference)
    bool wide;                // partial masks: y1 - y0 > 1 && x1 - x0 > 1
};

typedef __attribute__((address_space(1))) const float global_float;

// clamp(int64(roundf(m - 0.5)), 0, hi) of a box minimum m (never NaN, +inf when every corner was
// NaN): for 0.5 <= m < 2^23, m - 0.5 is exact and roundf (halves away from zero) gives floor(m); for
// m < 0.5 the rounded value is at most 0 and clamps to 0, as floor(m) does; from hi up both give hi.
// So it is floor(m) clamped, and for the clamped, non-negative m truncation is the floor.
__device__ __forceinline__ int32_t
clamp_round_min(float m, float hi)
{
    return int32_t(__builtin_amdgcn_fmed3f(m, 0.0f, hi));
}

// Lower clamp test of a box minimum m: roundf(m - 0.5f) >= 0  <=>  m - 0.5f > -0.5  <=>  m > 2^-26 for
// every float m.  The float after -0.5 is -0.5 + 2^-25, and -0.5 + 2^-26 is the tie between the two,
// which rounds to the even -0.5, so m - 0.5f stays -0.5 up to m = 2^-26 and exceeds it above; NaN
// fails both tests.
constexpr float kMinAboveHalf = 0x1p-26f;

template <bool PARTIAL>
__device__ __forceinline__ void
child_window(const PixelBox& bb, const float* __restrict__ I, uint32_t ld, float Hm1, float Wm1, ChildWindow& cw)
{
    const int32_t x0 = clamp_round_min(bb.minx, Wm1), y0 = clamp_round_min(bb.miny, Hm1);
    const int32_t x1 = clamp_round(bb.ux, Wm1), y1 = clamp_round(bb.uy, Hm1);
    // box size minus one row and plus one column: |dy| < 2^23 and |dx1| < 2^23 (H, W < 2^23)
    const int32_t dy = y1 - y0, dx1 = x1 - x0 + 1;
    bool same = true;
    if constexpr (PARTIAL)
    {
        // roundf(e) lies in [0, n - 1] iff -0.5 < e < n - 0.5, for e0 = m - 0.5 iff m > 2^-26 and for
        // e1 = p + 0.5 iff u < n - 0.5.  The box minimum never exceeds its maximum unless every corner is
        // NaN (minimum +inf, maximum NaN: u fails its test), so two tests per axis tell whether the clamp
        // changed any of the four rounded bounds.
        if (!(bb.minx > kMinAboveHalf && bb.miny > kMinAboveHalf && bb.ux < Wm1 + 0.5f && bb.uy < Hm1 + 0.5f))
        {
            // clamped somewhere: compare with the unclamped box area in int64 (wrap-around like the
            // GPU reference); its maxima start at -FLT_MAX, which an all-NaN maximum keeps (the pixel
            // maxima are u - 0.5, exactly)
            const float rx0 = roundf(bb.minx + -0.5f), ry0 = roundf(bb.miny + -0.5f);
            const float rx1 = roundf(fmaxf(bb.ux + -0.5f, -FLT_MAX) + 0.5f);
            const float ry1 = roundf(fmaxf(bb.uy + -0.5f, -FLT_MAX) + 0.5f);
            const uint64_t fy = uint64_t(f2i64_sat(ry1)) - uint64_t(f2i64_sat(ry0)) + 1u;
            const uint64_t fx = uint64_t(f2i64_sat(rx1)) - uint64_t(f2i64_sat(rx0)) + 1u;
            same = int64_t(fy * fx) == int64_t(dy + 1) * int64_t(dx1);
        }
        cw.wide = dy > 1 && dx1 > 2;
    }
    cw.same = same;
    // 32-bit byte offsets from the camera's tiled plane (a plane holds fewer than 2^30 floats), so the
    // reads take the scalar-base + vector-offset form when the plane base is wave-uniform: the entries
    // (y0 - 1, x0 - 1), (y0 - 1, x1), (y1, x0 - 1), (y1, x1) at padded rows y0 + kIntegralRow0 - 1,
    // y1 + kIntegralRow0 and columns x0 + kIntegralCol0 - 1, x1 + kIntegralCol0
    const auto G = (gptr<const char>)I;
    const uint32_t r0 = integral_row_offset(uint32_t(y0) + uint32_t(kIntegralRow0 - 1), ld);
    const uint32_t r1 = integral_row_offset(uint32_t(y1) + uint32_t(kIntegralRow0), ld);
    // (column x1 + kIntegralCol0 is kIntegralCol0 / 8 whole tiles right of column x1: that shift rides in
    // the loads' immediate offset)
    static_assert(kIntegralCol0 % 8 == 0, "tile-aligned column shift");
    constexpr uint32_t kShift1 = 4u * uint32_t(kIntegralCol0 / 8 * 32);
    const uint32_t c0 = integral_col_offset(uint32_t(x0) + uint32_t(kIntegralCol0 - 1));
    const uint32_t c1 = integral_col_offset(uint32_t(x1));
    cw.i11 = *(global_float*)(G + kShift1 + (r1 + c1) * 4u);
    cw.i00 = *(global_float*)(G + (r0 + c0) * 4u);
    cw.i10 = *(global_float*)(G + (r1 + c0) * 4u);
    cw.i01 = *(global_float*)(G + kShift1 + (r0 + c1) * 4u);
    // (dy + 1) * dx1 = dy * dx1 + dx1 exactly in 32 bits (|area| <= H * W < 2^30): one signed 24-bit
    // multiply-add, then one rounding to float like float(int64 area)
    int32_t area;
    asm("v_mad_i32_i24 %0, %1, %2, %3" : "=v"(area) : "v"(dy), "v"(dx1), "v"(dx1));
    cw.area = float(area);
}

// Decision of one child for one camera from its window (VH:258-280 and
// VH:381-412).  Returns true when the camera classifies the child as empty.
template <bool PARTIAL>
__device__ __forceinline__ bool
child_decide(const ChildWindow& cw, bool fully_inside, uint32_t bit, uint32_t& refine, uint32_t& inside_any)
{
    const float sum = ((cw.i11 + cw.i00) - cw.i10) - cw.i01;
    if constexpr (!PARTIAL)
    {
        if (sum <= kMargin)
            return true;
        if (!(sum >= cw.area - kMargin))
            refine |= bit;
        return false;
    }
    else
    {
        if (fully_inside)
            inside_any |= bit;
        if (sum <= kMargin && cw.same)
            return true;
        if (sum >= cw.area - kMargin && cw.same)
            return false;
        if (cw.wide)
            refine |= bit;
        return false;
    }
}

// Largest magnitude of three values; NaN if any of them is NaN.
__device__ __forceinline__ float
max_abs3_nan(float a, float b, float c)
{
    return __builtin_elementwise_maximum(__builtin_elementwise_maximum(fabsf(a), fabsf(b)), fabsf(c));
}

// Carving divides only to take the pixel coordinate q + 1 (OpenGL) or
// q - 0.5 (OpenCV) of a quotient q.  With every operand magnitude at most
// 2^40 (hi, NaN failing) and the denominator's at least 2^-40 (lo_d), the
// shared-reciprocal division gives those pixel coordinates exactly: a
// numerator of at least 2^-80 keeps the IEEE division's scaling and fix-up
// idle (see div2_shared), and a smaller one, zero included, gives |q| < 2^-40
// on both routes, which leaves q + 1 at 1 and q - 0.5 at -0.5.
__device__ __forceinline__ bool
carve_div_in_range(float hi, float lo_d)
{
    return hi <= 0x1p40f && lo_d >= 0x1p-40f;
}

// Pixel coordinate of a projected coordinate q (VH:163-170): OpenGL maps
// normalized device coordinates with image_utils.h:67-71 (t * 0.5 is exact, so
// fmaf(t, 0.5, -0.5) == (t / 2) - 0.5), OpenCV subtracts the pixel centre.
// Every step is a correctly rounded operation that is non-decreasing in its
// operand (size >= 1), so the mapping is non-decreasing; it maps NaN, and only
// NaN, to NaN (infinities stay infinite, overflow gives an infinity) and never
// yields -0, so it commutes with the box extremes (Box).
template <bool GL>
__device__ __forceinline__ float
to_pixel(float q, float size)
{
    if constexpr (GL)
        return fmaf((q + 1.0f) * size, 0.5f, -0.5f);
    else
        return q - 0.5f;
}

// u = p + 0.5 of a box maximum's pixel coordinate p = to_pixel(q) in fewer operations: OpenCV q itself,
// OpenGL ((q + 1) * size) * 0.5 (the halving is exact).  For every float q and image size n, u gives
// the same upper window bound clamp_round(u, n - 1), the same clamp test u < n - 0.5 and, where the
// box minimum can pass its fully-inside test (p >= 0.5), the same fully-inside test u < n - 1 as the
// rounded p + 0.5 and the test p < n - 1.5 do, and u - 0.5 rounds back to p exactly (checked on the
// host for all 2^32 floats, both conventions and n from 1 to 2^23 - 1).
template <bool GL>
__device__ __forceinline__ float
to_upper(float q, float size)
{
    if constexpr (GL)
        return ((q + 1.0f) * size) * 0.5f;
    else
        return q;
}

// The pixel box of a box of quotients: the minima mapped by to_pixel, the maxima by to_upper.
template <bool GL>
__device__ __forceinline__ PixelBox
pixel_box(const Box& q, float fW, float fH)
{
    return PixelBox{ to_pixel<GL>(q.minx, fW), to_pixel<GL>(q.miny, fH), to_upper<GL>(q.maxx, fW),
                     to_upper<GL>(q.maxy, fH) };
}

// Projects one z-slice (N x N points, 3 x 3 of a parent's lattice or 2 x 2 of a
// child's) for one camera and reduces it to the quotient boxes of its 2 x 2 point
// groups, box a + (N - 1) b for x offset a and y offset b.  The fused row products are shared along the
// lattice axes: fmaf(A2, z, A3) per slice, fmaf(A1, y, .) per row and
// fmaf(A0, x, .) per point, the nested fmaf chain of VH:150-153.  The
// quotients take the shared-reciprocal division, checked once for the whole
// slice (carve_div_in_range; the largest magnitude propagates NaN, so a NaN
// operand fails the check too); a slice that fails is projected again with
// the IEEE division (rare: a lattice point on a camera's principal plane, or
// non-finite input), and `nanpts` gets bit u + Nv for each point whose
// quotients hold a NaN.  A slice that passes has finite quotients only.
template <bool GL, int N>
__device__ __forceinline__ void
lattice_slice(const CarveCamera& cam, const float (&wx)[N], const float (&wy)[N], float wz,
              Box (&win)[(N - 1) * (N - 1)], uint32_t& nanpts)
{
    const float ax = fmaf(cam.x2, wz, cam.x3);
    const float ay = fmaf(cam.y2, wz, cam.y3);
    const float ad = fmaf(cam.d2, wz, cam.d3);
    float ppx[N][N], ppy[N][N]; // [v][u] quotients
    float hi = 0.0f, lo = 0.0f;
#pragma unroll
    for (int v = 0; v < N; ++v)
    {
        const float bx = fmaf(cam.x1, wy[v], ax);
        const float by = fmaf(cam.y1, wy[v], ay);
        const float bd = fmaf(cam.d1, wy[v], ad);
        float h = 0.0f, l = 0.0f;
#pragma unroll
        for (int u = 0; u < N; ++u)
        {
            const float cx = fmaf(cam.x0, wx[u], bx);
            const float cy = fmaf(cam.y0, wx[u], by);
            const float cd = fmaf(cam.d0, wx[u], bd);
            const float hu = max_abs3_nan(cx, cy, cd);
            h = u == 0 ? hu : __builtin_elementwise_maximum(h, hu);
            l = u == 0 ? fabsf(cd) : fminf(l, fabsf(cd));
            div2_unchecked(cx, cy, cd, ppx[v][u], ppy[v][u]); // cx / cd, cy / cd when in range
        }
        hi = v == 0 ? h : __builtin_elementwise_maximum(hi, h);
        lo = v == 0 ? l : fminf(lo, l);
    }
    nanpts = 0u;
    if (carve_div_in_range(hi, lo))
    {
        // every quotient is finite: the boxes take the single-instruction minimum / maximum
#pragma unroll
        for (int bb = 0; bb + 1 < N; ++bb)
#pragma unroll
            for (int a = 0; a + 1 < N; ++a)
            {
                const float mnx0 = min_nn(ppx[bb][a], ppx[bb][a + 1]);
                const float mnx1 = min_nn(ppx[bb + 1][a], ppx[bb + 1][a + 1]);
                const float mny0 = min_nn(ppy[bb][a], ppy[bb][a + 1]);
                const float mny1 = min_nn(ppy[bb + 1][a], ppy[bb + 1][a + 1]);
                const float mxx0 = max_nn(ppx[bb][a], ppx[bb][a + 1]);
                const float mxx1 = max_nn(ppx[bb + 1][a], ppx[bb + 1][a + 1]);
                const float mxy0 = max_nn(ppy[bb][a], ppy[bb][a + 1]);
                const float mxy1 = max_nn(ppy[bb + 1][a], ppy[bb + 1][a + 1]);
                win[a + (N - 1) * bb] = Box{ min_nn(mnx0, mnx1), min_nn(mny0, mny1), max_nn(mxx0, mxx1), max_nn(mxy0, mxy1) };
            }
        return;
    }
#pragma unroll
    for (int v = 0; v < N; ++v)
    {
        const float bx = fmaf(cam.x1, wy[v], ax);
        const float by = fmaf(cam.y1, wy[v], ay);
        const float bd = fmaf(cam.d1, wy[v], ad);
#pragma unroll
        for (int u = 0; u < N; ++u)
        {
            const float cx = fmaf(cam.x0, wx[u], bx);
            const float cy = fmaf(cam.y0, wx[u], by);
            const float cd = fmaf(cam.d0, wx[u], bd);
            ppx[v][u] = cx / cd;
            ppy[v][u] = cy / cd;
            if (ppx[v][u] != ppx[v][u] || ppy[v][u] != ppy[v][u])
                nanpts |= 1u << (u + N * v);
        }
    }
    // NaN quotients are left out (fminf / fmaxf); an all-NaN group gets the box (+inf, -inf)
#pragma unroll
    for (int bb = 0; bb + 1 < N; ++bb)
#pragma unroll
        for (int a = 0; a + 1 < N; ++a)
        {
            const float mnx0 = fminf(ppx[bb][a], ppx[bb][a + 1]);
            const float mnx1 = fminf(ppx[bb + 1][a], ppx[bb + 1][a + 1]);
            const float mny0 = fminf(ppy[bb][a], ppy[bb][a + 1]);
            const float mny1 = fminf(ppy[bb + 1][a], ppy[bb + 1][a + 1]);
            const float mxx0 = fmaxf(ppx[bb][a], ppx[bb][a + 1]);
            const float mxx1 = fmaxf(ppx[bb + 1][a], ppx[bb + 1][a + 1]);
            const float mxy0 = fmaxf(ppy[bb][a], ppy[bb][a + 1]);
            const float mxy1 = fmaxf(ppy[bb + 1][a], ppy[bb + 1][a + 1]);
            win[a + (N - 1) * bb] = Box{ fminf(fminf(mnx0, mnx1), INFINITY), fminf(fminf(mny0, mny1), INFINITY),
                                   fmaxf(fmaxf(mxx0, mxx1), -INFINITY), fmaxf(fmaxf(mxy0, mxy1), -INFINITY) };
        }
}

// The four children of layer cz (children 4cz .. 4cz + 3) between slices cz
// (`lo`) and cz + 1 (`hi`): their windows, with the integral reads only
// issued.  A child is fully inside the frame (VH:358-362, needed for partial
// masks at the last level only) when none of its 8 corners is NaN and its
// pixel box satisfies 1 <= roundf(p) <= n - 2 on both axes, i.e.
// 0.5 <= p < n - 1.5, which for the maxima is u < n - 1 (to_upper).
struct LayerWindows
{
    ChildWindow cw[4];
    bool inside[4];
};

template <bool PARTIAL, bool GL>
__device__ __forceinline__ void
layer_windows(int cz, const Box (&lo)[4], const Box (&hi)[4], uint32_t nanpts, uint32_t alive, bool last,
              const float* __restrict__ I, uint32_t ld, float fW, float fH, float Hm1, float Wm1, float Hlim,
              float Wlim, LayerWindows& L)
{
#pragma unroll
    for (int q = 0; q < 4; ++q)
    {
        L.inside[q] = false;
        if (alive & (1u << (4 * cz + q)))
        {
            const PixelBox bb = pixel_box<GL>(box_merge(lo[q], hi[q]), fW, fH);
            child_window<PARTIAL>(bb, I, ld, Hm1, Wm1, L.cw[q]);
            if (PARTIAL && last)
            {
                const int a = q & 1, b = q >> 1;
                const uint32_t mm = ((3u << a) | (3u << (a + 3))) << (3 * b); // the group's points in a slice
                L.inside[q] = (nanpts & (mm | (mm << 9))) == 0u && bb.minx >= 0.5f && bb.miny >= 0.5f &&
                              bb.ux < Wlim && bb.uy < Hlim;
            }
        }
    }
}

// Decisions of the live children of layer cz; returns the children this
// camera finds empty.
template <bool PARTIAL>
__device__ __forceinline__ uint32_t
layer_decide(int cz, const LayerWindows& L, uint32_t alive, uint32_t& refine, uint32_t& inside_any)
{
    uint32_t dead = 0u;
#pragma unroll
    for (int q = 0; q < 4; ++q)
    {
        const uint32_t bit = 1u << (4 * cz + q);
        if (!(alive & bit))
            continue;
        if (child_decide<PARTIAL>(L.cw[q], L.inside[q], bit, refine, inside_any))
            dead |= bit;
    }
    return dead;
}

// Projects the 3x3x3 lattice of one parent for one camera and classifies the
// live children.  `dead` collects children found empty by this camera.
template <bool PARTIAL, bool GL>
__device__ __forceinline__ uint32_t
parent_camera(const SceneDev& s,
              const float (&wx)[3],
              const float (&wy)[3],
              const float (&wz)[3],
              int32_t b,
              uint32_t alive,
              bool last,
              uint32_t& refine,
              uint32_t& inside_any)
{
    const float fH = float(s.H), fW = float(s.W);
    const float Hm1 = float(s.H - 1), Wm1 = float(s.W - 1);
    const float Wlim = float(s.W) - 1.0f, Hlim = float(s.H) - 1.0f; // fully-inside limits of u
    const uint32_t ld = uint32_t(integral_pitch(s.W));
    const CarveCamera cam = load_camera(s.transforms + 16 * b, GL);
    // the camera's tiled plane (common.h)
    const float* I = s.integral + int64_t(b) * integral_rows(s.H) * ld;

    // one z-slice of the lattice at a time (only two slices of windows live); the reads of the lower
    // layer are in flight while the top slice is projected and the upper layer's reads are issued
    Box w0[4], w1[4];
    uint32_t n0 = 0u, n1 = 0u;
    lattice_slice<GL>(cam, wx, wy, wz[0], w0, n0);
    lattice_slice<GL>(cam, wx, wy, wz[1], w1, n1);
    LayerWindows L0, L1;
    layer_windows<PARTIAL, GL>(0, w0, w1, n0 | (n1 << 9), alive, last, I, ld, fW, fH, Hm1, Wm1, Hlim, Wlim, L0);
    lattice_slice<GL>(cam, wx, wy, wz[2], w0, n0);
    layer_windows<PARTIAL, GL>(1, w1, w0, n1 | (n0 << 9), alive, last, I, ld, fW, fH, Hm1, Wm1, Hlim, Wlim, L1);
    return layer_decide<PARTIAL>(0, L0, alive, refine, inside_any) | layer_decide<PARTIAL>(1, L1, alive, refine, inside_any);
}

// Whether camera b can be left out for a parent cell: its mask is 1 in every pixel that the windows of the cell's
// children can hold, and the box sums of such windows are certain to classify as full, so the camera empties and
// refines none of the children; with partial masks it also sees all of them fully inside the frame.
//
// The cell's centre projects to q = n / d.  For any point of the cell, n and d differ from the centre's by at most
// the half cell size h times their coefficients, so |q - q_centre| <= h sum |A_i - q_centre D_i| / (|d| - h sum
// |D_i|), with the rounding errors of all of them bounded by 2^-20 of their largest magnitudes over the cube
// (CullCamera).  A window reaches at most one pixel past the projected corners; half a pixel more covers the
// partial masks' frame margin, a quarter the approximate quotients here.  A centre in tile t covers tiles within
// ceil(reach / 4) of t, all solid when t's distance exceeds that.  Any NaN fails the test (it ends in a reach that
// no distance covers).
struct SkipProbe
{
    float reach; // how far the windows may reach from the centre's pixel, NaN or too large: not skipped
    uint32_t at; // map byte of the centre's tile
    bool inside; // FIELD: every point of the cell projects well inside the image, with operands of at most 2^40
                 // and denominators of at least 2^-40
};

// FIELD: for the field, whose factor is 1 over solid pixels whatever the box sums, without CullCamera::reach.
template <bool GL, bool FIELD>
__device__ __forceinline__ SkipProbe
skip_probe(const SceneDev& s, int32_t b, float half, float wx, float wy, float wz)
{
    const CarveCamera cam = load_camera(s.transforms + 16 * b, GL);
    const CullCamera cull = s.cull[b];
    const float nx = fmaf(cam.x0, wx, fmaf(cam.x1, wy, fmaf(cam.x2, wz, cam.x3)));
    const float ny = fmaf(cam.y0, wx, fmaf(cam.y1, wy, fmaf(cam.y2, wz, cam.y3)));
    const float nd = fmaf(cam.d0, wx, fmaf(cam.d1, wy, fmaf(cam.d2, wz, cam.d3)));
    const float rd = __builtin_amdgcn_rcpf(nd);
    const float qx = nx * rd, qy = ny * rd;
    const float lx = fabsf(fmaf(-qx, cam.d0, cam.x0)) + fabsf(fmaf(-qx, cam.d1, cam.x1)) +
                     fabsf(fmaf(-qx, cam.d2, cam.x2));
    const float ly = fabsf(fmaf(-qy, cam.d0, cam.y0)) + fabsf(fmaf(-qy, cam.d1, cam.y1)) +
                     fabsf(fmaf(-qy, cam.d2, cam.y2));
    const float den = fabsf(nd) - fmaf(half, cull.sum_d, cull.ed);
    float ex = fmaf(half, lx, fmaf(fabsf(qx), cull.ed, cull.ex));
    float ey = fmaf(half, ly, fmaf(fabsf(qy), cull.ed, cull.ey));
    float px, py;
    if constexpr (GL)
    {
        const float hw = 0.5f * float(s.W), hh = 0.5f * float(s.H);
        ex *= hw;
        ey *= hh;
        px = fmaf(qx, hw, hw - 0.5f);
        py = fmaf(qy, hh, hh - 0.5f);
    }
    else
    {
        px = qx - 0.5f;
        py = qy - 0.5f;
    }
    const float reach = fmaf(__builtin_elementwise_maximum(ex, ey), __builtin_amdgcn_rcpf(den), 1.75f);
    const int32_t tx = int32_t(floorf(px * (1.0f / kSolidTile))), ty = int32_t(floorf(py * (1.0f / kSolidTile)));
    const bool in = uint32_t(tx) < uint32_t(s.solid_w) && uint32_t(ty) < uint32_t(s.solid_h);
    SkipProbe p;
    p.at = in ? uint32_t(ty) * uint32_t(s.solid_w) + uint32_t(tx) : 0u;
    p.reach = in && den > 0.0f && (FIELD || reach <= cull.reach) ? reach : 1e30f;
    if constexpr (FIELD) // the error bounds are 2^-20 of the operands' largest magnitudes
        p.inside = den >= 0x1p-40f && cull.ex <= 0x1p20f && cull.ey <= 0x1p20f && cull.ed <= 0x1p20f &&
                   px - p.reach >= 0.0f && py - p.reach >= 0.0f && px + p.reach <= float(s.W - 1) &&
                   py + p.reach <= float(s.H - 1);
    return p;
}

// The probes of kSkipBatch cameras and their map bytes are in flight together.
constexpr int kSkipBatch = 4;

// Which of the cameras b0, b0 + step, ... below `end` (kSkipBatch of them) the lane can skip, as bits.
template <bool GL>
__device__ __forceinline__ uint32_t
carve_skips(const SceneDev& s, int32_t b0, int32_t step, int32_t end, float half, float wx, float wy, float wz)
{
    SkipProbe p[kSkipBatch];
    int32_t d[kSkipBatch];
#pragma unroll
    for (int u = 0; u < kSkipBatch; ++u)
        p[u] = skip_probe<GL, false>(s, min(b0 + u * step, end - 1), half, wx, wy, wz);
#pragma unroll
    for (int u = 0; u < kSkipBatch; ++u)
        d[u] = as_global(s.solid + int64_t(min(b0 + u * step, end - 1)) * s.solid_h * s.solid_w)[p[u].at];
    uint32_t skips = 0u;
#pragma unroll
    for (int u = 0; u < kSkipBatch; ++u)
        if (p[u].reach <= float(kSolidTile * (d[u] - 1)))
            skips |= 1u << u;
    return skips;
}

// Whether testing the cameras of a level-li cell is worth it.  A cell that is large beside the object lies on the
// outlines of most silhouettes, so the level decides (share of the cameras that a wavefront of 64 parents of a
// 50-camera 1080p hull still tests, by level of the parents: 5 97 %, 6 78 %, 7 53 %, 8 38 %); and a cell of more
// pixels than the maps' distances reach past is in no map's solid part, whatever its level.
constexpr int32_t kCullLevel = 7;
constexpr int32_t kCullPixels = 16;

__host__ __device__ __forceinline__ bool
cull_level(const SceneDev& s, int32_t li)
{
    return s.solid != nullptr && li >= kCullLevel && ((s.H > s.W ? s.H : s.W) >> li) <= kCullPixels;
}

__device__ __forceinline__ bool
cull_pays(const SceneDev& s, int32_t li)
{
    return cull_level(s, li) && s.culls != 0;
}

// Cameras c0 .. c0 + n - 1 (n <= 64) that some lane of the wavefront (all in one scene) cannot skip; with G
// lanes per parent the lanes of a group (j: lane in its group) test them in turn.
template <bool GL, int G>
__device__ __forceinline__ uint64_t
carve_needed(const SceneDev& s, int32_t c0, int32_t n, int32_t j, float half, float wx, float wy, float wz)
{
    uint64_t need = 0;
    for (int32_t k = 0; k < n; k += kSkipBatch * G)
    {
        const uint32_t skips = carve_skips<GL>(s, c0 + k + j, G, c0 + n, half, wx, wy, wz);
#pragma unroll
        for (int u = 0; u < kSkipBatch; ++u)
        {
            const int32_t first = k + u * G; // camera c0 + first + j is the lane's
            if (first >= n)
                break;
            uint64_t m = __ballot((skips & (1u << u)) == 0u && first + j < n);
#pragma unroll
            for (int off = 32; off >= G; off >>= 1)
                m |= m >> off; // the groups' answers
            if constexpr (G < 64)
                m &= (uint64_t(1) << G) - 1u;
            need |= m << first;
        }
    }
    return need;
}

__device__ __forceinline__ void
lattice_world(const SceneDev& s, uint32_t px, uint32_t py, uint32_t pz, int32_t li, float (&wx)[3], float (&wy)[3],
              float (&wz)[3])
{
    const float inv = __builtin_ldexpf(1.0f, -(li + 1)); // 1 / resolution_children, exact
#pragma unroll
    for (int u = 0; u < 3; ++u)
    {
        wx[u] = grid_to_world(2 * px + u, inv, s.length, s.corner[0]);
        wy[u] = grid_to_world(2 * py + u, inv, s.length, s.corner[1]);
        wz[u] = grid_to_world(2 * pz + u, inv, s.length, s.corner[2]);
    }
}

// All cameras in index order for one parent; returns the occupancy mask.  CULL: cameras may be left out.  A launch in
// which no scene can leave out any (carve_culls) runs a copy without that code, here and in the split kernels
// (64 mixed scenes, us with and without it where it never applies: 100 635 parents, 4 lanes, 460 and 422; 455 118, 2
// lanes, 760 and 688).
template <bool PARTIAL, bool GL, bool UNIFORM, bool CULL>
__device__ uint32_t
classify_parent(const SceneDev& s, uint32_t px, uint32_t py, uint32_t pz, int32_t li, bool last, uint32_t& tests)
{
    float wx[3], wy[3], wz[3];
    lattice_world(s, px, py, pz, li, wx, wy, wz);
    uint32_t alive = 0xffu, refine = 0u, inside_any = 0u;
    if constexpr (UNIFORM && CULL)
    {
        // the cameras that some lane needs, in index order; a skipped camera counts as a test of every live child
        const float half = 0.5f * s.length * __builtin_ldexpf(1.0f, -li);
        for (int32_t c0 = 0; c0 < s.B && !__all(alive == 0u); c0 += 64)
        {
            const int32_t n = min(s.B - c0, 64);
            uint64_t need = n < 64 ? (uint64_t(1) << n) - 1u : ~uint64_t(0);
            if (cull_pays(s, li))
            {
                need = carve_needed<GL, 1>(s, c0, n, 0, half, wx[1], wy[1], wz[1]);
                if (PARTIAL && int32_t(__popcll(need)) < n)
                    inside_any = 0xffu; // a skipped camera sees all children fully inside
            }
            for (; need != 0u; need &= need - 1u)
            {
                if (__all(alive == 0u))
                    break;
                const int32_t b = c0 + int32_t(__builtin_ctzll(need));
                if (alive == 0u)
                    continue;
                const uint32_t dead =
                    parent_camera<PARTIAL, GL>(s, wx, wy, wz, b, alive, last, refine, inside_any);
                tests += uint32_t(b + 1) * uint32_t(__popc(dead));
                alive &= ~dead;
            }
        }
        tests += uint32_t(s.B) * uint32_t(__popc(alive));
    }
    else
        for (int32_t b = 0; b < s.B; ++b)
        {
            if (alive == 0u)
                break;
            tests += __popc(alive);
            alive &= ~parent_camera<PARTIAL, GL>(s, wx, wy, wz, b, alive, last, refine, inside_any);
        }
    uint32_t occ = refine & alive; // should_refine && !is_empty
    if (PARTIAL && last)
        occ &= inside_any; // (!last_children || fully_inside_one_frame)
    return occ;
}

template <bool PARTIAL, bool GL, bool UNIFORM, bool CULL>
__device__ __forceinline__ uint32_t
classify_entry(const SceneDev& s, uint64_t key, int32_t step, uint32_t& tests)
{
    const int32_t li = step - s.start; // the scene's own octree level
    if (li >= s.level)
        return 0u;
    return classify_parent<PARTIAL, GL, UNIFORM, CULL>(s, key_x(key), key_y(key), key_z(key), li, li == s.level - 1,
                                                       tests);
}

// UNIFORM = true for a descriptor shared by the whole wave.  The flag changes
// no arithmetic; it keeps the wave-uniform and the per-lane instantiations
// apart, so that the compiler cannot merge the two calls into one per-lane copy.
template <bool UNIFORM, bool CULL>
__device__ __forceinline__ uint32_t
classify_scene(const SceneDev& s, uint64_t key, int32_t level_i, uint32_t& tests)
{
    if (s.partial)
        return s.opengl ? classify_entry<true, true, UNIFORM, CULL>(s, key, level_i, tests)
                        : classify_entry<true, false, UNIFORM, CULL>(s, key, level_i, tests);
    return s.opengl ? classify_entry<false, true, UNIFORM, CULL>(s, key, level_i, tests)
                    : classify_entry<false, false, UNIFORM, CULL>(s, key, level_i, tests);
}

// Classification of the kCarveThreads parents of logical block lb (all threads of the block call it).
template <bool CULL>
__device__ __forceinline__ void
classify_block(const uint64_t* __restrict__ parents,
               uint32_t n,
               int32_t step,
               const SceneDev* __restrict__ scenes,
               uint8_t* __restrict__ child_mask,
               uint32_t* __restrict__ block_counts,
               unsigned long long* __restrict__ tests_out,
               uint32_t lb,
               uint32_t* lds)
{
    const uint32_t t = lb * kCarveThreads + threadIdx.x;
    uint32_t mask = 0u, tests = 0u;
    if (t < n)
    {
        const uint64_t key = parents[t];
        const uint32_t sid = key_scene(key);
        const uint32_t s0 = __builtin_amdgcn_readfirstlane(sid);
        if (__all(sid == s0)) // the whole wave carves one scene: camera data and integral bases are scalar
            mask = classify_scene<true, CULL>(wave_uniform(scenes[s0]), key, step, tests);
        else
            mask = classify_scene<false, false>(scenes[sid], key, step, tests);
        child_mask[t] = uint8_t(mask);
    }
    uint32_t total;
    block_exclusive_sum(__popc(mask), lds, total);
    if (threadIdx.x == 0)
        block_counts[lb] = total;
    uint32_t tsum;
    block_exclusive_sum(tests, lds, tsum);
    if (threadIdx.x == 0 && tests_out != nullptr)
        atomicAdd(tests_out, (unsigned long long)tsum);
}

template <bool CULL>
__global__ __launch_bounds__(kCarveThreads) void
carve_classify_kernel(const uint64_t* __restrict__ parents,
                      uint32_t n,
                      int32_t level_i,
                      const SceneDev* __restrict__ scenes,
                      uint8_t* __restrict__ child_mask,
                      uint32_t* __restrict__ block_counts,
                      unsigned long long* __restrict__ tests_out)
{
    __shared__ uint32_t lds[kCarveThreads / 64];
    const uint32_t lb = xcd_block(blockIdx.x, gridDim.x); // neighbouring parents read neighbouring pixels
    classify_block<CULL>(parents, n, level_i, scenes, child_mask, block_counts, tests_out, lb, lds);
}

// Device-driven form of carve_classify_kernel for a level whose size only the device knows
// (min(*dev_n, cap)): a persistent grid of workgroups (a multiple of 8) takes blocks of kCarveThreads
// parents from a work queue.  There is one queue per XCD (cursors[8], zero at start): hardware
// workgroup w runs on XCD w % 8 and takes that XCD's blocks, runs of 16 consecutive blocks whose run
// index is w % 8 modulo 8 -- the order xcd_block gives a launch-per-level grid -- so neighbouring
// parents still share an L2, and the workgroups of an XCD balance its blocks among themselves.
template <bool CULL>
__global__ __launch_bounds__(kCarveThreads, 4) void
carve_classify_queue_kernel(const uint64_t* __restrict__ parents,
                            const unsigned long long* __restrict__ dev_n,
                            uint32_t cap,
                            int32_t step,
                            const SceneDev* __restrict__ scenes,
                            uint8_t* __restrict__ child_mask,
                            uint32_t* __restrict__ block_counts,
                            unsigned long long* __restrict__ tests_out,
                            uint32_t* __restrict__ cursors)
{
    __shared__ uint32_t lds[kCarveThreads / 64];
    __shared__ uint32_t next;
    const uint32_t n = uint32_t(min(*dev_n, (unsigned long long)cap));
    const uint32_t nblocks = (n + kCarveThreads - 1) / kCarveThreads;
    const uint32_t xcd = blockIdx.x & 7u;
    for (;;)
    {
        if (threadIdx.x == 0)
            next = atomicAdd(cursors + xcd, 1u);
        __syncthreads();
        const uint32_t k = next;
        __syncthreads();
        const uint64_t lb = (uint64_t(k / 16u) * 8u + xcd) * 16u + (k % 16u); // increases with k
        if (lb >= nblocks)
            break;
        classify_block<CULL>(parents, n, step, scenes, child_mask, block_counts, tests_out, uint32_t(lb), lds);
    }
}

// Small levels are latency-bound with one thread per parent (a chain of up to
// B dependent camera iterations).  Here G lanes share a parent and take the
// cameras b = j, j + G, ...; the result flags are ORs over cameras and a
// child is empty if any camera says so, so the lanes combine exactly by
// OR / min across the group.  The canonical early-exit count is rebuilt from
// the first camera that found each child empty.
template <int G, bool PARTIAL, bool GL, bool CULL>
__device__ __forceinline__ void
classify_split(const SceneDev& s, uint64_t key, int32_t level_i, int32_t j, uint32_t& refine, uint32_t& inside,
               uint32_t (&first_empty)[8])
{
    float wx[3], wy[3], wz[3];
    lattice_world(s, key_x(key), key_y(key), key_z(key), level_i, wx, wy, wz);
    const bool last = level_i == s.level - 1;
    // The group takes its cameras in rounds of G (lane j: camera b0 + j) and shares the children
    // found empty after every round, so no lane goes on with children another lane has emptied
    // and the group stops when all children are empty.  A child emptied in a round was live for
    // every camera before it, so the smallest camera of that round that emptied it is its first.
    // All lanes of a group have the same parent, so they run the same rounds.
    uint32_t alive = 0xffu;
    // CULL, with several rounds of cameras: those that no parent of the wavefront needs are left out first.  The
    // lanes of a group test the cameras in turn, the groups' answers are ORed into one mask per 64 cameras, and its
    // cameras go to the lanes in rounds.  (Groups of 16 and 64 lanes have few rounds to save.)
    const bool cull = CULL && s.B >= 4 * G && cull_pays(s, level_i);
    const float half = 0.5f * s.length * __builtin_ldexpf(1.0f, -level_i);
    uint64_t need = 0;
    int32_t c0 = 0, b0 = 0; // first camera of the mask; next camera to look at
    for (;;)
    {
        int32_t b = b0 + j; // the lane's camera, s.B or more for none
        if (cull)
        {
            while (need == 0 && b0 < s.B)
            {
                c0 = b0;
                const int32_t n = min(s.B - c0, 64);
                if constexpr (CULL)
                    need = carve_needed<GL, G>(s, c0, n, j, half, wx[1], wy[1], wz[1]);
                if (PARTIAL && int32_t(__popcll(need)) < n)
                    inside = 0xffu; // a skipped camera sees all children fully inside
                b0 = c0 + n;
            }
            if (need == 0)
                break;
            b = s.B;
#pragma unroll
            for (int q = 0; q < G; ++q)
            {
                if (need == 0)
                    break;
                b = j == q ? c0 + int32_t(__builtin_ctzll(need)) : b;
                need &= need - 1u;
            }
        }
        else
        {
            if (b0 >= s.B)
                break;
            b0 += G;
        }
        uint32_t dead = 0u;
        if (b < s.B && (!CULL || alive != 0u))
            dead = parent_camera<PARTIAL, GL>(s, wx, wy, wz, b, alive, last, refine, inside);
#pragma unroll
        for (int c = 0; c < 8; ++c)
            if (dead & (1u << c))
                first_empty[c] = uint32_t(b);
        alive &= ~dead;
#pragma unroll
        for (int off = G / 2; off >= 1; off >>= 1)
            alive &= uint32_t(__shfl_xor(int(alive), off, G));
        if (CULL ? __all(alive == 0u) : alive == 0u)
            break;
    }
}

// Scene flags and the classification of one parent by lane j of its group;
// UNIFORM as for classify_scene.
template <int G, bool UNIFORM, bool CULL>
__device__ __forceinline__ void
split_scene(const SceneDev& s, uint64_t key, int32_t step, int32_t j, int32_t& B, bool& partial, bool& last,
            bool& active, uint32_t& refine, uint32_t& inside, uint32_t (&first_empty)[8])
{
    const int32_t level_i = step - s.start; // the scene's own octree level
    B = s.B;
    partial = s.partial != 0;
    last = level_i == s.level - 1;
    active = level_i < s.level;
    if (!active)
        return;
    if (partial)
    {
        if (s.opengl)
            classify_split<G, true, true, UNIFORM && CULL>(s, key, level_i, j, refine, inside, first_empty);
        else
            classify_split<G, true, false, UNIFORM && CULL>(s, key, level_i, j, refine, inside, first_empty);
    }
    else
    {
        if (s.opengl)
            classify_split<G, false, true, UNIFORM && CULL>(s, key, level_i, j, refine, inside, first_empty);
        else
            classify_split<G, false, false, UNIFORM && CULL>(s, key, level_i, j, refine, inside, first_empty);
    }
}

template <int G, bool CULL>
__global__ __launch_bounds__(256) void
carve_classify_split_kernel(const uint64_t* __restrict__ parents,
                            uint32_t n,
                            int32_t level_i,
                            const SceneDev* __restrict__ scenes,
                            uint8_t* __restrict__ child_mask,
                            unsigned long long* __restrict__ tests_out,
                            const unsigned long long* __restrict__ dev_n) // optional: n = min(n, *dev_n)
{
    __shared__ uint32_t lds[256 / 64];
    if (dev_n != nullptr)
        n = uint32_t(min((unsigned long long)n, *dev_n));
    const uint32_t gt = xcd_block(blockIdx.x, gridDim.x) * 256 + threadIdx.x;
    const uint32_t p = gt / G;
    const int32_t j = int32_t(gt % G);
    uint32_t refine = 0u, inside = 0u;
    uint32_t first_empty[8];
#pragma unroll
    for (int c = 0; c < 8; ++c)
        first_empty[c] = 0xffffffffu;
    bool active = false, partial = false, last = false;
    int32_t B = 0;
    if (p < n)
    {
        const uint64_t key = parents[p];
        const uint32_t sid = key_scene(key);
        const uint32_t s0 = __builtin_amdgcn_readfirstlane(sid);
        if (__all(sid == s0))
            split_scene<G, true, CULL>(wave_uniform(scenes[s0]), key, level_i, j, B, partial, last, active, refine,
                                       inside, first_empty);
        else
            split_scene<G, false, false>(scenes[sid], key, level_i, j, B, partial, last, active, refine, inside,
                                         first_empty);
    }
#pragma unroll
    for (int off = G / 2; off >= 1; off >>= 1)
    {
        refine |= __shfl_xor(refine, off, G);
        inside |= __shfl_xor(inside, off, G);
#pragma unroll
        for (int c = 0; c < 8; ++c)
            first_empty[c] = min(first_empty[c], uint32_t(__shfl_xor(int(first_empty[c]), off, G)));
    }
    uint32_t tests = 0u;
    if (j == 0 && p < n)
    {
        uint32_t dead = 0u;
        if (active)
        {
#pragma unroll
            for (int c = 0; c < 8; ++c)
            {
                const bool d = first_empty[c] != 0xffffffffu;
                dead |= d ? (1u << c) : 0u;
                tests += d ? first_empty[c] + 1u : uint32_t(B);
            }
        }
        uint32_t occ = active ? (refine & ~dead) : 0u;
        if (partial && last)
            occ &= inside;
        child_mask[p] = uint8_t(occ);
    }
    uint32_t tsum;
    block_exclusive_sum(tests, lds, tsum);
    if (threadIdx.x == 0 && tests_out != nullptr)
        atomicAdd(tests_out, (unsigned long long)tsum);
}

// The smallest levels: a lane per parent, child and camera.  A level of a few hundred parents leaves most of the chip
// idle whatever its split, and its time is the chain of one lane: the split kernel's projects 27 lattice points and
// reads 8 windows per camera.  Here the 8 wavefronts of a block take a child each (8 points and a window per camera),
// and the lanes of a wavefront G cameras of 64 / G parents; G is the power of two from 8 that holds the scenes'
// cameras, 64 at most.  Points shared by children are projected again, so it only pays while the chip has room, up to
// about kChildWaves wavefronts (split kernel of 64 lanes -> this one, us; 437 parents of 8 cameras 15.9 -> 8.5, 1891
// 17.1 -> 9.6; 421 of 50 31 -> 21; 1523 of 64, 12184 wavefronts, 55 -> 57; 7396 of 50 93 -> 128).
constexpr int kChildThreads = 512;
constexpr uint64_t kChildWaves = 8192;

template <bool PARTIAL, bool GL>
__device__ __forceinline__ bool
child_camera(const SceneDev& s, const float (&wx)[2], const float (&wy)[2], const float (&wz)[2], int32_t b, bool last,
             uint32_t& refine, uint32_t& inside)
{
    const uint32_t ld = uint32_t(integral_pitch(s.W));
    const CarveCamera cam = load_camera(s.transforms + 16 * b, GL);
    Box lo[1], hi[1];
    uint32_t n0 = 0u, n1 = 0u;
    lattice_slice<GL>(cam, wx, wy, wz[0], lo, n0);
    lattice_slice<GL>(cam, wx, wy, wz[1], hi, n1);
    const PixelBox bb = pixel_box<GL>(box_merge(lo[0], hi[0]), float(s.W), float(s.H));
    ChildWindow cw;
    child_window<PARTIAL>(bb, s.integral + int64_t(b) * integral_rows(s.H) * ld, ld, float(s.H - 1), float(s.W - 1), cw);
    const bool in = PARTIAL && last && (n0 | n1) == 0u && bb.minx >= 0.5f && bb.miny >= 0.5f &&
                    bb.ux < float(s.W) - 1.0f && bb.uy < float(s.H) - 1.0f;
    return child_decide<PARTIAL>(cw, in, 1u, refine, inside);
}

// One child by the lanes of its group (j of G): the group takes its cameras in rounds, as in classify_split.
template <bool PARTIAL, bool GL>
__device__ __forceinline__ void
classify_child(const SceneDev& s, uint64_t key, int32_t level_i, uint32_t c, int32_t j, int32_t G, uint32_t& refine,
               uint32_t& inside, uint32_t& first_empty)
{
    const float inv = __builtin_ldexpf(1.0f, -(level_i + 1));
    float wx[2], wy[2], wz[2];
#pragma unroll
    for (uint32_t u = 0; u < 2; ++u)
    {
        wx[u] = grid_to_world(2 * key_x(key) + (c & 1u) + u, inv, s.length, s.corner[0]);
        wy[u] = grid_to_world(2 * key_y(key) + ((c >> 1) & 1u) + u, inv, s.length, s.corner[1]);
        wz[u] = grid_to_world(2 * key_z(key) + (c >> 2) + u, inv, s.length, s.corner[2]);
    }
    const bool last = level_i == s.level - 1;
    for (int32_t b0 = 0; b0 < s.B && first_empty == 0xffffffffu; b0 += G)
    {
        const int32_t b = b0 + j;
        if (b < s.B && child_camera<PARTIAL, GL>(s, wx, wy, wz, b, last, refine, inside))
            first_empty = uint32_t(b);
        for (int off = G / 2; off >= 1; off >>= 1)
            first_empty = min(first_empty, uint32_t(__shfl_xor(int(first_empty), off, 64)));
    }
}

__device__ __forceinline__ void
child_scene(const SceneDev& s, uint64_t key, int32_t step, uint32_t c, int32_t j, int32_t G, uint32_t& occupied,
            uint32_t& tests)
{
    const int32_t level_i = step - s.start;
    if (level_i >= s.level)
        return;
    uint32_t refine = 0u, inside = 0u, first_empty = 0xffffffffu;
    if (s.partial != 0)
    {
        if (s.opengl)
            classify_child<true, true>(s, key, level_i, c, j, G, refine, inside, first_empty);
        else
            classify_child<true, false>(s, key, level_i, c, j, G, refine, inside, first_empty);
    }
    else
    {
        if (s.opengl)
            classify_child<false, true>(s, key, level_i, c, j, G, refine, inside, first_empty);
        else
            classify_child<false, false>(s, key, level_i, c, j, G, refine, inside, first_empty);
    }
    for (int off = G / 2; off >= 1; off >>= 1)
    {
        refine |= uint32_t(__shfl_xor(int(refine), off, 64));
        inside |= uint32_t(__shfl_xor(int(inside), off, 64));
    }
    const bool dead = first_empty != 0xffffffffu;
    tests = dead ? first_empty + 1u : uint32_t(s.B);
    occupied = dead ? 0u : refine;
    if (s.partial != 0 && level_i == s.level - 1)
        occupied &= inside;
}

__global__ __launch_bounds__(kChildThreads) void
carve_classify_child_kernel(const uint64_t* __restrict__ parents, uint32_t n, int32_t step,
                            const SceneDev* __restrict__ scenes, int32_t G, uint8_t* __restrict__ child_mask,
                            unsigned long long* __restrict__ tests_out,
                            const unsigned long long* __restrict__ dev_n) // optional: n = min(n, *dev_n)
{
    __shared__ uint32_t found[8][8]; // child, group: tests * 2 + occupied
    if (dev_n != nullptr)
        n = uint32_t(min((unsigned long long)n, *dev_n));
    const uint32_t per = 64u / uint32_t(G), p0 = blockIdx.x * per;
    if (p0 >= n)
        return;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t c = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)));
    const uint32_t group = lane / uint32_t(G), p = p0 + group;
    const int32_t j = int32_t(lane & uint32_t(G - 1));
    uint32_t occupied = 0u, tests = 0u;
    if (p < n)
    {
        const uint64_t key = parents[p];
        const uint32_t sid = key_scene(key), s0 = __builtin_amdgcn_readfirstlane(sid);
        if (__all(sid == s0))
            child_scene(wave_uniform(scenes[s0]), key, step, c, j, G, occupied, tests);
        else
            child_scene(scenes[sid], key, step, c, j, G, occupied, tests);
    }
    if (j == 0)
        found[c][group] = 2u * tests + occupied;
    __syncthreads();
    if (threadIdx.x >= 64u)
        return;
    uint32_t sum = 0u;
    if (lane < per && p0 + lane < n)
    {
        uint32_t mask = 0u;
#pragma unroll
        for (uint32_t k = 0; k < 8u; ++k)
        {
            const uint32_t f = found[k][lane];
            mask |= (f & 1u) << k;
            sum += f >> 1;
        }
        child_mask[p0 + lane] = uint8_t(mask);
    }
    sum = __reduce_add_sync(0xffffffffffffffffull, sum);
    if (lane == 0 && tests_out != nullptr)
        atomicAdd(tests_out, (unsigned long long)sum);
}

__device__ __forceinline__ uint32_t
popc4(const uint4& v)
{
    return uint32_t(__popc(v.x) + __popc(v.y) + __popc(v.z) + __popc(v.w));
}

__global__ __launch_bounds__(kCarveThreads) void
carve_count_kernel(const uint8_t* __restrict__ child_mask, uint32_t n, uint32_t* __restrict__ block_counts,
                   const unsigned long long* __restrict__ dev_n) // optional: n = min(n, *dev_n)
{
    __shared__ uint32_t lds[kCarveThreads / 64];
    if (dev_n != nullptr)
        n = uint32_t(min((unsigned long long)n, *dev_n));
    const uint32_t t = blockIdx.x * kCarveThreads + threadIdx.x;
    const uint32_t mask = (t < n) ? child_mask[t] : 0u;
    uint32_t total;
    block_exclusive_sum(__popc(mask), lds, total);
    if (threadIdx.x == 0)
        block_counts[blockIdx.x] = total;
}

// The kept children of a parent whose scene ends at child_level are leaf
// cells: their bits go into the scene's leaf-cell bitmap (rows of
// cell_row_words words; the 2 x 2 x 2 children touch at most 4 words, one per
// (y, z) row).  Parents whose children share a word (same scene, z, y and
// x / 16) often sit in consecutive lanes (x-neighbours among the children of
// one grandparent are listed together): the wave ORs the words of such runs
// together (a segmented reduction over runs of up to 16 lanes; a key that
// recurs further on just starts another run) and only the first lane of each
// run issues the atomics.  Every lane of the wave calls this; `mask` is 0 for
// lanes without children.
__device__ __forceinline__ void
mark_leaf_children_wave(const SceneDev* __restrict__ scenes, int32_t child_step, uint64_t key, uint32_t mask)
{
    uint32_t w[4] = { 0u, 0u, 0u, 0u };
    uint32_t* row0 = nullptr;
    uint64_t row_step = 0, plane_step = 0;
    bool mark = false;
    if (mask != 0u)
    {
        const SceneDev& sd = scenes[key_scene(key)];
        if (sd.level == child_step - sd.start)
        {
            mark = true;
            const uint32_t cx = 2 * key_x(key), cy = 2 * key_y(key), cz = 2 * key_z(key);
            const uint64_t R = uint64_t(1) << sd.level;
            row_step = sd.cell_row_words;
            plane_step = R * row_step;
            row0 = sd.cells + uint64_t(cz) * plane_step + uint64_t(cy) * row_step + (cx >> 5);
#pragma unroll
            for (int r = 0; r < 4; ++r) // r = b + 2c: children (x = 0, 1; y = b; z = c)
                w[r] = ((mask >> (2 * r)) & 3u) << (cx & 31u);
        }
    }
    // run key: the parent's key with the low 4 bits of x cleared (x / 16 picks the word)
    const uint64_t K = mark ? (key & ~uint64_t(15)) : ~uint64_t(0);
    const uint32_t klo = uint32_t(K), khi = uint32_t(K >> 32);
#pragma unroll
    for (int d = 1; d < 16; d <<= 1)
    {
        // every lane shuffles (no short-circuit around a cross-lane read); lanes past the end read
        // their own values, which leaves them unchanged
        const uint32_t olo = uint32_t(__shfl_down(int(klo), d, 64));
        const uint32_t ohi = uint32_t(__shfl_down(int(khi), d, 64));
        const bool same = (olo == klo) & (ohi == khi);
#pragma unroll
        for (int r = 0; r < 4; ++r)
        {
            const uint32_t o = uint32_t(__shfl_down(int(w[r]), d, 64));
            w[r] |= same ? o : 0u;
        }
    }
    const int lane = int(threadIdx.x & 63);
    const uint32_t plo = uint32_t(__shfl_up(int(klo), 1, 64));
    const uint32_t phi = uint32_t(__shfl_up(int(khi), 1, 64));
    const bool first = (lane == 0) | (plo != klo) | (phi != khi);
    if (mark && first)
    {
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (w[r] != 0u)
                atomicOr(row0 + uint64_t(r >> 1) * plane_step + uint64_t(r & 1) * row_step, w[r]);
    }
}

// The kept children of a block's parents, one contiguous range of the list from `first`: assembled in LDS at `off` and
// written with coalesced stores.  All threads of the block call this.
__device__ __forceinline__ void
write_children(uint64_t* stage, uint64_t key, uint32_t mask, uint32_t off, uint32_t total, uint64_t first,
               uint64_t* __restrict__ children, uint64_t out_cap, int32_t child_step,
               const SceneDev* __restrict__ scenes, bool mark_leaves)
{
    if (mask != 0u)
    {
        const uint32_t s = key_scene(key), x = 2 * key_x(key), y = 2 * key_y(key), z = 2 * key_z(key);
        // VH:694-711: children of a parent in child order (x bit, y bit, z bit)
#pragma unroll
        for (int c = 0; c < 8; ++c)
            if (mask & (1u << c))
                stage[off++] = pack_key(s, x + (c & 1), y + ((c >> 1) & 1), z + ((c >> 2) & 1));
    }
    __syncthreads();
    uint64_t* dst = children + first;
    for (uint32_t q = threadIdx.x; q < total; q += kCarveThreads)
        if (first + q < out_cap)
            dst[q] = stage[q];
    if (mark_leaves)
        mark_leaf_children_wave(scenes, child_step, key, mask);
}

__global__ __launch_bounds__(kCarveThreads) void
carve_scatter_kernel(const uint64_t* __restrict__ parents,
                     uint32_t n,
                     const uint8_t* __restrict__ child_mask,
                     const uint32_t* __restrict__ block_offsets,
                     uint64_t* __restrict__ children,
                     int32_t child_step,
                     const SceneDev* __restrict__ scenes,
                     bool mark_leaves,
                     const unsigned long long* __restrict__ dev_n, // optional: n = min(n, *dev_n)
                     uint64_t out_cap)                             // children past this index are dropped
{
    __shared__ uint32_t lds[kCarveThreads / 64];
    __shared__ uint64_t stage[kCarveThreads * 8];
    if (dev_n != nullptr)
        n = uint32_t(min((unsigned long long)n, *dev_n));
    const uint32_t t = blockIdx.x * kCarveThreads + threadIdx.x;
    const uint32_t mask = (t < n) ? child_mask[t] : 0u;
    const uint64_t key = (t < n) ? parents[t] : 0; // read with the mask, ahead of the block sum
    uint32_t total;
    const uint32_t off = block_exclusive_sum(__popc(mask), lds, total);
    write_children(stage, key, mask, off, total, block_offsets[blockIdx.x], children, out_cap, child_step, scenes,
                   mark_leaves);
}

// Count, scan and scatter of a level of at most kCompactParents in one launch: every block sums the masks of all
// parents before its own (a byte each, a few 16-byte loads per thread from L2), so no block waits for another, and
// the last one has the total for the host.  Small levels spend their time in launches: a level-7 hull of 8 cameras
// 420 -> 384 us, a level-8 one of 10 540 -> 487.  At kCompactParents a thread reads 32 groups of masks at most.
__global__ __launch_bounds__(kCarveThreads) void
carve_compact_kernel(const uint64_t* __restrict__ parents, uint32_t n, const uint8_t* __restrict__ child_mask,
                     uint64_t* __restrict__ children, int32_t child_step, const SceneDev* __restrict__ scenes,
                     bool mark_leaves, unsigned long long* __restrict__ total_out, ScanNotify note)
{
    __shared__ uint32_t lds[kCarveThreads / 64];
    __shared__ uint64_t stage[kCarveThreads * 8];
    const uint32_t t = blockIdx.x * kCarveThreads + threadIdx.x;
    const uint32_t mask = (t < n) ? child_mask[t] : 0u;
    const uint64_t key = (t < n) ? parents[t] : 0;
    uint32_t before = 0u;
#pragma unroll 4
    for (uint32_t g = threadIdx.x; g < blockIdx.x * (kCarveThreads / 16u); g += kCarveThreads)
        before += popc4(reinterpret_cast<const uint4*>(child_mask)[g]);
    // one block sum of both: at most 8 children of 256 parents in the low 12 bits, the sum before above
    static_assert(uint64_t(kCompactParents) * 8u <= uint64_t(1) << 20, "sums fit 20 bits");
    uint32_t both;
    const uint32_t mine = block_exclusive_sum((before << 12) | __popc(mask), lds, both);
    const uint32_t first = both >> 12, total = both & 4095u;
    if (blockIdx.x + 1 == gridDim.x && threadIdx.x == 0)
    {
        const unsigned long long all = first + total;
        *total_out = all;
        if (note.slot != nullptr)
        {
            note.slot[0] = all;
            note.slot[1] = note.extra != nullptr ? *note.extra : 0ull;
            __hip_atomic_store(note.slot + 2, note.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
    write_children(stage, key, mask, mine & 4095u, total, first, children, ~uint64_t(0), child_step, scenes,
                   mark_leaves);
}

// Lanes per parent and child of the kernel for the smallest levels, 0: too many wavefronts for it.
static int32_t
child_lanes(uint32_t n, int32_t max_cameras)
{
    int32_t G = 8;
    while (G < max_cameras && G < 64)
        G *= 2;
    return uint64_t(n) * uint64_t(G) / 8u <= kChildWaves ? G : 0;
}

bool
carve_culls(const SceneDev* scenes, size_t n, int32_t step)
{
    return std::any_of(scenes, scenes + n, [&](const SceneDev& s) {
        const int32_t li = step - s.start;
        return li < s.level && cull_level(s, li);
    });
}

int32_t
launch_carve_classify(const uint64_t* parents,
                      uint32_t n,
                      int32_t level_i,
                      const SceneDev* scenes,
                      uint8_t* child_mask,
                      uint32_t* block_counts,
                      unsigned long long* tests,
                      const CarveTuning& tune,
                      int32_t max_cameras,
                      bool culls,
                      hipStream_t st,
                      const unsigned long long* dev_n,
                      int32_t split_hint,
                      uint32_t* cursors,
                      bool counts)
{
    if (n == 0)
        return 0;
    int32_t split = dev_n != nullptr ? split_hint : carve_split_factor(n, tune);
    if (split == kChildSplit)
        split = 64; // a plan's hint, from the level that its capacity rounds up
    const int32_t G = split == 64 ? child_lanes(n, max_cameras) : 0;
    // fewer lanes when they still hold a parent's cameras in one round: the others would idle (8197 parents of 8
    // cameras: 64 lanes 38 us, 16 15; 7421 of 10: 38, 21)
    if (split == 64 && G == 0 && max_cameras <= 16)
        split = 16;
    if (split == 16 && max_cameras <= 4)
        split = 4;
    const uint64_t nb = blocks_for(n, kCarveThreads);
    if (dev_n != nullptr && split == 1)
    {
        // persistent workgroups: as many as the CUs hold at the kernel's occupancy (3 per CU), a multiple
        // of 8 so that every XCD's queue is served
        const uint64_t grid = std::max<uint64_t>(8, std::min<uint64_t>(768, (nb + 7) / 8 * 8));
        const auto kernel = culls ? carve_classify_queue_kernel<true> : carve_classify_queue_kernel<false>;
        kernel<<<unsigned(grid), kCarveThreads, 0, st>>>(parents, dev_n, n, level_i, scenes, child_mask, block_counts,
                                                         tests, cursors);
        THULL_LAUNCH_CHECK();
        return split;
    }
    if (split == 1)
    {
        const auto kernel = culls ? carve_classify_kernel<true> : carve_classify_kernel<false>;
        kernel<<<nb, kCarveThreads, 0, st>>>(parents, n, level_i, scenes, child_mask, block_counts, tests);
        THULL_LAUNCH_CHECK();
        return split;
    }
    if (G > 0)
        carve_classify_child_kernel<<<blocks_for(n, 64 / G), kChildThreads, 0, st>>>(parents, n, level_i, scenes, G,
                                                                                     child_mask, tests, dev_n);
    else
    {
        const auto kernel = split == 64  ? carve_classify_split_kernel<64, false>
                            : split == 16 ? carve_classify_split_kernel<16, false>
                            : split == 4  ? (culls ? carve_classify_split_kernel<4, true>
                                                   : carve_classify_split_kernel<4, false>)
                                          : (culls ? carve_classify_split_kernel<2, true>
                                                   : carve_classify_split_kernel<2, false>);
        kernel<<<blocks_for(int64_t(n) * split, 256), 256, 0, st>>>(parents, n, level_i, scenes, child_mask, tests,
                                                                    dev_n);
    }
    THULL_LAUNCH_CHECK();
    if (counts)
    {
        carve_count_kernel<<<nb, kCarveThreads, 0, st>>>(child_mask, n, block_counts, dev_n);
        THULL_LAUNCH_CHECK();
    }
    return G > 0 ? kChildSplit : split;
}

int32_t
carve_split_factor(uint32_t n, const CarveTuning& tune)
{
    // small levels split each parent's cameras over G lanes to fill the chip
    int32_t g = 1;
    if (n <= tune.max_parents[0])
        g = 64;
    else if (n <= tune.max_parents[1])
        g = 16;
    else if (n <= tune.max_parents[2])
        g = 4;
    else if (n <= tune.max_parents[3])
        g = 2;
    // the split kernel numbers its lanes n * G with 32-bit thread ids: thresholds set high enough to
    // pass that bound fall back to fewer lanes per parent (the results do not depend on G)
    while (g > 1 && uint64_t(n) * uint64_t(g) >= (uint64_t(1) << 31))
        g = g == 64 ? 16 : (g == 16 ? 4 : (g == 4 ? 2 : 1));
    return g;
}

void
launch_carve_scatter(const uint64_t* parents,
                     uint32_t n,
                     const uint8_t* child_mask,
                     const uint32_t* block_offsets,
                     uint64_t* children,
                     int32_t child_step,
                     const SceneDev* scenes,
                     bool mark_leaves,
                     hipStream_t st,
                     const unsigned long long* dev_n,
                     uint64_t out_cap)
{
    if (n == 0)
        return;
    carve_scatter_kernel<<<blocks_for(n, kCarveThreads), kCarveThreads, 0, st>>>(
            parents, n, child_mask, block_offsets, children, child_step, scenes, mark_leaves, dev_n, out_cap);
    THULL_LAUNCH_CHECK();
}

void
launch_carve_compact(const uint64_t* parents, uint32_t n, const uint8_t* child_mask, uint64_t* children,
                     int32_t child_step, const SceneDev* scenes, bool mark_leaves, unsigned long long* total,
                     const ScanNotify& note, hipStream_t st)
{
    THULL_CHECK(n > 0 && n <= kCompactParents, "level size of a one-launch compaction");
    carve_compact_kernel<<<blocks_for(n, kCarveThreads), kCarveThreads, 0, st>>>(
            parents, n, child_mask, children, child_step, scenes, mark_leaves, total, note);
    THULL_LAUNCH_CHECK();
}

// ===========================================================================
// Corner vertices (VH:770-825)
//
// Instead of sorting the 8 corner ids of every leaf and removing duplicates,
// the corners are set in a bitmap of the (R+1)^3 grid whose rows are padded
// to whole 32-bit words.  The bitmap order is the (z, y, x) order of the
// reference's sorted ravel ids, so a popcount prefix over the words yields the
// sorted unique vertex list directly, and also serves as the rank dictionary
// (vertex -> list position) of marching cubes.
// ===========================================================================

// Leaf cells of the scenes whose target level is `level`: the children that
// carving step level-1 kept, read from the parents' child masks.  A parent
// owns a 2x2 block of bits in four cell rows, and both bits of a row sit in
// one word (2 px is even), so it issues at most four atomics.
// Level-0 scenes: the root cell is the only leaf.
__global__ void
mark_root_cells_kernel(const SceneDev* __restrict__ scenes, int32_t first, int32_t nscenes)
{
    const int32_t s = first + int32_t(blockIdx.x * 256 + threadIdx.x);
    if (s < first + nscenes && scenes[s].level == 0)
        scenes[s].cells[0] = 1u;
}

// Vertex bitmap = leaf cells dilated by {0,1}^3: vertex (x, y, z) is a corner
// of cell (x - dx, y - dy, z - dz).  One thread per vertex word, no atomics.
// The reads of a word (the words xw and xw - 1 of 4 cell rows) are issued
// unconditionally, out-of-range ones from word 0 with their result masked, so
// that the reads of several words are in flight together.
struct DilateReads
{
    uint32_t c[4] = { 0u, 0u, 0u, 0u }; // cell words xw of rows (dy, dz), r = dy + 2 dz (0 when out of range)
    uint32_t p[4] = { 0u, 0u, 0u, 0u }; // words xw - 1 of the same rows, read by lane 0 of a wave only
    bool first_in_row = true;           // xw == 0: no word xw - 1
};

// Position of a vertex word in its scene's bitmap: word xw of row y + z (R + 1)
// (rows of row_words words, R + 1 rows per plane).  Walking a thread's words
// (a fixed stride apart) moves the position by a fixed (rows, words) step, so
// only the first word of a scene needs divisions.
struct WordPos
{
    uint32_t xw, y, z;
};

__device__ __forceinline__ WordPos
word_pos(const SceneDev& s, uint64_t local)
{
    const uint32_t R1 = (1u << s.level) + 1u;
    const uint64_t row = div_u64_u32(local, s.row_words);
    WordPos q;
    q.xw = uint32_t(local - row * s.row_words);
    const uint64_t zq = div_u64_u32(row, R1);
    q.y = uint32_t(row - zq * R1);
    q.z = uint32_t(zq);
    return q;
}

// Issues the reads of word q (UNIFORM as for classify_scene: keeps the
// wave-uniform and per-lane copies apart).  The lanes of a wave hold
// consecutive words, so word xw - 1 of a row is the previous lane's word xw:
// only lane 0 reads it.
template <bool UNIFORM>
__device__ __forceinline__ void
dilate_issue(const SceneDev& s, const WordPos& q, bool lane0, DilateReads& d)
{
    const int32_t R = int32_t(1) << s.level;
    const uint32_t rwc = s.cell_row_words;
    const uint32_t* plane = s.cells; // a scene's cell bitmap holds fewer than 2^32 words
    d.first_in_row = q.xw == 0u;
#pragma unroll
    for (int r = 0; r < 4; ++r)
    {
        const int32_t cz = int32_t(q.z) - (r >> 1), cy = int32_t(q.y) - (r & 1);
        const bool rowok = cz >= 0 && cz < R && cy >= 0 && cy < R;
        const uint32_t base = (uint32_t(cz) * uint32_t(R) + uint32_t(cy)) * rwc;
        d.c[r] = (rowok && q.xw < rwc) ? plane[base + q.xw] : 0u;
        if (lane0)
            d.p[r] = (rowok && q.xw > 0 && q.xw - 1 < rwc) ? plane[base + q.xw - 1] : 0u;
    }
}

// Every lane of the wave calls this (cross-lane reads).
__device__ __forceinline__ uint32_t
dilate_combine(const DilateReads& d, bool lane0)
{
    uint32_t out = 0u;
#pragma unroll
    for (int r = 0; r < 4; ++r)
    {
        const uint32_t prev = uint32_t(__shfl_up(int(d.c[r]), 1, 64));
        const uint32_t pw = d.first_in_row ? 0u : (lane0 ? d.p[r] : prev);
        out |= d.c[r] | (d.c[r] << 1) | (pw >> 31);
    }
    return out;
}

// Each block covers a tile of 256 ITEMS consecutive words, each thread one word per
// 256, in batches of up to 4 words whose reads are in flight together.  The block
// also sums the popcounts of its words: the first pass of the exclusive scan
// that numbers the vertices.  Small bitmaps take 2 words per thread, so that there
// are blocks for the chip (dilation + numbering, us, with 16 -> 2: level 7, 84 000
// words, 16 + 20 -> 5 + 6; level 9, 4.5 million, 26 + 32 -> 24 + 22; level 10, 36
// million, 122 + 139 -> 161 + 158).
constexpr int kVertexItems = 2;
constexpr uint64_t kSmallTileWords = uint64_t(1) << 23;

template <int ITEMS>
__global__ __launch_bounds__(kScanThreads) void
dilate_cells_kernel(uint32_t* __restrict__ verts,
                    uint64_t nwords,
                    const uint64_t* __restrict__ scene_word_begin,
                    const SceneDev* __restrict__ scenes,
                    int32_t nscenes,
                    uint32_t* __restrict__ block_sums)
{
    constexpr int kBatch = ITEMS < 4 ? ITEMS : 4;
    __shared__ uint32_t lds[kScanThreads / 64];
    const uint64_t w0 = uint64_t(blockIdx.x) * (kScanThreads * ITEMS) + threadIdx.x;
    const bool lane0 = (threadIdx.x & 63) == 0;
    const auto begin = [&](int32_t i) { return scene_word_begin[i]; };
    // all lanes take part in the lookup ballot before any diverge
    int32_t lo = find_segment_rising(begin, nscenes, w0);
    // first word of scene lo + 1, kept in a register (the scan of scene boundaries reads memory only
    // when a thread's words enter the next scene)
    uint64_t next_begin = lo + 1 < nscenes ? begin(lo + 1) : ~uint64_t(0);
    int32_t at = -1;           // scene of the position below
    WordPos q{ 0u, 0u, 0u };   // position of the previous word of this thread in scene `at`
    uint32_t step_w = 0u, step_r = 0u, R1 = 0u, rw = 0u;
    uint32_t count = 0u;
    for (int k0 = 0; k0 < ITEMS; k0 += kBatch)
    {
        DilateReads d[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; ++u)
        {
            const uint64_t w = w0 + uint64_t(k0 + u) * kScanThreads;
            if (w < nwords)
            {
                while (w >= next_begin)
                {
                    ++lo;
                    next_begin = lo + 1 < nscenes ? begin(lo + 1) : ~uint64_t(0);
                }
                const SceneDev& sd = scenes[lo];
                if (lo != at)
                {
                    // first word of this thread in the scene: divisions, and the per-stride step
                    q = word_pos(sd, w - begin(lo));
                    at = lo;
                    rw = sd.row_words;
                    R1 = (1u << sd.level) + 1u;
                    step_r = uint32_t(kScanThreads) / rw;
                    step_w = uint32_t(kScanThreads) - step_r * rw;
                }
                else
                {
                    q.xw += step_w;
                    uint32_t dr = step_r;
                    if (q.xw >= rw)
                    {
                        q.xw -= rw;
                        ++dr;
                    }
                    q.y += dr;
                    if (dr < R1)
                    {
                        if (q.y >= R1)
                        {
                            q.y -= R1;
                            ++q.z;
                        }
                    }
                    else
                        q = word_pos(sd, w - begin(lo)); // tiny grids: more rows per stride than per plane
                }
                const int32_t l0 = __builtin_amdgcn_readfirstlane(lo);
                if (__all(lo == l0))
                    dilate_issue<true>(wave_uniform(scenes[l0]), q, lane0, d[u]);
                else
                    dilate_issue<false>(sd, q, lane0, d[u]);
            }
        }
#pragma unroll
        for (int u = 0; u < kBatch; ++u)
        {
            const uint64_t w = w0 + uint64_t(k0 + u) * kScanThreads;
            const uint32_t out = dilate_combine(d[u], lane0); // all lanes: cross-lane reads
            if (w < nwords)
            {
                verts[w] = out;
                count += __popc(out);
            }
        }
    }
    uint32_t total;
    block_exclusive_sum(count, lds, total);
    if (threadIdx.x == 0)
        block_sums[blockIdx.x] = total;
}

void
launch_mark_root_cells(const SceneDev* scenes, int32_t first, int32_t nscenes, hipStream_t st)
{
    if (nscenes <= 0)
        return;
    mark_root_cells_kernel<<<blocks_for(nscenes, 256), 256, 0, st>>>(scenes, first, nscenes);
    THULL_LAUNCH_CHECK();
}

void
launch_dilate_cells(uint32_t* verts, uint64_t nwords, const uint64_t* scene_word_begin, const SceneDev* scenes,
                    int32_t nscenes, uint32_t* block_sums, hipStream_t st)
{
    if (nwords == 0)
        return;
    const auto kernel = nwords <= kSmallTileWords ? dilate_cells_kernel<kVertexItems> : dilate_cells_kernel<kScanItems>;
    kernel<<<vertex_tiles(nwords), kScanThreads, 0, st>>>(verts, nwords, scene_word_begin, scenes, nscenes, block_sums);
    THULL_LAUNCH_CHECK();
}

uint32_t
vertex_tiles(uint64_t nwords)
{
    const uint64_t tile = nwords <= kSmallTileWords ? kScanThreads * kVertexItems : kScanTile;
    return uint32_t((nwords + tile - 1) / tile);
}

// Second pass of the vertex numbering fused with the vertex extraction.  Wave
// w of a block takes the block's words [w * 64 ITEMS, (w + 1) * 64 ITEMS) in ITEMS
// steps of 64 consecutive words (one per lane, coalesced); a wave prefix sum of
// the popcounts plus a running total turn the block offsets of the dilation
// pass into the exclusive prefix of every word (stored for the marching-cubes
// rank lookups), and each set bit's packed key is written at prefix[word] +
// rank, i.e. in bitmap order = per scene (z, y, x) order; adjacent lanes write
// adjacent keys.
template <int ITEMS>
__global__ __launch_bounds__(kScanThreads) void
prefix_extract_kernel(const uint32_t* __restrict__ bitmap,
                      uint64_t nwords,
                      const uint32_t* __restrict__ block_offsets,
                      const uint64_t* __restrict__ scene_word_begin,
                      const SceneDev* __restrict__ scenes,
                      int32_t nscenes,
                      uint32_t* __restrict__ prefix,
                      uint64_t* __restrict__ vertices)
{
    constexpr int kSteps = ITEMS, kWaveWords = 64 * ITEMS;
    __shared__ uint32_t wave_total[kScanThreads / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint64_t wbase = uint64_t(blockIdx.x) * (kScanThreads * ITEMS) + uint64_t(wave) * kWaveWords;
    uint32_t v[kSteps];
    uint32_t total = 0;
#pragma unroll
    for (int k = 0; k < kSteps; ++k)
    {
        const uint64_t w = wbase + 64 * k + lane;
        v[k] = w < nwords ? bitmap[w] : 0u;
        total += __popc(v[k]);
    }
    // wave total, then the offsets of the waves before this one
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1)
        total += __shfl_xor(total, d, 64);
    if (lane == 0)
        wave_total[wave] = total;
    __syncthreads();
    uint32_t run = block_offsets[blockIdx.x];
    for (int q = 0; q < wave; ++q)
        run += wave_total[q];
    const auto begin = [&](int32_t i) { return scene_word_begin[i]; };
    int32_t lo = find_segment_rising(begin, nscenes, wbase + lane);
    // the scene's first word, the next scene's first word and the scene's row geometry, kept in
    // registers: memory is read only when a thread's words enter another scene
    uint64_t cur_begin = begin(lo), next_begin = lo + 1 < nscenes ? begin(lo + 1) : ~uint64_t(0);
    int32_t at = -1;
    uint32_t rw = 1u, R1 = 1u;
#pragma unroll
    for (int k = 0; k < kSteps; ++k)
    {
        const uint64_t w = wbase + 64 * k + lane;
        const uint32_t c = __popc(v[k]);
        const uint32_t inc = wave_inclusive_sum(c);
        const uint32_t pos = run + inc - c;
        run += __shfl(inc, 63, 64);
        if (w >= nwords)
            continue;
        prefix[w] = pos;
        while (w >= next_begin)
        {
            ++lo;
            cur_begin = next_begin;
            next_begin = lo + 1 < nscenes ? begin(lo + 1) : ~uint64_t(0);
        }
        uint32_t word = v[k];
        if (word == 0u)
            continue;
        if (lo != at)
        {
            rw = scenes[lo].row_words;
            R1 = (1u << scenes[lo].level) + 1u;
            at = lo;
        }
        const uint64_t local = w - cur_begin;
        const uint64_t row = div_u64_u32(local, rw);
        const uint32_t xw = uint32_t(local - row * rw);
        const uint64_t zq = div_u64_u32(row, R1);
        const uint32_t y = uint32_t(row - zq * R1), z = uint32_t(zq);
        uint32_t o = pos;
        while (word != 0u)
        {
            const uint32_t bit = __builtin_ctz(word);
            vertices[o++] = pack_key(uint32_t(lo), xw * 32u + bit, y, z);
            word &= word - 1u;
        }
    }
}

void
launch_prefix_extract(const uint32_t* bitmap,
                      uint64_t nwords,
                      const uint32_t* block_offsets,
                      const uint64_t* scene_word_begin,
                      const SceneDev* scenes,
                      int32_t nscenes,
                      uint32_t* prefix,
                      uint64_t* vertices,
                      hipStream_t st)
{
    if (nwords == 0)
        return;
    const auto kernel =
            nwords <= kSmallTileWords ? prefix_extract_kernel<kVertexItems> : prefix_extract_kernel<kScanItems>;
    kernel<<<vertex_tiles(nwords), kScanThreads, 0, st>>>(bitmap, nwords, block_offsets, scene_word_begin, scenes,
                                                          nscenes, prefix, vertices);
    THULL_LAUNCH_CHECK();
}

// ===========================================================================
// Corner vertices by bricks
//
// In a large scene nearly all words of the bitmaps are empty (99 % at level 11), and the bricks of up to 8 x 8 x 8
// cells that the octree kept say where they are not.  A thread takes groups of 4 words (rows are padded to whole
// groups); only those that a kept brick can reach (a flag per group and 8 x 8 rows) are dilated, counted and
// numbered.  Lookups go from vertices of cells to their neighbours, so groups with such neighbours are zeroed; no
// other word of the vertex bitmap is written or read, and prefixes only hold in groups with vertices.
// Bound by VALU issue and the latency of short waves; a level-11 hull of 50 1080p cameras (71 M groups, 1.1 GB):
// dilation 0.94 -> 0.26 ms, prefixes and keys 0.99 -> 0.27.
// ===========================================================================

__device__ __forceinline__ bool
brick_of_list(const SceneDev& s, const BrickList& l)
{
    return s.bricks != nullptr && s.start + s.level - s.brick_shift == l.step;
}

__device__ __forceinline__ uint64_t
brick_bit(uint32_t x, uint32_t y, uint32_t z, int32_t level)
{
    return (((uint64_t(z) << level) + y) << level) + x;
}

__global__ __launch_bounds__(256) void
mark_bricks_kernel(const BrickList* __restrict__ lists, int32_t nlists, uint64_t total,
                   const SceneDev* __restrict__ scenes)
{
    const uint64_t i = uint64_t(blockIdx.x) * 256 + threadIdx.x;
    const int32_t q = find_segment_rising([&](int32_t k) { return lists[k].begin; }, nlists, i);
    if (i >= total)
        return;
    const BrickList l = lists[q];
    const uint64_t key = l.keys[i - l.begin];
    const SceneDev& s = scenes[key_scene(key)];
    if (!brick_of_list(s, l))
        return;
    const uint64_t bit = brick_bit(key_x(key), key_y(key), key_z(key), s.level - s.brick_shift);
    atomicOr(s.bricks + (bit >> 5), 1u << uint32_t(bit & 31u));
}

void
launch_mark_bricks(const BrickList* lists, int32_t nlists, uint64_t waves, const SceneDev* scenes, hipStream_t st)
{
    if (waves == 0)
        return;
    mark_bricks_kernel<<<blocks_for(int64_t(waves), 256), 256, 0, st>>>(lists, nlists, waves, scenes);
    THULL_LAUNCH_CHECK();
}

// A group of 4 vertex words of a scene, group q.x of row q.y of plane q.z.
struct WordGroup
{
    uint32_t x, y, z;
};

__device__ __forceinline__ WordGroup
word_group(const SceneDev& s, uint64_t g)
{
    const uint32_t R1 = (1u << s.level) + 1u, per = s.row_words / 4u;
    const uint64_t row = div_u64_u32(g, per), z = div_u64_u32(row, R1);
    return WordGroup{ uint32_t(g - row * per), uint32_t(row - z * R1), uint32_t(z) };
}

// The group `step` groups further on, rows = step / per and rest = step % per.
__device__ __forceinline__ void
next_group(const SceneDev& s, WordGroup& q, uint32_t rows, uint32_t rest)
{
    const uint32_t R1 = (1u << s.level) + 1u, per = s.row_words / 4u;
    q.x += rest;
    uint32_t up = rows;
    if (q.x >= per)
    {
        q.x -= per;
        ++up;
    }
    q.y += up;
    while (q.y >= R1)
    {
        q.y -= R1;
        ++q.z;
    }
}

// Rows of group flags along y and z: the vertices of 2^shift rows share a flag.
__device__ __forceinline__ uint32_t
flag_rows(const SceneDev& s)
{
    return (1u << (s.level - s.brick_shift)) + 1u;
}

// (The vertex bitmaps that fit the memory have fewer than 2^32 flags.)
__device__ __forceinline__ uint8_t
group_flag(const SceneDev& s, const WordGroup& q)
{
    const uint32_t i =
            ((q.z >> s.brick_shift) * flag_rows(s) + (q.y >> s.brick_shift)) * (s.row_words / 4u) + q.x;
    return as_global(s.group_flags)[i];
}

// Flags of the word groups (columns 128 x .. 128 x + 127 of 2^shift rows and planes): 2: a kept brick may hold a cell
// that touches a vertex of the group, 1: one that touches a vertex next to one of the group, 0: neither.
__global__ __launch_bounds__(256) void
group_flags_kernel(const SceneDev* __restrict__ scenes)
{
    const SceneDev s = wave_uniform(scenes[blockIdx.y]);
    if (s.bricks == nullptr)
        return;
    const int32_t sh = s.brick_shift, level = s.level - sh;
    const uint32_t n = flag_rows(s), per = s.row_words / 4u, nb = 1u << level;
    const uint64_t total = uint64_t(n) * n * per;
    for (uint64_t i = uint64_t(blockIdx.x) * 256 + threadIdx.x; i < total; i += uint64_t(gridDim.x) * 256)
    {
        const uint64_t row = div_u64_u32(i, per), bz = div_u64_u32(row, n);
        const uint32_t x0 = uint32_t(i - row * per) * 128u, by = uint32_t(row - bz * n);
        const uint32_t last = (1u << s.level) - 1u; // last cell of an axis
        // bricks of the cells x0 - 1 .. x0 + 127 and of x0 - 2 .. x0 + 128
        const uint32_t t0 = (max(x0, 1u) - 1u) >> sh, t1 = min(x0 + 127u, last) >> sh;
        const uint32_t w0 = (max(x0, 2u) - 2u) >> sh, w1 = min(x0 + 128u, last) >> sh;
        uint32_t flag = 0u;
        if (x0 <= last + 1u) // else padding
        {
            const uint64_t near = (uint64_t(2) << (w1 - w0)) - 1u; // at most 18 bricks
            const uint64_t own = ((uint64_t(2) << (t1 - t0)) - 1u) << (t0 - w0);
#pragma unroll
            for (int r = 0; r < 9; ++r)
            {
                const uint32_t y = by + uint32_t(r % 3 - 1), z = uint32_t(bz) + uint32_t(r / 3 - 1);
                if (y >= nb || z >= nb) // -1 wraps past nb
                    continue;
                const uint64_t bit = brick_bit(w0, y, z, level);
                const uint32_t b = uint32_t(bit & 31u);
                const auto w = as_global(s.bricks) + (bit >> 5);
                uint64_t v = w[0];
                if (b + w1 - w0 >= 32u)
                    v |= uint64_t(w[1]) << 32;
                v >>= b;
                if ((v & near) != 0u)
                    flag = max(flag, r % 3 < 2 && r / 3 < 2 && (v & own) != 0u ? 2u : 1u);
            }
        }
        as_global(s.group_flags)[i] = uint8_t(flag);
    }
}

// The group's words: leaf cells dilated by {0,1}^3, as in dilate_cells_kernel.
__device__ __forceinline__ uint4
dilate_group(const SceneDev& s, const WordGroup& q)
{
    const int32_t R = int32_t(1) << s.level;
    const uint32_t rwc = s.cell_row_words, xw = 4u * q.x;
    uint32_t out[4] = { 0u, 0u, 0u, 0u };
#pragma unroll
    for (int r = 0; r < 4; ++r)
    {
        const int32_t cz = int32_t(q.z) - (r >> 1), cy = int32_t(q.y) - (r & 1);
        if (cz < 0 || cz >= R || cy < 0 || cy >= R)
            continue;
        const uint32_t* row = s.cells + (uint64_t(cz) * uint32_t(R) + uint32_t(cy)) * rwc;
        uint32_t c[5] = { 0u, 0u, 0u, 0u, 0u }; // words xw - 1 .. xw + 3
        if (xw > 0u && xw <= rwc)
            c[0] = row[xw - 1u];
        if ((rwc & 3u) == 0u)
        {
            if (xw < rwc)
            {
                const uint4 v = *reinterpret_cast<const uint4*>(row + xw);
                c[1] = v.x;
                c[2] = v.y;
                c[3] = v.z;
                c[4] = v.w;
            }
        }
        else
        {
#pragma unroll
            for (uint32_t k = 0; k < 4u; ++k)
                if (xw + k < rwc)
                    c[k + 1] = row[xw + k];
        }
#pragma unroll
        for (int k = 0; k < 4; ++k)
            out[k] |= c[k + 1] | (c[k + 1] << 1) | (c[k] >> 31);
    }
    return make_uint4(out[0], out[1], out[2], out[3]);
}

constexpr int kTileGroups = kScanTile / 4;
constexpr int kGroupSteps = kTileGroups / kScanThreads; // groups per thread

// The scene of a tile's first word, and whether the whole tile lies in it.
__device__ __forceinline__ int32_t
tile_scene(const uint64_t* __restrict__ scene_word_begin, int32_t nscenes, uint64_t nwords, bool& one)
{
    const uint64_t w0 = uint64_t(blockIdx.x) * kScanTile;
    const int32_t q = find_segment_uniform([&](int32_t i) { return scene_word_begin[i]; }, nscenes, w0);
    one = q + 1 >= nscenes || scene_word_begin[q + 1] >= min(w0 + kScanTile, nwords);
    return q;
}

// First pass: vertex words, the popcount sum of each tile and per 64 groups the bits of those with vertices (and of
// every scene's first group), kTileGroups / 64 words per tile.  The flags of a thread's groups are loaded together.
__global__ __launch_bounds__(kScanThreads) void
dilate_groups_kernel(uint4* __restrict__ verts, uint64_t nwords, const uint64_t* __restrict__ scene_word_begin,
                     const SceneDev* __restrict__ scenes, int32_t nscenes, uint32_t* __restrict__ block_sums,
                     uint64_t* __restrict__ filled)
{
    __shared__ uint32_t lds[kScanThreads / 64];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    bool one;
    const int32_t q0 = tile_scene(scene_word_begin, nscenes, nwords, one);
    const uint64_t g0 = uint64_t(blockIdx.x) * kTileGroups + wave * (kTileGroups / 4) + lane;
    uint32_t count = 0u;
    uint64_t bits[kGroupSteps];
    const auto group = [&](const SceneDev& s, uint64_t g, const WordGroup& q, uint8_t flag) {
        const bool first = (q.x | q.y | q.z) == 0u;
        uint32_t c = 0u;
        if (flag != 0 || first)
        {
            uint4 v = make_uint4(0u, 0u, 0u, 0u);
            if (flag == 2)
                v = dilate_group(s, q);
            verts[g] = v;
            c = popc4(v);
        }
        count += c;
        return c != 0u || first;
    };
    if (one)
    {
        const SceneDev s = wave_uniform(scenes[q0]);
        const uint32_t per = s.row_words / 4u, rows = 64u / per, rest = 64u - rows * per;
        WordGroup q[kGroupSteps];
        uint8_t flag[kGroupSteps];
        q[0] = word_group(s, g0 - scene_word_begin[q0] / 4u);
#pragma unroll
        for (int k = 1; k < kGroupSteps; ++k)
        {
            q[k] = q[k - 1];
            next_group(s, q[k], rows, rest);
        }
#pragma unroll
        for (int k = 0; k < kGroupSteps; ++k)
            flag[k] = 4 * (g0 + uint32_t(64 * k)) < nwords ? group_flag(s, q[k]) : 0;
#pragma unroll
        for (int k = 0; k < kGroupSteps; ++k)
        {
            const uint64_t g = g0 + uint32_t(64 * k);
            bool any = false;
            if (4 * g < nwords)
                any = group(s, g, q[k], flag[k]);
            bits[k] = __ballot(any);
        }
    }
    else
    {
        int32_t q = q0;
#pragma unroll 1
        for (int k = 0; k < kGroupSteps; ++k)
        {
            const uint64_t g = g0 + uint32_t(64 * k);
            bool any = false;
            if (4 * g < nwords)
            {
                while (q + 1 < nscenes && scene_word_begin[q + 1] <= 4 * g)
                    ++q;
                const WordGroup at = word_group(scenes[q], g - scene_word_begin[q] / 4u);
                any = group(scenes[q], g, at, group_flag(scenes[q], at));
            }
            const uint64_t m = __ballot(any);
#pragma unroll
            for (int i = 0; i < kGroupSteps; ++i)
                bits[i] = i == k ? m : bits[i];
        }
    }
    if (lane == 0)
#pragma unroll
        for (int k = 0; k < kGroupSteps; ++k)
            filled[uint64_t(blockIdx.x) * (kTileGroups / 64) + wave * kGroupSteps + uint32_t(k)] = bits[k];
    uint32_t total;
    block_exclusive_sum(count, lds, total);
    if (threadIdx.x == 0)
        block_sums[blockIdx.x] = total;
}

// Second pass: prefixes and vertex keys of the groups of the first pass's bits.  Wavefront w takes the tile's groups
// [w * 256, w * 256 + 256) in steps of 64, as there.
__global__ __launch_bounds__(kScanThreads) void
extract_groups_kernel(const uint4* __restrict__ bitmap, const uint64_t* __restrict__ filled,
                      const uint32_t* __restrict__ block_offsets, const uint64_t* __restrict__ scene_word_begin,
                      const SceneDev* __restrict__ scenes, int32_t nscenes, uint4* __restrict__ prefix,
                      uint64_t* __restrict__ vertices)
{
    __shared__ uint32_t wave_total[kScanThreads / 64];
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)));
    const uint64_t g0 = uint64_t(blockIdx.x) * kTileGroups + wave * (kTileGroups / 4) + lane;
    const uint64_t* const fb = filled + uint64_t(blockIdx.x) * (kTileGroups / 64) + wave * kGroupSteps;
    uint64_t bits[kGroupSteps];
    uint4 v[kGroupSteps];
    uint32_t n = 0u;
#pragma unroll
    for (int k = 0; k < kGroupSteps; ++k)
        bits[k] = fb[k];
#pragma unroll
    for (int k = 0; k < kGroupSteps; ++k)
    {
        v[k] = make_uint4(0u, 0u, 0u, 0u);
        if ((bits[k] >> lane) & 1u)
            v[k] = bitmap[g0 + uint32_t(64 * k)];
    }
#pragma unroll
    for (int k = 0; k < kGroupSteps; ++k)
        n += popc4(v[k]);
    const uint32_t mine = __reduce_add_sync(0xffffffffffffffffull, n);
    if (lane == 0)
        wave_total[wave] = mine;
    __syncthreads();
    if ((bits[0] | bits[1] | bits[2] | bits[3]) == 0u)
        return;
    uint32_t run = block_offsets[blockIdx.x];
    for (uint32_t q = 0; q < wave; ++q)
        run += wave_total[q];
    // the scene of the wave's first group; most waves lie in one
    int32_t q0 = find_segment_uniform([&](int32_t i) { return scene_word_begin[i]; }, nscenes, 4u * (g0 - lane));
#pragma unroll
    for (int k = 0; k < kGroupSteps; ++k)
    {
        if (bits[k] == 0u)
            continue;
        const uint32_t c = popc4(v[k]), inc = wave_inclusive_sum(c);
        uint32_t pos = run + inc - c;
        run += uint32_t(__shfl(int(inc), 63, 64));
        if (((bits[k] >> lane) & 1u) == 0u)
            continue;
        const uint32_t w[4] = { v[k].x, v[k].y, v[k].z, v[k].w };
        uint32_t p[4];
#pragma unroll
        for (int q = 0; q < 4; ++q)
        {
            p[q] = pos;
            pos += uint32_t(__popc(w[q]));
        }
        const uint64_t g = g0 + uint32_t(64 * k);
        prefix[g] = make_uint4(p[0], p[1], p[2], p[3]);
        int32_t scene = q0;
        while (scene + 1 < nscenes && scene_word_begin[scene + 1] <= 4 * g)
            ++scene;
        const WordGroup at = word_group(scenes[scene], g - scene_word_begin[scene] / 4u);
#pragma unroll
        for (int q = 0; q < 4; ++q)
        {
            uint32_t o = p[q];
            for (uint32_t m = w[q]; m != 0u; m &= m - 1u)
                vertices[o++] = pack_key(uint32_t(scene), 128u * at.x + 32u * uint32_t(q) + uint32_t(__builtin_ctz(m)),
                                         at.y, at.z);
        }
    }
}

uint64_t
filled_words(uint64_t nwords)
{
    return uint64_t(scan_blocks(nwords)) * (kTileGroups / 64);
}

uint64_t
group_flag_bytes(int32_t level, int32_t brick_shift, uint32_t row_words)
{
    const uint64_t n = (uint64_t(1) << (level - brick_shift)) + 1;
    return n * n * (row_words / 4u);
}

void
launch_group_flags(const SceneDev* scenes, int32_t nscenes, uint64_t most, hipStream_t st)
{
    constexpr int32_t kMostScenes = 32768; // of one grid
    for (int32_t s = 0; s < nscenes; s += kMostScenes)
    {
        const dim3 grid(unsigned(std::min<uint64_t>((most + 255) / 256, 2048)),
                        unsigned(std::min(nscenes - s, kMostScenes)));
        group_flags_kernel<<<grid, 256, 0, st>>>(scenes + s);
        THULL_LAUNCH_CHECK();
    }
}

void
launch_dilate_groups(uint32_t* verts, uint64_t nwords, const uint64_t* scene_word_begin, const SceneDev* scenes,
                     int32_t nscenes, uint32_t* block_sums, uint64_t* filled, hipStream_t st)
{
    if (nwords == 0)
        return;
    dilate_groups_kernel<<<scan_blocks(nwords), kScanThreads, 0, st>>>(
            reinterpret_cast<uint4*>(verts), nwords, scene_word_begin, scenes, nscenes, block_sums, filled);
    THULL_LAUNCH_CHECK();
}

void
launch_extract_groups(const uint32_t* bitmap, uint64_t nwords, const uint64_t* filled,
                      const uint32_t* block_offsets, const uint64_t* scene_word_begin, const SceneDev* scenes,
                      int32_t nscenes, uint32_t* prefix, uint64_t* vertices, hipStream_t st)
{
    if (nwords == 0)
        return;
    extract_groups_kernel<<<scan_blocks(nwords), kScanThreads, 0, st>>>(
            reinterpret_cast<const uint4*>(bitmap), filled, block_offsets, scene_word_begin, scenes, nscenes,
            reinterpret_cast<uint4*>(prefix), vertices);
    THULL_LAUNCH_CHECK();
}

// ===========================================================================
// Self-test of the division shortcuts against the IEEE division on random
// operands in (and at the edges of) their fast ranges and beyond them, and of
// clamp_round against clamp(roundf(v)) on rounding boundaries and special values.
// ===========================================================================

__device__ __forceinline__ uint32_t
mix32(uint64_t x)
{
    x ^= x >> 33;
    x *= 0xff51afd7ed558ccdull;
    x ^= x >> 33;
    x *= 0xc4ceb9fe1a85ec53ull;
    x ^= x >> 33;
    return uint32_t(x);
}

__device__ __forceinline__ float
test_operand(uint64_t key)
{
    const uint32_t r = mix32(key), m = mix32(key ^ 0x9e3779b97f4a7c15ull);
    // exponents -44..43 (the fast range is 2^-40 .. 2^40), mantissas random, all ones or zero
    const int32_t e = int32_t(r % 88u) - 44;
    const uint32_t mant = (m & 3u) == 0u ? 0x7fffffu : (m & 3u) == 1u ? 0u : (m >> 9);
    return __uint_as_float(((r >> 31) << 31) | (uint32_t(e + 127) << 23) | mant);
}

// A numerator for the carving check: one in four is tiny (2^-149 .. 2^-60,
// subnormals included) or zero, the others as test_operand.
__device__ __forceinline__ float
test_numerator(uint64_t key)
{
    const uint32_t r = mix32(key ^ 0x5851f42d4c957f2dull);
    if ((r & 3u) != 0u)
        return test_operand(key);
    const uint32_t m = mix32(key ^ 0x14057b7ef767814full);
    const uint32_t bits = ((r >> 2) % 90u == 0u) ? 0u : (m % 0x21800000u); // 0x21800000 = 2^-60
    return __uint_as_float(((r >> 31) << 31) | bits);
}

// The reference's window bound: clamp(int64(roundf(v)), 0, hi).
__device__ __forceinline__ int32_t
clamp_round_ref(float v, float hi)
{
    const float r = roundf(v);
    if (r != r)
        return 0;
    return int32_t(fminf(fmaxf(r, 0.0f), hi));
}

__global__ __launch_bounds__(256) void
div2_check_kernel(uint64_t count, uint64_t seed, unsigned long long* mismatches)
{
    const uint64_t i = uint64_t(blockIdx.x) * 256 + threadIdx.x;
    uint32_t bad = 0u;
    if (i < count)
    {
        const uint64_t k = seed * 0x100000001b3ull + 3 * i;
        const float nx = test_operand(k), ny = test_operand(k + 1), d = test_operand(k + 2);
        float qx, qy;
        div2_shared(nx, ny, d, qx, qy);
        const float rx = nx / d, ry = ny / d;
        bad = (__float_as_uint(qx) != __float_as_uint(rx) ? 1u : 0u) + (__float_as_uint(qy) != __float_as_uint(ry) ? 1u : 0u);

        // carving: operands with a carve_div_in_range denominator give the pixel coordinates of the
        // IEEE quotients in both conventions, tiny and zero numerators included
        const float tx = test_numerator(k), ty = test_numerator(k + 1);
        if (carve_div_in_range(max_abs3_nan(tx, ty, d), fabsf(d)))
        {
            float cx, cy;
            div2_unchecked(tx, ty, d, cx, cy);
            const float ex = tx / d, ey = ty / d;
            const float fW = float(1u + mix32(k ^ 7u) % 4096u);
            bad += __float_as_uint(to_pixel<true>(cx, fW)) != __float_as_uint(to_pixel<true>(ex, fW)) ? 1u : 0u;
            bad += __float_as_uint(to_pixel<true>(cy, fW)) != __float_as_uint(to_pixel<true>(ey, fW)) ? 1u : 0u;
            bad += __float_as_uint(to_pixel<false>(cx, fW)) != __float_as_uint(to_pixel<false>(ex, fW)) ? 1u : 0u;
            bad += __float_as_uint(to_pixel<false>(cy, fW)) != __float_as_uint(to_pixel<false>(ey, fW)) ? 1u : 0u;
        }

        // clamp_round on quarter steps around the rounding boundaries, one ulp either side, and
        // specials (NaN, infinities, signed zeros, huge values)
        const uint32_t c = mix32(k ^ 0xabcdefull);
        const float hi = float(c % 3000u);
        float v = float(int32_t(c >> 12) % 8200 - 4100) * 0.25f;
        if ((c & 0x30u) != 0u && v != 0.0f) // one ulp away from zero or towards it
            v = __uint_as_float(__float_as_uint(v) + ((c & 0x30u) == 0x10u ? 1u : 0xffffffffu));
        switch (c & 0xf00u)
        {
        case 0x100u: v = __uint_as_float(0x7fc00000u); break;
        case 0x200u: v = INFINITY; break;
        case 0x300u: v = -INFINITY; break;
        case 0x400u: v = -0.0f; break;
        case 0x500u: v = 3.0e38f; break;
        case 0x600u: v = -3.0e38f; break;
        default: break;
        }
        bad += clamp_round(v, hi) != clamp_round_ref(v, hi) ? 1u : 0u;

        // every float of [0, 2^23] (every value the clamp of clamp_round can pass on, for any image
        // size): its rounding instruction against roundf, and the lower clamp test of child_window
        // for m = +-u
        for (uint64_t bits = i; bits <= 0x4b000000ull; bits += count)
        {
            const float u = __uint_as_float(uint32_t(bits));
            bad += clamp_round(u, 8388607.0f) != clamp_round_ref(u, 8388607.0f) ? 1u : 0u;
            bad += (u + -0.5f > -0.5f) != (u > kMinAboveHalf) ? 1u : 0u;
            bad += (-u + -0.5f > -0.5f) != (-u > kMinAboveHalf) ? 1u : 0u;
        }
    }
    bad = __reduce_add_sync(0xffffffffffffffffull, bad);
    if ((threadIdx.x & 63) == 0 && bad != 0u)
        atomicAdd(mismatches, (unsigned long long)bad);
}

void
launch_div2_check(uint64_t count, uint64_t seed, unsigned long long* mismatches, hipStream_t st)
{
    if (count == 0)
        return;
    div2_check_kernel<<<blocks_for(int64_t(count), 256), 256, 0, st>>>(count, seed, mismatches);
    THULL_LAUNCH_CHECK();
}

// ===========================================================================
// Field (VH:419-520, camera loop VH:847)
//
// The reference launches one kernel per camera, each re-reading and
// re-writing the value array.  Here one thread owns a vertex and multiplies
// the camera samples in camera order 0..B-1 in a register, which gives the
// same float product.
// ===========================================================================

// Bilinear sample of one camera's mask at the projection of a world point
// (VH:470-530, IU:162-214): the four reads are issued by field_sample and
// combined by field_factor, so that the reads of several cameras are in
// flight together.  `skip`: a partial-mask camera that does not see the point
// well (VH:513-518) leaves the product unchanged.
// PAIR (images at least 2 columns wide): each of the two rows is read as one pair of
// adjacent columns.  The loaded values are only combined in field_factor, after the reads
// of all cameras in flight have been issued.
template <typename T>
struct FieldSample
{
    typedef T pair_t __attribute__((ext_vector_type(2), aligned(sizeof(T))));
    pair_t p0, p1; // two adjacent columns of rows y0 and y1
    float ty, tx;
    bool i00, i10, i01, i11;
    bool first0, first1; // column x0 (x0 + 1) is the pair's first element
    bool skip;
};

// Row (or column) y0 = int64(roundf(p - 0.5)) of the bilinear sample at pixel coordinate p
// (IU:162-214), as a float clamped to [-2, 2^30].  For p in [0.25, 2^23), p - 0.5 is exact and
// roundf (halves away from zero) of it is floor(p), which the clamp leaves unchanged; this is the
// path of every in-image sample.  Elsewhere the value is carried as a float clamped to
// [-2, 2^30], which changes neither the rows it selects nor ty = p - y0: a value the clamp moves
// (or the reference's saturation would) leaves all four samples outside the image, and such a
// factor is +0 for full masks (lerps of zeros with any finite weight; an infinite p gives NaN
// either way) and never taken for partial masks (only cameras that see the point inside the image
// count); a NaN p gives a NaN weight either way.
__device__ __forceinline__ void
sample_rows(float px, float py, float& fx, float& fy)
{
    if (__builtin_elementwise_minimum(px, py) >= 0.25f && __builtin_elementwise_maximum(px, py) < 0x1p23f)
    {
        fy = floorf(py);
        fx = floorf(px);
    }
    else
    {
        fy = fminf(fmaxf(roundf(py + -0.5f), -2.0f), 1073741824.0f);
        fx = fminf(fmaxf(roundf(px + -0.5f), -2.0f), 1073741824.0f);
    }
}

// PARTIAL: the scene's masks are partial.  OFF32: the camera's mask plane holds fewer than 2^31
// bytes and a row fewer than 2^24, so the reads take 32-bit byte offsets (24-bit row products)
// from the plane base (scalar when the plane is).
template <typename T, bool PAIR, bool PARTIAL, bool OFF32>
__device__ __forceinline__ void
field_sample(const SceneDev& s, int32_t b, float wx, float wy, float wz, FieldSample<T>& f)
{
    const auto T4 = as_global(s.transforms + 16 * b);
    const float fH = float(s.H), fW = float(s.W);
    const float cx = fmaf(T4[0], wx, fmaf(T4[1], wy, fmaf(T4[2], wz, T4[3])));
    const float cy = fmaf(T4[4], wx, fmaf(T4[5], wy, fmaf(T4[6], wz, T4[7])));
    float px, py;
    if (s.opengl != 0)
    {
        const float cw = fmaf(T4[12], wx, fmaf(T4[13], wy, fmaf(T4[14], wz, T4[15])));
        float qx, qy;
        div2_shared(cx, cy, cw, qx, qy); // cx / cw, cy / cw
        px = unnormalize_ndc(qx, fW);
        py = unnormalize_ndc(qy, fH);
    }
    else
    {
        const float cz = fmaf(T4[8], wx, fmaf(T4[9], wy, fmaf(T4[10], wz, T4[11])));
        float qx, qy;
        div2_shared(cx, cy, cz, qx, qy); // cx / cz, cy / cz
        px = qx - 0.5f;
        py = qy - 0.5f;
    }
    f.skip = false;
    if constexpr (PARTIAL)
    {
        // VH:513-518: only cameras whose rounded pixel lies inside with margin 1;
        // 1 <= roundf(p) <= n - 2  <=>  0.5 <= p < n - 1.5 (roundf rounds halves up for p >= 0)
        f.skip = !((px >= 0.5f) & (px < float(s.W) - 1.5f) & (py >= 0.5f) & (py < float(s.H) - 1.5f));
    }
    float fx, fy;
    sample_rows(px, py, fx, fy);
    // rows / columns as unsigned integers: -1 wraps to 2^32 - 1, so y0 in [0, H) <=> iy < H and
    // y0 + 1 in [0, H) <=> iy + 1 < H (the range tests are exact in float for integral values and
    // H, W < 2^24)
    const uint32_t H = uint32_t(s.H), W = uint32_t(s.W);
    const uint32_t iy = uint32_t(int32_t(fy));
    const uint32_t ix = uint32_t(int32_t(fx));
    const bool y0in = iy < H, y1in = iy + 1u < H;
    const bool x0in = ix < W, x1in = ix + 1u < W;
    f.i00 = y0in && x0in;
    f.i10 = y1in && x0in;
    f.i01 = y0in && x1in;
    f.i11 = y1in && x1in;
    // in-plane offsets (H * W < 2^31); a sample outside the image reads an element inside and is
    // replaced by padding
    typedef __attribute__((address_space(1))) const T global_t;
    global_t* M = (global_t*)(static_cast<const T*>(s.masks) + int64_t(b) * s.H * s.W);
    if constexpr (PAIR)
    {
        // columns ix and ix + 1 of a row are read as one pair (one load of 2 elements, element
        // alignment) starting at column xa = clamp(ix, 0, W - 2): for ix in [0, W - 2] the pair is
        // (ix, ix + 1); ix = W - 1 is the pair's second element, ix = -1 makes ix + 1 = 0 its first.
        // Rows outside the image read row 0.
        typedef __attribute__((address_space(1))) const typename FieldSample<T>::pair_t global_pair_t;
        const uint32_t xa = uint32_t(min(max(int32_t(ix), 0), int32_t(W) - 2));
        if constexpr (OFF32)
        {
            // byte offsets: each row's pair from its own 24-bit multiply-add r * pitch + xb, which is
            // meaningless, and unused, when row r is outside (the multiply reads the low 24 bits of
            // r, so iy = -1 is 2^24 - 1 there: row iy + 1 = 0 cannot be derived from row iy's
            // product); rows outside read row 0
            const auto G = (gptr<const char>)M;
            const uint32_t pitch = W * uint32_t(sizeof(T)), xb = xa * uint32_t(sizeof(T));
            uint32_t r0, r1; // one v_mad_u32_u24 each, which hipcc does not select here by itself (it
                             // takes a 64-bit multiply-add)
            asm("v_mad_u32_u24 %0, %1, %2, %3" : "=v"(r0) : "v"(iy), "v"(pitch), "v"(xb));
            asm("v_mad_u32_u24 %0, %1, %2, %3" : "=v"(r1) : "v"(iy + 1u), "v"(pitch), "v"(xb));
            f.p0 = *(global_pair_t*)(G + (y0in ? r0 : xb));
            f.p1 = *(global_pair_t*)(G + (y1in ? r1 : xb));
        }
        else
        {
            const uint32_t ra = y0in ? iy : 0u, rb = y1in ? iy + 1u : 0u;
            f.p0 = *(global_pair_t*)(M + (ra * W + xa));
            f.p1 = *(global_pair_t*)(M + (rb * W + xa));
        }
        f.first0 = ix == xa;
        f.first1 = ix + 1u == xa;
    }
    else
    {
        const uint32_t o00 = iy * W + ix;
        f.p0.x = M[f.i00 ? o00 : 0u];
        f.p0.y = M[f.i01 ? o00 + 1u : 0u];
        f.p1.x = M[f.i10 ? o00 + W : 0u];
        f.p1.y = M[f.i11 ? o00 + W + 1u : 0u];
        f.first0 = true;
        f.first1 = false;
    }
    f.ty = py - fy;
    f.tx = px - fx;
}

template <typename T>
__device__ __forceinline__ float
field_factor(const FieldSample<T>& f, float pad)
{
    float a0 = float(f.p0.x), b0 = float(f.p0.y), a1 = float(f.p1.x), b1 = float(f.p1.y);
    // An empty asm statement hides that these values were loaded, so the selects below stay
    // selects: the compiler otherwise turns a select of a loaded value into branches around it.
    asm("" : "+v"(a0), "+v"(b0), "+v"(a1), "+v"(b1));
    const float v00 = f.i00 ? (f.first0 ? a0 : b0) : pad;
    const float v10 = f.i10 ? (f.first0 ? a1 : b1) : pad;
    const float v01 = f.i01 ? (f.first1 ? a0 : b0) : pad;
    const float v11 = f.i11 ? (f.first1 ? a1 : b1) : pad;
    const float l0 = lerp_ref(v00, v10, f.ty);
    const float l1 = lerp_ref(v01, v11, f.ty);
    return lerp_ref(l0, l1, f.tx);
}

// The cameras of a field product, in index order: all of a scene's, or those whose bit is set in the words' `need`
// (in LDS, the same for the whole wavefront).
struct AllCameras
{
    int32_t b = 0, B;
    __device__ __forceinline__ explicit AllCameras(int32_t n) : B(n) {}
    __device__ __forceinline__ int32_t left() const { return B - b; }
    template <int N>
    __device__ __forceinline__ bool inside() const { return false; }
    __device__ __forceinline__ int32_t next() { return b++; }
};

struct CameraWord
{
    uint64_t need;
    uint64_t inside; // cameras in whose images all points project well inside (SkipProbe::inside)
};

struct NeededCameras
{
    static constexpr int32_t kWords = 16; // cameras past 64 * kWords are always needed
    const CameraWord* words;
    int32_t B, w = -1;
    uint64_t m = 0; // cameras left in word w, 0 only at the end
    uint64_t in = 0;
    __device__ __forceinline__ NeededCameras(const CameraWord* c, int32_t n) : words(c), B(n) { advance(); }
    static __device__ __forceinline__ uint64_t
    uniform(uint64_t v)
    {
        // (the builtin returns a signed value)
        return (uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(uint32_t(v >> 32)))) << 32) |
               uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(uint32_t(v))));
    }
    __device__ __forceinline__ void
    advance()
    {
        while (m == 0 && 64 * (w + 1) < B)
        {
            ++w;
            m = B - 64 * w < 64 ? (uint64_t(1) << (B - 64 * w)) - 1u : ~uint64_t(0);
            in = 0;
            if (w < kWords)
            {
                m &= uniform(words[w].need);
                in = uniform(words[w].inside);
            }
        }
    }
    __device__ __forceinline__ int32_t left() const { return __popcll(m); }
    // whether the next N cameras (N <= left()) are `inside` ones
    template <int N>
    __device__ __forceinline__ bool
    inside() const
    {
        uint64_t rest = m;
#pragma unroll
        for (int u = 0; u < N; ++u)
            rest &= rest - 1u;
        return ((m ^ rest) & ~in) == 0;
    }
    __device__ __forceinline__ int32_t
    next()
    {
        const int32_t b = 64 * w + int32_t(__builtin_ctzll(m));
        m &= m - 1u;
        advance();
        return b;
    }
};

// field_sample and field_factor for a camera in whose image the point is known to project well inside
// (SkipProbe::inside): the division needs no range test (a numerator too small for the shared reciprocal leaves
// q + 1 and q - 0.5 as the IEEE quotient does, carve_div_in_range), the sample no bounds tests and no padding, and
// partial masks count the camera.  About half the VALU instructions of field_sample.
template <typename T>
struct InsideSample
{
    typedef T pair_t __attribute__((ext_vector_type(2), aligned(sizeof(T))));
    pair_t p0, p1;
    float ty, tx;
};

template <typename T, bool OFF32>
__device__ __forceinline__ void
inside_sample(const SceneDev& s, int32_t b, float wx, float wy, float wz, InsideSample<T>& f)
{
    const auto T4 = as_global(s.transforms + 16 * b);
    const bool gl = s.opengl != 0;
    const auto D = T4 + (gl ? 12 : 8);
    const float cx = fmaf(T4[0], wx, fmaf(T4[1], wy, fmaf(T4[2], wz, T4[3])));
    const float cy = fmaf(T4[4], wx, fmaf(T4[5], wy, fmaf(T4[6], wz, T4[7])));
    const float cd = fmaf(D[0], wx, fmaf(D[1], wy, fmaf(D[2], wz, D[3])));
    float qx, qy;
    div2_unchecked(cx, cy, cd, qx, qy);
    const float px = gl ? unnormalize_ndc(qx, float(s.W)) : qx - 0.5f;
    const float py = gl ? unnormalize_ndc(qy, float(s.H)) : qy - 0.5f;
    const float fx = floorf(px), fy = floorf(py);
    const uint32_t ix = uint32_t(fx), iy = uint32_t(fy);
    typedef __attribute__((address_space(1))) const typename InsideSample<T>::pair_t global_pair_t;
    const T* M = static_cast<const T*>(s.masks) + int64_t(b) * s.H * s.W;
    if constexpr (OFF32)
    {
        const auto G = (gptr<const char>)M;
        const uint32_t pitch = uint32_t(s.W) * uint32_t(sizeof(T)), xb = ix * uint32_t(sizeof(T));
        uint32_t r0; // one v_mad_u32_u24 (see field_sample)
        asm("v_mad_u32_u24 %0, %1, %2, %3" : "=v"(r0) : "v"(iy), "v"(pitch), "v"(xb));
        f.p0 = *(global_pair_t*)(G + r0);
        f.p1 = *(global_pair_t*)(G + (r0 + pitch));
    }
    else
    {
        const auto G = as_global(M);
        f.p0 = *(global_pair_t*)(G + (uint64_t(iy) * uint32_t(s.W) + ix));
        f.p1 = *(global_pair_t*)(G + (uint64_t(iy + 1u) * uint32_t(s.W) + ix));
    }
    f.ty = py - fy;
    f.tx = px - fx;
}

template <typename T>
__device__ __forceinline__ float
inside_factor(const InsideSample<T>& f)
{
    const float l0 = lerp_ref(float(f.p0.x), float(f.p1.x), f.ty);
    const float l1 = lerp_ref(float(f.p0.y), float(f.p1.y), f.ty);
    return lerp_ref(l0, l1, f.tx);
}

// Product over the cameras, in camera order, of the bilinear mask samples at
// a grid vertex (VH:470-530); masks of element type T (float32 or uint8).
template <typename T, bool PAIR, bool PARTIAL, bool OFF32, typename Cameras>
__device__ __forceinline__ float
field_product(const SceneDev& s, float wx, float wy, float wz, Cameras cams)
{
    const float pad = PARTIAL ? 1.0f : 0.0f; // ones padding (partial) or zeros padding (full), IU:162-214
    constexpr int U = 4; // cameras whose reads are in flight together
    float value = 1.0f;
    while (cams.left() > 0)
    {
        while (cams.left() >= U)
        {
            if constexpr (PAIR)
                if (cams.template inside<U>())
                {
                    InsideSample<T> f[U];
#pragma unroll
                    for (int u = 0; u < U; ++u)
                        inside_sample<T, OFF32>(s, cams.next(), wx, wy, wz, f[u]);
#pragma unroll
                    for (int u = 0; u < U; ++u)
                        value *= inside_factor<T>(f[u]);
                    continue;
                }
            FieldSample<T> f[U];
#pragma unroll
            for (int u = 0; u < U; ++u)
                field_sample<T, PAIR, PARTIAL, OFF32>(s, cams.next(), wx, wy, wz, f[u]);
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (!PARTIAL || !f[u].skip)
                    value *= field_factor<T>(f[u], pad);
        }
        // the rest of a camera word: the next word's cameras go U at a time again
        for (int32_t rest = cams.left(); rest > 0; --rest)
        {
            FieldSample<T> f;
            field_sample<T, PAIR, PARTIAL, OFF32>(s, cams.next(), wx, wy, wz, f);
            if (!PARTIAL || !f.skip)
                value *= field_factor<T>(f, pad);
        }
    }
    return value;
}

// Field value at grid point (x, y, z) of scene s.
template <typename T, typename Cameras>
__device__ __forceinline__ float
field_value(const SceneDev& s, uint32_t x, uint32_t y, uint32_t z, Cameras cams)
{
    const float inv = __builtin_ldexpf(1.0f, -s.level);
    const float wx = grid_to_world(x, inv, s.length, s.corner[0]);
    const float wy = grid_to_world(y, inv, s.length, s.corner[1]);
    const float wz = grid_to_world(z, inv, s.length, s.corner[2]);
    if (s.W < 2)
        return s.partial != 0 ? field_product<T, false, true, false>(s, wx, wy, wz, cams)
                              : field_product<T, false, false, false>(s, wx, wy, wz, cams);
    if (uint64_t(s.H) * uint64_t(s.W) * sizeof(T) < (uint64_t(1) << 31) && s.W * int32_t(sizeof(T)) < (1 << 24))
        return s.partial != 0 ? field_product<T, true, true, true>(s, wx, wy, wz, cams)
                              : field_product<T, true, false, true>(s, wx, wy, wz, cams);
    return s.partial != 0 ? field_product<T, true, true, false>(s, wx, wy, wz, cams)
                          : field_product<T, true, false, false>(s, wx, wy, wz, cams);
}

// One thread per vertex in numbering order (packed keys).  The gathers of a wave are bound by the
// vector-memory path (distinct mask lines per instruction); ordering a wave's vertices in 4 x 4 x 4
// tiles would cut those lines by about 40 %, but whole tiles are too uneven a unit of work (up to
// 2048 vertices) for a persistent walk, so the kernel keeps the numbering order.  Six waves per SIMD: 80
// VGPRs, which the compiler passed by 2 when the loop over the cameras was written otherwise.
__global__ __launch_bounds__(256, 6) void
field_kernel(const uint64_t* __restrict__ vertices, uint32_t n, const SceneDev* __restrict__ scenes,
             float* __restrict__ values)
{
    const uint32_t i = xcd_block(blockIdx.x, gridDim.x) * 256 + threadIdx.x;
    if (i >= n)
        return;
    const uint64_t key = vertices[i];
    const uint32_t sid = key_scene(key);
    const uint32_t s0 = __builtin_amdgcn_readfirstlane(sid);
    float value;
    if (__all(sid == s0))
    {
        const SceneDev s = wave_uniform(scenes[s0]); // scalar camera data
        value = s.mask_dtype == kF32
                    ? field_value<float>(s, key_x(key), key_y(key), key_z(key), AllCameras(s.B))
                    : field_value<uint8_t>(s, key_x(key), key_y(key), key_z(key), AllCameras(s.B));
    }
    else
    {
        const SceneDev s = scenes[sid];
        value = s.mask_dtype == kF32
                    ? field_value<float>(s, key_x(key), key_y(key), key_z(key), AllCameras(s.B))
                    : field_value<uint8_t>(s, key_x(key), key_y(key), key_z(key), AllCameras(s.B));
    }
    values[i] = value;
}

void
launch_field(const uint64_t* vertices, uint32_t n, const SceneDev* scenes, float* values, hipStream_t st)
{
    if (n == 0)
        return;
    field_kernel<<<blocks_for(n, 256), 256, 0, st>>>(vertices, n, scenes, values);
    THULL_LAUNCH_CHECK();
}

// ===========================================================================
// Field by bricks
//
// For scenes with solid maps a wavefront takes the vertices of one brick of up to 8 x 8 x 8 cells.  One test per
// camera (a lane each) finds the cameras whose mask is 1 under the whole brick: their bilinear samples are of
// four ones, their factor is exactly 1, and they are left out of all products of the brick.  The vertices of a
// brick also project closer together than 64 consecutive vertices of the numbering, so the reads of the other
// cameras touch fewer lines.  Bound by VALU issue.  Field of a level-11 hull of 50 1080p cameras 1.89 -> 0.78 ms, of a
// level-10 hull of 32 partial 2048^2 ones 1.14 -> 0.27, of a level-9 hull of 64 blurred 1024^2 ones 0.41 -> 0.16.
//
// A vertex on the faces between bricks belongs to the last of the kept bricks it touches, in (z, y, x) order.
// ===========================================================================

// Neighbours of a brick that come after it in (z, y, x) order among those that a vertex at (px, py, pz) of its box
// touches, 0: low, 1: inside, 2: high side per axis; neighbour (dx, dy, dz) is bit (dz + 1) * 9 + (dy + 1) * 3 +
// dx + 1.
__device__ __forceinline__ uint32_t
brick_after(uint32_t px, uint32_t py, uint32_t pz)
{
    // neighbours touched along an axis
    constexpr uint32_t X = 0b001001001001001001001001001u, Y = 0b000000111000000111000000111u, Z = 0b111111111u;
    const uint32_t tx = px == 0u ? 3u * X : px == 1u ? 2u * X : 6u * X;
    const uint32_t ty = py == 0u ? Y | (Y << 3) : py == 1u ? Y << 3 : (Y << 3) | (Y << 6);
    const uint32_t tz = pz == 0u ? Z | (Z << 9) : pz == 1u ? Z << 9 : (Z << 9) | (Z << 18);
    return tx & ty & tz & (0x7ffffffu << 14 & 0x7ffffffu); // the neighbours after the brick's own bit 13
}

constexpr int kBrickRows = ((1 << kBrickShift) + 1) * ((1 << kBrickShift) + 1); // rows of vertices, 81
constexpr int kBrickVerts = kBrickRows * ((1 << kBrickShift) + 1);
constexpr int kNeedWords = NeededCameras::kWords;

__global__ __launch_bounds__(256) void
field_bricks_kernel(const BrickList* __restrict__ lists, int32_t nlists, uint64_t total,
                    const SceneDev* __restrict__ scenes, const uint32_t* __restrict__ bitmap,
                    const uint32_t* __restrict__ prefix, float* __restrict__ values)
{
    __shared__ CameraWord need_lds[4][kNeedWords];
    __shared__ uint32_t first_lds[4][kBrickRows + 3]; // rank of a row's first vertex
    __shared__ uint16_t bits_lds[4][kBrickRows + 3];  // a row's vertices
    __shared__ uint16_t queue_lds[4][kBrickVerts + 7];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint64_t item = uint64_t(xcd_block(blockIdx.x, gridDim.x)) * 4u + wave;
    if (item >= total)
        return;
    const BrickList l = lists[find_segment_uniform([&](int32_t k) { return lists[k].begin; }, nlists, item)];
    const uint64_t key = l.keys[item - l.begin];
    const uint32_t sid = uint32_t(__builtin_amdgcn_readfirstlane(key_scene(key)));
    if (!brick_of_list(scenes[sid], l)) // a cell of a scene whose bricks are in another list
        return;
    const SceneDev s = wave_uniform(scenes[sid]);
    const int32_t shift = s.brick_shift, level = s.level - shift;
    const uint32_t side = 1u << shift, nb = 1u << level;
    const uint32_t bx = __builtin_amdgcn_readfirstlane(key_x(key)), by = __builtin_amdgcn_readfirstlane(key_y(key)),
                   bz = __builtin_amdgcn_readfirstlane(key_z(key));
    CameraWord* const need = need_lds[wave];
    uint32_t* const first = first_lds[wave];
    uint16_t* const bits = bits_lds[wave];
    uint16_t* const queue = queue_lds[wave];
    // occupied neighbours
    uint32_t kept = 0u;
    {
        const int32_t n = int32_t(min(lane, 26u));
        const uint32_t x = bx + uint32_t(n % 3 - 1), y = by + uint32_t(n / 3 % 3 - 1), z = bz + uint32_t(n / 9 - 1);
        bool on = lane < 27u && x < nb && y < nb && z < nb; // -1 wraps past nb
        if (on)
        {
            const uint64_t bit = brick_bit(x, y, z, level);
            on = (s.bricks[bit >> 5] >> uint32_t(bit & 31u)) & 1u;
        }
        kept = uint32_t(__ballot(on));
    }
    // cameras that are needed
    const int32_t words = (s.B + 63) / 64;
    for (int32_t w = 0; w < words && w < kNeedWords; ++w)
    {
        const int32_t b = 64 * w + int32_t(lane);
        bool needed = b < s.B, inside = false;
        if (needed && s.solid != nullptr && shift > 0)
        {
            const float inv = __builtin_ldexpf(1.0f, -s.level), half = 0.5f * s.length * __builtin_ldexpf(1.0f, -level);
            const float cx = grid_to_world((bx << shift) + side / 2u, inv, s.length, s.corner[0]);
            const float cy = grid_to_world((by << shift) + side / 2u, inv, s.length, s.corner[1]);
            const float cz = grid_to_world((bz << shift) + side / 2u, inv, s.length, s.corner[2]);
            const SkipProbe p = s.opengl != 0 ? skip_probe<true, true>(s, b, half, cx, cy, cz)
                                              : skip_probe<false, true>(s, b, half, cx, cy, cz);
            const int32_t d = as_global(s.solid + int64_t(b) * s.solid_h * s.solid_w)[p.at];
            needed = !(p.reach <= float(kSolidTile * (d - 1)));
            inside = p.inside;
        }
        const CameraWord m{ __ballot(needed), __ballot(inside) };
        if (lane == 0)
            need[w] = m;
    }
    // the vertices of the brick's rows
    const uint32_t R1 = (1u << s.level) + 1u, rows1 = side + 1u;
    uint32_t queued = 0u;
    for (uint32_t r0 = 0; r0 < rows1 * rows1; r0 += 64)
    {
        const uint32_t r = r0 + lane;
        uint32_t own = 0u;
        if (r < rows1 * rows1)
        {
            const uint32_t rz = r / rows1, ry = r - rz * rows1;
            const uint32_t x0 = bx << shift, sh = x0 & 31u;
            const uint64_t row = uint64_t((bz << shift) + rz) * R1 + (by << shift) + ry;
            const uint64_t w = s.bitmap_offset + row * s.row_words + (x0 >> 5);
            const uint32_t word = bitmap[w];
            // the last vertex of a row may be the first bit of the next word
            const uint32_t next = sh + side == 32u ? bitmap[w + 1] : 0u;
            // prefixes hold where their group has vertices
            const uint64_t at = word == 0u && sh + side == 32u ? w + 1 : w;
            uint32_t v = ((word >> sh) | (next << 1 << (31u - sh))) & ((2u << side) - 1u);
            first[r] = prefix[at] + uint32_t(__popc(word & ((1u << sh) - 1u)));
            bits[r] = uint16_t(v);
            const uint32_t py = ry == 0u ? 0u : ry == side ? 2u : 1u, pz = rz == 0u ? 0u : rz == side ? 2u : 1u;
            if ((kept & brick_after(0u, py, pz)) != 0u)
                v &= ~1u;
            if ((kept & brick_after(1u, py, pz)) != 0u)
                v &= 1u | (1u << side);
            if ((kept & brick_after(2u, py, pz)) != 0u)
                v &= ~(1u << side);
            own = v;
        }
        const uint32_t n = uint32_t(__popc(own)), inc = wave_inclusive_sum(n);
        for (uint32_t at = queued + inc - n; own != 0u; own &= own - 1u)
            queue[at++] = uint16_t((r << 4) | uint32_t(__builtin_ctz(own)));
        queued += uint32_t(__shfl(int(inc), 63, 64));
    }
    wave_lds_sync();
    for (uint32_t q = lane; q - lane < queued; q += 64)
    {
        const bool on = q < queued;
        const uint32_t e = queue[on ? q : 0u], r = e >> 4, b = e & 15u;
        const uint32_t rz = r / rows1, ry = r - rz * rows1;
        const uint32_t x = (bx << shift) + b, y = (by << shift) + ry, z = (bz << shift) + rz;
        const float value = s.mask_dtype == kF32 ? field_value<float>(s, x, y, z, NeededCameras(need, s.B))
                                                 : field_value<uint8_t>(s, x, y, z, NeededCameras(need, s.B));
        if (on)
            values[first[r] + uint32_t(__popc(uint32_t(bits[r]) & ((1u << b) - 1u)))] = value;
    }
}

void
launch_field_bricks(const BrickList* lists, int32_t nlists, uint64_t waves, const SceneDev* scenes,
                    const uint32_t* bitmap, const uint32_t* prefix, float* values, hipStream_t st)
{
    if (waves == 0)
        return;
    field_bricks_kernel<<<blocks_for(int64_t(waves), 4), 256, 0, st>>>(lists, nlists, waves, scenes, bitmap, prefix,
                                                                       values);
    THULL_LAUNCH_CHECK();
}

__global__ __launch_bounds__(256) void
fill_u32_kernel(uint32_t* __restrict__ dst, uint64_t n, uint32_t value)
{
    const uint64_t stride = uint64_t(gridDim.x) * 256u;
    for (uint64_t i = uint64_t(blockIdx.x) * 256u + threadIdx.x; i < n; i += stride)
        dst[i] = value;
}


void
launch_fill_u32(uint32_t* dst, uint64_t n, uint32_t value, hipStream_t st)
{
    if (n == 0)
        return;
    const uint64_t blocks = std::min<uint64_t>((n + 255) / 256, 8192);
    fill_u32_kernel<<<unsigned(blocks), 256, 0, st>>>(dst, n, value);
    THULL_LAUNCH_CHECK();
}

// ===========================================================================
// Candidate wireframes (VH:1022-1058)
//
// Cell c of a level-i candidate list (ravel id x + y R + z R^2, R = 2^i) gives
// the 8 corners of the cell in cube_vertex order (x bit, y bit, z bit) at
// fmaf(length / R, corner index, cube corner) per axis, and 12 edges between
// them in edge_to_vertex_table order.  One thread per cell; the 24 floats and
// 24 int64 values of a cell are written as whole rows.
// ===========================================================================

// Corner pairs of the 12 cube edges (corner i at (i & 1, i >> 1 & 1, i >> 2 & 1)) in the order the
// reference's wireframes list them (edge_to_vertex_table, marching_cubes_table.h:335-338): the edge
// order is part of the output.
__constant__ uint8_t kWireEdges[12][2] = { { 0, 1 }, { 1, 5 }, { 4, 5 }, { 0, 4 }, { 2, 3 }, { 3, 7 },
                                           { 6, 7 }, { 2, 6 }, { 0, 2 }, { 1, 3 }, { 5, 7 }, { 4, 6 } };

__global__ __launch_bounds__(256) void
wireframe_kernel(const int64_t* __restrict__ cells, uint32_t n, int32_t level, float cx, float cy, float cz,
                 float scale, float* __restrict__ verts, int64_t* __restrict__ edges)
{
    const uint32_t t = blockIdx.x * 256 + threadIdx.x;
    if (t >= n)
        return;
    const uint64_t id = uint64_t(cells[t]);
    const uint64_t mask = (uint64_t(1) << level) - 1u;
    const uint32_t x = uint32_t(id & mask), y = uint32_t((id >> level) & mask), z = uint32_t(id >> (2 * level));
    float v[24];
#pragma unroll
    for (int i = 0; i < 8; ++i)
    {
        v[3 * i + 0] = fmaf(scale, float(x + (i & 1)), cx);
        v[3 * i + 1] = fmaf(scale, float(y + ((i >> 1) & 1)), cy);
        v[3 * i + 2] = fmaf(scale, float(z + ((i >> 2) & 1)), cz);
    }
    float* dv = verts + 24 * uint64_t(t);
#pragma unroll
    for (int i = 0; i < 24; ++i)
        dv[i] = v[i];
    int64_t* de = edges + 24 * uint64_t(t);
    const int64_t base = 8 * int64_t(t);
#pragma unroll
    for (int i = 0; i < 12; ++i)
    {
        de[2 * i + 0] = base + kWireEdges[i][0];
        de[2 * i + 1] = base + kWireEdges[i][1];
    }
}

void
launch_wireframe(const int64_t* cells, uint32_t n, int32_t level, const float corner[3], float length, float* verts,
                 int64_t* edges, hipStream_t st)
{
    if (n == 0)
        return;
    // VH:1038-1040: cube_length / float(resolution), a division by a power of two
    const float scale = length / float(int64_t(1) << level);
    wireframe_kernel<<<blocks_for(n, 256), 256, 0, st>>>(cells, n, level, corner[0], corner[1], corner[2], scale,
                                                          verts, edges);
    THULL_LAUNCH_CHECK();
}

} // namespace thull
