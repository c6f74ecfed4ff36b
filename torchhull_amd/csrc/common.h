// Shared definitions of the MI355X visual-hull library: device-side scalar
// semantics, scene descriptors, error handling and launch helpers.
//
// Floating-point rule of this library: every translation unit is compiled
// with -ffp-contract=off, so the only fused multiply-adds are the explicit
// fmaf() calls below, placed where the reference calls fmaf or where nvcc
// contracts `a + b * c` by default.  Division is IEEE (hipcc's default
// correctly rounded f32 divide), roundf rounds halves away from zero and
// fminf/fmaxf ignore NaN operands, as in CUDA.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <stdexcept>
#include <string>

namespace thull
{

// ---------------------------------------------------------------------------
// Error handling
// ---------------------------------------------------------------------------

struct Error : std::runtime_error
{
    using std::runtime_error::runtime_error;
};

#define THULL_CHECK(cond, msg)                                                                                         \
    do                                                                                                                 \
    {                                                                                                                  \
        if (!(cond))                                                                                                   \
            throw ::thull::Error(std::string("Check failed: ") + #cond + ". " + (msg));                               \
    } while (0)

#define THULL_HIP(expr)                                                                                                \
    do                                                                                                                 \
    {                                                                                                                  \
        hipError_t err_ = (expr);                                                                                      \
        if (err_ != hipSuccess)                                                                                        \
            throw ::thull::Error(std::string("HIP error ") + hipGetErrorString(err_) + " at " + __FILE__ + ":" +       \
                                 std::to_string(__LINE__) + " (" #expr ")");                                           \
    } while (0)

#define THULL_LAUNCH_CHECK() THULL_HIP(hipGetLastError())

// ---------------------------------------------------------------------------
// Element types crossing the C ABI (values of thull_dtype in the public header)
// ---------------------------------------------------------------------------

enum DType : int32_t
{
    kBool = 0,
    kU8 = 1,
    kI8 = 2,
    kI16 = 3,
    kI32 = 4,
    kI64 = 5,
    kF16 = 6,
    kF32 = 7,
    kF64 = 8,
};

// ---------------------------------------------------------------------------
// Packed cell / vertex keys.  A grid point of scene s is packed as
//   s << 48 | z << 32 | y << 16 | x     (x, y, z < 2^16, s < 2^16)
// so that the octree queues and the vertex list carry their scene and
// coordinates without any division.  Within one scene the packed order is the
// (z, y, x) lexicographic order, i.e. the order of the reference's ravel
// index x + y*R + z*R*R.
// ---------------------------------------------------------------------------

__host__ __device__ __forceinline__ uint64_t
pack_key(uint32_t s, uint32_t x, uint32_t y, uint32_t z)
{
    return (uint64_t(s) << 48) | (uint64_t(z) << 32) | (uint64_t(y) << 16) | uint64_t(x);
}
__host__ __device__ __forceinline__ uint32_t
key_scene(uint64_t k)
{
    return uint32_t(k >> 48);
}
__host__ __device__ __forceinline__ uint32_t
key_x(uint64_t k)
{
    return uint32_t(k) & 0xffffu;
}
__host__ __device__ __forceinline__ uint32_t
key_y(uint64_t k)
{
    return uint32_t(k >> 16) & 0xffffu;
}
__host__ __device__ __forceinline__ uint32_t
key_z(uint64_t k)
{
    return uint32_t(k >> 32) & 0xffffu;
}

// ---------------------------------------------------------------------------
// Device scalar semantics of the reference
// ---------------------------------------------------------------------------

// float -> int64 as CUDA's cvt.rzi.s64.f32 (static_cast<int64_t>(float)):
// truncation, saturation to the int64 range, NaN -> 0.
__device__ __forceinline__ int64_t
f2i64_sat(float f)
{
    if (fabsf(f) < 2147483648.0f)
        return int64_t(int32_t(f));
    if (f != f)
        return 0;
    if (f >= 9223372036854775808.0f)
        return INT64_MAX;
    if (f < -9223372036854775808.0f)
        return INT64_MIN;
    return int64_t(f);
}

// clamp(int64(roundf-ed value r), 0, hi) evaluated in float: r is an
// integral float, +-inf or NaN; NaN maps to 0 like the saturating conversion.
__device__ __forceinline__ int32_t
clamp_rounded(float r, float hi)
{
    return int32_t(fminf(fmaxf(r, 0.0f), hi));
}

// image_utils.h:67-71: ((c + 1) * size) / 2 - 0.5, every step rounded.  The
// halving is exact, so fmaf(t, 0.5, -0.5) rounds once, like (t / 2) - 0.5.
__device__ __forceinline__ float
unnormalize_ndc(float c, float size)
{
    float t = c + 1.0f;
    t = t * size;
    return fmaf(t, 0.5f, -0.5f);
}

// math.h:19-23
__device__ __forceinline__ float
lerp_ref(float v0, float v1, float t)
{
    return fmaf(t, v1, fmaf(-t, v0, v0));
}

// Two IEEE quotients nx / d and ny / d with one shared reciprocal.
//
// hipcc's correctly rounded float division is div_scale(n) and div_scale(d)
// (operands scaled by 2^+-64 when exponents are extreme), r = rcp(d),
// r += r * (1 - d * r), q = n * r, two corrections q += r * (n - d * q) (the
// second through div_fmas, which undoes the scaling) and div_fixup (NaN,
// infinities, zeros, overflow).  When 2^-40 <= |n|, |d| <= 2^40, div_scale
// scales nothing (exponent gap < 96, no denormal operand, quotient or
// reciprocal) and div_fixup passes the quotient through, so the same
// operations without them give the same bits; the reciprocal does not depend
// on the numerator, so both quotients share it.  Other operands take the
// plain division.
//
// A NaN operand fails the range test (the magnitude bounds propagate NaN) and
// takes the plain division.
__device__ __forceinline__ void
div2_unchecked(float nx, float ny, float d, float& qx, float& qy)
{
    float r = __builtin_amdgcn_rcpf(d);
    r = fmaf(fmaf(-d, r, 1.0f), r, r);
    float a = nx * r, b = ny * r;
    a = fmaf(fmaf(-d, a, nx), r, a);
    b = fmaf(fmaf(-d, b, ny), r, b);
    qx = fmaf(fmaf(-d, a, nx), r, a);
    qy = fmaf(fmaf(-d, b, ny), r, b);
}

// Largest and smallest magnitude of three operands; NaN if any of them is NaN
// (one v_maximum3 / v_minimum3, with no quieting of the operands first).
__device__ __forceinline__ float
max_abs3(float a, float b, float c)
{
    return __builtin_elementwise_maximum(__builtin_elementwise_maximum(fabsf(a), fabsf(b)), fabsf(c));
}
__device__ __forceinline__ float
min_abs3(float a, float b, float c)
{
    return __builtin_elementwise_minimum(__builtin_elementwise_minimum(fabsf(a), fabsf(b)), fabsf(c));
}

// True when every operand magnitude between lo and hi lies in [2^-40, 2^40].
__device__ __forceinline__ bool
div2_in_range(float hi, float lo)
{
    return hi <= 0x1p40f && lo >= 0x1p-40f;
}

__device__ __forceinline__ void
div2_shared(float nx, float ny, float d, float& qx, float& qy)
{
    if (div2_in_range(max_abs3(nx, ny, d), min_abs3(nx, ny, d)))
        div2_unchecked(nx, ny, d, qx, qy);
    else
    {
        qx = nx / d;
        qy = ny / d;
    }
}

// Orders the LDS accesses of one wavefront's lanes around this point, for lanes that exchange
// data through LDS without a workgroup barrier (a wavefront's LDS instructions execute in order).
__device__ __forceinline__ void
wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Grid coordinate -> world coordinate: corner + v / res * length, contracted
// by nvcc to fmaf(v / res, length, corner) (visual_hull_cuda.cu:206-213).
// res is a power of two, so v / res is exact and equal to v * inv_res.
__device__ __forceinline__ float
grid_to_world(uint32_t v, float inv_res, float length, float corner)
{
    return fmaf(float(v) * inv_res, length, corner);
}

// ---------------------------------------------------------------------------
// Padded, tiled integral-image layout used by carving.  Per camera a plane of
// integral_rows(H) rows (H + kIntegralRow0 rounded up to a multiple of 4) of
// pitch integral_pitch(W) floats (a multiple of 32); element (y, x) is at
// padded row Y = y + kIntegralRow0, column X = x + kIntegralCol0.  Row
// kIntegralRow0 - 1 and column kIntegralCol0 - 1 hold zeros: they are the
// entries y = -1 and x = -1 that the box sums read at the image border.  The
// plane is stored in tiles of 4 rows x 8 columns, one 128-byte line each, tile
// (Y / 4, X / 8) at float Y / 4 * 4 * pitch + X / 8 * 32 and (Y, X) at
// (Y % 4) * 8 + X % 8 inside it: the four corner reads of a wavefront's child
// windows, which spread over a few rows and columns of pixels, touch a quarter
// fewer distinct lines than in row-major order (a gather costs about one L1
// tag cycle per distinct line).  The image's rows start at a tile row and its
// columns at a tile column, so the integral passes write whole lines.  Entries
// outside the image and its zero row and column are never read.
// ---------------------------------------------------------------------------

constexpr int64_t kIntegralCol0 = 32;
constexpr int64_t kIntegralRow0 = 4;

__host__ __device__ __forceinline__ int64_t
integral_pitch(int64_t W)
{
    return (W + kIntegralCol0 + 31) & ~int64_t(31);
}

__host__ __device__ __forceinline__ int64_t
integral_rows(int64_t H)
{
    return (H + kIntegralRow0 + 3) & ~int64_t(3);
}

// Float offset of padded row Y's tile row plus Y's row inside the tile, (Y & ~3) * pitch + (Y & 3) * 8,
// taken as (Y & ~3) * (pitch - 8) + 8 Y (one and, one shift, one 24-bit multiply-add; pitch >= 32,
// pitch and Y below 2^24 and the result below 2^30, as the plane is).
__device__ __forceinline__ uint32_t
integral_row_offset(uint32_t Y, uint32_t pitch)
{
    return __umul24(Y & ~3u, pitch - 8u) + (Y << 3);
}

// Float offset of padded column X's tile plus X's column inside the tile: (X / 8) * 32 + X % 8, taken as
// X + 3 (X & ~7) with one 24-bit multiply-add (X < 2^24), which hipcc does not select here by itself
// (it takes a 64-bit multiply-add).
__device__ __forceinline__ uint32_t
integral_col_offset(uint32_t X)
{
    uint32_t r;
    asm("v_mad_u32_u24 %0, %1, 3, %2" : "=v"(r) : "v"(X & ~7u), "v"(X));
    return r;
}

// ---------------------------------------------------------------------------
// Solid maps: per camera one byte per tile of 4 x 4 pixels, the Chebyshev distance in tiles (at most
// kSolidReach) to the nearest tile that is not solid, 0 for such a tile itself.  A tile is solid when it lies
// inside the image and all its pixels are exactly 1; what lies outside the image counts as not solid.
// ---------------------------------------------------------------------------

constexpr int kSolidTile = 4;
constexpr int kSolidReach = 15;

// Per camera: how far a carving window may reach from its cell's centre for the camera to be skipped
// (carve_skips), and bounds of the projection's rounding errors over the scene's cube.
struct CullCamera
{
    float reach;      // pixels; negative: never skipped
    float sum_d;      // sum of the magnitudes of the denominator row's first three coefficients
    float ex, ey, ed; // rounding errors of the two numerators and the denominator
    float pad_[3];
};

// ---------------------------------------------------------------------------
// Scene descriptor (device side).  One per scene of a batch.
// ---------------------------------------------------------------------------

struct SceneDev
{
    const void* masks;      // [B,H,W] contiguous, element type mask_dtype
    const float* integral;  // B planes of the padded integral-image layout (integral_pitch)
    const float* transforms; // [B,16] float32
    int32_t mask_dtype;
    int32_t B, H, W;
    int32_t level;          // target octree level
    int32_t partial;        // masks_partial
    int32_t opengl;         // transforms convention
    float corner[3];
    float length;
    // carving step at which the scene's root cell is classified: the scene's octree level at carving
    // step i is i - start (0 for the scenes a batch starts with, later for scenes that join it)
    int32_t start;
    // bitmap of grid vertices (R+1)^3 with rows padded to `row_words` 32-bit words
    uint64_t bitmap_offset; // in words, into the batch's vertex bitmap
    uint32_t row_words;
    // bitmap of leaf cells R^3 with rows padded to `cell_row_words` words
    uint32_t cell_row_words;
    uint32_t* cells;        // the scene's leaf-cell bitmap
    // solid maps (null: none) of solid_h x solid_w tiles per camera, and one CullCamera per camera
    const uint8_t* solid;
    const CullCamera* cull;
    int32_t solid_h, solid_w;
    // field by bricks (null: not used): one bit per brick of 2^brick_shift cells per side of the scene's octree,
    // set for the bricks among the kept cells
    uint32_t* bricks;
    uint8_t* group_flags; // with bricks: flags of the groups of 4 words of the vertex bitmap (group_flags_kernel)
    int32_t brick_shift;
    int32_t culls; // set by the solid map pass: some camera's CullCamera::reach lets carving skip it
};

// Bricks of the field are at most 8 cells per side.
constexpr int kBrickShift = 3;

// ---------------------------------------------------------------------------
// Global-memory pointers.  Pointers read from a table in device memory are
// generic (flat) to the compiler; casting them to the global address space
// gives global loads and stores, which carry no LDS dependency and take
// scalar base addresses.
// ---------------------------------------------------------------------------

template <typename T>
using gptr = __attribute__((address_space(1))) T*;

template <typename T>
__device__ __forceinline__ gptr<T>
as_global(T* p)
{
    return (gptr<T>)p;
}

typedef float float4_v __attribute__((ext_vector_type(4)));

// 16-byte load through a global pointer (p 16-byte aligned).
__device__ __forceinline__ float4
ld_float4(gptr<const float> p)
{
    const float4_v v = *(gptr<const float4_v>)p;
    return make_float4(v.x, v.y, v.z, v.w);
}

// ---------------------------------------------------------------------------
// Segment lookup: index of the last segment whose first element is <= v, for
// a non-decreasing table begin(0..n-1).
// ---------------------------------------------------------------------------

// v wave-uniform, every lane of the wave active.  Up to 64 segments take one
// load per lane and a ballot; larger tables use a binary search.
template <typename F>
__device__ __forceinline__ int32_t
find_segment_uniform(F begin, int32_t n, uint64_t v)
{
    if (n <= 64)
    {
        const int32_t lane = int32_t(threadIdx.x & 63);
        const bool le = lane < n && begin(lane) <= v;
        const uint64_t m = __ballot(le);
        return m == 0 ? 0 : 63 - __builtin_clzll(m);
    }
    int32_t lo = 0, hi = n - 1;
    while (lo < hi)
    {
        const int32_t mid = (lo + hi + 1) >> 1;
        if (begin(mid) <= v)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

// v non-decreasing with the lane index (lane 0 holds the wave's smallest v),
// every lane of the wave active: the segment of lane 0's v, then a short walk
// forward per lane.
template <typename F>
__device__ __forceinline__ int32_t
find_segment_rising(F begin, int32_t n, uint64_t v)
{
    const uint64_t v0 = (uint64_t(__builtin_amdgcn_readfirstlane(uint32_t(v >> 32))) << 32) |
                        uint64_t(__builtin_amdgcn_readfirstlane(uint32_t(v)));
    int32_t s = find_segment_uniform(begin, n, v0);
    while (s + 1 < n && begin(s + 1) <= v)
        ++s;
    return s;
}

// A descriptor (scene, grid) with every 32-bit word read from the first
// active lane: for a descriptor that all active lanes share, the compiler then
// keeps it, and what it loads through its pointers, in scalar registers.
template <typename T>
__device__ __forceinline__ T
wave_uniform(const T& s)
{
    constexpr int kWords = sizeof(T) / 4;
    static_assert(sizeof(T) % 4 == 0, "descriptor is a whole number of words");
    uint32_t w[kWords];
    __builtin_memcpy(w, &s, sizeof(T));
#pragma unroll
    for (int i = 0; i < kWords; ++i)
        w[i] = __builtin_amdgcn_readfirstlane(w[i]);
    T u;
    __builtin_memcpy(&u, w, sizeof(T));
    return u;
}

// Logical block of hardware workgroup `bid` of a 1-D grid of `nblocks`.  The
// dispatcher hands workgroups to the 8 XCDs round-robin (workgroup i to XCD
// i % 8), and every XCD has its own L2.  This bijection gives each XCD runs of
// C consecutive logical blocks (neighbouring cells, vertices or pixels, which
// read neighbouring data) while consecutive runs still rotate over the XCDs,
// so work that varies along the grid (scenes with more cameras) stays spread
// evenly.  Workgroups past the last whole round of 8 C keep their index.
template <uint32_t C = 16>
__device__ __forceinline__ uint32_t
xcd_block(uint32_t bid, uint32_t nblocks)
{
    constexpr uint32_t kXcds = 8;
    if (bid >= nblocks / (kXcds * C) * (kXcds * C))
        return bid;
    const uint32_t x = bid % kXcds, k = bid / kXcds;
    return ((k / C) * kXcds + x) * C + k % C;
}

// Quotient of a 64-bit value by a 32-bit divisor, through the 32-bit divide
// when the dividend fits (the common case; 64-bit division is a long
// software sequence).
__device__ __forceinline__ uint64_t
div_u64_u32(uint64_t a, uint32_t b)
{
    if ((a >> 32) == 0u)
        return uint32_t(a) / b;
    return a / b;
}

// ---------------------------------------------------------------------------
// Launch helpers
// ---------------------------------------------------------------------------

// Host-to-device copies of small host tables (job lists, scene descriptors)
// in stream order.  The implementation stages the bytes in pinned memory when
// upload() is called, so the copy neither blocks the host nor reads the host
// table later (a copy from pageable memory waits for the stream's earlier work).
struct Uploader
{
    virtual void upload(void* dst, const void* src, size_t bytes, hipStream_t st) = 0;

protected:
    ~Uploader() = default;
};

inline unsigned
blocks_for(int64_t n, int threads)
{
    return unsigned((n + threads - 1) / threads);
}

} // namespace thull
