// Gaussian mask blur for CDNA4.
//
// Reference (vc-bonn/torchhull, src/torchhull/_C/src/gaussian_blur_cuda.cu, GB):
// sparse band blur GB:288-507 (edge pixels GB:116-142, 3x3 tile window
// GB:144-178, per-pixel convolution GB:180-286), dense blur GB:20-114.
//
// The reference builds the band as a sorted unique list of tile ids (sort +
// unique of 9 ids per edge pixel).  Here the band is a per-tile flag grid: one
// pass marks every tile that holds an edge pixel, and the output pass treats a
// pixel as a band pixel when any tile of the 3x3 window around its tile is
// marked, which is the same set (the reference's clamped window of an edge
// tile never leaves the tile grid, so membership is symmetric).  Band pixels
// get the convolution with the reference's tap order (x offset outer, y
// offset inner), its accumulation in the output type (fused multiply-add for
// float and double, per-operation binary16 rounding for half) and its final
// division by the weight sum; every other pixel is the converted input.
//
// A block of output pixels without band pixels is read at most once more: none
// of its tiles is an edge tile, so every pixel of the block equals its right
// and lower neighbours, and the block holds one value.  The output pass writes
// that value, converted, from one read; only an image holding a negative zero
// (equal to +0 but not the same bits, flagged by the edge pass) copies such
// blocks pixel by pixel.

#include <type_traits>
#include <vector>

#include <hip/hip_fp16.h>

#include "kernels.h"

namespace thull
{

template <typename T>
struct OutOps;

template <>
struct OutOps<float>
{
    using W = float;
    __device__ static float zero() { return 0.0f; }
    __device__ static float mac(float acc, float w, float x) { return fmaf(w, x, acc); }
    __device__ static float add(float a, float b) { return a + b; }
    __device__ static float div(float a, float b) { return a / b; }
    __device__ static float from_float(float v) { return v; }
    __device__ static float from_double(double v) { return float(v); }
};

template <>
struct OutOps<double>
{
    __device__ static double zero() { return 0.0; }
    __device__ static double mac(double acc, double w, double x) { return fma(w, x, acc); }
    __device__ static double add(double a, double b) { return a + b; }
    __device__ static double div(double a, double b) { return a / b; }
    __device__ static double from_float(float v) { return double(v); }
    __device__ static double from_double(double v) { return v; }
};

template <>
struct OutOps<__half>
{
    // c10::Half arithmetic: compute in float, round to binary16 after every operation
    __device__ static __half zero() { return __float2half(0.0f); }
    __device__ static __half mac(__half acc, __half w, __half x)
    {
        const __half prod = __float2half(__half2float(w) * __half2float(x));
        return __float2half(__half2float(acc) + __half2float(prod));
    }
    __device__ static __half add(__half a, __half b) { return __float2half(__half2float(a) + __half2float(b)); }
    __device__ static __half div(__half a, __half b) { return __float2half(__half2float(a) / __half2float(b)); }
    __device__ static __half from_float(float v) { return __float2half(v); }
    __device__ static __half from_double(double v) { return __float2half(float(v)); }
};

// static_cast<BlurredImageT>(input value)
template <typename To, typename Ti>
__device__ __forceinline__ To
convert_in(Ti v)
{
    if constexpr (std::is_same_v<Ti, double>)
        return OutOps<To>::from_double(v);
    else if constexpr (std::is_same_v<Ti, __half>)
        return OutOps<To>::from_float(__half2float(v));
    else if constexpr (std::is_same_v<To, double>)
        return double(v);
    else
        return OutOps<To>::from_float(float(v));
}

// Element read through a global pointer; binary16 values are read as their bits.
template <typename T>
__device__ __forceinline__ T
ld(gptr<const T> p, int64_t i)
{
    if constexpr (std::is_same_v<T, __half>)
        return __ushort_as_half(((gptr<const unsigned short>)p)[i]);
    else
        return p[i];
}

template <typename T>
__device__ __forceinline__ void
st(gptr<T> p, int64_t i, T v)
{
    if constexpr (std::is_same_v<T, __half>)
        ((gptr<unsigned short>)p)[i] = __half_as_ushort(v);
    else
        p[i] = v;
}

// Pixel comparison in the input type (GB:140); half compares as float.
template <typename Ti>
__device__ __forceinline__ bool
differs(Ti a, Ti b)
{
    if constexpr (std::is_same_v<Ti, __half>)
        return __half2float(a) != __half2float(b);
    else
        return a != b;
}

// A floating-point value with the bits of -0 (equal to +0 under differs, so the edge test cannot
// see it); integers have none.
template <typename Ti>
__device__ __forceinline__ bool
negative_zero(Ti v)
{
    if constexpr (std::is_same_v<Ti, __half>)
        return __half_as_ushort(v) == 0x8000u;
    else if constexpr (std::is_same_v<Ti, float>)
        return __float_as_uint(v) == 0x80000000u;
    else if constexpr (std::is_same_v<Ti, double>)
        return uint64_t(__double_as_longlong(v)) == 0x8000000000000000ull;
    else
        return false;
}

// The value of the next lane of the wavefront (lane 63: its own); every lane must execute it.
template <typename T>
__device__ __forceinline__ T
lane_down1(T v)
{
    if constexpr (sizeof(T) == 8)
    {
        const uint64_t u = __builtin_bit_cast(uint64_t, v);
        const uint32_t lo = uint32_t(__shfl_down(int(uint32_t(u)), 1, 64));
        const uint32_t hi = uint32_t(__shfl_down(int(uint32_t(u >> 32)), 1, 64));
        return __builtin_bit_cast(T, (uint64_t(hi) << 32) | lo);
    }
    else
    {
        uint32_t u = 0u;
        __builtin_memcpy(&u, &v, sizeof(T));
        u = uint32_t(__shfl_down(int(u), 1, 64));
        T r;
        __builtin_memcpy(&r, &u, sizeof(T));
        return r;
    }
}

// image_utils.h:129-160 (border not repeated)
__device__ __forceinline__ int64_t
reflect_index(int64_t i, int64_t n)
{
    if (i >= 0 && i < n)
        return i;
    if (n == 1)
        return 0;
    // one reflection (the common case of a halo narrower than the image); at i = 1 - n the
    // reference's formula below gives 0, not n - 1
    if (i < 0 && i > 1 - n)
        return -i;
    if (i >= n && i < 2 * n - 1)
        return 2 * n - 2 - i;
    const int64_t p = n - 1;
    const int64_t flips = i / p + (i < 0 ? 1 : 0);
    int64_t rem = i % p;
    if (rem < 0)
        rem += p;
    return (flips % 2 == 0) ? rem : p - rem;
}

// One blur job: B images of H x W.  Blocks of all jobs are flattened into one
// launch per pass; `*_begin` is the job's first block.
struct BlurJob
{
    const void* in;
    void* out;
    uint8_t* flags;      // B * TH * TW edge-tile flags, then B negative-zero flags (sparse)
    uint8_t* bflags;     // B * oby * obx band-block flags (sparse)
    int32_t B, H, W;
    int32_t TH, TW;      // tile grid (W / ts + 1, H / ts + 1)
    uint32_t bx, by;     // pixel blocks per image (x, y) of the pass running
    uint32_t obx, oby;   // 64 x RB output blocks per image (x, y) of the output pass
    uint64_t p_begin;    // first pixel block of this job
};

__device__ __forceinline__ int32_t
find_blur_job(const BlurJob* jobs, int32_t n, uint64_t blk)
{
    return find_segment_uniform([&](int32_t i) { return jobs[i].p_begin; }, n, blk);
}

constexpr int kBlurBX = 64;
// edge-flag tiles around one pixel block with a zero border: at most (64 / ts + 5) x (RB / ts + 5)
// for ts >= 1, RB <= 64
constexpr int kBlurMaxFlagTiles = (kBlurBX + 5) * (64 + 5); // pixel block: 64 columns x RB rows, 256 threads

// Marks every output block (64 x orb pixels) that holds a pixel of a band tile of an edge tile in
// tile columns txl..txh and rows tyl..tyh: the tiles of their 3 x 3 windows, clamped to the image
// (GB:154-176).  Blocks are marked from the bounding rectangle of a thread's edge tiles, so a marked
// block may still hold no band pixel; an unmarked block holds none.
__device__ __forceinline__ void
mark_band_blocks(const BlurJob& j, int32_t b, int32_t txl, int32_t txh, int32_t tyl, int32_t tyh, int32_t ts,
                 int32_t orb)
{
    const int64_t xl = int64_t(max(txl - 1, 0)) * ts, xh = min(int64_t(txh + 2) * ts, int64_t(j.W)) - 1;
    const int64_t yl = int64_t(max(tyl - 1, 0)) * ts, yh = min(int64_t(tyh + 2) * ts, int64_t(j.H)) - 1;
    const auto F = as_global(j.bflags + int64_t(b) * j.oby * j.obx);
    for (int64_t by = yl / orb; by <= yh / orb; ++by)
        for (int64_t bx = xl / kBlurBX; bx <= xh / kBlurBX; ++bx)
            F[by * j.obx + bx] = 1;
}

// Edge pixels (GB:116-142) marked into their tile's flag, the output blocks
// of the output pass (64 x orb pixels) that their band tiles reach into the
// band-block flags, and images holding a negative zero into their
// negative-zero flag.  Every writer stores the same value 1, so the plain
// byte stores need no atomics; flags are zeroed beforehand.  Wave w of a
// block tests RB / 4 consecutive rows of the block; all of a thread's pixels
// are loaded before any flag is stored.
template <typename Ti, int RB>
__global__ __launch_bounds__(256) void
blur_edge_flags_kernel(const BlurJob* __restrict__ jobs, int32_t njobs, int32_t ts, int32_t orb)
{
    constexpr int R = RB / 4;
    // runs of consecutive blocks (neighbours to the right and below) on one XCD: the lines a block
    // reads past its own columns and rows are its neighbours' and come from the same L2
    const uint64_t blk = xcd_block(blockIdx.x, gridDim.x);
    const BlurJob j = jobs[find_blur_job(jobs, njobs, blk)]; // by value: no reloads after stores
    const uint32_t local = uint32_t(blk - j.p_begin);
    const uint32_t per = j.bx * j.by;
    const int32_t b = int32_t(local / per);
    const uint32_t r = local - uint32_t(b) * per;
    const int32_t by = int32_t(r / j.bx), bx = int32_t(r - uint32_t(by) * j.bx);
    const int32_t H = j.H, W = j.W;
    const int32_t x = bx * kBlurBX + int32_t(threadIdx.x & 63);
    const int32_t yb = by * RB + int32_t(threadIdx.x >> 6) * R;
    if (x >= W || yb >= H)
        return;
    const auto I = as_global(static_cast<const Ti*>(j.in) + int64_t(b) * H * W + x);
    const bool has_right = x + 1 < W;
    Ti c[R + 1], rt[R];
#pragma unroll
    for (int q = 0; q <= R; ++q)
    {
        const bool in = yb + q < H; // row yb + q exists (q == R: the row below the thread's last row)
        c[q] = in ? ld(I, int64_t(yb + q) * W) : (q > 0 ? c[q - 1] : Ti{});
    }
    // the right neighbour is the next lane's pixel (same rows), read for the last lane only
    const bool last_lane = (threadIdx.x & 63u) == 63u;
#pragma unroll
    for (int q = 0; q < R; ++q)
    {
        const Ti nb = lane_down1(c[q]);
        rt[q] = has_right ? nb : c[q];
        if (last_lane && has_right && yb + q < H)
            rt[q] = ld(I, int64_t(yb + q) * W + 1);
    }
    bool nz = false;
#pragma unroll
    for (int q = 0; q <= R; ++q)
        nz = nz || negative_zero(c[q]); // c[R] and absent rows repeat pixels of the image
    if (nz)
        j.flags[int64_t(j.B) * j.TH * j.TW + b] = 1;
    const auto F = as_global(j.flags + int64_t(b) * j.TH * j.TW + x / ts);
    int32_t eyl = -1, eyh = -1; // first and last edge row of the thread
#pragma unroll
    for (int q = 0; q < R; ++q)
    {
        if (yb + q >= H)
            break;
        if (differs(rt[q], c[q]) || differs(c[q + 1], c[q]))
        {
            F[((yb + q) / ts) * j.TW] = 1;
            eyl = eyl < 0 ? yb + q : eyl;
            eyh = yb + q;
        }
    }
    if (eyl >= 0)
        mark_band_blocks(j, b, x / ts, x / ts, eyl / ts, eyh / ts, ts, orb);
}

// float32 images with W % 4 == 0: each thread tests 4 consecutive pixels of
// its rows with 16-byte loads (256 columns per block).
template <int RB>
__global__ __launch_bounds__(256) void
blur_edge_flags_f32x4_kernel(const BlurJob* __restrict__ jobs, int32_t njobs, int32_t ts, int32_t orb)
{
    constexpr int R = RB / 4;
    // runs of consecutive blocks (neighbours to the right and below) on one XCD: the lines a block
    // reads past its own columns and rows are its neighbours' and come from the same L2
    const uint64_t blk = xcd_block(blockIdx.x, gridDim.x);
    const BlurJob j = jobs[find_blur_job(jobs, njobs, blk)]; // by value: no reloads after stores
    const uint32_t local = uint32_t(blk - j.p_begin);
    const uint32_t per = j.bx * j.by;
    const int32_t b = int32_t(local / per);
    const uint32_t r = local - uint32_t(b) * per;
    const int32_t by = int32_t(r / j.bx), bx = int32_t(r - uint32_t(by) * j.bx);
    const int32_t H = j.H, W = j.W;
    const int32_t lane = int32_t(threadIdx.x & 63), wave = int32_t(threadIdx.x >> 6);
    const int32_t x = (bx * 64 + lane) * 4;
    const int32_t yb = by * RB + wave * R;
    const bool live = x < W && yb < H;
    const auto I = as_global(static_cast<const float*>(j.in) + int64_t(b) * H * W + x);
    const bool has_right = x + 4 < W;
    float4 c[R + 1];
    float rt[R];
#pragma unroll
    for (int q = 0; q < R; ++q)
    {
        const bool in = live && yb + q < H;
        c[q] = in ? ld_float4(I + int64_t(yb + q) * W) : (q > 0 ? c[q - 1] : float4{});
    }
    // the row below a wavefront's rows is the next wavefront's first row (same columns): shared
    // through LDS, so the rows of a block are read once; the block's last wavefront reads its own
    static_assert(RB % 4 == 0, "four wavefronts of RB / 4 rows");
    __shared__ float4_v first[4][64];
    first[wave][lane] = float4_v{ c[0].x, c[0].y, c[0].z, c[0].w };
    __syncthreads();
    if (!live)
        return;
    if (yb + R < H)
    {
        if (wave < 3)
        {
            const float4_v v = first[wave + 1][lane];
            c[R] = make_float4(v.x, v.y, v.z, v.w);
        }
        else
            c[R] = ld_float4(I + int64_t(yb + R) * W);
    }
    else
        c[R] = c[R - 1];
    // the right neighbour of the 4 pixels is the next lane's first pixel (same rows), read for the
    // last lane only
    const bool last_lane = (threadIdx.x & 63u) == 63u;
#pragma unroll
    for (int q = 0; q < R; ++q)
    {
        const float nb = lane_down1(c[q].x);
        rt[q] = has_right ? nb : c[q].w;
        if (last_lane && has_right && yb + q < H)
            rt[q] = I[int64_t(yb + q) * W + 4];
    }
    bool nz = false;
#pragma unroll
    for (int q = 0; q <= R; ++q)
        nz = nz || negative_zero(c[q].x) || negative_zero(c[q].y) || negative_zero(c[q].z) || negative_zero(c[q].w);
    if (nz)
        j.flags[int64_t(j.B) * j.TH * j.TW + b] = 1;
    const auto F = as_global(j.flags + int64_t(b) * j.TH * j.TW);
    int32_t exl = x + 3, exh = x, eyl = -1, eyh = -1; // bounding rectangle of the thread's edge pixels
#pragma unroll
    for (int q = 0; q < R; ++q)
    {
        if (yb + q >= H)
            break;
        const float4 u = c[q], d = c[q + 1];
        const bool e0 = (u.y != u.x) || (d.x != u.x);
        const bool e1 = (u.z != u.y) || (d.y != u.y);
        const bool e2 = (u.w != u.z) || (d.z != u.z);
        const bool e3 = (rt[q] != u.w) || (d.w != u.w);
        if (e0 || e1 || e2 || e3)
        {
            const auto row = F + ((yb + q) / ts) * j.TW;
            if (e0)
                row[x / ts] = 1;
            if (e1)
                row[(x + 1) / ts] = 1;
            if (e2)
                row[(x + 2) / ts] = 1;
            if (e3)
                row[(x + 3) / ts] = 1;
            exl = min(exl, e0 ? x : e1 ? x + 1 : e2 ? x + 2 : x + 3);
            exh = max(exh, e3 ? x + 3 : e2 ? x + 2 : e1 ? x + 1 : x);
            eyl = eyl < 0 ? yb + q : eyl;
            eyh = yb + q;
        }
    }
    if (eyl >= 0)
        mark_band_blocks(j, b, exl / ts, exh / ts, eyl / ts, eyh / ts, ts, orb);
}

// Band pixels of a 64 x RB block are convolved from an LDS tile with a halo
// of k/2 (reflect-padded at the image border); blocks without band pixels
// only convert and copy.  `norm` is the reference's sum of the weights in tap
// order and output precision, the same for every pixel.  KT > 0 fixes the
// kernel size at compile time (k == KT); KT == 0 takes it from `k`.
template <typename Ti, typename To, int RB, int KT>
__global__ __launch_bounds__(256) void
blur_tile_kernel(const BlurJob* __restrict__ jobs,
                 int32_t njobs,
                 int32_t k_rt,
                 int32_t ts_rt,
                 bool sparse,
                 const To* __restrict__ weights,
                 To norm,
                 bool vec4)
{
    extern __shared__ unsigned char smem_raw[];
    To* tile = reinterpret_cast<To*>(smem_raw);
    constexpr int P = RB / 4; // pixels per thread
    const int32_t k = KT > 0 ? KT : k_rt;
    const int32_t ts = KT > 0 ? (KT / 2 > 0 ? KT / 2 : 1) : ts_rt; // compile-time divisor when KT is fixed
    const uint64_t blk = xcd_block(blockIdx.x, gridDim.x); // halos of neighbouring blocks share one L2
    const BlurJob j = jobs[find_blur_job(jobs, njobs, blk)]; // by value: no reloads after stores
    const uint32_t local = uint32_t(blk - j.p_begin);
    const uint32_t per = j.bx * j.by;
    const int32_t b = int32_t(local / per);
    const uint32_t rr = local - uint32_t(b) * per;
    const int32_t by = int32_t(rr / j.bx), bx = int32_t(rr - uint32_t(by) * j.bx);
    const int32_t H = j.H, W = j.W;
    const int32_t h = k / 2;
    const int32_t LW = kBlurBX + 2 * h, LH = RB + 2 * h;
    const int32_t x0 = bx * kBlurBX, y0 = by * RB;
    const auto I = as_global(static_cast<const Ti*>(j.in) + int64_t(b) * H * W);
    const auto O = as_global(static_cast<To*>(j.out) + int64_t(b) * H * W);
    const int32_t lx = int32_t(threadIdx.x & 63), ly0 = int32_t(threadIdx.x >> 6);
    const int32_t x = x0 + lx;
    const bool dense = !sparse && k > 1;
    const bool use_flags = sparse && k > 1;
    // float32 rows of a multiple of 4 pixels, 16-byte aligned: a block without band pixels is
    // written with 16-byte stores (thread t: columns x0 + 4 (t % 16) .. + 3 of rows y0 + t / 16 + 16 r)
    constexpr bool kF32 = std::is_same_v<Ti, float> && std::is_same_v<To, float>;
    constexpr int R4 = RB / 16;
    const int32_t cx4 = x0 + 4 * int32_t(threadIdx.x & 15), ry4 = y0 + int32_t(threadIdx.x >> 4);
    // pixel q of this thread: (x, y0 + ly0 P + q), P consecutive rows; rows past H count as absent
    const int32_t yt = y0 + ly0 * P;
    int32_t nq = H - yt;
    nq = x < W ? min(max(nq, 0), P) : 0;
    uint32_t band = 0u;
    // a block that the edge pass left unmarked holds no pixel of a band tile; its band flag, the
    // image's negative-zero flag and its first pixel are read together
    bool flat_block = false, flat_bits = false;
    To v0{};
    if (use_flags)
    {
        flat_block = j.bflags[(int64_t(b) * j.oby + by) * j.obx + bx] == 0;
        flat_bits = j.flags[int64_t(j.B) * j.TH * j.TW + b] == 0;
        v0 = convert_in<To>(ld(I, int64_t(y0) * W + x0));
    }
    if (dense)
        band = nq >= 32 ? 0xffffffffu : ((1u << nq) - 1u);
    else if (use_flags && !flat_block)
    {
        // Band tiles (GB:154-176): a tile is a band tile when an edge tile lies in its 3x3 window,
        // clamped to the tile grid.  The edge flags of the block's tiles and their neighbours go to
        // LDS with a border of zeros (tiles outside the grid), the block's band tiles are derived
        // there from fixed 3 x 3 windows, and each pixel reads its tile's bit.  Both tables occupy
        // the start of the pixel tile, which is staged only after the barrier below.
        uint8_t* ef = smem_raw;
        uint8_t* btl = smem_raw + kBlurMaxFlagTiles;
        const int32_t tx_lo = x0 / ts, tx_hi = min(x0 + kBlurBX - 1, W - 1) / ts;
        const int32_t ty_lo = y0 / ts, ty_hi = min(y0 + RB - 1, H - 1) / ts;
        const int32_t ex_lo = max(tx_lo - 1, 0), ex_hi = min(tx_hi + 1, j.TW - 1);
        const int32_t ey_lo = max(ty_lo - 1, 0), ey_hi = min(ty_hi + 1, j.TH - 1);
        const int32_t ew = ex_hi - ex_lo + 1, eh = ey_hi - ey_lo + 1;
        const int32_t pw = ew + 2, ph = eh + 2; // padded: tile (ex_lo + c - 1, ey_lo + r - 1) at r * pw + c
        const auto E = as_global(j.flags + uint64_t(b) * j.TH * j.TW);
        for (int32_t r = ly0; r < ph; r += 4)
            for (int32_t c = lx; c < pw; c += 64)
            {
                const bool in = r >= 1 && r <= eh && c >= 1 && c <= ew;
                ef[r * pw + c] = in ? E[int64_t(ey_lo + r - 1) * j.TW + (ex_lo + c - 1)] : uint8_t(0);
            }
        __syncthreads();
        const int32_t bw = tx_hi - tx_lo + 1, bh = ty_hi - ty_lo + 1;
        const int32_t ox = tx_lo - ex_lo + 1, oy = ty_lo - ey_lo + 1; // padded position of tile (tx_lo, ty_lo)
        for (int32_t r = ly0; r < bh; r += 4)
            for (int32_t c = lx; c < bw; c += 64)
            {
                const uint8_t* e = ef + (oy + r) * pw + (ox + c);
                btl[r * bw + c] = uint8_t(e[-pw - 1] | e[-pw] | e[-pw + 1] | e[-1] | e[0] | e[1] | e[pw - 1] | e[pw] |
                                          e[pw + 1]);
            }
        __syncthreads();
        const int32_t bx_t = x / ts - tx_lo;
#pragma unroll
        for (int q = 0; q < P; ++q)
            if (q < nq && btl[((yt + q) / ts - ty_lo) * bw + bx_t] != 0)
                band |= 1u << q;
    }
    if (flat_block || !__syncthreads_or(band != 0u))
    {
        // With edge flags, no band pixel means that no tile of the block is an edge tile: every
        // pixel equals its right and lower neighbours in the image, so the block holds the value
        // of its first pixel (x0, y0), and, unless the image holds a negative zero, the same bits.
        if (use_flags && flat_bits)
        {
            const To v = v0;
            if constexpr (kF32)
            {
                if (vec4)
                {
                    if (cx4 >= W)
                        return;
                    const float4_v v4 = { v, v, v, v };
#pragma unroll
                    for (int r = 0; r < R4; ++r)
                        if (ry4 + 16 * r < H)
                            *(gptr<float4_v>)(O + int64_t(ry4 + 16 * r) * W + cx4) = v4;
                    return;
                }
            }
#pragma unroll
            for (int q = 0; q < P; ++q)
                if (q < nq)
                    st(O, int64_t(yt + q) * W + x, v);
            return;
        }
        if constexpr (kF32)
        {
            if (vec4)
            {
                if (cx4 >= W)
                    return;
                float4_v pre[R4];
#pragma unroll
                for (int r = 0; r < R4; ++r)
                    if (ry4 + 16 * r < H)
                        pre[r] = *(gptr<const float4_v>)(I + int64_t(ry4 + 16 * r) * W + cx4);
#pragma unroll
                for (int r = 0; r < R4; ++r)
                    if (ry4 + 16 * r < H)
                        *(gptr<float4_v>)(O + int64_t(ry4 + 16 * r) * W + cx4) = pre[r];
                return;
            }
        }
        To v[P];
#pragma unroll
        for (int q = 0; q < P; ++q)
            if (q < nq)
                v[q] = convert_in<To>(ld(I, int64_t(yt + q) * W + x)); // images.clone().to(dtype) (GB:444)
#pragma unroll
        for (int q = 0; q < P; ++q)
            if (q < nq)
                st(O, int64_t(yt + q) * W + x, v[q]);
        return;
    }
    // stage the block and its halo, converted to the output type (GB:221)
    bool staged = false;
    if constexpr (kF32)
    {
        // float32 block away from the image border: no reflection, and the rows are read with
        // aligned 16-byte loads from column x0 - hx (hx: the halo rounded up to 4 columns); each
        // loaded column c lands at tile column c - (x0 - h) when that is inside the tile
        const int32_t hx = (h + 3) & ~3;
        if (vec4 && x0 >= hx && x0 + kBlurBX + hx <= W && y0 >= h && y0 + RB + h <= H)
        {
            constexpr int kVB = 4; // loads in flight per thread
            const int32_t n4 = (kBlurBX + 2 * hx) / 4;
            const int32_t items = LH * n4;
            const auto src = I + (int64_t(y0 - h) * W + (x0 - hx));
            for (int32_t t0 = int32_t(threadIdx.x); t0 < items; t0 += 256 * kVB)
            {
                float4_v v[kVB];
#pragma unroll
                for (int u = 0; u < kVB; ++u)
                {
                    const int32_t t = t0 + 256 * u;
                    if (t < items)
                    {
                        const int32_t r = t / n4, kq = t - r * n4;
                        v[u] = *(gptr<const float4_v>)(src + (int64_t(r) * W + 4 * kq));
                    }
                }
#pragma unroll
                for (int u = 0; u < kVB; ++u)
                {
                    const int32_t t = t0 + 256 * u;
                    if (t < items)
                    {
                        const int32_t r = t / n4, kq = t - r * n4;
                        const int32_t c0 = 4 * kq - hx + h;
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (c0 + e >= 0 && c0 + e < LW)
                                tile[r * LW + c0 + e] = v[u][e];
                    }
                }
            }
            staged = true;
        }
    }
    // elsewhere thread (lx, ly0) stages columns lx and lx + 64 of rows ly0, ly0 + 4, ... (reflect
    // padding); reads go out in batches of 2 columns x 8 rows before the batch is stored
    constexpr int kStageRows = 8;
    if (!staged)
    {
        const int32_t cxa = lx, cxb = 64 + lx;
        const bool inb = cxb < LW; // LW <= 128 when the halo fits in LDS with RB >= 16
        const int64_t xa = reflect_index(x0 + cxa - h, W), xb = inb ? reflect_index(x0 + cxb - h, W) : 0;
        for (int32_t t0 = ly0; t0 < LH; t0 += 4 * kStageRows)
        {
            To va[kStageRows], vb[kStageRows];
#pragma unroll
            for (int u = 0; u < kStageRows; ++u)
            {
                const int32_t ty = t0 + 4 * u;
                const int64_t row = reflect_index(y0 + min(ty, LH - 1) - h, H) * W;
                va[u] = ty < LH ? convert_in<To>(ld(I, row + xa)) : OutOps<To>::zero();
                vb[u] = (inb && ty < LH) ? convert_in<To>(ld(I, row + xb)) : OutOps<To>::zero();
            }
#pragma unroll
            for (int u = 0; u < kStageRows; ++u)
            {
                const int32_t ty = t0 + 4 * u;
                if (ty < LH)
                {
                    tile[ty * LW + cxa] = va[u];
                    if (inb)
                        tile[ty * LW + cxb] = vb[u];
                }
            }
        }
        for (int32_t cx = 128 + lx; cx < LW; cx += 64) // halos wider than 32 pixels
        {
            const int64_t xx = reflect_index(x0 + cx - h, W);
            for (int32_t ty = ly0; ty < LH; ty += 4)
                tile[ty * LW + cx] = convert_in<To>(ld(I, reflect_index(y0 + ty - h, H) * W + xx));
        }
    }
    __syncthreads();
    if (x >= W)
        return;
    if constexpr (KT > 0)
    {
        // GB:217-230 per pixel: x offset i outer, y offset j inner.  The thread's P pixels are
        // consecutive rows of one column, so for each i the column's P + KT - 1 tile values are read
        // once and every pixel's accumulator takes its KT taps from them, in the same order.
        To acc[P];
#pragma unroll
        for (int q = 0; q < P; ++q)
            acc[q] = OutOps<To>::zero();
        if (band != 0u)
        {
#pragma unroll
            for (int32_t i = 0; i < KT; ++i)
            {
                const To* col = tile + (lx + i) + (ly0 * P) * LW;
                To c[P + KT - 1];
#pragma unroll
                for (int t = 0; t < P + KT - 1; ++t)
                    c[t] = col[t * LW];
#pragma unroll
                for (int q = 0; q < P; ++q)
#pragma unroll
                    for (int32_t jj = 0; jj < KT; ++jj)
                        acc[q] = OutOps<To>::mac(acc[q], weights[i * KT + jj], c[q + jj]);
            }
        }
#pragma unroll
        for (int q = 0; q < P; ++q)
        {
            if (q >= nq)
                break;
            const int32_t ly = ly0 * P + q;
            const To result = (band & (1u << q)) ? (sparse ? OutOps<To>::div(acc[q], norm) : acc[q])
                                                 : tile[(ly + h) * LW + lx + h];
            st(O, int64_t(y0 + ly) * W + x, result);
        }
        return;
    }
    // Other sizes: the same with the taps of a column taken kTaps at a time, so that a tile value read once
    // still serves up to kTaps pixels of the thread (10 dense 1080p images, k = 11: 0.50 ms with one tile read
    // and one weight read per tap and pixel, 0.14 ms so, 0.097 ms with the taps compiled in; float64 and float16
    // outputs, which take this loop for every size: k = 5 0.20 -> 0.12 and 0.22 -> 0.09, k = 11 0.69 -> 0.27 and
    // 0.59 -> 0.19, sparse k = 3 0.102 -> 0.096 and 0.091).
    constexpr int kTaps = 8;
    To acc[P];
#pragma unroll
    for (int q = 0; q < P; ++q)
        acc[q] = OutOps<To>::zero();
    if (band != 0u)
    {
        for (int32_t i = 0; i < k; ++i)
        {
            const To* col = tile + (lx + i) + (ly0 * P) * LW;
            const To* wcol = weights + i * k;
            for (int32_t j0 = 0; j0 < k; j0 += kTaps)
            {
                const int32_t taps = min(k - j0, kTaps); // values j0 .. j0 + P + taps - 2 of the column
                To c[P + kTaps - 1];
#pragma unroll
                for (int t = 0; t < P + kTaps - 1; ++t)
                    if (t < P - 1 + taps)
                        c[t] = col[(j0 + t) * LW];
#pragma unroll
                for (int32_t jj = 0; jj < kTaps; ++jj)
                {
                    if (jj >= taps)
                        break;
                    const To w = wcol[j0 + jj];
#pragma unroll
                    for (int q = 0; q < P; ++q)
                        acc[q] = OutOps<To>::mac(acc[q], w, c[q + jj]);
                }
            }
        }
    }
    // With an early exit this loop stays a loop for __half, and acc an array in private memory (dense k = 3 85 us
    // instead of 75); float64 is 2 % faster with it (dense k = 11 303 us and 310).
    constexpr bool kExit = !std::is_same_v<To, __half>;
#pragma unroll
    for (int q = 0; q < P; ++q)
    {
        if (q >= nq)
        {
            if constexpr (kExit)
                break;
            else
                continue;
        }
        const int32_t ly = ly0 * P + q;
        const To result = (band & (1u << q)) ? (sparse ? OutOps<To>::div(acc[q], norm) : acc[q])
                                             : tile[(ly + h) * LW + lx + h];
        st(O, int64_t(y0 + ly) * W + x, result);
    }
}

// Edge-tile flags and negative-zero flags of B images with a TH x TW tile grid, in whole 32-bit
// words (they are cleared by a fill kernel).
static int64_t
flag_region_bytes(int64_t B, int64_t TH, int64_t TW, int64_t oby, int64_t obx)
{
    return (B * (TH * TW + 1 + oby * obx) + 3) & ~int64_t(3);
}

int64_t
blur_tile_flag_bytes(int64_t B, int64_t H, int64_t W, int kernel_size)
{
    const int64_t ts = kernel_size / 2;
    if (ts <= 0 || B == 0)
        return 0;
    // output blocks of 16 rows at the least
    return flag_region_bytes(B, H / ts + 1, W / ts + 1, (H + 15) / 16, (W + kBlurBX - 1) / kBlurBX);
}

size_t
blur_job_bytes(size_t n)
{
    return 2 * n * sizeof(BlurJob); // a table for either pass
}

template <typename Ti, typename To, int RB>
static void
run_blur_rb(std::vector<BlurJob>& jobs, BlurJob* djobs, Uploader& up, int k, bool sparse, const To* weights, To norm,
            uint8_t* flags, hipStream_t st)
{
    const int32_t ts = k / 2;
    const bool use_band = sparse && k > 1;
    // the edge pass reads 4 pixels per thread with 16-byte loads for float32 images of width % 4 == 0
    bool vec = std::is_same_v<Ti, float>;
    for (auto& j : jobs)
        vec = vec && (j.W % 4 == 0) && (reinterpret_cast<uintptr_t>(j.in) % 16 == 0);
    // the float32 edge pass takes blocks of kEdgeRows rows (fewer registers per thread, more waves)
    constexpr int kEdgeRows = RB > 32 ? 32 : RB;
    uint64_t pb = 0, eb = 0, fbytes = 0;
    for (auto& j : jobs)
    {
        j.by = blocks_for(j.H, vec ? kEdgeRows : RB);
        j.bx = blocks_for(j.W, vec ? 4 * kBlurBX : kBlurBX);
        j.p_begin = eb; // edge-pass blocks first
        eb += uint64_t(j.bx) * j.by * j.B;
        j.obx = blocks_for(j.W, kBlurBX);
        j.oby = blocks_for(j.H, RB);
        if (use_band)
        {
            j.TH = j.H / ts + 1;
            j.TW = j.W / ts + 1;
            j.flags = flags + fbytes;
            j.bflags = j.flags + int64_t(j.B) * (int64_t(j.TH) * j.TW + 1);
            fbytes += uint64_t(flag_region_bytes(j.B, j.TH, j.TW, j.oby, j.obx));
        }
    }
    const int32_t n = int32_t(jobs.size());
    // the tile pass has its own block layout: a second table behind the first, and one copy for both (a copy
    // between the passes kept 30 1080p images waiting: 162 -> 160 us, nothing on images seen for the first time)
    jobs.resize(2 * size_t(n));
    for (int32_t i = 0; i < n; ++i)
    {
        BlurJob& j = jobs[n + i];
        j = jobs[i];
        j.by = j.oby; // the output pass's blocks: the band-block flags' grid
        j.bx = j.obx;
        j.p_begin = pb;
        pb += uint64_t(j.bx) * j.by * j.B;
    }
    if (pb == 0)
        return;
    THULL_CHECK(pb < (uint64_t(1) << 31), "blur batch too large");
    up.upload(djobs, jobs.data(), jobs.size() * sizeof(BlurJob), st);
    if (use_band)
    {
        THULL_CHECK(eb < (uint64_t(1) << 31), "blur batch too large");
        launch_fill_u32(reinterpret_cast<uint32_t*>(flags), fbytes / 4, 0u, st);
        if (vec)
        {
            if constexpr (std::is_same_v<Ti, float>)
                blur_edge_flags_f32x4_kernel<kEdgeRows>
                    <<<unsigned(eb), 256, 0, st>>>(djobs, n, ts, RB);
        }
        else
            blur_edge_flags_kernel<Ti, RB><<<unsigned(eb), 256, 0, st>>>(djobs, n, ts, RB);
        THULL_LAUNCH_CHECK();
    }
    djobs += n;
    const int32_t h = k / 2;
    // the pixel tile, which also holds the two band-tile tables before it is staged
    const size_t lds = std::max(size_t(kBlurBX + 2 * h) * (RB + 2 * h) * sizeof(To), size_t(2 * kBlurMaxFlagTiles));
    // blocks without band pixels copy with 16-byte accesses when every image allows it
    bool vec4 = std::is_same_v<Ti, float> && std::is_same_v<To, float>;
    for (const auto& j : jobs)
        vec4 = vec4 && j.W % 4 == 0 && reinterpret_cast<uintptr_t>(j.in) % 16 == 0 &&
               reinterpret_cast<uintptr_t>(j.out) % 16 == 0;
    const int32_t tsl = ts > 0 ? ts : 1;
    // float outputs of the odd sizes up to 15 take a kernel with the taps unrolled (10 dense 1080p images, taps
    // 8 at a time and unrolled: k = 11 0.140 and 0.097 ms; the runtime loop over taps took 0.50 and, k = 13, 0.66;
    // unrolling rows only costs k = 15 4 %)
    constexpr bool spec = std::is_same_v<To, float> && (std::is_same_v<Ti, float> || std::is_same_v<Ti, uint8_t>);
    if (spec && k == 3)
        blur_tile_kernel<Ti, To, RB, spec ? 3 : 0><<<unsigned(pb), 256, lds, st>>>(djobs, n, k, tsl, sparse, weights,
                                                                                   norm, vec4);
    else if (spec && k == 5)
        blur_tile_kernel<Ti, To, RB, spec ? 5 : 0><<<unsigned(pb), 256, lds, st>>>(djobs, n, k, tsl, sparse, weights,
                                                                                   norm, vec4);
    else if (spec && k == 7)
        blur_tile_kernel<Ti, To, RB, spec ? 7 : 0><<<unsigned(pb), 256, lds, st>>>(djobs, n, k, tsl, sparse, weights,
                                                                                   norm, vec4);
    else if (spec && k == 9)
        blur_tile_kernel<Ti, To, RB, spec ? 9 : 0><<<unsigned(pb), 256, lds, st>>>(djobs, n, k, tsl, sparse, weights,
                                                                                   norm, vec4);
    else if (spec && k == 11)
        blur_tile_kernel<Ti, To, RB, spec ? 11 : 0><<<unsigned(pb), 256, lds, st>>>(djobs, n, k, tsl, sparse, weights,
                                                                                    norm, vec4);
    else if (spec && k == 13 && RB == 64)
        blur_tile_kernel<Ti, To, RB, spec ? 13 : 0><<<unsigned(pb), 256, lds, st>>>(djobs, n, k, tsl, sparse, weights,
                                                                                    norm, vec4);
    else if (spec && k == 15 && RB == 64)
        blur_tile_kernel<Ti, To, RB, spec ? 15 : 0><<<unsigned(pb), 256, lds, st>>>(djobs, n, k, tsl, sparse, weights,
                                                                                    norm, vec4);
    else
        blur_tile_kernel<Ti, To, RB, 0><<<unsigned(pb), 256, lds, st>>>(djobs, n, k, tsl, sparse, weights, norm,
                                                                         vec4);
    THULL_LAUNCH_CHECK();
}

template <typename Ti, typename To>
static void
run_blur(std::vector<BlurJob>& jobs, BlurJob* djobs, Uploader& up, int k, bool sparse, const To* weights, To norm,
         uint8_t* flags, hipStream_t st)
{
    const int32_t h = k / 2;
    if (size_t(kBlurBX + 2 * h) * (64 + 2 * h) * sizeof(To) <= 48 * 1024)
        run_blur_rb<Ti, To, 64>(jobs, djobs, up, k, sparse, weights, norm, flags, st);
    else if (size_t(kBlurBX + 2 * h) * (16 + 2 * h) * sizeof(To) <= 48 * 1024)
        run_blur_rb<Ti, To, 16>(jobs, djobs, up, k, sparse, weights, norm, flags, st);
    else
        throw Error("kernel_size too large for the LDS tile");
}

template <typename Ti>
static void
run_blur_out(std::vector<BlurJob>& jobs, BlurJob* djobs, Uploader& up, int k, bool sparse, const void* weights,
             double norm, int32_t out_dtype, uint8_t* flags, hipStream_t st)
{
    switch (out_dtype)
    {
    case kF16:
        run_blur<Ti, __half>(jobs, djobs, up, k, sparse, static_cast<const __half*>(weights), __float2half(float(norm)),
                             flags, st);
        break;
    case kF32:
        run_blur<Ti, float>(jobs, djobs, up, k, sparse, static_cast<const float*>(weights), float(norm), flags, st);
        break;
    case kF64:
        run_blur<Ti, double>(jobs, djobs, up, k, sparse, static_cast<const double*>(weights), norm, flags, st);
        break;
    default:
        throw Error("gaussian_blur: output dtype must be floating point");
    }
}

// Blurs a batch of images of one input dtype into outputs of one output dtype.
// `weights` is a device table of k*k weights in the output type; `norm` the
// weight sum in the output type (exactly representable in double).
void
launch_gaussian_blur_batch(const BlurImage* imgs, int32_t n, int32_t in_dtype, int k, bool sparse,
                           const void* weights, double norm, int32_t out_dtype, uint8_t* flags, void* job_buf,
                           Uploader& up, hipStream_t st)
{
    std::vector<BlurJob> jobs;
    for (int32_t i = 0; i < n; ++i)
    {
        const BlurImage& im = imgs[i];
        if (im.B == 0 || im.H == 0 || im.W == 0)
            continue;
        THULL_CHECK(im.H < (int64_t(1) << 31) && im.W < (int64_t(1) << 31) && im.H * im.W < (int64_t(1) << 40),
                    "image too large");
        BlurJob j{};
        j.in = im.in;
        j.out = im.out;
        j.B = int32_t(im.B);
        j.H = int32_t(im.H);
        j.W = int32_t(im.W);
        jobs.push_back(j);
    }
    if (jobs.empty())
        return;
    BlurJob* djobs = static_cast<BlurJob*>(job_buf);
    switch (in_dtype)
    {
    case kBool:
    case kU8:
        run_blur_out<uint8_t>(jobs, djobs, up, k, sparse, weights, norm, out_dtype, flags, st);
        break;
    case kI8:
        run_blur_out<int8_t>(jobs, djobs, up, k, sparse, weights, norm, out_dtype, flags, st);
        break;
    case kI16:
        run_blur_out<int16_t>(jobs, djobs, up, k, sparse, weights, norm, out_dtype, flags, st);
        break;
    case kI32:
        run_blur_out<int32_t>(jobs, djobs, up, k, sparse, weights, norm, out_dtype, flags, st);
        break;
    case kI64:
        run_blur_out<int64_t>(jobs, djobs, up, k, sparse, weights, norm, out_dtype, flags, st);
        break;
    case kF16:
        run_blur_out<__half>(jobs, djobs, up, k, sparse, weights, norm, out_dtype, flags, st);
        break;
    case kF32:
        run_blur_out<float>(jobs, djobs, up, k, sparse, weights, norm, out_dtype, flags, st);
        break;
    case kF64:
        run_blur_out<double>(jobs, djobs, up, k, sparse, weights, norm, out_dtype, flags, st);
        break;
    default:
        throw Error("gaussian_blur: unsupported input dtype");
    }
}

} // namespace thull
