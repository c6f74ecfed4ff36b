// Marching cubes for CDNA4 over a sorted vertex set (sparse) or a dense grid.
//
// Reference (vc-bonn/torchhull, src/torchhull/_C/src/marching_cubes_cuda.cu, MC):
// classification MC:146-223, generation MC:242-374, interpolation MC:72-97,
// edge keys MC:99-112, unique vertices MC:674-693.
//
// The reference emits a triangle soup, keys every soup vertex by
// (ravel(lower endpoint) << 3 | direction) and runs unique_dim (a full sort)
// to build the compact mesh, whose vertices come out in ascending key order.
// This implementation reaches the same mesh without sorting: an output vertex
// is a grid edge (p, d) owned by its lower endpoint p.  An edge is emitted iff
// its endpoints lie on different sides of the isolevel and at least one of the
// (up to four) cells around it is complete; for a complete cell the case table
// lists exactly its sign-changing edges, so this is the set of edges the
// reference's soup contains.  The vertex list is sorted by ravel index, so an
// exclusive scan of popcount(edge mask) over it numbers the edges in the
// reference's ascending key order, and a face corner finds its vertex index
// by a rank lookup of p.  Duplicate soup vertices of the reference are
// bit-identical (same endpoints and values), so computing each edge's position
// once gives the same coordinates.

#include <algorithm>
#include <type_traits>

#include "mc_cases.h"
#include "kernels.h"
#include "scan.h"

namespace thull
{

__constant__ McCaseTable c_cases = mc_build_case_table();

// Case corner b -> offset (bit0 x, bit1 y, bit2 z) in the cell.
__constant__ uint8_t c_corner_off[8] = { 0b000, 0b001, 0b101, 0b100, 0b010, 0b011, 0b111, 0b110 };
// the same table for compile-time indexing in unrolled loops
constexpr uint8_t c_corner_off_host[8] = { 0b000, 0b001, 0b101, 0b100, 0b010, 0b011, 0b111, 0b110 };
// Edge e -> lower endpoint offset (bits as above) and axis (0 x, 1 y, 2 z).
__constant__ uint8_t c_edge_low[12] = { kMcEdgeLow[0], kMcEdgeLow[1], kMcEdgeLow[2],  kMcEdgeLow[3],
                                        kMcEdgeLow[4], kMcEdgeLow[5], kMcEdgeLow[6],  kMcEdgeLow[7],
                                        kMcEdgeLow[8], kMcEdgeLow[9], kMcEdgeLow[10], kMcEdgeLow[11] };
__constant__ uint8_t c_edge_axis[12] = { kMcEdgeAxis[0], kMcEdgeAxis[1], kMcEdgeAxis[2],  kMcEdgeAxis[3],
                                         kMcEdgeAxis[4], kMcEdgeAxis[5], kMcEdgeAxis[6],  kMcEdgeAxis[7],
                                         kMcEdgeAxis[8], kMcEdgeAxis[9], kMcEdgeAxis[10], kMcEdgeAxis[11] };

constexpr uint32_t kInfoComplete = 1u << 8;
constexpr int kInfoSignShift = 9;

struct BitmapLookup
{
    const uint32_t* bitmap;
    const uint32_t* prefix;

    __device__ __forceinline__ bool
    find(const McGrid& g, uint32_t x, uint32_t y, uint32_t z, uint32_t& pos) const
    {
        const uint64_t w = g.bitmap_offset + (uint64_t(z) * g.dims[1] + y) * g.row_words + (x >> 5);
        const uint32_t word = bitmap[w];
        const uint32_t pre = prefix[w]; // read with the word, not after the presence test
        const uint32_t bit = x & 31u;
        if (((word >> bit) & 1u) == 0u)
            return false;
        pos = pre + __popc(word & ((1u << bit) - 1u));
        return true;
    }

    // Split lookup for batching: probe() issues the bitmap and prefix reads,
    // present() and rank() use them, so that the probes of several points are
    // in flight together.
    struct Probe
    {
        uint32_t word, pre, bit;
    };
    __device__ __forceinline__ Probe
    probe(const McGrid& g, uint32_t x, uint32_t y, uint32_t z) const
    {
        const uint64_t w = g.bitmap_offset + (uint64_t(z) * g.dims[1] + y) * g.row_words + (x >> 5);
        return Probe{ bitmap[w], prefix[w], x & 31u };
    }
    __device__ __forceinline__ bool
    present(const Probe& p) const
    {
        return ((p.word >> p.bit) & 1u) != 0u;
    }
    __device__ __forceinline__ uint32_t
    rank(const Probe& p) const
    {
        return p.pre + __popc(p.word & ((1u << p.bit) - 1u));
    }
};

struct VertexRef
{
    uint32_t scene, x, y, z;
};

__device__ __forceinline__ VertexRef
vertex_ref(const McPlan& p, uint64_t i)
{
    const uint64_t k = p.vertices[i];
    return VertexRef{ key_scene(k), key_x(k), key_y(k), key_z(k) };
}

template <typename V>
__device__ __forceinline__ V
value_at(const McPlan& p, uint32_t pos)
{
    return static_cast<const V*>(p.values)[pos];
}

// MC:72-97
__device__ __forceinline__ void
interpolate_vertex(float iso, const uint32_t p1[3], const uint32_t p2[3], float v1, float v2, float out[3])
{
    const float eps = 1e-5f;
    if (fabsf(iso - v1) < eps)
    {
        out[0] = float(p1[0]);
        out[1] = float(p1[1]);
        out[2] = float(p1[2]);
        return;
    }
    if (fabsf(iso - v2) < eps)
    {
        out[0] = float(p2[0]);
        out[1] = float(p2[1]);
        out[2] = float(p2[2]);
        return;
    }
    if (fabsf(v1 - v2) < eps)
    {
        out[0] = float(p1[0]);
        out[1] = float(p1[1]);
        out[2] = float(p1[2]);
        return;
    }
    const float t = (iso - v1) / (v2 - v1);
#pragma unroll
    for (int a = 0; a < 3; ++a)
        out[a] = lerp_ref(float(p1[a]), float(p2[a]), t);
}

__device__ __forceinline__ void
finish_vertex(const McGrid& g, const float v[3], float* out)
{
#pragma unroll
    for (int a = 0; a < 3; ++a)
    {
        float r = v[a];
        if (g.out_mode == 1)
        {
            r = r * g.scale[a]; // verts *= scale (MC:528)
            r = r - 1.0f;       // verts -= 1 (MC:529)
        }
        else if (g.out_mode == 2)
        {
            r = fmaf(g.scale[a], r, g.corner[a]); // to_global_coordinates (visual_hull_cuda.cu:929-937)
        }
        out[a] = r;
    }
}

// ---------------------------------------------------------------------------
// Pass 1: cell case, completeness and edge sign changes per vertex
// ---------------------------------------------------------------------------

// The two corners x and x + 1 of one (y, z) row of a cell share a bitmap word (and its prefix): 3 row
// words plus the vertex's own word are read instead of 7 words and 7 prefixes, and the +x neighbour of a
// present vertex i is vertex i + 1.
struct RowProbe
{
    uint64_t w;     // word of x
    uint32_t word;  // bitmap word of x
    uint32_t pre;   // prefix of that word (read with it)
    uint32_t next;  // bitmap word of x + 1 when x % 32 == 31 (else unused)
    bool p0, p1;    // x, x + 1 present (x + 1 only when inside the grid)
};

__device__ __forceinline__ RowProbe
row_probe(const BitmapLookup& lk, const McGrid& g, uint32_t x, uint32_t y, uint32_t z, bool in_row, bool inx)
{
    RowProbe q{};
    if (!in_row)
        return q;
    q.w = g.bitmap_offset + (uint64_t(z) * g.dims[1] + y) * g.row_words + (x >> 5);
    const uint32_t b = x & 31u;
    // word x + 1 is the next word when x % 32 == 31 (inside the row: x + 1 is in the grid), else
    // the same word: both reads are issued together, with no branch around the second
    q.word = lk.bitmap[q.w];
    q.next = lk.bitmap[q.w + ((inx && b == 31u) ? 1u : 0u)];
    q.pre = lk.prefix[q.w];
    q.p0 = ((q.word >> b) & 1u) != 0u;
    if (inx)
        q.p1 = (b != 31u ? (q.word >> (b + 1u)) & 1u : q.next & 1u) != 0u;
    return q;
}

template <typename V, bool UNIFORM>
__device__ __forceinline__ void
mc_classify_vertex(const McPlan& p, const BitmapLookup& lk, const McGrid& g, uint64_t i, const VertexRef& r,
                   uint32_t& info, uint32_t& ntv)
{
    const V iso = static_cast<V>(p.iso);
    constexpr uint32_t corner[7] = { 1u, 4u, 3u, 2u, 5u, 6u, 7u };
    bool found[7];
    bool inx, iny, inz;
    inx = r.x + 1 < g.dims[0];
    iny = r.y + 1 < g.dims[1];
    inz = r.z + 1 < g.dims[2];
    // rows (dy, dz) = (0, 0), (1, 0), (0, 1), (1, 1); row (0, 0) holds the vertex itself
    const RowProbe q00 = row_probe(lk, g, r.x, r.y, r.z, true, inx);
    const RowProbe q10 = row_probe(lk, g, r.x, r.y + 1, r.z, iny, inx);
    const RowProbe q01 = row_probe(lk, g, r.x, r.y, r.z + 1, inz, inx);
    const RowProbe q11 = row_probe(lk, g, r.x, r.y + 1, r.z + 1, iny && inz, inx);
    // corners 1 (x+1,y,z), 4 (x,y+1,z), 3 (x,y,z+1), 2 (x+1,y,z+1), 5 (x+1,y+1,z), 6 (x+1,y+1,z+1), 7 (x,y+1,z+1)
    found[0] = q00.p1;
    found[1] = q10.p0;
    found[2] = q01.p0;
    found[3] = q01.p1;
    found[4] = q10.p1;
    found[5] = q11.p1;
    found[6] = q11.p0;
    bool complete = inx && iny && inz; // MC:199
#pragma unroll
    for (int k = 0; k < 7; ++k)
        complete = complete && found[k];
    // Values are read as pairs of consecutive vertices, the corners x and x + 1 of a row: the
    // vertex itself and its +x neighbour (which follows it when present), and in the rows
    // (y + 1, z), (y, z + 1), (y + 1, z + 1) the first present corner x' at rank r of x and, in a
    // complete cell, x + 1 at r + 1.  A pair starts at a = min(r, nverts - 2) (some neighbour is
    // present whenever one is read, so nverts >= 2), and the value of r is its first element when
    // a == r, else its second (r = nverts - 1); the second corner of a pair is only read in a
    // complete cell, where r + 1 < nverts.
    typedef V pair_t __attribute__((ext_vector_type(2), aligned(sizeof(V))));
    typedef __attribute__((address_space(1))) const pair_t global_pair_t;
    const V* vals = static_cast<const V*>(p.values);
    const uint32_t last2 = uint32_t(p.nverts) - 2u; // used only when nverts >= 2
    V vg, vrow[4][2] = {}; // entries of absent corners are never compared
    if (found[0])
    {
        const pair_t v2 = *(global_pair_t*)(vals + i); // i + 1 < nverts
        vg = v2.x;
        vrow[0][1] = v2.y;
    }
    else
        vg = vals[i];
    const auto row_pair = [&](const RowProbe& q, int row) {
        const uint32_t b = r.x & 31u;
        const uint32_t r0 = q.pre + __popc(q.word & ((1u << b) - 1u));
        const uint32_t a = min(r0, last2);
        const pair_t v2 = *(global_pair_t*)(vals + a);
        vrow[row][0] = a == r0 ? v2.x : v2.y;
        vrow[row][1] = v2.y;
    };
    if (found[1] || complete)
        row_pair(q10, 1);
    if (found[2] || complete)
        row_pair(q01, 2);
    if (complete)
        row_pair(q11, 3);
    // case-corner order 1, 4, 3, 2, 5, 6, 7: (x+1,y,z), (x,y+1,z), (x,y,z+1), (x+1,y,z+1),
    // (x+1,y+1,z), (x+1,y+1,z+1), (x,y+1,z+1)
    const V cv[7] = { vrow[0][1], vrow[1][0], vrow[2][0], vrow[2][1], vrow[1][1], vrow[3][1], vrow[3][0] };
    const bool below_g = vg < iso;
    bool below[7];
#pragma unroll
    for (int k = 0; k < 7; ++k)
        below[k] = (k < 3 ? found[k] : complete) && cv[k] < iso;
    uint32_t sc = 0u;
#pragma unroll
    for (int d = 0; d < 3; ++d)
        if (found[d] && below[d] != below_g)
            sc |= 1u << d;
    uint32_t ci = 0u; // missing corner or boundary vertex: cubeindex 0 (MC:206-211)
    if (complete)
    {
        ci = below_g ? 1u : 0u;
#pragma unroll
        for (int k = 0; k < 7; ++k)
            ci |= below[k] ? (1u << corner[k]) : 0u;
    }
    info = ci | (complete ? kInfoComplete : 0u) | (sc << kInfoSignShift);
    ntv = complete ? uint32_t(c_cases.count[ci]) : 0u;
}

template <typename V>
__global__ __launch_bounds__(256) void
mc_classify_kernel(McPlan p, BitmapLookup lk, uint32_t* __restrict__ info, uint32_t* __restrict__ ntv)
{
    const uint64_t i = uint64_t(xcd_block(blockIdx.x, gridDim.x)) * 256 + threadIdx.x;
    if (i >= p.nverts)
        return;
    const VertexRef r = vertex_ref(p, i);
    const uint32_t s0 = __builtin_amdgcn_readfirstlane(r.scene);
    uint32_t inf, n;
    if (__all(r.scene == s0)) // one grid for the whole wave: scalar grid parameters
        mc_classify_vertex<V, true>(p, lk, wave_uniform(p.grids[s0]), i, r, inf, n);
    else
        mc_classify_vertex<V, false>(p, lk, p.grids[r.scene], i, r, inf, n);
    info[i] = inf;
    ntv[i] = n;
}

// ---------------------------------------------------------------------------
// Pass 2: emitted edges per vertex
// ---------------------------------------------------------------------------

// Emitted edges of a vertex with sign-change bits sc (info word inf).
// UNIFORM as for mc_classify_vertex: keeps the wave-uniform and per-lane copies apart.
template <bool UNIFORM>
__device__ __forceinline__ uint32_t
mc_vertex_emask(const McPlan& p, const BitmapLookup& lk, const McGrid& g, const uint32_t* __restrict__ info,
                const VertexRef& r, uint32_t inf, uint32_t sc)
{
    if (inf & kInfoComplete) // the vertex's own cell is complete: every sign-changing edge is emitted
        return sc;
    // cells sharing the edge from (x,y,z) along axis d: origins minus the two other unit vectors.
    // The six cells other than the vertex's own that these edges touch, (dx, dy, dz) offsets
    // 010, 001, 011, 100, 101, 110 (bit 2: x, 1: y, 0: z), are looked up together: all bitmap reads,
    // then all info reads, instead of one cell after the other.
    constexpr uint32_t off[6] = { 2u, 1u, 3u, 4u, 5u, 6u };
    // cells each axis needs: axis x: 010 001 011, axis y: 100 001 101, axis z: 100 010 110
    uint32_t need = 0u;
    if (sc & 1u)
        need |= 0b000111u;
    if (sc & 2u)
        need |= 0b011010u;
    if (sc & 4u)
        need |= 0b101001u;
    BitmapLookup::Probe pr[6];
    bool ok[6];
#pragma unroll
    for (int k = 0; k < 6; ++k)
    {
        const uint32_t dx = (off[k] >> 2) & 1u, dy = (off[k] >> 1) & 1u, dz = off[k] & 1u;
        ok[k] = (need & (1u << k)) && r.x >= dx && r.y >= dy && r.z >= dz;
        if (ok[k])
            pr[k] = lk.probe(g, r.x - dx, r.y - dy, r.z - dz);
    }
    uint32_t inf_k[6];
#pragma unroll
    for (int k = 0; k < 6; ++k)
    {
        ok[k] = ok[k] && lk.present(pr[k]);
        inf_k[k] = ok[k] ? info[lk.rank(pr[k])] : 0u;
    }
    uint32_t complete = 0u;
#pragma unroll
    for (int k = 0; k < 6; ++k)
        complete |= (inf_k[k] & kInfoComplete) ? (1u << k) : 0u;
    uint32_t m = 0u;
    if ((sc & 1u) && (complete & 0b000111u))
        m |= 1u;
    if ((sc & 2u) && (complete & 0b011010u))
        m |= 2u;
    if ((sc & 4u) && (complete & 0b101001u))
        m |= 4u;
    return m;
}

__global__ __launch_bounds__(256) void
mc_edges_kernel(McPlan p, BitmapLookup lk, const uint32_t* __restrict__ info, uint32_t* __restrict__ emask)
{
    const uint64_t i = uint64_t(xcd_block(blockIdx.x, gridDim.x)) * 256 + threadIdx.x;
    if (i >= p.nverts)
        return;
    // the vertex's own reads are issued together, ahead of the sign-change test (the empty asm keeps the
    // compiler from moving the key's read behind the test: 62 instead of 57 us on 24 mixed scenes)
    const uint32_t inf = info[i];
    VertexRef r = vertex_ref(p, i);
    asm volatile("" : "+v"(r.scene), "+v"(r.x), "+v"(r.y), "+v"(r.z));
    const uint32_t sc = (inf >> kInfoSignShift) & 7u;
    uint32_t m = 0u;
    if (sc != 0u)
    {
        const uint32_t s0 = __builtin_amdgcn_readfirstlane(r.scene);
        if (__all(r.scene == s0)) // one grid for the active lanes: scalar grid parameters
            m = mc_vertex_emask<true>(p, lk, wave_uniform(p.grids[s0]), info, r, inf, sc);
        else
            m = mc_vertex_emask<false>(p, lk, p.grids[r.scene], info, r, inf, sc);
    }
    emask[i] = m;
}

// ---------------------------------------------------------------------------
// Pass 3: output vertices (compact mesh)
// ---------------------------------------------------------------------------

// The output vertices of a wavefront's 64 grid vertices are one contiguous
// range (vbase is an exclusive prefix in vertex order): they are assembled in
// LDS and written with coalesced stores.
constexpr int kMcWaves = 256 / 64;

// Output vertices of the emitted edges m of vertex i into out (3 floats each).
// UNIFORM as for mc_classify_vertex: keeps the wave-uniform and per-lane copies apart.
template <typename V, bool UNIFORM>
__device__ __forceinline__ void
mc_edge_vertices(const McPlan& p, const BitmapLookup& lk, const McGrid& g, uint64_t i, const VertexRef& r, uint32_t m,
                 float v1, float* out)
{
    const uint32_t p1[3] = { r.x, r.y, r.z };
    // the far endpoints of the emitted edges (present: each edge has a sign change); reads batched
    // (the +x endpoint of a present vertex i is vertex i + 1)
    BitmapLookup::Probe pr[3];
#pragma unroll
    for (int d = 1; d < 3; ++d)
        if (m & (1u << d))
            pr[d] = lk.probe(g, r.x + (d == 0), r.y + (d == 1), r.z + (d == 2));
    float v2[3];
#pragma unroll
    for (int d = 0; d < 3; ++d)
        if (m & (1u << d))
            v2[d] = float(value_at<V>(p, d == 0 ? uint32_t(i) + 1u : lk.rank(pr[d])));
    uint32_t o = 0u;
#pragma unroll
    for (int d = 0; d < 3; ++d)
    {
        if (!(m & (1u << d)))
            continue;
        const uint32_t p2[3] = { r.x + (d == 0), r.y + (d == 1), r.z + (d == 2) };
        float v[3];
        interpolate_vertex(p.iso, p1, p2, v1, v2[d], v);
        finish_vertex(g, v, out + 3 * o);
        ++o;
    }
}

// Active-vertex gathering: a wavefront walks a run of consecutive 64-vertex chunks and
// queues the vertices that emit something (in LDS, in vertex order); every full queue of 64 is
// processed with all lanes busy.  The outputs of a batch of queued vertices are still one
// contiguous range (the vertices between them emit nothing), assembled in LDS and written with
// coalesced stores.
// 64-vertex chunks per wavefront: at most kMcVertexChunks and kMcFaceChunks (measured on the mixed
// workload: 16 and 32 chunks, 148 vs 153 and 182 us for the vertices; 8, 16 and 32 chunks, 283, 278 and
// 308 us for the faces), fewer for lists that would leave CUs idle (mc_chunks).
constexpr int kMcVertexChunks = 8;
constexpr int kMcFaceChunks = 16;

struct McQueue
{
    uint32_t v[128];
};

// Appends the lanes' vertex i where `active` to the queue of q entries; returns the new count.
__device__ __forceinline__ uint32_t
mc_enqueue(McQueue& Q, uint32_t q, bool active, uint32_t i)
{
    const uint64_t m = __ballot(active);
    const uint32_t lane = threadIdx.x & 63u;
    if (active)
        Q.v[q + uint32_t(__popcll(m & ((uint64_t(1) << lane) - 1u)))] = i;
    return q + uint32_t(__popcll(m));
}

// Moves queue entries 64 .. q - 1 to the front; returns q - 64.
__device__ __forceinline__ uint32_t
mc_dequeue64(McQueue& Q, uint32_t q)
{
    const uint32_t lane = threadIdx.x & 63u;
    wave_lds_sync();
    const uint32_t t = lane + 64u < q ? Q.v[lane + 64u] : 0u;
    wave_lds_sync();
    if (lane + 64u < q)
        Q.v[lane] = t;
    wave_lds_sync();
    return q - 64u;
}

// Output vertices of the first nb queued vertices (nb >= 1).
template <typename V>
__device__ __forceinline__ void
mc_vertices_batch(const McPlan& p, const BitmapLookup& lk, const McQueue& Q, uint32_t nb,
                  const uint32_t* __restrict__ emask, const uint32_t* __restrict__ vbase, float* __restrict__ verts,
                  float* stage)
{
    const uint32_t lane = threadIdx.x & 63u;
    const bool on = lane < nb;
    const uint32_t i = on ? Q.v[lane] : 0u;
    const uint32_t m = on ? emask[i] : 0u;
    const uint32_t out = on ? vbase[i] : 0u;
    const VertexRef r = on ? vertex_ref(p, i) : VertexRef{};
    const float v1 = on ? float(value_at<V>(p, i)) : 0.0f; // stored as float (MC:343)
    // batch range [V0, V1) of output vertices; lane 0 holds the smallest vertex
    const uint32_t V0 = __builtin_amdgcn_readfirstlane(out);
    uint32_t end = on ? out + uint32_t(__popc(m & 7u)) : 0u;
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1)
        end = max(end, __shfl_xor(end, d, 64));
    if (on)
    {
        const uint32_t s0 = __builtin_amdgcn_readfirstlane(r.scene);
        float* o = stage + 3 * (out - V0);
        if (__all(r.scene == s0)) // one grid for the active lanes: scalar grid parameters
            mc_edge_vertices<V, true>(p, lk, wave_uniform(p.grids[s0]), i, r, m, v1, o);
        else
            mc_edge_vertices<V, false>(p, lk, p.grids[r.scene], i, r, m, v1, o);
    }
    wave_lds_sync();
    const uint32_t nf = 3u * (end - V0);
    float* dst = verts + 3 * uint64_t(V0);
    for (uint32_t q = lane; q < nf; q += 64)
        dst[q] = stage[q];
    wave_lds_sync();
}

template <typename V>
__global__ __launch_bounds__(256) void
mc_vertices_kernel(McPlan p, BitmapLookup lk, int chunks, const uint32_t* __restrict__ emask,
                   const uint32_t* __restrict__ vbase, float* __restrict__ verts)
{
    __shared__ float stage[kMcWaves][64 * 3 * 3];
    __shared__ McQueue queue[kMcWaves];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint64_t v0 = (uint64_t(xcd_block(blockIdx.x, gridDim.x)) * kMcWaves + wave) * (64u * uint32_t(chunks));
    uint32_t q = 0u; // queued vertices (wave-uniform)
    for (int c = 0; c < chunks; ++c)
    {
        const uint64_t i = v0 + 64u * uint32_t(c) + lane;
        if (v0 + 64u * uint32_t(c) >= p.nverts)
            break;
        const bool valid = i < p.nverts;
        const uint32_t m = valid ? emask[i] : 0u;
        q = mc_enqueue(queue[wave], q, m != 0u, uint32_t(i));
        if (q >= 64u)
        {
            wave_lds_sync();
            mc_vertices_batch<V>(p, lk, queue[wave], 64u, emask, vbase, verts, stage[wave]);
            q = mc_dequeue64(queue[wave], q);
        }
    }
    if (q > 0u)
    {
        wave_lds_sync();
        mc_vertices_batch<V>(p, lk, queue[wave], q, emask, vbase, verts, stage[wave]);
    }
}

// ---------------------------------------------------------------------------
// Pass 4: faces (and soup vertices)
// ---------------------------------------------------------------------------

template <typename V>
__global__ __launch_bounds__(256) void
mc_faces_kernel(McPlan p,
                BitmapLookup lk,
                const uint32_t* __restrict__ info,
                const uint32_t* __restrict__ tbase,
                const uint32_t* __restrict__ emask,
                const uint32_t* __restrict__ vbase,
                const uint32_t* __restrict__ scene_vstart,
                const uint32_t* __restrict__ scene_tstart,
                bool unique,
                float* __restrict__ soup_verts,
                int64_t* __restrict__ faces)
{
    const uint64_t i = uint64_t(xcd_block(blockIdx.x, gridDim.x)) * 256 + threadIdx.x;
    if (i >= p.nverts)
        return;
    const uint32_t inf = info[i];
    if (!(inf & kInfoComplete))
        return;
    const uint32_t ci = inf & 0xffu;
    const int count = c_cases.count[ci];
    if (count == 0)
        return;
    const VertexRef r = vertex_ref(p, i);
    const McGrid& g = p.grids[r.scene];
    const uint32_t t0 = tbase[i];
    const uint32_t ts = scene_tstart[r.scene];
    const uint32_t vs = unique ? scene_vstart[r.scene] : 0u;
    for (int k = 0; k < count; ++k)
    {
        const int e = c_cases.edges[ci][k];
        const uint32_t lo = c_edge_low[e];
        const int axis = c_edge_axis[e];
        const uint32_t q1[3] = { r.x + (lo & 1u), r.y + ((lo >> 1) & 1u), r.z + ((lo >> 2) & 1u) };
        uint32_t pos1 = 0;
        lk.find(g, q1[0], q1[1], q1[2], pos1); // corner of a complete cell
        const uint32_t tv = t0 + uint32_t(k) - ts; // triangle-vertex index within the scene
        int64_t idx;
        if (unique)
        {
            idx = int64_t(vbase[pos1] + __popc(emask[pos1] & ((1u << axis) - 1u)) - vs);
        }
        else
        {
            const uint32_t q2[3] = { q1[0] + (axis == 0), q1[1] + (axis == 1), q1[2] + (axis == 2) };
            uint32_t pos2 = 0;
            lk.find(g, q2[0], q2[1], q2[2], pos2);
            float v[3];
            interpolate_vertex(p.iso, q1, q2, float(value_at<V>(p, pos1)), float(value_at<V>(p, pos2)), v);
            finish_vertex(g, v, soup_verts + 3 * uint64_t(t0 + uint32_t(k)));
            idx = int64_t(tv); // faces = arange (MC:691-692)
        }
        int col = k % 3;
        if (g.flip && col != 0)
            col = 3 - col; // flip_faces swaps columns 1 and 2 (visual_hull_cuda.cu:951-954)
        faces[3 * uint64_t((t0 + uint32_t(k)) / 3u) + col] = idx;
    }
}

// Faces of the compact mesh: per complete cell, the vertex index of each of
// its triangle corners (an edge's rank in the edge numbering), written at the
// cell's triangle-vertex slots (tbase, a multiple of 3) with flip_faces'
// column swap.  The slots of a wavefront's 64 cells are one contiguous range
// (tbase is an exclusive prefix in vertex order): they are assembled in LDS
// and written with coalesced stores.
constexpr int kMcMaxTriVerts = 15; // triangle vertices of one cell (5 triangles)

constexpr int
mc_max_case_count()
{
    const McCaseTable t = mc_build_case_table();
    int m = 0;
    for (int c = 0; c < 256; ++c)
        m = t.count[c] > m ? t.count[c] : m;
    return m;
}
static_assert(mc_max_case_count() <= kMcMaxTriVerts, "face staging holds kMcMaxTriVerts slots per cell");

// Vertex indices v[0 .. count) of the triangle corners of a cell of case ci, from the vertex base vb and edge
// mask em of its corners (meaningful where the corner is the lower endpoint of one of the case's edges).  The
// indices of the cell's 12 edges go to the lane's row of an LDS table first, which the triangle corners then
// pick from: selecting each corner's base and mask from the 8 registers took 36 VALU instructions per triangle
// corner, and every lane of a batch runs as many corners as the largest cell.  Faces
// of 24 mixed scenes: 138 -> 123 us, of a 400^3 sphere band 29 -> 25, of a level-7 hull 7.7 -> 5.7.
constexpr uint32_t kMcEdgeRow = 13; // odd: the lanes' rows start in different banks
static_assert(kMcEdgeRow <= kMcMaxTriVerts, "the edge table and the face staging share their LDS");

__device__ __forceinline__ void
case_faces(uint32_t ci, int count, uint32_t vs, const uint32_t (&vb)[8], const uint32_t (&em)[8], uint32_t* lds,
           uint32_t (&v)[kMcMaxTriVerts])
{
    uint32_t* row = lds + (threadIdx.x & 63u) * kMcEdgeRow;
    // the case's edges, all 15 in one 16-byte read
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    const u32x4 ids = *reinterpret_cast<const u32x4*>(&c_cases.edges[ci][0]);
    const uint32_t id[4] = { ids.x, ids.y, ids.z, ids.w };
#pragma unroll
    for (int e = 0; e < 12; ++e)
        row[e] = vb[kMcEdgeLow[e]] + __popc(em[kMcEdgeLow[e]] & ((1u << kMcEdgeAxis[e]) - 1u)) - vs;
#pragma unroll
    for (int k = 0; k < kMcMaxTriVerts; ++k)
        if (k - k % 3 < count)
            v[k] = row[(id[k >> 2] >> (8 * (k & 3))) & 0xffu];
}

// The indices to the lane's slots `out` of the staging that shares its LDS with the edge tables; every lane of the
// wavefront has read its table before.  flip_faces swaps columns 1 and 2 (visual_hull_cuda.cu:951-954).
__device__ __forceinline__ void
stage_faces(int count, bool flip, const uint32_t (&v)[kMcMaxTriVerts], uint32_t* out)
{
#pragma unroll
    for (int t = 0; t < kMcMaxTriVerts; t += 3)
        if (t < count)
        {
            out[t] = v[t];
            out[t + 1] = flip ? v[t + 2] : v[t + 1];
            out[t + 2] = flip ? v[t + 1] : v[t + 2];
        }
}

// Vertex indices of the triangle corners of complete cell i (case ci, count corners).
// UNIFORM as for mc_classify_vertex: keeps the wave-uniform and per-lane copies apart.
template <bool UNIFORM>
__device__ __forceinline__ void
mc_cell_faces(const McPlan& p, const BitmapLookup& lk, const McGrid& g, uint64_t i, const VertexRef& r, uint32_t ci,
              int count, uint32_t vs, const uint32_t* __restrict__ emask, const uint32_t* __restrict__ vbase,
              uint32_t* lds, uint32_t (&v)[kMcMaxTriVerts])
{
    // vertex base and edge mask of every corner that is the lower endpoint of one of the case's
    // edges (corner 0 is this vertex); all corners of a complete cell are present, reads batched
    const uint32_t lows = c_cases.lows[ci];
    uint32_t vb[8] = {}, em[8] = {};
    // corners 2q and 2q + 1 (x and x + 1) of row q = (dy, dz) are consecutive present
    // vertices: one bitmap word and prefix give the row's rank, and the two corners' vertex
    // bases and edge masks are read as pairs (element-aligned 8-byte loads)
    typedef uint32_t pair_t __attribute__((ext_vector_type(2), aligned(4)));
    typedef __attribute__((address_space(1))) const pair_t global_pair_t;
    uint32_t pos[4];
    pos[0] = uint32_t(i);
    uint64_t w[4];
    uint32_t word[4];
    const uint32_t b = r.x & 31u;
#pragma unroll
    for (int q = 1; q < 4; ++q)
        if (lows & (3u << (2 * q)))
        {
            w[q] = g.bitmap_offset + (uint64_t(r.z + (q >> 1)) * g.dims[1] + (r.y + (q & 1))) * g.row_words +
                   (r.x >> 5);
            word[q] = lk.bitmap[w[q]];
        }
#pragma unroll
    for (int q = 1; q < 4; ++q)
        if (lows & (3u << (2 * q)))
            pos[q] = lk.prefix[w[q]] + __popc(word[q] & ((1u << b) - 1u));
#pragma unroll
    for (int q = 0; q < 4; ++q)
        if (lows & (3u << (2 * q)))
        {
            const pair_t v2 = *(global_pair_t*)(vbase + pos[q]);
            const pair_t e2 = *(global_pair_t*)(emask + pos[q]);
            vb[2 * q] = v2.x;
            vb[2 * q + 1] = v2.y;
            em[2 * q] = e2.x;
            em[2 * q + 1] = e2.y;
        }
    case_faces(ci, count, vs, vb, em, lds, v);
}

// Faces of the first nb queued complete cells (nb >= 1).
__device__ __forceinline__ void
mc_faces_batch(const McPlan& p, const BitmapLookup& lk, const McQueue& Q, uint32_t nb,
               const uint32_t* __restrict__ info, const uint32_t* __restrict__ tbase, const uint32_t* __restrict__ emask,
               const uint32_t* __restrict__ vbase, const uint32_t* __restrict__ scene_vstart,
               int64_t* __restrict__ faces, uint32_t* stage)
{
    const uint32_t lane = threadIdx.x & 63u;
    const bool on = lane < nb;
    const uint32_t i = on ? Q.v[lane] : 0u;
    const uint32_t inf = on ? info[i] : 0u;
    const uint32_t t0 = on ? tbase[i] : 0u;
    const VertexRef r = on ? vertex_ref(p, i) : VertexRef{};
    const uint32_t ci = inf & 0xffu;
    const int count = on ? c_cases.count[ci] : 0;
    // batch range [T0, T1) of triangle-vertex slots; lane 0 holds the smallest cell
    const uint32_t T0 = __builtin_amdgcn_readfirstlane(t0);
    uint32_t end = on ? t0 + uint32_t(count) : 0u;
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1)
        end = max(end, __shfl_xor(end, d, 64));
    uint32_t v[kMcMaxTriVerts];
    bool flip = false;
    if (on)
    {
        const uint32_t s0 = __builtin_amdgcn_readfirstlane(r.scene);
        flip = p.grids[r.scene].flip != 0;
        if (__all(r.scene == s0)) // one grid for the active lanes: scalar grid parameters
            mc_cell_faces<true>(p, lk, wave_uniform(p.grids[s0]), i, r, ci, count,
                                __builtin_amdgcn_readfirstlane(scene_vstart[s0]), emask, vbase, stage, v);
        else
            mc_cell_faces<false>(p, lk, p.grids[r.scene], i, r, ci, count, scene_vstart[r.scene], emask, vbase, stage,
                                 v);
    }
    wave_lds_sync();
    if (on)
        stage_faces(count, flip, v, stage + (t0 - T0));
    wave_lds_sync();
    const uint32_t n = end - T0;
    int64_t* dst = faces + uint64_t(T0);
    for (uint32_t q = lane; q < n; q += 64)
        dst[q] = int64_t(stage[q]);
    wave_lds_sync();
}

// The complete cells with triangles are gathered like the vertices of mc_vertices_kernel.
__global__ __launch_bounds__(256) void
mc_faces_unique_kernel(McPlan p,
                       BitmapLookup lk,
                       int chunks,
                       const uint32_t* __restrict__ info,
                       const uint32_t* __restrict__ tbase,
                       const uint32_t* __restrict__ emask,
                       const uint32_t* __restrict__ vbase,
                       const uint32_t* __restrict__ scene_vstart,
                       int64_t* __restrict__ faces)
{
    __shared__ uint32_t stage[kMcWaves][64 * kMcMaxTriVerts];
    __shared__ McQueue queue[kMcWaves];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint64_t v0 = (uint64_t(xcd_block(blockIdx.x, gridDim.x)) * kMcWaves + wave) * (64u * uint32_t(chunks));
    uint32_t q = 0u; // queued cells (wave-uniform)
    for (int c = 0; c < chunks; ++c)
    {
        const uint64_t i = v0 + 64u * uint32_t(c) + lane;
        if (v0 + 64u * uint32_t(c) >= p.nverts)
            break;
        const uint32_t inf = i < p.nverts ? info[i] : 0u;
        const bool active = (inf & kInfoComplete) && c_cases.count[inf & 0xffu] > 0;
        q = mc_enqueue(queue[wave], q, active, uint32_t(i));
        if (q >= 64u)
        {
            wave_lds_sync();
            mc_faces_batch(p, lk, queue[wave], 64u, info, tbase, emask, vbase, scene_vstart, faces, stage[wave]);
            q = mc_dequeue64(queue[wave], q);
        }
    }
    if (q > 0u)
    {
        wave_lds_sync();
        mc_faces_batch(p, lk, queue[wave], q, info, tbase, emask, vbase, scene_vstart, faces, stage[wave]);
    }
}

// ---------------------------------------------------------------------------
// Dense volumes (MC:146-178, MC:242-306, MC:376-533)
//
// Every grid point of a dense volume is present, so which edges are emitted and which case a cell has
// follows from one bit per point: whether its value is below the isolevel.  The volume is read once into
// that bitmap (rows padded to 32-bit words), and the rest of the work is done on words of 32 points: the
// sign-changing edges of a word are the XOR of it with the words one step along x, y and z (every edge of a
// volume of at least 2 points per axis belongs to a cell, so all of them are emitted), the cells with
// triangles are those whose 8 corner bits differ.  The words' counts of output vertices and triangle
// vertices are scanned in tiles of kDenseTile words, and the two output passes visit the words with a count
// only: a vertex of the mesh has the index of its edge in the order (point, axis), which is its word's
// first vertex plus three popcounts.
//
// A 500^3 float32 volume moves 0.5 GB once (the sign pass) and about 60 MB of words; with five 32-bit values
// per grid point, as the sparse passes keep them, it moved 6 GB.  500^3: 2.53 ms -> 0.28 ms (the sign pass
// 0.10 ms at 5.1 TB/s, counts 0.03, vertices 0.04, faces 0.07); 61 x 83 x 71 float64: 85 -> 54 us.
// ---------------------------------------------------------------------------

// Words per workgroup of the counting pass (one per thread) and per entry of the scanned
// tile counts.
constexpr int kDenseTile = 256;

// Edge masks of a word's 32 points along x, y and z, and the index of its first output vertex (written by
// the vertex pass).  Words that emit no edge have no record.
struct alignas(16) DenseEdges
{
    uint32_t x, y, z, first;
};

// A word's counts: output vertices in the low byte (at most 96), triangle vertices above.
__device__ __forceinline__ uint32_t
dense_verts(uint32_t c)
{
    return c & 0xffu;
}
__device__ __forceinline__ uint32_t
dense_tris(uint32_t c)
{
    return c >> 8;
}

// Sign bits.  A lane reads 4 consecutive points in each of kSignRows consecutive rows (16-byte loads of
// float32, element-aligned, all in flight together); 8 lanes assemble a word.  Bound by the one read of the
// volume.
constexpr int kSignRows = 4;

template <typename V>
__global__ __launch_bounds__(256) void
mc_dense_signs_kernel(const V* __restrict__ volume, uint32_t W, uint32_t rows, uint32_t row_words, float isolevel,
                      uint32_t* __restrict__ signs)
{
    typedef V quad_t __attribute__((ext_vector_type(4), aligned(sizeof(V))));
    typedef __attribute__((address_space(1))) const quad_t global_quad_t;
    const V iso = static_cast<V>(isolevel);
    const uint32_t quads = row_words * 8u; // per row, a multiple of 8: the 8 lanes of a word stay together
    const uint64_t t = uint64_t(blockIdx.x) * 256 + threadIdx.x;
    const uint64_t r0 = div_u64_u32(t, quads) * kSignRows;
    const uint32_t quad = uint32_t(t - (r0 / kSignRows) * quads);
    const uint32_t x = quad * 4u;
    const auto src = as_global(volume);
    quad_t v[kSignRows] = {};
    uint32_t n = 0u; // points of this lane's quad inside the row
    if (x < W)
        n = min(W - x, 4u);
#pragma unroll
    for (int q = 0; q < kSignRows; ++q)
        if (r0 + q < rows)
        {
            const uint64_t at = (r0 + q) * W + x;
            if (n == 4u)
                v[q] = *(global_quad_t*)(src + at);
            else
            {
                if (n > 0u)
                    v[q].x = src[at];
                if (n > 1u)
                    v[q].y = src[at + 1];
                if (n > 2u)
                    v[q].z = src[at + 2];
            }
        }
    const uint32_t sub = threadIdx.x & 7u, inside = (1u << n) - 1u;
    uint32_t mine = 0u;
#pragma unroll
    for (int q = 0; q < kSignRows; ++q)
    {
        uint32_t b = (v[q].x < iso ? 1u : 0u) | (v[q].y < iso ? 2u : 0u) | (v[q].z < iso ? 4u : 0u) |
                     (v[q].w < iso ? 8u : 0u);
        b = (b & inside) << (4u * sub);
        b |= uint32_t(__shfl_xor(int(b), 1, 64));
        b |= uint32_t(__shfl_xor(int(b), 2, 64));
        b |= uint32_t(__shfl_xor(int(b), 4, 64));
        if (sub == uint32_t(q))
            mine = b;
    }
    if (sub < uint32_t(kSignRows) && r0 + sub < rows)
        as_global(signs)[(r0 + sub) * row_words + quad / 8u] = mine;
}

// Position of a word: row = y + z H and the points of it inside the volume.
struct DenseWord
{
    uint32_t row, xw, z;
    bool iny, inz;   // rows y + 1 and z + 1 exist
    uint32_t points; // bits of points inside the volume
    uint32_t stepx;  // bits of points with a +x neighbour
};

__device__ __forceinline__ DenseWord
dense_word(const McDense& d, uint32_t w)
{
    DenseWord q;
    q.row = w / d.row_words;
    q.xw = w - q.row * d.row_words;
    q.z = q.row / d.dims[1];
    q.iny = q.row - q.z * d.dims[1] + 1u < d.dims[1];
    q.inz = q.z + 1u < d.dims[2];
    const uint32_t left = d.dims[0] - q.xw * 32u; // points of the row from this word on, at least 1
    q.points = left >= 32u ? 0xffffffffu : (1u << left) - 1u;
    q.stepx = left > 32u ? 0xffffffffu : q.points >> 1;
    return q;
}

// Sign words of a word's four rows (dy, dz) = (0, 0), (1, 0), (0, 1), (1, 1) and of the points one step along
// x from them; rows outside the volume read as the word's own (their results are masked).
struct DenseSigns
{
    uint32_t s[4], x[4];
};

__device__ __forceinline__ DenseSigns
dense_signs(const McDense& d, const DenseWord& q, uint32_t w)
{
    const auto S = as_global(d.signs);
    const uint32_t next = q.xw + 1u < d.row_words ? 1u : 0u;
    const uint32_t oy = q.iny ? d.row_words : 0u, oz = q.inz ? d.row_words * d.dims[1] : 0u;
    DenseSigns g;
#pragma unroll
    for (int r = 0; r < 4; ++r)
    {
        const uint32_t at = w + ((r & 1) ? oy : 0u) + ((r >> 1) ? oz : 0u);
        g.s[r] = S[at];
        g.x[r] = S[at + next];
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
        g.x[r] = (g.s[r] >> 1) | (g.x[r] << 31);
    return g;
}

// Cells of the word with triangles: complete cells whose corners differ.
__device__ __forceinline__ uint32_t
dense_active(const DenseWord& q, const DenseSigns& g)
{
    uint32_t any = 0u, all = 0xffffffffu;
#pragma unroll
    for (int r = 0; r < 4; ++r)
    {
        any |= g.s[r] | g.x[r];
        all &= g.s[r] & g.x[r];
    }
    return (q.iny && q.inz) ? (any & ~all & q.stepx) : 0u;
}

// Case of the cell at bit b: case corner k is the point at offset c_corner_off[k].
__device__ __forceinline__ uint32_t
dense_case(const DenseSigns& g, uint32_t b)
{
    uint32_t ci = 0u;
#pragma unroll
    for (int k = 0; k < 8; ++k)
    {
        const int o = c_corner_off_host[k];
        ci |= ((((o & 1) ? g.x[o >> 1] : g.s[o >> 1]) >> b) & 1u) << k;
    }
    return ci;
}

// Edge masks and counts of every word, and the sums of each tile of words.
__global__ __launch_bounds__(256) void
mc_dense_count_kernel(McDense d, DenseEdges* __restrict__ edges, uint32_t* __restrict__ counts,
                      uint32_t* __restrict__ tile_verts, uint32_t* __restrict__ tile_tris)
{
    __shared__ uint8_t case_count[256];
    __shared__ uint32_t sums[2];
    case_count[threadIdx.x] = c_cases.count[threadIdx.x];
    if (threadIdx.x < 2)
        sums[threadIdx.x] = 0u;
    __syncthreads();
    const uint64_t wl = uint64_t(blockIdx.x) * kDenseTile + threadIdx.x;
    uint32_t nv = 0u, nt = 0u;
    if (wl < d.nwords)
    {
        const uint32_t w = uint32_t(wl);
        const DenseWord q = dense_word(d, w);
        const DenseSigns g = dense_signs(d, q, w);
        DenseEdges e;
        e.x = (g.s[0] ^ g.x[0]) & q.stepx;
        e.y = q.iny ? (g.s[0] ^ g.s[1]) & q.points : 0u;
        e.z = q.inz ? (g.s[0] ^ g.s[2]) & q.points : 0u;
        e.first = 0u;
        nv = uint32_t(__popc(e.x) + __popc(e.y) + __popc(e.z));
        for (uint32_t act = dense_active(q, g); act != 0u; act &= act - 1u)
            nt += case_count[dense_case(g, uint32_t(__builtin_ctz(act)))];
        if (nv != 0u)
            edges[w] = e;
        counts[w] = nv | (nt << 8);
    }
    nv = __reduce_add_sync(0xffffffffffffffffull, nv);
    nt = __reduce_add_sync(0xffffffffffffffffull, nt);
    if ((threadIdx.x & 63) == 0)
    {
        atomicAdd(&sums[0], nv);
        atomicAdd(&sums[1], nt);
    }
    __syncthreads();
    if (threadIdx.x == 0)
    {
        tile_verts[blockIdx.x] = sums[0];
        tile_tris[blockIdx.x] = sums[1];
    }
}

// The output passes run single wavefronts of 64 words, one per lane.
constexpr uint32_t kDenseWaves = kDenseTile / 64;

// First output of each lane's word: the tile's offset plus the counts of the tile's words before it.  `own` is
// the lane's count, `total` the wavefront's.
template <typename Count>
__device__ __forceinline__ uint32_t
dense_first(const McDense& d, const uint32_t* __restrict__ counts, const uint32_t* __restrict__ tile_first,
            Count count, uint32_t& own, uint32_t& total)
{
    const uint32_t q = blockIdx.x % kDenseWaves;
    const uint64_t w = uint64_t(blockIdx.x) * 64u + threadIdx.x;
    uint32_t before = 0u;
#pragma unroll
    for (uint32_t k = 1; k < kDenseWaves; ++k)
        before += k <= q ? count(counts[w - 64u * k]) : 0u; // words of the wavefronts before: all inside
    own = w < d.nwords ? count(counts[w]) : 0u;
    const uint32_t inc = wave_inclusive_sum(own);
    total = uint32_t(__shfl(int(inc), 63, 64));
    return tile_first[blockIdx.x / kDenseWaves] + __reduce_add_sync(0xffffffffffffffffull, before) + inc - own;
}

// The lanes' set bits, one entry (lane << 5 | bit) each, in lane order; returns their number.
__device__ __forceinline__ uint32_t
dense_enqueue(uint16_t* queue, uint32_t bits)
{
    const uint32_t n = uint32_t(__popc(bits)), inc = wave_inclusive_sum(n);
    for (uint32_t at = inc - n; bits != 0u; bits &= bits - 1u)
        queue[at++] = uint16_t((threadIdx.x << 5) | uint32_t(__builtin_ctz(bits)));
    wave_lds_sync();
    return uint32_t(__shfl(int(inc), 63, 64));
}

// Output vertices of the compact mesh.  A lane records its word's first vertex and queues its points that emit
// an edge; the wavefront then takes the queued points 64 at a time.  Bound by the latency of the value reads.
template <typename V>
__global__ __launch_bounds__(64) void
mc_dense_vertices_kernel(McDense d, McGrid g, const V* __restrict__ volume, float iso,
                         const uint32_t* __restrict__ counts, const uint32_t* __restrict__ tile_verts,
                         DenseEdges* __restrict__ edges, float* __restrict__ verts)
{
    __shared__ DenseEdges rec[64];
    __shared__ uint16_t queue[64 * 32];
    const uint32_t lane = threadIdx.x;
    const uint64_t w0 = uint64_t(blockIdx.x) * 64u; // the wavefront's first word
    uint32_t c, total;
    const uint32_t first = dense_first(d, counts, tile_verts, dense_verts, c, total);
    if (total == 0u)
        return;
    uint32_t points = 0u;
    if (c != 0u)
    {
        DenseEdges r = edges[w0 + lane];
        r.first = first;
        edges[w0 + lane].first = first;
        rec[lane] = r;
        points = r.x | r.y | r.z;
    }
    const uint32_t n = dense_enqueue(queue, points);
    const uint32_t step[3] = { 1u, d.dims[0], d.dims[0] * d.dims[1] };
    for (uint32_t k = lane; k < n; k += 64)
    {
        const uint32_t e = queue[k], b = e & 31u, lt = (1u << b) - 1u;
        const DenseEdges r = rec[e >> 5];
        const DenseWord q = dense_word(d, uint32_t(w0) + (e >> 5));
        const uint32_t x = q.xw * 32u + b, y = q.row - q.z * d.dims[1];
        const uint32_t i = q.row * d.dims[0] + x; // fewer than 2^32 points
        const bool on[3] = { ((r.x >> b) & 1u) != 0u, ((r.y >> b) & 1u) != 0u, ((r.z >> b) & 1u) != 0u };
        const float v1 = float(volume[i]); // stored as float (MC:343)
        float v2[3];
#pragma unroll
        for (int a = 0; a < 3; ++a)
            v2[a] = on[a] ? float(volume[i + step[a]]) : 0.0f;
        uint64_t o = 3 * uint64_t(r.first + uint32_t(__popc(r.x & lt) + __popc(r.y & lt) + __popc(r.z & lt)));
        const uint32_t p1[3] = { x, y, q.z };
#pragma unroll
        for (int a = 0; a < 3; ++a)
            if (on[a])
            {
                const uint32_t p2[3] = { x + (a == 0), y + (a == 1), q.z + (a == 2) };
                float v[3];
                interpolate_vertex(iso, p1, p2, v1, v2[a], v);
                finish_vertex(g, v, verts + o);
                o += 3;
            }
    }
}

// Faces, and the vertices of a triangle soup.  As the vertex pass, with the cells that have triangles; a cell's
// first triangle vertex is the running total of the cells before it.  The slots of 64 queued cells are one
// contiguous range, assembled in LDS and written with coalesced stores.
template <typename V, bool UNIQUE>
__global__ __launch_bounds__(64) void
mc_dense_faces_kernel(McDense d, McGrid g, const V* __restrict__ volume, float iso,
                      const uint32_t* __restrict__ counts, const uint32_t* __restrict__ tile_tris,
                      const DenseEdges* __restrict__ edges, float* __restrict__ soup_verts,
                      int64_t* __restrict__ faces)
{
    __shared__ DenseSigns signs[64];
    __shared__ uint16_t queue[64 * 32];
    __shared__ uint32_t stage[UNIQUE ? 64 * kMcMaxTriVerts : 1];
    const uint32_t lane = threadIdx.x;
    const uint64_t w0 = uint64_t(blockIdx.x) * 64u; // the wavefront's first word
    uint32_t c, total;
    const uint32_t first = dense_first(d, counts, tile_tris, dense_tris, c, total);
    if (total == 0u)
        return;
    uint32_t run = __builtin_amdgcn_readfirstlane(first); // first triangle vertex of the cells taken next
    uint32_t cells = 0u;
    if (c != 0u)
    {
        const DenseWord q = dense_word(d, uint32_t(w0) + lane);
        const DenseSigns s = dense_signs(d, q, uint32_t(w0) + lane);
        cells = dense_active(q, s);
        signs[lane] = s;
    }
    const uint32_t n = dense_enqueue(queue, cells);
    const uint32_t wy = d.row_words, wz = d.row_words * d.dims[1];
    for (uint32_t k0 = 0; k0 < n; k0 += 64)
    {
        const bool on = k0 + lane < n;
        const uint32_t e = on ? queue[k0 + lane] : 0u;
        const uint32_t b = e & 31u, w = uint32_t(w0) + (e >> 5);
        const uint32_t ci = on ? dense_case(signs[e >> 5], b) : 0u;
        const int count = on ? c_cases.count[ci] : 0;
        const uint32_t inc = wave_inclusive_sum(uint32_t(count));
        const uint32_t off = inc - uint32_t(count); // of the cell's slots in this batch
        const uint32_t slots = uint32_t(__shfl(int(inc), 63, 64));
        if constexpr (UNIQUE)
        {
            uint32_t v[kMcMaxTriVerts];
            if (on)
            {
                // corners 2q and 2q + 1 (x and x + 1) of row q = (dy, dz): same word unless x is its last point
                const uint32_t lows = c_cases.lows[ci];
                uint32_t vb[8], em[8];
#pragma unroll
                for (int q = 0; q < 4; ++q)
                {
                    const uint32_t wq = w + ((q & 1) ? wy : 0u) + ((q >> 1) ? wz : 0u);
                    DenseEdges r{};
                    if (lows & ((b != 31u ? 3u : 1u) << (2 * q))) // a corner that emits an edge: its word has a record
                        r = edges[wq];
                    DenseEdges r1 = r;
                    if (b == 31u && (lows & (2u << (2 * q))))
                        r1 = edges[wq + 1u];
                    const uint32_t b1 = (b + 1u) & 31u, lt = (1u << b) - 1u, lt1 = (1u << b1) - 1u;
                    vb[2 * q] = r.first + uint32_t(__popc(r.x & lt) + __popc(r.y & lt) + __popc(r.z & lt));
                    em[2 * q] = ((r.x >> b) & 1u) | (((r.y >> b) & 1u) << 1) | (((r.z >> b) & 1u) << 2);
                    vb[2 * q + 1] = r1.first + uint32_t(__popc(r1.x & lt1) + __popc(r1.y & lt1) + __popc(r1.z & lt1));
                    em[2 * q + 1] = ((r1.x >> b1) & 1u) | (((r1.y >> b1) & 1u) << 1) | (((r1.z >> b1) & 1u) << 2);
                }
                case_faces(ci, count, 0u, vb, em, stage, v);
            }
            wave_lds_sync();
            if (on)
                stage_faces(count, false, v, stage + off);
            wave_lds_sync();
            for (uint32_t s = lane; s < slots; s += 64)
                faces[uint64_t(run) + s] = int64_t(stage[s]);
            wave_lds_sync();
        }
        else if (on)
        {
            const DenseWord q = dense_word(d, w);
            const uint32_t x = q.xw * 32u + b, y = q.row - q.z * d.dims[1];
            const uint64_t t0 = uint64_t(run) + off;
            for (int k = 0; k < count; ++k)
            {
                const int id = c_cases.edges[ci][k];
                const uint32_t lo = c_edge_low[id], axis = c_edge_axis[id];
                const uint32_t q1[3] = { x + (lo & 1u), y + ((lo >> 1) & 1u), q.z + ((lo >> 2) & 1u) };
                const uint32_t q2[3] = { q1[0] + (axis == 0u), q1[1] + (axis == 1u), q1[2] + (axis == 2u) };
                const float v1 = float(volume[(q1[2] * d.dims[1] + q1[1]) * d.dims[0] + q1[0]]);
                const float v2 = float(volume[(q2[2] * d.dims[1] + q2[1]) * d.dims[0] + q2[0]]);
                float v[3];
                interpolate_vertex(iso, q1, q2, v1, v2, v);
                finish_vertex(g, v, soup_verts + 3 * (t0 + uint32_t(k)));
                faces[t0 + uint32_t(k)] = int64_t(t0 + uint32_t(k)); // faces = arange (MC:515-519)
            }
        }
        run += slots;
    }
}

uint32_t
mc_dense_tiles(uint64_t nwords)
{
    return uint32_t((nwords + kDenseTile - 1) / kDenseTile);
}

size_t
mc_dense_edge_bytes(uint64_t nwords)
{
    return size_t(nwords) * sizeof(DenseEdges);
}

void
launch_mc_dense_counts(const McDense& d, const void* volume, int32_t value_type, float iso, void* edges,
                       uint32_t* counts, uint32_t* tile_verts, uint32_t* tile_tris, hipStream_t st)
{
    const uint32_t rows = d.dims[1] * d.dims[2];
    const uint64_t threads = uint64_t(d.row_words) * 8u * ((uint64_t(rows) + kSignRows - 1) / kSignRows);
    const unsigned nb = unsigned((threads + 255) / 256);
    if (value_type == kMcF64)
        mc_dense_signs_kernel<double>
            <<<nb, 256, 0, st>>>(static_cast<const double*>(volume), d.dims[0], rows, d.row_words, iso, d.signs);
    else
        mc_dense_signs_kernel<float>
            <<<nb, 256, 0, st>>>(static_cast<const float*>(volume), d.dims[0], rows, d.row_words, iso, d.signs);
    THULL_LAUNCH_CHECK();
    mc_dense_count_kernel<<<mc_dense_tiles(d.nwords), 256, 0, st>>>(d, static_cast<DenseEdges*>(edges), counts,
                                                                    tile_verts, tile_tris);
    THULL_LAUNCH_CHECK();
}

void
launch_mc_dense_mesh(const McDense& d, const McGrid& g, const void* volume, int32_t value_type, float iso,
                     const uint32_t* counts, const uint32_t* tile_verts, const uint32_t* tile_tris, void* edges,
                     bool unique, float* verts, int64_t* faces, hipStream_t st)
{
    const unsigned nb = unsigned((d.nwords + 63) / 64);
    DenseEdges* e = static_cast<DenseEdges*>(edges);
    const auto run = [&](auto* vol) {
        using V = std::remove_const_t<std::remove_pointer_t<decltype(vol)>>;
        if (unique)
        {
            mc_dense_vertices_kernel<V><<<nb, 64, 0, st>>>(d, g, vol, iso, counts, tile_verts, e, verts);
            THULL_LAUNCH_CHECK();
            mc_dense_faces_kernel<V, true><<<nb, 64, 0, st>>>(d, g, vol, iso, counts, tile_tris, e, verts, faces);
        }
        else
            mc_dense_faces_kernel<V, false><<<nb, 64, 0, st>>>(d, g, vol, iso, counts, tile_tris, e, verts, faces);
        THULL_LAUNCH_CHECK();
    };
    if (value_type == kMcF64)
        run(static_cast<const double*>(volume));
    else
        run(static_cast<const float*>(volume));
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------

// Chunks per wavefront of the gathering kernels: `most` where that still gives kMcTargetWaves wavefronts
// (16 per CU), else as many as give them, since a wavefront walks its chunks one after the other and each
// batch is a chain of dependent reads.  Level-7 hull of 8 cameras (about 60 000 vertices): faces 42 -> 7.7 us
// and vertices 16 -> 4.9 us; sparse 400^3 sphere band (1.5 million): faces 51 -> 29 us.
constexpr uint64_t kMcTargetWaves = 4096;

static int
mc_chunks(uint64_t nverts, int most)
{
    return int(std::min<uint64_t>(uint64_t(most), std::max<uint64_t>(1, nverts / (64u * kMcTargetWaves))));
}

// Workgroups of the gathering kernels: kMcWaves wavefronts of `chunks` 64-vertex chunks each.
static unsigned
mc_gather_blocks(uint64_t nverts, int chunks)
{
    const uint64_t per = uint64_t(kMcWaves) * 64u * uint64_t(chunks);
    return unsigned((nverts + per - 1) / per);
}

template <typename F>
static void
dispatch_mc(const McPlan& p, F&& f)
{
    if (p.value_type == kMcF64)
        f(double{});
    else
        f(float{});
}

void
launch_mc_classify(const McPlan& p, uint32_t* info, uint32_t* ntv, hipStream_t st)
{
    if (p.nverts == 0)
        return;
    const BitmapLookup lk{ p.bitmap, p.prefix };
    dispatch_mc(p, [&](auto vt) {
        using VT = decltype(vt);
        mc_classify_kernel<VT><<<blocks_for(int64_t(p.nverts), 256), 256, 0, st>>>(p, lk, info, ntv);
    });
    THULL_LAUNCH_CHECK();
}

void
launch_mc_edges(const McPlan& p, const uint32_t* info, uint32_t* emask, hipStream_t st)
{
    if (p.nverts == 0)
        return;
    mc_edges_kernel<<<blocks_for(int64_t(p.nverts), 256), 256, 0, st>>>(p, BitmapLookup{ p.bitmap, p.prefix }, info,
                                                                        emask);
    THULL_LAUNCH_CHECK();
}

void
launch_mc_vertices(const McPlan& p, const uint32_t* emask, const uint32_t* vbase, float* verts, hipStream_t st)
{
    if (p.nverts == 0)
        return;
    const BitmapLookup lk{ p.bitmap, p.prefix };
    dispatch_mc(p, [&](auto vt) {
        using VT = decltype(vt);
        const int chunks = mc_chunks(p.nverts, kMcVertexChunks);
        mc_vertices_kernel<VT><<<mc_gather_blocks(p.nverts, chunks), 256, 0, st>>>(p, lk, chunks, emask, vbase,
                                                                                      verts);
    });
    THULL_LAUNCH_CHECK();
}

void
launch_mc_faces(const McPlan& p,
                const uint32_t* info,
                const uint32_t* ntv_base,
                const uint32_t* emask,
                const uint32_t* vbase,
                const uint32_t* scene_vstart,
                const uint32_t* scene_tstart,
                bool unique,
                float* soup_verts,
                int64_t* faces,
                hipStream_t st)
{
    if (p.nverts == 0)
        return;
    const BitmapLookup lk{ p.bitmap, p.prefix };
    dispatch_mc(p, [&](auto vt) {
        using VT = decltype(vt);
        const int chunks = mc_chunks(p.nverts, kMcFaceChunks);
        if (unique)
            mc_faces_unique_kernel<<<mc_gather_blocks(p.nverts, chunks), 256, 0, st>>>(
                    p, lk, chunks, info, ntv_base, emask, vbase, scene_vstart, faces);
        else
            mc_faces_kernel<VT><<<blocks_for(int64_t(p.nverts), 256), 256, 0, st>>>(
                    p, lk, info, ntv_base, emask, vbase, scene_vstart, scene_tstart, unique, soup_verts, faces);
    });
    THULL_LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------
// Sparse COO input (MC:756-815): vertex bitmap of the nonzero entries
// ---------------------------------------------------------------------------

// One lane per entry reads its four indices, so this is also where they are checked: an entry outside the
// volume marks nothing and raises *bad.  Coalesced entries are sorted, so the entries of one bitmap word sit
// in consecutive lanes: the lanes of such a run OR their bits together (a segmented reduction between run
// heads, any run length) and its first lane issues the one atomic.  Bound by the 32 bytes per entry.
// 400^3 sphere band, 1.5 million entries: 70 us with one atomic per entry and three index rows, now 12 us
// with four; the checks as reductions over the index rows took another 650 us.
__global__ __launch_bounds__(256) void
mark_coo_kernel(const int64_t* __restrict__ coo, uint64_t nnz, const McGrid* __restrict__ grid,
                uint32_t* __restrict__ bitmap, unsigned long long* __restrict__ bad)
{
    const uint64_t i = uint64_t(blockIdx.x) * 256 + threadIdx.x;
    const int lane = int(threadIdx.x & 63);
    const McGrid g = *grid;
    uint64_t w = ~uint64_t(0);
    uint32_t bits = 0u;
    bool out = false;
    if (i < nnz)
    {
        const int64_t b = coo[i], z = coo[1 * nnz + i], y = coo[2 * nnz + i], x = coo[3 * nnz + i];
        out = b < 0 || x < 0 || y < 0 || z < 0 || x >= g.dims[0] || y >= g.dims[1] || z >= g.dims[2];
        if (!out)
        {
            w = g.bitmap_offset + (uint64_t(z) * g.dims[1] + uint64_t(y)) * g.row_words + uint64_t(x >> 5);
            bits = 1u << uint32_t(x & 31);
        }
    }
    if (__any(out) && lane == 0)
        atomicOr(bad, 1ull);
    // every lane takes part in the shuffles
    const uint32_t plo = uint32_t(__shfl_up(int(uint32_t(w)), 1, 64));
    const uint32_t phi = uint32_t(__shfl_up(int(uint32_t(w >> 32)), 1, 64));
    const bool head = lane == 0 || plo != uint32_t(w) || phi != uint32_t(w >> 32);
    const uint64_t later = (__ballot(head) >> lane) >> 1; // run heads after this lane
    const int len = later == 0 ? 64 - lane : 1 + __builtin_ctzll(later); // lanes of the run from this one on
#pragma unroll
    for (int d = 1; d < 64; d <<= 1)
    {
        const uint32_t o = uint32_t(__shfl_down(int(bits), d, 64));
        bits |= d < len ? o : 0u;
    }
    if (head && bits != 0u)
        atomicOr(bitmap + w, bits);
}

void
launch_mark_coo(const int64_t* coo, uint64_t nnz, const McGrid* grid, uint32_t* bitmap, unsigned long long* bad,
                hipStream_t st)
{
    if (nnz == 0)
        return;
    mark_coo_kernel<<<blocks_for(int64_t(nnz), 256), 256, 0, st>>>(coo, nnz, grid, bitmap, bad);
    THULL_LAUNCH_CHECK();
}

__global__ __launch_bounds__(256) void
extract_grid_vertices_kernel(const uint32_t* __restrict__ bitmap, const uint32_t* __restrict__ prefix,
                             uint64_t nwords, const McGrid* __restrict__ grid, uint64_t* __restrict__ vertices)
{
    const uint64_t w = uint64_t(blockIdx.x) * 256 + threadIdx.x;
    if (w >= nwords)
        return;
    uint32_t word = bitmap[w];
    if (word == 0u)
        return;
    const McGrid g = *grid;
    const uint64_t row = div_u64_u32(w, g.row_words);
    const uint32_t xw = uint32_t(w - row * g.row_words);
    const uint64_t zq = div_u64_u32(row, g.dims[1]);
    const uint32_t y = uint32_t(row - zq * g.dims[1]), z = uint32_t(zq);
    uint32_t pos = prefix[w];
    while (word != 0u)
    {
        const uint32_t b = __builtin_ctz(word);
        vertices[pos++] = pack_key(0u, xw * 32u + b, y, z);
        word &= word - 1u;
    }
}

void
launch_extract_grid_vertices(const uint32_t* bitmap, const uint32_t* prefix, uint64_t nwords, const McGrid* grid,
                             uint64_t* vertices, hipStream_t st)
{
    if (nwords == 0)
        return;
    extract_grid_vertices_kernel<<<blocks_for(int64_t(nwords), 256), 256, 0, st>>>(bitmap, prefix, nwords, grid,
                                                                                   vertices);
    THULL_LAUNCH_CHECK();
}

} // namespace thull
