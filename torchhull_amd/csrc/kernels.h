// Host-side launchers of the device kernels (one translation unit each).
#pragma once

#include "common.h"

namespace thull
{

// ---- integral image (vh_kernels.hip) ----
// float32 integral image of masks [B,H,W] of element type `dtype`, equal to
// torch::cumsum(.., 1, f32) followed by cumsum(.., 2, f32) on CUDA.
// `job_buf` is device scratch of integral_job_bytes(number of tensors) bytes;
// `carry` holds integral_carry_floats(B, H, W) floats per tensor.
constexpr size_t kIntegralJobBytes = 128; // integral_job_bytes(1) at most
size_t integral_job_bytes(size_t njobs);
uint64_t integral_carry_floats(int64_t B, int64_t H, int64_t W);
void launch_integral_image(const void* masks, int32_t dtype, int64_t B, int64_t H, int64_t W, float* out, float* carry,
                           void* job_buf, Uploader& up, hipStream_t st);
// The same integral images, for many mask tensors in one launch per pass, in
// the padded, tiled layout carving reads (integral_pitch, integral_rows in common.h): the zero row
// and column make the zero padding of image_utils.h:84-97 branch-free.
// `carry` holds the sum over requests of integral_carry_floats.
struct IntegralRequest
{
    const void* masks;
    int32_t dtype;
    int64_t B, H, W;
    float* padded;
    // solid maps (common.h), built with the integral images where `solid` is not null: the maps and the cameras'
    // bounds, and scratch of solid_scratch_bytes(B, H, W) bytes
    uint8_t* solid;
    CullCamera* cull;
    void* solid_scratch;
    int32_t* culls; // the scene's SceneDev::culls on the device
    const float* transforms;
    int32_t opengl;
    float corner[3];
    float length;
};
uint64_t solid_map_bytes(int64_t B, int64_t H, int64_t W);
uint64_t solid_scratch_bytes(int64_t B, int64_t H, int64_t W);
size_t solid_job_bytes(size_t njobs);
// `solid_jobs`: solid_job_bytes(n) bytes of device scratch, unused without solid maps.
void launch_integral_images_padded(const IntegralRequest* req, int32_t n, float* carry, void* job_buf,
                                   void* solid_jobs, Uploader& up, hipStream_t st);

// ---- octree carving (vh_kernels.hip) ----
constexpr int kCarveThreads = 256;

// Classifies the 8 children of each parent; writes an 8-bit occupancy mask per
// parent and the number of occupied children per block of kCarveThreads
// parents.  `tests` accumulates the number of camera tests (early exit).
// Returns the kernel that ran: the number of lanes that share one parent's cameras (1: one thread
// per parent, carve_classify_kernel; 2/4/16/64: carve_classify_split_kernel<G>) or kChildSplit.
// Lanes per parent by level size: G = 64 for at most max_parents[0] parents, 16 up to max_parents[1],
// 4 up to max_parents[2], 2 up to max_parents[3], else 1.  Of the levels with 64, the smallest take a
// lane per parent, child and camera, and lanes that the launch's cameras would leave idle are not
// launched: 16 for at most 16 cameras, 4 for at most 4.
constexpr int32_t kChildSplit = 8; // carve_classify_child_kernel
struct CarveTuning
{
    uint32_t max_parents[4] = { 16384u, 131072u, 1048576u, 1048576u }; // G = 64, 16, 4, 2 up to these sizes
};
int32_t carve_split_factor(uint32_t n, const CarveTuning& tune);
// Whether carving of some scene may leave out cameras at a step (host descriptors).
bool carve_culls(const SceneDev* scenes, size_t n, int32_t step);
// `step`: the carving step (a scene's octree level is step - its start).  `max_cameras`: the most cameras of a scene.
// `culls`: carve_culls of the launch's scenes.
// Device-driven levels (dev_n non-null): the level holds min(*dev_n, n) parents, n being the list's
// capacity; the lanes per parent are `split_hint`, and with one lane per parent a persistent queue
// kernel runs (carve_classify_queue_kernel, `cursors`: 8 words, zero at start).
int32_t launch_carve_classify(const uint64_t* parents, uint32_t n, int32_t step, const SceneDev* scenes,
                              uint8_t* child_mask, uint32_t* block_counts, unsigned long long* tests,
                              const CarveTuning& tune, int32_t max_cameras, bool culls, hipStream_t st,
                              const unsigned long long* dev_n = nullptr, int32_t split_hint = 0,
                              uint32_t* cursors = nullptr, bool counts = true);

// Writes the occupied children of every parent, parent-major and child-minor,
// at `block_offsets[block]` + the in-block prefix.  With `mark_leaves`, the
// children of parents whose scene ends at carving step `child_step` (scene
// level + start) are also set in their scene's leaf-cell bitmap.
// Device-driven levels: n is a capacity, dev_n the size, and children past out_cap are dropped.
void launch_carve_scatter(const uint64_t* parents, uint32_t n, const uint8_t* child_mask,
                          const uint32_t* block_offsets, uint64_t* children, int32_t child_step,
                          const SceneDev* scenes, bool mark_leaves, hipStream_t st,
                          const unsigned long long* dev_n = nullptr, uint64_t out_cap = ~uint64_t(0));
// Block counts, their scan and launch_carve_scatter of a level of at most kCompactParents parents in one launch
// (masks 16-byte aligned); total and note as in exclusive_scan.
struct ScanNotify;
constexpr uint32_t kCompactParents = 1u << 17;
void launch_carve_compact(const uint64_t* parents, uint32_t n, const uint8_t* child_mask, uint64_t* children,
                          int32_t child_step, const SceneDev* scenes, bool mark_leaves, unsigned long long* total,
                          const ScanNotify& note, hipStream_t st);
// Sets the root cell of every level-0 scene among scenes first .. first + nscenes - 1.
void launch_mark_root_cells(const SceneDev* scenes, int32_t first, int32_t nscenes, hipStream_t st);
// Vertex bitmap (all words, no clearing needed) = leaf cells dilated by {0,1}^3.
// Also writes the popcount sum of every tile of words to block_sums
// (vertex_tiles(nwords) entries), the first pass of the vertex numbering.
uint32_t vertex_tiles(uint64_t nwords);
void launch_dilate_cells(uint32_t* verts, uint64_t nwords, const uint64_t* scene_word_begin, const SceneDev* scenes,
                         int32_t nscenes, uint32_t* block_sums, hipStream_t st);

// Fills n 32-bit words with `value` (a kernel, so that it can sit in a captured graph).
void launch_fill_u32(uint32_t* dst, uint64_t n, uint32_t value, hipStream_t st);

// From the exclusive block offsets of those sums: prefix[word] (exclusive
// popcount prefix) and the packed key of every set bit of the bitmap at
// prefix[word] + rank.  `scene_word_begin` has nscenes + 1 entries.
void launch_prefix_extract(const uint32_t* bitmap, uint64_t nwords, const uint32_t* block_offsets,
                           const uint64_t* scene_word_begin, const SceneDev* scenes, int32_t nscenes,
                           uint32_t* prefix, uint64_t* vertices, hipStream_t st);

// Self-test: div2_shared against the IEEE division on `count` random operand
// triples; adds the number of differing quotients to *mismatches.
void launch_div2_check(uint64_t count, uint64_t seed, unsigned long long* mismatches, hipStream_t st);

// One octree list that holds bricks: the cells kept up to a carving step.
struct BrickList
{
    const uint64_t* keys;
    uint32_t count;
    int32_t step;
    uint64_t begin; // first wavefront of this list
};
// Marks the bricks of the lists (scenes whose brick level is reached at the list's step) in their scenes' brick
// bitmaps, which are zero.  `waves`: the summed counts of the lists.
void launch_mark_bricks(const BrickList* lists, int32_t nlists, uint64_t waves, const SceneDev* scenes,
                        hipStream_t st);
// Flags of the groups of 4 words of the scenes' vertex bitmaps that marked bricks reach, group_flag_bytes per scene
// (`most`: the largest scene's).
uint64_t group_flag_bytes(int32_t level, int32_t brick_shift, uint32_t row_words);
void launch_group_flags(const SceneDev* scenes, int32_t nscenes, uint64_t most, hipStream_t st);
// launch_dilate_cells and launch_prefix_extract for scenes whose group flags are set: rows of whole groups of 4 words,
// every scene's words a multiple of 4, and prefixes only of groups with vertices and of every scene's first group.
// `filled`: filled_words(nwords) words of bits of those groups, from the first launch to the second.
uint64_t filled_words(uint64_t nwords);
void launch_dilate_groups(uint32_t* verts, uint64_t nwords, const uint64_t* scene_word_begin, const SceneDev* scenes,
                          int32_t nscenes, uint32_t* block_sums, uint64_t* filled, hipStream_t st);
void launch_extract_groups(const uint32_t* bitmap, uint64_t nwords, const uint64_t* filled,
                           const uint32_t* block_offsets, const uint64_t* scene_word_begin, const SceneDev* scenes,
                           int32_t nscenes, uint32_t* prefix, uint64_t* vertices, hipStream_t st);
// Field values by bricks: as launch_field for all vertices of the lists' bricks, written at the vertices' ranks.
void launch_field_bricks(const BrickList* lists, int32_t nlists, uint64_t waves, const SceneDev* scenes,
                         const uint32_t* bitmap, const uint32_t* prefix, float* values, hipStream_t st);

// Field value of every vertex: product over cameras of the bilinear mask sample.
void launch_field(const uint64_t* vertices, uint32_t n, const SceneDev* scenes, float* values, hipStream_t st);

// Wireframe of n level-`level` cells (ravel ids): verts float32 [8n,3], edges int64 [12n,2].
void launch_wireframe(const int64_t* cells, uint32_t n, int32_t level, const float corner[3], float length, float* verts,
                      int64_t* edges, hipStream_t st);

// ---- marching cubes (mc_kernels.hip) ----

// Grid description for marching cubes.  Vertex positions of the sparse passes are ranks in the batch bitmap.
struct McGrid
{
    uint32_t dims[3];       // grid vertices per axis
    uint32_t row_words;     // bitmap words per (y, z) row
    uint64_t bitmap_offset; // first bitmap word of this grid
    int32_t out_mode;       // 0: grid units, 1: local [-1, 1] (v * scale - 1), 2: world (fmaf(scale, v, corner))
    float scale[3];
    float corner[3];
    int32_t flip;           // swap face columns 1 and 2
};

enum McValueType : int32_t
{
    kMcF32 = 0,
    kMcF64 = 1,
};

struct McPlan
{
    // inputs
    const McGrid* grids;      // device, one per scene
    const uint64_t* vertices; // packed keys
    uint64_t nverts;          // vertex count
    const void* values;       // [nverts] f32 or f64
    int32_t value_type;
    float iso;
    const uint32_t* bitmap;   // grid vertices
    const uint32_t* prefix;   // exclusive popcount prefix per word
};

// Pass 1: per vertex info word (case, complete bit, edge sign-change bits) and
// number of triangle vertices of its cell.
void launch_mc_classify(const McPlan& p, uint32_t* info, uint32_t* ntv, hipStream_t st);
// Pass 2: 3-bit mask of the emitted edges starting at each vertex.
void launch_mc_edges(const McPlan& p, const uint32_t* info, uint32_t* emask, hipStream_t st);
// Pass 3: one output vertex per emitted edge, at vbase[i] + rank within emask.
void launch_mc_vertices(const McPlan& p, const uint32_t* emask, const uint32_t* vbase, float* verts, hipStream_t st);
// Pass 4: faces of every active cell; unique: indices through emask/vbase,
// soup: vertices interpolated per triangle corner.  scene_vstart / scene_tstart
// give the first output vertex / triangle-vertex of each scene.
void launch_mc_faces(const McPlan& p, const uint32_t* info, const uint32_t* ntv_base, const uint32_t* emask,
                     const uint32_t* vbase, const uint32_t* scene_vstart, const uint32_t* scene_tstart, bool unique,
                     float* soup_verts, int64_t* faces, hipStream_t st);

// Dense volumes [D,H,W] (x fastest) of at least 2 points per axis and fewer than 2^32 points.
struct McDense
{
    uint32_t dims[3];   // points along x, y, z
    uint32_t row_words; // 32-point words per row
    uint64_t nwords;    // row_words * dims[1] * dims[2]
    uint32_t* signs;    // [nwords] one bit per point: value below the isolevel
};
uint32_t mc_dense_tiles(uint64_t nwords);
size_t mc_dense_edge_bytes(uint64_t nwords);
// Sign bits, edge masks (`edges`, mc_dense_edge_bytes) and counts of every word ([nwords]), and the counts of
// output vertices and triangle vertices of every tile (mc_dense_tiles entries each).
void launch_mc_dense_counts(const McDense& d, const void* volume, int32_t value_type, float iso, void* edges,
                            uint32_t* counts, uint32_t* tile_verts, uint32_t* tile_tris, hipStream_t st);
// The mesh, from the exclusive prefixes of the tile counts; soups (unique false) have a vertex per triangle corner.
void launch_mc_dense_mesh(const McDense& d, const McGrid& g, const void* volume, int32_t value_type, float iso,
                          const uint32_t* counts, const uint32_t* tile_verts, const uint32_t* tile_tris, void* edges,
                          bool unique, float* verts, int64_t* faces, hipStream_t st);

// Grid-vertex bitmap of a sparse COO volume: marks (x, y, z) = (idx[3], idx[2], idx[1]).  An entry outside the
// volume (or with a negative index idx[0]) marks nothing and sets *bad.
void launch_mark_coo(const int64_t* coo, uint64_t nnz, const McGrid* grid, uint32_t* bitmap, unsigned long long* bad,
                     hipStream_t st);
// Packed keys (scene 0) of the set bits of a single-grid bitmap.
void launch_extract_grid_vertices(const uint32_t* bitmap, const uint32_t* prefix, uint64_t nwords, const McGrid* grid,
                                  uint64_t* vertices, hipStream_t st);

// ---- gaussian blur (blur_kernels.hip) ----
struct BlurImage
{
    const void* in;  // [B,H,W]
    void* out;       // [B,H,W] of the output dtype
    int64_t B, H, W;
};
int64_t blur_tile_flag_bytes(int64_t B, int64_t H, int64_t W, int kernel_size);
size_t blur_job_bytes(size_t n);
// `flags`: sum over images of blur_tile_flag_bytes(B, H, W, k) bytes (sparse, k > 1; 4-byte aligned).
void launch_gaussian_blur_batch(const BlurImage* imgs, int32_t n, int32_t in_dtype, int kernel_size, bool sparse,
                                const void* weights, double norm, int32_t out_dtype, uint8_t* flags, void* job_buf,
                                Uploader& up, hipStream_t st);

} // namespace thull
