/*
 * torchhull_amd: C ABI of the MI355X (gfx950) visual-hull library.
 *
 * Plain pointers and sizes only.  Every device pointer refers to memory of the
 * context's device; `stream` is a hipStream_t (NULL = the default stream).
 * Every entry point returns 0 on success and a nonzero status on failure; the
 * message is then available from thull_last_error() (thread-local).  Calls on
 * one context are not thread-safe: use one context per host thread.
 *
 * Each declaration cites the reference interface it replaces
 * (vc-bonn/torchhull, paths relative to the repository root).
 */
#ifndef TORCHHULL_AMD_H
#define TORCHHULL_AMD_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define THULL_ABI_VERSION 1

/* Element types (thull_dtype). */
enum thull_dtype
{
    THULL_BOOL = 0,
    THULL_U8 = 1,
    THULL_I8 = 2,
    THULL_I16 = 3,
    THULL_I32 = 4,
    THULL_I64 = 5,
    THULL_F16 = 6,
    THULL_F32 = 7,
    THULL_F64 = 8
};

typedef struct thull_ctx thull_ctx;

/* ABI version of the loaded library (THULL_ABI_VERSION). */
int thull_abi_version(void);

/* Message of the last failed call on this thread ("" if none). */
const char* thull_last_error(void);

/* Context: a device plus pooled device memory reused across calls.
 * Replaces the per-call torch caching-allocator / stdgpu allocations of the
 * reference (src/torchhull/_C/include/torchhull/stdgpu_allocator.h:36-49). */
int thull_ctx_create(int device, thull_ctx** out);
int thull_ctx_destroy(thull_ctx* ctx);
/* Peak pooled device bytes and currently reserved bytes. */
int thull_ctx_memory(thull_ctx* ctx, int64_t* peak_bytes, int64_t* reserved_bytes);
/* Release pooled memory that holds no result. */
int thull_ctx_trim(thull_ctx* ctx);

/* Carving launch shape by octree level size, with no counterpart in the reference
 * (its carving launches one thread per node): max_parents holds 4 values; a level of
 * at most max_parents[0] parents splits each parent's cameras over 64 lanes, up to
 * max_parents[1] over 16, up to max_parents[2] over 4, up to max_parents[3] over 2,
 * larger levels use one lane per parent.  Of the levels with 64 lanes the smallest take a lane
 * per parent, child and camera instead, and lanes that the scenes' cameras would leave idle are
 * not used (16 lanes for at most 16 cameras, 4 for at most 4).  Values are non-decreasing; the results do
 * not depend on them.  torchhull_amd.tuning measures and stores the fastest values
 * for a device. */
int thull_ctx_set_carve_tuning(thull_ctx* ctx, const uint32_t* max_parents);
int thull_ctx_get_carve_tuning(thull_ctx* ctx, uint32_t* max_parents);

/* Replay of captured carving loops, with no counterpart in the reference (its level loop waits on the
 * host after every launch, src/torchhull/_C/src/visual_hull_cuda.cu:634-751).  When enabled, the
 * first visual-hull run of a batch shape (scene count and each scene's B, H, W, level and flags) is
 * carved host-driven and leaves a plan: capacity-sized level lists and a hipGraph of every level's
 * launches, whose kernels read the level sizes from device memory (a persistent work-queue kernel
 * classifies the large levels).  Later runs of that shape replay the graph with no host wait between
 * levels; a replay whose levels outgrow the capacities is carved again host-driven.  Results do not
 * depend on it.  Up to 4 plans per context; thull_ctx_trim releases them. */
int thull_ctx_set_graph_replay(thull_ctx* ctx, int32_t enabled);
/* Graphs captured, runs replayed and replays that overflowed, since the context was created. */
int thull_ctx_graph_stats(thull_ctx* ctx, int64_t* captures, int64_t* replays, int64_t* overflows);

/* One visual-hull problem (the arguments of torchhull.visual_hull,
 * src/torchhull/_C/python/bindings.cpp:12-21). */
typedef struct thull_scene
{
    const void* masks;        /* device [B,H,W] contiguous; dtype THULL_F32, THULL_U8 or THULL_BOOL */
    int32_t mask_dtype;
    const float* transforms;  /* device [B,4,4] float32 row-major */
    int64_t B, H, W;
    int32_t level;            /* >= 0 */
    int32_t masks_partial;    /* bool */
    int32_t opengl;           /* 1: "opengl", 0: "opencv" */
    float cube_corner_bfl[3];
    float cube_length;        /* > 0 */
} thull_scene;

/* Per-scene result sizes of thull_visual_hull_run. */
typedef struct thull_vh_counts
{
    int64_t num_verts;  /* mesh vertices (soup: 3 * num_faces) */
    int64_t num_faces;
    int64_t num_field;  /* sparse field entries (grid vertices of the leaves) */
    int32_t num_levels; /* candidate lists kept (level + 1 unless carving emptied early) */
    int32_t pad_;
} thull_vh_counts;

/* Carves and meshes `n_scenes` scenes in one batch: integral images, level-
 * synchronous octree carving, corner vertices, field, sparse marching cubes
 * at isolevel 0.5, world coordinates and face flip.  Replaces
 * visual_hull_cuda (src/torchhull/_C/src/visual_hull.cpp:34-58) with
 * sparse_visual_hull_field_cuda_ravelled (src/torchhull/_C/src/visual_hull_cuda.cu:582-894),
 * marching_cubes_cuda_sparse (src/torchhull/_C/src/marching_cubes_cuda.cu:709-754) and
 * to_global_coordinates_and_flip_faces_ (src/torchhull/_C/src/visual_hull_cuda.cu:958-1020).
 * Results stay in the context until the next run; `counts` is host memory of
 * n_scenes entries.  Blocks until the sizes are known. */
int thull_visual_hull_run(thull_ctx* ctx,
                          const thull_scene* scenes,
                          int32_t n_scenes,
                          int32_t unique_verts,
                          void* stream,
                          thull_vh_counts* counts);

/* Join callback of thull_visual_hull_run_join: called on the calling thread before carving step `step`
 * (1, 2, ...) of a run that needs `last_step` steps; it may write up to `max_out` more scenes to `out` and
 * returns how many it wrote (0: none; a negative value aborts the run).  A scene that joins at step s
 * carves its level 0 at step s, so one with level <= last_step - step ends with the scenes in flight.
 * Its device buffers must stay valid, and their contents ready in stream order, until the run returns. */
typedef int32_t (*thull_join_fn)(void* user, int32_t step, int32_t last_step, thull_scene* out, int32_t max_out);

/* thull_visual_hull_run whose octree loop admits more scenes at every level boundary (continuous
 * batching): each carving launch classifies the cells of every scene in flight, each scene at its own
 * octree level, and scenes that join start at level 0 beside deeper ones.  No counterpart in the
 * reference (its visual_hull_cuda, src/torchhull/_C/src/visual_hull.cpp:34-58, carves one scene per
 * call).  `counts` has room for max_scenes entries; *n_total receives the number of scenes run (the
 * n_scenes given, then the joined ones in join order).  Every scene's result equals its result alone. */
int thull_visual_hull_run_join(thull_ctx* ctx,
                               const thull_scene* scenes,
                               int32_t n_scenes,
                               int32_t unique_verts,
                               void* stream,
                               thull_join_fn join,
                               void* user,
                               int32_t max_scenes,
                               thull_vh_counts* counts,
                               int32_t* n_total);

/* Copies scene `scene`'s mesh: verts float32 [num_verts,3], faces int64 [num_faces,3]. */
int thull_visual_hull_fetch_mesh(thull_ctx* ctx, int32_t scene, float* verts, int64_t* faces, void* stream);
/* Copies every scene's mesh at once, scene after scene: verts float32 [sum num_verts,3],
 * faces int64 [sum num_faces,3] (face indices relative to each scene's own vertices). */
int thull_visual_hull_fetch_all(thull_ctx* ctx, float* verts, int64_t* faces, void* stream);

/* Copies scene `scene`'s sparse field as COO: indices int64 [4,num_field] rows (0, z, y, x),
 * values float32 [num_field]; replaces sparse_visual_hull_field_cuda
 * (src/torchhull/_C/src/visual_hull_cuda.cu:896-914, to_sparse_coo_tensor :543-580). */
int thull_visual_hull_fetch_field(thull_ctx* ctx, int32_t scene, int64_t* indices, float* values, void* stream);

/* Number of candidates of single-scene runs at `level` (0..num_levels-1), and their
 * ravelled ids (x + y*2^level + z*4^level) in carving order; replaces the candidate
 * list of visual_hull_with_candidate_voxels (src/torchhull/_C/src/visual_hull.cpp:85-109). */
int thull_visual_hull_candidates_count(thull_ctx* ctx, int32_t level, int64_t* count);
int thull_visual_hull_fetch_candidates(thull_ctx* ctx, int32_t level, int64_t* out, void* stream);

/* Wireframe of `n` candidate cells of level `level` (ravel ids x + y*2^level + z*4^level, device
 * int64): verts float32 [8n,3] at fmaf(cube_length / 2^level, corner index, cube_corner_bfl) per axis
 * (cube_corner_bfl is host memory, 3 floats), edges int64 [12n,2] into those vertices.  Replaces
 * to_wireframe / candidate_voxels_to_wireframes_cuda (src/torchhull/_C/src/visual_hull_cuda.cu:1022-1111).
 * Works on any context; does not touch the context's results. */
int thull_candidate_wireframe(thull_ctx* ctx, const int64_t* cells, int64_t n, int32_t level,
                              const float* cube_corner_bfl, float cube_length, float* verts, int64_t* edges,
                              void* stream);

/* Camera tests (child-camera classifications, early exit included) and children
 * tested at each carving step of the last run, summed over its scenes; host arrays of
 * `max_levels` entries.  Instrumentation for throughput accounting. */
int thull_visual_hull_stats(thull_ctx* ctx, int32_t max_levels, int64_t* camera_tests, int64_t* children);

/* Optional HIP-event timing of every carving classification launch of later runs
 * (no counterpart in the reference; instrumentation for roofline accounting). */
int thull_profile_enable(thull_ctx* ctx, int32_t enabled);
/* Per carving step i of the last run: classification kernel time (ms, 0 when
 * profiling is off), parent cells, camera tests, resulting child cells and the
 * kernel used (split = 1: one thread per parent; 2/4/16/64: lanes per parent; 8: a lane per parent,
 * child and camera, the kernel of the smallest levels; 0: one thread per parent in the persistent
 * work-queue kernel of a replayed carving loop, whose launches a profiled replay runs eagerly, each
 * timed). */
int thull_profile_carve(thull_ctx* ctx, int32_t max_levels, float* ms, int64_t* parents, int64_t* tests,
                        int64_t* next, int32_t* split);

/* Marching cubes on a dense volume [1,D,H,W] (value dtype THULL_F32 or THULL_F64)
 * or a coalesced sparse COO volume (indices int64 [4,nnz], values [nnz]).
 * return_local_coords maps to [-1,1]; otherwise grid units.  Replaces
 * marching_cubes_cuda (src/torchhull/_C/src/marching_cubes_cuda.cu:817-831). */
int thull_marching_cubes_dense_run(thull_ctx* ctx,
                                   const void* volume,
                                   int32_t dtype,
                                   int64_t D,
                                   int64_t H,
                                   int64_t W,
                                   float isolevel,
                                   int32_t return_local_coords,
                                   int32_t unique_verts,
                                   void* stream,
                                   int64_t* num_verts,
                                   int64_t* num_faces);
int thull_marching_cubes_sparse_run(thull_ctx* ctx,
                                    const int64_t* indices,
                                    const void* values,
                                    int32_t dtype,
                                    int64_t nnz,
                                    int64_t D,
                                    int64_t H,
                                    int64_t W,
                                    float isolevel,
                                    int32_t return_local_coords,
                                    int32_t unique_verts,
                                    void* stream,
                                    int64_t* num_verts,
                                    int64_t* num_faces);
int thull_marching_cubes_fetch(thull_ctx* ctx, float* verts, int64_t* faces, void* stream);

/* Gaussian blur of images [B,H,W] (channel 0 of [B,H,W,1]) into out [B,H,W] of
 * out_dtype (THULL_F16, THULL_F32 or THULL_F64); sparse = band blur.  Replaces
 * gaussian_blur_cuda (src/torchhull/_C/src/gaussian_blur_cuda.cu:509-518). */
int thull_gaussian_blur(thull_ctx* ctx,
                        const void* images,
                        int32_t in_dtype,
                        int64_t B,
                        int64_t H,
                        int64_t W,
                        int32_t kernel_size,
                        float sigma,
                        int32_t sparse,
                        void* out,
                        int32_t out_dtype,
                        void* stream);

/* The same blur for `n` image tensors of one input dtype in one launch per pass:
 * images[i] / outs[i] are device [B,H,W] tensors with sizes[3i..3i+2] = (B, H, W).
 * Batched form of gaussian_blur_cuda (src/torchhull/_C/src/gaussian_blur_cuda.cu:509-518). */
int thull_gaussian_blur_batch(thull_ctx* ctx,
                              int32_t n,
                              const void* const* images,
                              int32_t in_dtype,
                              const int64_t* sizes,
                              int32_t kernel_size,
                              float sigma,
                              int32_t sparse,
                              void* const* outs,
                              int32_t out_dtype,
                              void* stream);

/* float32 integral image of masks [B,H,W] (dtype THULL_F32/U8/BOOL); equal to the
 * reference's integral_image (src/torchhull/_C/src/visual_hull_cuda.cu:76-90). */
int thull_integral_image(thull_ctx* ctx,
                         const void* masks,
                         int32_t dtype,
                         int64_t B,
                         int64_t H,
                         int64_t W,
                         float* out,
                         void* stream);

/* The same integral image with nothing allocated: no counterpart in the reference; for callers that
 * cannot allocate device memory (code under HIP graph capture, serving loops, harnesses that forbid
 * hipMalloc).  The column carries and the job descriptor live in a 32 MiB static device array per GPU
 * instead of the context's pool, so B * (ceil(H / 32) - 1) * W carry floats must fit 32 MiB - 256 bytes
 * (larger inputs are rejected with an error).  Every call on one GPU shares that array: calls that
 * overlap in time on one GPU (different streams or host threads) race.  The context's results are not
 * touched. */
int thull_integral_image_noalloc(thull_ctx* ctx,
                                 const void* masks,
                                 int32_t dtype,
                                 int64_t B,
                                 int64_t H,
                                 int64_t W,
                                 float* out,
                                 void* stream);

/* Self-test with no counterpart in the reference: the carving and field kernels
 * divide two numerators by one denominator with a shared reciprocal whenever the
 * operands lie in [2^-40, 2^40] (the IEEE division otherwise).  This runs that
 * helper and the IEEE division on `count` random operand triples on the device
 * and returns the number of quotients whose bits differ (expected 0). */
int thull_selftest_division(thull_ctx* ctx, uint64_t count, uint64_t seed, uint64_t* mismatches, void* stream);

#ifdef __cplusplus
}
#endif

#endif /* TORCHHULL_AMD_H */
