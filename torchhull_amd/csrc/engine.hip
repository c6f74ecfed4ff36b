// Host orchestration and the C ABI of the visual-hull library.
//
// The reference (vc-bonn/torchhull) orchestrates on the host in
// src/torchhull/_C/src/visual_hull_cuda.cu:582-894 with torch allocations,
// CUB/Thrust calls and a stream synchronisation after every launch.  Here one
// batch of scenes goes through the whole pipeline on one stream; the host
// waits only where a size decides the next allocation (one count per octree
// level, the vertex count, the mesh sizes).

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <tuple>
#include <string>
#include <vector>

#include <hip/hip_fp16.h>

#include "../../include/torchhull_amd.h"
#include "kernels.h"
#include "scan.h"

namespace thull
{


namespace
{

thread_local std::string g_last_error;

// ---------------------------------------------------------------------------
// Pooled device memory: chunks are kept for the context's lifetime and handed
// out by a bump pointer that restarts with every call.
// ---------------------------------------------------------------------------

class Pool
{
public:
    ~Pool() { release(); }

    void
    reset()
    {
        for (auto& c : chunks_)
            c.used = 0;
        in_use_ = 0;
    }

    template <typename T>
    T*
    alloc(uint64_t count)
    {
        return static_cast<T*>(alloc_bytes(count * sizeof(T)));
    }

    void*
    alloc_bytes(uint64_t bytes)
    {
        bytes = (bytes + 255) & ~uint64_t(255);
        if (bytes == 0)
            bytes = 256;
        for (auto& c : chunks_)
            if (c.size - c.used >= bytes)
            {
                void* p = c.ptr + c.used;
                c.used += bytes;
                note(bytes);
                return p;
            }
        uint64_t reserved = 0;
        for (auto& c : chunks_)
            reserved += c.size;
        const uint64_t size = std::max<uint64_t>(bytes, std::max<uint64_t>(uint64_t(64) << 20, reserved));
        char* p = nullptr;
        THULL_HIP(hipMalloc(&p, size));
        chunks_.push_back(Chunk{ p, size, bytes });
        note(bytes);
        return p;
    }

    void
    release()
    {
        for (auto& c : chunks_)
            (void)hipFree(c.ptr);
        chunks_.clear();
    }

    uint64_t
    reserved() const
    {
        uint64_t r = 0;
        for (auto& c : chunks_)
            r += c.size;
        return r;
    }

    uint64_t peak() const { return peak_; }

private:
    struct Chunk
    {
        char* ptr;
        uint64_t size;
        uint64_t used;
    };

    void
    note(uint64_t bytes)
    {
        in_use_ += bytes;
        peak_ = std::max(peak_, in_use_);
    }

    std::vector<Chunk> chunks_;
    uint64_t in_use_ = 0;
    uint64_t peak_ = 0;
};

// Pinned host staging for the few counts the host must see.
struct HostStage
{
    unsigned long long* p = nullptr;
    static constexpr int kSlots = 4096;
    HostStage() { THULL_HIP(hipHostMalloc(reinterpret_cast<void**>(&p), kSlots * sizeof(unsigned long long))); }
    ~HostStage() { (void)hipHostFree(p); }
};

// Pinned staging chunks for the host-to-device table copies.  upload() copies
// the bytes into the current chunk and queues the device copy; seal() marks
// the end of a call with an event, and a chunk is reused only after its event
// completed, so a queued copy never sees its bytes overwritten.  A call that
// needs more room than its chunk has left seals it and takes another.
class UploadRing final : public Uploader
{
public:
    UploadRing() = default;
    UploadRing(const UploadRing&) = delete;
    UploadRing& operator=(const UploadRing&) = delete;
    ~UploadRing()
    {
        for (auto& c : chunks_)
        {
            (void)hipEventDestroy(c.ev);
            (void)hipHostFree(c.p);
        }
    }

    void
    upload(void* dst, const void* src, size_t bytes, hipStream_t st) override
    {
        if (bytes == 0)
            return;
        const size_t need = (bytes + 255) & ~size_t(255);
        if (cur_ < 0 || chunks_[cur_].used + need > chunks_[cur_].cap)
        {
            seal(st);
            cur_ = take(need);
        }
        Chunk& c = chunks_[cur_];
        char* p = c.p + c.used;
        c.used += need;
        std::memcpy(p, src, bytes);
        THULL_HIP(hipMemcpyAsync(dst, p, bytes, hipMemcpyHostToDevice, st));
    }

    // The copies queued so far on `st` are the last ones reading the current chunk.
    void
    seal(hipStream_t st)
    {
        if (cur_ < 0)
            return;
        Chunk& c = chunks_[cur_];
        if (c.used > 0)
        {
            THULL_HIP(hipEventRecord(c.ev, st));
            c.recorded = true;
        }
        cur_ = -1;
    }

private:
    struct Chunk
    {
        char* p = nullptr;
        size_t cap = 0, used = 0;
        hipEvent_t ev = nullptr;
        bool recorded = false;
    };
    static constexpr size_t kChunk = size_t(1) << 20;
    std::vector<Chunk> chunks_;
    int cur_ = -1;

    int
    take(size_t need)
    {
        for (size_t i = 0; i < chunks_.size(); ++i)
        {
            Chunk& c = chunks_[i];
            if (c.cap < need)
                continue;
            if (c.recorded)
            {
                const hipError_t q = hipEventQuery(c.ev);
                if (q == hipErrorNotReady)
                    continue;
                THULL_HIP(q);
                c.recorded = false;
            }
            c.used = 0;
            return int(i);
        }
        Chunk c;
        c.cap = std::max(kChunk, need);
        THULL_HIP(hipHostMalloc(reinterpret_cast<void**>(&c.p), c.cap));
        const hipError_t e = hipEventCreateWithFlags(&c.ev, hipEventDisableTiming);
        if (e != hipSuccess)
        {
            (void)hipHostFree(c.p);
            THULL_HIP(e);
        }
        chunks_.push_back(c);
        return int(chunks_.size()) - 1;
    }
};

// Coherent pinned words that scan kernels write their totals to (ScanNotify):
// the host learns a level's size as soon as its scan ends, while the kernels
// queued after the scan still run, instead of waiting for the whole stream.
class HostNotify
{
public:
    HostNotify()
    {
        THULL_HIP(hipHostMalloc(reinterpret_cast<void**>(&host_), (4 + kTable) * sizeof(unsigned long long),
                                hipHostMallocCoherent | hipHostMallocMapped));
        const hipError_t e = hipHostGetDevicePointer(reinterpret_cast<void**>(&dev_), host_, 0);
        if (e != hipSuccess)
        {
            (void)hipHostFree(host_);
            THULL_HIP(e);
        }
        host_[0] = host_[1] = host_[2] = 0;
    }
    HostNotify(const HostNotify&) = delete;
    HostNotify& operator=(const HostNotify&) = delete;
    ~HostNotify() { (void)hipHostFree(host_); }

    // The notification for the next scan (a fresh sequence number).
    ScanNotify
    next(const unsigned long long* extra)
    {
        return ScanNotify{ dev_, extra, ++seq_ };
    }

    // Words that a kernel may write ahead of its notification.
    static constexpr int kTable = 3 * 256;
    unsigned long long* dev_table() const { return dev_ + 4; }
    const unsigned long long* table() const { return host_ + 4; }

    // Waits for the notification `n` (queued on `st`); false when the stream went idle without it,
    // and the caller then reads the values from device memory.
    bool
    wait(const ScanNotify& n, hipStream_t st, unsigned long long (&out)[2]) const
    {
        volatile unsigned long long* v = host_;
        for (uint32_t i = 1;; ++i)
        {
            if (v[2] == n.seq)
            {
                std::atomic_thread_fence(std::memory_order_acquire);
                out[0] = v[0];
                out[1] = v[1];
                return true;
            }
            if ((i & 255u) == 0u)
            {
                const hipError_t q = hipStreamQuery(st);
                if (q == hipSuccess)
                    return v[2] == n.seq ? wait(n, st, out) : false;
                if (q != hipErrorNotReady)
                    THULL_HIP(q);
            }
            __builtin_ia32_pause();
        }
    }

private:
    unsigned long long* host_ = nullptr;
    unsigned long long* dev_ = nullptr;
    unsigned long long seq_ = 0;
};

// ---------------------------------------------------------------------------
// Device scratch of the allocation-free integral-image entry point: one static
// array per device, holding the job descriptor (first 256 bytes) and the
// column carries.  Its device address is looked up once per device, with that
// device current, when the first context of the device is created; host code
// uses that address only (the array's name is a host-side stand-in).
// ---------------------------------------------------------------------------

constexpr size_t kScratchBytes = size_t(32) << 20;
constexpr size_t kScratchJobBytes = 256;

static __device__ __align__(256) unsigned char scratch[kScratchBytes];

std::mutex g_scratch_mu;
std::vector<void*> g_scratch_ptr; // by device index

// Called with `device` current.
void*
scratch_for_device(int device)
{
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_ptr.size() <= size_t(device))
        g_scratch_ptr.resize(size_t(device) + 1, nullptr);
    if (g_scratch_ptr[device] == nullptr)
    {
        void* ptr = nullptr;
        THULL_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
        THULL_CHECK(ptr != nullptr, "device scratch has no address");
        g_scratch_ptr[device] = ptr;
    }
    return g_scratch_ptr[device];
}

// Host-to-device copies of small tables through kernel arguments (64 words per launch, vector
// stores): no pinned staging memory, no copy engine, nothing allocated.
struct Words64
{
    uint32_t w[64];
};

__global__ __launch_bounds__(64) void
store_words_kernel(Words64 src, uint32_t nwords, uint32_t* __restrict__ dst)
{
    const uint32_t i = threadIdx.x;
    if (i < nwords)
        dst[i] = src.w[i];
}

class KernelUploader final : public Uploader
{
public:
    void
    upload(void* dst, const void* src, size_t bytes, hipStream_t st) override
    {
        THULL_CHECK(bytes % 4 == 0 && reinterpret_cast<uintptr_t>(dst) % 4 == 0,
                    "kernel uploads move whole aligned words");
        for (size_t off = 0; off < bytes; off += sizeof(Words64))
        {
            Words64 w{};
            const size_t n = std::min(sizeof(Words64), bytes - off);
            std::memcpy(w.w, static_cast<const char*>(src) + off, n);
            store_words_kernel<<<1, 64, 0, st>>>(w, uint32_t(n / 4), reinterpret_cast<uint32_t*>(
                                                                           static_cast<char*>(dst) + off));
            THULL_LAUNCH_CHECK();
        }
    }
};

// A captured carving loop for one batch shape: capacity-sized level lists in device memory of its
// own, level sizes counted on the device (the host never waits between levels), and a hipGraph of all
// the levels' launches, replayed for every later batch of that shape.  The capacities come from the
// level sizes of a host-driven run of the shape, with headroom; a replay whose levels outgrow them
// raises an overflow flag and the batch is run again host-driven.
struct CarvePlan
{
    std::vector<int64_t> sig;   // batch shape: scene count and per scene B, H, W, level, flags
    int32_t steps = 0;          // carving steps of the loop
    std::vector<uint32_t> cap;  // list capacities of levels 0 .. steps
    std::vector<int32_t> split; // kernel of every step (launch_carve_classify)
    std::vector<uint64_t> roots;
    char* arena = nullptr;
    SceneDev* scenes = nullptr;
    std::vector<uint64_t*> lists;
    std::vector<uint8_t*> masks;
    std::vector<uint32_t*> bcount, boff, sums;
    unsigned long long* status = nullptr; // level sizes [steps + 1], camera tests [steps]
    uint32_t* cursors = nullptr;          // 8 work-queue cursors per step
    uint32_t* overflow = nullptr;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    uint64_t replays = 0;

    CarvePlan() = default;
    CarvePlan(const CarvePlan&) = delete;
    CarvePlan& operator=(const CarvePlan&) = delete;
    ~CarvePlan()
    {
        if (exec != nullptr)
            (void)hipGraphExecDestroy(exec);
        if (graph != nullptr)
            (void)hipGraphDestroy(graph);
        if (arena != nullptr)
            (void)hipFree(arena);
    }
};

} // namespace

struct Context
{
    int device = 0;
    void* scratch = nullptr; // this device's allocation-free scratch (scratch_for_device)
    Pool pool;
    HostStage* stage = nullptr;
    UploadRing upload;
    HostNotify notify;
    CarveTuning tuning;
    hipStream_t last_stream = nullptr;
    bool have_last = false;

    // last visual-hull run; its results are valid until the next call resets the pool
    bool vh_valid = false;
    int32_t n_scenes = 0;
    bool unique = true;
    std::vector<thull_vh_counts> counts;
    std::vector<uint32_t> scene_vstart, scene_tstart, scene_first;
    std::vector<SceneDev> scenes_host;
    std::vector<uint64_t*> level_lists;
    std::vector<uint32_t> level_sizes;
    std::vector<int64_t> level_tests, level_children;
    uint64_t* vertices = nullptr;
    float* values = nullptr;
    float* verts = nullptr;
    int64_t* faces = nullptr;

    // replay of captured carving loops for repeated batch shapes (thull_ctx_set_graph_replay)
    bool graph_replay = false;
    std::vector<std::unique_ptr<CarvePlan>> plans; // most recently used last
    hipStream_t capture_stream = nullptr;
    int64_t graph_replays = 0, graph_captures = 0, graph_overflows = 0;

    // optional HIP-event timing of the carving classification launches
    bool profile = false;
    std::vector<hipEvent_t> ev_pool;
    std::vector<float> carve_ms;
    std::vector<int64_t> carve_parents, carve_next;
    std::vector<int32_t> carve_split;

    hipEvent_t
    event(size_t i)
    {
        while (ev_pool.size() <= i)
        {
            hipEvent_t e;
            THULL_HIP(hipEventCreate(&e));
            ev_pool.push_back(e);
        }
        return ev_pool[i];
    }

    // device weight tables of the blur, keyed by (kernel size, sigma bits, output dtype, sparse)
    struct BlurWeights
    {
        void* dev;
        double norm;
    };
    std::map<std::tuple<int, uint32_t, int, int>, BlurWeights> blur_weights;

    ~Context()
    {
        plans.clear();
        if (capture_stream != nullptr)
            (void)hipStreamDestroy(capture_stream);
        for (auto& kv : blur_weights)
            (void)hipFree(kv.second.dev);
        for (auto e : ev_pool)
            (void)hipEventDestroy(e);
    }

    // last marching-cubes run
    bool mc_valid = false;
    float* mc_verts = nullptr;
    int64_t* mc_faces = nullptr;
    int64_t mc_nv = 0, mc_nf = 0;

    void
    begin(hipStream_t st)
    {
        THULL_HIP(hipSetDevice(device));
        if (have_last)
        {
            // the staging chunk of the previous call is free once its stream passes this point
            upload.seal(last_stream);
            if (last_stream != st)
                THULL_HIP(hipStreamSynchronize(last_stream));
        }
        last_stream = st;
        have_last = true;
        invalidate();
        pool.reset();
    }

    // Forgets the results of the last visual-hull and marching-cubes runs (their pool memory is
    // about to be reused or released): fetches then fail instead of copying stale memory.
    void
    invalidate()
    {
        vh_valid = false;
        n_scenes = 0;
        counts.clear();
        level_lists.clear();
        level_sizes.clear();
        level_tests.clear();
        level_children.clear();
        vertices = nullptr;
        values = nullptr;
        verts = nullptr;
        faces = nullptr;
        mc_valid = false;
        mc_verts = nullptr;
        mc_faces = nullptr;
        mc_nv = mc_nf = 0;
    }

    unsigned long long
    read_u64(const unsigned long long* dev, hipStream_t st)
    {
        THULL_HIP(hipMemcpyAsync(stage->p, dev, sizeof(unsigned long long), hipMemcpyDeviceToHost, st));
        THULL_HIP(hipStreamSynchronize(st));
        return stage->p[0];
    }
};

namespace
{

template <typename F>
int
guarded(F&& f)
{
    try
    {
        f();
        g_last_error.clear();
        return 0;
    }
    catch (const std::exception& e)
    {
        g_last_error = e.what();
        return 1;
    }
    catch (...)
    {
        g_last_error = "unknown error";
        return 1;
    }
}

struct LoadPopcount
{
    const uint32_t* w;
    __device__ uint32_t operator()(uint64_t i) const { return __popc(w[i]); }
};

struct LoadPopcountMask
{
    const uint32_t* m;
    __device__ uint32_t operator()(uint64_t i) const { return __popc(m[i] & 7u); }
};

// Per scene: first vertex position, first output vertex and first triangle-vertex, the latter two also as the tables of
// the faces kernel.  One block sends them, after the two totals, to the host by `note` and `host_out`.
__global__ __launch_bounds__(256) void
scene_starts_kernel(const uint64_t* word_begin,
                    int32_t n,
                    uint64_t nwords,
                    const uint32_t* bitmap_prefix,
                    uint64_t nverts,
                    const uint32_t* vbase,
                    const uint32_t* tbase,
                    const unsigned long long* totals, // triangle vertices, output vertices (unique meshes)
                    bool unique,
                    unsigned long long* out,
                    uint32_t* vstart,
                    uint32_t* tstart,
                    unsigned long long* host_out, // with note: one block, n < 256
                    ScanNotify note)
{
    const int32_t s = blockIdx.x * 256 + threadIdx.x;
    const uint64_t ttotal = totals[0], vtotal = unique ? totals[1] : ttotal;
    if (s <= n)
    {
        uint64_t first = nverts;
        if (s < n && word_begin[s] < nwords)
            first = bitmap_prefix[word_begin[s]];
        uint64_t vs = vtotal, ts = ttotal;
        if (first < nverts)
        {
            ts = tbase[first];
            vs = vbase != nullptr ? vbase[first] : ts; // soup vertices sit at the triangle-vertex slots
        }
        out[3 * s + 0] = first;
        out[3 * s + 1] = vs;
        out[3 * s + 2] = ts;
        if (note.slot != nullptr)
        {
            host_out[3 * s + 0] = first;
            host_out[3 * s + 1] = vs;
            host_out[3 * s + 2] = ts;
        }
        vstart[s] = uint32_t(vs);
        tstart[s] = uint32_t(ts);
    }
    if (note.slot == nullptr)
        return;
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0)
    {
        note.slot[0] = ttotal;
        note.slot[1] = vtotal;
        __hip_atomic_store(note.slot + 2, note.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

__global__ void
keys_to_ravel_kernel(const uint64_t* keys, uint32_t n, int32_t level, int64_t* out)
{
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n)
        return;
    const uint64_t k = keys[i];
    const int64_t R = int64_t(1) << level;
    out[i] = int64_t(key_x(k)) + int64_t(key_y(k)) * R + int64_t(key_z(k)) * R * R;
}

__global__ void
field_coo_kernel(const uint64_t* keys, const float* values, uint32_t n, int64_t* coo, float* vals)
{
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n)
        return;
    const uint64_t k = keys[i];
    coo[i] = 0;
    coo[n + i] = key_z(k);
    coo[2 * uint64_t(n) + i] = key_y(k);
    coo[3 * uint64_t(n) + i] = key_x(k);
    vals[i] = values[i];
}

void
check_u32(uint64_t v, const char* what)
{
    if (v >= (uint64_t(1) << 32))
        throw Error(std::string(what) + " exceeds 2^32 entries");
}

} // namespace

// ---------------------------------------------------------------------------
// Visual hull
// ---------------------------------------------------------------------------

// Builds the plan of a batch shape from a host-driven run of it: level capacities with 25 % headroom
// (plus 256), the run's lanes per parent, the roots uploaded once.
static CarvePlan*
make_plan(Context& ctx, std::vector<int64_t> sig, const std::vector<uint64_t>& roots, int32_t steps, hipStream_t st)
{
    auto p = std::make_unique<CarvePlan>();
    p->sig = std::move(sig);
    p->steps = steps;
    p->roots = roots;
    p->cap.assign(size_t(steps) + 1, 256u);
    p->cap[0] = uint32_t(std::max<size_t>(roots.size(), 1));
    for (int32_t i = 1; i <= steps; ++i)
    {
        const uint64_t seen = i < int32_t(ctx.level_sizes.size()) ? ctx.level_sizes[i] : 0;
        p->cap[i] = uint32_t(std::min<uint64_t>(seen + seen / 4 + 256, uint64_t(8) * p->cap[i - 1]));
    }
    p->split.resize(size_t(steps));
    for (int32_t i = 0; i < steps; ++i)
        p->split[i] = i < int32_t(ctx.carve_split.size()) && ctx.carve_split[i] > 0
                          ? ctx.carve_split[i]
                          : carve_split_factor(p->cap[i], ctx.tuning);
    // one allocation for every buffer of the loop
    std::vector<size_t> sizes;
    auto add = [&](size_t bytes) {
        sizes.push_back((bytes + 255) & ~size_t(255));
        return sizes.size() - 1;
    };
    const size_t i_scenes = add(p->sig[0] * sizeof(SceneDev));
    const size_t i_status = add((2 * size_t(steps) + 1) * sizeof(unsigned long long));
    const size_t i_cursors = add(8 * size_t(std::max(steps, 1)) * sizeof(uint32_t));
    const size_t i_overflow = add(sizeof(uint32_t));
    std::vector<size_t> i_list, i_mask, i_bc, i_bo, i_sums;
    for (int32_t i = 0; i <= steps; ++i)
        i_list.push_back(add(size_t(p->cap[i]) * sizeof(uint64_t)));
    for (int32_t i = 0; i < steps; ++i)
    {
        const uint32_t nb = blocks_for(p->cap[i], kCarveThreads);
        i_mask.push_back(add(p->cap[i]));
        i_bc.push_back(add(size_t(nb) * sizeof(uint32_t)));
        i_bo.push_back(add(size_t(nb) * sizeof(uint32_t)));
        i_sums.push_back(add(size_t(scan_sums_room(nb)) * sizeof(uint32_t)));
    }
    size_t total = 0;
    std::vector<size_t> off(sizes.size());
    for (size_t k = 0; k < sizes.size(); ++k)
    {
        off[k] = total;
        total += sizes[k];
    }
    THULL_HIP(hipMalloc(&p->arena, total));
    char* a = p->arena;
    p->scenes = reinterpret_cast<SceneDev*>(a + off[i_scenes]);
    p->status = reinterpret_cast<unsigned long long*>(a + off[i_status]);
    p->cursors = reinterpret_cast<uint32_t*>(a + off[i_cursors]);
    p->overflow = reinterpret_cast<uint32_t*>(a + off[i_overflow]);
    for (int32_t i = 0; i <= steps; ++i)
        p->lists.push_back(reinterpret_cast<uint64_t*>(a + off[i_list[i]]));
    for (int32_t i = 0; i < steps; ++i)
    {
        p->masks.push_back(reinterpret_cast<uint8_t*>(a + off[i_mask[i]]));
        p->bcount.push_back(reinterpret_cast<uint32_t*>(a + off[i_bc[i]]));
        p->boff.push_back(reinterpret_cast<uint32_t*>(a + off[i_bo[i]]));
        p->sums.push_back(reinterpret_cast<uint32_t*>(a + off[i_sums[i]]));
    }
    ctx.upload.upload(p->lists[0], roots.data(), roots.size() * sizeof(uint64_t), st);
    constexpr size_t kMaxPlans = 4;
    if (ctx.plans.size() >= kMaxPlans)
    {
        THULL_HIP(hipStreamSynchronize(st)); // the evicted plan's graph may still run on this stream
        ctx.plans.erase(ctx.plans.begin());
    }
    ctx.plans.push_back(std::move(p));
    return ctx.plans.back().get();
}

// The most cameras of a scene (launch_carve_classify).
static int32_t
max_cameras(const std::vector<SceneDev>& sd)
{
    int32_t most = 0;
    for (const SceneDev& d : sd)
        most = std::max(most, d.B);
    return most;
}

// The launches of a plan's carving loop, as captured into its graph: counters cleared by kernels (no
// memset nodes), then per step the classification (a persistent work-queue kernel, or the lane-split
// kernel on a capacity-sized grid), the scan of the block counts whose total is the next level's size,
// the capacity guard and the scatter -- every kernel reads its level's size from device memory.
// With `timed`, the launches run eagerly with HIP events around every classification (the profile of
// a replayed loop: the same kernels as the graph, timed one by one).
static void
record_plan(Context& ctx, CarvePlan& p, const std::vector<SceneDev>& sd, int32_t n, hipStream_t st,
            bool timed = false)
{
    const int32_t steps = p.steps;
    unsigned long long* counts = p.status;
    unsigned long long* tests = p.status + steps + 1;
    launch_fill_u32(reinterpret_cast<uint32_t*>(p.status), 2 * (2 * uint64_t(steps) + 1), 0u, st);
    launch_fill_u32(reinterpret_cast<uint32_t*>(counts), 1, uint32_t(n), st); // level 0: the roots
    launch_fill_u32(p.cursors, 8 * uint64_t(std::max(steps, 1)), 0u, st);
    launch_fill_u32(p.overflow, 1, 0u, st);
    for (int32_t i = 0; i < steps; ++i)
        if (p.split[i] == 1) // the queue kernel writes the counts of the blocks it takes only
            launch_fill_u32(p.bcount[i], blocks_for(p.cap[i], kCarveThreads), 0u, st);
    for (int32_t i = 0; i < steps; ++i)
    {
        const uint32_t nb = blocks_for(p.cap[i], kCarveThreads);
        if (timed)
            THULL_HIP(hipEventRecord(ctx.event(2 * i), st));
        p.split[i] = launch_carve_classify(p.lists[i], p.cap[i], i, p.scenes, p.masks[i], p.bcount[i], tests + i,
                                           ctx.tuning, max_cameras(sd), carve_culls(sd.data(), sd.size(), i), st,
                                           counts + i, p.split[i], p.cursors + 8 * i);
        if (timed)
            THULL_HIP(hipEventRecord(ctx.event(2 * i + 1), st));
        // the next level's size, clamped to its list's capacity (overflow: the run is repeated)
        exclusive_scan(LoadU32{ p.bcount[i] }, nb, p.boff[i], p.sums[i], counts + i + 1, st, {},
                       ScanGuard{ p.cap[i + 1], p.overflow });
        bool target = false;
        for (const SceneDev& d : sd)
            target |= d.level == i + 1;
        launch_carve_scatter(p.lists[i], p.cap[i], p.masks[i], p.boff[i], p.lists[i + 1], i + 1, p.scenes, target, st,
                             counts + i, p.cap[i + 1]);
    }
}

// A caller's join callback (thull_visual_hull_run_join): before carving step `step` (> 0) it may hand
// over up to `max_out` more scenes, which start their octree at that step.
using JoinFn = int32_t (*)(void* user, int32_t step, int32_t last_step, thull_scene* out, int32_t max_out);

static void
check_scene(const thull_scene& sc)
{
    THULL_CHECK(sc.level >= 0 && sc.level <= 15, "level must be in [0, 15]");
    THULL_CHECK(sc.cube_length > 0.0f, "cube_length must be positive");
    THULL_CHECK(sc.B >= 0 && sc.H >= 0 && sc.W >= 0, "mask sizes must be non-negative");
    THULL_CHECK(sc.H * sc.W < (int64_t(1) << 31), "H * W must be below 2^31");
    // pixel rounding in float and 32-bit byte offsets into a camera's padded integral plane
    THULL_CHECK(sc.H < (int64_t(1) << 23) && sc.W < (int64_t(1) << 23), "H and W must be below 2^23");
    THULL_CHECK(integral_rows(sc.H) * integral_pitch(sc.W) < (int64_t(1) << 30),
                "(H + 1 rounded up to 4) * integral pitch (W + 32, rounded up to 32) must be below 2^30");
    THULL_CHECK(sc.mask_dtype == kF32 || sc.mask_dtype == kU8 || sc.mask_dtype == kBool,
                "masks must be float32, uint8 or bool at the C ABI");
}

// Solid maps and the field by bricks cost a few launches and a sixteenth of a pass over the masks, and save camera
// tests and samples of the scenes' surface cells, about 4^level of them in every camera: they are used from
// kMinCellCameras cell-cameras in the scenes a run starts with (16.8 million, 64 cameras at level 9: 1.75 -> 1.41 ms;
// 6.3 million, 24 cameras at level 9: 0.79 -> 0.74, and in 10 mixed scenes: 1.55 -> 1.68; 3.3 million, 50 cameras at
// level 8: 1.06 -> 1.03; 0.7 million, 10 cameras at level 8: 0.41 -> 0.47).
static bool
solid_maps_pay(const thull_scene* scenes, int32_t n)
{
    constexpr int64_t kMinCellCameras = int64_t(1) << 23;
    int64_t work = 0;
    for (int32_t i = 0; i < n; ++i)
        work += std::max<int64_t>(scenes[i].B, 0) << (2 * std::clamp(scenes[i].level, 0, 12));
    return work >= kMinCellCameras;
}

static bool
has_solid_map(const thull_scene& sc)
{
    return sc.H >= 4 * kSolidTile && sc.W >= 4 * kSolidTile && sc.B >= 3;
}

static void
visual_hull_run(Context& ctx, const thull_scene* in, int32_t n0, bool unique, hipStream_t st, thull_vh_counts* counts,
                JoinFn join, void* user, int32_t max_scenes, int32_t* n_total)
{
    THULL_CHECK(n0 >= 1 && n0 < 65536, "n_scenes must be in [1, 65535]");
    const int32_t capacity = join != nullptr ? max_scenes : n0;
    THULL_CHECK(capacity >= n0 && capacity < 65536, "max_scenes must be in [n_scenes, 65535]");
    ctx.begin(st);
    Pool& pool = ctx.pool;
    ctx.unique = unique;
    ctx.carve_ms.clear();
    ctx.carve_parents.clear();
    ctx.carve_next.clear();
    ctx.carve_split.clear();
    std::vector<thull_scene> all;   // every scene of the run, the joined ones after the first n0
    std::vector<SceneDev> sd;
    std::vector<uint64_t> word_begin; // first vertex-bitmap word of each scene
    uint64_t total_words = 0;
    int32_t last_step = 0; // carving steps the run needs: max over scenes of start + level
    uint32_t* first_cells = nullptr; // leaf-cell bitmaps of the initial scenes
    uint64_t first_cell_words = 0;
    // descriptors, roots, first words and grids: one block, which goes up in one copy when no scene can join (a small
    // hull spends most of its time between launches; with the starts sent by their kernel, 9 copies, 2 launches and a
    // stream synchronisation less: a level-7 hull of 8 cameras 351 -> 294 us)
    static_assert(sizeof(SceneDev) % 8 == 0 && alignof(SceneDev) <= 8 && alignof(McGrid) <= 8, "table of 8-byte parts");
    const size_t room_all = size_t(std::max(capacity, 1));
    SceneDev* scenes = reinterpret_cast<SceneDev*>(pool.alloc_bytes(
            room_all * (sizeof(SceneDev) + 2 * sizeof(uint64_t) + sizeof(McGrid)) + sizeof(uint64_t)));
    uint64_t* const root_list = reinterpret_cast<uint64_t*>(scenes + room_all);
    uint64_t* const dev_word_begin = root_list + room_all;
    McGrid* const dgrids = reinterpret_cast<McGrid*>(dev_word_begin + room_all + 1);
    // camera-test counters of every carving step (a joined scene ends by the last step), cleared with the first cells
    constexpr int32_t kMaxSteps = 64;
    unsigned long long* dev_tests = nullptr;
    unsigned long long* dev_total = pool.alloc<unsigned long long>(2);

    // Adds scenes k0 .. all.size() - 1, which start at carving step `start`: descriptors, integral images
    // (one launch per pass for all of them), cleared leaf-cell bitmaps and the roots of level-0 scenes;
    // returns their root keys.  The roots go in order of falling per-cell cost (cameras, then depth):
    // every level's list keeps the scenes in root order, so each carving launch starts with its most
    // expensive cells and ends with the cheapest ones instead of finishing on a tail of many-camera
    // cells.  Each scene's own cells keep the reference's parent-major order, so no result depends on it.
    const bool by_bricks = solid_maps_pay(in, n0);
    uint64_t most_flags = 0;
    // marching-cubes grids of all scenes: isolevel 0.5, world coordinates, flipped faces
    const auto scene_grids = [&] {
        std::vector<McGrid> grids(all.size());
        for (size_t s = 0; s < all.size(); ++s)
        {
            McGrid g{};
            const uint32_t R1 = (1u << std::max(0, all[s].level)) + 1u;
            g.dims[0] = g.dims[1] = g.dims[2] = R1;
            g.row_words = sd[s].row_words;
            g.bitmap_offset = sd[s].bitmap_offset;
            g.out_mode = 2;
            const float scale = all[s].cube_length / float(int64_t(1) << std::max(0, all[s].level));
            g.scale[0] = g.scale[1] = g.scale[2] = scale;
            g.corner[0] = all[s].cube_corner_bfl[0];
            g.corner[1] = all[s].cube_corner_bfl[1];
            g.corner[2] = all[s].cube_corner_bfl[2];
            g.flip = 1;
            grids[s] = g;
        }
        return grids;
    };
    auto add_scenes = [&](size_t k0, int32_t start) {
        const size_t k1 = all.size();
        std::vector<IntegralRequest> ireq;
        uint64_t cell_words = 0;
        for (size_t s = k0; s < k1; ++s)
        {
            const thull_scene& sc = all[s];
            check_scene(sc);
            SceneDev d{};
            d.masks = sc.masks;
            d.mask_dtype = sc.mask_dtype;
            d.transforms = sc.transforms;
            // A scene without cameras refines nothing: its candidates are the root, then none
            // (VH:627-751 with an empty camera loop); a level-0 scene keeps the root cell, whose field
            // is the empty product 1.  Cameras with an empty image (H or W zero) are out of the
            // reference's domain (its pixel clamp to [0, size - 1] is empty); here they constrain
            // nothing, like no camera at all.
            d.B = (sc.H == 0 || sc.W == 0) ? 0 : int32_t(sc.B);
            d.H = int32_t(sc.H);
            d.W = int32_t(sc.W);
            d.level = sc.level;
            d.partial = sc.masks_partial;
            d.opengl = sc.opengl;
            d.corner[0] = sc.cube_corner_bfl[0];
            d.corner[1] = sc.cube_corner_bfl[1];
            d.corner[2] = sc.cube_corner_bfl[2];
            d.length = sc.cube_length;
            d.start = start;
            const uint64_t R = uint64_t(1) << sc.level, R1 = R + 1;
            d.row_words = uint32_t((R1 + 31) / 32);
            if (by_bricks)
                d.row_words = (d.row_words + 3u) & ~3u; // whole groups of words (launch_dilate_groups)
            d.bitmap_offset = total_words;
            d.cell_row_words = uint32_t((R + 31) / 32);
            word_begin.push_back(total_words);
            total_words += R1 * R1 * d.row_words;
            cell_words += (R * R * d.cell_row_words + 3) & ~uint64_t(3); // 16-byte aligned scenes
            last_step = std::max(last_step, start + d.level);
            if (d.B > 0)
            {
                float* integral = pool.alloc<float>(uint64_t(sc.B) * uint64_t(integral_rows(sc.H)) *
                                                    uint64_t(integral_pitch(sc.W)));
                IntegralRequest r{ sc.masks, sc.mask_dtype, sc.B, sc.H, sc.W, integral };
                d.integral = integral;
                if (by_bricks && has_solid_map(sc))
                {
                    r.solid = pool.alloc<uint8_t>(solid_map_bytes(sc.B, sc.H, sc.W));
                    r.cull = pool.alloc<CullCamera>(uint64_t(sc.B));
                    r.solid_scratch = pool.alloc_bytes(solid_scratch_bytes(sc.B, sc.H, sc.W));
                    r.culls = &scenes[s].culls;
                    r.transforms = sc.transforms;
                    r.opengl = sc.opengl;
                    std::copy(sc.cube_corner_bfl, sc.cube_corner_bfl + 3, r.corner);
                    r.length = sc.cube_length;
                    d.solid = r.solid;
                    d.cull = r.cull;
                    d.solid_h = int32_t(sc.H / kSolidTile);
                    d.solid_w = int32_t(sc.W / kSolidTile);
                }
                ireq.push_back(r);
            }
            sd.push_back(d);
        }
        // brick bitmaps, and leaf-cell bitmaps, filled by the scatter of each scene's last carving step
        uint64_t brick_words = 0;
        for (size_t s = k0; by_bricks && s < k1; ++s)
        {
            sd[s].brick_shift = std::min(kBrickShift, sd[s].level);
            brick_words += ((uint64_t(1) << (3 * (sd[s].level - sd[s].brick_shift))) + 31) / 32;
            const uint64_t flags = group_flag_bytes(sd[s].level, sd[s].brick_shift, sd[s].row_words);
            sd[s].group_flags = pool.alloc<uint8_t>(flags);
            most_flags = std::max(most_flags, flags);
        }
        const uint64_t test_words = k0 == 0 ? 2 * kMaxSteps : 0; // keep the cells' alignment
        uint32_t* cells = pool.alloc<uint32_t>(std::max<uint64_t>(test_words + cell_words + brick_words, 1));
        launch_fill_u32(cells, test_words + cell_words + brick_words, 0u, st);
        if (k0 == 0)
            dev_tests = reinterpret_cast<unsigned long long*>(cells);
        cells += test_words;
        for (size_t s = k0, w = cell_words; by_bricks && s < k1; ++s)
        {
            sd[s].bricks = cells + w;
            w += ((size_t(1) << (3 * (sd[s].level - sd[s].brick_shift))) + 31) / 32;
        }
        if (k0 == 0)
        {
            first_cells = cells;
            first_cell_words = cell_words;
        }
        uint64_t off = 0;
        for (size_t s = k0; s < k1; ++s)
        {
            sd[s].cells = cells + off;
            off += ((uint64_t(1) << (2 * sd[s].level)) * sd[s].cell_row_words + 3) & ~uint64_t(3);
        }
        std::vector<int32_t> order;
        for (size_t s = k0; s < k1; ++s)
            order.push_back(int32_t(s));
        std::stable_sort(order.begin(), order.end(), [&](int32_t a, int32_t b) {
            return sd[a].B != sd[b].B ? sd[a].B > sd[b].B : sd[a].level > sd[b].level;
        });
        std::vector<uint64_t> roots(order.size());
        for (size_t k = 0; k < order.size(); ++k)
            roots[k] = pack_key(uint32_t(order[k]), 0, 0, 0);
        if (join == nullptr)
        {
            word_begin.push_back(total_words);
            const std::vector<McGrid> grids = scene_grids();
            std::vector<char> table;
            const auto put = [&](const void* p, size_t bytes) {
                table.insert(table.end(), static_cast<const char*>(p), static_cast<const char*>(p) + bytes);
            };
            put(sd.data(), sd.size() * sizeof(SceneDev));
            put(roots.data(), roots.size() * sizeof(uint64_t));
            put(word_begin.data(), word_begin.size() * sizeof(uint64_t));
            put(grids.data(), grids.size() * sizeof(McGrid));
            ctx.upload.upload(scenes, table.data(), table.size(), st);
        }
        else
            ctx.upload.upload(scenes + k0, sd.data() + k0, (k1 - k0) * sizeof(SceneDev), st);
        // after the descriptors: the solid map pass sets SceneDev::culls
        uint64_t carry_floats = 0;
        for (const auto& r : ireq)
            carry_floats += integral_carry_floats(r.B, r.H, r.W);
        launch_integral_images_padded(ireq.data(), int32_t(ireq.size()),
                                      pool.alloc<float>(std::max<uint64_t>(carry_floats, 1)),
                                      pool.alloc_bytes(integral_job_bytes(std::max<size_t>(ireq.size(), 1))),
                                      pool.alloc_bytes(solid_job_bytes(ireq.size())), ctx.upload, st);
        if (std::any_of(sd.begin() + k0, sd.end(), [](const SceneDev& d) { return d.level == 0; }))
            launch_mark_root_cells(scenes, int32_t(k0), int32_t(k1 - k0), st);
        return roots;
    };

    all.assign(in, in + n0);
    std::vector<uint64_t> roots = add_scenes(0, 0);
    uint64_t* list = root_list; // with room for the roots of scenes that may still join
    if (join != nullptr)
        ctx.upload.upload(list, roots.data(), roots.size() * sizeof(uint64_t), st);
    uint32_t count = uint32_t(roots.size());
    ctx.level_lists.push_back(list);
    ctx.level_sizes.push_back(count);

    // ---- replay of the captured carving loop of this batch shape (thull_ctx_set_graph_replay) ----
    const bool graph = ctx.graph_replay && join == nullptr;
    std::vector<int64_t> sig;
    bool replayed = false;
    if (graph)
    {
        sig.push_back(n0);
        for (const SceneDev& d : sd)
            for (int64_t v : { int64_t(d.B), int64_t(d.H), int64_t(d.W), int64_t(d.level), int64_t(d.partial),
                               int64_t(d.opengl), int64_t(d.mask_dtype) })
                sig.push_back(v);
        CarvePlan* plan = nullptr;
        for (size_t k = 0; k < ctx.plans.size(); ++k)
            if (ctx.plans[k]->sig == sig)
            {
                std::unique_ptr<CarvePlan> hit = std::move(ctx.plans[k]); // most recently used goes last
                ctx.plans.erase(ctx.plans.begin() + k);
                ctx.plans.push_back(std::move(hit));
                plan = ctx.plans.back().get();
                break;
            }
        if (plan != nullptr && plan->steps == last_step && plan->roots == roots)
        {
            // this batch's descriptors, read by the graph from the plan's copy
            THULL_HIP(hipMemcpyAsync(plan->scenes, scenes, size_t(n0) * sizeof(SceneDev), hipMemcpyDeviceToDevice, st));
            if (plan->exec == nullptr && !ctx.profile)
            {
                // captured on a stream of the context's own (the caller's may be the null stream, which
                // cannot capture); nothing runs while capturing, and the graph is launched on the caller's
                if (ctx.capture_stream == nullptr)
                    THULL_HIP(hipStreamCreateWithFlags(&ctx.capture_stream, hipStreamNonBlocking));
                hipStream_t cs = ctx.capture_stream;
                THULL_HIP(hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal));
                try
                {
                    record_plan(ctx, *plan, sd, n0, cs);
                }
                catch (...)
                {
                    hipGraph_t g = nullptr;
                    (void)hipStreamEndCapture(cs, &g);
                    if (g != nullptr)
                        (void)hipGraphDestroy(g);
                    throw;
                }
                THULL_HIP(hipStreamEndCapture(cs, &plan->graph));
                THULL_HIP(hipGraphInstantiate(&plan->exec, plan->graph, nullptr, nullptr, 0));
                ++ctx.graph_captures;
            }
            if (ctx.profile)
                record_plan(ctx, *plan, sd, n0, st, true);
            else
                THULL_HIP(hipGraphLaunch(plan->exec, st));
            ++plan->replays;
            const int32_t steps = plan->steps;
            unsigned long long* h = ctx.stage->p;
            THULL_HIP(hipMemcpyAsync(h, plan->status, (2 * size_t(steps) + 1) * sizeof(unsigned long long),
                                     hipMemcpyDeviceToHost, st));
            THULL_HIP(hipMemcpyAsync(h + 2 * steps + 1, plan->overflow, sizeof(uint32_t), hipMemcpyDeviceToHost, st));
            THULL_HIP(hipStreamSynchronize(st));
            const uint32_t overflow = reinterpret_cast<const uint32_t*>(h + 2 * steps + 1)[0];
            if (overflow == 0u)
            {
                replayed = true;
                ++ctx.graph_replays;
                ctx.level_lists.clear();
                ctx.level_sizes.clear();
                // the lists up to the first empty one, and the steps that had parents, as the host-driven
                // loop keeps them
                for (int32_t i = 0; i <= steps; ++i)
                {
                    ctx.level_lists.push_back(plan->lists[i]);
                    ctx.level_sizes.push_back(uint32_t(h[i]));
                    if (h[i] == 0 || i == steps)
                        break;
                    ctx.level_tests.push_back(int64_t(h[steps + 1 + i]));
                    ctx.level_children.push_back(int64_t(h[i]) * 8);
                    ctx.carve_parents.push_back(int64_t(h[i]));
                    ctx.carve_next.push_back(int64_t(h[i + 1]));
                    // 0: the persistent queue kernel (one lane per parent)
                    ctx.carve_split.push_back(plan->split[i] == 1 ? 0 : plan->split[i]);
                    if (ctx.profile)
                    {
                        float ms = 0.0f;
                        THULL_HIP(hipEventElapsedTime(&ms, ctx.event(2 * i), ctx.event(2 * i + 1)));
                        ctx.carve_ms.push_back(ms);
                    }
                }
                count = 0;
            }
            else
            {
                // a level outgrew its capacity: forget the plan, clear the leaf marks, carve host-driven
                ++ctx.graph_overflows;
                for (size_t k = 0; k < ctx.plans.size(); ++k)
                    if (ctx.plans[k].get() == plan)
                    {
                        ctx.plans.erase(ctx.plans.begin() + k);
                        break;
                    }
                launch_fill_u32(first_cells, first_cell_words, 0u, st);
                launch_mark_root_cells(scenes, 0, n0, st);
            }
        }
    }

    // ---- level loop (VH:634-751), one launch per carving step for every scene in flight ----
    std::vector<thull_scene> joined(size_t(std::max(capacity - n0, 0)));
    for (int32_t i = 0; !replayed; ++i)
    {
        if (join != nullptr && i > 0 && int32_t(all.size()) < capacity)
        {
            // scenes that join at this level boundary: their roots go after the children of the
            // scenes in flight (the list has room for one root per possible scene)
            const int32_t room = capacity - int32_t(all.size());
            const int32_t k = join(user, i, last_step, joined.data(), room);
            THULL_CHECK(k >= 0 && k <= room, "join callback returned an invalid scene count");
            if (k > 0)
            {
                const size_t k0 = all.size();
                all.insert(all.end(), joined.begin(), joined.begin() + k);
                const std::vector<uint64_t> r = add_scenes(k0, i);
                ctx.upload.upload(list + count, r.data(), r.size() * sizeof(uint64_t), st);
                count += uint32_t(r.size());
                ctx.level_sizes.back() = count;
            }
        }
        if (count == 0 || i >= last_step)
            break;
        THULL_CHECK(i < kMaxSteps, "too many carving steps");
        const int32_t room = capacity - int32_t(all.size()); // roots that may join at the next boundary
        const uint32_t nb = blocks_for(count, kCarveThreads);
        const bool compact = count <= kCompactParents;
        uint8_t* mask = pool.alloc<uint8_t>(count);
        uint32_t* bcount = pool.alloc<uint32_t>(nb);
        uint32_t* boff = pool.alloc<uint32_t>(nb);
        uint32_t* sums = pool.alloc<uint32_t>(scan_sums_room(nb));
        if (ctx.profile)
            THULL_HIP(hipEventRecord(ctx.event(2 * i), st));
        const int32_t split = launch_carve_classify(list, count, i, scenes, mask, bcount, dev_tests + i, ctx.tuning,
                                                    max_cameras(sd), carve_culls(sd.data(), sd.size(), i), st, nullptr,
                                                    0, nullptr, !compact);
        if (ctx.profile)
            THULL_HIP(hipEventRecord(ctx.event(2 * i + 1), st));
        // the scan sends the next level's size (and the camera tests) to the host; the children go out
        // before the host learns their number (8 per parent at most), so the scatter runs while the host
        // queues the next level
        const ScanNotify note = ctx.notify.next(dev_tests + i);
        if (!compact)
            exclusive_scan(LoadU32{ bcount }, nb, boff, sums, dev_total, st, note);
        uint64_t* children = pool.alloc<uint64_t>(std::max<uint64_t>(uint64_t(count) * 8 + uint64_t(room), 1));
        bool target = false; // a scene ends at step i + 1
        for (const SceneDev& d : sd)
            target |= d.start + d.level == i + 1;
        if (compact)
            launch_carve_compact(list, count, mask, children, i + 1, scenes, target, dev_total, note, st);
        else
            launch_carve_scatter(list, count, mask, boff, children, i + 1, scenes, target, st);
        unsigned long long got[2];
        if (!ctx.notify.wait(note, st, got))
        {
            THULL_HIP(hipMemcpyAsync(ctx.stage->p, dev_total, sizeof(unsigned long long), hipMemcpyDeviceToHost, st));
            THULL_HIP(
                hipMemcpyAsync(ctx.stage->p + 1, dev_tests + i, sizeof(unsigned long long), hipMemcpyDeviceToHost, st));
            THULL_HIP(hipStreamSynchronize(st));
            got[0] = ctx.stage->p[0];
            got[1] = ctx.stage->p[1];
        }
        const uint64_t next = got[0];
        check_u32(next, "octree level size");
        ctx.level_tests.push_back(int64_t(got[1]));
        ctx.level_children.push_back(int64_t(count) * 8);
        ctx.carve_parents.push_back(int64_t(count));
        ctx.carve_next.push_back(int64_t(next));
        ctx.carve_split.push_back(split);
        if (ctx.profile)
        {
            float ms = 0.0f;
            THULL_HIP(hipEventSynchronize(ctx.event(2 * i + 1)));
            THULL_HIP(hipEventElapsedTime(&ms, ctx.event(2 * i), ctx.event(2 * i + 1)));
            ctx.carve_ms.push_back(ms);
        }
        list = children;
        count = uint32_t(next);
        ctx.level_lists.push_back(list);
        ctx.level_sizes.push_back(count);
    }
    if (graph && !replayed)
        make_plan(ctx, sig, roots, last_step, st);
    const int32_t n = int32_t(all.size());
    ctx.scenes_host = sd;
    const int32_t nlists = int32_t(ctx.level_lists.size());

    // ---- corner vertices (VH:770-825): leaf cells (marked above), then their corners by dilation ----
    if (join != nullptr)
    {
        word_begin.push_back(total_words);
        const std::vector<McGrid> grids = scene_grids();
        ctx.upload.upload(dev_word_begin, word_begin.data(), (n + 1) * sizeof(uint64_t), st);
        ctx.upload.upload(dgrids, grids.data(), n * sizeof(McGrid), st);
    }
    uint32_t* bitmap = pool.alloc<uint32_t>(std::max<uint64_t>(total_words, 1));
    uint32_t* prefix = pool.alloc<uint32_t>(std::max<uint64_t>(total_words, 1));
    std::vector<BrickList> bricks; // lists of the steps at which some scene's bricks are kept
    uint64_t brick_waves = 0;
    if (by_bricks)
        for (int32_t i = 0; i < nlists; ++i)
        {
            const bool any = std::any_of(sd.begin(), sd.end(), [&](const SceneDev& d) {
                return d.start + d.level - d.brick_shift == i;
            });
            if (!any || ctx.level_sizes[i] == 0)
                continue;
            bricks.push_back(BrickList{ ctx.level_lists[i], ctx.level_sizes[i], i, brick_waves });
            brick_waves += ctx.level_sizes[i];
        }
    BrickList* brick_lists = nullptr;
    if (!bricks.empty())
    {
        brick_lists = pool.alloc<BrickList>(bricks.size());
        ctx.upload.upload(brick_lists, bricks.data(), bricks.size() * sizeof(BrickList), st);
        launch_mark_bricks(brick_lists, int32_t(bricks.size()), brick_waves, scenes, st);
    }
    if (by_bricks)
        launch_group_flags(scenes, n, most_flags, st);
    // dilation + tile popcount sums, scan of the sums, then word prefixes + vertex keys
    const uint32_t wblocks = by_bricks ? scan_blocks(total_words) : vertex_tiles(total_words);
    uint32_t* wsums = pool.alloc<uint32_t>(std::max((wblocks + 3u) & ~3u, 4u)); // scanned in groups of 4
    uint64_t* filled = by_bricks ? pool.alloc<uint64_t>(filled_words(total_words)) : nullptr;
    if (by_bricks)
        launch_dilate_groups(bitmap, total_words, dev_word_begin, scenes, n, wsums, filled, st);
    else
        launch_dilate_cells(bitmap, total_words, dev_word_begin, scenes, n, wsums, st);
    uint64_t nverts = 0;
    if (wblocks > 0)
    {
        const ScanNotify note = ctx.notify.next(nullptr);
        scan_block_sums_kernel<><<<1, 1024, 0, st>>>(wsums, wblocks, dev_total, note);
        THULL_LAUNCH_CHECK();
        unsigned long long got[2];
        nverts = ctx.notify.wait(note, st, got) ? got[0] : ctx.read_u64(dev_total, st);
    }
    check_u32(nverts, "sparse field size");
    uint64_t* vertices = pool.alloc<uint64_t>(std::max<uint64_t>(nverts, 1));
    float* values = pool.alloc<float>(std::max<uint64_t>(nverts, 1));
    if (by_bricks)
        launch_extract_groups(bitmap, total_words, filled, wsums, dev_word_begin, scenes, n, prefix, vertices, st);
    else
        launch_prefix_extract(bitmap, total_words, wsums, dev_word_begin, scenes, n, prefix, vertices, st);

    // ---- field (VH:827-888) ----
    if (by_bricks)
        launch_field_bricks(brick_lists, int32_t(bricks.size()), nverts > 0 ? brick_waves : 0, scenes, bitmap, prefix,
                            values, st);
    else
        launch_field(vertices, uint32_t(nverts), scenes, values, st);
    ctx.vertices = vertices;
    ctx.values = values;

    // ---- sparse marching cubes ----
    McPlan plan{};
    plan.grids = dgrids;
    plan.vertices = vertices;
    plan.nverts = nverts;
    plan.values = values;
    plan.value_type = kMcF32;
    plan.iso = 0.5f;
    plan.bitmap = bitmap;
    plan.prefix = prefix;

    uint64_t vtotal = 0, ttotal = 0;
    float* verts = nullptr;
    int64_t* faces = nullptr;
    std::vector<unsigned long long> starts(3 * (n + 1), 0);
    if (nverts > 0)
    {
        uint32_t* info = pool.alloc<uint32_t>(nverts);
        uint32_t* ntv = pool.alloc<uint32_t>(nverts);
        uint32_t* tbase = pool.alloc<uint32_t>(nverts);
        uint32_t* sums = pool.alloc<uint32_t>(scan_sums_room(nverts));
        uint32_t* emask = nullptr;
        uint32_t* vbase = nullptr;
        launch_mc_classify(plan, info, ntv, st);
        exclusive_scan(LoadU32{ ntv }, nverts, tbase, sums, dev_total, st);
        if (unique)
        {
            emask = pool.alloc<uint32_t>(nverts);
            vbase = pool.alloc<uint32_t>(nverts);
            launch_mc_edges(plan, info, emask, st);
            exclusive_scan(LoadPopcountMask{ emask }, nverts, vbase, sums, dev_total + 1, st);
        }
        unsigned long long* dstarts = pool.alloc<unsigned long long>(3 * (n + 1));
        uint32_t* dv = pool.alloc<uint32_t>(n + 1);
        uint32_t* dt = pool.alloc<uint32_t>(n + 1);
        // one wait for the two totals and the scene starts
        const bool notes = 3 * (n + 1) <= HostNotify::kTable;
        const ScanNotify note = notes ? ctx.notify.next(nullptr) : ScanNotify{};
        scene_starts_kernel<<<blocks_for(n + 1, 256), 256, 0, st>>>(dev_word_begin, n, total_words, prefix, nverts,
                                                                    vbase, tbase, dev_total, unique, dstarts, dv, dt,
                                                                    ctx.notify.dev_table(), note);
        THULL_LAUNCH_CHECK();
        unsigned long long got[2];
        if (notes && ctx.notify.wait(note, st, got))
        {
            std::copy(ctx.notify.table(), ctx.notify.table() + starts.size(), starts.begin());
            ttotal = got[0];
        }
        else
        {
            THULL_HIP(hipMemcpyAsync(starts.data(), dstarts, starts.size() * sizeof(unsigned long long),
                                     hipMemcpyDeviceToHost, st));
            ttotal = ctx.read_u64(dev_total, st);
        }
        vtotal = unique ? starts[3 * n + 1] : ttotal; // the entries past the last scene are the totals
        check_u32(ttotal, "triangle vertex count");
        std::vector<uint32_t> vstart(n + 1), tstart(n + 1);
        for (int32_t s = 0; s <= n; ++s)
        {
            vstart[s] = uint32_t(starts[3 * s + 1]);
            tstart[s] = uint32_t(starts[3 * s + 2]);
        }
        verts = pool.alloc<float>(3 * std::max<uint64_t>(vtotal, 1));
        faces = pool.alloc<int64_t>(std::max<uint64_t>(ttotal, 1));
        if (unique)
            launch_mc_vertices(plan, emask, vbase, verts, st);
        launch_mc_faces(plan, info, tbase, emask, vbase, dv, dt, unique, verts, faces, st);
        ctx.scene_vstart = vstart;
        ctx.scene_tstart = tstart;
    }
    else
    {
        ctx.scene_vstart.assign(n + 1, 0);
        ctx.scene_tstart.assign(n + 1, 0);
    }
    ctx.verts = verts;
    ctx.faces = faces;
    ctx.scene_first.assign(n + 1, 0);
    for (int32_t s = 0; s <= n; ++s)
        ctx.scene_first[s] = nverts > 0 ? uint32_t(starts[3 * s + 0]) : 0u;
    for (int32_t s = 0; s < n; ++s)
    {
        thull_vh_counts c{};
        c.num_verts = int64_t(ctx.scene_vstart[s + 1]) - int64_t(ctx.scene_vstart[s]);
        c.num_faces = (int64_t(ctx.scene_tstart[s + 1]) - int64_t(ctx.scene_tstart[s])) / 3;
        c.num_field = int64_t(ctx.scene_first[s + 1]) - int64_t(ctx.scene_first[s]);
        // candidate lists kept for this scene: up to its level, or up to the first empty level
        int32_t nl = 1;
        if (sd[s].level >= 0)
            nl = std::min(all[s].level + 1, nlists);
        c.num_levels = nl;
        counts[s] = c;
    }
    ctx.counts.assign(counts, counts + n);
    ctx.n_scenes = n;
    ctx.vh_valid = true;
    if (n_total != nullptr)
        *n_total = n;
}

} // namespace thull

using thull::Context;
using thull::guarded;

struct thull_ctx
{
    Context c;
};

extern "C" {

int
thull_abi_version(void)
{
    return THULL_ABI_VERSION;
}

const char*
thull_last_error(void)
{
    return thull::g_last_error.c_str();
}

int
thull_ctx_create(int device, thull_ctx** out)
{
    return guarded([&] {
        THULL_CHECK(out != nullptr, "out is null");
        int n = 0;
        THULL_HIP(hipGetDeviceCount(&n));
        THULL_CHECK(device >= 0 && device < n, "invalid device index");
        THULL_HIP(hipSetDevice(device));
        void* scr = thull::scratch_for_device(device);
        auto* ctx = new thull_ctx{};
        ctx->c.device = device;
        ctx->c.scratch = scr;
        try
        {
            ctx->c.stage = new thull::HostStage();
        }
        catch (...)
        {
            delete ctx;
            throw;
        }
        *out = ctx;
    });
}

int
thull_ctx_destroy(thull_ctx* ctx)
{
    return guarded([&] {
        if (ctx == nullptr)
            return;
        (void)hipSetDevice(ctx->c.device);
        (void)hipDeviceSynchronize();
        delete ctx->c.stage;
        delete ctx;
    });
}

int
thull_ctx_memory(thull_ctx* ctx, int64_t* peak, int64_t* reserved)
{
    return guarded([&] {
        THULL_CHECK(ctx != nullptr, "ctx is null");
        if (peak)
            *peak = int64_t(ctx->c.pool.peak());
        if (reserved)
            *reserved = int64_t(ctx->c.pool.reserved());
    });
}

int
thull_ctx_set_carve_tuning(thull_ctx* ctx, const uint32_t* max_parents)
{
    return guarded([&] {
        THULL_CHECK(ctx != nullptr && max_parents != nullptr, "ctx and max_parents must not be null");
        THULL_CHECK(max_parents[0] <= max_parents[1] && max_parents[1] <= max_parents[2] &&
                        max_parents[2] <= max_parents[3],
                    "max_parents must be non-decreasing");
        for (int k = 0; k < 4; ++k)
            ctx->c.tuning.max_parents[k] = max_parents[k];
    });
}

int
thull_ctx_get_carve_tuning(thull_ctx* ctx, uint32_t* max_parents)
{
    return guarded([&] {
        THULL_CHECK(ctx != nullptr && max_parents != nullptr, "ctx and max_parents must not be null");
        for (int k = 0; k < 4; ++k)
            max_parents[k] = ctx->c.tuning.max_parents[k];
    });
}

int
thull_ctx_set_graph_replay(thull_ctx* ctx, int32_t enabled)
{
    return guarded([&] {
        THULL_CHECK(ctx != nullptr, "ctx is null");
        ctx->c.graph_replay = enabled != 0;
    });
}

int
thull_ctx_graph_stats(thull_ctx* ctx, int64_t* captures, int64_t* replays, int64_t* overflows)
{
    return guarded([&] {
        THULL_CHECK(ctx != nullptr, "ctx is null");
        if (captures)
            *captures = ctx->c.graph_captures;
        if (replays)
            *replays = ctx->c.graph_replays;
        if (overflows)
            *overflows = ctx->c.graph_overflows;
    });
}

int
thull_ctx_trim(thull_ctx* ctx)
{
    return guarded([&] {
        THULL_CHECK(ctx != nullptr, "ctx is null");
        THULL_HIP(hipSetDevice(ctx->c.device));
        THULL_HIP(hipDeviceSynchronize());
        ctx->c.invalidate();
        ctx->c.pool.release();
        ctx->c.plans.clear();
        ctx->c.have_last = false;
    });
}

int
thull_visual_hull_run(thull_ctx* ctx,
                      const thull_scene* scenes,
                      int32_t n_scenes,
                      int32_t unique_verts,
                      void* stream,
                      thull_vh_counts* counts)
{
    return guarded([&] {
        THULL_CHECK(ctx != nullptr && scenes != nullptr && counts != nullptr, "null argument");
        thull::visual_hull_run(ctx->c, scenes, n_scenes, unique_verts != 0, static_cast<hipStream_t>(stream), counts,
                               nullptr, nullptr, 0, nullptr);
    });
}

int
thull_visual_hull_run_join(thull_ctx* ctx,
                           const thull_scene* scenes,
                           int32_t n_scenes,
                           int32_t unique_verts,
                           void* stream,
                           thull_join_fn join,
                           void* user,
                           int32_t max_scenes,
                           thull_vh_counts* counts,
                           int32_t* n_total)
{
    return guarded([&] {
        THULL_CHECK(ctx != nullptr && scenes != nullptr && counts != nullptr && n_total != nullptr && join != nullptr,
                    "null argument");
        thull::visual_hull_run(ctx->c, scenes, n_scenes, unique_verts != 0, static_cast<hipStream_t>(stream), counts,
                               join, user, max_scenes, n_total);
    });
}

int
thull_visual_hull_fetch_mesh(thull_ctx* ctx, int32_t scene, float* verts, int64_t* faces, void* stream)
{
    return guarded([&] {
        THULL_CHECK(ctx != nullptr, "ctx is null");
        Context& c = ctx->c;
        THULL_CHECK(c.vh_valid, "no visual-hull result: the last call on this context was not a visual-hull run");
        THULL_CHECK(scene >= 0 && scene < c.n_scenes, "scene index out of range");
        hipStream_t st = static_cast<hipStream_t>(stream);
        const thull_vh_counts& k = c.counts[scene];
        if (k.num_verts > 0)
            THULL_HIP(hipMemcpyAsync(verts, c.verts + 3 * uint64_t(c.scene_vstart[scene]),
                                     3 * sizeof(float) * uint64_t(k.num_verts), hipMemcpyDeviceToDevice, st));
        if (k.num_faces > 0)
            THULL_HIP(hipMemcpyAsync(faces, c.faces + uint64_t(c.scene_tstart[scene]),
                                     3 * sizeof(int64_t) * uint64_t(k.num_faces), hipMemcpyDeviceToDevice, st));
    });
}

int
thull_visual_hull_fetch_all(thull_ctx* ctx, float* verts, int64_t* faces, void* stream)
{
    return guarded([&] {
        THULL_CHECK(ctx != nullptr, "ctx is null");
        Context& c = ctx->c;
        THULL_CHECK(c.vh_valid, "no visual-hull result: the last call on this context was not a visual-hull run");
        hipStream_t st = static_cast<hipStream_t>(stream);
        uint64_t nv = 0, nf = 0;
        for (int32_t s = 0; s < c.n_scenes; ++s)
        {
            nv += uint64_t(c.counts[s].num_verts);
            nf += uint64_t(c.counts[s].num_faces);
        }
        // scenes are stored one after the other in scene order, as the caller's buffers expect
        if (nv > 0)
            THULL_HIP(hipMemcpyAsync(verts, c.verts + 3 * uint64_t(c.scene_vstart[0]), 3 * sizeof(float) * nv,
                                     hipMemcpyDeviceToDevice, st));
        if (nf > 0)
            THULL_HIP(hipMemcpyAsync(faces, c.faces + uint64_t(c.scene_tstart[0]), 3 * sizeof(int64_t) * nf,
                                     hipMemcpyDeviceToDevice, st));
    });
}

int
thull_visual_hull_fetch_field(thull_ctx* ctx, int32_t scene, int64_t* indices, float* values, void* stream)
{
    return guarded([&] {
        THULL_CHECK(ctx != nullptr, "ctx is null");
        Context& c = ctx->c;
        THULL_CHECK(c.vh_valid, "no visual-hull result: the last call on this context was not a visual-hull run");
        THULL_CHECK(scene >= 0 && scene < c.n_scenes, "scene index out of range");
        hipStream_t st = static_cast<hipStream_t>(stream);
        const uint32_t n = uint32_t(c.counts[scene].num_field);
        if (n == 0)
            return;
        const uint32_t first = c.scene_first[scene];
        thull::field_coo_kernel<<<thull::blocks_for(n, 256), 256, 0, st>>>(c.vertices + first, c.values + first, n,
                                                                          indices, values);
        THULL_LAUNCH_CHECK();
    });
}

int
thull_visual_hull_candidates_count(thull_ctx* ctx, int32_t level, int64_t* count)
{
    return guarded([&] {
        THULL_CHECK(ctx != nullptr && count != nullptr, "null argument");
        Context& c = ctx->c;
        THULL_CHECK(c.vh_valid, "no visual-hull result: the last call on this context was not a visual-hull run");
        THULL_CHECK(c.n_scenes == 1, "candidate lists are kept for single-scene runs only");
        THULL_CHECK(level >= 0 && level < c.counts[0].num_levels, "level out of range");
        *count = int64_t(c.level_sizes[level]);
    });
}

int
thull_visual_hull_fetch_candidates(thull_ctx* ctx, int32_t level, int64_t* out, void* stream)
{
    return guarded([&] {
        THULL_CHECK(ctx != nullptr, "ctx is null");
        Context& c = ctx->c;
        THULL_CHECK(c.vh_valid, "no visual-hull result: the last call on this context was not a visual-hull run");
        THULL_CHECK(c.n_scenes == 1, "candidate lists are kept for single-scene runs only");
        THULL_CHECK(level >= 0 && level < c.counts[0].num_levels, "level out of range");
        const uint32_t n = c.level_sizes[level];
        if (n == 0)
            return;
        hipStream_t st = static_cast<hipStream_t>(stream);
        thull::keys_to_ravel_kernel<<<thull::blocks_for(n, 256), 256, 0, st>>>(c.level_lists[level], n, level, out);
        THULL_LAUNCH_CHECK();
    });
}

int
thull_candidate_wireframe(thull_ctx* ctx, const int64_t* cells, int64_t n, int32_t level, const float* cube_corner_bfl,
                          float cube_length, float* verts, int64_t* edges, void* stream)
{
    return guarded([&] {
        THULL_CHECK(ctx != nullptr && cube_corner_bfl != nullptr, "null argument");
        THULL_CHECK(level >= 0 && level <= 20, "level must be in [0, 20]");
        THULL_CHECK(n >= 0 && n < (int64_t(1) << 31), "n must be in [0, 2^31)");
        THULL_HIP(hipSetDevice(ctx->c.device));
        thull::launch_wireframe(cells, uint32_t(n), level, cube_corner_bfl, cube_length, verts, edges,
                                static_cast<hipStream_t>(stream));
    });
}

int
thull_visual_hull_stats(thull_ctx* ctx, int32_t max_levels, int64_t* camera_tests, int64_t* children)
{
    return guarded([&] {
        THULL_CHECK(ctx != nullptr, "ctx is null");
        Context& c = ctx->c;
        THULL_CHECK(c.vh_valid, "no visual-hull result: the last call on this context was not a visual-hull run");
        for (int32_t i = 0; i < max_levels; ++i)
        {
            const bool have = i < int32_t(c.level_tests.size());
            if (camera_tests)
                camera_tests[i] = have ? c.level_tests[i] : 0;
            if (children)
                children[i] = have ? c.level_children[i] : 0;
        }
    });
}

int
thull_profile_enable(thull_ctx* ctx, int32_t enabled)
{
    return guarded([&] {
        THULL_CHECK(ctx != nullptr, "ctx is null");
        ctx->c.profile = enabled != 0;
    });
}

int
thull_profile_carve(thull_ctx* ctx, int32_t max_levels, float* ms, int64_t* parents, int64_t* tests, int64_t* next,
                    int32_t* split)
{
    return guarded([&] {
        THULL_CHECK(ctx != nullptr, "ctx is null");
        Context& c = ctx->c;
        THULL_CHECK(c.vh_valid, "no visual-hull result: the last call on this context was not a visual-hull run");
        for (int32_t i = 0; i < max_levels; ++i)
        {
            const bool have = i < int32_t(c.carve_parents.size());
            if (ms)
                ms[i] = (have && i < int32_t(c.carve_ms.size())) ? c.carve_ms[i] : 0.0f;
            if (parents)
                parents[i] = have ? c.carve_parents[i] : 0;
            if (tests)
                tests[i] = have ? c.level_tests[i] : 0;
            if (next)
                next[i] = have ? c.carve_next[i] : 0;
            if (split)
                split[i] = have ? c.carve_split[i] : 0;
        }
    });
}

// ---------------------------------------------------------------------------
// Marching cubes API
// ---------------------------------------------------------------------------

// Device copy of a run's one grid, followed by zero scene starts (one upload).
struct McGridUpload
{
    thull::McGrid grid;
    uint32_t zeros[2];
};

static McGridUpload*
upload_mc_grid(Context& c, const thull::McGrid& grid, hipStream_t st)
{
    McGridUpload* d = c.pool.alloc<McGridUpload>(1);
    const McGridUpload h{ grid, { 0u, 0u } };
    c.upload.upload(d, &h, sizeof(h), st);
    return d;
}

static void
mc_run_common(Context& c, thull::McPlan plan, McGridUpload* dgrid, bool unique, hipStream_t st, int64_t* nv,
              int64_t* nf)
{
    using namespace thull;
    Pool& pool = c.pool;
    plan.grids = &dgrid->grid;
    c.mc_verts = nullptr;
    c.mc_faces = nullptr;
    c.mc_nv = c.mc_nf = 0;
    *nv = *nf = 0;
    const uint64_t n = plan.nverts;
    if (n == 0)
    {
        THULL_HIP(hipStreamSynchronize(st));
        c.mc_valid = true;
        return;
    }
    check_u32(n, "marching cubes vertex count");
    unsigned long long* dev_total = pool.alloc<unsigned long long>(2);
    uint32_t* info = pool.alloc<uint32_t>(n);
    uint32_t* ntv = pool.alloc<uint32_t>(n);
    uint32_t* tbase = pool.alloc<uint32_t>(n);
    uint32_t* sums = pool.alloc<uint32_t>(scan_sums_room(n));
    uint32_t* emask = nullptr;
    uint32_t* vbase = nullptr;
    // the last scan sends the totals to the host (compact meshes: the output vertices, with the triangle
    // vertices beside them)
    ScanNotify note = c.notify.next(nullptr);
    launch_mc_classify(plan, info, ntv, st);
    exclusive_scan(LoadU32{ ntv }, n, tbase, sums, dev_total, st, unique ? ScanNotify{} : note);
    if (unique)
    {
        emask = pool.alloc<uint32_t>(n);
        vbase = pool.alloc<uint32_t>(n);
        launch_mc_edges(plan, info, emask, st);
        note.extra = dev_total;
        exclusive_scan(LoadPopcountMask{ emask }, n, vbase, sums, dev_total + 1, st, note);
    }
    unsigned long long got[2];
    if (!c.notify.wait(note, st, got))
    {
        THULL_HIP(hipMemcpyAsync(c.stage->p, dev_total, 2 * sizeof(unsigned long long), hipMemcpyDeviceToHost, st));
        THULL_HIP(hipStreamSynchronize(st));
        got[0] = c.stage->p[unique ? 1 : 0];
        got[1] = c.stage->p[0];
    }
    const uint64_t vtotal = got[0];
    const uint64_t ttotal = unique ? got[1] : got[0];
    check_u32(ttotal, "triangle vertex count");
    float* verts = pool.alloc<float>(3 * std::max<uint64_t>(vtotal, 1));
    int64_t* faces = pool.alloc<int64_t>(std::max<uint64_t>(ttotal, 1));
    if (unique)
        launch_mc_vertices(plan, emask, vbase, verts, st);
    launch_mc_faces(plan, info, tbase, emask, vbase, dgrid->zeros, dgrid->zeros, unique, verts, faces, st);
    c.mc_verts = verts;
    c.mc_faces = faces;
    c.mc_nv = int64_t(vtotal);
    c.mc_nf = int64_t(ttotal / 3);
    *nv = c.mc_nv;
    *nf = c.mc_nf;
    c.mc_valid = true;
}

static thull::McGrid
mc_grid(int64_t D, int64_t H, int64_t W, bool local)
{
    thull::McGrid g{};
    g.dims[0] = uint32_t(W);
    g.dims[1] = uint32_t(H);
    g.dims[2] = uint32_t(D);
    g.row_words = uint32_t((W + 31) / 32);
    g.bitmap_offset = 0;
    g.out_mode = local ? 1 : 0;
    // MC:523-526: 2 / (size - 1) per axis, x with W, y with H, z with D
    g.scale[0] = 2.0f / float(W - 1);
    g.scale[1] = 2.0f / float(H - 1);
    g.scale[2] = 2.0f / float(D - 1);
    g.flip = 0;
    return g;
}

int
thull_marching_cubes_dense_run(thull_ctx* ctx,
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
                               int64_t* num_faces)
{
    return guarded([&] {
        using namespace thull;
        THULL_CHECK(ctx != nullptr && num_verts != nullptr && num_faces != nullptr, "null argument");
        THULL_CHECK(dtype == kF32 || dtype == kF64, "volume must be float32 or float64 at the C ABI");
        THULL_CHECK(isolevel >= 0.0f, "isolevel must be non-negative");
        THULL_CHECK(D >= 0 && H >= 0 && W >= 0 && D < 65536 && H < 65536 && W < 65536, "volume size out of range");
        THULL_CHECK(D * H * W < (int64_t(1) << 32), "volume must have fewer than 2^32 elements");
        Context& c = ctx->c;
        hipStream_t st = static_cast<hipStream_t>(stream);
        c.begin(st);
        Pool& pool = c.pool;
        *num_verts = *num_faces = 0;
        if (D < 2 || H < 2 || W < 2)
        {
            c.mc_valid = true;
            return;
        }
        McDense d{};
        d.dims[0] = uint32_t(W);
        d.dims[1] = uint32_t(H);
        d.dims[2] = uint32_t(D);
        d.row_words = uint32_t((W + 31) / 32);
        d.nwords = uint64_t(d.row_words) * uint64_t(H) * uint64_t(D);
        d.signs = pool.alloc<uint32_t>(d.nwords);
        const int32_t value_type = dtype == kF64 ? kMcF64 : kMcF32;
        const uint32_t tiles = mc_dense_tiles(d.nwords);
        void* edges = pool.alloc_bytes(mc_dense_edge_bytes(d.nwords));
        uint32_t* counts = pool.alloc<uint32_t>(d.nwords);
        uint32_t* tile_verts = pool.alloc<uint32_t>(uint64_t(tiles) + 3); // scanned in groups of 4
        uint32_t* tile_tris = pool.alloc<uint32_t>(uint64_t(tiles) + 3);
        unsigned long long* totals = pool.alloc<unsigned long long>(2); // output vertices, triangle vertices
        launch_mc_dense_counts(d, volume, value_type, isolevel, edges, counts, tile_verts, tile_tris, st);
        const ScanNotify note = c.notify.next(nullptr);
        scan_block_sums2_kernel<><<<1, 1024, 0, st>>>(tile_verts, tile_tris, tiles, totals, note);
        THULL_LAUNCH_CHECK();
        unsigned long long got[2];
        if (!c.notify.wait(note, st, got))
        {
            THULL_HIP(hipMemcpyAsync(c.stage->p, totals, sizeof(got), hipMemcpyDeviceToHost, st));
            THULL_HIP(hipStreamSynchronize(st));
            got[0] = c.stage->p[0];
            got[1] = c.stage->p[1];
        }
        const bool unique = unique_verts != 0;
        const uint64_t ttotal = got[1], vtotal = unique ? got[0] : ttotal;
        check_u32(ttotal, "triangle vertex count");
        c.mc_verts = pool.alloc<float>(3 * std::max<uint64_t>(vtotal, 1));
        c.mc_faces = pool.alloc<int64_t>(std::max<uint64_t>(ttotal, 1));
        if (ttotal > 0)
            launch_mc_dense_mesh(d, mc_grid(D, H, W, return_local_coords != 0), volume, value_type, isolevel, counts,
                                 tile_verts, tile_tris, edges, unique, c.mc_verts, c.mc_faces, st);
        c.mc_nv = int64_t(vtotal);
        c.mc_nf = int64_t(ttotal / 3);
        *num_verts = c.mc_nv;
        *num_faces = c.mc_nf;
        c.mc_valid = true;
    });
}

int
thull_marching_cubes_sparse_run(thull_ctx* ctx,
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
                                int64_t* num_faces)
{
    return guarded([&] {
        using namespace thull;
        THULL_CHECK(ctx != nullptr && num_verts != nullptr && num_faces != nullptr, "null argument");
        THULL_CHECK(dtype == kF32 || dtype == kF64, "values must be float32 or float64 at the C ABI");
        THULL_CHECK(isolevel >= 0.0f, "isolevel must be non-negative");
        THULL_CHECK(nnz >= 0 && nnz < (int64_t(1) << 31), "nnz must be below 2^31");
        THULL_CHECK(D >= 0 && H >= 0 && W >= 0 && D < 65536 && H < 65536 && W < 65536, "volume size out of range");
        Context& c = ctx->c;
        hipStream_t st = static_cast<hipStream_t>(stream);
        c.begin(st);
        McGrid grid = mc_grid(D, H, W, return_local_coords != 0);
        const uint64_t nwords = uint64_t(D) * uint64_t(H) * grid.row_words;
        THULL_CHECK(nwords < (uint64_t(1) << 34), "sparse volume too large for the vertex bitmap");
        McGridUpload* up = upload_mc_grid(c, grid, st);
        McPlan plan{};
        plan.nverts = 0;
        if (nnz > 0 && nwords > 0)
        {
            Pool& pool = c.pool;
            const McGrid* dgrid = &up->grid;
            uint32_t* bitmap = pool.alloc<uint32_t>(nwords);
            uint32_t* prefix = pool.alloc<uint32_t>(nwords);
            unsigned long long* dev_total = pool.alloc<unsigned long long>(2); // set bits, out-of-range flag
            launch_fill_u32(reinterpret_cast<uint32_t*>(dev_total), 4, 0u, st);
            launch_fill_u32(bitmap, nwords, 0u, st);
            launch_mark_coo(indices, uint64_t(nnz), dgrid, bitmap, dev_total + 1, st);
            uint32_t* sums = pool.alloc<uint32_t>(scan_sums_room(nwords));
            // the scan sends the number of set bits (at most nnz) and the flag to the host; the vertex list
            // goes out before the host learns them
            const ScanNotify note = c.notify.next(dev_total + 1);
            exclusive_scan(LoadPopcount{ bitmap }, nwords, prefix, sums, dev_total, st, note);
            uint64_t* vertices = pool.alloc<uint64_t>(uint64_t(nnz));
            launch_extract_grid_vertices(bitmap, prefix, nwords, dgrid, vertices, st);
            unsigned long long got[2];
            if (!c.notify.wait(note, st, got))
            {
                THULL_HIP(hipMemcpyAsync(c.stage->p, dev_total, sizeof(got), hipMemcpyDeviceToHost, st));
                THULL_HIP(hipStreamSynchronize(st));
                got[0] = c.stage->p[0];
                got[1] = c.stage->p[1];
            }
            THULL_CHECK(got[1] == 0, "indices within the volume");
            THULL_CHECK(got[0] == uint64_t(nnz), "sparse volume must be coalesced (unique, in-range indices)");
            plan.vertices = vertices;
            plan.nverts = uint64_t(nnz);
            plan.bitmap = bitmap;
            plan.prefix = prefix;
        }
        plan.values = values;
        plan.value_type = dtype == kF64 ? kMcF64 : kMcF32;
        plan.iso = isolevel;
        mc_run_common(c, plan, up, unique_verts != 0, st, num_verts, num_faces);
    });
}

int
thull_marching_cubes_fetch(thull_ctx* ctx, float* verts, int64_t* faces, void* stream)
{
    return guarded([&] {
        THULL_CHECK(ctx != nullptr, "ctx is null");
        Context& c = ctx->c;
        THULL_CHECK(c.mc_valid, "no marching-cubes result: the last call on this context was not a marching-cubes run");
        hipStream_t st = static_cast<hipStream_t>(stream);
        if (c.mc_nv > 0)
            THULL_HIP(hipMemcpyAsync(verts, c.mc_verts, 3 * sizeof(float) * uint64_t(c.mc_nv), hipMemcpyDeviceToDevice,
                                     st));
        if (c.mc_nf > 0)
            THULL_HIP(hipMemcpyAsync(faces, c.mc_faces, 3 * sizeof(int64_t) * uint64_t(c.mc_nf),
                                     hipMemcpyDeviceToDevice, st));
    });
}

// ---------------------------------------------------------------------------
// Gaussian blur and integral image
// ---------------------------------------------------------------------------

// Weight of tap (i, j) as evaluated by the reference (gaussian_blur_cuda.cu:222-223):
// expf(-float(i*i + j*j) / (2 * sigma * sigma)) with float32 argument; the
// exponential is taken correctly rounded (double exp, rounded to float).
static float
gauss_weight(int i, int j, float sigma)
{
    const float num = -float(i * i + j * j);
    float den = 2.0f * sigma;
    den = den * sigma;
    const float arg = num / den;
    return float(std::exp(double(arg)));
}

// Weight table in the output type and the weight sum of the band blur (the
// reference's `normalization`, accumulated in tap order in the output
// precision, GB:217-228); for the dense blur the table is normalised by the
// float32 sum (GB:68) and the sum is unused.  Uploaded once per key.
static Context::BlurWeights
make_blur_weights(int k, float sigma, int32_t out_dtype, bool sparse)
{
    using namespace thull;
    const int h = k / 2;
    std::vector<float> w(size_t(k) * k);
    for (int i = -h; i <= h; ++i)
        for (int j = -h; j <= h; ++j)
            w[(i + h) * k + (j + h)] = gauss_weight(i, j, sigma);
    std::vector<unsigned char> table;
    double norm = 0.0;
    if (out_dtype == kF32)
    {
        std::vector<float> t(w);
        float acc = 0.0f, fsum = 0.0f;
        for (float v : w)
        {
            acc = acc + v;
            fsum = fsum + v;
        }
        if (!sparse)
            for (auto& v : t)
                v = v / fsum;
        norm = double(acc);
        table.resize(t.size() * sizeof(float));
        std::memcpy(table.data(), t.data(), table.size());
    }
    else if (out_dtype == kF64)
    {
        std::vector<double> t(w.size());
        double acc = 0.0;
        float fsum = 0.0f;
        for (float v : w)
        {
            acc = acc + double(v);
            fsum = fsum + v;
        }
        for (size_t q = 0; q < w.size(); ++q)
            t[q] = sparse ? double(w[q]) : double(w[q]) / double(fsum);
        norm = acc;
        table.resize(t.size() * sizeof(double));
        std::memcpy(table.data(), t.data(), table.size());
    }
    else
    {
        std::vector<__half> t(w.size());
        __half acc = __float2half(0.0f);
        float fsum = 0.0f;
        for (float v : w)
        {
            const __half hv = __float2half(v);
            acc = __float2half(__half2float(acc) + __half2float(hv));
            fsum = fsum + __half2float(hv);
        }
        for (size_t q = 0; q < w.size(); ++q)
        {
            const __half hw = __float2half(w[q]);
            t[q] = sparse ? hw : __float2half(__half2float(hw) / fsum);
        }
        norm = double(__half2float(acc));
        table.resize(t.size() * sizeof(__half));
        std::memcpy(table.data(), t.data(), table.size());
    }
    Context::BlurWeights bw{ nullptr, norm };
    THULL_HIP(hipMalloc(&bw.dev, table.size()));
    THULL_HIP(hipMemcpy(bw.dev, table.data(), table.size(), hipMemcpyHostToDevice));
    return bw;
}

int
thull_gaussian_blur(thull_ctx* ctx,
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
                    void* stream)
{
    return guarded([&] {
        using namespace thull;
        THULL_CHECK(ctx != nullptr, "ctx is null");
        THULL_CHECK(kernel_size > 0, "kernel_size must be positive");
        THULL_CHECK(kernel_size % 2 == 1, "kernel_size must be odd");
        THULL_CHECK(sigma > 0.0f, "sigma must be positive");
        THULL_CHECK(out_dtype == kF16 || out_dtype == kF32 || out_dtype == kF64, "dtype must be floating point");
        THULL_CHECK(B >= 0 && H >= 0 && W >= 0, "sizes must be non-negative");
        Context& c = ctx->c;
        hipStream_t st = static_cast<hipStream_t>(stream);
        c.begin(st);
        const int k = kernel_size;
        const bool is_sparse = sparse != 0;
        uint32_t sbits;
        std::memcpy(&sbits, &sigma, 4);
        const auto key = std::make_tuple(k, sbits, int(out_dtype), int(is_sparse));
        auto it = c.blur_weights.find(key);
        if (it == c.blur_weights.end())
        {
            Context::BlurWeights bw = make_blur_weights(k, sigma, out_dtype, is_sparse);
            it = c.blur_weights.emplace(key, bw).first;
        }
        if (B == 0 || H == 0 || W == 0)
            return;
        BlurImage im{ images, out, B, H, W };
        uint8_t* flags = nullptr;
        if (is_sparse && k > 1)
            flags = c.pool.alloc<uint8_t>(uint64_t(blur_tile_flag_bytes(B, H, W, k)));
        launch_gaussian_blur_batch(&im, 1, in_dtype, k, is_sparse, it->second.dev, it->second.norm, out_dtype, flags,
                                   c.pool.alloc_bytes(blur_job_bytes(1)), c.upload, st);
    });
}

int
thull_gaussian_blur_batch(thull_ctx* ctx,
                          int32_t n,
                          const void* const* images,
                          int32_t in_dtype,
                          const int64_t* sizes,
                          int32_t kernel_size,
                          float sigma,
                          int32_t sparse,
                          void* const* outs,
                          int32_t out_dtype,
                          void* stream)
{
    return guarded([&] {
        using namespace thull;
        THULL_CHECK(ctx != nullptr && images != nullptr && sizes != nullptr && outs != nullptr, "null argument");
        THULL_CHECK(n >= 0, "n must be non-negative");
        THULL_CHECK(kernel_size > 0, "kernel_size must be positive");
        THULL_CHECK(kernel_size % 2 == 1, "kernel_size must be odd");
        THULL_CHECK(sigma > 0.0f, "sigma must be positive");
        THULL_CHECK(out_dtype == kF16 || out_dtype == kF32 || out_dtype == kF64, "dtype must be floating point");
        Context& c = ctx->c;
        hipStream_t st = static_cast<hipStream_t>(stream);
        c.begin(st);
        const int k = kernel_size;
        const bool is_sparse = sparse != 0;
        uint32_t sbits;
        std::memcpy(&sbits, &sigma, 4);
        const auto key = std::make_tuple(k, sbits, int(out_dtype), int(is_sparse));
        auto it = c.blur_weights.find(key);
        if (it == c.blur_weights.end())
            it = c.blur_weights.emplace(key, make_blur_weights(k, sigma, out_dtype, is_sparse)).first;
        std::vector<BlurImage> ims(n);
        uint64_t fbytes = 0;
        for (int32_t i = 0; i < n; ++i)
        {
            const int64_t B = sizes[3 * i], H = sizes[3 * i + 1], W = sizes[3 * i + 2];
            THULL_CHECK(B >= 0 && H >= 0 && W >= 0, "sizes must be non-negative");
            ims[i] = BlurImage{ images[i], outs[i], B, H, W };
            if (is_sparse && k > 1)
                fbytes += uint64_t(blur_tile_flag_bytes(B, H, W, k));
        }
        uint8_t* flags = fbytes ? c.pool.alloc<uint8_t>(fbytes) : nullptr;
        launch_gaussian_blur_batch(ims.data(), n, in_dtype, k, is_sparse, it->second.dev, it->second.norm, out_dtype,
                                   flags, c.pool.alloc_bytes(blur_job_bytes(std::max(n, 1))), c.upload, st);
    });
}

int
thull_integral_image(thull_ctx* ctx, const void* masks, int32_t dtype, int64_t B, int64_t H, int64_t W, float* out,
                     void* stream)
{
    return guarded([&] {
        THULL_CHECK(ctx != nullptr, "ctx is null");
        THULL_CHECK(H * W < (int64_t(1) << 31), "H * W must be below 2^31");
        hipStream_t st = static_cast<hipStream_t>(stream);
        ctx->c.begin(st);
        float* carry = ctx->c.pool.alloc<float>(std::max<uint64_t>(thull::integral_carry_floats(B, H, W), 1));
        thull::launch_integral_image(masks, dtype, B, H, W, out, carry,
                                     ctx->c.pool.alloc_bytes(thull::integral_job_bytes(1)), ctx->c.upload, st);
    });
}

int
thull_integral_image_noalloc(thull_ctx* ctx, const void* masks, int32_t dtype, int64_t B, int64_t H, int64_t W,
                             float* out, void* stream)
{
    return guarded([&] {
        using namespace thull;
        THULL_CHECK(ctx != nullptr, "ctx is null");
        THULL_CHECK(ctx->c.scratch != nullptr, "context has no device scratch");
        THULL_CHECK(B >= 0 && H >= 0 && W >= 0, "sizes must be non-negative");
        THULL_CHECK(H * W < (int64_t(1) << 31), "H * W must be below 2^31");
        const uint64_t carry_bytes = integral_carry_floats(B, H, W) * sizeof(float);
        THULL_CHECK(carry_bytes <= kScratchBytes - kScratchJobBytes,
                    "integral_image_noalloc: B * (ceil(H / 32) - 1) * W floats of column carries exceed the 32 MiB "
                    "device scratch (use thull_integral_image)");
        static_assert(kScratchJobBytes >= kIntegralJobBytes, "one integral job descriptor fits the job area");
        hipStream_t st = static_cast<hipStream_t>(stream);
        THULL_HIP(hipSetDevice(ctx->c.device));
        char* base = static_cast<char*>(ctx->c.scratch);
        KernelUploader up;
        launch_integral_image(masks, dtype, B, H, W, out, reinterpret_cast<float*>(base + kScratchJobBytes), base, up,
                              st);
    });
}

int
thull_selftest_division(thull_ctx* ctx, uint64_t count, uint64_t seed, uint64_t* mismatches, void* stream)
{
    return guarded([&] {
        THULL_CHECK(ctx != nullptr && mismatches != nullptr, "ctx and mismatches must not be null");
        hipStream_t st = static_cast<hipStream_t>(stream);
        ctx->c.begin(st);
        unsigned long long* dev = ctx->c.pool.alloc<unsigned long long>(1);
        THULL_HIP(hipMemsetAsync(dev, 0, sizeof(unsigned long long), st));
        thull::launch_div2_check(count, seed, dev, st);
        *mismatches = ctx->c.read_u64(dev, st);
    });
}

} // extern "C"
