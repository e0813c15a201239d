// Internal runtime of the C ABI: the context, its device buffers and the
// chunk driver shared by the plain frame loop, the batch API and the server.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <string>
#include <vector>

#include "../../../include/cudatracer.h"
#include "../device/dev_common.h"
#include "../device/launch.h"

struct ChunkStats {
    uint64_t primary = 0, extension = 0, shadow = 0, samples = 0;
    double extend_ms = 0, shade_ms = 0, connect_ms = 0, other_ms = 0, total_ms = 0, tail_ms = 0;
    uint64_t work[4] = {0, 0, 0, 0};  // closest-hit node/tri tests, shadow node/tri tests
    int extend_launches = 0;
    int chunks = 0;
};

#ifndef CT_LANES
#define CT_LANES 2
#endif
// Pipelines the chunk driver rotates through.
constexpr int kLanes = CT_LANES;
// The bounce from which a chunk's remaining bounces run in one k_paths
// launch (tail_bounce): with roulette, rr_start + CT_TAIL_AFTER_ROULETTE;
// without, max_depth - CT_TAIL_BEFORE_END (0: no tail).
#ifndef CT_TAIL_AFTER_ROULETTE
#define CT_TAIL_AFTER_ROULETTE 0
#endif
#ifndef CT_TAIL_BEFORE_END
#define CT_TAIL_BEFORE_END 0
#endif
constexpr int kTailAfterRoulette = CT_TAIL_AFTER_ROULETTE;
constexpr int kTailBeforeEnd = CT_TAIL_BEFORE_END;
static_assert(kLanes >= 2, "at least two lanes");

// One of the pipelines the chunk driver rotates through.  Each lane
// has its own queue views (a half of the context's path buffers), counters,
// chunk tables, streams, events and captured bounce loop, so the chunks of
// the two lanes run concurrently and fill each other's launch tails.
struct Lane {
    ctd::Queues q{};
    hipStream_t stream = nullptr;
    hipEvent_t resolved = nullptr;   // after this lane's latest resolve
    unsigned long long* wstats = nullptr;
    ctd::ViewDesc* d_views = nullptr;
    uint32_t d_views_cap = 0;
    ctd::Segment* d_segs = nullptr;
    uint32_t d_segs_cap = 0;
    ctd::ChunkHdr* d_hdr = nullptr;
    uint32_t* h_read = nullptr;      // pinned, written by the device: counters, error flag (Queues::err), work counters
    uint32_t* h_read_dev = nullptr;  // its device address
    uint32_t* h_stage = nullptr;     // pinned upload staging of the chunk tables, read by k_stage
    uint32_t* h_stage_dev = nullptr; // its device address
    size_t h_stage_bytes = 0;
    // captured bounce loop
    hipGraphExec_t graph_exec = nullptr;
    std::string graph_key;
    hipEvent_t ev[2 * (3 * ctd::kMaxBounce + 8)] = {};
    int n_events = 0;
    uint32_t gen = 0;  // generation of the lane's latest chunk (ChunkHdr::gen)
    // the chunk in flight (launched, not yet finished)
    bool pending = false;
    uint32_t n_paths = 0;
    int max_depth = 0;
    bool timed = false, count = false, clock = false;
    bool nee = false;  // the chunk ends with a launch for the last bounce's shadow rays
    int tail = -1;     // the chunk's k_paths bounce, or -1
};
constexpr int kHostWords = 16;  // in ct_ctx::h_flag: the words of a tree build
// h_read layout (uint32 words)
constexpr int kReadErr = ctd::kReadCounters;
constexpr int kReadWork = ctd::kReadCounters + 2;  // 4 x uint64, 8-byte aligned
constexpr int kReadWords = kReadWork + 8;

struct ct_ctx;

namespace ctr {
// Device memory, counted against the context's budget.
int dalloc(ct_ctx* c, void** p, size_t bytes, const char* what);
void dfree(ct_ctx* c, void* p);
int hip_fail(ct_ctx* c, hipError_t e, const char* what);

// Results to the caller's memory.  To memory the runtime knows (pinned by the
// caller) by its copy: 33 MB (a 1080p float image, or a 4K byte image) 0.59 ms.
// To pageable memory through pinned slots: while the caller's thread copies one
// slot to its place, the device fills the next ones.  The runtime's own copy does
// the two in turn: 33 MB 1.85 ms, the thread's memcpy 0.8-0.9 ms of it.  Textured
// 1080p frame with its float image 5.83 to 5.15 ms, 4K frame with its byte image
// 7.61 to 6.95 ms.  For one thread at a time.  Pinning takes 0.4 ms a MB, so the
// slots are small (four of 2 MB served no better) and made at the second result: a
// context's first goes by the runtime's copy, as do results of up to 1 MB in
// device memory, where there is little to overlap, and all of them where no
// slots can be had.
class ReadBack {
  public:
    // bytes of results to dst, in parts; put(dev, offset, n) enqueues on
    // stream s a kernel that writes the n bytes from `offset` on to a slot (its
    // device address).  Offsets are multiples of 512 KiB.  s is idle when it
    // returns a CT_ code.
    template <class Put>
    int run(ct_ctx* c, void* dst, size_t bytes, hipStream_t s, const char* what, Put put) {
        const hipMemoryType type = type_of(dst);
        const bool to_known = type != hipMemoryTypeUnregistered, first = !host_ && !used_;
        used_ = used_ || !to_known;
        hipError_t e;
        if (to_known || first || init() != hipSuccess) {
            // by the runtime's copy, from a buffer in device memory (kept for
            // the next known destination)
            const int r = buffer(c, bytes, what);
            if (r == CT_OK) {
                e = put(buf_, 0, bytes);
                if (e == hipSuccess) e = hipMemcpyAsync(dst, buf_, bytes, hipMemcpyDeviceToHost, s);
                const hipError_t f = hipStreamSynchronize(s);
                if (!to_known) drop(c);
                if (e == hipSuccess) e = f;
                return e == hipSuccess ? CT_OK : hip_fail(c, e, what);
            }
            if (type == hipMemoryTypeDevice || init() != hipSuccess) return r;
        }
        e = parts(dst, bytes, s, put);
        return e == hipSuccess ? CT_OK : hip_fail(c, e, what);
    }
    // device memory; queue() leaves a result that needs no slots to be waited
    // for with s, so that many small ones cost one wait (each on its own: 12 us
    // against 3)
    hipError_t queue(void* dst, const void* src, size_t bytes, hipStream_t s) {
        return through_slots(dst, bytes) ? copy_parts(dst, src, bytes, s)
                                         : hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s);
    }
    hipError_t copy(void* dst, const void* src, size_t bytes, hipStream_t s) {
        if (through_slots(dst, bytes)) return copy_parts(dst, src, bytes, s);
        const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s);
        const hipError_t f = hipStreamSynchronize(s);
        return e != hipSuccess ? e : f;
    }
    void release();

  private:
    static constexpr size_t kSlots = 4, kSlot = 512u << 10, kDirect = 1u << 20;
    hipError_t init();
    static hipMemoryType type_of(const void* p) {
        hipPointerAttribute_t a{};
        if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type;
        (void)hipGetLastError();
        return hipMemoryTypeUnregistered;
    }
    bool through_slots(const void* dst, size_t bytes) {
        if (bytes <= kDirect || type_of(dst) != hipMemoryTypeUnregistered) return false;
        const bool first = !host_ && !used_;
        used_ = true;
        return !first && init() == hipSuccess;
    }
    int buffer(ct_ctx* c, size_t bytes, const char* what) {
        if (buf_bytes_ >= bytes) return CT_OK;
        drop(c);
        const int r = dalloc(c, reinterpret_cast<void**>(&buf_), bytes, what);
        if (r == CT_OK) buf_bytes_ = bytes;
        return r;
    }
    void drop(ct_ctx* c) {
        dfree(c, buf_);
        buf_ = nullptr;
        buf_bytes_ = 0;
    }
    // through the slots, which are there
    template <class Put>
    hipError_t parts(void* dst, size_t bytes, hipStream_t s, Put put) {
        hipError_t e = hipSuccess;
        // up to 1.5 MB in one part: a further part's launch and wait cost what
        // the overlap would give (at 2 MB one part took 118 us, four 106, and
        // the runtime's copy 113)
        const size_t part = bytes <= 3 * kSlot ? 3 * kSlot : kSlot;
        const size_t n = (bytes + part - 1) / part;
        auto size = [&](size_t k) { return std::min(part, bytes - k * part); };
        for (size_t put_n = 0, k = 0; k < n && e == hipSuccess; ++k) {
            for (; put_n < n && put_n < k + kSlots && e == hipSuccess; ++put_n) {
                const size_t o = put_n % kSlots * kSlot;
                e = put(dev_ + o, put_n * part, size(put_n));
                if (e == hipSuccess) e = hipEventRecord(ev_[put_n % kSlots], s);
            }
            if (e == hipSuccess) e = hipEventSynchronize(ev_[k % kSlots]);
            if (e == hipSuccess) std::memcpy(static_cast<char*>(dst) + k * part, host_ + k % kSlots * kSlot, size(k));
        }
        const hipError_t f = hipStreamSynchronize(s);
        return e != hipSuccess ? e : f;
    }
    hipError_t copy_parts(void* dst, const void* src, size_t bytes, hipStream_t s) {
        return parts(dst, bytes, s, [&](char* dev, size_t offset, size_t n) {
            return ctk::launch_copy_out(static_cast<const char*>(src) + offset, n, dev, s);
        });
    }
    bool used_ = false;
    char *host_ = nullptr, *dev_ = nullptr, *buf_ = nullptr;
    size_t buf_bytes_ = 0;
    hipEvent_t ev_[kSlots] = {};
};
}  // namespace ctr

struct ct_ctx {
    int device = 0;
    Lane ln[kLanes];
    std::string err;
    std::string name;
    int num_cus = 0;
    uint64_t budget = 0, used = 0;
    std::vector<std::pair<void*, size_t>> allocs;

    ctk::LaunchShape shape;
    uint32_t chunk_default = 1u << 22;  // paths per chunk

    // scene
    bool has_scene = false;
    bool has_bvh2 = false, has_bvh4 = false;
    uint32_t wide_stack_bound = 0;  // worst-case stack of the wide tree (fast mode)
    ctd::DevScene sc{};
    std::vector<void*> scene_bufs;
    std::vector<ct_material> h_mats;
    std::vector<uint32_t> h_mat_idx, h_light_idx;
    std::vector<float> h_light_rows;  // 20 floats per light

    // plain frame accumulator
    int width = 0, height = 0;
    int32_t samples = 0;
    float4* accum = nullptr;
    ctr::ReadBack read;  // results on their way to the caller's arrays

    // path state: buffers of kLanes * lane_cap slots, lane k uses [k * lane_cap, (k + 1) * lane_cap)
    uint32_t lane_cap = 0;
    std::vector<void*> path_bufs;
    uint32_t spill_threads = 0;

    // error flag of the allocation-free entry point (pinned; its device
    // address), and from kHostWords on the words a tree build writes for the host
    uint32_t* h_flag = nullptr;
    uint32_t* h_flag_dev = nullptr;
    // this device's copy of the allocation-free entry point's scratch array
    // (its device address; runtime/noalloc.hip)
    void* scratch = nullptr;
};

// Return the failure of a HIP call as CT_ERR_DEVICE on context `c`.
#define HIPCHK(expr, what)                                       \
    do {                                                         \
        hipError_t e_ = (expr);                                  \
        if (e_ != hipSuccess) return ctr::hip_fail(c, e_, what); \
    } while (0)

namespace ctr {

int fail(ct_ctx* c, int code, const std::string& msg);

int validate_opts(ct_ctx* c, const ct_frame_opts& o);
// Option checks of validate_opts without touching the context's error string
// (for callers on other threads than the context's owner); *why gets the
// message of a failure.
int check_opts(const ct_ctx* c, const ct_frame_opts& o, const char** why);
// Finite position, forward and up, non-zero forward, plane distance > 0.
bool camera_ok(const ct_camera* cam);
// Device bytes of one path slot of the path-state buffers (every lane holds
// lane_cap slots): ray origin, direction and throughput (two sets), path
// words (two), hit, shadow origin, direction and colour (two sets), path
// radiance and the radiance terms (two sets each of shade's and connect's).
constexpr size_t kPathSlotBytes = 6 * 16 + 2 * 4 + 8 + 6 * 16 + 16 + 4 * 16;
// The arrays of the device-pointer entry points: float4 rays, (t, id) pairs.
inline ctd::RayArrays device_rays(const void* o, const void* d, void* hits) {
    ctd::RayArrays r{};
    r.o = static_cast<const float*>(o);
    r.d = static_cast<const float*>(d);
    r.stride = 4;
    r.hit_stride = 2;
    r.t = static_cast<float*>(hits);
    r.prim = static_cast<int*>(hits) + 1;
    return r;
}
// Zeroed pinned words the device can access, and their device address.
bool pinned_words(size_t words, uint32_t** host, uint32_t** dev);
// Path buffers for chunks of up to cap paths on each lane.
int ensure_paths(ct_ctx* c, uint32_t cap);
int ensure_tables(ct_ctx* c, Lane& L, uint32_t nviews, uint32_t nsegs);
void drop_graphs(ct_ctx* c);
// Wait for every lane's stream.
void sync_lanes(ct_ctx* c);
ctd::ViewDesc make_view(const ct_camera& cam, int width, int height, int spp, uint32_t frame_base,
                        uint64_t accum_offset);
// Stride of the pixel-strip order for n full strips (see ctd::pixel_of).
uint32_t strip_stride(uint32_t n);

// Split a list of (view, first_path, n) runs into chunks of at most cap paths
// and run them in order, alternating between the two lanes (a workload that
// fits one chunk is split in two so both lanes work on it).  Work the caller
// queued on lane 0's stream before the call is ordered before all of it; both
// lanes are idle when it returns.  Accumulator updates keep chunk order.
struct Run {
    uint32_t view, first_path, n;
};
// How run_paths runs the chunks: kRunTimed records an event pair around every
// kernel (per-stage times in ChunkStats), kRunCount counts node / triangle
// tests, kRunGraph replays each lane's captured bounce loop, kRunSerial
// runs one chunk at a time (nothing overlaps: per-kernel times are the
// kernels' own, for measurement), kRunClock measures the chunks' device time
// (ChunkStats::total_ms; kRunTimed does too).
enum RunFlags { kRunTimed = 1, kRunCount = 2, kRunGraph = 4, kRunSerial = 8, kRunClock = 16 };
int run_paths(ct_ctx* c, const std::vector<ctd::ViewDesc>& views, const std::vector<Run>& runs, uint32_t cap,
              float4* accum, const ct_frame_opts& o, int flags, ChunkStats* st);

}  // namespace ctr

namespace ctr {
// Trees and triangle records built on the device (allocated with dalloc;
// the caller owns them, also when the build fails part-way).
struct DeviceTrees {
    float4* tris = nullptr;
    ct_bvh_node* nodes2 = nullptr;
    ct_mbvh_node* nodes4 = nullptr;
    uint32_t n2 = 0, n4 = 0;
};
// Build the binary and quad trees of v's triangles on lane 0's stream; the
// result equals the host build byte for byte.  d_vert, d_idx: the view's
// vertices and indices in device memory.
int device_build(ct_ctx* c, const ct_scene_view* v, const float* d_vert, const uint32_t* d_idx, DeviceTrees* out,
                 ct_build_stats* st);
}  // namespace ctr

namespace ctr {
// Look up the device address of this device's scratch array (c->device
// current); once per device, kept for the process.
int scratch_init(ct_ctx* c);
}  // namespace ctr

// Set the launch shape (block, LDS stack depth) and size the persistent grid.
extern "C" void ctr_apply_shape(ct_ctx* c, int block, int lds_depth);
