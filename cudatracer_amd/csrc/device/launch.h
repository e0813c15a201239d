// Host-side launchers of the wavefront kernels (kernels.hip).
#pragma once

#include <algorithm>

#include "../../../include/cudatracer.h"
#include "dev_common.h"

namespace ctk {

// Launch geometry chosen by the runtime (and the autotuner).
struct LaunchShape {
    int block = 256;          // threads per block for extend / connect
    int lds_depth = 16;       // per-lane LDS stack entries
    int trace_blocks = 1024;  // largest persistent grid at full fill (sizes the stack spill area)
    int tail_blocks = 1024;   // k_paths' resident grid with two lanes a path (<= trace_blocks)
    int path_blocks = 1024;   // and with eight
    int grid2 = 1024, grid4 = 1024, grid8 = 1024, gridc = 1024;  // persistent grids per tree (c: compact quad)
    // Eighths of the resident blocks that the frame loop's persistent
    // traversal grids (grid2 ... gridc) fill.  Below 8 the other lane's shade
    // kernel runs beside a traversal launch instead of waiting for its waves
    // to retire.  3, 4, 5 and 6: the 259K-triangle atrium at 1080p 3.37, 3.31,
    // 3.37 and 3.41 ms, the 7.24M-triangle sphere at 4K 7.25, 6.83, 6.93 and
    // 6.87, 16 views of the small box 66.3, 63.0, 63.5 and 63.1.  The ray-level
    // launches always fill every slot (full2 ...).
    int trace_fill = 4;
    int full2 = 1024, full4 = 1024, full8 = 1024, fullc = 1024;
    int shade_blocks = 1024;  // grid-stride grid of shade
    int max_blocks = 65536;   // cap for the simple grid-stride kernels
};

// Persistent grids of the traversal kernels of each tree for ls.block and
// ls.lds_depth (resident blocks per CU x CUs); false if a kernel cannot run
// with that shape.
bool set_trace_grids(LaunchShape& ls, int num_cus);

// A chunk's header, views and segments (word counts) from its staging buffer
// to device memory, and its counters cleared.
hipError_t launch_stage(const uint32_t* stage, uint32_t view_words, uint32_t seg_words, ctd::ChunkHdr* hdr,
                        ctd::ViewDesc* views, ctd::Segment* segs, uint32_t* counters, hipStream_t s);
hipError_t launch_generate(const LaunchShape& ls, const ctd::ViewDesc* views, const ctd::Segment* segs,
                           const ctd::ChunkHdr* hdr, uint32_t max_n, const ctd::Queues& q, hipStream_t s);
// Closest hit for the n rays of r (the ray-level entry points); clears the
// counters it needs.
hipError_t launch_extend(const LaunchShape& ls, const ctd::DevScene& sc, const ctd::TraceOpts& to,
                         const ctd::Queues& q, const ctd::RayArrays& r, uint32_t n, hipStream_t s);
// The frame loop's traversal of bounce b: closest hit for the extension rays
// of bounce b and any hit for the shadow rays of bounce b - 1 in one launch
// (bounce = max_depth: the last bounce's shadow rays).  wstats (may be null)
// accumulates closest-hit node / triangle tests and any-hit node / triangle
// tests.
hipError_t launch_trace(const LaunchShape& ls, const ctd::DevScene& sc, const ctd::TraceOpts& to,
                        const ctd::Queues& q, const ctd::ChunkHdr* hdr, int sel, int bounce,
                        unsigned long long* wstats, hipStream_t s);
// The roulette tail of a chunk from bounce bounce0 on, after trace(bounce0):
// the remaining bounces of bounce0's extension queue (k_paths, two lanes a
// path) of at most n paths.
hipError_t launch_tail(const LaunchShape& ls, const ctd::DevScene& sc, const ctd::TraceOpts& to,
                       const ctd::ShadeOpts& so, const ctd::ViewDesc* views, const ctd::Segment* segs,
                       const ctd::ChunkHdr* hdr, const ctd::Queues& q, int sel, int bounce0, uint32_t n,
                       hipStream_t s);
// A chunk of n paths from the primary rays to their ends (k_paths).
hipError_t launch_paths(const LaunchShape& ls, const ctd::DevScene& sc, const ctd::TraceOpts& to,
                        const ctd::ShadeOpts& so, const ctd::ViewDesc* views, const ctd::Segment* segs,
                        const ctd::ChunkHdr* hdr, const ctd::Queues& q, uint32_t n, hipStream_t s);
hipError_t launch_shade(const LaunchShape& ls, const ctd::DevScene& sc, const ctd::ShadeOpts& so,
                        const ctd::ViewDesc* views, const ctd::Segment* segs, const ctd::ChunkHdr* hdr,
                        const ctd::Queues& q, int sel, int bounce, hipStream_t s);
hipError_t launch_resolve(const LaunchShape& ls, const ctd::ViewDesc* views, const ctd::Segment* segs,
                          const ctd::ChunkHdr* hdr, uint32_t max_tasks, const ctd::Queues& q, float4* accum,
                          uint32_t* counts, hipStream_t s);
// n bytes from device memory to `out`, the device address of pinned host memory.
hipError_t launch_copy_out(const void* src, size_t n, void* out, hipStream_t s);
hipError_t launch_tonemap(const float4* accum, uint32_t n, float samples, float4* out, hipStream_t s);
hipError_t launch_tonemap8(const float4* accum, uint32_t n, float samples, uint32_t* out, hipStream_t s);
// The fast node test's copy of a quad tree (8 float4 per node), its compact
// layout (4 uint4 per node) and the tree's plane / slot flags (*flags
// cleared first).
hipError_t launch_prepare_quad(const float4* nodes4, uint32_t n4, float4* fast, uint4* compact, uint32_t* flags,
                               hipStream_t s);
// The binary tree's plane flag (*flags cleared first).
hipError_t launch_prepare_binary(const float4* nodes2, uint32_t n2, uint32_t* flags, hipStream_t s);
// The shading records of n primitives (kPrimRows rows each) from the scene's
// arrays; uv may be null.
hipError_t launch_shading_records(const float* vert, const float* norm, const float* uv, const uint32_t* idx,
                                  const float* cn, const uint32_t* mat, uint32_t n, float4* out, hipStream_t s);
// The primitive ids of n triangle records from `first` on.
hipError_t launch_prim_ids(const float4* tris, uint32_t first, uint32_t n, uint32_t* out, hipStream_t s);
hipError_t launch_shadow_flags(const LaunchShape& ls, const ctd::DevScene& sc, const ctd::TraceOpts& to,
                               const ctd::Queues& q, const ctd::RayArrays& r, uint32_t n, hipStream_t s);

}  // namespace ctk
