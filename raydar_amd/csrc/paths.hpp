// The path kernel (paths.hip): whole camera paths of one scene in one launch.
#pragma once

#include <hip/hip_runtime.h>

#include "layout.hpp"

namespace rdh {

constexpr int kPathBlock = 256;                // threads of a workgroup
constexpr uint32_t kPathSlices = kSegments;  // slices of a work list at most

// The tree a launch walks: DevNode4 in memory, the same with leaves of one
// primitive, DevNode4C (the same leaves), DevNode4 in LDS, with one-primitive leaves.
enum PathTree : int { kTreeMemory, kTreeLeaf1, kTreeCompact, kTreeLds, kTreeLdsLeaf1 };

struct PathArgs {
  const DevJob *job;
  QueueCtl *ctl;                // (bounds-checked builds' violation mask)
  uint32_t *cursor;             // chunks of each slice handed out, kSegStride words apart;
                                // zero at launch
  // Camera-ray hits by rank, the pixels in the order their paths start
  // (tile_order_pixel): direction and distance; hit id (kNoHit) and pixel.
  float4 *cam_ray;
  uint2 *cam_hit;
  float4 *L;                    // radiance arena
  unsigned long long l_offset;  // slot of local sample 0, pixel 0
  DevNode4C *compact;           // kTreeCompact's nodes (launch_compact makes them)
  uint32_t n_nodes4;
  uint32_t npix;
  uint32_t sample_base;         // global index of local sample 0
  uint32_t spp;                 // samples of a group of ranks in the work list, below 2^24
  uint32_t samples;             // vk: samples a lane takes of its pixel, below 2^24
  uint32_t chunks;              // work list: groups of 64 ranks * spp
  uint32_t slices;              // slices it is dealt to, at most the launch's workgroups
  uint32_t first_block;         // the launch's first workgroup among all that share the list
  uint32_t request;             // chunks a wave asks for at once
  uint32_t step_groups;         // slices / spp and slices % spp: from one chunk of a
  uint32_t step_samples;        // slice to the next
  uint32_t refill;              // idle lanes at which a wave stops to shade and refill
  uint32_t lds_bvh_bytes;       // > 0: nodes and primitives copied to LDS
  uint32_t lds_obj_bytes;       // > 0: objects copied to LDS
  uint32_t stack_rows;          // traversal stack entries per lane
  PathTree tree;
  int vk;                       // Vulkan semantics: the work list holds each group once and
                                // the launch accumulates (L is not used)
  unsigned long long l_cap;     // radiance arena entries (bounds-checked builds)
};

// Bytes of the camera-hit table per pixel.
constexpr uint64_t kCamBytes = sizeof(float4) + sizeof(uint2);

// Weak: a host build without the device kernels has none of these, and the
// engine then runs the wavefront's launchers.
//
// Fill in what depends on the scene: the stack and what a workgroup copies into
// LDS (at most lds_bvh bytes of tree and lds_objects bytes of objects).
__attribute__((weak)) void plan_paths(PathArgs *a, const DevJob &j, uint64_t lds_bvh,
                                      uint64_t lds_objects);
// Workgroups of the kernel that fit on one CU, and its launch.
__attribute__((weak)) int path_blocks_per_cu(const PathArgs &a, bool record);
__attribute__((weak)) hipError_t launch_paths(const PathArgs &a, bool record, int grid,
                                              hipStream_t st);
__attribute__((weak)) hipError_t launch_compact(const PathArgs &a, hipStream_t st);
// Adds the radiance slots of `t` to the accumulator and writes the image bytes
// of the `samples` samples it then holds, for npix pixels; npix > 0.
__attribute__((weak)) hipError_t launch_finish(const DevJob *job, const DevTicket &t, uint32_t npix,
                                               const float4 *L, float samples, uchar4 *rgba,
                                               int max_grid, hipStream_t st);
// Parity-test entry (rd_debug_arith): `n` values by the short exact forms.
__attribute__((weak)) hipError_t launch_debug_arith(int which, const float *a, const float *b, uint32_t n,
                                                    float *out, hipStream_t st);

}  // namespace rdh
