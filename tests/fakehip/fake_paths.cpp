// The fake kernels (fake_kernels.cpp, included whole) with the path kernel's
// launchers (paths.hpp) beside them, so that the host code takes the route it
// takes on a GPU.  A launch drains the slices of the work list that its
// workgroups own and marks the radiance slots of the chunks it took; a pass is
// complete once all its launches together have taken every chunk once.  On the
// way they check what the real kernel would touch and rely on:
//   - the camera-hit table, the work-list counters, the half-size tree, the
//     radiance slots and the job's buffers are live and large enough
//   - the counters were cleared for this launch; slices, steps between a
//     slice's chunks and requests are what the kernel's arithmetic needs
//   - the camera hits and the half-size tree were made from the scene, camera
//     and image size that the job has now
//   - Vulkan semantics: passes continue the accumulator in sample order
// Test infrastructure only.
#define launch_tonemap device_launch_tonemap  // its image is device memory only
#include "fake_kernels.cpp"
#undef launch_tonemap

#include <atomic>
#include <cstring>

#include "../../raydar_amd/csrc/paths.hpp"

namespace rdh {

namespace {

// What a camera-hit table or a half-size tree was made from.
struct Made {
  uint64_t scene = 0;  // sequence number of the tree's upload
  uint32_t width = 0, height = 0, nodes = 0;
  float view[16] = {}, proj[16] = {}, position[3] = {};
  bool operator==(const Made &o) const {
    return scene == o.scene && width == o.width && height == o.height && nodes == o.nodes &&
           !std::memcmp(view, o.view, sizeof(view)) && !std::memcmp(proj, o.proj, sizeof(proj)) &&
           !std::memcmp(position, o.position, sizeof(position));
  }
};

struct PathPass {
  uint64_t taken = 0;
  std::vector<bool> chunk;
};

std::map<const void *, Made> g_cam, g_compact;               // by table / tree
std::map<std::pair<const void *, uint64_t>, PathPass> g_pass;  // by (arena or counters, first slot)
std::once_flag g_paths_hooked;

void hook_paths() {
  hook();
  std::call_once(g_paths_hooked, [] { fakehip::on_free([](const void *base, size_t size) {
    std::lock_guard<std::mutex> g(g_k);
    const char *b = (const char *)base, *e = b + size;
    for (auto *m : {&g_cam, &g_compact})
      for (auto it = m->begin(); it != m->end();) {
        const char *p = (const char *)it->first;
        it = p >= b && p < e ? m->erase(it) : std::next(it);
      }
    for (auto it = g_pass.begin(); it != g_pass.end();) {
      const char *p = (const char *)it->first.first;
      it = p >= b && p < e ? g_pass.erase(it) : std::next(it);
    }
  }); });
}

Made made_from(const DevJob &J) {
  Made m;
  m.scene = fakehip::last_write(J.nodes4, 128ull * J.n_nodes4);
  m.width = J.width;
  m.height = J.height;
  m.nodes = J.n_nodes4;
  std::memcpy(m.view, J.inv_view, sizeof(m.view));
  std::memcpy(m.proj, J.inv_proj, sizeof(m.proj));
  std::memcpy(m.position, J.position, sizeof(m.position));
  return m;
}

bool check_path_job(const DevJob *job, const char *k) {
  if (!need(job, sizeof(DevJob), k, "job record")) return false;
  const DevJob &J = *job;
  const uint64_t e_job = fakehip::last_write(job, sizeof(DevJob));
  bool ok = true;
  if (!e_job) err(k, "job record was never uploaded"), ok = false;
  struct Buf {
    const void *p;
    uint64_t bytes;
    const char *what;
  } bufs[] = {{J.nodes4, 128ull * J.n_nodes4, "4-wide BVH nodes"},
              {J.prims, 32ull * J.n_prims, "primitives"},
              {J.objects, 64ull * J.n_prims, "objects"}};
  for (const Buf &b : bufs) {
    if (!b.bytes || !need(b.p, b.bytes, k, b.what)) {
      err(k, std::string(b.what) + ": none");
      return false;
    }
    const uint64_t e = fakehip::last_write(b.p, b.bytes);
    if (!e || e > e_job)
      err(k, std::string(b.what) + (e ? " rewritten after the job's record" : " never uploaded")), ok = false;
  }
  return need(J.acc, 16ull * J.width * J.height, k, "accumulator") && ok;
}

void add_samples(const DevJob &J, uint32_t base, uint32_t n, const char *k) {
  uint64_t &samples = g_acc[J.acc];
  if (samples != base)
    err(k, "samples from " + std::to_string(base) + " on added to an accumulator of " + std::to_string(samples));
  samples = (uint64_t)base + n;
  J.acc[0] = (float)samples;
  J.acc[1] = (float)(J.seed & 0xffff);
}

void fake_paths(const PathArgs a, bool record, int grid) {
  fakehip::count_kernel();
  std::lock_guard<std::mutex> g(g_k);
  const char *k = record ? "paths (record)" : "paths";
  if (!check_path_job(a.job, k)) return;
  const DevJob &J = *a.job;
  if (a.npix != (uint64_t)J.width * J.height) return err(k, "pixels of another job");
  if (a.refill < 1 || a.refill > 64) return err(k, "refill " + std::to_string(a.refill));
  if (J.max_bounces < 1 || J.max_bounces > 255 || a.spp < 1 || a.spp >= 1u << 24) return err(k, "pass out of range");
  const uint32_t groups = (a.npix + 63) / 64;
  if (a.chunks != groups * a.spp) return err(k, "chunks of the work list");
  if (grid < 1 || a.slices < 1 || a.slices > kPathSlices || a.request < 1 || a.step_groups != a.slices / a.spp ||
      a.step_samples != a.slices % a.spp)
    return err(k, "slices of the work list");
  if (!need(a.cursor, 4ull * kSegments * kSegStride, k, "work-list counters")) return;
  if (!need(a.cam_ray, 16ull * a.npix, k, "camera rays") || !need(a.cam_hit, 8ull * a.npix, k, "camera hits")) return;
  const Made now = made_from(J);
  if (record) {
    g_cam[a.cam_ray] = now;
  } else {
    auto it = g_cam.find(a.cam_ray);
    if (it == g_cam.end() || !(it->second == now)) err(k, "camera hits of another scene, camera or image size");
    if (a.tree == kTreeCompact) {
      if (!need(a.compact, 64ull * J.n_nodes4, k, "half-size tree")) return;
      auto ct = g_compact.find(a.compact);
      if (ct == g_compact.end() || ct->second.scene != now.scene || ct->second.nodes != now.nodes)
        err(k, "half-size tree of another scene");
    }
  }
  const uint64_t slots = (uint64_t)a.spp * a.npix;
  const bool radiance = !record && !a.vk;
  if (radiance && !need(a.L + a.l_offset, 16 * slots, k, "radiance slots")) return;
  // the chunks of the slices that this launch's workgroups own
  const std::pair<const void *, uint64_t> key{radiance ? (const void *)a.L : (const void *)a.cursor,
                                              radiance ? a.l_offset : 0};
  std::set<uint32_t> own;
  for (int b = 0; b < grid && own.size() < a.slices; ++b) own.insert((uint32_t)(b + a.first_block) % a.slices);
  auto chunks_of = [&](uint32_t s) { return (a.chunks + a.slices - 1 - s) / a.slices; };
  bool any = false;  // (a launch may find the other pipes' launches have taken it all)
  for (uint32_t s : own) any |= a.cursor[s * kSegStride] < chunks_of(s);
  if (!any) return;
  PathPass &p = g_pass[key];
  if (p.chunk.size() != a.chunks) p.chunk.assign(a.chunks, false);
  if (radiance && p.taken == 0) {
    std::vector<LRange> &ranges = g_lmap[a.L];
    for (const LRange &r : ranges)
      if (r.off < a.l_offset + slots && a.l_offset < r.off + r.len)
        err(k, "radiance slots that sample " + std::to_string(r.sample_base) + " of another pass has not accumulated");
    ranges.push_back(LRange{a.l_offset, slots, false, 0, a.sample_base});
  }
  for (uint32_t s : own) {
    const uint32_t mine = chunks_of(s);
    uint32_t &cursor = a.cursor[s * kSegStride];
    while (cursor < mine) {
      const uint32_t w = cursor;
      cursor += a.request;
      uint32_t chunk = w * a.slices + s, group = chunk / a.spp, sample = chunk - group * a.spp;
      for (uint32_t n = 0; n < a.request && w + n < mine; ++n) {
        const uint32_t c = group * a.spp + sample;
        if (c >= a.chunks || p.chunk[c]) err(k, "chunk " + std::to_string(c) + " handed out twice or beyond the list");
        else p.chunk[c] = true, ++p.taken;
        group += a.step_groups;
        sample += a.step_samples;
        if (sample >= a.spp) sample -= a.spp, ++group;
      }
    }
    cursor += a.request;  // the other waves find it empty
  }
  if (p.taken < a.chunks) return;
  g_pass.erase(key);
  if (radiance) {
    for (LRange &r : g_lmap[a.L])
      if (r.off == a.l_offset && r.len == slots) r.complete = true;
  } else if (!record) {
    if (need(J.vk_rng, 4ull * a.npix, k, "random-number states")) add_samples(J, a.sample_base, a.samples, k);
  }
}

}  // namespace

std::atomic<uint64_t> g_tree_bytes{0};  // of the last planned pass, for the scenarios
std::atomic<bool> g_tree_in_lds{false};
std::atomic<int> g_fail_tonemaps{0};  // launches of it that fail

// The real plan's choices, with lines low enough for the scenarios to cross.
void plan_paths(PathArgs *a, const DevJob &j, uint64_t lds_bvh, uint64_t lds_objects) {
  a->stack_rows = j.stack4 + 4;
  const uint64_t tree = sizeof(DevNode4) * (uint64_t)j.n_nodes4 + sizeof(DevPrim) * (uint64_t)j.n_prims;
  const uint64_t objects = sizeof(DevObject) * (uint64_t)j.n_prims;
  const bool lds = tree <= lds_bvh && tree <= 24 * 1024, leaf1 = j.max_leaf == 1;
  a->tree = lds ? (leaf1 ? kTreeLdsLeaf1 : kTreeLds)
                : !leaf1 ? kTreeMemory
                         : !a->vk && (uint64_t)a->npix * a->samples >= 1u << 18 ? kTreeCompact : kTreeLeaf1;
  g_tree_bytes = tree;
  g_tree_in_lds = lds;
  a->lds_bvh_bytes = lds ? (uint32_t)tree : 0u;
  a->lds_obj_bytes = objects <= lds_objects ? (uint32_t)objects : 0u;
}

int path_blocks_per_cu(const PathArgs &a, bool) { return a.vk ? 4 : 5; }

hipError_t launch_paths(const PathArgs &a, bool record, int grid, hipStream_t st) {
  hook_paths();
  if (grid <= 0) return hipErrorInvalidValue;
  const PathArgs args = a;
  fakehip::enqueue(st, [args, record, grid] { fake_paths(args, record, grid); });
  return hipSuccess;
}

hipError_t launch_compact(const PathArgs &a, hipStream_t st) {
  hook_paths();
  const DevJob *job = a.job;
  DevNode4C *out = a.compact;
  const uint32_t n = a.n_nodes4;
  fakehip::enqueue(st, [job, out, n] {
    fakehip::count_kernel();
    std::lock_guard<std::mutex> g(g_k);
    if (!check_path_job(job, "compact") || !need(out, 64ull * n, "compact", "half-size tree")) return;
    if (n != job->n_nodes4) err("compact", "nodes of another job");
    g_compact[out] = made_from(*job);
  });
  return hipSuccess;
}

// The mark of fake_kernels.cpp's tonemap, written to the image's ends: device
// memory, or pinned memory, which the address checks of the host build know.
static void mark_image(const DevJob *job, uint64_t npix, float samples, uchar4 *rgba, const char *k) {
  if (!need(job, sizeof(DevJob), k, "job record")) return;
  const DevJob &J = *job;
  if (npix != (uint64_t)J.width * J.height) return err(k, "pixels of another job");
  if ((uint64_t)samples != g_acc[J.acc])
    err(k, "image of " + std::to_string((uint64_t)samples) + " samples with " + std::to_string(g_acc[J.acc]) +
               " accumulated");
  rgba[npix - 1] = rgba[0] = make_uchar4((unsigned char)(uint64_t)samples, (unsigned char)J.seed,
                                         (unsigned char)(J.seed >> 8), 0xA5);
}

hipError_t launch_tonemap(const DevJob *job, uint32_t n, float spp, uchar4 *out, DevCounters *, bool, int grid,
                          hipStream_t st, bool) {
  hook_paths();
  if (grid <= 0) return hipErrorInvalidValue;
  if (g_fail_tonemaps > 0) {
    --g_fail_tonemaps;
    return hipErrorInvalidValue;
  }
  fakehip::enqueue(st, [job, n, spp, out] {
    fakehip::count_kernel();
    std::lock_guard<std::mutex> g(g_k);
    mark_image(job, n, spp, out, "tonemap");
  });
  return hipSuccess;
}

hipError_t launch_finish(const DevJob *job, const DevTicket &t, uint32_t npix, const float4 *L, float samples,
                         uchar4 *rgba, int max_grid, hipStream_t st) {
  hook_paths();
  if (max_grid <= 0) return hipErrorInvalidValue;
  const DevTicket tt = t;
  fakehip::enqueue(st, [job, tt, npix, L, samples, rgba] {
    fake_accumulate(job, tt, L);
    std::lock_guard<std::mutex> g(g_k);
    mark_image(job, npix, samples, rgba, "finish");
  });
  return hipSuccess;
}

}  // namespace rdh
