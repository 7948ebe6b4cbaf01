// The stress driver (stress.cpp, included whole) on the fake kernels with the
// path kernel (fake_paths.cpp), and the scenarios that only it can take:
//   path_frames  frames, progressive passes, restarts and new scenes on one
//                renderer, both semantics, the tree in every form, options
//                that send single passes of a frame to the wavefront
//   lds_limit    the option that bounds a tree in LDS bounds the path kernel's
//   no_image     passes whose image fails: the samples are in the accumulator
//                and count
//   new_scenes   one new scene after another, with nothing rendered between
//   no_memory    image readback while the host has no memory for its threads
//   noalloc_large  rd_render_frame_noalloc of scenes beyond the reserved upload
//                memory, by the path kernel and the wavefront: nothing is
//                allocated or freed during a call, pinned memory neither
//   path_budget  a server whose budget a job fits without the path kernel's
//                tables, with them and with room to spare
// Test infrastructure only.
#include <atomic>
#include <cstdint>
#include <cstdlib>
#include <new>

#include "../../raydar_amd/csrc/transfer.hpp"

// The allocation of this thread that fails, counted down (0: none does).
static thread_local int t_fail_new = 0;
void *operator new(size_t n) {
  if (t_fail_new > 0 && --t_fail_new == 0) throw std::bad_alloc();
  if (void *p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void *operator new(size_t n, const std::nothrow_t &) noexcept { return std::malloc(n ? n : 1); }
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

namespace rdh {
extern std::atomic<uint64_t> g_tree_bytes;  // fake_paths.cpp
extern std::atomic<bool> g_tree_in_lds;
extern std::atomic<int> g_fail_tonemaps;
}  // namespace rdh

#define main stress_main
#include "stress.cpp"
#undef main

namespace {

// `first` samples by the path kernel and the wavefront in turns, then a restart
// and the whole frame at once.
void frame(rd_renderer *r, const JobSpec &j, bool vulkan, const std::string &what) {
  rd_set_max_sample_count(r, j.spp);
  rd_set_max_bounces(r, j.bounces);
  rd_set_seed(r, j.seed);
  rd_set_option(r, "semantics", vulkan ? 1 : 0);
  Out o;
  o.rgba.assign(4ull * j.scene->s.camera.resolution_x * j.scene->s.camera.resolution_y, 0);
  if (rd_new_frame(r, &j.scene->s) != RD_OK) return fail(what + ": " + rd_last_error(r));
  int produced = 1, pass = 0;
  rd_set_samples_per_pass(r, 3);
  while (produced && pass < 4) {
    if (!vulkan) rd_set_option(r, "block", pass % 2 ? 128 : 256);
    rd_set_option(r, "lds_bvh", pass % 3 ? 0 : 14336);
    if (rd_render_sample(r, nullptr, o.rgba.data(), o.rgba.size(), &produced) != RD_OK)
      return fail(what + ": " + rd_last_error(r));
    ++pass;
  }
  rd_set_option(r, "block", 256);
  rd_set_option(r, "lds_bvh", 14336);
  if (rd_restart_frame(r) != RD_OK) return fail(what + ": restart");
  rd_set_samples_per_pass(r, j.spp);
  if (rd_render_sample(r, nullptr, o.rgba.data(), o.rgba.size(), &produced) != RD_OK || !produced)
    return fail(what + ": " + rd_last_error(r));
  o.acc.assign(o.rgba.size(), 0.0f);
  if (rd_read_accumulator(r, o.acc.data(), o.acc.size()) != RD_OK) fail(what + ": accumulator");
  check_out(j, o, what);
}

void path_frames() {
  std::vector<JobSpec> jobs;
  uint64_t seed = 500;
  for (int n : {3, 60, 300, 900})
    for (auto wh : {std::pair<uint32_t, uint32_t>{3, 5}, {97, 61}, {640, 360}, {1100, 700}})
      jobs.push_back(JobSpec{clustered(seed, n, wh.first, wh.second), 11, 12, seed}), ++seed;
  for (int pipes : {0, 1, 3}) {
    rd_config cfg{1, 12};
    rd_renderer *r = nullptr;
    if (rd_create(&cfg, &r) != RD_OK) return fail("rd_create");
    rd_set_option(r, "pipes", pipes);
    rd_set_option(r, "queue", 1 << 18);
    for (size_t i = 0; i < jobs.size(); ++i)
      frame(r, jobs[(i * 7 + pipes) % jobs.size()], i % 3 == 2, "path frame " + std::to_string(i));
    rd_destroy(r);
  }
}

void lds_limit() {
  auto sc = clustered(3, 200, 64, 48);
  rd_config cfg{1, 4};
  rd_renderer *r = nullptr;
  if (rd_create(&cfg, &r) != RD_OK) return fail("rd_create");
  std::vector<uint8_t> img(4 * 64 * 48);
  auto in_lds = [&](int64_t limit) {
    if (limit >= 0 && rd_set_option(r, "lds_bvh", limit) != RD_OK) fail("lds_bvh");
    if (rd_render_frame(r, &sc->s, img.data(), img.size()) != RD_OK) fail(rd_last_error(r));
    return rdh::g_tree_in_lds.load();
  };
  if (!in_lds(-1)) fail("by default a tree that fits is walked from LDS");
  const int64_t tree = (int64_t)rdh::g_tree_bytes.load();
  if (tree <= 14336 + 8) return fail("the tree says nothing: " + std::to_string(tree));
  for (int64_t limit : {tree, tree + 1, (int64_t)131072})
    if (!in_lds(limit)) fail("tree in memory below a limit of " + std::to_string(limit));
  for (int64_t limit : {(int64_t)0, (int64_t)14335, (int64_t)14337, tree - 1})
    if (in_lds(limit)) fail("tree in LDS above a limit of " + std::to_string(limit));
  rd_destroy(r);
}

void no_image() {
  for (uint32_t side : {60u, 700u}) {  // images below and above a megabyte
    JobSpec j{clustered(side, 80, side, side), 12, 6, 77};
    rd_config cfg{12, 6};
    rd_renderer *r = nullptr;
    if (rd_create(&cfg, &r) != RD_OK) return fail("rd_create");
    rd_set_seed(r, j.seed);
    rd_set_samples_per_pass(r, 4);
    rd_set_option(r, "kernel_timing", 1);  // (the tonemap is then a launch of its own)
    Out o;
    o.rgba.assign(4ull * side * side, 0);
    if (rd_new_frame(r, &j.scene->s) != RD_OK) return fail(rd_last_error(r));
    for (int pass = 1, produced = 0; pass <= 3; ++pass) {
      rdh::g_fail_tonemaps = pass == 2;
      const rd_status st = rd_render_sample(r, nullptr, o.rgba.data(), o.rgba.size(), &produced);
      if (st != (pass == 2 ? RD_ERR_DEVICE : RD_OK)) fail("status of pass " + std::to_string(pass));
      if (rd_sample_count(r) != 4u * pass) fail(std::to_string(rd_sample_count(r)) + " samples counted");
    }
    o.acc.assign(o.rgba.size(), 0.0f);
    if (rd_read_accumulator(r, o.acc.data(), o.acc.size()) != RD_OK) fail("accumulator");
    check_out(j, o, "frame with a pass of no image");
    rd_destroy(r);
  }
}

void new_scenes() {
  // The first image's accumulator and bytes are more than a renderer keeps for reuse, so
  // the second scene has the former freed, with its clearing perhaps still queued.
  fakehip::set_max_delay_us(3000);
  for (int k = 0; k < 12; ++k) {
    auto big = clustered(k, 20, 16384, 16384), small = clustered(k, 20, 40, 30);
    rd_config cfg{2, 6};
    rd_renderer *r = nullptr;
    if (rd_create(&cfg, &r) != RD_OK) return fail("rd_create");
    if (rd_new_frame(r, &big->s) != RD_OK) fail(rd_last_error(r));
    if (k % 2 && rd_restart_frame(r) != RD_OK) fail(rd_last_error(r));
    if (rd_new_frame(r, &small->s) != RD_OK) fail(rd_last_error(r));
    std::vector<uint8_t> img(4 * 40 * 30);
    if (k % 3 == 0 && rd_render_frame(r, &small->s, img.data(), img.size()) != RD_OK) fail(rd_last_error(r));
    rd_destroy(r);
  }
  fakehip::set_max_delay_us(20);
}

void no_memory() {
  // the callback runs just before the reading threads are made
  constexpr uint64_t bytes = 9u << 20;
  hipStream_t stream;
  unsigned char *device = nullptr;
  if (hipStreamCreate(&stream) != hipSuccess || hipMalloc((void **)&device, bytes) != hipSuccess) return fail("setup");
  std::vector<unsigned char> src(bytes), dst(bytes);
  for (uint64_t i = 0; i < bytes; ++i) src[i] = (unsigned char)(i * 2654435761u >> 13);
  if (hipMemcpy(device, src.data(), bytes, hipMemcpyHostToDevice) != hipSuccess) return fail("setup");
  {
    rdh::HostTransfer transfer;
    for (int nth : {0, 1, 2, 3, 4}) {
      std::fill(dst.begin(), dst.end(), 0);
      const rdh::HostTransfer::Read read{dst.data(), device, bytes};
      const hipError_t e = transfer.read(&read, 1, stream, 0, [&] {
        t_fail_new = nth;
        return hipSuccess;
      });
      t_fail_new = 0;
      if (e != hipSuccess || dst != src) fail("read with allocation " + std::to_string(nth) + " failing");
    }
  }
  (void)hipFree(device);
  (void)hipStreamDestroy(stream);
}

void noalloc_large() {
  rd_config cfg{1, 12};
  rd_renderer *r = nullptr;
  if (rd_create(&cfg, &r) != RD_OK) return fail("rd_create");
  for (int n : {50, 1100, 1300, 5000, 30000, 60000, 50})
    for (int block : {256, 128}) {
      JobSpec j{clustered(n, n, 200, 150), 5, 12, (uint64_t)n};
      const std::string what = "noalloc " + std::to_string(n) + " objects, block " + std::to_string(block);
      rd_set_option(r, "block", block);
      rd_set_max_sample_count(r, j.spp);
      rd_set_seed(r, j.seed);
      Out o;
      o.rgba.assign(4ull * 200 * 150, 0);
      const auto before = fakehip::stats();
      if (rd_render_frame_noalloc(r, &j.scene->s, o.rgba.data(), o.rgba.size()) != RD_OK) {
        fail(what + ": " + rd_last_error(r));
        continue;
      }
      const auto after = fakehip::stats();
      if (after.mallocs != before.mallocs || after.frees != before.frees) fail(what + ": device memory allocated");
      if (after.host_mallocs != before.host_mallocs || after.host_frees != before.host_frees)
        fail(what + ": pinned memory allocated or freed");
      check_out(j, o, what);
    }
  rd_destroy(r);
}

void path_budget() {
  rd_server *s = nullptr;
  rd_server_config any{0, 8, 0, 65536, 0};
  if (rd_server_create(&any, &s) != RD_OK) return fail("server create");
  rd_server_stats st{};
  rd_server_stats_get(s, &st);
  const uint64_t engine = st.engine_bytes;
  rd_server_destroy(s);
  std::vector<JobSpec> jobs;
  for (int i = 0; i < 6; ++i) jobs.push_back(JobSpec{clustered(40 + i, 400, 1920, 1080 + 8 * i), 20, 6, 40ull + i});
  // bytes a pixel that the budget leaves each job, and at least what the job
  // reports to hold: accumulator, image and the tables of its kernel
  const struct {
    uint64_t per_pixel, held;
  } cases[] = {{29, 28}, {60, 44}, {100, 44}, {1000, 44}};
  for (const auto &c : cases) {
    const uint64_t npix = 1920ull * (1080 + 8 * 5);
    rd_server_config cfg{engine + c.per_pixel * npix + (1 << 20), 8, 0, 65536, 0};
    const std::string what = "budget of " + std::to_string(c.per_pixel) + " bytes a pixel";
    if (rd_server_create(&cfg, &s) != RD_OK) return fail(what + ": create");
    for (int round = 0; round < 2; ++round) {  // what ran before changes nothing
      std::vector<Out> outs(jobs.size());
      std::vector<uint64_t> ids(jobs.size(), 0);
      for (size_t i = 0; i < jobs.size(); ++i) {
        rd_job_desc d = desc(jobs[i], &outs[i], true, i % 2 == 0);
        if (rd_server_submit(s, &d, &ids[i]) != RD_OK) fail(what + ": " + rd_server_last_error(s));
      }
      for (size_t i = 0; i < jobs.size(); ++i) {
        rd_job_result r{};
        if (!ids[i]) continue;
        if (rd_server_wait(s, ids[i], -1, &r) != RD_OK || !r.done || r.status != RD_OK) {
          fail(what + ": job " + std::to_string(i) + ": " + rd_server_last_error(s));
          continue;
        }
        check_out(jobs[i], outs[i], what);
        const uint64_t px = (uint64_t)jobs[i].scene->s.camera.resolution_x * jobs[i].scene->s.camera.resolution_y;
        if (r.device_bytes < c.held * px || r.device_bytes > (c.held + 1) * px)
          fail(what + ": job holds " + std::to_string(r.device_bytes) + " bytes");
      }
    }
    rd_server_stats_get(s, &st);
    if (st.engine_bytes + st.hbm_peak > cfg.hbm_budget_bytes) fail(what + ": passed");
    rd_server_destroy(s);
  }
}

}  // namespace

int main(int argc, char **argv) {
  const std::string scenario = argc > 1 ? argv[1] : "";
  if (scenario != "path_frames" && scenario != "path_budget" && scenario != "noalloc_large" &&
      scenario != "lds_limit" && scenario != "no_memory" && scenario != "no_image" && scenario != "new_scenes")
    return stress_main(argc, argv);
  fakehip::set_max_delay_us(20);
  if (scenario == "path_frames") path_frames();
  if (scenario == "path_budget") path_budget();
  if (scenario == "noalloc_large") noalloc_large();
  if (scenario == "lds_limit") lds_limit();
  if (scenario == "no_memory") no_memory();
  if (scenario == "no_image") no_image();
  if (scenario == "new_scenes") new_scenes();
  device_clean(scenario.c_str());
  const auto st = fakehip::stats();
  std::printf("%llu kernels, %llu copies, %llu mallocs\n", (unsigned long long)st.kernels,
              (unsigned long long)st.copies, (unsigned long long)st.mallocs);
  if (g_fail) {
    std::printf("stress FAILED: %d problems\n", g_fail);
    return 1;
  }
  std::printf("stress ok\n");
  return 0;
}
