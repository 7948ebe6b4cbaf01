// The stress driver (stress.cpp, included whole) on the fake kernels with the
// path kernel (fake_paths.cpp), and the scenarios that only it can take:
//   path_frames  frames, progressive passes, restarts and new scenes on one
//                renderer, both semantics, the tree in every form, options
//                that send single passes of a frame to the wavefront
// Test infrastructure only.
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

}  // namespace

int main(int argc, char **argv) {
  const std::string scenario = argc > 1 ? argv[1] : "";
  if (scenario != "path_frames") return stress_main(argc, argv);
  fakehip::set_max_delay_us(20);
  path_frames();
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
