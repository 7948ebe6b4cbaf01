// Host check of the box walks' slab tests over the scales a scene may have
// (built with g++ by test_box_walk.py, no GPU): the 4-wide nodes and their
// half-size form (DevNode4C) against the linear scan (the reference's
// closest-hit rule, src/renderer/cpu.rs:344-352), which every walk must match
// whatever the rays' directions: random, axis-parallel (direction components
// that are exactly zero) and nearly so.
//
// compact() and entered() restate k_compact and the half-size nodes' slab test
// of paths.hip: FP16 planes are floats rounded to 11 significant bits here.
#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

#include "../raydar_amd/csrc/bvh.hpp"
#include "../raydar_amd/csrc/pathmath.hpp"

namespace rdh {
void set_global_error(const std::string &) {}
}  // namespace rdh

using namespace rdh;

struct Half4 {
  float origin[3], unit;
  float lo[3][4], hi[3][4];
};

static float half_down(float q) {
  if (std::fabs(q) < 0x1p-14f) return q < 0.0f ? -0x1p-14f : 0.0f;
  uint32_t b = fbits(q);
  if (q > 0.0f) return bitsf(b & ~0x1fffu);
  return bitsf((b + 0x1fffu) & ~0x1fffu);
}

static Half4 compact(const DevNode4 &nd) {
  Half4 c;
  const float *lo[3] = {nd.lo_x, nd.lo_y, nd.lo_z}, *hi[3] = {nd.hi_x, nd.hi_y, nd.hi_z};
  float slack[3], reach = 0.0f;
  auto used = [&](int k) { return !is_leaf(nd.child[k]) || leaf_count(nd.child[k]) > 0; };
  for (int x = 0; x < 3; ++x) {
    float a = INFINITY, b = -INFINITY;
    for (int k = 0; k < 4; ++k)
      if (used(k)) {
        a = std::fmin(a, lo[x][k]);
        b = std::fmax(b, hi[x][k]);
      }
    c.origin[x] = bitsf(fbits(0.5f * a + 0.5f * b) & 0xffff0000u);
    slack[x] = 0x1p-21f * (std::fabs(a) + std::fabs(b));
    reach = std::fmax(reach, std::fmax(std::fabs(a - c.origin[x]), std::fabs(b - c.origin[x])) + slack[x]);
  }
  uint32_t unit = (fbits(reach) + 0x7fffffu) & 0x7f800000u;
  unit = std::min(std::max(unit, 27u << 23), 247u << 23);
  c.unit = bitsf(unit);
  const float per = bitsf((254u << 23) - unit);
  for (int x = 0; x < 3; ++x)
    for (int k = 0; k < 4; ++k) {
      c.lo[x][k] = used(k) ? half_down((lo[x][k] - c.origin[x] - slack[x]) * per) : INFINITY;
      c.hi[x][k] = used(k) ? -half_down(-((hi[x][k] - c.origin[x] + slack[x]) * per)) : -INFINITY;
    }
  return c;
}

static bool entered(const Half4 &c, int k, const SlabNF &n, float tcull) {
  const float i[3] = {n.ix, n.iy, n.iz}, ns[3] = {n.nx, n.ny, n.nz}, fs[3] = {n.fx, n.fy, n.fz};
  float tn = 0.0f, tf = tcull;
  for (int x = 0; x < 3; ++x) {
    const bool neg = i[x] < 0.0f;
    const float s = c.unit * i[x];
    const float near = std::fmaf(neg ? c.hi[x][k] : c.lo[x][k], s, std::fmaf(c.origin[x], i[x], -ns[x]));
    const float far = std::fmaf(neg ? c.lo[x][k] : c.hi[x][k], s, std::fmaf(c.origin[x], i[x], -fs[x]));
    tn = std::fmax(tn, near);
    tf = std::fmin(tf, far);
  }
  return tn <= tf;
}

static void walk(const BuiltScene &b, const std::vector<Half4> *half, const RayPre &r, float *bt, uint32_t *bid) {
  *bt = 0.0f;
  *bid = kNoHit;
  if (!walkable(r)) {
    for (const DevPrim &p : b.prims) test_prim(r, p, bt, bid);
    return;
  }
  const SlabNF n = slab_nf(slab_ray(r, ray_tolerance(r, b.r0)));
  std::vector<int32_t> stack{0};
  while (!stack.empty()) {
    const int32_t node = stack.back();
    stack.pop_back();
    const DevNode4 &nd = b.nodes4[node];
    for (int k = 0; k < 4; ++k) {
      const float tcull = cull_limit(*bt, *bid);
      float t;
      auto plane = [&](const float *lo, const float *hi, bool neg) { return neg ? hi[k] : lo[k]; };
      const bool in = half ? entered((*half)[node], k, n, tcull)
                           : slab_hit_nf(n, plane(nd.lo_x, nd.hi_x, n.ox), plane(nd.hi_x, nd.lo_x, n.ox),
                                         plane(nd.lo_y, nd.hi_y, n.oy > 32), plane(nd.hi_y, nd.lo_y, n.oy > 32),
                                         plane(nd.lo_z, nd.hi_z, n.oz > 64), plane(nd.hi_z, nd.lo_z, n.oz > 64),
                                         tcull, &t);
      if (!in) continue;
      const int32_t c = nd.child[k];
      if (!is_leaf(c)) stack.push_back(c);
      else
        for (uint32_t j = leaf_first(c), e = j + leaf_count(c); j < e; ++j) test_prim(r, b.prims[j], bt, bid);
    }
  }
}

int main() {
  std::mt19937 g(77);
  std::uniform_real_distribution<float> u(-1.f, 1.f);
  std::vector<rd_object> unit(800);
  for (size_t i = 0; i < unit.size(); ++i) {
    rd_object &o = unit[i];
    std::memset(&o, 0, sizeof(o));
    o.kind = i % 2 ? RD_CUBE : RD_SPHERE;
    for (float &v : o.center) v = 8.f * u(g);
    o.size = 0.05f + 0.4f * std::fabs(u(g));
    o.ior = 1.5f;
  }
  int wrong = 0;
  for (int power : {-40, 0, 12, 20, 24, 25, 26, 27, 28, 29, 30, 40, 56, 60, 70}) {
    const float scale = std::ldexp(1.0f, power);
    std::vector<rd_object> objs = unit;
    for (rd_object &o : objs) {
      for (float &v : o.center) v *= scale;
      o.size *= scale;
      if (power > 56) o.kind = RD_CUBE;  // (a sphere's squares overflow)
    }
    rd_scene sc;
    std::memset(&sc, 0, sizeof(sc));
    sc.camera.resolution_x = sc.camera.resolution_y = 8;
    sc.object_count = (uint32_t)objs.size();
    sc.objects = objs.data();
    BuiltScene b;
    std::string err;
    if (!build_scene(sc, 1, &b, &err)) {
      std::printf("FAIL: %s\n", err.c_str());
      return 1;
    }
    std::vector<Half4> half;
    for (const DevNode4 &nd : b.nodes4) half.push_back(compact(nd));
    int bad[2] = {0, 0}, hits = 0;
    const int rays = 3000;
    for (int k = 0; k < rays; ++k) {
      float o[3], d[3];
      for (int a = 0; a < 3; ++a) {
        o[a] = scale * 9.f * u(g);
        d[a] = u(g);
      }
      const int axis = k % 3;
      if (k % 4 == 1) d[axis] = k % 8 == 1 ? 0.f : -0.f;                 // one zero component
      if (k % 4 == 2) d[axis] = d[(axis + 1) % 3] = k % 8 == 2 ? 0.f : -0.f;  // along an axis
      if (k % 4 == 3) d[axis] = std::ldexp(u(g), -(k / 4) % 100);        // nearly zero
      const RayPre r = ray_pre(f3(o[0], o[1], o[2]), f3(d[0], d[1], d[2]));
      float t, ts = 0.f;
      uint32_t id, is = kNoHit;
      for (const DevPrim &p : b.prims) test_prim(r, p, &ts, &is);
      hits += is != kNoHit;
      // (beyond 2^62 no scene takes the half-size form: plan_paths)
      for (int form = 0; form < (b.reach <= 0x1p62f ? 2 : 1); ++form) {
        walk(b, form ? &half : nullptr, r, &t, &id);
        bad[form] += id != is || (is != kNoHit && std::memcmp(&t, &ts, 4) != 0);
      }
    }
    std::printf("scale 2^%d: %d rays, %d hits, full nodes %d wrong, half-size %d wrong\n", power, rays, hits,
                bad[0], bad[1]);
    wrong += bad[0] + bad[1];
    if (hits < rays / 10) ++wrong;  // the rays must say something
  }
  if (wrong) return 1;
  std::printf("box walks ok\n");
  return 0;
}
