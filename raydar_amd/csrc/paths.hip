// Whole camera paths in one persistent kernel, for one scene whose 4-wide
// tree fits the traversal stack: the per-scene renderer's passes.
//
// A lane carries one path from its camera ray's hit to its last bounce: it
// walks the tree, waits until enough lanes of its wave have finished their
// walk, scatters with them, walks again, and takes the pass's next path when
// its own ends.  Path state never leaves the registers, so a pass moves the
// scene, the camera-hit table and one radiance record per path instead of
// about 120 bytes per bounce through queues, and it is one or two launches
// whatever its bounce limit instead of three per bounce with a readback
// between every few.  Radiance goes to the same arena slots as the wavefront kernels'
// (kernels.hip) and is accumulated by the same kernel in sample order: every
// draw is keyed by (pixel, sample, bounce), so the image is the same bit for
// bit.
//
// What bounds it: the issue of instructions, one of any kind (scalar ones too)
// per SIMD and about 2.1 cycles; for a tree outside LDS the L1's rate of node
// fetches as well.  Against the wavefront it gains most in shading: a turn
// shades only lanes that hit something (a wavefront tile is a third misses),
// and no lane waits for a path's record to come back from HBM.  A quarter of
// the instructions (1.41e10 -> 1.07e10 on the first case below, scalar ones
// 3.8e9 -> 1.9e9) went with: the inner loop of the walk, which looks at one
// ballot instead of three; visit order from integer min/med/max; a stack whose
// pops need no look at the depth; one division a sphere, exact short forms of
// the roots and reciprocals (pathmath.hpp); camera misses recorded as their
// radiance.  Measured, wavefront -> paths -> with those: 97 objects at 1080p,
// 64 spp 20.0 -> 12.7 -> 10.8 ms; 4096 objects 22.4 -> 18.5 -> 16.1 ms; a
// closed room at 960x540, 16 spp 6.1 -> 4.6 -> 3.8 ms; 183 objects at 4K, 8 spp
// 15.7 -> 10.2 -> 9.6 ms; 256x256, 16 spp, whole call 0.56 -> 0.32 -> 0.29 ms;
// one sample at 1080p with a new scene 1.28 -> 1.03 -> 0.94 ms.  With the steps
// whose figures stand beside them below: 10.0, 13.4, 3.5, 6.7, 0.22 and 0.68 ms.
#include <algorithm>

#include "kernel_util.hpp"
#include "paths.hpp"

namespace rdh {

namespace {

// Waves per SIMD the path kernel is compiled for: what its registers allow.
// Six spill 30 registers around the shading (97 objects at 1080p, 64 spp 12.8
// against 10.8 ms), four are too few (11.6 ms); with Vulkan semantics, whose
// lanes also hold the stream's state and the rank, four are the faster by 2 %.
constexpr int path_waves(bool record, bool vk) { return vk && !record ? 4 : 5; }

// A pooled walk puts the primitives of the leaves it enters on a per-lane list
// in LDS and tests one of each lane's once kPoolTests lanes have one, so that a
// test runs with many lanes instead of the few that entered a leaf in this
// step.  It pays where a step waits for memory: 4096 objects at 1080p, 64 spp
// 17.3 -> 16.0 ms, 183 at 4K, 8 spp 9.6 -> 9.4 (8 or 12 lanes alike, 16 16.3 ms,
// 24 17.6); a tree in LDS loses, as the rays' culling distances shrink later:
// 97 objects 10.8 -> 11.0 ms.  The list's rows: a step adds up to four and
// writes one past what it keeps, so it starts with at most four in it.
constexpr uint32_t kPoolTests = 12, kPoolRows = 8;
template <int BLOCK>
__host__ __device__ constexpr uint32_t pool_bytes() {
  return kPoolRows * BLOCK * (uint32_t)sizeof(uint16_t);
}

// Visit keys of the walk: see the sort in k_paths.
constexpr uint32_t kNoKey = 0xffffffffu;
constexpr uint32_t kNoNode = 0xffffu;  // no 4-wide tree with 16-bit entries has this index
__device__ __forceinline__ uint32_t umin(uint32_t a, uint32_t b) { return a < b ? a : b; }
__device__ __forceinline__ uint32_t umax(uint32_t a, uint32_t b) { return a > b ? a : b; }
__device__ __forceinline__ uint32_t umed3(uint32_t a, uint32_t b, uint32_t c) {
  return umin(umax(a, b), umax(umin(a, b), c));
}

// the FP16 numbers of a word (v_fma_mix takes them as they are)
__device__ __forceinline__ float half_lo(int w) { return (float)__builtin_bit_cast(_Float16, (uint16_t)w); }
__device__ __forceinline__ float half_hi(int w) {
  return (float)__builtin_bit_cast(_Float16, (uint16_t)((uint32_t)w >> 16));
}

// A walk's ray: dot(d, d) in [kMinDot, kMaxDot] besides walkable().
constexpr float kMinDot = 0x1p-20f, kMaxDot = 0x1p20f;

// hit_sphere (cpu.rs:34-62) for a ray of a walk; NaN or negative: no hit.  The
// reference returns t1 = (-k - s) / a if that is >= 0, else t2 = (-k + s) / a if
// that is.  With a in [2^-20, 2^20] the sign of t1 is its numerator's (s is 0
// or at least 2^-75, so a negative -k - s is at most -2^-99 unless s = 0, and
// its quotient no underflow; with s = 0 both numerators are the same), so one
// division does, and that by the ray's ya = RN(1/a) (div_rn).
__device__ __forceinline__ float sphere_distance(const RayPre &r, float ya, const DevPrim &p) {
  const float dC = r.dx * p.a[0] + r.dy * p.a[1] + r.dz * p.a[2];
  const float oC = r.ox * p.a[0] + r.oy * p.a[1] + r.oz * p.a[2];
  const float k = r.od - dC;
  const float c = r.oo - 2.0f * oC + p.a[3] - p.b[0];
  const float disc = k * k - r.a * c;
  const float s = sqrt_rn_normal(disc);  // NaN for a miss
  const float n1 = -k - s;
  const float n = n1 >= 0.0f ? n1 : -k + s;
  float t = div_rn(n, r.a, ya);
  // a tiny or overflown discriminant, a tiny numerator: as written (and -0 as
  // +0, which no comparison and no hit point tells apart)
  const bool slow = (fbits(disc) < 0x0f800000u) | ((int32_t)fbits(disc) >= 0x71800000) |
                    (fabsf(n) < 0x1p-60f);
  if (slow) {
    const float s0 = sqrtf(disc);
    const float m1 = -k - s0;
    t = (m1 >= 0.0f ? m1 : -k + s0) / r.a + 0.0f;
  }
  return t;
}

// hit_cube (cpu.rs:64-98) for a ray of a walk; NaN: no hit.  The six quotients
// by div_rn with the ray's i = RN(1/d), where d and the numerators allow.
template <bool VK>
__device__ __forceinline__ float cube_from(float q0, float q1, float q2, float q3, float q4, float q5) {
  const float tmin = fmaxf(fmaxf(fminf(q0, q1), fminf(q2, q3)), fminf(q4, q5));
  const float tmax = fminf(fminf(fmaxf(q0, q1), fmaxf(q2, q3)), fmaxf(q4, q5));
  if (VK) return !(tmax >= kVkTMin) || tmin > tmax ? NAN : tmin >= kVkTMin ? tmin : tmax;
  // tmax < 0 or tmin > tmax: no hit; from inside the exit
  return fmaxf(tmin, 0.0f) > tmax ? NAN : tmin < 0.0f ? tmax : tmin;
}
template <bool VK>
__device__ __forceinline__ float cube_distance(const RayPre &r, float ix, float iy, float iz,
                                               const DevPrim &p) {
  const float n0 = p.a[0] - r.ox, n1 = p.b[0] - r.ox, n2 = p.a[1] - r.oy;
  const float n3 = p.b[1] - r.oy, n4 = p.a[2] - r.oz, n5 = p.b[2] - r.oz;
  float t = cube_from<VK>(div_rn(n0, r.dx, ix), div_rn(n1, r.dx, ix), div_rn(n2, r.dy, iy),
                          div_rn(n3, r.dy, iy), div_rn(n4, r.dz, iz), div_rn(n5, r.dz, iz));
  const float nl = fminf(fminf(fminf(fabsf(n0), fabsf(n1)), fminf(fabsf(n2), fabsf(n3))),
                         fminf(fabsf(n4), fabsf(n5)));
  const float nh = fmaxf(fmaxf(fmaxf(fabsf(n0), fabsf(n1)), fmaxf(fabsf(n2), fabsf(n3))),
                         fmaxf(fabsf(n4), fabsf(n5)));
  const float dl = fminf(fminf(fabsf(r.dx), fabsf(r.dy)), fabsf(r.dz));
  const bool slow = !((nl >= 0x1p-60f) & (nh <= 0x1p60f) & (dl >= 0x1p-20f));
  if (slow) t = cube_from<VK>(n0 / r.dx, n1 / r.dx, n2 / r.dy, n3 / r.dy, n4 / r.dz, n5 / r.dz) + 0.0f;
  return t;
}

// A walk's best hit: distance bits above the object's index.  No distance is
// NaN in a walk (a sphere's is >= 0, and some component of d is not zero) or
// -0, so unsigned order is better_hit's: the smaller distance, then the lower
// index, with misses (NaN, negative) above the +inf that stands for no hit.
constexpr uint64_t kNoBest = ((uint64_t)0x7f800000u << 32) | kNoHit;

template <bool VK>
__device__ __forceinline__ void test_in_walk(const RayPre &r, float ya, float ix, float iy, float iz,
                                             const DevPrim &p, uint64_t *best) {
  const uint32_t tag = fbits(p.b[3]);
  const bool cube = (tag & kTagCube) != 0u;
  float t = NAN;
  if (__ballot(!cube) != 0) t = sphere_distance(r, ya, p);
  if (__ballot(cube) != 0) {
    const float tc = cube_distance<VK>(r, ix, iy, iz, p);
    t = cube ? tc : t;
  }
  if (VK && !(t >= kVkTMin && t <= kVkTMax)) t = NAN;
  const uint64_t key = ((uint64_t)fbits(t) << 32) | (tag & ~kTagCube);
  if (key < *best) *best = key;
}

// The camera rays' common origin.
template <bool VK>
__device__ __forceinline__ F3 camera_origin(const DevJob &J) {
  F3 o = f3(J.position[0], J.position[1], J.position[2]), d;
  if constexpr (VK) camera_ray_vk(J, 0, 0, &o, &d);
  return o;
}

// q in [-2, 2] as FP16, rounded down or up and never subnormal.
__device__ __forceinline__ uint16_t half_toward(float q, bool up) {
  if (up) q = -q;  // round down the negative
  uint16_t b;
  if (fabsf(q) < 0x1p-14f) {
    b = q < 0.0f ? 0x8400u : 0u;
  } else {
    const _Float16 h = (_Float16)q;
    b = __builtin_bit_cast(uint16_t, h);
    if ((float)h > q) b = (uint16_t)(q < 0.0f ? b + 1u : b - 1u);
  }
  return up ? (uint16_t)(b ^ 0x8000u) : b;
}

// DevNode4 -> DevNode4C, a thread per node; a few microseconds once a frame.
__global__ __launch_bounds__(64) void k_compact(const DevJob *job, DevNode4C *out, uint32_t n) {
  const uint32_t i = blockIdx.x * 64u + threadIdx.x;
  if (i >= n) return;
  const DevNode4 nd = load_constant(&job->nodes4)[i];
  bool used[4];
  uint32_t code[4], flags = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int32_t c = nd.child[k];
    used[k] = !is_leaf(c) || leaf_count(c) > 0;
    code[k] = is_leaf(c) ? (used[k] ? leaf_first(c) : 0u) : (uint32_t)c;
    if (is_leaf(c)) flags |= k < 3 ? 0x10000u << k : 0x80000000u;
  }
  float origin[3], slack[3], reach = 0.0f;
  auto place = [&](int x, const float *lo, const float *hi) {
    float a = INFINITY, b = -INFINITY;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (used[k]) {
        a = fminf(a, lo[k]);
        b = fmaxf(b, hi[k]);
      }
    // any origin will do; this one is near the middle
    origin[x] = bitsf(fbits(0.5f * a + 0.5f * b) & 0xffff0000u);
    // for the subtractions below
    slack[x] = 0x1p-21f * (fabsf(a) + fabsf(b));
    reach = fmaxf(reach, fmaxf(fabsf(a - origin[x]), fabsf(b - origin[x])) + slack[x]);
  };
  place(0, nd.lo_x, nd.hi_x);
  place(1, nd.lo_y, nd.hi_y);
  place(2, nd.lo_z, nd.hi_z);
  // the power of two at or above it
  const uint32_t unit = min(max((fbits(reach) + 0x7fffffu) & 0x7f800000u, 27u << 23), 247u << 23);
  const float per = bitsf((254u << 23) - unit);
  DevNode4C c;
  auto planes = [&](int x, const float *lo, const float *hi, uint16_t *p) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      p[k] = used[k] ? half_toward((lo[k] - origin[x] - slack[x]) * per, false) : 0x7c00u;
      p[4 + k] = used[k] ? half_toward((hi[k] - origin[x] + slack[x]) * per, true) : 0xfc00u;
    }
  };
  planes(0, nd.lo_x, nd.hi_x, c.x);
  planes(1, nd.lo_y, nd.hi_y, c.y);
  planes(2, nd.lo_z, nd.hi_z, c.z);
#pragma unroll
  for (int x = 0; x < 3; ++x) c.head[x] = fbits(origin[x]) | code[x];
  c.head[3] = unit | code[3] | flags;
  out[i] = c;
}

// RECORD: trace every pixel's camera ray and write its hit to the table, in
// the order the paths are handed out (tile_order_pixel).
// LDS trees and the primitives are copied into LDS by every workgroup; LEAF1:
// every leaf holds one primitive.
// VK (Vulkan semantics): a pixel's samples share one stream of random numbers,
// whose place after a sample depends on that sample's draws, so a lane keeps
// its pixel for all samples of the pass, one after another, with the stream's
// state in a register, and adds each to the accumulator itself (the order
// k_accumulate would take).  The camera ray has no draw in it here either.
// 97 objects, 1280x720, 16 spp: 8.1 -> 3.5 ms, which were 16 passes of one
// sample with 12 bounces of three launches each; 2.8 ms with the shorter walk.
template <int BLOCK, bool RECORD, PathTree TREE, bool VK>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(path_waves(RECORD, VK), 8)))
void k_paths(PathArgs a) {
  typedef uint16_t StackT;
  constexpr bool LDS = TREE == kTreeLds || TREE == kTreeLdsLeaf1;
  constexpr bool LEAF1 = TREE != kTreeMemory && TREE != kTreeLds;
  constexpr bool kCompact = TREE == kTreeCompact, kPooled = LEAF1 && !LDS;
  extern __shared__ __align__(16) unsigned char dynamic_lds[];
  // Job fields are scalar loads.  What a walk needs stays in registers; the
  // shading's fields are read again in every turn: held across the walk, they
  // overflowed into vector registers and those into scratch, whose traffic
  // shares the L1 with the node fetches (4096 objects at 1080p, 64 spp 20.7 ->
  // 18.5 ms; 183 objects at 4K, 8 spp 10.7 -> 9.9 ms; 97 objects in LDS -1%).
  const DevNode4 *nodes4 = load_constant(&a.job->nodes4);
  const DevPrim *prims = load_constant(&a.job->prims);
  const uint32_t n_nodes4 = load_constant(&a.job->n_nodes4), n_prims = load_constant(&a.job->n_prims);
  (void)n_nodes4;
  (void)nodes4;
  const uint32_t stack_bytes = (a.stack_rows * BLOCK * (uint32_t)sizeof(StackT) + 15u) & ~15u;
  // The lane's stack column: rows of kRow bytes, the last holding kNoNode for
  // good, so that a pop needs no look at the depth.
  constexpr uint32_t kRow = BLOCK * (uint32_t)sizeof(StackT);
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)dynamic_lds;
  const uint32_t stack_first = lds_base + (a.stack_rows - 2u) * kRow + threadIdx.x * (uint32_t)sizeof(StackT);
  typedef __attribute__((address_space(3))) StackT LdsStackT;
  auto stack_at = [](uint32_t off) -> LdsStackT & { return *(LdsStackT *)off; };
  stack_at(stack_first + kRow) = (StackT)kNoNode;
  // a pooled walk's primitives entered but not yet tested: kPoolRows rows
  const uint32_t pool_first = lds_base + stack_bytes + threadIdx.x * (uint32_t)sizeof(StackT);
  VecF4 *lds_nodes = reinterpret_cast<VecF4 *>(dynamic_lds + stack_bytes + (kPooled ? pool_bytes<BLOCK>() : 0u));
  const uint32_t node_vecs = LDS ? 8 * n_nodes4 : 0u, prim_vecs = LDS ? 2 * n_prims : 0u;
  VecF4 *lds_prims = lds_nodes + node_vecs;
  VecF4 *lds_objects = lds_prims + prim_vecs;
  const bool lds_obj = !RECORD && a.lds_obj_bytes != 0;
  if (LDS) {
    GlobalF4 *gn = (GlobalF4 *)nodes4, *gp = (GlobalF4 *)prims;
    for (uint32_t i = threadIdx.x; i < node_vecs; i += BLOCK) {
      VecF4 v = gn[i];
      if (LEAF1 && (i & 7u) == 6u) {
        // the children's codes: a one-primitive leaf's becomes its primitive's
        // index, with bit 16 + k for child k; an empty slot's is never entered
        VecI4 c = __builtin_bit_cast(VecI4, v);
        for (int k = 0; k < 4; ++k)
          if (is_leaf(c[k])) c[k] = (int32_t)(0x80000000u | 0x10000u << k | (leaf_first(c[k]) & 0xffffu));
        v = __builtin_bit_cast(VecF4, c);
      }
      lds_nodes[i] = v;
    }
    for (uint32_t i = threadIdx.x; i < prim_vecs; i += BLOCK) lds_prims[i] = gp[i];
  }
  if (lds_obj) {
    GlobalF4 *go = (GlobalF4 *)load_constant(&a.job->objects);
    for (uint32_t i = threadIdx.x; i < a.lds_obj_bytes / 16u; i += BLOCK) lds_objects[i] = go[i];
  }
  __syncthreads();

  const uint32_t lane = lane_id();
  // The work list: chunks of 64 ranks at one sample (the last group of ranks
  // may be smaller), the samples of a group one after another, dealt round-
  // robin to a.slices slices.  Each slice has a counter on a cache line of its
  // own, and a wave takes chunks from its workgroup's slice only: a counter
  // serves about 90 requests per microsecond whoever asks, 32 of them 2100,
  // and a dealt slice is a fair sample of the image, so the slices end
  // together.  (Waves that went on to other slices when theirs was used up
  // spent 0.3 ms of a 1080p recording asking around.)
  const uint32_t slice = (blockIdx.x + a.first_block) % a.slices;
  const uint32_t slice_chunks = (a.chunks + a.slices - 1u - slice) / a.slices;
  const float cull0 = VK ? cull_limit(kVkTMax, 0u) : INFINITY;  // with no hit yet
  // A lane is free (!has), or its path walks (nodes to visit: node != kNoNode;
  // with a pool, primitives to test: pool != pool_first), or waits to be shaded.
  bool has = false;
  uint32_t pool = pool_first;  // byte offset of the pool's next free entry
  // The wave's chunk (group, sample, paths handed out) and the chunks of its
  // last request still to come: wave-uniform.
  uint32_t group = 0, sample = 0, off = 64, left = 0;
  bool more = true;                // wave-uniform: the list may hold more
  // A turn hands out work until fewer than `few` lanes are free: at most
  // `refill`, so that the lanes left free never start a turn by themselves
  // (every turn shades a lane, hands out work or finds the list empty).
  const uint32_t few = a.refill < 16u ? a.refill : 16u;
  F3 o = f3(0.0f, 0.0f, 0.0f), d = o;
  F3 at = f3(1.0f, 1.0f, 1.0f), li = f3(0.0f, 0.0f, 0.0f);
  uint32_t pixel = 0, sb = 0;      // sample in the pass << 8 | bounce (RECORD: the rank)
  uint32_t vk_rank = 0, vk_state = 0;  // VK: the pixel's rank and random-number state
  uint64_t best = kNoBest;         // the walk's or the waiting path's hit
  float tcull = INFINITY;
  uint32_t node = kNoNode;
  uint32_t sp = 0;          // byte offset two rows past the next stack entry to write
  RayPre r;
  SlabNF nf;
  bool neg_x = false, neg_y = false, neg_z = false;  // (a compact tree's)
  float ya = 0.0f;  // RN(1 / dot(d, d))

  // The lane's path ends with radiance c.  VK: the pixel's next sample, if the
  // pass has one, waits at the camera ray's hit.
  auto finish = [&](const DevJob &J, F3 c) {
    if constexpr (VK) {
      float4 *acc = reinterpret_cast<float4 *>(J.acc) + pixel;
      const float4 v = *acc;
      *acc = make_float4(v.x + c.x, v.y + c.y, v.z + c.z, v.w + 1.0f);
      if ((sb >> 8) + 1u < a.samples) {
        const float4 cr = a.cam_ray[vk_rank];
        o = camera_origin<VK>(J);
        d = f3(cr.x, cr.y, cr.z);
        best = ((uint64_t)fbits(cr.w) << 32) | a.cam_hit[vk_rank].x;
        at = f3(1.0f, 1.0f, 1.0f);
        li = f3(0.0f, 0.0f, 0.0f);
        sb = ((sb >> 8) + 1u) << 8;
      } else {
        J.vk_rng[pixel] = vk_state;
        has = false;
      }
    } else {
      const unsigned long long slot =
          a.l_offset + (unsigned long long)(sb >> 8) * a.npix + pixel;
      a.L[chk(slot, a.l_cap, K_RADIANCE, a.ctl)] = make_float4(c.x, c.y, c.z, 1.0f);
      has = false;
    }
  };
  auto walking = [&]() { return kPooled ? node != kNoNode || pool != pool_first : node != kNoNode; };
  auto hit_id = [&]() { return (uint32_t)best; };
  auto hit_t = [&]() { return bitsf((uint32_t)(best >> 32)); };
  // the walk's culling distance (VK: hits beyond t_max do not count)
  auto cull = [&]() {
    const float c = hit_t() * 1.0001f + 1e-30f;
    return VK ? fminf(c, cull0) : c;
  };
  auto test = [&](uint32_t j) {
#ifdef RDH_CHECKED
    j = chk(j, n_prims, K_PRIM, a.ctl);
#endif
    DevPrim pr;
    if (LDS) {
      const VecF4 pa = lds_prims[2 * j], pb = lds_prims[2 * j + 1];
      pr.a[0] = pa.x; pr.a[1] = pa.y; pr.a[2] = pa.z; pr.a[3] = pa.w;
      pr.b[0] = pb.x; pr.b[1] = pb.y; pr.b[2] = pb.z; pr.b[3] = pb.w;
    } else {
      load_prim(prims, j, &pr);
    }
    test_in_walk<VK>(r, ya, nf.ix, nf.iy, nf.iz, pr, &best);
  };
  // off, a row further if key's sign bit is set: a shift and a shift-add (as
  // one expression the compiler makes it three instructions; with stack
  // addresses kept absolute and one comparison less a step 97 objects at 1080p,
  // 64 spp 10.30 -> 10.07 ms, 4096 objects 14.05 -> 13.37)
  auto row_if = [](uint32_t key, uint32_t off) {
    uint32_t bit = key >> 31;
    asm("" : "+v"(bit));
    off += bit * kRow;
    asm("" : "+v"(off));
    return off;
  };
  // the primitive of a one-primitive leaf (in LDS and compact trees the code's
  // lower half)
  auto leaf_prim = [&](int32_t code) { return (uint16_t)(LDS || kCompact ? code : code >> 4); };

  for (;;) {
    // ---- a turn: shade the lanes whose walk has ended, refill the free ones
    const DevJob J = load_constant(a.job);
    bool full = has && !walking(), fresh = false;
    if constexpr (RECORD) {
      if (full) {
        const bool hit = hit_id() != kNoHit;
        // a pixel whose camera ray leaves the scene: its samples' radiance
        const F3 c = add(f3(0.0f, 0.0f, 0.0f), mul(VK ? world_sample_vk(J, d) : world_sample(J, d),
                                                   f3(1.0f, 1.0f, 1.0f)));
        a.cam_ray[sb] = hit ? make_float4(d.x, d.y, d.z, hit_t()) : make_float4(c.x, c.y, c.z, 0.0f);
        a.cam_hit[sb] = make_uint2(hit_id(), pixel);
        has = full = false;
      }
    } else {
      if (full && hit_id() == kNoHit) {
        // cpu.rs:334-337 (raytrace.rgen:178)
        finish(J, add(li, mul(VK ? world_sample_vk(J, d) : world_sample(J, d), at)));
        full = has;
      }
    }
    // Free lanes take the next paths.  A camera path starts at its pixel's
    // recorded hit, so it is shaded in this turn with the lanes that finished
    // a walk; one that left the scene ends at once, and its lane asks again.
    while (more) {
      const uint64_t need = __ballot(!has);
      if ((uint32_t)__popcll(need) < few) break;
      const uint32_t in_group = a.npix - group * 64u;
      const uint32_t size = in_group < 64u ? in_group : 64u;
      if (off >= size) {
        // the next chunk of the request, or a new request
        off = 0;
        if (left > 0) {
          --left;
          group += a.step_groups;
          sample += a.step_samples;
          if (sample >= a.spp) {
            sample -= a.spp;
            ++group;
          }
        } else {
          uint32_t w = 0;
          if (lane == 0) w = atomicAdd(&a.cursor[slice * kSegStride], a.request);
          w = __builtin_amdgcn_readfirstlane(w);
          if (w >= slice_chunks) {
            more = false;
            break;
          }
          left = (slice_chunks - w < a.request ? slice_chunks - w : a.request) - 1u;
          const uint32_t chunk = w * a.slices + slice;
          group = __builtin_amdgcn_readfirstlane(chunk / a.spp);
          sample = chunk - group * a.spp;
        }
        continue;
      }
      const uint32_t k = off + lanes_below(need);
      if (!has && k < size) {
        const uint32_t rank = chk(group * 64u + k, a.npix, K_RADIANCE, a.ctl);
        has = true;
        if constexpr (RECORD) {
          pixel = tile_order_pixel(rank, J.width, J.height);
          if constexpr (VK) camera_ray_vk(J, pixel % J.width, pixel / J.width, &o, &d);
          else camera_ray(J, pixel % J.width, pixel / J.width, &o, &d);
          sb = rank;
          fresh = true;
        } else {
          const float4 cr = a.cam_ray[rank];
          const uint2 ch = a.cam_hit[rank];
          pixel = ch.y;
          sb = sample << 8;
          if constexpr (VK) {
            vk_rank = rank;
            vk_state = a.sample_base == 0 ? pixel % J.width + (pixel / J.width) * 1000u : J.vk_rng[pixel];
          }
          if (ch.x != kNoHit) {
            o = camera_origin<VK>(J);
            d = f3(cr.x, cr.y, cr.z);
            best = ((uint64_t)fbits(cr.w) << 32) | ch.x;
            // a camera path's attenuation and light (cpu.rs:253-254)
            at = f3(1.0f, 1.0f, 1.0f);
            li = f3(0.0f, 0.0f, 0.0f);
            full = true;
          } else if constexpr (VK) {
            // every sample of the pixel is this one and draws nothing
            float4 *acc = reinterpret_cast<float4 *>(J.acc) + pixel;
            float4 v = *acc;
            for (uint32_t i = 0; i < a.samples; ++i)
              v = make_float4(v.x + cr.x, v.y + cr.y, v.z + cr.z, v.w + 1.0f);
            *acc = v;
            J.vk_rng[pixel] = vk_state;
            has = false;
          } else {
            finish(J, f3(cr.x, cr.y, cr.z));
          }
        }
      }
      off += (uint32_t)__popcll(need);
    }
    if constexpr (!RECORD) {
      if (full) {
        const uint32_t oid = chk(hit_id(), J.n_prims, K_OBJECT, a.ctl);
        const DevObject ob = lds_obj ? object_from(lds_objects[4 * oid], lds_objects[4 * oid + 1],
                                                   lds_objects[4 * oid + 2], lds_objects[4 * oid + 3])
                                     : load_object(J.objects, oid);
        const HitRec h = closest_hit(o, d, hit_t(), ob);
        ScatterOut so;
        if constexpr (VK) {
          so = scatter_vk(d, h, ob, vk_state, at, li);
        } else {
          BounceDraws dr;
          dr.init(J.seed, pixel, a.sample_base + (sb >> 8), sb & 0xffu);
          so = scatter(d, h, ob, dr, at, li);
        }
        li = so.light;
        if ((sb & 0xffu) + 1u < J.max_bounces) {
          ++sb;
          o = so.o;
          d = so.d;
          at = so.atten;
          fresh = true;
        } else {
          finish(J, li);  // bounce budget spent: no sky term (cpu.rs:256)
        }
      }
    }
    // The walk's per-ray values, for the fresh rays and again (the same
    // values) for the lanes in mid-walk, which did not keep them.
    if (fresh || walking()) {
      r = ray_pre(o, d);
      if (fresh) {
        best = kNoBest;
        sp = stack_first - 2u * kRow;
        if (walkable(r) && r.a >= kMinDot && r.a <= kMaxDot) {
          node = 0;
        } else {
          // the linear scan, exact for every ray (cpu.rs:345-349); the lane
          // is shaded in the next turn
          float bt = 0.0f;
          uint32_t bid = kNoHit;
          for (uint32_t j = 0; j < J.n_prims; ++j) {
            DevPrim pr;
            load_prim(J.prims, j, &pr);
            if constexpr (VK) test_prim_vk(r, pr, &bt, &bid);
            else test_prim(r, pr, &bt, &bid);
          }
          best = ((uint64_t)fbits(bt) << 32) | bid;
        }
      }
      ya = rcp_rn_normal(r.a);
      nf = slab_nf(slab_ray(r, ray_tolerance(r, J.r0_tol)));
      neg_x = nf.ix < 0.0f;
      neg_y = nf.iy < 0.0f;
      neg_z = nf.iz < 0.0f;
      tcull = cull();
    }
    // ---- the walk, until enough lanes are out of it: with work left every
    // lane that does not walk can be put to use; once the list is empty one
    // is only worth shading, so the wave waits for three quarters of them
    const uint32_t walkers = (uint32_t)__popcll(__ballot(walking()));
    if (walkers == 0) {
      if (!more && __ballot(has) == 0) break;
      continue;
    }
    const uint32_t keep = more ? 64u - a.refill : walkers / 4u;
    for (;;) {
      const uint64_t at_nodes = __ballot(node != kNoNode);
      if constexpr (kPooled) {
        // Test one primitive a lane once many lanes have one, or a pool could
        // overflow in the next step, or nothing else is left to do.
        const uint64_t pending = __ballot(pool != pool_first);
        if ((uint32_t)__popcll(pending) >= kPoolTests || at_nodes == 0 ||
            __ballot(pool > pool_first + 4u * kRow) != 0) {
          if (pending == 0) break;
          if (pool != pool_first) {
            pool -= kRow;
            test(stack_at(pool));
            tcull = cull();
          }
          continue;
        }
        if ((uint32_t)__popcll(at_nodes | pending) <= keep) break;
      } else {
        if ((uint32_t)__popcll(at_nodes) <= keep) break;
      }
      if (__builtin_amdgcn_inverse_ballot_w64(at_nodes)) {
#ifdef RDH_CHECKED
        node = chk(node, n_nodes4, K_NODE, a.ctl);
#endif
        float t0, t1, t2, t3;
        uint32_t e0, e1, e2, e3;
        VecI4 ch;
        bool h0 = false, h1 = false, h2 = false, h3 = false;
        if constexpr (kCompact) {
          // DevNode4C: a plane's distance is (origin + h * unit) * i - n, as
          // fma(h, unit * i, fma(origin, i, -n)) with an exact first product
          // (unit is a power of two, and the product finite: plan_paths); the
          // inner one rounds by 2^-24 of the node origin's distance from the
          // ray's, which the 1e-6 L of every primitive's box covers (bvh.cpp).
          const __attribute__((address_space(1))) unsigned char *gb =
              (const __attribute__((address_space(1))) unsigned char *)a.compact;
          const uint32_t nb = node * (uint32_t)sizeof(DevNode4C);
          const VecI4 hd = *(GlobalI4 *)(gb + nb), wx = *(GlobalI4 *)(gb + (nb + 16u));
          const VecI4 wy = *(GlobalI4 *)(gb + (nb + 32u)), wz = *(GlobalI4 *)(gb + (nb + 48u));
          const float unit = bitsf((uint32_t)hd.w & 0x7f800000u);
          const float cx = bitsf((uint32_t)hd.x & 0xffff0000u), cy = bitsf((uint32_t)hd.y & 0xffff0000u);
          const float cz = bitsf((uint32_t)hd.z & 0xffff0000u);
          const float sx = unit * nf.ix, sy = unit * nf.iy, sz = unit * nf.iz;
          const float bnx = fmaf(cx, nf.ix, -nf.nx), bfx = fmaf(cx, nf.ix, -nf.fx);
          const float bny = fmaf(cy, nf.iy, -nf.ny), bfy = fmaf(cy, nf.iy, -nf.fy);
          const float bnz = fmaf(cz, nf.iz, -nf.nz), bfz = fmaf(cz, nf.iz, -nf.fz);
          const int xna = neg_x ? wx.z : wx.x, xnb = neg_x ? wx.w : wx.y;
          const int xfa = neg_x ? wx.x : wx.z, xfb = neg_x ? wx.y : wx.w;
          const int yna = neg_y ? wy.z : wy.x, ynb = neg_y ? wy.w : wy.y;
          const int yfa = neg_y ? wy.x : wy.z, yfb = neg_y ? wy.y : wy.w;
          const int zna = neg_z ? wz.z : wz.x, znb = neg_z ? wz.w : wz.y;
          const int zfa = neg_z ? wz.x : wz.z, zfb = neg_z ? wz.y : wz.w;
          auto enters = [&](float xn, float xf, float yn, float yf, float zn, float zf, float *t) {
            const float tn = fmaxf(fmaxf(fmaf(xn, sx, bnx), fmaf(yn, sy, bny)),
                                   fmaxf(fmaf(zn, sz, bnz), 0.0f));
            const float tf = fminf(fminf(fmaf(xf, sx, bfx), fmaf(yf, sy, bfy)),
                                   fminf(fmaf(zf, sz, bfz), tcull));
            *t = tn;
            return tn <= tf;
          };
          h0 = enters(half_lo(xna), half_lo(xfa), half_lo(yna), half_lo(yfa), half_lo(zna), half_lo(zfa), &t0);
          h1 = enters(half_hi(xna), half_hi(xfa), half_hi(yna), half_hi(yfa), half_hi(zna), half_hi(zfa), &t1);
          h2 = enters(half_lo(xnb), half_lo(xfb), half_lo(ynb), half_lo(yfb), half_lo(znb), half_lo(zfb), &t2);
          h3 = enters(half_hi(xnb), half_hi(xfb), half_hi(ynb), half_hi(yfb), half_hi(znb), half_hi(zfb), &t3);
          // keys as below, the leaf flag moved to the sign bit
          auto key = [](float t, int code, uint32_t flag) {
            return (flag & 0x80000000u) | (((uint32_t)code & 0xffffu) | (fbits(t) & 0x7fff0000u));
          };
          const uint32_t fl = (uint32_t)hd.w;
          e0 = h0 ? key(t0, hd.x, fl << 15) : kNoKey;
          e1 = h1 ? key(t1, hd.y, fl << 14) : kNoKey;
          e2 = h2 ? key(t2, hd.z, fl << 13) : kNoKey;
          e3 = h3 ? key(t3, hd.w, fl) : kNoKey;
          ch = hd;
        } else {
          // each axis's near and far planes of the four children, picked by the
          // ray's direction signs (slab_hit_nf)
          VecF4 xn, xf, yn, yf, zn, zf;
          if (LDS) {
            const unsigned char *np = reinterpret_cast<const unsigned char *>(lds_nodes + 8 * node);
            xn = *(const VecF4 *)(np + nf.ox); xf = *(const VecF4 *)((np - nf.ox) + 16);
            yn = *(const VecF4 *)(np + nf.oy); yf = *(const VecF4 *)((np - nf.oy) + 80);
            zn = *(const VecF4 *)(np + nf.oz); zf = *(const VecF4 *)((np - nf.oz) + 144);
            ch = *(const VecI4 *)(np + 96);
          } else {
            // 32-bit offsets from the tree's base keep the address arithmetic
            // out of 64-bit registers
            const __attribute__((address_space(1))) unsigned char *gb =
                (const __attribute__((address_space(1))) unsigned char *)nodes4;
            const uint32_t nb = node * (uint32_t)sizeof(DevNode4);
            xn = *(GlobalF4 *)(gb + (nb + nf.ox)); xf = *(GlobalF4 *)(gb + ((nb - nf.ox) + 16u));
            yn = *(GlobalF4 *)(gb + (nb + nf.oy)); yf = *(GlobalF4 *)(gb + ((nb - nf.oy) + 80u));
            zn = *(GlobalF4 *)(gb + (nb + nf.oz)); zf = *(GlobalF4 *)(gb + ((nb - nf.oz) + 144u));
            ch = *(GlobalI4 *)(gb + (nb + 96u));
          }
          h0 = slab_hit_nf(nf, xn.x, xf.x, yn.x, yf.x, zn.x, zf.x, tcull, &t0);
          h1 = slab_hit_nf(nf, xn.y, xf.y, yn.y, yf.y, zn.y, zf.y, tcull, &t1);
          h2 = slab_hit_nf(nf, xn.z, xf.z, yn.z, yf.z, zn.z, zf.z, tcull, &t2);
          h3 = slab_hit_nf(nf, xn.w, xf.w, yn.w, yf.w, zn.w, zf.w, tcull, &t3);
          // The entered inner children, nearest first.  A key is the entry
          // distance's upper 16 bits (it only orders the visits) above the
          // child's index; a leaf's code leaves the sign bit set, as kNoKey has
          // it, so those keys sort behind.  Seven integer min/med/max steps
          // order distance and child together (the float form took a compare
          // and four selects for each of five exchanges).
          e0 = h0 ? (fbits(t0) & 0x7fff0000u) | (uint32_t)ch.x : kNoKey;
          e1 = h1 ? (fbits(t1) & 0x7fff0000u) | (uint32_t)ch.y : kNoKey;
          e2 = h2 ? (fbits(t2) & 0x7fff0000u) | (uint32_t)ch.z : kNoKey;
          e3 = h3 ? (fbits(t3) & 0x7fff0000u) | (uint32_t)ch.w : kNoKey;
        }
        if constexpr (kPooled) {
          // the entered leaves' primitives go above the lane's others; a key
          // plus one has the sign bit set for a leaf's alone
          stack_at(pool) = leaf_prim(ch.x);
          pool = row_if(e0 + 1u, pool);
          stack_at(pool) = leaf_prim(ch.y);
          pool = row_if(e1 + 1u, pool);
          stack_at(pool) = leaf_prim(ch.z);
          pool = row_if(e2 + 1u, pool);
          stack_at(pool) = leaf_prim(ch.w);
          pool = row_if(e3 + 1u, pool);
        }
        const uint32_t lo = umin(umin(e0, e1), e2), mid = umed3(e0, e1, e2), hi = umax(umax(e0, e1), e2);
        const uint32_t r0 = umin(lo, e3), r1 = umed3(lo, mid, e3);
        const uint32_t r2 = umed3(mid, hi, e3), r3 = umax(hi, e3);
        // The stack grows downwards.  The farther ones go on it, farthest
        // first; an entry that is none (sign bit set) is written too and the
        // next one put over it.  The nearest is next, or the top of the stack
        // (kNoNode above the first).
#ifdef RDH_CHECKED
        // (one up: the first row of lane 0 is at 0, as is what chk puts in place)
        if (chk(sp - lds_base + 1u, stack_bytes - 2u * kRow + 1u, K_STACK, a.ctl) == 0u) sp = stack_first - 2u * kRow;
#endif
        stack_at(sp + 2u * kRow) = (StackT)r3;
        sp = row_if(r3, sp);
        stack_at(sp + kRow) = (StackT)r2;
        sp = row_if(r2, sp);
        stack_at(sp) = (StackT)r1;
        sp = row_if(r1, sp);
        const uint32_t popped = stack_at(sp);
        node = (int32_t)r0 < 0 ? popped : r0 & 0xffffu;
        sp = row_if(r0, sp) - 3u * kRow;
        if constexpr (LDS && LEAF1) {
          // the entered leaves' bits, and a primitive a trip: its half word of
          // the codes is picked by a byte permutation (selecting it by three
          // compares took 10 instructions a trip, and counting 12 a step; 97
          // objects at 1080p, 64 spp 10.63 -> 10.30 ms with plain branches to
          // the tests' slow forms, a closed room 3.67 -> 3.54)
          auto entered = [](bool h, int code) { return h ? (uint32_t)code : 0u; };
          uint32_t mask = (entered(h0, ch.x) | entered(h1, ch.y) | entered(h2, ch.z) | entered(h3, ch.w)) & 0xf0000u;
          if (mask != 0) {
            const uint32_t f01 = __builtin_amdgcn_perm(ch.y, ch.x, 0x05040100u);
            const uint32_t f23 = __builtin_amdgcn_perm(ch.w, ch.z, 0x05040100u);
            do {
              // bytes 2k + 1 and 2k, and zeros above (from 16 + k without a
              // constant in a register: 0x202 (16 + k) is 2020 + 202 k, hex)
              const uint32_t bit = (uint32_t)__builtin_ctz(mask);
              mask &= mask - 1u;
              test(__builtin_amdgcn_perm(f23, f01, (bit * 0x202u) ^ 0x0c0c2120u));
            } while (mask != 0);
            tcull = cull();
          }
        } else if constexpr (!kPooled) {
          // trip t tests f_k + t for the k-th hit leaf
          const uint32_t n0 = h0 && is_leaf(ch.x) ? leaf_count(ch.x) : 0u;
          const uint32_t p1 = n0 + (h1 && is_leaf(ch.y) ? leaf_count(ch.y) : 0u);
          const uint32_t p2 = p1 + (h2 && is_leaf(ch.z) ? leaf_count(ch.z) : 0u);
          const uint32_t n_leaf = p2 + (h3 && is_leaf(ch.w) ? leaf_count(ch.w) : 0u);
          const uint32_t f0 = leaf_first(ch.x), f1 = leaf_first(ch.y) - n0;
          const uint32_t f2 = leaf_first(ch.z) - p1, f3 = leaf_first(ch.w) - p2;
          for (uint32_t t = 0; t < n_leaf; ++t)
            test((t < n0 ? f0 : t < p1 ? f1 : t < p2 ? f2 : f3) + t);
          if (n_leaf) tcull = cull();
        }
      }
    }
  }
}

// k_accumulate and k_tonemap (kernels.hip) in one pass over the accumulator, a
// thread a pixel, which spares the image's read of it and a launch.  Bound by
// HBM for a large image (1080p, one sample: 15 + 9 us and 5 between -> 18), by
// its launch for a small one, whose bytes it writes to the host itself:
// 128x128, 8 spp, whole call 127 -> 107 us; 256x256, 16 spp 245 -> 227;
// 643x361, 7 spp 612 -> 587.
__global__ __launch_bounds__(256) void k_finish(const DevJob *job, DevTicket T, uint32_t npix,
                                                const float4 *L, float samples, uchar4 *rgba) {
  float4 *acc = reinterpret_cast<float4 *>(load_constant(&job->acc));
  for (uint32_t px = blockIdx.x * 256u + threadIdx.x; px < npix; px += gridDim.x * 256u) {
    float4 v = acc[px];
    for (uint32_t s = 0; s < T.spp; ++s) {
      const float4 c = L[T.l_offset + (uint64_t)s * npix + px];
      v = make_float4(v.x + c.x, v.y + c.y, v.z + c.z, v.w + 1.0f);
    }
    acc[px] = v;
    rgba[px] = make_uchar4(tonemap_channel(v.x, samples), tonemap_channel(v.y, samples),
                           tonemap_channel(v.z, samples), tonemap_channel(v.w, samples));
  }
}

__global__ __launch_bounds__(256) void k_debug_arith(int which, const float *a, const float *b, uint32_t n,
                                                     float *out) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= n) return;
  const float x = a[i], y = b[i];
  out[i] = which == 0   ? sqrt_rn(x)
           : which == 1 ? rcp_rn(x)
           : which == 2 ? div_rn(x, y, rcp_rn_normal(y))
           : which == 3 ? normalize(f3(x, y, 0.0f)).x
           : which == 4 ? sqrt_rn_normal(x)
                        : rcp_rn_normal(x);
}

template <bool VK>
const void *paths_fn_of(PathTree tree, bool record) {
  switch (tree) {
    case kTreeMemory:
      return record ? (const void *)k_paths<kPathBlock, true, kTreeMemory, VK>
                    : (const void *)k_paths<kPathBlock, false, kTreeMemory, VK>;
    case kTreeCompact:  // (not with Vulkan semantics: plan_paths)
      // camera rays share their nodes: recorded from the tree itself
      if constexpr (!VK)
        if (!record) return (const void *)k_paths<kPathBlock, false, kTreeCompact, VK>;
      [[fallthrough]];
    case kTreeLeaf1:
      return record ? (const void *)k_paths<kPathBlock, true, kTreeLeaf1, VK>
                    : (const void *)k_paths<kPathBlock, false, kTreeLeaf1, VK>;
    case kTreeLds:
      return record ? (const void *)k_paths<kPathBlock, true, kTreeLds, VK>
                    : (const void *)k_paths<kPathBlock, false, kTreeLds, VK>;
    default:
      return record ? (const void *)k_paths<kPathBlock, true, kTreeLdsLeaf1, VK>
                    : (const void *)k_paths<kPathBlock, false, kTreeLdsLeaf1, VK>;
  }
}

const void *paths_fn(const PathArgs &a, bool record) {
  return a.vk ? paths_fn_of<true>(a.tree, record) : paths_fn_of<false>(a.tree, record);
}

uint32_t dynamic_lds_bytes(const PathArgs &a, bool record) {
  return ((a.stack_rows * kPathBlock * 2u + 15u) & ~15u) +
         (a.tree == kTreeLeaf1 || a.tree == kTreeCompact ? pool_bytes<kPathBlock>() : 0u) +
         a.lds_bvh_bytes + (record ? 0u : a.lds_obj_bytes);
}

}  // namespace

// A tree is copied into LDS by every workgroup as long as that costs none of
// the workgroups the registers allow on a CU (five, with Vulkan semantics
// four); the objects too if they fit beside it.  183 objects (17 KB) at 4K, 8
// spp: 9.2 ms from memory, 8.0 from LDS.  Larger workgroups that share a copy
// were slower than the walk in memory: 640 threads 300 objects 1.33 -> 1.45 ms,
// 500 objects 1.46 -> 1.69 (1280x720, 16 spp, whole call).
//
// A larger tree of one-primitive leaves is walked as DevNode4C, four 16-byte
// loads a node instead of seven, where that outweighs a third more instructions:
// in a large tree, whose node fetches miss the L1, and in a long pass, whose
// rate counts and not the latency of its last paths.  1280x720, 16 spp, full ->
// compact: 1000 objects (455 nodes) 1.03 -> 1.04 ms, 1400 (621) 1.24 -> 1.23,
// 2000 1.56 -> 1.50, 2400 1.78 -> 1.66, 4096 (1777) 2.63 -> 2.26, 8000 4.62 ->
// 4.01; 1080p, 2 spp: 2400 1.06 -> 1.10, 4096 1.28 -> 1.33, 8000 1.71 -> 1.73,
// 14000 2.07 -> 1.97: the line is nodes times paths, where no pass measured loses
// (8000 objects in the short pass come to 1.45e10) and 2000 in the long one, at
// 1.3e10, leave 4 % behind.  With Vulkan semantics
// (four waves per SIMD, more registers) the full nodes are faster at every
// size: 2400 2.48 against 2.26, 4096 2.92 and 2.56, 14000 5.55 and 5.28.  Nor for
// scenes beyond 2^62, where a node's unit times 1/d (at most 2^60) could overflow.
void plan_paths(PathArgs *a, const DevJob &j, uint64_t lds_bvh, uint64_t lds_objects) {
  constexpr uint64_t kCompactNodes = 768, kCompactWork = 14ull << 30;
  constexpr float kCompactReach = 0x1p62f;
  const bool compact = !a->vk && j.n_nodes4 >= kCompactNodes && j.reach <= kCompactReach &&
                       (uint64_t)a->npix * a->samples * j.n_nodes4 >= kCompactWork;
  a->stack_rows = j.stack4 + 4;  // a sentinel below, and three written above the top
  const bool leaf1 = j.max_leaf == 1;
  const uint64_t blocks = 4 * path_waves(false, a->vk) / (kPathBlock / 64);
  const uint64_t room = 160 * 1024 / blocks - 1024, stack = 2ull * a->stack_rows * kPathBlock + 16;
  const uint64_t tree = sizeof(DevNode4) * (uint64_t)j.n_nodes4 + sizeof(DevPrim) * (uint64_t)j.n_prims;
  const uint64_t objects = sizeof(DevObject) * (uint64_t)j.n_prims;
  const bool lds = tree <= lds_bvh && stack + tree <= room;
  a->tree = lds ? (leaf1 ? kTreeLdsLeaf1 : kTreeLds)
                : !leaf1 ? kTreeMemory : compact ? kTreeCompact : kTreeLeaf1;
  a->lds_bvh_bytes = lds ? (uint32_t)tree : 0u;
  const uint64_t used = stack + (lds ? tree : pool_bytes<kPathBlock>());
  a->lds_obj_bytes = objects <= lds_objects && used + objects <= room ? (uint32_t)objects : 0u;
}

int path_blocks_per_cu(const PathArgs &a, bool record) {
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, paths_fn(a, record), kPathBlock,
                                                   dynamic_lds_bytes(a, record)) != hipSuccess) {
    (void)hipGetLastError();
    return 1;
  }
  return std::max(1, n);
}

hipError_t launch_paths(const PathArgs &a, bool record, int grid, hipStream_t st) {
  PathArgs args = a;
  void *kargs[] = {&args};
  return hipLaunchKernel(paths_fn(a, record), dim3(grid), dim3(kPathBlock), kargs,
                         dynamic_lds_bytes(a, record), st);
}

hipError_t launch_compact(const PathArgs &a, hipStream_t st) {
  k_compact<<<(a.n_nodes4 + 63) / 64, 64, 0, st>>>(a.job, a.compact, a.n_nodes4);
  return hipGetLastError();
}

hipError_t launch_finish(const DevJob *job, const DevTicket &t, uint32_t npix, const float4 *L, float samples,
                         uchar4 *rgba, int max_grid, hipStream_t st) {
  const uint32_t grid = std::min<uint32_t>((npix + 255u) / 256u, (uint32_t)max_grid);
  k_finish<<<grid, 256, 0, st>>>(job, t, npix, L, samples, rgba);
  return hipGetLastError();
}

hipError_t launch_debug_arith(int which, const float *a, const float *b, uint32_t n, float *out, hipStream_t st) {
  if (n == 0) return hipSuccess;
  k_debug_arith<<<(uint32_t)((n + 255ull) / 256), 256, 0, st>>>(which, a, b, n, out);
  return hipGetLastError();
}

}  // namespace rdh
