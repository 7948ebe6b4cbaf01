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
// What bounds it: VALU issue (99% busy on 97 objects in LDS), then the node
// fetches of a tree outside LDS.  Against the wavefront it gains most in
// shading: a turn shades only lanes that hit something (a wavefront tile is a
// third misses), and no lane waits for a path's record to come back from HBM.
// 77% of the lanes work in an average VALU instruction (wavefront: 54% in
// extend, 58% in shade).  Measured, wavefront -> paths: 97 objects at 1080p,
// 64 spp 20.0 -> 12.8 ms; 4096 objects 19.9 -> 17.7 ms; a closed room at
// 960x540, 16 spp 6.1 -> 4.3 ms; 256x256, 16 spp, whole call 0.56 -> 0.31 ms;
// one sample at 1080p with a new scene 1.28 -> 1.00 ms.
#include <algorithm>

#include "kernel_util.hpp"
#include "paths.hpp"

namespace rdh {

namespace {

// Waves per SIMD the path kernel is compiled for.
#ifndef RDH_PATH_WAVES
#define RDH_PATH_WAVES 6
#endif
constexpr int path_waves(bool record, bool vk) { return vk && !record ? 5 : RDH_PATH_WAVES; }

// The camera rays' common origin.
template <bool VK>
__device__ __forceinline__ F3 camera_origin(const DevJob &J) {
  F3 o = f3(J.position[0], J.position[1], J.position[2]), d;
  if constexpr (VK) camera_ray_vk(J, 0, 0, &o, &d);
  return o;
}

// RECORD: trace every pixel's camera ray and write its hit to the table, in
// the order the paths are handed out (tile_order_pixel).
// LDS: the tree and the primitives are copied into LDS by every workgroup.
// LEAF1: every leaf holds one primitive.
// VK (Vulkan semantics): a pixel's samples share one stream of random numbers,
// whose place after a sample depends on that sample's draws, so a lane keeps
// its pixel for all samples of the pass, one after another, with the stream's
// state in a register, and adds each to the accumulator itself (the order
// k_accumulate would take).  The camera ray has no draw in it here either.
// 97 objects, 1280x720, 16 spp: 8.1 -> 3.5 ms, which were 16 passes of one
// sample with 12 bounces of three launches each; 5 waves per SIMD, as the
// stream and rank do not fit the registers of 6.
template <int BLOCK, bool RECORD, bool LDS, bool LEAF1, bool VK>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(path_waves(RECORD, VK), 8)))
void k_paths(PathArgs a) {
  typedef uint16_t StackT;
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
  const uint32_t stack_bytes = (a.stack_rows * BLOCK * (uint32_t)sizeof(StackT) + 15u) & ~15u;
  StackT *stk = reinterpret_cast<StackT *>(dynamic_lds) + threadIdx.x;
  VecF4 *lds_nodes = reinterpret_cast<VecF4 *>(dynamic_lds + stack_bytes);
  const uint32_t node_vecs = LDS ? 8 * n_nodes4 : 0u, prim_vecs = LDS ? 2 * n_prims : 0u;
  VecF4 *lds_prims = lds_nodes + node_vecs;
  VecF4 *lds_objects = lds_prims + prim_vecs;
  const bool lds_obj = !RECORD && a.lds_obj_bytes != 0;
  if (LDS) {
    GlobalF4 *gn = (GlobalF4 *)nodes4, *gp = (GlobalF4 *)prims;
    for (uint32_t i = threadIdx.x; i < node_vecs; i += BLOCK) lds_nodes[i] = gn[i];
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
  const uint32_t slice = blockIdx.x % a.slices;
  const uint32_t slice_chunks = (a.chunks + a.slices - 1u - slice) / a.slices;
  const float cull0 = VK ? cull_limit(kVkTMax, 0u) : INFINITY;  // with no hit yet
  // A lane is walking (active), waits to be shaded (full) or is free.
  bool active = false, full = false;
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
  float bt = 0.0f, tcull = INFINITY;
  uint32_t bid = kNoHit;
  int32_t node = 0;
  int sp = 0;
  RayPre r;
  SlabNF nf;

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
        bt = cr.w;
        bid = a.cam_hit[vk_rank].x;
        at = f3(1.0f, 1.0f, 1.0f);
        li = f3(0.0f, 0.0f, 0.0f);
        sb = ((sb >> 8) + 1u) << 8;
        full = true;
      } else {
        J.vk_rng[pixel] = vk_state;
      }
      return;
    }
    const unsigned long long slot =
        a.l_offset + (unsigned long long)(sb >> 8) * a.npix + pixel;
    a.L[chk(slot, a.l_cap, K_RADIANCE, a.ctl)] = make_float4(c.x, c.y, c.z, 1.0f);
  };

  for (;;) {
    const uint64_t walking = __ballot(active), waiting = __ballot(full);
    // With work left every lane that is not walking can be put to use; once
    // the list is empty a lane is only worth shading when it waits, and the
    // wave shades when three quarters of its live lanes do.
    const uint32_t live = (uint32_t)__popcll(walking | waiting);
    const bool turn = more ? 64u - (uint32_t)__popcll(walking) >= a.refill
                           : 4u * (uint32_t)__popcll(waiting) >= 3u * live;
    if (turn || walking == 0) {
      if (!more && live == 0) break;
      const DevJob J = load_constant(a.job);
      if constexpr (RECORD) {
        if (full) {
          a.cam_ray[sb] = make_float4(d.x, d.y, d.z, bid == kNoHit ? 0.0f : bt);
          a.cam_hit[sb] = make_uint2(bid, pixel);
          full = false;
        }
      } else if (full && bid == kNoHit) {
        // cpu.rs:334-337 (raytrace.rgen:178)
        full = false;
        finish(J, add(li, mul(VK ? world_sample_vk(J, d) : world_sample(J, d), at)));
      }
      // Free lanes take the next paths.  A camera path starts at its pixel's
      // recorded hit, so it is shaded in this turn with the lanes that
      // finished a walk; one that left the scene ends at once, and its lane
      // asks again.
      bool fresh = false;
      while (more) {
        const uint64_t need = __ballot(!active && !full);
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
        if (!active && !full && k < size) {
          const uint32_t rank = chk(group * 64u + k, a.npix, K_RADIANCE, a.ctl);
          if constexpr (RECORD) {
            pixel = tile_order_pixel(rank, J.width, J.height);
            if (VK) camera_ray_vk(J, pixel % J.width, pixel / J.width, &o, &d);
            else camera_ray(J, pixel % J.width, pixel / J.width, &o, &d);
            sb = rank;
            fresh = true;
            full = true;  // (until its walk starts below)
          } else {
            const float4 cr = a.cam_ray[rank];
            const uint2 ch = a.cam_hit[rank];
            o = camera_origin<VK>(J);
            d = f3(cr.x, cr.y, cr.z);
            bt = cr.w;
            bid = ch.x;
            pixel = ch.y;
            sb = sample << 8;
            // a camera path's attenuation and light (cpu.rs:253-254)
            at = f3(1.0f, 1.0f, 1.0f);
            li = f3(0.0f, 0.0f, 0.0f);
            if constexpr (VK) {
              vk_rank = rank;
              vk_state = a.sample_base == 0 ? pixel % J.width + (pixel / J.width) * 1000u : J.vk_rng[pixel];
            }
            if (bid != kNoHit) {
              full = true;
            } else {
              const F3 c = add(li, mul(VK ? world_sample_vk(J, d) : world_sample(J, d), at));
              if constexpr (VK) {
                // every sample of the pixel is this one and draws nothing
                float4 *acc = reinterpret_cast<float4 *>(J.acc) + pixel;
                float4 v = *acc;
                for (uint32_t k = 0; k < a.samples; ++k)
                  v = make_float4(v.x + c.x, v.y + c.y, v.z + c.z, v.w + 1.0f);
                *acc = v;
                J.vk_rng[pixel] = vk_state;
              } else {
                finish(J, c);
              }
            }
          }
        }
        off += (uint32_t)__popcll(need);
      }
      if (!RECORD && full) {
        const uint32_t oid = chk(bid, J.n_prims, K_OBJECT, a.ctl);
        const DevObject ob = lds_obj ? object_from(lds_objects[4 * oid], lds_objects[4 * oid + 1],
                                                   lds_objects[4 * oid + 2], lds_objects[4 * oid + 3])
                                     : load_object(J.objects, oid);
        const HitRec h = closest_hit(o, d, bt, ob);
        ScatterOut so;
        if constexpr (VK) {
          so = scatter_vk(d, h, ob, vk_state, at, li);
        } else {
          BounceDraws dr;
          dr.init(J.seed, pixel, a.sample_base + (sb >> 8), sb & 0xffu);
          so = scatter(d, h, ob, dr, at, li);
        }
        li = so.light;
        full = false;
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
      // The walk's per-ray values, for the fresh rays and again (the same
      // values) for the lanes in mid-walk, which did not keep them.
      if (fresh || active) {
        r = ray_pre(o, d);
        if (fresh) {
          bt = 0.0f;
          bid = kNoHit;
          node = 0;
          sp = 0;
          active = walkable(r);
          full = !active;
          if (full)  // the linear scan, exact for every ray (cpu.rs:345-349)
            for (uint32_t j = 0; j < J.n_prims; ++j) {
              DevPrim pr;
              load_prim(J.prims, j, &pr);
              if (VK) test_prim_vk(r, pr, &bt, &bid);
              else test_prim(r, pr, &bt, &bid);
            }
        }
        nf = slab_nf(slab_ray(r, ray_tolerance(r, J.r0_tol)));
        tcull = VK && bid == kNoHit ? cull0 : cull_limit(bt, bid);
      }
      continue;
    }
    if (active) {
#ifdef RDH_CHECKED
      node = (int32_t)chk((uint32_t)node, n_nodes4, K_NODE, a.ctl);
#endif
      // each axis's near and far planes of the four children, picked by the
      // ray's direction signs (slab_hit_nf)
      VecF4 xn, xf, yn, yf, zn, zf;
      VecI4 ch;
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
        const uint32_t nb = (uint32_t)node * (uint32_t)sizeof(DevNode4);
        xn = *(GlobalF4 *)(gb + (nb + nf.ox)); xf = *(GlobalF4 *)(gb + ((nb - nf.ox) + 16u));
        yn = *(GlobalF4 *)(gb + (nb + nf.oy)); yf = *(GlobalF4 *)(gb + ((nb - nf.oy) + 80u));
        zn = *(GlobalF4 *)(gb + (nb + nf.oz)); zf = *(GlobalF4 *)(gb + ((nb - nf.oz) + 144u));
        ch = *(GlobalI4 *)(gb + (nb + 96u));
      }
      float t0, t1, t2, t3;
      const bool h0 = slab_hit_nf(nf, xn.x, xf.x, yn.x, yf.x, zn.x, zf.x, tcull, &t0);
      const bool h1 = slab_hit_nf(nf, xn.y, xf.y, yn.y, yf.y, zn.y, zf.y, tcull, &t1);
      const bool h2 = slab_hit_nf(nf, xn.z, xf.z, yn.z, yf.z, zn.z, zf.z, tcull, &t2);
      const bool h3 = slab_hit_nf(nf, xn.w, xf.w, yn.w, yf.w, zn.w, zf.w, tcull, &t3);
      const bool l0 = h0 && is_leaf(ch.x), l1 = h1 && is_leaf(ch.y);
      const bool l2 = h2 && is_leaf(ch.z), l3 = h3 && is_leaf(ch.w);
      // trip t tests f_k + t for the k-th hit leaf (one primitive each with
      // LEAF1: trip t is that leaf's first primitive)
      const uint32_t n0 = l0 ? (LEAF1 ? 1u : leaf_count(ch.x)) : 0u;
      const uint32_t p1 = n0 + (l1 ? (LEAF1 ? 1u : leaf_count(ch.y)) : 0u);
      const uint32_t p2 = p1 + (l2 ? (LEAF1 ? 1u : leaf_count(ch.z)) : 0u);
      const uint32_t n_leaf = p2 + (l3 ? (LEAF1 ? 1u : leaf_count(ch.w)) : 0u);
      const uint32_t f0 = leaf_first(ch.x), f1 = leaf_first(ch.y) - (LEAF1 ? 0u : n0);
      const uint32_t f2 = leaf_first(ch.z) - (LEAF1 ? 0u : p1);
      const uint32_t f3 = leaf_first(ch.w) - (LEAF1 ? 0u : p2);
      // The next node and the stack are settled before the primitive tests
      // (they depend only on this node's boxes), so the children's keys and
      // ids are dead while the primitives are tested.
      const bool i0 = h0 && !l0, i1 = h1 && !l1, i2 = h2 && !l2, i3 = h3 && !l3;
      const int cnt = (int)i0 + (int)i1 + (int)i2 + (int)i3;
      int32_t c0;
      if (__ballot(cnt > 1) == 0) {
        // no lane entered two inner children: nothing to order or push
        c0 = i0 ? ch.x : i1 ? ch.y : i2 ? ch.z : ch.w;
      } else {
        float k0 = i0 ? t0 : INFINITY, k1 = i1 ? t1 : INFINITY;
        float k2 = i2 ? t2 : INFINITY, k3 = i3 ? t3 : INFINITY;
        int32_t c1 = ch.y, c2 = ch.z, c3 = ch.w;
        c0 = ch.x;
        order_pair(k0, c0, k1, c1);
        order_pair(k2, c2, k3, c3);
        order_pair(k0, c0, k2, c2);
        order_pair(k1, c1, k3, c3);
        order_pair(k1, c1, k2, c2);
#ifdef RDH_CHECKED
        sp = (int)chk((uint32_t)sp + 2u, a.stack_rows, K_STACK, a.ctl) - 2;
        if (sp < 0) sp = 0;
#endif
        stk[sp * BLOCK] = (StackT)(cnt == 4 ? c3 : cnt == 3 ? c2 : c1);
        stk[(sp + 1) * BLOCK] = (StackT)(cnt == 4 ? c2 : c1);
        stk[(sp + 2) * BLOCK] = (StackT)c1;
      }
      const int top = sp > 0 ? sp - 1 : 0;
      const int32_t popped = (int32_t)stk[top * BLOCK];
      const bool done = cnt == 0 && sp == 0;
      if (cnt > 0) {
        node = c0;
        sp += cnt - 1;
      } else if (sp > 0) {
        node = popped;
        sp = top;
      }
      if (n_leaf) {
        for (uint32_t t = 0; t < n_leaf; ++t) {
          DevPrim pr;
          uint32_t j = LEAF1 ? (t < n0 ? f0 : t < p1 ? f1 : t < p2 ? f2 : f3)
                             : (t < n0 ? f0 + t : t < p1 ? f1 + t : t < p2 ? f2 + t : f3 + t);
#ifdef RDH_CHECKED
          j = chk(j, n_prims, K_PRIM, a.ctl);
#endif
          if (LDS) {
            const VecF4 pa = lds_prims[2 * j], pb = lds_prims[2 * j + 1];
            pr.a[0] = pa.x; pr.a[1] = pa.y; pr.a[2] = pa.z; pr.a[3] = pa.w;
            pr.b[0] = pb.x; pr.b[1] = pb.y; pr.b[2] = pb.z; pr.b[3] = pb.w;
          } else {
            load_prim(prims, j, &pr);
          }
          if (VK) test_prim_vk(r, pr, &bt, &bid);
          else test_prim(r, pr, &bt, &bid);
        }
        tcull = VK && bid == kNoHit ? cull0 : cull_limit(bt, bid);
      }
      if (done) {
        active = false;
        full = true;
      }
    }
  }
}

constexpr int kPathBlock = 256;

template <bool RECORD, bool VK>
const void *paths_fn_of(bool lds, bool leaf1) {
  return lds ? (leaf1 ? (const void *)k_paths<kPathBlock, RECORD, true, true, VK>
                      : (const void *)k_paths<kPathBlock, RECORD, true, false, VK>)
             : (leaf1 ? (const void *)k_paths<kPathBlock, RECORD, false, true, VK>
                      : (const void *)k_paths<kPathBlock, RECORD, false, false, VK>);
}

const void *paths_fn(const PathArgs &a, bool record) {
  const bool lds = a.lds_bvh_bytes > 0, leaf1 = a.leaf1 != 0;
  if (a.vk) return record ? paths_fn_of<true, true>(lds, leaf1) : paths_fn_of<false, true>(lds, leaf1);
  return record ? paths_fn_of<true, false>(lds, leaf1) : paths_fn_of<false, false>(lds, leaf1);
}

uint32_t dynamic_lds_bytes(const PathArgs &a, bool record) {
  return ((a.stack_rows * kPathBlock * 2u + 15u) & ~15u) + a.lds_bvh_bytes +
         (record ? 0u : a.lds_obj_bytes);
}

}  // namespace

int path_blocks_per_cu(const PathArgs &a, bool record) {
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
          &n, paths_fn(a, record), kPathBlock,
          dynamic_lds_bytes(a, record)) != hipSuccess) {
    (void)hipGetLastError();
    return 1;
  }
  return std::max(1, n);
}

hipError_t launch_paths(const PathArgs &a, bool record, int grid, hipStream_t st) {
  PathArgs args = a;
  void *kargs[] = {&args};
  return hipLaunchKernel(paths_fn(a, record), dim3(grid),
                         dim3(kPathBlock), kargs, dynamic_lds_bytes(a, record), st);
}

}  // namespace rdh
