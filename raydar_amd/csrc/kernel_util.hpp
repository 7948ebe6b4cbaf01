// Device helpers shared by the wavefront kernels (kernels.hip) and the path
// kernel (paths.hip): checked indexing, wave-lane masks, scalar and vector
// loads of the scene, the camera paths' pixel order.
#pragma once

#include "kernels.hpp"
#include "pathmath.hpp"

namespace rdh {

namespace {

// Bounds-checked builds (-DRDH_CHECKED) pass every computed index through
// chk(): an index outside its buffer sets bit `bit` of QueueCtl::violation
// (the host then fails the render) and is replaced by 0, so the access
// itself stays inside the buffer.  Production builds compile chk() away.
enum CheckBit {
  K_SLOT = 0, K_TICKET, K_JOB, K_NODE, K_PRIM, K_STACK, K_OBJECT, K_RADIANCE
};
template <class I>
__device__ __forceinline__ I chk(I i, I n, CheckBit bit, QueueCtl *ctl) {
#ifdef RDH_CHECKED
  if (i >= n) {
    atomicOr(&ctl->violation, 1u << bit);
    return I(0);
  }
#endif
  (void)n; (void)bit; (void)ctl;
  return i;
}

__device__ __forceinline__ uint32_t lanes_below(uint64_t mask) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                   __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}
__device__ __forceinline__ uint32_t lane_id() { return lanes_below(~0ull); }

// A record of a table that no kernel writes during a launch, read through
// the constant address space: at a wave-uniform address that is a scalar
// load.  The pointer is rebuilt from its integer value, which the compiler
// cannot fold back to a global pointer (a plain cast it folds, and the loads
// stay vector loads).  The host pass of the compiler only checks the body.
template <class T>
__device__ __forceinline__ T load_constant(const T *p) {
#if defined(__HIP_DEVICE_COMPILE__)
  return *(const __attribute__((address_space(4))) T *)(uintptr_t)p;
#else
  return *p;
#endif
}

// Scene buffers are reached through pointers read from the job table, which
// the compiler cannot place in an address space; these loads name the global
// space explicitly so they become global_load (not flat_load, which also
// waits on the LDS counter the traversal stack uses).
typedef float VecF4 __attribute__((ext_vector_type(4)));
typedef float VecF2 __attribute__((ext_vector_type(2)));
typedef int VecI4 __attribute__((ext_vector_type(4)));
typedef unsigned int VecU4 __attribute__((ext_vector_type(4)));
typedef unsigned int VecU2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(1))) const VecF4 GlobalF4;
typedef __attribute__((address_space(1))) const VecF2 GlobalF2;
typedef __attribute__((address_space(1))) const VecI4 GlobalI4;
typedef __attribute__((address_space(1))) const VecU4 GlobalU4;
typedef __attribute__((address_space(1))) const VecU2 GlobalU2;
typedef __attribute__((address_space(1))) VecF4 GlobalF4Out;
typedef __attribute__((address_space(1))) VecF2 GlobalF2Out;
typedef __attribute__((address_space(1))) VecU4 GlobalU4Out;
typedef __attribute__((address_space(1))) VecU2 GlobalU2Out;

__device__ __forceinline__ void load_prim(const DevPrim *prims, uint32_t j, DevPrim *p) {
  GlobalF4 *s = (GlobalF4 *)(prims + j);
  const VecF4 a = s[0], b = s[1];
  p->a[0] = a.x; p->a[1] = a.y; p->a[2] = a.z; p->a[3] = a.w;
  p->b[0] = b.x; p->b[1] = b.y; p->b[2] = b.z; p->b[3] = b.w;
}

__device__ __forceinline__ DevObject object_from(VecF4 g, VecF4 m0, VecF4 m1, VecF4 m2) {
  DevObject o;
  o.geo[0] = g.x; o.geo[1] = g.y; o.geo[2] = g.z; o.geo[3] = g.w;
  o.m0[0] = m0.x; o.m0[1] = m0.y; o.m0[2] = m0.z; o.m0[3] = m0.w;
  o.m1[0] = m1.x; o.m1[1] = m1.y; o.m1[2] = m1.z; o.m1[3] = m1.w;
  o.m2[0] = m2.x; o.m2[1] = m2.y; o.m2[2] = m2.z; o.m2[3] = m2.w;
  return o;
}
__device__ __forceinline__ DevObject load_object(const DevObject *objects, uint32_t id) {
  GlobalF4 *s = (GlobalF4 *)(objects + id);
  return object_from(s[0], s[1], s[2], s[3]);
}

// Pixel of the r-th camera path of a sample: 8x8 tiles, row by row inside a
// tile and tile by tile along each band of 8 rows (the columns right of the
// last whole tile row-major inside the band; a last band of fewer than 8 rows
// row-major), a permutation of [0, W*H).  A wave's 64 consecutive paths then
// start from one 8x8 tile instead of 64 pixels of one row: their rays and,
// after a bounce, their origins stay close together, which the closest-hit
// kernel's node fetches and traversal order profit from.  A path's draws,
// radiance slot and accumulation are keyed by its pixel, so the order changes
// no result.
__device__ __forceinline__ uint32_t tile_order_pixel(uint32_t r, uint32_t W, uint32_t H) {
  const uint32_t band_px = 8u * W;
  const uint32_t band = r / band_px;
  if ((band + 1u) * 8u > H) return r;
  const uint32_t q = r - band * band_px;
  const uint32_t full = W & ~7u;
  uint32_t x, y;
  if (q < full * 8u) {
    x = (q >> 6) * 8u + (q & 7u);
    y = band * 8u + ((q >> 3) & 7u);
  } else {
    const uint32_t e = q - full * 8u, rw = W - full;
    x = full + e % rw;
    y = band * 8u + e / rw;
  }
  return y * W + x;
}

// Comparator of the 4-wide traversal's sorting network: (ka, ca) gets the
// smaller key (a strictly smaller kb swaps, as the host traversal does).
__device__ __forceinline__ void order_pair(float &ka, int32_t &ca, float &kb, int32_t &cb) {
  const bool sw = kb < ka;
  const float k = sw ? kb : ka;
  const int32_t c = sw ? cb : ca;
  kb = sw ? ka : kb;
  cb = sw ? ca : cb;
  ka = k;
  ca = c;
}

}  // namespace

}  // namespace rdh
