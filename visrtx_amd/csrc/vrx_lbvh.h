// vrx_lbvh.h -- node layout and build entry shared by the HIP translation units.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/vrx_hip.h"
#include "vrx_math.h"

namespace vrx {

// 64-byte BVH2 node holding the boxes of both children (see lbvh.hip).
struct alignas(16) Node {
  float4 a, b, c;
  uint4 d;
};
static_assert(sizeof(Node) == 64, "Node must be 64 bytes");

__device__ __forceinline__ Node gld_node(const Node *nodes, size_t i)
{
  typedef float f4v __attribute__((ext_vector_type(4)));
  typedef unsigned int u4v __attribute__((ext_vector_type(4)));
  const __attribute__((address_space(1))) f4v *q =
      (const __attribute__((address_space(1))) f4v *)(nodes + i);
  f4v a = q[0], b = q[1], c = q[2];
  u4v d = ((const __attribute__((address_space(1))) u4v *)(nodes + i))[3];
  Node n;
  n.a = make_float4(a.x, a.y, a.z, a.w);
  n.b = make_float4(b.x, b.y, b.z, b.w);
  n.c = make_float4(c.x, c.y, c.z, c.w);
  n.d = make_uint4(d.x, d.y, d.z, d.w);
  return n;
}

// 128-byte 4-wide node (one HBM line): the boxes of up to four children in
// SoA form and their links (bit 31 = leaf, as in Node); slots at or beyond
// `count` are unused.
struct alignas(16) Node4 {
  float4 lox, loy, loz, hix, hiy, hiz;
  uint4 link;
  uint4 meta; // x = count (2..4)
};
static_assert(sizeof(Node4) == 128, "Node4 must be 128 bytes");

__device__ __forceinline__ Node4 gld_node4(const Node4 *nodes, size_t i)
{
  typedef float f4v __attribute__((ext_vector_type(4)));
  typedef unsigned int u4v __attribute__((ext_vector_type(4)));
  const __attribute__((address_space(1))) f4v *q =
      (const __attribute__((address_space(1))) f4v *)(nodes + i);
  f4v a = q[0], b = q[1], c = q[2], d = q[3], e = q[4], f = q[5];
  const __attribute__((address_space(1))) u4v *u =
      (const __attribute__((address_space(1))) u4v *)(nodes + i);
  u4v l = u[6], m = u[7];
  Node4 n;
  n.lox = make_float4(a.x, a.y, a.z, a.w);
  n.loy = make_float4(b.x, b.y, b.z, b.w);
  n.loz = make_float4(c.x, c.y, c.z, c.w);
  n.hix = make_float4(d.x, d.y, d.z, d.w);
  n.hiy = make_float4(e.x, e.y, e.z, e.w);
  n.hiz = make_float4(f.x, f.y, f.z, f.w);
  n.link = make_uint4(l.x, l.y, l.z, l.w);
  n.meta = make_uint4(m.x, m.y, m.z, m.w);
  return n;
}

// 64-byte packed 4-wide node: the boxes of up to four children on a grid of
// 8-bit steps.  Plane q of an axis lies at origin + q * scale; a child's
// planes enclose its box by at least kPackMargin steps (vrx_bvh_pack), which
// covers the rounding of the traversal's plane distances.  Byte c of the
// lo / hi words belongs to child c; an unused slot holds kPackEmpty.
// The traversal is bound by its box-test arithmetic and by the L1 data path
// of its node fetches: half the bytes of Node4 (and of the two BVH2 levels it
// spans) relieve the second, the one-FMA planes the first.  Against BVH2
// nodes, the faster of the two older forms on these scenes: 10M spheres
// 1920x1080 raycast frame 580 -> 502 us, AO 16 spp 14.9 -> 11.6 ms; 1M lit
// spheres 5.1 -> 3.9 ms; 64 views of 9.4M instanced triangles 13.8 -> 13.2 ms
// (against Node4).
struct alignas(16) Node4p {
  float ox, oy, oz, sx;
  float sy, sz;
  uint32_t lox, loy, loz, hix, hiy, hiz;
  uint4 link;
};
static_assert(sizeof(Node4p) == 64, "Node4p must be 64 bytes");

// link of an unused slot: a leaf no BVH has (n < 2^31 - 1)
constexpr uint32_t kPackEmpty = 0xFFFFFFFEu;
constexpr double kPackMargin = 1.0 / 64.0;

__device__ __forceinline__ Node4p gld_node4p(const Node4p *nodes, size_t i)
{
  typedef float f4v __attribute__((ext_vector_type(4)));
  typedef unsigned int u4v __attribute__((ext_vector_type(4)));
  const __attribute__((address_space(1))) u4v *u =
      (const __attribute__((address_space(1))) u4v *)(nodes + i);
  const f4v a = ((const __attribute__((address_space(1))) f4v *)(nodes + i))[0];
  const u4v b = u[1], c = u[2], d = u[3];
  Node4p n;
  n.ox = a.x; n.oy = a.y; n.oz = a.z; n.sx = a.w;
  n.sy = __uint_as_float(b.x); n.sz = __uint_as_float(b.y);
  n.lox = b.z; n.loy = b.w;
  n.loz = c.x; n.hix = c.y; n.hiy = c.z; n.hiz = c.w;
  n.link = make_uint4(d.x, d.y, d.z, d.w);
  return n;
}

// What a walk needs of an instance, one 128-byte line, in the order of the
// instance level's sorted leaves (after its packed nodes): entering an
// instance is one fetch instead of a chain of three (leaf id, entry,
// geometry), and hits read the rest.
struct alignas(128) InstRec {
  float inv[12];          // world -> object
  const void *nodes;      // packed nodes of the geometry
  const void *leaves;
  const uint32_t *ids;
  uint32_t entry, flags;  // kInst* | type << 8
  float box[6];           // the entry's exact box
  float opacity;
  uint32_t pad[5];
};
static_assert(sizeof(InstRec) == 128, "InstRec must be 128 bytes");
constexpr uint32_t kInstIdentity = 1, kInstBoxed = 2, kInstCull = 4, kInstCaps = 8, kInstEmpty = 16;

__host__ __device__ __forceinline__ size_t inst_rec_offset(uint32_t n)
{
  return ((size_t)(n - 1) * sizeof(Node4p) + 127) & ~size_t(127);
}

int bvh_pack_impl(const vrx_bvh *bvh, uint32_t n, hipStream_t s);

// float4s per leaf record
template <int T>
constexpr int record_quads()
{
  return T == VRX_SPHERE ? 1
      : (T == VRX_CYLINDER || T == VRX_CONE || T == VRX_CURVE) ? 2 : (T == VRX_TRIANGLE ? 3 : 0);
}

// box of a leaf record (the bounds rule of the build's prim_box)
template <int T>
__device__ __forceinline__ void record_box(const float4 *L, v3 &lo, v3 &hi)
{
  if constexpr (T == VRX_SPHERE) {
    const float4 a = L[0];
    lo = mk(a.x - a.w, a.y - a.w, a.z - a.w);
    hi = mk(a.x + a.w, a.y + a.w, a.z + a.w);
  } else if constexpr (T == VRX_CYLINDER) {
    const float4 a = L[0], b = L[1];
    v3 mn = vmin(mk(a.x, a.y, a.z), mk(b.x, b.y, b.z)), mx = vmax(mk(a.x, a.y, a.z), mk(b.x, b.y, b.z));
    lo = mk(mn.x - a.w, mn.y - a.w, mn.z - a.w);
    hi = mk(mx.x + a.w, mx.y + a.w, mx.z + a.w);
  } else if constexpr (T == VRX_CONE) {
    const float4 a = L[0], b = L[1];
    v3 mn = vmin(mk(a.x, a.y, a.z), mk(b.x, b.y, b.z)), mx = vmax(mk(a.x, a.y, a.z), mk(b.x, b.y, b.z));
    float r = fmaxf(a.w, b.w);
    lo = mk(mn.x - r, mn.y - r, mn.z - r);
    hi = mk(mx.x + r, mx.y + r, mx.z + r);
  } else if constexpr (T == VRX_CURVE) {
    const float4 a = L[0], b = L[1];
    lo = vmin(mk(a.x - a.w, a.y - a.w, a.z - a.w), mk(b.x - b.w, b.y - b.w, b.z - b.w));
    hi = vmax(mk(a.x + a.w, a.y + a.w, a.z + a.w), mk(b.x + b.w, b.y + b.w, b.z + b.w));
  } else if constexpr (T == VRX_TRIANGLE) {
    const float4 a = L[0], b = L[1], c = L[2];
    v3 v0 = mk(a.x, a.y, a.z), v1 = mk(b.x, b.y, b.z), v2 = mk(c.x, c.y, c.z);
    lo = vmin(vmin(v0, v1), v2);
    hi = vmax(vmax(v0, v1), v2);
  }
}

size_t leaf_record_bytes(int type);
void bvh_sizes(int32_t type, uint32_t n, vrx_bvh_sizes *o);
int bvh_build_impl(const vrx_prims *p, const vrx_bvh *out, void *d_ws, size_t ws_bytes,
    uint32_t *codes_out, float *cbox_out, hipStream_t s);

} // namespace vrx
