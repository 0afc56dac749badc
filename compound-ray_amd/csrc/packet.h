// Wave-packet traversal of the 64-wide tree (wide_bvh.h), gfx950.
//
// The 64 rays of a wave are samples of one or a few neighbouring ommatidia.
// The wave walks the tree together, and a step tests a node's 64 children
// twice:
//   - lane l tests child l against the packet's bounds (the four planes and
//     the depth range of the rays' frustum): one pass of about 45 VALU
//     instructions rejects most of the 64 boxes;
//   - each child left is tested by every lane against its own ray (14
//     instructions, the box read from its lane into scalar registers), and is
//     entered when any lane's ray enters it before its closest hit.
// Every lane tests the triangles of an entered leaf; entered nodes are
// walked nearest first, the others wait in LDS.
//
// What bounds it: VALU issue.  A wave64 instruction takes a SIMD four cycles,
// and the 4-wide packet walk spent 25 instructions on each of 160-250 boxes
// per 64 rays, three quarters of which no ray entered, and up to 53 dependent
// node fetches; here a packet makes 3-14 fetches and 10-150 ray tests.
//
// A lane tests a superset of the triangles that its own ray's boxes hold, and
// keeps the exact (t, id) minimum, so the result is that of any other walk.
#pragma once

#include <hip/hip_runtime.h>

#include "bvh_format.h"
#include "eyecore.h"
#include "wide_bvh.h"

namespace eye {
namespace {

struct Hit {
  float t, b1, b2;
  uint32_t k;   // canonical triangle position
  uint32_t id;  // original triangle id, 0xffffffff for a miss
  float det;    // during traversal b1, b2 hold V, W of the closest hit and det its
                // determinant; finish_hit divides them (b1 = V / det, b2 = W / det)
};

__device__ __forceinline__ void finish_hit(Hit& h) {
  if (h.id != 0xffffffffu) {
    h.b1 = h.b1 / h.det;
    h.b2 = h.b2 / h.det;
  }
}

__device__ __forceinline__ float lane_f(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ float first_f(float v) {
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

// Wave-wide maxima of six values, each in its VGPR at once: six DPP maxima
// per value (four within rows of 16 lanes, two across rows), the values taking
// turns, which also keeps the two wait states between a write and its DPP read.
// The compiler's form of one step is a copy, a wait, a DPP move, two
// canonicalising maxima and the maximum: 435 VALU instructions for a packet's
// bounds, 230 so.  Every lane of the wave takes part.
__device__ __forceinline__ void wave_max6(float& a, float& b, float& c, float& d, float& e, float& f) {
#define EYE_DPP_STEP(ctrl)                      \
  "v_max_f32_dpp %0, %0, %0 " ctrl "\n\t"       \
  "v_max_f32_dpp %1, %1, %1 " ctrl "\n\t"       \
  "v_max_f32_dpp %2, %2, %2 " ctrl "\n\t"       \
  "v_max_f32_dpp %3, %3, %3 " ctrl "\n\t"       \
  "v_max_f32_dpp %4, %4, %4 " ctrl "\n\t"       \
  "v_max_f32_dpp %5, %5, %5 " ctrl "\n\t"
  asm volatile("s_nop 1\n\t"
               EYE_DPP_STEP("quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf")
               EYE_DPP_STEP("quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf")
               EYE_DPP_STEP("row_half_mirror row_mask:0xf bank_mask:0xf")
               EYE_DPP_STEP("row_mirror row_mask:0xf bank_mask:0xf")
               EYE_DPP_STEP("row_bcast:15 row_mask:0xa bank_mask:0xf")
               EYE_DPP_STEP("row_bcast:31 row_mask:0xc bank_mask:0xf")
               "s_nop 1"
               : "+v"(a), "+v"(b), "+v"(c), "+v"(d), "+v"(e), "+v"(f));
#undef EYE_DPP_STEP
  a = lane_f(a, 63);
  b = lane_f(b, 63);
  c = lane_f(c, 63);
  d = lane_f(d, 63);
  e = lane_f(e, 63);
  f = lane_f(f, 63);
}
// The maximum of a value that is not negative in any lane: compared as bits.
template <int kCtrl, int kRows = 0xf>
__device__ __forceinline__ int dpp_i(int i) {
  return __builtin_amdgcn_update_dpp(i, i, kCtrl, kRows, 0xf, false);
}
__device__ __forceinline__ float wave_max_depth(float v) {
  int i = __float_as_int(v);
  i = max(i, dpp_i<0xb1>(i));
  i = max(i, dpp_i<0x4e>(i));
  i = max(i, dpp_i<0x141>(i));
  i = max(i, dpp_i<0x140>(i));
  i = max(i, dpp_i<0x142, 0xa>(i));
  i = max(i, dpp_i<0x143, 0xc>(i));
  return __int_as_float(__builtin_amdgcn_readlane(i, 63));
}

// The frustum around a packet's rays, wave-uniform: a frame (u, v, w) with w
// along the first ray, the ranges of the rays' slopes d.u / d.w and d.v / d.w,
// and the rays' starts' offsets from the four planes.  Margins cover the
// rounding of these values; that of the box tests is in the boxes' padding.
struct PacketBounds {
  V3 u, v, w;
  float a0, a1, b0, b1;       // slopes
  float oa0, oa1, ob0, ob1;   // plane offsets
  float near;                 // smallest start depth along w
  float spread;               // largest origin depth beyond it
  float reach;                // largest depth along w per unit of t
  float pad;                  // far origins only: added to half extents
};

// Whether the box may meet the frustum, and its depth beyond the starts along
// w (a number: the boxes are bounded, kWideFarthest).
__device__ __forceinline__ bool bounds_meet(const PacketBounds& B, const V3& c, const V3& h, float* depth) {
  const float cu = fmaf(c.z, B.u.z, fmaf(c.y, B.u.y, c.x * B.u.x));
  const float cv = fmaf(c.z, B.v.z, fmaf(c.y, B.v.y, c.x * B.v.x));
  const float cw = fmaf(c.z, B.w.z, fmaf(c.y, B.w.y, c.x * B.w.x));
  const float ru = fmaf(h.z, fabsf(B.u.z), fmaf(h.y, fabsf(B.u.y), h.x * fabsf(B.u.x)));
  const float rv = fmaf(h.z, fabsf(B.v.z), fmaf(h.y, fabsf(B.v.y), h.x * fabsf(B.v.x)));
  const float rw = fmaf(h.z, fabsf(B.w.z), fmaf(h.y, fabsf(B.w.y), h.x * fabsf(B.w.x)));
  const float fa1 = fmaf(-fabsf(B.a1), rw, fmaf(-B.a1, cw, cu)), fa0 = fmaf(-fabsf(B.a0), rw, fmaf(B.a0, cw, -cu));
  const float fb1 = fmaf(-fabsf(B.b1), rw, fmaf(-B.b1, cw, cv)), fb0 = fmaf(-fabsf(B.b0), rw, fmaf(B.b0, cw, -cv));
  *depth = cw - rw - B.near;
  return !(fa1 > B.oa1 + ru) && !(fa0 > B.oa0 + ru) && !(fb1 > B.ob1 + rv) && !(fb0 > B.ob0 + rv) &&
         !(cw + rw < B.near);
}

// One ray as the packet tests need it.  Components ok*, s* are permuted by the
// ray's axes (k), the watertight test's order.
struct PacketRay {
  float ix, iy, iz;      // reciprocal direction
  float nx, ny, nz;      // -origin * reciprocal
  float okx, oky, okz;   // origin
  float sx, sy, sz;      // shear and scale
  float tmin;
  int k;                 // kx | ky << 2 | kz << 4
};

// Whether the ray enters the box before `limit`.  The rounding of the test is
// within the boxes' padding.
__device__ __forceinline__ bool ray_meets(const PacketRay& r, float cx, float cy, float cz, float hx, float hy,
                                          float hz, float limit) {
  const float tx = fmaf(cx, r.ix, r.nx), ty = fmaf(cy, r.iy, r.ny), tz = fmaf(cz, r.iz, r.nz);
  const float ax = fabsf(r.ix), ay = fabsf(r.iy), az = fabsf(r.iz);
  const float tn = fmaxf(fmaxf(fmaf(-hx, ax, tx), fmaf(-hy, ay, ty)), fmaxf(fmaf(-hz, az, tz), r.tmin));
  const float tf = fminf(fminf(fmaf(hx, ax, tx), fmaf(hy, ay, ty)), fminf(fmaf(hz, az, tz), limit));
  return tn <= tf;
}

// Wave-uniform records read through the constant address space: scalar loads,
// once per wave, into scalar registers that the vector tests use directly.
typedef float f8v __attribute__((ext_vector_type(8)));
typedef float f4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(4))) const f8v k8v;
typedef __attribute__((address_space(4))) const f4v k4v;

// The watertight test of eyecore.h's intersect_triangle_raw, the same
// operations on the same values, with the corners' components already in the
// ray's axis order.
__device__ __forceinline__ void test_triangle(const PacketRay& r, const V3& a, const V3& b, const V3& c, uint32_t id,
                                              uint32_t pos, Hit& h) {
  const float az = a.z - r.okz, bz = b.z - r.okz, cz = c.z - r.okz;
  const float ax = (a.x - r.okx) - r.sx * az, ay = (a.y - r.oky) - r.sy * az;
  const float bx = (b.x - r.okx) - r.sx * bz, by = (b.y - r.oky) - r.sy * bz;
  const float cx = (c.x - r.okx) - r.sx * cz, cy = (c.y - r.oky) - r.sy * cz;
  const float U = cx * by - cy * bx;
  const float V = ax * cy - ay * cx;
  const float W = bx * ay - by * ax;
  const float det = U + V + W;
  // two signs among the edges, or none of any size
  if ((fminf(fminf(U, V), W) < 0.0f) & (fmaxf(fmaxf(U, V), W) > 0.0f) | (det == 0.0f)) return;
  const float T = U * (r.sz * az) + V * (r.sz * bz) + W * (r.sz * cz);
  const float t = T / det;
  if (t >= r.tmin && (t < h.t || (t == h.t && id < h.id))) {
    h.t = t;
    h.b1 = V;
    h.b2 = W;
    h.det = det;
    h.k = pos;
    h.id = id;
  }
}

// A leaf's triangles, each three rows (x, y, z) of its corners' components.
// When all rays share the axis order, the rows are read in that order.
template <bool kShared>
__device__ __forceinline__ void test_leaf64(const float4* tris, int32_t code, const PacketRay& r, int axes, Hit& h) {
  const uint32_t cnt = leaf_count(code);
  const k4v* rows = (const k4v*)(tris + 3 * (size_t)leaf_first(code));
  for (uint32_t q = 0; q < cnt; ++q, rows += 3) {
    const f4v x = rows[kShared ? axes & 3 : 0], y = rows[kShared ? (axes >> 2) & 3 : 1],
              z = rows[kShared ? axes >> 4 : 2];
    const f4v tag = rows[0];
    const f4v pos = rows[1];
    V3 a = v3(x.x, y.x, z.x), b = v3(x.y, y.y, z.y), c = v3(x.z, y.z, z.z);
    if (!kShared) {
      const int kx = r.k & 3, ky = (r.k >> 2) & 3, kz = r.k >> 4;
      a = v3(comp(a.x, a.y, a.z, kx), comp(a.x, a.y, a.z, ky), comp(a.x, a.y, a.z, kz));
      b = v3(comp(b.x, b.y, b.z, kx), comp(b.x, b.y, b.z, ky), comp(b.x, b.y, b.z, kz));
      c = v3(comp(c.x, c.y, c.z, kx), comp(c.x, c.y, c.z, ky), comp(c.x, c.y, c.z, kz));
    }
    test_triangle(r, a, b, c, __float_as_uint(tag.w), __float_as_uint(pos.w), h);
  }
}

// Node fetches in units of the canonical tree's 128-byte nodes.
constexpr uint32_t kWideFetch = sizeof(WideNode64) / 128;

// The walk of the lanes `in`.  Every lane of the wave takes part (ballots and
// lane reads).  stack: the wave's LDS column (wide_stack entries).  fetched /
// tris count node bytes / 128 and leaf triangles (wave-uniform).  kFar: the
// origins lie far outside the scene, whose boxes' padding does not cover
// them, or rays start behind theirs and may hit there, at a negative t.
template <bool kShared, bool kFar>
__device__ __forceinline__ void walk64(const WideNode64* nodes, const float4* wtris, int root, const PacketBounds& B,
                                       const PacketRay& r, bool in, int axes, uint2* stack, Hit& h,
                                       uint32_t& fetched, uint32_t& tris) {
  const int lane = (int)(threadIdx.x & 63);
  int sp = 0;
  int node = root;
  const auto cull_limit = [](float t) { return kFar ? fmaf(fabsf(t), kCullSlack - 1.0f, t) : t * kCullSlack; };
  float limit = in ? cull_limit(h.t) : -INFINITY;
  // Depth beyond which every ray has a closer hit: depths count from the
  // starts, a hit's t from its ray's origin.
  float horizon = INFINITY;
  for (;;) {
    node = __builtin_amdgcn_readfirstlane(node);
    fetched += kWideFetch;
    const WideChild* kids = nodes[node].child;
    const float4 lo = reinterpret_cast<const float4*>(kids + lane)[0];
    const float4 hi = reinterpret_cast<const float4*>(kids + lane)[1];
    const V3 c = v3(lo.x, lo.y, lo.z);
    const V3 e = kFar ? v3(hi.x + B.pad, hi.y + B.pad, hi.z + B.pad) : v3(hi.x, hi.y, hi.z);
    const int ref = __float_as_int(lo.w);
    float depth;
    const bool meets = bounds_meet(B, c, e, &depth) && !(depth > horizon) && ref != kChildEmpty;
    uint64_t leaves = __ballot(meets && ref < 0);
    uint64_t inner = __ballot(meets && ref >= 0);
    const k8v* boxes = (const k8v*)kids;
    const auto any_ray = [&](const f8v& x) {
      const float p = kFar ? B.pad : 0.0f;
      return __ballot(ray_meets(r, x[0], x[1], x[2], kFar ? x[4] + p : x[4], kFar ? x[5] + p : x[5],
                                kFar ? x[6] + p : x[6], limit)) != 0ull;
    };
    bool closer = false;
    if (leaves != 0ull) {
      f8v box = boxes[__builtin_ctzll(leaves)];
      do {
        leaves &= leaves - 1;
        // the next box is on its way while this one is tested
        const f8v next = boxes[leaves != 0ull ? __builtin_ctzll(leaves) : 0];
        if (any_ray(box)) {
          const int32_t code = __float_as_int(box[3]);
          tris += leaf_count(code);
          const float before = h.t;
          test_leaf64<kShared>(wtris, code, r, axes, h);
          limit = in ? cull_limit(h.t) : -INFINITY;
          closer = closer || __ballot(h.t < before) != 0ull;
        }
        box = next;
      } while (leaves != 0ull);
    }
    if (closer) horizon = wave_max_depth(in ? (kFar ? fmaxf(h.t, 0.0f) : h.t) : 0.0f) * B.reach + B.spread;
    uint64_t kept = 0ull;
    if (inner != 0ull) {
      int l = __builtin_ctzll(inner);
      f8v box = boxes[l];
      do {
        inner &= inner - 1;
        const int ln = inner != 0ull ? __builtin_ctzll(inner) : 0;
        const f8v next = boxes[ln];
        if (any_ray(box)) kept |= 1ull << l;
        box = next;
        l = ln;
      } while (inner != 0ull);
    }
    if (kept != 0ull) {
      // rank 0: the farthest; the nearest is walked next, the rest wait
      const int n = __popcll(kept);
      int next = __builtin_ctzll(kept);
      if (n > 1) {
        int rank = 0;
        for (uint64_t m = kept; m != 0ull; m &= m - 1) {
          const int l = __builtin_ctzll(m);
          const float dl = lane_f(depth, l);
          rank += (dl > depth || (dl == depth && l > lane)) ? 1 : 0;
        }
        const bool here = ((kept >> lane) & 1ull) != 0ull;
        if (here && rank < n - 1) stack[sp + rank] = make_uint2((uint32_t)ref, __float_as_uint(depth));
        next = __builtin_ctzll(__ballot(here && rank == n - 1));
        sp += n - 1;
      }
      node = __builtin_amdgcn_readlane(ref, next);
      continue;
    }
    bool found = false;
    while (sp > 0 && !found) {
      --sp;
      const uint2 w = stack[sp];
      node = (int)w.x;
      found = !(first_f(__uint_as_float(w.y)) > horizon);
    }
    if (!found) break;
  }
}

// Rays further than this slope from a packet's first ray, or whose origin is
// further from its than the scene's longest extent times kPacketSpread, go
// in a packet of their own: a wave of several ommatidia may hold several
// cones, or several eyes.
constexpr float kPacketSlope = 1.0f;
constexpr float kPacketSpread = 1.0f / 256.0f;
constexpr float kFarStart = 1e30f;
constexpr float kLeastComponent = 1e-37f;   // per unit of the scene's coordinates

// The offsets and depths of B for rays that start `back` <= 0 times d behind
// their origins o, all of them within `out` of 0 along each axis.  From starts
// so far behind that they cannot be computed with (tmin may be infinite) the
// packet has no bounds.
__device__ __forceinline__ void bound_starts_behind(PacketBounds& B, const V3& o, const V3& d, float back, bool in,
                                                    float out) {
  const V3 p = v3(fmaf(back, d.x, o.x), fmaf(back, d.y, o.y), fmaf(back, d.z, o.z));
  const float away = fabsf(p.x) + fabsf(p.y) + fabsf(p.z);
  const float pu = dot(p, B.u), pv = dot(p, B.v), pw = dot(p, B.w);
  float oa1 = pu - B.a1 * pw, oa0 = B.a0 * pw - pu, ob1 = pv - B.b1 * pw, ob0 = B.b0 * pw - pv, nr = -pw,
        fr = dot(o, B.w);
  wave_max6(oa0, oa1, ob0, ob1, nr, fr);
  const float m = 8.0f * kWidePad * fmaxf(out, wave_max_depth(in && away < kFarStart ? away : 0.0f));
  const bool bounded = __ballot(in && !(away < kFarStart)) == 0ull;
  B.oa0 = first_f(bounded ? oa0 + m : INFINITY);
  B.oa1 = first_f(bounded ? oa1 + m : INFINITY);
  B.ob0 = first_f(bounded ? ob0 + m : INFINITY);
  B.ob1 = first_f(bounded ? ob1 + m : INFINITY);
  B.near = first_f(bounded ? -nr - m : -INFINITY);
  B.spread = first_f(bounded ? (fr + nr) + 2.0f * m : INFINITY);
}

// Closest hits of the wave's rays (ray, rp: this lane's) in the tree of T.
struct WideTree {
  const WideNode64* nodes;
  const float4* tris;
  int root;
  int stack;      // LDS entries per wave
  float spread;   // how far apart the origins of one packet may be
  float range;    // origins this far out are covered by the boxes' padding
  float least;    // smaller direction components count as this
};

__device__ __forceinline__ void closest_hit_wide(const WideTree& T, const Ray& ray, const RayPre& rp, bool active,
                                                 uint2* stack, uint32_t* fault, Hit& h, uint32_t& fetched,
                                                 uint32_t& tris, float slope = kPacketSlope) {
  h.t = rp.tmax;
  h.b1 = h.b2 = 0.0f;
  h.k = 0xffffffffu;
  h.id = 0xffffffffu;
  if (T.nodes == nullptr) return;
  // A wave that has lost lanes cannot walk (child l is lane l's to test): it
  // flags the launch for the host and returns misses.
  if (__ballot(1) != ~0ull) {
    if (fault) *fault = 1u;
    return;
  }
  PacketRay r;
  r.okx = comp(rp.ox, rp.oy, rp.oz, rp.kx);
  r.oky = comp(rp.ox, rp.oy, rp.oz, rp.ky);
  r.okz = comp(rp.ox, rp.oy, rp.oz, rp.kz);
  r.sx = rp.sx; r.sy = rp.sy; r.sz = rp.sz;
  r.k = rp.kx | rp.ky << 2 | rp.kz << 4;
  // A component near 0 counts as one whose reciprocal times any coordinate of the
  // scene is finite; what that moves a point sideways is far below the boxes'
  // padding.  (From an origin so far out that the product is not, the ray runs
  // past every box, as its test then finds.)
  r.ix = __builtin_amdgcn_rcpf(fabsf(ray.dx) < T.least ? copysignf(T.least, ray.dx) : ray.dx);
  r.iy = __builtin_amdgcn_rcpf(fabsf(ray.dy) < T.least ? copysignf(T.least, ray.dy) : ray.dy);
  r.iz = __builtin_amdgcn_rcpf(fabsf(ray.dz) < T.least ? copysignf(T.least, ray.dz) : ray.dz);
  r.nx = -(ray.ox * r.ix); r.ny = -(ray.oy * r.iy); r.nz = -(ray.oz * r.iz);
  // A ray with a not-a-number or an origin beyond 1e30 hits nothing: its shears
  // or the triangle test's products are not numbers.  Directions beyond these
  // lengths are the caller's to scale.
  const float size = fabsf(ray.dx) + fabsf(ray.dy) + fabsf(ray.dz);
  const float far = fmaxf(fmaxf(fabsf(ray.ox), fabsf(ray.oy)), fabsf(ray.oz));
  uint64_t left = __ballot(active && size > 1e-36f && size < 1e37f && far < 1e30f);
  while (left != 0ull) {
    const int first = __builtin_ctzll(left);
    PacketBounds B;
    const V3 d = v3(ray.dx, ray.dy, ray.dz) * __builtin_amdgcn_rcpf(size);
    const V3 d0 = v3(lane_f(d.x, first), lane_f(d.y, first), lane_f(d.z, first));
    const V3 w = d0 * __builtin_amdgcn_rsqf(dot(d0, d0));
    const bool level = fabsf(w.y) < 0.9f;
    const V3 s = v3(level ? w.z : 0.0f, level ? 0.0f : -w.z, level ? -w.x : w.y);
    const V3 u = s * __builtin_amdgcn_rsqf(dot(s, s));
    const V3 v = cross(w, u);
    B.u = v3(first_f(u.x), first_f(u.y), first_f(u.z));
    B.v = v3(first_f(v.x), first_f(v.y), first_f(v.z));
    B.w = v3(first_f(w.x), first_f(w.y), first_f(w.z));
    const V3 o0 = v3(lane_f(ray.ox, first), lane_f(ray.oy, first), lane_f(ray.oz, first));
    const V3 gap = v3(ray.ox, ray.oy, ray.oz) - o0;
    const float k = dot(d, B.w);
    const float rk = __builtin_amdgcn_rcpf(k);
    float a = dot(d, B.u) * rk, b = dot(d, B.v) * rk;
    const bool in = ((left >> (threadIdx.x & 63)) & 1ull) != 0ull && k > 0.0f && fabsf(a) < slope &&
                    fabsf(b) < slope && fabsf(gap.x) + fabsf(gap.y) + fabsf(gap.z) <= T.spread;
    left &= ~(__ballot(in) | (1ull << first));
    // lanes of other packets take no hits here: their axes may differ
    r.tmin = in ? rp.tmin : INFINITY;
    a = in ? a : 0.0f;
    b = in ? b : 0.0f;
    const float margin = 8e-6f;   // slopes are below 1
    float a0 = -a, a1 = a, b0 = -b, b1 = b, reach = in ? k * size : 0.0f, out = in ? far : 0.0f;
    wave_max6(a0, a1, b0, b1, reach, out);
    B.a0 = first_f(-a0 - margin);
    B.a1 = first_f(a1 + margin);
    B.b0 = first_f(-b0 - margin);
    B.b1 = first_f(b1 + margin);
    B.reach = reach * 1.0002f;
    B.pad = 2.0f * kWidePad * out;
    const V3 o = v3(in ? ray.ox : o0.x, in ? ray.oy : o0.y, in ? ray.oz : o0.z);
    const bool behind = __ballot(in && rp.tmin < 0.0f) != 0ull;
    if (behind) {
      bound_starts_behind(B, o, v3(ray.dx, ray.dy, ray.dz), in ? fminf(rp.tmin, 0.0f) : 0.0f, in, out);
    } else {
      const float pu = dot(o, B.u), pv = dot(o, B.v), pw = dot(o, B.w);
      float oa1 = pu - B.a1 * pw, oa0 = B.a0 * pw - pu, ob1 = pv - B.b1 * pw, ob0 = B.b0 * pw - pv, nr = pw, fr = pw;
      // one start for all rays (samples of one ommatidium): no reductions
      if (__ballot(o.x != o0.x || o.y != o0.y || o.z != o0.z) != 0ull) {
        nr = -nr;
        wave_max6(oa0, oa1, ob0, ob1, nr, fr);
        nr = -nr;
      }
      const float m = 8.0f * kWidePad * out;
      B.oa0 = first_f(oa0 + m);
      B.oa1 = first_f(oa1 + m);
      B.ob0 = first_f(ob0 + m);
      B.ob1 = first_f(ob1 + m);
      B.near = first_f(nr - m);
      B.spread = first_f((fr - nr) + 2.0f * m);
    }
    const int axes = __builtin_amdgcn_readlane(r.k, first);
    if (behind || out > T.range)
      walk64<false, true>(T.nodes, T.tris, T.root, B, r, in, axes, stack, h, fetched, tris);
    else if (__ballot(in && r.k != axes) == 0ull)
      walk64<true, false>(T.nodes, T.tris, T.root, B, r, in, axes, stack, h, fetched, tris);
    else
      walk64<false, false>(T.nodes, T.tris, T.root, B, r, in, axes, stack, h, fetched, tris);
  }
  finish_hit(h);
}

}  // namespace
}  // namespace eye
