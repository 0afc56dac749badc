// gfx950 render kernels: fused Gaussian-cone ray generation + wide BVH
// traversal + shading (replacing __raygen__ommatidium, the OptiX traversal,
// __closesthit__radiance and the miss programs, libEyeRenderer3/shaders.cu:664-811),
// and the per-ommatidium wave reduction + projection (shaders.cu:341-406).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>

#include "launch_grid.h"
#include "packet.h"
#include "render.h"

namespace eye {
namespace {

constexpr int kTraceThreads = 256;
// XCDs of the device: workgroup b runs on XCD b % kXcds, each with its own L2.
constexpr uint32_t kXcds = 8;
constexpr int kPacketStackMax = 128;  // two VGPRs of 64 lanes

struct SceneView {
  const WideNode* nodes;
  const float4* tris;
  const float4* cols;
  const uint32_t* texels;
  const TexView* textures;
  WideTree wide;
  int node_count;
  int sky_mode;
  uint32_t* fault;   // host-visible word set when a packet traversal is entered by a partial wave
};

SceneView view_of(const DeviceScene& s) {
  SceneView v;
  v.nodes = s.nodes;
  v.tris = s.tris;
  v.cols = s.cols;
  v.texels = s.texels;
  v.textures = s.textures;
  float ext = 0.0f;
  for (int a = 0; a < 3; ++a) ext = std::max(ext, s.centroid_hi[a] - s.centroid_lo[a]);
  v.wide = WideTree{s.wide_nodes, s.wide_tris, s.wide_root, s.wide_stack, ext * kPacketSpread,
                    kWideRange * s.wide_radius, std::max(1e-30f, s.wide_farthest * kLeastComponent)};
  v.node_count = s.node_count;
  v.sky_mode = s.sky_mode;
  v.fault = s.fault;
  return v;
}

__device__ __forceinline__ void test_leaf(const float4* tris, int32_t code, const RayPre& rp, Hit& h) {
  const uint32_t first = leaf_first(code);
  const uint32_t cnt = leaf_count(code);
  for (uint32_t q = 0; q < cnt; ++q) {
    const uint32_t k = first + q;
    const float4 a = tris[3 * (size_t)k + 0];
    const float4 b = tris[3 * (size_t)k + 1];
    const float4 c = tris[3 * (size_t)k + 2];
    float t, vv, ww, det;
    if (intersect_triangle_raw(rp, v3(a.x, a.y, a.z), v3(b.x, b.y, b.z), v3(c.x, c.y, c.z), &t, &vv, &ww, &det)) {
      const uint32_t id = __float_as_uint(a.w);
      if (t < h.t || (t == h.t && id < h.id)) {
        h.t = t;
        h.b1 = vv;
        h.b2 = ww;
        h.det = det;
        h.k = k;
        h.id = id;
      }
    }
  }
}

// A wave-uniform leaf (packet traversal, every lane of the wave executing).
// Triangle records are 12 dwords (three float4: vertex xyz, and the original
// id in the first record's w).  One coalesced load puts dword j of up to five
// consecutive records on lane j; v_readlane then hands each record to the
// scalar unit.  A leaf of n triangles costs ceil(n / 5) dependent memory round
// trips instead of n, and the tested values are the same bits.
__device__ __forceinline__ void test_leaf_wave(const float4* tris, int32_t code, const RayPre& rp, Hit& h) {
  constexpr uint32_t kPerLoad = 5;
  const uint32_t first = leaf_first(code);
  const uint32_t cnt = leaf_count(code);
  const int lane = (int)(threadIdx.x & 63);
  const int* words = reinterpret_cast<const int*>(tris + 3 * (size_t)first);
  for (uint32_t q0 = 0; q0 < cnt; q0 += kPerLoad) {
    const uint32_t m = cnt - q0 < kPerLoad ? cnt - q0 : kPerLoad;
    const int v = lane < (int)(12 * m) ? words[12 * (size_t)q0 + lane] : 0;
    for (uint32_t q = 0; q < m; ++q) {
      const int o = (int)(12 * q);
      const V3 a = v3(__int_as_float(__builtin_amdgcn_readlane(v, o + 0)),
                      __int_as_float(__builtin_amdgcn_readlane(v, o + 1)),
                      __int_as_float(__builtin_amdgcn_readlane(v, o + 2)));
      const uint32_t id = (uint32_t)__builtin_amdgcn_readlane(v, o + 3);
      const V3 b = v3(__int_as_float(__builtin_amdgcn_readlane(v, o + 4)),
                      __int_as_float(__builtin_amdgcn_readlane(v, o + 5)),
                      __int_as_float(__builtin_amdgcn_readlane(v, o + 6)));
      const V3 c = v3(__int_as_float(__builtin_amdgcn_readlane(v, o + 8)),
                      __int_as_float(__builtin_amdgcn_readlane(v, o + 9)),
                      __int_as_float(__builtin_amdgcn_readlane(v, o + 10)));
      float t, vv, ww, det;
      if (intersect_triangle_raw(rp, a, b, c, &t, &vv, &ww, &det)) {
        if (t < h.t || (t == h.t && id < h.id)) {
          h.t = t;
          h.b1 = vv;
          h.b2 = ww;
          h.det = det;
          h.k = first + q0 + q;
          h.id = id;
        }
      }
    }
  }
}

// Inserts (key, child) into the list of the first n entries of (keys,
// children), kept in increasing key order; among equal keys the earlier
// insertion stays first.  Every index is a compile-time constant, so the
// lists stay in registers (scalar registers when the values are
// wave-uniform): a list indexed by a run-time count would be placed in scratch.
template <typename K>
__device__ __forceinline__ void sorted_insert(K (&keys)[kBvhWidth], int (&children)[kBvhWidth], int n, K key,
                                              int child) {
  int pos = 0;
#pragma unroll
  for (int i = 0; i < kBvhWidth; ++i) pos += (i < n && !(key < keys[i])) ? 1 : 0;
#pragma unroll
  for (int j = kBvhWidth - 1; j >= 0; --j) {
    const K below_k = j > 0 ? keys[j - 1] : key;
    const int below_c = j > 0 ? children[j - 1] : child;
    keys[j] = j < pos ? keys[j] : (j == pos ? key : below_k);
    children[j] = j < pos ? children[j] : (j == pos ? child : below_c);
  }
}

// Closest hit over the kBvhWidth-wide BVH.  `stack` points at this lane's column of
// an LDS array laid out [depth][blockDim.x].  The result is independent of
// the traversal order: the (t, id) pair is minimised lexicographically.  At a
// node, the entry distances of all child boxes use the culling limit of
// the hit found before the node; the slots are taken in order: leaves are
// tested at once, internal children are visited nearest first (equal
// distances in slot order).
template <bool kStats, bool kParallel>
__device__ __forceinline__ void closest_hit_impl(const SceneView& S, const RayPre& rp, uint32_t* stack,
                                                 int stride, Hit& h, uint32_t* nodes_visited,
                                                 uint32_t* tris_tested) {
  h.t = rp.tmax;
  h.b1 = h.b2 = 0.0f;
  h.k = 0xffffffffu;
  h.id = 0xffffffffu;
  if (S.node_count == 0) return;
  int sp = 0;
  int node = 0;
  for (;;) {
    if (kStats) ++*nodes_visited;
    const float4* np = reinterpret_cast<const float4*>(S.nodes + node);
    const float limit = h.t * kCullSlack;
    int ni = 0;
    int ic[kBvhWidth];
    float it[kBvhWidth];
#pragma unroll
    for (int hf = 0; hf < kBvhHalves; ++hf) {
      const float4* q = np + 8 * hf;
      const float4 lx = q[0], hx = q[1], ly = q[2], hy = q[3], lz = q[4], hz = q[5];
      const int4 ch = reinterpret_cast<const int4*>(q)[6];
      float te[kHalfWidth];
      te[0] = slab_enter<kParallel>(rp, lx.x, hx.x, ly.x, hy.x, lz.x, hz.x, limit);
      te[1] = slab_enter<kParallel>(rp, lx.y, hx.y, ly.y, hy.y, lz.y, hz.y, limit);
      te[2] = slab_enter<kParallel>(rp, lx.z, hx.z, ly.z, hy.z, lz.z, hz.z, limit);
      te[3] = slab_enter<kParallel>(rp, lx.w, hx.w, ly.w, hy.w, lz.w, hz.w, limit);
      const int32_t cc[kHalfWidth] = {ch.x, ch.y, ch.z, ch.w};
#pragma unroll
      for (int s = 0; s < kHalfWidth; ++s) {
        const int32_t c = cc[s];
        if (c == kChildEmpty || !(te[s] < INFINITY)) continue;
        if (child_is_leaf(c)) {
          if (kStats) *tris_tested += leaf_count(c);
          test_leaf(S.tris, c, rp, h);
        } else {
          sorted_insert(it, ic, ni, te[s], c);
          ++ni;
        }
      }
    }
    if (ni == 0) {
      if (sp == 0) break;
      --sp;
      node = (int)stack[sp * stride];
      continue;
    }
    // internal children are in near-to-far order: push all but the nearest,
    // farthest first, and visit the nearest
#pragma unroll
    for (int a = kBvhWidth - 1; a >= 1; --a) {
      if (a < ni) {
        stack[sp * stride] = (uint32_t)ic[a];
        ++sp;
      }
    }
    node = ic[0];
  }
}

// Rays with an exactly axis-parallel direction take the variant with the
// parallel-slab rule; all others the plain slab test.
template <bool kStats = false>
__device__ __forceinline__ void closest_hit(const SceneView& S, const RayPre& rp, uint32_t* stack, int stride,
                                            Hit& h, uint32_t* nodes_visited = nullptr,
                                            uint32_t* tris_tested = nullptr) {
  if (rp.par != 0)
    closest_hit_impl<kStats, true>(S, rp, stack, stride, h, nodes_visited, tris_tested);
  else
    closest_hit_impl<kStats, false>(S, rp, stack, stride, h, nodes_visited, tris_tested);
  finish_hit(h);
}

__device__ __forceinline__ V3 shade(const float4* cols, const uint32_t* texels, const TexView* textures, int sky_mode,
                                    const Hit& h, float dx, float dy, float dz) {
  if (h.id == 0xffffffffu) return sky_colour(sky_mode, dx, dy, dz);
  const float4 c0 = cols[3 * (size_t)h.k + 0];
  const float4 c1 = cols[3 * (size_t)h.k + 1];
  const uint32_t word = __float_as_uint(c0.w);
  if (colour_mode(word) == kTextureColour) {
    const float uv[6] = {c0.x, c0.y, c0.z, c1.x, c1.y, c1.z};
    return shade_texture(h.b1, h.b2, uv, texels, textures[texture_index(word)]);
  }
  const float4 c2 = cols[3 * (size_t)h.k + 2];
  return shade_hit(h.b1, h.b2, v3(c0.x, c0.y, c0.z), v3(c1.x, c1.y, c1.z), v3(c2.x, c2.y, c2.z), word);
}
__device__ __forceinline__ V3 shade(const SceneView& S, const Hit& h, float dx, float dy, float dz) {
  return shade(S.cols, S.texels, S.textures, S.sky_mode, h, dx, dy, dz);
}

// Maps a ray number to (pose, ommatidium, sample, samples of that ommatidium).
__device__ __forceinline__ void locate_ray(const EyeLaunch& L, uint64_t r, int* pose, int* omm, int* sample,
                                           int* n) {
  const uint64_t p = r / L.rays_per_pose;
  const uint32_t local = (uint32_t)(r - p * L.rays_per_pose);
  *pose = (int)p;
  if (L.offsets == nullptr) {
    const int i = (int)(local / (uint32_t)L.spp);
    *omm = i;
    *sample = (int)(local - (uint32_t)i * (uint32_t)L.spp);
    *n = L.spp;
    return;
  }
  // last i with offsets[i] <= local (empty ommatidia are skipped naturally)
  int lo = 0, hi = L.omm_count - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (L.offsets[mid] <= local) lo = mid;
    else hi = mid - 1;
  }
  *omm = lo;
  *sample = (int)(local - L.offsets[lo]);
  *n = (int)(L.offsets[lo + 1] - L.offsets[lo]);
}

// ---------------------------------------------------------------------------
// Wave-packet traversal of the 4-wide tree (trace mode 1; trace mode 2, the
// default, walks the 64-wide tree, packet.h).  The 64 rays of a wave are
// samples of one or two neighbouring ommatidia: nearly the same origin and
// direction.  The wave walks the BVH together: the node index is wave-uniform, each
// lane tests the children against its own ray and closest hit, a child is
// entered when any lane's ray enters it, and every active lane tests the
// triangles of an entered leaf.  Each lane still computes the exact
// lexicographic (t, id) minimum over the triangles its ray can hit (a lane
// only ever visits a superset of the nodes its own traversal would), so
// results are identical to per-ray traversal whatever the visiting order.
//
// A step is one long chain of dependent instructions, so the step keeps off
// LDS: the wave's stack lives in two VGPRs, entry k in lane k & 63 of
// stack[k >> 6] (a lane select to push, v_readlane to pop; kPacketStackMax
// entries), and entered children are ordered nearest first by the entry
// distance of the first lane that enters them, read with v_readlane and
// compared as bits on the scalar unit (entry distances are >= tmin >= 0,
// where the float order is the integer order).
// ---------------------------------------------------------------------------
__device__ __forceinline__ void stack_push(int& s0, int& s1, int lane, int sp, int v) {
  if (sp < 64)
    s0 = lane == sp ? v : s0;
  else
    s1 = lane == sp - 64 ? v : s1;
}
__device__ __forceinline__ int stack_top(int s0, int s1, int sp) {
  return sp < 64 ? __builtin_amdgcn_readlane(s0, sp) : __builtin_amdgcn_readlane(s1, sp - 64);
}

// One node of a packet step: tests its leaf children (every lane, against
// its own ray) and appends the internal children that any lane enters to
// ic / ik (child, ordering key).
template <bool kParallel>
__device__ __forceinline__ void packet_visit(const SceneView& S, const RayPre& rp, bool active, int node, Hit& h,
                                             int (&ic)[kBvhWidth], uint32_t (&ik)[kBvhWidth], int& ni,
                                             uint32_t& tris) {
  // every slot's entry distance uses the culling limit of the hit found
  // before the node, also after the first half's leaves have been tested
  const float limit = h.t * kCullSlack;
#pragma unroll
  for (int hf = 0; hf < kBvhHalves; ++hf) {
    const float4* np = reinterpret_cast<const float4*>(S.nodes + node) + 8 * hf;
    const float4 lx = np[0], hx = np[1], ly = np[2], hy = np[3], lz = np[4], hz = np[5];
    const int4 ch = reinterpret_cast<const int4*>(np)[6];
    const float slo_x[kHalfWidth] = {lx.x, lx.y, lx.z, lx.w}, shi_x[kHalfWidth] = {hx.x, hx.y, hx.z, hx.w};
    const float slo_y[kHalfWidth] = {ly.x, ly.y, ly.z, ly.w}, shi_y[kHalfWidth] = {hy.x, hy.y, hy.z, hy.w};
    const float slo_z[kHalfWidth] = {lz.x, lz.y, lz.z, lz.w}, shi_z[kHalfWidth] = {hz.x, hz.y, hz.z, hz.w};
    const int32_t cc[kHalfWidth] = {ch.x, ch.y, ch.z, ch.w};
#pragma unroll
    for (int s = 0; s < kHalfWidth; ++s) {
      const int32_t c = cc[s];
      // the child word is wave-uniform: an empty slot is skipped on the
      // scalar unit before its slab test (the tree's empty slots are ~18 %)
      if (c == kChildEmpty) continue;
      const float te = slab_enter<kParallel>(rp, slo_x[s], shi_x[s], slo_y[s], shi_y[s], slo_z[s], shi_z[s], limit);
      const bool mine = active && te < INFINITY;
      if (__ballot(mine) == 0ull) continue;
      if (child_is_leaf(c)) {
        tris += leaf_count(c);
        // inactive lanes test a dummy ray whose result is discarded
        test_leaf_wave(S.tris, c, rp, h);
      } else {
        // order key: the entry distance of the first lane that enters the child
        const uint64_t m = __ballot(mine);
        const int lead = __builtin_amdgcn_readfirstlane(__ffsll((long long)m) - 1);
        const uint32_t key = (uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(te), lead);
        sorted_insert(ik, ic, ni, key, c);
        ++ni;
      }
    }
  }
}

// steps / tris count the packet's node visits and the triangles of the leaves
// it enters (wave-uniform: what the wave fetches from memory).
template <bool kParallel>
__device__ __forceinline__ void closest_hit_packet_impl(const SceneView& S, const RayPre& rp, bool active, Hit& h,
                                                        uint32_t& steps, uint32_t& tris) {
  int sp = 0;
  int node = 0;
  int stk0 = 0, stk1 = 0;
  const int lane = (int)(threadIdx.x & 63);
  for (;;) {
    node = __builtin_amdgcn_readfirstlane(node);
    int ni = 0;
    int ic[kBvhWidth];
    uint32_t ik[kBvhWidth];
    ++steps;
    packet_visit<kParallel>(S, rp, active, node, h, ic, ik, ni, tris);
    if (ni == 0) {
      if (sp == 0) break;
      --sp;
      node = stack_top(stk0, stk1, sp);
      continue;
    }
    // entered children are in near-to-far order: push all but the nearest,
    // farthest first, and visit the nearest
#pragma unroll
    for (int a = kBvhWidth - 1; a >= 1; --a) {
      if (a < ni) {
        stack_push(stk0, stk1, lane, sp, ic[a]);
        ++sp;
      }
    }
    node = ic[0];
  }
}

__device__ __forceinline__ void closest_hit_packet(const SceneView& S, const RayPre& rp, bool active, Hit& h,
                                                   uint32_t& steps, uint32_t& tris) {
  h.t = rp.tmax;
  h.b1 = h.b2 = 0.0f;
  h.k = 0xffffffffu;
  h.id = 0xffffffffu;
  if (S.node_count == 0) return;
  // The stack's entry k lives in lane k & 63, written by a lane select: a
  // lane outside EXEC would drop its entries.  Every caller enters with the
  // whole wave; a partial wave is flagged to the host, which discards the
  // launch's results, and returns misses instead of walking the tree.
  if (__ballot(1) != ~0ull) {
    if (S.fault) *S.fault = 1u;
    return;
  }
  if (__ballot(active && rp.par != 0) != 0ull)
    closest_hit_packet_impl<true>(S, rp, active, h, steps, tris);
  else
    closest_hit_packet_impl<false>(S, rp, active, h, steps, tris);
  finish_hit(h);
}

// The closest hits of a wave's rays by packet traversal kTrav; lds: the
// block's dynamic LDS (wide walk: a stack per wave).
template <int kTrav>
__device__ __forceinline__ void packet_hits(const SceneView& S, const Ray& ray, const RayPre& rp, bool active,
                                            uint32_t* lds, Hit& h, uint32_t& steps, uint32_t& tris) {
  if (kTrav == kUnitPacketWide) {
    uint2* stack = reinterpret_cast<uint2*>(lds) + (size_t)(threadIdx.x >> 6) * (size_t)S.wide.stack;
    closest_hit_wide(S.wide, ray, rp, active, stack, S.fault, h, steps, tris);
  } else {
    closest_hit_packet(S, rp, active, h, steps, tris);
  }
}

// The value of lane (lane ^ M), M a power of two below 64, without an
// address register: ds_swizzle in bit mode (and 0x1f, xor M) within each
// 32-lane half for M <= 16, and gfx950's v_permlane32_swap across the halves
// for M = 32.  __shfl_xor needs a (lane ^ M) * 4 address per mask, which the
// compiler computes once per kernel and keeps live (in the unit renderer, six
// of them spilled to scratch and reloaded in every round).
template <int M>
__device__ __forceinline__ uint32_t lane_xor(uint32_t v) {
  static_assert(M >= 1 && M <= 32 && (M & (M - 1)) == 0, "power of two below 64");
  if constexpr (M == 32) {
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return (threadIdx.x & 32u) ? r[0] : r[1];
  } else {
    return (uint32_t)__builtin_amdgcn_ds_swizzle((int)v, (M << 10) | 0x1f);
  }
}
template <int M>
__device__ __forceinline__ float lane_xor(float v) {
  return __uint_as_float(lane_xor<M>(__float_as_uint(v)));
}

__device__ __forceinline__ float wave_sum(float v) {
  v = v + lane_xor<32>(v);
  v = v + lane_xor<16>(v);
  v = v + lane_xor<8>(v);
  v = v + lane_xor<4>(v);
  v = v + lane_xor<2>(v);
  v = v + lane_xor<1>(v);
  return v;
}

// Segmented form of wave_sum: lanes [a, a + seg) with a a multiple of seg
// (a power of two) sum their values; lane a ends with the total.  For a unit
// whose samples occupy lanes a .. a + n - 1 (n <= seg, other lanes 0) this is
// bit-identical to wave_sum over a wave holding the same samples in lanes
// 0 .. n - 1: the butterfly steps with offset >= seg only add zeros there.
template <int M>
__device__ __forceinline__ float segment_step(float v, int seg) {
  const float w = lane_xor<M>(v);
  return M < seg ? v + w : v;
}
__device__ __forceinline__ float segment_sum(float v, int seg) {
  v = segment_step<32>(v, seg);
  v = segment_step<16>(v, seg);
  v = segment_step<8>(v, seg);
  v = segment_step<4>(v, seg);
  v = segment_step<2>(v, seg);
  v = segment_step<1>(v, seg);
  return v;
}

// Bitonic sort of one value per lane, largest first, across the 64 lanes.
template <int K, int J>
__device__ __forceinline__ uint32_t sort_step(uint32_t v, int lane) {
  const uint32_t o = lane_xor<J>(v);
  const bool take_max = ((lane & J) == 0) == ((lane & K) == 0);
  return take_max ? (o > v ? o : v) : (o < v ? o : v);
}
template <int K, int J>
__device__ __forceinline__ uint32_t sort_merge(uint32_t v, int lane) {
  v = sort_step<K, J>(v, lane);
  if constexpr (J > 1) v = sort_merge<K, J / 2>(v, lane);
  return v;
}
__device__ __forceinline__ uint32_t wave_sort_desc(uint32_t v) {
  const int lane = (int)(threadIdx.x & 63);
  v = sort_merge<2, 1>(v, lane);
  v = sort_merge<4, 2>(v, lane);
  v = sort_merge<8, 4>(v, lane);
  v = sort_merge<16, 8>(v, lane);
  v = sort_merge<32, 16>(v, lane);
  v = sort_merge<64, 32>(v, lane);
  return v;
}

__device__ __forceinline__ int pow2_at_least(uint32_t n) {
  int s = 1;
  while ((uint32_t)s < n) s <<= 1;
  return s;
}

// Workgroups are handed to the 8 XCDs round-robin (block b to XCD b % 8),
// and each XCD has its own L2.  Logical blocks are therefore dealt to XCDs in
// runs of kXcdRun consecutive blocks: the processing order is the Morton order of the
// ommatidial axes, so an XCD's resident waves look in neighbouring directions
// and share BVH nodes in its L2, while runs still alternate between XCDs so
// that each gets its share of costly directions.  The mapping is a
// bijection, so results do not depend on it.
__device__ __forceinline__ uint32_t xcd_run_block(uint32_t b, uint32_t blocks, uint32_t run) {
  const uint32_t span = kXcds * run;
  if (b >= (blocks / span) * span) return b;
  const uint32_t x = b % kXcds, j = b / kXcds;
  return ((j / run) * kXcds + x) * run + j % run;
}

// Unit renderer.  A wave takes units_per_grab consecutive units of the
// processing order and renders them in rounds: a unit of more than 32 samples
// fills the wave alone (lane l takes samples l, l + 64, ...); smaller units are
// packed side by side into power-of-two lane segments, so the lanes of a
// wave stay busy when sample counts are small (adaptive pilots, uneven
// counts).  Each unit's colour is the same canonical sum either way.
//
// The workgroup dispatcher is the work queue: a grid has a wave per grab.  A
// persistent grid with atomic counters per XCD spent 0.6 of its 0.70 ms on
// those counters when 12,461 small units were rendered (all waves look
// through all slices before they exit).
//
// Packet variants: six waves per SIMD (at most 80 VGPRs); five and four are
// 4 and 13 % slower on the bee eye's batch.  The multi-pass instances spill at
// six (68 bytes of scratch per lane, 84 with statistics; the uneven batch
// writes 42 GB for 0.33 GB of colours), at five 8 and 16 bytes, at four none,
// and are faster all the same: uneven batch 60.4 ms, 61.4 at five and 68.0 at
// four; adaptive renders of the bee eye 13.0, 13.6 and 14.7, of 2.1 M
// ommatidia 20.1, 20.6 and 22.0.  The per-ray variant's LDS stack
// columns allow few resident blocks anyway; four waves (128 VGPRs) keep its
// traversal loop free of scratch.
//
// What a round needs after the walk is read anew from the kernel arguments
// (fresh_args): held in scalar registers across it, the arguments spill.
//
// kOnePass: every unit has the same count of at most 64 samples, so a round's
// lanes trace once, the sums need no registers across the traversal, and the
// segments need no packing.
// Packet workgroups are one wave: waves of uneven work then leave no slot idle
// until their workgroup's last one ends (against four waves: bee eye's batch
// 17.8 -> 16.0 ms, uneven batch 71.1 -> 63.6).
constexpr int unit_threads(int traversal) { return traversal == kUnitPerRay ? kTraceThreads : 64; }

struct RenderArgs {
  SceneView S;
  UnitLaunch U;
  Pose pose;            // the one pose when U.poses is null
  uint32_t omm_magic;   // floor(2^32 / omm_count), at most 2^32 - 1
  uint32_t blocks;      // workgroups of work; the grid strides over them
  uint32_t run;         // consecutive ones on one XCD
  // split launches: chunks per unit and the reciprocal of split_unit, tasks, 1 / spp
  uint32_t chunks, chunk_magic, tasks;
  float inv;
  uint32_t ways_log;   // packet tasks: log2 of the waves a task's rays are dealt to
};
typedef __attribute__((address_space(4))) const RenderArgs KernelArgs;

__device__ __forceinline__ KernelArgs* fresh_args() {
  KernelArgs* p = (KernelArgs*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return p;
}

__device__ __forceinline__ Pose pose_of(KernelArgs* K, uint32_t p) {
  if (K->U.poses) return K->U.poses[p];
  Pose P;
  for (int a = 0; a < 3; ++a) {
    P.pos[a] = K->pose.pos[a];
    P.x[a] = K->pose.x[a];
    P.y[a] = K->pose.y[a];
    P.z[a] = K->pose.z[a];
  }
  return P;
}

// What a traversal needs of the scene.
__device__ __forceinline__ SceneView walk_view(KernelArgs* K) {
  SceneView S;
  S.nodes = K->S.nodes;
  S.tris = K->S.tris;
  S.wide = WideTree{K->S.wide.nodes, K->S.wide.tris, K->S.wide.root, K->S.wide.stack, K->S.wide.spread,
                    K->S.wide.range, K->S.wide.least};
  S.node_count = K->S.node_count;
  S.fault = K->S.fault;
  return S;
}

// Pose and place in the processing order of unit u: u / omm_count by the
// magic reciprocal, whose estimate is exact or one too small.
__device__ __forceinline__ void split_unit(uint32_t u, uint32_t n, uint32_t magic, uint32_t* p, uint32_t* k) {
  uint32_t q = __umulhi(u, magic);
  uint32_t rest = u - q * n;
  if (rest >= n) {
    ++q;
    rest -= n;
  }
  *p = q;
  *k = rest;
}

template <bool kStats, bool kSamples, int kTrav, bool kOnePass = false>
__global__ __launch_bounds__(unit_threads(kTrav), kTrav == kUnitPerRay ? 4 : 6) void k_render_units(RenderArgs A) {
  // LDS: per-ray traversal a stack column per lane, laid out
  // [depth][blockDim.x]; wide packets a stack per wave
  extern __shared__ uint32_t unit_lds[];
  const int lane = threadIdx.x & 63;
  uint32_t* lane_stack = unit_lds + threadIdx.x;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t units = (uint32_t)((uint64_t)A.U.pose_count * (uint64_t)A.U.omm_count);
  uint32_t w_steps = 0, w_tris = 0;   // packet node fetches and leaf triangles of this wave
  for (uint32_t b = blockIdx.x; b < fresh_args()->blocks; b += gridDim.x) {
    const uint32_t G0 = (uint32_t)fresh_args()->U.units_per_grab;
    const uint64_t first = (uint64_t)(xcd_run_block(b, fresh_args()->blocks, fresh_args()->run) *
                                          (unit_threads(kTrav) / 64) + wave) * G0;
    if (first >= units) continue;   // whole wave
    const uint32_t base = (uint32_t)first;
    const int G = (int)min(G0, units - base);
    // lane g < G holds the sample count of a unit; rounds take the grab's
    // units largest first, so that power-of-two segments tile the 64 lanes
    // without gaps.  Sorted position q holds unit offset order[q] (units above
    // 32 samples, which fill whole rounds, compare equal).
    uint32_t my_n = 0;
    int order = lane;
    if (!kOnePass) {
      KernelArgs* K = fresh_args();
      if (lane < G) {
        uint32_t p, k;
        split_unit(base + (uint32_t)lane, (uint32_t)K->U.omm_count, K->omm_magic, &p, &k);
        const uint32_t i = K->U.order ? K->U.order[k] : k;
        my_n = K->U.unit_counts ? K->U.unit_counts[p * (uint32_t)K->U.omm_count + i]
                                : K->U.omm_counts ? K->U.omm_counts[i] : (uint32_t)K->U.spp;
      }
      const uint32_t key = wave_sort_desc(lane < G ? ((min(my_n, 64u) + 1u) << 6) | (uint32_t)lane : 0u);
      order = (int)(key & 63u);
      my_n = (uint32_t)__shfl((int)my_n, order);
    }
    int g = 0;
    while (g < G) {
      // ---- build a round: which unit (slot) each lane serves ----
      int slot = -1, seg_off = 0, seg = 64;
      int g_end = g + 1;
      uint32_t n;
      if (kOnePass) {
        n = (uint32_t)fresh_args()->U.spp;
        const int log_seg = n <= 1u ? 0 : 32 - __builtin_clz(n - 1u);
        seg = 1 << log_seg;
        slot = g + (lane >> log_seg);
        seg_off = lane & ~(seg - 1);
        g_end = min(G, g + (64 >> log_seg));
        if (slot >= G) slot = -1;
      } else {
        const uint32_t n_first = (uint32_t)__builtin_amdgcn_readlane((int)my_n, g);
        if (n_first > 32u) {
          slot = g;
        } else {
          int cursor = 0;
          g_end = g;
          while (g_end < G) {
            const uint32_t nj = (uint32_t)__builtin_amdgcn_readlane((int)my_n, g_end);
            if (nj > 32u) break;
            const int sj = pow2_at_least(nj);
            const int a = (cursor + sj - 1) & ~(sj - 1);
            if (a + sj > 64) break;
            if (lane >= a && lane < a + sj) {
              slot = g_end;
              seg_off = a;
              seg = sj;
            }
            cursor = a + sj;
            ++g_end;
          }
        }
        n = (uint32_t)__shfl((int)my_n, slot < 0 ? 0 : slot);   // every lane takes part
      }
      // ---- this lane's unit ----
      const int unit_off = kOnePass ? max(slot, 0) : __shfl(order, slot < 0 ? 0 : slot);
      if (slot < 0) n = 0u;
      uint32_t p, i;
      {
        KernelArgs* K = fresh_args();
        split_unit(base + (uint32_t)unit_off, (uint32_t)K->U.omm_count, K->omm_magic, &p, &i);
        if (K->U.order) i = K->U.order[i];
      }
      // The lane's place in the round, the one register of round bookkeeping
      // kept across the traversal: bit 16 set when the lane serves a unit,
      // bits 8-10 log2 of its segment, bits 0-6 the lane's first sample in
      // its unit (lane - segment start).
      const uint32_t desc = (slot >= 0 ? 0x10000u : 0u) | ((uint32_t)__builtin_ctz((unsigned)seg) << 8) |
                            (uint32_t)(lane - seg_off);
      float r = 0.0f, gg = 0.0f, bl = 0.0f;
      float sr = 0.0f, sg = 0.0f, sb = 0.0f, sd = 0.0f, sd2 = 0.0f, sh = 0.0f;
      for (uint32_t c0 = 0; __ballot(c0 + (desc & 127u) < n) != 0ull; c0 += 64u) {
        const bool active = c0 + (desc & 127u) < n;
        Ray ray;
        if (active) {
          KernelArgs* K = fresh_args();
          const U4 rnd = sample_randoms(K->U.seed, K->U.eye, i, K->U.sample_base + c0 + (desc & 127u), K->U.frame,
                                        K->U.pose_base + p);
          ray = generate_ray(K->U.cones[i], pose_of(K, p), rnd);
        } else {
          ray.ox = ray.oy = ray.oz = 0.0f;
          ray.dx = ray.dy = 0.0f;
          ray.dz = 1.0f;
          ray.tmin = 0.0f;
          ray.tmax = 1.0f;
        }
        Hit h;
        {
          KernelArgs* K = fresh_args();
          const SceneView S = walk_view(K);
          const RayPre rp = precompute_ray(ray);
          if (kTrav == kUnitPerRay) {
            h.t = rp.tmax;
            h.k = h.id = 0xffffffffu;
            h.b1 = h.b2 = 0.0f;
            if (active) closest_hit(S, rp, lane_stack, (int)blockDim.x, h);
          } else {
            packet_hits<kTrav>(S, ray, rp, active, unit_lds, h, w_steps, w_tris);
          }
        }
        if (active) {
          KernelArgs* K = fresh_args();
          const V3 c = shade(K->S.cols, K->S.texels, K->S.textures, K->S.sky_mode, h, ray.dx, ray.dy, ray.dz);
          const float inv = 1.0f / (float)n;
          r = r + c.x * inv;
          gg = gg + c.y * inv;
          bl = bl + c.z * inv;
          const bool hit = h.id != 0xffffffffu;
          if (kSamples)
            K->U.samples[K->U.sample_offsets[p * (uint32_t)K->U.omm_count + i] + c0 + (desc & 127u)] =
                make_float4(c.x, c.y, c.z, hit ? h.t : -1.0f);
          if (kStats) {
            sr += c.x * c.x;
            sg += c.y * c.y;
            sb += c.z * c.z;
            const float idp = hit ? 1.0f / (1.0f + h.t) : 0.0f;
            sd += idp;
            sd2 += idp * idp;
            sh += hit ? 1.0f : 0.0f;
          }
        }
        if (kOnePass) break;
      }
      const int seg_len = 1 << ((desc >> 8) & 7u);
      r = segment_sum(r, seg_len);
      gg = segment_sum(gg, seg_len);
      bl = segment_sum(bl, seg_len);
      if (kStats) {
        sr = segment_sum(sr, seg_len);
        sg = segment_sum(sg, seg_len);
        sb = segment_sum(sb, seg_len);
        sd = segment_sum(sd, seg_len);
        sd2 = segment_sum(sd2, seg_len);
        sh = segment_sum(sh, seg_len);
      }
      if ((desc & 0x1007fu) == 0x10000u) {   // the first lane of a unit's segment
        KernelArgs* K = fresh_args();
        const uint32_t out = p * (uint32_t)K->U.omm_count + i;
        K->U.colours[out] = make_float4(r, gg, bl, (float)n);
        if (kStats) {
          // E[c^2] - E[c]^2 with E[c] the unit's mean colour
          const float inv = 1.0f / (float)(n > 0u ? n : 1u);
          const float vr = fmaxf(sr * inv - r * r, 0.0f);
          const float vg = fmaxf(sg * inv - gg * gg, 0.0f);
          const float vb = fmaxf(sb * inv - bl * bl, 0.0f);
          const float md = sd * inv;
          K->U.stats[2 * (size_t)out] = make_float4(vr, vg, vb, sh * inv);
          K->U.stats[2 * (size_t)out + 1] = make_float4(md, fmaxf(sd2 * inv - md * md, 0.0f), 0.0f, 0.0f);
        }
      }
      g = g_end;
    }
  }
  unsigned long long* counts = fresh_args()->U.packet_counts;
  if (counts && lane == 0 && w_steps != 0u) {
    atomicAdd(counts, (unsigned long long)w_steps);
    atomicAdd(counts + 1, (unsigned long long)w_tris);
  }
}

// Split launch of one pose's units with a uniform sample count n: task t is
// chunk t % C of unit t / C of the processing order (C = ceil(n / 64)), so
// that a single pose's few units still fill the GPU.  A wave traces one
// task; lane l keeps the scaled colour of its one sample in `partial` (three
// planes of 64 floats per task), and k_reduce_tasks adds a unit's chunks lane
// by lane in chunk order and then across the wave, which gives the same sums
// as k_render_units (there a lane adds samples l, l + 64, ... in this order).
//
// Two kernels, because completing units inside the task kernel (a counter
// per unit, behind a device-scope fence per task that writes back the XCD's
// L2) cost more than the traversal: 1,000 ommatidia x 3,200 samples 1.19 ms
// in the task kernel against 0.17 and 0.012 in the two, 1 sample 53 against
// 23 us.
//
// A unit of one chunk needs no partial sums: its wave writes the colour.  Where
// the frame shows ommatidium x in pixel x of its first row, the wave that
// knows a colour writes its pixel too (`frame`, `frame_width`).
//
// Why no persistent task loop: a loop whose body takes its task from a lane-0
// atomic broadcast with __shfl and ends in lane-0-only stores is compiled
// with the lane-0 branch leaving the loop on its own; the other 63 lanes
// then go round without lane 0, read 0 from the broadcast (a permute from a
// disabled lane) and, for C = 1, never leave.  Every wave here runs
// straight through, and its lane-dependent branches rejoin before the next
// cross-lane operation.
__device__ __forceinline__ uchar4 make_color(float4 c) {
  return make_uchar4(encode_channel(c.x), encode_channel(c.y), encode_channel(c.z), 255);
}

// Lane 0: the unit's colour, and its pixel.
__device__ __forceinline__ void put_unit(KernelArgs* K, uint32_t i, float r, float g, float b) {
  const float4 c = make_float4(r, g, b, (float)(uint32_t)K->U.spp);
  K->U.colours[i] = c;
  if (K->U.host_colours) K->U.host_colours[i] = c;
  if (K->U.frame_pixels && i < (uint32_t)K->U.frame_width) {
    const uchar4 pixel = make_color(c);
    K->U.frame_pixels[i] = pixel;
    if (K->U.host_pixels) K->U.host_pixels[i] = pixel;
  }
}

constexpr uint32_t kTaskFloats = 3 * 64;   // of `partial`, per task

__device__ __forceinline__ void put_partial(KernelArgs* K, uint32_t t, int lane, float r, float g, float b) {
  float* slot = K->U.chunk_partial + (size_t)t * kTaskFloats + lane;
  slot[0] = r;
  slot[64] = g;
  slot[128] = b;
}

// One wave per unit: bound by reading 12 bytes per sample.
__global__ __launch_bounds__(kTraceThreads) void k_reduce_tasks(RenderArgs A) {
  const int lane = threadIdx.x & 63;
  const uint32_t u = blockIdx.x * (kTraceThreads / 64) + (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  if (u >= (uint32_t)A.U.omm_count) return;   // whole wave
  const uint32_t n = (uint32_t)A.U.spp, chunks = A.chunks;
  const float* src = A.U.chunk_partial + (size_t)u * chunks * kTaskFloats + lane;
  float r = 0.0f, g = 0.0f, b = 0.0f;
  const uint32_t whole = n / 64u;   // chunks in which this lane has a sample, the last one apart
  uint32_t q = 0;
  for (; q + 8u <= whole; q += 8u) {
    float v[8][3];
#pragma unroll
    for (int k = 0; k < 8; ++k)
#pragma unroll
      for (int c = 0; c < 3; ++c) v[k][c] = src[(size_t)(q + k) * kTaskFloats + 64 * c];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      r = r + v[k][0];
      g = g + v[k][1];
      b = b + v[k][2];
    }
  }
  for (; q < chunks; ++q)
    if (q * 64u + (uint32_t)lane < n) {
      r = r + src[(size_t)q * kTaskFloats];
      g = g + src[(size_t)q * kTaskFloats + 64];
      b = b + src[(size_t)q * kTaskFloats + 128];
    }
  r = segment_sum(r, 64);
  g = segment_sum(g, 64);
  b = segment_sum(b, 64);
  if (lane == 0) put_unit(fresh_args(), A.U.order ? A.U.order[u] : u, r, g, b);
}

// The rays of a task one per lane (an LDS stack column per lane): lanes past n
// skip the traversal.
template <bool kSamples>
__global__ __launch_bounds__(kTraceThreads, 5) void k_render_chunks(RenderArgs A) {
  extern __shared__ uint32_t lane_stacks[];
  const int lane = threadIdx.x & 63;
  const uint32_t t = xcd_run_block(blockIdx.x, gridDim.x, 16u) * (kTraceThreads / 64) +
                     (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  if (t >= A.tasks) return;  // whole wave
  uint32_t u, j;
  split_unit(t, A.chunks, A.chunk_magic, &u, &j);
  const uint32_t i = A.U.order ? A.U.order[u] : u;
  const uint32_t s = j * 64u + (uint32_t)lane;
  float r = 0.0f, g = 0.0f, b = 0.0f;
  if (s < (uint32_t)A.U.spp) {
    const U4 rnd = sample_randoms(A.U.seed, A.U.eye, i, A.U.sample_base + s, A.U.frame, A.U.pose_base);
    const Ray ray = generate_ray(A.U.cones[i], A.pose, rnd);
    const RayPre rp = precompute_ray(ray);
    Hit h;
    closest_hit(A.S, rp, lane_stacks + threadIdx.x, (int)blockDim.x, h);
    const V3 c = shade(A.S, h, ray.dx, ray.dy, ray.dz);
    r = c.x * A.inv;
    g = c.y * A.inv;
    b = c.z * A.inv;
    if (kSamples)
      A.U.samples[A.U.sample_offsets[i] + s] = make_float4(c.x, c.y, c.z, h.id != 0xffffffffu ? h.t : -1.0f);
  }
  put_partial(fresh_args(), t, lane, r, g, b);
}

// Which of 2^ways_log waves traces a sample: by its azimuth about the axis (the
// sign of the splay, then the spin), so that a wave's rays share a sector of
// the cone; by lane when no more than a ray is left for each (count_log: bits
// of the task's ray count).
__device__ __forceinline__ uint32_t cone_sector(const U4& rnd, uint32_t ways_log, uint32_t count_log, int lane) {
  if (ways_log == 0u) return 0u;
  if (ways_log + 1u >= count_log) return (uint32_t)lane & ((1u << ways_log) - 1u);
  // a Box-Muller cosine is negative in the second and third quarter turn
  const uint32_t back = ((rnd.b >> 30) + 1u) >> 1 & 1u;
  return ways_log == 1u ? back : back << (ways_log - 1u) | rnd.c >> (33u - ways_log);
}

// The rays of a task as one packet, in workgroups of one wave.  kSplit: the
// launch records its tasks' packet steps and, with a list from the last
// launch's (split_flag), traces the listed tasks first, as several packets.
template <bool kSamples, int kTrav, bool kSplit>
__global__ __launch_bounds__(64, 6) void k_render_tasks(RenderArgs A) {
  extern __shared__ uint32_t task_lds[];
  const int lane = threadIdx.x & 63;
  const uint32_t wv = xcd_run_block(blockIdx.x, gridDim.x, 64u);
  // With a long-task split the first kSplitSubWaves waves trace the listed
  // tasks: 4 waves per tier-0 task (wave w: part w % 4 of tier-0 task w / 4),
  // then 2 per tier-1 task, then one per tier-2 task (whole); the rest every
  // other task in order.
  const bool split = kSplit && A.U.split_flag != nullptr;
  const uint32_t sub_waves = split ? (uint32_t)kSplitSubWaves : 0u;
  uint32_t t;
  int part = -1, ways = 1;
  if (wv < sub_waves) {
    constexpr uint32_t r0 = 4u * kSplit4Max, r1 = r0 + 2u * kSplit2Max;
    uint32_t tier, k, first;
    if (wv < r0) {
      tier = 0u;
      k = wv >> 2;
      part = (int)(wv & 3u);
      ways = 4;
      first = 0u;
    } else if (wv < r1) {
      tier = 1u;
      k = (wv - r0) >> 1;
      part = (int)((wv - r0) & 1u);
      ways = 2;
      first = kSplit4Max;
    } else {
      tier = 2u;
      k = wv - r1;
      first = kSplit4Max + kSplit2Max;
    }
    const uint32_t listed = (uint32_t)__builtin_amdgcn_readfirstlane((int)A.U.split_count[tier]);
    if (k >= listed) return;  // whole wave
    t = (uint32_t)__builtin_amdgcn_readfirstlane((int)A.U.split_list[first + k]);
  } else {
    t = (wv - sub_waves) >> A.ways_log;
    if (t >= A.tasks) return;  // whole wave
    if (split && __builtin_amdgcn_readfirstlane((int)A.U.split_flag[t]) != 0) return;  // traced listed
  }
  uint32_t u, j;
  split_unit(t, A.chunks, A.chunk_magic, &u, &j);
  const uint32_t i = (uint32_t)__builtin_amdgcn_readfirstlane((int)(A.U.order ? A.U.order[u] : u));
  const uint32_t s = j * 64u + (uint32_t)lane;
  const bool active = s < (uint32_t)A.U.spp;
  Ray ray;
  uint32_t sector = 0;
  if (active) {
    const U4 rnd = sample_randoms(A.U.seed, A.U.eye, i, A.U.sample_base + s, A.U.frame, A.U.pose_base);
    ray = generate_ray(A.U.cones[i], A.pose, rnd);
    sector = cone_sector(rnd, A.ways_log, 32 - __builtin_clz(min(64u, (uint32_t)A.U.spp) | 1u), lane);
  } else {
    ray.ox = ray.oy = ray.oz = 0.0f;
    ray.dx = ray.dy = 0.0f;
    ray.dz = 1.0f;
    ray.tmin = 0.0f;
    ray.tmax = 1.0f;
  }
  // A split packet traces the lanes whose rays rank part * 64 / ways ..
  // (part + 1) * 64 / ways - 1 by elevation (the direction's y, ties by
  // lane): rays of neighbouring elevation fan out less than the whole chunk.
  bool mine = active;
  const bool dealt = !kSplit && A.ways_log != 0u;
  if (dealt) {
    mine = active && sector == (wv & ((1u << A.ways_log) - 1u));
    if (__ballot(mine) == 0ull) return;
  }
  if (part >= 0) {
    const uint32_t bits = __float_as_uint(ray.dy);
    const uint32_t key = ((bits & 0x80000000u) ? ~bits : (bits | 0x80000000u)) & ~63u;
    const uint32_t sorted = wave_sort_desc(key | (uint32_t)lane);
    // sorted position q holds lane (sorted & 63): send q back to that lane
    const int rank = __builtin_amdgcn_ds_permute((int)((sorted & 63u) * 4u), lane);
    mine = active && (rank >> (ways == 4 ? 4 : 5)) == part;
  }
  Hit h;
  uint32_t w_steps = 0, w_tris = 0;
  {
    const SceneView S = walk_view(fresh_args());
    packet_hits<kTrav>(S, ray, precompute_ray(ray), mine, task_lds, h, w_steps, w_tris);
  }
  KernelArgs* K = fresh_args();
  if (K->U.packet_counts && lane == 0) {
    atomicAdd(K->U.packet_counts, (unsigned long long)w_steps);
    atomicAdd(K->U.packet_counts + 1, (unsigned long long)w_tris);
  }
  if (kSplit && K->U.split_cost && lane == 0) atomicAdd(K->U.split_cost + t, w_steps);
  float r = 0.0f, g = 0.0f, b = 0.0f;
  if (mine) {
    const V3 c = shade(K->S.cols, K->S.texels, K->S.textures, K->S.sky_mode, h, ray.dx, ray.dy, ray.dz);
    r = c.x * K->inv;
    g = c.y * K->inv;
    b = c.z * K->inv;
    if (kSamples)
      K->U.samples[K->U.sample_offsets[i] + s] = make_float4(c.x, c.y, c.z, h.id != 0xffffffffu ? h.t : -1.0f);
  }
  if (!kSplit && K->chunks == 1u && !dealt) {
    // the unit's only chunk
    r = segment_sum(0.0f + r, 64);
    g = segment_sum(0.0f + g, 64);
    b = segment_sum(0.0f + b, 64);
    if (lane == 0) put_unit(K, i, r, g, b);
    return;
  }
  // a split packet writes its own lanes' terms; the other packets of its
  // task write the rest
  if ((part < 0 && !dealt) || mine) put_partial(K, t, lane, r, g, b);
}

// Failure-handling probe of the packet traversal's partial-wave guard: one
// wave traces 64 rays, lanes at or above active_lanes skip the call (their
// ids stay 0xfffffffe).
template <int kTrav>
__global__ __launch_bounds__(64) void k_packet_guard_probe(SceneView S, const Ray* __restrict__ rays,
                                                           int active_lanes, int32_t* __restrict__ ids) {
  extern __shared__ uint32_t probe_lds[];
  const int lane = (int)(threadIdx.x & 63);
  Hit h;
  h.id = 0xfffffffeu;
  if (lane < active_lanes) {
    const Ray ray = rays[lane];
    uint32_t steps = 0, tris = 0;
    packet_hits<kTrav>(S, ray, precompute_ray(ray), true, probe_lds, h, steps, tris);
  }
  ids[lane] = (int32_t)h.id;
}

// Long-task split plan, one workgroup launched before the task kernel: it
// takes a histogram of the last
// launch's per-task packet steps (bins of 8 steps, the last one open), and
// picks each tier's threshold: the smallest multiple of 8 steps at or above
// the tier's minimum with at most the tiers' combined room (tier 0: 128
// tasks, tiers 0-1: 1,024, tiers 0-2: 3,072) at or above it (none when even
// the open top bin holds more).  It lists the tasks by tier and flags them,
// and clears every task's step count for this launch to fill in.
constexpr int kSplitPlanThreads = 1024;
constexpr int kSplitPlanPer = 16;   // step counts a thread holds at once
static_assert(kSplitBins <= kSplitPlanThreads, "one thread per histogram bin");

__device__ __forceinline__ uint32_t split_threshold(uint32_t over, uint32_t min_steps) {
  const uint32_t b = max(over, min_steps / 8u);
  return b >= (uint32_t)kSplitBins ? 0xffffffffu : b * 8u;
}

__global__ __launch_bounds__(kSplitPlanThreads) void k_split_plan(uint32_t* __restrict__ cost, uint64_t tasks,
                                                                   uint32_t* __restrict__ flag,
                                                                   uint32_t* __restrict__ list,
                                                                   uint32_t* __restrict__ count) {
  __shared__ uint32_t hist[kSplitBins];
  __shared__ uint32_t listed[3];
  const uint32_t tid = threadIdx.x;
  for (uint32_t b = tid; b < (uint32_t)kSplitBins; b += kSplitPlanThreads) hist[b] = 0u;
  if (tid < 3u) listed[tid] = 0u;
  __syncthreads();
  // a round's loads are all issued before its histogram updates; only tasks
  // of at least kSplitEarlyMinSteps enter the histogram (shorter ones are
  // never listed, and the threshold searches start there or above)
  const uint64_t per_round = (uint64_t)kSplitPlanThreads * kSplitPlanPer;
  uint32_t c[kSplitPlanPer];
  for (uint64_t base = 0; base < tasks; base += per_round) {
#pragma unroll
    for (int k = 0; k < kSplitPlanPer; ++k) {
      const uint64_t t = base + (uint64_t)k * kSplitPlanThreads + tid;
      c[k] = t < tasks ? cost[t] : 0u;
    }
#pragma unroll
    for (int k = 0; k < kSplitPlanPer; ++k)
      if (c[k] >= kSplitEarlyMinSteps) atomicAdd(&hist[min(c[k] / 8u, (uint32_t)kSplitBins - 1u)], 1u);
  }
  __syncthreads();
  // suffix counts S[b] = tasks in bins b .. kSplitBins - 1 fall as b grows,
  // so the bins with S[b] above a room are a prefix of the bins
  for (uint32_t off = 1; off < (uint32_t)kSplitBins; off <<= 1) {
    const uint32_t v = tid + off < (uint32_t)kSplitBins ? hist[tid + off] : 0u;
    __syncthreads();
    if (tid < (uint32_t)kSplitBins) hist[tid] += v;
    __syncthreads();
  }
  const bool bin = tid < (uint32_t)kSplitBins;
  const uint32_t over0 = (uint32_t)__syncthreads_count(bin && hist[tid] > (uint32_t)kSplit4Max);
  const uint32_t over1 = (uint32_t)__syncthreads_count(bin && hist[tid] > (uint32_t)(kSplit4Max + kSplit2Max));
  const uint32_t over2 = (uint32_t)__syncthreads_count(bin && hist[tid] > (uint32_t)kSplitListMax);
  const uint32_t th0 = split_threshold(over0, kSplitMinSteps);
  const uint32_t th1 = split_threshold(over1, kSplitMinSteps);
  const uint32_t th2 = split_threshold(over2, kSplitEarlyMinSteps);
  for (uint64_t base = 0; base < tasks; base += per_round) {
    if (tasks > per_round) {   // one round: the step counts are still held
#pragma unroll
      for (int k = 0; k < kSplitPlanPer; ++k) {
        const uint64_t t = base + (uint64_t)k * kSplitPlanThreads + tid;
        c[k] = t < tasks ? cost[t] : 0u;
      }
    }
#pragma unroll
    for (int k = 0; k < kSplitPlanPer; ++k) {
      const uint64_t t = base + (uint64_t)k * kSplitPlanThreads + tid;
      if (t < tasks) {
        uint32_t f = 0u;
        const uint32_t tier = c[k] >= th0 ? 0u : c[k] >= th1 ? 1u : c[k] >= th2 ? 2u : 3u;
        if (tier < 3u) {
          const uint32_t room = tier == 0u ? kSplit4Max : tier == 1u ? kSplit2Max : kSplit1Max;
          const uint32_t first = tier == 0u ? 0u : tier == 1u ? kSplit4Max : kSplit4Max + kSplit2Max;
          const uint32_t slot = atomicAdd(&listed[tier], 1u);
          if (slot < room) {
            list[first + slot] = (uint32_t)t;
            f = tier + 1u;
          }
        }
        flag[t] = f;
        cost[t] = 0u;
      }
    }
  }
  __syncthreads();
  if (tid == 0) {
    count[0] = min(listed[0], (uint32_t)kSplit4Max);
    count[1] = min(listed[1], (uint32_t)kSplit2Max);
    count[2] = min(listed[2], (uint32_t)kSplit1Max);
    count[3] = th0;
    count[4] = th1;
    count[5] = th2;
  }
}

__global__ void k_fill_u32(uint32_t* __restrict__ p, uint32_t n, uint32_t v) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// Traversal work counters of the same rays (nodes visited, triangles tested),
// summed over the launch: the algorithmic memory traffic of the trace kernel.
__global__ __launch_bounds__(kTraceThreads) void k_trace_stats(SceneView S, EyeLaunch L, uint64_t total,
                                                               unsigned long long* __restrict__ totals) {
  extern __shared__ uint32_t lds_stack[];
  const uint64_t r = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  uint32_t nv = 0, nt = 0, hit = 0;
  if (r < total) {
    int p, i, s, n;
    locate_ray(L, r, &p, &i, &s, &n);
    const U4 rnd = sample_randoms(L.seed, L.eye, (uint32_t)i, (uint32_t)s, L.frame, L.pose_base + (uint32_t)p);
    const Ray ray = generate_ray(cone_of(L.omms[i]), L.poses[p], rnd);
    Hit h;
    closest_hit<true>(S, precompute_ray(ray), lds_stack + threadIdx.x, blockDim.x, h, &nv, &nt);
    hit = h.id != 0xffffffffu ? 1u : 0u;
  }
  unsigned long long a = nv, b = nt, c = hit;
  for (int m = 32; m >= 1; m >>= 1) {
    a += __shfl_xor(a, m);
    b += __shfl_xor(b, m);
    c += __shfl_xor(c, m);
  }
  if ((threadIdx.x & 63) == 0) {
    atomicAdd(&totals[0], a);
    atomicAdd(&totals[1], b);
    atomicAdd(&totals[2], c);
  }
}

// Once per upload of an eye: every ray of an ommatidium needs its cone, whose
// three divisions and two square roots took 100 of a ray's instructions
// (4,096 poses x 5,000 ommatidia of 8-256 samples 64.6 -> 59.9 ms).
__global__ void k_cones(const Ommatidium* __restrict__ omms, int n, Cone* __restrict__ cones) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) cones[i] = cone_of(omms[i]);
}

__global__ void k_generate_rays(EyeLaunch L, uint64_t total, Ray* __restrict__ rays) {
  const uint64_t r = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= total) return;
  int p, i, s, n;
  locate_ray(L, r, &p, &i, &s, &n);
  const U4 rnd = sample_randoms(L.seed, L.eye, (uint32_t)i, (uint32_t)s, L.frame, L.pose_base + (uint32_t)p);
  rays[r] = generate_ray(cone_of(L.omms[i]), L.poses[p], rnd);
}

__global__ __launch_bounds__(kTraceThreads) void k_trace_rays(SceneView S, const Ray* __restrict__ rays,
                                                              uint64_t n, int32_t* __restrict__ hit,
                                                              float* __restrict__ tbb) {
  extern __shared__ uint32_t lds_stack[];
  const uint64_t r = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  const RayPre rp = precompute_ray(rays[r]);
  Hit h;
  closest_hit(S, rp, lds_stack + threadIdx.x, blockDim.x, h);
  hit[r] = h.id == 0xffffffffu ? -1 : (int32_t)h.id;
  tbb[3 * r] = h.t;
  tbb[3 * r + 1] = h.b1;
  tbb[3 * r + 2] = h.b2;
}

// 2^log consecutive rays per one-wave workgroup, as packets of what of them is
// close together (free rays may point anywhere: a wide frustum around a few
// would walk far more than their own paths).  Rays without any order take a
// walk each, a box test per lane; a ray per lane in a tree of four children
// kept a wave of them until its longest ended, 350 us for any few.  Calls of
// traceRays, us, ray per lane / one ray per wave / 8: 500 rays in 2.2 M
// triangles 366 / 70 / 127, 5,000 511 / 172 / 228, 50,000 490 / 275 / 284,
// 300,007 1,253 / 1,181 / 1,183; in 19,602 triangles 500 146 / 53 / 71, 50,000
// 250 / 187 / 190, 300,007 728 / 844 / 808 (the one size where a ray per lane
// was faster; in the pieces of 131,072 rays that a call now makes of it, 638).
//
// Directions may have any length: beyond what the walk computes with (or where
// the distances' products come near subnormal numbers) they are scaled by a
// power of two, and the distances with them, exactly.
constexpr float kRaySlope = 0.0625f;
__device__ __forceinline__ int length_exponent(const Ray& ray) {
  const float big = fmaxf(fmaxf(fabsf(ray.dx), fabsf(ray.dy)), fabsf(ray.dz));
  return big < 0x1p-70f || big > 0x1p60f ? __builtin_amdgcn_frexp_expf(big) : 0;
}
__global__ __launch_bounds__(64, 6) void k_trace_packets(SceneView S, const Ray* __restrict__ rays, uint64_t n, int log,
                                                         int32_t* __restrict__ hit, float* __restrict__ tbb) {
  extern __shared__ uint32_t ray_lds[];
  const int lane = (int)(threadIdx.x & 63);
  const uint64_t r = ((uint64_t)blockIdx.x << log) + (uint64_t)lane;
  const bool inside = (lane >> log) == 0 && r < n;
  Ray ray = rays[inside ? r : 0];
  const int e = length_exponent(ray);
  ray.dx = ldexpf(ray.dx, -e);
  ray.dy = ldexpf(ray.dy, -e);
  ray.dz = ldexpf(ray.dz, -e);
  ray.tmin = ldexpf(ray.tmin, e);
  ray.tmax = ldexpf(ray.tmax, e);
  Hit h;
  uint32_t steps = 0, tris = 0;
  closest_hit_wide(S.wide, ray, precompute_ray(ray), inside, reinterpret_cast<uint2*>(ray_lds), S.fault, h, steps,
                   tris, kRaySlope);
  if (!inside) return;
  const bool miss = h.id == 0xffffffffu;
  hit[r] = miss ? -1 : (int32_t)h.id;
  tbb[3 * r] = miss ? rays[r].tmax : ldexpf(h.t, -e);
  tbb[3 * r + 1] = h.b1;
  tbb[3 * r + 2] = h.b2;
}

// One pixel of a regular camera per thread: primary ray, closest hit
// (per-ray LDS stack), shading or sky, make_color.  rays (nullable) receives
// the generated rays.  Frames take k_camera_tiles where there is a 64-wide
// tree.
__global__ __launch_bounds__(kTraceThreads) void k_camera_frame(SceneView S, CameraLaunch C,
                                                                uchar4* __restrict__ frame, Ray* __restrict__ rays) {
  extern __shared__ uint32_t lds_stack[];
  const int pixels = C.width * C.height;
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= pixels) return;
  const Ray r = camera_ray(C, p % C.width, p / C.width);
  if (rays) rays[p] = r;
  if (!frame) return;
  Hit h;
  closest_hit(S, precompute_ray(r), lds_stack + threadIdx.x, blockDim.x, h);
  const V3 c = shade(S, h, r.dx, r.dy, r.dz);
  frame[p] = make_color(make_float4(c.x, c.y, c.z, 0.0f));
}

// A tile of 2^wide_log x 2^high_log pixels, at most 64, per one-wave workgroup,
// its rays as one packet (641 x 361 pixels of a panorama over 2.2 M triangles:
// 367 us with a ray per lane and a tree of four children, 136 with tiles of
// four pixels).
__global__ __launch_bounds__(64, 6) void k_camera_tiles(SceneView S, CameraLaunch C, int tiles_x, int wide_log,
                                                        int high_log, uchar4* __restrict__ frame) {
  extern __shared__ uint32_t tile_lds[];
  const int lane = (int)(threadIdx.x & 63);
  const uint32_t tile = xcd_run_block(blockIdx.x, gridDim.x, 16u);
  const int x = ((int)(tile % (uint32_t)tiles_x) << wide_log) + (lane & ((1 << wide_log) - 1));
  const int y = ((int)(tile / (uint32_t)tiles_x) << high_log) + (lane >> wide_log);
  const bool inside = (lane >> wide_log >> high_log) == 0 && x < C.width && y < C.height;
  const Ray r = camera_ray(C, inside ? x : 0, inside ? y : 0);
  Hit h;
  uint32_t steps = 0, tris = 0;
  packet_hits<kUnitPacketWide>(S, r, precompute_ray(r), inside, tile_lds, h, steps, tris);
  if (!inside) return;
  const V3 c = shade(S, h, r.dx, r.dy, r.dz);
  frame[(size_t)y * C.width + x] = make_color(make_float4(c.x, c.y, c.z, 0.0f));
}

__global__ void k_frame_sdf(const float4* __restrict__ colours, int omm_count, uchar4* __restrict__ frame,
                            int width) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= width || x >= omm_count) return;
  frame[x] = make_color(colours[x]);
}

__global__ void k_frame_sd(const float4* __restrict__ colours, int omm_count, uchar4* __restrict__ frame,
                           int width, int height) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  const int y = blockIdx.y;
  if (x >= width || y >= height) return;
  const int i = (int)(((long long)x * omm_count) / width);
  frame[(size_t)y * width + x] = make_color(colours[i]);
}

// Column x shows ommatidium x's samples, row y its sample y.  offsets
// (nullable: spp samples each) is the per-ommatidium sample counts' prefix
// sum; rows at or beyond an ommatidium's count keep the frame's contents.
__global__ void k_frame_raw(const float4* __restrict__ samples, const uint32_t* __restrict__ offsets,
                            int omm_count, int spp, uchar4* __restrict__ frame, int width, int height) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  const int y = blockIdx.y;
  if (x >= width || y >= height || x >= omm_count) return;
  const size_t first = offsets ? (size_t)offsets[x] : (size_t)x * (size_t)spp;
  const uint32_t n = offsets ? offsets[x + 1] - offsets[x] : (uint32_t)spp;
  if ((uint32_t)y >= n) return;
  // the reference stores c / spp per sample and displays it unsummed
  const float4 v = samples[first + (size_t)y];
  const float inv = 1.0f / (float)n;
  frame[(size_t)y * width + x] = make_color(make_float4(v.x * inv, v.y * inv, v.z * inv, 0.0f));
}

__global__ void k_pack_rgb(const float4* __restrict__ colours, uint64_t n, float* __restrict__ rgb) {
  const uint64_t u = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= n) return;
  const float4 c = colours[u];
  rgb[3 * u] = c.x;
  rgb[3 * u + 1] = c.y;
  rgb[3 * u + 2] = c.z;
}

__global__ void k_copy_probe(const float4* __restrict__ src, float4* __restrict__ dst, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    dst[i] = src[i];
}

bool check_launch(const char* what, std::string* err) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    if (err) *err = std::string(what) + ": " + hipGetErrorString(e);
    return false;
  }
  return true;
}

size_t stack_bytes(const DeviceScene& s) {
  const int depth = s.stack_bound > 0 ? s.stack_bound : 1;
  return sizeof(uint32_t) * (size_t)depth * kTraceThreads;
}

}  // namespace

static int g_trace_mode = kTracePacketWide;
static const char* g_last_kernel = "";
static bool g_split = true;

using UnitsKernel = void (*)(RenderArgs);

// A uniform count of at most 64 samples per unit (the adaptive pilot, uniform
// batches of few samples): every round traces once.
static bool one_pass(const UnitLaunch& U) { return !U.omm_counts && !U.unit_counts && U.spp <= 64; }

template <int kTrav>
static UnitsKernel units_kernel_variant(const UnitLaunch& U) {
  const bool one = one_pass(U);
  if (U.stats && U.samples) return one ? k_render_units<true, true, kTrav, true> : k_render_units<true, true, kTrav>;
  if (U.stats) return one ? k_render_units<true, false, kTrav, true> : k_render_units<true, false, kTrav>;
  if (U.samples) return one ? k_render_units<false, true, kTrav, true> : k_render_units<false, true, kTrav>;
  return one ? k_render_units<false, false, kTrav, true> : k_render_units<false, false, kTrav>;
}

static UnitsKernel units_kernel_of(const UnitLaunch& U) {
  if (U.traversal == kUnitPerRay) return units_kernel_variant<kUnitPerRay>(U);
  if (U.traversal == kUnitPacketWide) return units_kernel_variant<kUnitPacketWide>(U);
  return units_kernel_variant<kUnitPacket>(U);
}

static int device_cus() {
  static int cus = 0;
  if (cus == 0) {
    int dev = 0;
    (void)hipGetDevice(&dev);
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
      cus = 256;
  }
  return cus;
}

// Dynamic LDS of a block of `waves` waves: a stack column per lane (per ray) or
// per wave (wide packets).
static size_t units_lds_bytes(const DeviceScene& scene, int traversal, int waves = kTraceThreads / 64) {
  if (traversal == kUnitPacketWide) return sizeof(uint2) * (size_t)std::max(scene.wide_stack, 1) * (size_t)waves;
  return traversal == kUnitPerRay ? stack_bytes(scene) : 0;
}

// The wide walk's LDS stacks hold kWideStackMax entries and the 4-wide packets'
// stack, in VGPR lanes, kPacketStackMax: a deeper tree (or no wide tree) takes
// the next of them, at last the per-ray traversal.
static int effective_traversal(const DeviceScene& scene, int traversal) {
  if (traversal == kUnitPacketWide && scene.node_count > 0 &&
      (!scene.wide_nodes || scene.wide_stack > kWideStackMax))
    traversal = kUnitPacket;
  return traversal != kUnitPerRay && scene.stack_bound > kPacketStackMax ? (int)kUnitPerRay : traversal;
}

int render_units_capacity(const DeviceScene& scene, const UnitLaunch& U_in) {
  UnitLaunch U = U_in;
  U.traversal = effective_traversal(scene, U.traversal);
  const int threads = unit_threads(U.traversal);
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(units_kernel_of(U)), threads,
                                                   units_lds_bytes(scene, U.traversal, threads / 64)) != hipSuccess ||
      per_cu <= 0)
    per_cu = 4 * kTraceThreads / threads;
  return std::max(1, device_cus() * per_cu * threads / kTraceThreads);
}

static uint32_t magic_of(int n) { return (uint32_t)std::min<uint64_t>(0xffffffffull, (1ull << 32) / (uint64_t)n); }

// A launch of few packets lasts as long as its longest ones: a wave walks up
// to 1,500 boxes and 500 triangles of a large scene for 64 rays that fan out
// (over 60,000 instructions, 100 us and more alone), while most SIMDs have run
// dry.  Such launches deal their rays to more and narrower packets, up to
// these many.  Every further packet costs its own ray generation, set-up and
// walk to its rays, which the short walks of a small scene repay sooner.
// Measured, us, by packets (rays each):
//   frames, 24,200 triangles: 1,000 x 100 samples 2k 76, 4k 63, 8k 65, 16k 71,
//     32k 91; 1,000 x 400 7k 85, 14k 82, 28k 100;
//   frames, 2.2 M triangles: 700 x 32 700 122, 11k 45, 22k 41; 2,000 x 64 2k
//     191, 16k 80, 32k 76, 64k 99; 5,500 x 128 11k 242, 22k 169, 44k 150, 88k
//     188; 5,500 x 500 44k 325, 88k 328;
//   cameras, 19,602 triangles: 641 x 361 3.6k 97, 7.2k 74, 14k 66, 29k 63, 58k
//     95; 1,280 x 720 14k 81, 29k 77, 58k 96;
//   cameras, 2.2 M triangles: 97 x 61 91 722, 5.9k (1) 36; 641 x 361 3.6k 366,
//     14k 167, 29k 144, 58k 136, 116k 237; 1,280 x 720 14k 312, 58k 202, 115k
//     254; 320 x 180 29k (2) 80, 58k (1) 123.
constexpr int kLargeScene = 1 << 18;   // triangles; between the measured sizes
static uint64_t task_packets(const DeviceScene& scene) { return scene.tri_count < kLargeScene ? 12288 : 49152; }
static uint64_t tile_packets(const DeviceScene& scene) { return scene.tri_count < kLargeScene ? 16384 : 65536; }

// log2 of the waves that each task of a split launch deals its rays to.
static int task_ways(const DeviceScene& scene, const UnitLaunch& U) {
  if (effective_traversal(scene, U.traversal) != kUnitPacketWide) return 0;
  const uint64_t chunks = U.spp > 64 ? ((uint64_t)U.spp + 63u) / 64u : 1u;
  const uint64_t tasks = (uint64_t)U.omm_count * chunks, most = task_packets(scene);
  int ways = 0;
  while ((std::min(U.spp, 64) >> ways) > 1 && (tasks << (ways + 1)) <= most) ++ways;
  return ways;
}
bool tasks_are_dealt(const DeviceScene& scene, const UnitLaunch& U) { return task_ways(scene, U) > 0; }

bool launch_render_units(const DeviceScene& scene, const UnitLaunch& U_in, hipStream_t stream, std::string* err) {
  UnitLaunch U = U_in;
  const uint64_t units = (uint64_t)U.pose_count * (uint64_t)U.omm_count;
  if (units == 0) {
    if (U.traced) (void)hipEventRecord(U.traced, stream);
    return true;
  }
  if (units > kMaxLaunchUnits) {
    if (err) *err = "render_units: too many units for one launch";
    return false;
  }
  if (!U.colours || (U.samples && !U.sample_offsets)) {
    if (err) *err = "render_units: incomplete launch description";
    return false;
  }
  if (U.traversal < kUnitPacket || U.traversal > kUnitPerRay) {
    if (err) *err = "render_units: unknown traversal";
    return false;
  }
  U.traversal = effective_traversal(scene, U.traversal);
  const size_t lds = units_lds_bytes(scene, U.traversal);
  if (lds > 160 * 1024) {
    if (err) *err = "render_units: BVH too deep for the LDS traversal stack";
    return false;
  }
  const int capacity = render_units_capacity(scene, U);
  const SceneView v = view_of(scene);
  RenderArgs A{};
  A.S = v;
  A.U = U;
  if (U.host_pose) A.pose = *U.host_pose;
  A.omm_magic = magic_of(U.omm_count);
  // Split launch: one pose, a uniform count and fewer units than two per wave
  // slot of the device, when the caller gave scratch: each unit's 64-sample
  // chunks are tasks of their own, one wave each.  With per-ray traversal
  // units of 32 samples or fewer stay in the unit kernel, which packs two or
  // more of them into a wave's lanes (a per-ray task would leave the other
  // lanes idle); the packet task kernel takes any count (a single pose still
  // renders sooner that way).  The slots are counted at the kernels' launch
  // bound (5 blocks of 4 waves per CU) or the unit kernel's occupancy if
  // higher, not lowered by the LDS the per-ray stack takes: a deep tree's
  // per-ray stack cuts the unit kernel to two blocks per CU, which leaves a
  // single pose badly balanced.
  const uint64_t chunks = U.spp > 64 ? ((uint64_t)U.spp + 63u) / 64u : 1u;
  const uint64_t resident_waves = (uint64_t)std::max(capacity, device_cus() * 5) * (kTraceThreads / 64);
  const bool packet_tasks = U.traversal != kUnitPerRay;
  const uint64_t tasks = units * chunks;
  if (g_split && U.host_pose && !U.omm_counts && !U.unit_counts && !U.stats && (U.spp > 32 || packet_tasks) &&
      units < 2 * resident_waves && U.chunk_partial && tasks + (uint64_t)kSplitSubWaves <= max_grid(64) &&
      tasks * kTaskFloats <= U.chunk_partial_cap) {
    A.chunks = (uint32_t)chunks;
    A.chunk_magic = magic_of((int)chunks);
    A.tasks = (uint32_t)tasks;
    A.inv = 1.0f / (float)(uint32_t)U.spp;
    bool reduce = chunks > 1;
    if (packet_tasks) {
      const bool have_split = U.split_cost && U.split_flag && U.split_list && U.split_count && U.split_tasks == tasks;
      if (have_split && U.split_plan) {
        hipLaunchKernelGGL(k_split_plan, dim3(1), dim3(kSplitPlanThreads), 0, stream, U.split_cost, tasks,
                           U.split_flag, U.split_list, U.split_count);
      } else {
        A.U.split_flag = nullptr;
        if (have_split)  // no steps of these tasks yet: record them, split nothing
          hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)((tasks + 255) / 256)), dim3(256), 0, stream, U.split_cost,
                             (uint32_t)tasks, 0u);
        else
          A.U.split_cost = nullptr;
      }
      const bool wide = U.traversal == kUnitPacketWide;
      constexpr int kW = kUnitPacketWide, kP = kUnitPacket;
      // the variant without the split's code keeps the registers of the plain task kernel
      auto kernel = U.samples ? (wide ? k_render_tasks<true, kW, false> : k_render_tasks<true, kP, false>)
                              : (wide ? k_render_tasks<false, kW, false> : k_render_tasks<false, kP, false>);
      if (A.U.split_cost) {
        kernel = U.samples ? (wide ? k_render_tasks<true, kW, true> : k_render_tasks<true, kP, true>)
                           : (wide ? k_render_tasks<false, kW, true> : k_render_tasks<false, kP, true>);
        reduce = true;
      }
      if (!A.U.split_cost) A.ways_log = (uint32_t)task_ways(scene, U);
      if (A.ways_log != 0u) reduce = true;
      const uint64_t waves = (tasks << A.ways_log) + (A.U.split_flag ? (uint64_t)kSplitSubWaves : 0u);
      hipLaunchKernelGGL(kernel, dim3((unsigned)waves), dim3(64), units_lds_bytes(scene, U.traversal, 1), stream, A);
      g_last_kernel = "k_render_tasks";
    } else {
      // per-ray traversal: an LDS stack column per lane
      const unsigned grid = (unsigned)((tasks + (kTraceThreads / 64) - 1) / (kTraceThreads / 64));
      if (U.samples)
        hipLaunchKernelGGL(k_render_chunks<true>, dim3(grid), dim3(kTraceThreads), lds, stream, A);
      else
        hipLaunchKernelGGL(k_render_chunks<false>, dim3(grid), dim3(kTraceThreads), lds, stream, A);
      reduce = true;
      g_last_kernel = "k_render_chunks";
    }
    if (U.traced && hipEventRecord(U.traced, stream) != hipSuccess) {
      if (err) *err = "render_tasks: event";
      return false;
    }
    if (reduce)
      hipLaunchKernelGGL(k_reduce_tasks, dim3((unsigned)((units + 3) / 4)), dim3(kTraceThreads), 0, stream, A);
    if (U.frame_done) *U.frame_done = U.frame_pixels != nullptr;
    if (U.host_done) *U.host_done = U.host_colours != nullptr;
    return check_launch("render_tasks", err);
  }
  // Units per wave: as given, or (0) as many as leave four waves for every
  // resident slot, at most auto_grab_max, but enough to fill a wave's lanes
  // where that does not leave too few packets (733 ommatidia x 15 samples x 17
  // poses: 3,115 waves of four units 183 us with all else, 12,461 of one 115).
  if (A.U.units_per_grab <= 0) {
    uint64_t fill = 1;
    const uint64_t few = U.traversal == kUnitPacketWide ? task_packets(scene) : 0;
    if (one_pass(U))
      for (uint64_t seg = 64; seg > 1 && seg / 2 >= (uint64_t)std::max(U.spp, 1) && units / (2 * fill) >= few; seg /= 2)
        fill *= 2;
    A.U.units_per_grab = (int)std::max<uint64_t>(
        fill, std::min<uint64_t>((uint64_t)std::max(U.auto_grab_max, 1), units / (4 * resident_waves)));
  }
  A.U.units_per_grab = std::min(A.U.units_per_grab, kMaxUnitsPerGrab);
  const int threads = unit_threads(U.traversal);
  const UnitGrid shape = unit_grid(units, A.U.units_per_grab, threads, U.blocks);
  A.blocks = shape.blocks;
  // eight runs of consecutive workgroups per XCD: long enough for its L2 to
  // hold a pose's surroundings, short enough to even out the XCDs' work (4 to
  // 16 runs within 1 %, 64 runs 3-10 % slower)
  A.run = std::max<uint32_t>(1u, A.blocks / (kXcds * 8u));
  hipLaunchKernelGGL(units_kernel_of(U), dim3(shape.grid), dim3(threads),
                     units_lds_bytes(scene, U.traversal, threads / 64), stream, A);
  if (U.traced) (void)hipEventRecord(U.traced, stream);
  g_last_kernel = "k_render_units";
  return check_launch("render_units", err);
}

const char* last_render_kernel() { return g_last_kernel; }
void set_split_launches(bool on) { g_split = on; }

void set_trace_mode(int mode) { g_trace_mode = mode; }
int trace_mode() { return g_trace_mode; }
int unit_traversal_of(int mode) {
  return mode == kTracePerRay ? kUnitPerRay : mode == kTracePacketWide ? kUnitPacketWide : kUnitPacket;
}
int trace_mode_of(int traversal) {
  return traversal == kUnitPerRay ? kTracePerRay : traversal == kUnitPacketWide ? kTracePacketWide : kTracePacket;
}

bool launch_copy_probe(const float4* src, float4* dst, size_t n, hipStream_t stream, std::string* err) {
  if (n == 0) return true;
  const size_t blocks = std::min<size_t>((n + 255) / 256, 256 * 32);
  hipLaunchKernelGGL(k_copy_probe, dim3((unsigned)blocks), dim3(256), 0, stream, src, dst, n);
  return check_launch("copy_probe", err);
}

bool launch_trace_stats(const DeviceScene& scene, const EyeLaunch& L, unsigned long long* totals,
                        hipStream_t stream, std::string* err) {
  const uint64_t total = L.rays_per_pose * (uint64_t)L.pose_count;
  if (total == 0) return true;
  const size_t lds = stack_bytes(scene);
  if (lds > 160 * 1024) {
    if (err) *err = "trace: BVH too deep for the LDS traversal stack";
    return false;
  }
  const uint64_t blocks = (total + kTraceThreads - 1) / kTraceThreads;
  hipLaunchKernelGGL(k_trace_stats, dim3((unsigned)blocks), dim3(kTraceThreads), lds, stream, view_of(scene), L,
                     total, totals);
  return check_launch("trace_stats", err);
}

bool launch_frame_single_dim_fast(const float4* colours, int omm_count, uchar4* frame, int width,
                                  hipStream_t stream, std::string* err) {
  if (width <= 0 || omm_count <= 0) return true;
  hipLaunchKernelGGL(k_frame_sdf, dim3((width + 255) / 256), dim3(256), 0, stream, colours, omm_count, frame, width);
  return check_launch("frame", err);
}

bool launch_frame_single_dim(const float4* colours, int omm_count, uchar4* frame, int width, int height,
                             hipStream_t stream, std::string* err) {
  if (width <= 0 || height <= 0 || omm_count <= 0) return true;
  hipLaunchKernelGGL(k_frame_sd, dim3((width + 255) / 256, height), dim3(256), 0, stream, colours, omm_count,
                     frame, width, height);
  return check_launch("frame", err);
}

bool launch_frame_raw_samples(const float4* samples, const uint32_t* offsets, int omm_count, int spp,
                              uchar4* frame, int width, int height, hipStream_t stream, std::string* err) {
  if (width <= 0 || height <= 0 || omm_count <= 0) return true;
  hipLaunchKernelGGL(k_frame_raw, dim3((width + 255) / 256, height), dim3(256), 0, stream, samples, offsets,
                     omm_count, spp, frame, width, height);
  return check_launch("frame", err);
}

bool launch_camera_frame(const DeviceScene& scene, const CameraLaunch& C, uchar4* frame, Ray* rays,
                         hipStream_t stream, std::string* err) {
  if (C.width <= 0 || C.height <= 0) return true;
  const long long pixels = (long long)C.width * C.height;
  if (pixels > 0x7fffffffLL) {
    if (err) *err = "camera: frame too large";
    return false;
  }
  // the smallest tile (1, 1 x 2, 2 x 2 .. 8 x 8 pixels) that makes no more
  // than tile_packets tiles; single rays are worth a wave only while few
  int log = 0;
  if (pixels > 16384) log = 1;
  while (log < 6 && pixels > (long long)(tile_packets(scene) << log)) ++log;
  const int wide_log = log / 2, high_log = log - wide_log;
  const long long tiles_x = ((long long)C.width + (1 << wide_log) - 1) >> wide_log;
  const long long tiles_y = ((long long)C.height + (1 << high_log) - 1) >> high_log;
  if (frame && !rays && scene.node_count > 0 && (uint64_t)(tiles_x * tiles_y) <= max_grid(64) &&
      effective_traversal(scene, kUnitPacketWide) == kUnitPacketWide) {
    hipLaunchKernelGGL(k_camera_tiles, dim3((unsigned)(tiles_x * tiles_y)), dim3(64),
                       units_lds_bytes(scene, kUnitPacketWide, 1), stream, view_of(scene), C, (int)tiles_x,
                       wide_log, high_log, frame);
    return check_launch("camera_frame", err);
  }
  const size_t lds = stack_bytes(scene);
  if (lds > 160 * 1024) {
    if (err) *err = "camera: BVH too deep for the LDS traversal stack";
    return false;
  }
  hipLaunchKernelGGL(k_camera_frame, dim3((unsigned)((pixels + kTraceThreads - 1) / kTraceThreads)),
                     dim3(kTraceThreads), lds, stream, view_of(scene), C, frame, rays);
  return check_launch("camera_frame", err);
}

bool launch_pack_rgb(const float4* colours, uint64_t n, float* rgb, hipStream_t stream, std::string* err) {
  if (n == 0) return true;
  hipLaunchKernelGGL(k_pack_rgb, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, colours, n, rgb);
  return check_launch("pack_rgb", err);
}

bool launch_cones(const Ommatidium* omms, int omm_count, Cone* cones, hipStream_t stream, std::string* err) {
  if (omm_count <= 0) return true;
  hipLaunchKernelGGL(k_cones, dim3((unsigned)((omm_count + 255) / 256)), dim3(256), 0, stream, omms, omm_count, cones);
  return check_launch("cones", err);
}

bool launch_generate_rays(const EyeLaunch& L, Ray* rays, hipStream_t stream, std::string* err) {
  const uint64_t total = L.rays_per_pose * (uint64_t)L.pose_count;
  if (total == 0) return true;
  hipLaunchKernelGGL(k_generate_rays, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, stream, L, total, rays);
  return check_launch("generate_rays", err);
}

bool launch_packet_guard_probe(const DeviceScene& scene, const Ray* rays, int active_lanes, int32_t* ids,
                               hipStream_t stream, std::string* err) {
  const int trav = effective_traversal(scene, kUnitPacketWide);
  if (trav == kUnitPerRay) {
    if (err) *err = "packet probe: BVH too deep for the packet traversal";
    return false;
  }
  const size_t lds = units_lds_bytes(scene, trav, 1);
  if (trav == kUnitPacketWide)
    hipLaunchKernelGGL(k_packet_guard_probe<kUnitPacketWide>, dim3(1), dim3(64), lds, stream, view_of(scene), rays,
                       active_lanes, ids);
  else
    hipLaunchKernelGGL(k_packet_guard_probe<kUnitPacket>, dim3(1), dim3(64), lds, stream, view_of(scene), rays,
                       active_lanes, ids);
  return check_launch("packet_guard_probe", err);
}

bool launch_trace_rays(const DeviceScene& scene, const Ray* rays, uint64_t n, int32_t* hit, float* tbb,
                       hipStream_t stream, std::string* err) {
  if (n == 0) return true;
  const int log = n > 16384 ? 3 : 0;
  const uint64_t packets = (n + (1u << log) - 1) >> log;
  if (scene.node_count > 0 && packets <= max_grid(64) &&
      effective_traversal(scene, kUnitPacketWide) == kUnitPacketWide) {
    hipLaunchKernelGGL(k_trace_packets, dim3((unsigned)packets), dim3(64),
                       units_lds_bytes(scene, kUnitPacketWide, 1), stream, view_of(scene), rays, n, log, hit, tbb);
    return check_launch("trace_rays", err);
  }
  const size_t lds = stack_bytes(scene);
  if (lds > 160 * 1024) {
    if (err) *err = "trace: BVH too deep for the LDS traversal stack";
    return false;
  }
  hipLaunchKernelGGL(k_trace_rays, dim3((unsigned)((n + kTraceThreads - 1) / kTraceThreads)), dim3(kTraceThreads),
                     lds, stream, view_of(scene), rays, n, hit, tbb);
  return check_launch("trace_rays", err);
}

}  // namespace eye
