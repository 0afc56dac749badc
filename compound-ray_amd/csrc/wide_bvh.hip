// GPU build of the 64-wide traversal tree (rules in wide_bvh.h).  Bound by
// memory passes over the triangles: the 63-bit sort's eight passes move 24
// bytes per triangle each way, the rest about 200 bytes per triangle.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <string>
#include <vector>

#include "bvh_format.h"
#include "device_scene.h"
#include "radix.h"
#include "scan.h"
#include "wide_bvh.h"

namespace eye {
namespace {

constexpr int kBuildThreads = 256;
inline unsigned blocks_of(size_t n) { return (unsigned)((n + kBuildThreads - 1) / kBuildThreads); }

// Bit i of the low 21 bits of v moves to bit 3i.
__device__ __forceinline__ uint64_t expand_bits21(uint64_t v) {
  v &= 0x1fffffull;
  v = (v | v << 32) & 0x1f00000000ffffull;
  v = (v | v << 16) & 0x1f0000ff0000ffull;
  v = (v | v << 8) & 0x100f00f00f00f00full;
  v = (v | v << 4) & 0x10c30c30c30c30c3ull;
  return (v | v << 2) & 0x1249249249249249ull;
}

__device__ __forceinline__ void tri_box(const float4* tris, size_t k, float lo[3], float hi[3]) {
  const float4 a = tris[3 * k], b = tris[3 * k + 1], c = tris[3 * k + 2];
  lo[0] = fminf(fminf(a.x, b.x), c.x);
  lo[1] = fminf(fminf(a.y, b.y), c.y);
  lo[2] = fminf(fminf(a.z, b.z), c.z);
  hi[0] = fmaxf(fmaxf(a.x, b.x), c.x);
  hi[1] = fmaxf(fmaxf(a.y, b.y), c.y);
  hi[2] = fmaxf(fmaxf(a.z, b.z), c.z);
}

__global__ __launch_bounds__(kBuildThreads) void k_wide_codes(const float4* __restrict__ tris, int n, float ox,
                                                             float oy, float oz, float scale,
                                                             uint64_t* __restrict__ codes,
                                                             uint32_t* __restrict__ ids,
                                                             uint32_t* __restrict__ beyond) {
  const int i = blockIdx.x * kBuildThreads + threadIdx.x;
  if (i >= n) return;
  const auto within = [](const float4& v) {   // false for a not-a-number
    return (fabsf(v.x) <= kWideFarthest) & (fabsf(v.y) <= kWideFarthest) & (fabsf(v.z) <= kWideFarthest);
  };
  if (!(within(tris[3 * (size_t)i]) & within(tris[3 * (size_t)i + 1]) & within(tris[3 * (size_t)i + 2]))) *beyond = 1u;
  float lo[3], hi[3];
  tri_box(tris, (size_t)i, lo, hi);
  const float o[3] = {ox, oy, oz};
  uint64_t code = 0;
  for (int a = 0; a < 3; ++a) {
    const float q = ((lo[a] + hi[a]) * 0.5f - o[a]) * scale;
    code |= expand_bits21((uint64_t)fminf(fmaxf(q, 0.0f), 2097151.0f)) << (2 - a);
  }
  codes[i] = code;
  ids[i] = (uint32_t)i;
}

// Common-prefix length of sorted keys i and j, equal keys told apart by index.
__device__ __forceinline__ int prefix64(const uint64_t* codes, int n, int i, int j) {
  if (j < 0 || j >= n) return -1;
  const uint64_t x = codes[i] ^ codes[j];
  return x != 0 ? __clzll((long long)x) : 64 + __clz((int)((uint32_t)i ^ (uint32_t)j));
}

// Karras' internal node i of n - 1: the range of keys it covers and its
// parenthood.  Combined indexing: internal nodes 0 .. n-2, leaf k at n-1+k.
__global__ __launch_bounds__(kBuildThreads) void k_wide_radix_tree(const uint64_t* __restrict__ codes, int n,
                                                                  int2* __restrict__ range,
                                                                  int32_t* __restrict__ parent) {
  const int i = blockIdx.x * kBuildThreads + threadIdx.x;
  if (i < n) range[n - 1 + i] = make_int2(i, i);
  if (i == 0) parent[0] = -1;
  if (i >= n - 1) return;
  const int d = prefix64(codes, n, i, i + 1) > prefix64(codes, n, i, i - 1) ? 1 : -1;
  const int low = prefix64(codes, n, i, i - d);
  int reach = 2;
  while (prefix64(codes, n, i, i + reach * d) > low) reach *= 2;
  int len = 0;
  for (int t = reach / 2; t >= 1; t /= 2)
    if (prefix64(codes, n, i, i + (len + t) * d) > low) len += t;
  const int j = i + len * d;
  const int own = prefix64(codes, n, i, j);
  int s = 0;
  for (int t = len; t > 1;) {
    t = (t + 1) / 2;
    if (prefix64(codes, n, i, i + (s + t) * d) > own) s += t;
  }
  const int split = i + s * d + (d < 0 ? -1 : 0);
  const int first = min(i, j), last = max(i, j);
  const int left = split == first ? n - 1 + split : split;
  const int right = split + 1 == last ? n - 1 + split + 1 : split + 1;
  range[i] = make_int2(first, last);
  parent[left] = i;
  parent[right] = i;
}

// Units a binary node covers: start[] is the exclusive prefix sum of the unit
// starts (start[n] = their number); null: every triangle is a unit.
__device__ __forceinline__ int units_in(const uint32_t* start, int2 r) {
  return start ? (int)(start[r.y + 1] - start[r.x]) : r.y - r.x + 1;
}

// Flags the first triangle of every largest subtree of at most `most` units
// (the next level's units): in `unit` all of them, in `made` those of two or
// more units, which become nodes; `node_of` keeps the binary node at the start.
__global__ __launch_bounds__(kBuildThreads) void k_wide_mark(const int2* __restrict__ range,
                                                            const int32_t* __restrict__ parent, int n, int most,
                                                            const uint32_t* __restrict__ start,
                                                            uint32_t* __restrict__ unit, uint32_t* __restrict__ made,
                                                            int32_t* __restrict__ node_of) {
  const int x = blockIdx.x * kBuildThreads + threadIdx.x;
  if (x >= 2 * n - 1) return;
  const int2 r = range[x];
  const int c = units_in(start, r);
  if (c > most) return;
  if (x != 0 && units_in(start, range[parent[x]]) <= most) return;
  unit[r.x] = 1u;
  made[r.x] = c > 1 ? 1u : 0u;
  node_of[r.x] = x;
}

// A level's units.
struct Units {
  float* box;       // 6 per unit: lo x, y, z, hi x, y, z
  int32_t* ref;     // leaf code or node number
  int32_t* need;    // deferred children a walk of the unit's subtree can hold
};

// Level 0: leaves.  `start`: exclusive prefix sum of the leaf starts.
__global__ __launch_bounds__(kBuildThreads) void k_wide_leaves(const int2* __restrict__ range,
                                                              const int32_t* __restrict__ node_of,
                                                              const uint32_t* __restrict__ start, int n,
                                                              const float4* __restrict__ tris,
                                                              const uint32_t* __restrict__ ids, Units out) {
  const int i = blockIdx.x * kBuildThreads + threadIdx.x;
  if (i >= n || start[i + 1] == start[i]) return;
  const int2 r = range[node_of[i]];
  float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
  for (int k = r.x; k <= r.y; ++k) {
    float l[3], h[3];
    tri_box(tris, (size_t)ids[k], l, h);
    for (int a = 0; a < 3; ++a) {
      lo[a] = fminf(lo[a], l[a]);
      hi[a] = fmaxf(hi[a], h[a]);
    }
  }
  const uint32_t u = start[i];
  for (int a = 0; a < 3; ++a) {
    out.box[6 * (size_t)u + a] = lo[a];
    out.box[6 * (size_t)u + 3 + a] = hi[a];
  }
  out.ref[u] = encode_leaf((uint32_t)r.x, (uint32_t)(r.y - r.x + 1));
  out.need[u] = 0;
}

__device__ __forceinline__ WideChild child_of(const float lo[3], const float hi[3], int32_t ref, float radius) {
  float c[3], h[3];
  for (int a = 0; a < 3; ++a) {
    c[a] = (lo[a] + hi[a]) * 0.5f;
    const float e = fmaxf(hi[a] - c[a], c[a] - lo[a]);
    h[a] = (e * (1.0f + 2.0f * kWidePad) + (fabsf(c[a]) + radius) * kWidePad) + 1e-30f;
  }
  return WideChild{c[0], c[1], c[2], ref, h[0], h[1], h[2], 0.0f};
}

__device__ __forceinline__ WideChild empty_child() {
  return WideChild{0.0f, 0.0f, 0.0f, kChildEmpty, 0.0f, 0.0f, 0.0f, 0.0f};
}

// One wave per unit of the new level: a unit of one old unit is that unit; any
// other becomes node base + rank, whose children are its old units in order.
__global__ __launch_bounds__(kBuildThreads) void k_wide_level(const int2* __restrict__ range,
                                                             const int32_t* __restrict__ node_at, int count,
                                                             const uint32_t* __restrict__ old_start,
                                                             const uint32_t* __restrict__ rank, int base, float radius,
                                                             Units in, Units out, WideNode64* __restrict__ nodes) {
  const int u = (int)(blockIdx.x * (kBuildThreads / 64) + (threadIdx.x >> 6));
  const int lane = (int)(threadIdx.x & 63);
  if (u >= count) return;   // whole wave
  const int2 r = range[node_at[u]];
  const uint32_t c0 = old_start[r.x], c1 = old_start[r.y + 1];
  const bool have = (uint32_t)lane < c1 - c0;
  const size_t src = (size_t)c0 + (size_t)lane;
  float lo[3], hi[3];
  for (int a = 0; a < 3; ++a) {
    lo[a] = have ? in.box[6 * src + a] : INFINITY;
    hi[a] = have ? in.box[6 * src + 3 + a] : -INFINITY;
  }
  const int32_t ref = have ? in.ref[src] : kChildEmpty;
  int need = have ? in.need[src] : 0;
  if (c1 - c0 == 1u) {
    if (lane == 0) {
      for (int a = 0; a < 3; ++a) {
        out.box[6 * (size_t)u + a] = lo[a];
        out.box[6 * (size_t)u + 3 + a] = hi[a];
      }
      out.ref[u] = ref;
      out.need[u] = need;
    }
    return;
  }
  const int id = base + (int)rank[r.x];
  nodes[rank[r.x]].child[lane] = have ? child_of(lo, hi, ref, radius) : empty_child();
  const int inner = __popcll(__ballot(have && !child_is_leaf(ref)));
  for (int m = 32; m >= 1; m >>= 1) {
    for (int a = 0; a < 3; ++a) {
      lo[a] = fminf(lo[a], __shfl_xor(lo[a], m));
      hi[a] = fmaxf(hi[a], __shfl_xor(hi[a], m));
    }
    need = max(need, __shfl_xor(need, m));
  }
  if (lane == 0) {
    for (int a = 0; a < 3; ++a) {
      out.box[6 * (size_t)u + a] = lo[a];
      out.box[6 * (size_t)u + 3 + a] = hi[a];
    }
    out.ref[u] = id;
    out.need[u] = need + max(inner - 1, 0);
  }
}

// The new level's binary nodes, one per unit.
__global__ __launch_bounds__(kBuildThreads) void k_wide_units(const uint32_t* __restrict__ start,
                                                             const int32_t* __restrict__ node_of, int n,
                                                             int32_t* __restrict__ node_at) {
  const int i = blockIdx.x * kBuildThreads + threadIdx.x;
  if (i < n && start[i + 1] != start[i]) node_at[start[i]] = node_of[i];
}

// A scene of one leaf: its root holds that leaf alone.
__global__ void k_wide_single(Units in, float radius, WideNode64* __restrict__ nodes) {
  const int lane = (int)threadIdx.x;
  nodes[0].child[lane] = lane == 0 ? child_of(in.box, in.box + 3, in.ref[0], radius) : empty_child();
}

__global__ __launch_bounds__(kBuildThreads) void k_wide_gather(const float4* __restrict__ tris,
                                                              const uint32_t* __restrict__ ids, int n,
                                                              float4* __restrict__ out) {
  const int k = blockIdx.x * kBuildThreads + threadIdx.x;
  if (k >= n) return;
  const uint32_t id = ids[k];
  const float4 a = tris[3 * (size_t)id], b = tris[3 * (size_t)id + 1], c = tris[3 * (size_t)id + 2];
  out[3 * (size_t)k] = make_float4(a.x, b.x, c.x, a.w);
  out[3 * (size_t)k + 1] = make_float4(a.y, b.y, c.y, __uint_as_float(id));
  out[3 * (size_t)k + 2] = make_float4(a.z, b.z, c.z, 0.0f);
}

// Structure check before any walk: every child is a leaf inside the triangle
// array or a node of a lower number, every node but the root has one parent
// and every triangle is in one leaf.  Violations set *bad.
__global__ __launch_bounds__(kBuildThreads) void k_wide_count(const WideNode64* __restrict__ nodes, int count, int n,
                                                             uint32_t* __restrict__ parents,
                                                             uint32_t* __restrict__ covered,
                                                             uint32_t* __restrict__ bad) {
  const int x = (int)(blockIdx.x * (kBuildThreads / 64) + (threadIdx.x >> 6));
  if (x >= count) return;
  const int32_t c = nodes[x].child[threadIdx.x & 63].ref;
  if (c == kChildEmpty) return;
  if (child_is_leaf(c)) {
    const uint32_t f = leaf_first(c), k = leaf_count(c);
    if ((uint64_t)f + k > (uint64_t)n || k > (uint32_t)kWideLeaf)
      *bad = 1u;
    else
      for (uint32_t q = f; q < f + k; ++q) atomicAdd(&covered[q], 1u);
  } else if (c >= x) {
    *bad = 1u;
  } else {
    atomicAdd(&parents[c], 1u);
  }
}

__global__ __launch_bounds__(kBuildThreads) void k_wide_check(const uint32_t* __restrict__ parents, int count,
                                                             const uint32_t* __restrict__ covered, int n,
                                                             uint32_t* __restrict__ bad) {
  const int i = blockIdx.x * kBuildThreads + threadIdx.x;
  if (i < n && covered[i] != 1u) *bad = 1u;
  if (i < count && parents[i] != (i == count - 1 ? 0u : 1u)) *bad = 1u;
}

// Device allocations of one build, freed together unless taken.
struct Pool {
  std::vector<void*> held;
  std::string* err;
  bool ok = true;
  bool full = false;   // out of memory
  template <typename T>
  T* get(size_t n) {
    void* p = nullptr;
    if (!ok) return nullptr;
    const hipError_t e = hipMalloc(&p, sizeof(T) * std::max<size_t>(n, 1));
    if (e != hipSuccess) {
      if (err) *err = std::string("wide tree: hipMalloc: ") + hipGetErrorString(e);
      ok = false;
      full = e == hipErrorOutOfMemory;
      return nullptr;
    }
    held.push_back(p);
    return static_cast<T*>(p);
  }
  void drop(void* p) {
    held.erase(std::find(held.begin(), held.end(), p));
    (void)hipFree(p);
  }
  template <typename T>
  T* take(T* p) {
    held.erase(std::find(held.begin(), held.end(), (void*)p));
    return p;
  }
  ~Pool() {
    for (void* p : held) (void)hipFree(p);
  }
};

bool good(hipError_t e, const char* what, std::string* err) {
  if (e == hipSuccess) return true;
  if (err) *err = std::string("wide tree: ") + what + ": " + hipGetErrorString(e);
  return false;
}

// *unfit: the scene takes no wide tree.
bool build(DeviceScene* S, Pool& pool, ScanScratch* scan, bool* unfit, hipStream_t stream, std::string* err) {
  const int n = S->tri_count;
  const size_t N = (size_t)n;
  const int tiles = (int)((N + kSortTile - 1) / kSortTile);
  uint64_t *codes = pool.get<uint64_t>(N), *codes_b = pool.get<uint64_t>(N);
  uint32_t *ids = pool.get<uint32_t>(N), *ids_b = pool.get<uint32_t>(N);
  uint32_t* hist = pool.get<uint32_t>((size_t)kRadix * tiles);
  int2* range = pool.get<int2>(2 * N - 1);
  int32_t* parent = pool.get<int32_t>(2 * N - 1);
  uint32_t* bad = pool.get<uint32_t>(1);
  if (!pool.ok || !scan_reserve(scan, std::max((size_t)kRadix * tiles, N + 1), err, &pool.full)) return false;
  float ext = 0.0f;
  for (int a = 0; a < 3; ++a) ext = std::max(ext, S->centroid_hi[a] - S->centroid_lo[a]);
  float radius = ext;
  for (int a = 0; a < 3; ++a)
    radius = std::max(radius, std::max(std::fabs(S->centroid_lo[a]), std::fabs(S->centroid_hi[a])));
  const float scale = ext > 0.0f ? 2097152.0f / ext : 0.0f;
  if (!good(hipMemsetAsync(bad, 0, sizeof(uint32_t), stream), "clear", err)) return false;
  hipLaunchKernelGGL(k_wide_codes, dim3(blocks_of(N)), dim3(kBuildThreads), 0, stream, S->tris, n, S->centroid_lo[0],
                     S->centroid_lo[1], S->centroid_lo[2], scale, codes, ids, bad);
  uint32_t beyond = 0;
  if (!good(hipGetLastError(), "launch", err) ||
      !good(hipMemcpyAsync(&beyond, bad, sizeof(beyond), hipMemcpyDeviceToHost, stream), "extent", err) ||
      !good(hipStreamSynchronize(stream), "extent", err))
    return false;
  if (beyond) {
    *unfit = true;
    return true;
  }
  for (int shift = 0; shift < 64; shift += 8) {
    hipLaunchKernelGGL(k_sort_hist<uint64_t>, dim3(tiles), dim3(kSortThreads), 0, stream, codes, n, shift, hist,
                       tiles);
    if (!scan_exclusive_u32(scan, hist, (size_t)kRadix * tiles, stream, err)) return false;
    hipLaunchKernelGGL(k_sort_scatter<uint64_t>, dim3(tiles), dim3(kSortThreads), 0, stream, codes, ids, codes_b,
                       ids_b, n, shift, hist, tiles);
    std::swap(codes, codes_b);
    std::swap(ids, ids_b);
  }
  hipLaunchKernelGGL(k_wide_radix_tree, dim3(blocks_of(N)), dim3(kBuildThreads), 0, stream, codes, n, range, parent);
  // level 0: the leaves.  codes and codes_b are free from here: the start
  // tables of this level and the next live in them.
  uint32_t* start = reinterpret_cast<uint32_t*>(codes);      // n + 1 words of 2 n
  uint32_t* next = reinterpret_cast<uint32_t*>(codes_b);
  uint32_t* made = pool.get<uint32_t>(N + 1);
  int32_t* node_of = pool.get<int32_t>(N);
  if (!pool.ok) return false;
  const auto mark = [&](int most, const uint32_t* old, uint32_t* unit, uint32_t* units, uint32_t* nodes) {
    if (!good(hipMemsetAsync(unit, 0, sizeof(uint32_t) * (N + 1), stream), "clear", err) ||
        !good(hipMemsetAsync(made, 0, sizeof(uint32_t) * (N + 1), stream), "clear", err))
      return false;
    hipLaunchKernelGGL(k_wide_mark, dim3(blocks_of(2 * N - 1)), dim3(kBuildThreads), 0, stream, range, parent, n, most,
                       old, unit, made, node_of);
    return scan_exclusive_u32_total(scan, unit, unit, N + 1, stream, units, err) &&
           scan_exclusive_u32_total(scan, made, made, N + 1, stream, nodes, err);
  };
  uint32_t count = 0, fresh = 0;
  if (!mark(kWideLeaf, nullptr, start, &count, &fresh)) return false;
  Units cur{pool.get<float>(6 * (size_t)count), pool.get<int32_t>(count), pool.get<int32_t>(count)};
  if (!pool.ok) return false;
  hipLaunchKernelGGL(k_wide_leaves, dim3(blocks_of(N)), dim3(kBuildThreads), 0, stream, range, node_of, start, n,
                     S->tris, ids, cur);
  struct Level {
    WideNode64* nodes;
    int count;
  };
  std::vector<Level> levels;
  int total = 0;
  if (count == 1) {
    levels.push_back(Level{pool.get<WideNode64>(1), 1});
    if (!pool.ok) return false;
    hipLaunchKernelGGL(k_wide_single, dim3(1), dim3(64), 0, stream, cur, radius, levels.back().nodes);
    total = 1;
  }
  while (count > 1) {
    uint32_t units = 0;
    if (!mark(kWideWidth, start, next, &units, &fresh)) return false;
    if (units >= count || fresh == 0) {
      if (err) *err = "wide tree: a level did not shrink";
      return false;
    }
    Units out{pool.get<float>(6 * (size_t)units), pool.get<int32_t>(units), pool.get<int32_t>(units)};
    int32_t* node_at = pool.get<int32_t>(units);
    levels.push_back(Level{pool.get<WideNode64>(fresh), (int)fresh});
    if (!pool.ok) return false;
    hipLaunchKernelGGL(k_wide_units, dim3(blocks_of(N)), dim3(kBuildThreads), 0, stream, next, node_of, n, node_at);
    hipLaunchKernelGGL(k_wide_level, dim3(blocks_of((size_t)units * 64)), dim3(kBuildThreads), 0, stream, range,
                       node_at, (int)units, start, made, total, radius, cur, out,
                       levels.back().nodes);
    total += (int)fresh;
    if (!good(hipStreamSynchronize(stream), "level", err)) return false;
    pool.drop(cur.box);
    pool.drop(cur.ref);
    pool.drop(cur.need);
    pool.drop(node_at);
    cur = out;
    count = units;
    std::swap(start, next);
  }
  WideNode64* nodes = pool.get<WideNode64>((size_t)total);
  float4* tris = pool.get<float4>(3 * N);
  uint32_t* parents = pool.get<uint32_t>((size_t)total);
  if (!pool.ok) return false;
  size_t at = 0;
  for (const Level& l : levels) {
    if (!good(hipMemcpyAsync(nodes + at, l.nodes, sizeof(WideNode64) * (size_t)l.count, hipMemcpyDeviceToDevice,
                             stream), "nodes", err))
      return false;
    at += (size_t)l.count;
  }
  hipLaunchKernelGGL(k_wide_gather, dim3(blocks_of(N)), dim3(kBuildThreads), 0, stream, S->tris, ids, n, tris);
  if (!good(hipMemsetAsync(parents, 0, sizeof(uint32_t) * (size_t)total, stream), "clear", err) ||
      !good(hipMemsetAsync(made, 0, sizeof(uint32_t) * N, stream), "clear", err) ||
      !good(hipMemsetAsync(bad, 0, sizeof(uint32_t), stream), "clear", err))
    return false;
  hipLaunchKernelGGL(k_wide_count, dim3(blocks_of((size_t)total * 64)), dim3(kBuildThreads), 0, stream, nodes, total,
                     n, parents, made, bad);
  hipLaunchKernelGGL(k_wide_check, dim3(blocks_of(std::max(N, (size_t)total))), dim3(kBuildThreads), 0, stream,
                     parents, total, made, n, bad);
  uint32_t wrong = 0;
  int32_t need = 0;
  float box[6];
  if (!good(hipGetLastError(), "launch", err) ||
      !good(hipMemcpyAsync(box, cur.box, sizeof(box), hipMemcpyDeviceToHost, stream), "box", err) ||
      !good(hipMemcpyAsync(&wrong, bad, sizeof(wrong), hipMemcpyDeviceToHost, stream), "check", err) ||
      !good(hipMemcpyAsync(&need, cur.need, sizeof(need), hipMemcpyDeviceToHost, stream), "bound", err) ||
      !good(hipStreamSynchronize(stream), "build", err))
    return false;
  if (wrong) {
    if (err) *err = "wide tree: bad structure";
    return false;
  }
  S->wide_nodes = pool.take(nodes);
  S->wide_tris = pool.take(tris);
  S->wide_count = total;
  S->wide_root = total - 1;
  S->wide_stack = std::max(need, 1);
  S->wide_radius = radius;
  S->wide_farthest = 0.0f;
  for (float v : box) S->wide_farthest = std::max(S->wide_farthest, std::fabs(v));
  return true;
}

}  // namespace

bool build_wide_tree(DeviceScene* scene, hipStream_t stream, std::string* err) {
  if (scene->tri_count == 0) return true;
  ScanScratch scan;
  Pool pool;
  pool.err = err;
  bool unfit = false;
  const bool ok = build(scene, pool, &scan, &unfit, stream, err);
  scan_release(&scan);
  if (ok || !pool.full) return ok;
  // no room: packets walk the 4-wide tree
  (void)hipGetLastError();
  if (err) err->clear();
  return true;
}

void free_wide_tree(DeviceScene* scene) {
  if (scene->wide_nodes) (void)hipFree(scene->wide_nodes);
  if (scene->wide_tris) (void)hipFree(scene->wide_tris);
  scene->wide_nodes = nullptr;
  scene->wide_tris = nullptr;
  scene->wide_count = 0;
}

}  // namespace eye
