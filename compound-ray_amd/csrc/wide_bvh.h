// The 64-wide tree that wave packets walk, and its builder's interface.
//
// A wave of 64 lanes tests 64 child boxes at once, one per lane, against the
// bounds of its rays (packet.h), so a node has up to 64 children: a packet
// makes 3-15 dependent node fetches where the 4-wide tree needs 11-66.  The
// tree serves traversal only; the canonical 4-wide tree (bvh_format.h) stays
// for the per-ray kernels, the traversal statistics and inspection.  Which
// triangle a ray hits does not depend on the tree: the closest hit is the
// (t, id) minimum over every triangle the ray meets.
//
// Build (wide_bvh.hip), over the triangles in canonical order:
//   1. 63-bit Morton codes of the box centres in cubic cells (all three axes
//      divided by the longest extent, 21 bits each).  The canonical tree's
//      10 bits per axis, each axis by its own extent, cut a flat terrain
//      through its height as often as along it: over the 2.2M-triangle bee
//      scene a packet enters a quarter more boxes and triangles with them.
//   2. the binary radix tree over the sorted codes (Karras, HPG 2012);
//   3. units: leaves are its largest subtrees of at most kWideLeaf
//      triangles; then, level by level, the largest subtrees of at most 64
//      units become nodes, which are the units of the next level, until one is
//      left.  A subtree covers a contiguous run of sorted triangles, so a
//      node's children are consecutive units, found with two prefix sums, and
//      no bounds of the binary tree are ever needed.  Nodes hold 41 of 64
//      children on average; growing nodes from the top, largest box first,
//      leaves most bottom nodes with 2-8.
// Leaves of at most 4 triangles: against 2, a third fewer ray tests of boxes
// for half again as many of triangles, and half the node bytes (203 poses of
// the bee eye 17.2 -> 16.7 ms, its adaptive render 16.0 -> 15.1; the small
// scene's batch 66.8 -> 68.7).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string>

namespace eye {

struct DeviceScene;

constexpr int kWideWidth = 64;   // one child per lane
constexpr int kWideLeaf = 4;     // triangles per leaf, at most
// Deferred children a packet may hold at once (LDS, 8 bytes each per wave).  A
// tree that could need more is walked through the 4-wide tree instead.
constexpr int kWideStackMax = 512;

// Relative padding of box tests.
constexpr float kWidePad = 4.76837158203125e-7f;   // 2^-21

// Scenes with a vertex that is not a number or further out than this have no
// wide tree: boxes as centre and half extent would lose such corners (an
// infinite or overflowing centre is not inside its box), and a packet orders
// children by depths, which have to be numbers.  Their rays take the 4-wide
// walks, whose boxes keep both corners.
constexpr float kWideFarthest = 1.152921504606846976e18f;   // 2^60

// Boxes as centre and half extent: (c - o) / d -/+ h / |d| needs no choice of
// near and far planes.  Half extents are rounded up and padded by kWidePad of
// themselves, of the centre and of the scene's radius R (the largest
// coordinate).  With u = 2^-24, a test of an axis is off, as a length, by at most
//   2 u (|c - o| + h)  the reciprocal, to one ulp
//   u |o|              its product with the origin
//   u |c - o|          the first FMA
//   u (|c - o| + h)    the second
// together 5 u |o| + 4 u |c| + 3 u h.  kWidePad = 8 u covers that for origins out
// to kWideRange R, so that no box loses a ray that meets it.  (At 3.9 R, of 8 M
// hits on corners of flat boxes one was lost.)  Packets from further out pad
// the boxes by their own origins, walk64's kFar.
constexpr float kWideRange = 1.5f;
struct WideChild {
  float cx, cy, cz;
  int32_t ref;                 // bvh_format.h's encoding: a node, a leaf of the wide order, or kChildEmpty
  float hx, hy, hz, unused;
};
struct alignas(32) WideNode64 {
  WideChild child[kWideWidth];
};
static_assert(sizeof(WideNode64) == 2048, "wide node layout");

// Builds scene->wide_* from the scene's canonical triangles; without room for
// it, or beyond kWideFarthest, they stay null.  False and `err` on failure (nothing is left allocated).
bool build_wide_tree(DeviceScene* scene, hipStream_t stream, std::string* err);
void free_wide_tree(DeviceScene* scene);

}  // namespace eye
