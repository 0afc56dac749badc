#include "batch.h"

#include <algorithm>
#include <cstdio>
#include <cstring>
#include <fstream>
#include <sstream>

namespace eye {

namespace {
template <typename T>
bool grow(T** p, size_t* cap, size_t n, std::string* err) {
  if (*cap >= n && *p) return true;
  if (*p) (void)hipFree(*p);
  *p = nullptr;
  *cap = 0;
  if (n == 0) return true;
  const hipError_t e = hipMalloc(p, sizeof(T) * n);
  if (e != hipSuccess) {
    if (err) *err = std::string("batch: hipMalloc failed: ") + hipGetErrorString(e);
    return false;
  }
  *cap = n;
  return true;
}

constexpr size_t kPackUnits = (size_t)1 << 23;   // 96 MiB of packed colours at most
constexpr size_t kHostUnits = 65536;             // 768 KiB of pinned ones

}  // namespace

std::vector<LaunchShape> LaunchTuner::candidates(int capacity) {
  std::vector<LaunchShape> out;
  const int cap = std::max(capacity, 1);
  // a wave per grab, or a grid that strides over the grabs: 4,096 poses x 5,000
  // uneven ommatidia 59.9 ms with a wave per grab, 70.1 with 2 cap blocks
  const int block_opts[3] = {0, cap, 2 * cap};
  for (int trav = kUnitPacket; trav <= kUnitPerRay; ++trav)
    for (int b : block_opts)
      for (int g : {1, 2, 4, 8, 16}) {
        LaunchShape sh;
        sh.units_per_grab = g;
        sh.blocks = b;
        sh.traversal = trav;
        out.push_back(sh);
      }
  return out;
}

std::string LaunchTuner::key_of(const DeviceScene& scene, const UnitLaunch& U, uint64_t samples_per_pose) {
  // The last word names the kernels that the shapes were timed on: files hold
  // shapes of others too (traversal 1 was once another walk, and blocks a
  // persistent grid's), which must not pass for these.
  char buf[160];
  std::snprintf(buf, sizeof(buf), "tris%d_nodes%d_leaf%d_omm%d_spp%llu_stats%d_rec%d_wide64", scene.tri_count,
                scene.node_count, scene.leaf_max, U.omm_count, (unsigned long long)samples_per_pose,
                U.stats ? 1 : 0, U.samples ? 1 : 0);
  return buf;
}

bool LaunchTuner::find(const std::string& key, LaunchShape* shape) const {
  for (size_t i = keys_.size(); i-- > 0;)
    if (keys_[i] == key) {
      *shape = shapes_[i];
      return true;
    }
  return false;
}

void LaunchTuner::put(const std::string& key, const LaunchShape& shape, double ms) {
  for (size_t i = 0; i < keys_.size(); ++i)
    if (keys_[i] == key) {
      shapes_[i] = shape;
      ms_[i] = ms;
      return;
    }
  keys_.push_back(key);
  shapes_.push_back(shape);
  ms_.push_back(ms);
}

bool LaunchTuner::load(const std::string& path, std::string* err) {
  std::ifstream f(path);
  if (!f) return true;  // no file yet: nothing cached
  std::string line;
  int lineno = 0;
  while (std::getline(f, line)) {
    ++lineno;
    if (line.empty() || line[0] == '#') continue;
    std::istringstream in(line);
    std::string key;
    LaunchShape sh;
    double ms = 0.0;
    if (!(in >> key >> sh.units_per_grab >> sh.blocks >> sh.traversal >> ms) || sh.units_per_grab < 1 ||
        sh.blocks < 0 || sh.traversal < kUnitPacket || sh.traversal > kUnitPerRay) {
      if (err) *err = "autotune cache " + path + ": bad entry on line " + std::to_string(lineno);
      return false;
    }
    put(key, sh, ms);
  }
  return true;
}

bool LaunchTuner::save(const std::string& path, std::string* err) const {
  std::ofstream f(path, std::ios::trunc);
  if (!f) {
    if (err) *err = "autotune cache " + path + ": cannot write";
    return false;
  }
  f << "# key units_per_grab blocks traversal ms\n";
  for (size_t i = 0; i < keys_.size(); ++i)
    f << keys_[i] << ' ' << shapes_[i].units_per_grab << ' ' << shapes_[i].blocks << ' ' << shapes_[i].traversal
      << ' ' << ms_[i] << '\n';
  return bool(f);
}

void BatchRenderer::release() {
  if (d_poses_) (void)hipFree(d_poses_);
  if (d_colours_) (void)hipFree(d_colours_);
  if (d_rgb_) (void)hipFree(d_rgb_);
  if (h_rgb_) (void)hipHostFree(h_rgb_);
  d_rgb_ = h_rgb_ = nullptr;
  rgb_cap_ = 0;
  if (ev0_) (void)hipEventDestroy(ev0_);
  if (ev1_) (void)hipEventDestroy(ev1_);
  d_poses_ = nullptr;
  d_colours_ = nullptr;
  ev0_ = ev1_ = nullptr;
  poses_cap_ = colours_cap_ = 0;
}

bool BatchRenderer::host_rgb() {
  if (h_rgb_) return true;
  void* p = nullptr;
  if (hipHostMalloc(&p, sizeof(float) * 3 * kHostUnits, hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  h_rgb_ = static_cast<float*>(p);
  return true;
}

bool BatchRenderer::prepare(const UnitLaunch& U, const std::vector<Pose>& poses, hipStream_t stream,
                            std::string* err) {
  const size_t np = poses.size();
  if (!ev0_ && (hipEventCreate(&ev0_) != hipSuccess || hipEventCreate(&ev1_) != hipSuccess)) {
    if (err) *err = "batch: event creation failed";
    return false;
  }
  const size_t units = np * (size_t)U.omm_count;
  if (!grow(&d_poses_, &poses_cap_, np, err)) return false;
  if (!grow(&d_colours_, &colours_cap_, units, err)) return false;
  if (hipMemcpyAsync(d_poses_, poses.data(), sizeof(Pose) * np, hipMemcpyHostToDevice, stream) != hipSuccess) {
    if (err) *err = "batch: pose upload failed";
    return false;
  }
  return true;
}

bool BatchRenderer::tune(const DeviceScene& scene, UnitLaunch U, const std::vector<Pose>& poses, int repeats,
                         hipStream_t stream, std::vector<TuneTrial>* trials, LaunchShape* best, std::string* err) {
  trials->clear();
  if (poses.empty() || U.omm_count == 0) {
    if (err) *err = "autotune: empty batch";
    return false;
  }
  if (!prepare(U, poses, stream, err)) return false;
  U.poses = d_poses_;
  U.pose_count = (int)poses.size();
  U.pose_base = 0;
  U.colours = d_colours_;
  U.stats = nullptr;
  U.samples = nullptr;
  const int capacity = render_units_capacity(scene, U);
  double best_ms = 1e300;
  for (const LaunchShape& sh : LaunchTuner::candidates(capacity)) {
    U.units_per_grab = sh.units_per_grab;
    U.blocks = sh.blocks;
    U.traversal = sh.traversal;
    if (!launch_render_units(scene, U, stream, err)) return false;  // untimed: caches, clocks
    double ms_min = 1e300;
    for (int r = 0; r < std::max(repeats, 1); ++r) {
      (void)hipEventRecord(ev0_, stream);
      if (!launch_render_units(scene, U, stream, err)) return false;
      (void)hipEventRecord(ev1_, stream);
      if (hipEventSynchronize(ev1_) != hipSuccess) {
        if (err) *err = "autotune: render failed";
        return false;
      }
      float ms = 0.0f;
      (void)hipEventElapsedTime(&ms, ev0_, ev1_);
      ms_min = std::min(ms_min, (double)ms);
    }
    trials->push_back(TuneTrial{sh, ms_min});
    if (ms_min < best_ms) {
      best_ms = ms_min;
      *best = sh;
    }
  }
  return true;
}

bool BatchRenderer::render(const DeviceScene& scene, UnitLaunch U, const std::vector<Pose>& poses, float* rgb,
                           hipStream_t stream, double* gpu_ms, std::string* err) {
  const size_t np = poses.size();
  *gpu_ms = 0.0;
  if (np == 0) return true;
  const size_t units = np * (size_t)U.omm_count;
  if (!prepare(U, poses, stream, err)) return false;
  U.poses = d_poses_;
  U.pose_count = (int)np;
  U.pose_base = 0;
  U.colours = d_colours_;
  (void)hipEventRecord(ev0_, stream);
  if (!launch_render_units(scene, U, stream, err)) return false;
  (void)hipEventRecord(ev1_, stream);
  // The colours are packed on the device, the first piece right behind the
  // render.  Small batches' go straight to pinned memory (a blocking copy
  // waits 20 us for any size); larger ones' are copied to the caller in
  // pieces of kPackUnits units.  1.1 M units: 1.1 ms less than a float4 copy
  // that the host repacks.
  const bool pinned = rgb && units <= kHostUnits && host_rgb();
  // without memory to pack into, the host repacks after all
  std::string no_memory;
  const bool packs = rgb && (pinned || grow(&d_rgb_, &rgb_cap_, 3 * std::min(kPackUnits, units), &no_memory));
  if (rgb && !packs) (void)hipGetLastError();
  const auto pack = [&](size_t first) {
    return launch_pack_rgb(d_colours_ + first, std::min(kPackUnits, units - first), pinned ? h_rgb_ : d_rgb_, stream,
                           err);
  };
  if (packs && !pack(0)) {
    (void)hipStreamSynchronize(stream);
    return false;
  }
  if ((pinned ? hipStreamSynchronize(stream) : hipEventSynchronize(ev1_)) != hipSuccess) {
    if (err) *err = "batch: render failed";
    return false;
  }
  float ms = 0.0f;
  (void)hipEventElapsedTime(&ms, ev0_, ev1_);
  *gpu_ms = ms;
  if (pinned) {
    memcpy(rgb, h_rgb_, sizeof(float) * 3 * units);
    return true;
  }
  if (rgb && !packs) {
    std::vector<float4> tmp(units);
    if (hipMemcpy(tmp.data(), d_colours_, sizeof(float4) * units, hipMemcpyDeviceToHost) != hipSuccess) {
      if (err) *err = "batch: readback failed";
      return false;
    }
    for (size_t i = 0; i < units; ++i) {
      rgb[3 * i] = tmp[i].x;
      rgb[3 * i + 1] = tmp[i].y;
      rgb[3 * i + 2] = tmp[i].z;
    }
    return true;
  }
  for (size_t first = 0; rgb && first < units; first += kPackUnits) {
    if (first != 0 && !pack(first)) return false;
    if (hipMemcpyAsync(rgb + 3 * first, d_rgb_, sizeof(float) * 3 * std::min(kPackUnits, units - first),
                       hipMemcpyDeviceToHost, stream) != hipSuccess ||
        hipStreamSynchronize(stream) != hipSuccess) {
      if (err) *err = "batch: readback failed";
      return false;
    }
  }
  return true;
}

}  // namespace eye
