// The sorted order of projected grids, as the gather reads it (the C ABI exports
// the reference's order, sorted again from the input's).
//
//   sort_order DIR TARGET N...
//
// For each N reads DIR/p4_N.f32 (float4 particles) and DIR/h_N.f32, builds the
// grid with TARGET particles per cell and writes the sorted cell keys and input
// indices to DIR/key_N.u32 and DIR/perm_N.u32.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <string>
#include <vector>

#include "gridbuild.hpp"

namespace {

template <class T>
std::vector<T> read_file(const std::string& path, size_t n) {
  std::vector<T> v(n);
  FILE* f = std::fopen(path.c_str(), "rb");
  if (!f || std::fread(v.data(), sizeof(T), n, f) != n) {
    std::fprintf(stderr, "cannot read %s\n", path.c_str());
    std::exit(2);
  }
  std::fclose(f);
  return v;
}

void write_file(const std::string& path, const std::vector<uint32_t>& v) {
  FILE* f = std::fopen(path.c_str(), "wb");
  if (!f || std::fwrite(v.data(), 4, v.size(), f) != v.size()) std::exit(2);
  std::fclose(f);
}

void sort_one(const std::string& dir, uint64_t target, uint64_t n) {
  const std::string tag = "_" + std::to_string(n);
  const auto p4 = read_file<float4>(dir + "/p4" + tag + ".f32", n);
  const auto h = read_file<float>(dir + "/h" + tag + ".f32", n);
  ilc::dbuf<float4> dp;
  ilc::dbuf<float> dh;
  ILC_HIP(hipMemcpy(dp.ensure(n), p4.data(), sizeof(float4) * n, hipMemcpyHostToDevice));
  ILC_HIP(hipMemcpy(dh.ensure(n), h.data(), sizeof(float) * n, hipMemcpyHostToDevice));
  ilc::grid_store gs;
  ilc::grid_scratch sc;
  const int parts = int(std::min<uint64_t>(1024, (n + ilc::kBlock - 1) / ilc::kBlock));
  sc.bbox_partial.ensure(size_t(parts) * ilc::kBboxWords);
  sc.bbox_dev.ensure(1);
  sc.flags.ensure(2);
  ilc::launch_bbox(dp.p, dh.p, n, sc.bbox_partial.p, parts, sc.bbox_dev.p, nullptr);
  ilc::bbox_result bb;
  ILC_HIP(hipMemcpy(&bb, sc.bbox_dev.p, sizeof(bb), hipMemcpyDeviceToHost));
  int32_t kz0 = 0;
  const ilc::grid_params g = ilc::plan_grid(bb, n, target, ILC_MODE_REFERENCE, &kz0);
  ilc::enqueue_grid_build(gs, sc, dp.p, dh.p, n, g, kz0, bb.max_h, ILC_KERNEL_QUARTIC_REF,
                          sc.flags.p, true, nullptr);
  std::vector<uint32_t> key(n), perm(n);
  ILC_HIP(hipMemcpy(key.data(), gs.key.p, 4 * n, hipMemcpyDeviceToHost));
  ILC_HIP(hipMemcpy(perm.data(), gs.perm.p, 4 * n, hipMemcpyDeviceToHost));
  write_file(dir + "/key" + tag + ".u32", key);
  write_file(dir + "/perm" + tag + ".u32", perm);
  std::printf("sorted %llu\n", (unsigned long long)n);
  std::fflush(stdout);
}

}  // namespace

int main(int argc, char** argv) {
  if (argc < 4) return 2;
  try {
    for (int k = 3; k < argc; ++k)
      sort_one(argv[1], std::strtoull(argv[2], nullptr, 10), std::strtoull(argv[k], nullptr, 10));
  } catch (const std::exception& e) {
    std::fprintf(stderr, "%s\n", e.what());
    return 1;
  }
  return 0;
}
