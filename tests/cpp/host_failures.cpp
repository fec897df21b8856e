// What the host runtime does when the device refuses memory, on the CPU: this
// program defines the HIP calls that libvdbgpu.so makes (device memory is host
// memory, kernels do nothing but what a scenario puts in their place) and
// fails one allocation at a time.
//
// Build: g++ -std=c++17 -rdynamic -Iinclude tests/cpp/host_failures.cpp -Lvdb_mapping_amd -lvdbgpu
// Usage: host_failures SCENARIO   (exit status 0 = all checks hold)
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <string>
#include <vector>

#include "vdbgpu.h"

// ------------------------------------------------------- stand-in for HIP --

namespace {

constexpr int kOutOfMemory = 2;  // hipErrorOutOfMemory

struct Dim3 {
  uint32_t x, y, z;
};

// Kernels by host function (the library registers them before this program's
// own globals are built).
std::map<const void*, std::string>& names() {
  static std::map<const void*, std::string> n;
  return n;
}
std::map<std::string, std::function<void(void**)>> g_kernels;  // stand-ins by kernel name
std::map<std::string, int> g_launches;
std::map<const void*, size_t> g_blocks;  // live allocations
long g_fail_in = 0;                      // the n-th allocation from here fails (0: none)
bool g_failed = false;
size_t g_pinned = 0;  // bytes ever allocated as pinned memory
size_t g_read = 0;    // bytes ever copied from the device

// The plain name of a kernel's symbol, _ZN6vdbgpu<length>k_name...
std::string plain(const char* mangled) {
  const char* p = std::strstr(mangled, "k_");
  if (!p) return mangled;
  const char* d = p;
  while (d > mangled && d[-1] >= '0' && d[-1] <= '9') --d;
  return std::string(p, std::strtoul(d, nullptr, 10));
}

int allocate(void** p, size_t bytes) {
  *p = nullptr;
  if (g_fail_in > 0 && --g_fail_in == 0) {
    g_failed = true;
    return kOutOfMemory;
  }
  *p = std::calloc(1, bytes ? bytes : 1);
  g_blocks[*p] = bytes;
  return 0;
}

int release(void* p) {
  if (!p) return 0;
  if (!g_blocks.erase(p)) {
    std::printf("free of an unknown block\n");
    std::exit(2);
  }
  std::free(p);
  return 0;
}

Dim3 g_grid, g_block;

}  // namespace

extern "C" {
void** __hipRegisterFatBinary(const void*) {
  static void* module;
  return &module;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  names()[host] = plain(name);
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t, void*) {
  g_grid = grid;
  g_block = block;
  return 0;
}
int __hipPopCallConfiguration(Dim3* grid, Dim3* block, size_t* shared, void** stream) {
  *grid = g_grid;
  *block = g_block;
  *shared = 0;
  *stream = nullptr;
  return 0;
}
int hipLaunchKernel(const void* host, Dim3, Dim3, void** args, size_t, void*) {
  const std::string& name = names()[host];
  ++g_launches[name];
  auto k = g_kernels.find(name);
  if (k != g_kernels.end()) k->second(args);
  return 0;
}
int hipMalloc(void** p, size_t bytes) { return allocate(p, bytes); }
int hipFree(void* p) { return release(p); }
int hipHostMalloc(void** p, size_t bytes, unsigned) {
  g_pinned += bytes;
  return allocate(p, bytes);
}
int hipHostFree(void* p) { return release(p); }
int hipHostGetDevicePointer(void** d, void* h, unsigned) {
  *d = h;
  return 0;
}
int hipMemcpy(void* d, const void* s, size_t n, int kind) {
  if (kind == 2) g_read += n;  // hipMemcpyDeviceToHost
  std::memcpy(d, s, n);
  return 0;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void*) { return hipMemcpy(d, s, n, kind); }
int hipMemsetAsync(void* d, int v, size_t n, void*) {
  std::memset(d, v, n);
  return 0;
}
int hipGetDevice(int* d) { return *d = 0; }
int hipSetDevice(int) { return 0; }
int hipGetDeviceCount(int* n) {
  *n = 1;
  return 0;
}
int hipDeviceGetAttribute(int* v, int, int) { return *v = 0; }  // 256 CUs by default, no virtual memory: plain pools
const char* hipGetErrorString(int e) { return e == kOutOfMemory ? "out of memory" : "error"; }
int hipGetLastError() { return 0; }
int hipStreamCreateWithFlags(void** s, unsigned) {
  *s = &g_grid;
  return 0;
}
int hipStreamDestroy(void*) { return 0; }
int hipStreamSynchronize(void*) { return 0; }
int hipStreamWaitEvent(void*, void*, unsigned) { return 0; }
int hipEventCreate(void** e) {
  *e = &g_grid;
  return 0;
}
int hipEventCreateWithFlags(void** e, unsigned) { return hipEventCreate(e); }
int hipEventDestroy(void*) { return 0; }
int hipEventQuery(void*) { return 0; }
int hipEventRecord(void*, void*) { return 0; }
int hipEventSynchronize(void*) { return 0; }
}  // extern "C"

// -------------------------------------------------------------- scenarios --

#define CHECK(cond)                                                       \
  do {                                                                    \
    if (!(cond)) {                                                        \
      std::printf("%s:%d: %s\n", __FILE__, __LINE__, #cond);              \
      std::exit(1);                                                       \
    }                                                                     \
  } while (0)

namespace {

template <class T>
T& arg(void** args, int i) {
  return *static_cast<T*>(args[i]);
}

vdbgpu_map* new_map(bool fast) {
  vdbgpu_map* m = nullptr;
  CHECK(vdbgpu_create(0.1, &m) == VDBGPU_OK);
  vdbgpu_config c{};
  c.max_range = 10.0;
  c.fast_mode = fast;
  c.prob_hit = 0.9;
  c.prob_miss = 0.1;
  c.prob_thres_min = 0.12;
  c.prob_thres_max = 0.97;
  CHECK(vdbgpu_set_config(m, &c) == VDBGPU_OK);
  CHECK(vdbgpu_add_source(m, "s", 10.0, 0.0) == VDBGPU_OK);
  return m;
}

void close_map(vdbgpu_map* m) {
  vdbgpu_destroy(m);
  CHECK(g_blocks.empty());
}

int edit(vdbgpu_map* m) {
  const float p[3] = {0.05f, 0.05f, 0.05f};
  return vdbgpu_set_points(m, p, 1, 12, 1);
}

int raytrace(vdbgpu_map* m) {
  const double o[3] = {0, 0, 0}, d[3] = {1, 0, 0}, len = 5;
  uint8_t hit = 0;
  double end[3];
  return vdbgpu_raytrace(m, 1, o, d, &len, &hit, end);
}

// A topology snapshot whose node bitmaps cannot grow: k_snapshot_nodes has put
// nodes into the hash that the bitmaps have no room for, so no query may run
// until a later build is through.
void snapshot() {
  struct Info {  // RtInfo
    int bbox[6];
    unsigned int nodes, leaves;
  };
  unsigned int nodes = 1;
  g_kernels["k_compact"] = [](void** a) { *arg<unsigned int*>(a, 3) = 1; };  // one listed leaf
  g_kernels["k_snapshot_nodes"] = [&](void** a) { arg<Info*>(a, 3)->nodes = nodes; };
  bool through = false;
  for (long k = 1; !through; ++k) {  // a map's first build
    vdbgpu_map* m = new_map(true);
    CHECK(edit(m) == VDBGPU_OK);
    g_fail_in = k;
    g_failed = false;
    const int r = vdbgpu_integrate(m);
    through = !g_failed;
    g_fail_in = 0;
    CHECK(r == (g_failed ? VDBGPU_DEVICE_ERROR : VDBGPU_OK));
    CHECK(raytrace(m) == (g_failed ? VDBGPU_NO_INTERSECTOR : VDBGPU_OK));
    CHECK(vdbgpu_integrate(m) == VDBGPU_OK && raytrace(m) == VDBGPU_OK);
    close_map(m);
    CHECK(k > 1 || !through);
  }
  through = false;
  for (long k = 1; !through; ++k) {
    vdbgpu_map* m = new_map(true);
    CHECK(edit(m) == VDBGPU_OK && vdbgpu_integrate(m) == VDBGPU_OK);
    CHECK(raytrace(m) == VDBGPU_OK);
    // the map grows: every allocation of the next build fails in turn
    nodes = 5000;
    CHECK(edit(m) == VDBGPU_OK);
    g_fail_in = k;
    g_failed = false;
    const int r = vdbgpu_integrate(m);
    through = !g_failed;
    g_fail_in = 0;
    CHECK(r == (g_failed ? VDBGPU_DEVICE_ERROR : VDBGPU_OK));
    const int before = g_launches["k_raytrace"];
    CHECK(raytrace(m) == (g_failed ? VDBGPU_NO_INTERSECTOR : VDBGPU_OK));
    CHECK(g_launches["k_raytrace"] == before + (g_failed ? 0 : 1));
    // a later build is whole again
    CHECK(vdbgpu_integrate(m) == VDBGPU_OK && raytrace(m) == VDBGPU_OK);
    nodes = 1;
    close_map(m);
    CHECK(k > 1 || !through);  // the growth allocates
  }
}

// Map sections: pinned staging comes a few chunks a read and stays bounded; a
// refused chunk is done without, a refused device buffer fails the read alone.
void section() {
  unsigned int leaves = 1100;
  g_kernels["k_compact"] = [](void** a) { *arg<unsigned int*>(a, 3) = 1; };
  g_kernels["k_scan_u64"] = [&](void** a) { *arg<unsigned int*>(a, 3) = leaves; };
  const int32_t box[6] = {0, 0, 0, 255, 255, 255};  // 32,768 cells
  std::vector<int32_t> o(3 * 32768);
  std::vector<float> v((size_t)512 * 32768);
  std::vector<uint64_t> w(8 * 32768);
  auto read = [&](vdbgpu_map* m) {
    return vdbgpu_export_section(m, box, 1, o.data(), v.data(), w.data(), 32768);
  };
  vdbgpu_map* m = new_map(false);
  CHECK(edit(m) == VDBGPU_OK);
  const size_t start = g_pinned;
  for (int k = 0; k < 40; ++k) {
    const size_t before = g_pinned;
    leaves = k < 20 ? 1100 : 30000;
    CHECK(read(m) == leaves);
    CHECK(g_pinned - before <= (size_t)leaves * 2124 / 3 + (1 << 20));
  }
  CHECK(g_pinned - start <= 16u << 20);
  CHECK(vdbgpu_release_scratch(m) == VDBGPU_OK && read(m) == leaves);
  close_map(m);
  bool through = false;
  for (long k = 1; !through; ++k) {
    m = new_map(false);
    CHECK(edit(m) == VDBGPU_OK);
    leaves = 200;
    CHECK(read(m) == 200);
    leaves = 3000;
    g_fail_in = k;
    g_failed = false;
    const int64_t n = read(m);
    through = !g_failed;
    g_fail_in = 0;
    CHECK(n == 3000 || (g_failed && n == -1));
    CHECK(read(m) == 3000 && read(m) == 3000);
    close_map(m);
    CHECK(k > 1 || !through);
  }
}

// An update set's export reads its entries, whatever room the set has.
void update_export() {
  constexpr int kLeaves = 100;
  g_kernels["k_compact"] = [](void** a) { *arg<unsigned int*>(a, 3) = kLeaves; };
  vdbgpu_map* m = new_map(false);
  vdbgpu_tuning t{256, 32, 16, 0.5, 1, 8};
  CHECK(vdbgpu_set_tuning(m, &t) == VDBGPU_OK);
  const std::vector<float> p(3 * 2000, 0.5f);
  const double origin[3] = {0, 0, 0};
  CHECK(vdbgpu_accumulate(m, "s", p.data(), 2000, 12, origin, 0) == VDBGPU_OK);
  std::vector<int32_t> o(3 * kLeaves);
  std::vector<uint64_t> v(8 * kLeaves), h(8 * kLeaves);
  const size_t before = g_read;
  CHECK(vdbgpu_export_update(m, "s", o.data(), v.data(), h.data(), kLeaves) == kLeaves);
  CHECK(g_read - before <= kLeaves * 136 + 4096);
  g_fail_in = 1;
  CHECK(vdbgpu_export_update(m, "s", o.data(), v.data(), h.data(), kLeaves) == -1);
  CHECK(vdbgpu_export_update(m, "s", o.data(), v.data(), h.data(), kLeaves - 1) == -kLeaves);
  close_map(m);
}

// The point export: tables for the leaves there are, and the host's own way when the
// device has no room for tables or points.
void points() {
  struct StatusHead {  // Status
    unsigned long long total, voxels, rays;
    unsigned int error, overflow, entries, leaf_count;
  };
  g_kernels["k_compact"] = [](void** a) { *arg<unsigned int*>(a, 3) = 1; };
  g_kernels["k_map_insert"] = [](void** a) { arg<StatusHead*>(a, 10)->leaf_count = 1; };
  g_kernels["k_point_leaves"] = [](void** a) {
    arg<StatusHead*>(a, 6)->entries = 1;
    arg<StatusHead*>(a, 6)->total = 1;
  };
  std::vector<float> xyz(3);
  bool through = false;
  for (long k = 1; !through; ++k) {
    vdbgpu_map* m = new_map(false);
    // many edits of one leaf: the host's bound of the leaf count is far above it
    for (int i = 0; i < 50; ++i) CHECK(edit(m) == VDBGPU_OK);
    vdbgpu_stats before{}, after{};
    CHECK(vdbgpu_get_stats(m, &before) == VDBGPU_OK);
    for (int i = 0; i < 50; ++i) CHECK(edit(m) == VDBGPU_OK);
    g_fail_in = k;
    g_failed = false;
    const int64_t n = vdbgpu_export_active_points(m, xyz.data(), 1);
    through = !g_failed;
    g_fail_in = 0;
    // (kernels write nothing here, so the host finds the leaf without an active voxel)
    CHECK(n == (g_failed ? 0 : 1));
    CHECK(vdbgpu_export_active_points(m, xyz.data(), 1) == 1);
    CHECK(vdbgpu_get_stats(m, &after) == VDBGPU_OK);
    CHECK(after.scratch_bytes - before.scratch_bytes <= 24 + 12);
    close_map(m);
    CHECK(k > 1 || !through);
  }
}

}  // namespace

int main(int argc, char** argv) {
  const std::map<std::string, void (*)()> scenarios = {{"snapshot", snapshot}, {"section", section}, {"update_export", update_export}, {"points", points}};
  const auto s = argc > 1 ? scenarios.find(argv[1]) : scenarios.end();
  if (s == scenarios.end()) return 3;
  s->second();
  std::printf("%s ok\n", argv[1]);
  return 0;
}
