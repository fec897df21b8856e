"""CPU check of the update set's probe sequence (device_common.h map_hash and kUpdStep): at the highest load the host
allows, full columns of four leaves, one layer of leaves and scattered ones need about the probes that linear probing of
independent keys needs, (1 + 1 / (1 - load)) / 2 of them for a key that is there; the sequence reaches every slot."""
import os
import subprocess


ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include <cstdio>
#include <random>
#include <vector>
#include "device_common.h"
using namespace vdbgpu;
static int failures = 0;
static void check(const char* what, const std::vector<uint64_t>& keys, uint32_t cap) {
  std::vector<uint64_t> slot(cap, ~0ull);
  auto probes = [&](uint64_t key) {
    uint32_t h = map_hash(key) & (cap - 1), n = 1;
    for (; slot[h] != ~0ull && slot[h] != key; ++n) h = (h + kUpdStep) & (cap - 1);
    slot[h] = key;
    return n;
  };
  for (uint64_t k : keys) probes(k);
  double sum = 0;
  for (uint64_t k : keys) sum += probes(k);
  const double load = (double)keys.size() / cap, mean = sum / keys.size(), want = (1 + 1 / (1 - load)) / 2;
  std::printf("%s: load %.2f, %.2f probes, %.2f expected\n", what, load, mean, want);
  failures += !(mean < 1.15 * want);
}
int main() {
  for (uint32_t log2cap : {12u, 16u, 20u}) {
    const uint32_t cap = 1u << log2cap, n = cap / 2;
    std::mt19937 rng(log2cap);
    const int side = (int)std::sqrt(n / 4.0) + 1;
    std::vector<uint64_t> columns, layer, any;
    for (int x = 0; x < side && columns.size() < n; ++x)
      for (int y = 0; y < side && columns.size() < n; ++y)
        for (int z = 0; z < 4; ++z) columns.push_back(leaf_key(8 * (x - 7), 8 * (y + 3), 8 * (z - 4)));
    check("columns", columns, cap);
    for (int x = 0; x < 2 * side && layer.size() < n; ++x)
      for (int y = 0; y < 2 * side && layer.size() < n; ++y) layer.push_back(leaf_key(8 * x, 8 * y, 0));
    check("layer", layer, cap);
    while (any.size() < n)
      any.push_back(leaf_key(8 * (int)(rng() % 4000), 8 * (int)(rng() % 4000), 8 * (int)(rng() % 4000)));
    check("scattered", any, cap);
    std::vector<char> seen(cap, 0);
    uint32_t h = 3, count = 0;
    for (uint32_t p = 0; p < cap; ++p, h = (h + kUpdStep) & (cap - 1)) count += !seen[h], seen[h] = 1;
    failures += count != cap;
  }
  std::printf("%d failures\n", failures);
  return failures != 0;
}
"""


def test_probe_lengths(tmp_path):
    src, exe = tmp_path / "update_hash.hip", str(tmp_path / "update_hash")
    src.write_text(SRC)
    subprocess.run(["hipcc", "--offload-host-only", "-O2", "-std=c++17",
                    "-I" + os.path.join(ROOT, "vdb_mapping_amd", "csrc"), str(src), "-o", exe], check=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout
