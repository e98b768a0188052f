"""Host-side rules of the library that are plain arithmetic
(rtspatial_amd/csrc/rules.h), compiled for the host and run on the CPU."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def evaluate(tmp_path, body):
    """The integers that a C++ function body prints."""
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("no g++")
    src, exe = tmp_path / "rules.cpp", tmp_path / "rules"
    src.write_text('#include <cstdio>\n#include <initializer_list>\n#include "rules.h"\nusing namespace rts;\nint main() {\n'
                   f"{body}\n}}\n")
    subprocess.run([gxx, "-std=c++17", "-Wall", f"-I{ROOT}/rtspatial_amd/csrc", str(src), "-o",
                    str(exe)], check=True)
    out = subprocess.run([str(exe)], stdout=subprocess.PIPE, check=True).stdout.decode()
    return [int(x) for x in out.split()]


def test_sort_reads_only_its_own_devices_memory_in_place(tmp_path):
    got = evaluate(tmp_path, """
  static uint32_t m[100];
  auto t = [&](bool dev, int owner, int device, int in, int ko, int vo) {
    std::printf("%d ", (int)sort_reads_in_place(dev, owner, device, m + in, m + ko, m + vo, 20));
  };
  t(true, 0, 0, 0, 20, 40);   // device memory, apart from both outputs
  t(true, 1, 1, 60, 20, 40);
  t(false, 0, 0, 0, 20, 40);  // host memory
  t(true, 1, 0, 0, 20, 40);   // another device's
  t(true, 0, 1, 0, 20, 40);
  t(true, 0, 0, 20, 20, 40);  // also an output
  t(true, 0, 0, 40, 20, 40);
  t(true, 0, 0, 25, 10, 60);  // overlapping an output's end, or its start
  t(true, 0, 0, 25, 70, 44);
  t(true, 0, 0, 20, 0, 40);   // next to both
""")
    assert got == [1, 1, 0, 0, 0, 0, 0, 0, 0, 1]


def test_a_wave_with_one_query_can_log_all_of_it(tmp_path):
    # Calls with a wave to a query, and fewer queries than fill a round of waves
    # over the XCDs: each wave's share of the log is a query's longest log.
    got = evaluate(tmp_path, """
  for (uint32_t n = 1; n <= 4096; n++)
    if (query_log_entries(n) / persistent_waves(n, 1, 8192) < kLogQueryMax) std::printf("%u ", n);
  std::printf("0 %u %u %u", persistent_waves(1, 1, 8192), persistent_waves(8193, 4, 8192),
              persistent_waves(1u << 26, 4, 8192));
  std::printf(" %d %d", (int)(query_log_entries(32768) == kLogMinEntries),
              (int)(query_log_entries(1u << 26) == kLogMaxEntries));
""")
    assert got == [0, 8, 2056, 8192, 1, 1]


def test_leaves_are_not_above_the_leaf_blocks(tmp_path):
    # At every depth: nodes above level D - 1, and neither that level's nor the
    # leaves, up to the last of 2^30 - 1.
    got = evaluate(tmp_path, """
  for (uint32_t d = 1; d <= 10; d++) {
    uint64_t leaf0 = 0, last = 0;  // last: first node of level d - 1
    for (uint32_t k = 0; k < d; k++) { last = leaf0; leaf0 = 8 * leaf0 + 1; }
    const uint64_t n = d == 10 ? (1ull << 30) - 1 : 1ull << (3 * d);
    uint64_t wrong = 0;
    for (const uint64_t i : {(uint64_t)0, last - 1, last, leaf0 - 1, leaf0, leaf0 + n / 3,
                       (uint64_t)((1ull << 29) - 1), (uint64_t)(1ull << 29),
                       (uint64_t)((1ull << 29) + 7), leaf0 + n - 1})
      if (i < leaf0 + n && i != ~0ull)
        wrong += above_leaf_blocks((uint32_t)i, (uint32_t)leaf0) != (i < last);
    std::printf("%d ", (int)wrong);
  }
""")
    assert got == [0] * 10
