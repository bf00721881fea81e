"""Which of the library's counters a launch meets on (csrc/kernels/sync_regions.h), host code alone: launches that may
run side by side have workspaces of their own, and no two such workspaces may ever share a region."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = r"""
#include <cstdio>
#include <thread>
#include <vector>
#include "sync_regions.h"
using namespace mlakv;
template <int N>
void Answer() {
  static SyncRegions<N> regions;
  unsigned long long address, bytes;
  while (std::scanf("%llu %llu", &address, &bytes) == 2) {
    std::printf("%d\n", regions.Of(WorkspaceName(reinterpret_cast<void*>(address), bytes)));
  }
}
int Threads() {  // eight threads name the same 300 workspaces, each in another order
  static SyncRegions<256> regions;
  std::vector<std::vector<int>> seen(8, std::vector<int>(300));
  std::vector<std::thread> threads;
  for (int t = 0; t < 8; ++t) {
    threads.emplace_back([&, t] {
      for (int i = 0; i < 300; ++i) {
        const int w = (i * 7 + t * 41) % 300;
        const int region = regions.Of(WorkspaceName(reinterpret_cast<void*>(0x7000000000ull + w * 0x2000000ull), 0x2000000));
        if (region >= 0) seen[t][w] = region;
        if (region < 0) seen[t][w] = -1;
      }
    });
  }
  for (auto& thread : threads) thread.join();
  for (int w = 0; w < 300; ++w) std::printf("%d %d\n", regions.Of(WorkspaceName(reinterpret_cast<void*>(0x7000000000ull + w * 0x2000000ull), 0x2000000)), w);
  for (const auto& one : seen) {
    for (int w = 0; w < 300; ++w) std::printf("%d %d\n", one[w], w);
  }
  return 0;
}
int main(int argc, char** argv) {
  if (argc > 1 && argv[1][0] == 't') return Threads();
  if (argc > 1 && argv[1][0] == 'p') {
    for (int parts = 0; parts <= 8; ++parts) std::printf("%d\n", PartsWithoutCounters(parts));
    return 0;
  }
  if (argc > 1 && argv[1][0] == 's') Answer<16>(); else Answer<4096>();
}
"""
PAGE = 8 << 20


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    source = tmp_path_factory.mktemp("sync_regions") / "regions.cpp"
    source.write_text(PROGRAM)
    binary = source.with_suffix("")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-Wall", "-Werror", "-I",
                    os.path.join(ROOT, "ascend-moe-engine_amd", "csrc", "kernels"), str(source), "-o", str(binary)], check=True)

    def run(mode, workspaces=()):
        text = "".join(f"{address} {size}\n" for address, size in workspaces)
        out = subprocess.run([str(binary), mode], input=text, capture_output=True, text=True, check=True).stdout
        return [tuple(map(int, line.split())) for line in out.splitlines()]

    return run


@pytest.mark.parametrize("size,gap", [(16 << 20, 0), (17_000_000 // 256 * 256, 0), (24 << 20, 512), (2 * PAGE, 256), (2 * PAGE - 256, 0),
                                      (65_792, 0), (16, 0), (300 << 20, 4096)])
def test_workspaces_that_do_not_overlap_have_regions_of_their_own(program, size, gap):
    workspaces = [(0x7F0000000100 + i * (size + gap), size) for i in range(1000)]
    given = [region for region, in program("many", workspaces * 2)]
    assert min(given) >= 0 and max(given) < 4096
    assert len(set(given[:1000])) == 1000 and given[1000:] == given[:1000]


def test_large_and_small_workspaces_side_by_side(program):
    workspaces, at = [], 0x7F0000000100
    for i in range(1500):
        size = (32_768, 2 * PAGE, 2 * PAGE - 16, 40 << 20, 16)[i % 5]
        workspaces.append((at, size))
        at += size
    given = [region for region, in program("many", workspaces)]
    assert min(given) >= 0 and len(set(given)) == 1500


def test_a_seventeenth_workspace_of_sixteen_regions_gets_none(program):
    workspaces = [(0x7F0000000000 + i * (24 << 20), 24 << 20) for i in range(17)]
    given = [region for region, in program("sixteen", workspaces + workspaces[::-1])]
    assert sorted(given[:16]) == list(range(16)) and given[16] == -1
    assert given[17:] == given[:17][::-1]  # those handed out stay, and the seventeenth still gets none


def test_a_workspace_carved_anew_keeps_to_few_names(program):
    # 16.9 MB anywhere in 256 MiB, 4000 times: at most a region per page
    workspaces = [(0x7F0000000000 + (i * 7919 * 512) % (256 << 20), 16_909_312) for i in range(4000)]
    given = [region for region, in program("many", workspaces)]
    assert min(given) >= 0 and len(set(given)) <= 34


def test_threads_agree_on_the_regions(program):
    given = program("threads")
    held = dict((w, region) for region, w in given[:300])
    assert sum(region >= 0 for region in held.values()) == 256
    assert len({region for region in held.values() if region >= 0}) == 256
    assert all(region in (held[w], -1) for region, w in given)  # (-1 for the 44 that came last)
    assert all(region == held[w] for region, w in given if held[w] < 0 or region >= 0)


def test_what_a_launch_without_counters_falls_to(program):
    # five to eight workgroups per unit: the 64-head kernel; two and four: one
    assert [parts for parts, in program("parts")] == [0, 1, 1, 1, 1, 0, 0, 0, 0]
