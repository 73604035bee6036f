"""The host's and the kernels' reckoning of work-group placement (``csrc/placement.h``) and the
per-op calls' counter blocks (``csrc/op_blocks.h``), on the CPU: the header is compiled into a
small program that counts what it finds wrong."""
from __future__ import annotations

import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "diffusorrt_amd",
                    "csrc")


def _run(tmp_path, body, *headers):
    src = tmp_path / "t.cpp"
    src.write_text("#include <cstdio>\n#include <initializer_list>\n" + "".join(f'#include {h if h[0] == "<" else chr(34) + h + chr(34)}\n' for h in headers) +
                   "int main() {\n  int wrong = 0;\n" + body + "  return wrong != 0;\n}\n")
    exe = tmp_path / "t"
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, str(src), "-o", str(exe), "-pthread"],
                   check=True, capture_output=True, text=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout


@pytest.mark.parametrize("n_xcc", [1, 2, 4, 8])
def test_rotation_is_the_same_for_every_work_group(tmp_path, n_xcc):
    _run(tmp_path, """
  const int n = %d;
  for (int r = 0; r < n; ++r)
    for (int i = 0; i < 512; ++i)
      if (drt::xcd_rotation((i + r) %% n, i, n) != r) { ++wrong; std::printf("r %%d i %%d\\n", r, i); }
""" % n_xcc, "placement.h")


def test_settled_word_keeps_other_reports(tmp_path):
    # 2: a bounded wait, 4: the fp16 range
    _run(tmp_path, """
  for (int r = 0; r < 8; ++r)
    for (int other : {0, 2, 4, 6}) {
      const int moved = 1 | drt::placement_bit(r);
      wrong += drt::settled_word(other, r, true) != other;
      wrong += drt::settled_word(moved | other, r, true) != other;
      wrong += drt::settled_word(moved | other, r, false) != (moved | other);
      for (int q = 0; q < 8; ++q) {
        if (q == r) continue;
        wrong += drt::settled_word(moved | other, q, true) != (moved | other);
        const int two = moved | drt::placement_bit(q) | other;
        wrong += drt::settled_word(two, r, true) != two || drt::settled_word(two, q, true) != two;
      }
      wrong += drt::settled_word(moved | other, -1, true) != (moved | other);
    }
""", "placement.h")


def test_a_launch_cut_in_two_leaves_a_counter(tmp_path):
    # KS slices of a block count in one L2, or (one launch) some in another: each L2 works on
    # its own copy of the counter and either may be the one written back last. The last of a
    # block sets it to zero. Later launches run whole; no remainder may come back to zero.
    _run(tmp_path, """
  for (int KS = 2; KS <= 16; ++KS)
    for (int a = 1; a < KS; ++a)
      for (int back = 0; back < 2; ++back) {
        int c = back ? a : KS - a;
        for (int launch = 0; launch < 64; ++launch) {
          wrong += c == 0;
          const int ks = 2 + (7 * KS + 5 * launch) % 15;  // another linear's slices
          for (int i = 0; i < ks; ++i)
            if (c++ == ks - 1) c = 0;
        }
        wrong += c == 0;
      }
  int c = 0;
  for (int i = 0; i < 5; ++i) if (c++ == 4) c = 0;
  wrong += c != 0;
""", "placement.h")


def test_a_wrong_xcd_count_shows(tmp_path):
    # eight XCDs taken for four or two: some of the first eight work-groups disagree
    _run(tmp_path, """
  for (int n : {2, 4})
    for (int r = 0; r < 8; ++r) {
      bool differs = false;
      for (int i = 0; i < 8; ++i) differs = differs || drt::xcd_rotation((i + r) % 8, i, n) != r;
      wrong += !differs;
    }
""", "placement.h")


def test_the_exchange_is_probed_on_each_stream(tmp_path):
    # stream 16 is round-robin, stream 32 (a CU mask, say) is not; one being captured is not
    # probed, takes the fenced form, and is probed by its next call
    _run(tmp_path, """
  drt::CounterBlocks blocks;
  int probes = 0;
  bool capturing = false;
  auto fenced = [&](std::uintptr_t s) {
    auto* b = blocks.of(s);
    return drt::CounterBlocks::fenced(*b, [&] { return capturing; },
                                      [&] { ++probes; return s == 32 ? -1 : 5; });
  };
  for (int i = 0; i < 3; ++i) wrong += fenced(16) || !fenced(32);
  wrong += probes != 2;
  capturing = true;
  wrong += !fenced(48) || probes != 2;
  wrong += fenced(16) || !fenced(32);
  capturing = false;
  wrong += fenced(48) || probes != 3;
  wrong += blocks.of(16)->index == blocks.of(32)->index || blocks.of(16) != blocks.of(16);
  for (std::uintptr_t s = 64; s < 64 + 29; ++s) wrong += !blocks.of(s);
  wrong += blocks.of(1000) != nullptr || !blocks.of(64);
""", "op_blocks.h")


def test_threads_on_one_stream_share_its_block_and_probe(tmp_path):
    _run(tmp_path, """
  drt::CounterBlocks blocks;
  std::atomic<int> probes{0}, odd{0};
  std::vector<std::thread> ts;
  for (int t = 0; t < 8; ++t)
    ts.emplace_back([&] {
      for (int i = 0; i < 200; ++i) {
        auto* b = blocks.of(16);
        if (drt::CounterBlocks::fenced(*b, [] { return false; },
                                       [&] { ++probes; std::this_thread::yield(); return 0; }) ||
            b->index != 0)
          ++odd;
      }
    });
  for (auto& t : ts) t.join();
  wrong += odd + (probes != 1);
""", "op_blocks.h", "<thread>", "<vector>")


def test_the_per_thread_handle_has_no_block(tmp_path):
    # one handle, as many streams as threads: they would count in one block at the same time
    _run(tmp_path, """
  drt::CounterBlocks blocks;
  wrong += blocks.of(2) != nullptr || !blocks.of(0) || !blocks.of(1);
""", "op_blocks.h")
