"""csrc/kept.h, the runtime's answers that the launchers keep: compiled for the host and checked there."""

import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "instantmimic_amd", "csrc")

PROGRAM = r"""
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <memory>
#include <thread>
#include <tuple>
#include <vector>
#include "kept.h"

#define CHECK(x) if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; }
using Key = std::tuple<int, const void *, int, size_t>;  // device, kernel, threads, LDS
using Occupancy = im::Kept<Key, int>;

int main() {
  const void *fn = (const void *)&std::puts;
  int n = 0, asked = 0;
  auto answer = [&](int v) { return [&asked, v](int &out) { ++asked; out = v; return 0; }; };
  {  // asked once per key; the device is part of it
    Occupancy kept;
    CHECK(kept.get(Key(0, fn, 256, 1024), answer(4), &n) == 0 && n == 4);
    CHECK(kept.get(Key(0, fn, 256, 1024), answer(9), &n) == 0 && n == 4 && asked == 1);
    CHECK(kept.get(Key(1, fn, 256, 1024), answer(2), &n) == 0 && n == 2 && asked == 2);
    CHECK(kept.get(Key(0, fn, 256, 2048), answer(3), &n) == 0 && n == 3 && asked == 3);
    CHECK(kept.get(Key(0, fn, 256, 1024), answer(9), &n) == 0 && n == 4 && asked == 3);
  }
  {  // an error is returned, leaves the caller's value and is asked again
    Occupancy kept;
    n = 7;
    CHECK(kept.get(Key(0, fn, 64, 0), [](int &out) { out = 1; return 4; }, &n) == 4 && n == 7);
    CHECK(kept.get(Key(0, fn, 64, 0), answer(5), &n) == 0 && n == 5);
  }
  {  // a plan's answers go with the plan: the same kernel address in the next plan is asked for
    auto plan = std::make_unique<Occupancy>();
    CHECK(plan->get(Key(0, fn, 256, 0), answer(6), &n) == 0 && n == 6);
    plan = std::make_unique<Occupancy>();
    CHECK(plan->get(Key(0, fn, 256, 0), answer(1), &n) == 0 && n == 1);
  }
  {  // bounded, and right beyond the bound
    im::Kept<int, int> kept;
    for (int k = 0; k < 3 * (int)im::Kept<int, int>::kMost; ++k) CHECK(kept.get(k, answer(k), &n) == 0 && n == k);
  }
  {  // several threads: one answer, asked once
    im::Kept<int, int> kept;
    std::atomic<int> asks{0}, wrong{0};
    std::vector<std::thread> threads;
    for (int t = 0; t < 8; ++t)
      threads.emplace_back([&] {
        for (int k = 0; k < 2000; ++k) {
          int v = -1;
          if (kept.get(k % 50, [&](int &out) { ++asks; out = 100 + k % 50; return 0; }, &v) != 0 || v != 100 + k % 50) ++wrong;
        }
      });
    for (auto &t : threads) t.join();
    CHECK(wrong == 0 && asks == 50);
  }
  std::puts("ok");
  return 0;
}
"""


def test_kept_answers(tmp_path):
    src, exe = tmp_path / "kept.cpp", tmp_path / "kept"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    done = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert done.returncode == 0 and done.stdout.strip() == "ok", done.stdout


def test_no_launcher_keeps_a_runtime_answer_in_a_plain_static():
    """An occupancy, a variant's resources or a device's size in a plain static knows neither the device
    nor the other threads (the native host path asks with the interpreter's lock released)."""
    import re

    for name in sorted(os.listdir(CSRC)):
        if name.endswith((".hip", ".cpp", ".h")):
            text = open(os.path.join(CSRC, name)).read()
            assert not re.search(r"^\s*static (bool|int|std::map\b[^;]*) \w+(\[\w+\])? *(=|;)", text, re.M), name
