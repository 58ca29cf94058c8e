"""The queue between the thread that builds a reply's steps and the one that launches them: what a launch throws, and who ends which step."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include "step_queue.h"

#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <memory>
#include <stdexcept>
#include <vector>

using namespace std::chrono_literals;
static std::atomic<int> ended{0};
static std::thread::id owner;
#define CHECK(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); exit(1); } } while (0)

struct Step {
  int n = -1;
  Step() = default;
  explicit Step(int i) : n(i) {}
  Step(Step&& o) : n(o.n) { o.n = -1; }
  Step& operator=(Step&& o) { std::swap(n, o.n); return *this; }
  ~Step() {
    if (n < 0) return;
    CHECK(std::this_thread::get_id() == owner);
    ++ended;
  }
};
typedef ug_llama::StepQueue<Step> Queue;

// Steps 0 .. steps - 1, the launch of `bad` throws, the caller gives up before pushing `quit`.  Returns how many were pushed.
static int drive(int steps, int bad, int quit, std::chrono::milliseconds launch, std::chrono::milliseconds build, std::vector<int>* ran, bool* threw) {
  int pushed = 0;
  *threw = false;
  ended = 0;
  try {
    Queue q([&](Step& s) {
      std::this_thread::sleep_for(launch);
      ran->push_back(s.n);
      if (s.n == bad) throw std::runtime_error("launch");
    });
    for (int i = 0; i < steps; ++i) {
      if (i == quit) throw std::logic_error("build");
      std::this_thread::sleep_for(build);
      Step s(i);
      ++pushed;
      q.push(std::move(s));
    }
    q.finish();
  } catch (const std::runtime_error&) {
    *threw = true;
  } catch (const std::logic_error&) {
  }
  return pushed;
}

int main() {
  owner = std::this_thread::get_id();
  for (auto launch : {0ms, 2ms})
    for (auto build : {0ms, 2ms}) {
      std::vector<int> ran;
      bool threw;
      CHECK(drive(20, -1, -1, launch, build, &ran, &threw) == 20 && !threw && ran.size() == 20 && ended == 20);
      for (int i = 0; i < 20; ++i) CHECK(ran[i] == i);
      for (int bad : {0, 1, 7, 18, 19}) {  // the last ones come out of finish
        ran.clear();
        const int pushed = drive(20, bad, -1, launch, build, &ran, &threw);
        CHECK(threw && ran.size() == (size_t)bad + 1 && ended == pushed && pushed <= bad + 2 + (int)Queue::kAhead);
      }
      for (int quit : {0, 1, 5}) {
        ran.clear();
        CHECK(drive(20, -1, quit, launch, build, &ran, &threw) == quit && !threw && ran.size() <= (size_t)quit && ended == quit);
        for (size_t i = 0; i < ran.size(); ++i) CHECK(ran[i] == (int)i);
      }
      ran.clear();
      CHECK(drive(0, -1, -1, launch, build, &ran, &threw) == 0 && !threw && ended == 0);
    }
  puts("ok");
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host compiler")
def test_exceptions_on_either_side(tmp_path):
    (tmp_path / "main.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I" + os.path.join(ROOT, "ug_amd", "csrc", "host"), str(tmp_path / "main.cpp"), "-o", str(tmp_path / "queue")], check=True)
    out = subprocess.run([str(tmp_path / "queue")], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout == "ok\n", out.stdout + out.stderr
