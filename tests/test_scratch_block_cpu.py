"""Blocks that grow: only a want of memory may be worked round; an error that an earlier launch left is the caller's to report."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include "scratch_block.h"

#include <cstdio>
#include <cstdlib>
#include <string>

using ughip::Grown;
#define CHECK(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); exit(1); } } while (0)

struct Fake {
  bool sync_ok = true, free_ok = true;
  Grown memory = Grown::YES;
  std::string calls;
  char place[2];
  bool synchronize() { return calls += "s", sync_ok; }
  bool free(void* p) {
    CHECK(p != nullptr);
    return calls += "f", free_ok;
  }
  Grown allocate(void** p, size_t bytes) { return calls += "a" + std::to_string(bytes), *p = place + 1, memory; }
};

int main() {
  for (bool had : {false, true}) {
    auto start = [&](Fake& f, void** block, size_t* have) { *block = had ? f.place : nullptr, *have = had ? 10 : 0; };
    const std::string before = had ? "sf" : "s";
    void* block;
    size_t have;
    Fake f;
    start(f, &block, &have);
    CHECK(ughip::grow_block(f, &block, &have, have, 5) == Grown::YES && f.calls.empty() && (block != nullptr) == had);
    CHECK(ughip::grow_block(f, &block, &have, 11, 5) == Grown::YES && f.calls == before + "a11" && have == 11 && block == f.place + 1);
    Fake g;
    start(g, &block, &have);
    CHECK(ughip::grow_block(g, &block, &have, 11, 64) == Grown::YES && g.calls == before + "a64" && have == 64);
    Fake late;  // something launched before has failed: nothing is freed or allocated, and it is not a want of memory
    late.sync_ok = false;
    late.memory = Grown::NO_MEMORY;
    start(late, &block, &have);
    CHECK(ughip::grow_block(late, &block, &have, 11, 5) == Grown::FAILED && late.calls == "s" && (block != nullptr) == had && have == (had ? 10u : 0u));
    for (Grown why : {Grown::NO_MEMORY, Grown::FAILED}) {
      Fake none;
      none.memory = why;
      start(none, &block, &have);
      CHECK(ughip::grow_block(none, &block, &have, 11, 5) == why && none.calls == before + "a11" && block == nullptr && have == 0);
    }
    if (had) {
      Fake kept;
      kept.free_ok = false;
      start(kept, &block, &have);
      CHECK(ughip::grow_block(kept, &block, &have, 11, 5) == Grown::FAILED && kept.calls == "sf" && block == kept.place && have == 10);
    }
  }
  puts("ok");
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host compiler")
def test_what_growing_a_block_can_come_to(tmp_path):
    (tmp_path / "main.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I" + os.path.join(ROOT, "ug_amd", "csrc", "ughip"), str(tmp_path / "main.cpp"), "-o", str(tmp_path / "grow")], check=True)
    out = subprocess.run([str(tmp_path / "grow")], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout == "ok\n", out.stdout + out.stderr
