"""The gate of the resident solves (host code, compiled here by itself): which
solves run side by side on a device, in which order they are let in, and how
long none is tried after one gave up."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <thread>
#include <vector>
#include "ohm_resident_gate.h"
using namespace ohm;
#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); std::exit(1); } } while (0)
static void nap() { std::this_thread::sleep_for(std::chrono::milliseconds(50)); }
int main() {
  // places come in eights, a whole device at most
  CHECK(ResidentGate::places(1, 256) == 8 && ResidentGate::places(9, 256) == 16);
  CHECK(ResidentGate::places(300, 256) == 256 && ResidentGate::places(256, 256) == 256);
  // two devices do not wait for each other, nor do two solves that fit
  {
    ResidentPass a(0, 256, 256), b(1, 256, 256);
  }
  {
    ResidentPass a(0, 100, 256), b(0, 130, 256);  // 104 + 136 places
    std::atomic<int> in{0};
    std::thread t([&] { ResidentPass c(0, 17, 256); in = 1; });  // 24: 16 are left
    nap();
    CHECK(in == 0);
    std::thread late([&] { ResidentPass d(0, 1, 256); CHECK(in == 1); in = 2; });  // fits, but asked later
    nap();
    CHECK(in == 0);
    resident_gate(0).leave(104);
    t.join();
    late.join();
    CHECK(in == 2);
    resident_gate(0).enter(104, 256);
  }
  // many threads never exceed the device
  std::atomic<int> used{0};
  std::vector<std::thread> pool;
  for (int k = 0; k < 16; k++)
    pool.emplace_back([&, k] {
      for (int i = 0; i < 200; i++) {
        const int p = ResidentGate::places(1 + 37 * k % 250, 256);
        ResidentPass pass(0, 1 + 37 * k % 250, 256);
        CHECK(used.fetch_add(p) + p <= 256);
        used.fetch_sub(p);
      }
    });
  for (auto &t : pool) t.join();
  // a give-up closes the gate for 1, 2, 4 ... 32 s; a finished solve opens it
  ResidentGate g;
  int64_t now = 1000, want = 1000;
  for (int k = 0; k < 8; k++) {
    CHECK(g.open(now));
    g.report(true, now);
    CHECK(!g.open(now) && !g.open(now + want - 1) && g.open(now + want));
    now += want;
    want = want < 32000 ? 2 * want : want;
    if (want > 32000) want = 32000;
  }
  g.report(false, now);
  CHECK(g.open(now));
  g.report(true, now);
  CHECK(!g.open(now + 999) && g.open(now + 1000));
  std::printf("ok\n");
}
"""


def test_resident_gate(tmp_path):
    src, exe = tmp_path / "gate.cpp", tmp_path / "gate"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-pthread",
                    "-I" + os.path.join(ROOT, "ohmnivore_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
