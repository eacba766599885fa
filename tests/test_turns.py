"""Which solvers' frames may be on a device together (csrc/turns.hpp), on the
host: a small program against the header walks the protocol with made-up
completion queries.  Kernels that wait for their other workgroups must not
meet an ordinary launch of the tile kernel, so a frame has to stay announced
until its completion has been seen, also while its owner waits for it."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <thread>
#include "turns.hpp"
using namespace avbd;
#define CHECK(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); exit(1); } } while (0)

struct Solver {
  Turn t;
  bool complete[2] = {false, false};
  Turns& all;
  explicit Solver(Turns& a, int device = 0) : all(a) {
    t.device = device;
    t.done = [this](int k) {
      CHECK(t.open == Launch::Ends);  // a query may end the capture of a frame being submitted
      return complete[k];
    };
    all.join(&t);
  }
  ~Solver() { all.leave(&t); }
  bool begin(Launch want, Launch expect) {
    Launch got = Launch::Ends;
    return all.begin(&t, want, &got) && got == expect;
  }
  bool refused(Launch want) {
    Launch got;
    return !all.begin(&t, want, &got);
  }
  void submit(int k) {
    complete[k] = false;
    all.end(&t, k);
  }
};

// a frame alone is ordinary; others beside it are cooperative or wait
void announced() {
  Turns all;
  Solver a(all), b(all), grid(all);
  CHECK(a.begin(Launch::Tiles, Launch::Tiles));
  CHECK(b.begin(Launch::Tiles, Launch::Apart));
  b.all.end(&b.t, -1);
  CHECK(grid.refused(Launch::Apart));
  a.submit(1);
  CHECK(grid.refused(Launch::Apart));
  CHECK(a.begin(Launch::Tiles, Launch::Tiles));  // its own frame before it is in the same stream
  CHECK(grid.refused(Launch::Apart));
  a.submit(0);
  a.complete[1] = true;
  CHECK(grid.refused(Launch::Apart));
  a.complete[0] = true;
  CHECK(grid.begin(Launch::Apart, Launch::Apart));
  CHECK(a.begin(Launch::Tiles, Launch::Apart));
  a.submit(1);
  CHECK(b.begin(Launch::Tiles, Launch::Apart));
  b.all.end(&b.t, -1);
  grid.submit(0);
  grid.complete[0] = a.complete[1] = true;
  CHECK(b.begin(Launch::Tiles, Launch::Tiles));
  b.all.end(&b.t, -1);
}

// while its owner waits for a frame, the others still see it
void waited_for() {
  Turns all;
  Solver a(all), b(all), grid(all);
  CHECK(a.begin(Launch::Tiles, Launch::Tiles));
  a.submit(0);
  const int r = all.retire(&a.t, 0, [&] {
    CHECK(grid.refused(Launch::Apart));
    CHECK(b.begin(Launch::Tiles, Launch::Apart));
    b.all.end(&b.t, -1);
    a.complete[0] = true;
    return 7;
  });
  CHECK(r == 7);
  CHECK(grid.begin(Launch::Apart, Launch::Apart));
}

// devices are apart, and a solver that left is not seen
void apart() {
  Turns all;
  Solver other(all, 1), grid(all);
  CHECK(other.begin(Launch::Tiles, Launch::Tiles));
  CHECK(grid.begin(Launch::Apart, Launch::Apart));
  all.end(&grid.t, -1);
  {
    Solver a(all);
    CHECK(a.begin(Launch::Tiles, Launch::Tiles));
    CHECK(grid.refused(Launch::Apart));
  }
  CHECK(grid.begin(Launch::Apart, Launch::Apart));
}

// four threads, every choice checked against what is on the device
void threads() {
  Turns all;
  std::mutex m;
  int ordinary = 0, cooperative = 0, grids = 0;
  auto run = [&](bool tiles) {
    Solver s(all);
    for (int i = 0; i < 4000; i++) {
      Launch got;
      if (!all.begin(&s.t, tiles ? Launch::Tiles : Launch::Apart, &got)) {
        std::this_thread::yield();
        i--;
        continue;
      }
      {
        std::lock_guard<std::mutex> g(m);
        (got == Launch::Tiles ? ordinary : tiles ? cooperative : grids)++;
        CHECK(ordinary <= 1);
        CHECK(!(ordinary && grids));
      }
      all.end(&s.t, i & 1);
      all.retire(&s.t, i & 1, [&] {
        std::lock_guard<std::mutex> g(m);
        (got == Launch::Tiles ? ordinary : tiles ? cooperative : grids)--;
        return 0;
      });
    }
  };
  std::thread a(run, true), b(run, true), c(run, false), d(run, false);
  a.join(), b.join(), c.join(), d.join();
}

int main(int, char** argv) {
  const std::string name = argv[1];
  if (name == "announced") announced();
  else if (name == "waited_for") waited_for();
  else if (name == "apart") apart();
  else if (name == "threads") threads();
  else return 2;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("turns")
    (d / "main.cpp").write_text("#include <string>\n" + PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", os.path.join(ROOT, "avbd-metal_amd", "csrc"),
                    str(d / "main.cpp"), "-o", str(d / "turns")], check=True, timeout=120)
    return str(d / "turns")


@pytest.mark.parametrize("name", ["announced", "waited_for", "apart", "threads"])
def test_turns(program, name):
    r = subprocess.run([program, name], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
