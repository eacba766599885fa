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
#include <atomic>
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
  explicit Solver(Turns& a, int device = 0, bool grid = false) : all(a) {
    t.device = device;
    t.grid = grid;
    t.done = [this](int k) {
      CHECK(!t.submitting);  // a query may end the capture of a frame being submitted
      return complete[k];
    };
    all.join(&t);
  }
  ~Solver() { all.leave(&t); }
  std::vector<std::pair<Turn*, int>> after;  // what the last frame begun has to run after
  bool begin(Launch want, Launch expect, bool lasting = false) {
    Launch got = Launch::Ends;
    after.clear();
    return all.begin(&t, want, lasting, &got, [&](Turn* o, int k) { after.push_back({o, k}); }) && got == expect;
  }
  bool behind(std::vector<std::pair<Turn*, int>> frames) {  // a grid-wide frame may begin, behind these
    const bool ok = begin(Launch::Apart, Launch::Apart) && after == frames;
    all.end(&t, -1);
    return ok;
  }
  bool refused(Launch want) {
    Launch got;
    return !all.begin(&t, want, false, &got, [](Turn*, int) { CHECK(false); });
  }
  void submit(int k) {
    complete[k] = false;
    all.end(&t, k);
  }
  void finish(int k) {
    submit(k);
    complete[k] = true;
    all.retire(&t, k, [] { return 0; });
  }
};

// a frame alone is ordinary; others beside it are cooperative or come after it
void announced() {
  Turns all;
  Solver a(all), b(all), grid(all);
  CHECK(a.begin(Launch::Tiles, Launch::Tiles));
  CHECK(b.begin(Launch::Tiles, Launch::Apart));
  b.all.end(&b.t, -1);
  CHECK(grid.refused(Launch::Apart));  // its completion is not recorded yet
  a.submit(1);
  CHECK(grid.behind({{&a.t, 1}}));
  CHECK(a.begin(Launch::Tiles, Launch::Tiles));  // its own frame before it is in the same stream
  CHECK(grid.refused(Launch::Apart));
  a.submit(0);
  CHECK(grid.behind({{&a.t, 0}, {&a.t, 1}}));
  a.complete[1] = true;
  CHECK(grid.behind({{&a.t, 0}}));
  CHECK(grid.begin(Launch::Apart, Launch::Apart));
  CHECK(a.begin(Launch::Tiles, Launch::Apart));  // the grid-wide frame is still to come
  a.submit(1);
  a.complete[0] = true;
  CHECK(b.begin(Launch::Tiles, Launch::Apart));
  b.submit(0);
  grid.submit(0);
  CHECK(grid.behind({}));  // cooperative frames are kept apart by the runtime
  grid.complete[0] = a.complete[1] = true;
  CHECK(a.begin(Launch::Tiles, Launch::Apart));
  a.all.end(&a.t, -1);
  b.complete[0] = true;
  CHECK(a.begin(Launch::Tiles, Launch::Tiles));
  a.all.end(&a.t, -1);
}

// a solver whose frame ends by itself, with a tile frame before it in flight, may be capturing
void mixed() {
  Turns all;
  Solver a(all), b(all), grid(all);
  CHECK(a.begin(Launch::Tiles, Launch::Tiles));
  a.submit(0);
  CHECK(a.begin(Launch::Ends, Launch::Ends));
  CHECK(grid.refused(Launch::Apart));
  CHECK(b.begin(Launch::Tiles, Launch::Apart));
  b.all.end(&b.t, -1);
  a.submit(1);
  CHECK(grid.behind({{&a.t, 0}}));
  a.complete[0] = true;
  CHECK(a.begin(Launch::Ends, Launch::Ends));
  CHECK(grid.refused(Launch::Apart));  // not asked while it submits
  a.finish(0);
  CHECK(a.begin(Launch::Ends, Launch::Ends));
  CHECK(grid.behind({}));
  CHECK(b.begin(Launch::Tiles, Launch::Tiles));
  b.finish(0);
  a.finish(1);
}

// while its owner waits for a frame, the others still see it
void waited_for() {
  Turns all;
  Solver a(all), b(all), grid(all);
  CHECK(a.begin(Launch::Tiles, Launch::Tiles));
  a.submit(0);
  const int r = all.retire(&a.t, 0, [&] {
    CHECK(grid.behind({{&a.t, 0}}));
    CHECK(b.begin(Launch::Tiles, Launch::Apart));
    b.all.end(&b.t, -1);
    a.complete[0] = true;
    return 7;
  });
  CHECK(r == 7);
  CHECK(grid.behind({}));
}

// a frame that stays open while it runs never keeps a grid-wide solver waiting that joined before it
void lasting() {
  Turns all;
  Solver a(all), b(all);
  CHECK(a.begin(Launch::Tiles, Launch::Tiles, true));
  a.finish(0);
  {
    Solver far(all, 1, true), grid(all, 0, true);
    CHECK(a.begin(Launch::Tiles, Launch::Apart, true));
    CHECK(grid.behind({}));
    a.finish(1);
    CHECK(a.begin(Launch::Tiles, Launch::Tiles, false));
    a.finish(0);
  }
  Solver far(all, 1, true);
  CHECK(a.begin(Launch::Tiles, Launch::Tiles, true));
  a.finish(1);
}

// devices are apart, and a solver that left is not seen
void apart() {
  Turns all;
  Solver other(all, 1), grid(all);
  CHECK(other.begin(Launch::Tiles, Launch::Tiles));
  CHECK(grid.behind({}));
  other.submit(0);
  CHECK(grid.behind({}));
  {
    Solver a(all);
    CHECK(a.begin(Launch::Tiles, Launch::Tiles));
    CHECK(grid.refused(Launch::Apart));
  }
  CHECK(grid.behind({}));
}

// four threads, every choice checked against what is on the device: a
// completed frame's event is set, a frame ordered behind others waits for theirs
void threads() {
  Turns all;
  std::atomic<int> ordinary{0}, grids{0};
  auto run = [&](bool tiles) {
    Turn t;
    std::atomic<bool> complete[2] = {{true}, {true}};
    t.grid = !tiles;
    t.done = [&](int k) { return complete[k].load(); };
    all.join(&t);
    for (int i = 0; i < 3000; i++) {
      const int k = i & 1;
      Launch got;
      while (!all.begin(&t, tiles ? Launch::Tiles : Launch::Apart, i % 7 == 0, &got, [](Turn*, int) {}))
        std::this_thread::yield();
      complete[k] = false;
      if (got == Launch::Tiles) {
        CHECK(++ordinary == 1);
        CHECK(grids == 0);
      }
      all.end(&t, k);
      all.retire(&t, k, [&] {
        if (!tiles) {  // the device runs it once the frames before it have ended
          while (ordinary) std::this_thread::yield();
          ++grids;
          CHECK(ordinary == 0);
          --grids;
        }
        if (got == Launch::Tiles) --ordinary;
        complete[k] = true;
        return 0;
      });
    }
    all.leave(&t);
  };
  std::thread a(run, true), b(run, true), c(run, false), d(run, false);
  a.join(), b.join(), c.join(), d.join();
}

int main(int, char** argv) {
  const std::string name = argv[1];
  if (name == "announced") announced();
  else if (name == "mixed") mixed();
  else if (name == "waited_for") waited_for();
  else if (name == "lasting") lasting();
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


@pytest.mark.parametrize("name", ["announced", "mixed", "waited_for", "lasting", "apart", "threads"])
def test_turns(program, name):
    r = subprocess.run([program, name], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
