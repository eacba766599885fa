// turns.hpp -- which solvers' frames may be on a device together.
//
// Kernels whose workgroups wait for each other (the tile kernel, the grid-wide
// sweeps and the cooperative color repair) need all of them resident.
// Cooperative launches of one process are kept apart by the runtime, but one
// costs 36 to 110 us of gaps, so the tile kernel is launched the ordinary way
// where that is safe: beside kernels that end by themselves, and beside one
// tile kernel more (two of its workgroups fit a CU).  Every solver whose frames
// hold such kernels has an entry here, and a frame stays announced from the
// choice of its launch until its completion has been seen:
//   - a tile frame is ordinary while no other solver's waiting frame is
//     announced, cooperative otherwise;
//   - a frame of grid-wide kernels is ordered, on the device, after the
//     ordinary tile frames of other solvers.  It has to wait on the host only
//     while such a solver is submitting, and a frame that its solver
//     iterates to a residual, which stays open for as long as it runs, is
//     ordinary only where no other solver has grid-wide kernels at all.
//
// No HIP calls: an entry brings its own completion query.
#pragma once
#include <algorithm>
#include <functional>
#include <mutex>
#include <vector>

namespace avbd {

enum class Launch : unsigned char {
  Ends,   // every kernel of the frame ends by itself
  Apart,  // kernels that wait, launched cooperatively
  Tiles,  // the tile kernel, launched the ordinary way
};

// One solver's entry.  Up to `event` all is set before it joins; the rest belongs to Turns.
struct Turn {
  int device = 0;
  bool grid = false;                   // some of its frames hold grid-wide kernels
  std::function<bool(int slot)> done;  // has the frame submitted in this slot completed?
  void* event[2] = {};                 // what its owner records behind a frame, for the frames ordered after it
  bool submitting = false;             // a frame is being submitted (or iterated to a residual)
  Launch open = Launch::Ends;          // what that frame holds
  Launch slot[2] = {Launch::Ends, Launch::Ends};  // frames submitted and not seen to complete
};

class Turns {
 public:
  void join(Turn* t) {
    std::lock_guard<std::mutex> g(m_);
    list_.push_back(t);
  }
  void leave(Turn* t) {
    std::lock_guard<std::mutex> g(m_);
    list_.erase(std::remove(list_.begin(), list_.end(), t), list_.end());
  }
  // Announces t's next frame, which holds `want`; *got is how to launch it.  A
  // solver with an entry announces frames that end by themselves too.
  // after(o, k): the frame has to run after the one in o's slot k.  `lasting`:
  // it stays open while it runs.  False: not now, nothing announced.
  template <typename After>
  bool begin(Turn* t, Launch want, bool lasting, Launch* got, After&& after) {
    std::lock_guard<std::mutex> g(m_);
    bool others = false;
    for (Turn* o : list_) {
      if (o == t || o->device != t->device) continue;
      // its events are left alone while it submits: it may be capturing, which a query of them would end
      for (int k = 0; k < 2 && !o->submitting; k++)
        if (o->slot[k] != Launch::Ends && o->done(k)) o->slot[k] = Launch::Ends;
      if (want == Launch::Apart && o->submitting)
        for (Launch l : {o->open, o->slot[0], o->slot[1]})
          if (l == Launch::Tiles) return false;
      for (Launch l : {o->open, o->slot[0], o->slot[1]}) others |= l != Launch::Ends;
      others |= lasting && o->grid;
    }
    if (want == Launch::Apart)
      for (Turn* o : list_)
        for (int k = 0; k < 2; k++)
          if (o != t && o->device == t->device && o->slot[k] == Launch::Tiles) after(o, k);
    *got = t->open = want == Launch::Tiles && others ? Launch::Apart : want;
    t->submitting = true;
    return true;
  }
  // The frame is submitted in `slot`, its completion recorded there; slot < 0: it left nothing on the device.
  void end(Turn* t, int slot) {
    std::lock_guard<std::mutex> g(m_);
    if (slot >= 0) t->slot[slot] = t->open;
    t->open = Launch::Ends;
    t->submitting = false;
  }
  // Waits for the slot's frame (`wait`), which stays announced meanwhile.
  template <typename Wait>
  auto retire(Turn* t, int slot, Wait&& wait) -> decltype(wait()) {
    const auto r = wait();
    std::lock_guard<std::mutex> g(m_);
    t->slot[slot] = Launch::Ends;
    return r;
  }

 private:
  std::mutex m_;
  std::vector<Turn*> list_;
};

}  // namespace avbd
