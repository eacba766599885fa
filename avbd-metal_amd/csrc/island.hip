// island.hip -- contact-aware coloring and the whole solve of rigid scenes
// whose bodies fall into independent islands, one workgroup per island.
//
// An island is a set of dynamic bodies that no joint, spring or possible
// contact links to a body outside it (found at create from the constraint
// graph and the collision groups).  Gauss-Seidel order only has to hold
// inside one, so a workgroup runs all iterations, colors and duals of its
// island with workgroup barriers; the grid-wide sweep needs one dependent
// launch (or grid barrier) per color and iteration.
#include "sweep.hpp"

namespace avbd {

// global writes of this workgroup visible to its own later reads
__device__ __forceinline__ void block_sync() {
  __threadfence_block();
  __syncthreads();
}

// ---------------------------------------------------------------------------
// coloring: the 20 Jacobi passes of the parallel rule (40_solver.metal:
// 320-386) on colors held in LDS.  A pass that changes no body of the island
// leaves it at the rule's fixed point, so stopping there equals running on.
// Neighbour lists are packed in LDS once when they fit, else every pass
// walks the adjacency.  Two launches in place of 26 (passes, repair,
// validation, bucket lists); 4096 scenes: 26 us, and 36 us where the
// repair runs (the grid-wide repair alone took 268 us).
// ---------------------------------------------------------------------------
constexpr uint32_t kIslandNbrLds = 4096;
constexpr uint32_t kNoNbr = 0xFFFFu;

struct IslandColors {
  uint8_t c[2][kIslandMax];
  uint16_t off[kIslandMax], deg[kIslandMax];
  uint16_t nbr[kIslandNbrLds];
  uint32_t total;
};

// the masks of neighbor_masks (sweep.hpp) over local indices: bodies of an
// island are ascending, so local order is body order
template <typename F>
__device__ __forceinline__ void island_neighbors(const DeviceState& S, const IslandColors& I, uint32_t i, uint32_t v,
                                                 bool packed, F&& f) {
  if (packed) {
    for (uint32_t k = 0; k < I.deg[i]; k++) {
      const uint32_t j = I.nbr[I.off[i] + k];
      if (j != kNoNbr) f(j);
    }
    return;
  }
  auto visit = [&](uint32_t b) {
    if (body_dynamic(S, b)) f(S.islandLocal[b]);
  };
  const uint32_t ss = S.sAdjStart[v], sc = S.sAdjCount[v], ds = S.dAdjStart[v], dc = S.dAdjCount[v];
  for (uint32_t k = 0; k < sc; k++) for_each_neighbor(S, S.sAdjList[ss + k], v, false, visit);
  for (uint32_t k = 0; k < dc; k++) for_each_neighbor(S, S.dAdjList[ds + k], v, false, visit);
}
__device__ __forceinline__ ColorMasks island_masks(const DeviceState& S, const IslandColors& I, const uint8_t* colors,
                                                   uint32_t i, uint32_t v, bool packed) {
  ColorMasks m{0ull, 0ull, false};
  const uint32_t my = colors[i];
  island_neighbors(S, I, i, v, packed, [&](uint32_t j) {
    const uint32_t c = colors[j];
    const uint64_t bit = c < 64 ? (1ull << c) : 0ull;
    m.all |= bit;
    if (j < i) {
      m.lower |= bit;
      if (c == my) m.conflict = true;
    }
  });
  return m;
}
// packs the neighbour lists; every adjacency entry of a rigid scene has one
// other participant.  Returns whether they fit.
__device__ __forceinline__ bool island_pack(const DeviceState& S, IslandColors& I, const uint32_t* body, uint32_t n) {
  if (threadIdx.x == 0) I.total = 0;
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) {
    const uint32_t v = body[i], d = S.sAdjCount[v] + S.dAdjCount[v];
    const uint32_t o = atomicAdd(&I.total, d);
    I.off[i] = (uint16_t)(o < kIslandNbrLds ? o : 0u);
    I.deg[i] = (uint16_t)(d < kNoNbr ? d : kNoNbr);
  }
  __syncthreads();
  if (I.total > kIslandNbrLds) return false;
  for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) {
    const uint32_t v = body[i];
    uint32_t o = I.off[i];
    auto put = [&](uint32_t b) { I.nbr[o++] = (uint16_t)(body_dynamic(S, b) ? S.islandLocal[b] : kNoNbr); };
    const uint32_t ss = S.sAdjStart[v], sc = S.sAdjCount[v], ds = S.dAdjStart[v], dc = S.dAdjCount[v];
    for (uint32_t k = 0; k < sc; k++) for_each_neighbor(S, S.sAdjList[ss + k], v, false, put);
    for (uint32_t k = 0; k < dc; k++) for_each_neighbor(S, S.dAdjList[ds + k], v, false, put);
  }
  __syncthreads();
  return true;
}

__global__ void __launch_bounds__(kIslandThreads) k_island_color(DeviceState S) {
  __shared__ IslandColors I;
  const uint32_t s0 = S.islandStart[blockIdx.x], n = S.islandStart[blockIdx.x + 1] - s0;
  const uint32_t* body = S.islandBody + s0;
  for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) I.c[0][i] = (uint8_t)S.colors[body[i]];
  const bool packed = island_pack(S, I, body, n);
  __syncthreads();
  uint32_t cur = 0;
  bool open = true;
  for (uint32_t pass = 0; pass < kColorPasses && open; pass++) {
    bool changed = false;
    for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) {
      const uint32_t my = I.c[cur][i];
      const ColorMasks m = island_masks(S, I, I.c[cur], i, body[i], packed);
      uint32_t out;
      if (m.conflict) {
        const uint64_t f = ~m.lower;
        out = f ? (uint32_t)__builtin_ctzll(f) : 63u;
        changed = true;
      } else {
        const uint64_t f = ~m.all;
        const uint32_t best = f ? (uint32_t)__builtin_ctzll(f) : my;
        out = best < my ? best : my;
        changed |= best < my;
      }
      I.c[cur ^ 1u][i] = (uint8_t)out;
    }
    open = __syncthreads_or(changed) != 0;
    cur ^= 1u;
  }
  if (open && threadIdx.x == 0) S.colorFlags[kColorPasses - 1] = 1u;  // some island is unfinished: all are repaired
  for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) S.colors[body[i]] = I.c[cur][i];
}

// When some island's passes did not settle, every island takes the serial
// greedy coloring (the lowest color unused by its lower-index neighbours,
// 40_solver.metal:387-436) and is validated.  A body is final once its
// lower-index neighbours are, so applying the rule until nothing changes
// reaches that coloring in any order, in at most n + 1 passes.
__global__ void __launch_bounds__(kIslandThreads) k_island_repair(DeviceState S) {
  if (S.colorFlags[kColorPasses - 1] == 0u) return;
  __shared__ IslandColors I;
  const uint32_t s0 = S.islandStart[blockIdx.x], n = S.islandStart[blockIdx.x + 1] - s0;
  const uint32_t* body = S.islandBody + s0;
  for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) I.c[0][i] = (uint8_t)S.colors[body[i]];
  const bool packed = island_pack(S, I, body, n);
  __syncthreads();
  uint32_t cur = 0;
  bool open = true;
  for (uint32_t pass = 0; pass <= n && open; pass++) {
    bool changed = false;
    for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) {
      const uint64_t f = ~island_masks(S, I, I.c[cur], i, body[i], packed).lower;
      const uint32_t out = f ? (uint32_t)__builtin_ctzll(f) : 63u;
      changed |= out != I.c[cur][i];
      I.c[cur ^ 1u][i] = (uint8_t)out;
    }
    open = __syncthreads_or(changed) != 0;
    cur ^= 1u;
  }
  for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) {
    if (island_masks(S, I, I.c[cur], i, body[i], packed).conflict) atomicAdd(&S.counters[CTR_COLOR_CONFLICTS], 1u);
    S.colors[body[i]] = I.c[cur][i];
  }
}

// S.colorFlags must be zero on entry (cleared with the frame's counters)
void launch_island_coloring(hipStream_t st, const DeviceState& S, uint32_t numIslands, uint32_t threads) {
  hipLaunchKernelGGL(k_island_color, dim3(numIslands), dim3(threads), 0, st, S);
  hipLaunchKernelGGL(k_island_repair, dim3(numIslands), dim3(threads), 0, st, S);
}

// ---------------------------------------------------------------------------
// solve: P.iterations sweeps of a workgroup's islands.
//
// Bound by instruction issue along a wave: one color of the sweep is about
// 2300 instructions (two manifold stamps, the reduction, the 6x6 LDL^T),
// 5 to 6 us however few bodies it has, and one dual 2 to 3 us.  Four lanes a
// body measured best (4096 scenes: 1, 2, 8 lanes 2.00, 1.80, 2.02 ms a frame
// against 1.81), 64 bodies a workgroup as good as 32 or 128; splitting the
// listed contacts over the threads took the dual of 128 bodies from 20 us
// (eight lanes per body, its manifolds in turn) to the time of a color.
// 4096 batched scenes: this kernel 0.65 ms, the frame 3.35 -> 1.84 ms with the
// coloring above; 64 scenes 0.30, the frame 1.18 -> 0.64 ms; a 10-cube stack
// 0.144 (20 colors and 10 duals, 4.8 us each), the frame 0.48 -> 0.29 ms.
// ---------------------------------------------------------------------------
// f(manifold, contacts) for every active manifold of the workgroup's bodies,
// split over its threads; one of two dynamic bodies belongs to its first
template <typename F>
__device__ __forceinline__ void island_manifolds(const DeviceState& S, const uint32_t* body, uint32_t n, F&& f) {
  for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) {
    const uint32_t v = body[i], ds = S.dAdjStart[v], dc = S.dAdjCount[v];
    for (uint32_t k = 0; k < dc; k++) {
      const uint32_t m = S.dAdjList[ds + k] & kAdjIndexMask;
      const U4 h = S.manifolds[m].header;
      if (h.x == v || !body_dynamic(S, h.x)) f(m, h.z);
    }
  }
}

template <int L>
__global__ void __launch_bounds__(kIslandThreads) k_island_solve(DeviceState S, StepParams P) {
  if (P.convCheck && S.counters[CTR_CONV_DONE] != 0u) return;
  __shared__ uint32_t order[kIslandMax];  // bodies by color
  __shared__ uint32_t contact[kIslandContacts], contacts;  // manifold << 3 | slot of every contact of the workgroup
  __shared__ uint32_t start[kMaxColors + 1], cursor[kMaxColors];
  const uint32_t tid = threadIdx.x, nt = blockDim.x;
  const uint32_t s0 = S.islandStart[blockIdx.x], n = S.islandStart[blockIdx.x + 1] - s0;
  const uint32_t* body = S.islandBody + s0;
  if (tid < kMaxColors) cursor[tid] = 0;
  if (tid == 0) contacts = 0;
  __syncthreads();
  for (uint32_t i = tid; i < n; i += nt) atomicAdd(&cursor[S.colors[body[i]] & 63u], 1u);
  __syncthreads();
  if (tid < 64) {
    const uint32_t c = cursor[tid];
    uint32_t x = c;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t y = __shfl_up(x, d, 64);
      if (tid >= (uint32_t)d) x += y;
    }
    start[tid + 1] = x;
    if (tid == 0) start[0] = 0;
    cursor[tid] = x - c;
  }
  __syncthreads();
  // a color's bodies are independent, so their order inside it is free
  for (uint32_t i = tid; i < n; i += nt) {
    const uint32_t v = body[i];
    order[atomicAdd(&cursor[S.colors[v] & 63u], 1u)] = v;
  }
  __syncthreads();
  island_manifolds(S, order, n, [&](uint32_t m, uint32_t count) {
    const uint32_t at = atomicAdd(&contacts, count);
    for (uint32_t k = 0; k < count; k++)
      if (at + k < kIslandContacts) contact[at + k] = m * kMaxContacts + k;
  });
  __syncthreads();
  const bool listed = contacts <= kIslandContacts;
  const uint32_t lane = tid & (L - 1), group = tid / L, groups = nt / L, waveFirst = (tid & ~63u) / L;
  const uint32_t j0 = S.islandJointStart[blockIdx.x], j1 = S.islandJointStart[blockIdx.x + 1];
  const uint32_t p0 = S.islandSpringStart[blockIdx.x], p1 = S.islandSpringStart[blockIdx.x + 1];
  for (uint32_t it = 0; it < P.iterations; it++) {
    for (uint32_t c = 0; c < kMaxColors; c++) {
      const uint32_t e = start[c + 1];
      if (start[c] == e) continue;
      for (uint32_t b0 = start[c]; b0 + waveFirst < e; b0 += groups) {
        const bool active = b0 + group < e;
        primal_group<L, kModeGeneral>(S, P, active, body_work(S, active, active ? order[b0 + group] : 0u), lane, c);
      }
      block_sync();
      if (e == n) break;
    }
    for (uint32_t q = j0 + tid; q < j1; q += nt) dual_joint(S, P, S.islandJoint[q]);
    for (uint32_t q = p0 + tid; q < p1; q += nt) dual_spring(S, P, S.islandSpring[q]);
    if (listed)
      for (uint32_t q = tid; q < contacts; q += nt) dual_contact(S, P, contact[q] / kMaxContacts, contact[q] % kMaxContacts);
    else
      island_manifolds(S, order, n, [&](uint32_t m, uint32_t count) {
        for (uint32_t k = 0; k < count; k++) dual_contact(S, P, m, k);
      });
    block_sync();
  }
}

void launch_island_solve(hipStream_t st, const DeviceState& S, const StepParams& P, uint32_t numIslands, int lanes,
                         uint32_t threads) {
  switch (lanes) {
    case 4: hipLaunchKernelGGL(k_island_solve<4>, dim3(numIslands), dim3(threads), 0, st, S, P); break;
    case 8: hipLaunchKernelGGL(k_island_solve<8>, dim3(numIslands), dim3(threads), 0, st, S, P); break;
    case 16: hipLaunchKernelGGL(k_island_solve<16>, dim3(numIslands), dim3(threads), 0, st, S, P); break;
    default: hipLaunchKernelGGL(k_island_solve<32>, dim3(numIslands), dim3(threads), 0, st, S, P); break;
  }
}

}  // namespace avbd
