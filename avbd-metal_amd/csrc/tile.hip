// tile.hip -- the whole solve of a tetrahedral scene in one launch: every
// workgroup keeps a tile of bodies, and tiles exchange positions through
// versioned records instead of meeting at a grid barrier.
//
// Gauss-Seidel by color only orders a body against its neighbours: it must
// read the neighbours of lower colors after, and those of higher colors
// before, their update of the same sweep.  A tile therefore waits, before
// each color, for its halo bodies of the color before it and for nothing
// else.  Each float of a position travels in one 64-bit word beside the
// version (sweep count) that wrote it, so a reader polls the data itself: no
// fence, no flag, no write-back of caches.  Overwriting is safe without a
// second buffer: before a body's next update its tile has waited for every
// adjacent tile's bodies that read the old one.
//
// Bound by the chain of a color: poll a halo word (about 1 us from the store
// in the other tile), gather from LDS, stamp, reduce and solve (1 to 1.4 us
// at one wave per SIMD).  One launch per color spent 5.2 us on the same color:
// the launch, five dependent loads that miss the cold L2, and the solve.
// 9261 vertices: 1.29 -> 0.70 ms a frame, two frames iterated to residual 1e-4
// 33.0 -> 17.5 ms; 125 vertices 1.03 -> 0.52 ms a frame.  This kernel takes 0.469
// and 0.401 ms of them, 2.6 and 2.2 us a color or dual.  Contacts kept in
// LDS took the tiles on the ground, which the others wait for, from 2.25 to
// 1.5 us a color and their dual from 2.3 to 0.5 us; fetching the next color's
// records a color ahead changed nothing.
#include "sweep.hpp"

namespace avbd {

// Partner of a manifold between a particle and a static body (the only kind
// in frames this kernel runs): the particle's pose comes from the tile.
struct TilePose {
  const F4* lin;
  const F4* ang;
  uint32_t self;
  F4 pos;
  __device__ __forceinline__ F4 L(uint32_t b, uint32_t, bool) const { return b == self ? pos : lin[b]; }
  __device__ __forceinline__ F4 A(uint32_t b, uint32_t, bool) const { return ang[b]; }
};

// The single contact point of a particle with a static body, in LDS: what
// contact_force reads, with the terms that stay fixed over a frame (rotations,
// the static side) folded to one vector each, added in the same places.
struct GroundContact {
  V3 n, t1, C0, lam, pen, kA, kB, init;
  float dynF, statF, sign, stick;  // sign: the particle is side A (+1) or B (-1)
  uint32_t manifold;
};
constexpr uint32_t kTouchAny = 1u, kTouchFast = 2u;

__device__ __forceinline__ void ground_load(const DeviceState& S, uint32_t mi, uint32_t self, GroundContact& g) {
  const ManifoldRec& m = S.manifolds[mi];
  const ContactRec& c = m.c[0];
  const uint32_t a = m.header.x, b = m.header.y;
  const F4 qA = S.posAng[a], qB = S.posAng[b];
  const V3 rA = (m.header.w & 2u) ? xyz(c.rA) : q_rotate(qA, xyz(c.rA));
  const V3 rB = (m.header.w & 4u) ? xyz(c.rB) : q_rotate(qB, xyz(c.rB));
  const V3 dA = q_sub(qA, S.initAng[a]), dB = q_sub(qB, S.initAng[b]);
  g.n = xyz(m.basisN);
  g.t1 = xyz(m.basisT1);
  const V3 t2 = cross(g.n, g.t1);
  g.dynF = m.basisN.w;
  g.statF = m.basisT1.w;
  g.C0 = xyz(c.C0);
  g.lam = xyz(c.lambda);
  g.pen = xyz(c.penalty);
  g.stick = c.rB.w;
  g.kA = v3(dot(cross(rA, g.n), dA), dot(cross(rA, g.t1), dA), dot(cross(rA, t2), dA));
  g.kB = v3(dot(cross(rB, g.n), dB), dot(cross(rB, g.t1), dB), dot(cross(rB, t2), dB));
  g.init = xyz(S.initLin[self]);
  g.sign = self == a ? 1.0f : -1.0f;
  g.manifold = mi;
}
__device__ __forceinline__ void ground_store(const DeviceState& S, const GroundContact& g) {
  ContactRec& c = S.manifolds[g.manifold].c[0];
  c.lambda = f4(g.lam, 0.0f);
  c.penalty = f4(g.pen, 0.0f);
  c.rB.w = g.stick;
}
// contact_force (stamps.hpp) for the particle's displacement dq
__device__ __forceinline__ V3 ground_force(const GroundContact& g, V3 dq, float alpha, V3 t2, V3& C, float& fs,
                                           float& bounds) {
  C = g.C0 * (1.0f - alpha);
  C += v3(dot(g.n, dq), dot(g.t1, dq), dot(t2, dq)) * g.sign;
  C += g.kA;
  C -= g.kB;
  V3 F = g.pen * C + g.lam;
  F.x = fminf(F.x, 0.0f);
  bounds = fabsf(F.x) * g.statF;
  fs = sqrtf(F.y * F.y + F.z * F.z);
  if (fs > bounds && fs > 0.0f) {
    const float dyn = fabsf(F.x) * g.dynF;
    F.y *= dyn / fs;
    F.z *= dyn / fs;
  }
  return F;
}
__device__ __forceinline__ void stamp_ground(const GroundContact& g, V3 xs, V3 ls, float alpha, Acc& acc) {
  const V3 t2 = cross(g.n, g.t1);
  V3 C;
  float fs, bounds;
  const V3 F = ground_force(g, (xs - g.init) + ls, alpha, t2, C, fs, bounds);
  const V3 j0 = g.n * g.sign, j1 = g.t1 * g.sign, j2 = t2 * g.sign;
  acc_lin_outer(acc, j0, g.pen.x);
  acc_lin_outer(acc, j1, g.pen.y);
  acc_lin_outer(acc, j2, g.pen.z);
  acc.gl += j0 * F.x + j1 * F.y + j2 * F.z;
}
// dual_contact (sweep.hpp) at the particle's position (w its mass)
__device__ __forceinline__ void dual_ground(const StepParams& P, GroundContact& g, F4 pos) {
  V3 C;
  float fs, bounds;
  V3 F = ground_force(g, xyz(pos) - g.init, P.alpha, cross(g.n, g.t1), C, fs, bounds);
  F.x = fmaxf(F.x, -fminf(P.lambdaMax, fmaxf(10.0f, 1.0e5f * pos.w)));
  g.lam = F;
  if (F.x < 0.0f) g.pen.x = fminf(g.pen.x + P.betaLin * fabsf(C.x), kPenaltyMax);
  if (fs <= bounds) {
    g.pen.y = fminf(g.pen.y + P.betaLin * fabsf(C.y), kPenaltyMaxT);
    g.pen.z = fminf(g.pen.z + P.betaLin * fabsf(C.z), kPenaltyMaxT);
    g.stick = sqrtf(C.y * C.y + C.z * C.z) < kStickThresh ? 1.0f : 0.0f;
  }
}

// LDS writes visible to the workgroup; global stores stay in flight
__device__ __forceinline__ void lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

constexpr int kTileLanes = 32;
constexpr uint32_t kTileSpins = 1u << 20;

__global__ void __launch_bounds__(kTileThreads) k_tile_solve(DeviceState S, StepParams P, uint32_t colors) {
  if (P.convCheck && S.counters[CTR_CONV_DONE] != 0u) return;
  if (S.counters[CTR_DYN_CONTACT] != 0u) {
    // contacts between dynamic bodies couple bodies the halos do not hold:
    // this frame sweeps grid-wide (rare: the host then leaves this path)
    grid_sweeps<kTileLanes, kModeTet>(S, P, colors, 0u);
    __syncthreads();
    if (threadIdx.x == 0 && atomicAdd(&S.tileEpoch[1], 1u) == gridDim.x - 1u) {
      S.tileEpoch[1] = 0u;
      S.counters[CTR_GBAR] = 0u;
    }
    return;
  }
  __shared__ F4 hi[kTileLocal], lo[kTileLocal];   // positions of own and halo bodies, high (w mass) and low parts
  __shared__ GroundContact ground[kTileOwn];
  __shared__ uint8_t touch[kTileOwn];
  const uint32_t tid = threadIdx.x, nt = blockDim.x;
  const uint32_t lane = tid & (kTileLanes - 1), group = tid / kTileLanes, groups = nt / kTileLanes;
  const uint32_t tiles = gridDim.x, tile = S.tileOrder[blockIdx.x];
  const uint32_t* own = S.tileOwn + tile * (colors + 1);    // per color: range of tileWork
  const uint32_t* halo = S.tileHalo + tile * (colors + 2);  // per color, then static: range of tileHaloBody
  const uint32_t base = S.tileEpoch[0];
  for (uint32_t i = own[0] + tid; i < own[colors]; i += nt) {
    const U4 w = S.tileWork[i];
    hi[w.w] = S.posLin[w.x];
    lo[w.w] = S.posLo[w.x];
  }
  for (uint32_t i = halo[0] + tid; i < halo[colors + 1]; i += nt) {
    const U2 h = S.tileHaloBody[i];
    hi[h.y] = S.posLin[h.x];
    lo[h.y] = S.posLo[h.x];
  }
  // contacts of the own bodies: the usual one, a single point against a static
  // body, is kept in LDS for the whole launch
  bool any = false, fast = false;
  for (uint32_t i = own[0] + tid; i < own[colors]; i += nt) {
    const U4 w = S.tileWork[i];
    const uint32_t dc = S.dAdjCount[w.x];
    uint32_t kind = dc ? kTouchAny : 0u;
    if (dc == 1u) {
      const uint32_t m = S.dAdjList[S.dAdjStart[w.x]] & kAdjIndexMask;
      if (S.manifolds[m].header.z == 1u) {
        kind = kTouchFast;
        ground_load(S, m, w.x, ground[w.w]);
      }
    }
    touch[w.w] = (uint8_t)kind;
    any |= kind == kTouchAny;
    fast |= kind == kTouchFast;
  }
  const bool anyContact = __syncthreads_or(any) != 0, fastContact = __syncthreads_or(fast) != 0;
  uint32_t* fail = &S.counters[CTR_GBAR_FAIL];
  for (uint32_t it = 0; it < P.iterations; it++) {
    for (uint32_t c = 0; c < colors; c++) {
      const uint32_t w0 = own[c], w1 = own[c + 1];
      // the color's records do not depend on other tiles: load them before waiting
      U4 work = U4{0u, 0u, 0u, 0u};
      TetSlot slot;
      TileSlotIdx idx;
      F4 inert = F4{0, 0, 0, 0};
      float rad = 0.0f;
      auto fetch = [&](uint32_t i) {
        work = S.tileWork[i];
        if (lane < work.z) {
          slot = S.tetSlots[work.y + lane];
          idx = S.tileIdx[work.y + lane];
        }
        inert = S.inertLin[work.x];
        rad = fabsf(S.shape[work.x].w);
      };
      if (w0 + group < w1) fetch(w0 + group);
      if (it + c > 0) {
        const uint32_t pc = c ? c - 1 : colors - 1, tag = base + it + (c ? 1u : 0u);
        const uint32_t h0 = halo[pc], words = (halo[pc + 1] - h0) * 6u;
        for (uint32_t q = tid; q < words; q += nt) {
          const U2 h = S.tileHaloBody[h0 + q / 6u];
          const uint32_t k = q % 6u;
          const uint64_t* word = S.tileX + 6ull * h.x + k;
          uint64_t v = __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          // bounded: a tile that gives up records the failure, and then none waits
          for (uint32_t spins = 0; (uint32_t)(v >> 32) != tag; spins++) {
            if (spins >= kTileSpins || ((spins & 255u) == 255u && __hip_atomic_load(fail, __ATOMIC_RELAXED,
                                                                                   __HIP_MEMORY_SCOPE_AGENT) != 0u)) {
              if (spins >= kTileSpins) atomicAdd(fail, 1u);
              break;
            }
            v = __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          }
          float* to = k < 3u ? &hi[h.y].x + k : &lo[h.y].x + (k - 3u);
          *to = __uint_as_float((uint32_t)v);
        }
      }
      lds_sync();
      for (uint32_t i = w0 + group; i < w1; i += groups) {
        if (i != w0 + group) fetch(i);
        const F4 pl = hi[work.w], pLo = lo[work.w];
        const V3 xs = xyz(pl), ls = xyz(pLo);
        Acc acc;
        acc_zero(acc);
        for (uint32_t k = lane; k < work.z; k += kTileLanes) {
          if (k != lane) {
            slot = S.tetSlots[work.y + k];
            idx = S.tileIdx[work.y + k];
          }
          V3 x[3], l[3];
#pragma unroll
          for (int o = 0; o < 3; o++) {
            x[o] = xyz(hi[idx.o[o]]);
            l[o] = xyz(lo[idx.o[o]]);
          }
          stamp_tet_slot_e(slot, split_edge(x[0], l[0], xs, ls), split_edge(x[1], l[1], xs, ls),
                           split_edge(x[2], l[2], xs, ls), acc);
        }
        // contacts follow the tets on the lanes, as in the per-color kernel
        const uint32_t kind = touch[work.w], first = (kTileLanes - (work.z % kTileLanes)) % kTileLanes;
        if (kind == kTouchFast && lane == first) {
          stamp_ground(ground[work.w], xs, ls, P.alpha, acc);
        } else if (kind == kTouchAny) {
          const uint32_t ds = S.dAdjStart[work.x], dc = S.dAdjCount[work.x];
          const TilePose pose{S.posLin, S.posAng, work.x, pl};
          for (uint32_t k = (lane + first) % kTileLanes; k < dc; k += kTileLanes)
            stamp_manifold(S.manifolds[S.dAdjList[ds + k] & kAdjIndexMask], work.x, false, pose, S.initLin, S.initAng,
                           P.alpha, acc, ls);
        }
        acc.l00 = group_sum<kTileLanes>(acc.l00);
        acc.l10 = group_sum<kTileLanes>(acc.l10);
        acc.l11 = group_sum<kTileLanes>(acc.l11);
        acc.l20 = group_sum<kTileLanes>(acc.l20);
        acc.l21 = group_sum<kTileLanes>(acc.l21);
        acc.l22 = group_sum<kTileLanes>(acc.l22);
        acc.gl = group_sum3<kTileLanes>(acc.gl);
        // every lane holds the totals: all solve, each stores one word
        const float mass = pl.w, md = mass / (P.dt * P.dt);
        acc.l00 += md; acc.l11 += md; acc.l22 += md;
        acc.gl += ((xs - xyz(inert)) + ls) * md;
        V3 dx = solve3x3(acc.l00, acc.l10, acc.l11, acc.l20, acc.l21, acc.l22, -acc.gl);
        V3 hiN = xs, loN = ls;
        if (finite3(dx)) {
          const float maxLin = 0.35f * rad, l2 = dot(dx, dx);
          if (l2 > maxLin * maxLin) dx *= maxLin * rsq(l2);
          two_sum3(xs, ls + dx, hiN, loN);
        }
        if (lane < 6 && tiles > 1) {
          const float f = lane == 0 ? hiN.x : lane == 1 ? hiN.y : lane == 2 ? hiN.z : lane == 3 ? loN.x : lane == 4 ? loN.y : loN.z;
          __hip_atomic_store(S.tileX + 6ull * work.x + lane,
                             (uint64_t)(base + it + 1u) << 32 | (uint64_t)__float_as_uint(f), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
        } else if (lane == 6) {
          hi[work.w] = S.posLin[work.x] = f4(hiN, mass);
        } else if (lane == 7) {
          lo[work.w] = S.posLo[work.x] = f4(loN, 0.0f);
        }
      }
    }
    if (fastContact) {
      lds_sync();
      for (uint32_t i = own[0] + tid; i < own[colors]; i += nt) {
        const U4 w = S.tileWork[i];
        if (touch[w.w] == kTouchFast) dual_ground(P, ground[w.w], hi[w.w]);
      }
    }
    if (anyContact) {
      __syncthreads();  // the positions stored by this workgroup, read back by the dual
      for (uint32_t i = own[0] + tid / kMaxContacts; i < own[colors]; i += nt / kMaxContacts) {
        const U4 w = S.tileWork[i];
        if (touch[w.w] != kTouchAny) continue;
        const uint32_t ds = S.dAdjStart[w.x], dc = S.dAdjCount[w.x];
        for (uint32_t k = 0; k < dc; k++) dual_contact(S, P, S.dAdjList[ds + k] & kAdjIndexMask, tid % kMaxContacts);
      }
      __syncthreads();
    }
  }
  if (fastContact) {
    lds_sync();
    for (uint32_t i = own[0] + tid; i < own[colors]; i += nt) {
      const uint32_t w = S.tileWork[i].w;
      if (touch[w] == kTouchFast) ground_store(S, ground[w]);
    }
  }
  // the last workgroup out opens the next launch's versions
  if (tid == 0 && atomicAdd(&S.tileEpoch[1], 1u) == tiles - 1u) {
    S.tileEpoch[1] = 0u;
    S.tileEpoch[0] = base + P.iterations;
  }
}

// Waits inside, so all workgroups have to be resident: as an ordinary launch
// when no other kernel that waits is in flight, cooperative otherwise.  A
// cooperative launch goes through a queue of its own and cost 36 to 110 us of
// gaps around the kernel.
hipError_t launch_tile_solve(hipStream_t st, const DeviceState& S, const StepParams& P, uint32_t tiles,
                             uint32_t colors, uint32_t threads, bool cooperative) {
  if (!cooperative) {
    hipLaunchKernelGGL(k_tile_solve, dim3(tiles), dim3(threads), 0, st, S, P, colors);
    return hipGetLastError();
  }
  DeviceState s = S;
  StepParams p = P;
  void* args[] = {&s, &p, &colors};
  return hipLaunchCooperativeKernel((const void*)k_tile_solve, dim3(tiles), dim3(threads), args, 0, st);
}

bool tile_fits(uint32_t threads) {
  int per = 0;
  return hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k_tile_solve, (int)threads, 0) == hipSuccess && per > 1;
}

}  // namespace avbd
