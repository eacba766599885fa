// sweep.hpp -- device functions shared by the sweep kernels (solve.hip) and
// the island kernels (island.hip): neighbour enumeration, the lane-split
// primal of one body, the dual update of one constraint.
#pragma once
#include "kernels.hpp"
#include "stamps.hpp"

namespace avbd {

__device__ __forceinline__ bool body_dynamic(const DeviceState& S, uint32_t b) {
  return b != kWorld && S.posLin[b].w > 0.0f;
}

// ---------------------------------------------------------------------------
// neighbour enumeration for coloring: the other dynamic participants of an
// adjacency entry (40_solver.metal:260-318)
// ---------------------------------------------------------------------------
template <typename F>
__device__ __forceinline__ void for_each_neighbor(const DeviceState& S, uint32_t entry, uint32_t self, bool staticOnly,
                                                  F&& f) {
  uint32_t kind = entry >> kAdjShift, idx = entry & kAdjIndexMask;
  if (kind == FK_TET) {
    U4 ids = S.tets[idx].ids;
    uint32_t v[4] = {ids.x, ids.y, ids.z, ids.w};
    for (int k = 0; k < 4; k++)
      if (v[k] != self) f(v[k]);
  } else if (kind == FK_JOINT) {
    U4 h = S.joints[idx].header;
    f(h.x == self ? h.y : h.x);
  } else if (kind == FK_SPRING || kind == FK_PSPRING) {
    U4 h = S.springs[idx].header;
    f(h.x == self ? h.y : h.x);
  } else if (kind == FK_MANIFOLD && !staticOnly) {
    U4 h = S.manifolds[idx].header;
    f(h.x == self ? h.y : h.x);
  }
}

struct ColorMasks {
  uint64_t lower, all;
  bool conflict;
};
__device__ __forceinline__ ColorMasks neighbor_masks(const DeviceState& S, uint32_t v, const uint32_t* colors,
                                                     uint32_t myColor) {
  ColorMasks m{0ull, 0ull, false};
  auto visit = [&](uint32_t nb) {
    if (nb == kWorld || !body_dynamic(S, nb)) return;
    uint32_t c = colors[nb];
    uint64_t bit = c < 64 ? (1ull << c) : 0ull;
    m.all |= bit;
    if (nb < v) {
      m.lower |= bit;
      if (c == myColor) m.conflict = true;
    }
  };
  uint32_t s = S.sAdjStart[v], n = S.sAdjCount[v];
  for (uint32_t k = 0; k < n; k++) for_each_neighbor(S, S.sAdjList[s + k], v, false, visit);
  s = S.dAdjStart[v];
  n = S.dAdjCount[v];
  for (uint32_t k = 0; k < n; k++) for_each_neighbor(S, S.dAdjList[s + k], v, false, visit);
  return m;
}

// ---------------------------------------------------------------------------
// lane-split primal: L lanes stamp one body's adjacency slice each, DPP /
// ds_swizzle butterflies reduce the block system, lane 0 solves
// (40_solver.metal:1544-1685 re-mapped onto wave64).
// ---------------------------------------------------------------------------
template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}
__device__ __forceinline__ float swz16_f(float v) {
  return __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), 0x401F));
}
// Sum over aligned groups of L lanes; every lane of a group gets the total.
template <int L>
__device__ __forceinline__ float group_sum(float v) {
  if (L >= 2) v += dpp_f<0xB1>(v);    // quad_perm [1,0,3,2]: xor 1
  if (L >= 4) v += dpp_f<0x4E>(v);    // quad_perm [2,3,0,1]: xor 2
  if (L >= 8) v += dpp_f<0x141>(v);   // row_half_mirror: other quad of 8
  if (L >= 16) v += dpp_f<0x140>(v);  // row_mirror: other half of 16
  if (L >= 32) v += swz16_f(v);       // ds_swizzle xor 16
  return v;
}
template <int L>
__device__ __forceinline__ V3 group_sum3(V3 v) {
  return v3(group_sum<L>(v.x), group_sum<L>(v.y), group_sum<L>(v.z));
}

// Isotropic limiter (40_solver.metal:1361-1382): a particle's total
// displacement from the pose its bound holds around stays within
// max(0.45 sqrt(bound), 0.2 r); `cut` reports a truncation (counted for the
// refresh check and the frame's diagnostics by ogc_count).
__device__ __forceinline__ V3 ogc_truncate(const DeviceState& S, uint32_t body, V3 cur, V3 dx, float rad, bool& cut) {
  const float d2 = as_float(S.ogcBound[body]);
  if (!(d2 < 1e37f)) return dx;
  const float bv = fmaxf(0.45f * sqrtf(d2), 0.2f * rad);
  const V3 anchor = xyz(S.ogcPrev[body]);
  V3 tot = (cur + dx) - anchor;
  const float t2 = dot(tot, tot);
  if (t2 > bv * bv) {
    tot = tot * (bv / sqrtf(t2));
    dx = (anchor + tot) - cur;
    cut = true;
  }
  return dx;
}
// The wave's truncations in one pair of atomics (the lanes still running
// here are the solving lanes of the wave's bodies): per-body atomics on
// the two shared counters serialize when most particles are held back.
__device__ __forceinline__ void ogc_count(const DeviceState& S, bool cut) {
  const uint64_t m = __ballot(cut);
  if (m != 0ull && __lane_id() == (uint32_t)(__ffsll((unsigned long long)__activemask()) - 1)) {
    const uint32_t n = (uint32_t)__popcll(m);
    atomicAdd(&S.counters[CTR_OGC], n);
    atomicAdd(&S.counters[CTR_OGC_TRUNC], n);
  }
}

// Gathers and stamps one body's entries (lane-strided), reduces, and lane 0
// solves and writes.  Must be reached by whole waves (EXEC full) because of
// the ballot and DPP reductions; inactive groups pass active = false.
template <int L, int MODE>
__device__ __forceinline__ void primal_group(const DeviceState& S, const StepParams& P, bool active, U4 work,
                                             uint32_t lane, uint32_t color) {
  constexpr bool SOFT = MODE == kModeTet;
  const uint32_t body = work.x;
  bool rigid = MODE == kModeGeneral && active && S.shape[body].w >= 0.0f;
  const bool anyRigid = MODE == kModeGeneral && __ballot(rigid) != 0ull;
  Acc acc;
  acc_zero(acc);
  if (active) {
    PoseView pv{S.posLin, S.posAng, S.posLinSnap, S.posAngSnap, true};
    const V3 xs = xyz(S.posLin[body]), ls = xyz(S.posLo[body]);
    const uint32_t ss = work.y, sc = work.z;
    const uint32_t ds = S.dAdjStart[body], dc = S.dAdjCount[body];
    if (SOFT) {
      // particle colors: static entries are tets, per-frame entries manifolds.
      // Each lane first issues all of its slot-record loads of a batch, then
      // all position gathers, then the arithmetic.
      constexpr int B = L >= 32 ? 1 : (L == 16 ? 2 : 4);
      for (uint32_t base = lane; base < sc; base += L * B) {
        TetSlot r[B];
#pragma unroll
        for (int i = 0; i < B; i++) {
          uint32_t k = base + i * L;
          if (k < sc) r[i] = S.tetSlots[ss + k];
        }
        V3 x[B][3], lo[B][3];
#pragma unroll
        for (int i = 0; i < B; i++) {
          if (base + i * L < sc) {
            x[i][0] = xyz(S.posLin[r[i].other.x]);
            x[i][1] = xyz(S.posLin[r[i].other.y]);
            x[i][2] = xyz(S.posLin[r[i].other.z]);
            lo[i][0] = xyz(S.posLo[r[i].other.x]);
            lo[i][1] = xyz(S.posLo[r[i].other.y]);
            lo[i][2] = xyz(S.posLo[r[i].other.z]);
          }
        }
#pragma unroll
        for (int i = 0; i < B; i++)
          if (base + i * L < sc)
            stamp_tet_slot_e(r[i], split_edge(x[i][0], lo[i][0], xs, ls), split_edge(x[i][1], lo[i][1], xs, ls),
                             split_edge(x[i][2], lo[i][2], xs, ls), acc);
      }
      // contact entries continue the lane round-robin after the tets
      for (uint32_t k = (lane + L - (sc % L)) % L; k < dc; k += L) {
        uint32_t entry = S.dAdjList[ds + k];
        if ((entry >> kAdjShift) == FK_SOFT)
          stamp_soft(S.soft[entry & kSoftIndexMask], body, (entry >> kSoftSameShift) & 15u, pv, S.initLin, S.initAng,
                     P.alpha, acc);
        else
          stamp_manifold(S.manifolds[entry & kAdjIndexMask], body, false, pv, S.initLin, S.initAng, P.alpha, acc, ls);
      }
    } else if (MODE == kModeParticle) {
      // particles: cloth slots inline, any other static entry generically.  An
      // entry's word and slot are loaded while the one before is stamped, and the
      // first contact's word with the first slot: every pass of the loops
      // started with two dependent round trips to memory before (a color of the
      // draped 256^2 sheet took 19.4 us, 16.9 now, at 114 VGPRs against 104:
      // four waves per SIMD either way).
      uint32_t k = lane, kd = (lane + L - (sc % L)) % L;
      uint32_t entry = 0, contact = kd < dc ? S.dAdjList[ds + kd] : 0u;
      ClothSlot slot{};
      if (k < sc) {
        entry = S.sAdjList[ss + k];
        if (ss + k < S.numClothSlots) slot = S.clothSlots[ss + k];
      }
      while (k < sc) {
        const uint32_t next = k + L;
        uint32_t nextEntry = 0;
        ClothSlot nextSlot{};
        if (next < sc) {
          nextEntry = S.sAdjList[ss + next];
          if (ss + next < S.numClothSlots) nextSlot = S.clothSlots[ss + next];
        }
        uint32_t kind = entry >> kAdjShift;
        if (kind >= FK_MEMBRANE) stamp_cloth_slot(kind, slot, pv, xs, S.springs, P.alpha, acc);
        else stamp_entry(S, pv, entry, ss + k, body, xs, ls, false, P.alpha, P.dt, acc);
        k = next;
        entry = nextEntry;
        slot = nextSlot;
      }
      while (kd < dc) {
        const uint32_t next = kd + L;
        const uint32_t nextContact = next < dc ? S.dAdjList[ds + next] : 0u;
        if ((contact >> kAdjShift) == FK_SOFT)
          stamp_soft(S.soft[contact & kSoftIndexMask], body, (contact >> kSoftSameShift) & 15u, pv, S.initLin, S.initAng,
                     P.alpha, acc);
        else
          stamp_manifold(S.manifolds[contact & kAdjIndexMask], body, false, pv, S.initLin, S.initAng, P.alpha, acc, ls);
        kd = next;
        contact = nextContact;
      }
    } else {
      // static entries round-robin over the lanes; each contact manifold
      // split over the lanes contact by contact (a body's few manifolds
      // carry up to 8 contacts each), other per-frame entries round-robin
      for (uint32_t k = lane; k < sc; k += L) stamp_entry(S, pv, S.sAdjList[ss + k], ss + k, body, xs, ls, rigid,
                                                           P.alpha, P.dt, acc);
      for (uint32_t j = 0; j < dc; j++) {
        const uint32_t entry = S.dAdjList[ds + j];
        if ((entry >> kAdjShift) == FK_MANIFOLD)
          stamp_manifold(S.manifolds[entry & kAdjIndexMask], body, rigid, pv, S.initLin, S.initAng, P.alpha, acc, ls,
                         lane, (uint32_t)L);
        else if ((sc + j) % L == lane)
          stamp_entry(S, pv, entry, ss + sc + j, body, xs, ls, rigid, P.alpha, P.dt, acc);
      }
    }
  }
  acc.l00 = group_sum<L>(acc.l00);
  acc.l10 = group_sum<L>(acc.l10);
  acc.l11 = group_sum<L>(acc.l11);
  acc.l20 = group_sum<L>(acc.l20);
  acc.l21 = group_sum<L>(acc.l21);
  acc.l22 = group_sum<L>(acc.l22);
  acc.gl = group_sum3<L>(acc.gl);
  if (anyRigid) {
    acc.a00 = group_sum<L>(acc.a00);
    acc.a10 = group_sum<L>(acc.a10);
    acc.a11 = group_sum<L>(acc.a11);
    acc.a20 = group_sum<L>(acc.a20);
    acc.a21 = group_sum<L>(acc.a21);
    acc.a22 = group_sum<L>(acc.a22);
    acc.cr.r0 = group_sum3<L>(acc.cr.r0);
    acc.cr.r1 = group_sum3<L>(acc.cr.r1);
    acc.cr.r2 = group_sum3<L>(acc.cr.r2);
    acc.ga = group_sum3<L>(acc.ga);
  }
  if (!active || lane != 0) return;
  F4 pl = S.posLin[body];
  const V3 lo = xyz(S.posLo[body]);
  float mass = pl.w, dt2 = P.dt * P.dt;
  float md = mass / dt2;
  acc.l00 += md; acc.l11 += md; acc.l22 += md;
  acc.gl += ((xyz(pl) - xyz(S.inertLin[body])) + lo) * md;
  V3 dxL, dxA = v3s(0);
  float rad = fabsf(S.shape[body].w);
  if (rigid) {
    F4 q = S.posAng[body];
    M3 inertia = m3_scale(world_inertia(q, xyz(S.props[body])), 1.0f / dt2);
    acc_ang_m3(acc, inertia);
    acc.ga += m3_mul(inertia, q_sub(q, S.inertAng[body]));
    solve6x6(lower_to_m3(acc.l00, acc.l10, acc.l11, acc.l20, acc.l21, acc.l22),
             lower_to_m3(acc.a00, acc.a10, acc.a11, acc.a20, acc.a21, acc.a22), acc.cr, -acc.gl, -acc.ga, dxL, dxA);
    if (!finite3(dxL) || !finite3(dxA)) return;
    float a2 = dot(dxA, dxA);
    if (a2 > 0.25f) dxA *= 0.5f * rsq(a2);
  } else {
    dxL = solve3x3(acc.l00, acc.l10, acc.l11, acc.l20, acc.l21, acc.l22, -acc.gl);
    if (!finite3(dxL)) return;
  }
  float maxLin = 0.35f * rad;
  float l2 = dot(dxL, dxL);
  if (l2 > maxLin * maxLin) dxL *= maxLin * rsq(l2);
  if (P.isoOn) {
    bool cut = false;
    if (!rigid) dxL = ogc_truncate(S, body, xyz(pl), dxL, rad, cut);
    ogc_count(S, cut);
  }
  // (hi, lo) + dx, renormalised exactly: hi = f32(hi + t), lo = the error term
  V3 hiN, loN;
  two_sum3(xyz(pl), lo + dxL, hiN, loN);
  S.posLin[body] = f4(hiN, mass);
  S.posLo[body] = f4(loN, 0.0f);
  if (rigid) S.posAng[body] = q_addw(S.posAng[body], dxA);
}

// (body, static CSR start, static CSR count) of a body of a device-built palette
__device__ __forceinline__ U4 body_work(const DeviceState& S, bool active, uint32_t body) {
  return active ? U4{body, S.sAdjStart[body], S.sAdjCount[body], 0u} : U4{0u, 0u, 0u, 0u};
}

// ---------------------------------------------------------------------------
// augmented-Lagrangian dual + penalty ramp (40_solver.metal:1689-1910)
// ---------------------------------------------------------------------------
__device__ __forceinline__ void dual_joint(const DeviceState& S, const StepParams& P, uint32_t gid) {
  JointRec& j = S.joints[gid];
  if (j.header.z != 0) return;
  uint32_t a = j.header.x, b = j.header.y;
  float torqueArm = j.C0Lin.w;
  V3 penLin = xyz(j.penaltyLin);
  if (dot(penLin, penLin) > 0.0f) {
    V3 pA = a == kWorld ? xyz(j.rA) : xform(xyz(S.posLin[a]), S.posAng[a], xyz(j.rA));
    V3 pB = xform(xyz(S.posLin[b]), S.posAng[b], xyz(j.rB));
    V3 C = pA - pB;
    if (j.header.w & 1u) {
      C -= xyz(j.C0Lin) * P.alpha;
      V3 l = penLin * C + xyz(j.lambdaLin);
      j.lambdaLin = f4(v3(clampf(l.x, -P.lambdaMax, P.lambdaMax), clampf(l.y, -P.lambdaMax, P.lambdaMax),
                          clampf(l.z, -P.lambdaMax, P.lambdaMax)),
                       j.lambdaLin.w);
    }
    float cap = fminf(j.rA.w, kPenaltyMax);
    V3 np = penLin + vabs(C) * P.betaLin;
    j.penaltyLin = f4(v3(fminf(np.x, cap), fminf(np.y, cap), fminf(np.z, cap)), j.penaltyLin.w);
  }
  V3 penAng = xyz(j.penaltyAng);
  if (dot(penAng, penAng) > 0.0f) {
    F4 qA = a == kWorld ? F4{0, 0, 0, 1} : S.posAng[a];
    V3 C;
    if (j.hingeAxis.w != 0.0f) {
      V3 aB = q_rotate(S.posAng[b], xyz(j.hingeAxis));
      V3 aA = q_rotate(q_mul(qA, j.restRel), xyz(j.hingeAxis));
      C = cross(aA, aB) * torqueArm;
    } else {
      C = q_sub(q_mul(qA, j.restRel), S.posAng[b]) * torqueArm;
    }
    if (j.header.w & 2u) {
      C -= xyz(j.C0Ang) * P.alpha;
      V3 l = penAng * C + xyz(j.lambdaAng);
      j.lambdaAng = f4(v3(clampf(l.x, -P.lambdaMax, P.lambdaMax), clampf(l.y, -P.lambdaMax, P.lambdaMax),
                          clampf(l.z, -P.lambdaMax, P.lambdaMax)),
                       j.lambdaAng.w);
    }
    float cap = fminf(j.rB.w, kPenaltyMax);
    V3 np = penAng + vabs(C) * P.betaAng;
    j.penaltyAng = f4(v3(fminf(np.x, cap), fminf(np.y, cap), fminf(np.z, cap)), j.penaltyAng.w);
  }
  float fracture = j.C0Ang.w;
  V3 la = xyz(j.lambdaAng);
  float lin2 = (j.header.w & 8u) ? dot(xyz(j.lambdaLin), xyz(j.lambdaLin)) : 0.0f;
  if ((j.header.w & 4u) && dot(la, la) + lin2 > fracture * fracture) {
    j.penaltyLin = F4{0, 0, 0, 0};
    j.penaltyAng = F4{0, 0, 0, 0};
    j.lambdaLin = F4{0, 0, 0, 0};
    j.lambdaAng = F4{0, 0, 0, 0};
    j.header.z = 1;
  }
}

__device__ __forceinline__ void dual_spring(const DeviceState& S, const StepParams& P, uint32_t si) {
  SpringRec& sp = S.springs[si];
  if (sp.header.z == 0) return;
  uint32_t a = sp.header.x, b = sp.header.y;
  V3 pA = xform(xyz(S.posLin[a]), S.posAng[a], xyz(sp.rA));
  V3 pB = xform(xyz(S.posLin[b]), S.posAng[b], xyz(sp.rB));
  float C = length(pA - pB) - sp.rB.w - sp.dual.z * P.alpha;
  float mA = S.posLin[a].w, mB = S.posLin[b].w;
  float big = 3.402823466e38f;
  float mMin = fminf(mA > 0.0f ? mA : big, mB > 0.0f ? mB : big);
  float cap = fminf(P.lambdaMax, fmaxf(2.0f, 5.0e3f * mMin));
  sp.dual.x = clampf(0.98f * sp.dual.x + sp.dual.y * C, 0.0f, cap);
  if (C > 0.0f) sp.dual.y = fminf(sp.dual.y + C * P.betaLin, fminf(sp.rA.w, kPenaltyMax));
}

// One item per contact slot (kMaxContacts per manifold): a contact's update
// reads only its own record and the manifold's shared header, basis and
// body poses, so the slots of a manifold run on adjacent lanes and their
// records load as one contiguous span instead of a serial loop per thread.
__device__ __forceinline__ void dual_contact(const DeviceState& S, const StepParams& P, uint32_t gid, uint32_t i) {
  ManifoldRec& m = S.manifolds[gid];
  uint32_t n = m.header.z;
  if (i >= n) return;
  uint32_t a = m.header.x, b = m.header.y;
  bool rA_round = (m.header.w & 2u) != 0, rB_round = (m.header.w & 4u) != 0;
  V3 dqAL = xyz(S.posLin[a]) - xyz(S.initLin[a]);
  V3 dqAA = q_sub(S.posAng[a], S.initAng[a]);
  V3 dqBL = xyz(S.posLin[b]) - xyz(S.initLin[b]);
  V3 dqBA = q_sub(S.posAng[b], S.initAng[b]);
  float mA = S.posLin[a].w, mB = S.posLin[b].w;
  float big = 3.402823466e38f;
  float minMass = fminf(mA > 0.0f ? mA : big, mB > 0.0f ? mB : big);
  float lamCap = fminf(P.lambdaMax, fmaxf(10.0f, 1.0e5f * minMass));
  V3 nrm = xyz(m.basisN), t1 = xyz(m.basisT1), t2 = cross(nrm, t1);
  {
    V3 rAW = rA_round ? xyz(m.c[i].rA) : q_rotate(S.posAng[a], xyz(m.c[i].rA));
    V3 rBW = rB_round ? xyz(m.c[i].rB) : q_rotate(S.posAng[b], xyz(m.c[i].rB));
    V3 C;
    float fs, bnd;
    V3 F = contact_force(m, (int)i, dqAL, dqAA, dqBL, dqBA, rAW, rBW, P.alpha, nrm, t1, t2, C, fs, bnd);
    F.x = fmaxf(F.x, -lamCap);
    m.c[i].lambda = f4(F, 0.0f);
    V3 pen = xyz(m.c[i].penalty);
    if (F.x < 0.0f) pen.x = fminf(pen.x + P.betaLin * fabsf(C.x), kPenaltyMax);
    if (fs <= bnd) {
      pen.y = fminf(pen.y + P.betaLin * fabsf(C.y), kPenaltyMaxT);
      pen.z = fminf(pen.z + P.betaLin * fabsf(C.z), kPenaltyMaxT);
      m.c[i].rB.w = sqrtf(C.y * C.y + C.z * C.z) < kStickThresh ? 1.0f : 0.0f;
    }
    m.c[i].penalty = f4(pen, 0.0f);
  }
}

// element contact dual: the quadratic stage only (the log-barrier stage is
// dual-free), mass-scaled normal cap, penalties capped at 1e6
// (40_solver.metal:1689-1727)
__device__ __forceinline__ void dual_soft(const DeviceState& S, const StepParams& P, uint32_t gid) {
  SoftRec& sc = S.soft[gid];
  PoseView pv{S.posLin, S.posAng, S.posLin, S.posAng, false};
  V3 n, t1, t2, rAW;
  V3 C = soft_contact_C(sc, pv, 0u, S.initLin, S.initAng, P.alpha, n, t1, t2, rAW);
  V3 F = xyz(sc.penalty) * C + xyz(sc.lambda);
  F.x = fminf(F.x, 0.0f);
  float bnd = fabsf(F.x) * sc.normal.w;
  float fs = sqrtf(F.y * F.y + F.z * F.z);
  if (fs > bnd && fs > 0.0f) {
    F.y *= bnd / fs;
    F.z *= bnd / fs;
  }
  F.x = fmaxf(F.x, -sc.C0.w);
  sc.lambda = f4(F, sc.lambda.w);
  V3 pen = xyz(sc.penalty);
  if (F.x < 0.0f) pen.x = fminf(pen.x + P.betaLin * fabsf(C.x), kPenaltyMaxT);
  if (fs <= bnd) {
    pen.y = fminf(pen.y + P.betaLin * fabsf(C.y), kPenaltyMaxT);
    pen.z = fminf(pen.z + P.betaLin * fabsf(C.z), kPenaltyMaxT);
  }
  sc.penalty = f4(pen, sc.penalty.w);
}

// one item of the fused dual pass over [joints | springs | manifolds | soft],
// plus the next iteration's pose snapshot over bodies
__device__ __forceinline__ void dual_item(const DeviceState& S, const StepParams& P, uint32_t gid, uint32_t numPairs) {
  if (gid < P.numJoints) { dual_joint(S, P, gid); return; }
  uint32_t si = gid - P.numJoints;
  if (si < P.numSprings) { dual_spring(S, P, si); return; }
  uint32_t mi = si - P.numSprings;
  if (mi < numPairs * kMaxContacts) { dual_contact(S, P, mi / kMaxContacts, mi % kMaxContacts); return; }
  dual_soft(S, P, mi - numPairs * kMaxContacts);
}

// Grid barrier (every workgroup resident).
// Every wait is bounded: past the spin bound a block records CTR_GBAR_FAIL
// and proceeds, and once any block has given up later barriers do not wait,
// so the grid always drains.
// One release (cache write-back) before arriving, relaxed polling of the
// arrival counter, and one acquire (cache invalidate) once it is reached:
// an acquire load inside the spin would invalidate the L2 on every poll.
__device__ __forceinline__ void grid_barrier(uint32_t* bar, uint32_t* fail, uint32_t target) {
  __syncthreads();
  if (threadIdx.x == 0) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    __hip_atomic_fetch_add(bar, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    uint32_t spins = 0;
    while (__hip_atomic_load(bar, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < target &&
           __hip_atomic_load(fail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0u) {
      __builtin_amdgcn_s_sleep(1);
      if (++spins > (1u << 20)) {
        atomicAdd(fail, 1u);
        break;
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  }
  __syncthreads();
}

// XCD-aware block order: the hardware deals consecutive workgroups to the
// 8 XCDs round-robin; remapping gives each XCD one contiguous slice of the
// color list so neighbour gathers of adjacent bodies share that XCD's L2.
__device__ __forceinline__ uint32_t xcd_block(uint32_t b, uint32_t n) {
  const uint32_t X = 8;
  uint32_t per = (n + X - 1) / X;
  uint32_t r = (b % X) * per + b / X;
  return r;
}

// Every sweep of the whole grid, a grid barrier after each color and each dual
template <int L, int MODE>
__device__ __forceinline__ void grid_sweeps(const DeviceState& S, const StepParams& P, uint32_t numColors,
                                            uint32_t barrierBase) {
  const uint32_t groupsPerBlock = blockDim.x / L;
  const uint32_t lane = threadIdx.x & (L - 1);
  const uint32_t block = gridDim.x % 8u ? blockIdx.x : xcd_block(blockIdx.x, gridDim.x);
  const uint32_t gslot = block * groupsPerBlock + threadIdx.x / L;
  const uint32_t ngroups = gridDim.x * groupsPerBlock;
  uint32_t* bar = &S.counters[CTR_GBAR];
  uint32_t* fail = &S.counters[CTR_GBAR_FAIL];
  uint32_t epoch = barrierBase;
  const uint32_t colorsUsed = numColors ? numColors : S.colorStart[kMaxColors + 1];
  const uint32_t numPairs = S.counters[CTR_PAIRS];
  const uint32_t dualTotal = P.numJoints + P.numSprings + numPairs * kMaxContacts + S.counters[CTR_SOFT];
  const uint32_t tid = blockIdx.x * blockDim.x + threadIdx.x, nthreads = gridDim.x * blockDim.x;
  for (uint32_t it = 0; it < P.iterations; it++) {
    for (uint32_t c = 0; c < colorsUsed; c++) {
      uint32_t s = S.colorStart[c], e = S.colorStart[c + 1];
      uint32_t count = e - s;
      uint32_t rounds = (count + ngroups - 1) / ngroups;
      for (uint32_t r = 0; r < rounds; r++) {
        uint32_t slot = r * ngroups + gslot;
        bool active = slot < count;
        primal_group<L, MODE>(S, P, active,
                              numColors ? (active ? S.colorWork[s + slot] : U4{0u, 0u, 0u, 0u})
                                        : body_work(S, active, active ? S.colorList[s + slot] : 0u),
                              lane, c);
      }
      epoch += gridDim.x;
      grid_barrier(bar, fail, epoch);
    }
    for (uint32_t g = tid; g < dualTotal; g += nthreads) dual_item(S, P, g, numPairs);
    for (uint32_t b = tid; b < P.numBodies; b += nthreads) {
      S.posLinSnap[b] = S.posLin[b];
      S.posAngSnap[b] = S.posAng[b];
    }
    epoch += gridDim.x;
    grid_barrier(bar, fail, epoch);
  }
}

}  // namespace avbd
