// Brick tiles shared by the forward and reverse gather passes.
//
// A workgroup owns one brick of 4x4x4 cells.  After the counting sort the
// brick's particles are contiguous and all their neighbours lie in the brick's
// 6x6x6-cell halo; tile slots number the halo's particles (halo cells in
// (z, y, x) order, particles of a cell in sorted order).  Fluid neighbour
// lists hold 16-bit tile slots, eight per 16-byte pack, packs stored
// pack-major (nbr8[p * N + i]).
#pragma once
#include "dfr_kernels.h"

namespace dfr {

constexpr int HALO = 216;

template <int NT> struct TileHdr {
  uint32_t cstart[HALO];      // first particle (global sorted index) of each halo cell
  uint32_t coff[HALO + 1];    // tile slot of each halo cell's first particle
  uint32_t scan[NT / 64 + 1];
  uint32_t own_begin, own_end, total;
  int bx, by, bz;
};

template <int NT>
__device__ inline void tile_setup(const GridDesc& g, const uint32_t* __restrict__ fstart, uint32_t brick,
                                  TileHdr<NT>& T) {
  const int bx = (int)(brick % (uint32_t)g.bn[0]);
  const int by = (int)((brick / (uint32_t)g.bn[0]) % (uint32_t)g.bn[1]);
  const int bz = (int)(brick / ((uint32_t)g.bn[0] * (uint32_t)g.bn[1]));
  const int t = threadIdx.x;
  uint32_t cnt = 0;
  if (t < HALO) {
    const int cx = 4 * bx - 1 + t % 6, cy = 4 * by - 1 + (t / 6) % 6, cz = 4 * bz - 1 + t / 36;
    uint32_t st = 0;
    if (cx >= 0 && cy >= 0 && cz >= 0 && cx < g.n[0] && cy < g.n[1] && cz < g.n[2]) {
      const uint32_t key = cell_key(g, cx, cy, cz);
      st = fstart[key];
      cnt = fstart[key + 1] - st;
    }
    T.cstart[t] = st;
  }
  uint32_t total;
  const uint32_t ex = block_exclusive_scan<NT>(cnt, T.scan, total);
  if (t < HALO) T.coff[t] = ex;
  if (t == 0) {
    T.coff[HALO] = total;
    T.total = total;
    T.own_begin = fstart[brick * 64u];
    T.own_end = fstart[brick * 64u + 64u];
    T.bx = bx; T.by = by; T.bz = bz;
  }
  __syncthreads();
}

// Global sorted index of a tile slot (slot < total).
template <int NT> __device__ inline uint32_t tile_global(const TileHdr<NT>& T, uint32_t slot) {
  int lo = 0, hi = HALO - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (T.coff[mid] <= slot) lo = mid; else hi = mid - 1;
  }
  return T.cstart[lo] + (slot - T.coff[lo]);
}

// Halo cell index of the cell (cx, cy, cz) + (dx, dy, dz) for a particle of the brick.
template <int NT>
__device__ inline int halo_cell(const TileHdr<NT>& T, int cx, int cy, int cz, int dx, int dy, int dz) {
  return (cz + dz - 4 * T.bz + 1) * 36 + (cy + dy - 4 * T.by + 1) * 6 + (cx + dx - 4 * T.bx + 1);
}

// Two-phase halo staging: every thread first resolves its slots to particle
// indices (LDS-only binary searches, independent), then issues all its global
// loads before writing LDS, so the loads are in flight together.  CAP is the
// largest capacity (registers per thread); slots >= total are skipped.
template <int NT, int CAP = TILE_CAP> constexpr int per_thread() { return (CAP + NT - 1) / NT; }

template <int NT, int CAP = TILE_CAP>
__device__ inline void tile_indices(const TileHdr<NT>& T, uint32_t total, uint32_t* js) {
#pragma unroll
  for (int r = 0; r < per_thread<NT, CAP>(); ++r) {
    const uint32_t s = threadIdx.x + r * NT;
    js[r] = (s < total) ? tile_global<NT>(T, s) : 0u;
  }
}

// Uniform early exit for bricks that own no particle (about half of a tank's
// bricks lie above the free surface): two scalar loads, no halo setup.
__device__ inline bool brick_empty(const uint32_t* __restrict__ fstart, uint32_t brick) {
  return fstart[brick * 64u] == fstart[brick * 64u + 64u];
}

__device__ inline uint32_t pack_get(const uint4& v, int u) {
  const uint32_t w = (u < 2) ? v.x : (u < 4) ? v.y : (u < 6) ? v.z : v.w;
  return (u & 1) ? (w >> 16) : (w & 0xffffu);
}

struct PassArgs {
  StepConst c;
  GridDesc g;
  const uint32_t* fstart;
  const float4* pos;
  float4* vel;
  const float4* bpos;
  const float4* bvel;
  const float4* bx0;
  const uint4* nbr8;
  const uint4* thdr;      // brick headers and halo slot maps written by the build
  const uint32_t* tmap;
  const uint32_t* nbrB;
  const uint32_t* cnt;
  int nb_static;
  int cap;  // halo slots staged in LDS (larger halos read global memory)
  int parts_log2;  // workgroups per brick: 2^parts_log2 (NbrBufs)
};

inline unsigned nbricks(const GridDesc& g) { return (unsigned)(g.bn[0] * g.bn[1] * g.bn[2]); }

inline PassArgs make_args(const StepConst& c, const GridDesc& g, GridBufs& gb, FluidBufs& f, BoundaryBufs& b,
                          NbrBufs& nb) {
  PassArgs a;
  a.c = c; a.g = g; a.fstart = gb.fstart; a.pos = f.pos; a.vel = f.vel; a.bpos = b.pos; a.bvel = b.vel;
  a.bx0 = b.x0; a.nbr8 = nb.nbr8; a.nbrB = nb.nbrB; a.cnt = nb.cnt; a.nb_static = b.n - b.nd;
  a.thdr = nb.thdr; a.tmap = nb.tmap;
  a.cap = nb.cap;
  a.parts_log2 = nb.parts_log2;
  return a;
}

// The passes that run once a step: one workgroup per brick at every size.
inline PassArgs whole_bricks(PassArgs a) {
  a.parts_log2 = 0;
  return a;
}
// Workgroups of a gather pass.
inline unsigned pass_grid(const GridDesc& g, int parts_log2) { return nbricks(g) << parts_log2; }

// A pass's view of its brick: the particles of its own that this workgroup
// handles (all of them, or one of 2^parts_log2 ranges of whole wavefronts of
// four lanes a particle; each stages the whole halo).  The build leaves, per
// brick, a header (own particle range, halo total) and the halo's slot -> particle map, so a pass
// starts with one header load and coalesced map loads; only a halo beyond the
// LDS capacity sets up the cell table for the binary-search fallback.
struct BrickView {
  uint32_t own_begin, own_end, total;
  uint32_t brick, block;  // block: this workgroup's number in the pass
  bool in_lds;
};
template <int NT, class Args>
__device__ inline bool brick_open(const Args& a, TileHdr<NT>& T, BrickView& B) {
  B.block = xcd_block();
  B.brick = B.block >> a.parts_log2;
  const uint4 h = a.thdr[B.brick];
  const uint32_t parts = 1u << a.parts_log2, part = B.block & (parts - 1u);
  const uint32_t per = (((h.y - h.x + parts - 1u) >> a.parts_log2) + 15u) & ~15u;
  B.own_begin = h.x + (parts > 1u ? part * per : 0u);
  B.own_end = parts > 1u ? min(B.own_begin + per, h.y) : h.y;
  if (B.own_begin >= B.own_end) return false;  // no own particle (uniform exit)
  B.total = h.z;
  B.in_lds = h.z <= (uint32_t)a.cap;
  if (!B.in_lds) tile_setup<NT>(a.g, a.fstart, B.brick, T);
  return true;
}
template <int NT, int CAP = TILE_CAP>
__device__ inline void map_indices(const uint32_t* __restrict__ tmap, uint32_t brick, uint32_t total, uint32_t* js) {
#pragma unroll
  for (int r = 0; r < per_thread<NT, CAP>(); ++r) {
    const uint32_t s = threadIdx.x + r * NT;
    js[r] = (s < total) ? tmap[(size_t)brick * TILE_CAP + s] : 0u;
  }
}

// Visits the nF fluid neighbour slots of particle i in list order: a loop over
// the packs with the eight slots of a pack unrolled, the pack two ahead in
// flight (a compact loop body keeps the instruction stream small).
template <class Body>
__device__ inline void for_fluid_slots(const uint4* __restrict__ nbr8, size_t stride, uint32_t i, uint32_t nF,
                                       Body&& body) {
  // rows past the last used one are read as that row again (in bounds, in
  // cache) and never used
  const uint32_t np = (nF + PACK - 1) / PACK;
  const uint32_t last = np > 0 ? np - 1 : 0;
  uint4 cur = nbr8[i];
  uint4 nxt = nbr8[(size_t)min(1u, last) * stride + i];
#pragma unroll 1
  for (uint32_t p = 0; p < np; ++p) {
    const uint4 pk = cur;
    cur = nxt;
    nxt = nbr8[(size_t)min(p + 2, last) * stride + i];
    const uint32_t base = p * PACK;
#pragma unroll
    for (int u = 0; u < PACK; ++u)
      if (base + (uint32_t)u < nF) body(pack_get(pk, u));
  }
}

// Branch-free visit of the same slots for LDS-staged halos.  Within a pack the
// slots go in groups of G: `load(s)` of every slot of a group is issued before
// the first `body`, so the group's LDS reads are in flight together, then
// `body(v, live)` runs in slot order.  `live` is false for the slots past nF
// in the last pack; those hold slot 0 (a staged slot, so the read stays in
// bounds), and the body must select their contribution to zero.  A group
// wholly past nF is skipped.
template <int G, class Load, class Body>
__device__ inline void for_fluid_groups(const uint4* __restrict__ nbr8, size_t stride, uint32_t i, uint32_t nF,
                                        Load&& load, Body&& body) {
  static_assert(PACK % G == 0, "the group size divides the pack");
  const uint32_t np = (nF + PACK - 1) / PACK;
  const uint32_t last = np > 0 ? np - 1 : 0;
  uint4 cur = nbr8[i];
  uint4 nxt = nbr8[(size_t)min(1u, last) * stride + i];
#pragma unroll 1
  for (uint32_t p = 0; p < np; ++p) {
    const uint4 pk = cur;
    cur = nxt;
    nxt = nbr8[(size_t)min(p + 2, last) * stride + i];
    const uint32_t rem = nF - p * PACK;  // >= 1
#pragma unroll
    for (int g0 = 0; g0 < PACK; g0 += G) {
      if (g0 > 0 && rem <= (uint32_t)g0) break;
      decltype(load(0u)) v[G];
#pragma unroll
      for (int u = 0; u < G; ++u) v[u] = load(pack_get(pk, g0 + u));
#pragma unroll
      for (int u = 0; u < G; ++u) body(v[u], (uint32_t)(g0 + u) < rem);
    }
  }
}

// The same with four lanes per particle, for the reverse passes (see
// dfr_spread.h): lane l takes the slots 2 l and 2 l + 1 of each pack, two
// packs a round; the partial sums of the lanes are added at the end (lane_sum).
template <int G, int L, class Load, class Body>
__device__ inline void for_fluid_lanes(const uint4* __restrict__ nbr8, size_t stride, uint32_t i, uint32_t nF, int l,
                                       Load&& load, Body&& body) {
  if constexpr (L == 1) {
    for_fluid_groups<G>(nbr8, stride, i, nF, load, body);
  } else {
    static_assert(L == 4, "a pack holds four pairs of slots");
    const uint32_t* __restrict__ words = reinterpret_cast<const uint32_t*>(nbr8);
    const uint32_t np = (nF + PACK - 1) / PACK;
    const uint32_t last = np > 0 ? np - 1 : 0;
    auto word = [&](uint32_t p) { return words[((size_t)min(p, last) * stride + i) * 4 + l]; };
    uint32_t a = word(0), b = word(1), a2 = word(2), b2 = word(3);
#pragma unroll 1
    for (uint32_t p = 0; p < np; p += 2) {
      const uint32_t s0 = a & 0xffffu, s1 = a >> 16, s2 = b & 0xffffu, s3 = b >> 16;
      a = a2; b = b2;
      a2 = word(p + 4); b2 = word(p + 5);
      const uint32_t e = p * PACK + 2u * (uint32_t)l;
      // rows past the last one repeat it: their slots are not live
      const auto v0 = load(s0), v1 = load(s1), v2 = load(s2), v3 = load(s3);
      body(v0, e < nF);
      body(v1, e + 1u < nF);
      body(v2, e + (uint32_t)PACK < nF);
      body(v3, e + (uint32_t)PACK + 1u < nF);
    }
  }
}

// Sum over the L lanes of a particle (consecutive lanes), in every lane.
template <int L> __device__ inline float lane_sum(float x) {
  if constexpr (L == 4) {
    x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0xB1, 0xf, 0xf, true));  // quad_perm [1,0,3,2]
    x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x4E, 0xf, 0xf, true));  // quad_perm [2,3,0,1]
  }
  return x;
}

// Visits the nB boundary neighbours of particle i in list order, G at a time:
// the group's sample indices are loaded first, then the group's sample data
// (`load(j)`), so a group costs two dependent trips to memory instead of two
// per neighbour; `body(v, j, u)` then runs for the group's neighbours in order,
// u their place in the group.
// With L lanes per particle, lane l takes every L-th neighbour from l on.
template <uint32_t G = 4, uint32_t L = 1, class Load, class Body>
__device__ inline void for_boundary_groups(const uint32_t* __restrict__ nbrB, size_t stride, uint32_t i,
                                           uint32_t nB, Load&& load, Body&& body, uint32_t l = 0) {
#pragma unroll 1
  for (uint32_t k0 = l; k0 < nB; k0 += G * L) {
    uint32_t jj[G];
#pragma unroll
    for (uint32_t u = 0; u < G; ++u) jj[u] = nbrB[(size_t)min(k0 + u * L, nB - 1) * stride + i];
    decltype(load(0u)) v[G];
#pragma unroll
    for (uint32_t u = 0; u < G; ++u) v[u] = load(jj[u]);
#pragma unroll
    for (uint32_t u = 0; u < G; ++u)
      if (k0 + u * L < nB) body(v[u], jj[u], u);
  }
}

// ---------------------------------------------------------------------------
// Four lanes per particle in the step's own passes (L = 4: small scenes, see
// dfr_spread.h).  The lanes of a quad evaluate different pairs; every lane
// then adds all pairs' terms in list order, reading each from the lane that has
// it (a quad broadcast costs one instruction), so the sums are those of one lane
// per particle bit for bit.  `term` forms what a pair contributes (Terms), `acc`
// adds it; with L = 1 they run one after the other.  This pays for two to four
// terms a pair: the reverse passes' seven to twelve took 9.2 us in place of 6.7
// (delta, 2,000 particles).
// ---------------------------------------------------------------------------
template <int N> struct Terms {
  float f[N];
};
template <int K, int N> __device__ inline Terms<N> quad_bcast(const Terms<N>& t) {
  Terms<N> o;
#pragma unroll
  for (int n = 0; n < N; ++n)
    o.f[n] = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(t.f[n]), K * 0x55, 0xf, 0xf, true));
  return o;
}

// Fluid pairs: lane l of the quad takes slots 2 l and 2 l + 1 of each pack.
template <int G, int L, class Load, class Term, class Acc>
__device__ inline void for_fluid_terms(const uint4* __restrict__ nbr8, size_t stride, uint32_t i, uint32_t nF, int l,
                                       Load&& load, Term&& term, Acc&& acc) {
  if constexpr (L == 1) {
    for_fluid_groups<G>(nbr8, stride, i, nF, load, [&](const auto& v, bool live) { acc(term(v, live)); });
  } else {
    static_assert(L == 4, "a pack holds four pairs of slots");
    const uint32_t* __restrict__ words = reinterpret_cast<const uint32_t*>(nbr8);
    const uint32_t np = (nF + PACK - 1) / PACK;
    const uint32_t last = np > 0 ? np - 1 : 0;
    auto word = [&](uint32_t p) { return words[((size_t)min(p, last) * stride + i) * 4 + l]; };
    uint32_t w0 = word(0), w1 = word(1), w2 = word(2);
#pragma unroll 1
    for (uint32_t p = 0; p < np; ++p) {
      const uint32_t s0 = w0 & 0xffffu, s1 = w0 >> 16;
      w0 = w1; w1 = w2; w2 = word(p + 3);
      const uint32_t e = p * PACK + 2u * (uint32_t)l;
      const auto v0 = load(s0), v1 = load(s1);
      const auto t0 = term(v0, e < nF), t1 = term(v1, e + 1u < nF);
      acc(quad_bcast<0>(t0)); acc(quad_bcast<0>(t1));
      acc(quad_bcast<1>(t0)); acc(quad_bcast<1>(t1));
      acc(quad_bcast<2>(t0)); acc(quad_bcast<2>(t1));
      acc(quad_bcast<3>(t0)); acc(quad_bcast<3>(t1));
    }
  }
}

// The same order with the particles read from global memory (a halo beyond the LDS
// capacity): four slots a round, lane l of the quad takes the l-th, one pair a lane in
// flight (two spill a register of the velocity update).
template <class Load, class Term, class Acc>
__device__ inline void for_fluid_terms_rolled(const uint4* __restrict__ nbr8, size_t stride, uint32_t i, uint32_t nF,
                                              int l, Load&& load, Term&& term, Acc&& acc) {
  const uint16_t* __restrict__ slots = reinterpret_cast<const uint16_t*>(nbr8);
#pragma unroll 1
  for (uint32_t k0 = 0; k0 < nF; k0 += 4) {
    const uint32_t k = k0 + (uint32_t)l;  // of the same pack as k0; past the list's end a pack holds slot 0
    const auto t = term(load((uint32_t)slots[((size_t)(k / PACK) * stride + i) * PACK + k % PACK]), k < nF);
    acc(quad_bcast<0>(t));
    acc(quad_bcast<1>(t));
    acc(quad_bcast<2>(t));
    acc(quad_bcast<3>(t));
  }
}

// Which product of a boundary pair's three is rounded by itself, and whether its
// share is added fused, has always gone by the neighbour's place u in its group
// of the one-lane loop; both forms take it from u, so that a particle's sums are
// the same bits by either.
__device__ inline float place_dot(uint32_t u, float ax, float ay, float az, float bx, float by, float bz) {
  const bool x_first = (u & 2u) == 0u;
  const float a0 = x_first ? ax : ay, b0 = x_first ? bx : by, a1 = x_first ? ay : ax, b1 = x_first ? by : bx;
  return fmaf(az, bz, fmaf(a1, b1, a0 * b0));
}

// Boundary samples: lane l of the quad takes neighbours l and l + 4 of each
// eight; `term(v, j, u)` runs once per neighbour (its side effects too), u the
// neighbour's place in its group of G.
template <uint32_t G, int L, class Load, class Term, class Acc>
__device__ inline void for_boundary_terms(const uint32_t* __restrict__ nbrB, size_t stride, uint32_t i, uint32_t nB,
                                          int l, Load&& load, Term&& term, Acc&& acc) {
  static_assert(4 % G == 0, "a lane's neighbours have one place in their groups");
  if constexpr (L == 1) {
    for_boundary_groups<G>(nbrB, stride, i, nB, load,
                           [&](const auto& v, uint32_t j, uint32_t u) { acc(term(v, j, u), u); });
  } else {
#pragma unroll 1
    for (uint32_t k0 = 0; k0 < nB; k0 += 8) {
      const uint32_t ka = k0 + (uint32_t)l, kb = ka + 4u, u = (uint32_t)l % G;
      const uint32_t ja = nbrB[(size_t)min(ka, nB - 1) * stride + i], jb = nbrB[(size_t)min(kb, nB - 1) * stride + i];
      const auto va = load(ja), vb = load(jb);
      decltype(term(va, ja, u)) ta{}, tb{};
      if (ka < nB) ta = term(va, ja, u);
      if (kb < nB) tb = term(vb, jb, u);
      acc(quad_bcast<0>(ta), 0u);
      if (k0 + 1 < nB) acc(quad_bcast<1>(ta), 1u % G);
      if (k0 + 2 < nB) acc(quad_bcast<2>(ta), 2u % G);
      if (k0 + 3 < nB) acc(quad_bcast<3>(ta), 3u % G);
      if (k0 + 4 < nB) acc(quad_bcast<0>(tb), 0u);
      if (k0 + 5 < nB) acc(quad_bcast<1>(tb), 1u % G);
      if (k0 + 6 < nB) acc(quad_bcast<2>(tb), 2u % G);
      if (k0 + 7 < nB) acc(quad_bcast<3>(tb), 3u % G);
    }
  }
}

// Halo slot records in LDS: the fields a pass gathers per neighbour,
// interleaved so one slot is one or two 16-byte reads.
struct Slot6 {
  float4 a;
  float2 b;
};
struct Slot8 {
  float4 a, b;
};

// Same visit order without unrolling, for the global-memory fallback (a halo
// beyond the LDS capacity): keeps the rare path out of the unrolled hot loop.
// With four lanes per particle, lane l takes the slots it takes from LDS.
template <int L = 1, class Body>
__device__ inline void for_fluid_slots_rolled(const uint4* __restrict__ nbr8, size_t stride, uint32_t i,
                                              uint32_t nF, Body&& body, int l = 0) {
  if constexpr (L == 1) {
#pragma unroll 1
    for (uint32_t k = 0; k < nF; ++k) {
      const uint4 v = nbr8[(size_t)(k >> 3) * stride + i];
      body(pack_get(v, (int)(k & 7u)));
    }
  } else {
    constexpr uint32_t W = PACK / L;  // slots of a pack that a lane takes
#pragma unroll 1
    for (uint32_t m = 0;; ++m) {
      const uint32_t k = (m / W) * PACK + W * (uint32_t)l + m % W;
      if ((m / W) * PACK >= nF) break;
      if (k >= nF) continue;
      const uint4 v = nbr8[(size_t)(k >> 3) * stride + i];
      body(pack_get(v, (int)(k & 7u)));
    }
  }
}

}  // namespace dfr
