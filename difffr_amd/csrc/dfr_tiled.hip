// Brick-tiled neighbour build and gather passes.
//
// A workgroup owns one brick of 4x4x4 cells.  After the counting sort the
// brick's particles are contiguous, and every neighbour of them lies in the
// brick's 6x6x6-cell halo.  The workgroup stages the halo's particle data in
// LDS with coalesced loads (cell ranges are contiguous), so the per-neighbour
// gathers of all passes read LDS instead of L2.  Fluid neighbour lists store
// 16-bit slots into the halo ("tile slots"; slot order = halo cells in
// (z, y, x) order, particles of a cell in sorted order), eight slots per
// 16-byte pack, packs stored pack-major (nbr8[p * N + i]) so that a wavefront
// reads and writes 1 KB per instruction.  Boundary neighbours keep 32-bit
// sample indices.
//
// A halo larger than the LDS capacity is served from global memory through the
// same slot -> particle mapping (binary search over the halo cell offsets).
#include "dfr_tile.h"

namespace dfr {

// ---------------------------------------------------------------------------
// Neighbour build (CompactNSearch::find_neighbors replacement).
// ---------------------------------------------------------------------------
constexpr int BB = PASS_BLOCK;  // build workgroup: one particle of the brick per thread

// Fluid neighbour slots of one particle as they are found: a 16-entry ring per
// thread in LDS (entry e of thread t at ring[e * BB + t], so a wavefront's
// writes are consecutive), one 16-bit write per candidate.  Eight pending slots
// leave as one pack of the pack-major list; packing costs as much as testing
// eight candidates, so the lanes of a wavefront store together, when some
// lane's ring might not take another chunk of four (in nearly every chunk some
// lane reaches eight).
constexpr int RING = 16;
struct PackWriter {
  uint16_t* ring;  // this block's ring
  int t;
  uint32_t n = 0;   // slots accepted
  uint32_t np = 0;  // packs written
  __device__ inline void push(uint32_t s) {
    ring[(n & (RING - 1)) * BB + t] = (uint16_t)s;
    ++n;
  }
  // Branch-free push: the slot is written at the next free entry either way
  // (an entry past the accepted ones, which the next push overwrites; at most
  // RING - 4 are pending before a chunk, so it never holds one) and counted if
  // d2 < h2 (compare and add with carry).
  __device__ inline void push_if(uint32_t s, float h2, float d2) {
    ring[(n & (RING - 1)) * BB + t] = (uint16_t)s;
    asm("v_cmp_gt_f32 vcc, %1, %2\n\tv_addc_co_u32 %0, vcc, 0, %0, vcc" : "+v"(n) : "s"(h2), "v"(d2) : "vcc");
  }
  __device__ inline void store(uint4* __restrict__ nbr8, size_t stride, uint32_t i, uint32_t count) {
    uint32_t w[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t e0 = np * PACK + 2 * k, e1 = e0 + 1;
      const uint32_t lo = (2 * k < (int)count) ? ring[(e0 & (RING - 1)) * BB + t] : 0u;
      const uint32_t hi = (2 * k + 1 < (int)count) ? ring[(e1 & (RING - 1)) * BB + t] : 0u;
      w[k] = lo | (hi << 16);
    }
    if (np < (uint32_t)NPACK) nbr8[(size_t)np * stride + i] = make_uint4(w[0], w[1], w[2], w[3]);
    ++np;
  }
  __device__ inline void flush_full(uint4* __restrict__ nbr8, size_t stride, uint32_t i) {
    if (n - np * PACK >= (uint32_t)PACK) store(nbr8, stride, i, PACK);
  }
  // after a chunk of up to four pushes: keeps room for the next one
  __device__ inline void flush_chunk(uint4* __restrict__ nbr8, size_t stride, uint32_t i) {
    if (__any(n - np * PACK > (uint32_t)(RING - 4))) flush_full(nbr8, stride, i);
  }
  __device__ inline uint32_t finish(uint4* __restrict__ nbr8, size_t stride, uint32_t i) {
    flush_full(nbr8, stride, i);  // at most RING - 4 pending: fewer than a pack are left
    const uint32_t rest = n - np * PACK;
    if (rest > 0u) store(nbr8, stride, i, rest);
    return n;
  }
};

// Bound by vector issue: 270 candidates a particle at rest density, walked as
// nine rows by each lane, so a wavefront takes the longest row of its cells
// nine times (1.6 times the mean in a packing with 8 to 27 particles a cell).
// 13 instructions a candidate with whole chunks free of the row-end test and the
// lanes storing together; 16, with a store in nearly every chunk, took 247 us
// at 1M, this form 225 (483k: 144 and 132).  One cell a wavefront with the
// candidates in the lanes and ballots for the lists: 379 us (the scalar work
// per round of 64 outweighs the balanced lanes).
//
// Dynamic LDS: x, y, z of the halo in three arrays of a fixed stride, so one
// address serves a chunk of four candidates (immediate offsets); a chunk reads
// up to three slots past its row's end, which stay inside the arrays because
// a halo is staged only if it has at most BSTRIDE - 4 slots (three workgroups
// of 640 threads still fit a CU's LDS).
constexpr int BSTRIDE = 2304;
__global__ void __launch_bounds__(BB)
k_build_tiled(const float4* __restrict__ pos, int nf, GridDesc g, const uint32_t* __restrict__ fstart,
              const float4* __restrict__ bpos, const uint32_t* __restrict__ bstart,
              const uint32_t* __restrict__ bperm, float h2, int maxb, int cap, uint4* __restrict__ nbr8,
              uint32_t* __restrict__ nbrB, uint32_t* __restrict__ cnt, uint32_t* __restrict__ overflow,
              uint4* __restrict__ thdr, uint32_t* __restrict__ tmap) {
  __shared__ TileHdr<BB> T;
  __shared__ uint32_t bcs[HALO], bcn[HALO];  // boundary sample range of each halo cell
  __shared__ uint16_t ring[RING * BB];
  extern __shared__ float lds[];
  const uint32_t brick = xcd_block();
  if (brick_empty(fstart, brick)) {
    if (threadIdx.x == 0) thdr[brick] = make_uint4(0u, 0u, 0u, 0u);
    return;
  }
  tile_setup<BB>(g, fstart, brick, T);
  if (threadIdx.x == 0) thdr[brick] = make_uint4(T.own_begin, T.own_end, T.total, 0u);
  if (T.own_begin == T.own_end) return;
  const uint32_t total = T.total;
  const int t = threadIdx.x;
  if (t == 0) atomicMax(&overflow[3], total);
  if (total > 65535u) {
    // tile slots are 16-bit: leave empty lists (safe for every pass) and report
    for (uint32_t i = T.own_begin + t; i < T.own_end; i += BB) cnt[i] = 0u;
    if (t == 0) atomicMax(&overflow[0], total);
    return;
  }
  if (t < HALO) {
    const int cx = 4 * T.bx - 1 + t % 6, cy = 4 * T.by - 1 + (t / 6) % 6, cz = 4 * T.bz - 1 + t / 36;
    uint32_t st = 0, n = 0;
    if (cx >= 0 && cy >= 0 && cz >= 0 && cx < g.n[0] && cy < g.n[1] && cz < g.n[2]) {
      const uint32_t key = cell_key(g, cx, cy, cz);
      st = bstart[key];
      n = bstart[key + 1] - st;
    }
    bcs[t] = st;
    bcn[t] = n;
  }
  const bool in_lds = total <= (uint32_t)min(cap, BSTRIDE - 4);
  float* lx = lds; float* ly = lds + BSTRIDE; float* lz = lds + 2 * BSTRIDE;
  // the halo's slot -> particle map, for every slot a pass could stage
  constexpr int PTB = per_thread<BB>();
  uint32_t js[PTB];
  {
    const uint32_t mapped = min(total, (uint32_t)TILE_CAP);
    tile_indices<BB>(T, mapped, js);
#pragma unroll
    for (int r = 0; r < PTB; ++r) {
      const uint32_t s = t + r * BB;
      if (s < mapped) tmap[(size_t)brick * TILE_CAP + s] = js[r];
    }
  }
  if (in_lds) {
    float4 q[PTB];
#pragma unroll
    for (int r = 0; r < PTB; ++r)
      if (t + r * BB < (int)total) q[r] = pos[js[r]];
#pragma unroll
    for (int r = 0; r < PTB; ++r) {
      const uint32_t s = t + r * BB;
      if (s < total) { lx[s] = q[r].x; ly[s] = q[r].y; lz[s] = q[r].z; }
    }
  }
  __syncthreads();
  const size_t stride = (size_t)nf;
  for (uint32_t i = T.own_begin + t; i < T.own_end; i += BB) {
    const float4 p = pos[i];
    int cx, cy, cz;
    cell_coords(g, p.x, p.y, p.z, cx, cy, cz);
    const int hc0 = halo_cell<BB>(T, cx, cy, cz, 0, 0, 0);
    const uint32_t self = T.coff[hc0] + (i - T.cstart[hc0]);
    PackWriter pw{ring, t};
    // the three x-neighbour cells of a (dz, dy) row are consecutive halo
    // cells, so their candidates form one contiguous slot range; the centre
    // row goes as the two ranges either side of the particle's own slot
    // (ranges 4 and 5), which keeps the candidate order and needs no
    // per-candidate self test
    for (int row = 0; row < 10; ++row) {
      const int rr = row < 5 ? row : row - 1;
      const int dz = rr / 3 - 1, dy = rr % 3 - 1;
      const int hm = halo_cell<BB>(T, cx, cy, cz, -1, dy, dz);
      uint32_t r0 = T.coff[hm], r1 = T.coff[hm + 3];
      if (row == 4) r1 = self;
      if (row == 5) r0 = self + 1;
      if (in_lds) {
        uint32_t s0 = r0;
        auto chunk = [&](bool tail) {
          float qx[4], qy[4], qz[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const uint32_t s = s0 + u;  // <= r1 + 2 <= total + 2 < BSTRIDE
            qx[u] = lx[s]; qy[u] = ly[s]; qz[u] = lz[s];
          }
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const uint32_t s = s0 + u;
            float d2 = dist2_exact(p.x, p.y, p.z, qx[u], qy[u], qz[u]);
            if (tail && u > 0 && s >= r1) d2 = h2;  // past the row's end
            pw.push_if(s, h2, d2);
          }
          pw.flush_chunk(nbr8, stride, i);
        };
        // whole chunks need no test for the row's end
        for (; s0 + 4u <= r1; s0 += 4) chunk(false);
        if (s0 < r1) chunk(true);
      } else {
        for (uint32_t s = r0; s < r1; ++s) {
          const float4 q = pos[tile_global<BB>(T, s)];
          if (dist2_exact(p.x, p.y, p.z, q.x, q.y, q.z) < h2) pw.push(s);
          pw.flush_full(nbr8, stride, i);
        }
      }
    }
    uint32_t nF = pw.finish(nbr8, stride, i);
    uint32_t nB = 0;
    for (int dz = -1; dz <= 1; ++dz)
      for (int dy = -1; dy <= 1; ++dy)
        for (int dx = -1; dx <= 1; ++dx) {
          const int hc = halo_cell<BB>(T, cx, cy, cz, dx, dy, dz);
          const uint32_t n = bcn[hc];
          if (n == 0) continue;
          const uint32_t st = bcs[hc];
          // four samples at a time: their indices, then their positions, then the tests in order
          for (uint32_t k0 = 0; k0 < n; k0 += 4) {
            uint32_t jj[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) jj[u] = bperm[st + min(k0 + u, n - 1)];
            float4 q[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) q[u] = bpos[jj[u]];
#pragma unroll
            for (int u = 0; u < 4; ++u)
              if (k0 + u < n && dist2_exact(p.x, p.y, p.z, q[u].x, q[u].y, q[u].z) < h2) {
                if (nB < (uint32_t)maxb) nbrB[(size_t)nB * stride + i] = jj[u];
                ++nB;
              }
          }
        }
    if (nF > (uint32_t)MAXF) { atomicMax(&overflow[0], nF); nF = MAXF; }
    if (nB > (uint32_t)maxb) { atomicMax(&overflow[2], nB); nB = maxb; }
    cnt[i] = nF | (nB << 16);
  }
}

// ---------------------------------------------------------------------------
// The same lists for scenes of a few bricks, where the build costs one
// wavefront's chain.  A wavefront takes up to eight particles of one cell: the
// particles share their candidates (nine rows of three halo cells, about 270 at
// rest density), so the lanes hold the candidates, 64 a round, and the
// particles are tested one after the other against a whole round; the accept
// mask is a ballot, a slot's place in the list its rank in the mask, and the
// particle itself drops out by its slot.  2^cell_parts_log2 workgroups share a
// brick, each with the whole halo and its share of the 64 cells.
// Against k_build_tiled, us: 1,000 particles 15 (45), 8,000 22 (44), 28,000 35
// (48), 56,000 53 (61); from 98,000 (79 against 72) the scalar work per round
// costs more than the short chains give.
// ---------------------------------------------------------------------------
constexpr int CNR = 6;             // rounds of 64 candidates kept in registers
constexpr int CP = 8;              // particles a wavefront takes at a time
constexpr int BW = BB / 64;
__device__ inline uint32_t rfl(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }
__device__ inline uint32_t rdl(uint32_t v, int lane) { return (uint32_t)__builtin_amdgcn_readlane((int)v, lane); }
__device__ inline float rdl(float v, int lane) { return __uint_as_float(rdl(__float_as_uint(v), lane)); }
// rank of this lane among the set bits of a wave mask, plus base
__device__ inline uint32_t mask_rank(unsigned long long m, uint32_t base) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, base));
}

__global__ void __launch_bounds__(BB)
k_build_cells(const float4* __restrict__ pos, int nf, GridDesc g, const uint32_t* __restrict__ fstart,
              const float4* __restrict__ bpos, const uint32_t* __restrict__ bstart,
              const uint32_t* __restrict__ bperm, float h2, int maxb, int cap, int cell_parts_log2,
              uint4* __restrict__ nbr8, uint32_t* __restrict__ nbrB, uint32_t* __restrict__ cnt,
              uint32_t* __restrict__ overflow, uint4* __restrict__ thdr, uint32_t* __restrict__ tmap) {
  __shared__ TileHdr<BB> T;
  __shared__ uint32_t bcs[HALO], bcn[HALO];  // boundary sample range of each halo cell
  __shared__ uint32_t bpre[BW][28];          // boundary candidates before each of a cell's 27 neighbour cells
  __shared__ __attribute__((aligned(16))) uint16_t list[BW][CP][MAXF];
  __shared__ uint32_t next_item;
  extern __shared__ float lds[];
  const uint32_t blk = xcd_block();
  const uint32_t brick = blk >> cell_parts_log2, part = blk & ((1u << cell_parts_log2) - 1u);
  if (brick_empty(fstart, brick)) {
    if (threadIdx.x == 0 && part == 0u) thdr[brick] = make_uint4(0u, 0u, 0u, 0u);
    return;
  }
  tile_setup<BB>(g, fstart, brick, T);
  if (threadIdx.x == 0 && part == 0u) thdr[brick] = make_uint4(T.own_begin, T.own_end, T.total, 0u);
  const uint32_t total = T.total;
  const int t = threadIdx.x;
  if (t == 0 && part == 0u) atomicMax(&overflow[3], total);
  if (total > 65535u) {
    // tile slots are 16-bit: leave empty lists (safe for every pass) and report
    if (part == 0u)
      for (uint32_t i = T.own_begin + t; i < T.own_end; i += BB) cnt[i] = 0u;
    if (t == 0) atomicMax(&overflow[0], total);
    return;
  }
  if (t < HALO) {
    const int cx = 4 * T.bx - 1 + t % 6, cy = 4 * T.by - 1 + (t / 6) % 6, cz = 4 * T.bz - 1 + t / 36;
    uint32_t st = 0, n = 0;
    if (cx >= 0 && cy >= 0 && cz >= 0 && cx < g.n[0] && cy < g.n[1] && cz < g.n[2]) {
      const uint32_t key = cell_key(g, cx, cy, cz);
      st = bstart[key];
      n = bstart[key + 1] - st;
    }
    bcs[t] = st;
    bcn[t] = n;
  }
  // items: four per cell, item m of a cell takes its particles 8 m.. + 8 (and every 32nd from there)
  const uint32_t item_end = (part + 1u) * (256u >> cell_parts_log2);
  if (t == 0) next_item = part * (256u >> cell_parts_log2);
  const bool in_lds = total <= (uint32_t)min(cap, BSTRIDE - 4);
  float* lx = lds; float* ly = lds + BSTRIDE; float* lz = lds + 2 * BSTRIDE;
  constexpr int PTB = per_thread<BB>();
  uint32_t js[PTB];
  tile_indices<BB>(T, min(total, (uint32_t)TILE_CAP), js);
#pragma unroll
  for (int r = 0; r < PTB; ++r) {
    const uint32_t s = t + r * BB;
    if (part == 0u && s < min(total, (uint32_t)TILE_CAP)) tmap[(size_t)brick * TILE_CAP + s] = js[r];
  }
  if (in_lds) {
    float4 q[PTB];
#pragma unroll
    for (int r = 0; r < PTB; ++r)
      if (t + r * BB < (int)total) q[r] = pos[js[r]];
#pragma unroll
    for (int r = 0; r < PTB; ++r) {
      const uint32_t s = t + r * BB;
      if (s < total) { lx[s] = q[r].x; ly[s] = q[r].y; lz[s] = q[r].z; }
    }
  }
  __syncthreads();
  const size_t stride = (size_t)nf;
  const int lane = t & 63;
  const int wv = (int)rfl((uint32_t)t >> 6);
  while (true) {
    uint32_t item = 0;
    if (lane == 0) item = atomicAdd(&next_item, 1u);
    item = rfl(item);
    if (item >= item_end) break;
    const uint32_t cell = item >> 2;
    // cell coordinates in the brick from its Morton number
    const int x = (int)((cell & 1u) | ((cell >> 2) & 2u)), y = (int)(((cell >> 1) & 1u) | ((cell >> 3) & 2u)),
              z = (int)(((cell >> 2) & 1u) | ((cell >> 4) & 2u));
    const int hc0 = (z + 1) * 36 + (y + 1) * 6 + (x + 1);
    const uint32_t self0 = rfl(T.coff[hc0]);
    const uint32_t own = rfl(T.coff[hc0 + 1]) - self0;
    if ((item & 3u) * CP >= own) continue;
    const uint32_t i0 = rfl(T.cstart[hc0]);
    // candidate t of row r is slot t + off[r]; the row starts at candidate pre[r]
    uint32_t off[9], pre[9], ncand = 0;
    {
      const int rr = min(lane, 8);
      const int hm = hc0 + (rr / 3 - 1) * 36 + (rr % 3 - 1) * 6 - 1;
      const uint32_t v0 = T.coff[hm], v1 = T.coff[hm + 3];
#pragma unroll
      for (int r = 0; r < 9; ++r) {
        const uint32_t r0 = rdl(v0, r);
        pre[r] = ncand;
        off[r] = r0 - ncand;
        ncand += rdl(v1, r) - r0;
      }
    }
    // boundary candidates of the 27 cells
    uint32_t nbc = 0;
    {
      uint32_t n = 0;
      if (lane < 27) n = bcn[hc0 + (lane / 9 - 1) * 36 + ((lane / 3) % 3 - 1) * 6 + (lane % 3 - 1)];
      if (__ballot(n > 0u) != 0ull) {
        uint32_t inc = n;
#pragma unroll
        for (int o = 1; o < 32; o <<= 1) {
          const uint32_t u = __shfl_up(inc, o, 64);
          if (lane >= o) inc += u;
        }
        if (lane < 27) bpre[wv][lane] = inc - n;
        nbc = rdl(inc, 26);
        __threadfence_block();
        __builtin_amdgcn_wave_barrier();
      }
    }
    float qx[CNR], qy[CNR], qz[CNR];
    uint32_t sl[CNR];
    bool loaded = false;
    for (uint32_t b0 = (item & 3u) * CP; b0 < own; b0 += 4 * CP) {
      const uint32_t nk = min(own - b0, (uint32_t)CP);
      // lanes 0..7 hold the particles
      float px = 0.f, py = 0.f, pz = 0.f;
      if ((uint32_t)lane < nk) {
        const float4 p = pos[i0 + b0 + lane];
        px = p.x; py = p.y; pz = p.z;
      }
      uint32_t myF = 0, myB = 0;  // counts of particle b0 + lane / 8
      for (uint32_t g0 = 0; g0 < ncand; g0 += CNR * 64) {
        if (!loaded) {
#pragma unroll
          for (int r = 0; r < CNR; ++r) {
            const uint32_t tc = g0 + r * 64 + lane;
            uint32_t o = off[0];
#pragma unroll
            for (int w = 1; w < 9; ++w) o = tc >= pre[w] ? off[w] : o;
            const uint32_t s = tc + o;
            sl[r] = s;
            qx[r] = 1.0e30f; qy[r] = 0.f; qz[r] = 0.f;  // no candidate: never within reach
            if (tc < ncand) {
              if (in_lds) {
                qx[r] = lx[s]; qy[r] = ly[s]; qz[r] = lz[s];
              } else {
                const float4 q = pos[tile_global<BB>(T, s)];
                qx[r] = q.x; qy[r] = q.y; qz[r] = q.z;
              }
            }
          }
          loaded = ncand <= (uint32_t)(CNR * 64);
        }
        for (uint32_t k = 0; k < nk; ++k) {
          const uint32_t ps = self0 + b0 + k;
          const float kx = rdl(px, (int)k), ky = rdl(py, (int)k), kz = rdl(pz, (int)k);
          uint16_t* L = list[wv][k];
          uint32_t n = g0 == 0u ? 0u : rdl(myF, (int)(8u * k));
#pragma unroll
          for (int r = 0; r < CNR; ++r) {
            if (g0 + r * 64u >= ncand) break;
            const bool hit = dist2_exact(kx, ky, kz, qx[r], qy[r], qz[r]) < h2 && sl[r] != ps;
            const unsigned long long m = __ballot(hit);
            const uint32_t at = mask_rank(m, n);
            if (hit && at < (uint32_t)MAXF) L[at] = (uint16_t)sl[r];
            n += (uint32_t)__popcll(m);
          }
          if ((uint32_t)(lane >> 3) == k) myF = n;
        }
      }
      for (uint32_t g0 = 0; g0 < nbc; g0 += 64) {
        const uint32_t tc = g0 + lane;
        uint32_t j = 0;
        float bx = 1.0e30f, by = 0.f, bz = 0.f;
        if (tc < nbc) {
          int lo = 0, hi = 26;  // the cell holding candidate tc
          while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (bpre[wv][mid] <= tc) lo = mid; else hi = mid - 1;
          }
          j = bperm[bcs[hc0 + (lo / 9 - 1) * 36 + ((lo / 3) % 3 - 1) * 6 + (lo % 3 - 1)] + (tc - bpre[wv][lo])];
          const float4 q = bpos[j];
          bx = q.x; by = q.y; bz = q.z;
        }
        for (uint32_t k = 0; k < nk; ++k) {
          const bool hit = dist2_exact(rdl(px, (int)k), rdl(py, (int)k), rdl(pz, (int)k), bx, by, bz) < h2;
          const unsigned long long m = __ballot(hit);
          const uint32_t at = mask_rank(m, rdl(myB, (int)(8u * k)));
          if (hit && at < (uint32_t)maxb) nbrB[(size_t)at * stride + (i0 + b0 + k)] = j;
          if ((uint32_t)(lane >> 3) == k) myB += (uint32_t)__popcll(m);
        }
      }
      // the lists leave: eight lanes per particle, a 16-byte pack each
      __threadfence_block();
      __builtin_amdgcn_wave_barrier();
      const uint32_t k = (uint32_t)lane >> 3;
      if (k < nk) {
        const uint32_t i = i0 + b0 + k;
        const uint32_t nF = min(myF, (uint32_t)MAXF), nB = min(myB, (uint32_t)maxb);
        for (uint32_t p = lane & 7u; p * PACK < nF; p += 8) {
          uint4 v = *reinterpret_cast<const uint4*>(&list[wv][k][p * PACK]);
          const uint32_t left = nF - p * PACK;  // entries past the list's end are slot 0
          auto keep = [&](uint32_t w, uint32_t e) { return left >= e + 2u ? w : (left > e ? w & 0xffffu : 0u); };
          nbr8[(size_t)p * stride + i] = make_uint4(keep(v.x, 0), keep(v.y, 2), keep(v.z, 4), keep(v.w, 6));
        }
        if ((lane & 7) == 0) {
          if (myF > (uint32_t)MAXF) atomicMax(&overflow[0], myF);
          if (myB > (uint32_t)maxb) atomicMax(&overflow[2], myB);
          cnt[i] = nF | (nB << 16);
        }
      }
      __threadfence_block();
      __builtin_amdgcn_wave_barrier();
    }
  }
}

// ---------------------------------------------------------------------------
// Gather passes: PASS_BLOCK threads per brick.  Dynamic LDS per slot:
// x, y, z (+ per-pass fields).
// ---------------------------------------------------------------------------
constexpr int PB = PASS_BLOCK;
constexpr int PT = per_thread<PB>();
// The velocity update stages 4 floats per slot, so LDS would fit four 640-thread
// workgroups but the CU holds at most 32 wavefronts: 512 threads keep four.
// With four lanes per particle a workgroup's 160 particles fill 640 threads.
template <int L> constexpr int velocity_block() { return L == 1 ? 512 : PASS_BLOCK; }

// TimeStep::computeDensities (TimeStep.cpp:147-202) + computeDFSPHFactor
// (TimeStepDiffDFSPH.cpp:883-962) + the first loop of warmstartDivergenceSolve
// (:1720-1732), one pass.
__global__ void __launch_bounds__(PB) __attribute__((amdgpu_waves_per_eu(8, 8)))
k_density_factor_t(PassArgs a, float* __restrict__ rho, float* __restrict__ alpha, float4* __restrict__ s_out,
                   float* __restrict__ badv, float* __restrict__ kappav, int div_warm, int divergence_on,
                   float2* __restrict__ aux) {
  __shared__ TileHdr<PB> T;
  extern __shared__ float4 lds4[];
  const StepConst& c = a.c;
  const int cap = a.cap;
  BrickView B;
  if (!brick_open<PB>(a, T, B)) return;
  const uint32_t total = B.total;
  const bool in_lds = B.in_lds;
  float4* LA = lds4;                                          // x, y, z, vx
  float2* LB = reinterpret_cast<float2*>(lds4 + cap);         // vy, vz
  const int t = threadIdx.x;
  if (in_lds) {
    uint32_t js[PT];
    map_indices<PB>(a.tmap, B.brick, total, js);
    float4 q[PT], v[PT];
#pragma unroll
    for (int r = 0; r < PT; ++r)
      if (t + r * PB < (int)total) {
        q[r] = a.pos[js[r]];
        v[r] = divergence_on ? a.vel[js[r]] : make_float4(0.f, 0.f, 0.f, 0.f);
      }
#pragma unroll
    for (int r = 0; r < PT; ++r) {
      const uint32_t s = t + r * PB;
      if (s < total) {
        LA[s] = make_float4(q[r].x, q[r].y, q[r].z, v[r].x);
        LB[s] = make_float2(v[r].y, v[r].z);
      }
    }
  }
  __syncthreads();
  const size_t stride = (size_t)c.nf;
  for (uint32_t i = B.own_begin + t; i < B.own_end; i += PB) {
    const float4 p = a.pos[i];
    float4 vi = make_float4(0.f, 0.f, 0.f, 0.f);
    if (divergence_on) vi = a.vel[i];
    const uint32_t cc = a.cnt[i];
    const uint32_t nF = cc & 0xffffu, nB = cc >> 16;
    float dens = c.V_f * c.K.w0;
    float sumsq = 0.f, gx = 0.f, gy = 0.f, gz = 0.f, delta = 0.f;
    // sums over fluid neighbours without the common factor V_f (applied once)
    float wsum = 0.f, sq = 0.f, fgx = 0.f, fgy = 0.f, fgz = 0.f, fdelta = 0.f;
    // a slot that is not live contributes W = 0 and gradW = 0 (exact no-ops)
    auto pair = [&](float qx, float qy, float qz, float vx, float vy, float vz, bool live) {
      const float rx = p.x - qx, ry = p.y - qy, rz = p.z - qz;
      const PairKernel kw = cubic_pair(c.K, rx * rx + ry * ry + rz * rz, live);
      const float kc = kw.c;
      wsum += kw.W;
      const float wx = kc * rx, wy = kc * ry, wz = kc * rz;
      sq += wx * wx + wy * wy + wz * wz;
      fgx += wx; fgy += wy; fgz += wz;
      if (divergence_on) fdelta += (vi.x - vx) * wx + (vi.y - vy) * wy + (vi.z - vz) * wz;
    };
    if (in_lds) {
      for_fluid_groups<2>(a.nbr8, stride, i, nF, [&](uint32_t s) { return Slot6{LA[s], LB[s]}; },
                          [&](const Slot6& q, bool live) {
                            pair(q.a.x, q.a.y, q.a.z, q.a.w, q.b.x, q.b.y, live);
                          });
    } else {
      for_fluid_slots_rolled(a.nbr8, stride, i, nF, [&](uint32_t s) {
        const uint32_t j = tile_global<PB>(T, s);
        const float4 q = a.pos[j];
        const float4 v = divergence_on ? a.vel[j] : make_float4(0.f, 0.f, 0.f, 0.f);
        pair(q.x, q.y, q.z, v.x, v.y, v.z, true);
      });
    }
    dens += c.V_f * wsum;
    sumsq = c.V_f * c.V_f * sq;
    gx = c.V_f * fgx; gy = c.V_f * fgy; gz = c.V_f * fgz;
    delta = c.V_f * fdelta;
    float bdens = 0.f;  // boundary part of the density sum (a feature of the learned warm start)
    for_boundary_groups(
        a.nbrB, stride, i, nB,
        [&](uint32_t j) { return Slot8{a.bpos[j], divergence_on ? a.bvel[j] : make_float4(0.f, 0.f, 0.f, 0.f)}; },
        [&](const Slot8& s, uint32_t, uint32_t) {
          const float4 q = s.a, vb = s.b;
          const float rx = p.x - q.x, ry = p.y - q.y, rz = p.z - q.z;
          const PairKernel kw = cubic_pair(c.K, rx * rx + ry * ry + rz * rz);
          dens += q.w * kw.W;
          bdens += q.w * kw.W;
          const float wx = kw.c * rx, wy = kw.c * ry, wz = kw.c * rz;
          gx += q.w * wx; gy += q.w * wy; gz += q.w * wz;
          if (divergence_on) delta += q.w * ((vi.x - vb.x) * wx + (vi.y - vb.y) * wy + (vi.z - vb.z) * wz);
        });
    rho[i] = dens * c.rho0;
    if (aux) aux[i] = make_float2(delta, bdens);
    s_out[i] = make_float4(-gx, -gy, -gz, 0.f);
    sumsq += gx * gx + gy * gy + gz * gz;
    alpha[i] = (sumsq > c.eps) ? -1.f / sumsq : 0.f;
    if (divergence_on) {
      float d = fmaxf(delta, 0.f);
      if (nF + nB < 20u) d = 0.f;
      badv[i] = d;
      if (div_warm) {
        const float invH = 1.f / c.dt;
        kappav[i] = (d > 0.f) ? 0.5f * fmaxf(kappav[i], -0.5f) * invH : 0.f;
      }
    }
  }
}

// Jacobi velocity update shared by the two warm starts and every iteration of
// both solves (TimeStepDiffDFSPH.cpp:1024-1055, :1101-1197, :1753-1784,
// :1826-1902): v_i -= dt sum_j (k_i + k_j) grad_p_ij over fluid pairs with
// |k_i + k_j| > eps; when |k_i| > eps each boundary neighbour b changes v_i by
// -dt k_i grad_p_ib and receives f = -m_i dv / dt (BoundaryModel::addForce,
// BoundaryModel.h:46-58), summed here in FP64 per dynamic body.
// LDS per slot: x, y, z, k.
template <int L, int VB>
__global__ void __launch_bounds__(VB) __attribute__((amdgpu_waves_per_eu(8, 8)))
k_velocity_update_t(PassArgs a, const float* __restrict__ kfield, float* __restrict__ kappa_acc,
                    RigidDev* __restrict__ rig, const int* __restrict__ stop, IterTapeOut tape) {
  constexpr int VT = per_thread<VB>();
  __shared__ TileHdr<VB> T;
  extern __shared__ float4 lds4[];
  const StepConst& c = a.c;
  if (stop && *stop) return;
  BrickView B;
  if (!brick_open<VB>(a, T, B)) return;
  const uint32_t total = B.total;
  const bool in_lds = B.in_lds;
  float4* LS = lds4;  // x, y, z, k
  const int t = threadIdx.x;
  if (in_lds) {
    uint32_t js[VT];
    map_indices<VB>(a.tmap, B.brick, total, js);
    float4 q[VT];
    float kk[VT];
#pragma unroll
    for (int r = 0; r < VT; ++r)
      if (t + r * VB < (int)total) { q[r] = a.pos[js[r]]; kk[r] = kfield[js[r]]; }
#pragma unroll
    for (int r = 0; r < VT; ++r) {
      const uint32_t s = t + r * VB;
      if (s < total) LS[s] = make_float4(q[r].x, q[r].y, q[r].z, kk[r]);
    }
  }
  __syncthreads();
  const size_t stride = (size_t)c.nf;
  const float invH = 1.f / c.dt;
  // The particle loop runs the same number of times on every lane of a wave, so
  // the coupling partials of each round are reduced over the wave at its end
  // (and are not live across the next round's fluid pair loop).
  const int l = t % L;  // lane of the particle
  for (uint32_t base = B.own_begin; base < B.own_end; base += VB / L) {
    const uint32_t i = base + t / L;
    int cb = -1;
    double F0 = 0, F1 = 0, F2 = 0, T0 = 0, T1 = 0, T2 = 0;
    if (i < B.own_end) {
      const float ki = kfield[i];
      const float4 p = a.pos[i];
      float4 vi = a.vel[i];
      if (l == 0) {
        if (kappa_acc) kappa_acc[i] += ki;
        if (tape.v) tape.v[i] = vi;
        if (tape.k) tape.k[i] = ki;
        if (tape.b) tape.b[i] = tape.bsrc[i];
      }
      const uint32_t cc = a.cnt[i];
      const uint32_t nF = cc & 0xffffu, nB = cc >> 16;
      // v_i -= dt (k_i + k_j) grad_p_ij = dt V_f (k_i + k_j) c_ij r_ij; dt V_f applied once
      float ux = 0.f, uy = 0.f, uz = 0.f;
      // pairs with |k_i + k_j| <= eps (and slots that are not live) add s = 0
      auto pair = [&](float qx, float qy, float qz, float kj, bool live) {
        const float kSum = ki + kj;
        const float rx = p.x - qx, ry = p.y - qy, rz = p.z - qz;
        const float s = kSum * cubic_grad_c(c.K, rx * rx + ry * ry + rz * rz, live && fabsf(kSum) > c.eps);
        return Terms<4>{{s, rx, ry, rz}};
      };
      auto add = [&](const Terms<4>& q) {
        ux += q.f[0] * q.f[1]; uy += q.f[0] * q.f[2]; uz += q.f[0] * q.f[3];
      };
      if (in_lds) {
        for_fluid_terms<2, L>(a.nbr8, stride, i, nF, l, [&](uint32_t s) { return LS[s]; },
                              [&](const float4& q, bool live) { return pair(q.x, q.y, q.z, q.w, live); }, add);
      } else if constexpr (L == 1) {
        for_fluid_slots_rolled(a.nbr8, stride, i, nF, [&](uint32_t s) {
          const uint32_t j = tile_global<VB>(T, s);
          const float4 q = a.pos[j];
          add(pair(q.x, q.y, q.z, kfield[j], true));
        });
      } else {
        // each lane reads its own pairs' particles; all four walking the whole list took
        // 31 us for 12 (recompute 32 for 12) at 8,000 particles, 38 for 16 (53 for 20) at 24,000
        auto far = [&](uint32_t s) {
          const uint32_t j = tile_global<VB>(T, s);
          float4 q = a.pos[j];
          q.w = kfield[j];
          return q;
        };
        for_fluid_terms_rolled(a.nbr8, stride, i, nF, l, far,
                               [&](const float4& q, bool live) { return pair(q.x, q.y, q.z, q.w, live); }, add);
      }
      {
        const float dv = c.dt * c.V_f;
        vi.x += dv * ux; vi.y += dv * uy; vi.z += dv * uz;
      }
      if (fabsf(ki) > c.eps) {
        auto load = [&](uint32_t j) { return a.bpos[j]; };
        for_boundary_terms<2, L>(a.nbrB, stride, i, nB, l, load, [&](const float4& q, uint32_t j, uint32_t) {
          const float rx = p.x - q.x, ry = p.y - q.y, rz = p.z - q.z;
          const float sc = cubic_grad_c(c.K, rx * rx + ry * ry + rz * rz);
          const float gpx = -q.w * (sc * rx), gpy = -q.w * (sc * ry), gpz = -q.w * (sc * rz);
          const float am = -c.dt * 1.f * ki;
          const float dvx = am * gpx, dvy = am * gpy, dvz = am * gpz;
          if ((int)j >= a.nb_static) {
            const int body = (int)a.bx0[j].w;
            if (rig[body].dynamic) {
              if (body != cb && cb >= 0) {
                atomicAdd(&rig[cb].F[0], F0); atomicAdd(&rig[cb].F[1], F1); atomicAdd(&rig[cb].F[2], F2);
                atomicAdd(&rig[cb].T[0], T0); atomicAdd(&rig[cb].T[1], T1); atomicAdd(&rig[cb].T[2], T2);
                F0 = F1 = F2 = T0 = T1 = T2 = 0.0;
              }
              cb = body;
              const float fx = -c.m_f * dvx * invH, fy = -c.m_f * dvy * invH, fz = -c.m_f * dvz * invH;
              const double rxd = (double)q.x - rig[body].x[0], ryd = (double)q.y - rig[body].x[1],
                           rzd = (double)q.z - rig[body].x[2];
              F0 += fx; F1 += fy; F2 += fz;
              T0 += ryd * fz - rzd * fy; T1 += rzd * fx - rxd * fz; T2 += rxd * fy - ryd * fx;
            }
          }
          return Terms<3>{{gpx, gpy, gpz}};
        }, [&](const Terms<3>& q, uint32_t u) {
          const float am = -c.dt * 1.f * ki;
          if (u == 0u) {
#pragma clang fp contract(off)
            const float dx = am * q.f[0], dy = am * q.f[1], dz = am * q.f[2];
            vi.x += dx; vi.y += dy; vi.z += dz;
          } else {
            vi.x = fmaf(am, q.f[0], vi.x); vi.y = fmaf(am, q.f[1], vi.y); vi.z = fmaf(am, q.f[2], vi.z);
          }
        });
      }
      if (l == 0) a.vel[i] = vi;
    }
    // Wave-level FP64 reduction of the round's coupling partials, one body at a time.
    while (true) {
      const unsigned long long m = __ballot(cb >= 0);
      if (m == 0ull) break;
      const int src = __ffsll((long long)m) - 1;
      const int b0 = __shfl(cb, src, 64);
      const bool mine = (cb == b0);
      const double a0 = wave_sum_d(mine ? F0 : 0.0), a1 = wave_sum_d(mine ? F1 : 0.0),
                   a2 = wave_sum_d(mine ? F2 : 0.0);
      const double a3 = wave_sum_d(mine ? T0 : 0.0), a4 = wave_sum_d(mine ? T1 : 0.0),
                   a5 = wave_sum_d(mine ? T2 : 0.0);
      if ((threadIdx.x & 63) == 0) {
        atomicAdd(&rig[b0].F[0], a0); atomicAdd(&rig[b0].F[1], a1); atomicAdd(&rig[b0].F[2], a2);
        atomicAdd(&rig[b0].T[0], a3); atomicAdd(&rig[b0].T[1], a4); atomicAdd(&rig[b0].T[2], a5);
      }
      if (mine) cb = -1;
    }
  }
}

// TimeStepDiffDFSPH::computeDensityChange (:1977-2041) or computeDensityAdv
// (:1926-1975) for every particle, followed by the residual sum of
// divergenceSolveIteration / pressureSolveIteration (:1906-1916, :1203-1213)
// and k_i = b_i alpha_i kcoef for the next Jacobi update (mode 0 divergence,
// 1 pressure); mode 2 is the first loop of warmstartPressureSolve (:987-999).
// LDS per slot: x, y, z, vx, vy, vz.
template <int L>
__global__ void __launch_bounds__(PB) __attribute__((amdgpu_waves_per_eu(6, 8)))
k_recompute_t(PassArgs a, int mode, float kcoef, const float* __restrict__ rho, const float* __restrict__ alpha,
              float* __restrict__ badv, float* __restrict__ kf, float* __restrict__ kappa, double* __restrict__ err,
              const float* __restrict__ kpred, const int* __restrict__ stop) {
  __shared__ TileHdr<PB> T;
  extern __shared__ float4 lds4[];
  const StepConst& c = a.c;
  if (stop && *stop) return;
  const int cap = a.cap;
  const bool residual = err && (mode == RECOMPUTE_DIV || mode == RECOMPUTE_PRESSURE);
  BrickView B;
  if (!brick_open<PB>(a, T, B)) {
    if (residual && threadIdx.x == 0) err[B.block] = 0.0;
    return;
  }
  const uint32_t total = B.total;
  const bool in_lds = B.in_lds;
  float4* LA = lds4;                                          // x, y, z, vx
  float2* LB = reinterpret_cast<float2*>(lds4 + cap);         // vy, vz
  const int t = threadIdx.x;
  if (in_lds) {
    uint32_t js[PT];
    map_indices<PB>(a.tmap, B.brick, total, js);
    float4 q[PT], v[PT];
#pragma unroll
    for (int r = 0; r < PT; ++r)
      if (t + r * PB < (int)total) { q[r] = a.pos[js[r]]; v[r] = a.vel[js[r]]; }
#pragma unroll
    for (int r = 0; r < PT; ++r) {
      const uint32_t s = t + r * PB;
      if (s < total) {
        LA[s] = make_float4(q[r].x, q[r].y, q[r].z, v[r].x);
        LB[s] = make_float2(v[r].y, v[r].z);
      }
    }
  }
  __syncthreads();
  const size_t stride = (size_t)c.nf;
  double e = 0.0;
  const int l = t % L;  // lane of the particle
  for (uint32_t i = B.own_begin + t / L; i < B.own_end; i += PB / L) {
    const float4 p = a.pos[i];
    const float4 vi = a.vel[i];
    const uint32_t cc = a.cnt[i];
    const uint32_t nF = cc & 0xffffu, nB = cc >> 16;
    float delta = 0.f;
    float fdelta = 0.f;  // fluid part without the common factor V_f
    auto pair = [&](float qx, float qy, float qz, float vx, float vy, float vz, bool live) {
      const float rx = p.x - qx, ry = p.y - qy, rz = p.z - qz;
      const float sc = cubic_grad_c(c.K, rx * rx + ry * ry + rz * rz, live);
      return Terms<2>{{sc, (vi.x - vx) * rx + (vi.y - vy) * ry + (vi.z - vz) * rz}};
    };
    auto add = [&](const Terms<2>& q) { fdelta += q.f[0] * q.f[1]; };
    if (in_lds) {
      for_fluid_terms<4, L>(a.nbr8, stride, i, nF, l, [&](uint32_t s) { return Slot6{LA[s], LB[s]}; },
                            [&](const Slot6& q, bool live) {
                              return pair(q.a.x, q.a.y, q.a.z, q.a.w, q.b.x, q.b.y, live);
                            }, add);
    } else if constexpr (L == 1) {
      for_fluid_slots_rolled(a.nbr8, stride, i, nF, [&](uint32_t s) {
        const uint32_t j = tile_global<PB>(T, s);
        const float4 q = a.pos[j];
        const float4 v = a.vel[j];
        add(pair(q.x, q.y, q.z, v.x, v.y, v.z, true));
      });
    } else {
      auto far = [&](uint32_t s) {
        const uint32_t j = tile_global<PB>(T, s);
        const float4 q = a.pos[j], v = a.vel[j];
        return Slot6{make_float4(q.x, q.y, q.z, v.x), make_float2(v.y, v.z)};
      };
      for_fluid_terms_rolled(a.nbr8, stride, i, nF, l, far, [&](const Slot6& q, bool live) {
        return pair(q.a.x, q.a.y, q.a.z, q.a.w, q.b.x, q.b.y, live);
      }, add);
    }
    delta = c.V_f * fdelta;
    for_boundary_terms<4, L>(a.nbrB, stride, i, nB, l, [&](uint32_t j) { return Slot8{a.bpos[j], a.bvel[j]}; },
                             [&](const Slot8& s, uint32_t, uint32_t u) {
                               const float4 q = s.a, vb = s.b;
                               const float rx = p.x - q.x, ry = p.y - q.y, rz = p.z - q.z;
                               const float sc = cubic_grad_c(c.K, place_dot(u, rx, ry, rz, rx, ry, rz));
                               return Terms<2>{{q.w * sc, place_dot(u, vi.x - vb.x, vi.y - vb.y, vi.z - vb.z,
                                                                       rx, ry, rz)}};
                             }, [&](const Terms<2>& q, uint32_t) { delta += q.f[0] * q.f[1]; });
    if (l != 0) continue;
    float b;
    if (mode == 0) {
      b = fmaxf(delta, 0.f);
      if (nF + nB < 20u) b = 0.f;
      kf[i] = b * alpha[i] * kcoef;
      e += (double)(c.rho0 * b);
    } else {
      b = fmaxf(rho[i] / c.rho0 + c.dt * delta, 1.f);
      if (mode == 1) {
        kf[i] = (b - 1.f) * alpha[i] * kcoef;
        e += (double)(c.rho0 * b - c.rho0);
      } else if (mode == PRESSURE_WARMSTART) {
        const float invH2 = 1.f / (c.dt * c.dt);
        kappa[i] = (b > 1.f) ? 0.5f * fmaxf(kappa[i], -0.00025f) * invH2 : 0.f;
      } else {  // learned warm start: the predicted stiffness (stored units)
        const float invH2 = 1.f / (c.dt * c.dt);
        kappa[i] = (b > 1.f) ? kpred[i] * invH2 : 0.f;
      }
    }
    badv[i] = b;
  }
  if (residual) block_sum_double<PB>(e, err + B.block);
}

// Expands tile slots back to sorted fluid indices (diagnostics).
__global__ void __launch_bounds__(BB)
k_expand_lists(GridDesc g, const uint32_t* __restrict__ fstart, int nf, const uint4* __restrict__ nbr8,
               const uint32_t* __restrict__ cnt, uint32_t* __restrict__ out) {
  __shared__ TileHdr<BB> T;
  const uint32_t brick = blockIdx.x;
  tile_setup<BB>(g, fstart, brick, T);
  if (T.own_begin == T.own_end) return;
  const size_t stride = (size_t)nf;
  for (uint32_t i = T.own_begin + threadIdx.x; i < T.own_end; i += BB) {
    const uint32_t nF = cnt[i] & 0xffffu;
    uint32_t k = 0;
    for_fluid_slots(nbr8, stride, i, nF, [&](uint32_t s) { out[(size_t)(k++) * stride + i] = tile_global<BB>(T, s); });
  }
}

// Copies a step's lists to another set of buffers: the rows and map entries in
// use, which is all that a pass reads.  A thread per particle, a workgroup per
// brick for the maps; bound by memory.  Whole buffers hold 128 fluid slots (2 bytes)
// and maxb boundary samples (4) a particle and 2,560 map entries a brick, some 570 MB
// at 1M particles; the entries in use take 40 us there (250,000: 14.5), and a pass of
// four recorded steps with their reverse went from 8454 to 8284 us (six
// checkpointed ones at 250,000: 8167 to 8076).
__global__ void __launch_bounds__(DFR_BLOCK)
k_copy_lists(ListBufs d, ListBufs s, uint32_t n, uint32_t maxb, uint32_t bricks, uint32_t particle_blocks) {
  if (blockIdx.x < particle_blocks) {
    const uint32_t i = blockIdx.x * DFR_BLOCK + threadIdx.x;
    if (i >= n) return;
    const uint32_t cc = s.cnt[i];
    const uint32_t np = ((cc & 0xffffu) + PACK - 1) / PACK, nB = min(cc >> 16, maxb);
    d.cnt[i] = cc;
#pragma unroll
    for (uint32_t p = 0; p < (uint32_t)NPACK; ++p)
      if (p < np) d.nbr8[(size_t)p * n + i] = s.nbr8[(size_t)p * n + i];
    for (uint32_t k = 0; k < nB; ++k) d.nbrB[(size_t)k * n + i] = s.nbrB[(size_t)k * n + i];
    return;
  }
  const uint32_t brick = blockIdx.x - particle_blocks;
  if (brick >= bricks) return;
  const uint4 h = s.thdr[brick];
  if (threadIdx.x == 0) d.thdr[brick] = h;
  const uint32_t m = min(h.z, (uint32_t)TILE_CAP);
  for (uint32_t k = threadIdx.x; k < m; k += DFR_BLOCK)
    d.tmap[(size_t)brick * TILE_CAP + k] = s.tmap[(size_t)brick * TILE_CAP + k];
}

// ---------------------------------------------------------------------------

void launch_build_tiled(FluidBufs& f, BoundaryBufs& b, const GridDesc& g, GridBufs& gb, NbrBufs& nb, float h2,
                        hipStream_t s) {
  const size_t shm = sizeof(float) * 3 * (size_t)BSTRIDE;
  // workgroups per brick of k_build_cells: 2,000 particles 17 us with 8, 21 with 4; 28,000: 41 and 35
  const int cell_parts_log2 = f.n < 16384 ? 3 : 2;
  if (nb.by_cells)
    hipLaunchKernelGGL(k_build_cells, dim3(nbricks(g) << cell_parts_log2), dim3(BB), shm, s, f.pos, f.n, g, gb.fstart,
                       b.pos, gb.bstart, gb.bperm, h2, nb.maxb, nb.cap, cell_parts_log2, nb.nbr8, nb.nbrB, nb.cnt,
                       nb.overflow, nb.thdr, nb.tmap);
  else
    hipLaunchKernelGGL(k_build_tiled, dim3(nbricks(g)), dim3(BB), shm, s, f.pos, f.n, g, gb.fstart, b.pos, gb.bstart,
                       gb.bperm, h2, nb.maxb, nb.cap, nb.nbr8, nb.nbrB, nb.cnt, nb.overflow, nb.thdr, nb.tmap);
}

void launch_density_factor_t(const StepConst& c, const GridDesc& g, GridBufs& gb, FluidBufs& f, BoundaryBufs& b,
                             NbrBufs& nb, int div_warm, int divergence_on, float2* aux, hipStream_t s) {
  const size_t shm = sizeof(float) * (size_t)nb.cap * 6;
  hipLaunchKernelGGL(k_density_factor_t, dim3(nbricks(g)), dim3(PB), shm, s, whole_bricks(make_args(c, g, gb, f, b, nb)),
                     f.rho, f.alpha, f.s, f.badv, f.kappav, div_warm, divergence_on, aux);
}

void launch_velocity_update_t(const StepConst& c, const GridDesc& g, GridBufs& gb, FluidBufs& f, BoundaryBufs& b,
                              NbrBufs& nb, RigidDev* rig, const float* kfield, float* kappa_acc, hipStream_t s,
                              const int* stop, IterTapeOut tape) {
  const size_t shm = sizeof(float) * (size_t)nb.cap * 4;
  const PassArgs a = make_args(c, g, gb, f, b, nb);
  const dim3 grid(pass_grid(g, nb.parts_log2));
  constexpr int V1 = velocity_block<1>(), V4 = velocity_block<4>();
  if (nb.parts_log2 > 0)
    hipLaunchKernelGGL((k_velocity_update_t<4, V4>), grid, dim3(V4), shm, s, a, kfield, kappa_acc, rig, stop, tape);
  else
    hipLaunchKernelGGL((k_velocity_update_t<1, V1>), grid, dim3(V1), shm, s, a, kfield, kappa_acc, rig, stop, tape);
}

void launch_recompute_t(const StepConst& c, const GridDesc& g, GridBufs& gb, FluidBufs& f, BoundaryBufs& b,
                        NbrBufs& nb, int mode, float kcoef, double* err_slot, hipStream_t s, const float* kpred,
                        const int* stop) {
  const size_t shm = sizeof(float) * (size_t)nb.cap * 6;
  hipLaunchKernelGGL(nb.parts_log2 > 0 ? k_recompute_t<4> : k_recompute_t<1>, dim3(pass_grid(g, nb.parts_log2)),
                     dim3(PB), shm, s, make_args(c, g, gb, f, b, nb), mode, kcoef, f.rho, f.alpha, f.badv, f.kf,
                     f.kappa, err_slot, kpred, stop);
}

void launch_expand_lists(const GridDesc& g, GridBufs& gb, FluidBufs& f, NbrBufs& nb, uint32_t* out, hipStream_t s) {
  hipLaunchKernelGGL(k_expand_lists, dim3(nbricks(g)), dim3(BB), 0, s, g, gb.fstart, f.n, nb.nbr8, nb.cnt, out);
}

void launch_copy_lists(const ListBufs& d, const ListBufs& src, int n, int maxb, const GridDesc& g,
                       hipStream_t s) {
  const unsigned pb = (unsigned)((n + DFR_BLOCK - 1) / DFR_BLOCK);
  hipLaunchKernelGGL(k_copy_lists, dim3(pb + nbricks(g)), dim3(DFR_BLOCK), 0, s, d, src, (uint32_t)n,
                     (uint32_t)maxb, nbricks(g), pb);
}

void set_tiled_kernel_attributes() {
  const int shm6 = (int)(sizeof(float) * TILE_CAP * 6), shm4 = (int)(sizeof(float) * TILE_CAP * 4);
  for (const void* k : {(const void*)k_density_factor_t, (const void*)k_recompute_t<1>, (const void*)k_recompute_t<4>})
    (void)hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, shm6);
  for (const void* k : {(const void*)k_velocity_update_t<1, velocity_block<1>()>,
                        (const void*)k_velocity_update_t<4, velocity_block<4>()>})
    (void)hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, shm4);
  for (const void* k : {(const void*)k_build_tiled, (const void*)k_build_cells})
    (void)hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)(sizeof(float) * 3 * BSTRIDE));
}

}  // namespace dfr
