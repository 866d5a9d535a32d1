// Batched per-query preprocessing on gfx950: up to 64 queries per pass.
//
// Replaces, for a whole batch at once, the per-query host BFS and the
// admission kernels of the reference: cal_query_dist (src/Graph.h:111-142),
// initialReductionRules (src/helpers.cc:207-248), CompressTask
// (src/helpers.cc:250-313), the Thrust offset scan (main.cu:208-211) and
// NeighborUpdate (src/helpers.cc:317-368).
//
// Query b of the batch owns bit b of a 64-bit mask per vertex:
//   elig[v]  queries whose BFS may enter v (core[v] > kl0_b).  The host
//            numbers the queries by ascending kl0, so elig[v] is the mask of
//            the first cnt(v) bits: one compare per query, no table.
//   vis[v]   queries whose BFS reached v (= v is kept for them); a level's
//            finds join it when the next level, or ms_count, reads them.
//   fr / nf  queries for which v is in the current / next frontier (three
//            buffers in turn: the third is cleared for the level after).
// Level 0 pushes from the query vertices (top-down).  Every later level is
// bottom-up (pull): every vertex that some active query still wants ORs the
// frontier masks of its neighbours, stopping once it has every bit it
// wants.  No atomics, and the adjacency of a vertex is read once per level
// for all 64 queries.  Kept vertex v of query b gets local id
//   base[g][b] + rank of v among group g's vertices kept by b
// (g = v / 64, ranks by ballot), so local ids ascend with original ids as
// the reference's compaction order does.  The local degree and adjacency
// passes read the adjacency of each kept vertex once for every query of
// the batch that kept it; a 64 x 64 bit transpose of the per-neighbour keep
// masks gives every query its own bits.
//
// Outputs per query b (device pointers in MsQuery): loff[K+1] (exclusive
// scan of local degrees, loff[K] = nnz), ldist[K], lcore[K], lorig[K] and
// ladj[nnz] (local ids, ascending per vertex).
//
// Every kernel adds the bytes its loads and stores name (each element once)
// to a counter: the algorithmic traffic of the batched pass.
#include "scs_internal.h"

#define MS_BITS 64

__device__ __forceinline__ u64 ms_or(u64 x) {
  u32 lo = (u32)x, hi = (u32)(x >> 32);
  for (int o = 32; o > 0; o >>= 1) {
    lo |= __shfl_xor(lo, o);
    hi |= __shfl_xor(hi, o);
  }
  return ((u64)hi << 32) | lo;
}
__device__ __forceinline__ u64 ms_sum(u64 x) {
  u32 lo = (u32)x, hi = (u32)(x >> 32);
  // 64-bit add through two 32-bit halves with carry
  for (int o = 32; o > 0; o >>= 1) {
    const u32 olo = __shfl_xor(lo, o), ohi = __shfl_xor(hi, o);
    const u32 nlo = lo + olo;
    hi = hi + ohi + (nlo < lo ? 1u : 0u);
    lo = nlo;
  }
  return ((u64)hi << 32) | lo;
}
__device__ __forceinline__ u64 ms_shfl64(u64 x, int src) {
  const u32 lo = __shfl((u32)x, src), hi = __shfl((u32)(x >> 32), src);
  return ((u64)hi << 32) | lo;
}
// One add per wave into one of MS_BYTE_SLOTS counters, each on its own
// 128-byte line: adds to a single address serialise at the L2 (about 12 ns
// each), which had made the count, not the work, bound the wide launches.
__device__ __forceinline__ void ms_count_bytes(unsigned long long* ctr, u64 b) {
  b = ms_sum(b);
  const u32 slot = ((blockIdx.x * blockDim.x + threadIdx.x) >> 6) & (MS_BYTE_SLOTS - 1);
  if ((threadIdx.x & 63) == 0 && b) atomicAdd(ctr + slot * MS_BYTE_STRIDE, (unsigned long long)b);
}
__device__ __forceinline__ u64 ms_below() {
  const u32 lane = threadIdx.x & 63;
  return lane ? (~0ull >> (64 - lane)) : 0ull;
}
__device__ __forceinline__ u64 ms_shfl_xor64(u64 x, int m) {
  const u32 lo = __shfl_xor((u32)x, m), hi = __shfl_xor((u32)(x >> 32), m);
  return ((u64)hi << 32) | lo;
}
// 64 x 64 bit transpose across the wave: on entry lane j holds row j, on
// exit lane b holds column b (bit j of lane b = bit b of row j).  Six
// butterfly stages; at stage j the pair (lane, lane ^ j) swaps the j x j
// blocks off the diagonal.
__device__ __forceinline__ u64 ms_transpose(u64 a) {
  const u32 lane = threadIdx.x & 63;
  const u64 M[6] = {0x00000000FFFFFFFFull, 0x0000FFFF0000FFFFull, 0x00FF00FF00FF00FFull,
                    0x0F0F0F0F0F0F0F0Full, 0x3333333333333333ull, 0x5555555555555555ull};
#pragma unroll
  for (int s = 0; s < 6; s++) {
    const int j = 32 >> s;
    const u64 p = ms_shfl_xor64(a, j);
    const u64 up = ((p >> j) ^ a) & M[s];           // lane has bit j set
    const u64 dn = (((a >> j) ^ p) & M[s]) << j;    // lane has bit j clear
    a ^= (lane & (u32)j) ? up : dn;
  }
  return a;
}
// Inclusive sum over the wave's lanes.
__device__ __forceinline__ u32 ms_wave_incl(u32 x) {
  const u32 lane = threadIdx.x & 63;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const u32 y = __shfl_up(x, o);
    if (lane >= (u32)o) x += y;
  }
  return x;
}
__device__ __forceinline__ u64 ms_uniform64(u64 x) {
  // readfirstlane is signed: the low word must not spread its top bit
  return ((u64)(u32)__builtin_amdgcn_readfirstlane((u32)(x >> 32)) << 32) |
         (u32)__builtin_amdgcn_readfirstlane((u32)x);
}
// The wave number as a wave-uniform value.
__device__ __forceinline__ u32 ms_wave_id() {
  return __builtin_amdgcn_readfirstlane((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
}

// elig/vis/fr for every vertex; level flags cleared.
__global__ void __launch_bounds__(256) ms_init(u32 n, const u32* __restrict__ core,
                                               const MsBatch* __restrict__ B,
                                               u64* __restrict__ elig, u64* __restrict__ vis,
                                               u64* __restrict__ fr, u64* __restrict__ nf,
                                               u64* __restrict__ xf, u32* __restrict__ flags,
                                               u32 nflags,
                                               unsigned long long* bytes) {
  const u32 tid = blockIdx.x * blockDim.x + threadIdx.x;
  const u32 nt = gridDim.x * blockDim.x;
  u64 nb = 0;
  for (u32 v = tid; v < n; v += nt) {
    const u32 c = core[v];
    u32 cnt = 0;
    const u32 nbq = B->nb;
    for (u32 b = 0; b < nbq; b++) cnt += B->kl0[b] < c ? 1u : 0u;
    elig[v] = cnt >= 64 ? ~0ull : ((1ull << cnt) - 1ull);
    vis[v] = 0;
    fr[v] = 0;
    nf[v] = 0;
    xf[v] = 0;
    nb += 4 + 40;
  }
  for (u32 i = tid; i < nflags; i += nt) flags[i] = 0;
  ms_count_bytes(bytes, nb);
}

// Query vertices: visited and in the first frontier, distance 0.
__global__ void ms_seed(const MsBatch* __restrict__ B, u64* __restrict__ vis,
                        u64* __restrict__ fr, u16* __restrict__ dist16) {
  const u32 b = threadIdx.x;
  if (b < B->nb) {
    const u32 q = B->q[b];
    atomicOr((unsigned long long*)&vis[q], (unsigned long long)(1ull << b));
    atomicOr((unsigned long long*)&fr[q], (unsigned long long)(1ull << b));
    dist16[(u64)q * MS_BITS + b] = 0;
  }
}

// Level 0, top-down: the frontier is the query vertices themselves, so
// rather than every eligible vertex scanning its adjacency for them (the
// bottom-up form of the later levels), the wave of query b pushes bit b to
// the eligible neighbours of q_b.  The atomicOr on vis decides which wave
// reached a vertex first for a bit, so each (vertex, query) is taken once.
// Sets flags[0] if anything was reached.
__global__ void __launch_bounds__(64) ms_push0(const i64* __restrict__ off,
                                               const int32_t* __restrict__ adj,
                                               const MsBatch* __restrict__ B, u64 act,
                                               const u64* __restrict__ elig, u64* __restrict__ vis,
                                               u64* __restrict__ nf, u16* __restrict__ dist16,
                                               u32* __restrict__ flag0, unsigned long long* bytes) {
  const u32 b = blockIdx.x, lane = threadIdx.x;
  if (!((act >> b) & 1ull)) return;
  const u32 q = B->q[b];
  const u64 bit = 1ull << b;
  const i64 b0 = off[q], e0 = off[q + 1];
  bool found = false;
  u64 nbytes = lane == 0 ? 20 : 0;
  for (i64 j = b0 + lane; j < e0; j += 64) {
    const u32 w = (u32)adj[j];
    nbytes += 12;
    if (elig[w] & bit) {
      const u64 old = atomicOr((unsigned long long*)&vis[w], (unsigned long long)bit);
      if (!(old & bit)) {
        atomicOr((unsigned long long*)&nf[w], (unsigned long long)bit);
        dist16[(u64)w * MS_BITS + b] = 1;
        found = true;
        nbytes += 18;
      }
    }
  }
  if (__ballot(found) && lane == 0) atomicOr(flag0, 1u);
  ms_count_bytes(bytes, nbytes);
}

// One BFS level for every query whose depth bound exceeds `level` (act).
// Runs only if the previous level found something (flag_prev).  A 16-lane
// segment takes one adjacency unit (at most MS_UNIT entries; four units per
// wave) and reads 64 entries per step, stopping once it holds every bit it
// wants.  A hub's units are spread over waves; each ORs what it found into nf,
// which the level two before this one cleared for the hubs.  vis takes in the
// current frontier here (vis | fr is the same whichever unit of a hub wrote
// it), so no unit depends on another's finds of this level.
//
// Bound: the frontier gathers (8 bytes from a 64-byte line each, 16M of them
// on the 500,000-vertex graph), and on hub-heavy graphs the longest wave: with
// whole vertices per segment, and ids dealt out modulo the waves, an R-MAT
// graph's hubs (ids with few bits set) met in one wave, and its second level
// took 424 us where the 500,000-vertex graph's took 255; both take under 120 now (36 and 119).

__device__ __forceinline__ u64 ms_seg_or(u64 x) {
  u32 lo = (u32)x, hi = (u32)(x >> 32);
  for (int o = 8; o > 0; o >>= 1) {
    lo |= __shfl_xor(lo, o, 16);
    hi |= __shfl_xor(hi, o, 16);
  }
  return ((u64)hi << 32) | lo;
}
// The bits of a find to the distance row of v, by the segment's lanes.
__device__ __forceinline__ void ms_seg_dist(u16* __restrict__ dist16, u32 v, u64 acc, u32 level) {
  for (u32 b = threadIdx.x & 15; b < 64; b += 16)
    if ((acc >> b) & 1ull) dist16[(u64)v * MS_BITS + b] = (u16)(level + 1);
}
// Sets the level flag once: later waves read it from the L2 and skip the
// atomic, so the finders do not queue on one address.
__device__ __forceinline__ void ms_set_flag(u32* flag, bool found) {
  if (__ballot(found) && (threadIdx.x & 63) == 0 &&
      __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0)
    atomicOr(flag, 1u);
}

__global__ void __launch_bounds__(256) ms_level(const int32_t* __restrict__ adj,
                                                const MsUnit* __restrict__ units, u32 nunits,
                                                const MsHub* __restrict__ hubs, u32 nhubs,
                                                u32 level, u64 act, const u64* __restrict__ elig,
                                                u64* vis, const u64* fr, u64* nf, u64* clr,
                                                u16* __restrict__ dist16,
                                                const u32* __restrict__ flag_prev,
                                                u32* __restrict__ flag_cur,
                                                unsigned long long* bytes) {
  if (level > 0 && *flag_prev == 0) return;
  const u32 lane = threadIdx.x & 63, seg = lane >> 4, sl = lane & 15;
  const u64 wid = ms_wave_id();
  const u64 nw = ((u64)gridDim.x * blockDim.x) >> 6;
  for (u32 i = blockIdx.x * blockDim.x + threadIdx.x; i < nhubs; i += gridDim.x * blockDim.x)
    clr[hubs[i].u] = 0;
  u64 nbytes = 0;
  bool found = false;
  for (u64 k0 = wid * 4; k0 < nunits; k0 += nw * 4) {
    const bool in = k0 + seg < nunits;
    const MsUnit U = units[in ? k0 + seg : nunits - 1];
    const u32 v = U.u, len = (u32)(U.pos >> 48);
    const i64 b0 = (i64)(U.pos & 0xFFFFFFFFFFFFull);
    const u64 visv = vis[v], frv = fr[v], seen = visv | frv;
    const u64 want = in ? elig[v] & act & ~seen : 0ull;
    if (in && sl == 0) {
      nbytes += 16 + 24;
      if (frv & ~visv) {
        vis[v] = seen;
        nbytes += 8;
      }
    }
    // 64 entries per segment step: each lane issues its four adjacency
    // loads, then its four frontier gathers, so a step costs two memory
    // round trips
    u64 acc = 0;
    u32 j = sl;
    bool active = want != 0 && len != 0;
    while (__ballot(active)) {
      u64 x = 0;
      if (active) {
        u32 w[4];
#pragma unroll
        for (int t = 0; t < 4; t++)
          w[t] = j + 16 * t < len ? (u32)__builtin_nontemporal_load(&adj[b0 + j + 16 * t]) : v;
#pragma unroll
        for (int t = 0; t < 4; t++)
          if (j + 16 * t < len) {
            x |= fr[w[t]];
            nbytes += 12;
          }
        x &= want;
      }
      acc |= ms_seg_or(x);
      j += 64;
      if (active && (acc == want || j - sl >= len)) active = false;
    }
    if (in) {
      if (U.h == MS_NOHUB) {
        if (sl == 0) {
          nf[v] = acc;
          nbytes += 8;
        }
      } else if (acc && sl == 0) {
        atomicOr((unsigned long long*)&nf[v], (unsigned long long)acc);
        nbytes += 8;
      }
      if (acc) {
        found = true;
        ms_seg_dist(dist16, v, acc, level);
        if (sl == 0) nbytes += 2ull * (u32)__popcll(acc);
      }
    }
  }
  ms_set_flag(flag_cur, found);
  ms_count_bytes(bytes, nbytes);
}

// Kept counts.  A wave takes a chunk of `ch` groups of 64 vertices, lane b counting
// for query b: gcnt[g * 64 + b] = query b's kept vertices in the chunk's groups
// before g, cbase[c * 64 + b] = those in chunk c.  vis takes in the last
// level's finds (lf; bits already there when the search ended earlier).  At
// most 256 chunks: enough waves for the count, and few rows for the one wave
// that scans them.
__global__ void __launch_bounds__(256) ms_count(u32 n, u32 G, u32 ch, u64* __restrict__ vis,
                                                const u64* __restrict__ lf, u64 valid,
                                                u32* __restrict__ gcnt, u32* __restrict__ cbase,
                                                unsigned long long* bytes) {
  const u32 lane = threadIdx.x & 63;
  const u32 c = ms_wave_id();
  const u32 g0 = c * ch;
  if (g0 >= G) return;
  const u32 g1 = min(G, g0 + ch);
  u64 nbytes = 0;
  u32 run = 0;
  for (u32 g = g0; g < g1; g += 8) {
    u64 m[8], f[8];
#pragma unroll
    for (int t = 0; t < 8; t++) {
      const u64 v = (u64)(g + t) * 64 + lane;
      const bool in = g + t < g1 && v < n;
      m[t] = in ? vis[v] : 0ull;
      f[t] = in ? lf[v] : 0ull;
    }
#pragma unroll
    for (int t = 0; t < 8; t++) {
      if (g + t >= g1) break;
      const u64 v = (u64)(g + t) * 64 + lane;
      if (f[t] & ~m[t]) vis[v] = m[t] | f[t];
      if (v < n) nbytes += 16;
      gcnt[(u64)(g + t) * 64 + lane] = run;
      run += (u32)__popcll(ms_transpose((m[t] | f[t]) & valid));
      nbytes += 4;
    }
  }
  cbase[(u64)c * 64 + lane] = run;
  ms_count_bytes(bytes, nbytes + 4);
}

// Chunk counts -> exclusive bases in place; K_b -> tot[b].  One wave, lane =
// query, eight coalesced rows in flight.  (One wave per query over the
// group counts, 256 bytes apart per lane, took 62 us on 500,000 vertices;
// counting by chunks first leaves 253 rows.)
__global__ void __launch_bounds__(64) ms_bscan(u32 C, u32* __restrict__ cbase,
                                               u32* __restrict__ tot, unsigned long long* bytes) {
  const u32 b = threadIdx.x;
  u32 run = 0;
  for (u32 c = 0; c < C; c += 8) {
    u32 x[8];
#pragma unroll
    for (int t = 0; t < 8; t++) x[t] = cbase[(u64)min(c + t, C - 1) * 64 + b];
#pragma unroll
    for (int t = 0; t < 8; t++)
      if (c + t < C) {
        cbase[(u64)(c + t) * 64 + b] = run;
        run += x[t];
      }
  }
  tot[b] = run;
  ms_count_bytes(bytes, (u64)C * 8 + 4);
}

// Columns of the local-id rows (locid, one row per vertex): the groups of
// eight queries that the pass takes, packed, so that a batch which leaves few
// queries to it has rows of 8 or 16 entries instead of 64, whose gathers the
// caches can hold (500,000 vertices: 16 MB instead of 128).
struct MsCols {
  u32 rank;    // 4 bits per group of eight queries: its place in a row
  u32 stride;  // entries per row
  __device__ __forceinline__ u32 group(u32 g) const { return ((rank >> (4 * g)) & 15u) * 8; }
  __device__ __forceinline__ u32 col(u32 b) const { return group(b >> 3) + (b & 7); }
};

// Local ids, and per kept vertex: orig id, distance, core number.
__global__ void __launch_bounds__(256) ms_scatter(u32 n, u32 G, u32 ch,
                                                  const u64* __restrict__ vis,
                                                  u64 valid, const u32* __restrict__ gcnt,
                                                  const u32* __restrict__ cbase,
                                                  const u32* __restrict__ core,
                                                  const u16* __restrict__ dist16,
                                                  const MsBatch* __restrict__ B,
                                                  u32* __restrict__ locid, MsCols cols,
                                                  u32* __restrict__ qloc,
                                                  unsigned long long* bytes) {
  const u32 lane = threadIdx.x & 63;
  const u32 wid = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const u32 nw = (gridDim.x * blockDim.x) >> 6;
  const u64 below = ms_below();
  // lane b holds query b's output pointers and vertex; the per-query loop
  // below takes them by shuffles, so its stores wait on no memory load
  const MsQuery Qb = B->P[lane];
  const u32 qb = B->q[lane];
  u64 nbytes = 0;
  for (u32 g = wid; g < G; g += nw) {
    const u64 v = (u64)g * 64 + lane;
    const u64 m = v < n ? vis[v] & valid : 0;
    // lane b: query b's first id in the group
    const u32 gb = gcnt[(u64)g * 64 + lane] + cbase[(u64)(g / ch) * 64 + lane];
    u32 cv = 0;
    if (m) {
      cv = core[v];
      nbytes += 12;
    }
    u64 any = ms_or(m);
    // eight queries at a time: their distance loads are in flight together
    // before the stores that need them
    while (any) {
      int bb[8];
      u32 dv[8];
#pragma unroll
      for (int t = 0; t < 8; t++) {
        bb[t] = any ? __ffsll((unsigned long long)any) - 1 : -1;
        any &= any - 1;  // 0 stays 0
      }
#pragma unroll
      for (int t = 0; t < 8; t++)
        dv[t] = (bb[t] >= 0 && ((m >> bb[t]) & 1ull)) ? (u32)dist16[v * MS_BITS + bb[t]] : 0u;
#pragma unroll
      for (int t = 0; t < 8; t++) {
        const int b = bb[t];
        if (b < 0) break;
        const u64 bal = __ballot((m >> b) & 1ull);
        const u32 base = (u32)__shfl((int)gb, b), qv = (u32)__shfl((int)qb, b);
        u32* const lorig = (u32*)ms_shfl64((u64)Qb.lorig, b);
        u32* const ldist = (u32*)ms_shfl64((u64)Qb.ldist, b);
        u32* const lcore = (u32*)ms_shfl64((u64)Qb.lcore, b);
        if ((m >> b) & 1ull) {
          const u32 id = base + (u32)__popcll(bal & below);
          lorig[id] = (u32)v;
          ldist[id] = dv[t];
          lcore[id] = cv;
          locid[v * cols.stride + cols.col(b)] = id;
          if ((u32)v == qv) qloc[b] = id;
          nbytes += 4 + 2 + 12 + 4;
        }
      }
    }
  }
  ms_count_bytes(bytes, nbytes);
}

// Whole-graph queries (gmask): query b's distance array over every vertex of
// the graph, SCS_DIST_NONE where b does not keep the vertex.  Lane = vertex,
// so each query's 64 values of a group are one coalesced store; a lane reads
// its vertex's row of 64 distances as eight 16-byte loads, all in flight, so a
// row's line is fetched once.  Bound: stores (4 bytes per query and vertex).
// 500,000 vertices, 59 such queries: 41 us; one 2-byte load per query and
// vertex, eight queries at a time, took 102.
__global__ void __launch_bounds__(256) ms_gdist(u32 n, u32 G, const u64* __restrict__ vis,
                                                u64 gmask, const u16* __restrict__ dist16,
                                                const MsBatch* __restrict__ B,
                                                unsigned long long* bytes) {
  const u32 lane = threadIdx.x & 63;
  const u32 wid = ms_wave_id();
  const u32 nw = (gridDim.x * blockDim.x) >> 6;
  const u64 dp = (u64)B->P[lane].ldist;
  u64 nbytes = 0;
  for (u32 g = wid; g < G; g += nw) {
    const u64 v = (u64)g * 64 + lane;
    const bool in = v < n;
    const u64 vv = in ? v : (u64)n - 1;
    const u64 m = in ? vis[vv] & gmask : 0ull;
    uint4 d[8];
#pragma unroll
    for (int t = 0; t < 8; t++)
      if ((gmask >> (8 * t)) & 0xFFull) d[t] = *(const uint4*)&dist16[vv * MS_BITS + 8 * t];
    if (in) nbytes += 8 + 4ull * (u32)__popcll(gmask) + 2ull * (u32)__popcll(m);
#pragma unroll
    for (int t = 0; t < 8; t++) {
      const u32 x[4] = {d[t].x, d[t].y, d[t].z, d[t].w};
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const int b = 8 * t + i;
        if (!((gmask >> b) & 1ull)) continue;
        const u32 dv = (x[i >> 1] >> (16 * (i & 1))) & 0xFFFFu;
        u32* const o = (u32*)ms_shfl64(dp, b);
        if (in) o[v] = (m >> b) & 1ull ? dv : SCS_DIST_NONE;
      }
    }
  }
  ms_count_bytes(bytes, nbytes);
}

// One adjacency unit (at most MS_UNIT entries) as the local degree and
// adjacency passes take it: lane i holds entries i, i+64, i+128, i+192 (0 past
// the unit's end), lane b query b's local id of the unit's vertex.  A wave
// loads the next unit while it works on this one, so a unit costs two round
// trips less than its chain of header, entries, keep masks and rows; the keep
// masks of the entries, gathers all over the graph, are read only for a vertex
// that some query of the pass keeps.
struct MsUnitRegs {
  u32 u, h, len, id, w[4];
  u64 mu;  // the pass's queries that keep u
};
__device__ __forceinline__ void ms_unit_load(const int32_t* __restrict__ adj, const MsUnit& U,
                                             const u64* __restrict__ vis, u64 valid,
                                             const u32* __restrict__ locid, const MsCols& cols,
                                             MsUnitRegs& R) {
  const u32 lane = threadIdx.x & 63;
  const i64 b0 = (i64)(U.pos & 0xFFFFFFFFFFFFull);
  R.u = U.u;
  R.h = U.h;
  R.len = (u32)(U.pos >> 48);
  R.mu = vis[U.u] & valid;
  R.id = locid[(u64)U.u * cols.stride + cols.col(lane)];
#pragma unroll
  for (int t = 0; t < 4; t++) R.w[t] = lane + 64u * t < R.len ? (u32)adj[b0 + lane + 64 * t] : 0u;
}
// mw[t] = the queries that keep entry t.
__device__ __forceinline__ void ms_unit_masks(const u64* __restrict__ vis, const MsUnitRegs& R,
                                              u64 mw[4], u64& nbytes) {
  const u32 lane = threadIdx.x & 63;
#pragma unroll
  for (int t = 0; t < 4; t++) {
    mw[t] = 0;
    if (lane + 64u * t < R.len) {
      mw[t] = vis[R.w[t]];
      nbytes += 12;
    }
  }
}

// Local degree of every (query, kept vertex).  One wave per adjacency unit;
// lane b counts query b's kept neighbours in the unit as the popcount of
// column b of the transposed keep masks.  A single-unit vertex writes
// loff[id] directly; a hub's units write partial counts to hubcnt, which
// ms_hubsum turns into unit offsets and the degree.
// Bound: round trips.  500,000 vertices, 16M entries, 5 queries: 137 us, 164 with
// one unit at a time.
__global__ void __launch_bounds__(256) ms_degree(const int32_t* __restrict__ adj,
                                                 const MsUnit* __restrict__ units, u32 nunits,
                                                 const u64* __restrict__ vis, u64 valid,
                                                 const u32* __restrict__ locid, MsCols cols,
                                                 const MsBatch* __restrict__ B,
                                                 u32* __restrict__ hubcnt,
                                                 unsigned long long* bytes) {
  const u32 lane = threadIdx.x & 63;
  const u32 wid = ms_wave_id();
  const u32 nw = (gridDim.x * blockDim.x) >> 6;
  if (wid >= nunits) return;
  u32* const loff = B->P[lane].loff;
  u64 nbytes = 0;
  MsUnitRegs N;
  ms_unit_load(adj, units[wid], vis, valid, locid, cols, N);
  MsUnit Un = units[(u64)wid + nw < nunits ? wid + nw : wid];
  for (u64 k = wid; k < nunits; k += nw) {
    const MsUnitRegs R = N;
    if (k + nw < nunits) {
      ms_unit_load(adj, Un, vis, valid, locid, cols, N);
      if (k + 2ull * nw < nunits) Un = units[k + 2ull * nw];
    }
    if (lane == 0) nbytes += 16 + 8;
    if (!R.mu) continue;
    u64 mw[4];
    ms_unit_masks(vis, R, mw, nbytes);
    u32 cnt = 0;
#pragma unroll
    for (int t = 0; t < 4; t++)
      if (64u * t < R.len) cnt += (u32)__popcll(ms_transpose(mw[t] & R.mu));
    if (R.h == MS_NOHUB) {
      if ((R.mu >> lane) & 1ull) {
        loff[R.id] = cnt;
        nbytes += 8;
      }
    } else {
      hubcnt[(u64)R.h * 64 + lane] = cnt;
      nbytes += 4;
    }
  }
  ms_count_bytes(bytes, nbytes);
}

// One wave per hub vertex: lane b turns the hub's per-unit counts into
// exclusive unit offsets (in place) and writes the degree to loff[id].
__global__ void __launch_bounds__(256) ms_hubsum(const MsHub* __restrict__ hubs, u32 nhubs,
                                                 const u64* __restrict__ vis, u64 valid,
                                                 const u32* __restrict__ locid, MsCols cols,
                                                 const MsBatch* __restrict__ B,
                                                 u32* __restrict__ hubcnt,
                                                 unsigned long long* bytes) {
  const u32 lane = threadIdx.x & 63;
  const u32 wid = ms_wave_id();
  const u32 nw = (gridDim.x * blockDim.x) >> 6;
  u64 nbytes = 0;
  for (u32 k = wid; k < nhubs; k += nw) {
    const MsHub H = hubs[k];
    const u64 mu = vis[H.u] & valid;
    if (lane == 0) nbytes += 16 + 8;
    if (!mu) continue;
    u32 run = 0;
    for (u32 t = 0; t < H.nu; t++) {
      u32* p = &hubcnt[(u64)(H.h0 + t) * 64 + lane];
      const u32 c = *p;
      *p = run;
      run += c;
    }
    nbytes += (u64)H.nu * 8;
    if ((mu >> lane) & 1ull) {
      const u32 id = locid[(u64)H.u * cols.stride + cols.col(lane)];
      B->P[lane].loff[id] = run;
      nbytes += 8;
    }
  }
  ms_count_bytes(bytes, nbytes);
}

// Exclusive scan of every valid query's loff[0..K) in place, loff[K] = nnz
// -> tot[64 + b], in three passes with no LDS: chunk sums, chunk bases per
// query, then each chunk rescanned from its base.  A chunk is MS_SCAN_CHUNK
// entries, one wave, 64 contiguous entries per lane (16 aligned 16-byte
// loads: loff starts on an arena granule).  Wave w of the first and last
// passes takes query w / cmax, chunk w % cmax.
#define MS_SCAN_CHUNK 4096

__device__ __forceinline__ u32 ms_lane_load(const u32* __restrict__ a, u64 i0, u32 K, uint4 v[16]) {
  u32 s = 0;
  if (i0 + 64 <= K) {
    const uint4* p = (const uint4*)(a + i0);
#pragma unroll
    for (int k = 0; k < 16; k++) v[k] = p[k];
  } else {
#pragma unroll
    for (int k = 0; k < 16; k++) {
      const u64 i = i0 + 4 * k;
      v[k].x = i < K ? a[i] : 0u;
      v[k].y = i + 1 < K ? a[i + 1] : 0u;
      v[k].z = i + 2 < K ? a[i + 2] : 0u;
      v[k].w = i + 3 < K ? a[i + 3] : 0u;
    }
  }
#pragma unroll
  for (int k = 0; k < 16; k++) s += v[k].x + v[k].y + v[k].z + v[k].w;
  return s;
}

__global__ void __launch_bounds__(256) ms_loff_sum(const MsBatch* __restrict__ B,
                                                   const u32* __restrict__ tot, u64 valid,
                                                   u32 cmax, u32* __restrict__ csum) {
  const u32 lane = threadIdx.x & 63;
  const u32 wid = ms_wave_id();
  const u32 b = wid / cmax, c = wid % cmax;
  if (b >= 64 || !((valid >> b) & 1ull)) return;
  const u32 K = tot[b];
  const u64 c0 = (u64)c * MS_SCAN_CHUNK;
  if (c0 >= K) return;
  const u64 i0 = c0 + 64ull * lane;
  uint4 v[16];
  const u32 s = i0 < K ? ms_lane_load(B->P[b].loff, i0, K, v) : 0u;
  const u32 t = __shfl(ms_wave_incl(s), 63);
  if (lane == 0) csum[(u64)b * cmax + c] = t;
}

// One wave per query: chunk sums -> exclusive chunk bases; loff[K] and
// tot[64 + b] get the total.
__global__ void __launch_bounds__(64) ms_loff_base(const MsBatch* __restrict__ B,
                                                   u32* __restrict__ tot, u64 valid, u32 cmax,
                                                   u32* __restrict__ csum) {
  const u32 b = blockIdx.x, lane = threadIdx.x;
  if (!((valid >> b) & 1ull)) return;
  const u32 K = tot[b];
  const u32 nc = (K + MS_SCAN_CHUNK - 1) / MS_SCAN_CHUNK;
  const u32 per = (nc + 63) / 64;
  const u32 c0 = min(nc, lane * per), c1 = min(nc, c0 + per);
  u32* cs = csum + (u64)b * cmax;
  u32 s = 0;
  for (u32 c = c0; c < c1; c++) s += cs[c];
  const u32 incl = ms_wave_incl(s);
  u32 run = incl - s;
  for (u32 c = c0; c < c1; c++) {
    const u32 x = cs[c];
    cs[c] = run;
    run += x;
  }
  if (lane == 63) {
    B->P[b].loff[K] = incl;
    tot[64 + b] = incl;
  }
}

__global__ void __launch_bounds__(256) ms_loff_apply(const MsBatch* __restrict__ B,
                                                     const u32* __restrict__ tot, u64 valid,
                                                     u32 cmax, const u32* __restrict__ csum,
                                                     unsigned long long* bytes) {
  const u32 lane = threadIdx.x & 63;
  const u32 wid = ms_wave_id();
  const u32 b = wid / cmax, c = wid % cmax;
  if (b >= 64 || !((valid >> b) & 1ull)) return;
  const u32 K = tot[b];
  const u64 c0 = (u64)c * MS_SCAN_CHUNK;
  if (c0 >= K) return;
  u32* a = B->P[b].loff;
  const u64 i0 = c0 + 64ull * lane;
  uint4 v[16];
  const u32 s = i0 < K ? ms_lane_load(a, i0, K, v) : 0u;
  u32 run = csum[(u64)b * cmax + c] + ms_wave_incl(s) - s;
  u64 nbytes = 0;
  if (i0 < K) {
    uint4 o[16];
#pragma unroll
    for (int k = 0; k < 16; k++) {
      o[k].x = run; run += v[k].x;
      o[k].y = run; run += v[k].y;
      o[k].z = run; run += v[k].z;
      o[k].w = run; run += v[k].w;
    }
    if (i0 + 64 <= K) {
      uint4* p = (uint4*)(a + i0);
#pragma unroll
      for (int k = 0; k < 16; k++) p[k] = o[k];
      nbytes = 64 * 8;
    } else {
#pragma unroll
      for (int k = 0; k < 16; k++) {
        const u64 i = i0 + 4 * k;
        if (i < K) a[i] = o[k].x;
        if (i + 1 < K) a[i + 1] = o[k].y;
        if (i + 2 < K) a[i + 2] = o[k].z;
        if (i + 3 < K) a[i + 3] = o[k].w;
      }
      nbytes = (K - i0) * 8;
    }
  }
  ms_count_bytes(bytes, nbytes);
}

// Local adjacency: for every (query, kept vertex u), the local ids of u's
// kept neighbours in ascending order at ladj[loff[id(u)] ..].
// One wave per adjacency unit.  Query b's entries of the unit go to its
// write position dst_b, in neighbour order; column b of the transposed keep
// masks says which neighbours query b keeps.  The work is cut into tiles of
// 8 queries x 8 neighbours: lane (ji, qi) = (lane / 8, lane % 8) takes query
// 8 qb + qi and neighbour 8 jb + ji.  A store instruction then writes eight
// runs of up to eight consecutive entries and a load instruction reads eight
// pieces of eight entries of the locid rows, where a whole-row or whole-column
// form touches 64 lines with one of the two.
//
// FEW: one group of eight queries at a time, for batches that leave at most
// MS_FILL_FEW queries to this pass: groups without a query that keeps the
// vertex and tiles past the unit's end are passed over, and the registers that
// saves let twice the waves hide the round trips.  Else four groups at a time,
// with all their 32 row loads in flight and no branches between them.
// 500,000 vertices, 5 queries: 354 us, 525 before; 131,072 (R-MAT), 35 queries:
// 314, 312 before.
// Ids from per-group keep bits (16 bytes per query and 64 vertices) in place
// of the rows were 1.5 times slower; non-temporal stores 2.7 times.
#define MS_FILL_FEW 16
template <bool FEW>
__global__ void __launch_bounds__(256, FEW ? 6 : 1) ms_fill(const int32_t* __restrict__ adj,
                                               const MsUnit* __restrict__ units, u32 nunits,
                                               const u64* __restrict__ vis, u64 valid,
                                               const u32* __restrict__ locid, MsCols cols,
                                               const MsBatch* __restrict__ B,
                                               const u32* __restrict__ hubcnt,
                                               unsigned long long* bytes) {
  constexpr u32 QG = FEW ? 1 : 4;
  constexpr u64 GMASK = (1ull << (QG * 8)) - 1ull;
  const u32 lane = threadIdx.x & 63;
  const u32 wid = ms_wave_id();
  const u32 nw = (gridDim.x * blockDim.x) >> 6;
  if (wid >= nunits) return;
  const u32 qi = lane % 8, ji = lane / 8;
  const u32 below = (1u << ji) - 1u;
  const u32* const loff = B->P[lane].loff;
  u32* const ladj = B->P[lane].ladj;
  u64 nbytes = 0;
  MsUnitRegs N;
  ms_unit_load(adj, units[wid], vis, valid, locid, cols, N);
  MsUnit Un = units[(u64)wid + nw < nunits ? wid + nw : wid];
  for (u64 k = wid; k < nunits; k += nw) {
    const MsUnitRegs R = N;
    if (k + nw < nunits) {
      ms_unit_load(adj, Un, vis, valid, locid, cols, N);
      if (k + 2ull * nw < nunits) Un = units[k + 2ull * nw];
    }
    if (lane == 0) nbytes += 16 + 8;
    const u64 mu = ms_uniform64(R.mu);
    if (!mu) continue;
    const u32 len = __builtin_amdgcn_readfirstlane(R.len);
    u64 mw[4];
    ms_unit_masks(vis, R, mw, nbytes);
    // lane b: where query b's entries of this unit go
    u64 dst = 0;
    if ((mu >> lane) & 1ull) {
      const u32 part = R.h != MS_NOHUB ? hubcnt[(u64)R.h * 64 + lane] : 0u;
      dst = (u64)(ladj + loff[R.id] + part);
      nbytes += 8;
    }
    u64 col[4];  // lane b: bit j = query b keeps entry 64t + j
#pragma unroll
    for (int t = 0; t < 4; t++) col[t] = 64u * t < len ? ms_transpose(mw[t] & mu) : 0ull;
#pragma unroll
    for (int t = 0; t < 4; t++) nbytes += 8ull * (u32)__popcll(col[t]);
    for (u32 qb0 = 0; qb0 < 8; qb0 += QG) {
      if (!((mu >> (qb0 * 8)) & GMASK)) continue;  // none of these queries keeps the vertex
      __attribute__((address_space(1))) u32* dq[QG];
#pragma unroll
      for (u32 x = 0; x < QG; x++)
        dq[x] = (__attribute__((address_space(1))) u32*)ms_shfl64(dst, (int)((qb0 + x) * 8 + qi));
#pragma unroll
      for (int t = 0; t < 4; t++) {
        if (64u * t >= len) break;
        const u32 nj = FEW ? (min(64u, len - 64u * t) + 7) / 8 : 8u;  // blocks to take
        u32 wj[8];  // an entry is 0 past the unit's end, so every row index is a vertex
#pragma unroll
        for (u32 jb = 0; jb < 8; jb++)
          if (jb < nj) wj[jb] = (u32)__shfl(R.w[t], (int)(jb * 8 + ji));
        u32 r[QG][8];
#pragma unroll
        for (u32 x = 0; x < QG; x++)
#pragma unroll
          for (u32 jb = 0; jb < 8; jb++)
            if (jb < nj)
              r[x][jb] = locid[(u64)wj[jb] * cols.stride + cols.group(qb0 + x) + qi];
#pragma unroll
        for (u32 x = 0; x < QG; x++) {
          const u32 clo = __shfl((u32)col[t], (int)((qb0 + x) * 8 + qi));
          const u32 chi = __shfl((u32)(col[t] >> 32), (int)((qb0 + x) * 8 + qi));
#pragma unroll
          for (u32 jb = 0; jb < 8; jb++)
            if (jb < nj) {
              const u32 bits = ((jb < 4 ? clo : chi) >> (8 * (jb & 3))) & 0xFFu;
              if ((bits >> ji) & 1u) dq[x][__popc(bits & below)] = r[x][jb];
              dq[x] += __popc(bits);
            }
        }
      }
    }
  }
  ms_count_bytes(bytes, nbytes);
}

// ---------------------------------------------------------------------------
// Launchers.  B points to the batch header in device memory.
// ---------------------------------------------------------------------------
// Grid-stride kernels launch at most one generation of resident waves
// (2048 blocks of four waves = 8 waves on each SIMD of 256 CUs).
#define MS_GRID 2048
static MsCols ms_cols(u64 valid) {
  MsCols c{0, 0};
  for (u32 g = 0; g < 8; g++)
    if ((valid >> (8 * g)) & 0xFFull) {
      c.rank |= (c.stride / 8) << (4 * g);
      c.stride += 8;
    }
  return c;
}
static u32 ms_blocks(u64 threads, u32 cap) {
  u64 b = (threads + 255) / 256;
  if (b == 0) b = 1;
  return (u32)(b < cap ? b : cap);
}

extern "C" hipError_t scs_launch_ms_init(u32 n, const u32* core, const MsBatch* B, u64* elig,
                                         u64* vis, u64* fr, u64* nf, u64* xf, u32* flags,
                                         u32 nflags, unsigned long long* bytes, hipStream_t s) {
  ms_init<<<ms_blocks(n, MS_GRID), 256, 0, s>>>(n, core, B, elig, vis, fr, nf, xf, flags, nflags,
                                                bytes);
  return hipGetLastError();
}
extern "C" hipError_t scs_launch_ms_push0(const i64* off, const int32_t* adj, u32 nb,
                                          const MsBatch* B, u64 act, const u64* elig, u64* vis,
                                          u64* nf, u16* dist16, u32* flag0,
                                          unsigned long long* bytes, hipStream_t s) {
  ms_push0<<<nb, 64, 0, s>>>(off, adj, B, act, elig, vis, nf, dist16, flag0, bytes);
  return hipGetLastError();
}
extern "C" hipError_t scs_launch_ms_seed(const MsBatch* B, u64* vis, u64* fr, u16* dist16,
                                         hipStream_t s) {
  ms_seed<<<1, 64, 0, s>>>(B, vis, fr, dist16);
  return hipGetLastError();
}
extern "C" hipError_t scs_launch_ms_level(const int32_t* adj, const MsUnit* units, u32 nunits,
                                          const MsHub* hubs, u32 nhubs, u32 level, u64 act,
                                          const u64* elig, u64* vis, const u64* fr, u64* nf,
                                          u64* clr, u16* dist16, const u32* flag_prev,
                                          u32* flag_cur, unsigned long long* bytes,
                                          hipStream_t s) {
  ms_level<<<ms_blocks(((u64)nunits + 3) / 4 * 64, MS_GRID), 256, 0, s>>>(
      adj, units, nunits, hubs, nhubs, level, act, elig, vis, fr, nf, clr, dist16, flag_prev,
      flag_cur, bytes);
  return hipGetLastError();
}
static u32 ms_chunk(u32 G) { return G ? (G + 255) / 256 : 1; }
// Kept counts and their bases: gcnt holds G * 64 words, cbase one row of 64
// per chunk.
extern "C" hipError_t scs_launch_ms_count(u32 n, u32 G, u64* vis, const u64* lf, u64 valid,
                                          u32* gcnt, u32* cbase, u32* tot,
                                          unsigned long long* bytes, hipStream_t s) {
  const u32 ch = ms_chunk(G), C = (G + ch - 1) / ch;
  if (C) ms_count<<<(C + 3) / 4, 256, 0, s>>>(n, G, ch, vis, lf, valid, gcnt, cbase, bytes);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  ms_bscan<<<1, 64, 0, s>>>(C, cbase, tot, bytes);
  return hipGetLastError();
}
extern "C" u64 scs_ms_count_rows(u32 G) { return G ? (G + ms_chunk(G) - 1) / ms_chunk(G) : 1; }
extern "C" hipError_t scs_launch_ms_gdist(u32 n, u32 G, const u64* vis, u64 gmask,
                                          const u16* dist16, const MsBatch* B,
                                          unsigned long long* bytes, hipStream_t s) {
  ms_gdist<<<ms_blocks((u64)G * 64, MS_GRID), 256, 0, s>>>(n, G, vis, gmask, dist16, B, bytes);
  return hipGetLastError();
}
extern "C" hipError_t scs_launch_ms_scatter(u32 n, u32 G, const u64* vis, u64 valid,
                                            const u32* gcnt, const u32* cbase, const u32* core,
                                            const u16* dist16,
                                            const MsBatch* B, u32* locid, u32* qloc,
                                            unsigned long long* bytes, hipStream_t s) {
  ms_scatter<<<ms_blocks((u64)G * 64, MS_GRID), 256, 0, s>>>(n, G, ms_chunk(G), vis, valid, gcnt, cbase,
                                                          core, dist16,
                                                          B, locid, ms_cols(valid), qloc, bytes);
  return hipGetLastError();
}
// Local degrees, then the hubs' unit offsets (nhubs may be 0).
extern "C" hipError_t scs_launch_ms_degree(const int32_t* adj, const MsUnit* units, u32 nunits,
                                           const MsHub* hubs, u32 nhubs, const u64* vis,
                                           u64 valid, const u32* locid, const MsBatch* B,
                                           u32* hubcnt, unsigned long long* bytes,
                                           hipStream_t s) {
  ms_degree<<<ms_blocks((u64)nunits * 64, MS_GRID), 256, 0, s>>>(adj, units, nunits, vis, valid,
                                                                locid, ms_cols(valid), B, hubcnt,
                                                                bytes);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || nhubs == 0) return e;
  ms_hubsum<<<ms_blocks((u64)nhubs * 64, MS_GRID), 256, 0, s>>>(hubs, nhubs, vis, valid, locid, ms_cols(valid), B,
                                                             hubcnt, bytes);
  return hipGetLastError();
}
// cmax = chunks of the largest valid K (>= 1); csum holds nb * cmax words.
extern "C" hipError_t scs_launch_ms_scan_loff(u32 nb, const MsBatch* B, u32* tot, u64 valid,
                                              u32 cmax, u32* csum, unsigned long long* bytes,
                                              hipStream_t s) {
  const u32 blocks = (u32)(((u64)nb * cmax + 3) / 4);
  ms_loff_sum<<<blocks, 256, 0, s>>>(B, tot, valid, cmax, csum);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  ms_loff_base<<<nb, 64, 0, s>>>(B, tot, valid, cmax, csum);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  ms_loff_apply<<<blocks, 256, 0, s>>>(B, tot, valid, cmax, csum, bytes);
  return hipGetLastError();
}
// packed: the queries that scatter and degree took (valid may have lost some
// since, for want of room; the rows keep their columns).
extern "C" hipError_t scs_launch_ms_fill(const int32_t* adj, const MsUnit* units, u32 nunits,
                                         const u64* vis, u64 valid, u64 packed, const u32* locid,
                                         const MsBatch* B, const u32* hubcnt,
                                         unsigned long long* bytes, hipStream_t s) {
  const u32 blocks = ms_blocks((u64)nunits * 64, MS_GRID);
  if (__builtin_popcountll(valid) <= MS_FILL_FEW)
    ms_fill<true><<<blocks, 256, 0, s>>>(adj, units, nunits, vis, valid, locid, ms_cols(packed), B, hubcnt, bytes);
  else
    ms_fill<false><<<blocks, 256, 0, s>>>(adj, units, nunits, vis, valid, locid, ms_cols(packed), B, hubcnt, bytes);
  return hipGetLastError();
}
