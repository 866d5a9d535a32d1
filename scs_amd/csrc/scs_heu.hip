// Greedy lower bounds on the GPU: the reference's CSSC_heu
// (inc/heuristic.h:321-348), the best of its three greedy constructions
// heu2 (:8-120), heu3 (:125-239) and heu4 (:242-317), one block of eight
// waves per construction of each query.
//
// The reference drives each construction with a std::priority_queue that
// holds stale duplicates.  Its pop order reduces to a deterministic choice
// per step, which a block makes with a reduction instead of a heap:
//   heu2  add the frontier vertex with the largest (count of H-neighbours,
//         id); every increment of a count pushes, so the largest pushed key
//         of a vertex is its current count;
//   heu3  add the frontier vertex with the largest (key, id), where key is
//         the largest score ever pushed for it (scores can fall, and a
//         stale larger entry is popped first);
//   heu4  peel the vertex of S with the smallest (degree in S, id); degrees
//         only fall, so the smallest pushed key of a vertex is its current
//         degree.
// heu3's score of v sums 1/deg(w) over v's neighbours w in H in ascending
// id order, then adds deg(v)/dmax, as the reference's adjacency scan does,
// so the doubles are bit-identical.  heu4 drops the reference's +1 on q when
// q is popped alone (inc/heuristic.h:259), as the host version does.
//
// Candidates sit in an append-only list.  Each block of 64 list positions
// keeps the largest key of its members; keys only rise while a vertex is a
// candidate, so a rise is an atomic max on its block, and only the block of
// the vertex chosen in a step is recomputed.  A step costs the chosen
// vertex's adjacency, shared by the eight waves, and one pass over the block
// keys.
//
// heu3 keeps, for each vertex, one bit per member of H (in joining order) that
// it is adjacent to, and H sorted by id with each member's term 1/deg: a score
// is then a walk over the at most h members, the same for every lane, instead
// of over the vertex's adjacency.
//
// Bound: latency of the steps' dependent loads (offsets, neighbours, their
// records, the keys): 512 lanes share a chosen hub's thousands of neighbours,
// four in flight each.  64 queries on a 100,000-vertex, 1.5M-edge power-law
// graph take 4.8 ms, 108.5 ms with one wave per construction and scores that
// walked adjacency lists; 8 queries on 4,000 vertices 0.9 and 4.6 ms.
#include "scs_internal.h"

#define HEU_T 512     // threads per block
#define HEU_NW (HEU_T / 64)
#define HEU_SMALL 32  // heu4: members of at most this degree are counted by one lane
#define HEU_LDSB 64   // heu4: block keys held in LDS (4,096 members)

struct HeuArgs {
  const u32* off;  // n+1, 32-bit offsets of the resident graph
  const u32* adj;
  u32 dmax, nq, hcap;
  const u32* ql;
  const u32* qh;
  const u32* qq;
  u8* zs;  // arrays that are zero between queries
  u8* gs;  // the others
  HeuLayout lay;
  u32* kl;     // nq
  u32* hsize;  // nq (sizes above hcap are reported, H is cut at hcap)
  u32* H;      // nq * hcap
  u32* kl3;    // 3 * nq: heu2, heu3, heu4 of each query
  u32* hs3;    // 3 * nq
  u32* H3;     // 3 * nq * hcap
};

#define LANE (threadIdx.x & 63u)
#define WAVE (threadIdx.x >> 6)

// One vertex's state in a construction.  sta: 0 untouched, 1 candidate (heu4:
// in S), 2 in H.  cnt: H-neighbours.  deg: degree inside H (heu4: inside S).
struct __attribute__((aligned(16))) HV {
  u32 cnt, deg, pos, sta;
};

// One 1,280-byte piece of the CU's LDS, which an engine that admits through this
// kernel leaves free beside its search waves.
struct HL {
  u64 wmax[HEU_NW];
  u32 wmin[HEU_NW];
  u32 m;        // candidates in the list
  u32 dv[2];    // H-neighbours of the chosen vertex (by step parity)
  u32 rank[2];  // members of H with a smaller id (by step parity)
  u32 best[2];  // heu3: largest id + 1 among the equal keys (by step parity)
  u32 mindeg, remove;
  u64 bk[HEU_LDSB];
};

__device__ __forceinline__ u32 h_sum(u32 x) {
  for (int o = 32; o > 0; o >>= 1) x += (u32)__shfl_xor((int)x, o);
  return x;
}
__device__ __forceinline__ u32 h_min(u32 x) {
  for (int o = 32; o > 0; o >>= 1) x = min(x, (u32)__shfl_xor((int)x, o));
  return x;
}
__device__ __forceinline__ u64 h_max64(u64 x) {
  for (int o = 32; o > 0; o >>= 1) {
    const u32 lo = (u32)__shfl_xor((int)(u32)x, o), hi = (u32)__shfl_xor((int)(u32)(x >> 32), o);
    const u64 y = ((u64)hi << 32) | lo;
    x = y > x ? y : x;
  }
  return x;
}
__device__ __forceinline__ u64 h_below() { return LANE ? (~0ull >> (64 - LANE)) : 0ull; }

struct HW {
  const u32* off;
  const u32* adj;
  u32 dmax, W;
  HV* hv;
  u64* key;   // heu3: bits of the largest score pushed, plus one
  u64* mask;  // heu3: W words per vertex, bit j = adjacent to the j-th member of H
  u32* list;
  u32* rmv;
  u32* th;
  u32* hsort;    // heu3: H sorted by id (two rows of hrow words, by step
  u32 hrow;      // parity), and each member's joining number (two more rows)
  double* term;  // heu3: 1/deg of the sorted members (0 for degree 0)
  u64* bkey;     // per block of 64 list positions: the largest member key (0 = none)
  HL* L;
};

// Candidate keys, larger is chosen first, 0 = not a candidate.
//   heu2: (count of H-neighbours + 1, id)
//   heu4: the complement of (degree in S, id), so the smallest pair is largest
//   heu3: the bits of the (non-negative) double key, plus one; ties are broken
//         by id when the chosen vertex is looked up
__device__ __forceinline__ u64 k2(u32 cnt, u32 x) { return ((u64)(cnt + 1) << 32) | x; }
__device__ __forceinline__ u64 k4(u32 deg, u32 x) { return ~(((u64)deg << 32) | x); }
// block keys are raised by atomics at the L2; reads go past the L1
__device__ __forceinline__ u64 hld64(const u64* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void hst64(u64* p, u64 v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void bump(HW& w, u32 p, u64 k) {
  atomicMax((unsigned long long*)&w.bkey[p >> 6], (unsigned long long)k);
}
__device__ __forceinline__ HV hget(const HW& w, u32 x) { return w.hv[x]; }

// Places in the list for the wave's lanes with `on` (call on all lanes).
__device__ __forceinline__ u32 push_pos(HW& w, bool on) {
  const u64 b = __ballot(on);
  u32 base = 0;
  if (b) {
    const int first = __ffsll((unsigned long long)b) - 1;
    if (LANE == (u32)first) base = atomicAdd(&w.L->m, (u32)__popcll(b));
    base = (u32)__shfl((int)base, first);
  }
  return base + (u32)__popcll(b & h_below());
}

// Largest k and smallest mn over the block; one barrier.
__device__ __forceinline__ void block_red(HL& L, u64& k, u32& mn) {
  k = h_max64(k);
  mn = h_min(mn);
  if (LANE == 0) {
    L.wmax[WAVE] = k;
    L.wmin[WAVE] = mn;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < HEU_NW; i++) {
    k = L.wmax[i] > k ? L.wmax[i] : k;
    mn = min(mn, L.wmin[i]);
  }
}

// This thread's share of the largest block key, without block bv.
__device__ __forceinline__ u64 max_blocks(const HW& w, u32 m, u32 bv) {
  const u32 nblk = (m + 63) / 64;
  u64 k = 0;
  for (u32 b0 = threadIdx.x; b0 < nblk; b0 += 4 * HEU_T) {
    u64 x[4];
#pragma unroll
    for (int t = 0; t < 4; t++) x[t] = hld64(&w.bkey[min(b0 + t * HEU_T, nblk - 1)]);
#pragma unroll
    for (int t = 0; t < 4; t++)
      if (b0 + t * HEU_T < nblk && b0 + t * HEU_T != bv && x[t] > k) k = x[t];
  }
  return k;
}

// Every array the run touched back to zero: the candidates' state and the
// block keys.
__device__ __forceinline__ void cleanup(HW& w, bool masks) {
  __syncthreads();
  const u32 m = w.L->m;
  for (u32 i = threadIdx.x; i < m; i += HEU_T) {
    const u32 x = w.list[i];
    w.hv[x] = HV{0, 0, 0, 0};
    if (masks) {
      w.key[x] = 0;
      for (u32 k = 0; k < w.W; k++) w.mask[(u64)x * w.W + k] = 0;
    }
  }
  const u32 nblk = (m + 63) / 64;
  for (u32 b = threadIdx.x; b < nblk; b += HEU_T) hst64(&w.bkey[b], 0ull);
}

// q as the only candidate, with key k.
__device__ __forceinline__ void seed(HW& w, u32 q, u64 k) {
  if (threadIdx.x == 0) {
    HL& L = *w.L;
    w.hv[q] = HV{0, 0, 0, 1};
    w.list[0] = q;
    hst64(&w.bkey[0], k);
    L.m = 1;
    L.dv[0] = L.dv[1] = L.rank[0] = L.rank[1] = L.best[0] = L.best[1] = 0;
  }
  __syncthreads();
}

// heu2 (inc/heuristic.h:8-120): H grows from q by the frontier vertex with
// the most H-neighbours (ties: larger id); the best prefix of size in
// [N1, N2] by minimum degree (ties: the later one) is kept.
__device__ __forceinline__ void heu2(HW& w, u32 N1, u32 N2, u32 q, u32* outH, u32 hcap,
                                     u32& osize, u32& okl) {
  HL& L = *w.L;
  seed(w, q, k2(0, q));
  u32 nH = 0, tkl = 0, tsize = 0;
  u64 M = k2(0, q);
  while (M) {
    const u32 v = (u32)M, par = nH & 1;
    const u32 b0 = w.off[v], e0 = w.off[v + 1], pv = w.hv[v].pos;
    if (threadIdx.x == 0) {
      w.th[nH] = v;
      w.hv[v].sta = 2;
      L.dv[par ^ 1] = 0;
    }
    nH++;
    u32 dv = 0;
    for (u32 j0 = b0; j0 < e0; j0 += 4 * HEU_T) {
      u32 nb[4];
      HV h[4];
#pragma unroll
      for (int t = 0; t < 4; t++) nb[t] = w.adj[min(j0 + t * HEU_T + threadIdx.x, e0 - 1)];
#pragma unroll
      for (int t = 0; t < 4; t++) h[t] = hget(w, nb[t]);
#pragma unroll
      for (int t = 0; t < 4; t++) {
        const bool in = j0 + t * HEU_T + threadIdx.x < e0;
        const u32 c = h[t].cnt + 1;
        const bool fresh = in && h[t].sta == 0;
        const u32 p = push_pos(w, fresh);
        if (in && h[t].sta == 2) {
          w.hv[nb[t]].deg = h[t].deg + 1;
          dv++;
        } else if (fresh) {
          w.hv[nb[t]] = HV{c, 0, p, 1};
          w.list[p] = nb[t];
          bump(w, p, k2(c, nb[t]));
        } else if (in) {
          w.hv[nb[t]].cnt = c;
          bump(w, h[t].pos, k2(c, nb[t]));
        }
      }
    }
    dv = h_sum(dv);
    if (LANE == 0 && dv) atomicAdd(&L.dv[par], dv);
    __syncthreads();
    // v's degree, v's block without v, the next choice, H's minimum degree
    const u32 dvt = L.dv[par], m = L.m;
    if (threadIdx.x == 0) w.hv[v].deg = dvt;
    u64 k = max_blocks(w, m, pv >> 6);
    if (WAVE == 0) {
      const u32 p = (pv & ~63u) + LANE;
      u64 kk = 0;
      if (p < m) {
        const u32 x = w.list[p];
        const HV h = hget(w, x);
        if (x != v && h.sta == 1) kk = k2(h.cnt, x);
      }
      kk = h_max64(kk);
      if (LANE == 0) hst64(&w.bkey[pv >> 6], kk);
      k = kk > k ? kk : k;
    }
    u32 mn = 0xffffffffu;
    if (nH >= N1)
      for (u32 i = threadIdx.x; i < nH; i += HEU_T)
        mn = min(mn, i == nH - 1 ? dvt : w.hv[w.th[i]].deg);
    block_red(L, k, mn);
    if (nH >= N1 && mn >= tkl) {
      tkl = mn;
      tsize = nH;
    }
    if (nH == N2) break;
    M = k;
  }
  for (u32 i = threadIdx.x; i < tsize && i < hcap; i += HEU_T) outH[i] = w.th[i];
  osize = tsize;
  okl = tkl;
  cleanup(w, false);
}

// Sum of the terms of x's H-neighbours in ascending id order, for the wave's
// 64 vertices at once: the sorted members go by one after another (64 of them
// in the lanes' registers, read out with readlane), and a lane adds the term
// when its vertex has the member's bit.  WN: words of a vertex's bits (0 = more
// than four: a word is loaded when it is needed).
template <int WN>
__device__ __forceinline__ double walk_members(const HW& w, u32 nH, const u32* hj, u32 x, bool on) {
  const u64* row = w.mask + (u64)x * w.W;
  u64 mk[WN ? WN : 1];
#pragma unroll
  for (int i = 0; i < (WN ? WN : 1); i++) mk[i] = WN && on ? row[i] : 0ull;
  double sc = 0.0;
  for (u32 r0 = 0; r0 < nH; r0 += 64) {
    const u32 cnt = min(64u, nH - r0), rl = r0 + min(LANE, cnt - 1);
    const u64 tb = (u64)__double_as_longlong(w.term[rl]);
    const u32 jl = hj[rl];
    for (u32 r = 0; r < cnt; r++) {
      const u32 j = __builtin_amdgcn_readlane(jl, r);
      const u32 lo = __builtin_amdgcn_readlane((u32)tb, r);
      const u32 hi = __builtin_amdgcn_readlane((u32)(tb >> 32), r);
      u64 word = 0;
      if (WN) {
#pragma unroll
        for (int i = 0; i < (WN ? WN : 1); i++)
          if ((j >> 6) == (u32)i) word = mk[i];
      } else if (on) {
        word = row[j >> 6];
      }
      const double t = __longlong_as_double((long long)(((u64)hi << 32) | lo));
      if ((word >> (j & 63)) & 1ull) sc += t;
    }
  }
  return sc;
}

// heu3 (inc/heuristic.h:125-239): H grows from q by the frontier vertex of
// largest connection score (the largest score pushed for it).
__device__ __forceinline__ void heu3(HW& w, u32 N1, u32 N2, u32 q, u32* outH, u32 hcap,
                                     u32& osize, u32& okl) {
  HL& L = *w.L;
  seed(w, q, 1ull);
  if (threadIdx.x == 0) w.key[q] = 1ull;
  u32 nH = 0, tkl = 0, tsize = 0, v = q;
  while (true) {
    const u32 par = nH & 1, jn = nH;
    const u32 b0 = w.off[v], e0 = w.off[v + 1], pv = w.hv[v].pos;
    const u32 *hid = w.hsort + par * w.hrow, *hj = hid + 2 * w.hrow;
    u32 *hidn = w.hsort + (par ^ 1) * w.hrow, *hjn = hidn + 2 * w.hrow;
    if (threadIdx.x == 0) {
      w.th[nH] = v;
      w.hv[v].sta = 2;
      L.dv[par ^ 1] = 0;
      L.rank[par ^ 1] = 0;
      L.best[par] = 0;
    }
    nH++;
    // counts, degrees and bits of v's neighbours; H's sorted list with a gap
    // for v
    u32 dv = 0;
    for (u32 j0 = b0; j0 < e0; j0 += 4 * HEU_T) {
      u32 nb[4];
      HV h[4];
      u64 mw[4];
#pragma unroll
      for (int t = 0; t < 4; t++) nb[t] = w.adj[min(j0 + t * HEU_T + threadIdx.x, e0 - 1)];
#pragma unroll
      for (int t = 0; t < 4; t++) {
        h[t] = hget(w, nb[t]);
        mw[t] = w.mask[(u64)nb[t] * w.W + (jn >> 6)];
      }
#pragma unroll
      for (int t = 0; t < 4; t++) {
        if (j0 + t * HEU_T + threadIdx.x >= e0) continue;
        if (h[t].sta == 2) {
          w.hv[nb[t]].deg = h[t].deg + 1;
          dv++;
        } else {
          w.hv[nb[t]].cnt = h[t].cnt + 1;
          w.mask[(u64)nb[t] * w.W + (jn >> 6)] = mw[t] | (1ull << (jn & 63));
        }
      }
    }
    u32 below = 0;
    for (u32 i = threadIdx.x; i < jn; i += HEU_T) {
      const u32 id = hid[i], to = i + (id > v ? 1u : 0u);
      hidn[to] = id;
      hjn[to] = hj[i];
      below += id < v ? 1u : 0u;
    }
    dv = h_sum(dv);
    below = h_sum(below);
    if (LANE == 0) {
      if (dv) atomicAdd(&L.dv[par], dv);
      if (below) atomicAdd(&L.rank[par], below);
    }
    __syncthreads();
    const u32 dvt = L.dv[par], rank = L.rank[par];
    u32 mn = 0xffffffffu;
    for (u32 i = threadIdx.x; i < nH; i += HEU_T) {
      u32 d;
      if (i == rank) {
        hidn[i] = v;
        hjn[i] = jn;
        w.hv[v].deg = dvt;
        d = dvt;
      } else {
        d = w.hv[hidn[i]].deg;
      }
      mn = min(mn, d);
      w.term[i] = d ? 1.0 / (double)d : 0.0;
    }
    __syncthreads();
    // scores of v's neighbours outside H, against the degrees after v joined;
    // a vertex whose only H-neighbour is v needs no walk: its sum is v's term
    const double termv = dvt != 0 ? 1.0 / (double)dvt : 0.0;
    const u32 wn = (nH + 63) / 64;
    for (u32 j0 = b0 + WAVE * 64; j0 < e0; j0 += HEU_T) {
      const bool in = j0 + LANE < e0;
      const u32 nb = w.adj[min(j0 + LANE, e0 - 1)];
      const HV h = hget(w, nb);
      const u32 dg = w.off[nb + 1] - w.off[nb];
      const u64 old = w.key[nb];
      const bool out = in && h.sta != 2, many = out && h.cnt > 1;
      double sc = 0.0 + termv;
      if (__ballot(many)) {
        double s2;
        if (wn == 1)
          s2 = walk_members<1>(w, nH, hjn, nb, many);
        else if (wn == 2)
          s2 = walk_members<2>(w, nH, hjn, nb, many);
        else if (wn <= 4 && w.W >= 4)
          s2 = walk_members<4>(w, nH, hjn, nb, many);
        else
          s2 = walk_members<0>(w, nH, hjn, nb, many);
        if (many) sc = s2;
      }
      sc += (double)dg / (double)w.dmax;
      const u64 k = (u64)__double_as_longlong(sc) + 1ull;
      const bool fresh = out && h.sta == 0;
      const u32 p = push_pos(w, fresh);
      if (fresh) {
        w.hv[nb].pos = p;
        w.hv[nb].sta = 1;
        w.list[p] = nb;
        w.key[nb] = k;
        bump(w, p, k);
      } else if (out && k > old) {
        w.key[nb] = k;
        bump(w, h.pos, k);
      }
    }
    __syncthreads();
    const u32 m = L.m;
    u64 M = max_blocks(w, m, pv >> 6);
    if (WAVE == 0) {
      const u32 p = (pv & ~63u) + LANE;
      u64 kk = 0;
      if (p < m) {
        const u32 x = w.list[p];
        if (w.hv[x].sta == 1) kk = w.key[x];
      }
      kk = h_max64(kk);
      if (LANE == 0) hst64(&w.bkey[pv >> 6], kk);
      M = kk > M ? kk : M;
    }
    if (nH < N1) mn = 0xffffffffu;
    block_red(L, M, mn);
    if (nH >= N1 && mn >= tkl) {
      tkl = mn;
      tsize = nH;
    }
    if (nH == N2 || M == 0) break;
    // the largest id among the candidates whose key is M
    const u32 nblk = (m + 63) / 64;
    for (u32 b0 = WAVE * 64; b0 < nblk; b0 += HEU_T) {
      const u32 b = b0 + LANE;
      u64 bm = __ballot(b < nblk && hld64(&w.bkey[min(b, nblk - 1)]) == M);
      while (bm) {
        const u32 p = (b0 + (u32)(__ffsll((unsigned long long)bm) - 1)) * 64 + LANE;
        bm &= bm - 1;
        if (p < m) {
          const u32 x = w.list[p];
          if (w.hv[x].sta == 1 && w.key[x] == M) atomicMax(&L.best[par], x + 1);
        }
      }
    }
    __syncthreads();
    const u32 best = L.best[par];
    if (best == 0) break;  // keys and members disagree: stop (never seen)
    v = best - 1;
  }
  for (u32 i = threadIdx.x; i < tsize && i < hcap; i += HEU_T) outH[i] = w.th[i];
  osize = tsize;
  okl = tkl;
  cleanup(w, true);
}

// heu4 (inc/heuristic.h:242-317): S = q and its neighbours; peel the vertex
// of smallest (degree in S, id) until N1 remain, keeping the peel prefix
// whose popped degree is the largest with |S left| in [N1, N2].  The degrees
// are counted by the whole block; the peeling, one vertex after another, is
// one wave's, without block barriers.  Up to 4,096 members' block keys are in
// LDS.
template <bool INLDS>
__device__ __forceinline__ void peel4(HW& w, u32 m, u32 N1, u32 N2, u32 q) {
  HL& L = *w.L;
  const u32 nblk = (m + 63) / 64;
  u32 nr = 0, rmv_idx = 0, mindeg = 0;
  while (true) {
    u64 M = 0;
    if (INLDS) {
      M = LANE < nblk ? L.bk[LANE] : 0ull;
    } else {
      for (u32 b0 = LANE; b0 < nblk; b0 += 256) {
        u64 x[4];
#pragma unroll
        for (int t = 0; t < 4; t++) x[t] = hld64(&w.bkey[min(b0 + 64u * t, nblk - 1)]);
#pragma unroll
        for (int t = 0; t < 4; t++) M = x[t] > M ? x[t] : M;
      }
    }
    M = h_max64(M);
    if (M == 0) break;
    const u64 best = ~M;
    const u32 v = (u32)best;
    u32 d = (u32)(best >> 32);
    const u32 remain = m - nr;
    if (v == q) d -= 1;
    if (remain >= N1 && remain <= N2 && d > mindeg) {
      mindeg = d;
      rmv_idx = nr;
    }
    if (remain == N1) break;
    // v's block without v, from the degrees before v's neighbours lose it
    // (their keys only rise), while v's adjacency is on its way
    const u32 b0 = w.off[v], e0 = w.off[v + 1], bv = w.hv[v].pos >> 6;
    const u32 p = bv * 64 + LANE;
    u32 x = w.adj[min(b0 + LANE, e0 - 1)];
    const u32 y = w.list[min(p, m - 1)];
    const HV hy = hget(w, y);
    u64 kk = h_max64(p < m && y != v && hy.sta ? k4(hy.deg, y) : 0ull);
    if (LANE == 0) {
      w.hv[v].sta = 0;
      w.rmv[nr] = v;
      if (INLDS)
        L.bk[bv] = kk;
      else
        hst64(&w.bkey[bv], kk);
    }
    nr++;
    // the key is in place before the rises below reach it
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    for (u32 j0 = b0; j0 < e0; j0 += 64) {
      const bool in = j0 + LANE < e0;
      const u32 xn = w.adj[min(j0 + 64 + LANE, e0 - 1)];
      const HV h = hget(w, x);
      if (in && h.sta) {
        w.hv[x].deg = h.deg - 1;
        const u64 k = k4(h.deg - 1, x);
        if (INLDS)
          atomicMax((unsigned long long*)&L.bk[h.pos >> 6], (unsigned long long)k);
        else
          bump(w, h.pos, k);
      }
      x = xn;
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
  }
  if (LANE == 0) {
    L.mindeg = mindeg;
    L.remove = rmv_idx;
  }
}

__device__ __forceinline__ void heu4(HW& w, u32 N1, u32 N2, u32 q, u32* outH, u32 hcap, u32& osize,
                                     u32& okl) {
  HL& L = *w.L;
  osize = 0;
  okl = 0;
  const u32 qb = w.off[q], qe = w.off[q + 1];
  if (qe - qb < N1 - 1u) return;
  const u32 m = 1 + (qe - qb), nblk = (m + 63) / 64;
  const bool inlds = nblk <= HEU_LDSB;
  for (u32 i = threadIdx.x; i < m; i += HEU_T) {
    const u32 x = i ? w.adj[qb + i - 1] : q;
    w.list[i] = x;
    w.hv[x] = HV{0, 0, i, 1};
  }
  if (threadIdx.x == 0) L.m = m;
  __syncthreads();
  // degree of each member inside S (q: one more, as the reference counts it)
  for (u32 i0 = WAVE * 64; i0 < m; i0 += HEU_T) {
    const u32 i = i0 + LANE;
    const bool on = i < m;
    u32 x = 0, b = 0, e = 0, c = 0;
    if (on) {
      x = w.list[i];
      b = w.off[x];
      e = w.off[x + 1];
    }
    const bool big = on && (e - b) > HEU_SMALL;
    if (on && !big) {
      for (u32 k = b; k < e; k += 4) {
        u32 y[4], s[4];
#pragma unroll
        for (int t = 0; t < 4; t++) y[t] = w.adj[min(k + t, e - 1)];
#pragma unroll
        for (int t = 0; t < 4; t++) s[t] = w.hv[y[t]].sta;
#pragma unroll
        for (int t = 0; t < 4; t++) c += k + t < e ? s[t] : 0u;
      }
    }
    u64 bm = __ballot(big);
    while (bm) {
      const int src = __ffsll((unsigned long long)bm) - 1;
      bm &= bm - 1;
      const u32 bb = (u32)__shfl((int)b, src), be = (u32)__shfl((int)e, src);
      u32 cc = 0;
      for (u32 k = bb; k < be; k += 256) {
        u32 y[4], s[4];
#pragma unroll
        for (int t = 0; t < 4; t++) y[t] = w.adj[min(k + 64u * t + LANE, be - 1)];
#pragma unroll
        for (int t = 0; t < 4; t++) s[t] = w.hv[y[t]].sta;
#pragma unroll
        for (int t = 0; t < 4; t++) cc += k + 64u * t + LANE < be ? s[t] : 0u;
      }
      cc = h_sum(cc);
      if (LANE == (u32)src) c = cc;
    }
    c += x == q ? 1u : 0u;
    if (on) w.hv[x].deg = c;
    const u64 kk = h_max64(on ? k4(c, x) : 0ull);
    if (LANE == 0) {
      if (inlds)
        L.bk[i0 >> 6] = kk;
      else
        hst64(&w.bkey[i0 >> 6], kk);
    }
  }
  __syncthreads();
  if (WAVE == 0) {
    if (inlds)
      peel4<true>(w, m, N1, N2, q);
    else
      peel4<false>(w, m, N1, N2, q);
  }
  __syncthreads();
  const u32 rmv_idx = L.remove, mindeg = L.mindeg;
  // H = S without the first rmv_idx peeled vertices, in S order
  for (u32 i = threadIdx.x; i < m; i += HEU_T) w.hv[w.list[i]].sta = 1;
  __syncthreads();
  for (u32 i = threadIdx.x; i < rmv_idx; i += HEU_T) w.hv[w.rmv[i]].sta = 0;
  __syncthreads();
  if (WAVE == 0) {
    u32 base = 0;
    for (u32 i0 = 0; i0 < m; i0 += 256) {
      u32 x[4], s[4];
#pragma unroll
      for (int t = 0; t < 4; t++) x[t] = w.list[min(i0 + 64u * t + LANE, m - 1)];
#pragma unroll
      for (int t = 0; t < 4; t++) s[t] = w.hv[x[t]].sta;
#pragma unroll
      for (int t = 0; t < 4; t++) {
        const bool keep = i0 + 64u * t + LANE < m && s[t];
        const u64 bal = __ballot(keep);
        const u32 p = base + (u32)__popcll(bal & h_below());
        if (keep && p < hcap) outH[p] = x[t];
        base += (u32)__popcll(bal);
      }
    }
  }
  osize = m - rmv_idx;
  okl = mindeg;
  cleanup(w, false);
}

// Three blocks per query, one per construction (block 3i + c runs heu2, heu3
// or heu4 of query i in its own workspace).
__global__ void __launch_bounds__(HEU_T, 4) scs_heu_kernel(HeuArgs A) {
  __shared__ HL L;
  const u32 bi = blockIdx.x, qi = bi / 3, which = bi % 3;
  if (qi >= A.nq) return;
  u8* const z = A.zs + (u64)qi * A.lay.zstride + A.lay.zpart[which];
  u8* const g = A.gs + (u64)qi * A.lay.gstride + A.lay.gpart[which];
  HW w;
  w.off = A.off;
  w.adj = A.adj;
  w.dmax = A.dmax;
  w.W = A.lay.words;
  w.hv = (HV*)z;
  w.bkey = (u64*)(z + A.lay.bkey);
  w.key = (u64*)(z + A.lay.key);
  w.mask = (u64*)(z + A.lay.mask);
  w.list = (u32*)g;
  w.th = w.rmv = (u32*)(g + A.lay.th);  // heu2 and heu3 use one, heu4 the other
  w.hsort = (u32*)(g + A.lay.hsort);
  w.hrow = A.lay.hrow;
  w.term = (double*)(g + A.lay.term);
  w.L = &L;
  const u32 l = A.ql[qi], h = A.qh[qi], q = A.qq[qi];
  u32* out = A.H3 + (u64)bi * A.hcap;
  u32 sz = 0, kk = 0;
  if (which == 0)
    heu2(w, l, h, q, out, A.hcap, sz, kk);
  else if (which == 1)
    heu3(w, l, h, q, out, A.hcap, sz, kk);
  else
    heu4(w, l, h, q, out, A.hcap, sz, kk);
  if (threadIdx.x == 0) {
    A.kl3[bi] = kk;
    A.hs3[bi] = sz;
  }
}

// CSSC_heu's pick (inc/heuristic.h:321-348): heu4 when it ties with both,
// else heu3 when it ties with heu2, else heu2.
__global__ void __launch_bounds__(64) scs_heu_pick(HeuArgs A) {
  const u32 qi = blockIdx.x;
  if (qi >= A.nq) return;
  const u32 k2 = A.kl3[3 * qi], k3 = A.kl3[3 * qi + 1], k4 = A.kl3[3 * qi + 2];
  const u32 c = (k4 >= k3 && k4 >= k2) ? 2u : (k3 >= k2 ? 1u : 0u);
  const u32 sz = A.hs3[3 * qi + c];
  const u32* src = A.H3 + (u64)(3 * qi + c) * A.hcap;
  u32* out = A.H + (u64)qi * A.hcap;
  for (u32 i = LANE; i < sz && i < A.hcap; i += 64) out[i] = src[i];
  if (LANE == 0) {
    A.kl[qi] = c == 2 ? k4 : (c == 1 ? k3 : k2);
    A.hsize[qi] = sz;
  }
}

static u64 heu_al(u64 x) { return (x + 255) & ~255ull; }

// Workspace of one query whose h is at most hmax, in three parts (heu2, heu3,
// heu4) of two areas: the arrays a block finds zeroed and leaves zeroed, whose
// layout depends on hmax, and the others, whose layout does not, so that runs
// with different hmax can share a workspace.
extern "C" HeuLayout scs_heu_layout(u32 n, u32 hmax) {
  HeuLayout L{};
  L.words = (hmax + 63) / 64;
  if (L.words == 3) L.words = 4;  // the walk takes 1, 2 or 4 words in registers
  u64 o = heu_al(16ull * n);  // records first
  L.bkey = o; o = heu_al(o + 8ull * ((n + 63) / 64 + 1));
  const u64 z24 = o;
  L.key = o; o = heu_al(o + 8ull * n);
  L.mask = o; o = heu_al(o + 8ull * L.words * n);
  L.zpart[1] = z24;
  L.zpart[2] = z24 + o;
  L.zstride = 2 * z24 + o;
  L.hrow = SCS_MAX_H + 24;
  o = heu_al(4ull * (n + 64));  // the list first
  L.th = o; o = heu_al(o + 4ull * (SCS_MAX_H + 64));
  const u64 g2 = o, g4 = heu_al(L.th + 4ull * (n + 64));
  L.hsort = o; o = heu_al(o + 16ull * L.hrow);
  L.term = o; o = heu_al(o + 8ull * L.hrow);
  L.gpart[1] = g2;
  L.gpart[2] = g2 + o;
  L.gstride = g2 + o + g4;
  return L;
}

// zs and gs hold nq workspaces; kl3/hs3/H3 hold the three constructions'
// results of each query, kl/hsize/H the picked one.
extern "C" hipError_t scs_launch_heu(const u32* off, const u32* adj, u32 dmax, u32 nq,
                                     const u32* ql, const u32* qh, const u32* qq, u8* zs,
                                     u8* gs, HeuLayout lay, u32 hcap, u32* kl, u32* hsize, u32* H,
                                     u32* kl3, u32* hs3, u32* H3, hipStream_t s) {
  HeuArgs A;
  A.off = off;
  A.adj = adj;
  A.dmax = dmax;
  A.nq = nq;
  A.hcap = hcap;
  A.ql = ql;
  A.qh = qh;
  A.qq = qq;
  A.zs = zs;
  A.gs = gs;
  A.lay = lay;
  A.kl = kl;
  A.hsize = hsize;
  A.H = H;
  A.kl3 = kl3;
  A.hs3 = hs3;
  A.H3 = H3;
  scs_heu_kernel<<<3 * nq, HEU_T, 0, s>>>(A);
  scs_heu_pick<<<nq, 64, 0, s>>>(A);
  return hipGetLastError();
}
