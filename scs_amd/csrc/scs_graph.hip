// Graph-level kernels for gfx950, once per graph: validation of a caller's CSR
// and core decomposition, replacing the reference's host-side linear-heap
// peeling (src/Graph.h:82-109).  Per-query preprocessing is batched in
// scs_prep.hip.
#include "scs_internal.h"

#include <mutex>

// ---------------------------------------------------------------------------
// Validation of a caller's CSR (offsets checked by the host: they ascend from
// 0 to nnz) and the 32-bit forms the search reads.  The search kernels need a
// simple undirected graph: every row strictly ascending, ids inside [0, n), no
// self-loops, and w in row v exactly when v is in row w.  A lane takes an
// entry, finds its row by search over the offsets and, when w > v, looks v up
// in row w; as many entries below the diagonal as above it leave none of those
// unmatched.  Bound: the searches' dependent loads.  3M entries take 266 us,
// 1,046 with a 16-lane segment per row (the longest row's), 4,000 on the host.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) csr_check(const i64* __restrict__ off,
                                                 const int32_t* __restrict__ adj, u32 n, u64 nnz,
                                                 u32* __restrict__ bad,
                                                 unsigned long long* __restrict__ above,
                                                 unsigned long long* __restrict__ below) {
  u64 up = 0, dn = 0;
  bool wrong = false;
  for (u64 j = (u64)blockIdx.x * blockDim.x + threadIdx.x; j < nnz;
       j += (u64)gridDim.x * blockDim.x) {
    u32 lo = 0, hi = n - 1;  // the last row whose offset is at most j
    while (lo < hi) {
      const u32 mid = lo + (hi - lo + 1) / 2;
      if ((u64)off[mid] <= j)
        lo = mid;
      else
        hi = mid - 1;
    }
    const u32 v = lo;
    const int32_t w = adj[j];
    if (w < 0 || (u32)w >= n || (u32)w == v || (j > (u64)off[v] && adj[j - 1] >= w)) {
      wrong = true;
      continue;
    }
    if ((u32)w < v) {
      dn++;
      continue;
    }
    up++;
    i64 a = off[w], b = off[w + 1];  // first entry >= v
    const i64 end = b;
    while (a < b) {
      const i64 mid = (a + b) >> 1;
      if ((i64)adj[mid] < (i64)v)
        a = mid + 1;
      else
        b = mid;
    }
    if (a == end || (i64)adj[a] != (i64)v) wrong = true;
  }
  for (int o = 32; o > 0; o >>= 1) {
    up += __shfl_xor(up, o);
    dn += __shfl_xor(dn, o);
  }
  const bool any = __ballot(wrong) != 0;
  if ((threadIdx.x & 63) == 0) {
    if (any) atomicOr(bad, 1u);
    if (up) atomicAdd(above, (unsigned long long)up);
    if (dn) atomicAdd(below, (unsigned long long)dn);
  }
}
__global__ void csr_narrow(const i64* __restrict__ off, u32 n, u32* __restrict__ off32,
                           u32* __restrict__ ident) {
  for (u64 v = (u64)blockIdx.x * blockDim.x + threadIdx.x; v <= n;
       v += (u64)gridDim.x * blockDim.x) {
    off32[v] = (u32)off[v];
    if (v < n) ident[v] = (u32)v;
  }
}
static u32 csr_blocks(u64 threads, u32 cap) {
  const u64 b = (threads + 255) / 256;
  return (u32)(b < 1 ? 1 : (b < cap ? b : cap));
}
// res: three u64 words, zeroed (bad, above, below).
extern "C" hipError_t scs_launch_csr_check(const i64* off, const int32_t* adj, u32 n, u64 nnz,
                                           u64* res, hipStream_t s) {
  csr_check<<<csr_blocks(nnz, 2048), 256, 0, s>>>(
      off, adj, n, nnz, (u32*)res, (unsigned long long*)(res + 1), (unsigned long long*)(res + 2));
  return hipGetLastError();
}
extern "C" hipError_t scs_launch_csr_narrow(const i64* off, u32 n, u32* off32, u32* ident,
                                            hipStream_t s) {
  csr_narrow<<<csr_blocks((u64)n + 1, 2048), 256, 0, s>>>(off, n, off32, ident);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Core decomposition: level-synchronous peeling in one persistent kernel.
// deg holds the remaining degree of a live vertex and, once it is peeled, its
// core number, so the output array is the only n-sized state that changes.
// At level k every block takes the vertices of its share with deg == k into
// its LDS queue, a grid barrier ends the scan, and each block then empties
// its queue: a neighbour whose degree falls to k joins the queue of the block
// that took it there, so a cascade inside a level needs no further barrier.
// Entries that do not fit the queue go to a list in device memory, which all
// blocks share out after the level's barrier.  Core numbers are unique, so
// the result equals any exact sequential peeling.
//
// Bound: latency.  A level costs two grid barriers (4 us each), a scan (10 us)
// and its longest cascade (queue, offsets, neighbours, degree atomics: 4 us a
// step); the innermost core, thousands of hubs that leave together, is bound
// by atomics on the same degrees (2 ms).  Chung-Lu graphs, 88K / 1.5M / 8M
// edges (16 / 76 / 206 levels): 0.43 / 1.9 / 6.7 ms, 3.0 / 17.0 / 40.7 ms
// before, with a launch and a host round trip per cascade step.  Blocks of
// 256 and 1,024 threads are 2-12 % slower on these three, 2,048 vertices per
// block and more 1.5 times slower on the first.
// ---------------------------------------------------------------------------
#define CORE_T 512          // threads per block
#define CORE_QCAP 4096      // LDS queue entries per block
#define CORE_EMPTY 0xffffffffu
#define CORE_VPB 256        // vertices per block at least
#define CORE_TIMEOUT 3000000000ull  // wall_clock64 ticks (100 MHz): 30 s
#define CORE_GRACE 20000ull         // the same, for the blocks to come: 200 us

enum { CORE_SCAN = 0, CORE_PEEL = 1, CORE_OVF = 2, CORE_DONE = 3 };

// Barrier and counters, 128-byte lines apart (a line that others poll makes
// an atomic on it wait).  Blocks arrive in CORE_GROUPS groups (by block
// number, which is how blocks are dealt to the XCDs), the last of a group
// arrives at the root: 32 + 8 serial adds instead of 256.  An arrival adds
// one in the low word and its count of vertices in the high word.
#define CORE_GROUPS 8
struct __attribute__((aligned(128))) CoreLine {
  u64 v;
  u64 pad[15];
};
struct CoreCtl {
  CoreLine grp[CORE_GROUPS];
  CoreLine go[CORE_GROUPS];  // what the group polls: step << 34 | op << 32 | k
  CoreLine root;
  CoreLine join;  // blocks that have come; high word: closed to others
  CoreLine nblk;  // blocks that take part (0 while join is open)
  u32 minrest, pad0[31];
  u32 ovf, pad1[31];
  // the root's last block only
  u32 k, o0, o1, peeled, failed;
};
#define CORE_CTL_WORDS 1024
static_assert(sizeof(CoreCtl) <= CORE_CTL_WORDS * sizeof(u32), "fits the counter words");

__device__ __forceinline__ u32 c_load(const u32* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void c_store(u32* p, u32 v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Place of vertex v's degree: an odd multiple modulo the power of two above
// n.  Generators and crawls number hubs first, and 32 hubs' degrees in one
// cache line make every decrement of any of them wait for the others.
#define CORE_MUL 0x9E3779B1u
#define CORE_INV 0x0E8B2F51u
__device__ __forceinline__ u32 core_pos(u32 v, u32 mask) { return (v * CORE_MUL) & mask; }

__global__ void core_init(const i64* __restrict__ off, u32 n, u32* __restrict__ deg, u32 mask,
                          CoreCtl* __restrict__ ctl) {
  for (u32 v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += gridDim.x * blockDim.x)
    deg[core_pos(v, mask)] = (u32)(off[v + 1] - off[v]);
  if (blockIdx.x == 0) {
    u32* w = (u32*)ctl;
    for (u32 i = threadIdx.x; i < sizeof(CoreCtl) / 4; i += blockDim.x) w[i] = 0;
    __syncthreads();
    if (threadIdx.x == 0) ctl->minrest = 0xffffffffu;
  }
}

struct CoreLds {
  u32 q[CORE_QCAP];
  u32 head, tail, pending, done;
  u32 found, op, k, o0, o1, mn;
  u32 rank, nblk;  // this block among those that take part
};
__device__ __forceinline__ u32 c_lget(const u32* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void c_lput(u32* p, u32 v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

__device__ __forceinline__ u64 c_add64(u64* p, u64 v) {
  return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void c_store64(u64* p, u64 v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Everything blocks exchange goes through agent-scope atomic loads, stores
// and adds, which act at the memory all XCDs share.  What one block must see
// after another is ordered by waiting for those operations alone: a release
// or acquire at agent scope would also write back the XCD's L2 or drop its
// lines, once per block and barrier (8 us of a 12 us step here).
__device__ __forceinline__ void c_order() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
  __builtin_amdgcn_s_waitcnt(0);
}
__device__ __forceinline__ u64 c_load64(const u64* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Which blocks take part: those that come before the join closes, which is when
// the last block of the grid has come, or CORE_GRACE after the first of those
// still waiting.  A block that comes later leaves at once, so no block ever
// waits for one that has found no room: on a stream with few CUs, beside
// another kernel or another peel, the peel runs with the blocks that are there
// (one is enough).  Their numbers are the block numbers when all have come,
// else the order of arrival.  False: this block leaves.
__device__ bool core_join(CoreCtl* C, CoreLds& L) {
  if (threadIdx.x == 0) {
    const u32 G = gridDim.x;
    u32 r = blockIdx.x, nb = 1;
    if (G > 1) {
      const u64 old = c_add64(&C->join.v, 1ull);
      nb = 0;
      if (!(old >> 32)) {
        r = (u32)old;
        const u64 t0 = wall_clock64();
        while ((nb = (u32)c_load64(&C->nblk.v)) == 0) {
          if (r + 1 == G || wall_clock64() - t0 > CORE_GRACE) {
            const u64 o = __hip_atomic_fetch_or(&C->join.v, 1ull << 32, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_AGENT);
            if (!(o >> 32)) c_store64(&C->nblk.v, o);
          } else {
            __builtin_amdgcn_s_sleep(1);
          }
        }
        if (nb == G) r = blockIdx.x;
      }
    }
    L.rank = r;
    L.nblk = nb;
  }
  __syncthreads();
  return L.nblk != 0;
}

// Grid barrier after step `gen`; the last block to arrive decides the next
// step for all.  scan: the barrier ends a scan that queued `count` vertices,
// else a peel that finished `count`.  The step comes back in L.  Each wave
// waits for its own operations before the block arrives: the block's barrier
// alone does not wait for stores and adds that return nothing (a degree's
// undone decrement, an overflow entry), and other blocks read those next.
__device__ void core_barrier(CoreCtl* C, CoreLds& L, u32 n, u32 gen, bool scan, u32 count) {
  c_order();
  __syncthreads();
  if (threadIdx.x == 0) {
    const u32 g = L.rank % CORE_GROUPS, G = L.nblk;
    const u32 ingrp = (G - g + CORE_GROUPS - 1) / CORE_GROUPS;
    const u32 ngrp = G < CORE_GROUPS ? G : CORE_GROUPS;
    if (scan && L.mn < c_load(&C->minrest)) atomicMin(&C->minrest, L.mn);
    c_order();
    const u64 mine = ((u64)count << 32) | 1ull;
    const u64 a = c_add64(&C->grp[g].v, mine) + mine;
    if ((u32)a == ingrp) {
      c_store64(&C->grp[g].v, 0ull);
      c_order();
      const u64 gm = (a & 0xFFFFFFFF00000000ull) | 1ull;
      const u64 r = c_add64(&C->root.v, gm) + gm;
      if ((u32)r == ngrp) {
        const u32 total = (u32)(r >> 32), k = c_load(&C->k);
        u32 op, nk = k;
        if (scan) {
          const u32 mr = c_load(&C->minrest);
          if (total) {
            op = CORE_PEEL;
          } else if (mr == 0xffffffffu) {
            op = CORE_DONE;
          } else {
            op = CORE_SCAN;
            nk = mr > k + 1 ? mr : k + 1;
          }
          c_store(&C->minrest, 0xffffffffu);
        } else {
          const u32 ov = c_load(&C->ovf), o1 = c_load(&C->o1), pe = c_load(&C->peeled) + total;
          c_store(&C->peeled, pe);
          if (ov > o1) {
            op = CORE_OVF;
            c_store(&C->o0, o1);
            c_store(&C->o1, ov);
          } else {
            op = pe >= n ? CORE_DONE : CORE_SCAN;
            nk = k + 1;
          }
        }
        c_store(&C->k, nk);
        c_store64(&C->root.v, 0ull);
        c_order();
        const u64 w = ((u64)(gen + 1) << 34) | ((u64)op << 32) | nk;
        for (u32 i = 0; i < ngrp; i++) c_store64(&C->go[i].v, w);
      }
    }
    // every block that takes part is running, so the wait ends; the time limit
    // only guards against a machine that stops some of them
    u64 w;
    const u64 t0 = wall_clock64();
    u32 spins = 0;
    bool bad = false;
    while ((u32)((w = c_load64(&C->go[g].v)) >> 34) != gen + 1) {
      __builtin_amdgcn_s_sleep(1);
      if ((++spins & 1023u) == 0 &&
          (c_load(&C->failed) || wall_clock64() - t0 > CORE_TIMEOUT)) {
        c_store(&C->failed, 1u);
        bad = true;
        break;
      }
    }
    c_order();
    L.op = bad ? (u32)CORE_DONE : (u32)(w >> 32) & 3u;
    L.k = (u32)w;
    if (L.op == CORE_OVF) {
      L.o0 = c_load(&C->o0);
      L.o1 = c_load(&C->o1);
    }
  }
  __syncthreads();
}

__device__ __forceinline__ void core_push(CoreCtl* C, CoreLds& L, u32* ovf, u32 v) {
  const u32 p = atomicAdd(&L.tail, 1u);
  if (p < CORE_QCAP) {
    atomicAdd(&L.pending, 1u);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    c_lput(&L.q[p], v);
  } else {
    c_store(&ovf[atomicAdd(&C->ovf, 1u)], v);
  }
}

// Peels v with one wave, four adjacency entries per lane in flight (the next
// four are loaded before this step's degree atomics).  Takes one from each
// live neighbour's degree; the lane that takes it to k queues the neighbour,
// and a decrement that lost the race against that one is undone.  Looking at
// the degree first costs a round trip per step of a cascade (4,000 vertices:
// 480 us, 370 without) and saves two atomics per peeled neighbour (500,000
// vertices: 7.2 ms, 12.7 without).
__device__ __forceinline__ void core_take(const i64* __restrict__ off,
                                          const int32_t* __restrict__ adj, CoreCtl* C, CoreLds& L,
                                          u32* ovf, u32* deg, u32 mask, u32 k, u32 v) {
  const u32 lane = threadIdx.x & 63;
  const i64 b = off[v], e = off[v + 1];
  if (b == e) return;
  u32 w[4], x[4];
#pragma unroll
  for (int t = 0; t < 4; t++) w[t] = b + lane + 64 * t < e ? (u32)adj[b + lane + 64 * t] : v;
  for (i64 j = b + lane; j - (i64)lane < e; j += 256) {
#pragma unroll
    for (int t = 0; t < 4; t++) x[t] = j + 256 + 64 * t < e ? (u32)adj[j + 256 + 64 * t] : v;
    u32 old[4];
    u32 d[4];
#pragma unroll
    for (int t = 0; t < 4; t++) d[t] = c_load(&deg[core_pos(w[t], mask)]);
#pragma unroll
    for (int t = 0; t < 4; t++)
      old[t] = w[t] != v && d[t] > k ? atomicSub(&deg[core_pos(w[t], mask)], 1u) : 0xffffffffu;
#pragma unroll
    for (int t = 0; t < 4; t++) {
      if (old[t] == k + 1)
        core_push(C, L, ovf, w[t]);
      else if (old[t] <= k)
        atomicAdd(&deg[core_pos(w[t], mask)], 1u);
      w[t] = x[t];
    }
  }
}

__global__ void __launch_bounds__(CORE_T) core_peel(const i64* __restrict__ off,
                                                    const int32_t* __restrict__ adj, u32 n,
                                                    u32* __restrict__ core, u32* __restrict__ deg,
                                                    u32 mask, u32* __restrict__ ovf,
                                                    CoreCtl* __restrict__ C) {
  __shared__ CoreLds L;
  if (!core_join(C, L)) return;
  const u32 rank = L.rank, nblk = L.nblk;
  const u32 nt = nblk * CORE_T, tid = rank * CORE_T + threadIdx.x;
  const u32 lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (u32 i = threadIdx.x; i < CORE_QCAP; i += CORE_T) L.q[i] = CORE_EMPTY;
  if (threadIdx.x == 0) {
    L.tail = L.head = L.pending = L.done = 0;
    L.op = CORE_SCAN;
    L.k = 0;
  }
  __syncthreads();
  // each pass of the loop ends in one grid barrier
  for (u32 gen = 0;; gen++) {
    const u32 op = L.op, k = L.k, o0 = L.o0, o1 = L.o1;
    if (op == CORE_DONE) break;
    if (op == CORE_SCAN) {
      if (threadIdx.x == 0) {
        L.found = 0;
        L.mn = 0xffffffffu;
      }
      __syncthreads();
      u32 mn = 0xffffffffu, fnd = 0;
      for (u64 p0 = tid; p0 <= mask; p0 += 4ull * nt) {
        u32 d[4];
#pragma unroll
        for (int t = 0; t < 4; t++) {
          const u64 p = p0 + (u64)t * nt;
          d[t] = p <= mask ? c_load(&deg[p]) : 0u;
        }
#pragma unroll
        for (int t = 0; t < 4; t++) {
          const u64 p = p0 + (u64)t * nt;
          const u32 v = ((u32)p * CORE_INV) & mask;
          if (p > mask || v >= n) continue;
          if (d[t] == k) {
            core_push(C, L, ovf, v);
            fnd++;
          } else if (d[t] > k) {
            mn = min(mn, d[t]);
          }
        }
      }
      for (int o = 32; o > 0; o >>= 1) {
        mn = min(mn, (u32)__shfl_xor((int)mn, o));
        fnd += (u32)__shfl_xor((int)fnd, o);
      }
      if ((threadIdx.x & 63) == 0) {
        if (fnd) atomicAdd(&L.found, fnd);
        atomicMin(&L.mn, mn);
      }
      __syncthreads();
      core_barrier(C, L, n, gen, true, L.found);
      continue;
    }
    u32 done = 0;
    if (op == CORE_OVF) {
      // this block's share of the entries that overflowed, a wave each
      for (u64 i = (u64)wave * nblk + rank; i < o1 - o0; i += (u64)nblk * (CORE_T / 64)) {
        core_take(off, adj, C, L, ovf, deg, mask, k, c_load(&ovf[o0 + i]));
        done++;
      }
    }
    // This block's queue, until its cascades end: a wave holds one ticket
    // (queue position) at a time, waits for its entry, and leaves when the
    // queue has no entry for it and none is being peeled (pending counts
    // entries queued and not yet peeled, so a wave that may still queue
    // others keeps it above zero).
    if (op == CORE_OVF) __syncthreads();
    while (true) {
      u32 h = 0, v = CORE_EMPTY;
      if (lane == 0) {
        h = atomicAdd(&L.head, 1u);
        if (h < CORE_QCAP) {
          while (true) {
            v = c_lget(&L.q[h]);
            __atomic_signal_fence(__ATOMIC_SEQ_CST);
            if (v != CORE_EMPTY || c_lget(&L.pending) == 0) break;
            __builtin_amdgcn_s_sleep(1);
          }
        }
      }
      v = __builtin_amdgcn_readfirstlane(v);
      if (v == CORE_EMPTY) break;
      core_take(off, adj, C, L, ovf, deg, mask, k, v);
      done++;
      // after this wave's pushes: a wave's LDS operations are done in order
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      if (lane == 0) atomicSub(&L.pending, 1u);
    }
    __syncthreads();
    for (u32 i = threadIdx.x; i < min(L.tail, (u32)CORE_QCAP); i += CORE_T) L.q[i] = CORE_EMPTY;
    if (lane == 0 && done) atomicAdd(&L.done, done);
    __syncthreads();
    done = L.done;
    __syncthreads();
    if (threadIdx.x == 0) L.tail = L.head = L.done = 0;
    core_barrier(C, L, n, gen, false, done);
  }
  for (u32 v = tid; v < n; v += nt) core[v] = c_load(&deg[core_pos(v, mask)]);
}

// ---------------------------------------------------------------------------
// Host-side launch helpers (C linkage inside the library).
// ---------------------------------------------------------------------------
// One block per CU at most (8 waves and 17 KB of LDS), fewer on small graphs,
// whose levels are too short for every CU to have a share.
static u32 core_blocks(u32 n) {
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      cus < 1)
    cus = 1;
  const u32 want = n / CORE_VPB + 1;
  return want < (u32)cus ? want : (u32)cus;
}

static u32 core_pow2(u32 n) {
  u32 b = 0;
  while ((1ull << b) < n) b++;
  return b;
}
// Words of scs_core_run's working memory: counters, degrees, overflow list.
extern "C" u64 scs_core_words(u32 n) { return CORE_CTL_WORDS + (1ull << core_pow2(n)) + n; }

// Core numbers of the CSR into core; tmp: scs_core_words(n) words on a
// 128-byte boundary, this call's own; blocks: of the grid (0 = as many as suit
// the graph).  Waits for the result.
extern "C" int scs_core_run(const i64* off, const int32_t* adj, u32 n, u32* core, u32* tmp,
                            hipStream_t s, u32 blocks) {
  if (n == 0) return SCS_OK;
  CoreCtl* C = (CoreCtl*)tmp;
  const u64 slots = 1ull << core_pow2(n);
  u32* deg = tmp + CORE_CTL_WORDS;
  u32* ovf = deg + slots;
  const u32 ib = (n + 255) / 256;
  core_init<<<ib < 4096 ? ib : 4096, 256, 0, s>>>(off, n, deg, (u32)(slots - 1), C);
  if (hipGetLastError() != hipSuccess) return SCS_EHIP;
  core_peel<<<blocks ? blocks : core_blocks(n), CORE_T, 0, s>>>(off, adj, n, core, deg, (u32)(slots - 1), ovf, C);
  if (hipGetLastError() != hipSuccess) return SCS_EHIP;
  u32 failed = 0;
  if (hipMemcpyAsync(&failed, &C->failed, sizeof(u32), hipMemcpyDeviceToHost, s) != hipSuccess ||
      hipStreamSynchronize(s) != hipSuccess)
    return SCS_EHIP;
  return failed ? SCS_EHIP : SCS_OK;
}

// ---------------------------------------------------------------------------
// Core numbers without allocation, for callers that cannot allocate device
// memory.  The working memory (overflow list, barrier and counter words) is
// this fixed device array; the host finds its per-device address once with
// hipGetSymbolAddress and passes that address to the kernels.
// Layout (words): counters[CORE_CTL_WORDS] | degrees | overflow list.
// ---------------------------------------------------------------------------
#define CORE_NA_MAX_N (1u << 20)
static __device__ __align__(256) u32 scratch[CORE_CTL_WORDS + 2u * CORE_NA_MAX_N];

#define CORE_NA_DEVICES 64
// The array of each device; its lock is held for a call, so calls on one
// device take turns and those on others do not wait for them.
static struct CoreScratch {
  std::mutex mu;
  u32* words = nullptr;
} g_scratch[CORE_NA_DEVICES];

extern "C" int scs_core_numbers_noalloc(const int64_t* d_off, const int32_t* d_adj, uint32_t n,
                                        uint32_t* d_core, void* stream) {
  if (!d_off || !d_core || (n && !d_adj)) return SCS_EINVAL;
  if (n > CORE_NA_MAX_N) return SCS_EBIG;
  if (n == 0) return SCS_OK;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= CORE_NA_DEVICES) return SCS_EHIP;
  CoreScratch& S = g_scratch[dev];
  std::lock_guard<std::mutex> lk(S.mu);
  if (!S.words) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return SCS_EHIP;
    S.words = (u32*)p;
  }
  return scs_core_run(d_off, d_adj, n, d_core, S.words, (hipStream_t)stream, 0);
}
