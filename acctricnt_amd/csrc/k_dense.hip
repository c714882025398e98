// Dense sources of the forward path (gfx950, wave64).
//
// The forward path (k_forward.hip) finds every triangle {a < b < c} at its
// middle vertex b: an element a of N(c) ∩ [0, b) that lies in N<(b).  The
// sources with many upper slots, the first ids of a degree-ordered graph
// (dense_sources in fwd_plan.h), hold most of that work, and their ids fit
// 16 bits, so they run on a layout of their own:
//
//   low lists   every vertex c's neighbors below the last dense source, as
//               16-bit ids relative to the graph's first vertex, its list
//               starting at a multiple of 8 ids (16 bytes) and padded with an
//               id that no list of a source holds: a lane loads 8 elements of
//               a probe with one 16-byte load and finds the probe once for
//               the 8;
//   hit rows    one bit per probe element.  Row t of c's matrix belongs to
//               the t-th neighbor b of c, has one bit per element of
//               N(c) ∩ [0, b), t of them, and starts at a byte: the byte a
//               lane has just decided is stored as it is.
//
// A triangle adds one to its three edges' counts.  (b, a) is counted where it
// is found, by the position of a in N<(b), in LDS.  (c, b) and (c, a) are the
// row and column sums of c's hit matrix: k_dense_rows reads every matrix once
// and adds them to c's lower slots, where an update of one 4-byte count per
// triangle by a global atomic took most of the pass before.  The lower slots
// then hold the complete counts and k_combine copies them to the upper
// slots.  Matrices of vertices with more than hit_cap dense neighbors are not
// kept (their size grows with the square), and none where the device has no
// memory left for them; their probes update the counts by atomics.
//
// Measured at R-MAT scale 22 (4.2M vertices, 128M slots, 94% of 7.2e9 probe
// elements at dense sources): counting 4.5 ms + 1.0 ms for the other sources
// and 0.8 ms for the sums, where the other form took 17.1 ms for all; the
// copy to the upper slots 1.25 ms against 2.2 ms for adding both; the whole
// pass 20.0 to 7.6 ms.  The triangle-only pass, 6.1 to 3.3 ms, is bound by the
// lists' traffic (16-bit ids halve it; 17.4 GB fetched), the per-slot counting by VALU (74%
// busy) and LDS (59%); its hit bytes and (b, a) counters cost 0.8 ms each.

#include <hip/hip_runtime.h>

#include <cstddef>

#include <hipcub/hipcub.hpp>

#include "acc_internal.h"
#include "flat_window.h"

namespace {

using accfwd::kChunk;
using accfwd::kWG;
using accfwd::kWaves;

constexpr uint32_t kCtrCap = 2048;    // (b, a) counters in LDS; positions beyond update the slot itself
constexpr uint32_t kRowSmall = 32;    // matrices of at most this many rows: two vertices a wave,
constexpr uint32_t kRowMid = 1024;    // at most this many: one wave each, more: one workgroup each
constexpr int kDenseU = 2;             // rows of 64 groups per round: 16-byte loads in flight per lane
constexpr uint32_t kNoRows = ~0u;     // hit base of a vertex whose matrix is not kept

// Bytes of the rows 0 .. t - 1 of a hit matrix: the sum of ceil(s / 8) over s < t.
__host__ __device__ __forceinline__ uint32_t row_bytes(uint32_t t) {
  if (t == 0) return 0;
  const uint32_t q = (t - 1) >> 3, r = (t - 1) & 7;
  return (q + 1) * (4 * q + r);
}

__device__ __forceinline__ unsigned long long wave_sum_u64(unsigned long long v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

__device__ __forceinline__ uint32_t wave_excl_scan(uint32_t v, int lane) {
  uint32_t x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  return x - v;
}

// Largest k in [0, 64) with X_k <= e, for X nondecreasing over the lanes and X_0 <= e.
__device__ __forceinline__ int lane_search(uint32_t X, uint32_t e) {
  int k = 0;
#pragma unroll
  for (int st = 32; st; st >>= 1)
    if (static_cast<uint32_t>(__shfl(X, k + st)) <= e) k += st;
  return k;
}

// Makes the wave's earlier LDS writes visible to all of its lanes.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

typedef __attribute__((address_space(3))) uint32_t lds_u32;
__device__ __forceinline__ void lds_add(uint32_t *p, uint32_t v) {
  __hip_atomic_fetch_add((lds_u32 *)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void lds_or(uint32_t *p, uint32_t v) {
  __hip_atomic_fetch_or((lds_u32 *)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// ---------------------------------------------------------------- tables
// Per vertex v (of a graph with first vertex base and limit dense sources): the
// number of lower neighbors below base + limit (rows) and the 8-id groups of
// its low list's place: whole 128-byte lines of 8 groups for a list of more than
// 4 (wide), which starts on a line; 4, 2 or 1 groups after all of those for a
// shorter one.  A probe then reads the lines its elements fill and not one
// more (R-MAT scale 22, triangle-only pass: 3.6 to 3.3 ms).
__global__ __launch_bounds__(256) void k_dense_count(const uint32_t *__restrict__ off, const uint32_t *__restrict__ hs,
                                                     const int32_t *__restrict__ adj, uint32_t n,
                                                     const uint32_t *__restrict__ gvoff,
                                                     const uint32_t *__restrict__ glimit, uint32_t graphs,
                                                     uint32_t *__restrict__ rows, uint32_t *__restrict__ wide,
                                                     uint32_t *__restrict__ narrow) {
  for (uint32_t v = blockIdx.x * 256u + threadIdx.x; v <= n; v += gridDim.x * 256u) {
    uint32_t r = 0;
    if (v < n) {
      uint32_t lo = 0, hi = graphs;  // the last graph starting at or before v
      while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (gvoff[mid] <= v) lo = mid; else hi = mid;
      }
      const int32_t end = static_cast<int32_t>(gvoff[lo] + glimit[lo]);
      const uint32_t s = off[v];
      uint32_t a = s, b = hs[v];
      while (a < b) {
        const uint32_t mid = a + ((b - a) >> 1);
        if (adj[mid] < end) a = mid + 1; else b = mid;
      }
      r = a - s;
      rows[v] = r;
    }
    const uint32_t G = (r + 7) >> 3;
    wide[v] = G > 4 ? (G + 7) & ~7u : 0;
    narrow[v] = G > 4 ? 0 : G == 3 ? 4 : G;
  }
}

// The first group of v's low list, from the prefixes of the wide and narrow places.
__device__ __forceinline__ uint32_t low_group(const uint32_t *__restrict__ wide0, const uint32_t *__restrict__ narrow0,
                                              uint32_t v, uint32_t n, uint32_t rows) {
  return rows > 32 ? wide0[v] : wide0[n] + narrow0[v];
}

// What the host needs of the tables: the matrices' total bytes, the lengths
// of the lists of vertices with large and medium matrices, the low groups;
// then the lists' fill counters.
struct DenseSizes {
  unsigned long long bytes;
  uint32_t lists[2];
  uint32_t groups;
  uint32_t filled[2];
};

// 0: a large matrix, 1: a medium one, 2: neither (small, none or not kept).
__device__ __forceinline__ int list_of(uint32_t rows, uint32_t cap) {
  return rows > cap || rows <= kRowSmall ? 2 : rows > kRowMid ? 0 : 1;
}

// Bytes of every vertex's matrix: 0 where it has none (under two rows) or is
// not kept (more than cap rows); and their sum and the lists' lengths, with
// one atomic each per workgroup of a small grid, since atomics on one address
// queue.  wide0 and narrow0 are the finished prefixes of the low groups.
__global__ __launch_bounds__(256) void k_dense_bytes(const uint32_t *__restrict__ rows,
                                                     const uint32_t *__restrict__ wide0,
                                                     const uint32_t *__restrict__ narrow0, uint32_t n, uint32_t cap,
                                                     uint32_t *__restrict__ bytes, DenseSizes *__restrict__ sizes) {
  __shared__ unsigned long long part[4];
  __shared__ uint32_t len[2];
  if (threadIdx.x < 2) len[threadIdx.x] = 0;
  __syncthreads();
  unsigned long long sum = 0;
  for (uint32_t v = blockIdx.x * 256u + threadIdx.x; v <= n; v += gridDim.x * 256u) {
    const uint32_t r = v < n ? rows[v] : 0;
    const uint32_t b = r >= 2 && r <= cap ? row_bytes(r) : 0;
    bytes[v] = b;
    sum += b;
    const int k = list_of(r, cap);
    if (k < 2) lds_add(&len[k], 1);
  }
  sum = wave_sum_u64(sum);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = sum;
  __syncthreads();
  if (threadIdx.x == 0) {
    sum = part[0] + part[1] + part[2] + part[3];
    if (sum) atomicAdd(&sizes->bytes, sum);
    if (blockIdx.x == 0) sizes->groups = wide0[n] + narrow0[n];
  }
  if (threadIdx.x < 2 && len[threadIdx.x]) atomicAdd(&sizes->lists[threadIdx.x], len[threadIdx.x]);
}

// The lists of vertices with large and medium matrices, in no order.  A
// workgroup counts its contiguous share of the vertices first, so that each
// list's length takes one atomic per workgroup (one per vertex queued on the
// two addresses for 3 ms at R-MAT scale 22).
__global__ __launch_bounds__(256) void k_dense_lists(const uint32_t *__restrict__ rows, uint32_t n, uint32_t cap,
                                                     uint32_t *__restrict__ large, uint32_t *__restrict__ mid,
                                                     DenseSizes *__restrict__ sizes) {
  __shared__ uint32_t at[2];
  const uint32_t span = n / gridDim.x + 1;
  const uint32_t lo = min(n, blockIdx.x * span), hi = min(n, lo + span);
  if (threadIdx.x < 2) at[threadIdx.x] = 0;
  __syncthreads();
  for (uint32_t v = lo + threadIdx.x; v < hi; v += 256) {
    const int k = list_of(rows[v], cap);
    if (k < 2) lds_add(&at[k], 1);
  }
  __syncthreads();
  if (threadIdx.x < 2) at[threadIdx.x] = atomicAdd(&sizes->filled[threadIdx.x], at[threadIdx.x]);
  __syncthreads();
  for (uint32_t v = lo + threadIdx.x; v < hi; v += 256) {
    const int k = list_of(rows[v], cap);
    if (k < 2) (k == 0 ? large : mid)[atomicAdd(&at[k], 1u)] = v;
  }
}

// Vertex records {first slot, first low group, hit base, rows} and the low
// lists: a wave takes 64 vertices and lays their groups end to end, each lane
// writing one group of 8 ids.
__global__ __launch_bounds__(256) void k_dense_fill(const uint32_t *__restrict__ off, const int32_t *__restrict__ adj,
                                                    uint32_t n, const uint32_t *__restrict__ gvoff,
                                                    const uint32_t *__restrict__ glimit, uint32_t graphs,
                                                    const uint32_t *__restrict__ rows,
                                                    const uint32_t *__restrict__ wide0,
                                                    const uint32_t *__restrict__ narrow0,
                                                    const uint32_t *__restrict__ byte0, uint32_t cap,
                                                    uint4 *__restrict__ vmeta, uint4 *__restrict__ low) {
  const int lane = threadIdx.x & 63;
  const uint32_t waves = gridDim.x * 4u;
  for (uint32_t v0 = 64 * __builtin_amdgcn_readfirstlane(blockIdx.x * 4u + (threadIdx.x >> 6)); v0 < n;
       v0 += 64 * waves) {
    const uint32_t v = v0 + lane;
    uint32_t o = 0, r = 0, g0 = 0, base = 0, limit = 0;
    if (v < n) {
      uint32_t lo = 0, hi = graphs;
      while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (gvoff[mid] <= v) lo = mid; else hi = mid;
      }
      base = gvoff[lo];
      limit = glimit[lo];
      o = off[v];
      r = rows[v];
      g0 = low_group(wide0, narrow0, v, n, r);
      vmeta[v] = make_uint4(o, g0, r > cap ? kNoRows : byte0[v], r);
    }
    const uint32_t G = wave_excl_scan((r + 7) >> 3, lane);
    const uint32_t total = __builtin_amdgcn_readfirstlane(__shfl(G + ((r + 7) >> 3), 63));
    for (uint32_t e0 = 0; e0 < total; e0 += 64) {
      const uint32_t e = e0 + lane;
      const int k = lane_search(G, e < total ? e : total - 1);
      const uint32_t ko = __shfl(o, k), kr = __shfl(r, k), kG = __shfl(G, k), kg0 = __shfl(g0, k);
      const uint32_t kbase = __shfl(base, k), klimit = __shfl(limit, k);
      if (e < total) {
        const uint32_t i0 = 8 * (e - kG);
        int32_t in[8];  // the array ends with room for the last list's group
        __builtin_memcpy(in, adj + ko + i0, sizeof(in));
        uint32_t w[4];
#pragma unroll
        for (int h = 0; h < 4; h++) {
          uint32_t id[2];
#pragma unroll
          for (int x = 0; x < 2; x++) {
            const uint32_t a = static_cast<uint32_t>(in[2 * h + x]) - kbase;
            id[x] = i0 + 2 * h + x < kr && a < klimit ? a : klimit;  // an id outside reads as padding
          }
          w[h] = id[0] | (id[1] << 16);
        }
        low[kg0 + (e - kG)] = make_uint4(w[0], w[1], w[2], w[3]);
      }
    }
  }
}

// ---------------------------------------------------------------- counting
// LDS of a counting workgroup.  The set of N<(b) is a bitmap over the 16-bit
// ids, at the start of LDS so that an id's word address needs no base: id a is
// bit 31 - (a mod 32) of word a / 32, so that a shift left by a's low five
// bits (which the shift takes by itself) leaves its membership in the sign
// bit and the members above it below.  upto[w] is the number of members in the words
// 0 .. w, so a member's position is upto[w] less the bits left after that shift.
// ctr: the (b, a) counters, dynamic.
struct DenseLds {
  uint32_t set[(1u << 16) / 32];
  uint16_t upto[(1u << 16) / 32];
  uint32_t P[kChunk];   // exclusive prefix of the probes' groups; T beyond the probes
  uint32_t cb[kChunk];  // first low group of each probe less its prefix
  uint32_t hb[kChunk];  // first hit byte of each probe's row less its prefix
  uint32_t wsum[kWaves];
  uint32_t direct;  // some probe's hits are not kept as a row
  uint32_t dbits[kChunk / 32];
  uint32_t pad[3];
  uint32_t ctr[1];
};
constexpr size_t kDenseLdsBytes = offsetof(DenseLds, ctr);
static_assert(kDenseLdsBytes % 16 == 0, "the set is cleared in 16-byte steps, the counters follow aligned");

// Workgroup w runs the units w, w + gridDim.x, ....  A unit is a dense source
// b with at most kChunk of its upper slots (b, c): the workgroup builds the
// set of N<(b), lays the probes' 8-element groups end to end and gives every
// lane one group per row of 64.  The U rows of a round are loaded while the
// round before is decided.
template <int U, bool kSlots>
__global__ __launch_bounds__(kWG, 8) void k_dense(const uint4 *__restrict__ vmeta, const int32_t *__restrict__ adj,
                                                  const uint32_t *__restrict__ rev, const uint4 *__restrict__ low,
                                                  const FwdUnit *__restrict__ units, uint32_t n_units,
                                                  uint32_t set_words, uint32_t ctr_cap, int32_t *__restrict__ cnt,
                                                  uint8_t *__restrict__ hits, unsigned long long *total) {
  extern __shared__ __align__(16) unsigned char dense_lds[];
  DenseLds &S = *reinterpret_cast<DenseLds *>(dense_lds);
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  uint32_t found = 0;
  for (uint32_t t = blockIdx.x; t < n_units; t += gridDim.x) {
    const FwdUnit u = units[t];
    const uint4 mb = vmeta[u.b];  // a dense source's lower list is its low list
    const uint32_t nl = mb.w;
    const uint32_t nup = u.j1 - u.j0;
    if (!kSlots && nl == 0) continue;  // the middle of no triangle (with outputs its rows of zeros are written)
    uint32_t len = 0, cb = 0, hb = 0;
    bool direct = false;
    if (static_cast<uint32_t>(tid) < nup) {
      const int32_t c = adj[u.j0 + tid];
      const uint32_t p = rev[u.j0 + tid];
      const uint4 mc = vmeta[c];
      const uint32_t L = p - mc.x;  // |N(c) ∩ [0, b)|, and the row
      if (L < mc.w) {
        len = (L + 7) >> 3;
        cb = mc.y;
        if (kSlots) {
          direct = !hits || mc.z == kNoRows;
          hb = direct ? 0 : mc.z + row_bytes(L);
        }
      }
    }
    for (uint32_t i = 4 * tid; i < set_words; i += 4 * kWG)
      *reinterpret_cast<uint4 *>(S.set + i) = make_uint4(0, 0, 0, 0);
    const uint32_t nctr = nl < ctr_cap ? nl : ctr_cap;
    if (kSlots) {
      for (uint32_t i = tid; i < nctr; i += kWG) S.ctr[i] = 0;
      if (tid == 0) S.direct = 0;
      if (tid < static_cast<int>(kChunk / 32)) S.dbits[tid] = 0;
    }
    const uint32_t excl = wave_excl_scan(len, lane);
    if (lane == 63) S.wsum[wave] = excl + len;
    __syncthreads();
    uint32_t before = 0, T = 0;
#pragma unroll
    for (int w = 0; w < kWaves; w++) {
      const uint32_t ws = S.wsum[w];
      before += w < wave ? ws : 0;
      T += ws;
    }
    T = __builtin_amdgcn_readfirstlane(T);
    S.P[tid] = static_cast<uint32_t>(tid) < nup ? before + excl : T;
    if (static_cast<uint32_t>(tid) < nup) {
      S.cb[tid] = cb - (before + excl);
      if (kSlots) {
        S.hb[tid] = hb - (before + excl);
        if (direct) {
          S.direct = 1;
          lds_or(&S.dbits[tid >> 5], 1u << (tid & 31));
        }
      }
    }
    const uint16_t *const lb = reinterpret_cast<const uint16_t *>(low + mb.y);
    for (uint32_t i = tid; i < nl; i += kWG) {
      const uint32_t a = lb[i];
      lds_or(&S.set[a >> 5], 0x80000000u >> (a & 31));
      // the list's last id in a word closes the word's count
      if (kSlots && (i + 1 == nl || (static_cast<uint32_t>(lb[i + 1]) >> 5) != (a >> 5)))
        S.upto[a >> 5] = static_cast<uint16_t>(i + 1);
    }
    __syncthreads();
    constexpr uint32_t kStride = kWaves * 64 * U;
    uint32_t e0 = static_cast<uint32_t>(wave) * 64 * U;
    if (e0 < T) {
      struct Round {
        uint4 v[U];
        int k[U];
      };
      // the round at f0, or the last one again past the end
      auto fetch = [&](uint32_t f0, Round &r) {
        const uint32_t f1 = accflat::round_last<U>(f0, T);
        accflat::lds_search<U>(S.P, f0, f1, lane, r.k);
#pragma unroll
        for (int q = 0; q < U; q++) {
          const uint32_t e = f0 + 64 * q + lane;
          r.v[q] = low[S.cb[r.k[q]] + min(e, f1)];  // past T: the round's last group
        }
      };
      const bool wide = __builtin_amdgcn_readfirstlane(nl) > ctr_cap;  // positions beyond the LDS counters
      const bool unit_direct = kSlots && __builtin_amdgcn_readfirstlane(S.direct) != 0;
      auto decide = [&](uint32_t f0, const Round &r) {
#pragma unroll
        for (int q = 0; q < U; q++) {
          const uint32_t e = f0 + 64 * q + lane;
          const uint32_t p[4] = {r.v[q].x, r.v[q].y, r.v[q].z, r.v[q].w};
          uint32_t w[8], x[8];
#pragma unroll
          for (int i = 0; i < 8; i++)
            w[i] = i & 1 ? (p[i >> 1] >> 19) & 0x1ffcu : (p[i >> 1] >> 3) & 0x1ffcu;  // byte address of the word
#pragma unroll
          for (int i = 0; i < 8; i++)
            x[i] = *reinterpret_cast<const uint32_t *>(reinterpret_cast<const unsigned char *>(S.set) + w[i]);
          uint32_t h = 0;  // element i in bit 7 - i
#pragma unroll
          for (int i = 0; i < 8; i++) {
            x[i] <<= (i & 1 ? p[i >> 1] >> 16 : p[i >> 1]) & 31;
            h = __builtin_amdgcn_alignbit(h, x[i], 31);
          }
          if (!kSlots) {
            found += e < T ? __popc(h) : 0;
            continue;
          }
          if (e >= T) continue;
#pragma unroll
          for (int i = 0; i < 8; i++)
            if (static_cast<int32_t>(x[i]) < 0) {
              const uint32_t upto =
                  *reinterpret_cast<const uint16_t *>(reinterpret_cast<const unsigned char *>(S.upto) + (w[i] >> 1));
              const uint32_t pos = upto - __popc(x[i]);
              if (!wide || pos < ctr_cap)
                lds_add(&S.ctr[pos], 1);
              else
                atomicAdd(&cnt[mb.x + pos], 1);
            }
          const int k = r.k[q];
          if (unit_direct && ((S.dbits[k >> 5] >> (k & 31)) & 1u)) {
            // the counts of (c, a) and (c, b) by atomics
            const uint32_t oc = vmeta[adj[u.j0 + k]].x;
            const uint32_t i0 = 8 * (e - S.P[k]);
            for (uint32_t y = h; y; y &= y - 1) atomicAdd(&cnt[oc + i0 + 7 - __builtin_ctz(y)], 1);
            if (h) atomicAdd(&cnt[rev[u.j0 + k]], __popc(h));
          } else {
            hits[S.hb[k] + e] = static_cast<uint8_t>(h);
          }
        }
      };
      // two rounds per turn, so that their registers need no copies
      Round r0, r1;
      fetch(e0, r0);
      for (;;) {
        const uint32_t e1 = e0 + kStride;  // wave-uniform
        if (e1 < T) fetch(e1, r1);
        decide(e0, r0);
        if (e1 >= T) break;
        e0 = e1 + kStride;
        if (e0 < T) fetch(e0, r0);
        decide(e1, r1);
        if (e0 >= T) break;
      }
    }
    __syncthreads();
    if (kSlots) {
      for (uint32_t i = tid; i < nctr; i += kWG) {
        const uint32_t v = S.ctr[i];
        if (v) atomicAdd(&cnt[mb.x + i], static_cast<int>(v));
      }
      __syncthreads();
    }
  }
  if (!kSlots) {
    const unsigned long long w = wave_sum_u64(found);
    if (lane == 0 && w) atomicAdd(total + (blockIdx.x % accfwd::kTriParts) * accfwd::kTriStride, w);
  }
}

// ---------------------------------------------------------------- hit matrices
// Sum over the 2^log lanes of a group (consecutive lanes, log <= 3: a tile's words) in its last lane.
__device__ __forceinline__ uint32_t group_sum(uint32_t x, int log) {
  if (log > 0) x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);   // row_shr:1
  if (log > 1) x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);   // row_shr:2
  if (log > 2) x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);   // row_shr:4
  return x;
}

// Word w (32 columns) of row t of the matrix at H: the row's bytes beyond its
// end, where the next row starts, are masked off.  The matrices' array ends
// with room for the word's overhang.
__device__ __forceinline__ uint32_t row_word(const uint8_t *__restrict__ H, uint32_t t, uint32_t w) {
  const uint32_t nb = (t + 7) >> 3;
  if (4 * w >= nb) return 0;
  uint32_t x;
  __builtin_memcpy(&x, H + row_bytes(t) + 4 * w, 4);
  const uint32_t left = nb - 4 * w;
  return left >= 4 ? x : x & ((1u << (8 * left)) - 1);
}

// Sums of the 32 columns of a word.  Four rows at a time go through
// carry-save adders into a word of ones, one of twos and a carry of fours; the
// carries are counted in the four bytes of eight words, byte j of a[k] for column
// 8 j + 7 - k (element i of a group is bit 7 - i of its byte): 37 instructions
// for four rows, where counting every row in the bytes takes 96.
struct ColumnSums {
  uint32_t ones = 0, twos = 0;
  uint32_t a[8] = {};
  static __device__ __forceinline__ uint32_t carry(uint32_t x, uint32_t y, uint32_t z) { return (x & y) | (z & (x ^ y)); }
  __device__ __forceinline__ void add(const uint32_t (&x)[4]) {
    const uint32_t t0 = carry(x[0], x[1], ones);
    ones ^= x[0] ^ x[1];
    const uint32_t t1 = carry(x[2], x[3], ones);
    ones ^= x[2] ^ x[3];
    const uint32_t f = carry(t0, t1, twos);
    twos ^= t0 ^ t1;
#pragma unroll
    for (int k = 0; k < 8; k++) a[k] += (f >> k) & 0x01010101u;
  }
  // Adds the sums over the lanes of a column (lane mod 2^log) to to[0 .. 31]
  // and starts again.  At most 255 rows in all since the last time, so that the
  // bytes hold the sums; every lane calls it.  (Left to LDS atomics, the lanes of a
  // column queue on one address: the kernel took 1.35 ms.)
  __device__ __forceinline__ void flush(uint32_t *to, int log, bool in, int lane) {
    uint32_t v[8];
#pragma unroll
    for (int k = 0; k < 8; k++) v[k] = 4 * a[k] + 2 * ((twos >> k) & 0x01010101u) + ((ones >> k) & 0x01010101u);
    for (int o = 1 << log; o < 64; o <<= 1)
#pragma unroll
      for (int k = 0; k < 8; k++) v[k] += __shfl_xor(v[k], o, 64);
    if (in && lane < (1 << log)) {
#pragma unroll
      for (int k = 0; k < 8; k++)
#pragma unroll
        for (int j = 0; j < 4; j++) lds_add(&to[8 * j + 7 - k], (v[k] >> (8 * j)) & 255u);
    }
    *this = ColumnSums{};
  }
};

// One large or medium matrix of d rows in tiles of kTileWords words (256
// columns), from the tile's first column down, so that little of the triangle
// above the diagonal is read as nothing: 2^log lanes per row, one word each,
// 64 >> log rows a step, kTurns waves taking turns at the steps.  Row and column sums
// are added to sums[] in LDS.
constexpr uint32_t kTileWords = 8;
static_assert(kTileWords <= 8, "group_sum adds groups of up to 8 lanes");
template <uint32_t kTurns>
__device__ __forceinline__ void sum_matrix(const uint8_t *__restrict__ H, uint32_t d, uint32_t *sums, int wave,
                                           int lane) {
  constexpr int kRows = 4;  // rows in flight per lane
  for (uint32_t col0 = 0; col0 < d; col0 += 32 * kTileWords) {
    const uint32_t words = min(kTileWords, (d - col0 + 31) / 32);
    const int log = words > 1 ? 32 - __builtin_clz(words - 1) : 0;
    const uint32_t rpw = 64u >> log;
    const uint32_t q = lane & ((1u << log) - 1);
    const uint32_t w = col0 / 32 + q;
    const bool last = q == (1u << log) - 1;
    const uint32_t step = kTurns * rpw;
    ColumnSums c;
    uint32_t added = 0;
    // wave-uniform loop; every lane reaches the reductions
    for (uint32_t t0 = col0 + wave * rpw; t0 < d; t0 += kRows * step) {
      uint32_t x[kRows];
#pragma unroll
      for (int r = 0; r < kRows; r++) {
        const uint32_t t = t0 + step * r + (lane >> log);
        x[r] = t < d ? row_word(H, t, w) : 0;
      }
      if (added + kRows * rpw > 255) {
        c.flush(sums + 32 * w, log, 32 * w < d, lane);
        added = 0;
      }
#pragma unroll
      for (int r = 0; r < kRows; r += 2) {
        // two rows' sums (at most 256 each) in one word
        const uint32_t rs = group_sum(__popc(x[r]) | (__popc(x[r + 1]) << 16), log);
        const uint32_t t = t0 + step * r + (lane >> log);
        if (last && (rs & 0xffffu)) lds_add(&sums[t], rs & 0xffffu);
        if (last && (rs >> 16)) lds_add(&sums[t + step], rs >> 16);
      }
      c.add(x);
      added += kRows * rpw;
    }
    c.flush(sums + 32 * w, log, 32 * w < d, lane);
  }
}

// x of the lane whose number differs in the bits of M (within 32 lanes).
template <int M>
__device__ __forceinline__ uint32_t swizzle_xor(uint32_t x) {
  return static_cast<uint32_t>(__builtin_amdgcn_ds_swizzle(static_cast<int>(x), (M << 10) | 0x1f));
}

// The transpose of the 32 x 32 bits held one row per lane by each half of the
// wave (t = lane mod 32): bit p of lane t becomes bit t of lane p.  Step J
// exchanges the off-diagonal J x J blocks of every 2J x 2J block.
template <int J>
__device__ __forceinline__ uint32_t transpose_step(uint32_t x, uint32_t t) {
  constexpr uint32_t kLow = J == 16 ? 0x0000ffffu : J == 8 ? 0x00ff00ffu : J == 4 ? 0x0f0f0f0fu : J == 2 ? 0x33333333u : 0x55555555u;
  const uint32_t y = swizzle_xor<J>(x);
  const bool hi = t & J;
  const uint32_t keep = hi ? ~kLow : kLow;
  const uint32_t moved = __builtin_amdgcn_alignbit(y, y, hi ? J : 32 - J);  // rotated right by J, or left
  return (x & keep) | (moved & ~keep);
}
__device__ __forceinline__ uint32_t transpose32(uint32_t x, uint32_t t) {
  x = transpose_step<16>(x, t);
  x = transpose_step<8>(x, t);
  x = transpose_step<4>(x, t);
  x = transpose_step<2>(x, t);
  return transpose_step<1>(x, t);
}

// Adds the row and column sums of every hit matrix to its vertex's lower
// slots: 0.81 ms for 0.93 GB of matrices at R-MAT scale 22 (1.12 ms with one
// tile of all columns per matrix, four waves to it and every row counted in
// bytes), VALU and the latency of short matrices.  Workgroups [0, n_large) take one large matrix each, the next ones
// four medium matrices each (one per wave; sum_matrix).  The others go over
// all vertices for the small ones, `span` vertices a wave (a power of two up
// to 64): two vertices at a time, lane t of each half holding row t as one
// word; the row sums are popcounts, and the column sums those of the
// transposed matrix.
__global__ __launch_bounds__(256) void k_dense_rows(const uint4 *__restrict__ vmeta, uint32_t n,
                                                    const uint32_t *__restrict__ large, uint32_t n_large,
                                                    const uint32_t *__restrict__ mid_v, uint32_t n_mid,
                                                    uint32_t span, const uint8_t *__restrict__ hits,
                                                    int32_t *__restrict__ cnt) {
  __shared__ uint32_t sums[accdense::kMaxRows];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (blockIdx.x < n_large) {
    const uint4 m = vmeta[large[blockIdx.x]];
    const uint32_t d = __builtin_amdgcn_readfirstlane(m.w);
    for (uint32_t i = threadIdx.x; i < ((d + 31) & ~31u); i += 256) sums[i] = 0;
    __syncthreads();
    sum_matrix<4>(hits + m.z, d, sums, wave, lane);
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < d; i += 256) {
      const uint32_t v = sums[i];
      if (v) cnt[m.x + i] += static_cast<int>(v);
    }
    return;
  }
  const uint32_t blk = blockIdx.x - n_large, mid_blocks = (n_mid + 3) / 4;
  if (blk < mid_blocks) {
    const uint32_t i = __builtin_amdgcn_readfirstlane(blk * 4 + wave);
    if (i >= n_mid) return;
    const uint4 m = vmeta[mid_v[i]];
    const uint32_t d = __builtin_amdgcn_readfirstlane(m.w);
    uint32_t *const own = sums + wave * kRowMid;
    for (uint32_t s = lane; s < ((d + 31) & ~31u); s += 64) own[s] = 0;
    wave_lds_sync();
    sum_matrix<1>(hits + m.z, d, own, 0, lane);
    wave_lds_sync();
    for (uint32_t s = lane; s < d; s += 64) {
      const uint32_t v = own[s];
      if (v) cnt[m.x + s] += static_cast<int>(v);
    }
    return;
  }
  const uint32_t waves = (gridDim.x - n_large - mid_blocks) * 4u;
  const uint32_t t = lane & 31;
  for (uint32_t v0 = span * ((blk - mid_blocks) * 4u + wave); v0 < n; v0 += span * waves) {
    const uint32_t v = v0 + lane;
    uint4 m = make_uint4(0, 0, 0, 0);
    if (static_cast<uint32_t>(lane) < span && v < n) m = vmeta[v];
    unsigned long long todo = __ballot(m.w >= 2 && m.w <= kRowSmall && m.z != kNoRows);
    while (todo) {  // wave-uniform
      const int k0 = __builtin_ctzll(todo);
      todo &= todo - 1;
      const int k1 = todo ? __builtin_ctzll(todo) : k0;
      const bool two = todo != 0;
      todo &= todo - 1;
      const int k = lane < 32 ? k0 : k1;
      const uint32_t o = __shfl(m.x, k), hb = __shfl(m.z, k);
      const uint32_t dk = __shfl(m.w, k);
      const uint32_t d = lane < 32 || two ? dk : 0;
      const uint32_t x = t < d ? row_word(hits + hb, t, 0) : 0;
      const uint32_t c = __popc(x) + swizzle_xor<7>(__popc(transpose32(x, t)));
      if (t < d && c) cnt[o + t] += static_cast<int>(c);
    }
  }
}

unsigned grid_for(uint64_t items, int cus, unsigned per_cu) {
  const uint64_t want = (items + 255) / 256;
  const uint64_t cap = static_cast<uint64_t>(cus > 0 ? cus : 256) * per_cu;
  return static_cast<unsigned>(want < cap ? (want ? want : 1) : cap);
}

}  // namespace

namespace accdense {

void free_tables(acc_graph *g) {
  DensePlan &p = g->dense;
  for (void *q : {static_cast<void *>(p.d_vmeta), static_cast<void *>(p.d_low), static_cast<void *>(p.d_large),
                  static_cast<void *>(p.d_hits)})
    g->ctx->pool.free(q);
  p.d_vmeta = nullptr;
  p.d_low = nullptr;
  p.d_large = nullptr;
  p.d_hits = nullptr;
  g->device_bytes -= p.bytes + p.hits_held;
  p.bytes = p.hits_held = 0;
  p.no_hits = false;
  p.tables = false;
}

int build_tables(acc_graph *g) {
  DensePlan &p = g->dense;
  if (p.tables) return ACC_OK;
  const uint32_t n = g->n, graphs = static_cast<uint32_t>(p.limit.size());
  hipStream_t st = g->ctx->stream;
  const int cus = g->ctx->num_cus;
  const size_t n1 = static_cast<size_t>(n) + 1;
  // scratch: the sizes, rows, wide and narrow places and their prefixes, bytes
  // and their prefix, the graphs' first vertices and limits
  size_t t_scan = 0;
  uint32_t *w = nullptr;
  ACC_HIP_TRY(hipcub::DeviceScan::ExclusiveSum(nullptr, t_scan, w, w, static_cast<int>(n1), st));
  const size_t words = 8 + 6 * n1 + 2 * static_cast<size_t>(graphs);
  const size_t scan_at = (sizeof(uint32_t) * words + 255) / 256 * 256;
  static_assert(sizeof(DenseSizes) <= 8 * sizeof(uint32_t), "the sizes lie before the rows");
  if (g->ctx->pool.alloc(reinterpret_cast<void **>(&w), scan_at + t_scan + 16) != hipSuccess)
    return acc_set_error(ACC_ENOMEM, "hipMalloc of the dense tables' scratch failed");
  auto *const sizes = reinterpret_cast<DenseSizes *>(w);
  uint32_t *const rows = w + 8;
  uint32_t *const wide = rows + n1, *const narrow = wide + n1, *const wide0 = narrow + n1, *const narrow0 = wide0 + n1;
  uint32_t *const byte0 = narrow0 + n1, *const len = wide;  // the places are done with once summed
  uint32_t *const gvoff = byte0 + n1, *const glimit = gvoff + graphs;
  void *const temp = reinterpret_cast<char *>(w) + scan_at;
  auto fail = [&](int rc) {
    (void)hipStreamSynchronize(st);
    g->ctx->pool.free(w);
    free_tables(g);
    return rc;
  };
  auto device = [&](hipError_t err) {
    return fail(acc_set_error(ACC_EDEVICE, std::string("dense tables: ") + hipGetErrorString(err)));
  };
  hipError_t e = hipMemcpyAsync(gvoff, p.first.data(), sizeof(uint32_t) * graphs, hipMemcpyHostToDevice, st);
  if (e == hipSuccess)
    e = hipMemcpyAsync(glimit, p.limit.data(), sizeof(uint32_t) * graphs, hipMemcpyHostToDevice, st);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(k_dense_count, dim3(grid_for(n1, cus, 8)), dim3(256), 0, st, g->d_off, g->d_hs, g->d_adj, n,
                       gvoff, glimit, graphs, rows, wide, narrow);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipcub::DeviceScan::ExclusiveSum(temp, t_scan, wide, wide0, static_cast<int>(n1), st);
  if (e == hipSuccess) e = hipcub::DeviceScan::ExclusiveSum(temp, t_scan, narrow, narrow0, static_cast<int>(n1), st);
  // the largest cap whose matrices stay within the limit
  const uint64_t most = most_hit_bytes(g->m);
  DenseSizes h{};
  p.hit_cap = 2 * kMaxRows;
  do {
    p.hit_cap /= 2;
    if (e == hipSuccess) e = hipMemsetAsync(sizes, 0, sizeof(DenseSizes), st);
    if (e == hipSuccess) {
      hipLaunchKernelGGL(k_dense_bytes, dim3(grid_for(n1, cus, 1)), dim3(256), 0, st, rows, wide0, narrow0, n, p.hit_cap, len,
                         sizes);
      e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpyAsync(&h, sizes, sizeof(h), hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e != hipSuccess) return device(e);
  } while (h.bytes > most);  // a cap of 8 rows stays within it
  p.hit_bytes = h.bytes;
  p.n_large = h.lists[0];
  p.n_mid = h.lists[1];
  const size_t b_meta = sizeof(uint4) * static_cast<size_t>(n), b_low = sizeof(uint4) * (h.groups + size_t(1)),
               b_lists = sizeof(uint32_t) * (static_cast<size_t>(p.n_large) + p.n_mid + 1);
  if (g->ctx->pool.alloc(reinterpret_cast<void **>(&p.d_vmeta), b_meta) != hipSuccess ||
      g->ctx->pool.alloc(reinterpret_cast<void **>(&p.d_low), b_low) != hipSuccess ||
      g->ctx->pool.alloc(reinterpret_cast<void **>(&p.d_large), b_lists) != hipSuccess)
    return fail(acc_set_error(ACC_ENOMEM, "hipMalloc of the dense tables failed"));
  p.d_mid = p.d_large + p.n_large;
  p.bytes = b_meta + b_low + b_lists;
  g->device_bytes += p.bytes;
  e = hipcub::DeviceScan::ExclusiveSum(temp, t_scan, len, byte0, static_cast<int>(n1), st);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(k_dense_fill, dim3(grid_for(static_cast<uint64_t>(n) * 4, cus, 8)), dim3(256), 0, st, g->d_off,
                       g->d_adj, n, gvoff, glimit, graphs, rows, wide0, narrow0, byte0, p.hit_cap, p.d_vmeta, p.d_low);
    e = hipGetLastError();
  }
  if (e == hipSuccess && p.n_large + p.n_mid) {
    hipLaunchKernelGGL(k_dense_lists, dim3(grid_for(n1, cus, 2)), dim3(256), 0, st, rows, n, p.hit_cap, p.d_large,
                       p.d_mid, sizes);
    e = hipGetLastError();
  }
  if (e != hipSuccess) return device(e);
  g->ctx->pool.free(w);  // its next use comes later on the same stream
  p.tables = true;
  return ACC_OK;
}

int ensure(acc_graph *g, bool slots) {
  DensePlan &p = g->dense;
  if (!p.n_units) return ACC_OK;
  ACC_TRY(build_tables(g));
  if (!slots || p.d_hits || p.no_hits) return ACC_OK;
  // a caller who records the stream gets a pass by atomics: nothing is allocated under it
  hipStreamCaptureStatus recording = hipStreamCaptureStatusNone;
  ACC_HIP_TRY(hipStreamIsCapturing(g->ctx->stream, &recording));
  if (recording != hipStreamCaptureStatusNone) return ACC_OK;
  const uint64_t bytes = p.hit_bytes + 16;
  if (g->ctx->pool.alloc(reinterpret_cast<void **>(&p.d_hits), bytes) != hipSuccess) {
    (void)hipGetLastError();
    p.d_hits = nullptr;
    p.no_hits = true;
    return ACC_OK;
  }
  p.hits_held = bytes;
  g->device_bytes += bytes;
  // a share writes only its own sources' rows: the others read as no hits
  return clear_hits(g);
}

int clear_hits(acc_graph *g) {
  DensePlan &p = g->dense;
  if (p.d_hits && p.hit_bytes && (g->shard_lo != 0 || g->shard_hi != g->n))
    ACC_HIP_TRY(hipMemsetAsync(p.d_hits, 0, p.hit_bytes, g->ctx->stream));
  return ACC_OK;
}

template <bool kSlots>
static int launch_t(acc_graph *g, unsigned long long *total) {
  const DensePlan &p = g->dense;
  const uint64_t cap = static_cast<uint64_t>(g->persist) * static_cast<uint64_t>(g->ctx->num_cus);
  const unsigned grid = static_cast<unsigned>(g->persist && cap < p.n_units ? cap : p.n_units);
  const uint32_t words = (p.most / 32 + 4) & ~3u;  // the padding id, most, included
  const uint32_t ctr = kSlots ? std::min(kCtrCap, p.max_low) : 0;
  hipLaunchKernelGGL((k_dense<kDenseU, kSlots>), dim3(grid), dim3(kWG), kDenseLdsBytes + sizeof(uint32_t) * ctr, g->ctx->stream,
                     p.d_vmeta, g->d_adj, g->d_rev, p.d_low, p.d_units, p.n_units, words, ctr, g->d_cnt, p.d_hits,
                     total);
  ACC_HIP_TRY(hipGetLastError());
  return ACC_OK;
}

int launch_count(acc_graph *g) { return g->dense.n_units ? launch_t<true>(g, nullptr) : ACC_OK; }

int launch_triangles(acc_graph *g, unsigned long long *total) {
  return g->dense.n_units ? launch_t<false>(g, total) : ACC_OK;
}

int launch_rows(acc_graph *g) {
  const DensePlan &p = g->dense;
  // few vertices a wave while the graph is too small to give every wave slot
  // of the device 16 (a wave's pairs of vertices run one after another)
  const uint32_t slots = static_cast<uint32_t>(g->ctx->num_cus > 0 ? g->ctx->num_cus : 256) * 32;
  uint32_t span = 2;
  while (span < 16 && static_cast<uint64_t>(span) * slots < g->n) span *= 2;
  const unsigned small = grid_for(static_cast<uint64_t>(g->n) * 64 / span, g->ctx->num_cus, 8);
  hipLaunchKernelGGL(k_dense_rows, dim3(p.n_large + (p.n_mid + 3) / 4 + small), dim3(256), 0, g->ctx->stream,
                     p.d_vmeta, g->n, p.d_large, p.n_large, p.d_mid, p.n_mid, span, p.d_hits, g->d_cnt);
  ACC_HIP_TRY(hipGetLastError());
  return ACC_OK;
}

}  // namespace accdense
