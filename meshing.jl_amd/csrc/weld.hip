// weld.hip -- exact-coordinate vertex welding of a triangle mesh on the
// device: the opt-in step after Marching Cubes, whose cubes each emit their
// own copy of a vertex they share (src/algorithmtypes.jl:17-19).
//
// Two vertices weld when their three coordinates have identical bit
// patterns.  The welded vertices keep their order of first appearance and
// the faces are renumbered (1-based) to them, so the result is what a
// first-appearance `unique` over the vertex tuples gives on the host.
//
//   k_weld_bounds   (large tables only) one block sorts 4096 x coordinates
//                   sampled evenly over the vertices and keeps their
//                   quantiles as the bounds of the table's 64 x regions
//   k_weld_insert   open-addressing hash table over the coordinate bits,
//                   first within each block's 1024 vertices in LDS, then
//                   over the whole mesh for the block's first appearances:
//                   the first vertex of a key claims a slot (CAS from -1),
//                   equal keys then lower it to their smallest index
//                   (atomic min, only when smaller than what the slot
//                   showed), so every slot ends holding the first appearance
//                   of its key; each vertex notes its slot
//   k_weld_rep      per vertex: its key's first appearance (one table load
//                   per local key); per tile of 4096 vertices: its count of
//                   first appearances
//   k_weld_tiles    one block: exclusive prefix of the tile counts, total =
//                   welded count
//   k_weld_pos      exclusive prefix of the first appearances = their new
//                   index (reduce-then-scan: no block waits on another), and
//                   the first appearances themselves to their new slots
//   k_weld_faces    face indices renumbered to the new index of their
//                   vertex's first appearance (out-of-range indices are
//                   counted and left as they are)
//
// The vertex indices in the table, the first appearances and the new indices
// are 32-bit (I = uint32_t) for meshes of up to 2^31 vertices: every pass
// moves half the bytes of these, and a line of the table holds twice the slots.
// 384^3 Float32 value noise mesh against 64-bit indices: k_weld_rep 455 -> 349
// us, prefix and compaction 295 -> 193, the call 2553 -> 2151.
//
// A key's home slot in a large table is its x region's block of slots plus
// the hash's low bits inside it.  Vertices of a mesh are emitted cell by
// cell with x outermost, so the blocks in flight at any moment work in one
// or two of the 64 regions rather than all over the table (on the 272 M
// vertex Marching Cubes mesh of 1024^3 value noise: Float64 7% faster,
// Float32 level; 512 regions and none were slower); the regions come from
// quantiles of the x values, so each takes a like share of the keys whatever
// their distribution, and keys whose x equals several bounds (a plane
// x = const) spread over those regions by the hash.  Placement only changes
// where keys sit: the table still ends holding each key's smallest index,
// and a probe that runs past its region goes on into the next one.
//
// Every probe loop ends: each table has more slots than keys (the global
// one at least 1.25 times the vertices, the local one twice its window),
// slots never return to empty, and a probe stops at an empty slot or at its
// own key.
#include "device.h"

namespace msh {
namespace {

__device__ __forceinline__ uint64_t mix64(uint64_t h) {
  // SplitMix64 finaliser (Steele, Lea, Flood, "Fast splittable
  // pseudorandom number generators", OOPSLA 2014)
  h ^= h >> 30;
  h *= 0xBF58476D1CE4E5B9ull;
  h ^= h >> 27;
  h *= 0x94D049BB133111EBull;
  h ^= h >> 31;
  return h;
}

template <typename W>
__device__ __forceinline__ uint64_t key_hash(W x, W y, W z) {
  uint64_t h = mix64((uint64_t)x + 0x9E3779B97F4A7C15ull);
  h = mix64(h ^ (uint64_t)y);
  return mix64(h ^ (uint64_t)z);
}

__global__ void k_fill_i64(int64_t* __restrict__ p, int64_t n, int64_t v) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// Atomics on table slots (an empty slot holds all ones).
__device__ __forceinline__ uint32_t slot_cas(uint32_t* p, uint32_t want, uint32_t v) {
  return atomicCAS(p, want, v);
}
__device__ __forceinline__ uint64_t slot_cas(uint64_t* p, uint64_t want, uint64_t v) {
  return atomicCAS((unsigned long long*)p, (unsigned long long)want, (unsigned long long)v);
}
__device__ __forceinline__ void slot_min(uint32_t* p, uint32_t v) { atomicMin(p, v); }
__device__ __forceinline__ void slot_min(uint64_t* p, uint64_t v) {
  atomicMin((unsigned long long*)p, (unsigned long long)v);
}

// An IEEE bit pattern as an unsigned integer whose order is the numeric
// order (-0 before +0, NaNs beyond the infinities of their sign).
__device__ __forceinline__ uint64_t ordered(uint32_t b) {
  return (b & 0x80000000u) ? (uint64_t)(uint32_t)~b : (uint64_t)(b | 0x80000000u);
}
__device__ __forceinline__ uint64_t ordered(uint64_t b) {
  return (b >> 63) ? ~b : b | (1ull << 63);
}

constexpr int kWeldSample = 4096;     // x coordinates sorted for the region bounds
constexpr int kWeldRegions = 64;      // regions of a large table (measured: 64 beat 512 and none)
constexpr int kWeldSortBlock = kWeldSample / 4;  // a wave sorts 256 of them by itself

// One block: bounds[r - 1] = the (r / nreg) quantile of the sampled x
// coordinates (as ordered integers), r = 1 .. nreg - 1 (bitonic sort in LDS).
// One block's chain of steps, alone on the device: a step of stride 128 or
// less stays within the 256 values of a wave and needs no barrier of the
// block, which leaves 15 of the 78 (37 us; 60 with a barrier each).
template <typename W>
__global__ __launch_bounds__(kWeldSortBlock) void k_weld_bounds(const W* __restrict__ v,
                                                               int64_t nv, int nreg,
                                                               uint64_t* __restrict__ bounds) {
  __shared__ uint64_t s[kWeldSample];
  for (int k = threadIdx.x; k < kWeldSample; k += kWeldSortBlock)
    s[k] = ordered(v[3 * ((int64_t)k * nv / kWeldSample)]);
  __syncthreads();
  for (int size = 2; size <= kWeldSample; size <<= 1)
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
#pragma unroll
      for (int q = 0; q < 2; ++q) {  // the wave's 128 pairs
        const int i = wave_id() * 2 * kWave + q * kWave + lane_id();
        const int k = 2 * i - (i & (stride - 1)), p = k + stride;
        const uint64_t a = s[k], b = s[p];
        if ((a > b) == ((k & size) == 0)) {  // ascending runs where k & size is 0
          s[k] = b;
          s[p] = a;
        }
      }
      if (stride > 2 * kWave || (stride == 1 && size >= 4 * kWave))
        __syncthreads();
      else
        wave_sync();
    }
  for (int r = threadIdx.x + 1; r < nreg; r += kWeldSortBlock)
    bounds[r - 1] = s[(int64_t)r * kWeldSample / nreg];
}

// Home slot of a key with hash h: region (from x and the nreg - 1 sorted
// bounds in bnd) in the bits from rbits up, the hash's low bits below.
template <typename W>
__device__ __forceinline__ uint64_t home_slot(W x, uint64_t h, const uint64_t* bnd, int nreg,
                                              int rbits) {
  const uint64_t low = h & ((1ull << rbits) - 1);
  if (nreg == 1) return low;
  const uint64_t o = ordered(x);
  int a = 0, b = nreg - 1;  // c = bounds below o
  while (a < b) {
    const int m = (a + b) >> 1;
    if (bnd[m] < o) a = m + 1; else b = m;
  }
  const int c = a;
  uint64_t r = c;
  if (c < nreg - 1 && bnd[c] == o) {  // o is a bound: e = bounds at or below o
    b = nreg - 1;
    while (a < b) {
      const int m = (a + b) >> 1;
      if (bnd[m] <= o) a = m + 1; else b = m;
    }
    r += (h >> 32) % (uint64_t)(a - c + 1);
  }
  return (r << rbits) | low;
}

// Global insert of vertex i with key (x, y, z), probing from slot h:
// returns its slot.
template <typename W, typename I>
__device__ __forceinline__ uint32_t global_insert(const W* __restrict__ v, I i, W x, W y, W z,
                                                  uint64_t h, I* table, uint64_t mask) {
  constexpr I kFree = (I)~(I)0;
  while (true) {
    // a plain load first: a CAS on a taken slot measured slower
    I cur = __hip_atomic_load(&table[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (cur == kFree) {
      cur = slot_cas(&table[h], kFree, i);
      if (cur == kFree) break;  // claimed
    }
    // every index a slot ever holds has the slot's key, so this compare
    // does not depend on which of them it reads
    const W* k = v + 3 * (int64_t)cur;
    if (k[0] == x && k[1] == y && k[2] == z) {
      // a slot only ever decreases: above what it showed, i cannot lower it
      if (i < cur) slot_min(&table[h], i);
      break;
    }
    h = (h + 1) & mask;
  }
  return (uint32_t)h;
}

constexpr int kWeldLT = 1024;          // vertices per block: the local pass's window
constexpr int kWeldLS = 2 * kWeldLT;   // local hash slots
constexpr int kWeldBlock = 512;        // its threads

// Copies of a vertex sit close together in extraction order (the cubes
// around an edge are neighbours in the same or the next cell row), so each
// block first welds its 1024 consecutive vertices in LDS and sends only
// the first appearance of each local key to the global table; each vertex
// notes that local first appearance, whose slot k_weld_rep reads once for
// all of them.  Bound by the latency of the table's loads and atomics, which
// go past the L2s: a longer window sends fewer, a shorter one leaves more
// blocks to overlap theirs.  384^3 Float32 value noise mesh: 512 vertices and
// 256 threads 1149 us, 1024 and 512 1074, 2048 and 512 1144, 2048 and 1024
// 1073 (and k_weld_rep 384 us instead of 357), 4096 and 1024 1354.
template <typename W, typename I>
__global__ __launch_bounds__(kWeldBlock) void k_weld_insert(const W* __restrict__ v, int64_t nv,
                                                        I* table, uint64_t mask,
                                                        const uint64_t* __restrict__ bounds,
                                                        int nreg, int rbits,
                                                        uint32_t* __restrict__ slot,
                                                        uint16_t* __restrict__ lrep) {
  __shared__ W key[3 * kWeldLT];
  __shared__ uint32_t lt[kWeldLS];  // local slot -> smallest local index of its key
  __shared__ uint64_t bnd[kWeldRegions - 1];
  constexpr uint32_t kEmpty = 0xFFFFFFFFu;
  constexpr int PER = kWeldLT / kWeldBlock;
  const int64_t base = (int64_t)blockIdx.x * kWeldLT;
  const int n = nv - base < kWeldLT ? (int)(nv - base) : kWeldLT;
  for (int k = threadIdx.x; k < kWeldLS; k += kWeldBlock) lt[k] = kEmpty;
  for (int k = threadIdx.x; k < nreg - 1; k += kWeldBlock) bnd[k] = bounds[k];
  for (int k = threadIdx.x; k < 3 * n; k += kWeldBlock) key[k] = v[3 * base + k];
  __syncthreads();
  uint32_t ls[PER];
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int j = threadIdx.x + q * kWeldBlock;
    ls[q] = 0;
    if (j >= n) continue;
    const W x = key[3 * j], y = key[3 * j + 1], z = key[3 * j + 2];
    uint32_t h = (uint32_t)key_hash(x, y, z) & (kWeldLS - 1);
    while (true) {
      uint32_t cur = __hip_atomic_load(&lt[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      if (cur == kEmpty) {
        cur = atomicCAS(&lt[h], kEmpty, (uint32_t)j);
        if (cur == kEmpty) break;
      }
      if (key[3 * cur] == x && key[3 * cur + 1] == y && key[3 * cur + 2] == z) {
        if ((uint32_t)j < cur) atomicMin(&lt[h], (uint32_t)j);
        break;
      }
      h = (h + 1) & (kWeldLS - 1);
    }
    ls[q] = h;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int j = threadIdx.x + q * kWeldBlock;
    if (j >= n) continue;
    const uint32_t l = lt[ls[q]];
    lrep[base + j] = (uint16_t)l;
    if (l == (uint32_t)j) {
      const W x = key[3 * j], y = key[3 * j + 1], z = key[3 * j + 2];
      const uint64_t h = home_slot(x, key_hash(x, y, z), bnd, nreg, rbits);
      slot[base + j] = global_insert<W, I>(v, (I)(base + j), x, y, z, h, table, mask);
    }
  }
}

constexpr int kWeldTile = 4096;                 // vertices per prefix tile
constexpr int kWeldPer = kWeldTile / kBlock;     // per thread in k_weld_pos
static_assert(kWeldLT % kWeldBlock == 0 && kWeldTile % kWeldLT == 0 && kWeldLT <= 65536,
              "windows of whole waves inside one prefix tile, 16-bit local indices");

// Same windows as k_weld_insert: the local first appearances read their
// key's smallest index from the table, the others take it from them.
template <typename I>
__global__ __launch_bounds__(kWeldBlock) void k_weld_rep(int64_t nv, const I* __restrict__ table,
                                                     const uint32_t* __restrict__ slot,
                                                     const uint16_t* __restrict__ lrep,
                                                     I* __restrict__ rep,
                                                     uint32_t* __restrict__ tilecnt) {
  __shared__ I res[kWeldLT];
  constexpr int PER = kWeldLT / kWeldBlock;
  const int64_t base = (int64_t)blockIdx.x * kWeldLT;
  const int n = nv - base < kWeldLT ? (int)(nv - base) : kWeldLT;
  uint16_t l[PER];
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int j = threadIdx.x + q * kWeldBlock;
    l[q] = 0;
    if (j < n) {
      l[q] = lrep[base + j];
      if (l[q] == j) res[j] = table[slot[base + j]];
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int j = threadIdx.x + q * kWeldBlock;
    const int64_t i = base + j;
    bool first = false;
    if (j < n) {
      const I r = res[l[q]];  // the smallest index of i's key
      rep[i] = r;
      first = r == (I)i;
    }
    // a wave's 64 vertices here are consecutive and lie in one tile
    const uint64_t b = __ballot(first);
    if (lane_id() == 0 && b != 0) atomicAdd(&tilecnt[i / kWeldTile], (uint32_t)__popcll(b));
  }
}

// Exclusive prefix of the first appearances in three steps: the tile counts (above),
// their prefix in one block (here), then each tile's own (k_weld_pos).
__global__ __launch_bounds__(1024) void k_weld_tiles(const uint32_t* __restrict__ tilecnt,
                                                     int64_t ntiles, int64_t* __restrict__ tileoff,
                                                     int64_t* __restrict__ total) {
  __shared__ int64_t s_w[1024 / kWave];
  const int t = threadIdx.x, lane = lane_id(), wv = t / kWave;
  const int64_t per = (ntiles + 1023) / 1024;
  const int64_t lo = t * per, hi = lo + per < ntiles ? lo + per : ntiles;
  int64_t sum = 0;
  for (int64_t k = lo; k < hi; ++k) sum += tilecnt[k];
  const int64_t incl = (int64_t)wave_incl_scan64((uint64_t)sum);
  if (lane == kWave - 1) s_w[wv] = incl;
  __syncthreads();
  int64_t before = 0;
  for (int q = 0; q < wv; ++q) before += s_w[q];
  int64_t run = before + incl - sum;
  for (int64_t k = lo; k < hi; ++k) {
    tileoff[k] = run;
    run += tilecnt[k];
  }
  if (t == 1023) *total = before + incl;
}

// One tile per block in kWeldPer rounds of 256 consecutive vertices, so
// every load and store of a round is one coalesced stretch.  A first
// appearance goes to its new slot as soon as that is known: a pass of its own
// would read the vertices' new indices again.
template <typename W, typename I>
__global__ __launch_bounds__(kBlock) void k_weld_pos(const W* __restrict__ v,
                                                     const I* __restrict__ rep, int64_t nv,
                                                     const int64_t* __restrict__ tileoff,
                                                     I* __restrict__ pos, W* __restrict__ out) {
  __shared__ uint32_t s_w[kWeldPer][kWaves];
  const int lane = lane_id(), wv = threadIdx.x / kWave;
  const int64_t base = (int64_t)blockIdx.x * kWeldTile + threadIdx.x;
  bool f[kWeldPer];
  uint32_t below[kWeldPer];
#pragma unroll
  for (int q = 0; q < kWeldPer; ++q) {
    const int64_t i = base + q * kBlock;
    f[q] = i < nv && rep[i] == (I)i;
    const uint64_t b = __ballot(f[q]);
    below[q] = lanes_below(b);
    if (lane == 0) s_w[q][wv] = (uint32_t)__popcll(b);
  }
  __syncthreads();
  int64_t run = tileoff[blockIdx.x];
#pragma unroll
  for (int q = 0; q < kWeldPer; ++q) {
    uint32_t before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      before += w < wv ? s_w[q][w] : 0u;
      all += s_w[q][w];
    }
    const int64_t i = base + q * kBlock;
    if (f[q]) {  // (only first appearances are asked for their new index)
      const int64_t o = run + before + below[q];
      pos[i] = (I)o;
      out[3 * o] = v[3 * i];
      out[3 * o + 1] = v[3 * i + 1];
      out[3 * o + 2] = v[3 * i + 2];
    }
    run += all;
  }
}

template <typename I>
__global__ void k_weld_faces(const int64_t* f, int64_t* out, int64_t n,  // (may be the same)
                             const I* __restrict__ rep, const I* __restrict__ pos, int64_t nv,
                             unsigned long long* __restrict__ bad) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  int64_t j = f[k];
  if (j >= 1 && j <= nv)
    j = (int64_t)pos[rep[j - 1]] + 1;  // the new index of the vertex's first appearance
  else
    atomicAdd(bad, 1ull);
  out[k] = j;
}

unsigned grid_of(int64_t n) { return (unsigned)((n + kBlock - 1) / kBlock); }

template <typename W, typename I>
hipError_t weld_t(const WeldArgs& a, hipStream_t st) {
  const W* v = (const W*)a.verts;
  I* table = (I*)a.table;
  I* rep = (I*)a.rep;
  I* pos = (I*)a.pos;
  hipLaunchKernelGGL(k_fill_i64, dim3(1), dim3(kBlock), 0, st, a.bad, (int64_t)1, (int64_t)0);
  if (a.nverts > 0) {
    // (room is whole 256 bytes: the last word may reach past the slots)
    const int64_t words = (a.nslots * (int64_t)sizeof(I) + 7) / 8;
    hipLaunchKernelGGL(k_fill_i64, dim3(grid_of(words)), dim3(kBlock), 0, st, a.table, words,
                       (int64_t)-1);
    const unsigned nwin = (unsigned)((a.nverts + kWeldLT - 1) / kWeldLT);
    // x regions only where the table outgrows the caches (2^23 slots and up)
    int lg = 0;
    while (((int64_t)1 << lg) < a.nslots) ++lg;
    const int nreg = lg >= 23 ? kWeldRegions : 1;
    int rbits = lg;
    for (int r = nreg; r > 1; r >>= 1) --rbits;
    if (nreg > 1)
      hipLaunchKernelGGL((k_weld_bounds<W>), dim3(1), dim3(kWeldSortBlock), 0, st, v, a.nverts,
                         nreg, a.bounds);
    hipLaunchKernelGGL((k_weld_insert<W, I>), dim3(nwin), dim3(kWeldBlock), 0, st, v, a.nverts, table,
                       (uint64_t)(a.nslots - 1), (const uint64_t*)a.bounds, nreg, rbits, a.slot,
                       a.lrep);
    const int64_t ntiles = (a.nverts + kWeldTile - 1) / kWeldTile;
    hipLaunchKernelGGL(k_fill_i64, dim3(grid_of((ntiles + 1) / 2)), dim3(kBlock), 0, st,
                       (int64_t*)a.tilecnt, (ntiles + 1) / 2, (int64_t)0);
    hipLaunchKernelGGL((k_weld_rep<I>), dim3(nwin), dim3(kWeldBlock), 0, st, a.nverts,
                       (const I*)table, (const uint32_t*)a.slot, (const uint16_t*)a.lrep, rep,
                       a.tilecnt);
    hipLaunchKernelGGL(k_weld_tiles, dim3(1), dim3(1024), 0, st, (const uint32_t*)a.tilecnt,
                       ntiles, a.tileoff, a.total);
    hipLaunchKernelGGL((k_weld_pos<W, I>), dim3((unsigned)ntiles), dim3(kBlock), 0, st, v,
                       (const I*)rep, a.nverts, (const int64_t*)a.tileoff, pos, (W*)a.verts_out);
  }
  if (a.nfaces > 0)
    hipLaunchKernelGGL((k_weld_faces<I>), dim3(grid_of(3 * a.nfaces)), dim3(kBlock), 0, st, a.faces,
                       a.faces_out, 3 * a.nfaces, (const I*)rep, (const I*)pos, a.nverts,
                       (unsigned long long*)a.bad);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_weld(const WeldArgs& a, hipStream_t st) {
  const bool narrow = a.index_bytes == 4;
  if (a.out_kind == K_F32)
    return narrow ? weld_t<uint32_t, uint32_t>(a, st) : weld_t<uint32_t, uint64_t>(a, st);
  return narrow ? weld_t<uint64_t, uint32_t>(a, st) : weld_t<uint64_t, uint64_t>(a, st);
}

}  // namespace msh
