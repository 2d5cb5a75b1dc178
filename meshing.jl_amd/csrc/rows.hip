// rows.hip -- the first two passes of the row kernels (see rows.h): the
// sample bits of the whole field, and the vertex and face counts of every
// unit from the bits.  Their scan is the one of the other kernels
// (kernels.hip) over these units.
#include <algorithm>
#include <cmath>

#include "rows.h"

#define MSH_LUT static __constant__
#include "luts.h"

namespace msh {
namespace {

// ---------------------------------------------------------------------------
// Sample bits.  A block takes 64 * E * WX columns along x and PW words along
// a plane's (y, w) order; WX of its waves lie side by side along x, the
// others share the words, each lane making the words of its E neighbouring
// columns from loads of E samples (16 at a time, all in flight at once).  The
// words meet in LDS so that a column's PW words leave together.  Every sample
// is read once and only once: this pass is bound by HBM reads, which reach
// 5.4 to 5.7 TB/s of the 6.8 that a linear read gets here (each load takes 256
// or 512 bytes of a plane).  NT: non-temporal loads.
template <typename T, int E>
struct __attribute__((packed, aligned(sizeof(T)))) Vec {
  T v[E];
};

template <typename T, int E, bool NT>
__device__ __forceinline__ Vec<T, E> load_vec(const char* p) {
  if constexpr (!NT) {
    return *(const Vec<T, E>*)p;
  } else if constexpr (E == 1) {
    return {{__builtin_nontemporal_load((const T*)p)}};
  } else {
    static_assert(E == 2, "one or two samples");
    typedef T T2 __attribute__((ext_vector_type(2), aligned(sizeof(T))));
    const T2 v = __builtin_nontemporal_load((const T2*)p);
    return {{v.x, v.y}};
  }
}

template <typename T, int PW, int E, int WX, bool NT>
__device__ __forceinline__ void bits_tile(const VolArgs& a, int64_t t) {
  constexpr int PPW = PW * WX / kWaves, X = kWave * E * WX, ZB = 16;
  __shared__ uint32_t words[X][PW + 1];
  const Geom g = a.g;
  const T thr = (T)a.thr;
  const int lane = lane_id(), wv = wave_id() / WX, wx = wave_id() % WX;
  const uint32_t nxt = (uint32_t)(g.nx + X - 1) / X;
  const uint32_t tq = (uint32_t)t / nxt;
  const int xb = (int)((uint32_t)t - tq * nxt) * X;
  const uint32_t q0 = tq * PW, nq = (uint32_t)g.ny * (uint32_t)a.sw;
  const uint64_t pbytes = (uint64_t)g.nx * (uint64_t)g.ny * sizeof(T);
  // the lane's columns; at the row's end they move back to end with it (two
  // lanes then make the same words)
  const int xl = min(xb + (wx * kWave + lane) * E, g.nx - E);
  const uint32_t xo = (uint32_t)xl * (uint32_t)sizeof(T);
#pragma unroll 1
  for (int p = 0; p < PPW; ++p) {
    const uint32_t q = q0 + (uint32_t)(wv * PPW + p);
    uint32_t word[E];
#pragma unroll
    for (int e = 0; e < E; ++e) word[e] = 0;
    if (q < nq) {
      const uint32_t y = q / (uint32_t)a.sw, w = q - y * (uint32_t)a.sw;
      const int n = min(32, g.nz - 32 * (int)w);  // samples of this word
      const char* col = (const char*)a.f + (uint64_t)(32 * w) * pbytes +
                        (uint64_t)y * (uint64_t)g.nx * sizeof(T);
#pragma unroll
      for (int zb = 0; zb < 32; zb += ZB) {
        Vec<T, E> v[ZB];
#pragma unroll
        for (int z = 0; z < ZB; ++z)
          v[z] = load_vec<T, E, NT>(col + (uint64_t)min(zb + z, n - 1) * pbytes + xo);
#pragma unroll
        for (int z = 0; z < ZB; ++z)
#pragma unroll
          for (int e = 0; e < E; ++e) word[e] |= v[z].v[e] < thr ? 1u << (zb + z) : 0u;
      }
      if (n < 32)
#pragma unroll
        for (int e = 0; e < E; ++e) word[e] &= (1u << n) - 1u;
    }
#pragma unroll
    for (int e = 0; e < E; ++e)
      if (xl + e >= xb) words[xl + e - xb][wv * PPW + p] = word[e];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < X * PW / kBlock; ++k) {
    const int i = threadIdx.x + k * kBlock;
    const int x = i / PW, p = i % PW;
    if (xb + x < g.nx && q0 + p < nq) a.bits[(int64_t)(xb + x) * a.xs + q0 + p] = words[x][p];
  }
}

// A field of few columns along x leaves most of a tile's lanes on columns that
// others have: its columns are dealt to the lanes along x and y alike, as they
// lie in memory, and a lane makes kNarrowWords words of its column (2, 8, 16 and
// 32 x 2048 x 2048 Float32 124, 128, 147 and 188 us by the tiles above, 10, 24,
// 48 and 125 so; 48 x 1024 x 1024 takes 39 by those), as long as that makes
// blocks enough to fill the device.
constexpr int kNarrow = 32, kNarrowWords = 4;
__host__ __device__ inline int64_t narrow_tiles(const VolArgs& a) {  // 0: not by these
  const int64_t n = ((int64_t)a.g.nx * a.g.ny + kBlock - 1) / kBlock *
                    ((a.sw + kNarrowWords - 1) / kNarrowWords);
  return a.g.nx <= kNarrow && n >= 256 ? n : 0;
}
template <typename T, bool NT>
__device__ __forceinline__ void narrow_tile(const VolArgs& a, int64_t t) {
  const Geom g = a.g;
  const T thr = (T)a.thr;
  // (below 2^31: kMaxBlocks holds ny under 2^26)
  const uint32_t cols = (uint32_t)g.nx * (uint32_t)g.ny, nb = (cols + kBlock - 1) / kBlock;
  const uint32_t tw = (uint32_t)t / nb, c = ((uint32_t)t - tw * nb) * kBlock + threadIdx.x;
  if (c >= cols) return;
  const uint32_t y = c / (uint32_t)g.nx, x = c - y * (uint32_t)g.nx;
  const uint64_t pbytes = (uint64_t)cols * sizeof(T);
  uint32_t* const out = a.bits + (int64_t)x * a.xs + (int64_t)y * a.sw;
#pragma unroll 1
  for (int k = 0; k < kNarrowWords; ++k) {
    const int w = (int)tw * kNarrowWords + k;
    if (w >= a.sw) return;
    const int n = min(32, g.nz - 32 * w);  // samples of this word
    const char* col = (const char*)a.f + (uint64_t)(32 * w) * pbytes + (uint64_t)c * sizeof(T);
    Vec<T, 1> v[32];
#pragma unroll
    for (int z = 0; z < 32; ++z) v[z] = load_vec<T, 1, NT>(col + (uint64_t)min(z, n - 1) * pbytes);
    uint32_t word = 0;
#pragma unroll
    for (int z = 0; z < 32; ++z) word |= v[z].v[0] < thr ? 1u << z : 0u;
    out[w] = n < 32 ? word & ((1u << n) - 1u) : word;
  }
}
template <typename T, bool NT>
__global__ __launch_bounds__(kBlock) void k_bits_narrow(VolArgs a) {
  if (blockIdx.x == 0 && threadIdx.x < 2) a.groups.n[threadIdx.x] = 0;  // for the scan
  narrow_tile<T, NT>(a, blockIdx.x);
}

template <typename T, int PW, int E, int WX, bool NT>
__global__ __launch_bounds__(kBlock) void k_bits(VolArgs a) {
  if (blockIdx.x == 0 && threadIdx.x < 2) a.groups.n[threadIdx.x] = 0;  // for the scan
  bits_tile<T, PW, E, WX, NT>(a, blockIdx.x);
}

// Batched: a block per tile of the launch; the map names its volume.
template <typename T, int PW, int E>
__global__ __launch_bounds__(kBlock) void k_bits_b(const VolArgs* __restrict__ vols,
                                                   const int32_t* __restrict__ bmap, int64_t gbase) {
  const int64_t b = gbase + blockIdx.x;
  const VolArgs a = vols[__builtin_amdgcn_readfirstlane(bmap[b])];
  if (narrow_tiles(a) > 0)
    narrow_tile<T, false>(a, b - a.bblk0);
  else
    bits_tile<T, PW, E, 1, false>(a, b - a.bblk0);
}

// ---------------------------------------------------------------------------
// Counts, from the bits alone.  A wave counts kCountUnits units one after
// another.  Marching Cubes: a cell's vertices are its crossing edges, 12
// population counts of XORed words for 32 cells at once.  Its faces are its
// vertices less 2 for each loop its surface makes, and a cell has one loop
// unless a face of it is ambiguous (its corners alternate around the level)
// or two opposite corners are cut off by themselves: those few cells, found
// by ANDs of the same words, take their further loops from the table.
constexpr int kBatchPW = 8;
constexpr int kCountUnits = 2;  // (1: 32^3 0.6 us faster, 1024^3 30 us slower)
constexpr int kCountTile = kCountUnits * kWaves;

__device__ __forceinline__ uint32_t mc_word_counts(const CellWord& r, const uint8_t* extra) {
  const uint32_t x0 = r.c00.c ^ r.c10.c, x1 = r.c01.c ^ r.c11.c, x2 = r.c00.s ^ r.c10.s,
                 x3 = r.c01.s ^ r.c11.s;  // edges along x at y, y+1, above y, above y+1
  const uint32_t y0 = r.c00.c ^ r.c01.c, y1 = r.c10.c ^ r.c11.c, y2 = r.c00.s ^ r.c01.s,
                 y3 = r.c10.s ^ r.c11.s;  // along y at x, x+1, above x, above x+1
  const uint32_t z0 = r.c00.c ^ r.c00.s, z1 = r.c10.c ^ r.c10.s, z2 = r.c01.c ^ r.c01.s,
                 z3 = r.c11.c ^ r.c11.s;  // along z at (x,y) (x+1,y) (x,y+1) (x+1,y+1)
  const uint32_t m = r.valid;
  const uint32_t act = (x0 | x1 | x2 | x3 | y0 | y1 | y2 | y3 | z0 | z1 | z2 | z3) & m;
  if (__ballot(act != 0) == 0) return 0;
  const uint32_t v = __popc(x0 & m) + __popc(x1 & m) + __popc(x2 & m) + __popc(x3 & m) +
                     __popc(y0 & m) + __popc(y1 & m) + __popc(y2 & m) + __popc(y3 & m) +
                     __popc(z0 & m) + __popc(z1 & m) + __popc(z2 & m) + __popc(z3 & m);
  uint32_t more = (x0 & y1 & x1) | (x2 & y3 & x3) | (x0 & z1 & x2) | (x1 & z3 & x3) |
                  (y0 & z2 & y2) | (y1 & z3 & y3);
  more |= (x0 & y0 & z0) & (x3 & y3 & z3);
  more |= (x0 & y1 & z1) & (x3 & y2 & z2);
  more |= (x1 & y0 & z2) & (x2 & y3 & z1);
  more |= (x1 & y1 & z3) & (x2 & y2 & z0);
  more &= m;
  uint32_t f = v - 2u * __popc(act);
  while (more != 0) {
    const int b = __builtin_ctz(more);
    more &= more - 1;
    f -= extra[cell_case(r, b)];
  }
  return v | (f << 16);
}

// Surface nets: a vertex per active cell, and two faces for each of its
// crossing edges at corner 0 whose four cells exist.
__device__ __forceinline__ uint32_t sn_word_counts(const CellWord& r, bool xin) {
  const uint32_t ym = r.y > 0 ? ~0u : 0u, zm = r.w > 0 ? ~0u : ~1u, xm = xin ? ~0u : 0u;
  const uint32_t m = r.valid;
  const uint32_t q = __popc((r.c00.c ^ r.c10.c) & m & ym & zm) +
                     __popc((r.c00.c ^ r.c01.c) & m & zm & xm) +
                     __popc((r.c00.c ^ r.c00.s) & m & xm & ym);
  return __popc(active_cells(r)) | (q << 17);
}

// Marching Tetrahedra.  Faces: a tetrahedron whose corners differ has one
// where an odd number of them is below the level and two where two are.
// Vertices: crossing edges that the cell owns, the seven that end at its far
// corner and, on the volume's first layers, those whose end corner lies on
// the layer (src/marching_tetrahedra.jl:67-84: the first voxel to request an
// edge owns its vertex).
constexpr int kMtA[19] = {0, 1, 3, 0, 4, 5, 7, 4, 0, 1, 2, 3, 0, 0, 0, 4, 1, 3, 0};
constexpr int kMtB[19] = {1, 2, 2, 3, 5, 6, 6, 7, 4, 5, 6, 7, 2, 7, 5, 6, 6, 6, 6};
constexpr int kMtXyz[8] = {0, 2, 3, 1, 4, 6, 7, 5};  // dx | dy << 1 | dz << 2
constexpr int kMtTets[6][2] = {{2, 1}, {7, 3}, {3, 2}, {1, 5}, {4, 7}, {5, 4}};  // beside 0 and 6

__device__ __forceinline__ uint32_t mt_word_counts(const CellWord& r, bool x0) {
  const uint32_t w[8] = {r.c00.c, r.c01.c, r.c11.c, r.c10.c, r.c00.s, r.c01.s, r.c11.s, r.c10.s};
  const uint32_t m = r.valid;
  if (__ballot(active_cells(r) != 0) == 0) return 0;
  uint32_t f = 0;
  const uint32_t odd06 = w[0] ^ w[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    const uint32_t p = w[kMtTets[k][0]], q = w[kMtTets[k][1]];
    const uint32_t odd = (odd06 ^ p ^ q) & m;
    const uint32_t differ = ((w[0] | w[6] | p | q) & ~(w[0] & w[6] & p & q)) & m;
    f += __popc(odd) + 2u * __popc(differ & ~odd);
  }
  const bool y0 = r.y == 0, z0 = r.w == 0;
  uint32_t v = 0;
#pragma unroll
  for (int e = 0; e < 19; ++e) {
    const int back = 7 & ~kMtXyz[kMtB[e]];  // axes on which the edge's end corner is at 0
    if (back == 0) {
      v += __popc((w[kMtA[e]] ^ w[kMtB[e]]) & m);
    } else if (back == 4) {
      v += z0 ? (w[kMtA[e]] ^ w[kMtB[e]]) & m & 1u : 0u;
    }
  }
  if (__ballot(x0 || y0) != 0) {
#pragma unroll
    for (int e = 0; e < 19; ++e) {
      const int back = 7 & ~kMtXyz[kMtB[e]];
      if (!(back & 3)) continue;
      uint32_t own = (back & 4) ? (z0 ? 1u : 0u) : ~0u;
      if ((back & 1) && !x0) own = 0;
      if ((back & 2) && !y0) own = 0;
      v += __popc((w[kMtA[e]] ^ w[kMtB[e]]) & m & own);
    }
  }
  return v | (f << 16);
}

// The parts of a shared unit (rows.h): cut where the vertices before a word,
// of v in all, pass the next multiple of v / parts.
__device__ __forceinline__ void note_parts(const VolArgs& a, int method, uint32_t u, uint32_t all,
                                           uint32_t before) {
  const uint32_t v = all & 0xFFFF, parts = rows_parts(rows_cuts(method), v);
  if (__builtin_expect(parts == 0, 1)) return;
  const uint32_t lane = (uint32_t)lane_id();
  uint32_t first = 0;  // lane p: part p's first word
  for (uint32_t p = 1; p < parts; ++p) {
    const uint32_t words = (uint32_t)__popcll(__ballot((before & 0xFFFF) * parts < p * v));
    first = lane == p ? words : first;
  }
  const uint32_t pre =
      (uint32_t)__builtin_amdgcn_ds_bpermute((int)(min(first, (uint32_t)kWave - 1u) << 2), (int)before);
  if (lane < parts) a.parts[u].pre[lane] = first < (uint32_t)kWave ? pre : all;
  if (lane < parts) a.parts[u].word[lane] = (uint8_t)first;
}

template <int METHOD>
__device__ __forceinline__ void rows_count_tile(const VolArgs& a, int64_t t, const uint8_t* extra) {
  const int lane = lane_id();
  const uint32_t u0 = (uint32_t)t * kCountTile + (uint32_t)(wave_id() * kCountUnits);
  uint32_t* __restrict__ cnt = a.cnt + a.ubase;
#pragma unroll
  for (int k = 0; k < kCountUnits; ++k) {
    const uint32_t u = u0 + (uint32_t)k;
    if (u >= (uint32_t)a.g.units) return;
    const uint32_t x = u / (uint32_t)a.upx, g = u - x * (uint32_t)a.upx;
    const CellWord r = load_cells(a, (int)x, (int)g, lane);
    uint32_t n = 0;  // vertices | faces << 16
    if constexpr (METHOD == MC) n = mc_word_counts(r, extra);
    if constexpr (METHOD == MT) n = mt_word_counts(r, x == 0);
    if constexpr (METHOD == SN) n = sn_word_counts(r, x > 0);
    const uint32_t incl = wave_scan_dpp(n);
    if (lane == kWave - 1) cnt[u] = incl;
    note_parts(a, METHOD, u, (uint32_t)__builtin_amdgcn_readlane((int)incl, kWave - 1), incl - n);
    if constexpr (METHOD != MC)
      a.wpre[64 * (int64_t)u + lane] = (uint16_t)((incl - n) & 0xFFFF);
  }
}

// Marching Cubes: twice the loops of a case beyond its first
template <int METHOD>
__device__ __forceinline__ void count_table(uint8_t* extra) {
  if constexpr (METHOD == MC) {
    const uint32_t m = nat_to_mc(threadIdx.x);
    const int v = (int)(MC_CASE_VERTS[m] & 0xF), f = (int)(MC_CASE_TRIS[m] & 7);
    extra[threadIdx.x] = (uint8_t)(v > 0 ? v - f - 2 : 0);
    __syncthreads();
  }
}

// The scan of a volume of one scan tile, by the last block to finish its
// counts (the others' counts are visible to it: each block makes its own
// visible to the device before it adds itself to `done`).  Small volumes are
// launches and little else: two launches fewer, 32^3 Float32 sphere call
// 40.5 -> 36.9 us.
template <int METHOD>
__device__ __forceinline__ void scan_tail(const VolArgs& a, const ScanTail& t) {
  __shared__ bool last;
  __shared__ uint64_t s_w[kWaves];
  __syncthreads();
  if (threadIdx.x == 0) {
    __threadfence();
    last = atomicAdd(t.done, 1u) == gridDim.x - 1;
    __threadfence();
  }
  __syncthreads();
  if (!last) return;
  const int units = (int)a.g.units, base = (int)threadIdx.x * kScanItems;
  uint32_t c[kScanItems];
  uint64_t sum = 0;  // vertices | faces << 32
#pragma unroll
  for (int q = 0; q < kScanItems; ++q) {
    c[q] = base + q < units
               ? __hip_atomic_load(&a.cnt[base + q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
               : 0u;
    sum += (uint64_t)(c[q] & 0xFFFF) | ((uint64_t)(c[q] >> 16) << 32);
  }
  const uint64_t incl = wave_incl_scan64(sum);
  __shared__ ShareSums sums;
  const ShareOut share{a.groups, {rows_group_cap(METHOD, 0), rows_group_cap(METHOD, 1)},
                       (uint32_t)rows_emit_waves(METHOD), rows_cuts(METHOD), 0};
  const uint32_t groups = share_count(share, c, &sums);
  if (lane_id() == kWave - 1) s_w[wave_id()] = incl;
  __syncthreads();
  uint64_t before = 0, all = 0;
#pragma unroll
  for (int q = 0; q < kWaves; ++q) {
    before += q < wave_id() ? s_w[q] : 0ull;
    all += s_w[q];
  }
  const uint64_t excl = before + incl - sum;
  int64_t rv = (int64_t)(excl & 0xFFFFFFFFu), rf = (int64_t)(excl >> 32);
#pragma unroll
  for (int q = 0; q < kScanItems; ++q) {
    if (base + q < units) {
      t.voff[base + q] = rv;
      t.foff[base + q] = rf;
    }
    rv += c[q] & 0xFFFF;
    rf += c[q] >> 16;
  }
  const uint32_t shared = share_list(share, base, c, &sums, groups, true);
  if (threadIdx.x == 0) {
    const int64_t nv = (int64_t)(all & 0xFFFFFFFFu), nf = (int64_t)(all >> 32);
    t.totals[0] = 0;
    t.totals[1] = nv;
    t.totals[2] = 0;
    t.totals[3] = nf;
    *t.done = 0;
    t.host[0] = (int64_t)(shared & 0xFFFF) | ((int64_t)(shared >> 16) << 32);
    t.host[1] = nv;
    t.host[3] = nf;
    __threadfence_system();
  }
}

template <int METHOD>
__global__ __launch_bounds__(kBlock) void k_rows_count(VolArgs a, ScanTail tail) {
  __shared__ uint8_t extra[256];
  if (tail.done && blockIdx.x == 0)
    for (int i = threadIdx.x; i < tail.coords.nx + tail.coords.ny + tail.coords.nz; i += kBlock)
      tail.coords.out[i] = coord_at(tail.coords, i);
  count_table<METHOD>(extra);
  rows_count_tile<METHOD>(a, blockIdx.x, extra);
  if (tail.done) scan_tail<METHOD>(a, tail);
}

template <int METHOD>
__global__ __launch_bounds__(kBlock) void k_rows_count_b(const VolArgs* __restrict__ vols,
                                                         const int32_t* __restrict__ cmap,
                                                         int64_t gbase) {
  __shared__ uint8_t extra[256];
  count_table<METHOD>(extra);
  const int64_t b = gbase + blockIdx.x;
  const VolArgs a = vols[__builtin_amdgcn_readfirstlane(cmap[b])];
  rows_count_tile<METHOD>(a, b - a.cblk0, extra);
}

}  // namespace

// ---------------------------------------------------------------------------
// Host side.

bool rows_geom(const Plan& p, Geom* g, RowsGeom* r) {
  if (g->units == 0) return false;
  r->sw = (g->nz + 31) / 32;
  r->cw = (g->nz - 1 + 31) / 32;
  const int64_t words = (int64_t)(g->ny - 1) * r->cw, plane = (int64_t)g->ny * r->sw;
  if (plane >= (1ll << 30)) return false;  // word numbers of an x plane are 32-bit
  // vertices one x plane and one row apart are told apart by 32 bits
  // (a cell owns at most 13)
  if (p.method != MC && (int64_t)(g->ny + 1) * g->nz * (p.method == MT ? 13 : 1) >= (1ll << 31))
    return false;
  // the surface nets emit leaves p + mu (p - p) out for a finite p
  // (rows_sn.hip): every coordinate is finite between ends of this size
  if (p.method == SN)
    for (int k = 0; k < 3; ++k)
      if (!(std::fabs(p.a[k]) <= 0x1p1022 && std::fabs(p.b[k]) <= 0x1p1022)) return false;
  r->upx = (int32_t)((words + 63) / 64);
  r->xs = (plane + 31) / 32 * 32;
  const int64_t units = (int64_t)(g->nx - 1) * r->upx;
  r->blocks = std::max((int64_t)(g->nx + 127) / 128 * ((plane + 3) / 4),
                       (int64_t)(g->nx / 2 + 1) * r->upx);
  if (r->blocks >= kMaxBlocks) return false;
  g->units = units;
  return true;
}

size_t rows_bytes(const Geom& g, const RowsGeom& r) {
  return align256((size_t)g.nx * (size_t)r.xs * 4 + 4);
}

size_t rows_prefix_bytes(const Plan& p, const Geom& g) {
  return align256((size_t)g.units * ((p.method == MC ? 0 : 64 * sizeof(uint16_t)) +
                                     sizeof(RowsParts)));
}

void rows_vol(const RowsGeom& r, void* bits, void* prefixes, VolArgs* a) {
  a->bits = (uint32_t*)bits;
  a->parts = (RowsParts*)prefixes;
  a->wpre = (uint16_t*)(a->parts + a->g.units);
  a->xs = r.xs;
  a->sw = r.sw;
  a->cw = r.cw;
  a->upx = r.upx;
  a->cwm = (uint32_t)std::min<uint64_t>((1ull << 32) / (uint64_t)r.cw, 0xFFFFFFFFull);
  a->cwn = (65536u + (uint32_t)r.cw - 1u) / (uint32_t)r.cw;
  a->cntiles = (a->g.units + kCountTile - 1) / kCountTile;
  // (a batch's tiles are those of a small volume: its volumes fill the device)
  a->bntiles = narrow_tiles(*a);
  if (a->bntiles == 0)
    a->bntiles = (int64_t)((a->g.nx + 2 * kWave - 1) / (2 * kWave)) *
                 (((int64_t)a->g.ny * a->sw + kBatchPW - 1) / kBatchPW);
}

// Units a wave emits one after another: one where a unit alone has cells
// enough to fill the queue's steps, several on sparse fields, whose units
// would each pay the way to the first sample for a few cells (1024^3 Float32
// sphere, 12 vertices a unit: 8 units 158 us, 1 unit 349 us; 1024^3 Float64
// value noise, 520 vertices a unit: 1 unit 5.4 ms, 8 units 6.0 ms), as long
// as the waves fill the device.  One where the vertices are not known yet
// (a batch lays its tiles out before it counts): nverts < 0.
void rows_emit_tiling(VolArgs* a, int64_t nverts) {
  const int64_t waves = rows_emit_waves(a->method), nxb = (a->g.nx - 1 + waves - 1) / waves;
  const int64_t full = a->method == MC ? 256 : 64;  // about 64 cells
  a->ue = 1;
  while (nverts >= 0 && a->ue < kMaxUE && nverts * 2 * a->ue <= full * a->g.units &&
         waves * nxb * ((a->upx + 2 * a->ue - 1) / (2 * a->ue)) >= 32768)
    a->ue *= 2;
  a->ntiles = nxb * ((a->upx + a->ue - 1) / a->ue);
}

template <typename T, int PW, int E, int WX, bool NT>
static void launch_bits_e(const VolArgs& a, hipStream_t st) {
  constexpr int X = kWave * E * WX;
  const int64_t nxt = (a.g.nx + X - 1) / X, nq = (int64_t)a.g.ny * a.sw;
  hipLaunchKernelGGL((k_bits<T, PW, E, WX, NT>), dim3((unsigned)(nxt * ((nq + PW - 1) / PW))),
                     dim3(kBlock), 0, st, a);
}

// A field of up to twice the last-level cache (256 MB) is read through it, so
// that the emit finds samples there: with non-temporal loads the 256^3 Float32
// gyroid's emit takes 50 us instead of 35, and surface nets of 384 x 320 x 448
// Float64 noise (440 MB) 596 us a call instead of 570, although their bits
// take 67 instead of 77; at 512^3 Float32 both are level.  Its tiles have 32
// words of a column, whose 128 bytes leave as a line; 8 where those are too
// few to fill the device (256^3 Float32 11.8 us, 18 with 32), or 4 (32^3 4.2
// us, 5.3 with 8).  A larger field is read past the cache, by waves side by
// side along x where that pads no more than the narrower tile does: 1024^3
// Float32 0.91 -> 0.79 ms (0.82 with the narrower tile), Float64 1.68 -> 1.51
// ms (1.51).
template <typename T>
static void launch_bits_t(const VolArgs& a, hipStream_t st) {
  const bool large = (int64_t)a.g.nx * a.g.ny * a.g.nz * (int64_t)sizeof(T) > (512ll << 20);
  if (narrow_tiles(a) > 0) {
    hipLaunchKernelGGL((large ? k_bits_narrow<T, true> : k_bits_narrow<T, false>),
                       dim3((unsigned)narrow_tiles(a)), dim3(kBlock), 0, st, a);
    return;
  }
  const int64_t nq = (int64_t)a.g.ny * a.sw, x128 = (a.g.nx + 127) / 128, x256 = (a.g.nx + 255) / 256;
  if (large)
    2 * x256 == x128 ? launch_bits_e<T, 32, 1, 4, true>(a, st)
                     : launch_bits_e<T, 32, 2, 1, true>(a, st);
  else if (x128 * ((nq + 31) / 32) >= 2048)
    launch_bits_e<T, 32, 2, 1, false>(a, st);
  else
    x128 * ((nq + 7) / 8) >= 256 ? launch_bits_e<T, 8, 2, 1, false>(a, st)
                                 : launch_bits_e<T, 4, 2, 1, false>(a, st);
}

hipError_t launch_rows_count(const Plan& p, const VolArgs& a, const ScanTail& tail, hipStream_t st) {
  if (a.cntiles == 0) return hipSuccess;
  if (p.T == K_F32)
    launch_bits_t<float>(a, st);
  else
    launch_bits_t<double>(a, st);
  const auto k = p.method == MC ? k_rows_count<MC> : p.method == MT ? k_rows_count<MT> : k_rows_count<SN>;
  hipLaunchKernelGGL(k, dim3((unsigned)a.cntiles), dim3(kBlock), 0, st, a, tail);
  return hipGetLastError();
}

hipError_t launch_rows_bits_batch(int T, const RowsBatch& b, hipStream_t st) {
  const dim3 grid((unsigned)b.nblocks);
  if (T == K_F32)
    hipLaunchKernelGGL((k_bits_b<float, kBatchPW, 2>), grid, dim3(kBlock), 0, st, b.vols, b.map, b.gbase);
  else
    hipLaunchKernelGGL((k_bits_b<double, kBatchPW, 2>), grid, dim3(kBlock), 0, st, b.vols, b.map, b.gbase);
  return hipGetLastError();
}

hipError_t launch_rows_count_batch(int method, const RowsBatch& b, hipStream_t st) {
  const auto k = method == MC ? k_rows_count_b<MC> : method == MT ? k_rows_count_b<MT> : k_rows_count_b<SN>;
  hipLaunchKernelGGL(k, dim3((unsigned)b.nblocks), dim3(kBlock), 0, st, b.vols, b.map, b.gbase);
  return hipGetLastError();
}

hipError_t launch_rows_emit(const Plan& p, int cxclass, const VolArgs& a, const RowsBatch* b,
                            hipStream_t st) {
  if (p.method == MC) return launch_rows_mc(p, cxclass, a, b, st);
  if (p.method == MT) return launch_rows_mt(p, cxclass, a, b, st);
  return launch_rows_sn(p, cxclass, a, b, st);
}

}  // namespace msh
