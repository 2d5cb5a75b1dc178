// rows_mt.hip -- Marching Tetrahedra emit of the row kernels (see rows.h;
// src/marching_tetrahedra.jl:105-163).
//
// As in rows_mc.hip a wave queues the active cells of up to a.ue units from
// the bits, in emission order, and emits a full queue slot-parallel.  A face
// names vertices of its own cell and of the cells at -x, -y and -z (the
// first voxel to request an edge owns its vertex,
// src/marching_tetrahedra.jl:67-84).  Away from the low faces of the volume a
// cell owns the vertices of the seven edges that end at its far corner, so
// the vertices of a word's cells below bit b are seven population counts of
// XORed words, which carry-save adders bring down to three; a cell's own
// first vertex comes from the scan, those of the cells one step back along x
// and y from such counts of their words (and the vertex counts that the count
// pass keeps per word), and those one step back along z are one cell less.
// The 27 sample bits around a cell give the cases of all its owners, and so
// the ranks of its 19 edges among their vertices: a lane works this out for
// one cell of the queue and leaves it in LDS, where a face vertex is one sum.
// Cells whose owners lie on the volume's first layers, which own more edges,
// take these from the constant tables.
//
// Emit, before (halo5.hip) -> now: 256^3 Float32 gyroid 158 -> 90 us, 512^3
// Float32 value noise 2.05 -> 1.55 ms.
// Bound by vector issue (54% of the SIMDs' cycles on the noise, 38% on the
// gyroid) and the latency of each step at 2.8 and 1.6 waves a SIMD on average
// (128 registers and 40 KB of LDS a block would let it hold 4).  A queue of 64
// cells with all 19 edge numbers in LDS, which saves three look-ups a face
// vertex, was slower (100 us, 1.70 ms): a unit is then read about twice as
// often.
#include <type_traits>

#include "rows.h"

#define MSH_LUT static __constant__
#include "luts.h"

namespace msh {
namespace {

constexpr int kCells = 128;  // cells queued at a time, per wave

// The 19 edges of a voxel in the order of src/lut/mt.jl, corners in its order,
// and the corners' coordinates (dx | dy << 1 | dz << 2).
constexpr int kMtA[19] = {0, 1, 3, 0, 4, 5, 7, 4, 0, 1, 2, 3, 0, 0, 0, 4, 1, 3, 0};
constexpr int kMtB[19] = {1, 2, 2, 3, 5, 6, 6, 7, 4, 5, 6, 7, 2, 7, 5, 6, 6, 6, 6};
constexpr int kMtXyz[8] = {0, 2, 3, 1, 4, 6, 7, 5};
// An edge's owner is one cell back along the axes on which its end corner has
// coordinate 0 ..
constexpr int mt_back(int e) { return 7 & ~kMtXyz[kMtB[e]]; }
// .. where the edge ends at the far corner: its place among the seven that do
constexpr int kMtOwned[7] = {5, 6, 10, 15, 16, 17, 18};
constexpr int mt_slot(int e) {
  for (int s = 0; s < 7; ++s)
    if (kMtXyz[kMtA[kMtOwned[s]]] == (kMtXyz[kMtA[e]] | mt_back(e))) return s;
  return 0;
}
constexpr uint64_t mt_backs() {
  uint64_t k = 0;
  for (int e = 0; e < 19; ++e) k |= (uint64_t)mt_back(e) << (3 * e);
  return k;
}

// A cell's case with z fastest: bit 2 j + dz, columns j (x,y) (x+1,y) (x,y+1)
// (x+1,y+1); its Marching Tetrahedra corner order.
__device__ __forceinline__ uint32_t zcase_to_mt(uint32_t c) {
  return (c & 1u) | (((c >> 4) & 1u) << 1) | (((c >> 6) & 1u) << 2) | (((c >> 2) & 1u) << 3) |
         (((c >> 1) & 1u) << 4) | (((c >> 5) & 1u) << 5) | (((c >> 7) & 1u) << 6) |
         (((c >> 3) & 1u) << 7);
}
// vertices of a cell that owns the seven edges at its far corner
__device__ __forceinline__ uint32_t owned7(uint32_t zc) {
  const uint32_t p = __popc(zc);
  return (zc & 0x80u) ? 8u - p : p;
}

struct MtImage {
  uint16_t face[256 * 12];  // edges of each face, 5 bits each
  uint32_t rank7[256];      // rank of each owned edge among the cell's vertices, 4 bits a slot
  uint32_t own7[256];       // edges of the cell's vertices, as slots, 4 bits each
  uint8_t nf[256];          // faces
};
static __device__ __align__(16) MtImage g_mt_image;

__global__ __launch_bounds__(kBlock) void k_mt_image() {
  const uint32_t zc = threadIdx.x, m = zcase_to_mt(zc);
  const int nf = MT_NF[m];
  g_mt_image.nf[zc] = (uint8_t)nf;
  for (int q = 0; q < 12; ++q)
    g_mt_image.face[zc * 12 + q] =
        q < nf ? (uint16_t)(MT_FACE[m * 36 + 3 * q] | (MT_FACE[m * 36 + 3 * q + 1] << 5) |
                            (MT_FACE[m * 36 + 3 * q + 2] << 10))
               : (uint16_t)0;
  uint32_t rank = 0, own = 0;
#pragma unroll
  for (int s = 0; s < 7; ++s) {
    const int e = kMtOwned[s];
    // (class 0: an edge that does not cross has no rank and is not asked for)
    rank |= (uint32_t)(MT_RANK[m * 19 + e] & 15) << (4 * s);
    for (int q = 0; q < (int)MT_NOWN[m]; ++q)
      if (MT_OWN_EDGES[m * 20 + q] == e) own |= (uint32_t)s << (4 * q);
  }
  g_mt_image.rank7[zc] = rank;
  g_mt_image.own7[zc] = own;
}

// A column's word with the samples below and above it: {hi, lo} >> b holds
// samples b - 1, b, b + 1 in its low bits.
struct Col3 {
  uint32_t lo, hi;  // lo: samples -1 .. 30, hi: 31, 32
};
__device__ __forceinline__ Col col_of(const Col3& k) {
  return {__builtin_amdgcn_alignbit(k.hi, k.lo, 1), __builtin_amdgcn_alignbit(k.hi, k.lo, 2)};
}

__device__ __forceinline__ void full_add(uint32_t a, uint32_t b, uint32_t c, uint32_t* s,
                                         uint32_t* carry) {
  *s = a ^ b ^ c;
  *carry = (a & b) | (c & (a ^ b));
}

// Counts of the vertices of a word's cells, bit-sliced: cell b has
// sum over i of ((p[i] >> b) & 1) << i vertices.
struct Planes {
  uint32_t p[5];
};
// first: the cells' class along x and y (bits 0, 1); z0: cell 0 is the
// volume's first along z.  EDGE: the word may have first-layer cells.
template <bool EDGE>
__device__ __forceinline__ Planes owned_planes(const Col& a, const Col& b, const Col& c,
                                               const Col& d, uint32_t first, bool z0) {
  // corners in Marching Tetrahedra order
  const uint32_t w[8] = {a.c, c.c, d.c, b.c, a.s, c.s, d.s, b.s};
  uint32_t m[7];
#pragma unroll
  for (int s = 0; s < 7; ++s) m[s] = w[kMtA[kMtOwned[s]]] ^ w[6];
  Planes r{};
  uint32_t s0, s1, c0, c1, c2;
  full_add(m[0], m[1], m[2], &s0, &c0);
  full_add(m[3], m[4], m[5], &s1, &c1);
  full_add(s0, s1, m[6], &r.p[0], &c2);
  full_add(c0, c1, c2, &r.p[1], &r.p[2]);
  if constexpr (EDGE) {
#pragma unroll
    for (int e = 0; e < 19; ++e) {
      constexpr int none = 0;
      const int back = mt_back(e);
      if (back == none) continue;
      uint32_t own = (back & 4) ? (z0 ? 1u : 0u) : ~0u;
      if ((back & 1) && !(first & 1)) own = 0;
      if ((back & 2) && !(first & 2)) own = 0;
      uint32_t k = (w[kMtA[e]] ^ w[kMtB[e]]) & own;
#pragma unroll
      for (int i = 0; i < 5; ++i) {
        const uint32_t n = r.p[i] & k;
        r.p[i] ^= k;
        k = n;
      }
    }
  }
  return r;
}

template <typename T, typename M, typename A, typename Out, int CXM>
__device__ __forceinline__ void rows_mt_tile(const VolArgs& a, const RowsBlock& blk) {
  constexpr int VW = (kCells * 13 + 64) / 64 + 1, FW = (kCells * 12 + 64) / 64 + 1;
  struct Owners {
    int32_t first[8][64];  // first vertex of the owner one step back along (bits of) the index,
                           // counted from the queue's first
    uint32_t rank[3][64];  // ranks of the cell's edges among their owners' vertices, 4 bits each
  };
  struct Wave {
    union {
      Out v[192];
      Owners own;
    } u;
    int32_t fstage[192];
    uint64_t vbits[VW], fbits[FW];      // slot o starts a cell
    uint32_t list[kCells];              // word of the wave's | bit << 9 | z case << 14 | cells back << 22
                                        // | owners on a first layer << 25
    uint32_t around[kCells];            // the 27 samples around the cell's corner 0
    uint32_t d10[kCells], d01[kCells], d11[kCells];  // how far back the owners' first vertices are
    uint32_t face[kCells];  // cells with faces: cell | z case << 7 | cells back << 15 | first slot << 18
    uint16_t lpv[kCells], lpf[kCells];  // first vertex and face slot
    uint8_t vcell[kCells];  // cells with vertices
  };
  struct Smem {
    MtImage tab;
    uint4 edge[19];  // byte offsets of the edge's corners, then their (dx,dy,dz) | .. << 3
    Wave wave[kWaves];
  };
  __shared__ __align__(16) Smem sm;
  static_assert(sizeof(MtImage) % 16 == 0, "copied in 16-byte words");
  const Geom g = a.g;
  const uint32_t pbytes = (uint32_t)((int64_t)g.nx * g.ny * (int64_t)sizeof(T));
  const uint32_t rbytes = (uint32_t)g.nx * (uint32_t)sizeof(T);
  const int lane = lane_id();
  const RowsWork work = rows_work<MT>(a, blk);
  const int x = work.x, g0 = work.g0, g1 = work.g1;
  const uint32_t cnt = work.cnt;
  // a tile whose units are all empty ends here, before its tables
  if (!__syncthreads_or(cnt != 0)) return;
  for (int q = threadIdx.x; q < (int)(sizeof(MtImage) / 16); q += kBlock)
    ((uint4*)&sm.tab)[q] = ((const uint4*)&g_mt_image)[q];
  if (threadIdx.x < 19) {
    const uint32_t ew = MT_EDGE[threadIdx.x];
    const int ca = ew & 0xF, cb = ew >> 4;
    auto off = [&](int c) {
      return (mt_dz(c) ? pbytes : 0u) + (mt_dy(c) ? rbytes : 0u) +
             (mt_dx(c) ? (uint32_t)sizeof(T) : 0u);
    };
    sm.edge[threadIdx.x] = make_uint4(
        off(ca), off(cb),
        (uint32_t)(mt_dx(ca) | (mt_dy(ca) << 1) | (mt_dz(ca) << 2) | (mt_dx(cb) << 3) |
                   (mt_dy(cb) << 4) | (mt_dz(cb) << 5)), 0u);
  }
  __syncthreads();
  Wave& wm = sm.wave[wave_id()];
  const uint64_t todo = __ballot(cnt != 0);  // bit i: unit g0 + i has outputs
  if (todo == 0) return;
  for (int q = lane; q < VW; q += kWave) wm.vbits[q] = 0;
  for (int q = lane; q < FW; q += kWave) wm.fbits[q] = 0;
  const char* __restrict__ f = (const char*)a.f + (int64_t)x * (int64_t)sizeof(T);
  Out* __restrict__ verts = (Out*)a.verts;
  int64_t* __restrict__ faces = a.faces;
  const M iso = (M)a.iso;
  const A eps = (A)a.eps, ome = (A)a.ome;
  const int cxm = CXM >= 0 ? CXM : a.cxmask;
  const bool cx32 = cxm & 1, cy32 = (cxm >> 1) & 1, cz32 = (cxm >> 2) & 1;
  const double* __restrict__ yp = a.coords + g.nx;
  const double* __restrict__ zp = yp + g.ny;
  const double x0 = a.coords[x], x1 = a.coords[x + 1];
  const WordBase wb = word_base(a, g0);
  int64_t vb, fb;     // the queue's first outputs ..
  uint32_t vph, fph;  // .. beyond a multiple of 64 records
  uint32_t V, F;      // slots of the queue, from that multiple
  int nc = 0, nv = 0, nf = 0;  // its cells, those with vertices, with faces
  auto start = [&](int64_t v, int64_t f) {  // at a unit's outputs
    vb = v;
    fb = f;
    V = vph = (uint32_t)vb & 63u;
    F = fph = (uint32_t)fb & 63u;
  };

  struct Fetch {
    T va, vb;
    Pair<double> y, z;
    uint32_t ends;
  };
  auto emit = [&]() {
    wave_sync();
    int before = 0;
    auto fetch = [&](uint32_t o0, Fetch& r) {
      // (a lane without a vertex reads one of the queue's again)
      const uint32_t o = min(max(o0 + lane, vph), V - 1);
      const uint64_t word = wm.vbits[min(o0, V - 1) >> 6];
      const int ki = o0 >= V ? nv - 1 : before + __popcll(word & (~0ull >> (kWave - 1 - (o & 63)))) - 1;
      before += __popcll(word);
      const int c = wm.vcell[ki];
      const uint32_t e = wm.list[c], q = o - wm.lpv[c], zc = (e >> 14) & 0xFF;
      int y, w;
      word_pos(a, wb, e & 511, &y, &w);
      const uint32_t z = 32u * (uint32_t)w + ((e >> 9) & 31);
      const uint32_t slot = (sm.tab.own7[zc] >> (4 * (q & 7))) & 15;
      uint32_t ed = slot < 2 ? 5 + slot : slot == 2 ? 10u : 12 + slot;  // kMtOwned
      const uint32_t cls = (x == 0 ? 1u : 0u) | (y == 0 ? 2u : 0u) | (z == 0 ? 4u : 0u);
      if (cls != 0) {
        uint32_t own = MT_OWN_EDGES[(cls * 256 + zcase_to_mt(zc)) * 20 + q];
        // used here, so that the wait for this rare load is in the branch:
        // after it, it would stop every step until all loads and stores are back
        asm volatile("" : "+v"(own));
        ed = own;
      }
      const uint4 ew = sm.edge[ed];
      const char* cell = f + (uint64_t)z * pbytes + (uint64_t)(uint32_t)y * rbytes;
      r.va = *(const T*)(cell + ew.x);
      r.vb = *(const T*)(cell + ew.y);
      r.y = *(const Pair<double>*)(yp + y);
      r.z = *(const Pair<double>*)(zp + z);
      r.ends = ew.z;
    };
    auto place = [&](uint32_t o0, const Fetch& r) {
      // vertPos (src/marching_tetrahedra.jl:42-55)
      const uint32_t en = r.ends;
      const M rr = (iso - (M)r.va) / (M)(r.vb - r.va);
      const A aw = jl_min<A>(jl_max<A>((A)rr, eps), ome);
      const A bw = (A)1 - aw;
      const A wx = (A)(en & 1) * bw + (A)((en >> 3) & 1) * aw;
      const A wy = (A)((en >> 1) & 1) * bw + (A)((en >> 4) & 1) * aw;
      const A wz = (A)((en >> 2) & 1) * bw + (A)((en >> 5) & 1) * aw;
      wm.u.v[3 * lane] = (Out)mt_axis<A>(cx32, wx, x0, x1);
      wm.u.v[3 * lane + 1] = (Out)mt_axis<A>(cy32, wy, r.y.a, r.y.b);
      wm.u.v[3 * lane + 2] = (Out)mt_axis<A>(cz32, wz, r.z.a, r.z.b);
      wave_sync();
      store_records(verts + 3 * (vb - (int64_t)vph + (int64_t)o0), wm.u.v,
                    o0 == 0 ? (int)vph : 0, (int)V - (int)o0);
      wave_sync();
    };
    if (nv > 0) {
      Fetch p, q;
      fetch(0, p);
      for (uint32_t o0 = 0; o0 < V; o0 += 2 * kWave) {
        fetch(o0 + kWave, q);
        place(o0, p);
        fetch(o0 + 2 * kWave, p);
        place(o0 + kWave, q);
      }
    }
    // faces, 64 cells at a time
    before = 0;
    for (int c0 = 0; c0 < nc; c0 += kWave) {
      {
        const int c = min(c0 + lane, nc - 1);
        const uint32_t e = wm.list[c], n = wm.around[c];
        const uint32_t nb = (e >> 22) & 7;
        const int32_t s0 = (int32_t)wm.lpv[c] - (int32_t)vph;
        // z case of the cell one step back along the bits of d
        auto zcase = [&](int d) -> uint32_t {
          const int i = 3 * (3 * (1 - (d & 1)) + (1 - ((d >> 1) & 1))) + (1 - (d >> 2));
          return ((n >> i) & 3u) | (((n >> (i + 9)) & 3u) << 2) | (((n >> (i + 3)) & 3u) << 4) |
                 (((n >> (i + 12)) & 3u) << 6);
        };
        int32_t s[8];
        s[0] = s0;
        s[1] = s0 - (int32_t)wm.d10[c];
        s[2] = s0 - (int32_t)wm.d01[c];
        s[3] = s0 - (int32_t)wm.d11[c];
        uint32_t rank[3] = {0, 0, 0};
        uint32_t back[4];  // vertices of the cells one step back along z
        {
          uint32_t r7[8];
#pragma unroll
          for (int d = 0; d < 8; ++d) {
            const uint32_t zc = zcase(d);
            r7[d] = sm.tab.rank7[zc];
            if (d >= 4) back[d - 4] = owned7(zc);
          }
#pragma unroll
          for (int ed = 0; ed < 19; ++ed)
            rank[ed >> 3] |= ((r7[mt_back(ed)] >> (4 * mt_slot(ed))) & 15u) << (4 * (ed & 7));
        }
        if (__ballot((e >> 25) & 1) != 0) {
          // owners on a first layer: their classes' tables
          int y, w;
          word_pos(a, wb, e & 511, &y, &w);
          const int z = 32 * w + (int)((e >> 9) & 31);
          if ((e >> 25) & 1) {
            rank[0] = rank[1] = rank[2] = 0;
            auto cls = [&](uint32_t d) -> uint32_t {
              return (x - (int)(d & 1) == 0 ? 1u : 0u) | (y - (int)((d >> 1) & 1) == 0 ? 2u : 0u) |
                     (z - (int)(d >> 2) == 0 ? 4u : 0u);
            };
#pragma unroll 1
            for (uint32_t ed = 0; ed < 19; ++ed) {
              const uint32_t d = (uint32_t)(mt_backs() >> (3 * ed)) & 7u & nb;
              const uint32_t zc = zcase((int)d), m = zcase_to_mt(zc);
              const uint32_t e2 = MT_SHIFT[ed * 8 + d];
              rank[ed >> 3] |= (uint32_t)(MT_RANK[(cls(d) * 256 + m) * 19 + e2] & 15)
                               << (4 * (ed & 7));
            }
#pragma unroll
            for (uint32_t d = 4; d < 8; ++d)
              if ((d & nb) == d) back[d - 4] = MT_NOWN[cls(d) * 256 + zcase_to_mt(zcase((int)d))];
          }
        }
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          wm.u.own.first[d][lane] = s[d];
          wm.u.own.first[d + 4][lane] = s[d] - (int32_t)back[d];
        }
#pragma unroll
        for (int i = 0; i < 3; ++i) wm.u.own.rank[i][lane] = rank[i];
        wave_sync();
      }
      const uint32_t F0 = wm.lpf[c0], F1 = c0 + kWave < nc ? wm.lpf[c0 + kWave] : F;
      for (uint32_t o0 = F0 & ~63u; o0 < F1; o0 += kWave) {
        const uint32_t o = o0 + lane;
        const uint64_t word = wm.fbits[o0 >> 6];
        const int k = before + __popcll(word & (~0ull >> (kWave - 1 - lane))) - 1;
        if (o >= F0 && o < F1) {
          const uint32_t e = wm.face[k];
          const uint32_t fw = sm.tab.face[((e >> 7) & 0xFF) * 12 + (o - (e >> 18))];
          const uint32_t nb = (e >> 15) & 7;
          const int l = (int)(e & 63);
#pragma unroll
          for (int m = 0; m < 3; ++m) {
            const uint32_t ed = (fw >> (5 * m)) & 31;
            const uint32_t d = (uint32_t)(mt_backs() >> (3 * ed)) & nb;
            wm.fstage[3 * lane + m] = wm.u.own.first[d][l] +
                                      (int32_t)((wm.u.own.rank[ed >> 3][l] >> (4 * (ed & 7))) & 15u);
          }
        }
        wave_sync();
        const int64_t first = vb + 1;
        store_records(faces + 3 * (fb - (int64_t)fph + (int64_t)o0), wm.fstage, (int)F0 - (int)o0,
                      (int)F1 - (int)o0, [first](int32_t v) { return first + (int64_t)v; });
        wave_sync();
        if (o0 + kWave <= F1) before += __popcll(word);  // (the next cells start in this word)
      }
    }
    for (uint32_t q = lane; q < (V + 63) / 64; q += kWave) wm.vbits[q] = 0;
    for (uint32_t q = lane; q < (F + 63) / 64; q += kWave) wm.fbits[q] = 0;
    wave_sync();
    vb += (int64_t)(V - vph);
    fb += (int64_t)(F - fph);
    vph = (uint32_t)vb & 63u;
    fph = (uint32_t)fb & 63u;
    V = vph;
    F = fph;
    nc = nv = nf = 0;
  };

  int gi = g0 + __builtin_ctzll(todo), done = 0;  // `done` cells of unit gi are through ..
  uint32_t udone = work.vpre;                     // .. with this many vertices
  start(readlane64(work.voff, gi - g0) + (int64_t)work.vpre,
        readlane64(work.foff, gi - g0) + (int64_t)work.fpre);
#pragma unroll 1
  while (gi < g1) {
    bool gap = false;  // before the next unit
    {
      int y, w;
      word_pos(a, word_base(a, gi), (uint32_t)lane, &y, &w);
      const bool ok = y < g.ny - 1;
      const int left = g.nz - 1 - 32 * w;
      const uint32_t valid = !ok ? 0u : left >= 32 ? ~0u : (1u << left) - 1u;
      // the nine columns around the word, (x-1 .. x+1) by (y-1 .. y+1)
      Col3 k[9];
      {
        const uint32_t* __restrict__ p = a.bits + (int64_t)x * a.xs;
        const uint32_t i = (uint32_t)y * (uint32_t)a.sw + (uint32_t)w;
#pragma unroll
        for (int cx = 0; cx < 3; ++cx)
#pragma unroll
          for (int cy = 0; cy < 3; ++cy) {
            Col3 r{0, 0};
            if (ok && (cx > 0 || x > 0) && (cy > 0 || y > 0)) {
              const uint32_t* __restrict__ q = p + (int64_t)(cx - 1) * a.xs;
              const uint32_t j = i + (uint32_t)(cy - 1) * (uint32_t)a.sw;
              const uint32_t c = q[j], n = q[j + 1], m = w > 0 ? q[j - 1] : 0u;
              r.lo = __builtin_amdgcn_alignbit(c, m, 31);
              r.hi = (c >> 31) | ((n & 1u) << 1);
            }
            k[3 * cx + cy] = r;
          }
      }
      const Col c00 = col_of(k[4]), c10 = col_of(k[7]), c01 = col_of(k[5]), c11 = col_of(k[8]);
      const uint32_t act = work.has(lane) ? active_of(c00, c10, c01, c11, valid) : 0u;
      uint32_t above = 0;
#pragma unroll
      for (int i = 0; i < 9; ++i) above |= k[i].hi << (2 * i);
      const uint32_t incl = wave_scan_dpp(__popc(act));
      const int total = __builtin_amdgcn_readlane((int)incl, kWave - 1);
      // the words at -x, -y and both: how far back their first vertices are
      // from this word's, and their cells' vertices
      uint32_t w10 = 0, w01 = 0, w11 = 0, pre = 0;
      {
        const uint32_t q = (uint32_t)gi * 64u + (uint32_t)lane, cw = (uint32_t)a.cw;
        // (read from its lane before the branch: that lane may not take it)
        const int64_t unit = readlane64(work.voff, gi - g0) + a.sz[0];
        if (act != 0) {
          pre = a.wpre[64 * ((int64_t)x * a.upx + gi) + lane];
          const int64_t mine = unit + (int64_t)pre;
          if (x > 0) w10 = (uint32_t)(mine - word_vertex(a, x - 1, q));
          if (y > 0) w01 = (uint32_t)(mine - word_vertex(a, x, q - cw));
          if (x > 0 && y > 0) w11 = (uint32_t)(mine - word_vertex(a, x - 1, q - cw));
        }
      }
      Planes p10, p01, p11;
      const Col m0 = col_of(k[0]), m1 = col_of(k[1]), m2 = col_of(k[2]), m3 = col_of(k[3]),
                m6 = col_of(k[6]);
      const bool edge = __ballot(act != 0 && (x < 2 || y < 2)) != 0;
      uint32_t ex = 0;  // vertices that cell 0 owns beyond its class as the first along z
      if (edge) {
        const uint32_t fx0 = x == 1 ? 1u : 0u, fx = x == 0 ? 1u : 0u;
        const uint32_t fy0 = y == 1 ? 2u : 0u, fy = y == 0 ? 2u : 0u;
        p10 = owned_planes<true>(m1, c00, m2, c01, fx0 | fy, w == 0);
        p01 = owned_planes<true>(m3, m6, c00, c10, fx | fy0, w == 0);
        p11 = owned_planes<true>(m0, m3, m1, c00, fx0 | fy0, w == 0);
      } else {
        p10 = owned_planes<false>(m1, c00, m2, c01, 0, false);
        p01 = owned_planes<false>(m3, m6, c00, c10, 0, false);
        p11 = owned_planes<false>(m0, m3, m1, c00, 0, false);
        if (w == 0) {
          // the three edges of the cell's own level that end at (1, 1, 0)
          auto three = [](const Col& a, const Col& b, const Col& c, const Col& d) {
            return ((a.c ^ d.c) & 1u) + ((b.c ^ d.c) & 1u) + ((c.c ^ d.c) & 1u);
          };
          ex = three(m1, c00, m2, c01) | (three(m3, m6, c00, c10) << 8) |
               (three(m0, m3, m1, c00) << 16);
        }
      }
      while (done < total && nc < kCells) {
        const int take = min(min(kCells - nc, kWave), total - done);
        const bool in = lane < take;
        int L, b;
        listed_cell(act, incl, done, take, wm.list + nc, &L, &b);
        auto from = [&](uint32_t v) { return (uint32_t)__builtin_amdgcn_ds_bpermute(L << 2, (int)v); };
        const uint32_t hi = from(above), lowm = (1u << b) - 1u;
        uint32_t n27 = 0;
#pragma unroll
        for (int i = 0; i < 9; ++i)
          n27 |= (__builtin_amdgcn_alignbit((hi >> (2 * i)) & 3u, from(k[i].lo), (uint32_t)b) & 7u) << (3 * i);
        const uint32_t zc = ((n27 >> 13) & 3u) | (((n27 >> 22) & 3u) << 2) |
                            (((n27 >> 16) & 3u) << 4) | (((n27 >> 25) & 3u) << 6);
        const int cy = (int)from((uint32_t)y), cw = (int)from((uint32_t)w);
        const int cz = 32 * cw + b;
        const uint32_t cls = (x == 0 ? 1u : 0u) | (cy == 0 ? 2u : 0u) | (cz == 0 ? 4u : 0u);
        uint32_t cv = owned7(zc);
        if (in && cls != 0) cv = MT_NOWN[cls * 256 + zcase_to_mt(zc)];
        const uint32_t cf = sm.tab.nf[zc];
        const uint32_t pk = in ? cv | (cf << 16) : 0u;
        const uint32_t inc = wave_scan_dpp(pk);
        const uint32_t sv = V + ((inc - pk) & 0xFFFF), sf = F + ((inc - pk) >> 16);
        // vertices of the word's cells below this one, and of the words back
        const uint32_t mine = udone + ((inc - pk) & 0xFFFF) - from(pre);
        auto below = [&](const Planes& p) {
          uint32_t s = __popc(from(p.p[0]) & lowm) + 2u * __popc(from(p.p[1]) & lowm) +
                       4u * __popc(from(p.p[2]) & lowm);
          if (edge) s += 8u * __popc(from(p.p[3]) & lowm) + 16u * __popc(from(p.p[4]) & lowm);
          return s;
        };
        const uint32_t exl = from(ex);  // (every lane reads: no branch around it)
        const uint32_t xx = b > 0 ? exl : 0u;
        const uint32_t d10 = from(w10) + mine - below(p10) - (xx & 0xFF);
        const uint32_t d01 = from(w01) + mine - below(p01) - ((xx >> 8) & 0xFF);
        const uint32_t d11 = from(w11) + mine - below(p11) - ((xx >> 16) & 0xFF);
        const uint64_t withv = __ballot((pk & 0xFFFF) != 0), withf = __ballot((pk >> 16) != 0);
        if (in) {
          const uint32_t nb = (x > 0 ? 1u : 0u) | (cy > 0 ? 2u : 0u) | (cz > 0 ? 4u : 0u);
          const uint32_t near = (x < 2 || cy < 2 || cz < 2) ? 1u : 0u;
          const int c = nc + lane;
          wm.list[c] = ((uint32_t)L + 64u * (uint32_t)(gi - g0)) | ((uint32_t)b << 9) | (zc << 14) | (nb << 22) |
                       (near << 25);
          wm.around[c] = n27;
          wm.d10[c] = d10;
          wm.d01[c] = d01;
          wm.d11[c] = d11;
          wm.lpv[c] = (uint16_t)sv;
          wm.lpf[c] = (uint16_t)sf;
          if (pk & 0xFFFF) {
            wm.vcell[nv + (int)lanes_below(withv)] = (uint8_t)c;
            atomicOr((unsigned long long*)&wm.vbits[sv >> 6], 1ull << (sv & 63));
          }
          if (pk >> 16) {
            wm.face[nf + (int)lanes_below(withf)] = (uint32_t)c | (zc << 7) | (nb << 15) | (sf << 18);
            atomicOr((unsigned long long*)&wm.fbits[sf >> 6], 1ull << (sf & 63));
          }
        }
        const uint32_t sum = (uint32_t)__builtin_amdgcn_readlane((int)inc, kWave - 1);
        V += sum & 0xFFFF;
        F += sum >> 16;
        udone += sum & 0xFFFF;
        nv += __popcll(withv);
        nf += __popcll(withf);
        nc += take;
        done += take;
      }
      if (done >= total) {  // the next unit with outputs
        const uint64_t rest = (todo >> (gi - g0)) & ~1ull;
        const int gn = rest ? gi + __builtin_ctzll(rest) : g1;
        gap = gn < g1 && work.gap(gi - g0, gn - g0);
        gi = gn;
        done = 0;
        udone = 0;
      }
    }
    if (nc == kCells || ((gi == g1 || gap) && nc > 0)) emit();
    if (gap) {
      int64_t v, f;
      work.unit_offsets(a, gi - g0, &v, &f);
      start(v, f);
    }
  }
}

template <typename T, typename M, typename A, typename Out, int CXM>
__global__ __launch_bounds__(kBlock, 4) void k_rows_mt(VolArgs a) {
  const RowsBlock b = rows_block(a);
  if (!b.none) rows_mt_tile<T, M, A, Out, CXM>(a, b);
}

// Batched: a block per group or tile of the launch.
template <typename T, typename M, typename A, typename Out, int CXM>
__global__ __launch_bounds__(kBlock, 4) void k_rows_mt_b(const VolArgs* __restrict__ vols,
    const int32_t* __restrict__ emap, int64_t gbase, const RowsGroup* __restrict__ groups,
    const uint32_t* __restrict__ ngroups, int32_t xblocks) {
  RowsBlock b = rows_block(emap, gbase, groups, ngroups, xblocks);
  if (b.none) return;
  const VolArgs a = batch_volume(vols, b.vol);
  b.tile -= a.eblk0;
  rows_mt_tile<T, M, A, Out, CXM>(a, b);
}

}  // namespace

// ---------------------------------------------------------------------------
// Host side.

hipError_t launch_mt_image(hipStream_t st) {
  hipLaunchKernelGGL(k_mt_image, dim3(1), dim3(kBlock), 0, st);
  return hipGetLastError();
}

template <typename T, typename M, typename A, typename Out, int CXM>
static hipError_t rows_mt_cx(const VolArgs& a, const RowsBatch* b, hipStream_t st) {
  if (b)
    hipLaunchKernelGGL((k_rows_mt_b<T, M, A, Out, CXM>), dim3((unsigned)(b->xblocks + b->nblocks)),
                       dim3(kBlock), 0, st, b->vols, b->map, b->gbase, b->groups,
                       b->ngroups, b->xblocks);
  else
    hipLaunchKernelGGL((k_rows_mt<T, M, A, Out, CXM>), dim3((unsigned)(a.xblocks + a.ntiles)),
                       dim3(kBlock), 0, st, a);
  return hipGetLastError();
}

template <typename T, typename M, typename A, typename Out>
static hipError_t rows_mt_t(int cxclass, const VolArgs& a, const RowsBatch* b, hipStream_t st) {
  switch (cxclass) {
    case 1: return rows_mt_cx<T, M, A, Out, 0>(a, b, st);
    case 2: return rows_mt_cx<T, M, A, Out, 7>(a, b, st);
    default: return rows_mt_cx<T, M, A, Out, -1>(a, b, st);
  }
}

hipError_t launch_rows_mt(const Plan& p, int cxclass, const VolArgs& a, const RowsBatch* b,
                          hipStream_t st) {
  if ((b ? b->nblocks : a.ntiles) == 0) return hipSuccess;
  if (p.T == K_F32 && p.M == K_F32 && p.A == K_F32 && p.Out == K_F32)
    return rows_mt_t<float, float, float, float>(cxclass, a, b, st);
  if (p.T == K_F32 && p.M == K_F32 && p.A == K_F32) return rows_mt_t<float, float, float, double>(cxclass, a, b, st);
  if (p.T == K_F32 && p.M == K_F32) return rows_mt_t<float, float, double, double>(cxclass, a, b, st);
  if (p.T == K_F32) return rows_mt_t<float, double, double, double>(cxclass, a, b, st);
  return rows_mt_t<double, double, double, double>(cxclass, a, b, st);
}

}  // namespace msh
