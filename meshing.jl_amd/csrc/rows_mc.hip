// rows_mc.hip -- Marching Cubes emit of the row kernels (see rows.h;
// src/marching_cubes.jl:27-92).
//
// A wave emits up to a.ue consecutive units, whose outputs are one run of each
// array.  The active cells come from the bits (no sample is read to classify)
// and are queued in emission order across the units; lane k of a step looks
// cell k's counts up and a wave scan places them.  A full queue (and the last
// one) is emitted slot-parallel: lane o takes vertex slot o (and face slot
// o), finds its cell from a bitmap of the slots at which a cell starts, and
// reads the two samples of its edge from the field.  Slots are numbered so
// that slot 0 of a step of 64 falls on a multiple of 64 records of the
// output: a step stages its records in LDS and writes whole lines.
//
// The kernel with lanes along x (mc5.hip) gives every open row a few dozen
// bytes per z chunk, about two writes a line, and classifies every cell twice
// over; here a unit's run is kilobytes long and the empty cells cost one AND
// of words for 32 of them.  Emit, before -> now: 256^3 Float32 gyroid 80 ->
// 35 us, 301 x 217 x 389 Float32 value noise (rows not 16-byte aligned) 449
// -> 160 us, 1024^3 Float64 value noise 7.0 -> 4.8 ms.  The last reads 5.1 GB
// and writes 9.8 GB, 2.9 ms at the rate of a copy; the rest is the wait of
// the gathers (the two samples and two pairs of coordinates of 64 vertices
// that lie on dozens of lines) for their turn in the address unit, at 4
// waves a SIMD.  Blocks of 8 and 16 waves, whose planes share the lines, were
// slower (5.1 and 5.2 ms): a block then lasts as long as its slowest wave.
#include <type_traits>

#include "rows.h"

#define MSH_LUT static __constant__
#include "luts.h"

namespace msh {
namespace {

constexpr int kCells = 256;  // cells queued at a time, per wave

struct McImage {
  uint64_t lv[256], lt[256];  // MC_CASE_VERTS and MC_CASE_TRIS by natural case
  uint32_t cnt[256];          // vertices | faces << 16
};
static __device__ __align__(16) McImage g_mc_image;

__global__ __launch_bounds__(kBlock) void k_mc_image() {
  const uint32_t c = threadIdx.x, m = nat_to_mc(c);
  g_mc_image.lv[c] = MC_CASE_VERTS[m];
  g_mc_image.lt[c] = MC_CASE_TRIS[m];
  g_mc_image.cnt[c] = (uint32_t)(MC_CASE_VERTS[m] & 0xF) | ((uint32_t)(MC_CASE_TRIS[m] & 0x7) << 16);
}

template <typename T, typename M, typename Out, int CXM>
__device__ __forceinline__ void rows_mc_tile(const VolArgs& a, const RowsBlock& blk) {
  constexpr int VW = (kCells * 12 + 64) / 64 + 1, FW = (kCells * 5 + 64) / 64 + 1;
  struct Wave {
    union {
      Out v[192];
      int64_t f[192];
    } stage;
    uint64_t vbits[VW], fbits[FW];      // slot o starts a cell
    uint32_t list[kCells];              // word of the wave's | bit << 9 | case << 14
    uint16_t lpv[kCells], lpf[kCells];  // first vertex and face slot
  };
  struct Smem {
    McImage tab;
    uint4 edge[12];  // byte offsets of the edge's corners, then their (dx,dy,dz) | .. << 3
    Wave wave[kWaves];
  };
  __shared__ __align__(16) Smem sm;
  static_assert(sizeof(McImage) % 16 == 0, "copied in 16-byte words");
  const Geom g = a.g;
  const uint32_t pbytes = (uint32_t)((int64_t)g.nx * g.ny * (int64_t)sizeof(T));
  const uint32_t rbytes = (uint32_t)g.nx * (uint32_t)sizeof(T);
  const int lane = lane_id();
  const RowsWork work = rows_work<MC>(a, blk);
  const int x = work.x, g0 = work.g0, g1 = work.g1;
  const uint32_t cnt = work.cnt;
  // a tile whose units are all empty ends here, before its tables
  if (!__syncthreads_or(cnt != 0)) return;
  for (int q = threadIdx.x; q < (int)(sizeof(McImage) / 16); q += kBlock)
    ((uint4*)&sm.tab)[q] = ((const uint4*)&g_mc_image)[q];
  if (threadIdx.x < 12) {
    const uint32_t ew = MC_EDGE[threadIdx.x];
    const int ca = ew & 0xF, cb = ew >> 4;
    auto off = [&](int c) {
      return (mc_dz(c) ? pbytes : 0u) + (mc_dy(c) ? rbytes : 0u) +
             (mc_dx(c) ? (uint32_t)sizeof(T) : 0u);
    };
    sm.edge[threadIdx.x] = make_uint4(
        off(ca), off(cb),
        (uint32_t)(mc_dx(ca) | (mc_dy(ca) << 1) | (mc_dz(ca) << 2) | (mc_dx(cb) << 3) |
                   (mc_dy(cb) << 4) | (mc_dz(cb) << 5)), 0u);
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
  const int cxm = CXM >= 0 ? CXM : a.cxmask;
  const bool cx32 = cxm & 1, cy32 = (cxm >> 1) & 1, cz32 = (cxm >> 2) & 1;
  const double* __restrict__ yp = a.coords + g.nx;
  const double* __restrict__ zp = yp + g.ny;
  const double x0 = a.coords[x], x1 = a.coords[x + 1];
  const WordBase wb = word_base(a, g0);
  int64_t vb, fb;     // the queue's first outputs ..
  uint32_t vph, fph;  // .. beyond a multiple of 64 records
  uint32_t V, F;      // slots of the queue, from that multiple
  int nc = 0;         // its cells
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
  auto flush = [&]() {
    wave_sync();
    int before = 0;
    auto fetch = [&](uint32_t o0, Fetch& r) {
      // (a lane without a vertex reads one of the queue's again)
      const uint32_t o = min(max(o0 + lane, vph), V - 1);
      const uint64_t word = wm.vbits[min(o0, V - 1) >> 6];
      // (past the end: the last vertex of the last cell)
      const int ki = o0 >= V ? nc - 1 : before + __popcll(word & (~0ull >> (kWave - 1 - (o & 63)))) - 1;
      before += __popcll(word);
      const uint32_t e = wm.list[ki];
      const uint32_t ed = (uint32_t)(sm.tab.lv[(e >> 14) & 0xFF] >> (4 + 4 * (o - wm.lpv[ki]))) & 0xF;
      const uint4 ew = sm.edge[ed];
      int y, w;
      word_pos(a, wb, e & 511, &y, &w);
      const uint32_t z = 32u * (uint32_t)w + ((e >> 9) & 31);
      const char* cell = f + (uint64_t)z * pbytes + (uint64_t)(uint32_t)y * rbytes;
      r.va = *(const T*)(cell + ew.x);
      r.vb = *(const T*)(cell + ew.y);
      r.y = *(const Pair<double>*)(yp + y);
      r.z = *(const Pair<double>*)(zp + z);
      r.ends = ew.z;
    };
    auto place = [&](uint32_t o0, const Fetch& r) {
      const uint32_t en = r.ends;
      const M mu = (iso - (M)r.va) / (M)(r.vb - r.va);
      wm.stage.v[3 * lane] = (Out)lerp_axis<M>(cx32, mu, (en & 1) ? x1 : x0, (en & 8) ? x1 : x0);
      wm.stage.v[3 * lane + 1] =
          (Out)lerp_axis<M>(cy32, mu, (en & 2) ? r.y.b : r.y.a, (en & 16) ? r.y.b : r.y.a);
      wm.stage.v[3 * lane + 2] =
          (Out)lerp_axis<M>(cz32, mu, (en & 4) ? r.z.b : r.z.a, (en & 32) ? r.z.b : r.z.a);
      wave_sync();
      store_records(verts + 3 * (vb - (int64_t)vph + (int64_t)o0), wm.stage.v,
                    o0 == 0 ? (int)vph : 0, (int)V - (int)o0);
      wave_sync();
    };
    // The samples and coordinates of the next 64 vertices are on their way
    // while these are placed.  Two buffers in turn; an odd last step is
    // followed by one that stores nothing (an exit between the two would
    // make the compiler wait for the first buffer before it refills it).
    Fetch p, q;
    fetch(0, p);
    for (uint32_t o0 = 0; o0 < V; o0 += 2 * kWave) {
      fetch(o0 + kWave, q);
      place(o0, p);
      fetch(o0 + 2 * kWave, p);
      place(o0 + kWave, q);
    }
    before = 0;
    for (uint32_t o0 = 0; o0 < F; o0 += kWave) {
      const uint32_t o = o0 + lane;
      const uint64_t word = wm.fbits[o0 >> 6];
      const int ki = before + __popcll(word & (~0ull >> (kWave - 1 - lane))) - 1;
      before += __popcll(word);
      if (o >= fph && o < F) {
        const uint64_t w = sm.tab.lt[(wm.list[ki] >> 14) & 0xFF] >> (3 + 12 * (o - wm.lpf[ki]));
        // the cell's first vertex, 1-based
        const int64_t first = vb - (int64_t)vph + (int64_t)wm.lpv[ki] + 1;
        wm.stage.f[3 * lane] = first + (int64_t)(w & 0xF);
        wm.stage.f[3 * lane + 1] = first + (int64_t)((w >> 4) & 0xF);
        wm.stage.f[3 * lane + 2] = first + (int64_t)((w >> 8) & 0xF);
      }
      wave_sync();
      store_records(faces + 3 * (fb - (int64_t)fph + (int64_t)o0), wm.stage.f,
                    o0 == 0 ? (int)fph : 0, (int)F - (int)o0);
      wave_sync();
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
    nc = 0;
  };

  int gi = g0 + __builtin_ctzll(todo);
  start(readlane64(work.voff, gi - g0) + (int64_t)work.vpre,
        readlane64(work.foff, gi - g0) + (int64_t)work.fpre);
  RawWords raw = load_raw(a, x, gi, lane);
#pragma unroll 1
  while (gi < g1) {
    const CellWord r = cell_word(raw);
    const uint64_t rest = (todo >> (gi - g0)) & ~1ull;
    const int gn = rest ? gi + __builtin_ctzll(rest) : g1;
    if (gn < g1) raw = load_raw(a, x, gn, lane);  // the next unit's words, meanwhile
    const bool gap = gn < g1 && work.gap(gi - g0, gn - g0);
    const uint32_t act = work.has(lane) ? active_cells(r) : 0u;
    const uint32_t incl = wave_scan_dpp(__popc(act));
    const int total = __builtin_amdgcn_readlane((int)incl, kWave - 1);
    for (int lo = 0; lo < total;) {
      // the next cells of the unit that fit the queue, at most 64
      const int take = min(min(kCells - nc, kWave), total - lo);
      const int c = nc + lane;
      const bool in = lane < take;
      int L, b;
      listed_cell(act, incl, lo, take, wm.list + nc, &L, &b);
      const uint32_t cs = cell_case_of(r, L, b);
      const uint32_t pk = in ? sm.tab.cnt[cs] : 0u;
      const uint32_t inc = wave_scan_dpp(pk);
      const uint32_t sv = V + ((inc - pk) & 0xFFFF), sf = F + ((inc - pk) >> 16);
      if (in) {
        wm.list[c] = ((uint32_t)L + 64u * (uint32_t)(gi - g0)) | ((uint32_t)b << 9) | (cs << 14);
        wm.lpv[c] = (uint16_t)sv;
        wm.lpf[c] = (uint16_t)sf;
        atomicOr((unsigned long long*)&wm.vbits[sv >> 6], 1ull << (sv & 63));
        atomicOr((unsigned long long*)&wm.fbits[sf >> 6], 1ull << (sf & 63));
      }
      const uint32_t sum = (uint32_t)__builtin_amdgcn_readlane((int)inc, kWave - 1);
      V += sum & 0xFFFF;
      F += sum >> 16;
      nc += take;
      lo += take;
      if (nc == kCells || (lo == total && (gn == g1 || gap))) flush();
    }
    if (gap) {
      int64_t v, f;
      work.unit_offsets(a, gn - g0, &v, &f);
      start(v, f);
    }
    gi = gn;
  }
}

template <typename T, typename M, typename Out, int CXM>
__global__ __launch_bounds__(kBlock) void k_rows_mc(VolArgs a) {
  const RowsBlock b = rows_block(a);
  if (!b.none) rows_mc_tile<T, M, Out, CXM>(a, b);
}

// Batched: a block per group or tile of the launch.
template <typename T, typename M, typename Out, int CXM>
__global__ __launch_bounds__(kBlock) void k_rows_mc_b(const VolArgs* __restrict__ vols,
    const int32_t* __restrict__ emap, int64_t gbase, const RowsGroup* __restrict__ groups,
    const uint32_t* __restrict__ ngroups, int32_t xblocks) {
  RowsBlock b = rows_block(emap, gbase, groups, ngroups, xblocks);
  if (b.none) return;
  const VolArgs a = batch_volume(vols, b.vol);
  b.tile -= a.eblk0;
  rows_mc_tile<T, M, Out, CXM>(a, b);
}

}  // namespace

// ---------------------------------------------------------------------------
// Host side.

hipError_t launch_mc_image(hipStream_t st) {
  hipLaunchKernelGGL(k_mc_image, dim3(1), dim3(kBlock), 0, st);
  return hipGetLastError();
}

template <typename T, typename M, typename Out, int CXM>
static hipError_t rows_mc_cx(const VolArgs& a, const RowsBatch* b, hipStream_t st) {
  if (b)
    hipLaunchKernelGGL((k_rows_mc_b<T, M, Out, CXM>), dim3((unsigned)(b->xblocks + b->nblocks)),
                       dim3(kBlock), 0, st, b->vols, b->map, b->gbase, b->groups,
                       b->ngroups, b->xblocks);
  else
    hipLaunchKernelGGL((k_rows_mc<T, M, Out, CXM>), dim3((unsigned)(a.xblocks + a.ntiles)),
                       dim3(kBlock), 0, st, a);
  return hipGetLastError();
}

template <typename T, typename M, typename Out>
static hipError_t rows_mc_t(int cxclass, const VolArgs& a, const RowsBatch* b, hipStream_t st) {
  switch (cxclass) {
    case 1: return rows_mc_cx<T, M, Out, 0>(a, b, st);
    case 2: return rows_mc_cx<T, M, Out, 7>(a, b, st);
    default: return rows_mc_cx<T, M, Out, -1>(a, b, st);
  }
}

hipError_t launch_rows_mc(const Plan& p, int cxclass, const VolArgs& a, const RowsBatch* b,
                          hipStream_t st) {
  if ((b ? b->nblocks : a.ntiles) == 0) return hipSuccess;
  if (p.T == K_F32 && p.M == K_F32 && p.Out == K_F32) return rows_mc_t<float, float, float>(cxclass, a, b, st);
  if (p.T == K_F32 && p.M == K_F32) return rows_mc_t<float, float, double>(cxclass, a, b, st);
  if (p.T == K_F32) return rows_mc_t<float, double, double>(cxclass, a, b, st);
  return rows_mc_t<double, double, double>(cxclass, a, b, st);
}

}  // namespace msh
