// rows_sn.hip -- Naive Surface Nets emit of the row kernels (see rows.h; the
// method is this library's own, oracle/cpu_ref.cpp sn_isosurface).
//
// As in rows_mc.hip a wave queues the active cells of up to a.ue units from
// the bits, in emission order, and emits a full queue.  Every active cell has
// one vertex, so a vertex's number is the count of active cells before it:
// the vertices that a quad names beside its own cell's come from the active
// bits of the words at -x, -y and both and from the vertex counts that the
// count pass keeps per word, a population count each and no look-up of
// another cell.  In the emit lane k of a step owns cell k: it reads the cell's
// eight samples (four loads of two, a step ahead) and sums the crossing
// points of its edges in registers; the faces are then written slot-parallel
// as in rows_mc.hip.  A unit that does not fit the queue is read again after
// the emit, which so needs no registers for it.
//
// Emit, before (halo5.hip) -> now: 256^3 Float32 gyroid 114 -> 34 us,
// 384 x 320 x 448 Float64 value noise 774 -> 419 us.  Bound by vector issue
// (53% of the SIMDs' cycles there, 51% on the gyroid, most of it the divisions
// and interpolations of the edges) and by the latency of each step's look-ups
// at 2.7 and 2.3 waves a SIMD on average (94 registers, Float64 114, would
// let it hold 5 or 4); holding the samples of a step in registers while its
// unit is listed (122 registers) was slower, and so were caps on the
// registers, which spill.
#include <type_traits>

#include "rows.h"

namespace msh {
namespace {

constexpr int kCells = 256;  // cells queued at a time, per wave

// Two waves a block: a block keeps its registers and LDS until its slowest
// wave is done, and there are no tables to share (256^3 Float32 gyroid emit 37
// us with four waves, 34 with two, 41 with one; 384 x 320 x 448 Float64 noise
// 483, 427 and 438).
constexpr int kSnWaves = rows_emit_waves(SN);
constexpr int kSnBlock = kSnWaves * kWave;

// The 12 cube edges in Marching Cubes order (src/lut/mc.jl _mc_edge_list),
// corners in natural order (bits 0, 1, 2: dx, dy, dz).
struct SnEdges {
  int a[12], b[12];
};
constexpr SnEdges kSnEdges = {{0, 1, 3, 2, 4, 5, 7, 6, 0, 1, 3, 2}, {1, 3, 2, 0, 5, 7, 6, 4, 4, 5, 7, 6}};

template <typename T, typename M, typename Out, int CXM>
__device__ __forceinline__ void rows_sn_tile(const VolArgs& a, const RowsBlock& blk) {
  constexpr int FW = (kCells * 6 + 64) / 64 + 1;
  struct Wave {
    union {
      Out v[192];
      int64_t f[192];
    } stage;
    uint64_t fbits[FW];     // face slot o starts a cell
    uint32_t list[kCells];  // word of the wave's | bit << 9 | case << 14
    uint32_t d10[kCells], d01[kCells], d11[kCells];  // how far back the vertices at -x, -y, both are
    uint32_t face[kCells];  // cells with faces: cell | axes << 8 | below << 11 | slot << 12
  };
  __shared__ __align__(16) Wave waves[kSnWaves];
  const Geom g = a.g;
  const uint32_t pbytes = (uint32_t)((int64_t)g.nx * g.ny * (int64_t)sizeof(T));
  const uint32_t rbytes = (uint32_t)g.nx * (uint32_t)sizeof(T);
  const int lane = lane_id();
  const RowsWork work = rows_work<SN>(a, blk);
  const int x = work.x, g0 = work.g0, g1 = work.g1;
  const uint32_t cnt = work.cnt;
  const uint64_t todo = __ballot(cnt != 0);  // bit i: unit g0 + i has outputs
  if (todo == 0) return;
  Wave& wm = waves[wave_id()];
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
  int64_t vb, fb;  // the queue's first outputs

  const WordBase wb = word_base(a, g0);
  int nc = 0;      // cells in the queue
  uint32_t F = 0;  // its face slots, from the last multiple of 64 records in the output
  uint32_t fph;
  int nf = 0;  // its cells with faces
  auto start = [&](int64_t v, int64_t f) {  // at a unit's outputs
    vb = v;
    fb = f;
    F = fph = (uint32_t)fb & 63u;
  };

  struct Fetch {
    Pair<T> s00, s01, s10, s11;  // (y, z) (y+1, z) (y, z+1) (y+1, z+1), samples x and x+1
    Pair<double> y, z;
    uint32_t cs;
  };
  auto emit = [&]() {
    wave_sync();
    // slot o of a step of 64 vertices is cell o - vph
    const int vph = (int)((uint32_t)vb & 63u), V = vph + nc;
    auto fetch = [&](int o0, Fetch& r) {
      // (a lane without a cell reads one of the queue's again)
      const uint32_t e = wm.list[min(max(o0 + lane - vph, 0), nc - 1)];
      int y, w;
      word_pos(a, wb, e & 511, &y, &w);
      const uint32_t z = 32u * (uint32_t)w + ((e >> 9) & 31);
      const char* p = f + (uint64_t)z * pbytes + (uint64_t)(uint32_t)y * rbytes;
      const char* q = p + pbytes;
      r.s00 = *(const Pair<T>*)p;
      r.s01 = *(const Pair<T>*)(p + rbytes);
      r.s10 = *(const Pair<T>*)q;
      r.s11 = *(const Pair<T>*)(q + rbytes);
      r.y = *(const Pair<double>*)(yp + y);
      r.z = *(const Pair<double>*)(zp + z);
      r.cs = (e >> 14) & 0xFF;
    };
    auto place = [&](int o0, const Fetch& r) {
      const T v[8] = {r.s00.a, r.s00.b, r.s01.a, r.s01.b, r.s10.a, r.s10.b, r.s11.a, r.s11.b};
      const double px[2] = {x0, x1}, py[2] = {r.y.a, r.y.b}, pz[2] = {r.z.a, r.z.b};
      // the mean of the crossing points of the cell's edges, each interpolated
      // as vertex_interp does (src/marching_cubes.jl:100-104), summed in edge
      // order, per axis in promote(M, axis type)
      float fx = 0.f, fy = 0.f, fz = 0.f;
      double dx = 0.0, dy = 0.0, dz = 0.0;
      const bool sx = sizeof(M) == 4 && cx32, sy = sizeof(M) == 4 && cy32,
                 sz = sizeof(M) == 4 && cz32;
      int n = 0;
#pragma unroll
      for (int e = 0; e < 12; ++e) {
        const int ca = kSnEdges.a[e], cb = kSnEdges.b[e];
        if (((r.cs >> ca) ^ (r.cs >> cb)) & 1) {
          const M mu = (iso - (M)v[ca]) / (M)(v[cb] - v[ca]);
          // along an axis on which the edge's ends agree p1 + mu * (p2 - p1)
          // is the end itself, or NaN where mu is not finite (an infinite
          // end would make it NaN too: rows_geom takes finite ones only)
          const double nz = (double)(mu * (M)0);
          const int ax = ca ^ cb;  // 1, 2, 4: the edge's axis
          const double qx = ax == 1 ? lerp_axis<M>(cx32, mu, px[ca & 1], px[cb & 1]) : px[ca & 1] + nz;
          const double qy = ax == 2 ? lerp_axis<M>(cy32, mu, py[(ca >> 1) & 1], py[(cb >> 1) & 1])
                                    : py[(ca >> 1) & 1] + nz;
          const double qz = ax == 4 ? lerp_axis<M>(cz32, mu, pz[ca >> 2], pz[cb >> 2]) : pz[ca >> 2] + nz;
          if (sx) fx = fx + (float)qx; else dx = dx + qx;
          if (sy) fy = fy + (float)qy; else dy = dy + qy;
          if (sz) fz = fz + (float)qz; else dz = dz + qz;
          ++n;
        }
      }
      wm.stage.v[3 * lane] = (Out)(sx ? (double)(fx / (float)n) : dx / (double)n);
      wm.stage.v[3 * lane + 1] = (Out)(sy ? (double)(fy / (float)n) : dy / (double)n);
      wm.stage.v[3 * lane + 2] = (Out)(sz ? (double)(fz / (float)n) : dz / (double)n);
      wave_sync();
      store_records(verts + 3 * (vb - (int64_t)vph + (int64_t)o0), wm.stage.v, o0 == 0 ? vph : 0, V - o0);
      wave_sync();
    };
    Fetch p, q;
    fetch(0, p);
    for (int o0 = 0; o0 < V; o0 += 2 * kWave) {
      fetch(o0 + kWave, q);
      place(o0, p);
      fetch(o0 + 2 * kWave, p);
      if (o0 + kWave < V) place(o0 + kWave, q);
    }
    int before = 0;
    for (uint32_t o0 = 0; o0 < F; o0 += kWave) {
      const uint32_t o = o0 + lane;
      const uint64_t word = wm.fbits[o0 >> 6];
      const int k = before + __popcll(word & (~0ull >> (kWave - 1 - lane))) - 1;
      before += __popcll(word);
      if (o >= fph && o < F) {
        const uint32_t e = wm.face[k];
        const int c = (int)(e & 255);
        const uint32_t ax = (e >> 8) & 7, q = o - (e >> 12);
        const bool below = (e >> 11) & 1;
        // the (q >> 1)-th of the cell's axes, in x, y, z order
        const uint32_t first = ax & (0u - ax), rest = ax ^ first;
        const uint32_t pick = (q >> 1) == 0 ? first : (q >> 1) == 1 ? (rest & (0u - rest)) : 4u;
        // the cells around that edge: one step back along the next axis, along
        // both, along the one after (a step along z is one vertex back)
        const uint32_t d10 = wm.d10[c], d01 = wm.d01[c], d11 = wm.d11[c];
        const uint32_t q1 = pick == 1 ? d01 : pick == 2 ? 1u : d10;
        const uint32_t q2 = pick == 1 ? d01 + 1u : pick == 2 ? d10 + 1u : d11;
        const uint32_t q3 = pick == 1 ? 1u : pick == 2 ? d10 : d01;
        const uint32_t a1 = below ? q1 : q3, a3 = below ? q3 : q1;
        const int64_t me = vb + c + 1;
        wm.stage.f[3 * lane] = me;
        wm.stage.f[3 * lane + 1] = me - (int64_t)((q & 1) ? q2 : a1);
        wm.stage.f[3 * lane + 2] = me - (int64_t)((q & 1) ? a3 : q2);
      }
      wave_sync();
      store_records(faces + 3 * (fb - (int64_t)fph + (int64_t)o0), wm.stage.f,
                    o0 == 0 ? (int)fph : 0, (int)F - (int)o0);
      wave_sync();
    }
    for (uint32_t q = lane; q < (F + 63) / 64; q += kWave) wm.fbits[q] = 0;
    wave_sync();
    vb += nc;
    fb += (int64_t)(F - fph);
    fph = (uint32_t)fb & 63u;
    F = fph;
    nc = nf = 0;
  };

  int gi = g0 + __builtin_ctzll(todo), done = 0;  // `done` cells of unit gi are through
  start(readlane64(work.voff, gi - g0) + (int64_t)work.vpre,
        readlane64(work.foff, gi - g0) + (int64_t)work.fpre);
#pragma unroll 1
  while (gi < g1) {
    bool gap = false;  // before the next unit
    {
      const CellWord r = load_cells(a, x, gi, lane);
      const BackWords k = load_back(a, x, r);
      const uint32_t act = work.has(lane) ? active_cells(r) : 0u;
      const uint32_t a10 = active_of(k.x0, r.c00, k.x1, r.c01, r.valid);
      const uint32_t a01 = active_of(k.y0, k.y1, r.c00, r.c10, r.valid);
      const uint32_t a11 = active_of(k.xy, k.y0, k.x0, r.c00, r.valid);
      const uint32_t incl = wave_scan_dpp(__popc(act));
      const int total = __builtin_amdgcn_readlane((int)incl, kWave - 1);
      // cells of the unit before the word
      const int at = (int)work.vpre + (int)incl - (int)__popc(act);
      // how far back the first vertices of the words at -x, -y and both are
      // from this word's (only a quad's cells are asked for, and they exist)
      uint32_t w10 = 0, w01 = 0, w11 = 0;
      {
        const int64_t mine = readlane64(work.voff, gi - g0) + a.sz[0] + at;
        const uint32_t q = (uint32_t)gi * 64u + (uint32_t)lane, cw = (uint32_t)a.cw;
        const bool some = act != 0;
        if (some && x > 0) w10 = (uint32_t)(mine - word_vertex(a, x - 1, q));
        if (some && r.y > 0) w01 = (uint32_t)(mine - word_vertex(a, x, q - cw));
        if (some && x > 0 && r.y > 0) w11 = (uint32_t)(mine - word_vertex(a, x - 1, q - cw));
      }
      // quads only where the cells at -1 exist: the axes of corner 0's edges
      // that a cell of the word may have faces on (bit 0 of the column: z > 0)
      const uint32_t has = (r.y > 0 ? 1u : 0u) | (x > 0 ? 2u : 0u) | (r.w > 0 ? 4u : 0u);
      while (done < total && nc < kCells) {
        const int take = min(min(kCells - nc, kWave), total - done);
        const bool in = lane < take;
        int L, b;
        listed_cell(act, incl, done, take, wm.list + nc, &L, &b);
        auto from = [&](uint32_t v) { return (uint32_t)__builtin_amdgcn_ds_bpermute(L << 2, (int)v); };
        const uint32_t c = cell_case_of(r, L, b);
        const uint32_t lowm = (1u << b) - 1u;
        const uint32_t mine = __popc(from(act) & lowm);
        const uint32_t d10 = from(w10) + mine - __popc(from(a10) & lowm);
        const uint32_t d01 = from(w01) + mine - __popc(from(a01) & lowm);
        const uint32_t d11 = from(w11) + mine - __popc(from(a11) & lowm);
        const uint32_t h = from(has);
        const bool yin = h & 1, xin = h & 2, zin = (h & 4) || b > 0;
        const uint32_t c0 = c & 1u;
        const uint32_t axes = (uint32_t)(c0 != ((c >> 1) & 1) && yin && zin) |
                              ((uint32_t)(c0 != ((c >> 2) & 1) && zin && xin) << 1) |
                              ((uint32_t)(c0 != ((c >> 4) & 1) && xin && yin) << 2);
        const uint32_t n = in ? 2u * __popc(axes) : 0u;
        const uint32_t inc = wave_scan_dpp(n), sf = F + inc - n;
        const uint64_t with = __ballot(n != 0);
        if (in) {
          wm.list[nc + lane] = ((uint32_t)L + 64u * (uint32_t)(gi - g0)) | ((uint32_t)b << 9) | (c << 14);
          wm.d10[nc + lane] = d10;
          wm.d01[nc + lane] = d01;
          wm.d11[nc + lane] = d11;
        }
        if (n != 0) {
          wm.face[nf + (int)lanes_below(with)] = (uint32_t)(nc + lane) | (axes << 8) | (c0 << 11) | (sf << 12);
          atomicOr((unsigned long long*)&wm.fbits[sf >> 6], 1ull << (sf & 63));
        }
        F += (uint32_t)__builtin_amdgcn_readlane((int)inc, kWave - 1);
        nf += __popcll(with);
        nc += take;
        done += take;
      }
      if (done >= total) {  // the next unit with outputs
        const uint64_t rest = (todo >> (gi - g0)) & ~1ull;
        const int gn = rest ? gi + __builtin_ctzll(rest) : g1;
        gap = gn < g1 && work.gap(gi - g0, gn - g0);
        gi = gn;
        done = 0;
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

template <typename T, typename M, typename Out, int CXM>
__global__ __launch_bounds__(kSnBlock) void k_rows_sn(VolArgs a) {
  const RowsBlock b = rows_block(a);
  if (!b.none) rows_sn_tile<T, M, Out, CXM>(a, b);
}

// Batched: a block per group or tile of the launch.  Turns
// over the XCDs from 16384 blocks, as many waves as in the other methods'
// batches (32 mixed volumes 605 us a batch, 624 with turns from 8192).
template <typename T, typename M, typename Out, int CXM>
__global__ __launch_bounds__(kSnBlock) void k_rows_sn_b(const VolArgs* __restrict__ vols,
    const int32_t* __restrict__ emap, int64_t gbase, const RowsGroup* __restrict__ groups,
    const uint32_t* __restrict__ ngroups, int32_t xblocks) {
  RowsBlock b = rows_block(emap, gbase, groups, ngroups, xblocks, 16384);
  if (b.none) return;
  const VolArgs a = batch_volume(vols, b.vol);
  b.tile -= a.eblk0;
  rows_sn_tile<T, M, Out, CXM>(a, b);
}

}  // namespace

// ---------------------------------------------------------------------------
// Host side.

template <typename T, typename M, typename Out, int CXM>
static hipError_t rows_sn_cx(const VolArgs& a, const RowsBatch* b, hipStream_t st) {
  if (b)
    hipLaunchKernelGGL((k_rows_sn_b<T, M, Out, CXM>), dim3((unsigned)(b->xblocks + b->nblocks)),
                       dim3(kSnBlock), 0, st, b->vols, b->map, b->gbase, b->groups,
                       b->ngroups, b->xblocks);
  else
    hipLaunchKernelGGL((k_rows_sn<T, M, Out, CXM>), dim3((unsigned)(a.xblocks + a.ntiles)),
                       dim3(kSnBlock), 0, st, a);
  return hipGetLastError();
}

template <typename T, typename M, typename Out>
static hipError_t rows_sn_t(int cxclass, const VolArgs& a, const RowsBatch* b, hipStream_t st) {
  switch (cxclass) {
    case 1: return rows_sn_cx<T, M, Out, 0>(a, b, st);
    case 2: return rows_sn_cx<T, M, Out, 7>(a, b, st);
    default: return rows_sn_cx<T, M, Out, -1>(a, b, st);
  }
}

hipError_t launch_rows_sn(const Plan& p, int cxclass, const VolArgs& a, const RowsBatch* b,
                          hipStream_t st) {
  if ((b ? b->nblocks : a.ntiles) == 0) return hipSuccess;
  if (p.T == K_F32 && p.M == K_F32 && p.Out == K_F32) return rows_sn_t<float, float, float>(cxclass, a, b, st);
  if (p.T == K_F32 && p.M == K_F32) return rows_sn_t<float, float, double>(cxclass, a, b, st);
  if (p.T == K_F32) return rows_sn_t<float, double, double>(cxclass, a, b, st);
  return rows_sn_t<double, double, double>(cxclass, a, b, st);
}

}  // namespace msh
