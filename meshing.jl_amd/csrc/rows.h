// rows.h -- device helpers of the row kernels (rows.hip: sample bits and
// counts; rows_mc.hip, rows_sn.hip, rows_mt.hip: the emits).
//
// A "column" (x, y) of samples keeps one bit per sample, set below the
// level, 32 samples along z per word, z fastest in memory: word w of column
// (x, y) is bits[x * xs + y * sw + w] (sw words a column, xs words an x
// plane, rounded up to whole 128-byte lines).  Cells along z come 32 to a
// word too (cw words a cell row), so 32 cells are classified at once from
// the words of their four columns and those words moved down by one sample.
//
// A unit is 64 consecutive words of cells at one x in emission order (y,
// then z): one lane a word, upx units an x plane, unit u = x * upx + g.  The
// units' order is the reference's emission order (x outermost, z innermost,
// src/marching_cubes.jl:40), so a unit's vertices and faces are one run of
// each output array.
#pragma once
#include "device.h"

namespace msh {

// Word w of a column and the same moved down by one sample: bit b of c is
// the sample at z = 32 w + b, bit b of s the one above it.
struct Col {
  uint32_t c, s;
};

// The cell words of a lane: (y, w) of word q = g * 64 + lane of an x plane,
// its four columns (x, y), (x+1, y), (x, y+1), (x+1, y+1) and the cells that
// exist; lanes past the plane's last word have none.
struct CellWord {
  uint32_t valid;
  int y, w;
  Col c00, c10, c01, c11;
};
// (y, w) of word q0 + i of an x plane, q0 = g * 64 and i < 64 * kMaxUE: q0 is
// divided in scalar registers (cwm gives the quotient or one less); the
// lanes' distance t from that row's start is below cw + 512, where a 16-bit
// reciprocal is exact for short rows and a few compares serve the long ones.
constexpr int kMaxUE = 8;  // units a wave emits, at most
constexpr int kShortRow = 120;  // the reciprocal is exact up to 125 words
struct WordBase {
  uint32_t y0, w0;
};
__device__ __forceinline__ WordBase word_base(const VolArgs& a, int g) {
  const uint32_t cw = (uint32_t)a.cw, q0 = (uint32_t)g * 64u;
  uint32_t y0 = __umulhi(q0, a.cwm), w0 = q0 - y0 * cw;
  if (w0 >= cw) {
    ++y0;
    w0 -= cw;
  }
  return {y0, w0};
}
__device__ __forceinline__ void word_pos(const VolArgs& a, const WordBase& o, uint32_t i, int* y,
                                         int* w) {
  const uint32_t cw = (uint32_t)a.cw, t = o.w0 + i;
  uint32_t dy;
  if (cw < (uint32_t)kShortRow) {
    dy = (t * a.cwn) >> 16;
  } else {  // t < cw + 512 < 6 cw
    dy = (t >= cw) + (t >= 2 * cw) + (t >= 3 * cw) + (t >= 4 * cw) + (t >= 5 * cw);
  }
  *y = (int)(o.y0 + dy);
  *w = (int)(t - dy * cw);
}

// A lane's cell words as loaded: the four columns' words and the next ones.
struct RawWords {
  uint32_t c[4], n[4];  // (x, y) (x+1, y) (x, y+1) (x+1, y+1)
  uint32_t valid;
  int y, w;
};
__device__ __forceinline__ RawWords load_raw(const VolArgs& a, int x, int g, int lane) {
  RawWords r{};
  int y, w;
  word_pos(a, word_base(a, g), (uint32_t)lane, &y, &w);
  r.y = y;
  r.w = w;
  if (y >= a.g.ny - 1) return r;
  const int left = a.g.nz - 1 - 32 * w;  // cells from this word on
  r.valid = left >= 32 ? ~0u : (1u << left) - 1u;
  // a plane's words are counted in 32 bits; the word after a column's last
  // one is the next column's or the padding behind the plane: its bits
  // belong to no cell
  const uint32_t* __restrict__ p0 = a.bits + (int64_t)x * a.xs;
  const uint32_t* __restrict__ p1 = p0 + a.xs;
  const uint32_t i = (uint32_t)y * (uint32_t)a.sw + (uint32_t)w, j = i + (uint32_t)a.sw;
  r.c[0] = p0[i];
  r.n[0] = p0[i + 1];
  r.c[1] = p1[i];
  r.n[1] = p1[i + 1];
  r.c[2] = p0[j];
  r.n[2] = p0[j + 1];
  r.c[3] = p1[j];
  r.n[3] = p1[j + 1];
  return r;
}
__device__ __forceinline__ CellWord cell_word(const RawWords& r) {
  CellWord c{};
  c.valid = r.valid;
  c.y = r.y;
  c.w = r.w;
  c.c00 = {r.c[0], __builtin_amdgcn_alignbit(r.n[0], r.c[0], 1)};
  c.c10 = {r.c[1], __builtin_amdgcn_alignbit(r.n[1], r.c[1], 1)};
  c.c01 = {r.c[2], __builtin_amdgcn_alignbit(r.n[2], r.c[2], 1)};
  c.c11 = {r.c[3], __builtin_amdgcn_alignbit(r.n[3], r.c[3], 1)};
  return c;
}
__device__ __forceinline__ CellWord load_cells(const VolArgs& a, int x, int g, int lane) {
  return cell_word(load_raw(a, x, g, lane));
}
// cells with samples on both sides of the level
__device__ __forceinline__ uint32_t active_cells(const CellWord& r) {
  const uint32_t any = r.c00.c | r.c10.c | r.c01.c | r.c11.c | r.c00.s | r.c10.s | r.c01.s | r.c11.s;
  const uint32_t all = r.c00.c & r.c10.c & r.c01.c & r.c11.c & r.c00.s & r.c10.s & r.c01.s & r.c11.s;
  return any & ~all & r.valid;
}
// case of cell b in natural order: (x,y) (x+1,y) (x,y+1) (x+1,y+1), then above
__device__ __forceinline__ uint32_t cell_case(const CellWord& r, int b) {
  return ((r.c00.c >> b) & 1u) | (((r.c10.c >> b) & 1u) << 1) | (((r.c01.c >> b) & 1u) << 2) |
         (((r.c11.c >> b) & 1u) << 3) | (((r.c00.s >> b) & 1u) << 4) |
         (((r.c10.s >> b) & 1u) << 5) | (((r.c01.s >> b) & 1u) << 6) |
         (((r.c11.s >> b) & 1u) << 7);
}
// the same for cell b of lane L's word
__device__ __forceinline__ uint32_t cell_case_of(const CellWord& r, int L, int b) {
  auto from = [&](uint32_t v) {
    return ((uint32_t)__builtin_amdgcn_ds_bpermute(L << 2, (int)v) >> b) & 1u;
  };
  return from(r.c00.c) | (from(r.c10.c) << 1) | (from(r.c01.c) << 2) | (from(r.c11.c) << 3) |
         (from(r.c00.s) << 4) | (from(r.c10.s) << 5) | (from(r.c01.s) << 6) | (from(r.c11.s) << 7);
}

// The place of the r-th set bit of x (r below its population count).
__device__ __forceinline__ uint32_t nth_bit(uint32_t x, uint32_t r) {
  uint32_t p = 0;
#pragma unroll
  for (uint32_t s = 16; s > 0; s >>= 1) {
    const uint32_t c = __popc((x >> p) & ((1u << s) - 1u));
    const bool up = r >= c;
    r -= up ? c : 0u;
    p += up ? s : 0u;
  }
  return p;
}

// Cell lo + lane of a unit whose lanes hold the words' active cells act,
// incl = their inclusive count: its word's lane and its bit (0 from `take`
// on).  Each word with cells marks its first one's place in mark[0, take);
// the word of a place is the last one marked at or before it.  (A loop over
// the bits of each lane's word waits for the fullest word: 301 x 217 x 389
// Float32 Marching Cubes emit 174 us so, 160 us this way; 512^3 tetrahedra
// 1584 and 1553.)
__device__ __forceinline__ void listed_cell(uint32_t act, uint32_t incl, int lo, int take,
                                            uint32_t* mark, int* word, int* bit) {
  const int lane = lane_id();
  const bool in = lane < take;
  if (in) mark[lane] = 0;
  wave_sync();
  const uint32_t start = incl - (uint32_t)__popc(act), d = start - (uint32_t)lo;
  if (act != 0 && d < (uint32_t)take) mark[d] = (uint32_t)lane;
  wave_sync();
  // (place 0 may lie inside a word: the first one that ends past lo)
  const uint32_t w0 = (uint32_t)__popcll(__ballot((int)incl <= lo));
  uint32_t w = in ? mark[lane] : 0u;
  w = lane == 0 ? w0 : w;
  w = wave_max_dpp(w);
  const uint32_t wact = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(w << 2), (int)act);
  const uint32_t wstart = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(w << 2), (int)start);
  const uint32_t b = nth_bit(wact, (uint32_t)(lo + lane) - wstart) & 31u;
  *word = in ? (int)w : 0;
  *bit = in ? (int)b : 0;
}

// The five columns around a lane's cell words that hold corners of the cells
// at -x, -y and both: (x-1, y) (x-1, y+1) (x, y-1) (x+1, y-1) (x-1, y-1).
// Zero where they do not exist.
struct BackWords {
  Col x0, x1, y0, y1, xy;
};
__device__ __forceinline__ BackWords load_back(const VolArgs& a, int x, const CellWord& r) {
  BackWords k{};
  if (r.valid == 0) return k;
  const uint32_t* __restrict__ p0 = a.bits + (int64_t)x * a.xs;
  const uint32_t sw = (uint32_t)a.sw, i = (uint32_t)r.y * sw + (uint32_t)r.w;
  auto col = [](const uint32_t* __restrict__ p, uint32_t j) -> Col {
    const uint32_t c = p[j];
    return {c, __builtin_amdgcn_alignbit(p[j + 1], c, 1)};
  };
  if (r.y > 0) {
    k.y0 = col(p0, i - sw);
    k.y1 = col(p0 + a.xs, i - sw);
  }
  if (x > 0) {
    const uint32_t* __restrict__ pm = p0 - a.xs;
    k.x0 = col(pm, i);
    k.x1 = col(pm, i + sw);
    if (r.y > 0) k.xy = col(pm, i - sw);
  }
  return k;
}
// active cells of the word of columns a, b, c, d
__device__ __forceinline__ uint32_t active_of(const Col& a, const Col& b, const Col& c, const Col& d,
                                              uint32_t valid) {
  return ((a.c | b.c | c.c | d.c | a.s | b.s | c.s | d.s) &
          ~(a.c & b.c & c.c & d.c & a.s & b.s & c.s & d.s)) & valid;
}
// First vertex (in the volume's numbering) of cell word q of x plane x.
__device__ __forceinline__ int64_t word_vertex(const VolArgs& a, int x, uint32_t q) {
  const int64_t u = (int64_t)x * a.upx + (q >> 6);
  return a.voff[a.ubase + u] + (int64_t)a.wpre[64 * u + (q & 63)];
}

// ---------------------------------------------------------------------------
// Shared units.  A wave takes a unit's cells one queue after another, so a
// unit of a surface that runs along its x plane, up to 2048 cells where most
// have a few dozen, keeps one wave at work long after the rest of the device
// is idle (a plane x = const in 256^3 Float32: 32 such units, Marching Cubes
// call 184 us, tetrahedra 448).  Units of many outputs are therefore cut into
// parts of neighbouring words with about the same number of vertices
// (rows_parts, note_parts): the count pass leaves where they start, the scan
// lists the parts in groups (RowsGroup), and the emit's first blocks take a
// group each, a part a wave, while the waves of the tiles leave these units
// out (81 us and 106).  Where many units are full a wave takes a quarter of one,
// and where that is too many (rows_group_cap) the device is full without this.

// What a wave of an emit block works on: units [g0, g1) of x plane x, or with
// a group a part of one unit.
struct RowsWork {
  int x, g0, g1;
  uint32_t cnt;         // lane i: unit g0 + i's counts, 0 if it has none or others take it
  uint32_t shared;      // bit i: others take unit g0 + i
  int64_t voff, foff;   // lane i: where the unit's outputs start
  int w0, wn;           // its words: wn from w0 on
  uint32_t vpre, fpre;  // the unit's outputs before them
  __device__ bool has(int lane) const { return (uint32_t)(lane - w0) < (uint32_t)wn; }
  // (again for a unit behind a shared one, so that the lanes need not keep them)
  __device__ void unit_offsets(const VolArgs& a, int i, int64_t* v, int64_t* f) const {
    const int64_t u = a.ubase + (int64_t)x * a.upx + g0 + i;
    *v = a.voff[u] - a.sz[0];
    *f = a.foff[u] - a.sz[2];
  }
  // shared units between i and the next one of the wave, j?
  __device__ bool gap(int i, int j) const {
    return ((shared >> i) & ((1u << (j - i)) - 1u)) != 0;
  }
};

static_assert(rows_emit_waves(MC) == kWaves && rows_emit_waves(MT) == kWaves, "their blocks");

// Emit tile t: W x planes (one a wave of the block, so its waves read the
// same lines) by a.ue units.  Tiles go over 32 planes along x (a 128-byte line
// of Float32 samples), then along the planes, then to the next 32, so the
// tiles in flight on an XCD share their lines in its L2.
template <int W>
__device__ __forceinline__ void rows_tile(const VolArgs& a, int64_t t, int* x, int* g0) {
  constexpr uint32_t G = 32 / W;  // blocks of 32 planes
  const uint32_t nxb = (uint32_t)(a.g.nx - 1 + W - 1) / W;
  const uint32_t gb = (uint32_t)(a.upx + a.ue - 1) / (uint32_t)a.ue;
  const uint32_t full = nxb / G, rest = nxb - full * G;
  const uint32_t grp = (uint32_t)t / (G * gb);
  uint32_t r, n = G, first = grp;
  if (grp >= full) {
    first = full;
    n = rest;
  }
  r = (uint32_t)t - first * G * gb;
  const uint32_t gi = r / n;
  *x = (int)(first * G + (r - gi * n)) * W + wave_id();
  *g0 = (int)gi * a.ue;
}

// Emit tile of block b.  Blocks are dealt round-robin to the 8 XCDs; a launch
// of few blocks gives each XCD one run of tiles (xcd_tile), a larger one runs
// of 32 in turn, so tiles that share lines meet in one L2 and a field whose
// surface lies in a part of its planes still keeps every XCD busy (1024^3
// Float32 sphere emit 158 -> 132 us; the 2048 blocks of a 256^3 gyroid are
// 36 us in one run an XCD and 39 in turns; surface nets of 384 x 320 x 448
// Float64 noise, 13440 blocks of two waves, 458 and 430).  `few`: the blocks
// from which a launch takes turns.
__device__ __forceinline__ int64_t rows_block_tile(int64_t b, int64_t nb, int64_t few = 8192) {
  constexpr int64_t C = 32;
  if (nb < few) return xcd_tile(b, nb);
  if (b >= nb / (8 * C) * (8 * C)) return b;
  // (turned by one XCD a round: the y range of a plane is not one XCD's)
  const int64_t round = (b >> 3) / C, at = (b >> 3) % C;
  return (round * 8 + (((b & 7) + round) & 7)) * C + at;
}

// Group of block b < nb of a single emit's, n or more: none.  The n groups lie
// in the list about as their units do, so where most units are shared a row of
// cols groups is an x plane, and neighbours along x read the same lines.  As the
// tiles do (rows_tile), the blocks go over 32 planes along x, then along the
// planes, and each XCD gets one run of that order.  Dealt as they are listed,
// neighbours meet in one L2 only where cols is a multiple of 8, and then they do
// it best (cols 1 here).  Value noise, calls in us, a wave a unit / as listed /
// this order: Marching Cubes of 180^3, 17 columns, Float32 126 / 141 / 118 and
// Float64 139 / 170 / 133, of 144^3, 12, Float64 120 / 130 / 115; tetrahedra of
// 180^3 268 / 246 / 232; 128^3, 8, Float64 138 / 106 / 113.
__host__ __device__ inline uint32_t group_of_block(uint32_t b, uint32_t nb, uint32_t n, uint32_t cols) {
  if (cols == 1) return b;
  const uint32_t rows = (n + cols - 1) / cols, j = (uint32_t)xcd_tile(b, nb);
  if (j >= rows * cols) return n;
  const uint32_t first = j / (32 * cols) * 32, of = min(rows - first, 32u), r = j - first * cols;
  return (first + r % of) * cols + r / of;
}

// An emit block's work: a group of shared parts (the first blocks; those past
// the last group have none) or a tile.
struct RowsBlock {
  bool none = false;
  const RowsGroup* grp = nullptr;
  bool share = false;  // the launch's tiles leave shared units out
  int64_t tile = 0;    // of the volume
  int vol = 0;
};
__device__ __forceinline__ RowsBlock rows_block(const VolArgs& a) {
  // (worked out for a tile first: a branch on a kernel argument ahead of it
  // would put the reads of the others behind the wait for that one)
  RowsBlock r;
  r.tile = rows_block_tile((int64_t)blockIdx.x - a.xblocks, a.ntiles);
  r.share = a.xblocks > 0;
  if (__builtin_expect((int)blockIdx.x < a.xblocks, 0)) {
    const uint32_t i = group_of_block(blockIdx.x, (uint32_t)a.xblocks, a.shared, a.gcols);
    r.none = i >= a.shared;
    r.grp = a.taken + i;
    r.share = false;
  }
  return r;
}
__device__ __forceinline__ RowsBlock rows_block(const int32_t* __restrict__ map, int64_t gbase,
                                                const RowsGroup* __restrict__ groups,
                                                const uint32_t* __restrict__ ngroups,
                                                int32_t xblocks, int64_t few = 8192) {
  RowsBlock r;
  if (__builtin_expect((int)blockIdx.x < xblocks, 0)) {
    r.none = blockIdx.x >= *ngroups;
    r.grp = groups + blockIdx.x;
    if (!r.none) r.vol = __builtin_amdgcn_readfirstlane((int)r.grp->vol);
  } else {
    r.tile = gbase + rows_block_tile((int64_t)blockIdx.x - xblocks, (int64_t)gridDim.x - xblocks, few);
    r.vol = __builtin_amdgcn_readfirstlane(map[r.tile]);
    r.share = xblocks > 0;
  }
  return r;
}
template <int METHOD>
__device__ __forceinline__ RowsWork rows_work(const VolArgs& a, const RowsBlock& b) {
  const RowsGroup* const grp = b.grp;
  const bool share = b.share;
  constexpr int W = rows_emit_waves(METHOD);
  const int lane = lane_id();
  RowsWork k{};
  // (a group's block: any tile, replaced below)
  rows_tile<W>(a, grp ? 0 : b.tile, &k.x, &k.g0);
  k.g1 = min(k.g0 + a.ue, a.upx);
  k.wn = kWave;
  if (__builtin_expect(grp != nullptr, 0)) {
    const uint32_t u = grp->unit, step = grp->step;
    const uint32_t part = grp->first + step * (uint32_t)__builtin_amdgcn_readfirstlane(wave_id());
    const RowsParts& cut = a.parts[u];
    const uint32_t pre = cut.pre[part];
    k.x = (int)(u / (uint32_t)a.upx);
    k.g0 = (int)(u - (uint32_t)k.x * (uint32_t)a.upx);
    k.g1 = k.g0 + 1;
    k.w0 = cut.word[part];
    k.wn = (part + step < grp->parts ? (int)cut.word[part + step] : kWave) - k.w0;
    k.vpre = pre & 0xFFFF;
    k.fpre = pre >> 16;
  }
  if (k.x < a.g.nx - 1 && lane < k.g1 - k.g0) {
    const int64_t u = a.ubase + (int64_t)k.x * a.upx + k.g0 + lane;
    k.cnt = a.cnt[u];
    k.voff = a.voff[u] - a.sz[0];
    k.foff = a.foff[u] - a.sz[2];
  }
  const bool others = share && rows_parts(rows_cuts(METHOD), k.cnt & 0xFFFF) > 0;
  k.shared = (uint32_t)__ballot(others);  // (of kMaxUE units)
  k.cnt = others ? 0u : k.cnt;
  return k;
}

// Two neighbouring values in one load (aligned as one of them).
template <typename T>
struct __attribute__((packed, aligned(sizeof(T)))) Pair {
  T a, b;
};

// What the emits take of volume v of a batch, read as constant memory (it is, from
// the upload on): scalar loads, and pointers that the compiler knows to be
// global.  As flat ones, two registers an address, they cost Marching Cubes 98
// registers instead of 80 and made the tetrahedra kernel spill.
__device__ __forceinline__ VolArgs batch_volume(const VolArgs* vols, int v) {
  const auto* s = (const __attribute__((address_space(4))) VolArgs*)vols +
                  __builtin_amdgcn_readfirstlane(v);
  VolArgs a{};
  a.f = s->f;
  a.g.nx = s->g.nx;
  a.g.ny = s->g.ny;
  a.g.nz = s->g.nz;
  a.iso = s->iso;
  a.eps = s->eps;
  a.ome = s->ome;
  a.cxmask = s->cxmask;
  a.coords = s->coords;
  a.cnt = s->cnt;
  a.voff = s->voff;
  a.foff = s->foff;
  a.sz = s->sz;
  a.verts = s->verts;
  a.faces = s->faces;
  a.ubase = s->ubase;
  a.bits = s->bits;
  a.wpre = s->wpre;
  a.parts = s->parts;
  a.xs = s->xs;
  a.sw = s->sw;
  a.cw = s->cw;
  a.upx = s->upx;
  a.ue = s->ue;
  a.cwm = s->cwm;
  a.cwn = s->cwn;
  a.eblk0 = s->eblk0;
  return a;
}

// 64 records of three values from LDS to the output, each through `value`:
// records [s0, s1) of the 64 at `out`, the wave's lanes on consecutive
// values, so that every line is written whole by one store instruction.
// Buffer stores: a value outside the records gets an offset past the buffer
// and is dropped, so there is no branch, and a wait for loads issued before
// does not wait for the stores.
// Non-temporal: a line is written once and whole, and kept out of the L2 it
// leaves room there for the samples that the waves nearby share (301 x 217 x
// 389 Float32 value noise 250 -> 172 us, 1024^3 Float64 5.39 -> 4.97 ms).
struct Same {
  template <typename V>
  __device__ V operator()(V v) const { return v; }
};
template <typename O, typename V, class F = Same>
__device__ __forceinline__ void store_records(O* __restrict__ out, const V* stage, int s0, int s1,
                                              F value = F{}) {
  const __amdgpu_buffer_rsrc_t r = buffer_rsrc(out, 192 * sizeof(O));
  const int lane = lane_id();
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const int e = lane + 64 * j;
    const int off = e >= 3 * s0 && e < 3 * s1 ? e * (int)sizeof(O) : 0x7FFFFFFF;
    const O v = value(stage[e]);
    if constexpr (sizeof(O) == 4) {
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r, off, 0, 2);
    } else {
      typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
      __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, off, 0, 2);
    }
  }
}

__device__ __forceinline__ int64_t readlane64(int64_t v, int l) {
  return ((int64_t)__builtin_amdgcn_readlane((int)((uint64_t)v >> 32), l) << 32) |
         (int64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, l);
}

}  // namespace msh
