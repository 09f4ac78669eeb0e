// Cell-list neighbor search on a dense grid (gfx950).
//
// Build: key = cell of the wrapped position -> per-cell histogram (atomics
// give a provisional slot) -> exclusive scan -> scatter -> rank by original
// index within the cell (makes the order deterministic), with positions and
// supports moved into cell order in the same pass.
// Query: a wave takes the queries of one cell together (row_search.h); the
// three cells of a row are one contiguous slice of the sorted arrays unless
// the row wraps around a periodic x boundary.
#include "common.h"
#include "row_search.h"

namespace dsph {

int scan_exclusive(const int32_t* in, int64_t n, int32_t* out, void* ws, size_t ws_bytes, hipStream_t st);
size_t scan_ws(int64_t n);
// Tile run tables of a square list over the grid (k_tile_runs).
int launch_tile_runs(int64_t nq, const dsph_grid* grid, const dsph_domain* domain, const int32_t* cell_start,
                     int32_t* tile_runs, int32_t* tile_n, hipStream_t st);
int scan_read_total(const void* ws, int64_t* total_host, hipStream_t st);

struct GridDev {
  int nc[2];
  float hcell;
};

__device__ __forceinline__ int cell_coord(float x, const Dom& d, int k, const GridDev& g) {
  // clamped in float before the conversion: NaN (fmaxf returns the other
  // operand) and out-of-range coordinates land in an edge cell
  const float f = fminf(fmaxf(floorf(__fdiv_rn(x - d.min[k], g.hcell)), 0.0f), (float)(g.nc[k] - 1));
  return (int)f;
}

__global__ void __launch_bounds__(kBlock) k_cell_keys(const float2* __restrict__ pos, int n, Dom d, GridDev g,
                                                      int32_t* __restrict__ keys, int32_t* __restrict__ slot,
                                                      int32_t* __restrict__ cell_count,
                                                      float2* __restrict__ wrapped) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  const bool valid = i < n;
  int key = 0;
  if (valid) {
    float2 p = pos[i];
    float wx = wrap_coord(p.x, d, 0), wy = wrap_coord(p.y, d, 1);
    int cx = cell_coord(wx, d, 0, g), cy = cell_coord(wy, d, 1, g);
    key = cy * g.nc[0] + cx;
    keys[i] = key;
    if (wrapped) wrapped[i] = make_float2(wx, wy);
  }
  const int sl = wave_slot(cell_count, key, valid);
  if (valid) slot[i] = sl;
}

// Particles of each cell side by side, in any order (`order`, scratch).
__global__ void __launch_bounds__(kBlock) k_cell_scatter(int n, const int32_t* __restrict__ keys,
                                                         const int32_t* __restrict__ slot,
                                                         const int32_t* __restrict__ cell_start,
                                                         int32_t* __restrict__ order) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  order[cell_start[keys[i]] + slot[i]] = i;
}

// The final order, by original index within each cell: particle i goes to its
// rank in the cell (cell_rank, row_search.h), with its sorted position,
// support and rank in the same pass.  A cell over DSPH_CELL_MAX is a diverged
// state that the search reports: it is left unranked.
__global__ void __launch_bounds__(kBlock) k_cell_rank(int n, Dom d, const int32_t* __restrict__ keys,
                                                      const int32_t* __restrict__ slot,
                                                      const int32_t* __restrict__ cell_start,
                                                      const int32_t* __restrict__ order,
                                                      const float2* __restrict__ pos, const float* __restrict__ h,
                                                      int32_t* __restrict__ sort_index, float2* __restrict__ spos,
                                                      float* __restrict__ sh, int32_t* __restrict__ rank) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int p = cell_rank(i, keys[i], slot, cell_start, order, DSPH_CELL_MAX);
  const float2 x = pos[i];
  sort_index[p] = i;
  spos[p] = make_float2(wrap_coord(x.x, d, 0), wrap_coord(x.y, d, 1));
  if (sh) sh[p] = h[i];
  if (rank) rank[i] = p;
}

__global__ void __launch_bounds__(kBlock) k_wrap(const float2* __restrict__ pos, int n, Dom d,
                                                 float2* __restrict__ out) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float2 p = pos[i];
  out[i] = make_float2(wrap_coord(p.x, d, 0), wrap_coord(p.y, d, 1));
}

struct SearchArgs {
  Dom d;
  GridDev g;
  const int32_t* cs;
  const float2* rpos;
  const float* rh;
  const float2* qpos;
  const float* qh;
  float h0;
  int mode;
  int wrapped;
  int nq;
  int nref;
};

// The queries from row0 on, for a launch of their own.
inline SearchArgs queries_from(SearchArgs a, int row0, int64_t rows) {
  a.qpos += row0;
  if (a.qh) a.qh += row0;
  a.nq = (int)rows;
  return a;
}

// A candidate reference particle: wrapped position and support.
struct Cand {
  float2 x;
  float h;
};

__device__ __forceinline__ bool keep_pair(float2 qi, float hi, float2 rj, float hj, const SearchArgs& a) {
  float dx = mod_offset(qi.x - rj.x, a.d, 0);
  float dy = mod_offset(qi.y - rj.y, a.d, 1);
  return within_support(dist2_exact(dx, dy), pick_h(a.mode, hi, hj));
}

// keep_pair for a candidate range that does not cross a periodic seam: the
// plain difference is the min-image offset there (mod_offset returns it
// unchanged), so it is not evaluated.
__device__ __forceinline__ bool keep_pair_near(float2 qi, float hi, float2 rj, float hj, const SearchArgs& a) {
  return within_support(dist2_exact(qi.x - rj.x, qi.y - rj.y), pick_h(a.mode, hi, hj));
}

// A periodic axis of fewer than 7 cells: adjacent cells (the last one up to
// two cells wide) may hold pairs farther apart than half the domain, so
// every range takes mod_offset.  From 7 cells on, two adjacent cells span
// less than L - 5 L / 8 < L / 2, so only ranges across the seam can.
__device__ __forceinline__ bool small_periodic_grid(const SearchArgs& a) {
  return (a.d.periodic[0] && a.g.nc[0] < 7) || (a.d.periodic[1] && a.g.nc[1] < 7);
}

constexpr int kRangeMax = 3 * DSPH_CELL_MAX;

// The rows of cells dy = -1, 0, 1 around the query at qi, one per `part`
// 0..2 (threads of one workgroup share a query's three rows), and the
// query's cell.  A slice longer than three cells of DSPH_CELL_MAX is left out
// and sets `over`, as does a query cell of more than DSPH_CELL_MAX particles
// (a diverged state: the work stays bounded, the caller reports it).
__device__ __forceinline__ CellRow query_cell_row(const SearchArgs& a, float2 qi, int part, int& cell, bool& over) {
  const int ncx = a.g.nc[0], ncy = a.g.nc[1];
  const int cx = cell_coord(qi.x, a.d, 0, a.g), cy = cell_coord(qi.y, a.d, 1, a.g);
  cell = cy * ncx + cx;
  if (part == 1) {
    if (a.cs[cell + 1] - a.cs[cell] > DSPH_CELL_MAX) over = true;  // the query's own cell
  }
  int yy = cy + part - 1;
  if (a.d.periodic[1])
    yy = yy < 0 ? yy + ncy : (yy >= ncy ? yy - ncy : yy);
  else if (yy < 0 || yy >= ncy)
    return CellRow{0, 0, 0, 0};
  const bool wraps = a.d.periodic[0] && (cx == 0 || cx == ncx - 1);
  const bool seam = small_periodic_grid(a) || wraps || yy != cy + part - 1;
  return cell_row(a.cs + (int64_t)yy * ncx, ncx, cx, a.d.periodic[0], seam, kRangeMax, over);
}

__device__ __forceinline__ float2 query_pos(const SearchArgs& a, int i) {
  const float2 p = a.qpos[i];
  return a.wrapped ? p : make_float2(wrap_coord(p.x, a.d, 0), wrap_coord(p.y, a.d, 1));
}

// A workgroup's kRows queries and their cell rows in LDS.
template <int kRows>
struct Queries {
  CellRow rows[3][kRows];
  float x[kRows], y[kRows], h[kRows];
  int cell[kRows];  // -1: past the last query
};

// put(part, r, row) sees every cell row stored.
template <int kRows, class Put>
__device__ __forceinline__ void load_queries(const SearchArgs& a, int i0, Queries<kRows>& Q, bool& over,
                                             const Put& put) {
  const int r = threadIdx.x % kRows, part = threadIdx.x / kRows;
  if (part >= 3) return;
  const int i = i0 + r;
  CellRow cr{0, 0, 0, 0};
  float2 qi = make_float2(0.f, 0.f);
  float hi = 0.f;
  int cell = -1;
  if (i < a.nq) {
    qi = query_pos(a, i);
    hi = h_of(a.qh, i, a.h0);
    cr = query_cell_row(a, qi, part, cell, over);
  }
  Q.rows[part][r] = cr;
  if (part == 0) {
    Q.x[r] = qi.x;
    Q.y[r] = qi.y;
    Q.h[r] = hi;
    Q.cell[r] = cell;
  }
  put(part, r, cr);
}

// The rows of this wave's quarter of the workgroup's queries: value / put /
// spill as scan_rows takes them, with the row's number in the
// workgroup; done(r, n): row r has n entries (one lane per row).  The
// min-image is evaluated only for cell rows at a periodic seam (elsewhere the
// plain difference is the offset).  kH: supports per particle (else the
// uniform a.h0).
template <int kRows, bool kH, bool kDirect, bool kMaySparse, class Value, class Put, class Spill, class Done>
__device__ __forceinline__ void scan_queries(const SearchArgs& a, const Queries<kRows>& Q, int depth,
                                             const Value& value, const Put& put, const Spill& spill,
                                             const Done& done) {
  constexpr int kMine = kRows / 4;
  const int lane = threadIdx.x & 63;
  const int r0 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * kMine;
  const int own = r0 + (lane < kMine ? lane : 0);
  const float qx = Q.x[own], qy = Q.y[own], qh = Q.h[own];
  const int cell = lane < kMine ? Q.cell[own] : -1;
  auto rows = [&](int p, int k) { return Q.rows[p][r0 + k]; };
  const WaveQuery mine{qx, qy, qh, 0};
  auto val = [&](int p, int k, bool first, int j) { return value(p, r0 + k, first, j); };
  auto in = [&](int k, int pos, int v) { put(r0 + k, pos, v); };
  auto out = [&](int k, int pos, int v) { spill(r0 + k, pos, v); };
  int n;
  if (kH) {
    auto keep = [&](const Cand& c, const auto& q, bool seam) {
      const float2 qi = make_float2(q.x(), q.y());
      return seam ? keep_pair(qi, q.h(), c.x, c.h, a) : keep_pair_near(qi, q.h(), c.x, c.h, a);
    };
    n = scan_rows<kMine, kDirect, kMaySparse>(
        cell, depth, rows, mine, [&](int j) { return Cand{a.rpos[j], h_of(a.rh, j, a.h0)}; }, val,
        [&](const Cand& c, const auto& q, bool seam) {
          return LaneTest{__builtin_amdgcn_ballot_w64(keep(c, q, seam)), 0};
        },
        [](const Cand&, const auto&, bool) { return false; }, in, out);
  } else {
    const NearTest within(a.h0);
    auto d2 = [&](const float2& x, const auto& q, bool seam) {
      float dx = q.x() - x.x, dy = q.y() - x.y;
      if (seam) {
        dx = mod_offset(dx, a.d, 0);
        dy = mod_offset(dy, a.d, 1);
      }
      return dist2_exact(dx, dy);
    };
    n = scan_rows<kMine, kDirect, kMaySparse>(
        cell, depth, rows, mine, [&](int j) { return a.rpos[j]; }, val,
        [&](const float2& x, const auto& q, bool seam) { return within(d2(x, q, seam)); },
        [&](const float2& x, const auto& q, bool seam) { return within.exact(d2(x, q, seam)); }, in, out);
  }
  if (cell >= 0) done(own, n);
}

// Supports that differ between particles.
static bool varied_support(const SearchArgs& a) { return a.rh || a.qh; }

// Few enough queries for the 16-query workgroups: with supports per particle
// (a Verlet search, ~36 particles a cell, rows staged 128 deep) a query is
// several times the work and the larger workgroups leave a tail for longer
// (102k queries, count + fill: 55 + 139 us with 16, 87 + 183 with 64).
static bool small_query_set(const SearchArgs& a) {
  return a.nq < (varied_support(a) ? (1 << 18) : kRowSmall);
}

// Whether most cells may be sparse enough for scan_rows_sparse: only then do
// the kernels look for waves that are (0.25 us of a 10 us fill of a 64^2 box).
static bool may_be_sparse(const SearchArgs& a) {
  return (int64_t)a.nref * 9 < (int64_t)a.g.nc[0] * a.g.nc[1] * kSparse;
}

template <int kRows, bool kH, bool kMaySparse>
__global__ void __launch_bounds__(kBlock) k_neighbor_count(SearchArgs a, int32_t* __restrict__ counts) {
  __shared__ Queries<kRows> Q;
  const int i0 = blockIdx.x * kRows;
  bool over = false;  // counted without the skipped ranges; the host checks the cells
  load_queries<kRows>(a, i0, Q, over, [](int, int, const CellRow&) {});
  __syncthreads();
  scan_queries<kRows, kH, false, kMaySparse>(
      a, Q, INT32_MAX, [](int, int, bool, int) { return 0; }, [](int, int, int) {}, [](int, int, int) {},
      [&](int r, int n) { counts[i0 + r] = n; });
}

// With `d16` the 16-bit modular delta (j - i) mod nref of every entry is
// written beside it (rows = reference slots); a delta beyond int16 sets *ovf.
// With `map` (and no d16) the entry is map[j]: the reference slot's index in
// the caller's own order (its sort index), as dsph_remap_neighbors would
// write it afterwards.
__device__ __forceinline__ void put_entry(int32_t* __restrict__ nbr, int16_t* __restrict__ d16,
                                          const int32_t* __restrict__ map, int64_t o, int j, int i, int nref,
                                          bool& bad) {
  nbr[o] = map ? map[j] : j;
  if (d16) {
    int d = j - i;
    const int half = nref / 2;
    if (d > half) d -= nref;
    if (d < -half) d += nref;
    if (d > 32767 || d < -32767) {
      bad = true;
      d = 0;
    }
    d16[o] = (int16_t)d;
  }
}

// Tile slots written by the fill (fixed-width layout, rows = reference
// slots): 256 consecutive rows are a tile of the list; each entry also gets
// its neighbor's slot, j + run_d[u] for the run u holding j.  The tile runs
// come first (they depend on the cells only).
struct FillTiles {
  int32_t* runs;        // run tables, kTileRunStride ints per tile
  int32_t* n;           // particles per tile (set to -1 here when unusable)
  uint16_t* slot;       // per entry, beside nbr
  int cap;
};

// Largest tile whose staged (run << 12 | slot) values stay 16 bits.
constexpr int kFillTileMax = 4095;
constexpr int kNoRun = INT32_MIN;

// Where the rows go.  Fixed width w > 0 (slice s at s * 64 * w, no count
// pass): counts[i] = min(entries, w), *row_ovf set when a row has more
// entries than w (the list is then incomplete).  Else sliced ELL (slice !=
// NULL): the rest of the slice's columns padded with -1.  Else CSR: entries
// at off[i] + n.  Writes stay below `cap` and inside the row's own range.
struct FillOut {
  const int32_t* off;
  const int32_t* slice;
  int32_t* nbr;
  int64_t cap;
  int16_t* d16;
  int32_t* ovf;
  int width;
  int32_t* counts;
  int32_t* row_ovf;
  const int32_t* map;
  int depth;  // staged entries per row (0: CSR)
  // fixed width without a pass before the fill: the slice offsets are written
  // here, and the overflow bits are OR-ed into *row_ovf (not cleared)
  int32_t* slices_out;
};

// Neighbor rows [blockIdx * kRows, + kRows).  In the sliced layouts the first
// `depth` entries of every row are staged in LDS (rows side by side, one
// padding column: a wave writes one row at consecutive entries, so the odd
// stride of kRows + 1 spreads them over the banks) and written column
// by column after the scan, so each store covers whole lines; an entry past
// them is written as it is found.  A CSR row is contiguous and takes no
// staging.  kTiles: with tile slots (T), staged as (u << 12) | slot with u
// the run of the candidate range, as ~j for a range outside the tile's runs
// (tile_n = -1 then); a tile that does not fit T.cap (or kFillTileMax) is
// filled without slots.
template <int kRows, bool kTiles, bool kH, bool kCsr, bool kMaySparse>
__global__ void __launch_bounds__(kBlock) k_neighbor_fill(SearchArgs a, FillOut F, FillTiles T) {
  extern __shared__ int32_t stage[];
  __shared__ Queries<kRows> Q;
  __shared__ int2 run_add[kTiles ? 3 : 1][kTiles ? kRows : 1];
  __shared__ int found[kRows];
  __shared__ int rt_s[kTileMaxRuns], rt_e[kTileMaxRuns], rt_d[kTileMaxRuns];
  __shared__ int offs[kCsr ? kRows + 1 : 1];  // the rows' first entries
  const int i0 = blockIdx.x * kRows;
  const int tile = i0 / kBlock;
  if (kCsr && threadIdx.x <= kRows) offs[threadIdx.x] = F.off[i0 + (int)threadIdx.x < a.nq ? i0 + threadIdx.x : a.nq];
  bool fit = false;
  int R = 0;
  if (kTiles) {
    // a workgroup of the same tile may set tile_n to -1 meanwhile: whoever
    // reads that fills without slots, which no one then reads
    const int S = T.n[tile];
    fit = __syncthreads_and(S >= 0 && S <= T.cap && S <= kFillTileMax);
    if (fit) R = load_run_table(T.runs, tile, rt_s, rt_e, rt_d);
    __syncthreads();
    if (S > kFillTileMax && S <= T.cap && threadIdx.x == 0) T.n[tile] = -1;
  }
  bool bad = false, tbad = false, over = false;
  load_queries<kRows>(a, i0, Q, over, [&](int part, int r, const CellRow& cr) {
    if (kTiles && fit) {
      // what a candidate of each range adds to j for its staged value
      auto run_of = [&](int b, int len) {
        int u = -1;
        for (int k = 0; k < R; ++k) u = (b >= rt_s[k] && b + len <= rt_e[k]) ? k : u;
        if (u < 0 && len > 0) tbad = true;
        return u < 0 ? kNoRun : (u << 12) + rt_d[u];
      };
      run_add[part][r] = make_int2(run_of(cr.b0, cr.len0), run_of(cr.b1, cr.len1 & (kSeamBit - 1)));
    }
  });
  __syncthreads();
  const bool slots = kTiles && fit;
  auto row_of = [&](int i, int64_t& base, int64_t& step, int64_t& len) {
    if (kCsr) {
      base = offs[i - i0];
      step = 1;
      len = (int64_t)offs[i - i0 + 1] - base;
    } else if (F.width > 0) {
      base = (int64_t)(i >> 6) * 64 * F.width + (i & 63);
      step = 64;
      len = F.width;
    } else {
      const int s = i >> 6;
      base = (int64_t)F.slice[s] + (i & 63);
      step = 64;
      len = ((int64_t)F.slice[s + 1] - F.slice[s]) >> 6;
    }
  };
  // slot of the reference particle a staged value stands for
  auto ref_of = [&](int v) { return !slots ? v : (v >= 0 ? (v & 0xfff) - rt_d[v >> 12] : ~v); };
  scan_queries<kRows, kH, kCsr, kMaySparse>(
      a, Q, kCsr ? 0 : F.depth,
      [&](int p, int r, bool first, int j) {
        if (!slots) return j;
        const int2 add = run_add[kTiles ? p : 0][kTiles ? r : 0];
        const int ad = first ? add.x : add.y;
        return ad == kNoRun ? ~j : j + ad;
      },
      [&](int r, int pos, int v) { stage[__umul24(pos, kRows + 1) + r] = v; },
      [&](int r, int pos, int v) {
        const int i = i0 + r;
        int64_t base, step, len;
        row_of(i, base, step, len);
        const int64_t o = base + pos * step;
        if (pos < len && o < F.cap) {
          put_entry(F.nbr, F.d16, F.map, o, ref_of(v), i, a.nref, bad);
          if (slots && v >= 0) T.slot[o] = (uint16_t)(v & 0xfff);
        }
      },
      [&](int r, int n) { found[r] = n; });
  if (kTiles && tbad) T.n[tile] = -1;
  auto overflow = [&](int bit) { F.slices_out ? atomicOr(F.row_ovf, bit) : atomicMax(F.row_ovf, bit); };
  if (F.width > 0 && over) overflow(2);
  if (F.slices_out && threadIdx.x == 0) {
    if ((i0 & 63) == 0) F.slices_out[i0 >> 6] = (i0 >> 6) * 64 * F.width;
    const int last = (a.nq + 63) >> 6;
    if (blockIdx.x == 0) F.slices_out[last] = last * 64 * F.width;
  }
  if (kCsr) {
    if (bad) *F.ovf = 1;
    return;
  }
  __syncthreads();
  const int r = threadIdx.x % kRows, i = i0 + r;
  if (i < a.nq) {
    const int n = found[r];
    int64_t base, step, len;
    row_of(i, base, step, len);
    if (F.width > 0 && threadIdx.x < kRows) {
      // entries past the row's count are never read: no padding
      F.counts[i] = n < len ? n : (int32_t)len;
      if (n > len) overflow(1);
    }
    {
      const int staged = (int)(n < F.depth ? (n < len ? n : len) : (F.depth < len ? F.depth : len));
      constexpr int kStep = kBlock / kRows;
      int c = threadIdx.x / kRows;
      if (!slots && !F.d16 && base + (int64_t)staged * 64 <= F.cap) {
        // plain entries: four gathers through the map in flight
        for (; c + 3 * kStep < staged; c += 4 * kStep) {
          int j[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) j[u] = stage[(c + u * kStep) * (kRows + 1) + r];
          if (F.map) {
#pragma unroll
            for (int u = 0; u < 4; ++u) j[u] = F.map[j[u]];
          }
#pragma unroll
          for (int u = 0; u < 4; ++u) F.nbr[base + (int64_t)(c + u * kStep) * 64] = j[u];
        }
      }
      for (; c < staged; c += kStep) {
        const int64_t o = base + (int64_t)c * 64;
        if (o >= F.cap) break;
        const int v = stage[c * (kRows + 1) + r];
        put_entry(F.nbr, F.d16, F.map, o, ref_of(v), i, a.nref, bad);
        if (slots && v >= 0) T.slot[o] = (uint16_t)(v & 0xfff);
      }
      if (F.width == 0) {
        for (; c < len; c += kBlock / kRows) {
          const int64_t o = base + (int64_t)c * 64;
          if (c >= n && o < F.cap) F.nbr[o] = -1;
        }
      }
    }
  }
  if (bad) *F.ovf = 1;
}

// The list's rows from row0 (a multiple of 256) on.
static FillOut rows_from(FillOut F, int row0) {
  if (F.off) F.off += row0;
  if (F.slice) F.slice += row0 / 64;
  if (F.slices_out) F.slices_out += row0 / 64;
  if (F.width > 0) {
    const int64_t o = (int64_t)row0 * F.width;
    F.nbr += o;
    F.cap -= o;
    F.counts += row0;
  }
  return F;
}

static FillTiles tiles_from(FillTiles T, int row0, int width) {
  T.runs += (int64_t)(row0 / kBlock) * kTileRunStride;
  T.n += row0 / kBlock;
  T.slot += (int64_t)row0 * width;
  return T;
}

template <int kRows, bool kH, bool kMaySparse>
static void launch_fill_rows(const SearchArgs& a, const FillOut& F, const FillTiles* tiles, hipStream_t st) {
  const size_t lds = (size_t)F.depth * (kRows + 1) * sizeof(int32_t);
  auto go = [&](auto kernel) {
    in_launches(a.nq, kBlock / kRows, [&](int row0, int64_t rows) {
      kernel<<<grid_for(rows, kRows), kBlock, lds, st>>>(queries_from(a, row0, rows), rows_from(F, row0),
                                                         tiles ? tiles_from(*tiles, row0, F.width) : FillTiles{});
    });
  };
  if (tiles)
    go(k_neighbor_fill<kRows, true, kH, false, kMaySparse>);
  else if (F.depth > 0)
    go(k_neighbor_fill<kRows, false, kH, false, kMaySparse>);
  else
    go(k_neighbor_fill<kRows, false, kH, true, kMaySparse>);
}

__global__ void __launch_bounds__(kBlock) k_fixed_slices(int nslices, int width, int32_t* __restrict__ slice_off,
                                                         int32_t* __restrict__ row_ovf,
                                                         int32_t* __restrict__ d16_ovf) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s == 0) {
    if (row_ovf) *row_ovf = 0;
    if (d16_ovf) *d16_ovf = 0;
  }
  if (s <= nslices) slice_off[s] = s * 64 * width;
}

__global__ void k_set_flag(int32_t* flag, int v) {
  if (threadIdx.x == 0) *flag = v;
}

static int launch_fill(const SearchArgs& a, FillOut F, const FillTiles* tiles, hipStream_t st) {
  F.depth = F.width > 0 ? (F.width < kRowStage ? F.width : kRowStage) : (F.slice ? kRowStage : 0);
  const bool vary = varied_support(a);
  // several launches (in_launches): their rows count from each one's first, so
  // 16-bit deltas are given up as if one had not fitted, and the slice offsets
  // are written once more
  const bool several = (int64_t)a.nq * 4 > ((int64_t)1 << 31);
  if (several && F.d16) {
    k_set_flag<<<1, 64, 0, st>>>(F.ovf, 1);
    F.d16 = nullptr;
  }
  auto go = [&](auto sparse) {
    constexpr bool S = decltype(sparse)::value;
    if (small_query_set(a))
      vary ? launch_fill_rows<16, true, S>(a, F, tiles, st) : launch_fill_rows<16, false, S>(a, F, tiles, st);
    else
      vary ? launch_fill_rows<64, true, S>(a, F, tiles, st) : launch_fill_rows<64, false, S>(a, F, tiles, st);
  };
  may_be_sparse(a) ? go(std::true_type{}) : go(std::false_type{});
  if (several && F.slices_out) {
    const int nslices = (int)(((int64_t)a.nq + 63) / 64);
    k_fixed_slices<<<grid_for(nslices + 1), kBlock, 0, st>>>(nslices, F.width, F.slices_out, nullptr, nullptr);
  }
  return launch_status();
}

__global__ void __launch_bounds__(kBlock) k_zero_i32(int32_t* __restrict__ a, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) a[i] = 0;
}

// Longest row of every 64-row slice, times 64 (one wave per slice).
__global__ void __launch_bounds__(kBlock) k_slice_len(const int32_t* __restrict__ counts, int nq,
                                                      int32_t* __restrict__ slen) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  int v = i < nq ? counts[i] : 0;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    int t = __shfl_xor(v, o, 64);
    v = t > v ? t : v;
  }
  const int nslices = (nq + 63) >> 6;
  // 64 * (longest row) as int32; a row too long for that saturates, which
  // the scan then reports as an overflow of the int32 slice offsets
  if ((threadIdx.x & 63) == 0 && (i >> 6) < nslices)
    slen[i >> 6] = v > (INT32_MAX >> 6) ? INT32_MAX : (v < 0 ? -1 : v * 64);
}

inline GridDev make_grid(const dsph_grid& g) {
  GridDev o;
  o.nc[0] = g.ncell[0];
  o.nc[1] = g.ncell[1];
  o.hcell = g.hcell;
  return o;
}

inline size_t align256(size_t b) { return (b + 255) / 256 * 256; }

static int check_grid(const dsph_grid* g) {
  if (!g || g->ncell[0] < 1 || g->ncell[1] < 1 || !(g->hcell > 0.0f)) return DSPH_ERR_ARG;
  if ((int64_t)g->ncell[0] * g->ncell[1] >= (int64_t)INT32_MAX) return DSPH_ERR_DIM;
  return DSPH_OK;
}

static int make_search(SearchArgs& a, const dsph_domain* domain, const dsph_grid* grid, const int32_t* cell_start,
                       const float* sorted_pos, const float* sorted_h, int64_t nref, const float* qpos,
                       const float* qh, int64_t nq, int32_t wrapped, float h0, int32_t mode) {
  if (!domain || check_grid(grid) != DSPH_OK) return DSPH_ERR_ARG;
  // one periodic column: a cell row would be the same cell three times, which
  // is no two runs of slots (cell_row)
  if (domain->periodic[0] && grid->ncell[0] < 2) return DSPH_ERR_DIM;
  if (nq < 0 || nref < 0 || nq >= INT32_MAX || nref >= INT32_MAX) return DSPH_ERR_ARG;
  if (mode < 0 || mode > 2) return DSPH_ERR_ARG;
  if (nq > 0 && (!qpos || !cell_start)) return DSPH_ERR_ARG;
  if (nref > 0 && !sorted_pos) return DSPH_ERR_ARG;
  // Supports: a NULL array means the uniform h0, which must then be > 0.
  if (((mode != DSPH_MODE_GATHER && !sorted_h) || (mode != DSPH_MODE_SCATTER && !qh)) && !(h0 > 0.0f))
    return DSPH_ERR_ARG;
  a.d = make_dom(*domain);
  a.g = make_grid(*grid);
  a.cs = cell_start;
  a.rpos = reinterpret_cast<const float2*>(sorted_pos);
  a.rh = sorted_h;
  a.qpos = reinterpret_cast<const float2*>(qpos);
  a.qh = qh;
  a.nref = (int)nref;
  a.h0 = h0;
  a.mode = mode;
  a.wrapped = wrapped != 0;
  a.nq = (int)nq;
  return DSPH_OK;
}

}  // namespace dsph

using namespace dsph;

extern "C" int dsph_grid_dims(const dsph_domain* domain, float hsearch, dsph_grid* grid) {
  if (!domain || !grid || !(hsearch > 0.0f)) return DSPH_ERR_ARG;
  // Cells are kept 0.1% wider than the search radius so that float32
  // rounding of cell coordinates can never separate two particles closer
  // than the radius by two cells.
  const double hs = (double)hsearch * 1.001;
  double hc = 0.0;
  int nc[2];
  for (int k = 0; k < 2; ++k) {
    double L = (double)domain->max[k] - (double)domain->min[k];
    if (!(L > 0.0)) return DSPH_ERR_ARG;
    double n = std::floor(L / hs);
    if (n < 1.0) n = 1.0;
    double side = L / n;
    if (side > hc) hc = side;
  }
  // One square side for both axes: the larger one (reference compute_h).
  float hcell = (float)hc;
  if ((double)hcell < hs) hcell = nextafterf(hcell, INFINITY);
  for (int k = 0; k < 2; ++k) {
    double L = (double)domain->max[k] - (double)domain->min[k];
    double n;
    if (domain->periodic[k]) {
      // A periodic axis is tiled by floor(L/hcell) cells, each >= hcell wide
      // (the last cell absorbs the remainder), so the wrap keeps adjacency.
      // (+1e-4: hcell may have been rounded up by one float ulp; the last
      // cell is then at least (1-1e-4) hcell > the search radius wide.)
      n = std::floor(L / (double)hcell + 1e-4);
      if (n < 3.0) return DSPH_ERR_DIM;
    } else {
      n = std::ceil(L / (double)hcell);
      if (n < 1.0) n = 1.0;
    }
    if (n > 1e8) return DSPH_ERR_DIM;
    nc[k] = (int)n;
  }
  grid->ncell[0] = nc[0];
  grid->ncell[1] = nc[1];
  grid->hcell = hcell;
  grid->pad_ = 0;
  return DSPH_OK;
}

extern "C" size_t dsph_grid_build_workspace(int64_t n, const dsph_grid* grid) {
  if (!grid) return 0;
  int64_t ncell = (int64_t)grid->ncell[0] * grid->ncell[1];
  return align256((size_t)n * 4) * 3 + align256((size_t)ncell * 4) + scan_ws(ncell);
}

extern "C" int dsph_grid_build_wrapped(const dsph_domain* domain, const dsph_grid* grid, const float* pos,
                                       const float* h, int64_t n, int32_t* cell_start, int32_t* sort_index,
                                       int32_t* rank, float* sorted_pos, float* sorted_h, float* wrapped, void* ws,
                                       size_t ws_bytes, void* stream) {
  if (!domain || check_grid(grid) != DSPH_OK || n < 0 || n >= INT32_MAX) return DSPH_ERR_ARG;
  if (!cell_start || (n > 0 && (!pos || !sort_index || !sorted_pos))) return DSPH_ERR_ARG;
  if (sorted_h && !h) return DSPH_ERR_ARG;
  // A periodic axis is only valid when the cells tile it (L/hcell >= nc).
  for (int k = 0; k < 2; ++k) {
    if (domain->periodic[k] && grid->ncell[k] < 3) return DSPH_ERR_DIM;
  }
  const int64_t ncell = (int64_t)grid->ncell[0] * grid->ncell[1];
  if (!ws || ws_bytes < dsph_grid_build_workspace(n, grid)) return DSPH_ERR_CAPACITY;
  hipStream_t st = as_stream(stream);
  char* w = static_cast<char*>(ws);
  int32_t* keys = reinterpret_cast<int32_t*>(w);
  w += align256((size_t)n * 4);
  int32_t* slot = reinterpret_cast<int32_t*>(w);
  w += align256((size_t)n * 4);
  int32_t* order = reinterpret_cast<int32_t*>(w);
  w += align256((size_t)n * 4);
  int32_t* count = reinterpret_cast<int32_t*>(w);
  w += align256((size_t)ncell * 4);
  void* scan_w = w;
  size_t scan_b = scan_ws(ncell);

  Dom d = make_dom(*domain);
  GridDev g = make_grid(*grid);
  // a fill kernel rather than a memset node, so the call can be captured
  k_zero_i32<<<grid_for(ncell > 0 ? ncell : 1), kBlock, 0, st>>>(count, ncell);
  if (n > 0) {
    k_cell_keys<<<grid_for(n), kBlock, 0, st>>>(reinterpret_cast<const float2*>(pos), (int)n, d, g, keys, slot, count,
                                              reinterpret_cast<float2*>(wrapped));
    DSPH_LAUNCH_CHECK();
  }
  int s = scan_exclusive(count, ncell, cell_start, scan_w, scan_b, st);
  if (s != DSPH_OK) return s;
  if (n > 0) {
    k_cell_scatter<<<grid_for(n), kBlock, 0, st>>>((int)n, keys, slot, cell_start, order);
    k_cell_rank<<<grid_for(n), kBlock, 0, st>>>((int)n, d, keys, slot, cell_start, order,
                                                reinterpret_cast<const float2*>(pos), h, sort_index,
                                                reinterpret_cast<float2*>(sorted_pos), sorted_h, rank);
    DSPH_LAUNCH_CHECK();
  }
  return DSPH_OK;
}

extern "C" int dsph_grid_build(const dsph_domain* domain, const dsph_grid* grid, const float* pos, const float* h,
                               int64_t n, int32_t* cell_start, int32_t* sort_index, int32_t* rank,
                               float* sorted_pos, float* sorted_h, void* ws, size_t ws_bytes, void* stream) {
  return dsph_grid_build_wrapped(domain, grid, pos, h, n, cell_start, sort_index, rank, sorted_pos, sorted_h, nullptr,
                                 ws, ws_bytes, stream);
}

extern "C" int dsph_neighbor_count(const dsph_domain* domain, const dsph_grid* grid, const int32_t* cell_start,
                                   const float* sorted_pos, const float* sorted_h, int64_t nref, const float* qpos,
                                   const float* qh, int64_t nq, int32_t qpos_wrapped, float h_uniform, int32_t mode,
                                   int32_t* counts, void* stream) {
  SearchArgs a;
  int s = make_search(a, domain, grid, cell_start, sorted_pos, sorted_h, nref, qpos, qh, nq, qpos_wrapped,
                      h_uniform, mode);
  if (s != DSPH_OK) return s;
  if (nq > 0 && !counts) return DSPH_ERR_ARG;
  if (nq == 0) return DSPH_OK;
  hipStream_t st = as_stream(stream);
  const bool vary = varied_support(a);
  auto launch = [&](auto kernel, int per_block) {
    in_launches(nq, kBlock / per_block, [&](int row0, int64_t rows) {
      kernel<<<grid_for(rows, per_block), kBlock, 0, st>>>(queries_from(a, row0, rows), counts + row0);
    });
  };
  auto go = [&](auto sparse) {
    constexpr bool S = decltype(sparse)::value;
    if (small_query_set(a))
      vary ? launch(k_neighbor_count<16, true, S>, 16) : launch(k_neighbor_count<16, false, S>, 16);
    else
      vary ? launch(k_neighbor_count<64, true, S>, 64) : launch(k_neighbor_count<64, false, S>, 64);
  };
  may_be_sparse(a) ? go(std::true_type{}) : go(std::false_type{});
  return launch_status();
}

extern "C" int dsph_neighbor_fill(const dsph_domain* domain, const dsph_grid* grid, const int32_t* cell_start,
                                  const float* sorted_pos, const float* sorted_h, int64_t nref, const float* qpos,
                                  const float* qh, int64_t nq, int32_t qpos_wrapped, float h_uniform, int32_t mode,
                                  const int32_t* offsets, const int32_t* slice_off, int64_t layout_total,
                                  int32_t* nbr, int64_t capacity, void* stream) {
  SearchArgs a;
  int s = make_search(a, domain, grid, cell_start, sorted_pos, sorted_h, nref, qpos, qh, nq, qpos_wrapped,
                      h_uniform, mode);
  if (s != DSPH_OK) return s;
  if (nq == 0) return DSPH_OK;
  if ((!offsets && !slice_off) || (capacity > 0 && !nbr) || capacity < 0 || layout_total < 0) return DSPH_ERR_ARG;
  if (layout_total > capacity) return DSPH_ERR_CAPACITY;
  return launch_fill(a, FillOut{offsets, slice_off, nbr, capacity}, nullptr, as_stream(stream));
}

extern "C" int dsph_neighbor_fill16(const dsph_domain* domain, const dsph_grid* grid, const int32_t* cell_start,
                                    const float* sorted_pos, const float* sorted_h, int64_t nref, const float* qpos,
                                    const float* qh, int64_t nq, int32_t qpos_wrapped, float h_uniform, int32_t mode,
                                    const int32_t* offsets, const int32_t* slice_off, int64_t layout_total,
                                    int32_t* nbr, int16_t* nbr16, int64_t capacity, int32_t* overflow,
                                    void* stream) {
  SearchArgs a;
  int s = make_search(a, domain, grid, cell_start, sorted_pos, sorted_h, nref, qpos, qh, nq, qpos_wrapped,
                      h_uniform, mode);
  if (s != DSPH_OK) return s;
  if (!overflow || (capacity > 0 && !nbr16)) return DSPH_ERR_ARG;
  // the deltas are j - i modulo n: row i must be reference slot i
  if (nq != nref || !qpos_wrapped) return DSPH_ERR_ARG;
  hipStream_t st = as_stream(stream);
  k_set_flag<<<1, 64, 0, st>>>(overflow, 0);
  DSPH_LAUNCH_CHECK();
  if (nq == 0) return DSPH_OK;
  if ((!offsets && !slice_off) || (capacity > 0 && !nbr) || capacity < 0 || layout_total < 0) return DSPH_ERR_ARG;
  if (layout_total > capacity) return DSPH_ERR_CAPACITY;
  return launch_fill(a, FillOut{offsets, slice_off, nbr, capacity, nbr16, overflow}, nullptr, st);
}

namespace dsph {
static int fill_fixed(const dsph_domain* domain, const dsph_grid* grid, const int32_t* cell_start,
                      const float* sorted_pos, const float* sorted_h, int64_t nref, const float* qpos, const float* qh,
                      int64_t nq, int32_t qpos_wrapped, float h_uniform, int32_t mode, int32_t width, int32_t* counts,
                      int32_t* slice_off, int32_t* nbr, int64_t capacity, int16_t* nbr16, int32_t* delta_overflow,
                      int32_t* row_overflow, const int32_t* map, const FillTiles* tiles, void* stream,
                      bool accumulate = false) {
  SearchArgs a;
  int s = make_search(a, domain, grid, cell_start, sorted_pos, sorted_h, nref, qpos, qh, nq, qpos_wrapped,
                      h_uniform, mode);
  if (s != DSPH_OK) return s;
  if (width < 1 || width > 4096 || !row_overflow || !slice_off || (nbr16 && !delta_overflow)) return DSPH_ERR_ARG;
  // 16-bit deltas are j - i modulo n: row i must be reference slot i
  if (nbr16 && (nq != nref || !qpos_wrapped || map)) return DSPH_ERR_ARG;
  const int64_t nslices = (nq + 63) / 64;
  if (nslices * 64 * (int64_t)width >= INT32_MAX) return DSPH_ERR_ARG;
  if (capacity < nslices * 64 * (int64_t)width) return DSPH_ERR_CAPACITY;
  hipStream_t st = as_stream(stream);
  if (!accumulate || nq == 0) {
    k_fixed_slices<<<grid_for(nslices + 1), kBlock, 0, st>>>((int)nslices, width, slice_off,
                                                            accumulate ? nullptr : row_overflow, delta_overflow);
    DSPH_LAUNCH_CHECK();
  }
  if (nq == 0) return DSPH_OK;
  if (!counts || !nbr) return DSPH_ERR_ARG;
  if (tiles) {
    int s2 = launch_tile_runs(nq, grid, domain, cell_start, tiles->runs, tiles->n, st);
    if (s2 != DSPH_OK) return s2;
  }
  return launch_fill(a,
                     FillOut{nullptr, nullptr, nbr, capacity, nbr16, delta_overflow, width, counts, row_overflow, map,
                             0, accumulate ? slice_off : nullptr},
                     tiles, st);
}
}  // namespace dsph

extern "C" int dsph_neighbor_fill_fixed(const dsph_domain* domain, const dsph_grid* grid, const int32_t* cell_start,
                                        const float* sorted_pos, const float* sorted_h, int64_t nref,
                                        const float* qpos, const float* qh, int64_t nq, int32_t qpos_wrapped,
                                        float h_uniform, int32_t mode, int32_t width, int32_t* counts,
                                        int32_t* slice_off, int32_t* nbr, int64_t capacity, int16_t* nbr16,
                                        int32_t* delta_overflow, int32_t* row_overflow, void* stream) {
  return fill_fixed(domain, grid, cell_start, sorted_pos, sorted_h, nref, qpos, qh, nq, qpos_wrapped, h_uniform, mode,
                    width, counts, slice_off, nbr, capacity, nbr16, delta_overflow, row_overflow, nullptr, nullptr,
                    stream);
}

extern "C" int dsph_neighbor_fill_fixed_map(const dsph_domain* domain, const dsph_grid* grid,
                                            const int32_t* cell_start, const float* sorted_pos,
                                            const float* sorted_h, int64_t nref, const float* qpos, const float* qh,
                                            int64_t nq, int32_t qpos_wrapped, float h_uniform, int32_t mode,
                                            int32_t width, int32_t* counts, int32_t* slice_off, int32_t* nbr,
                                            int64_t capacity, const int32_t* map, int32_t* row_overflow,
                                            void* stream) {
  if (nref > 0 && !map) return DSPH_ERR_ARG;
  return fill_fixed(domain, grid, cell_start, sorted_pos, sorted_h, nref, qpos, qh, nq, qpos_wrapped, h_uniform, mode,
                    width, counts, slice_off, nbr, capacity, nullptr, nullptr, row_overflow, map, nullptr, stream);
}

extern "C" int dsph_neighbor_fill_fixed_or(const dsph_domain* domain, const dsph_grid* grid,
                                           const int32_t* cell_start, const float* sorted_pos, const float* sorted_h,
                                           int64_t nref, const float* qpos, const float* qh, int64_t nq,
                                           int32_t qpos_wrapped, float h_uniform, int32_t mode, int32_t width,
                                           int32_t* counts, int32_t* slice_off, int32_t* nbr, int64_t capacity,
                                           const int32_t* map, int32_t* row_overflow, void* stream) {
  return fill_fixed(domain, grid, cell_start, sorted_pos, sorted_h, nref, qpos, qh, nq, qpos_wrapped, h_uniform, mode,
                    width, counts, slice_off, nbr, capacity, nullptr, nullptr, row_overflow, map, nullptr, stream,
                    true);
}

extern "C" int dsph_neighbor_fill_fixed_tiles(const dsph_domain* domain, const dsph_grid* grid,
                                              const int32_t* cell_start, const float* sorted_pos,
                                              const float* sorted_h, int64_t nref, const float* qpos,
                                              const float* qh, int64_t nq, int32_t qpos_wrapped, float h_uniform,
                                              int32_t mode, int32_t width, int32_t* counts, int32_t* slice_off,
                                              int32_t* nbr, int64_t capacity, int16_t* nbr16,
                                              int32_t* delta_overflow, int32_t tile_cap, uint16_t* slot,
                                              int64_t slot_capacity, int32_t* tile_runs, int32_t* tile_n,
                                              int32_t* row_overflow, void* stream) {
  // the tiles of a list whose rows are the reference slots
  if (nq != nref || !qpos_wrapped) return DSPH_ERR_ARG;
  if (tile_cap < 1 || tile_cap > DSPH_TILE_MAX_CAP || slot_capacity < 0) return DSPH_ERR_ARG;
  if (nq > 0 && (!slot || !tile_runs || !tile_n)) return DSPH_ERR_ARG;
  if (width >= 1 && slot_capacity < ((nq + 63) / 64) * 64 * (int64_t)width) return DSPH_ERR_CAPACITY;
  FillTiles t{tile_runs, tile_n, slot, tile_cap};
  return fill_fixed(domain, grid, cell_start, sorted_pos, sorted_h, nref, qpos, qh, nq, qpos_wrapped, h_uniform, mode,
                    width, counts, slice_off, nbr, capacity, nbr16, delta_overflow, row_overflow, nullptr, &t,
                    stream);
}

extern "C" size_t dsph_sell_workspace(int64_t nq) {
  int64_t ns = (nq + 63) / 64;
  return align256((size_t)(ns > 0 ? ns : 1) * 4) + scan_ws(ns);
}

extern "C" int dsph_sell_layout(const int32_t* counts, int64_t nq, int32_t* slice_off, int64_t* total_host,
                                void* ws, size_t ws_bytes, void* stream) {
  if (nq < 0 || nq >= INT32_MAX || !slice_off || (nq > 0 && !counts)) return DSPH_ERR_ARG;
  if (!ws || ws_bytes < dsph_sell_workspace(nq)) return DSPH_ERR_CAPACITY;
  hipStream_t st = as_stream(stream);
  const int64_t ns = (nq + 63) / 64;
  int32_t* slen = static_cast<int32_t*>(ws);
  char* scan_w = static_cast<char*>(ws) + align256((size_t)(ns > 0 ? ns : 1) * 4);
  if (nq > 0) {
    k_slice_len<<<grid_for(nq), kBlock, 0, st>>>(counts, (int)nq, slen);
    DSPH_LAUNCH_CHECK();
  }
  int s = scan_exclusive(slen, ns, slice_off, scan_w, scan_ws(ns), st);
  if (s != DSPH_OK) return s;
  if (total_host) return scan_read_total(scan_w, total_host, st);
  return DSPH_OK;
}

extern "C" int dsph_wrap_positions(const dsph_domain* domain, const float* pos, int64_t n, float* out, void* stream) {
  if (!domain || n < 0 || n >= INT32_MAX) return DSPH_ERR_ARG;
  if (n == 0) return DSPH_OK;
  if (!pos || !out) return DSPH_ERR_ARG;
  k_wrap<<<grid_for(n), kBlock, 0, as_stream(stream)>>>(reinterpret_cast<const float2*>(pos), (int)n,
                                                        make_dom(*domain), reinterpret_cast<float2*>(out));
  return launch_status();
}

namespace dsph {
__global__ void __launch_bounds__(kBlock) k_remap(int32_t* __restrict__ nbr, int64_t entries,
                                                  const int32_t* __restrict__ map, int nmap) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= entries) return;
  const int32_t j = nbr[e];
  nbr[e] = (j >= 0 && j < nmap) ? map[j] : -1;
}
}  // namespace dsph

extern "C" int dsph_remap_neighbors(int32_t* nbr, int64_t entries, const int32_t* map, int64_t nmap, void* stream) {
  if (entries < 0 || nmap < 0 || nmap >= INT32_MAX || (entries > 0 && (!nbr || !map))) return DSPH_ERR_ARG;
  if (entries == 0) return DSPH_OK;
  const int64_t nb = (entries + kBlock - 1) / kBlock;
  if (nb >= INT32_MAX) return DSPH_ERR_ARG;
  k_remap<<<(int)nb, kBlock, 0, as_stream(stream)>>>(nbr, entries, map, (int)nmap);
  return launch_status();
}
