// Neighbor rows of the cell-list search, one cell at a time (gfx950).
//
// Queries arrive in cell order (up to the drift within a time step), so
// consecutive ones share the cell and with it all candidates.  A wave takes
// the queries of a cell together: its lanes hold the candidates of the three
// cell rows in registers (~48 of 64 lanes per row at 16 particles a cell)
// and the queries pass by one after the other as scalars.  A candidate test
// is then five VALU operations for 64 pairs, the kept mask is the compare's
// own result, and a kept candidate's place in the row is a count of the mask
// below it: the row keeps the order of a scan by one thread.
//
// One thread per query took 108 VALU issue slots per row (divergent ranges,
// per-lane candidate loads, exec-mask bookkeeping) and left searches below
// ~300k queries latency-bound (64 waves of ~150 dependent steps for a 64^2
// box; seam lanes ran nine ranges after the others' three).  Sixteen lanes
// per query fixed the latency but took ~150 slots per row.  Fixed-width fill,
// periodic box, one thread per query -> this: 64^2 93 -> 11 us, 256^2 99 ->
// 27, 512^2 109 -> 65, 1024^2 290 -> 178 us (with tile slots 313 -> 240);
// 1024^2 without a seam 160 -> 133 us.  Bound by scalar and vector issue.
#pragma once

#include <type_traits>

#include "common.h"

namespace dsph {

constexpr int kRowStage = 128;  // deepest staged row of the layouts without a fixed width

// Queries per workgroup of 256 threads, a quarter of them per wave: 64 (a
// slice of the sliced layout) share a cell's candidates between up to 16
// queries; 16 keeps every CU busy while there are fewer than kRowSmall
// (16 against 64 queries, us: 64^2 10.4 / 12.5, 256^2 22.4 / 18.0, 512^2
// 72 / 46).
constexpr int kRowSmall = 1 << 15;

// Candidates of a query (its three cell rows) up to which its wave takes
// scan_rows_sparse: 9 cells of 5 to 10.  Count and CSR fill in us, queries in
// cell order, bounds of 48 / 96 / 128: 1M at 5 a cell 85 + 181 / 60 + 93 / -,
// 1M at 16 a cell 88 + 206 / 88 + 207 / 90 + 206 (144 candidates: above).
constexpr int kSparse = 96;

// The candidates of one row of cells, at most two runs of sorted slots (two
// when the row wraps around the periodic x boundary), in scan order.  `len1`
// carries the seam flag: pairs of these ranges may cross a periodic seam.
struct CellRow {
  int b0, len0, b1, len1;
};
constexpr int kSeamBit = 1 << 30;

// Ranges of the cells cx-1 .. cx+1 of the row whose first cell is cs[0].  A
// slice longer than `longest` is left out and sets `over`, cell by cell in a
// wrapping row.  A periodic row has at least two cells (searches refuse one).
__device__ __forceinline__ CellRow cell_row(const int32_t* __restrict__ cs, int ncx, int cx, bool periodic_x,
                                            bool seam, int longest, bool& over) {
  CellRow r;
  r.len1 = 0;
  r.b1 = 0;
  auto clip = [&](int b, int e) {
    const int l = e - b;
    if (l > longest) {
      over = true;
      return 0;
    }
    return l;
  };
  if (!(periodic_x && (cx == 0 || cx == ncx - 1))) {
    const int x0 = cx - 1 < 0 ? 0 : cx - 1;
    const int x1 = cx + 1 > ncx - 1 ? ncx - 1 : cx + 1;
    r.b0 = cs[x0];
    r.len0 = clip(r.b0, cs[x1 + 1]);
  } else {
    // dx = -1, 0, 1: two of the three cells are neighbors in memory
    const int ca = cx == 0 ? ncx - 1 : cx - 1, cb = cx, cc = cx == ncx - 1 ? 0 : cx + 1;
    const int ba = cs[ca], bb = cs[cb], bc = cs[cc];
    const int la = clip(ba, cs[ca + 1]), lb = clip(bb, cs[cb + 1]), lc = clip(bc, cs[cc + 1]);
    if (cx == 0) {
      r.b0 = ba;
      r.len0 = la;
      r.b1 = lb > 0 ? bb : bc;
      r.len1 = lb + lc;
    } else {
      r.b0 = la > 0 ? ba : bb;
      r.len0 = la + lb;
      r.b1 = bc;
      r.len1 = lc;
    }
  }
  if (seam) r.len1 |= kSeamBit;
  return r;
}

// A candidate test of 64 lanes: the lanes that keep theirs, and the lanes
// that only the exact expression decides.
struct LaneTest {
  unsigned long long in, band;
};

// Sorted slot of particle i of cell `key`: the cell's first slot plus the
// count of smaller indices among its particles order[cell_start[key] ..].  One
// thread per particle with eight loads in flight; one thread per cell (a
// serial sort of 16 to 36 entries) took 14 us at 4k particles and 365 us on a
// grid of 36 a cell.  A cell of more than `longest` particles stays in
// provisional order.
__device__ __forceinline__ int cell_rank(int i, int key, const int32_t* __restrict__ slot,
                                         const int32_t* __restrict__ cell_start, const int32_t* __restrict__ order,
                                         int longest) {
  const int b = cell_start[key], e = cell_start[key + 1];
  if (e - b > longest) return b + slot[i];
  int r = 0;
  for (int a = b; a < e; a += 8) {
    int v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = order[a + u < e ? a + u : e - 1];
#pragma unroll
    for (int u = 0; u < 8; ++u) r += (a + u < e && v[u] < i) ? 1 : 0;
  }
  return b + r;
}

// d2 against one support h for all pairs, the thresholds of within_support:
// the compare's own masks.
struct NearTest {
  float h, lo, hi;
  __device__ __forceinline__ explicit NearTest(float support) : h(support) {
    const float hh = h * h;
    lo = hh * 0.999999f;
    hi = hh * 1.000001f;
  }
  __device__ __forceinline__ LaneTest operator()(float d2) const {
    LaneTest t;
    t.in = __builtin_amdgcn_ballot_w64(d2 < lo);
    t.band = ~(t.in | __builtin_amdgcn_ballot_w64(d2 > hi));
    return t;
  }
  __device__ __forceinline__ bool exact(float d2) const { return __fdiv_rn(sqrt_rn(d2), h) <= 1.0f; }
};

__device__ __forceinline__ float lane_value(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// Lanes [0, n) of the wave (n <= 0: none, n >= 64: all).
__device__ __forceinline__ unsigned long long first_lanes(int n) {
  return n >= 64 ? ~0ull : (n <= 0 ? 0ull : (1ull << n) - 1ull);
}

// Query k of the wave (the same k in all lanes) whose values lie in lane k, as
// scalars where they are used.
struct WaveQuery {
  float vx, vy, vh;
  int k;
  __device__ __forceinline__ float x() const { return lane_value(vx, k); }
  __device__ __forceinline__ float y() const { return lane_value(vy, k); }
  __device__ __forceinline__ float h() const { return lane_value(vh, k); }
};

// The query of this lane.
struct LaneQuery {
  float vx, vy, vh;
  int k;
  __device__ __forceinline__ float x() const { return vx; }
  __device__ __forceinline__ float y() const { return vy; }
  __device__ __forceinline__ float h() const { return vh; }
};

// The neighbor rows of the queries in `todo` (bit k: the query of lane k,
// k < 32, whose cell is `cell` there); returns each query's row length in its
// lane.  mine: the query of this lane (lanes without one: any); rows(p, k):
// cell row p = 0..2 of query k; load(j): candidate j;
// value(p, k, first, j): what a row gets for candidate j of cell row p of the
// queries in query k's cell (first: of its first range); test(c, q, seam): a
// LaneTest of every lane's candidate c against its query q (WaveQuery or
// LaneQuery), exact(c, q, seam) the expression itself; put(k, pos, value): entry pos < depth of row
// k, spill(k, pos, value): entry pos >= depth (kDirect: every entry).  All 64 lanes call it; no
// barrier inside.
//
// Vector and scalar issue are about equal here (~35 and ~33 a row), so the
// masks of a row's three cell rows are formed first and the checks that are
// rarely true (a pair in the band, a row past `depth`) made once per row.
template <bool kDirect, class Rows, class Load, class Value, class Test, class Exact, class Put,
          class Spill>
__device__ __forceinline__ int scan_rows_by_cell(uint32_t todo, int cell, int depth, const Rows& rows,
                                                 const WaveQuery& own, const Load& load, const Value& value,
                                                 const Test& test, const Exact& exact, const Put& put,
                                                 const Spill& spill) {
  using Cand = decltype(load(0));
  const int lane = threadIdx.x & 63;
  int found = 0;
  while (todo) {
    const int f = __ffs(todo) - 1;
    const int c = __builtin_amdgcn_readlane(cell, f);
    uint32_t same = (uint32_t)__builtin_amdgcn_ballot_w64(cell == c) & todo;
    todo &= ~same;
    CellRow R[3];
    int tot[3], longest = 0;
    bool seam = false;
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      const CellRow v = rows(p, f);
      R[p].b0 = __builtin_amdgcn_readfirstlane(v.b0);
      R[p].len0 = __builtin_amdgcn_readfirstlane(v.len0);
      R[p].b1 = __builtin_amdgcn_readfirstlane(v.b1);
      R[p].len1 = __builtin_amdgcn_readfirstlane(v.len1);
      seam = seam || (R[p].len1 & kSeamBit);
      tot[p] = R[p].len0 + (R[p].len1 & (kSeamBit - 1));
      longest = tot[p] > longest ? tot[p] : longest;
    }
    auto place_of = [](unsigned long long m, int n) {
      return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, n));
    };
    auto decide = [&](LaneTest t, const Cand& cd, const auto& q, bool at_seam) {
      return t.in | (__builtin_amdgcn_ballot_w64(exact(cd, q, at_seam)) & t.band);
    };
    // one query, candidates read as they come: any cell row
    auto general = [&](int k) {
      int n = 0;
      const WaveQuery qk{own.vx, own.vy, own.vh, k};
      for (int p = 0; p < 3; ++p) {
        const CellRow v = rows(p, f);
        const int b0 = __builtin_amdgcn_readfirstlane(v.b0), l0 = __builtin_amdgcn_readfirstlane(v.len0);
        const int b1 = __builtin_amdgcn_readfirstlane(v.b1), l1 = __builtin_amdgcn_readfirstlane(v.len1);
        const int total = l0 + (l1 & (kSeamBit - 1));
        const bool at_seam = (l1 & kSeamBit) != 0;
        for (int t0 = 0; t0 < total; t0 += 64) {
          const int t = t0 + lane, j = t + (t < l0 ? b0 : b1 - l0);
          const Cand cd = load(t < total ? j : 0);
          const unsigned long long m = decide(test(cd, qk, at_seam), cd, qk, at_seam) & first_lanes(total - t0);
          const int pos = place_of(m, n);
          if (__builtin_amdgcn_inverse_ballot_w64(m)) {
            if (kDirect || pos >= depth)
              spill(k, pos, value(p, k, t < l0, j));
            else
              put(k, pos, value(p, k, t < l0, j));
          }
          n += __popcll(m);
        }
      }
      return n;
    };
    // all queries of the cell, candidates in registers (up to 64 NC a row);
    // the cells of a seam have two ranges a row and take the min-image
    auto resident = [&](auto chunks, auto seam_cell) {
      constexpr int NC = decltype(chunks)::value;
      constexpr bool kSeam = decltype(seam_cell)::value;
      Cand cand[3][NC];
      int val[3][NC];
#pragma unroll
      for (int p = 0; p < 3; ++p) {
#pragma unroll
        for (int q = 0; q < NC; ++q) {
          const int t = q * 64 + lane;
          const bool first = !kSeam || t < R[p].len0;
          const int j = t + (first ? R[p].b0 : R[p].b1 - R[p].len0);
          cand[p][q] = load(t < tot[p] ? j : 0);
          val[p][q] = value(p, f, first, j);
        }
      }
      while (same) {
        const int k = __ffs(same) - 1;
        same &= same - 1;
        const WaveQuery qk{own.vx, own.vy, own.vh, k};
        unsigned long long m[3][NC];
        unsigned long long band = 0;
#pragma unroll
        for (int p = 0; p < 3; ++p) {
#pragma unroll
          for (int q = 0; q < NC; ++q) {
            const unsigned long long live = first_lanes(tot[p] - q * 64);
            const LaneTest t = test(cand[p][q], qk, kSeam && (R[p].len1 & kSeamBit));
            m[p][q] = t.in & live;
            band |= t.band & live;
          }
        }
        if (band) {
#pragma unroll
          for (int p = 0; p < 3; ++p) {
#pragma unroll
            for (int q = 0; q < NC; ++q) {
              const bool at_seam = kSeam && (R[p].len1 & kSeamBit);
              m[p][q] = decide(test(cand[p][q], qk, at_seam), cand[p][q], qk, at_seam) & first_lanes(tot[p] - q * 64);
            }
          }
        }
        int n = 0;
#pragma unroll
        for (int p = 0; p < 3; ++p) {
#pragma unroll
          for (int q = 0; q < NC; ++q) n += __popcll(m[p][q]);
        }
        found = lane == k ? n : found;
        if (!kDirect && n > depth) {
          general(k);
          continue;
        }
        n = 0;
#pragma unroll
        for (int p = 0; p < 3; ++p) {
#pragma unroll
          for (int q = 0; q < NC; ++q) {
            const int pos = place_of(m[p][q], n);
            if (__builtin_amdgcn_inverse_ballot_w64(m[p][q])) {
              if (kDirect)
                spill(k, pos, val[p][q]);
              else
                put(k, pos, val[p][q]);
            }
            n += __popcll(m[p][q]);
          }
        }
      }
    };
    // rows beyond 128 candidates (a 1.5 h Verlet cell row has ~108) are read
    // again for every query
    using std::integral_constant;
    if (longest == 0 || longest > 128) {
      while (same) {
        const int k = __ffs(same) - 1;
        same &= same - 1;
        const int n = general(k);
        found = lane == k ? n : found;
      }
    } else if (longest > 64) {
      if (seam)
        resident(integral_constant<int, 2>{}, std::true_type{});
      else
        resident(integral_constant<int, 2>{}, std::false_type{});
    } else if (seam) {
      resident(integral_constant<int, 1>{}, std::true_type{});
    } else {
      resident(integral_constant<int, 1>{}, std::false_type{});
    }
  }
  return found;
}

// scan_rows_by_cell for queries whose cell rows hold few candidates (up to
// kSparse each): all kMine queries of the wave at once, 64 / kMine lanes each
// over the candidates of the three cell rows end to end, four loads in flight.
// A cell's candidates in registers leave most lanes idle there, and its set-up
// (~330 cycles) comes with every one or two queries.  1M queries in cell order,
// count + CSR fill + fixed-width fill in us, by cell only / this: 0.5 a cell
// 157 + 256 + 225 / 32 + 42 + 49, 2 a cell 120 + 228 + 186 / 42 + 60 + 65, 5 a
// cell 92 + 204 + 156 / 60 + 93 + 89 (one thread per query: 29 + 45 + 47, 42 +
// 72 + 72, 57 + 127 + 108).
template <int kMine, bool kDirect, class Rows, class Load, class Value, class Test, class Exact, class Put,
          class Spill>
__device__ __forceinline__ int scan_rows_sparse(int end0, int end1, int total, bool seam, int depth, const Rows& rows,
                                                const LaneQuery& q, const Load& load, const Value& value,
                                                const Test& test, const Exact& exact, const Put& put,
                                                const Spill& spill) {
  constexpr int kLanes = 64 / kMine;
  const int lane = threadIdx.x & 63, k = lane / kLanes, g = lane % kLanes;
  int n = 0;
  using Cand = decltype(load(0));
  constexpr int U = 4;
  for (int t0 = 0; __builtin_amdgcn_ballot_w64(t0 < total); t0 += U * kLanes) {
    Cand c[U];
    int p[U], j[U];
    bool first[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int t = t0 + u * kLanes + g;
      p[u] = t < end0 ? 0 : (t < end1 ? 1 : 2);
      const CellRow v = rows(p[u], k);
      const int w = t - (p[u] == 0 ? 0 : (p[u] == 1 ? end0 : end1));
      first[u] = w < v.len0;
      j[u] = w + (first[u] ? v.b0 : v.b1 - v.len0);
      c[u] = load(t < total ? j[u] : 0);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const LaneTest in = test(c[u], q, seam);
      unsigned long long m = in.in;
      if (in.band) m |= __builtin_amdgcn_ballot_w64(exact(c[u], q, seam)) & in.band;
      m &= __builtin_amdgcn_ballot_w64(t0 + u * kLanes + g < total);
      const uint32_t mine = (uint32_t)(m >> (lane & ~(kLanes - 1))) & ((1u << kLanes) - 1u);
      if ((mine >> g) & 1u) {
        const int pos = n + __popc(mine & ((1u << g) - 1u));
        if (kDirect || pos >= depth)
          spill(k, pos, value(p[u], k, first[u], j[u]));
        else
          put(k, pos, value(p[u], k, first[u], j[u]));
      }
      n += __popc(mine);
    }
  }
  return __shfl(n, (lane % kMine) * kLanes, 64);
}

// The neighbor rows of a wave's kMine queries, by whichever of the two suits
// their candidates; arguments as for scan_rows_by_cell.
template <int kMine, bool kDirect, bool kMaySparse, class Rows, class Load, class Value, class Test, class Exact,
          class Put, class Spill>
__device__ __forceinline__ int scan_rows(int cell, int depth, const Rows& rows, const WaveQuery& own, const Load& load,
                                         const Value& value, const Test& test, const Exact& exact, const Put& put,
                                         const Spill& spill) {
  if constexpr (kMaySparse) {
    const int k = (threadIdx.x & 63) / (64 / kMine);
    int end[3], flags = 0, total = 0;
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      const CellRow v = rows(p, k);
      total += v.len0 + (v.len1 & (kSeamBit - 1));
      end[p] = total;
      flags |= v.len1;
    }
    if (__builtin_amdgcn_ballot_w64(total > kSparse) == 0) {
      // off a seam the min-image is the plain difference: all lanes take it
      // when one needs it
      const bool seam = __builtin_amdgcn_ballot_w64((flags & kSeamBit) != 0) != 0;
      const LaneQuery q{__shfl(own.vx, k, 64), __shfl(own.vy, k, 64), __shfl(own.vh, k, 64), k};
      return scan_rows_sparse<kMine, kDirect>(end[0], end[1], total, seam, depth, rows, q, load, value, test, exact,
                                              put, spill);
    }
  }
  const uint32_t todo = (uint32_t)__builtin_amdgcn_ballot_w64(cell >= 0);
  return scan_rows_by_cell<kDirect>(todo, cell, depth, rows, own, load, value, test, exact, put, spill);
}

}  // namespace dsph
