// kmi_march2d.h — K time steps of a D2Q9 lattice per pass, held in the registers of one wave.
//
// A wave owns a strip of columns, one per lane, and marches up y.  Level l (1 … K) is the
// state after l steps; in iteration s level l evaluates row s − (l − 1), so the row above it
// of level l − 1 has just been evaluated and the two rows it needs besides (its own row and
// the one below) wait in registers.  Level 1 pulls from HBM; the x neighbours of the others
// come from the neighbouring lanes (whole-wave DPP shifts), so no level touches LDS and no
// barrier is needed anywhere.  A lane of level l is exact when both neighbours of level l − 1
// are, so each inner edge of a strip loses one column per level: K − 1 lanes a side are halo
// and 64 − 2 (K − 1) columns are written (an edge on a wall needs no halo).  The rows above
// and below a chunk of rows are evaluated again the same way.
//
// What bounds it: the dependent loads and arithmetic of two waves per SIMD (the rows held take
// the registers of more), near the rate of memory in FP64.  Counters of a 2048² BGK launch, four
// steps: F64 154 µs for 360 MB read and 310 MB written (302 MB each without halos), 4.4 of the
// 5.5 TB/s of a copy, the VALU busy 50 % of the time; a wave issues in 40 % of its cycles, waits
// for its turn in 30 % and for a dependency in 30 %.  F32S: VALU busy 67 %, 53 / 17 / 30 %.
// Instructions, F32S MRT, K = 4: 443 per wave and iteration for 58 columns × 4 steps, against 405
// for 256 cells × 2 steps plus their halo and two barriers in the tile kernel.  Why registers
// and not LDS: a tile of W × H cells with a K-cell ring in LDS evaluates (W + 2K)(H + 2K) / WH
// cells (1.8 for 24×24, K = 4) and holds every wave at two barriers per step; a strip
// evaluates 64/58 in x and (rows + 3)/rows in y, and no wave waits for another.
//
// Per cell and step the arithmetic is the single-step kernel's, every intermediate value
// passes through the storage rounding, and each link from beyond a wall takes the cell's own
// opposite population of the previous level: bit-identical to K single-step launches.
#pragma once

#include "kmi_cell.h"

namespace kmi {

// Value of the lane below / above (whole wave; the outermost lane keeps its own value, which
// only ever reaches halo lanes).
template <int CTRL>
KMI_DEV int dpp_move(int v) {
  return __builtin_amdgcn_update_dpp(v, v, CTRL, 0xf, 0xf, false);
}
template <int CTRL, class R>
KMI_DEV R wave_shift(R v) {
  if constexpr (sizeof(R) == 4) {
    return __builtin_bit_cast(R, dpp_move<CTRL>(__builtin_bit_cast(int, v)));
  } else {
    const long long b = __builtin_bit_cast(long long, v);
    const unsigned lo = unsigned(dpp_move<CTRL>(int(b)));
    const int hi = dpp_move<CTRL>(int(b >> 32));
    return __builtin_bit_cast(R, (static_cast<long long>(hi) << 32) | lo);
  }
}
template <class R>
KMI_DEV R from_left(R v) { return wave_shift<0x138>(v); }  // wave_shr:1 — lane i takes lane i − 1
template <class R>
KMI_DEV R from_right(R v) { return wave_shift<0x130>(v); }  // wave_shl:1 — lane i takes lane i + 1

// Strips of a row of n columns for K levels: m strips, strip s covering [start(s), start(s + 1)).
// Between walls the two outer strips need no halo on their wall side, so they are K − 1 wider.
struct MarchStrips {
  int n, m, off;  // off: K − 1 between walls, 0 on a periodic axis
  KMI_HD int start(int s) const {
    return s <= 0 ? 0 : (s >= m ? n : off + int((long long)s * (n - 2 * off) / m));
  }
};
KMI_HD MarchStrips march_strips(int n, int K, bool periodic) {
  const int w = 64 - 2 * (K - 1), off = periodic ? 0 : K - 1;
  const int inner = n - 2 * off;
  const int m = inner <= w ? 1 : (inner + w - 1) / w;
  return MarchStrips{n, m, m == 1 ? 0 : off};
}

// Waves per SIMD the register budget is set for (K = 4: 111–138 VGPRs in FP32, 203–238 in
// FP64).  A tighter bound spills, and each reload waits for the row that is being pulled
// ahead: an earlier build that reloaded two registers per iteration at four waves ran 2048²
// F32S at 36–50 µs a step instead of 22.
template <int ST, int K>
constexpr int march_waves() { return sizeof(typename Store<ST>::real) == 4 ? (K >= 4 ? 3 : 4) : 2; }

// Rows per piece: `pieces(rows)` pieces of at most `rows` rows on 1024 SIMDs, `resident` of
// them per SIMD at a time.  A SIMD issues for its waves in turn, so a launch takes about
// (pieces per SIMD, rounded up) × (rows + 3) iterations — the 2 (K − 1) extra rows of a piece
// evaluate half their levels on average.  With more pieces than fit at once the last ones end
// in an uneven tail, about 1.5 pieces long; one wave alone issues about 10 % less than two.
// Measured (µs per step, periodic): 2048² F64 at 12 / 24 / 40 rows 46.9 / 44.8 / 40.5, 1024²
// F64 at 12 / 19 / 32 rows 12.3 / 11.3 / 14.6, 1024² F32 at 10 / 19 / 32 rows 8.1 / 9.1 / 12.3.
template <class Pieces>
inline int march_rows(int ny, int resident, Pieces&& pieces) {
  int best = 4;
  double cost = 1e300;
  for (int rows = 4; rows <= 128 && (rows == 4 || rows <= ny); ++rows) {
    const long long n = pieces(rows);
    const double per_simd = double((n + 1023) / 1024);
    double c = (per_simd + (n > 1024LL * resident ? 1.5 : 0.0)) * (rows + 3);
    if (n <= 1024) c *= 1.1;
    if (c < cost) cost = c, best = rows;
  }
  return best;
}

// Levels' carried rows: cc, cp, cm the c_y = 0, +1, −1 populations of the newest row but one
// of a level (the own row of the level above it), cq the c_y = +1 populations of the row
// below that.
template <class R>
struct MarchCarry {
  R cc[3], cp[3], cm[3], cq[3];
};

// Dom: the lattice (single or one of a batch) —
//   nx, ny, perx, pery               sizes, periodic axes
//   src(q), dst(q)                   population planes (uniform pointers)
//   ladd<q, ROWS>(v, wxm, wxp, wym, wyp)  Ladd terms of the faces a bounced link crosses
//   closures<ROWS>(fp, i, j)         Zou–He closures of the faces a cell lies on (ROWS: the
//                                    cell may lie on a y face; else on an x face at most)
//   collide(fp, fo)
// WX: some evaluated cell lies on a non-periodic x face.  Cells on y faces come up only in
// the first and last iterations of a chunk, which run the general form of an iteration.
template <int ST, int K, bool WX, class Dom>
KMI_DEV void march2d(const Dom& d, int xs, int xe, int y0, int y1) {
  using S = Store<ST>;
  using E = typename S::elem;
  using R = typename S::real;
  constexpr unsigned ES = sizeof(E);
  const int lane = threadIdx.x & 63;
  const int nx = d.nx, ny = d.ny;
  const bool perx = d.perx, pery = d.pery;
  // columns: lane 0 at xl, the last one that is needed at xr (lanes beyond repeat it)
  const int xl = (WX && !perx && xs == 0) ? 0 : xs - (K - 1);
  const int xr = (WX && !perx && xe == nx) ? nx - 1 : xe - 1 + (K - 1);
  const int ux = min(xl + lane, xr);
  const bool mine = xl + lane >= xs && xl + lane < xe;
  const int gx = ux < 0 ? ux + nx : (ux >= nx ? ux - nx : ux);
  const bool wxm = WX && !perx && gx == 0, wxp = WX && !perx && gx == nx - 1;
  const int xm = gx > 0 ? gx - 1 : (perx ? nx - 1 : 0), xp = gx < nx - 1 ? gx + 1 : (perx ? 0 : nx - 1);
  const unsigned ox[3] = {unsigned(xm) * ES, unsigned(gx) * ES, unsigned(xp) * ES};
  auto row_of = [&](int y) { return y < 0 ? y + ny : (y >= ny ? y - ny : y); };
  // Plane bases are uniform (scalar registers) and offsets within a plane 32-bit.
  auto elem = [](const E* plane, unsigned off) {
    return S::ld(reinterpret_cast<const E*>(reinterpret_cast<const char*>(plane) + off), 0);
  };

  // Level 1's populations of row s, pulled from HBM.  ROWS: the row may lie on a y face.
  R nxt[9];
  auto pull_row = [&](int s, auto on_rows) {
    constexpr bool ROWS = decltype(on_rows)::value;
    const int r = row_of(s);
    const bool wym = ROWS && !pery && r == 0, wyp = ROWS && !pery && r == ny - 1;
    const unsigned rows[3] = {unsigned(nx * (wym ? 0 : row_of(r - 1))) * ES, unsigned(nx * r) * ES,
                              unsigned(nx * (wyp ? r : row_of(r + 1))) * ES};
    sfor<9>([&](auto qc) {
      constexpr int q = decltype(qc)::value;
      constexpr int cx = Lat<9>::cx[q], cy = Lat<9>::cy[q], o = Lat<9>::opp[q];
      const bool wy = (cy > 0 && wym) || (cy < 0 && wyp);  // uniform
      const bool wx = (cx > 0 && wxm) || (cx < 0 && wxp);
      // a bounced link reads the cell's own opposite population
      const unsigned off = wy || wx ? rows[1] + ox[1] : rows[1 - cy] + ox[1 - cx];
      const E* p = wy ? d.src(o) : d.src(q);
      if constexpr (WX && cx != 0) p = wx ? d.src(o) : p;
      R v = elem(p, off);
      if constexpr (q != 0 && (WX || ROWS))
        if (wx || wy) v = d.template ladd<q, ROWS>(v, wxm, wxp, wym, wyp);
      nxt[q] = v;
    });
  };

  MarchCarry<R> carry[K - 1] = {};
  // first and last row of level l
  auto lo = [&](int l) { const int y = y0 - (K - l); return (pery || y > 0) ? y : 0; };
  auto hi = [&](int l) { const int y = y1 - 1 + (K - l); return (pery || y < ny) ? y : ny - 1; };

  // One iteration.  GENERAL: some level may have no row to evaluate, or one on a y face.
  auto iterate = [&](int s, auto general) {
    constexpr bool GENERAL = decltype(general)::value;
    R fp[9], prev[9] = {};
#pragma unroll
    for (int q = 0; q < 9; ++q) fp[q] = nxt[q];
    sfor<K>([&](auto lc) {
      constexpr int l = decltype(lc)::value + 1;
      const int y = s - (l - 1);
      R fo[9] = {};
      if (!GENERAL || (y >= lo(l) && y <= hi(l))) {
        const int j = row_of(y);
        if constexpr (l > 1) {
          MarchCarry<R>& c = carry[l - 2];
          fp[0] = c.cc[0];
          fp[1] = from_left(c.cc[1]);
          fp[3] = from_right(c.cc[2]);
          fp[2] = c.cq[0];
          fp[5] = from_left(c.cq[1]);
          fp[6] = from_right(c.cq[2]);
          fp[4] = prev[4];
          fp[7] = from_right(prev[7]);
          fp[8] = from_left(prev[8]);
          if constexpr (WX || GENERAL) {
            const bool wym = GENERAL && !pery && j == 0, wyp = GENERAL && !pery && j == ny - 1;
            const R own[9] = {c.cc[0], c.cc[1], c.cp[0], c.cc[2], c.cm[0], c.cp[1], c.cp[2], c.cm[1], c.cm[2]};
            sfor<8>([&](auto qc) {
              constexpr int q = decltype(qc)::value + 1;
              constexpr int cx = Lat<9>::cx[q], cy = Lat<9>::cy[q], o = Lat<9>::opp[q];
              if constexpr (cx != 0 || GENERAL) {
                const bool out = (cx > 0 && wxm) || (cx < 0 && wxp) || (cy > 0 && wym) || (cy < 0 && wyp);
                if (out) fp[q] = d.template ladd<q, GENERAL>(own[o], wxm, wxp, wym, wyp);
              }
            });
          }
        }
        if constexpr (WX || GENERAL) d.template closures<GENERAL>(fp, gx, j);
        d.collide(fp, fo);
        if constexpr (l == K) {
          if (mine) {
            const unsigned cell = unsigned(nx * j) * ES + ox[1];
            sfor<9>([&](auto qc) {
              constexpr int q = decltype(qc)::value;
              E* p = reinterpret_cast<E*>(reinterpret_cast<char*>(d.dst(q)) + cell);
              S::template st<false>(p, 0, fo[q]);
            });
          }
        } else {
#pragma unroll
          for (int q = 0; q < 9; ++q) fo[q] = storage_round<ST>(fo[q]);
        }
      }
      if constexpr (l > 1) {  // level l − 1 moves up a row
        MarchCarry<R>& c = carry[l - 2];
#pragma unroll
        for (int n = 0; n < 3; ++n) c.cq[n] = c.cp[n];
        c.cc[0] = prev[0], c.cc[1] = prev[1], c.cc[2] = prev[3];
        c.cp[0] = prev[2], c.cp[1] = prev[5], c.cp[2] = prev[6];
        c.cm[0] = prev[4], c.cm[1] = prev[7], c.cm[2] = prev[8];
      }
#pragma unroll
      for (int q = 0; q < 9; ++q) prev[q] = fo[q];
      // the next row's pull, in flight while levels 2 … K are evaluated
      if constexpr (l == 1)
        if (!GENERAL || s + 1 <= hi(1)) pull_row(s + 1, general);
    });
  };

  int s = lo(1);
  const int s1 = y1 - 1 + (K - 1);  // level K's last row y1 − 1 comes in this iteration
  pull_row(s, std::true_type{});
  // [a, b]: the iterations in which every level has a row to evaluate, none of them and not
  // the row that is pulled ahead on a y face
  int a = y0 + K - 1, b = s1 - 1;
  if (!pery) {
    a = max(a, K);       // level K's row is at least 1
    b = min(b, ny - 3);  // the row pulled ahead is at most ny − 2
  }
  for (; s < a && s <= s1; ++s) iterate(s, std::true_type{});
  for (; s <= b; ++s) iterate(s, std::false_type{});
  for (; s <= s1; ++s) iterate(s, std::true_type{});
}

// Whether a strip evaluates no cell on a non-periodic x face (WX = false applies).
KMI_HD bool march_inner(int nx, bool perx, int K, int xs, int xe) {
  return perx || (xs - (K - 1) >= 1 && xe - 1 + (K - 1) <= nx - 2);
}

}  // namespace kmi
