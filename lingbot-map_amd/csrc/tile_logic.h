// Which output tile a workgroup of the linears takes, and division by numbers that a launch fixes: plain index arithmetic, so that
// the same code can be built for the CPU and every tile accounted for there.
#ifndef LBM_TILE_LOGIC_H
#define LBM_TILE_LOGIC_H

#if defined(__HIPCC__)
#define LBM_TILE_FN __host__ __device__ __forceinline__
#else
#define LBM_TILE_FN inline
#endif

// t / d (0 <= t, 0 < d) and the remainder, given per = lbm_per(d): t x per / 2^32 is at most the quotient and less than two below
// it (32-bit division: a call works several out on its way to the launch).
// On a uniform value the compiler divides by way of a vector reciprocal and back: 40 instructions that wait for one
// another, in front of a launch's first load.  (qkv projection, proj, fc1 and fc2, two divisions each, and their sizes in one line of
// the scalar cache: 86 rows 25.3 -> 24.8 us, 261 28.7 -> 28.0, 1,004 43.0 -> 42.3, 2,008 60.5 -> 59.7.)
LBM_TILE_FN unsigned lbm_per(int d) { return d > 1 ? 0xffffffffu / (unsigned)d : 0xffffffffu; }
LBM_TILE_FN int lbm_divide(int t, int d, unsigned per, int& rest) {
  int q = (int)(((unsigned long long)(unsigned)t * per) >> 32);
  rest = t - q * d;
  if (rest >= d) {
    rest -= d;
    ++q;
  }
  return q;
}

// m_tiles x n_tiles tiles in panels of 1 << panel_shift column tiles; last_width: column tiles of the last panel where it has
// fewer (0: it does not); per_*: lbm_per of a panel's tiles and of last_width.
struct LbmTiles {
  int m_tiles, n_tiles;
  int panel_shift, last_width;
  unsigned per_panel, per_last;
};
LBM_TILE_FN void lbm_set_panels(LbmTiles& p, int panel_shift) {
  p.panel_shift = panel_shift;
  p.last_width = p.n_tiles & ((1 << panel_shift) - 1);
  p.per_panel = lbm_per(p.m_tiles << panel_shift);
  p.per_last = lbm_per(p.last_width);
}
// Workgroup b's tile.  Workgroups are dealt to the 8 XCDs round-robin (b % 8), 32 of a round of 256
// to each; an XCD's 32 take consecutive tiles of an order that walks panels of 8 column tiles row
// by row, i.e. 4 row tiles x 8 column tiles (8 x 4 in a last panel of 4): 12 operand tiles per
// k-step for the XCD's L2 to hold instead of 17 to 33, which is what sets the latency of the
// operand loads.  (Tiles of 64 columns x 32, 64 or 96 rows: panels of 4 or 8, see lbm_linear_panels.)
LBM_TILE_FN void lbm_tile_of_workgroup(int b, const LbmTiles& p, int& mt, int& nt) {
  const int x = b & 7, i = b >> 3;
  const int base = (i >> 5) * 256, left = p.m_tiles * p.n_tiles - base;
  const int in_round = left < 256 ? left : 256;
  const int t = base + x * (in_round >> 3) + (x < (in_round & 7) ? x : in_round & 7) + (i & 31);
  int rem;
  const int panel = lbm_divide(t, p.m_tiles << p.panel_shift, p.per_panel, rem);
  const int first = panel << p.panel_shift;
  if (p.n_tiles - first >= 1 << p.panel_shift) {
    mt = rem >> p.panel_shift;
    nt = first + (rem & ((1 << p.panel_shift) - 1));
  } else {
    int col;
    mt = lbm_divide(rem, p.last_width, p.per_last, col);
    nt = first + col;
  }
}

#endif  // LBM_TILE_LOGIC_H
