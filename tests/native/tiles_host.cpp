// CPU build of the arithmetic that gives a workgroup its tile (csrc/tile_logic.h).  Test infrastructure only.
#include "../../lingbot-map_amd/csrc/tile_logic.h"

// hits[mt * n_tiles + nt]: how many workgroups take that tile.  Returns the workgroups that take one outside the output.
extern "C" long long lbm_tiles_host(int m_tiles, int n_tiles, int panel_shift, int* hits) {
  LbmTiles p;
  p.m_tiles = m_tiles;
  p.n_tiles = n_tiles;
  lbm_set_panels(p, panel_shift);
  long long outside = 0;
  for (int b = 0; b < m_tiles * n_tiles; ++b) {
    int mt = -1, nt = -1;
    lbm_tile_of_workgroup(b, p, mt, nt);
    if (mt < 0 || mt >= m_tiles || nt < 0 || nt >= n_tiles) ++outside;
    else ++hits[mt * n_tiles + nt];
  }
  return outside;
}
// lbm_divide against the compiler's division; returns the first t of from, from + step, ... that differs, or -1
extern "C" long long lbm_divide_host(long long from, long long step, int d) {
  const unsigned per = lbm_per(d);
  for (long long t = from; t <= 0x7fffffffll; t += step) {
    int rest = -1;
    if (lbm_divide((int)t, d, per, rest) != (int)(t / d) || rest != (int)(t % d)) return t;
  }
  return -1;
}
