// CPU build of the arithmetic that decides which thread of a launch reads which line ahead (csrc/touch_logic.h): every thread of a
// launch is walked through and what it would read is counted.  Test infrastructure only.
#include "../../lingbot-map_amd/csrc/touch_logic.h"

// reads[r][line]: how often a launch of grid_x x grid_y workgroups of `threads` threads reads that line of range r (wave_first: the
// first thread of the wavefront that asks in a launch without workgroups of their own, or -1).  Returns the reads outside the ranges.
extern "C" long long lbm_touch_host(const unsigned* lines, const long long* at, unsigned wgs, unsigned grid_x, unsigned grid_y, unsigned threads,
                                    int wave_first, int* const* reads) {
  LbmTouch t;
  for (int r = 0; r < kTouchRanges; ++r) {
    t.at[r] = (const char*)at[r];
    t.lines[r] = lines[r];
  }
  t.wgs = wgs;
  long long outside = 0;
  for (unsigned y = 0; y < grid_y; ++y)
    for (unsigned x = 0; x < grid_x; ++x)
      for (unsigned thread = 0; thread < threads; ++thread) {
        if (y == 0 && (wave_first < 0 || (int)thread < wave_first || (int)thread >= wave_first + 64)) continue;
        const LbmTouchPlace p = lbm_touch_place(t, x, y, grid_x, thread, threads, wave_first >= 0);
        if (!p.step) continue;
        const LbmTouchPart part = lbm_touch_part(t, p.xcd, p.xcd_shift);
        for (unsigned line = p.first; line < part.end; line += p.step) {
          const long long byte = (long long)(size_t)lbm_touch_line(part, line);
          bool in = false;
          for (int r = 0; r < kTouchRanges && !in; ++r)
            if (byte >= at[r] && byte < at[r] + 128ll * lines[r] && (byte - at[r]) % 128 == 0) {
              ++reads[r][(byte - at[r]) / 128];
              in = true;
            }
          outside += !in;
        }
      }
  return outside;
}
