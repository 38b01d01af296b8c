// Which 128-byte lines of the ranges that a launch asks for ahead (lbm_linear_prefetch_hint) which thread of it reads: plain
// index arithmetic, so that the same code can be built for the CPU and every address looked at there.
#ifndef LBM_TOUCH_LOGIC_H
#define LBM_TOUCH_LOGIC_H

#include <stddef.h>

#if defined(__HIPCC__)
#define LBM_TOUCH_FN __host__ __device__ __forceinline__
#else
#define LBM_TOUCH_FN inline
#endif

constexpr int kTouchRanges = 4;
struct LbmTouch {
  const char* at[kTouchRanges];
  unsigned lines[kTouchRanges];   // 128-byte lines of each; 0: no range
  unsigned wgs;                   // workgroups with blockIdx.y > 0 that ask for them (any further ones end at once); 0 or at least 8
};

// CUs without a workgroup in the last round of a launch of `wgs` workgroups, one a CU
LBM_TOUCH_FN int lbm_idle_cus(long long wgs) { return (int)((256 - wgs % 256) % 256); }
constexpr int kTouchIdle = 32;

// one range more, up to kTouchRanges
LBM_TOUCH_FN void lbm_add_touch(LbmTouch& t, const void* ptr, size_t bytes) {
  if (!ptr || bytes < 128) return;
  for (int r = 0; r < kTouchRanges; ++r)
    if (!t.lines[r]) {
      t.at[r] = (const char*)ptr;
      t.lines[r] = (unsigned)(bytes / 128);
      return;
    }
}

// How a launch would ask for a hint: not at all, by wavefronts beside the computing ones, by workgroups of their own on idle CUs,
// and that beside tiles of 256 columns
enum LbmAsks { LBM_ASKS_NOT, LBM_ASKS_WAVES, LBM_ASKS_IDLE, LBM_ASKS_WIDE_IDLE };
// Which of a block's five launches (qkv projection, attention, proj, fc1, fc2) asks for which of the weights ahead, -1: none.  by[r]
// is for what launch 2 + r reads, the fourth the next block's first: the nearest of the three before it that can, but
// rather one of 256-column tiles with idle CUs than one that
// would do it by wavefronts beside the computing ones.  Three, since further ahead costs more than it saves once K/V and the
// rows of a few streams pass through the memory-side cache in between (ms a frame, three | any before it: two streams of 1,004
// rows 8.82 | 9.14, three anchor frames of 666 rows 7.37 | 7.68).  The nearest, since the 64 idle CUs of a qkv launch on 128 x 128
// tiles, which L2 binds, take from it what asking for all of them saves (1,004 rows 5.88, by wavefronts in between 5.86);
// 256-column tiles leave L2 the time (qkv projection, proj, fc1, fc2 of 2,008 rows: fc1's weights asked for by proj's wavefronts
// 66.5 us, by the qkv launch 64.9; of 3,000 rows 87.6, 86.7).
LBM_TOUCH_FN void lbm_deal_hints(const LbmAsks (&asks)[5], int (&by)[4]) {
  for (int r = 0; r < 4; ++r) {
    const int first = r > 0 ? r - 1 : 0;
    by[r] = -1;
    for (int l = 1 + r; l >= first && by[r] < 0; --l)
      if (asks[l] != LBM_ASKS_NOT) by[r] = l;
    if (by[r] >= 0 && asks[by[r]] == LBM_ASKS_WAVES)
      for (int l = by[r] - 1; l >= first; --l)
        if (asks[l] == LBM_ASKS_WIDE_IDLE) {
          by[r] = l;
          break;
        }
  }
}

// A thread's place: every `step`-th line from `first` on of the part of an XCD (all lines where xcd_shift is 0, else its
// eighth of each range); step 0: none.
struct LbmTouchPlace { unsigned xcd, xcd_shift, first, step; };
// Workgroups are dealt to the XCDs round-robin in the order of their linear index.
LBM_TOUCH_FN LbmTouchPlace lbm_touch_place(const LbmTouch& t, unsigned block_x, unsigned block_y, unsigned grid_x, unsigned thread,
                                           unsigned threads, bool wave) {
  if (block_y) {
    const unsigned i = (block_y - 1u) * grid_x + block_x;
    if (i >= t.wgs) return {0, 0, 0, 0};
    return {(grid_x + i) & 7u, 3u, (i >> 3) * threads + thread, ((t.wgs - (i & 7u) + 7u) >> 3) * threads};
  }
  if (!wave || t.wgs) return {0, 0, 0, 0};
  // A launch of 128 workgroups or more: an XCD's ask for the eighth of the lines that its own tiles of the next launch
  // are likely to read (weights by rows, panels of tiles by XCD), which then also waits in its L2 (a frame of 261 rows
  // 3.58 -> 3.55 ms, of 1,004 rows 6.61 -> 6.58).  The few of a smaller launch share all of them.
  if (grid_x >= 128u) return {block_x & 7u, 3u, (block_x >> 3) * 64u + (thread & 63u), ((grid_x - (block_x & 7u) + 7u) >> 3) * 64u};
  return {0, 0, block_x * 64u + (thread & 63u), grid_x * 64u};
}

// An XCD's part of the ranges, one behind the other: line i of it, i < end, is at base[r] + 128 i for the first r with i < until[r].
struct LbmTouchPart {
  size_t base[kTouchRanges];
  unsigned until[kTouchRanges], end;
};
LBM_TOUCH_FN LbmTouchPart lbm_touch_part(const LbmTouch& t, unsigned xcd, unsigned xcd_shift) {
  LbmTouchPart p;
  p.end = 0;
#pragma unroll
  for (int r = 0; r < kTouchRanges; ++r) {
    const unsigned lines = t.lines[r], share = (lines + (1u << xcd_shift) - 1u) >> xcd_shift;
    const unsigned begin = share * xcd < lines ? share * xcd : lines, count = lines - begin < share ? lines - begin : share;
    p.base[r] = (size_t)t.at[r] + ((size_t)begin - p.end) * 128;
    p.until[r] = p.end += count;
  }
  return p;
}
LBM_TOUCH_FN const char* lbm_touch_line(const LbmTouchPart& p, unsigned line) {
  size_t base = p.base[0];
#pragma unroll
  for (int r = 1; r < kTouchRanges; ++r) {
    const size_t next = p.base[r];   // (a value: of two lvalues ?: takes the address, and the array goes to memory)
    base = line >= p.until[r - 1] ? next : base;
  }
  return (const char*)(base + (size_t)line * 128);
}

#endif  // LBM_TOUCH_LOGIC_H
