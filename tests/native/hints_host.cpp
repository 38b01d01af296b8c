// What the library decides on the host about weights that a block's launches ask for ahead (csrc/touch_logic.h and the launches' own
// rules), for tests on the CPU.  Linked against the library; launches nothing.  Test infrastructure only.
#include "../../lingbot-map_amd/csrc/lbm_internal.h"

extern "C" void lbm_hints_deal(const int* asks, int* by) {
  LbmAsks a[5];
  int to[4];
  for (int l = 0; l < 5; ++l) a[l] = (LbmAsks)asks[l];
  lbm_deal_hints(a, to);
  for (int r = 0; r < 4; ++r) by[r] = to[r];
}

// The calling thread's pending hint: its ranges' addresses and 128-byte lines; it stays pending.
extern "C" void lbm_hints_pending(long long* at, unsigned* lines) {
  LbmTouch t;
  lbm_take_prefetch_hint(t);
  for (int r = 0; r < kTouchRanges; ++r) {
    at[r] = t.lines[r] ? (long long)(size_t)t.at[r] : 0;
    lines[r] = t.lines[r];
  }
  lbm_set_prefetch_hint(t);
}

// One attention launch in a fixed order: its rows per workgroup on the short-KV kernel (0: the split-KV schedule), its workgroups
// and each stream's splits; whether it asks for a hint.
extern "C" int lbm_hints_attention(const lbm_attn_stream* streams, int n, int heads, int own_rows, int* small, int* wgs, int* splits) {
  LbmAttnSchedule sch;
  lbm_attn_schedule(streams, n, heads, &sch, true);
  *small = sch.small;
  *wgs = sch.total_wgs;
  for (int i = 0; i < n; ++i) splits[i] = sch.s[i].n_splits;
  return lbm_attention_asks(sch, own_rows != 0);
}
