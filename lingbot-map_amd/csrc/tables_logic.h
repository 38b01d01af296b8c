// Page-table state machine of one stream, written so that the same code runs as one HIP
// workgroup (tid = threadIdx.x, nthr = blockDim.x, a barrier between phases) or as one host
// thread (tid = 0, nthr = 1) in the CPU build the table tests use.
//
// The policy is the reference's (lingbot_map/layers/flashinfer_cache.py): LIFO free list
// (:496, :538), anchor-then-window routing (:507-510), oldest-first eviction that returns
// pages to the tail of the free list (:252-254), packed special stream (:529-553),
// rollback to the free-list tail (:280-301).  No phase reads a word that the same phase
// writes, so the order of threads inside a phase does not matter.
#ifndef LBM_TABLES_LOGIC_H
#define LBM_TABLES_LOGIC_H

#include "../../include/lbm_paged_attn.h"
#include "tile_logic.h"

#if defined(__HIPCC__)
#define LBM_HD __host__ __device__ __forceinline__
#else
#define LBM_HD inline
#endif

struct LbmTablesLayout {
  int ppf;          // pages a frame takes
  int tpf;          // tokens of a frame stored in those pages
  int kpm;          // most pages a compacted frame keeps
  int ring_frames;  // capacity of the window ring, in frames
  int shift;        // of a power-of-two page size, -1: it is none
  int off_free_patch, off_free_special, off_anchor, off_window, off_special;
  int off_mem_pages, off_mem_tcum, off_mem_pcum;
  long long words;
};

LBM_HD int lbm_ceil_div(int a, int b) { return (a + b - 1) / b; }

// Sixteen wavefronts on one CU take the same instructions: a division is 40 of them, 0.3 us of a step that has a dozen.  So the
// layout is the launch's, pages are found by shifts, frames of the ring without remainders and threads' frames by a
// reciprocal.  With the barriers that lbm_tables_kernel no longer waits at, us a keyframe's step, before and now: 17 frames of 1,004 tokens
// 6.8, 6.0, of 261 4.9, 4.1, 5 of 100 4.5, 3.6; 300 of one token 4.6, 3.8; four streams of 1,004 7.0, 6.3; a plan alone 3.7, 3.45.
// The page and slot of token t of a page list; page sizes are powers of two in every configuration but one (page = patches per frame)
LBM_HD int lbm_page_of(const LbmTablesLayout& L, int page_size, int t, int& slot) {
  const int page = L.shift >= 0 ? t >> L.shift : t / page_size;
  slot = t - page * page_size;
  return page;
}
LBM_HD int lbm_pages_for(const LbmTablesLayout& L, int page_size, int tokens) {
  int slot;
  return lbm_page_of(L, page_size, tokens + page_size - 1, slot);
}
// a frame's place in the ring, i below twice its frames (head and count are at most its frames each)
LBM_HD int lbm_ring(const LbmTablesLayout& L, int i) { return i >= L.ring_frames ? i - L.ring_frames : i; }

LBM_HD bool lbm_geom_valid(const lbm_cache_geom& g) {
  if (g.layout != LBM_LAYOUT_TWO_STREAM && g.layout != LBM_LAYOUT_FRAME_PAGES) return false;
  if (g.page_size <= 0 || g.num_special_tokens < 0 || g.scale_frames < 0) return false;
  if (g.tokens_per_frame <= g.num_special_tokens) return false;  // flashinfer_cache.py:113
  if (g.patch_pages <= 0 || g.special_pages < 0 || g.memory_frames < 0) return false;
  if (g.pages_per_stream < g.patch_pages + g.special_pages) return false;
  return true;
}

LBM_HD LbmTablesLayout lbm_tables_layout(const lbm_cache_geom& g) {
  LbmTablesLayout L;
  const bool two = g.layout == LBM_LAYOUT_TWO_STREAM;
  L.tpf = two ? g.tokens_per_frame - g.num_special_tokens : g.tokens_per_frame;
  L.ppf = lbm_ceil_div(L.tpf, g.page_size);
  L.kpm = two ? 0 : lbm_ceil_div(g.num_special_tokens, g.page_size);
  L.ring_frames = g.patch_pages / L.ppf;
  L.shift = (g.page_size & (g.page_size - 1)) == 0 ? __builtin_ctz((unsigned)g.page_size) : -1;
  int off = LBM_HDR_WORDS;
  L.off_free_patch = off;   off += g.patch_pages;
  L.off_free_special = off; off += g.special_pages;
  L.off_anchor = off;       off += g.scale_frames * L.ppf;
  L.off_window = off;       off += L.ring_frames * L.ppf;
  L.off_special = off;      off += g.special_pages;
  L.off_mem_pages = off;    off += g.memory_frames * L.kpm;
  L.off_mem_tcum = off;     off += g.memory_frames + 1;
  L.off_mem_pcum = off;     off += g.memory_frames + 1;
  L.words = off;
  return L;
}

// Header snapshot taken by every thread at the start of a phase.
struct LbmHdr {
  int fc, na, wh, wc, nf, nfs, nsp, stc, nm, nmp, err;
};

LBM_HD LbmHdr lbm_hdr_load(const int32_t* st) {
  LbmHdr h;
  h.fc = st[LBM_HDR_FRAME_COUNT];      h.na = st[LBM_HDR_N_ANCHOR];
  h.wh = st[LBM_HDR_WIN_HEAD];         h.wc = st[LBM_HDR_WIN_COUNT];
  h.nf = st[LBM_HDR_N_FREE_PATCH];     h.nfs = st[LBM_HDR_N_FREE_SPECIAL];
  h.nsp = st[LBM_HDR_N_SPECIAL_PAGES]; h.stc = st[LBM_HDR_SPECIAL_TOKENS];
  h.nm = st[LBM_HDR_N_MEMORY];         h.nmp = st[LBM_HDR_N_MEMORY_PAGES];
  h.err = st[LBM_HDR_ERROR];
  return h;
}

LBM_HD void lbm_hdr_store(int32_t* st, const LbmHdr& h) {
  st[LBM_HDR_FRAME_COUNT] = h.fc;      st[LBM_HDR_N_ANCHOR] = h.na;
  st[LBM_HDR_WIN_HEAD] = h.wh;         st[LBM_HDR_WIN_COUNT] = h.wc;
  st[LBM_HDR_N_FREE_PATCH] = h.nf;     st[LBM_HDR_N_FREE_SPECIAL] = h.nfs;
  st[LBM_HDR_N_SPECIAL_PAGES] = h.nsp; st[LBM_HDR_SPECIAL_TOKENS] = h.stc;
  st[LBM_HDR_N_MEMORY] = h.nm;         st[LBM_HDR_N_MEMORY_PAGES] = h.nmp;
  st[LBM_HDR_ERROR] = h.err;
}

// ---------------------------------------------------------------------------- reset
// flashinfer_cache.py:423-432.  `h` is the header to commit after the phase.
LBM_HD void lbm_phase_reset(int32_t* st, const lbm_cache_geom& g, const LbmTablesLayout& L,
                            int page_base, int tid, int nthr, LbmHdr& h) {
  for (int i = tid; i < g.patch_pages; i += nthr) st[L.off_free_patch + i] = page_base + i;
  for (int i = tid; i < g.special_pages; i += nthr)
    st[L.off_free_special + i] = page_base + g.patch_pages + i;
  if (tid == 0) { st[L.off_mem_tcum] = 0; st[L.off_mem_pcum] = 0; }
  h = LbmHdr{};
  h.nf = g.patch_pages;
  h.nfs = g.special_pages;
}

// ---------------------------------------------------------------------------- rollback
// flashinfer_cache.py:268-301.
LBM_HD void lbm_phase_rollback(int32_t* st, const lbm_cache_geom& g, const LbmTablesLayout& L,
                               int tid, int nthr, LbmHdr& h) {
  const bool two = g.layout == LBM_LAYOUT_TWO_STREAM;
  const bool from_window = h.fc > g.scale_frames;
  int new_count = h.stc, n_pop = 0;
  if (two) {
    new_count = h.stc - g.num_special_tokens;
    n_pop = h.nsp - (new_count > 0 ? lbm_pages_for(L, g.page_size, new_count) : 0);
  }
  if (h.fc <= 0 || (from_window ? h.wc <= 0 : h.na <= 0) || new_count < 0) {
    h.err |= LBM_TERR_ROLLBACK;
    return;
  }
  const int32_t* src = from_window
      ? st + L.off_window + lbm_ring(L, h.wh + h.wc - 1) * L.ppf
      : st + L.off_anchor + (h.na - 1) * L.ppf;
  for (int j = tid; j < L.ppf; j += nthr) st[L.off_free_patch + h.nf + j] = src[L.ppf - 1 - j];
  for (int k = tid; k < n_pop; k += nthr)
    st[L.off_free_special + h.nfs + k] = st[L.off_special + h.nsp - 1 - k];
  if (from_window) h.wc -= 1; else h.na -= 1;
  h.nf += L.ppf;
  h.nfs += n_pop;
  h.nsp -= n_pop;
  h.stc = new_count;
  h.fc -= 1;
}

// ---------------------------------------------------------------------------- append
// Allocation half of append_frame: flashinfer_cache.py:474-553.  Writes the K row of every
// token of the new frame to rows_out[0 .. tokens_per_frame).
LBM_HD void lbm_phase_append(int32_t* st, const lbm_cache_geom& g, const LbmTablesLayout& L,
                             int32_t* rows_out, int tid, int nthr, LbmHdr& h) {
  const bool two = g.layout == LBM_LAYOUT_TWO_STREAM;
  const int S = g.page_size, n_sp = g.num_special_tokens, T = g.tokens_per_frame;
  const bool to_anchor = h.na < g.scale_frames;
  const int new_sp = two ? lbm_pages_for(L, S, h.stc + n_sp) - h.nsp : 0;
  int err = 0;
  if (h.nf < L.ppf) err |= LBM_TERR_PATCH_POOL;
  if (!to_anchor && h.wc >= L.ring_frames) err |= LBM_TERR_WINDOW_RING;
  if (new_sp > h.nfs) err |= LBM_TERR_SPECIAL_POOL;
  if (err) {
    h.err |= err;
    if (rows_out) for (int t = tid; t < T; t += nthr) rows_out[t] = -1;
    return;
  }
  const int32_t* fp = st + L.off_free_patch;
  int32_t* dst = to_anchor ? st + L.off_anchor + h.na * L.ppf
                           : st + L.off_window + lbm_ring(L, h.wh + h.wc) * L.ppf;
  for (int j = tid; j < L.ppf; j += nthr) dst[j] = fp[h.nf - 1 - j];
  if (rows_out) {
    for (int t = tid; t < T; t += nthr) {
      int page, slot;
      if (!two) {
        page = fp[h.nf - 1 - lbm_page_of(L, S, t, slot)];
      } else if (t >= n_sp) {
        page = fp[h.nf - 1 - lbm_page_of(L, S, t - n_sp, slot)];
      } else {
        const int pi = lbm_page_of(L, S, h.stc + t, slot);
        page = pi < h.nsp ? st[L.off_special + pi] : st[L.off_free_special + h.nfs - 1 - (pi - h.nsp)];
      }
      rows_out[t] = page * 2 * S + slot;
    }
  }
  for (int k = tid; k < new_sp; k += nthr)
    st[L.off_special + h.nsp + k] = st[L.off_free_special + h.nfs - 1 - k];
  if (to_anchor) h.na += 1; else h.wc += 1;
  h.nf -= L.ppf;
  h.nfs -= new_sp;
  h.nsp += new_sp;
  if (two) h.stc += n_sp;
  h.fc += 1;
}

// ---------------------------------------------------------------------------- evict
// flashinfer_cache.py:252-254; in the frame_pages layout the leading pages of an evicted
// frame stay as trajectory memory with `keep` valid tokens
// (lingbot_map/layers/attention.py:690-705), nothing is copied.
LBM_HD void lbm_phase_evict(int32_t* st, const lbm_cache_geom& g, const LbmTablesLayout& L,
                            int window, int keep, int tid, int nthr, LbmHdr& h) {
  const int n_ev = h.wc - window;
  if (n_ev <= 0) return;
  const bool two = g.layout == LBM_LAYOUT_TWO_STREAM;
  if (two || keep < 0) keep = 0;
  if (keep > g.num_special_tokens) keep = g.num_special_tokens;
  const int kp = keep ? lbm_pages_for(L, g.page_size, keep) : 0;
  if (keep && h.nm + n_ev > g.memory_frames) { h.err |= LBM_TERR_MEMORY_FULL; return; }
  const int per = L.ppf - kp;
  const int32_t* win = st + L.off_window;
  for (int i = tid; i < n_ev * per; i += nthr) {
    const int e = n_ev == 1 ? 0 : i / per, j = kp + i - e * per;
    st[L.off_free_patch + h.nf + i] = win[lbm_ring(L, h.wh + e) * L.ppf + j];
  }
  for (int i = tid; i < n_ev * kp; i += nthr) {
    const int e = n_ev == 1 ? 0 : i / kp, j = i - e * kp;
    st[L.off_mem_pages + h.nmp + i] = win[lbm_ring(L, h.wh + e) * L.ppf + j];
  }
  if (keep) {
    for (int e = tid; e < n_ev; e += nthr) {
      st[L.off_mem_tcum + h.nm + e + 1] = h.stc + (e + 1) * keep;
      st[L.off_mem_pcum + h.nm + e + 1] = h.nmp + (e + 1) * kp;
    }
    h.nm += n_ev;
    h.nmp += n_ev * kp;
    h.stc += n_ev * keep;
  }
  h.wh = lbm_ring(L, h.wh + n_ev);
  h.wc -= n_ev;
  h.nf += n_ev * per;
}

// ---------------------------------------------------------------------------- plan
// n (1 to 4) consecutive entries of a row table: first, first + step, ...; whole fours as one store (a table's entries are
// aligned to 4 bytes and no more, which is what the store needs).
LBM_HD void lbm_put_rows(int32_t* dst, int first, int step, int n) {
#ifdef __HIP_DEVICE_COMPILE__
  typedef int32_t four __attribute__((ext_vector_type(4), aligned(4)));
  if (n == 4) {
    *(four*)dst = four{first, first + step, first + 2 * step, first + 3 * step};
    return;
  }
#endif
  for (int j = 0; j < n; ++j) dst[j] = first + j * step;
}

// RUN token slots from t on (n_run of them; slot `slot` of page `pg` on) of frames my_group, my_group + groups, ...: BATCH
// frames at a time, so that their page-id loads are in flight together (no division per token, no load waiting on the
// previous frame's store).
template <int RUN, int BATCH>
LBM_HD void lbm_plan_run(int32_t* out, const int32_t* anchor, const int32_t* win, int S, const LbmTablesLayout& L, const LbmHdr& h,
                         int q_begin, bool newest_self, int limit, int t, int n_run, int pg, int slot, int my_group, int groups) {
  const int nfr = h.na + h.wc;
  for (int f0 = my_group; f0 < nfr; f0 += BATCH * groups) {
    int32_t page[BATCH];
#ifdef __HIP_DEVICE_COMPILE__
#pragma unroll
#endif
    for (int k = 0; k < BATCH; ++k) {
      const int f = f0 + k * groups < nfr ? f0 + k * groups : nfr - 1;
      int r = h.wh + f - h.na;                     // ring slot of window frame f - na
      if (r >= L.ring_frames) r -= L.ring_frames;  // wh < ring_frames and at most ring_frames window frames
      const int32_t* pages = f < h.na ? anchor + f * L.ppf : win + r * L.ppf;
      page[k] = pages[pg];
    }
#ifdef __HIP_DEVICE_COMPILE__
#pragma unroll
#endif
    for (int k = 0; k < BATCH; ++k) {
      const int f = f0 + k * groups;
      const int i = f * L.tpf + t;
      const bool own = newest_self && f == nfr - 1;
      if (RUN == 1) {
        if (f < nfr && i < limit) out[i] = own ? -1 - (q_begin + t) : page[k] * 2 * S + slot;
      } else if (f < nfr && i < limit) {
        lbm_put_rows(out + i, own ? -1 - (q_begin + t) : page[k] * 2 * S + slot, own ? -1 : 1,
                     n_run < limit - i ? n_run : limit - i);
      }
    }
  }
}

// The rows of the cached frames.  A thread owns runs of RUN token slots, u, u + nthr, ... of every frame (consecutive
// lanes write consecutive runs; RUN divides the page size).  Frames of fewer runs than there are threads are dealt to
// groups of `runs` threads, group i taking frames i, i + groups, ...: one thread would otherwise walk all frames of a
// one-token-per-frame cache by itself (10,000 frames: 1.4 ms).  Eight frames at a time; two where four-row runs leave a
// thread no more, since a frame that is not there costs its addresses and compares all the same (one workgroup, us a step
// with eight and with two: 197 tokens x 17 frames 6.1, 5.1; 261 x 17 5.9, 5.0; 1,004 x 5 6.3, 5.3).
struct LbmPlanDeal { int runs, groups; unsigned per_runs; };
LBM_HD LbmPlanDeal lbm_plan_deal(const LbmTablesLayout& L, int run, int nthr) {
  const int runs = lbm_ceil_div(L.tpf, run);
  return {runs, runs < nthr ? nthr / runs : 1, lbm_per(runs)};
}
template <int RUN>
LBM_HD void lbm_plan_frames(int32_t* out, const int32_t* st, int S, const LbmTablesLayout& L, const LbmHdr& h, const lbm_step_op& op,
                            const LbmPlanDeal& deal, bool newest_self, int limit, int tid, int nthr) {
  const int32_t* anchor = st + L.off_anchor;
  const int32_t* win = st + L.off_window;
  const int runs = deal.runs, groups = deal.groups;
  int my_group = 0, u_first = tid;
  if (groups > 1) {
    my_group = lbm_divide(tid, runs, deal.per_runs, u_first);
    if (my_group >= groups) u_first = runs;
  }
  for (int u = u_first; u < runs; u += groups > 1 ? runs : nthr) {
    const int t = u * RUN, n_run = RUN == 1 || L.tpf - t >= RUN ? RUN : L.tpf - t;
    int slot;
    const int pg = lbm_page_of(L, S, t, slot);
    if (RUN > 1 && h.na + h.wc <= 2 * groups)
      lbm_plan_run<RUN, 2>(out, anchor, win, S, L, h, op.q_begin, newest_self, limit, t, n_run, pg, slot, my_group, groups);
    else
      lbm_plan_run<RUN, 8>(out, anchor, win, S, L, h, op.q_begin, newest_self, limit, t, n_run, pg, slot, my_group, groups);
  }
}

// Four rows at a time where pages hold whole fours: a page id, its addresses and its compares serve four rows.  Frames of
// one token have nothing to share.  One workgroup, us a step with one row and with four: 17 frames of 1,004 tokens 9.5, 7.1,
// 21 frames 9.9, 7.2; 261 x 17 5.6, 5.0; 65 x 17 5.3, 4.6; 5 x 101 4.6, 4.6; 4 x 17 4.4, 4.5; 10,000 x 1 7.8, 9.3.
LBM_HD int lbm_rows_at_a_time(const lbm_cache_geom& g) { return (g.page_size & 3) == 0 && lbm_tables_layout(g).tpf >= 4 ? 4 : 1; }

// build_visible_page_table + compute_last_page_len (flashinfer_cache.py:438-470) with a
// valid length per page, plus the dense row table the attention kernel gathers through.
// Never writes more row entries than the host says the table holds (op.expect_kv_tokens, or the
// capacity it gives instead) and publishes a count within that bound, so a host/device
// disagreement cannot make the attention kernel read outside the table (it sets
// LBM_TERR_KV_COUNT instead).
// RUN: rows that a thread writes at a time, as lbm_rows_at_a_time says (0: asked here).  deal: lbm_plan_deal of them and of nthr, or null.
template <int RUN = 0>
LBM_HD void lbm_phase_plan(int32_t* st, const lbm_cache_geom& g, const LbmTablesLayout& L,
                           const lbm_step_op& op, int32_t* kv_rows, int32_t* page_ids,
                           int32_t* page_lens, int tid, int nthr, LbmHdr& h, const LbmPlanDeal* deal = nullptr) {
  const bool two = g.layout == LBM_LAYOUT_TWO_STREAM;
  const int S = g.page_size;
  const int nfr = h.na + h.wc;
  const int frame_tokens = nfr * L.tpf;
  const int self_n = op.self_tokens > 0 ? op.self_tokens : 0;
  // LBM_OP_PLAN_NEWEST_SELF: the newest cached frame (the one this step appended: the last of the
  // frame list) is named by the caller's own rows, in the place its pool rows would take
  const bool newest_self = (op.ops & LBM_OP_PLAN_NEWEST_SELF) != 0 && !two && nfr > 0;
  int total = frame_tokens + h.stc + self_n;
  // expect_kv_tokens >= 0: the host's own count, which must agree; < 0: the host does not track
  // the count and gives the capacity of this stream's part of kv_rows instead
  const bool counted = op.expect_kv_tokens >= 0;
  const int limit = counted ? op.expect_kv_tokens : -op.expect_kv_tokens;
  if (counted ? total != limit : total > limit) h.err |= LBM_TERR_KV_COUNT;
  const int32_t* anchor = st + L.off_anchor;
  const int32_t* win = st + L.off_window;
  if (kv_rows) {
    int32_t* out = kv_rows + op.kv_row_begin;
    const int run = RUN ? RUN : lbm_rows_at_a_time(g);
    const LbmPlanDeal dealt = deal ? *deal : lbm_plan_deal(L, run, nthr);
    if (RUN == 4 || (RUN == 0 && run == 4)) lbm_plan_frames<4>(out, st, S, L, h, op, dealt, newest_self, limit, tid, nthr);
    else lbm_plan_frames<1>(out, st, S, L, h, op, dealt, newest_self, limit, tid, nthr);
    if (two) {
      for (int c = tid; c < h.stc; c += nthr) {
        int slot;
        const int pg = lbm_page_of(L, S, c, slot);
        if (frame_tokens + c < limit) out[frame_tokens + c] = st[L.off_special + pg] * 2 * S + slot;
      }
    } else {
      for (int e = tid; e < h.nm; e += nthr) {
        const int t0 = st[L.off_mem_tcum + e], t1 = st[L.off_mem_tcum + e + 1];
        const int p0 = st[L.off_mem_pcum + e];
        for (int t = 0; t < t1 - t0; ++t) {
          int slot;
          const int pg = lbm_page_of(L, S, t, slot);
          if (frame_tokens + t0 + t < limit) out[frame_tokens + t0 + t] = st[L.off_mem_pages + p0 + pg] * 2 * S + slot;
        }
      }
    }
    for (int t = tid; t < self_n; t += nthr)
      if (frame_tokens + h.stc + t < limit) out[frame_tokens + h.stc + t] = -1 - (op.q_begin + t);
    if (counted)
      for (int i = total + tid; i < limit; i += nthr) out[i] = 0;
  }
  if (total > limit) total = limit;  // what the attention may read
  int n_pages = nfr * L.ppf + (two ? h.nsp : h.nmp);
  if (page_ids && page_lens) {
    int32_t* ids = page_ids + op.page_out_begin;
    int32_t* lens = page_lens + op.page_out_begin;
    for (int i = tid; i < nfr * L.ppf; i += nthr) {
      const int f = i / L.ppf, j = i % L.ppf;
      const int32_t* pages = f < h.na ? anchor + f * L.ppf
                                      : win + ((h.wh + f - h.na) % L.ring_frames) * L.ppf;
      ids[i] = pages[j];
      lens[i] = j < L.ppf - 1 ? S : L.tpf - (L.ppf - 1) * S;
    }
    int32_t* ids2 = ids + nfr * L.ppf;
    int32_t* lens2 = lens + nfr * L.ppf;
    if (two) {
      const int tail = h.stc % S;
      for (int k = tid; k < h.nsp; k += nthr) {
        ids2[k] = st[L.off_special + k];
        lens2[k] = (k < h.nsp - 1 || tail == 0) ? S : tail;
      }
    } else {
      for (int e = tid; e < h.nm; e += nthr) {
        const int keep = st[L.off_mem_tcum + e + 1] - st[L.off_mem_tcum + e];
        const int p0 = st[L.off_mem_pcum + e], p1 = st[L.off_mem_pcum + e + 1];
        for (int j = 0; j < p1 - p0; ++j) {
          ids2[p0 + j] = st[L.off_mem_pages + p0 + j];
          lens2[p0 + j] = j < p1 - p0 - 1 ? S : keep - (p1 - p0 - 1) * S;
        }
      }
    }
  }
  if (tid == 0) {
    st[LBM_HDR_PLAN_KV_TOKENS] = total;
    st[LBM_HDR_PLAN_N_PAGES] = n_pages;
  }
}

#endif  // LBM_TABLES_LOGIC_H
