// Index-only kernels: page-table maintenance (one workgroup per stream) and expansion of a
// FlashInfer-style page table into the row table the attention kernel gathers through.
// These kernels move a few KB of int32 per frame step; they are latency-bound, so each
// stream gets one 1024-thread workgroup and all requested operations run in one launch - except a
// plan that changes no table word, which is spread over several workgroups (lbm_launch_tables).
#include <hip/hip_runtime.h>
#include "tables_logic.h"
#include "lbm_internal.h"

constexpr int kTableThreads = 1024;
// A barrier that waits for no stores.  It is handed the tables: a kernel's own __restrict__ argument is memory that an asm
// statement may not touch unless it is given the address, clobbers or not, and loads and stores could move across.
__device__ __forceinline__ void lbm_bare_barrier(const int32_t* tables) { asm volatile("s_barrier" : : "s"(tables) : "memory"); }

template <int S>   // streams that there is room for, 1 or LBM_MAX_STREAMS (arguments that nobody reads are copied all the same: 0.2 us of the host)
struct LbmStepOps { lbm_step_op s[S]; };

// RUN: lbm_rows_at_a_time.  A kernel for each: with both forms of the plan in one, steps of the one-row form take longer
// (10,000 frames of one token 7.2 us apart, 7.4 in one; 2,000 5.7, 5.8).
//
// Between the phases.  A barrier that waits for the stores costs their trip to memory, and the plan's first load stands
// behind it.  It is needed where a phase reads what one before it wrote; elsewhere a bare one orders the threads: every load of
// a phase has come back when its stores leave, so no later phase overwrites what is still to be read (an eviction returns
// pages to where the append took its own, the last thread of the step writes the header that all begin with).  An eviction reads
// the appended frame only where no window is left; a plan that names the newest frame by the caller's rows reads none of its
// pages, and of an eviction only the memory lists that one with tokens to keep extends.
template <int S, int RUN>
__global__ __launch_bounds__(kTableThreads) void lbm_tables_kernel(
    int32_t* __restrict__ tables, lbm_cache_geom g, LbmTablesLayout L, LbmPlanDeal deal, int nthr, LbmStepOps<S> ops, int32_t* append_rows,
    int32_t* kv_rows, int32_t* page_ids, int32_t* page_lens) {
  const int b = S == 1 ? 0 : blockIdx.x;
  const lbm_step_op op = ops.s[b];
  // (more than one workgroup per stream only where every stream's operation is a plan alone: the
  // phases in front of it need the barriers below)
  const int tid = blockIdx.y * kTableThreads + threadIdx.x;
  if (op.ops == 0) {
    if (append_rows)
      for (int t = tid; t < g.tokens_per_frame; t += nthr) append_rows[op.q_begin + t] = -1;
    return;
  }
  int32_t* st = tables + (long long)b * L.words;
  LbmHdr h = lbm_hdr_load(st);
  // (all of it here: a bare barrier does not wait for loads that nobody has used yet)
  asm volatile("" : : "v"(h.fc), "v"(h.na), "v"(h.wh), "v"(h.wc), "v"(h.nf), "v"(h.nfs), "v"(h.nsp), "v"(h.stc), "v"(h.nm), "v"(h.nmp), "v"(h.err));
  if (op.ops & LBM_OP_RESET) {
    lbm_phase_reset(st, g, L, b * g.pages_per_stream, tid, nthr, h);
    __syncthreads();
  }
  if (op.ops & LBM_OP_ROLLBACK) {
    lbm_phase_rollback(st, g, L, tid, nthr, h);
    __syncthreads();
  }
  if (op.ops & LBM_OP_APPEND) {
    lbm_phase_append(st, g, L, append_rows ? append_rows + op.q_begin : nullptr, tid, nthr, h);
    if ((op.ops & LBM_OP_EVICT) && op.sliding_window < 1) __syncthreads();
    else lbm_bare_barrier(st);
  } else if (append_rows) {
    for (int t = tid; t < g.tokens_per_frame; t += nthr) append_rows[op.q_begin + t] = -1;
  }
  if (op.ops & LBM_OP_EVICT) {
    lbm_phase_evict(st, g, L, op.sliding_window, op.keep_tokens, tid, nthr, h);
    lbm_bare_barrier(st);
  }
  if (op.ops & LBM_OP_PLAN) {
    const bool own = (op.ops & LBM_OP_PLAN_NEWEST_SELF) && g.layout != LBM_LAYOUT_TWO_STREAM && !page_ids;
    if ((op.ops & (LBM_OP_APPEND | LBM_OP_EVICT)) && !(own && !((op.ops & LBM_OP_EVICT) && op.keep_tokens > 0))) __syncthreads();
    lbm_phase_plan<RUN>(st, g, L, op, kv_rows, page_ids, page_lens, tid, nthr, h, &deal);
  }
  if (tid == 0) lbm_hdr_store(st, h);
}

struct LbmPageSegs {
  int32_t page_begin[LBM_MAX_STREAMS + 1];
  int32_t kv_tokens[LBM_MAX_STREAMS];
  int32_t row_begin[LBM_MAX_STREAMS];
};

// One workgroup per stream: running exclusive scan of the page lengths in chunks of
// blockDim.x pages, then every thread writes the rows of its page.
__global__ __launch_bounds__(1024) void lbm_rows_from_pages_kernel(
    const int32_t* __restrict__ page_ids, const int32_t* __restrict__ page_lens,
    LbmPageSegs segs, int page_size, int32_t* __restrict__ kv_rows) {
  __shared__ int scan[1024];
  __shared__ int carry;
  const int b = blockIdx.x, tid = threadIdx.x, nthr = blockDim.x;
  const int p0 = segs.page_begin[b], p1 = segs.page_begin[b + 1];
  const int limit = segs.kv_tokens[b];
  int32_t* out = kv_rows + segs.row_begin[b];
  if (tid == 0) carry = 0;
  __syncthreads();
  for (int base = p0; base < p1; base += nthr) {
    const int p = base + tid;
    int len = 0, id = 0;
    if (p < p1) {
      len = page_lens[p];
      id = page_ids[p];
      len = len < 0 ? 0 : (len > page_size ? page_size : len);
    }
    scan[tid] = len;
    __syncthreads();
    for (int off = 1; off < nthr; off <<= 1) {
      const int v = tid >= off ? scan[tid - off] : 0;
      __syncthreads();
      scan[tid] += v;
      __syncthreads();
    }
    const int start = carry + scan[tid] - len;
    for (int s = 0; s < len; ++s)
      if (start + s < limit) out[start + s] = id * 2 * page_size + s;
    __syncthreads();
    if (tid == nthr - 1) carry += scan[tid];
    __syncthreads();
  }
  // A caller whose token count exceeds the table's total still gets defined rows.
  for (int i = carry + tid; i < limit; i += nthr) out[i] = 0;
}

template <int S>
static int lbm_launch_tables_of(int32_t* tables, const lbm_cache_geom& g, int n_streams,
                      const lbm_step_op* ops, int32_t* append_rows, int32_t* kv_rows,
                      int32_t* page_ids, int32_t* page_lens, hipStream_t stream) {
  LbmStepOps<S> o, plan;
  for (int i = 0; i < S; ++i) o.s[i] = plan.s[i] = lbm_step_op{};
  constexpr int32_t kPlanBits = LBM_OP_PLAN | LBM_OP_PLAN_NEWEST_SELF;
  bool changes = false;
  int most_rows = 0;
  for (int i = 0; i < n_streams; ++i) {
    o.s[i] = plan.s[i] = ops[i];
    plan.s[i].ops &= kPlanBits;
    changes = changes || (ops[i].ops & ~kPlanBits) != 0;
    if ((ops[i].ops & LBM_OP_PLAN) && kv_rows) {
      const int rows = ops[i].expect_kv_tokens < 0 ? -ops[i].expect_kv_tokens : ops[i].expect_kv_tokens;
      if (rows > most_rows) most_rows = rows;
    }
  }
  // Writing the rows is what takes time in a long plan.  A plan that follows no other operation reads the tables only and
  // takes one workgroup per 4,096 rows: 4.5 to 5.2 us from 4,096 rows to 65,000 (per 2,048 rows the same, per 8,192 up to
  // 0.2 more).  A step that also changes the tables needs a second launch for its plan then.  us, one launch and two: frames
  // of 1,004 tokens, 25,100 rows 6.9, 8.6, 33,132 7.4, 8.7, 41,164 8.8, 8.7, 65,260 9.9, 8.7; frames of one token, 10,000 rows
  // 7.4, 7.8, 20,000 9.3, 8.2, 40,000 12.9, 8.2.  The line lies between the two forms': 40,000 rows written four at a time,
  // 13,000 written one at a time.
  constexpr int kRowsPerGroup = 4096, kSplitRows = 24576, kMostGroups = 64;
  const int groups = most_rows <= kRowsPerGroup ? 1 : (most_rows + kRowsPerGroup - 1) / kRowsPerGroup;
  const bool wide = groups > 1 && (!changes || most_rows > kSplitRows);
  const int run = lbm_rows_at_a_time(g);
  const auto kernel = run == 4 ? lbm_tables_kernel<S, 4> : lbm_tables_kernel<S, 1>;
  const LbmTablesLayout L = lbm_tables_layout(g);
  auto launch = [&](int wgs, const LbmStepOps<S>& step, int32_t* rows) {
    const int nthr = wgs * kTableThreads;
    hipLaunchKernelGGL(kernel, dim3(n_streams, wgs), dim3(kTableThreads), 0, stream, tables, g, L, lbm_plan_deal(L, run, nthr), nthr, step, rows,
                       kv_rows, page_ids, page_lens);
    return lbm_check_launch("lbm_tables_kernel");
  };
  if (changes || !wide) {
    if (wide)
      for (int i = 0; i < n_streams; ++i) o.s[i].ops &= ~kPlanBits;
    const int rc = launch(1, o, append_rows);
    if (rc != LBM_OK || !wide) return rc;
  }
  // (append_rows was written by the launch in front, if it was asked for and there was one)
  return launch(groups < kMostGroups ? groups : kMostGroups, plan, changes ? nullptr : append_rows);
}

int lbm_launch_tables(int32_t* tables, const lbm_cache_geom& g, int n_streams,
                      const lbm_step_op* ops, int32_t* append_rows, int32_t* kv_rows,
                      int32_t* page_ids, int32_t* page_lens, hipStream_t stream) {
  return n_streams == 1 ? lbm_launch_tables_of<1>(tables, g, n_streams, ops, append_rows, kv_rows, page_ids, page_lens, stream)
                        : lbm_launch_tables_of<LBM_MAX_STREAMS>(tables, g, n_streams, ops, append_rows, kv_rows, page_ids, page_lens, stream);
}

int lbm_launch_rows_from_pages(const int32_t* page_ids, const int32_t* page_lens,
                               const int32_t* indptr, const int32_t* kv_tokens,
                               const int32_t* row_begin, int n_streams, int page_size,
                               int32_t* kv_rows, hipStream_t stream) {
  LbmPageSegs s;
  for (int i = 0; i <= LBM_MAX_STREAMS; ++i) s.page_begin[i] = 0;
  for (int i = 0; i < LBM_MAX_STREAMS; ++i) { s.kv_tokens[i] = 0; s.row_begin[i] = 0; }
  for (int i = 0; i < n_streams; ++i) {
    s.page_begin[i] = indptr[i];
    s.kv_tokens[i] = kv_tokens[i];
    s.row_begin[i] = row_begin[i];
  }
  s.page_begin[n_streams] = indptr[n_streams];
  hipLaunchKernelGGL(lbm_rows_from_pages_kernel, dim3(n_streams), dim3(1024), 0, stream,
                     page_ids, page_lens, s, page_size, kv_rows);
  return lbm_check_launch("lbm_rows_from_pages_kernel");
}
