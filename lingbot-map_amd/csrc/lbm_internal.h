// Declarations shared by the translation units of the library (not part of the C ABI).
#ifndef LBM_INTERNAL_H
#define LBM_INTERNAL_H

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>
#include "../../include/lbm_paged_attn.h"
#include "tile_logic.h"
#include "touch_logic.h"

// Records `msg` as the calling thread's last error and returns `code`.
int lbm_fail(int code, const char* fmt, ...);
// hipGetLastError() after a launch; LBM_OK or LBM_ERR_HIP with the kernel's name recorded.
int lbm_check_launch(const char* kernel_name);

int lbm_launch_tables(int32_t* tables, const lbm_cache_geom& g, int n_streams,
                      const lbm_step_op* ops, int32_t* append_rows, int32_t* kv_rows,
                      int32_t* page_ids, int32_t* page_lens, hipStream_t stream);
int lbm_launch_rows_from_pages(const int32_t* page_ids, const int32_t* page_lens,
                               const int32_t* indptr, const int32_t* kv_tokens,
                               const int32_t* row_begin, int n_streams, int page_size,
                               int32_t* kv_rows, hipStream_t stream);
int lbm_launch_append(const void* k, const void* v, int src_dtype, void* pool, int pool_dtype,
                      const int32_t* append_rows, int n_tokens, int num_heads, int head_dim,
                      int page_size, hipStream_t stream);

int lbm_launch_qkv_prepare(const void* qkv, int src_dtype, const float* q_norm_w, const float* q_norm_b,
                           const float* k_norm_w, const float* k_norm_b, float norm_eps, float q_scale,
                           const float* rope_cs, int rope_layout, void* q_out, void* k_out, void* v_out,
                           int dst_dtype, void* pool, const int32_t* append_rows, int n_tokens,
                           int num_heads, int page_size, hipStream_t stream);

int lbm_launch_residual_norm(const void* x, const void* y, int dtype, const float* gamma, const float* norm_w,
                             const float* norm_b, float eps, void* x_out, void* n_out, int rows, int cols,
                             hipStream_t stream);

int lbm_launch_linear(const void* a, const lbm_row_norm* a_norm, const void* w, const float* bias, const float* gamma,
                      const void* residual, void* out, float* out_stats, int M, int N, int K, int epilogue,
                      void* workspace, size_t workspace_bytes, hipStream_t stream);
int lbm_linear_stats_tiles_for(int M, int N);

void lbm_set_prefetch_hint(const LbmTouch& t);   // the calling thread's next launch asks for these ranges alone
void lbm_take_prefetch_hint(LbmTouch& t);
// The grid of a launch of `wgs` workgroups, one a CU: with t.wgs more that ask for t's ranges where its last round leaves
// kTouchIdle CUs without work (16 or 64: within 0.5 % of a frame for most sizes, but 16 three anchor frames of 666 rows 8 % slower).
dim3 lbm_touch_grid(LbmTouch& t, unsigned wgs);
// How lbm_linear_norm (heads 0) or the qkv projection of so many heads would ask for a hint
LbmAsks lbm_linear_asks(int M, int N, int K, int epilogue, int heads, bool may_split);
size_t lbm_linear_workspace_for(int M, int N, int K, int epilogue);

int lbm_launch_qkv_linear_prepare(const void* a, const lbm_row_norm* a_norm, const void* w, const float* bias, int M, int K,
                                  const float* q_norm_w, const float* q_norm_b, const float* k_norm_w,
                                  const float* k_norm_b, float norm_eps, float q_scale, const float* rope_cs, int rope_layout,
                                  void* q_out, void* k_out, void* v_out, void* pool, const int32_t* append_rows,
                                  int num_heads, int page_size, hipStream_t stream);

// Split-KV schedule of one attention call, computed on the host from token counts only.
struct LbmAttnStreamPlan {
  int32_t q_begin, q_rows, kv_row_begin, kv_tokens, live_at;
  int32_t n_qtiles, n_splits, tiles_per_split;
  int32_t wg_begin;    // first workgroup of this stream
  int32_t part_begin;  // first partial-result row (unit: q row of one split) in the workspace
  uint32_t per_qtiles; // lbm_per(n_qtiles), for the launch
};
struct LbmAttnSchedule {
  int32_t n_streams;
  int32_t total_wgs;
  int32_t small;       // query rows per workgroup of the in-workgroup split kernel (no partial results), 0: the split-KV kernel
  bool fixed_order;    // no rotation of a stream's pieces either (lbm_attn_schedule)
  int64_t part_rows;   // rows of partial results over all streams (0 when nothing is split)
  LbmAttnStreamPlan s[LBM_MAX_STREAMS];
};
// fixed_order: neither the schedule's rule for one stream's cache nor workgroups that begin at different pieces.
// lbm_block_run and calls with LBM_ATTN_FIXED_ORDER ask for it: 24 blocks make the last bits of an attention into 0.2 % of the
// last block's K and V, single values up to 7 %, and a model's results must not move with a schedule.  Needs at least the workspace of the other.
void lbm_attn_schedule(const lbm_attn_stream* streams, int n_streams, int num_heads,
                       LbmAttnSchedule* out, bool fixed_order);
// least: what a launch cannot do without; otherwise what it is fastest with
size_t lbm_attn_schedule_bytes(const LbmAttnSchedule& sch, int num_heads, int head_dim, bool least);

struct AttnCoreF32 {
  const float* q;
  const float* pool;
  float* out;
  const float* self_k;
  const float* self_v;
  const int32_t* kv_rows;
  const int32_t* live_kv_tokens;
  int num_heads;
  int page_size;
  float scale_log2;
  int n_streams;
  unsigned per_heads, per_eighth;   // lbm_per of the heads, and of an eighth of them where that is whole
  // the append carried by workgroups behind the attention's (LBM_ATTN_APPEND_APART; 0 tokens: none): row t of
  // self_k / self_v to pool row append_rows[t]
  const int32_t* append_rows;
  int append_tokens;
};
template <int S>   // room for so many streams, 1 or LBM_MAX_STREAMS (as AttnArgs of the bf16 kernels)
struct AttnArgsF32 : AttnCoreF32 {
  lbm_attn_stream s[S];
  int wg_begin[S + 1];     // beyond the streams: more than any workgroup's index
};
// fp32 attention at head_dim 64 on bf16 matrix instructions (paged_attn_f32_gfx950.hip)
template <int S>
int lbm_launch_attn_f32_d64(AttnArgsF32<S>& a, hipStream_t stream);

int lbm_launch_attention(const void* q, const void* pool, void* out, const void* self_k,
                         const void* self_v, const int32_t* kv_rows, const int32_t* live_kv_tokens,
                         const LbmAttnSchedule& sch,
                         int num_heads, int head_dim, int page_size, int dtype, float sm_scale,
                         void* workspace, size_t workspace_bytes, hipStream_t stream,
                         const int32_t* append_rows = nullptr, int append_tokens = 0, bool append_apart = false,
                         bool own_rows = false, const LbmTouch* touch = nullptr);
// Whether such a launch (bf16, no live counts, nothing to append) carries workgroups that ask for a hint: its kernel has them
// and CUs are idle
bool lbm_attention_asks(const LbmAttnSchedule& sch, bool own_rows);

#ifdef __HIPCC__
// 16 or 8 bytes stored past the L2 (device scope), for results that whole lines of neighbouring lanes leave.  A kernel ends
// when the lines its stores left dirty in the eight L2s have been written back, and the next launch waits for that: a chain
// of launches that write 2 MB each takes 1.91 us a launch with plain stores and 1.62 with these, one that also reads what the
// launch before it wrote 2.74 and 2.49 (the readers' L2s drop the lines at a launch's start either way).  Replayed
// aggregator frame of 1,004 rows 6.65 -> 6.49 ms, four streams 16.15 -> 15.90, eight anchor frames 24.7 -> 24.2.  Not for
// scattered 4- and 8-byte results (log-sum-exps, row statistics): those the L2 collects into lines, and past it the
// attention of four streams takes 1 % longer.
// (s_nop 1: two wait states before a vector instruction may write the registers that a 16-byte store still reads, which the
// compiler sees to behind its own stores and cannot behind inline asm)
__device__ __forceinline__ void lbm_store_through(void* dst, __attribute__((ext_vector_type(4))) unsigned int v) {
  asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" : : "v"(dst), "v"(v) : "memory");
}
__device__ __forceinline__ void lbm_store_through(void* dst, __attribute__((ext_vector_type(2))) unsigned int v) {
  asm volatile("global_store_dwordx2 %0, %1, off sc1" : : "v"(dst), "v"(v) : "memory");
}
// What workgroups with blockIdx.y > 0 do, thread by thread, and, where a kernel has one (`wave`), the wavefront beside the
// computing ones in a launch without such workgroups.  In a model every launch finds its weights in HBM - a frame walks
// through 600 MB of them, the caches hold 256 - and the loop's steps of look-ahead cover a trip to the memory-side cache, not
// that.  A caller that knows which memory launches behind this one will read says so, and these threads read one dword of every
// 128-byte line of it; the lines have then travelled while the launch computed.  (Plain loads whose results the compiler sees - a load
// whose result it does not know of could land in a register it has reused - eight in flight per lane.  The kernels call it
// in one place, behind a branch on a scalar register: called in two, its arguments were loaded in front of the computing
// path, 0.2 us of every launch.)
// Workgroups of their own where CUs are idle: a wavefront beside the computing ones takes its CU's vector memory path from
// them and may end after them, as 48 workgroups' wavefronts with 1,365 lines each did: qkv projection, proj, fc1 and fc2
// of 86 rows 34.6 us by wavefronts (34.2 without a hint, 25.3 with the weights in the caches), 27.1 by workgroups; 261 rows
// 33.4 -> 30.9, 566 rows 44.1 -> 41.8.
__device__ __forceinline__ void lbm_touch(const LbmTouch& t, unsigned threads, bool wave) {
  const LbmTouchPlace at = lbm_touch_place(t, blockIdx.x, blockIdx.y, gridDim.x, threadIdx.x, threads, wave);
  if (!at.step) return;
  const LbmTouchPart part = lbm_touch_part(t, at.xcd, at.xcd_shift);
  for (unsigned from = at.first; from < part.end; from += 8u * at.step) {
    unsigned got[8], folded = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const unsigned line = from + (unsigned)j * at.step;
      got[j] = line < part.end ? *(const __attribute__((address_space(1))) unsigned*)lbm_touch_line(part, line) : 0u;   // (from an integer it would be a flat load)
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) folded ^= got[j];
    asm volatile("" : : "v"(folded));
  }
}
// The append as workgroups of an attention launch: workgroup `wg` of those behind the attention's copies N 16-byte
// pieces of a K row and of the matching V row per thread (row_pieces: 16-byte pieces per row).
template <int N = 1>
__device__ __forceinline__ void lbm_append_pieces(const void* k, const void* v, void* pool, const int32_t* append_rows,
                                                  int append_tokens, int row_pieces, int page_size, int wg, int threads) {
  typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;
  // (the workgroup's first piece is uniform; from there 32 bits are enough)
  const long long base = (long long)wg * N * threads, left = (long long)append_tokens * row_pieces - base;
  const int t0 = (int)(base / row_pieces);
  const unsigned at0 = (unsigned)(base - (long long)t0 * row_pieces) + threadIdx.x;
  if ((long long)threadIdx.x >= left) return;
  u32x4 kk[N], vv[N];
  int row[N];
  unsigned piece[N];
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const bool there = (long long)(threadIdx.x + j * threads) < left;   // past the end: the thread's first once more, not stored
    const unsigned at = at0 + (there ? (unsigned)(j * threads) : 0u), t = at / (unsigned)row_pieces;
    piece[j] = at - t * (unsigned)row_pieces;
    const long long idx = (long long)t0 * row_pieces + at;
    row[j] = append_rows[t0 + (int)t];
    if (!there) row[j] = -1;
    kk[j] = ((const u32x4*)k)[idx];
    vv[j] = ((const u32x4*)v)[idx];
  }
#pragma unroll
  for (int j = 0; j < N; ++j) {
    if (row[j] < 0) continue;
    u32x4* dst = (u32x4*)pool + (long long)row[j] * row_pieces + piece[j];
    lbm_store_through(dst, kk[j]);
    lbm_store_through(dst + (long long)page_size * row_pieces, vv[j]);
  }
}
#endif

// Address and size of the library's static device scratch array on the current device (looked
// up once per device; no allocation).
int lbm_static_scratch(void** ptr, size_t* bytes);

#endif  // LBM_INTERNAL_H
