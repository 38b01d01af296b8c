// Ragged paged attention forward for gfx950: out = softmax(q k^T * scale) v over the K/V
// rows a row table names (pool pages in any order, partially filled pages already squeezed
// out by the table, optional read-only tail from the caller's own K/V).
//
// bf16 kernel, head_dim 64.  One workgroup = 8 wavefronts x 64 query rows of one head over
// one contiguous run of 64-token KV tiles (split-KV; partial results are merged by
// lbm_attn_combine_bf16_kernel).  Per tile a wavefront computes
//     S^T = K Q^T      v_mfma_f32_32x32x16_bf16, A = K rows from LDS, B = Q in registers; the
//                      softmax scale (in log2 units) is folded into Q, so S arrives ready
//                      for exp2
//     P   = exp2(S)    one query row per lane column; v_exp_f32 + v_cvt_pk_bf16_f32
//     O^T += V^T P^T   A = V^T read with ds_read_b64_tr_b16 from the row-major V tile,
//                      B = P^T straight from the registers the packing wrote
//     l   += 1^T P^T   row sums on the matrix pipe too (16x16x32 with a 0/1 selector)
// Common path: no softmax reference at all.  2^score is exact softmax arithmetic as long as
// nothing leaves the range of fp32 / bf16; a range check on O and l after the last tile
// decides, per workgroup, whether that held.  If not - scores beyond about +-100 in log2
// units - the workgroup repeats its split in an out-of-line function (lbm_attn_split_safe)
// with a reference m carried into the QK^T contraction as one more k-step: m is kHeadroom
// above the row maximum seen when it was last set and is only raised when a numerator
// reaches 2 (a bf16 numerator is >= 2 or infinite exactly when the top bit of its exponent
// field is set: a few OR instructions per half tile), with O, l and the scores in flight
// rescaled on that rare path.  The same extra k-step masks the rows past the last token on
// the ragged last tiles of either path.
//
// Why it is built this way.  Measured on MI355X with two wavefronts per SIMD: v_exp_f32 issues
// every ~4.6 ns per SIMD, v_cvt_pk_bf16_f32 (like v_max3_f32, v_dot2c_f32_bf16) every ~2.7 ns, plain
// fp32 adds and multiplies every ~1.4 ns, and a 32x32x16 MFMA occupies the matrix pipe for
// 13.8 ns.  With head_dim 64 every score needs one exp2 and half a packing instruction, so the
// vector ALU is as busy as the matrix pipe; everything that can run as an MFMA (scale, row
// sums, masking of the ragged tail, the reference subtraction of the repeat pass) does, and
// the vector ALU is left with exp2 and packing.
//
// Schedule.  Each wavefront runs a software pipeline over 32-token half tiles: while the
// vector ALU turns the scores of one half into numerators, the MFMAs of the next half's QK^T
// and of the previous half's PV and row sums are issued in between.  A half-step is one basic
// block written as 20 slices (22 with the extra k-step; one MFMA plus its share of the vector
// work and LDS reads each) fenced with sched_barrier, and the two wavefronts of a SIMD fill
// each other's issue gaps.  K/V tiles are shared by all eight waves through a three-stage
// LDS ring with one workgroup barrier per tile; the rows go from global memory straight into
// the ring (global_load_lds_dwordx4), no staging registers and no LDS store instructions.
#include <hip/hip_runtime.h>
#include <climits>
#include <mutex>
#include <type_traits>
#include "lbm_internal.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(8))) float f32x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;
typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;
typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef __attribute__((ext_vector_type(8))) short s16x8;

namespace {

constexpr int kKvTile = 64;             // KV tokens per tile
constexpr int kQPerWave = 64;           // query rows per wavefront (two 32-row MFMA blocks)
constexpr int kWaves = 8;
constexpr int kThreads = kWaves * 64;
constexpr int kQTile = kQPerWave * kWaves;
constexpr int kStages = 3;              // LDS ring depth
constexpr int kRingRow = 64;            // bf16 per row of a K/V tile in the LDS ring: 128 B, unpadded, 16-byte chunks swizzled
constexpr int kKStride = 72;            // bf16 per row of a padded patch (Q, output transpose): 144 B, b128 reads hit 64 distinct banks
constexpr float kHeadroom = 11.0f;      // the softmax reference is set this far above the row maxima (log2 units)

// 16-byte pieces of K and of V per thread of a workgroup that appends, in the split-KV launch.  In the short-KV launch and the
// merging one it is one: stored past the L2 they take no longer than they did with plain stores (us, plain and these:
// short-KV 65 rows over 325 tokens 7.0, 6.7, 261 over 4,437 20.9, 20.8, 500 over 2,000 14.8, 14.8; merge 1,004 rows over 17,068
// 6.3, 6.1, 505 over 8,585 5.7, 5.0).
constexpr int kAppendPieces = 4;

struct AttnCore {
  const unsigned short* q;
  const unsigned short* pool;
  unsigned short* out;
  const unsigned short* self_k;
  const unsigned short* self_v;
  const int32_t* kv_rows;
  const int32_t* live_kv_tokens;  // device-side token counts (NULL: the host's counts in the plan)
  unsigned short* part_o;  // split-KV partial outputs, normalised, bf16
  float* part_lse;
  int num_heads;
  int page_size;
  float scale_log2;
  // the append carried by workgroups behind those of the attention, or by the merging launch: row t of
  // self_k / self_v to pool row append_rows[t]
  const int32_t* append_rows;
  int append_tokens;
  int combine_blocks;      // blocks (per stream) of that launch that merge; those beyond them append
  unsigned per_heads, per_eighth;   // lbm_per of the heads, and of an eighth of them where that is whole
};
// S: streams that a launch's arguments have room for, 1 or LBM_MAX_STREAMS.  The runtime copies a launch's arguments on their way to
// the GPU: 0.4 us of the host for 0.9 KB of them that a launch of one stream does not read (82 and 261 own rows, whose calls wait for
// the host, 5.6 -> 5.25 and 5.7 -> 5.35 us).
template <int S>
struct AttnArgs : AttnCore {
  int32_t n_streams, total_wgs;
  LbmAttnStreamPlan s[S];
  int32_t first_wg[S];       // s[i].wg_begin, beyond the streams more than any workgroup
  LbmTouch touch;
};

// The first stream's plan, with everything else that a workgroup's first loads need of the arguments: asked for at once.  A launch
// finds its arguments in no cache; read where they are used - the workgroup count, the streams', the plan, the live counts'
// address, q's, k's - they were four to six trips one behind the other, with two integer divisions in between, in front of
// the first row's request.  us: 1,004 own rows 9.7 -> 9.2, 479 of 12 heads 6.3 -> 5.8, a block of 195 rows over 585 tokens 7.5 -> 6.9, of
// 261 over 4,437 20.7 -> 20.3, of four streams of 280 rows 23.5 -> 22.9, a read-only frame of 285 rows over 5,455 tokens 26.0 -> 24.9.
template <int S>
__device__ __forceinline__ LbmAttnStreamPlan lbm_first_plan(const AttnArgs<S>& a) {
  const LbmAttnStreamPlan sp = a.s[0];
  asm volatile("" : : "s"(a.total_wgs), "s"(a.n_streams), "s"(a.num_heads), "s"(a.per_heads), "s"(a.per_eighth), "s"(a.live_kv_tokens), "s"(a.q),
               "s"(a.self_k), "s"(a.self_v), "s"(a.pool), "s"(a.kv_rows), "s"(a.page_size), "s"(sp.q_begin), "s"(sp.q_rows), "s"(sp.kv_row_begin), "s"(sp.kv_tokens),
               "s"(sp.n_qtiles), "s"(sp.n_splits), "s"(sp.tiles_per_split), "s"(sp.wg_begin), "s"(sp.per_qtiles));
  return sp;
}
// A workgroup's plan where there are several streams
template <int S>
__device__ __forceinline__ void lbm_plan_of_workgroup(const AttnArgs<S>& a, LbmAttnStreamPlan& sp) {
  if (S == 1 || a.n_streams == 1) return;
  int b = 0;
#pragma unroll
  for (int i = 1; i < S; ++i) b += (int)((unsigned)(a.first_wg[i] - 1 - (int)blockIdx.x) >> 31);   // (no compare: its result would go by way of a vector register)
  sp = a.s[b];
}

// Exchange between lane l and lane l^32.  v_permlane32_swap swaps the upper half of its first
// register with the lower half of its second; fed two copies of x it leaves {x_lo, x_lo} in
// the first and {x_hi, x_hi} in the second.  Inline asm with the wait states from a VALU write to
// the permlane's read in it; the builtin compiles to the same instruction, provided that its two results
// are read by value (see float_bits).
__device__ __forceinline__ void swap_halves(float x, float& lo, float& hi) {
  float a = x, b = x;
  asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
  lo = a;
  hi = b;
}
// The same for neighbouring rows of 16 lanes: v_permlane16_swap swaps the odd rows of its first
// register with the even rows of its second; fed two copies of x it leaves rows {0, 0, 2, 2}
// in the first and rows {1, 1, 3, 3} in the second.
__device__ __forceinline__ void swap_rows(float x, float& even, float& odd) {
  float a = x, b = x;
  asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
  even = a;
  odd = b;
}
// Built with -fno-honor-nans, fmaxf chains become v_max3_f32 without NaN-quieting moves.
__device__ __forceinline__ float max3(float a, float b, float c) { return fmaxf(fmaxf(a, b), c); }
__device__ __forceinline__ float max2(float a, float b) { return fmaxf(a, b); }
__device__ __forceinline__ float swap_max(float x) {
  float lo, hi;
  swap_halves(x, lo, hi);
  return max2(lo, hi);
}
// A float's bits.  Vector elements go through it: __builtin_bit_cast(unsigned, v[i]) on an
// ext_vector lvalue takes the vector's address and so returns element 0 whatever i is.
__device__ __forceinline__ unsigned float_bits(float x) { return __builtin_bit_cast(unsigned, x); }

// loads of this wavefront still allowed in flight (expcnt and lgkmcnt untouched); its LDS accesses done
#define LBM_LOADS_LEFT(N) asm volatile("s_waitcnt vmcnt(%0)" : : "i"(N) : "memory")
#define LBM_LDS_DONE() asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory")

// LDS of the split-KV kernel, at namespace scope because the kernel and the out-of-line second
// pass below both work in it.
__shared__ __attribute__((aligned(1024))) unsigned short lds_k[kStages][kKvTile * kRingRow];
__shared__ __attribute__((aligned(1024))) unsigned short lds_v[kStages][kKvTile * kRingRow];
__shared__ __attribute__((aligned(16))) unsigned short lds_q[kWaves][kQPerWave * kKStride];   // per-wave patch: Q on the way in, O on the way out

// The repeat pass is a function of its own, not inlined: it is entered once in a blue moon,
// and compiled into the kernel body its registers would push the common path into scratch
// memory (spill stores and reloads on every launch, tens of MB of HBM traffic).
// (it takes the 130 bytes it needs, not the whole argument block with its sixteen stream plans:
// what is passed by value sizes the kernel's scratch frame)
__device__ __noinline__ void lbm_attn_split_safe(AttnCore a, LbmAttnStreamPlan sp);
__device__ __noinline__ void lbm_attn_pair_safe(AttnCore a, LbmAttnStreamPlan sp);

// LDS of the same with both splits of 256 query rows in one workgroup (PAIR below): a ring per split, and patches that
// the two wavefronts of the same 64 rows share.
__shared__ __attribute__((aligned(1024))) unsigned short lds_pair_k[2][kStages][kKvTile * kRingRow];
__shared__ __attribute__((aligned(1024))) unsigned short lds_pair_v[2][kStages][kKvTile * kRingRow];
__shared__ __attribute__((aligned(16))) unsigned short lds_pair_q[kWaves / 2][kQPerWave * kKStride];
__shared__ float lds_pair_lse[kWaves][32];   // log-sum-exps of the 32 rows that the other wavefront merges

// One workgroup's share of the split-KV attention: 512 query rows of one head over one run of
// KV tiles, start to finish.  SAFE = false is the common path (no softmax reference, range
// check at the end); when the check fails it writes nothing, hands the workgroup to the
// repeat pass and ends the program there, so that nothing of the common path is live across
// the call.  SAFE = true is the repeat with a reference that follows the row maxima.
//
// PAIR: launches whose streams attend to their own rows in order in two splits each (several streams' frame and encoder
// blocks).  Wavefronts 0-3 take 256 query rows over the first split, 4-7 the same rows over the second, each group from a
// ring of its own, and the two meet through LDS where the partial results of other launches go through memory to a second
// kernel: rounded to bf16 and weighted as there, the same bits.  As many workgroups as 512 rows x two splits make, or
// fewer; a group stages a tile by itself, twice the bytes into LDS per product, of which there were few (DMA of 32 KB per
// 2,300 cycles).
// OWN (and PAIR): token t of a stream is row kv_row_begin + t of the caller's K/V, addressed without the row table.  (The
// repeat pass of a launch that is not PAIR reads the table, which says the same.)
template <bool SAFE, bool PAIR, bool OWN = PAIR>
__device__ __forceinline__ void lbm_attn_split(const AttnCore& a, const LbmAttnStreamPlan& sp) {
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n32 = lane & 31, g = lane >> 5;
  constexpr int kRowWaves = PAIR ? kWaves / 2 : kWaves;      // wavefronts with query rows of their own
  constexpr int kPieces = kWaves / kRowWaves;                // 16-byte pieces of a tile's K (and V) rows per thread
  const int group = PAIR ? wave / kRowWaves : 0, rw = PAIR ? wave % kRowWaves : wave;
  unsigned short (*const ring_k)[kKvTile * kRingRow] = PAIR ? lds_pair_k[group] : lds_k;
  unsigned short (*const ring_v)[kKvTile * kRingRow] = PAIR ? lds_pair_v[group] : lds_v;
  unsigned short* const patch = PAIR ? lds_pair_q[rw] : lds_q[wave];

  // ---- which piece of this stream's work is this workgroup
  const int H = a.num_heads;
  const int local = (int)blockIdx.x - sp.wg_begin;
  const int n_hs = PAIR ? H : H * sp.n_splits;
  int qt, hs;
  if ((n_hs & 7) == 0) {
    // Workgroups are dealt to the 8 XCDs round-robin: keep the query tiles that share one
    // (head, split) - hence the same K/V rows - on one XCD so its L2 serves the re-reads.
    const int x = local & 7, i = local >> 3;
    hs = lbm_divide(i, sp.n_qtiles, sp.per_qtiles, qt) * 8 + x;
  } else {
    hs = lbm_divide(local, sp.n_qtiles, sp.per_qtiles, qt);
  }
  if (local >= sp.n_qtiles * n_hs) return;  // padding between streams
  int head = hs, split = group;
  if (!PAIR) split = lbm_divide(hs, H, a.per_heads, head);
  // With device-side token counts the split count stays the host's choice (it fixes the grid
  // and the workspace layout) and the tiles are dealt to the splits from the live count.
  const int kv_tokens = !OWN && a.live_kv_tokens ? a.live_kv_tokens[sp.live_at] : sp.kv_tokens;
  if (!PAIR && kv_tokens <= 0 && sp.n_splits == 1) {
    // nothing visible: the reference returns zeros (lingbot_map/layers/flashinfer_cache.py:368-370)
    for (int k = 0; k < kQPerWave / 8; ++k) {
      const int r = qt * kQTile + wave * kQPerWave + k * 8 + (lane >> 3);
      if (r < sp.q_rows)
        *(u32x4*)(a.out + ((size_t)(sp.q_begin + r) * H + head) * 64 + (lane & 7) * 8) = u32x4{0u, 0u, 0u, 0u};
    }
    return;
  }
  const int n_tiles = (max(kv_tokens, 0) + kKvTile - 1) / kKvTile;
  const int tiles_per_split = !OWN && a.live_kv_tokens ? max((n_tiles + sp.n_splits - 1) / sp.n_splits, 1) : sp.tiles_per_split;
  const int t0 = split * tiles_per_split;
  const int t1 = min(t0 + tiles_per_split, n_tiles);  // an empty split (t1 <= t0) contributes weight 0
  const int n = t1 - t0;
  const int n_most = PAIR ? max(min(tiles_per_split, n_tiles), 0) : n;   // tiles of the longer of the workgroup's splits, the first
  const unsigned row_bytes = (unsigned)H * 128u;

  // ---- tile staging: each thread moves one 16-byte piece of a K row and of a V row per tile,
  // global -> LDS without a stop in registers (global_load_lds_dwordx4: the wavefront's 64
  // pieces land on 1 KiB of consecutive LDS starting at M0, i.e. on eight 128-byte rows).  A
  // tile in the ring is therefore 64 unpadded rows, and what keeps the fragment reads off each
  // other's banks is the order of the eight 16-byte chunks within a row, which each lane
  // chooses by the global address it reads: chunk c of K row r sits at position
  // c ^ ((r >> 1) & 7) (the b128 fragment reads of 16 rows x one chunk hit all 64 banks), chunk
  // c of V row r at c ^ 4 ((r >> 1) & 1) (the 8-byte transposed reads touch four rows x 64
  // bytes; rows r+2 and r+3 move to the other half).  The compiler does not count these loads
  // (its own waits only get stricter by that); LBM_DMA_LANDED waits for them before the
  // barrier that publishes a tile.  M0 is declared clobbered, so the compiler keeps nothing of
  // its own in it across a load.
  // Rows past the last token re-read the last token (finite data; the softmax masks them).
  const int ld_r = (PAIR ? tid % (kRowWaves * 64) : tid) >> 3;
  const int ld_ck = ((lane & 7) ^ ((ld_r >> 1) & 7)) * 8, ld_cv = ((lane & 7) ^ (((ld_r >> 1) & 1) * 4)) * 8;
  const char* pool_k = (const char*)(a.pool + (size_t)head * 64 + ld_ck);
  const char* pool_v = (const char*)(a.pool + (size_t)head * 64 + ld_cv) + (size_t)a.page_size * row_bytes;
  const char* own_k = (const char*)(a.self_k + (size_t)head * 64 + ld_ck);
  const char* own_v = (const char*)(a.self_v + (size_t)head * 64 + ld_cv);
  const int32_t* rows = a.kv_rows + sp.kv_row_begin;
  const int last_token = max(kv_tokens - 1, 0);
  // Tiles past the end of this split re-read its last tile: the data lands in ring stages
  // nobody reads any more, and the code stays free of branches.
  // OWN: the "entry" of a tile is its first token.
  auto row_entry = [&](int t) -> int {
    const int first = max(min(t, t1 - 1), 0) * kKvTile;
    return OWN ? first : rows[min(first + ld_r, last_token)];
  };
  auto dma = [&](int e, const char* pool_base, const char* own_base, const unsigned short* lds_tile) {
#pragma unroll
    for (int k = 0; k < kPieces; ++k) {
      // negative entries name rows of the caller's own K/V (read-only tail of a non-keyframe)
      const char* base = OWN || e < 0 ? own_base : pool_base;
      const unsigned r = OWN ? (unsigned)(sp.kv_row_begin + min(e + ld_r + k * (kKvTile / kPieces), last_token)) : (unsigned)(e ^ (e >> 31));
      const char* src = base + (unsigned long long)r * row_bytes;
      const unsigned m0v = (unsigned)(size_t)(__attribute__((address_space(3))) const void*)(lds_tile + (k * kRowWaves + rw) * (8 * kRingRow));
      asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off"
                   :
                   : "v"(src), "s"(__builtin_amdgcn_readfirstlane(m0v))
                   : "memory", "m0");
    }
  };
#define LBM_DMA_LANDED() __builtin_amdgcn_s_waitcnt(0x0F70)   /* vmcnt(0); expcnt and lgkmcnt untouched */

  // The first tiles' rows are asked for before anything else: the row table entry, then the K/V
  // row it names, is the longest chain of memory latencies in front of the first MFMA, and the
  // Q rows below travel at the same time.
  const int e_t0 = row_entry(t0), e_t1 = row_entry(t0 + 1);
  int ek = row_entry(t0 + 2), ev = e_t1;   // entries of the loads of the first iteration
  dma(e_t0, pool_k, own_k, ring_k[0]);
  dma(e_t1, pool_k, own_k, ring_k[1]);
  dma(e_t0, pool_v, own_v, ring_v[0]);

  // ---- Q fragments (B operand of S^T = K Q^T): lane holds q row n32, d = ks*16 + g*8 .. +8.
  // Each wavefront reads its 64 query rows as whole 128-byte rows (eight lanes per row), parks
  // them in its own LDS patch and picks the fragments up from there; read directly in the
  // fragment layout every load instruction would touch 64 different rows with 16 bytes each.
  // The softmax scale and log2(e) are folded into Q here (one extra bf16 rounding of q; none
  // when the producer already multiplied q by them before its own rounding and the caller
  // passed sm_scale = 0), so the MFMA result is already the exponent of 2.
  bf16x8 qf[2][4];
  const int q_row0 = (qt * kRowWaves + rw) * kQPerWave;
  {
    constexpr int kRaw = kQPerWave / 8 / kPieces;            // (PAIR: half of them, the other group's wavefront the rest)
    u32x4 raw[kRaw];
#pragma unroll
    for (int k = 0; k < kRaw; ++k) {
      // rows past the stream's last query row re-read that row: their results are never stored,
      // and eight unconditional loads go out back to back (a load inside a conditional block
      // ends up with a wait for everything in flight behind it)
      const int r = max(min(q_row0 + (group * kRaw + k) * 8 + (lane >> 3), sp.q_rows - 1), 0);
      raw[k] = *(const u32x4*)(a.q + ((size_t)(sp.q_begin + r) * H + head) * 64 + (lane & 7) * 8);
    }
#pragma unroll
    for (int k = 0; k < kRaw; ++k)
      *(u32x4*)&patch[((group * kRaw + k) * 8 + (lane >> 3)) * kKStride + (lane & 7) * 8] = raw[k];
    __syncthreads();   // (a wavefront only reads its own patch, PAIR: the two that share it; the barrier orders writes and reads)
#pragma unroll
    for (int qb = 0; qb < 2; ++qb)
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        const bf16x8 rawf = __builtin_bit_cast(bf16x8, *(const u32x4*)&patch[(qb * 32 + n32) * kKStride + ks * 16 + g * 8]);
        f32x8 f = __builtin_convertvector(rawf, f32x8);
#pragma unroll
        for (int j = 0; j < 8; ++j) f[j] *= a.scale_log2;
        // (a q that already carries the scale - scale_log2 == 1 - comes back bit for bit: x * 1 is exact)
        qf[qb][ks] = __builtin_convertvector(f, bf16x8);
      }
  }
  // One more 16-wide step of the QK contraction carries the softmax reference: K side is the
  // constant row (-1, -1, 0, ...), Q side is (m_hi, m_lo, 0, ...) with m_hi + m_lo = m_run
  // exactly, so S arrives as score*scale - m_run at no vector-ALU cost.
  // A third element masks the rows past the last token: K side -1 on such rows (0 elsewhere),
  // Q side 2^100, so their scores arrive as about -2^100 and their numerators are exactly 0.
  u32x4 kaug_bits = {0u, 0u, 0u, 0u};
  if (g == 0) kaug_bits[0] = 0xBF80BF80u;
  u32x4 qaug_bits[2] = {{0u, 0u, 0u, 0u}, {0u, 0u, 0u, 0u}};
  if (g == 0) qaug_bits[0][1] = qaug_bits[1][1] = 0x7180u;  // bf16 2^100

  // Accumulators and softmax reference; (re)initialised at the start of each pass below.
  f32x16 o[2][2];
  float m_run[2];
  // Row sums (softmax denominators) are accumulated by the matrix pipe as well: a 16x16x32 MFMA
  // with a 0/1 selector as A and the numerators, exactly as they sit in the registers for PV,
  // as B.  Read as a 32x16 B operand the numerator registers hold, for column n, query n in
  // k rows 0-7 and 16-23 and query n+16 in k rows 8-15 and 24-31; selector row 0 picks the
  // former and row 1 the latter, so lane n < 16 ends up with the sums of query n (element 0)
  // and of query n+16 (element 1) of the block, and every other element stays 0.
  f32x4 lacc[2];
  const unsigned sel_word = (lane == 0 || lane == 32 || lane == 17 || lane == 49) ? 0x3F803F80u : 0u;
  const bf16x8 lsel = __builtin_bit_cast(bf16x8, u32x4{sel_word, sel_word, sel_word, sel_word});

  // Register state of the software pipeline.  A 64-token tile is processed as two 32-token
  // halves; while the vector ALU turns the scores of one half into softmax numerators, the
  // matrix pipe computes the scores of the next half and folds the numerators of the
  // previous half into O.  The two halves alternate between the A and B register sets.
  f32x16 sA[2], sB[2];        // s[qb][i]: kv = 32*half + 8*(i/4) + 4*g + i%4, q = qb*32 + n32
  bf16x8 pA[2][2], pB[2][2];  // numerators [qb][k-step] as the B operand of O^T += V^T P^T
  bf16x8 vnext[2];            // V^T fragments of the next PV's first k-step, read early

  // V^T fragment (A operand): lane holds d = db*32 + n32 and the kv rows
  // ks*16 + {4g..4g+3, 8+4g..8+4g+3} of the V tile in stage st
  auto v_frag = [&](int st, int ks, int db) -> bf16x8 {
    const int row = ks * 16 + 4 * g + ((lane & 15) >> 2);
    const int col = (db * 32 + ((lane >> 4) & 1) * 16 + (lane & 3) * 4) ^ (((lane >> 3) & 1) * 32);
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (s16x4 __attribute__((address_space(3)))*)&ring_v[st][row * kRingRow + col]);
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (s16x4 __attribute__((address_space(3)))*)&ring_v[st][(row + 8) * kRingRow + col]);
    s16x8 both;
    both[0] = lo[0]; both[1] = lo[1]; both[2] = lo[2]; both[3] = lo[3];
    both[4] = hi[0]; both[5] = hi[1]; both[6] = hi[2]; both[7] = hi[3];
    return __builtin_bit_cast(bf16x8, both);
  };
  // One k-step (16 kv rows) of O^T += V^T P^T; o[qb][db][i] is d = db*32 + 8*(i/4) + 4*g + i%4
  auto pv_step = [&](const bf16x8 (&va)[2], const bf16x8 (&p)[2][2], int kk) {
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
      for (int qb = 0; qb < 2; ++qb)
        o[qb][db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va[db], p[qb][kk], o[qb][db], 0, 0, 0);
  };
  // S^T = K Q^T - m_run for the 32 kv rows of half h of the K tile in stage st
  auto qk_half = [&](int st, int h, int n_valid, f32x16 (&sd)[2]) {
    f32x16 z;
#pragma unroll
    for (int i = 0; i < 16; ++i) z[i] = 0.f;
    u32x4 kb = kaug_bits;
    kb[1] = (g == 0 && h * 32 + n32 >= n_valid) ? 0xBF80u : 0u;
    const bf16x8 kaug = __builtin_bit_cast(bf16x8, kb);
#pragma unroll
    for (int qb = 0; qb < 2; ++qb)
      sd[qb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kaug, __builtin_bit_cast(bf16x8, qaug_bits[qb]), z, 0, 0, 0);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const bf16x8 ka = __builtin_bit_cast(
          bf16x8, *(const u32x4*)&ring_k[st][(h * 32 + n32) * kRingRow + ((ks * 2 + g) ^ ((n32 >> 1) & 7)) * 8]);
#pragma unroll
      for (int qb = 0; qb < 2; ++qb)
        sd[qb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka, qf[qb][ks], sd[qb], 0, 0, 0);
    }
  };
  // Row maxima of one half, per query block (the lane's own 16 scores, then the other
  // half-wave's through one swap).
  auto row_max = [&](const f32x16 (&sc)[2], float (&mx)[2]) {
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
      float m0 = max3(sc[qb][0], sc[qb][1], sc[qb][2]), m1 = max3(sc[qb][3], sc[qb][4], sc[qb][5]);
      m0 = max3(m0, sc[qb][6], sc[qb][7]);
      m1 = max3(m1, sc[qb][8], sc[qb][9]);
      m0 = max3(m0, sc[qb][10], sc[qb][11]);
      m1 = max3(m1, sc[qb][12], sc[qb][13]);
      m0 = max3(m0, sc[qb][14], sc[qb][15]);
      mx[qb] = swap_max(max2(m0, m1));
    }
  };
  // Numerators 2^s packed to bf16.
  auto numerators = [&](const f32x16 (&sc)[2], bf16x8 (&pd)[2][2]) {
#pragma unroll
    for (int qb = 0; qb < 2; ++qb)
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        f32x8 e;
#pragma unroll
        for (int j = 0; j < 8; ++j) e[j] = __builtin_amdgcn_exp2f(sc[qb][kk * 8 + j]);
        pd[qb][kk] = __builtin_convertvector(e, bf16x8);
      }
  };
  // Move the reference of query block qb to m_run + rise (rounded so that two bf16 values
  // carry it exactly) and return how far it moved.
  auto move_reference = [&](int qb, float rise) -> float {
    const float want = m_run[qb] + rise;
    const float hi = (float)(__bf16)want;
    const float lo = (float)(__bf16)(want - hi);
    const float d = (hi + lo) - m_run[qb];
    m_run[qb] = hi + lo;
    const bf16x2 pair = {(__bf16)hi, (__bf16)lo};
    qaug_bits[qb][0] = g == 0 ? __builtin_bit_cast(unsigned, pair) : 0u;
    return d;
  };
  // Rare path of a half-step: a numerator of `cur` came out as 2 or more, i.e. a score
  // exceeded the reference by at least 1 (in log2 units; an overflow to infinity included).
  // Nothing has consumed these numerators yet.  Raise the reference to kHeadroom above the row
  // maxima, rescale what is already expressed in the old one (O, the row sums, and the scores
  // of `cur` and of `next`, which the MFMAs of this half-step produced with the old reference)
  // and recompute the numerators, which are then at most 2^-kHeadroom.
  auto raise_reference = [&](f32x16 (&cur)[2], bf16x8 (&pd)[2][2], f32x16 (&next)[2]) {
    float mx[2];
    row_max(cur, mx);
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
      const float d = move_reference(qb, max2(mx[qb] + kHeadroom, 0.f));
      const float alpha = __builtin_amdgcn_exp2f(-d);
      // row sums: lane n < 16 holds query n in element 0 and query n + 16 in element 1
      const float alpha_hi = __builtin_bit_cast(
          float, __builtin_amdgcn_ds_bpermute(4 * ((lane & 15) + 16), __builtin_bit_cast(int, alpha)));
      lacc[qb][0] *= alpha;
      lacc[qb][1] *= alpha_hi;
#pragma unroll
      for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[qb][db][i] *= alpha;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        cur[qb][i] -= d;
        next[qb][i] -= d;
      }
    }
    numerators(cur, pd);
  };
// One half-step is one basic block of 22 MFMAs, written as 22 slices fenced by
// sched_barrier so that the interleaving is the one spelled out here.  Slice j issues MFMA j
//    0-3   O += V^T P^T, k-step 0 of `prev`        4-7   the same, k-step 1
//    8-11  row sums of `prev` (16x16x32)           12-13 reference step of the next scores
//   14-21  their four K steps
// then its share of the vector work on `cur` (two exp2 each in slices 0-15, the bf16 packing
// one slice later, then the OR of the packed words whose exponent bits tell whether any
// numerator reached 2) and the LDS reads of operands a few slices ahead of their MFMA.
//   cur/pd    scores of this half and where its numerators go
//   prev      numerators of the previous half; their V rows: k-step 0 already in vnext,
//             k-step 1 = k-step ks_pv of the V tile in stage st_pv
//   next      scores of the next half: K tile in stage st_qk, half h_qk, nv_qk valid tokens left
//   st_vn, ks_vn   V tile / k-step whose V^T goes to vnext for the following half-step
#define LBM_SLICE(j, cur, pd, prev, next, st_pv, ks_pv, st_qk, h_qk, st_vn, ks_vn, hook)           \
  {                                                                                              \
    /* ---- the MFMA of this slice */                                                            \
    if ((j) < 4)                                                                                 \
      o[(j) & 1][(j) >> 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(                            \
          vnext[(j) >> 1], prev[(j) & 1][0], o[(j) & 1][(j) >> 1], 0, 0, 0);                     \
    else if ((j) < 8)                                                                            \
      o[(j) & 1][((j) - 4) >> 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(                      \
          va[((j) - 4) >> 1], prev[(j) & 1][1], o[(j) & 1][((j) - 4) >> 1], 0, 0, 0);            \
    else if ((j) < 12)                                                                           \
      lacc[(j) & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(                                   \
          lsel, prev[(j) & 1][((j) - 8) >> 1], lacc[(j) & 1], 0, 0, 0);                          \
    else if ((j) < 14)                                                                           \
      next[(j) & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(                                   \
          kaug, __builtin_bit_cast(bf16x8, qaug_bits[(j) & 1]), zero16, 0, 0, 0);                \
    else                                                                                         \
      next[(j) & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(                                   \
          ka[((j) - 14) >> 1], qf[(j) & 1][((j) - 14) >> 1], next[(j) & 1], 0, 0, 0);            \
    /* ---- numerators of cur: exp2 of scores 2j, 2j+1; packing of the pair of slice j-1 */      \
    if ((j) < 16) {                                                                              \
      e[2 * (j)] = __builtin_amdgcn_exp2f(cur[(j) >> 3][(2 * (j)) & 15]);                        \
      e[2 * (j) + 1] = __builtin_amdgcn_exp2f(cur[(j) >> 3][(2 * (j) + 1) & 15]);                \
    }                                                                                            \
    if ((j) >= 1 && (j) <= 16) {                                                                 \
      constexpr int c = (j) - 1, ci = (2 * c) & 15;                                              \
      pd[c >> 3][ci >> 3][ci & 7] = (__bf16)e[2 * c];                                            \
      pd[c >> 3][ci >> 3][(ci & 7) + 1] = (__bf16)e[2 * c + 1];                                  \
    }                                                                                            \
    /* ---- OR of the packed numerators, one 4-word group per two slices once it is complete */  \
    if ((j) >= 5 && (j) <= 18 && (((j) - 5) & 3) < 2) {                                          \
      constexpr int grp = ((j) - 5) >> 2, w = (((j) - 5) & 3) * 2;                               \
      const u32x4 words = __builtin_bit_cast(u32x4, pd[grp >> 1][grp & 1]);                      \
      chk = ((j) == 5 ? 0u : chk) | words[w] | words[w + 1];                                     \
    }                                                                                            \
    /* ---- LDS reads */                                                                         \
    if ((j) == 0) va[0] = v_frag(st_pv, ks_pv, 0);                                               \
    if ((j) == 1) va[1] = v_frag(st_pv, ks_pv, 1);                                               \
    if ((j) == 10 || (j) == 12 || (j) == 14 || (j) == 16)                                        \
      ka[((j) - 10) >> 1] = __builtin_bit_cast(                                                  \
          bf16x8, *(const u32x4*)&ring_k[st_qk][((h_qk) * 32 + n32) * kRingRow + (((((j) - 10) >> 1) * 2 + g) ^ ((n32 >> 1) & 7)) * 8]); \
    if ((j) == 17) vnext[0] = v_frag(st_vn, ks_vn, 0);                                           \
    if ((j) == 18) vnext[1] = v_frag(st_vn, ks_vn, 1);                                           \
    hook(j)                                                                                      \
    __builtin_amdgcn_sched_barrier(0);                                                           \
  }
#define LBM_S4(j, ...) LBM_SLICE(j, __VA_ARGS__) LBM_SLICE(j + 1, __VA_ARGS__) LBM_SLICE(j + 2, __VA_ARGS__) LBM_SLICE(j + 3, __VA_ARGS__)
// `hot` tells whether a numerator of `cur` reached 2 (bf16 exponent field >= 128)
#define LBM_HALF_STEP(cur, pd, prev, next, st_pv, ks_pv, st_qk, h_qk, nv_qk, st_vn, ks_vn, hot, hook) \
  {                                                                                              \
    u32x4 kb = kaug_bits;                                                                        \
    kb[1] = (g == 0 && (h_qk) * 32 + n32 >= (nv_qk)) ? 0xBF80u : 0u;                             \
    const bf16x8 kaug = __builtin_bit_cast(bf16x8, kb);                                          \
    bf16x8 va[2], ka[4];                                                                         \
    float e[32];                                                                                 \
    unsigned chk;                                                                                \
    __builtin_amdgcn_sched_barrier(0);                                                           \
    LBM_S4(0, cur, pd, prev, next, st_pv, ks_pv, st_qk, h_qk, st_vn, ks_vn, hook)                       \
    LBM_S4(4, cur, pd, prev, next, st_pv, ks_pv, st_qk, h_qk, st_vn, ks_vn, hook)                       \
    LBM_S4(8, cur, pd, prev, next, st_pv, ks_pv, st_qk, h_qk, st_vn, ks_vn, hook)                       \
    LBM_S4(12, cur, pd, prev, next, st_pv, ks_pv, st_qk, h_qk, st_vn, ks_vn, hook)                      \
    LBM_S4(16, cur, pd, prev, next, st_pv, ks_pv, st_qk, h_qk, st_vn, ks_vn, hook)                      \
    LBM_SLICE(20, cur, pd, prev, next, st_pv, ks_pv, st_qk, h_qk, st_vn, ks_vn, hook)                   \
    LBM_SLICE(21, cur, pd, prev, next, st_pv, ks_pv, st_qk, h_qk, st_vn, ks_vn, hook)                   \
    /* the numerators exist before the test that follows, not only on its common branch */       \
    asm volatile("" : "+v"(pd[0][0]), "+v"(pd[0][1]), "+v"(pd[1][0]), "+v"(pd[1][1]));             \
    hot = (chk & 0x40004000u) != 0u;                                                             \
  }
// The same half-step without a softmax reference (scores go to exp2 as they come out of the
// QK^T product) and without the test: 20 slices, QK^T in slices 12-19 with its first k-step
// starting from zero.  Only for half-steps whose 32 KV rows are all valid tokens.
#define LBM_FSLICE(j, cur, pd, prev, next, st_pv, ks_pv, st_qk, h_qk, st_vn, ks_vn, hook)          \
  {                                                                                              \
    if ((j) < 4)                                                                                 \
      o[(j) & 1][(j) >> 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(                            \
          vnext[(j) >> 1], prev[(j) & 1][0], o[(j) & 1][(j) >> 1], 0, 0, 0);                     \
    else if ((j) < 8)                                                                            \
      o[(j) & 1][((j) - 4) >> 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(                      \
          va[((j) - 4) >> 1], prev[(j) & 1][1], o[(j) & 1][((j) - 4) >> 1], 0, 0, 0);            \
    else if ((j) < 12)                                                                           \
      lacc[(j) & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(                                   \
          lsel, prev[(j) & 1][((j) - 8) >> 1], lacc[(j) & 1], 0, 0, 0);                          \
    else if ((j) < 14)                                                                           \
      next[(j) & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka[0], qf[(j) & 1][0], zero16, 0, 0, 0); \
    else                                                                                         \
      next[(j) & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(                                   \
          ka[((j) - 12) >> 1], qf[(j) & 1][((j) - 12) >> 1], next[(j) & 1], 0, 0, 0);            \
    if ((j) < 16) {                                                                              \
      e[2 * (j)] = __builtin_amdgcn_exp2f(cur[(j) >> 3][(2 * (j)) & 15]);                        \
      e[2 * (j) + 1] = __builtin_amdgcn_exp2f(cur[(j) >> 3][(2 * (j) + 1) & 15]);                \
    }                                                                                            \
    if ((j) >= 1 && (j) <= 16) {                                                                 \
      constexpr int c = (j) - 1, ci = (2 * c) & 15;                                              \
      pd[c >> 3][ci >> 3][ci & 7] = (__bf16)e[2 * c];                                            \
      pd[c >> 3][ci >> 3][(ci & 7) + 1] = (__bf16)e[2 * c + 1];                                  \
    }                                                                                            \
    if ((j) == 0) va[0] = v_frag(st_pv, ks_pv, 0);                                               \
    if ((j) == 1) va[1] = v_frag(st_pv, ks_pv, 1);                                               \
    if ((j) == 8 || (j) == 10 || (j) == 12 || (j) == 14)                                         \
      ka[((j) - 8) >> 1] = __builtin_bit_cast(                                                   \
          bf16x8, *(const u32x4*)&ring_k[st_qk][((h_qk) * 32 + n32) * kRingRow + (((((j) - 8) >> 1) * 2 + g) ^ ((n32 >> 1) & 7)) * 8]); \
    if ((j) == 16) vnext[0] = v_frag(st_vn, ks_vn, 0);                                           \
    if ((j) == 17) vnext[1] = v_frag(st_vn, ks_vn, 1);                                           \
    hook(j)                                                                                      \
    __builtin_amdgcn_sched_barrier(0);                                                           \
  }
#define LBM_F4(j, ...) LBM_FSLICE(j, __VA_ARGS__) LBM_FSLICE(j + 1, __VA_ARGS__) LBM_FSLICE(j + 2, __VA_ARGS__) LBM_FSLICE(j + 3, __VA_ARGS__)
#define LBM_FAST_HALF_STEP(cur, pd, prev, next, st_pv, ks_pv, st_qk, h_qk, st_vn, ks_vn, hook)     \
  {                                                                                              \
    bf16x8 va[2], ka[4];                                                                         \
    float e[32];                                                                                 \
    __builtin_amdgcn_sched_barrier(0);                                                           \
    LBM_F4(0, cur, pd, prev, next, st_pv, ks_pv, st_qk, h_qk, st_vn, ks_vn, hook)                       \
    LBM_F4(4, cur, pd, prev, next, st_pv, ks_pv, st_qk, h_qk, st_vn, ks_vn, hook)                       \
    LBM_F4(8, cur, pd, prev, next, st_pv, ks_pv, st_qk, h_qk, st_vn, ks_vn, hook)                       \
    LBM_F4(12, cur, pd, prev, next, st_pv, ks_pv, st_qk, h_qk, st_vn, ks_vn, hook)                      \
    LBM_F4(16, cur, pd, prev, next, st_pv, ks_pv, st_qk, h_qk, st_vn, ks_vn, hook)                      \
  }
  f32x16 zero16;
#pragma unroll
  for (int i = 0; i < 16; ++i) zero16[i] = 0.f;

  // Iterations [0, n_fast) of this split see only complete 32-token halves (their own second
  // half and the first half of the tile after them) and take the half-step without reference;
  // the iterations around the ragged end of the KV list take the one with the masking k-step.
  const int n_fast = min(max((kv_tokens - 96) / kKvTile - t0 + (kv_tokens >= 96 ? 1 : 0), 0), n);

  // Two passes at most.  The first one uses no softmax reference at all: the numerators are
  // 2^score, which is exact softmax arithmetic as long as nothing leaves the range of fp32 /
  // bf16 (both carry 8 exponent bits and the relative precision does not depend on the
  // magnitude).  Scores in log2 units beyond about +-100 - unheard of behind a q/k LayerNorm -
  // make a row sum or an output overflow or vanish; the check after the pass sees that and the
  // whole workgroup repeats its split with a reference that follows the row maxima (pass 1).
  {
    constexpr bool safe = SAFE;
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
#pragma unroll
      for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[qb][db][i] = 0.f;
      lacc[qb] = f32x4{0.f, 0.f, 0.f, 0.f};
      m_run[qb] = 0.f;
      qaug_bits[qb][0] = 0u;
    }

    // ---- prologue: K(0), K(1), V(0) are on their way into the ring; the V stage the first PV
    // reads is zeroed
#pragma unroll
    for (int k = 0; k < kPieces; ++k)
      *(u32x4*)&ring_v[2][(k * kRowWaves * 64 + (PAIR ? tid % (kRowWaves * 64) : tid)) * 8] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int qb = 0; qb < 2; ++qb)
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) pB[qb][kk] = __builtin_bit_cast(bf16x8, u32x4{0u, 0u, 0u, 0u});
    LBM_DMA_LANDED();
    __syncthreads();
    qk_half(0, 0, kv_tokens - t0 * kKvTile, sA);
    if (safe) {
      // the reference starts kHeadroom above the maxima of the first half
      float mx[2];
      row_max(sA, mx);
#pragma unroll
      for (int qb = 0; qb < 2; ++qb) {
        const float d = move_reference(qb, mx[qb] + kHeadroom);
#pragma unroll
        for (int i = 0; i < 16; ++i) sA[qb][i] -= d;
      }
    }
    vnext[0] = v_frag(2, 2, 0);
    vnext[1] = v_frag(2, 2, 1);

    int st_k = 0, st_v = 0, st_vm1 = 2;  // stages of K(i), V(i), V(i-1)
    // Common frame of one tile iteration.  The loads of K(i+2) and V(i+1) into their ring
    // stages (free since the barrier that ended iteration i-1) and the fetch of the next row
    // entry are issued from inside the first half-step's slices (LBM_STAGING_HOOK), not in front
    // of it: after the barrier every wavefront goes straight to matrix instructions whose
    // operands it already holds, and the address arithmetic of the staging shares slices with
    // them instead of leaving the matrix pipe idle on all four SIMDs at once.  The loads have
    // the rest of the iteration to land; the wait for them sits right before the barrier that
    // ends it.  Past the last tile the data lands in stages nobody reads any more.  The row
    // entry fetched for K now serves V in the next iteration.
#define LBM_NO_HOOK(j)
#define LBM_STAGING_HOOK(j)                                                          \
    if ((j) == 1) dma(ek, pool_k, own_k, ring_k[st_k2]);                              \
    if ((j) == 2) dma(ev, pool_v, own_v, ring_v[st_v1]);                              \
    if ((j) == 3) {                                                                  \
      ev = ek;                                                                       \
      ek = row_entry(t + 3);                                                         \
    }
#define LBM_TILE_ITERATION(PRE, HALF0, HALF1)                                        \
    {                                                                                \
      const int t = t0 + i;                                                          \
      int st_k1 = st_k + 1; if (st_k1 >= kStages) st_k1 -= kStages;                  \
      int st_k2 = st_k1 + 1; if (st_k2 >= kStages) st_k2 -= kStages;                 \
      int st_v1 = st_v + 1; if (st_v1 >= kStages) st_v1 -= kStages;                  \
      PRE                                                                            \
      HALF0                                                                          \
      HALF1                                                                          \
      LBM_DMA_LANDED();                                                              \
      __syncthreads();                                                               \
      st_k = st_k1;                                                                  \
      st_vm1 = st_v;                                                                 \
      st_v = st_v1;                                                                  \
    }
    // The same frame with the ring stages as compile-time constants (the ring has three stages,
    // so three iterations bring it back to where it started): every LDS address of the
    // iteration is then one per-lane register plus an immediate offset, and the thirty-odd vector
    // and scalar instructions per tile that add a run-time stage base to it are gone.
#define LBM_TILE_ITERATION_AT(U, SK, HALF0, HALF1)                                   \
    {                                                                                \
      const int t = t0 + i + (U);                                                    \
      constexpr int st_k = (SK), st_v = (SK), st_vm1 = ((SK) + 2) % kStages;          \
      constexpr int st_k1 = ((SK) + 1) % kStages, st_k2 = ((SK) + 2) % kStages;       \
      constexpr int st_v1 = ((SK) + 1) % kStages;                                    \
      HALF0                                                                          \
      HALF1                                                                          \
      LBM_DMA_LANDED();                                                              \
      __syncthreads();                                                               \
    }
    int i = 0;
    // A wavefront whose 64 rows lie past the stream's last query row (an odd frame size in 512-row
    // tiles) only keeps the ring going for the others: its SIMD's time, and its power, go to the
    // wavefront it shares the SIMD with.
    if (q_row0 >= sp.q_rows) {
      for (; i < n; ++i)
        LBM_TILE_ITERATION(, dma(ek, pool_k, own_k, ring_k[st_k2]); dma(ev, pool_v, own_v, ring_v[st_v1]); ev = ek; ek = row_entry(t + 3);, )
    }
    // half 0 of tile i: softmax(sA) -> pA | PV(tile i-1, half 1) with pB | QK(tile i, half 1) -> sB
    // half 1 of tile i: softmax(sB) -> pB | PV(tile i, half 0) with pA | QK(tile i+1, half 0) -> sA
    const int n_f = safe ? 0 : n_fast;
#define LBM_FAST_ITERATION_AT(U, SK)                                                              \
      LBM_TILE_ITERATION_AT(U, SK,                                                                 \
        LBM_FAST_HALF_STEP(sA, pA, pB, sB, st_vm1, 3, st_k, 1, st_v, 0, LBM_STAGING_HOOK);,        \
        LBM_FAST_HALF_STEP(sB, pB, pA, sA, st_v, 1, st_k1, 0, st_v, 2, LBM_NO_HOOK);)
    for (; i + kStages <= n_f; i += kStages) {   // (entered with st_k = st_v = 0, st_vm1 = 2, and left so)
      LBM_FAST_ITERATION_AT(0, 0)
      LBM_FAST_ITERATION_AT(1, 1)
      LBM_FAST_ITERATION_AT(2, 2)
    }
#undef LBM_FAST_ITERATION_AT
#undef LBM_TILE_ITERATION_AT
    for (; i < n_f; ++i)
      LBM_TILE_ITERATION(
        ,
        LBM_FAST_HALF_STEP(sA, pA, pB, sB, st_vm1, 3, st_k, 1, st_v, 0, LBM_STAGING_HOOK);,
        LBM_FAST_HALF_STEP(sB, pB, pA, sA, st_v, 1, st_k1, 0, st_v, 2, LBM_NO_HOOK);
      )
    for (; i < n; ++i)
      LBM_TILE_ITERATION(
        const int n_valid = kv_tokens - t * kKvTile;
        bool hot;,
        LBM_HALF_STEP(sA, pA, pB, sB, st_vm1, 3, st_k, 1, n_valid, st_v, 0, hot, LBM_STAGING_HOOK);
        if (safe && __builtin_amdgcn_ballot_w64(hot)) raise_reference(sA, pA, sB);,
        /* after the last tile this QK reads a stale stage; its result is unused */
        LBM_HALF_STEP(sB, pB, pA, sA, st_v, 1, st_k1, 0, n_valid - kKvTile, st_v, 2, hot, LBM_NO_HOOK);
        if (safe && __builtin_amdgcn_ballot_w64(hot)) raise_reference(sB, pB, sA);
      )
#undef LBM_TILE_ITERATION
#undef LBM_STAGING_HOOK
#undef LBM_NO_HOOK
    for (; PAIR && i < n_most; ++i) __syncthreads();   // (the other group's last tiles)
    // PV and row sums of the last half: pB with half 1 of V(n-1), first k-step already in vnext
    {
      pv_step(vnext, pB, 0);
      bf16x8 va[2] = {v_frag(st_vm1, 3, 0), v_frag(st_vm1, 3, 1)};
      pv_step(va, pB, 1);
#pragma unroll
      for (int qb = 0; qb < 2; ++qb)
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
          lacc[qb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lsel, pB[qb][kk], lacc[qb], 0, 0, 0);
    }
    // Did the pass without reference stay in range?  Compared as integers (non-negative floats
    // order like their bit patterns; NaN, infinity and negative values land above every bound).
    bool bad = false;
    if (!safe && n > 0 && q_row0 < sp.q_rows) {
      unsigned top = 0u;
#pragma unroll
      for (int qb = 0; qb < 2; ++qb)
#pragma unroll
        for (int db = 0; db < 2; ++db)
#pragma unroll
          for (int i = 0; i < 16; ++i) top = max(top, float_bits(o[qb][db][i]) & 0x7FFFFFFFu);
      bad = top >= 0x7F800000u;
      if (lane < 16) {
#pragma unroll
        for (int qb = 0; qb < 2; ++qb)
#pragma unroll
          for (int h2 = 0; h2 < 2; ++h2) {
            const unsigned lb = float_bits(lacc[qb][h2]);
            bad = bad || lb < 0x12800000u /* 2^-90 */ || lb > 0x71800000u /* 2^100 */;
          }
      }
    }
    if (!safe && __builtin_amdgcn_readfirstlane(__syncthreads_or(bad))) {
      if (PAIR) lbm_attn_pair_safe(a, sp);
      else lbm_attn_split_safe(a, sp);
      __builtin_amdgcn_endpgm();
    }
  }
#undef LBM_FAST_HALF_STEP
#undef LBM_F4
#undef LBM_FSLICE
#undef LBM_HALF_STEP
#undef LBM_S4
#undef LBM_SLICE

  // ---- epilogue.  The accumulators hold O^T (a lane owns 4-element runs of 32 different
  // rows); written straight out that is 32 scattered 8-byte stores per instruction.  Each
  // wavefront instead transposes its rows through its Q patch (idle since the prologue) and
  // stores whole 128-byte rows, eight lanes per row.
  unsigned short* const stage = patch;
  const bool direct = PAIR || sp.n_splits == 1;
  unsigned short* dst = direct ? a.out : a.part_o;
  const size_t dst_row0 = direct ? (size_t)sp.q_begin : (size_t)sp.part_begin + (size_t)split * sp.q_rows;
  if (PAIR) {
    // A wavefront leaves one block of 32 rows of its partial result to the other group's wavefront of the same rows and
    // merges the other block: group 0 the first, group 1 the second.  Both partial results as lbm_attn_combine_bf16_kernel
    // finds them - normalised, bf16 - and its sums, in the order of the splits.  A lane reads what the same lane of the
    // other wavefront wrote.
    float lse[2], inv[2];
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
      const float sum_lo = lacc[qb][0], sum_hi = lacc[qb][1];
      const float l_lo = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(4 * (lane & 15), __builtin_bit_cast(int, sum_lo)));
      const float l_hi = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(4 * (lane & 15), __builtin_bit_cast(int, sum_hi)));
      const float l_tot = (n32 & 16) ? l_hi : l_lo;
      inv[qb] = l_tot > 0.f ? 1.0f / l_tot : 0.f;
      lse[qb] = m_run[qb] + __builtin_amdgcn_logf(l_tot);
    }
    auto partial = [&](int qb, int db, int c4) -> bf16x4 {
      f32x4 w;
#pragma unroll
      for (int e = 0; e < 4; ++e) w[e] = o[qb][db][c4 * 4 + e] * inv[qb];
      return __builtin_convertvector(w, bf16x4);
    };
    auto at = [&](int qb, int db, int c4) { return (bf16x4*)&stage[(qb * 32 + n32) * kKStride + db * 32 + c4 * 8 + g * 4]; };
    auto leave = [&](auto block) {
      constexpr int others = decltype(block)::value;
#pragma unroll
      for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int c4 = 0; c4 < 4; ++c4) *at(others, db, c4) = partial(others, db, c4);
      if (g == 0) lds_pair_lse[wave][n32] = lse[others];
    };
    auto merge = [&](auto block) {
      constexpr int mine = decltype(block)::value;   // (and the split that this wavefront summed)
      const float theirs = lds_pair_lse[wave ^ kRowWaves][n32];
      const float first = mine == 0 ? lse[mine] : theirs, second = mine == 0 ? theirs : lse[mine];
      float mx = fmaxf(first, second);
      if (mx == -INFINITY) mx = 0.f;
      const float w0 = __builtin_amdgcn_exp2f(first - mx), w1 = __builtin_amdgcn_exp2f(second - mx), wsum = w0 + w1;
      const float norm = wsum > 0.f ? 1.0f / wsum : 0.f;
#pragma unroll
      for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int c4 = 0; c4 < 4; ++c4) {
          const f32x4 x = __builtin_convertvector(partial(mine, db, c4), f32x4), y = __builtin_convertvector(*at(mine, db, c4), f32x4);
          f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            acc[e] += w0 * (mine == 0 ? x[e] : y[e]);
            acc[e] += w1 * (mine == 0 ? y[e] : x[e]);
            acc[e] *= norm;
          }
          *at(mine, db, c4) = __builtin_convertvector(acc, bf16x4);
        }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int row = mine * 32 + k * 8 + (lane >> 3);
        const u32x4 v = *(const u32x4*)&stage[row * kKStride + (lane & 7) * 8];
        const int r = q_row0 + row;
        if (r < sp.q_rows) lbm_store_through(dst + ((dst_row0 + r) * H + head) * 64 + (lane & 7) * 8, v);
      }
    };
    if (group == 0) leave(std::integral_constant<int, 1>{});
    else leave(std::integral_constant<int, 0>{});
    __syncthreads();
    if (group == 0) merge(std::integral_constant<int, 0>{});
    else merge(std::integral_constant<int, 1>{});
    return;
  }
#pragma unroll
  for (int qb = 0; qb < 2; ++qb) {
    // the row sum of query n32 of this block sits in lane n32 % 16, element n32 / 16
    // (both elements by value first, see float_bits)
    const float sum_lo = lacc[qb][0], sum_hi = lacc[qb][1];
    const float l_lo = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(4 * (lane & 15), __builtin_bit_cast(int, sum_lo)));
    const float l_hi = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(4 * (lane & 15), __builtin_bit_cast(int, sum_hi)));
    const float l_tot = (n32 & 16) ? l_hi : l_lo;
    const float inv = l_tot > 0.f ? 1.0f / l_tot : 0.f;
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
      for (int c4 = 0; c4 < 4; ++c4) {
        f32x4 w;
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = o[qb][db][c4 * 4 + e] * inv;
        *(bf16x4*)&stage[n32 * kKStride + db * 32 + c4 * 8 + g * 4] = __builtin_convertvector(w, bf16x4);
      }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int row = k * 8 + (lane >> 3);
      const u32x4 v = *(const u32x4*)&stage[row * kKStride + (lane & 7) * 8];
      const int r = q_row0 + qb * 32 + row;
      if (r < sp.q_rows) lbm_store_through(dst + ((dst_row0 + r) * H + head) * 64 + (lane & 7) * 8, v);
    }
    const int r = q_row0 + qb * 32 + n32;
    if (!direct && g == 0 && r < sp.q_rows)
      a.part_lse[(dst_row0 + r) * H + head] = m_run[qb] + __builtin_amdgcn_logf(l_tot);
  }
}

__device__ __noinline__ void lbm_attn_split_safe(AttnCore a, LbmAttnStreamPlan sp) { lbm_attn_split<true, false>(a, sp); }
__device__ __noinline__ void lbm_attn_pair_safe(AttnCore a, LbmAttnStreamPlan sp) { lbm_attn_split<true, true>(a, sp); }

}  // namespace

template <int S>
__global__ __launch_bounds__(kThreads, 1) void lbm_attn_bf16_d64_kernel(AttnArgs<S> a) {
  LbmAttnStreamPlan sp = lbm_first_plan(a);
  if (__builtin_expect((int)blockIdx.x >= a.total_wgs || blockIdx.y, 0)) {
    if (blockIdx.y)
      lbm_touch(a.touch, kThreads, false);
    else
      lbm_append_pieces<kAppendPieces>(a.self_k, a.self_v, const_cast<unsigned short*>(a.pool), a.append_rows, a.append_tokens,
                                       a.num_heads * 8, a.page_size, (int)blockIdx.x - a.total_wgs, kThreads);
    return;
  }
  lbm_plan_of_workgroup(a, sp);
  lbm_attn_split<false, false>(a, sp);
}

template <int S>
__global__ __launch_bounds__(kThreads, 1) void lbm_attn_bf16_d64_own_kernel(AttnArgs<S> a) {
  LbmAttnStreamPlan sp = lbm_first_plan(a);
  lbm_plan_of_workgroup(a, sp);
  lbm_attn_split<false, false, true>(a, sp);
}

// (its sch: n_qtiles and workgroups in tiles of 256 query rows, see the launch)
template <int S>
__global__ __launch_bounds__(kThreads, 1) void lbm_attn_bf16_d64_pair_kernel(AttnArgs<S> a) {
  LbmAttnStreamPlan sp = lbm_first_plan(a);
  lbm_plan_of_workgroup(a, sp);
  lbm_attn_split<false, true>(a, sp);
}

// ---------------------------------------------------------------------------- bf16, short KV
// Streams with at most kSmMaxKv KV tokens - the frame blocks' attention of a frame over itself
// (lingbot_map/layers/block.py:27-101: 1004 x 1004 tokens), the first frames of a stream - have
// too few KV tiles to amortise the split-KV machinery above (a workgroup per (512 rows, head,
// split) with a prologue of several tile-times, partial results through HBM and a second
// kernel).  Here one 8-wave workgroup owns 64 or 32 query rows of one head and the KV axis is split
// INSIDE it: wavefront w walks its own eighth of the KV axis in 32-token pieces with its own
// K/V ring in LDS (rows travel global -> LDS as whole 128-byte lines, two pieces ahead of the
// multiply), two wavefronts per SIMD covering each other's waits, and the eight partial
// results are summed through LDS at the end.  No workspace, no second kernel.  Same arithmetic
// as the main kernel's first pass: scores straight into exp2 without a reference, a range
// check at the end, and - only if that fails - a second pass with the textbook running-maximum
// recurrence.
namespace {
constexpr int kSmWaves = 8;
constexpr int kSmThreads = kSmWaves * 64;
// KV tokens up to which the kernel is a candidate.  Beyond them every workgroup would read a KV list that its
// XCD's L2 no longer holds for its neighbours (485 rows x 5,820 tokens: 38 us against 29 on the pair).
constexpr int kSmMaxKv = 4096;
constexpr int kSmMaxCacheKv = 4864;   // the same for one stream that attends to more than its own rows (lbm_attn_schedule)
constexpr int kSmPiece = 32;     // KV tokens per step of a wavefront
// KV tokens of a launch's longest stream beyond which the launch's workgroups begin at different pieces, those of its shorter
// streams too (lbm_attn_bf16_d64_small_kernel's TURN): 261 rows over 1,305 tokens 9.9 us in order, 10.1 so; 86 over 1,500
// 13.3, 11.6; 300 over 900 and 2,100 17.3, 16.7.  The shorter streams of such a launch in order instead (16 heads, K/V in
// HBM, all streams | the long ones only): 261 rows over 783 and 2,088 15.8 | 16.5, over 900 and 2,100 16.7 | 17.5, 330 over
// three times 990 and 1,980 24.5 | 25.4, but 201 over 804, 1,005 and 1,608 15.9 | 15.6, 261 over 261, 522, 1,305 and 2,349
// 20.2 | 19.7, 389 over 1,167 and 1,945 17.0 | 16.8.
constexpr int kSmTurnKv = 1408;
constexpr int kSmOStride = 68;   // floats per row of a partial output parked in LDS (4-bank shift per row)
constexpr int kSmPieceBytes = kSmPiece * 64 * 2;                                 // K (or V) rows of a piece, unpadded
constexpr int kSmOffLists = kSmWaves * 2 * 2 * kSmPieceBytes;                    // behind two stages of K and V per wavefront
constexpr int kSmListBytes = 256 + 2 * kSmPiece * 8;                             // a wavefront's row entries, and the K and V addresses they name
constexpr int kSmOffQ = kSmOffLists + kSmWaves * kSmListBytes;                   // Q on its way to the fragments
constexpr int lbm_sm_lds_bytes(int rows) {
  const int merge = kSmWaves * (rows * kSmOStride + 2 * rows) * 4, loop = kSmOffQ + rows * kKStride * 2;
  return merge > loop ? merge : loop;
}
static_assert(lbm_sm_lds_bytes(64) <= 160 * 1024, "LDS budget of the short-KV kernel");
}  // namespace

// QB: 32-row blocks of query rows per workgroup.  TURN: workgroups may begin at different pieces (an
// instance of its own: what it adds in front of the first load takes 0.2 us, 3 % of a launch on 261 own rows).
// OWN: token t of a stream is row kv_row_begin + t of the caller's K/V (LBM_ATTN_OWN_ROWS): the rows are asked for
// at once, without the trip to memory for their table entries and the one through LDS for their addresses (261
// rows 5.5 -> 5.2 us, 1,004 rows 11.4 -> 10.6, 2,000 rows 29.4 -> 26.3).
template <int S, int QB, bool TURN, bool OWN = false>
__global__ __launch_bounds__(kSmThreads, 1) void lbm_attn_bf16_d64_small_kernel(AttnArgs<S> a) {
  __shared__ __attribute__((aligned(16))) unsigned char lds_raw[lbm_sm_lds_bytes(32 * QB)];
  constexpr int kRows = 32 * QB;
  // (the wavefront index is uniform by construction; said so, or the loop over this wavefront's
  // pieces is compiled as divergent control flow)
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n32 = lane & 31, g = lane >> 5;
  // ---- which (stream, 64 query rows, head)
  LbmAttnStreamPlan sp = lbm_first_plan(a);
  if (__builtin_expect((int)blockIdx.x >= a.total_wgs || blockIdx.y, 0)) {
    if (blockIdx.y)
      lbm_touch(a.touch, kSmThreads, false);
    else
      lbm_append_pieces(a.self_k, a.self_v, const_cast<unsigned short*>(a.pool), a.append_rows, a.append_tokens, a.num_heads * 8, a.page_size,
                        (int)blockIdx.x - a.total_wgs, kSmThreads);
    return;
  }
  lbm_plan_of_workgroup(a, sp);
  const int H = a.num_heads;
  const int local = (int)blockIdx.x - sp.wg_begin;
  int q_tile, head;
  if ((H & 7) == 0) {   // the query blocks of one head on one XCD (blockIdx mod 8): its L2 serves their K/V
    const int x = local & 7, i = local >> 3;
    q_tile = lbm_divide(i, H >> 3, a.per_eighth, head);
    head = head * 8 + x;
  } else {
    q_tile = lbm_divide(local, H, a.per_heads, head);
  }
  if (q_tile >= sp.n_qtiles) return;   // padding between streams (whole workgroups)
  const int kv_tokens = max(a.live_kv_tokens ? a.live_kv_tokens[sp.live_at] : sp.kv_tokens, 0);
  const int n_pieces = (kv_tokens + kSmPiece - 1) / kSmPiece;
  const int pps = (n_pieces + kSmWaves - 1) / kSmWaves;
  const int p0 = wave * pps, p1 = min(p0 + pps, n_pieces);   // this wavefront's pieces (possibly none)
  // Where in its pieces it begins (TURN: the launch's longest stream decided that).  Over a cache the workgroups of a head, which start together, each begin at
  // another place and go round: all at the same one, they would ask HBM for the same two pieces per wavefront,
  // a quarter of what it takes to keep it busy, and wait for them together.  A ragged last piece stays the last
  // (it is masked there).  Attention to a stream's own rows, just written, keeps the order: an encoder's
  // results stay what they are.
  // (24 blocks with pools of their own, us per block: 261 rows over 2,349 tokens 16.3 -> 14.1, 600 over 3,600 25.3 ->
  // 23.6; 261 over 4,000 tokens, pools rotating through 600 MB, 25.1 -> 19.3.)
  int go_round = 0, turn = 0;
  if (TURN && pps > 2 && kv_tokens != sp.q_rows) {
    go_round = max(p1 - p0 - (p1 == n_pieces && kv_tokens % kSmPiece != 0 ? 1 : 0), 0);
    turn = min(__builtin_amdgcn_readfirstlane((int)((float)(q_tile * go_round) * __builtin_amdgcn_rcpf((float)sp.n_qtiles))), go_round);
  }
  auto piece = [&](int i) { return !TURN ? p0 + i : p0 + i + (i + turn < go_round ? turn : (i < go_round ? turn - go_round : 0)); };   // the i-th it takes
  const unsigned row_bytes = (unsigned)H * 128u;
  const int q_row0 = q_tile * kRows;
  if (n_pieces == 0) {
    // nothing visible: the reference returns zeros (lingbot_map/layers/flashinfer_cache.py:368-370).
    // Decided before the first load, so that every load below is unconditional.
    const int r = q_row0 + (tid >> 3);
    if (tid < kRows * 8 && r < sp.q_rows)
      *(u32x4*)(a.out + ((size_t)(sp.q_begin + r) * H + head) * 64 + (tid & 7) * 8) = u32x4{0u, 0u, 0u, 0u};
    return;
  }

  // ---- K/V rows of a piece travel global -> LDS directly (as in the main kernel: 1 KiB, eight rows, per
  // load; chunk c of K row r at c ^ ((r >> 1) & 7), of V row r at c ^ 4 ((r >> 1) & 1)) into one of
  // two stages of this wavefront's own, two pieces ahead of the multiply, their row entries three:
  // with one piece in registers, its entries and its rows one behind the other inside a step, a
  // step took two trips to memory, 1.1-1.35 us.
  unsigned char* ring = lds_raw + wave * (4 * kSmPieceBytes);        // [stage][K | V]
  int* entries = (int*)(lds_raw + kSmOffLists + wave * kSmListBytes);
  unsigned long long* sources = (unsigned long long*)(entries + 64); // [K | V][row of the piece]
  auto lds_at = [](const void* p) { return __builtin_amdgcn_readfirstlane((unsigned)(size_t)(__attribute__((address_space(3))) const void*)p); };
  const unsigned m0_ring = lds_at(ring), m0_entries = lds_at(entries);
  // lanes 0-31 work out where the piece's K rows are, lanes 32-63 where its V rows are
  const char* pool_rows = (const char*)(a.pool + (size_t)head * 64) + (g ? (size_t)a.page_size * row_bytes : 0);
  const char* own_rows = (const char*)((g ? a.self_v : a.self_k) + (size_t)head * 64);
  const int32_t* rows = a.kv_rows + sp.kv_row_begin;
  const int last_token = max(kv_tokens - 1, 0);
  const unsigned chunk_k[2] = {(unsigned)(((lane & 7) ^ (lane >> 4)) * 16), (unsigned)(((lane & 7) ^ (4 | (lane >> 4))) * 16)};
  const unsigned chunk_v = (unsigned)(((lane & 7) ^ (((lane >> 4) & 1) * 4)) * 16);
  // (tokens past the last re-read it: finite data, masked below)
  auto load_entries = [&](int i) {   // of the i-th piece (lanes 0-31) and the next
    const int pa = piece(i), pb = piece(i + 1);
    const int32_t* src = rows + min(TURN ? (g ? pb : pa) * kSmPiece + n32 : pa * kSmPiece + lane, last_token);
    asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dword %0, off" : : "v"(src), "s"(m0_entries) : "memory", "m0");
  };
  auto find_rows = [&](int e) {   // negative entries name rows of the caller's own K/V
    sources[lane] = (unsigned long long)((e < 0 ? own_rows : pool_rows) + (unsigned long long)(unsigned)(e ^ (e >> 31)) * row_bytes);
  };
  auto load_own_rows = [&](int pc, int stage) {
    const char* k = (const char*)(a.self_k + (size_t)head * 64) + (size_t)sp.kv_row_begin * row_bytes;
    const char* v = (const char*)(a.self_v + (size_t)head * 64) + (size_t)sp.kv_row_begin * row_bytes;
#pragma unroll
    for (int j = 0; j < 8; ++j) {   // K rows in j = 0..3, V rows in 4..7; tokens past the last re-read it
      const unsigned at = (unsigned)min(pc * kSmPiece + (j & 3) * 8 + (lane >> 3), last_token) * row_bytes + (j < 4 ? chunk_k[j & 1] : chunk_v);
      asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(at), "s"(j < 4 ? k : v), "s"(m0_ring + (unsigned)(stage * 2 * kSmPieceBytes + j * 1024)) : "memory", "m0");
    }
  };
  auto load_rows = [&](int stage) {
    unsigned long long at[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) at[j] = sources[j * 8 + (lane >> 3)];   // K rows in j = 0..3, V rows in 4..7
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const unsigned long long src = at[j] + (j < 4 ? chunk_k[j & 1] : chunk_v);
      asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(src), "s"(m0_ring + (unsigned)(stage * 2 * kSmPieceBytes + j * 1024)) : "memory", "m0");
    }
  };
  // pieces p0 and p0 + 1, as far as there are such, and the entries of the one after them on their way
  auto start = [&]() {
    if (OWN) {
      load_own_rows(p0, 0);
      if (p0 + 1 < p1) load_own_rows(p0 + 1, 1);
      return;
    }
    load_entries(0);
    LBM_LOADS_LEFT(0);
    const int e0 = entries[n32], e1 = entries[kSmPiece + n32];
    find_rows(e0);
    LBM_LDS_DONE();
    load_rows(0);
    if (p0 + 1 < p1) {
      find_rows(e1);
      LBM_LDS_DONE();
      load_entries(2);
      load_rows(1);
    }
  };
  const int q_r = max(min(q_row0 + (tid >> 3), sp.q_rows - 1), 0);   // rows past the last one re-read it (never stored)
  u32x4 q_raw = {};
  if (!OWN) q_raw = *(const u32x4*)(a.q + ((size_t)(sp.q_begin + q_r) * H + head) * 64 + (tid & 7) * 8);

  // ---- Q: the workgroup reads its rows once as whole rows, every wavefront picks its fragments up
  // from LDS; scale * log2(e) folded in (as in the main kernel)
  bf16x8 qf[QB][4];
  {
    unsigned short* patch_q = (unsigned short*)(lds_raw + kSmOffQ);
    if (OWN) {
      // Q travels to LDS directly as well, in front of K and V and unpadded (chunk c of row r at c ^ ((r >> 1) & 7)): a load
      // that the compiler sees would make it wait for everything behind
      if (QB == 2 || wave < 4) {
        const unsigned short* src = a.q + ((size_t)(sp.q_begin + q_r) * H + head) * 64 + ((tid & 7) ^ ((tid >> 4) & 7)) * 8;
        asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(src), "s"(lds_at(patch_q) + (unsigned)wave * 1024u) : "memory", "m0");
      }
      if (p0 < p1) start();
      if (p0 + 1 < p1) LBM_LOADS_LEFT(16);
      else if (p0 < p1) LBM_LOADS_LEFT(8);
      else LBM_LOADS_LEFT(0);
    } else {
      if (QB == 2 || tid < kRows * 8) *(u32x4*)&patch_q[(tid >> 3) * kKStride + (tid & 7) * 8] = q_raw;
      if (p0 < p1) start();
    }
    __syncthreads();
#pragma unroll
    for (int qb = 0; qb < QB; ++qb)
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        const bf16x8 rawf = __builtin_bit_cast(bf16x8, *(const u32x4*)&patch_q[
            OWN ? (qb * 32 + n32) * 64 + ((ks * 2 + g) ^ ((n32 >> 1) & 7)) * 8 : (qb * 32 + n32) * kKStride + ks * 16 + g * 8]);
        f32x8 f = __builtin_convertvector(rawf, f32x8);
#pragma unroll
        for (int j = 0; j < 8; ++j) f[j] *= a.scale_log2;
        qf[qb][ks] = __builtin_convertvector(f, bf16x8);
      }
  }

  auto v_frag = [&](const unsigned short* v, int ks, int db) -> bf16x8 {   // as in the main kernel, on this wave's ring
    const int row = ks * 16 + 4 * g + ((lane & 15) >> 2);
    const int col = (db * 32 + ((lane >> 4) & 1) * 16 + (lane & 3) * 4) ^ (((lane >> 3) & 1) * 32);
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)&v[row * 64 + col]);
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)&v[(row + 8) * 64 + col]);
    s16x8 both;
    both[0] = lo[0]; both[1] = lo[1]; both[2] = lo[2]; both[3] = lo[3];
    both[4] = hi[0]; both[5] = hi[1]; both[6] = hi[2]; both[7] = hi[3];
    return __builtin_bit_cast(bf16x8, both);
  };

  f32x16 o[QB][2];
  f32x4 lacc[QB];                // first pass: row sums on the matrix pipe (layout as in the main kernel)
  float m_run[QB], l_lane[QB];    // second pass: running maximum of the row, this lane's share of its sum
  const unsigned sel_word = (lane == 0 || lane == 32 || lane == 17 || lane == 49) ? 0x3F803F80u : 0u;
  const bf16x8 lsel = __builtin_bit_cast(bf16x8, u32x4{sel_word, sel_word, sel_word, sel_word});
  f32x16 zero16;
#pragma unroll
  for (int i = 0; i < 16; ++i) zero16[i] = 0.f;

  // One pass over this wavefront's pieces.  SAFE is a type, not a variable: with a branch per block of
  // scores the exponentials of one query block could not share the issue slots with the MFMAs of
  // the other.
  auto walk = [&](auto SAFE) {
    constexpr bool kSafe = decltype(SAFE)::value;
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
#pragma unroll
      for (int db = 0; db < 2; ++db) o[qb][db] = zero16;
      lacc[qb] = f32x4{0.f, 0.f, 0.f, 0.f};
      m_run[qb] = kSafe ? -INFINITY : 0.f;
      l_lane[qb] = 0.f;
    }
    if (p0 >= p1) return;
    bf16x8 ka[4];   // K fragments of the piece about to be multiplied
    auto read_k = [&](int stage) {
      const unsigned short* k = (const unsigned short*)(ring + stage * 2 * kSmPieceBytes);
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
        ka[ks] = __builtin_bit_cast(bf16x8, *(const u32x4*)&k[n32 * 64 + ((ks * 2 + g) ^ ((n32 >> 1) & 7)) * 8]);
    };
    // AHEAD: 2 - the piece two ahead is asked for, 1 - the next piece is the last, 0 - this one is
    auto step = [&](int at, auto AHEAD) {
      constexpr int kAhead = decltype(AHEAD)::value;
      const int stage = at & 1;
      const unsigned short* ring_v = (const unsigned short*)(ring + stage * 2 * kSmPieceBytes + kSmPieceBytes);
      // S^T = K Q^T for the piece's 32 kv rows: sc[qb][i] is kv = 8 (i / 4) + 4 g + i % 4, q = 32 qb + n32
      f32x16 sc[QB];
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) sc[qb] = zero16;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) sc[qb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka[ks], qf[qb][ks], sc[qb], 0, 0, 0);
      bf16x8 va[2][2];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int db = 0; db < 2; ++db) va[ks][db] = v_frag(ring_v, ks, db);
      if (kAhead == 0) {   // (the stream's ragged last piece is some wavefront's last piece)
        const int n_valid = kv_tokens - piece(at) * kSmPiece;
#pragma unroll
        for (int qb = 0; qb < QB; ++qb)
#pragma unroll
          for (int i = 0; i < 16; ++i)
            if (8 * (i >> 2) + 4 * g + (i & 3) >= n_valid) sc[qb][i] = -INFINITY;
      }
      bf16x8 p[QB][2];
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        if (kSafe) {
          float mx = max3(sc[qb][0], sc[qb][1], sc[qb][2]);
#pragma unroll
          for (int i = 3; i < 15; i += 2) mx = max3(mx, sc[qb][i], sc[qb][i + 1]);
          mx = swap_max(max2(mx, sc[qb][15]));
          const float m_new = max2(m_run[qb], mx);     // finite: the first row of a piece is a token
          const float alpha = __builtin_amdgcn_exp2f(m_run[qb] - m_new);   // 0 on the first piece
          m_run[qb] = m_new;
          l_lane[qb] *= alpha;
#pragma unroll
          for (int db = 0; db < 2; ++db)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[qb][db][i] *= alpha;
#pragma unroll
          for (int i = 0; i < 16; ++i) sc[qb][i] -= m_new;
        }
#pragma unroll
        for (int kk2 = 0; kk2 < 2; ++kk2) {
          f32x8 e;
#pragma unroll
          for (int j = 0; j < 8; ++j) e[j] = __builtin_amdgcn_exp2f(sc[qb][kk2 * 8 + j]);
          p[qb][kk2] = __builtin_convertvector(e, bf16x8);
          if (kSafe) {
#pragma unroll
            for (int j = 0; j < 8; ++j) l_lane[qb] += e[j];
          } else {
            lacc[qb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lsel, p[qb][kk2], lacc[qb], 0, 0, 0);
          }
        }
      }
      if (kAhead > 0) {   // the next piece has landed: its K fragments travel under this one's last MFMAs
        LBM_LOADS_LEFT(0);
        if (kAhead == 2 && !OWN) find_rows(entries[n32]);
        read_k(stage ^ 1);
      }
      if (kAhead == 2) {  // both buffers of this stage are read: the piece two ahead may come
        LBM_LDS_DONE();
        if (OWN) {
          load_own_rows(p0 + at + 2, stage);
        } else {
          load_entries(at + 3);
          load_rows(stage);
        }
      }
      // O^T += V^T P^T over the piece's two 16-row k-steps
#pragma unroll
      for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) {
          o[qb][db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va[0][db], p[qb][0], o[qb][db], 0, 0, 0);
          o[qb][db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va[1][db], p[qb][1], o[qb][db], 0, 0, 0);
        }
    };
    if (p0 + 1 < p1) LBM_LOADS_LEFT(8);
    else LBM_LOADS_LEFT(0);
    read_k(0);
    int at = 0;
    for (; at + 2 < p1 - p0; ++at) step(at, std::integral_constant<int, 2>());
    if (at + 1 < p1 - p0) step(at++, std::integral_constant<int, 1>());
    step(at, std::integral_constant<int, 0>());
  };
  walk(std::false_type());
  // range check of the pass without reference (integer compares, see the main kernel)
  bool bad = false;
  if (p0 < p1) {
    unsigned top = 0u;
#pragma unroll
    for (int qb = 0; qb < QB; ++qb)
#pragma unroll
      for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) top = max(top, float_bits(o[qb][db][i]) & 0x7FFFFFFFu);
    bad = top >= 0x7F800000u;
    if (lane < 16) {
#pragma unroll
      for (int qb = 0; qb < QB; ++qb)
#pragma unroll
        for (int h2 = 0; h2 < 2; ++h2) {
          const unsigned lb = float_bits(lacc[qb][h2]);
          bad = bad || lb < 0x12800000u /* 2^-90 */ || lb > 0x71800000u /* 2^100 */;
        }
    }
  }
  const bool safe = __syncthreads_or(bad);
  if (safe) {
    if (p0 < p1) start();
    walk(std::true_type());
  }

  // ---- merge the wavefronts' partial results through LDS (the rings are dead)
  LBM_LOADS_LEFT(0);
  __syncthreads();
  float* so = (float*)lds_raw + wave * (kRows * kSmOStride);
  float* sl = (float*)lds_raw + kSmWaves * (kRows * kSmOStride);   // [wave][64] row sums, then [wave][64] references
  float* sm = sl + kSmWaves * kRows;
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
      for (int c4 = 0; c4 < 4; ++c4)
        *(f32x4*)&so[(qb * 32 + n32) * kSmOStride + db * 32 + c4 * 8 + g * 4] =
            f32x4{o[qb][db][c4 * 4], o[qb][db][c4 * 4 + 1], o[qb][db][c4 * 4 + 2], o[qb][db][c4 * 4 + 3]};
    if (safe) {
      float lo, hi;
      swap_halves(l_lane[qb], lo, hi);
      if (g == 0) sl[wave * kRows + qb * 32 + n32] = lo + hi;
    } else if (lane < 16) {
      sl[wave * kRows + qb * 32 + lane] = lacc[qb][0];
      sl[wave * kRows + qb * 32 + 16 + lane] = lacc[qb][1];
    }
    if (g == 0) sm[wave * kRows + qb * 32 + n32] = (p0 < p1) ? m_run[qb] : -INFINITY;
  }
  __syncthreads();
  {
    // wavefront w finishes rows 4 QB w ...: 16 / QB lanes per row, 4 QB head dims each
    constexpr int kLanes = 16 / QB, kDims = 4 * QB;
    const int row = wave * (kRows / kSmWaves) + lane / kLanes, d0 = (lane % kLanes) * kDims;
    float mw[kSmWaves], mx = -INFINITY;
#pragma unroll
    for (int w = 0; w < kSmWaves; ++w) {
      mw[w] = sm[w * kRows + row];
      mx = max2(mx, mw[w]);
    }
    f32x4 acc[QB];
#pragma unroll
    for (int j = 0; j < QB; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    float l_tot = 0.f;
#pragma unroll
    for (int w = 0; w < kSmWaves; ++w) {
      // a wavefront without pieces (reference -inf) weighs nothing; with a common reference the weights are 1
      const float wgt = mw[w] > -INFINITY ? __builtin_amdgcn_exp2f(mw[w] - mx) : 0.f;
      l_tot += wgt * sl[w * kRows + row];
      const float* src = (const float*)lds_raw + w * (kRows * kSmOStride) + row * kSmOStride + d0;
#pragma unroll
      for (int j = 0; j < QB; ++j) acc[j] += *(const f32x4*)(src + 4 * j) * wgt;
    }
    const float inv = l_tot > 0.f ? 1.0f / l_tot : 0.f;   // nothing visible: zeros (flashinfer_cache.py:368-370)
    const int r = q_row0 + row;
    if (r < sp.q_rows) {
      unsigned short* dst = a.out + ((size_t)(sp.q_begin + r) * H + head) * 64 + d0;
      u32x2 y[QB];
#pragma unroll
      for (int j = 0; j < QB; ++j) y[j] = __builtin_bit_cast(u32x2, __builtin_convertvector(acc[j] * inv, bf16x4));
      if (QB == 2) lbm_store_through(dst, u32x4{y[0][0], y[0][1], y[QB - 1][0], y[QB - 1][1]});
      else lbm_store_through(dst, y[0]);
    }
  }
}

// Merge split-KV partial results: out = sum_s w_s * o_s with w_s = 2^(lse_s - max) / sum.
// One thread per (query row, head, 8 consecutive d).
//
// Up to NJ splits (n <= NJ): all 2 NJ loads - the log-sum-exps and the partial rows - are issued
// before the first use of any of them, one round trip of memory latency instead of three.  NJ is
// the next of 2, 4, 8, 16 above the split count, so that a launch with two splits (several streams'
// frame blocks) does not load its last split seven times over.  More than sixteen, few rows of few heads over a long list,
// go in batches of sixteen.  Bound by trips to memory there; us a launch, batches of 8 log-sum-exps and 4 rows from nine
// splits on, and these: 261 rows x 16 heads x 14 splits 5.6, 4.0; 261 x 8 x 26 8.0, 5.9; 520 x 4 x 30 8.5, 6.3; 65 x 1 x
// 64 13.9, 9.0.
template <int NJ>
__device__ __forceinline__ void lbm_combine_upto(const float* lse, const unsigned short* po, long long split_stride, int n,
                                                 float& wsum, f32x8& acc) {
  float t[NJ];
  bf16x8 v[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const long long s = min(j, n - 1);
    t[j] = lse[s * split_stride];
    v[j] = *(const bf16x8*)(po + s * split_stride * 64);
  }
  float mx = -INFINITY;
#pragma unroll
  for (int j = 0; j < NJ; ++j) mx = fmaxf(mx, t[j]);
  if (mx == -INFINITY) mx = 0.f;  // every split empty (no visible token): weights 0, output 0
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const float w = j < n ? __builtin_amdgcn_exp2f(t[j] - mx) : 0.f;
    const f32x8 vf = __builtin_convertvector(v[j], f32x8);
    wsum += w;
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] += w * vf[e];
  }
}

template <int S>
__global__ __launch_bounds__(256) void lbm_attn_combine_bf16_kernel(AttnArgs<S> a) {
  const LbmAttnStreamPlan sp = a.s[S == 1 ? 0 : blockIdx.y];
  asm volatile("" : : "s"(a.combine_blocks), "s"(a.num_heads), "s"(a.part_lse), "s"(a.part_o), "s"(a.out), "s"(sp.n_splits), "s"(sp.q_rows), "s"(sp.part_begin), "s"(sp.q_begin));   // (in one trip: lbm_first_plan)
  if ((int)blockIdx.x >= a.combine_blocks) {
    // The append's share of the launch (lbm_attn_run_append): the main kernel has read the pool,
    // the new frames' rows - attended to from the caller's tensors - now go into their pages.
    if (blockIdx.y == 0)
      lbm_append_pieces(a.self_k, a.self_v, const_cast<unsigned short*>(a.pool), a.append_rows, a.append_tokens, a.num_heads * 8, a.page_size,
                        (int)blockIdx.x - a.combine_blocks, 256);
    return;
  }
  if (sp.n_splits <= 1) return;
  const int H = a.num_heads;
  const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (long long)sp.q_rows * H * 8) return;
  const int d8 = (int)(idx & 7);
  const long long rh = idx >> 3;  // r * H + h
  const long long split_stride = (long long)sp.q_rows * H;
  const float* lse = a.part_lse + (long long)sp.part_begin * H + rh;
  const int n = sp.n_splits;
  const unsigned short* po = a.part_o + ((long long)sp.part_begin * H + rh) * 64 + d8 * 8;
  float wsum = 0.f;
  f32x8 acc;
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = 0.f;
  if (n <= 2) {
    lbm_combine_upto<2>(lse, po, split_stride, n, wsum, acc);
  } else if (n <= 4) {
    lbm_combine_upto<4>(lse, po, split_stride, n, wsum, acc);
  } else if (n <= 8) {
    lbm_combine_upto<8>(lse, po, split_stride, n, wsum, acc);
  } else if (n <= 16) {
    lbm_combine_upto<16>(lse, po, split_stride, n, wsum, acc);
  } else {
    // loads are issued in batches (the split count is a run-time value, a plain loop would
    // wait for each load in turn)
    float mx = -INFINITY;
    for (int s0 = 0; s0 < n; s0 += 16) {
      float t[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) t[j] = lse[min(s0 + j, n - 1) * split_stride];
#pragma unroll
      for (int j = 0; j < 16; ++j) mx = fmaxf(mx, t[j]);
    }
    if (mx == -INFINITY) mx = 0.f;
    for (int s0 = 0; s0 < n; s0 += 16) {
      float t[16];
      bf16x8 v[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const long long s = min(s0 + j, n - 1);
        t[j] = lse[s * split_stride];
        v[j] = *(const bf16x8*)(po + s * split_stride * 64);
      }
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const float w = s0 + j < n ? __builtin_amdgcn_exp2f(t[j] - mx) : 0.f;
        const f32x8 vf = __builtin_convertvector(v[j], f32x8);
        wsum += w;
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] += w * vf[e];
      }
    }
  }
  const float inv = wsum > 0.f ? 1.0f / wsum : 0.f;
  unsigned short* op = a.out + ((size_t)sp.q_begin * H + rh) * 64 + d8 * 8;
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] *= inv;
  lbm_store_through(op, __builtin_bit_cast(u32x4, __builtin_convertvector(acc, bf16x8)));
}

// ---------------------------------------------------------------------------- fp32, head_dim 128
// Same contract as the bf16 kernel for pools kept in fp32 (the reference's force_fp32 mode,
// lingbot_map/layers/flashinfer_cache.py:118-127,372-383) at the camera head's head_dim 128
// (lingbot_map/heads/camera_head.py:284-377: 16 heads of 128) for more query rows than the
// few-query kernels take; head_dim 64 is in paged_attn_f32_gfx950.hip.
// Full fp32 products and sums on the matrix pipe (v_mfma_f32_16x16x4_f32), exact running
// maximum, no split-KV across workgroups.  One workgroup per (64 query rows, head), two waves
// per 16 query rows.
//
// A lane is (n = lane % 16, g = lane / 16).  Scores are kept transposed, S^T = K Q^T: the
// 16x16x4 product takes K[kv = n][dim k_g] from every lane as A and Q[q = n][dim k_g] as B and
// leaves S^T[kv = 4g + i][q = n] in element i of lane (n, g), so a lane's four elements
// belong to ONE query row and the softmax statistics are per lane plus two cross-lane steps
// over g.  Which head dimension lane group g contributes in step t is free as long as A and B
// agree; dim = (D/4) g + t makes the K operand four consecutive floats per four steps (one
// ds_read_b128) and the Q operand a contiguous quarter row held in registers.  For O^T = V^T P^T
// the same freedom is used on the KV index: step (c, i) contracts kv = 16c + 4g + i over g,
// which is exactly where element i of the score block c already sits - P goes from the
// accumulator into the B operand without a shuffle.  Output block e takes head dimension
// (D/16) n + e from lane n as its A operand (one ds_read_b128 of V per lane and KV row covers
// four blocks), which leaves O^T[dim = (D/16)(4g + i) + e][q = n] in element i of block e:
// consecutive dims across the blocks, 16-byte stores.
namespace {
constexpr int kF32Rows = 64;
}  // namespace

// Maximum over the four lanes n, n + 16, n + 32, n + 48 that share a query row, on the vector
// ALU (no LDS round trip): rows of 16 lanes pairwise, then the two halves of the wavefront.
__device__ __forceinline__ float max_over_lane_groups(float x) {
  float a, b;
  swap_rows(x, a, b);
  x = fmaxf(a, b);
  swap_halves(x, a, b);
  return fmaxf(a, b);
}

template <int S>
__global__ __launch_bounds__(512) void lbm_attn_f32_kernel(AttnArgsF32<S> a) {
  constexpr int D = 128;
  // NG groups of four waves: wave w of every group owns the same 16 query rows, group j takes
  // KV tiles j, j + NG, ... (NG waves per SIMD, so one wave's softmax, LDS waits and barriers
  // overlap the others' matrix work); the partial results are merged through LDS at the end.
  constexpr int NG = 2;                        // wave groups = tiles staged per iteration
  constexpr int kThreadsF32 = 256 * NG;
  constexpr int kTile = 16;                    // KV tokens per tile = one 16-token score block
  constexpr int kStage = kTile * D / 256;      // floats of K (and of V) a thread stages per iteration
  constexpr int kRowThreads = D / kStage;      // threads that stage one row
  constexpr int LD = D + 4;                    // LDS row stride: rows stay 16-byte aligned and shift by 4 banks
  constexpr int NE = D / 16;                   // 16-dim output blocks
  constexpr int DG = D / 4;                    // head dims one lane group contributes to q.k
  static_assert(kThreadsF32 / kRowThreads == NG * kTile && kStage % 4 == 0, "the threads stage NG tiles");
  constexpr int kTileFloats = NG * kTile * LD;  // NG tiles of K (and as many again of V)
  constexpr int kMergeFloats = (NE * 4 + 2) * 256 * (NG / 2);
  constexpr int kLdsFloats = 2 * kTileFloats > kMergeFloats ? 2 * kTileFloats : kMergeFloats;
  __shared__ __attribute__((aligned(16))) float lds_raw[kLdsFloats];
  float (*lds_k)[LD] = (float (*)[LD])lds_raw;
  float (*lds_v)[LD] = (float (*)[LD])(lds_raw + kTileFloats);
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = (tid >> 6) & 3, grp = tid >> 8;
  const int n16 = lane & 15, g = lane >> 4;
  int b = 0;
  for (int i = 1; i < a.n_streams; ++i)
    if ((int)blockIdx.x >= a.wg_begin[i]) b = i;
  lbm_attn_stream sp = a.s[b];
  if (a.live_kv_tokens) sp.kv_tokens = max(a.live_kv_tokens[sp.live_at], 0);
  const int H = a.num_heads;
  const int local = (int)blockIdx.x - a.wg_begin[b];
  const int head = local % H, qt = local / H;
  const int r = qt * kF32Rows + wave * 16 + n16;   // this lane's query row
  const size_t row_elems = (size_t)H * D;
  const bool row_ok = r < sp.q_rows;

  // Q[r][DG g .. DG g + DG - 1], pre-multiplied by scale * log2(e)
  float q[DG];
  {
    const float* qp = a.q + ((size_t)(sp.q_begin + (row_ok ? r : 0)) * H + head) * D + DG * g;
#pragma unroll
    for (int d4 = 0; d4 < DG / 4; ++d4) {
      const f32x4 x = row_ok ? ((const f32x4*)qp)[d4] : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < 4; ++j) q[4 * d4 + j] = x[j] * a.scale_log2;
    }
  }
  f32x4 o[NE];
#pragma unroll
  for (int e = 0; e < NE; ++e) o[e] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;   // running maximum of the row; this lane's share of the row sum

  const int ld_r = tid / kRowThreads, ld_c = (tid % kRowThreads) * kStage;
  const int n_tiles = (sp.kv_tokens + kTile - 1) / kTile;
  const int n_iters = (n_tiles + NG - 1) / NG;
  // Two-deep prefetch: the row-table entry of iteration it + 2 is requested while iteration it
  // is computed, so the K/V loads of iteration it + 1 can be issued without waiting for it.
  f32x4 kk[kStage / 4], vv[kStage / 4];
  constexpr int kNoRow = INT32_MIN;   // not a row: past the end of the stream's KV
  auto entry = [&](int it) -> int {
    const int kvi = it * NG * kTile + ld_r;
    return kvi < sp.kv_tokens ? a.kv_rows[sp.kv_row_begin + kvi] : kNoRow;
  };
  auto fetch = [&](int e) {
#pragma unroll
    for (int i = 0; i < kStage / 4; ++i) kk[i] = vv[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (e != kNoRow) {
      const float *kp, *vp;
      if (e >= 0) {
        kp = a.pool + ((size_t)e * H + head) * D + ld_c;
        vp = kp + (size_t)a.page_size * row_elems;
      } else {
        const size_t off = ((size_t)(-1 - e) * H + head) * D + ld_c;
        kp = a.self_k + off;
        vp = a.self_v + off;
      }
#pragma unroll
      for (int i = 0; i < kStage / 4; ++i) {
        kk[i] = ((const f32x4*)kp)[i];
        vv[i] = ((const f32x4*)vp)[i];
      }
    }
  };
  int e_next = kNoRow;
  if (n_iters > 0) {
    fetch(entry(0));
    if (n_iters > 1) e_next = entry(1);
  }
  for (int it = 0; it < n_iters; ++it) {
    __syncthreads();  // the previous tiles are no longer being read
#pragma unroll
    for (int i = 0; i < kStage / 4; ++i) {
      *(f32x4*)&lds_k[ld_r][ld_c + 4 * i] = kk[i];
      *(f32x4*)&lds_v[ld_r][ld_c + 4 * i] = vv[i];
    }
    __syncthreads();
    if (it + 1 < n_iters) {                // in flight while these tiles are computed
      fetch(e_next);
      e_next = it + 2 < n_iters ? entry(it + 2) : kNoRow;
    }
    const int t = NG * it + grp;           // this wave's tile
    if (t >= n_tiles) continue;            // the last iteration may not have a tile for every group
    const int row0 = grp * kTile;

    // S^T block: sc[i] = score of kv token 4g + i of the tile for query row n16
    // every LDS operand of the tile is requested up front: the V reads complete under the
    // score MFMAs instead of stalling each output MFMA
    f32x4 kf[DG / 4];
#pragma unroll
    for (int d4 = 0; d4 < DG / 4; ++d4) kf[d4] = *(const f32x4*)&lds_k[row0 + n16][DG * g + 4 * d4];
    f32x4 vf[4][NE / 4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int h = 0; h < NE / 4; ++h) vf[i][h] = *(const f32x4*)&lds_v[row0 + 4 * g + i][NE * n16 + 4 * h];
    f32x4 sc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int d4 = 0; d4 < DG / 4; ++d4)
#pragma unroll
      for (int j = 0; j < 4; ++j) sc = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[d4][j], q[4 * d4 + j], sc, 0, 0, 0);
    const int n_valid = sp.kv_tokens - t * kTile;
    if (n_valid < kTile) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (4 * g + i >= n_valid) sc[i] = -INFINITY;
    }
    float mx = fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3]));
    mx = max_over_lane_groups(mx);
    mx = fmaxf(mx, m);                                    // finite: token 0 of every tile is valid
    const float alpha = __builtin_amdgcn_exp2f(m - mx);   // m = -inf on the first tile gives 0
    m = mx;
    l *= alpha;
#pragma unroll
    for (int e = 0; e < NE; ++e) o[e] *= alpha;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      sc[i] = __builtin_amdgcn_exp2f(sc[i] - m);
      l += sc[i];
    }
    // O^T += V^T P^T, contraction step i over kv = 4g + i; block e holds dims NE * m + e
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int e = 0; e < NE; ++e)
        o[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[i][e / 4][e % 4], sc[i], o[e], 0, 0, 0);
  }
  l += __shfl_xor(l, 16);
  l += __shfl_xor(l, 32);

  // merge the groups pairwise: the upper half of the remaining groups writes (o, m, l) per
  // lane, the lower half rescales and adds; the last round normalises and stores
  float* merge = lds_raw;
  const int slot = tid & 255;
#pragma unroll
  for (int stride = NG / 2; stride >= 1; stride /= 2) {
    __syncthreads();
    if (grp >= stride && grp < 2 * stride) {
      float* mb = merge + (size_t)(grp - stride) * (NE * 4 + 2) * 256;
#pragma unroll
      for (int e = 0; e < NE; ++e)
#pragma unroll
        for (int i = 0; i < 4; ++i) mb[(4 * e + i) * 256 + slot] = o[e][i];
      mb[(4 * NE) * 256 + slot] = m;
      mb[(4 * NE + 1) * 256 + slot] = l;
    }
    __syncthreads();
    if (grp < stride) {
      const float* mb = merge + (size_t)grp * (NE * 4 + 2) * 256;
      const float m1 = mb[(4 * NE) * 256 + slot], l1 = mb[(4 * NE + 1) * 256 + slot];
      const float mt = fmaxf(m, m1);
      // a group that saw no tile has m = -inf and contributes nothing
      const float w0 = m > -INFINITY ? exp2f(m - mt) : 0.f;
      const float w1 = m1 > -INFINITY ? exp2f(m1 - mt) : 0.f;
      l = l * w0 + l1 * w1;
      m = mt;
#pragma unroll
      for (int e = 0; e < NE; ++e)
#pragma unroll
        for (int i = 0; i < 4; ++i) o[e][i] = o[e][i] * w0 + mb[(4 * e + i) * 256 + slot] * w1;
    }
  }
  if (grp == 0 && row_ok) {
    const float inv = l > 0.f ? 1.0f / l : 0.f;   // no KV at all leaves zeros
    float* op = a.out + ((size_t)(sp.q_begin + r) * H + head) * D + NE * 4 * g;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int h = 0; h < NE / 4; ++h)
        *(f32x4*)(op + NE * i + 4 * h) =
            f32x4{o[4 * h][i], o[4 * h + 1][i], o[4 * h + 2][i], o[4 * h + 3][i]} * inv;
  }
}

// ---------------------------------------------------------------------------- fp32, few queries
// Streams with at most kDecQ query rows (the camera head: one token per frame attending to
// every frame so far, lingbot_map/heads/camera_head.py:296-346) are bound by reading K and V
// once - and, as long as the cache is short, by the latency of doing so - not by arithmetic, and
// have far too few rows for the matrix kernel's (64 rows, head) workgroups to fill the chip.
//
// D/4 lanes form a row group that takes a K row and its V row, 16 bytes a lane: a wavefront holds
// 64 / (D/4) row groups, a workgroup NW times as many, and the tokens of the workgroup's piece of
// the KV axis are dealt to them one by one.  A group asks for the K AND the V rows of eight
// or eleven tokens at once (V does not wait for the scores: one trip to memory per batch instead of two), and
// keeps the softmax state of its own tokens - maximum, sum, unnormalised output - in registers, so
// nothing crosses lanes inside the loop but the D/4-lane sum of a dot product (DPP) and there is no
// barrier in it; the groups meet through LDS once, at the end.
//
// Up to kDecOneTokens tokens one to four workgroups of eight or sixteen wavefronts take a (stream, head, query row) from
// start to finish: one launch, which also stores the caller's new rows (lbm_attn_run_append).
// Beyond that the KV axis is cut into chunks of 256 down to 64 tokens, one workgroup of four wavefronts
// each, which leave partial results for lbm_attn_f32_decode_merge_kernel.  Where the chip has workgroups to spare a
// chunk of 64 tokens is one batch of its eight row groups (head_dim 128): one trip to memory instead of four in a row.
namespace {
constexpr int kDecQ = 8;         // query rows per stream this path takes
constexpr int kDecBatch = 8;     // tokens a row group has in flight
constexpr int kDecOneBatch = 11; // the most where one workgroup takes everything, 16 or 32 (head_dim 128), 32 or 64 row groups
constexpr int kDecChunk = 256;   // tokens per chunk, as long as that makes at most kDecMaxChunks
constexpr int kDecFineChunk = 64, kDecFineWgs = 512, kDecFineChunks = 16;   // shorter chunks, within so many workgroups a launch and chunks a row
constexpr int kDecMaxChunks = 64;
constexpr int kDecOneTokens = 512;
constexpr int kDecOneWaves = 8, kDecChunkWaves = 4;

template <int S>   // streams that there is room for
struct DecodeArgs {
  AttnArgsF32<S> f;
  float* part;                           // [sum n_chunks][q_rows][H][D + 2]
  int n_chunks[S];
  int part_begin[S];                     // in (chunk, query row) units
  unsigned per_chunks[S];                // lbm_per(n_chunks)
  int max_q;                             // most query rows of any stream
  unsigned per_max_q;                    // lbm_per(max_q)
  // lbm_attn_run_append: rows of self_k / self_v that go into the pool once it has been read (NULL: none)
  const int32_t* append_rows;
  int append_tokens;
};
}  // namespace

// sum over the LPR = D/4 lanes that share a K row, on the vector ALU: four DPP steps inside a
// row of 16 lanes, and for 32-lane groups one exchange between neighbouring rows
template <int LPR>
__device__ __forceinline__ float row_group_sum(float v) {
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xf, 0xf, false));   // quad_perm [1,0,3,2]
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xf, 0xf, false));   // quad_perm [2,3,0,1]
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xf, 0xf, false));  // row_half_mirror
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x140, 0xf, 0xf, false));  // row_mirror
  if (LPR == 32) {
    float even, odd;
    swap_rows(v, even, odd);
    v = even + odd;
  }
  return v;
}

// grid: x = chunk of the KV axis, y = head, z = stream * max_q + query row.  ONE: the only chunk of
// its stream - the result goes to `out`; otherwise a partial.  VS: so many workgroups share a row, each with all of
// K and D / VS dimensions of V (z: one behind the others' rows, so that they meet in an XCD's L2) - the same sums for
// every output, from fewer bytes through a CU, which is what bounds a launch of few rows (a token of 128 floats is
// 1,024 bytes for one workgroup, 640 for each of four).  us, 16 heads, caches in HBM, VS 1, 2, 4: head_dim 128, 100
// tokens 4.9, 4.5, 4.4; 200 8.6, 7.4, 7.0; 300 10.6, 9.2, 8.2; four streams of 300 11.7, 10.1, 9.0; eight of them 12.5,
// 12.0, 13.6 (two workgroups per CU); head_dim 64, 300 tokens 6.8, 6.2, 5.8.
template <int S, int D, int NW, int NB, bool ONE, int VS = 1>
__global__ __launch_bounds__(NW * 64) void lbm_attn_f32_decode_kernel(DecodeArgs<S> a) {
#pragma clang fp contract(off)   // (products are fused by name: a stream's result does not depend on how many share its launch)
  constexpr int LPR = D / 4;         // lanes per K/V row, 16 bytes each
  constexpr int RPW = 64 / LPR;      // row groups of a wavefront
  constexpr int G = NW * RPW;        // row groups of the workgroup
  constexpr int DV = D / VS, VE = 4 / VS;   // dimensions of V: the workgroup's, a lane's
  typedef __attribute__((ext_vector_type(VE))) float vec;
  static_assert(ONE || VS == 1, "partials hold whole rows");
  __shared__ __attribute__((aligned(16))) float red_o[NW][DV];
  __shared__ float red_m[NW], red_l[NW];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // (what the first loads need of the arguments, the first stream's beside the launch's, in one trip and without divisions behind
  // it: see lbm_first_plan; sixteen caches of 300 tokens of 128 floats a frame 120 -> 111 us, one of 10,000 37.8 -> 37.2)
  lbm_attn_stream sp = a.f.s[0];
  int n_chunks = a.n_chunks[0], part_begin = ONE ? 0 : a.part_begin[0];
  unsigned per_chunks = ONE ? 0 : a.per_chunks[0];
  asm volatile("" : : "s"(a.f.q), "s"(a.f.pool), "s"(a.f.self_k), "s"(a.f.self_v), "s"(a.f.kv_rows), "s"(a.f.live_kv_tokens), "s"(a.f.num_heads), "s"(a.f.page_size),
               "s"(a.f.scale_log2), "s"(a.f.n_streams), "s"(a.max_q), "s"(a.per_max_q), "s"(sp.q_begin), "s"(sp.q_rows), "s"(sp.kv_row_begin), "s"(sp.kv_tokens), "s"(n_chunks),
               "s"(part_begin), "s"(per_chunks));
  const int rows_of_launch = VS == 1 ? 0 : a.f.n_streams * a.max_q;
  int vs = 0, z = blockIdx.z, qi;
#pragma unroll
  for (int i = 1; i < VS; ++i)
    if ((int)blockIdx.z >= i * rows_of_launch) vs = i, z = (int)blockIdx.z - i * rows_of_launch;
  const int b = lbm_divide(z, a.max_q, a.per_max_q, qi), head = blockIdx.y, chunk = blockIdx.x;
  if (S > 1 && b > 0) {
    sp = a.f.s[b];
    n_chunks = a.n_chunks[b];
    part_begin = ONE ? 0 : a.part_begin[b];
    per_chunks = ONE ? 0 : a.per_chunks[b];
  }
  if (chunk >= n_chunks || qi >= sp.q_rows) return;
  if (a.f.live_kv_tokens) sp.kv_tokens = max(a.f.live_kv_tokens[sp.live_at], 0);
  const int H = a.f.num_heads;
  const size_t row_elems = (size_t)H * D;
  int rest = 0;
  const int per = ONE ? sp.kv_tokens : lbm_divide(sp.kv_tokens + n_chunks - 1, n_chunks, per_chunks, rest);
  const int t_begin = ONE ? 0 : chunk * per, t_end = min(t_begin + per, sp.kv_tokens);
  const int grp = wave * RPW + lane / LPR, ln = lane % LPR;

  const f32x4 q4 = *(const f32x4*)(a.f.q + ((size_t)(sp.q_begin + qi) * H + head) * D + 4 * ln) * a.f.scale_log2;
  vec acc = {};
  float m = -INFINITY, l = 0.f;
  const int32_t* rows = a.f.kv_rows + sp.kv_row_begin;
  const size_t head_off = (size_t)head * D + 4 * ln, v_off = (size_t)a.f.page_size * row_elems;
  const size_t v_head_off = (size_t)head * D + vs * DV + VE * ln;
  // tokens past the end of the piece re-read its last token (weight 0): no load sits
  // inside a conditional block
  int e[NB];
  auto entries = [&](int t0) {
#pragma unroll
    for (int j = 0; j < NB; ++j) e[j] = rows[min(t0 + j * G + grp, t_end - 1)];
  };
  if (t_begin < t_end) entries(t_begin);
  for (int t0 = t_begin; t0 < t_end; t0 += NB * G) {
    f32x4 k[NB];
    vec v[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      // negative entries name rows of the caller's own K/V
      const size_t off = (size_t)(e[j] ^ (e[j] >> 31)) * row_elems;
      k[j] = *(const f32x4*)((e[j] < 0 ? a.f.self_k : a.f.pool) + off + head_off);
      v[j] = *(const vec*)((e[j] < 0 ? a.f.self_v : a.f.pool + v_off) + off + v_head_off);
    }
    if (t0 + NB * G < t_end) entries(t0 + NB * G);
    float s[NB], mx = m;
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      s[j] = row_group_sum<LPR>(fmaf(k[j][3], q4[3], fmaf(k[j][2], q4[2], fmaf(k[j][0], q4[0], k[j][1] * q4[1]))));
      if (t0 + j * G + grp >= t_end) {
        s[j] = -INFINITY;
        v[j] = vec{};   // (the last token's values may be infinite: 0 x inf)
      }
      mx = fmaxf(mx, s[j]);
    }
    // (a group that has not met a token yet keeps a reference of -inf and weights of 0)
    const float ref = mx > -INFINITY ? mx : 0.f;
    const float alpha = __builtin_amdgcn_exp2f(m - ref);
    m = mx;
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const float p = __builtin_amdgcn_exp2f(s[j] - ref);
      l = j == 0 ? fmaf(l, alpha, p) : l + p;
#pragma unroll
      for (int i = 0; i < VE; ++i) acc[i] = j == 0 ? fmaf(acc[i], alpha, v[j][i] * p) : fmaf(v[j][i], p, acc[i]);
    }
  }
  // ---- the row groups of a wavefront, then the wavefronts
#pragma unroll
  for (int step = LPR; step < 64; step *= 2) {
    const float m1 = __shfl_xor(m, step), l1 = __shfl_xor(l, step);
    const float mt = fmaxf(m, m1), ref = mt > -INFINITY ? mt : 0.f;
    const float w0 = __builtin_amdgcn_exp2f(m - ref), w1 = __builtin_amdgcn_exp2f(m1 - ref);
#pragma unroll
    for (int i = 0; i < VE; ++i) acc[i] = fmaf(acc[i], w0, __shfl_xor(acc[i], step) * w1);
    l = fmaf(l, w0, l1 * w1);
    m = mt;
  }
  if (lane < LPR) *(vec*)&red_o[wave][VE * ln] = acc;
  if (lane == 0) {
    red_m[wave] = m;
    red_l[wave] = l;
  }
  __syncthreads();     // (also: every wavefront has read what it needs of the pool)
  if (tid < DV) {
    float mx = red_m[0];
#pragma unroll
    for (int w = 1; w < NW; ++w) mx = fmaxf(mx, red_m[w]);
    const float ref = mx > -INFINITY ? mx : 0.f;
    // (sixteen wavefronts' in four sums of four: the longer chain's rounding would show)
    constexpr int kSums = NW == 16 ? 4 : 1;
    float os[kSums] = {}, ls[kSums] = {};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float wgt = __builtin_amdgcn_exp2f(red_m[w] - ref);
      ls[w % kSums] = fmaf(red_l[w], wgt, ls[w % kSums]);
      os[w % kSums] = fmaf(red_o[w][tid], wgt, os[w % kSums]);
    }
    const float o = kSums == 1 ? os[0] : (os[0] + os[kSums / 2]) + (os[1 % kSums] + os[kSums - 1]);
    const float lt = kSums == 1 ? ls[0] : (ls[0] + ls[kSums / 2]) + (ls[1 % kSums] + ls[kSums - 1]);
    if (ONE) {
      a.f.out[((size_t)(sp.q_begin + qi) * H + head) * D + vs * DV + tid] = lt > 0.f ? o / lt : 0.f;   // no token: zeros
    } else {
      float* pp = a.part + (((size_t)part_begin + (size_t)chunk * sp.q_rows + qi) * H + head) * (D + 2);
      pp[tid] = o;
      if (tid == 0) {
        pp[D] = mx;
        pp[D + 1] = lt;
      }
    }
  } else if (ONE && a.append_rows && tid < 2 * DV) {
    // this (stream, head)'s share of the append: one query row per stream (the launch checks; and where several
    // workgroups read a row of K, that no table names the row stored here)
    const int t = sp.q_begin, row = a.append_rows[t], d = vs * DV + tid - DV;
    if (row >= 0) {
      float* dst = const_cast<float*>(a.f.pool) + (size_t)row * row_elems + (size_t)head * D + d;
      const size_t src = ((size_t)t * H + head) * D + d;
      dst[0] = a.f.self_k[src];
      dst[v_off] = a.f.self_v[src];
    }
  }
}

// One row's merge by the 128 threads of a workgroup.  Thread c reads chunk c's maximum and sum (all chunks at once), the
// weights go through LDS, then thread d sums the weighted outputs.  Bound by trips to memory: the first kBatch chunks'
// outputs are asked for beside the maxima, before a weight is known, the others' together (40 chunks of 128 floats: six
// trips as batches of eight behind the weights 4.2 us, two so 4.0).  kBatch is the next of 8, 16 and 32 above the number of
// chunks: loads of chunks that are not there cost their issue all the same (us a launch, always 32 and these: 8 chunks 3.9,
// 3.4, 9 to 16 3.9, 3.55; 32 and more are the same either way).  The sums have no branches and their products are fused by
// name: behind a branch per chunk the compiler asked for some of the second batch's outputs only once the chunks before them had
// been added, and rounded one chunk's products apart from the others'.
constexpr int kDecMergeBatch = 32;
static_assert(kDecMaxChunks <= 2 * kDecMergeBatch, "two batches hold every chunk");
template <int D, int kBatch>
__device__ __forceinline__ void lbm_decode_merge_row(const float* base, size_t stride, int nc, float* out, float* w, float (*red)[2]) {
#pragma clang fp contract(off)
  const int tid = threadIdx.x;
  const int d = min(tid, D - 1), c_own = min(tid, nc - 1);      // (loads outside of conditional blocks: they go out together)
  float x[kBatch], m_c = base[c_own * stride + D], l_c = base[c_own * stride + D + 1];
#pragma unroll
  for (int j = 0; j < kBatch; ++j) x[j] = base[min(j, nc - 1) * stride + d];
  if (tid >= nc) m_c = -INFINITY, l_c = 0.f;
  float m = m_c;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
  if ((tid & 63) == 0) red[0][tid >> 6] = m;
  __syncthreads();
  m = fmaxf(red[0][0], red[0][1]);
  const float w_c = m_c > -INFINITY ? exp2f(m_c - m) : 0.f;   // a chunk without tokens weighs nothing
  if (tid < kDecMaxChunks) w[tid] = w_c;      // (0 for a chunk that is not there)
  float l = l_c * w_c;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) l += __shfl_xor(l, o);
  if ((tid & 63) == 0) red[1][tid >> 6] = l;
  __syncthreads();
  l = red[1][0] + red[1][1];
  if (tid >= D) return;
  float o = 0.f;
#pragma unroll
  for (int j = 0; j < kBatch; ++j) o = fmaf(j < nc ? x[j] : 0.f, w[j], o);
  if (kBatch == kDecMergeBatch && nc > kBatch) {
#pragma unroll
    for (int j = 0; j < kBatch; ++j) x[j] = base[min(kBatch + j, nc - 1) * stride + tid];
#pragma unroll
    for (int j = 0; j < kBatch; ++j) o = fmaf(kBatch + j < nc ? x[j] : 0.f, w[kBatch + j], o);
  }
  out[tid] = l > 0.f ? o / l : 0.f;
}

// one 128-thread workgroup per (stream, query row, head) merges the chunks' partials (and, grid z beyond the streams, stores
// the caller's new rows: the chunks' kernel has read the pool).
template <int S, int D>
__global__ __launch_bounds__(128) void lbm_attn_f32_decode_merge_kernel(DecodeArgs<S> a) {
  static_assert(kDecMaxChunks <= 128 && D <= 128, "one thread per chunk, one per head dimension");
  __shared__ float w[kDecMaxChunks];
  __shared__ float red[2][2];
  const int b = blockIdx.z, head = blockIdx.y, qi = blockIdx.x, tid = threadIdx.x;
  if (b >= a.f.n_streams) {
    for (int t = (b - a.f.n_streams) * a.max_q + qi; t < a.append_tokens; t += a.max_q * ((int)gridDim.z - a.f.n_streams)) {
      const int row = a.append_rows[t];
      if (row < 0 || tid >= D) continue;
      const size_t row_elems = (size_t)a.f.num_heads * D, src = (size_t)t * row_elems + (size_t)head * D + tid;
      float* dst = const_cast<float*>(a.f.pool) + (size_t)row * row_elems + (size_t)head * D + tid;
      dst[0] = a.f.self_k[src];
      dst[(size_t)a.f.page_size * row_elems] = a.f.self_v[src];
    }
    return;
  }
  const lbm_attn_stream sp = a.f.s[S == 1 ? 0 : b];
  if (qi >= sp.q_rows) return;
  const int H = a.f.num_heads, nc = a.n_chunks[S == 1 ? 0 : b];
  const size_t stride = (size_t)sp.q_rows * H * (D + 2);      // from one chunk's partial to the next
  const float* base = a.part + (((size_t)a.part_begin[S == 1 ? 0 : b] + qi) * H + head) * (D + 2);
  float* out = a.f.out + ((size_t)(sp.q_begin + qi) * H + head) * D;
  if (nc <= 8) lbm_decode_merge_row<D, 8>(base, stride, nc, out, w, red);
  else if (nc <= 16) lbm_decode_merge_row<D, 16>(base, stride, nc, out, w, red);
  else lbm_decode_merge_row<D, kDecMergeBatch>(base, stride, nc, out, w, red);
}

// Chunks per stream for the few-query path, and the floats of partials they need.  Depends on
// row and token counts only (never on the dtype), so the workspace query can include it.
//
// fine_chunks: chunks of 64 tokens up to so many per row, 0 for none.  As many as leave the launch at two workgroups
// per CU: beyond that its time is that of the bytes and not of the trips.  No more than sixteen a row, since the
// merge's time grows with them; but thirty-two for caches of 128 floats a row from 3,072 tokens up, where sixteen would be
// chunks of nearly 256 again.  (Beyond 8,192 tokens, or 4,096 of 64 floats, chunks of 256 are the more and decide,
// whole workgroups per CU or not.)  us a launch, 16 heads, caches in HBM, chunks of 256 | these: head_dim 128, one row over 500
// tokens 14.5 | 9.1, 700 14.9 | 10.1, 1,500 16.5 | 12.0, 3,000 18.3 | 16.7, 5,000 25.0 | 22.2; four streams of 1,000
// 20.4 | 17.9; head_dim 64, 700 11.1 | 9.4, 3,000 13.1 | 12.3, four streams of 1,000 13.9 | 12.8.  (Eight rows of one
// stream, that is four chunks a row: head_dim 64, 700 tokens 11.4 | 11.8, so not from there.)
static int lbm_decode_fine_chunks(const LbmAttnSchedule& sch, int num_heads, int head_dim) {
  long long rows = 0;
  int most = 0;
  for (int i = 0; i < sch.n_streams; ++i) {
    rows += sch.s[i].q_rows;
    if (sch.s[i].kv_tokens > most) most = sch.s[i].kv_tokens;
  }
  if (rows <= 0 || rows * num_heads * 8 > kDecFineWgs) return 0;
  const int fit = (int)(kDecFineWgs / (rows * num_heads)), cap = head_dim == 128 && most > 12 * kDecChunk ? 2 * kDecFineChunks : kDecFineChunks;
  return fit < cap ? fit : cap;
}
static int lbm_decode_chunks(int kv_tokens, int fine_chunks) {
  int n = (kv_tokens + kDecChunk - 1) / kDecChunk;
  const int fine = (kv_tokens + kDecFineChunk - 1) / kDecFineChunk, most = fine < fine_chunks ? fine : fine_chunks;
  if (n < most) n = most;
  return n < 1 ? 1 : (n > kDecMaxChunks ? kDecMaxChunks : n);
}
static bool lbm_decode_applies(const LbmAttnSchedule& sch) {
  for (int i = 0; i < sch.n_streams; ++i)
    if (sch.s[i].q_rows > kDecQ) return false;
  return sch.n_streams > 0;
}
static size_t lbm_decode_bytes(const LbmAttnSchedule& sch, int num_heads, int head_dim, int fine_chunks) {
  if (!lbm_decode_applies(sch)) return 0;
  size_t rows = 0;
  for (int i = 0; i < sch.n_streams; ++i) rows += (size_t)lbm_decode_chunks(sch.s[i].kv_tokens, fine_chunks) * sch.s[i].q_rows;
  return rows * num_heads * (head_dim + 2) * sizeof(float);
}

// ---------------------------------------------------------------------------- schedule
// How many KV splits each stream gets.  All workgroups of one launch compete for the 256 CUs
// (one 8-wave workgroup per CU at a time, handed out in blockIdx order), so the choice is a
// small scheduling problem: few long workgroups leave CUs idle at the end, many short ones
// pay the per-workgroup prologue/epilogue and more split-KV partials.  A handful of candidate
// tile counts per workgroup is priced with the measured costs below by simulating the
// hand-out (streams with the longest workgroups first), and the cheapest wins.  The result
// depends on row and tile counts only, and the last few are remembered per thread: a frame's blocks
// alternate between two or three of them (attention within the frame, over the cache, the encoder's), and pricing one
// takes the host 1 us with one stream and 3 with four.
namespace {
// Costs in us, fitted to back-to-back launches at 16 heads x 64 over 100-1,374 query rows and 100-17,000
// tokens, one to four streams (the choice is within 10 % of the best one measured in 19 of 20).  What a
// tile costs depends on how much of the chip works at once (`busy`, its wavefronts with rows to work on over
// the 2,048 it holds, up to 1): a full chip runs at a lower clock.
// A workgroup of the split-KV kernel with `waves` of its eight wavefronts on rows of the stream (up to
// four: one per SIMD):
double main_tile_us(int waves, double busy) { return waves <= 4 ? 0.70 + 0.96 * busy * busy : 1.18 + 0.42 * busy * busy; }
double main_fixed_us(int waves, double busy) {   // launch, prologue, epilogue
  return 5.7 + (waves <= 4 ? 20.0 : 4.0) * busy * busy * busy;
}
// The upper estimate (price_candidate with `wary`).
constexpr double kWaryTileUs = 1.95, kWaryFixedTiles = 3.0, kWaryCombineUs = 2.5, kWaryCombineBytesPerUs = 5.0e6;
constexpr double kCombineUs = 3.2;         // the merging launch
constexpr double kCombineBytesPerUs = 8.0e6;
// A workgroup of the short-KV kernel on 64 or 32 query rows: a step is eight 32-token pieces.
constexpr double kSmLaunchUs = 1.8;        // launch to first instruction
// Its counterpart for 64-row workgroups of the short-KV kernel: start and end, one 64-token tile.
constexpr double kWarySmallUs = 4.0, kWarySmallTileUs = 0.3625;
double small_fixed_us(int rows) { return rows == 64 ? 3.8 : 2.5; }
// (`busy` here: workgroups per CU)
double small_step_us(int rows, double busy) { return rows == 64 ? 0.88 + 0.30 * busy * busy : 0.74 + 0.12 * busy * busy; }

// `count` workgroups of `us` each
struct WorkgroupClass { double us; long long count; };
// When the last of them ends, each handed to the CU (of 256) that frees up first, longest first.  CUs that free up at the same
// time are one group: a class takes a whole group or the part of it that it has workgroups for, so there is at
// most one group more per class.  (Workgroup by workgroup, through a heap of finish times, a launch not seen before took the host 12
// to 120 us, twice in each frame of a stream that grows, now 1 to 2: five frames of 830 rows from an empty cache 340 -> 135 us,
// eight of 1,004 rows in fp32 1,182 -> 1,149.)
double makespan(WorkgroupClass* c, int n) {
  for (int i = 1; i < n; ++i)
    for (int j = i; j > 0 && c[j].us > c[j - 1].us; --j) { const WorkgroupClass t = c[j]; c[j] = c[j - 1]; c[j - 1] = t; }
  struct { double at; long long cus; } g[2 * LBM_MAX_STREAMS + 2];   // by time
  int groups = 1;
  g[0].at = 0.0;
  g[0].cus = 256;
  double last = 0.0;
  for (int i = 0; i < n; ++i)
    for (long long left = c[i].count; left > 0;) {
      const long long cus = left < g[0].cus ? left : g[0].cus;
      const double at = g[0].at + c[i].us;
      if (at > last) last = at;
      left -= cus;
      g[0].cus -= cus;
      int k = 0;
      if (g[0].cus == 0) {   // its place goes to the groups before the new one's
        --groups;
        for (; k < groups && g[k + 1].at < at; ++k) g[k] = g[k + 1];
        if (k < groups && g[k + 1].at == at) {
          g[k + 1].cus += cus;
          for (; k < groups; ++k) g[k] = g[k + 1];
        } else {
          g[k].at = at;
          g[k].cus = cus;
          ++groups;
        }
      } else {
        for (k = groups; k > 0 && g[k - 1].at > at; --k) g[k] = g[k - 1];
        if (g[k - 1].at == at) {   // (a workgroup of no time)
          g[k - 1].cus += cus;
          for (; k < groups; ++k) g[k] = g[k + 1];
        } else {
          g[k].at = at;
          g[k].cus = cus;
          ++groups;
        }
      }
    }
  return last;
}

struct ScheduleKey {
  int n_streams = -1, num_heads = 0;
  bool one_cache = false;
  int small = 0;   // query rows per workgroup of the short-KV kernel, 0: the split-KV pair
  int q_rows[LBM_MAX_STREAMS], n_tiles[LBM_MAX_STREAMS];
  int order[LBM_MAX_STREAMS], n_splits[LBM_MAX_STREAMS];
};
constexpr int kMemos = 8;
thread_local ScheduleKey g_schedules[kMemos];
thread_local int g_next_memo = 0;   // the entry the next new schedule replaces

// The split-KV kernel with about `tps` tiles per workgroup; the split counts it means go to n_splits_out.
// `wary`: an upper estimate - a full chip's cost for every workgroup, whole query tiles, partial
// results that are written and read back one after the other.
double price_candidate(const int* qt, const int* nt, int n_streams, int num_heads, int tps, const int* q_rows,
                       int* n_splits_out, bool wary) {
  double part_bytes = 0;
  long long active = 0;   // wavefronts with rows to work on
  int tiles[LBM_MAX_STREAMS];
  for (int i = 0; i < n_streams; ++i) {
    int ns = nt[i] > 0 ? (nt[i] + tps - 1) / tps : 1;
    if (ns > 64) ns = 64;
    if (ns < 1) ns = 1;
    tiles[i] = nt[i] > 0 ? (nt[i] + ns - 1) / ns : 0;
    n_splits_out[i] = nt[i] > 0 ? (nt[i] + tiles[i] - 1) / tiles[i] : 1;
    if (n_splits_out[i] > 1) part_bytes += (double)n_splits_out[i] * q_rows[i] * num_heads * (64 * 2 + 4);
    active += (long long)((q_rows[i] + kQPerWave - 1) / kQPerWave) * num_heads * n_splits_out[i];
  }
  const double busy = active < 2048 ? active / 2048.0 : 1.0;
  WorkgroupClass c[2 * LBM_MAX_STREAMS];
  int n = 0;
  for (int i = 0; i < n_streams; ++i) {   // whole query tiles, and the stream's last one
    if (qt[i] == 0) continue;
    if (wary) {
      c[n++] = {kWaryTileUs * (kWaryFixedTiles + tiles[i]), (long long)qt[i] * num_heads * n_splits_out[i]};
      continue;
    }
    const long long per_tile = (long long)num_heads * n_splits_out[i];
    const int last = (q_rows[i] - (qt[i] - 1) * kQTile + kQPerWave - 1) / kQPerWave;
    if (qt[i] > 1) c[n++] = {main_fixed_us(kWaves, busy) + tiles[i] * main_tile_us(kWaves, busy), (qt[i] - 1) * per_tile};
    c[n++] = {main_fixed_us(last, busy) + tiles[i] * main_tile_us(last, busy), per_tile};
  }
  const double merge = wary ? kWaryCombineUs + 2.0 * part_bytes / kWaryCombineBytesPerUs : kCombineUs + part_bytes / kCombineBytesPerUs;
  return makespan(c, n) + (part_bytes > 0 ? merge : 0.0);
}

// The short-KV kernel with `rows` query rows per workgroup.
double price_small(const int* nt, int n_streams, int num_heads, int rows, const int* q_rows) {
  long long wgs = 0;
  for (int i = 0; i < n_streams; ++i) wgs += (long long)((q_rows[i] + rows - 1) / rows) * num_heads;
  const double busy = wgs < 256 ? wgs / 256.0 : 1.0;
  WorkgroupClass c[LBM_MAX_STREAMS];
  for (int i = 0; i < n_streams; ++i) {
    const int steps = (nt[i] * (kKvTile / kSmPiece) + kSmWaves - 1) / kSmWaves;
    c[i] = {small_fixed_us(rows) + steps * small_step_us(rows, busy), (long long)((q_rows[i] + rows - 1) / rows) * num_heads};
  }
  return kSmLaunchUs + makespan(c, n_streams);
}
}  // namespace

void lbm_attn_schedule(const lbm_attn_stream* streams, int n_streams, int num_heads,
                       LbmAttnSchedule* out, bool fixed_order) {
  LbmAttnSchedule& sch = *out;
  sch = LbmAttnSchedule{};
  sch.n_streams = n_streams;
  sch.fixed_order = fixed_order;
  int qt[LBM_MAX_STREAMS], nt[LBM_MAX_STREAMS], q_rows[LBM_MAX_STREAMS];
  long long work = 0;
  int max_nt = 0;
  for (int i = 0; i < n_streams; ++i) {
    q_rows[i] = streams[i].q_rows;
    qt[i] = (streams[i].q_rows + kQTile - 1) / kQTile;
    nt[i] = (streams[i].kv_tokens + kKvTile - 1) / kKvTile;
    work += (long long)qt[i] * num_heads * nt[i];
    if (nt[i] > max_nt) max_nt = nt[i];
  }
  // The in-workgroup split kernel (one workgroup per 64 or 32 query rows and head, no partial results,
  // no second launch) is priced beside the split-KV plan while the KV of every stream is short: it wins
  // on one frame's 1,004 x 1,004 (10 us against 19) and on few query rows, where 512-row tiles leave most
  // of the chip idle (261 rows x 2,000 tokens: 11 against 16); the split-KV pair on long KV and once
  // several streams would take the CUs rounds of such workgroups.
  bool small_ok = n_streams > 0;
  for (int i = 0; i < n_streams; ++i) small_ok = small_ok && streams[i].kv_tokens <= kSmMaxKv;
  const bool one_cache = !fixed_order && n_streams == 1 && streams[0].kv_tokens != streams[0].q_rows && streams[0].kv_tokens <= kSmMaxCacheKv;
  int found = -1;
  for (int j = 0; j < kMemos && found < 0; ++j) {
    const ScheduleKey& m = g_schedules[j];
    bool hit = m.n_streams == n_streams && m.num_heads == num_heads && m.one_cache == one_cache;
    for (int i = 0; hit && i < n_streams; ++i) hit = m.q_rows[i] == q_rows[i] && m.n_tiles[i] == nt[i];
    if (hit) found = j;
  }
  const bool hit = found >= 0;
  if (!hit) {
    found = g_next_memo;
    g_next_memo = (g_next_memo + 1) % kMemos;
  }
  ScheduleKey& memo = g_schedules[found];
  if (!hit) {
    int best_splits[LBM_MAX_STREAMS], cand_splits[LBM_MAX_STREAMS], wary_splits[LBM_MAX_STREAMS];
    double best = -1.0;
    long long best_tps = 0;
    auto consider = [&](long long tps, bool wary) {
      if (tps < 2) tps = 2;
      if (tps > max_nt) tps = max_nt > 0 ? max_nt : 1;
      const double c = price_candidate(qt, nt, n_streams, num_heads, (int)tps, q_rows, cand_splits, wary);
      // A stream that the upper estimate leaves whole stays whole: split, its partial results would be rounded
      // to bf16 on their way through memory, and no time is worth a result with fewer bits.
      for (int i = 0; !wary && i < n_streams; ++i)
        if (wary_splits[i] == 1 && cand_splits[i] > 1) return;
      if (best < 0 || c < best) {
        best = c;
        best_tps = tps;
        for (int i = 0; i < n_streams; ++i) best_splits[i] = cand_splits[i];
      }
    };
    auto consider_all = [&](bool wary) {
      // the longest stream cut into 1..12 pieces, and the total work spread over 1..3 rounds of 256
      for (int k = 1; k <= 12; ++k) consider((max_nt + k - 1) / k, wary);
      for (int k = 1; k <= 3; ++k) consider((work + 256LL * k - 1) / (256LL * k), wary);
    };
    memo.small = 0;
    if (small_ok) {
      // The two kernels add the same products in different orders, and splitting rounds partial results to
      // bf16 on their way through memory: in a bf16 residual stream without LayerScale (the encoder) either
      // difference grows to 1.2 % over 24 blocks.  Launches this short are therefore dealt between them by fixed
      // estimates, not by the fitted costs, and the pair is the exception: it takes launches that even an
      // upper estimate puts 15 % ahead of 64-row workgroups (four streams of 1,004 tokens: 28 us against 43).
      double rows_us = 0.0, longest = 0.0;
      for (int i = 0; i < n_streams; ++i) {
        const double us = kWarySmallUs + kWarySmallTileUs * (nt[i] > 0 ? nt[i] : 1);
        const double wgs = (double)((q_rows[i] + kQPerWave - 1) / kQPerWave) * num_heads;
        if (wgs > 0 && us > longest) longest = us;
        rows_us += wgs * us;
      }
      const double wary_small = kSmLaunchUs + (rows_us / 256.0 > longest ? rows_us / 256.0 : longest);
      consider_all(true);
      // (32 and 64 rows per workgroup give the same bits where a stream attends to its own rows: the fitted costs choose)
      if (best < 0 || best >= 0.85 * wary_small)
        memo.small = price_small(nt, n_streams, num_heads, 32, q_rows) < price_small(nt, n_streams, num_heads, 64, q_rows) ? 32 : 64;
    } else {
      // The upper estimate's choice, unless the fitted costs see one that is 12 % ahead of it: that is as far as
      // they can be trusted between candidates (592 rows of four streams, 1,776-5,920 tokens: a choice that they
      // put 6 % ahead took 71 us against 68).
      consider_all(true);
      const long long wary_tps = best_tps;
      for (int i = 0; i < n_streams; ++i) wary_splits[i] = best_splits[i];
      best = -1.0;
      consider(wary_tps, false);
      const double wary_choice = best;
      best = -1.0;
      consider_all(false);
      if (best > 0.88 * wary_choice) {
        best = -1.0;
        consider(wary_tps, false);
      }
    }
    // One stream's attention to a cache: no encoder makes such a launch (theirs attend to their own rows), so the
    // fitted costs may give it to the short-KV kernel, up to 4,864 tokens and where they see the pair less than 8 %
    // ahead, up to 256 rows, where no SIMD has two of the pair's wavefronts at work, 4 % behind.  The costs were fitted to
    // K/V that caches hold and underrate both kernels from HBM, by more the longer the list; the two lines and the limit
    // are where the measured crossing (133 launches, 86-1,374 rows over 1,700-4,800 tokens, 8 to 16 heads, K/V from HBM)
    // leaves no launch slower: 63 change over, at 0.68 to 0.94 of the
    // pair's time, 0.84 in the mean; of the 70 that stay 27 would take 0.92.  us, 16 heads, pair and this kernel: 209 x
    // 2,976 19.1, 16.8; 261 x 4,437 23.1, 21.3; 420 x 4,800 26.8, 23.6; 1,004 x 4,800 32.2, 30.3; left to the pair: 209 x
    // 3,500 19.6, 19.1; 256 x 4,437 21.1, 22.1; 1,004 x 5,700 35.2, 35.1; 1,200 x 4,800 37.3, 50.5.  Several streams'
    // launches are priced less well and stay.
    if (!memo.small && one_cache) {
      const double pair_us = price_candidate(qt, nt, n_streams, num_heads, (int)best_tps, q_rows, cand_splits, false);
      const double us32 = price_small(nt, n_streams, num_heads, 32, q_rows), us64 = price_small(nt, n_streams, num_heads, 64, q_rows);
      if ((us32 < us64 ? us32 : us64) < (2 * q_rows[0] <= kQTile ? 0.96 : 1.08) * pair_us) memo.small = us32 < us64 ? 32 : 64;
    }
    memo.n_streams = n_streams;
    memo.num_heads = num_heads;
    memo.one_cache = one_cache;
    int tiles[LBM_MAX_STREAMS];
    for (int i = 0; i < n_streams; ++i) {
      memo.q_rows[i] = q_rows[i];
      memo.n_tiles[i] = nt[i];
      memo.n_splits[i] = best_splits[i];
      memo.order[i] = i;
      tiles[i] = nt[i] > 0 ? (memo.small ? nt[i] : (nt[i] + best_splits[i] - 1) / best_splits[i]) : 0;
    }
    for (int i = 1; i < n_streams; ++i)
      for (int j = i; j > 0 && tiles[memo.order[j]] > tiles[memo.order[j - 1]]; --j) {
        int t = memo.order[j]; memo.order[j] = memo.order[j - 1]; memo.order[j - 1] = t;
      }
  }
  if (memo.small) {
    sch.small = memo.small;
    int wg = 0;
    for (int oi = 0; oi < n_streams; ++oi) {
      const int i = memo.order[oi];
      // streams with the longest workgroups first, as below: the launch ends with short ones (261 rows over
      // 783 tokens and 261 over 2,088 in one launch: a frame of 24 blocks 479 us in the callers' order, 413 so)
      LbmAttnStreamPlan& p = sch.s[oi];
      p.q_begin = streams[i].q_begin;
      p.q_rows = streams[i].q_rows;
      p.kv_row_begin = streams[i].kv_row_begin;
      p.kv_tokens = streams[i].kv_tokens;
      p.live_at = streams[i].live_at;
      p.n_qtiles = (streams[i].q_rows + memo.small - 1) / memo.small;
      p.n_splits = 1;
      p.tiles_per_split = nt[i] > 0 ? nt[i] : 1;
      wg = (wg + 7) & ~7;   // each stream starts on XCD 0 so the in-kernel head -> XCD map lines up
      p.wg_begin = wg;
      p.part_begin = 0;
      // whole groups of 8 workgroups when the heads are dealt over the XCDs
      const int per_q = num_heads;
      wg += p.n_qtiles * per_q;
    }
    sch.total_wgs = wg;
    sch.part_rows = 0;
    return;
  }
  int wg = 0;
  long long part = 0;
  for (int oi = 0; oi < n_streams; ++oi) {
    const int i = memo.order[oi];
    LbmAttnStreamPlan& p = sch.s[oi];   // plans in launch order: blockIdx ranges ascend with the index
    p.q_begin = streams[i].q_begin;
    p.q_rows = streams[i].q_rows;
    p.kv_row_begin = streams[i].kv_row_begin;
    p.kv_tokens = streams[i].kv_tokens;
    p.live_at = streams[i].live_at;
    p.n_qtiles = qt[i];
    const int ns = memo.n_splits[i];
    p.tiles_per_split = nt[i] > 0 ? (nt[i] + ns - 1) / ns : 1;
    p.n_splits = nt[i] > 0 ? (nt[i] + p.tiles_per_split - 1) / p.tiles_per_split : 1;
    // keep each stream's first workgroup on XCD 0 so the in-kernel XCD mapping lines up
    wg = (wg + 7) & ~7;
    p.wg_begin = wg;
    p.part_begin = (int32_t)part;
    wg += p.n_qtiles * num_heads * p.n_splits;
    if (p.n_splits > 1) part += (long long)p.n_splits * p.q_rows;
  }
  sch.total_wgs = wg;
  sch.part_rows = part;
}

size_t lbm_attn_schedule_bytes(const LbmAttnSchedule& sch, int num_heads, int head_dim, bool least) {
  // bf16 partial outputs followed by one float log-sum-exp per (row, head); or, when every
  // stream has only a few query rows, the fp32 partials of the few-query path (the query does
  // not know the dtype, so it covers both)
  const size_t split_kv = (size_t)sch.part_rows * num_heads * (head_dim * 2 + 4);
  const size_t few_q = lbm_decode_bytes(sch, num_heads, head_dim, least ? 0 : lbm_decode_fine_chunks(sch, num_heads, head_dim));
  return split_kv > few_q ? split_kv : few_q;
}

namespace {
// The kernel that a launch on the split-KV schedule takes; own_rows: in order, with no live counts and nothing to append.
enum LbmSplitForm { kFormTable, kFormPair, kFormWhole };
LbmSplitForm lbm_split_form(const LbmAttnSchedule& sch, bool own_rows) {
  // Own rows in order, two splits per stream: both in one workgroup, no launch to merge (lbm_attn_split's PAIR).  us, two
  // kernels and this one: 16 heads, four streams of 833 rows 28.7, 18.8, of 1,004 32.0, 22.3, of 3,000 154, 140, of 5,000
  // 383, 361; 2 x 2,000 43.9, 34.9; 1 x 4,096 68.8, 61.0; four streams of 513 rows over 4,609 60.4, 56.1; from the line on,
  // eight streams of 257 rows over 4,097 54.1, 48.8, 12 heads 51.8, 47.8, of 300 52.1, 49.2, of 448 56.8, 50.7; six of 257
  // 58.8, 54.7; eight of 385 over 1,500 32.2, 25.9.  Up to 256 rows, which leave it half as many workgroups and those with half a
  // load each, the two kernels stay: eight streams of 40 rows over 4,097 45.8, 54.6; 12 heads, 255 rows over 4,223 44.5, 51.9.
  bool pair = own_rows;
  for (int i = 0; i < sch.n_streams; ++i) pair = pair && sch.s[i].n_splits == 2 && 2 * sch.s[i].q_rows > kQTile;
  if (pair) return kFormPair;
  // The same in one split.  us, with the table and without, 16 heads: 6 streams of 600 rows 21.6, 20.7; 8 x 1,004
  // 39.7, 38.7; 3 x 1,500 61.7, 58.3; 16 x 100 over 4,097 76.1, 71.6.
  bool whole = own_rows;
  for (int i = 0; i < sch.n_streams; ++i) whole = whole && sch.s[i].n_splits == 1;
  return whole ? kFormWhole : kFormTable;
}
}  // namespace

// (the kernels of own rows have no workgroups that ask)
bool lbm_attention_asks(const LbmAttnSchedule& sch, bool own_rows) {
  return (sch.small || lbm_split_form(sch, own_rows) == kFormTable) && lbm_idle_cus(sch.total_wgs) >= kTouchIdle;
}

namespace {
int lbm_launch_attention_only(const void* q, const void* pool, void* out, const void* self_k,
                              const void* self_v, const int32_t* kv_rows, const int32_t* live_kv_tokens,
                              const LbmAttnSchedule& sch, int num_heads, int head_dim, int page_size, int dtype,
                              float sm_scale, void* workspace, size_t workspace_bytes, hipStream_t stream, const int32_t* append_rows,
                              int append_tokens, bool append_apart, bool own_rows, const LbmTouch* touch, bool* appended);
}  // namespace

// append_rows (lbm_attn_run_append): rows of self_k / self_v that are stored in the pool after the
// attention has read it - inside the launch that merges the split-KV partials when the schedule has
// one, by lbm_kv_append_kernel behind the attention otherwise.  append_apart: the row tables name none of
// them, so nobody minds when they are stored, and the bf16 kernels and the fp32 head_dim 64 kernel carry
// them by workgroups of their own behind the others (a streamed frame of 261 rows over 2,349 tokens, us per block: 19.2 with
// a launch for the append, 16.3 without; fp32, 1,004 rows: 3 us a frame).
int lbm_launch_attention(const void* q, const void* pool, void* out, const void* self_k,
                         const void* self_v, const int32_t* kv_rows, const int32_t* live_kv_tokens,
                         const LbmAttnSchedule& sch,
                         int num_heads, int head_dim, int page_size, int dtype, float sm_scale,
                         void* workspace, size_t workspace_bytes, hipStream_t stream, const int32_t* append_rows, int append_tokens, bool append_apart, bool own_rows, const LbmTouch* touch) {
  bool appended = false;
  int rc = lbm_launch_attention_only(q, pool, out, self_k, self_v, kv_rows, live_kv_tokens, sch, num_heads, head_dim,
                                     page_size, dtype, sm_scale, workspace, workspace_bytes, stream, append_rows, append_tokens, append_apart, own_rows, touch, &appended);
  if (rc != LBM_OK || !append_rows || append_tokens <= 0 || appended) return rc;
  return lbm_launch_append(self_k, self_v, dtype, const_cast<void*>(pool), dtype, append_rows, append_tokens, num_heads,
                           head_dim, page_size, stream);
}

namespace {
template <int S>
int lbm_launch_f32(const AttnCoreF32& core, const LbmAttnSchedule& sch, int head_dim, void* workspace, size_t workspace_bytes, hipStream_t stream,
                   const int32_t* append_rows, int append_tokens, bool append_apart, bool* appended) {
  AttnArgsF32<S> f;
  static_cast<AttnCoreF32&>(f) = core;
  int wg = 0;
  for (int i = 0; i < S; ++i) {
    f.s[i] = lbm_attn_stream{0, 0, 0, 0, 0};
    f.wg_begin[i] = wg;
    if (i < sch.n_streams) {
      f.s[i] = lbm_attn_stream{sch.s[i].q_begin, sch.s[i].q_rows, sch.s[i].kv_row_begin, sch.s[i].kv_tokens, sch.s[i].live_at};
      wg += ((sch.s[i].q_rows + kF32Rows - 1) / kF32Rows) * f.num_heads;
    }
  }
  f.wg_begin[S] = wg;
  if (wg == 0) return LBM_OK;
  if (lbm_decode_applies(sch)) {
    DecodeArgs<S> d;
    d.f = f;
    d.part = (float*)workspace;
    d.append_rows = append_tokens > 0 ? append_rows : nullptr;
    d.append_tokens = append_tokens;
    int max_chunks = 0, max_q = 0, min_q = kDecQ, part = 0, most = 0;
    int fine = lbm_decode_fine_chunks(sch, f.num_heads, head_dim);
    if (workspace_bytes < lbm_decode_bytes(sch, f.num_heads, head_dim, fine)) fine = 0;   // a workspace for chunks of 256 serves too
    for (int i = 0; i < S; ++i) {
      d.n_chunks[i] = 0;
      d.part_begin[i] = part;
      if (i < sch.n_streams) {
        d.n_chunks[i] = lbm_decode_chunks(sch.s[i].kv_tokens, fine);
        part += d.n_chunks[i] * sch.s[i].q_rows;
        if (d.n_chunks[i] > max_chunks) max_chunks = d.n_chunks[i];
        if (sch.s[i].q_rows > max_q) max_q = sch.s[i].q_rows;
        if (sch.s[i].q_rows < min_q) min_q = sch.s[i].q_rows;
        if (sch.s[i].kv_tokens > most) most = sch.s[i].kv_tokens;
      }
    }
    if (max_q == 0) return LBM_OK;
    d.max_q = max_q;
    d.per_max_q = lbm_per(max_q);
    for (int i = 0; i < sch.n_streams; ++i) d.per_chunks[i] = lbm_per(d.n_chunks[i]);
    // One launch for short lists.  Up to two and a half trips to memory it is the faster form (us, one row of 16 heads
    // of 128, from the last-level cache and from HBM, against the chunked form: 300 tokens 7.0 and 8.2, 9.6 and 10.8;
    // 360 tokens 7.6 and 9.0, 8.9 and 9.9; 440 tokens 9.2 and 10.4, 9.1 and 10.3), beyond that it costs more than a
    // second launch (500 tokens 9.2 and 10.7, 8.0 and 9.0) unless fewer chunks fit (four streams, 500 tokens 10.0 and
    // 11.9, 11.1 and 12.4).  With one query row per stream and nothing to append beyond those rows it carries the
    // append as well.
    const int few = kDecOneWaves * 256 / head_dim, trip = kDecOneBatch * few;   // row groups of eight wavefronts, their tokens in flight
    if (most <= kDecOneTokens && (fine < kDecFineChunks || most <= trip * 5 / 2)) {
      for (int i = 0; i < sch.n_streams; ++i) d.n_chunks[i] = 1;
      unsigned covered = 0;   // rows 0 .. n_streams - 1 of the append, each some stream's query row
      for (int i = 0; i < sch.n_streams; ++i)
        if (sch.s[i].q_begin < LBM_MAX_STREAMS) covered |= 1u << sch.s[i].q_begin;
      const bool carries = d.append_rows && max_q == 1 && min_q == 1 && append_tokens == sch.n_streams &&
                           covered == (1u << append_tokens) - 1u;
      if (!carries) d.append_rows = nullptr;
      else *appended = true;
      // A row to four or two workgroups where that leaves one per CU, not for the shortest lists (16 tokens of 64
      // floats 2.75, 2.83), and not where a row to append may be one that another workgroup still has to read.
      const long long rows = (long long)f.num_heads * sch.n_streams * max_q;
      const int shares = (d.append_rows && !append_apart) || most <= 32 ? 1 : rows * 4 <= 256 ? 4 : rows * 2 <= 256 ? 2 : 1;
      // Sixteen wavefronts, each group with half as many tokens, where eight would make more than one trip (16 heads, K/V
      // from HBM, rows of a page each, us with eight and with sixteen: head_dim 128, 150 tokens 5.2, 5.3; 200 6.2, 5.8; 300
      // 7.2, 6.8; 440 9.4, 8.5; four streams of 300 8.5, 8.0, of 440 10.9, 10.0; head_dim 64, 300 tokens 5.1, 5.2; 400 6.0, 5.7).
      const bool many = most > trip;
      const int trips = many ? (most + 2 * trip - 1) / (2 * trip) : 1, groups = many ? 2 * few : few;
      const dim3 grid(1, f.num_heads, sch.n_streams * max_q * shares), block((many ? 2 : 1) * kDecOneWaves * 64);
      // As few trips as batches of eleven need, and batches no longer than so many trips need: a step loads its
      // batch whether the tokens are there or not, 0.13 us for 16 rows of 128 floats at a CU's 64 bytes per cycle.
      // us a launch, 16 heads, eight wavefronts, batches of eleven and these: head_dim 128, 16 tokens 4.3, 2.8; 64 4.3, 3.1; 100 4.3, 4.0;
      // 200 6.2, 5.7; head_dim 64, 100 tokens 4.2, 3.1; 400 6.2, 5.5.  (Ten: no better than eleven.)
      const int batch = (most + trips * groups - 1) / (trips * groups);
#define LBM_DECODE_ONE_VS(D, NW, NB, VS) hipLaunchKernelGGL((lbm_attn_f32_decode_kernel<S, D, NW, NB, true, VS>), grid, block, 0, stream, d);
#define LBM_DECODE_ONE_D(D, NW, NB)                                                                                                            \
  {                                                                                                                                          \
  if (shares == 4) LBM_DECODE_ONE_VS(D, NW, NB, 4)                                                                                           \
  else if (shares == 2) LBM_DECODE_ONE_VS(D, NW, NB, 2)                                                                                      \
  else LBM_DECODE_ONE_VS(D, NW, NB, 1)                                                                                                       \
  }
#define LBM_DECODE_ONE(NW, NB)                                                                                                                \
  {                                                                                                                                          \
  if (head_dim == 64) LBM_DECODE_ONE_D(64, NW, NB)                                                                                           \
  else LBM_DECODE_ONE_D(128, NW, NB)                                                                                                         \
  }
      static_assert(kDecOneTokens <= 8 * 2 * kDecOneWaves * 256 / 64, "head_dim 64 needs no longer batches of sixteen wavefronts than eight");
      if (many && batch <= 6) LBM_DECODE_ONE(2 * kDecOneWaves, 6)        // (more than half a trip of sixteen)
      else if (many && batch <= 8) LBM_DECODE_ONE(2 * kDecOneWaves, 8)
      else if (many) LBM_DECODE_ONE_D(128, 2 * kDecOneWaves, kDecOneBatch)
      else if (batch <= 2) LBM_DECODE_ONE(kDecOneWaves, 2)
      else if (batch <= 4) LBM_DECODE_ONE(kDecOneWaves, 4)
      else if (batch <= 6) LBM_DECODE_ONE(kDecOneWaves, 6)
      else if (batch <= 8) LBM_DECODE_ONE(kDecOneWaves, 8)
      else LBM_DECODE_ONE(kDecOneWaves, kDecOneBatch)
#undef LBM_DECODE_ONE
#undef LBM_DECODE_ONE_D
#undef LBM_DECODE_ONE_VS
      return lbm_check_launch("lbm_attn_f32_decode_kernel<one chunk>");
    }
    const dim3 grid(max_chunks, f.num_heads, sch.n_streams * max_q), block(kDecChunkWaves * 64);
    const dim3 mgrid(max_q, f.num_heads, sch.n_streams + (d.append_rows ? (append_tokens + max_q - 1) / max_q : 0));
    if (d.append_rows) *appended = true;
    if (head_dim == 64) {
      hipLaunchKernelGGL((lbm_attn_f32_decode_kernel<S, 64, kDecChunkWaves, kDecBatch, false>), grid, block, 0, stream, d);
      hipLaunchKernelGGL((lbm_attn_f32_decode_merge_kernel<S, 64>), mgrid, dim3(128), 0, stream, d);
    } else {
      hipLaunchKernelGGL((lbm_attn_f32_decode_kernel<S, 128, kDecChunkWaves, kDecBatch, false>), grid, block, 0, stream, d);
      hipLaunchKernelGGL((lbm_attn_f32_decode_merge_kernel<S, 128>), mgrid, dim3(128), 0, stream, d);
    }
    return lbm_check_launch("lbm_attn_f32_decode_kernel");
  }
  if (head_dim == 64) {
    if (append_apart && append_rows && append_tokens > 0) {
      f.append_rows = append_rows;
      f.append_tokens = append_tokens;
      *appended = true;
    }
    return lbm_launch_attn_f32_d64(f, stream);
  }
  hipLaunchKernelGGL(lbm_attn_f32_kernel<S>, dim3(wg), dim3(512), 0, stream, f);
  return lbm_check_launch("lbm_attn_f32_kernel");
}

template <int S>
int lbm_launch_bf16(const AttnCore& core, const LbmAttnSchedule& sch, hipStream_t stream, const int32_t* append_rows, int append_tokens,
                    bool append_apart, bool own_rows, const LbmTouch* touch, bool* appended) {
  AttnArgs<S> a;
  static_cast<AttnCore&>(a) = core;
  a.n_streams = sch.n_streams;
  a.total_wgs = sch.total_wgs;
  a.touch = touch ? *touch : LbmTouch{};
  for (int i = 0; i < sch.n_streams; ++i) a.s[i] = sch.s[i];
  auto streams_by_workgroup = [&]() {
    for (int i = 0; i < S; ++i) a.first_wg[i] = i < sch.n_streams ? a.s[i].wg_begin : 0x7fffffff;
    for (int i = 0; i < sch.n_streams; ++i) a.s[i].per_qtiles = lbm_per(a.s[i].n_qtiles);
  };
  streams_by_workgroup();
  if (sch.small) {
    unsigned blocks = (unsigned)sch.total_wgs;
    if (append_apart && append_rows && append_tokens > 0) {
      a.append_rows = append_rows;
      a.append_tokens = append_tokens;
      blocks += (unsigned)(((long long)append_tokens * a.num_heads * 8 + kSmThreads - 1) / kSmThreads);
      *appended = true;
    }
    bool turn = false;   // (for all streams over a cache; the kernel leaves out those with up to two pieces per wavefront, by the live count)
    for (int i = 0; i < sch.n_streams && !sch.fixed_order; ++i) turn = turn || (sch.s[i].kv_tokens != sch.s[i].q_rows && sch.s[i].kv_tokens > kSmTurnKv);
    const dim3 grid = lbm_touch_grid(a.touch, blocks), block(kSmThreads);
    // (own rows in order change where rows are read from, not the order of the sums: a launch that goes round keeps its table)
    if (own_rows && !turn) {
      if (sch.small == 64) hipLaunchKernelGGL((lbm_attn_bf16_d64_small_kernel<S, 2, false, true>), grid, block, 0, stream, a);
      else hipLaunchKernelGGL((lbm_attn_bf16_d64_small_kernel<S, 1, false, true>), grid, block, 0, stream, a);
      return lbm_check_launch("lbm_attn_bf16_d64_small_kernel<own rows>");
    }
    if (sch.small == 64 && turn) hipLaunchKernelGGL((lbm_attn_bf16_d64_small_kernel<S, 2, true>), grid, block, 0, stream, a);
    else if (sch.small == 64) hipLaunchKernelGGL((lbm_attn_bf16_d64_small_kernel<S, 2, false>), grid, block, 0, stream, a);
    else if (turn) hipLaunchKernelGGL((lbm_attn_bf16_d64_small_kernel<S, 1, true>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((lbm_attn_bf16_d64_small_kernel<S, 1, false>), grid, block, 0, stream, a);
    return lbm_check_launch("lbm_attn_bf16_d64_small_kernel");
  }
  const LbmSplitForm form = lbm_split_form(sch, own_rows && !a.live_kv_tokens && append_tokens <= 0);
  if (form == kFormPair) {
    int wg = 0;
    for (int i = 0; i < sch.n_streams; ++i) {
      LbmAttnStreamPlan& p = a.s[i];
      p.n_qtiles = (p.q_rows + kQTile / 2 - 1) / (kQTile / 2);
      wg = (wg + 7) & ~7;   // (a stream's first workgroup on XCD 0, as in the schedule)
      p.wg_begin = wg;
      wg += p.n_qtiles * a.num_heads;
    }
    streams_by_workgroup();
    hipLaunchKernelGGL(lbm_attn_bf16_d64_pair_kernel<S>, dim3((unsigned)wg), dim3(kThreads), 0, stream, a);
    return lbm_check_launch("lbm_attn_bf16_d64_pair_kernel");
  }
  if (form == kFormWhole) {
    hipLaunchKernelGGL(lbm_attn_bf16_d64_own_kernel<S>, dim3((unsigned)sch.total_wgs), dim3(kThreads), 0, stream, a);
    return lbm_check_launch("lbm_attn_bf16_d64_own_kernel");
  }
  // The append by workgroups behind the attention's: they run where CUs are done early (the last split of a list has fewer
  // tiles), and the launch that merges does not wait for them.  us a block, both builds' kernels: 1,004 rows over 17,068
  // tokens 71.6 + 6.6 for the merge and the append, 72.0 + 5.8; four streams of 1,004 rows 207.5 + 16.3, 209.3 + 11.7.
  unsigned wgs = (unsigned)sch.total_wgs;
  if (append_apart && append_rows && append_tokens > 0) {
    a.append_rows = append_rows;
    a.append_tokens = append_tokens;
    wgs += (unsigned)(((long long)append_tokens * a.num_heads * 8 + kThreads * kAppendPieces - 1) / (kThreads * kAppendPieces));
    *appended = true;
  }
  hipLaunchKernelGGL(lbm_attn_bf16_d64_kernel<S>, lbm_touch_grid(a.touch, wgs), dim3(kThreads), 0, stream, a);
  int rc = lbm_check_launch("lbm_attn_bf16_d64_kernel");
  if (rc != LBM_OK) return rc;
  if (sch.part_rows > 0) {
    int max_rows = 0;
    for (int i = 0; i < sch.n_streams; ++i)
      if (sch.s[i].n_splits > 1 && sch.s[i].q_rows > max_rows) max_rows = sch.s[i].q_rows;
    const long long threads = (long long)max_rows * a.num_heads * 8;
    unsigned blocks = (unsigned)((threads + 255) / 256);
    a.combine_blocks = (int)blocks;
    if (append_rows && append_tokens > 0 && !*appended) {
      a.append_rows = append_rows;
      a.append_tokens = append_tokens;
      blocks += (unsigned)(((long long)append_tokens * a.num_heads * 8 + 255) / 256);
      *appended = true;
    }
    hipLaunchKernelGGL(lbm_attn_combine_bf16_kernel<S>, dim3(blocks, sch.n_streams), dim3(256), 0, stream, a);
    rc = lbm_check_launch("lbm_attn_combine_bf16_kernel");
  }
  return rc;
}

int lbm_launch_attention_only(const void* q, const void* pool, void* out, const void* self_k,
                              const void* self_v, const int32_t* kv_rows, const int32_t* live_kv_tokens,
                              const LbmAttnSchedule& sch, int num_heads, int head_dim, int page_size, int dtype,
                              float sm_scale, void* workspace, size_t workspace_bytes, hipStream_t stream, const int32_t* append_rows,
                              int append_tokens, bool append_apart, bool own_rows, const LbmTouch* touch, bool* appended) {
  if (head_dim != 64 && !(head_dim == 128 && dtype == LBM_DTYPE_F32))
    return lbm_fail(LBM_ERR_UNSUPPORTED, "attention kernels cover head_dim 64 (bf16, fp32) and 128 (fp32), got %d", head_dim);
  if (dtype == LBM_DTYPE_F32) {
    AttnCoreF32 f;
    f.q = (const float*)q;
    f.pool = (const float*)pool;
    f.out = (float*)out;
    f.self_k = (const float*)self_k;
    f.self_v = (const float*)self_v;
    f.kv_rows = kv_rows;
    f.live_kv_tokens = live_kv_tokens;
    f.num_heads = num_heads;
    f.page_size = page_size;
    f.scale_log2 = sm_scale == 0.f ? 1.0f : sm_scale * 1.4426950408889634f;   // 0: q already carries scale * log2(e)
    f.per_heads = lbm_per(num_heads);
    f.per_eighth = lbm_per(num_heads >> 3);
    f.n_streams = sch.n_streams;
    f.append_rows = nullptr;
    f.append_tokens = 0;
    if (sch.n_streams == 1)
      return lbm_launch_f32<1>(f, sch, head_dim, workspace, workspace_bytes, stream, append_rows, append_tokens, append_apart, appended);
    return lbm_launch_f32<LBM_MAX_STREAMS>(f, sch, head_dim, workspace, workspace_bytes, stream, append_rows, append_tokens, append_apart, appended);
  }
  if (dtype != LBM_DTYPE_BF16) return lbm_fail(LBM_ERR_INVALID, "unknown dtype %d", dtype);
  AttnCore a;
  a.q = (const unsigned short*)q;
  a.pool = (const unsigned short*)pool;
  a.out = (unsigned short*)out;
  a.self_k = (const unsigned short*)self_k;
  a.self_v = (const unsigned short*)self_v;
  a.kv_rows = kv_rows;
  a.live_kv_tokens = live_kv_tokens;
  a.part_o = (unsigned short*)workspace;
  a.part_lse = (float*)(a.part_o + (size_t)sch.part_rows * num_heads * head_dim);
  a.num_heads = num_heads;
  a.page_size = page_size;
  a.scale_log2 = sm_scale == 0.f ? 1.0f : sm_scale * 1.4426950408889634f;   // 0: q already carries scale * log2(e)
  a.append_rows = nullptr;
  a.append_tokens = 0;
  a.combine_blocks = 0x7fffffff;
  a.per_heads = lbm_per(num_heads);
  a.per_eighth = lbm_per(num_heads >> 3);
  if (sch.total_wgs == 0) return LBM_OK;
  if (sch.n_streams == 1) return lbm_launch_bf16<1>(a, sch, stream, append_rows, append_tokens, append_apart, own_rows, touch, appended);
  return lbm_launch_bf16<LBM_MAX_STREAMS>(a, sch, stream, append_rows, append_tokens, append_apart, own_rows, touch, appended);
}
}  // namespace

// ---------------------------------------------------------------------------- static scratch
// Workspace for callers that cannot allocate (lbm_attn_run_static): split-KV partials and the
// few-query partials go into this file-scope device array instead of a caller's buffer.  Every
// GPU the library runs on holds its own copy at its own address until the process ends; the
// array's name is only a host-side handle, so the address is looked up once per device with
// that device current and the kernels get the looked-up pointer like any other workspace.
// Nothing in it has to start at zero: every partial a launch reads was written by that launch.
namespace {
constexpr size_t kStaticScratchBytes = (size_t)LBM_STATIC_SCRATCH_MIB << 20;
constexpr int kMaxDevices = 64;
}  // namespace
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];
static void* g_scratch_ptr[kMaxDevices];
static std::mutex g_scratch_mutex;

int lbm_static_scratch(void** ptr, size_t* bytes) {
  int dev = -1;
  const hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return lbm_fail(LBM_ERR_HIP, "hipGetDevice: %s", hipGetErrorString(e));
  if (dev < 0 || dev >= kMaxDevices) return lbm_fail(LBM_ERR_UNSUPPORTED, "device ordinal %d outside [0, %d)", dev, kMaxDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    const hipError_t es = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (es != hipSuccess || !p)
      return lbm_fail(LBM_ERR_HIP, "hipGetSymbolAddress(static scratch) on device %d: %s", dev, hipGetErrorString(es));
    g_scratch_ptr[dev] = p;
  }
  *ptr = g_scratch_ptr[dev];
  *bytes = kStaticScratchBytes;
  return LBM_OK;
}
