// bf16 linear layers of a transformer block for gfx950, with the elementwise work that follows
// them fused into the store:
//     out = epilogue(a @ w^T + bias)      a [M, K], w [N, K] (nn.Linear's weight), bf16 in and out
//   LBM_LINEAR_BIAS            the qkv projection                (lingbot_map/layers/attention.py:413)
//   LBM_LINEAR_BIAS_GELU       fc1 + exact (erf) GELU            (lingbot_map/layers/mlp.py:35-36)
//   LBM_LINEAR_BIAS_RESIDUAL   proj / fc2 + LayerScale + residual: x + gamma * (a @ w^T + bias)
//                              (attention.py:554, mlp.py:38, lingbot_map/layers/block.py:283,
//                              lingbot_map/layers/layer_scale.py:21-22)
// Roundings follow the sequence of separate bf16 torch ops: the linear's output is rounded to
// bf16, then each elementwise op rounds again.
//
// Around that, so that a transformer block needs no LayerNorm, residual or producer launch:
//   * the residual epilogue can leave the row statistics (mean, M2 per column tile) of what it
//     stores (block.py:283-285 feeding the next LayerNorm);
//   * a launch can take activations whose LayerNorm is still to be applied: the product runs on
//     the raw rows and the store applies rstd * (acc - mean * colsum(w)) + bias, the LayerNorm's
//     affine part folded into w and bias by the caller (block.py:194-195, 217; the normalised rows
//     are then never rounded to bf16, the folded weights are);
//   * the qkv projection can carry the pre-attention producer as its epilogue (kEpiQkvPrepare);
//   * a launch with few tiles and a long K can sum K in slices, by several workgroups per tile (SPLITK)
//     or by one (the KS of the small tiles).
//
// Shapes this is written for: M about 1,000 rows per stream (one frame), K, N in 1024 .. 4096.
// At that size a launch has only a few hundred tiles and 16-64 k-steps, so what counts is a
// tile count that matches the 256 CUs and a short prologue, not asymptotic throughput.  Three kernels: the
// one described here; smaller tiles for fewer rows and larger ones for more stand below with what differs.
//
// One workgroup = 8 wavefronts on a 128 x 128 tile of the output (TN = 64: 128 x 64, 256: 128 x 256).  The product
// is computed transposed, C^T = W A^T with v_mfma_f32_32x32x16_bf16 (A operand = 32 rows of W, B
// operand = 32 rows of the activations), so an accumulator register holds four consecutive output
// columns of one row.  The eight wavefronts are two groups of four: each group covers the whole
// tile (a wavefront owns 64 x TN / 2 of it) over its own half of every K slice, which gives each
// SIMD two wavefronts to cover each other's LDS and barrier waits without giving up the fragment
// reuse of the large per-wave tile; the two groups' sums meet through LDS once, at the end.
// Both operands are K-contiguous and travel global -> LDS directly (global_load_lds_dwordx4, no
// registers and no LDS store instructions in between) in 64-wide slices of K, four LDS stages (three
// of a 256-column tile), one slice less ahead of the multiply; rows are unpadded and their 16-byte chunks XOR-swizzled by
// the choice of source address, so the b128 fragment reads are free of bank conflicts.  One
// workgroup barrier per slice.  Two more wavefronts do the loading: a CU's vector memory path takes 64 bytes per
// cycle, so the 32 KB of a 128 x 128 step keep it busy as long as the multiply takes, and a wavefront that
// issues a load into a full path stands still with its MFMAs behind it (the tiles of 256 columns, whose
// accumulators leave no registers for a third wavefront per SIMD, load for themselves).  The tile leaves
// through LDS as whole rows: 16-byte stores, and the residual is read the same way.
#include <type_traits>
#include <hip/hip_runtime.h>
#include "lbm_internal.h"
#include "qkv_math.h"

#pragma clang fp contract(off)

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;
typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(2))) unsigned short u16x2;
typedef __attribute__((ext_vector_type(2))) short s16x2;

constexpr int kGK = 128;         // K granularity the launches accept
constexpr int kGM = 128;         // activation rows per tile
constexpr int kGThreads = 512;
constexpr int kGLoadWaves = 2;       // wavefronts that load the operands
constexpr int kGTouchThreads = 64;   // and one that only asks for the next launch's lines
// (256 columns: the accumulators leave no registers for a third wavefront per SIMD)
constexpr int lbm_linear_threads(int tn) { return kGThreads + (tn == 256 ? 0 : kGLoadWaves * 64 + kGTouchThreads); }
constexpr int lbm_rows_threads(int tm) { return tm / 32 * 4 * 64 + (kGLoadWaves * 64 + kGTouchThreads); }   // lbm_linear_bf16_rows_kernel
constexpr int kKS = 64;          // K elements per LDS stage
constexpr int kStagesG = 4;      // LDS stages: three being loaded while one is multiplied (six stages for the 64-column tile,
                                 // which has the room: slower, 8.4 -> 8.8 us for proj - the longer prologue costs more than the depth gains)

// what a workgroup's first loads need, in one line of the scalar cache
struct LinearOperands {
  const unsigned short* a;       // [M, K]
  const unsigned short* w;       // [N, K]
  int M, N, K;
};
struct LinearArgs : LinearOperands, LbmTiles {
  const float* bias;             // [N] or null
  const float* gamma;            // [N] LayerScale (RESIDUAL only) or null
  const unsigned short* res;     // [M, N] residual (RESIDUAL only)
  unsigned short* out;           // [M, N]
  // LBM_LINEAR_QKV_PREPARE: the fused pre-attention producer as the epilogue of the qkv projection
  const float* q_norm_w;         // all four null: no qk-norm
  const float* q_norm_b;
  const float* k_norm_w;
  const float* k_norm_b;
  const float* rope_cs;
  unsigned short* k_out;         // out is q_out; k_out / v_out may be null
  unsigned short* v_out;
  unsigned short* pool;
  const int32_t* append_rows;    // null: nothing is appended
  float eps;
  float q_scale;                 // q rows are multiplied by this in fp32 before their last rounding (1 = plain q)
  int num_heads, page_size;
  // LNA kernels: the rows of the activations are standardised, (x - mean) * rstd, without ever
  // being rewritten: the product runs on the raw rows and the store applies
  // rstd * (a @ w^T - mean * colsum(w)) + bias.  The statistics come from the launch that
  // produced the activations (one (mean, M2) pair per row and column tile of that launch).
  const float* ln_colsum;        // [N]: sum over k of w[n][k]
  const float* ln_stats;         // [M][ln_tiles][2]
  int ln_tiles;
  float ln_eps;
  // LBM_LINEAR_BIAS_RESIDUAL: (mean, M2) of every output row over each 2^stats_shift columns,
  // [M][N >> stats_shift][2], or null
  float* stats_out;
  int stats_shift;               // 6 or 7; 6 where the tiles have 64 columns
  LbmTouch touch;                // what launches behind this one will read (lbm_linear_prefetch_hint)
  // SPLITK kernels: K summed in k_splits slices by as many workgroups per tile.  Every one
  // parks its fp32 partial tile in `split_part` and takes a ticket from the tile's counter; the
  // one that draws the last ticket sums the partials in slice order (the same sum whoever is
  // last) and runs the epilogue.  Counters start at zero and are left at zero.
  int k_splits;
  unsigned* split_counters;      // [m_tiles * n_tiles]
  float* split_part;             // [m_tiles * n_tiles][k_splits][8 waves][NT * 16][64 lanes]
};
constexpr int kEpiQkvPrepare = 3;   // internal: reached through lbm_qkv_linear_prepare only

__device__ __forceinline__ float round_bf16(float f) { return (float)(__bf16)f; }
__device__ __forceinline__ float bf16_bits_to_f32(unsigned v) { return __builtin_bit_cast(float, v << 16); }
// The GELU of the fused fc1 epilogue (torch's exact-erf nn.GELU, lingbot_map/layers/mlp.py:24) acts
// on a value already rounded to bf16 and is rounded to bf16 again: a function from 16 bits to
// 16 bits.  Evaluated per element it costs about 32 vector instructions, 4 us of a 20 us launch;
// instead it is tabulated for |v| in [2^-12, 2^3) - 15 binades x 128 mantissas x 2 signs, 7.5 KB,
// exact values rounded once (gen_gelu_table.py) - and each workgroup pulls the table into LDS with
// one 16-byte LDS-direct load per thread, ahead of its first operand tiles, and looks the
// elements up, sixteen per lane at a time (gelu_of), so that their lookups overlap.
// Outside the table the function has closed forms that agree with torch's fp32 evaluation
// after the rounding to bf16: below 2^-12, 1 + erf differs from 1 by less than 2^-12 and
// v / 2 is the nearest bf16 value (zeros and denormals included); from 8 up erff is exactly
// +-1, so the result is v on the positive side (+inf and NaN included) and v * 0 on the
// negative side (-0, and NaN for -inf and NaN, like 0.5 * v * (1 - 1)).  Between -8 and -3,
// where torch's 1 + erff cancels and its result carries the last bits of its erff, the table
// holds the exact value, within one bf16 step of torch's.
constexpr int kGeluE0 = 127 - 12;              // biased exponent of the first tabulated binade
constexpr int kGeluHalf = 15 * 128;            // entries per sign
constexpr int kGeluEntries = 2 * kGeluHalf;
static __device__ __attribute__((aligned(16))) const unsigned short g_gelu_table[kGeluEntries] = {
#include "gelu_table.inc"
};
// GELU of sixteen values (x, rounded to bf16 here), rounded to bf16, from the table copy in LDS.  Two values
// share a register from their rounding on: their indices are one packed computation, the two lookups land in
// the halves of the result, and what lies outside the table is patched afterwards, only by wavefronts
// that hold such a value - ten vector instructions per element where one value at a time took 21 (fc1 of
// 8,040 rows 78.0 -> 75.7 us, 4,016 rows 38.9 -> 37.9, 1,004 rows 14.7 -> 14.5).
// The index is the entry's byte offset, made without a compare or a select: seven per element (with the column
// vectors read once per column block: 8,032 rows 78.1 -> 75.7, 4,016 rows 39.3 -> 37.9, 1,004 rows 14.8 -> 14.7).
// Of the 5 us that GELU then costs a 256 x 256 tile the lookups' bank conflicts are two.  (The table at the bottom of
// LDS, the offset its whole address: another 0.4 us of a 256-row tile in a loop, but whole frames 0.1 to 0.3 % slower.)
template <int C>
__device__ __forceinline__ void gelu_of(const f32x4 (&x)[C], const unsigned short* tab, bf16x4 (&y)[C]) {
  // byte offsets of the table's entries: twice the magnitude's bits, the sign shifted out
  const u16x2 lo = (unsigned short)(kGeluE0 << 8), hi = (unsigned short)((kGeluE0 << 8) + 2 * (kGeluHalf - 1));
  u16x2 in[2 * C], out[2 * C], beyond = {0, 0};
#pragma unroll
  for (int i = 0; i < 2 * C; ++i) {
    unsigned pair = __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{x[i >> 1][(i & 1) * 2], x[i >> 1][(i & 1) * 2 + 1]}, bf16x2));
    asm("" : "+v"(pair));   // (or the signs are taken from x, one compare and one select each)
    in[i] = __builtin_bit_cast(u16x2, pair);
    const u16x2 mag = in[i] << (unsigned short)1;
    const u16x2 held = __builtin_elementwise_max(__builtin_elementwise_min(mag, hi), lo);
    beyond |= mag ^ held;
    unsigned neg = __builtin_bit_cast(unsigned, in[i] >> (unsigned short)15);
    asm("" : "+v"(neg));    // (or they are: 0 or 1, to multiply with)
    const u16x2 at = __builtin_bit_cast(u16x2, neg) * (unsigned short)(2 * kGeluHalf) + (held - lo);
    const char* const bytes = (const char*)tab;
    out[i] = u16x2{*(const unsigned short*)(bytes + at[0]), *(const unsigned short*)(bytes + at[1])};
  }
  if (__builtin_amdgcn_ballot_w64(__builtin_bit_cast(unsigned, beyond) != 0u)) {
    // outside the table: v / 2 below it, v or v * 0 above it (see kGeluE0)
#pragma unroll
    for (int i = 0; i < 2 * C; ++i)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const unsigned b16 = in[i][e], mag = b16 & 0x7fffu;
        const float v = bf16_bits_to_f32(b16);
        const float o = mag < (unsigned)(kGeluE0 << 7) ? 0.5f * v : ((b16 & 0x8000u) ? v * 0.0f : v);
        if (mag - (unsigned)(kGeluE0 << 7) >= (unsigned)kGeluHalf) out[i][e] = __builtin_bit_cast(unsigned short, (__bf16)o);
      }
  }
#pragma unroll
  for (int c = 0; c < C; ++c)
    y[c] = __builtin_bit_cast(bf16x4, u32x2{__builtin_bit_cast(unsigned, out[2 * c]), __builtin_bit_cast(unsigned, out[2 * c + 1])});
}

// ---- pieces that the kernels below share

// s_waitcnt vmcnt(N), the other counters untouched
#define LBM_DMA_WAIT(N) __builtin_amdgcn_s_waitcnt(0x0F70 | ((N) & 15) | (((N) >> 4) << 14))

// LNA: the statistics of a row, held by four neighbouring lanes that take every fourth (mean, M2) partial each;
// equal-sized partials merge as mean = avg(mean_i), M2 = sum(M2_i) + n_i * sum((mean_i - mean)^2) (Chan et
// al.), variance = M2 / K.  Returns (rstd, -mean * rstd).  The partials are asked for before the operand
// tiles (loads return in order) and merged while those travel.
constexpr int kLnHeld = 4;     // partials a lane keeps in registers (up to 16 column tiles)
__device__ __forceinline__ void ask_row_stats(const LinearArgs& p, int row, int part, f32x2 (&held)[kLnHeld]) {
  const float* st = p.ln_stats + (size_t)row * p.ln_tiles * 2;
#pragma unroll
  for (int i = 0; i < kLnHeld; ++i)
    if (part + 4 * i < p.ln_tiles) held[i] = *(const f32x2*)(st + 2 * (part + 4 * i));
}
__device__ __forceinline__ f32x2 merge_row_stats(const LinearArgs& p, int row, int part, const f32x2 (&held)[kLnHeld]) {
  const float* st = p.ln_stats + (size_t)row * p.ln_tiles * 2;
  float sm = 0.f;
#pragma unroll
  for (int i = 0; i < kLnHeld; ++i)
    if (part + 4 * i < p.ln_tiles) sm += held[i][0];
  for (int i = part + 4 * kLnHeld; i < p.ln_tiles; i += 4) sm += st[2 * i];
  sm += lbm_qkv::lane_xor1(sm);
  sm += lbm_qkv::lane_xor2(sm);
  const float mean = sm / (float)p.ln_tiles;
  const float n_i = (float)p.K / (float)p.ln_tiles;
  float m2 = 0.f;
#pragma unroll
  for (int i = 0; i < kLnHeld; ++i)
    if (part + 4 * i < p.ln_tiles) {
      const float d = held[i][0] - mean;
      m2 += held[i][1] + n_i * d * d;
    }
  for (int i = part + 4 * kLnHeld; i < p.ln_tiles; i += 4) {
    const float d = st[2 * i] - mean;
    m2 += st[2 * i + 1] + n_i * d * d;
  }
  m2 += lbm_qkv::lane_xor1(m2);
  m2 += lbm_qkv::lane_xor2(m2);
  const float rstd = __builtin_amdgcn_rsqf(m2 / (float)p.K + p.ln_eps);
  return f32x2{rstd, -mean * rstd};
}

// Everything that a launch reads of its arguments, asked for at its start and at once.  In a model each launch finds them in no
// cache, and every line of them that is first read where it is needed - the epilogue's pointers, the statistics' behind
// the tile's - is a trip to memory of its own (frames, ms: 86 rows 2.73 -> 2.69, 261 rows 3.17 -> 3.13, 577 rows 4.56 -> 4.47, 1,004 rows
// 6.40 -> 6.32, four streams 15.10 -> 14.97; nothing in a loop over few launches).
template <int EPI, bool LNA, bool NORM>
__device__ __forceinline__ void hold_arguments(const LinearArgs& p) {
  constexpr bool res = EPI == LBM_LINEAR_BIAS_RESIDUAL, qkv = EPI == kEpiQkvPrepare;
  asm volatile("" : : "s"(p.a), "s"(p.w), "s"(p.M), "s"(p.N), "s"(p.K), "s"(p.m_tiles), "s"(p.n_tiles), "s"(p.panel_shift), "s"(p.last_width), "s"(p.per_panel),
               "s"(p.per_last), "s"(p.bias), "s"(p.out), "s"(res ? p.res : nullptr), "s"(res ? p.gamma : nullptr), "s"(res ? p.stats_out : nullptr),
               "s"(LNA ? p.ln_colsum : nullptr), "s"(LNA ? p.ln_stats : nullptr), "s"(LNA ? p.ln_tiles : 0), "s"(qkv ? p.rope_cs : nullptr), "s"(qkv ? p.k_out : nullptr),
               "s"(qkv ? p.pool : nullptr), "s"(qkv ? p.append_rows : nullptr), "s"(qkv ? p.num_heads : 0), "s"(qkv && NORM ? p.q_norm_w : nullptr));
}

// residual + branch, eight bf16 values
__device__ __forceinline__ u32x4 add_rows(u32x4 x, u32x4 v) {
  u32x4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float s0 = bf16_bits_to_f32(x[e] & 0xffffu) + bf16_bits_to_f32(v[e] & 0xffffu);
    const float s1 = bf16_bits_to_f32(x[e] >> 16) + bf16_bits_to_f32(v[e] >> 16);
    o[e] = (unsigned)__builtin_bit_cast(unsigned short, (__bf16)s0) | ((unsigned)__builtin_bit_cast(unsigned short, (__bf16)s1) << 16);
  }
  return o;
}

// (mean, M2) of a row's stored values (v: this lane's eight, from column col on), 64 or 128 columns at a
// time (shift 6 or 7): the 8 or 16 lanes that hold them are neighbours
__device__ __forceinline__ void store_row_stats(const LinearArgs& p, u32x4 v, int row, int col, int shift, int lane) {
  float x[8];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    x[2 * e] = bf16_bits_to_f32(v[e] & 0xffffu);
    x[2 * e + 1] = bf16_bits_to_f32(v[e] >> 16);
  }
  float sm = ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
  sm = lbm_qkv::sum_of_8(sm);
  if (shift == 7) sm += lbm_qkv::other_half_of_16(sm);
  const float mean = sm * (shift == 7 ? 1.0f / 128 : 1.0f / 64);
  float m2 = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) m2 += (x[e] - mean) * (x[e] - mean);
  m2 = lbm_qkv::sum_of_8(m2);
  if (shift == 7) m2 += lbm_qkv::other_half_of_16(m2);
  if (row < p.M && (lane & ((1 << (shift - 3)) - 1)) == 0) {
    float* so = p.stats_out + ((size_t)row * (p.N >> shift) + (col >> shift)) * 2;
    so[0] = mean;
    so[1] = m2;
  }
}

// The pre-attention producer on eight consecutive columns of the projection's output, rounded to bf16 (raw):
// the lanes of a (token, q|k|v, head) row of 64 are eight neighbours, exactly the producer's layout, so its
// LayerNorm, rotary embedding and scatter run on the tile as it leaves instead of in a pass of their own
// (lingbot_map/layers/attention.py:402-426, rope.py:438-461, flashinfer_cache.py:215-218).
template <int ROPE>
__device__ __forceinline__ void ask_rotary(const LinearArgs& p, int token, int c8, lbm_qkv::f32x4 (&cs)[4]) {
  if (ROPE == 1) {
    const lbm_qkv::f32x4* src = (const lbm_qkv::f32x4*)(p.rope_cs + ((long long)token * 32 + c8 * 4) * 2);
    cs[0] = src[0]; cs[1] = src[1];
  } else if (ROPE == 2) {
    const lbm_qkv::f32x4* src = (const lbm_qkv::f32x4*)(p.rope_cs + ((long long)token * 64 + c8 * 8) * 2);
    cs[0] = src[0]; cs[1] = src[1]; cs[2] = src[2]; cs[3] = src[3];
  }
}
template <int ROPE, bool NORM, bool READY = false>
__device__ __forceinline__ bf16x8 produce_row(u32x4 raw, int which, int c8, const lbm_qkv::f32x4 (&w4)[2], const lbm_qkv::f32x4 (&b4)[2],
                                              const lbm_qkv::f32x4 (&cs)[4], float eps, float post) {
  bf16x8 o8 = __builtin_bit_cast(bf16x8, raw);   // v rows leave as they are
  if (which < 2) {
    // q and k rows: the row's last rounding is the conversion that packs it
    float x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = __builtin_bit_cast(float, (i & 1) ? (raw[i >> 1] & 0xffff0000u) : (raw[i >> 1] << 16));
    lbm_qkv::norm_rope_unrounded<0, ROPE, NORM, READY>(x, w4, b4, cs, c8, eps, post);
#pragma unroll
    for (int i = 0; i < 8; ++i) o8[i] = (__bf16)x[i];
  }
  return o8;
}
__device__ __forceinline__ unsigned short* produced_rows(const LinearArgs& p, int which) { return which == 0 ? p.out : (which == 1 ? p.k_out : p.v_out); }
__device__ __forceinline__ void store_produced(const LinearArgs& p, unsigned short* plain, bf16x8 o8, int which, int token, int head, int c8, int pool_row) {
  const int H = p.num_heads;
  const long long nhd = ((long long)token * H + head) * 64 + c8 * 8;
  if (plain) lbm_store_through(plain + nhd, __builtin_bit_cast(u32x4, o8));
  if (which > 0 && pool_row >= 0) {
    const long long row_elems = (long long)H * 64;
    const long long d = (long long)pool_row * row_elems + (which == 2 ? (long long)p.page_size * row_elems : 0) + head * 64 + c8 * 8;
    lbm_store_through(p.pool + d, __builtin_bit_cast(u32x4, o8));
  }
}

// TN: output columns per tile (256, 128 or 64); a wavefront owns 64 x (TN / 2) of the tile.  Every
// output element is the same sum in the same order whatever TN is: they give the same bits.
// 256: bound by the multiply (a 64-wide step moves 48 KB for 1,024 cycles of MFMA, where 128 columns move 32 KB
// for 512); three stages, and no wavefronts beside the computing ones.
// ROPE / NORM: rotary layout (0 none, 1 interleaved, 2 half-split) and qk-LayerNorm of the
// kEpiQkvPrepare epilogue; 0 / false otherwise.
// LNA: the activations' rows are standardised by the store (see LinearArgs).
// SPLITK: several workgroups per tile, each over a slice of K (see LinearArgs).
template <int EPI, int TN, int ROPE = 0, bool NORM = false, bool LNA = false, bool SPLITK = false>
__global__ __launch_bounds__(lbm_linear_threads(TN), 1) void lbm_linear_bf16_kernel(LinearArgs p) {
  constexpr int NT = TN / 64;   // 32-column blocks of W per wavefront
  constexpr int kStages = TN == 256 ? kStagesG - 1 : kStagesG;
  // [stage][row][64]: 64-wide slices of K, kStages of them in flight or in use
  __shared__ __attribute__((aligned(16))) unsigned short lds_ops[kStages * (kGM + TN) * kKS];
  unsigned short (*const lds_a)[kGM * kKS] = (unsigned short (*)[kGM * kKS])lds_ops;
  unsigned short (*const lds_w)[TN * kKS] = (unsigned short (*)[TN * kKS])(lds_ops + kStages * kGM * kKS);
  __shared__ __attribute__((aligned(16))) unsigned short gelu_tab[EPI == LBM_LINEAR_BIAS_GELU ? kGeluEntries : 8];
  __shared__ __attribute__((aligned(8))) float ln_rows[LNA ? kGM * 2 : 2];   // per row of the tile: rstd, -mean * rstd
  __shared__ __attribute__((aligned(16))) float colvec[3][TN];               // bias, column sums of w (LNA), LayerScale

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  hold_arguments<EPI, LNA, NORM>(p);
  const int n32 = lane & 31, g = lane >> 5;
  const int kh = wave >> 2, ws = wave & 3;    // k half of this wave's group, its sub-tile
  // Workgroups are dealt to the 8 XCDs round-robin: an XCD keeps its own column tiles of W (read
  // from HBM once, by it alone) and walks all row tiles of the activations with them.
  // (the workgroups that share a tile under SPLITK land on the same XCD as well)
  int mt, nt, split = 0;
  {
    const int n_tiles_all = p.m_tiles * p.n_tiles;
    if (!SPLITK) {
      lbm_tile_of_workgroup((int)blockIdx.x, p, mt, nt);
    } else if ((p.n_tiles & 7) == 0) {
      const int x = blockIdx.x & 7;
      int i = blockIdx.x >> 3;
      split = i / (n_tiles_all >> 3);
      i -= split * (n_tiles_all >> 3);
      mt = i % p.m_tiles;
      nt = (i / p.m_tiles) * 8 + x;
    } else {
      int i = (int)blockIdx.x;
      if (SPLITK) {
        split = i / n_tiles_all;
        i -= split * n_tiles_all;
      }
      mt = i % p.m_tiles;
      nt = i / p.m_tiles;
    }
  }
  const int m0 = mt * kGM, n0 = nt * TN;
  const int wm = (ws & 1) * 64, wn = (ws >> 1) * (TN / 2);

  // ---- staging.  Operands travel global -> LDS without passing through registers
  // (global_load_lds_dwordx4: a wavefront's 64 lanes x 16 bytes land as one contiguous KB, i.e.
  // eight whole 128-byte rows of a 64-wide K slice; wavefront w covers rows 8 w .. 8 w + 7 of every
  // block of 64 rows).  Rows are not padded; instead the 16-byte chunk c of row r sits at chunk
  // position c ^ ((r >> 1) & 7), which the lane arranges by asking for the chunk that belongs at
  // ITS position - then the b128 fragment reads of 16 rows at one logical chunk hit all 64 banks.
  constexpr int kPassA = kGM / 64, kPassW = TN / 64;
  const int ld_r = wave * 8 + (lane >> 3);                                   // row within a block of 64
  const unsigned sw_c = (unsigned)(((lane & 7) ^ ((ld_r >> 1) & 7)) * 8);    // logical element offset this lane fetches
  unsigned a_off[kPassA];
#pragma unroll
  for (int j = 0; j < kPassA; ++j) a_off[j] = ((unsigned)min(m0 + ld_r + 64 * j, p.M - 1) * (unsigned)p.K + sw_c) * 2u;   // rows past M re-read the last row
  const unsigned w_off = ((unsigned)ld_r * (unsigned)p.K + sw_c) * 2u;
  const int nk = (SPLITK ? p.K / p.k_splits : p.K) / kKS;   // 64-wide steps of this workgroup
  const size_t k_first = SPLITK ? (size_t)split * nk * kKS : 0;
  const char* a_base = (const char*)(p.a + k_first);
  const char* w_base = (const char*)(p.w + (size_t)n0 * p.K + k_first);
  constexpr bool kLoaders = TN != 256;
  // (blockIdx.y is a scalar register: nothing is loaded to know)
  if (blockIdx.y || wave >= kGThreads / 64 + kGLoadWaves) {
    lbm_touch(p.touch, lbm_linear_threads(TN), true);
    return;
  }
  if (kLoaders && wave >= kGThreads / 64) {
    // A loading wavefront: every second KB - eight rows - of each step's operands.  The rows of a step are waited
    // for before the barrier that the computing wavefronts read them behind, and asked for behind the one that
    // frees their stage.  (M x N x K 1,004 x 3,072 x 1,024: 13.0 us with every wavefront loading its rows between
    // its own MFMAs, 11.8 with these; 1,004 x 4,096 x 1,024 + GELU 14.7 -> 13.4; 4,016 x 1,024 x 4,096 35.6 -> 34.0.)
    const int par = wave - kGThreads / 64, l8 = lane >> 3;
    constexpr int kUnitsA = kGM / 16, kLoads = kUnitsA + TN / 16;
    const unsigned chunk = (unsigned)(((lane & 7) ^ (4 * par + (lane >> 4))) * 8);   // rows 8 (2 u + par) + l8: bits 1 .. 3
    unsigned off[kLoads];
#pragma unroll
    for (int u = 0; u < kLoads; ++u) {
      const int row = u < kUnitsA ? min(m0 + 8 * (2 * u + par) + l8, p.M - 1) : 8 * (2 * (u - kUnitsA) + par) + l8;
      off[u] = ((unsigned)row * (unsigned)p.K + chunk) * 2u;
    }
    const unsigned lds_first = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(__attribute__((address_space(3))) unsigned short*)&lds_ops[0]) + (unsigned)par * 1024u;
    auto load_step = [&](int s) {
      const unsigned st = (unsigned)(s % kStages);
      const unsigned at_a = lds_first + st * (kGM * kKS * 2), at_w = lds_first + (kStages * kGM + st * TN) * (kKS * 2);
#pragma unroll
      for (int u = 0; u < kLoads; ++u) {
        const char* base = (u < kUnitsA ? a_base : w_base) + (size_t)s * (kKS * 2);
        const unsigned at = u < kUnitsA ? at_a + u * 2048u : at_w + (u - kUnitsA) * 2048u;
        asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off[u]), "s"(base), "s"(at) : "memory", "m0");
      }
    };
    __builtin_amdgcn_s_setprio(3);     // few instructions, and everybody waits for them
#pragma unroll
    for (int s = 0; s < kStages; ++s)
      if (s < nk) load_step(s);
    for (int s = -1; s < nk; ++s) {    // the barrier at the top of step s publishes the rows of step s + 1
      const int behind = nk - 2 - s;   // steps asked for behind those
      if (s < 0 && behind >= 3) LBM_DMA_WAIT(3 * kLoads);
      else if (behind >= 2) LBM_DMA_WAIT(2 * kLoads);
      else if (behind == 1) LBM_DMA_WAIT(kLoads);
      else LBM_DMA_WAIT(0);
      __builtin_amdgcn_s_barrier();
      if (s >= 0 && s + kStages < nk) load_step(s + kStages);
    }
    return;
  }
  // The loads are written as inline assembly: the compiler would otherwise wait for every
  // LDS-direct load in flight before any LDS read that might alias it (it cannot tell the two
  // buffers apart), which serialises load and multiply.  M0 carries the LDS address of the
  // wavefront's KB (declared as clobbered, so the compiler keeps nothing of its own in M0 across
  // the load).  The waits for these loads are placed
  // by hand (dma_wait) - the compiler's own counts only see fewer loads in flight than there
  // are, which makes its waits stricter, never laxer.
  auto dma_row = [&](const char* base, unsigned voff, const unsigned short* lds_dst) {
    const unsigned m0v = (unsigned)(size_t)(__attribute__((address_space(3))) const void*)lds_dst;
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1"
                 :
                 : "v"(voff), "s"(base), "s"(__builtin_amdgcn_readfirstlane(m0v))
                 : "memory", "m0");
  };
  auto dma_step = [&](int ks, int stage) {
#pragma unroll
    for (int j = 0; j < kPassA; ++j)
      dma_row(a_base + ks * (kKS * 2), a_off[j], &lds_a[stage][(64 * j + 8 * wave) * kKS]);
#pragma unroll
    for (int j = 0; j < kPassW; ++j)
      dma_row(w_base + ((size_t)(64 * j) * p.K + (size_t)ks * kKS) * 2, w_off, &lds_w[stage][(64 * j + 8 * wave) * kKS]);
  };
  // the same loads one by one, for the loop: M0 values and row offsets as integers, so that
  // nothing but two scalar adds and the load itself sits between the MFMAs
  const unsigned m0_a = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(__attribute__((address_space(3))) unsigned short*)&lds_a[0][0] + (unsigned)wave * 1024u);
  const unsigned m0_w = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(__attribute__((address_space(3))) unsigned short*)&lds_w[0][0] + (unsigned)wave * 1024u);
  unsigned w_offs[kPassW];
#pragma unroll
  for (int j = 0; j < kPassW; ++j) w_offs[j] = w_off + (unsigned)(64 * j) * (unsigned)p.K * 2u;
  auto dma_one = [&](int ks, int stage, int j) {
    const char* base = (j < kPassA ? a_base : w_base) + (size_t)ks * (kKS * 2);
    const unsigned voff = j < kPassA ? a_off[j < kPassA ? j : 0] : w_offs[j < kPassA ? 0 : j - kPassA];
    const unsigned m0v = j < kPassA ? m0_a + (unsigned)(stage * kGM * kKS * 2 + 64 * j * kKS * 2)
                                    : m0_w + (unsigned)(stage * TN * kKS * 2 + 64 * (j - kPassA) * kKS * 2);
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(voff), "s"(base), "s"(m0v) : "memory", "m0");
  };
  constexpr int kDmaPerStep = kPassA + kPassW;

  f32x16 acc[NT][2];   // [column block of W][row block of A]; element i: column 8 (i / 4) + 4 g + i % 4, row n32
#pragma unroll
  for (int a = 0; a < NT; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[a][b][i] = 0.f;

  // One 64-wide step: each wave group multiplies its 32-wide half.  The fragments of a step are
  // read during the step before it, one read in between two MFMAs (a burst of reads fills the LDS
  // queue and holds the MFMAs behind it back), into the other half of the fragment registers.
  const int sw_r = (n32 >> 1) & 7;
  bf16x8 wf[2][2][NT], af[2][2][2];   // [step parity][16-wide slice][block]
  auto read_one = [&](int stage, int buf, int i) {   // read i of a step's 2 (NT + 2), in the order the MFMAs use them
    const unsigned short* la = &lds_a[stage][0];
    const unsigned short* lw = &lds_w[stage][0];
    const int k16 = i / (NT + 2), j = i % (NT + 2);
    const int pos = ((kh * 4 + k16 * 2 + g) ^ sw_r) * 8;
    if (j == 0) wf[buf][k16][0] = __builtin_bit_cast(bf16x8, *(const u32x4*)&lw[(wn + n32) * kKS + pos]);
    else if (j <= 2) af[buf][k16][j - 1] = __builtin_bit_cast(bf16x8, *(const u32x4*)&la[(wm + ((j - 1) ^ kh) * 32 + n32) * kKS + pos]);
    else wf[buf][k16][j - 2] = __builtin_bit_cast(bf16x8, *(const u32x4*)&lw[(wn + (j - 2) * 32 + n32) * kKS + pos]);
  };
  auto read_slice = [&](int stage, int buf, int k16) {
#pragma unroll
    for (int i = 0; i < NT + 2; ++i) read_one(stage, buf, k16 * (NT + 2) + i);
  };
  auto read_step = [&](int stage, int buf) {
    read_slice(stage, buf, 0);
    read_slice(stage, buf, 1);
  };
  auto mfma_slice = [&](int buf, int k16) {
#pragma unroll
    for (int a = 0; a < NT; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
        acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[buf][k16][a], af[buf][k16][b], acc[a][b], 0, 0, 0);
  };

  // LNA, row statistics: row r of the tile is handled by threads 4 r .. 4 r + 3
  f32x2 ln_part[kLnHeld] = {};
  if (LNA) ask_row_stats(p, min(m0 + (tid >> 2), p.M - 1), tid & 3, ln_part);
  // The per-column vectors of the epilogue (bias, column sums of w, LayerScale) are asked for now
  // and parked in LDS behind the first operand loads; the loop's barriers publish them.
  float cv_bias = 0.f, cv_sum = 0.f, cv_gamma = 1.f;
  if (tid < TN) {
    if (p.bias) cv_bias = p.bias[n0 + tid];
    if (LNA) cv_sum = p.ln_colsum[n0 + tid];
    if (EPI == LBM_LINEAR_BIAS_RESIDUAL && p.gamma) cv_gamma = p.gamma[n0 + tid];
  }
  // The GELU table travels first (480 threads x 16 bytes; the loads return in order, so the wait
  // for the first operand tile covers it and the barrier behind that wait publishes it) ...
  if (EPI == LBM_LINEAR_BIAS_GELU && tid < kGeluEntries / 8)
    dma_row((const char*)g_gelu_table, (unsigned)tid * 16u, &gelu_tab[wave * 512]);
  // ... then the first steps of the tiles that load for themselves
#pragma unroll
  for (int i = 0; i < kStages - 1; ++i)
    if (!kLoaders && i < nk) dma_step(i, i);
  if (tid < TN) {
    colvec[0][tid] = cv_bias;
    colvec[1][tid] = cv_sum;
    colvec[2][tid] = cv_gamma;
  }
  if (LNA) {   // (read in the epilogue, many barriers from here)
    const f32x2 row = merge_row_stats(p, min(m0 + (tid >> 2), p.M - 1), tid & 3, ln_part);
    if ((tid & 3) == 0) *(f32x2*)&ln_rows[2 * (tid >> 2)] = row;
  }
  // Step 0's fragments: its rows have landed (later steps may still be in flight), barrier, read.
  LBM_DMA_WAIT(kLoaders ? 0 : kDmaPerStep);   // (0: the GELU table)
  __syncthreads();
  read_step(0, 0);
  if (!kLoaders && kStages - 1 < nk) dma_step(kStages - 1, kStages - 1);
  // Step s: the rows of step s + 1 have landed (whoever loads them waits until only the loads of steps
  // s + 2 and, with four stages, s + 3 are in flight), barrier (everyone's rows of step s + 1 are there, and everyone
  // holds the fragments of step s in registers, so its stage is free), then the MFMAs of step s with the
  // fragment reads of step s + 1 in between; the loads of step s + kStages go into the freed stage.
  static_assert(kStages == 4 || kStages == 3, "the waits below are written for a ring of three or four stages");
  constexpr int kUnroll = kStages == 4 ? 4 : 6;   // whole rounds of the ring and of the two fragment buffers
#define LBM_SGB(mask, n) __builtin_amdgcn_sched_group_barrier(mask, n, 0)
  for (int s0 = 0; s0 < nk; s0 += kUnroll) {
#pragma unroll
    for (int st = 0; st < kUnroll; ++st) {
      const int sidx = s0 + st;
      if (sidx < nk) {
        if (!kLoaders) {
          if (sidx + 2 < nk) LBM_DMA_WAIT(kDmaPerStep);
          else LBM_DMA_WAIT(0);
        }
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        const bool more = !kLoaders && sidx + kStages < nk;
#pragma unroll
        for (int k16 = 0; k16 < 2; ++k16) {
          read_slice((st + 1) % kStages, (st + 1) & 1, k16);   // (past the last step: stale rows, never used)
          mfma_slice(st & 1, k16);
#pragma unroll
          for (int i = 0; i < NT + 2; ++i) { LBM_SGB(0x008, 1); LBM_SGB(0x100, 1); }
          if (NT == 4) LBM_SGB(0x008, 2);
          __builtin_amdgcn_sched_barrier(0);
          if (more) {
#pragma unroll
            for (int j = 0; j < kDmaPerStep; ++j)
              if (j * 2 / kDmaPerStep == k16) dma_one(sidx + kStages, st % kStages, j);
          }
        }
      }
    }
  }
#undef LBM_SGB
  __syncthreads();

  // What the epilogue needs from global memory beyond the per-column vectors is asked for here,
  // all at once, and arrives while the wave groups exchange their sums (asked for where it is
  // used - per pass - every load would wait out a trip to L2 or HBM on its own, and behind the
  // stores of the pass before it; asked for before the multiply, it delays the first operand
  // tiles):
  // the residual rows of the store passes (a workgroup that shares its tile under SPLITK
  // asks only once it knows that it is the one to store).
  constexpr int kPieces = TN / 8;                 // 16-byte pieces per row of the tile
  constexpr int kRowsPerPass = kGThreads / kPieces;
  constexpr int kPasses = kGM / kRowsPerPass;
  u32x4 res_v[kPasses] = {};
  auto load_residual = [&]() {
#pragma unroll
    for (int j = 0; j < kPasses; ++j) {
      const int row = min(m0 + j * kRowsPerPass + tid / kPieces, p.M - 1);   // rows past M: read, never stored
      res_v[j] = *(const u32x4*)(p.res + (size_t)row * p.N + n0 + (tid % kPieces) * 8);
    }
  };
  if (EPI == LBM_LINEAR_BIAS_RESIDUAL && !SPLITK) load_residual();
  // The producer's own inputs - q/k norm weights, every pass's rotary table entries and pool rows -
  // are asked for now as well.
  const int H = p.num_heads;
  // 256 columns, four heads of q, k or v: the eight lanes of a head's row work on those columns of all four of a token, one set of
  // entries for the four (the registers hold no more: the second of the tile's two passes asks for its own when it comes)
  // (without norm and table rows of 512 bytes leave faster, as in the kernel below).
  constexpr bool kByToken = EPI == kEpiQkvPrepare && TN == 256 && (ROPE != 0 || NORM);
  constexpr int kTokens = kByToken ? kGM / 64 : kPasses, kRotary = kByToken ? 1 : kPasses;
  struct {
    int c, which, h, c8;
    lbm_qkv::f32x4 w4[2], b4[2], cs4[kRotary][4];
    int pool_row[kTokens];
  } pq = {};
  auto token_of = [&](int j) { return min(m0 + (kByToken ? j * 64 + (tid >> 3) : j * kRowsPerPass + tid / kPieces), p.M - 1); };
  if (EPI == kEpiQkvPrepare) {
    typedef lbm_qkv::f32x4 qf4;
    pq.c = kByToken ? (tid & 7) * 8 : (tid % kPieces) * 8;
    const int col = n0 + pq.c;                    // column of the projection: [q|k|v][head][64]
    pq.which = col / (H * 64);                    // uniform over the workgroup (H * 64 is a multiple of TN)
    pq.h = (col - pq.which * H * 64) >> 6;
    pq.c8 = (col & 63) >> 3;                      // = tid % 8: the lane's place in its row of 64
    if (NORM && pq.which < 2) {
      const qf4* wp = (const qf4*)((pq.which == 0 ? p.q_norm_w : p.k_norm_w) + pq.c8 * 8);
      const qf4* bp = (const qf4*)((pq.which == 0 ? p.q_norm_b : p.k_norm_b) + pq.c8 * 8);
      pq.w4[0] = wp[0]; pq.w4[1] = wp[1];
      pq.b4[0] = bp[0]; pq.b4[1] = bp[1];
    }
#pragma unroll
    for (int j = 0; j < kTokens; ++j) {
      const int t = token_of(j);
      if (pq.which < 2 && j < kRotary) ask_rotary<ROPE>(p, t, pq.c8, pq.cs4[j]);
      pq.pool_row[j] = -1;
      if (pq.which > 0 && p.append_rows) pq.pool_row[j] = p.append_rows[t];
    }
  }
  // ---- the two wave groups' sums meet: group 0 finishes row block 0 of every sub-tile, group 1
  // row block 1; each parks the other's half in LDS (the operand buffers are dead)
  float* xch = (float*)&lds_a[0][0];            // [wave][NT][4][64 lanes][4] floats
  static_assert(8 * NT * 16 * 64 * 4 <= (NT == 4 ? kStages * (kGM + TN) : kStages * kGM) * kKS * 2,
                "the exchanged halves fit the activation buffers (256 columns: all operand buffers)");
  // (the second wave group reads its activation fragments with the two row blocks swapped, so
  // for both groups acc[.][0] is the block they finish and acc[.][1] the one they hand over)
  f32x16 fin[NT];
  {
#pragma unroll
    for (int a = 0; a < NT; ++a)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        f32x4 give;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          give[e] = acc[a][1][q * 4 + e];
          fin[a][q * 4 + e] = acc[a][0][q * 4 + e];
        }
        *(f32x4*)&xch[(((wave * NT + a) * 4 + q) * 64 + lane) * 4] = give;
      }
    // (a barrier that waits for the LDS writes only: the loads asked for above stay in flight)
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const int peer = wave ^ 4;
#pragma unroll
    for (int a = 0; a < NT; ++a)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4 got = *(const f32x4*)&xch[(((peer * NT + a) * 4 + q) * 64 + lane) * 4];
#pragma unroll
        for (int e = 0; e < 4; ++e) fin[a][q * 4 + e] += got[e];
      }
    // (256 columns: the tile is staged below where the halves were exchanged)
    if (NT == 4) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  }
  const int b = kh;     // the row block this wave finishes
  if (SPLITK) {
    // Partials and counters travel as scope-qualified relaxed atomics, which go past the caches
    // that are not coherent between workgroups (the CU's and, between XCDs, the L2) - a
    // device-wide fence would write back and invalidate the whole L2 instead, once per
    // workgroup (measured: 60 us on a 25 us launch).  Order: every thread waits until its own
    // stores are acknowledged (an explicit s_waitcnt vmcnt(0): the stores are write-through, so an
    // acknowledged store is visible device-wide, and a workgroup-scope fence alone does not wait
    // for it), the barrier collects all threads, only then thread 0 draws the ticket.
    __shared__ unsigned ticket_lds;
    const int tile = mt * p.n_tiles + nt;
    constexpr int kPartFloats = 8 * NT * 16 * 64;                 // one workgroup's partial tile
    float* tile_part = p.split_part + (size_t)tile * p.k_splits * kPartFloats;
    float* mine = tile_part + (size_t)split * kPartFloats + (size_t)wave * (NT * 16 * 64);
#pragma unroll
    for (int a = 0; a < NT; ++a)
#pragma unroll
      for (int i = 0; i < 16; ++i)
        __hip_atomic_store(&mine[(a * 16 + i) * 64 + lane], fin[a][i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    LBM_DMA_WAIT(0);
    __syncthreads();
    if (tid == 0) ticket_lds = __hip_atomic_fetch_add(&p.split_counters[tile], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (ticket_lds != (unsigned)(p.k_splits - 1)) return;          // (uniform over the workgroup)
    if (tid == 0) __hip_atomic_store(&p.split_counters[tile], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // as the next launch expects it
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    if (EPI == LBM_LINEAR_BIAS_RESIDUAL) load_residual();
    // two slices: this workgroup's own sum is still in its registers and a + b = b + a; more
    // slices: all of them from memory, in slice order, so the sum does not depend on who is last
    const bool pair = p.k_splits == 2;
    if (!pair) {
#pragma unroll
      for (int a = 0; a < NT; ++a)
#pragma unroll
        for (int i = 0; i < 16; ++i) fin[a][i] = 0.f;
    }
    for (int sidx = pair ? 1 - split : 0; sidx < (pair ? 2 - split : p.k_splits); ++sidx) {
      const float* src = tile_part + (size_t)sidx * kPartFloats + (size_t)wave * (NT * 16 * 64);
#pragma unroll
      for (int a = 0; a < NT; ++a)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          fin[a][i] += __hip_atomic_load(&src[(a * 16 + i) * 64 + lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }

  // ---- epilogue.  In registers: + bias, round (the linear's output), GELU or LayerScale, round.
  // Then the tile goes through LDS and leaves as whole rows.
  constexpr int kCStride = TN + 4;   // bf16 per staged row: 8-byte writes of 32 rows hit 64 distinct banks
  unsigned short* stage = (unsigned short*)&lds_w[0][0];
  f32x2 row_f = {1.f, 0.f};   // this lane's output row: rstd, -mean * rstd
  if (LNA) row_f = *(const f32x2*)&ln_rows[2 * (wm + b * 32 + n32)];
  static_assert(kGM * kCStride <= kStages * TN * kKS, "the staged tile fits the weight buffers");
#pragma unroll
  for (int a = 0; a < NT; ++a) {
    f32x4 x[4];     // [c4]: columns wn + a * 32 + c4 * 8 + g * 4 and the three behind it
    bf16x4 y[4];
#pragma unroll
    for (int c4 = 0; c4 < 4; ++c4) {
      const int col = wn + a * 32 + c4 * 8 + g * 4;
      const f32x4 bias4 = *(const f32x4*)&colvec[0][col], colsum4 = *(const f32x4*)&colvec[1][col];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float lin = fin[a][c4 * 4 + e];
        if (LNA) lin = __builtin_fmaf(lin, row_f[0], row_f[1] * colsum4[e]);   // rstd * acc - mean * rstd * colsum
        x[c4][e] = lin + bias4[e];
      }
      if (EPI == LBM_LINEAR_BIAS_RESIDUAL && p.gamma) {
        const f32x4 gamma4 = *(const f32x4*)&colvec[2][col];
#pragma unroll
        for (int e = 0; e < 4; ++e) x[c4][e] = round_bf16(x[c4][e]) * gamma4[e];
      }
      y[c4] = __builtin_convertvector(x[c4], bf16x4);
    }
    if (EPI == LBM_LINEAR_BIAS_GELU) gelu_of<4>(x, gelu_tab, y);
#pragma unroll
    for (int c4 = 0; c4 < 4; ++c4)
      *(bf16x4*)&stage[(wm + b * 32 + n32) * kCStride + wn + a * 32 + c4 * 8 + g * 4] = y[c4];
  }
  __syncthreads();
  if (EPI == kEpiQkvPrepare) {
    unsigned short* const plain = produced_rows(p, pq.which);
    if (kByToken) {
#pragma unroll
      for (int j = 0; j < kTokens; ++j) {
        const int r = j * 64 + (tid >> 3);
        if (j > 0 && pq.which < 2) ask_rotary<ROPE>(p, token_of(j), pq.c8, pq.cs4[0]);
        if (pq.which < 2) lbm_qkv::ready_rotary<ROPE>(pq.cs4[0], pq.c8);
#pragma unroll
        for (int s = 0; s < TN / 64; ++s) {
          const u32x2 lo = *(const u32x2*)&stage[r * kCStride + s * 64 + pq.c], hi = *(const u32x2*)&stage[r * kCStride + s * 64 + pq.c + 4];
          const bf16x8 o8 = produce_row<ROPE, NORM, true>(u32x4{lo[0], lo[1], hi[0], hi[1]}, pq.which, pq.c8, pq.w4, pq.b4, pq.cs4[0], p.eps, pq.which == 0 ? p.q_scale : 1.0f);
          if (m0 + r < p.M) store_produced(p, plain, o8, pq.which, m0 + r, pq.h + s, pq.c8, pq.pool_row[j]);
        }
      }
      return;
    }
#pragma unroll
    for (int j = 0; j < kPasses; ++j) {
      const int r = j * kRowsPerPass + tid / kPieces;
      const u32x2 lo = *(const u32x2*)&stage[r * kCStride + pq.c], hi = *(const u32x2*)&stage[r * kCStride + pq.c + 4];
      // (rows past M are computed on the last token's entries and never stored)
      const bf16x8 o8 = produce_row<ROPE, NORM>(u32x4{lo[0], lo[1], hi[0], hi[1]}, pq.which, pq.c8, pq.w4, pq.b4, pq.cs4[kByToken ? 0 : j], p.eps, pq.which == 0 ? p.q_scale : 1.0f);
      if (m0 + r < p.M) store_produced(p, plain, o8, pq.which, m0 + r, pq.h, pq.c8, pq.pool_row[kByToken ? 0 : j]);
    }
    return;
  }
#pragma unroll
  for (int j = 0; j < kPasses; ++j) {
    const int r = j * kRowsPerPass + tid / kPieces, c = (tid % kPieces) * 8;
    const int row = m0 + r;
    // (an 8-byte aligned read of the padded row: two halves)
    const u32x2 lo = *(const u32x2*)&stage[r * kCStride + c], hi = *(const u32x2*)&stage[r * kCStride + c + 4];
    u32x4 v = {lo[0], lo[1], hi[0], hi[1]};
    if (row < p.M) {
      unsigned short* dst = p.out + (size_t)row * p.N + n0 + c;
      if (EPI == LBM_LINEAR_BIAS_RESIDUAL) v = add_rows(res_v[j], v);
      lbm_store_through(dst, v);
    }
    if (EPI == LBM_LINEAR_BIAS_RESIDUAL && p.stats_out) store_row_stats(p, v, row, n0 + c, TN == 64 ? 6 : p.stats_shift, tid);
  }
}

// ---------------------------------------------------------------------------- few rows
// The same product on tiles of 64 columns x 32, 64 or 96 rows, for launches whose 128-row tiles would leave CUs idle
// (a small image's 261 rows into 1,024 columns: 48 of 256) or share a tile between workgroups that meet in memory.
// Bound by the fill: a step moves (TM + 64) x 128 bytes through a CU's 64 bytes per cycle for TM x 64 x 64
// multiplications, a half to a quarter of that time on the matrix pipe, so what counts is how many CUs share the
// rows, and how little stands around the loop.  A wavefront owns a 32 x 32 block of the tile over its half of
// every 64-wide slice of K - the sums of the 128-row tiles, in their order: the same bits - and two others load, a
// 64-wide half each of 128-wide steps (half the barriers), three steps ahead.  Everything the store needs is asked
// for before the loop.  KS: the launches that sum K in slices (LinearArgs::k_splits) keep KS pairs of sums, one
// slice behind the other, and add them in slice order at the end: the bits of several workgroups that
// meet in memory, without the meeting (5 us of an fc2 launch).
// 96 rows: where 64-row tiles are more than one round of the CUs and 128-row tiles, at 192 rows a step to load instead of
// 160, are one: 257-384 rows x 4,096 columns, 321-480 x 3,072, 1,025-1,536 x 1,024.  (Three stages, not four: 40 KB each.)  us
// per launch on tiles of 128 and of 96 rows: 261 x 4,096 x 1,024 + GELU 8.4, 7.5, 384 rows 8.9, 7.9; 330 x 3,072 x 1,024
// with the producer 9.2, 8.4, 480 rows 9.9, 9.0; 1,200 x 1,024 x 1,024 7.8, 7.0, x 4,096 19.1, 17.8; 1,536 x 1,024 x 4,096
// 19.8, 19.6; 1,500 x 768 x 3,072 16.3, 14.3.
// us per launch, weights rotating through 24 layers, before (128 x 64 tiles) and after: M x N x K 81 x 3,072 x
// 1,024 with the producer 9.4 -> 6.1, 261 rows 10.1 -> 7.6; 261 x 1,024 x 1,024 8.1 -> 4.9, 1,004 rows 8.4 -> 6.4;
// 261 x 1,024 x 4,096 12.3 -> 10.1, 512 rows 14.6 -> 11.4, 1,004 rows 18.1 -> 15.3.  (Six stages instead of four: no
// faster.  What the last are bound by is L2: 256 CUs x 87 bytes per ns against 92 of a bare copy of such rows.)
template <int EPI, int TM, int KS = 1, int ROPE = 0, bool NORM = false, bool LNA = false>
__global__ __launch_bounds__(lbm_rows_threads(TM), 1) void lbm_linear_bf16_rows_kernel(LinearArgs p) {
  constexpr int kWaves = TM / 32 * 4;                      // computing wavefronts: (TM / 32) x 2 blocks of 32 x 32, two halves of K each
  constexpr int kHalf = (TM + 64) * kKS;                   // elements of one 64-wide half of a stage: rows of a, then of w
  constexpr int kStage = 2 * kHalf;
  constexpr int kStages = TM == 96 ? 3 : 4;
  __shared__ __attribute__((aligned(1024))) unsigned short ops[kStages * kStage];
  __shared__ __attribute__((aligned(16))) unsigned short gelu_tab[EPI == LBM_LINEAR_BIAS_GELU ? kGeluEntries : 8];
  __shared__ __attribute__((aligned(8))) float ln_rows[LNA ? TM * 2 : 2];                   // per row: rstd, -mean * rstd
  __shared__ __attribute__((aligned(16))) float colvec[3][64];                              // bias, column sums of w (LNA), LayerScale

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  hold_arguments<EPI, LNA, NORM>(p);
  int mt, nt;
  lbm_tile_of_workgroup((int)blockIdx.x, p, mt, nt);
  const int m0 = mt * TM, n0 = nt * 64;
  const int nk = p.K / (2 * kKS);                          // 128-wide steps

  if (blockIdx.y || wave >= kWaves) {
    // (blockIdx.y is a scalar register: nothing is loaded to know)
    if (blockIdx.y || wave == kWaves + 2) {
      lbm_touch(p.touch, lbm_rows_threads(TM), true);
      return;
    }
    // A loading wavefront, as in the kernel above: one 64-wide half of every step, eight whole rows per load.
    const int half = wave - kWaves;
    constexpr int kUnitsA = TM / 8, kUnitsW = 8, kLoads = kUnitsA + kUnitsW;
    const int l8 = lane >> 3, chunk = (lane & 7) ^ (lane >> 4);
    unsigned off[kLoads];
#pragma unroll
    for (int u = 0; u < kLoads; ++u) {
      const int row = u < kUnitsA ? min(m0 + 8 * u + l8, p.M - 1) : 8 * (u - kUnitsA) + l8;   // rows past M re-read the last row
      off[u] = ((unsigned)row * (unsigned)p.K + (unsigned)(chunk ^ (4 * (u & 1))) * 8u) * 2u;
    }
    const char* a_base = (const char*)(p.a + half * kKS);
    const char* w_base = (const char*)(p.w + (size_t)n0 * p.K + half * kKS);
    const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(__attribute__((address_space(3))) unsigned short*)&ops[0]) + (unsigned)(half * kHalf * 2);
    auto load_step = [&](int s) {
      const unsigned st = lds0 + (unsigned)(s % kStages) * (kStage * 2);
      const size_t at = (size_t)s * (2 * kKS * 2);
#pragma unroll
      for (int u = 0; u < kLoads; ++u) {
        const char* base = (u < kUnitsA ? a_base : w_base) + at;
        asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off[u]), "s"(base), "s"(st + u * 1024u) : "memory", "m0");
      }
    };
    __builtin_amdgcn_s_setprio(3);
#pragma unroll
    for (int i = 0; i < kStages - 1; ++i)
      if (i < nk) load_step(i);
    for (int s = -1; s < nk - 1; ++s) {   // the barrier at the top of step s publishes the rows of step s + 1
      const int behind = nk - 2 - s;      // steps that may be in flight behind those
      if (kStages > 3 && behind >= 2) LBM_DMA_WAIT(2 * kLoads);
      else if (behind >= 1) LBM_DMA_WAIT(kLoads);
      else LBM_DMA_WAIT(0);
      __builtin_amdgcn_s_barrier();
      if (s + kStages < nk) load_step(s + kStages);
    }
    return;
  }

  // ---- computing wavefronts
  const int n32 = lane & 31, g = lane >> 5;
  const int kh = wave & 1, sub = wave >> 1;
  const int wm = (sub >> 1) * 32, wn = (sub & 1) * 32;
  const int r = tid >> 3, c8 = tid & 7;                    // the row and the piece of it that this thread stores
  const int row = m0 + r, row_held = min(row, p.M - 1);
  // everything the store will need is asked for before the first step
  if (EPI == LBM_LINEAR_BIAS_GELU) {
#pragma unroll
    for (int i = 0; i < (kGeluEntries / 8 + kWaves * 64 - 1) / (kWaves * 64); ++i) {
      const int at = i * kWaves * 64 + tid;
      const unsigned m0v = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(__attribute__((address_space(3))) unsigned short*)&gelu_tab[0] + (unsigned)(i * kWaves + wave) * 1024u);
      if (at < kGeluEntries / 8)
        asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"((unsigned)at * 16u), "s"((const char*)g_gelu_table), "s"(m0v) : "memory", "m0");
    }
  }
  f32x2 ln_part[kLnHeld] = {};
  const bool ln_lane = LNA && tid < TM * 4;
  if (ln_lane) ask_row_stats(p, min(m0 + (tid >> 2), p.M - 1), tid & 3, ln_part);
  // (one value per thread: the vectors need not be aligned)
  float cv = 0.f;
  if (wave == 0 && p.bias) cv = p.bias[n0 + lane];
  if (LNA && wave == 1) cv = p.ln_colsum[n0 + lane];
  if (EPI == LBM_LINEAR_BIAS_RESIDUAL && wave == 2 && p.gamma) cv = p.gamma[n0 + lane];
  u32x4 res = {};
  if (EPI == LBM_LINEAR_BIAS_RESIDUAL) res = *(const u32x4*)(p.res + (size_t)row_held * p.N + n0 + c8 * 8);
  lbm_qkv::f32x4 w4[2] = {}, b4[2] = {}, cs4[4] = {};
  int which = 0, head = 0, pool_row = -1;
  if (EPI == kEpiQkvPrepare) {
    which = n0 / (p.num_heads * 64);
    head = nt - which * p.num_heads;
    if (NORM && which < 2) {
      const lbm_qkv::f32x4* wp = (const lbm_qkv::f32x4*)((which == 0 ? p.q_norm_w : p.k_norm_w) + c8 * 8);
      const lbm_qkv::f32x4* bp = (const lbm_qkv::f32x4*)((which == 0 ? p.q_norm_b : p.k_norm_b) + c8 * 8);
      w4[0] = wp[0]; w4[1] = wp[1];
      b4[0] = bp[0]; b4[1] = bp[1];
    }
    if (which < 2) ask_rotary<ROPE>(p, row_held, c8, cs4);
    else if (p.append_rows) pool_row = p.append_rows[row_held];
    if (which == 1 && p.append_rows) pool_row = p.append_rows[row_held];
  }
  if (ln_lane) {
    const f32x2 st = merge_row_stats(p, min(m0 + (tid >> 2), p.M - 1), tid & 3, ln_part);
    if ((tid & 3) == 0) *(f32x2*)&ln_rows[2 * (tid >> 2)] = st;
  }
  if (wave < 3) colvec[wave][lane] = cv;

  // fragments: row n32 of the block (the second half of K takes its columns of w with the halves of 16 swapped,
  // so that registers 0 .. 7 of either sum are the columns that its wavefront finishes)
  const int sw = (n32 >> 1) & 7;
  const unsigned short* fa = ops + (wm + n32) * kKS;
  const unsigned short* fw = ops + (TM + wn + (n32 ^ (kh * 16))) * kKS;
  int pos[2];
#pragma unroll
  for (int k16 = 0; k16 < 2; ++k16) pos[k16] = ((kh * 4 + k16 * 2 + g) ^ sw) * 8;
  bf16x8 wf[2][4], af[2][4];
  int stage_at = 0;          // elements to the stage that is read next
  auto read_step = [&](int buf) {
    const int stage = stage_at;
    stage_at = stage_at == (kStages - 1) * kStage ? 0 : stage_at + kStage;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int at = stage + (i >> 1) * kHalf + pos[i & 1];
      wf[buf][i] = __builtin_bit_cast(bf16x8, *(const u32x4*)(fw + at));
      af[buf][i] = __builtin_bit_cast(bf16x8, *(const u32x4*)(fa + at));
    }
  };
  f32x16 part[KS];
#pragma unroll
  for (int j = 0; j < KS; ++j)
#pragma unroll
    for (int i = 0; i < 16; ++i) part[j][i] = 0.f;
  auto step_barrier = [&]() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  step_barrier();
  read_step(0);
  const int seg = nk / KS;
#pragma unroll
  for (int j = 0; j < KS; ++j) {
    for (int s0 = 0; s0 < seg; s0 += 2) {
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        if (KS > 1 || s0 + st < seg) {          // (several sums: of an even number of steps each)
          if (j * seg + s0 + st + 1 < nk) {
            step_barrier();
            read_step(st ^ 1);
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) part[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[st][i], af[st][i], part[j], 0, 0, 0);
        }
      }
    }
  }
  LBM_DMA_WAIT(0);     // (the GELU table)
  step_barrier();      // everyone is done with the operands
  // ---- the two halves of K meet
  float* xch = (float*)&ops[0];              // [wave][KS][2][64 lanes][4]
  static_assert(kWaves * KS * 2 * 64 * 16 <= kStage * 2 * 2, "the exchanged sums fit the first two stages");
#pragma unroll
  for (int j = 0; j < KS; ++j)
#pragma unroll
    for (int c = 0; c < 2; ++c) *(f32x4*)&xch[(((wave * KS + j) * 2 + c) * 64 + lane) * 4] = f32x4{part[j][8 + 4 * c], part[j][9 + 4 * c], part[j][10 + 4 * c], part[j][11 + 4 * c]};
  step_barrier();
  f32x4 fin[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
#pragma unroll
    for (int j = 0; j < KS; ++j) {
      const f32x4 got = *(const f32x4*)&xch[((((wave ^ 1) * KS + j) * 2 + c) * 64 + lane) * 4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float both = part[j][4 * c + e] + got[e];
        fin[c][e] = j > 0 ? fin[c][e] + both : (KS > 2 ? 0.f + both : both);
      }
    }
  }
  // ---- epilogue
  constexpr int kCStride = 64 + 4;
  unsigned short* stage = &ops[2 * kStage];
  f32x2 row_f = {1.f, 0.f};
  if (LNA) row_f = *(const f32x2*)&ln_rows[2 * (wm + n32)];
  f32x4 x[2];
  bf16x4 y[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int col = wn + kh * 16 + c * 8 + g * 4;
    const f32x4 bias4 = *(const f32x4*)&colvec[0][col], colsum4 = *(const f32x4*)&colvec[1][col], gamma4 = *(const f32x4*)&colvec[2][col];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float lin = fin[c][e];
      if (LNA) lin = __builtin_fmaf(lin, row_f[0], row_f[1] * colsum4[e]);
      x[c][e] = lin + bias4[e];
      if (EPI == LBM_LINEAR_BIAS_RESIDUAL && p.gamma) x[c][e] = round_bf16(x[c][e]) * gamma4[e];
    }
    y[c] = __builtin_convertvector(x[c], bf16x4);
  }
  if (EPI == LBM_LINEAR_BIAS_GELU) gelu_of<2>(x, gelu_tab, y);
#pragma unroll
  for (int c = 0; c < 2; ++c) *(bf16x4*)&stage[(wm + n32) * kCStride + wn + kh * 16 + c * 8 + g * 4] = y[c];
  step_barrier();
  const u32x2 lo = *(const u32x2*)&stage[r * kCStride + c8 * 8], hi = *(const u32x2*)&stage[r * kCStride + c8 * 8 + 4];
  u32x4 v = {lo[0], lo[1], hi[0], hi[1]};
  if (EPI == kEpiQkvPrepare) {
    const bf16x8 o8 = produce_row<ROPE, NORM>(v, which, c8, w4, b4, cs4, p.eps, which == 0 ? p.q_scale : 1.0f);
    if (row < p.M) store_produced(p, produced_rows(p, which), o8, which, row, head, c8, pool_row);
    return;
  }
  if (EPI == LBM_LINEAR_BIAS_RESIDUAL) v = add_rows(res, v);
  if (row < p.M) lbm_store_through(p.out + (size_t)row * p.N + n0 + c8 * 8, v);
  if (EPI == LBM_LINEAR_BIAS_RESIDUAL && p.stats_out) store_row_stats(p, v, row, n0 + c8 * 8, 6, tid);
}

// ---------------------------------------------------------------------------- several streams' rows
// The same product on 256 x 256 (192 x 256, 128 x 256) tiles, for launches with enough rows to give most
// of the 256 CUs such a tile (four streams' 4,016 rows x the qkv projection's 3,072 or fc1's
// 4,096 columns): a 256 x 256 tile moves 64 KB of operands per 64 of K for 8.4 MFLOP - 128 FLOP
// per byte on the way from L2 into LDS, which is what bounds the 128 x 128 tiles above at 64.
// Eight wavefronts, each on 64 rows x 128 columns of the tile (96 x 64 of a 192-row tile, 64 x 64 of a 128-row
// one) over the whole K slice, no K split inside the workgroup and so no exchange at the end: one sum per
// element, the same bits whatever the tile.  Two LDS
// stages: a 64-wide step is 24-32 MFMAs per wavefront, longer than a trip to memory, so one step
// of prefetch is enough; the loads of a step are issued at the end of the step before the one
// they replace, right behind the barrier that frees its stage (a 128-row tile's step is half as long: three
// stages).  Same operand path (global -> LDS directly, swizzled 16-byte chunks), same
// epilogue arithmetic and rounding sequence.  Epilogues: bias, bias + GELU, and the
// pre-attention producer; the folded LayerNorm of the activations; not the residual forms (their
// 1,024 columns make too few such tiles).  The per-column vectors wait in LDS instead of
// registers (the accumulators take half the register file).  192- and 128-row tiles are for shapes whose
// 256-row tiles would leave CUs idle (4,016 x 3,072: 192 against 252 tiles; 2,008 x 3,072: 96 against 192:
// 33 us with the producer on the 132 tiles of 192 rows, 23 on these; 1,350 x 4,096 + GELU 27.7 -> 21.3).
constexpr int kBN = 256;
constexpr int kBCStride = kBN + 4;                          // bf16 per staged output row
constexpr int lbm_big_stages(int bm) { return bm == 128 ? 3 : 2; }
// Whether two more wavefronts load, as above: where the others can do with 168 registers, that is with up to 192 rows.
constexpr bool lbm_big_loaders(int bm) { return bm <= 192; }
constexpr int lbm_big_norm_rows(int epi, bool norm) { return epi == kEpiQkvPrepare && norm ? 4 : 1; }
constexpr int lbm_big_threads(int bm) { return kGThreads + (lbm_big_loaders(bm) ? kGLoadWaves * 64 : 0); }
constexpr int lbm_big_lds_bytes(int bm) {
  const int stages = lbm_big_stages(bm) * (bm + kBN) * kKS * 2;
  return bm * kBCStride * 2 > stages ? bm * kBCStride * 2 : stages;
}
static_assert(lbm_big_lds_bytes(256) + kGeluEntries * 2 + 2 * kBN * 4 + 256 * 8 <= 160 * 1024, "LDS budget of the 256 x 256 tile");

template <int BM, int EPI, int ROPE = 0, bool NORM = false, bool LNA = false>
__global__ __launch_bounds__(lbm_big_threads(BM), 1) void lbm_linear_bf16_big_kernel(LinearArgs p) {
  constexpr int kRowGroups = BM == 256 ? 4 : 2;             // wavefronts along the rows of the tile
  constexpr int kColGroups = 8 / kRowGroups;
  constexpr int RB = BM / 32 / kRowGroups, CB = kBN / 32 / kColGroups;   // 32 x 32 blocks per wavefront: 2 x 4 or 3 x 2
  constexpr int kStageBytes = (BM + kBN) * kKS * 2;
  __shared__ __attribute__((aligned(1024))) unsigned char lds_raw[lbm_big_lds_bytes(BM)];   // two operand stages, then the staged output tile
  __shared__ __attribute__((aligned(16))) float colvec[2][kBN];                             // bias, column sums of w (LNA)
  __shared__ __attribute__((aligned(16))) unsigned short gelu_tab[EPI == LBM_LINEAR_BIAS_GELU ? kGeluEntries : 8];
  __shared__ __attribute__((aligned(8))) float ln_rows[LNA ? BM * 2 : 2];                   // per row: rstd, -mean * rstd

  __shared__ __attribute__((aligned(16))) float qk_norm[lbm_big_norm_rows(EPI, NORM)][64];           // q's weight and bias, k's

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  hold_arguments<EPI, LNA, NORM>(p);
  const int n32 = lane & 31, g = lane >> 5;
  const int rg = wave % kRowGroups, cg = wave / kRowGroups;
  const int wm = rg * (RB * 32), wn = cg * (CB * 32);       // this wavefront's corner of the tile
  int mt, nt;
  lbm_tile_of_workgroup((int)blockIdx.x, p, mt, nt);
  const int m0 = mt * BM, n0 = nt * kBN;
  // The tile's columns in four slots of 64.  Where the producer has work to do, three tiles share four heads of q, k and v so that none
  // has more than three slots of q and k: q0 q1 k0 v0 | q2 k1 k2 v1 | q3 k3 v2 v3, a digit 4 x (q, k, v) + head for each slot.
  // The store is bound by the producer's vector instructions, and a launch of one round by its slowest tile: four slots of q
  // were 187 instructions per eight elements behind the loop, beside tiles of v with none.  Mixed, with a token's
  // entries rounded once for its slots instead of once for each and, the entries being few now, loading wavefronts on 192 rows too, us of
  // 16 heads x 1,024, interleaved and half-split entries, before and now: 2,008 rows 19.8, 20.4 -> 17.2, 17.4; 4,016 30.7, 33.1 -> 26.7, 27.0;
  // 5,000 38.1, 39.9 -> 34.0, 34.1; 8,040 59.8, 65.7 -> 52.1, 53.0.  Without norm and table slots of one kind stay: they leave as
  // rows of 512 bytes (mixed 2,008 rows 17.4 for 15.6, 8,040 51.2 for 46.2; q, k, v in turn instead of two neighbours where there are two 1 % more).
  constexpr bool kQkv = EPI == kEpiQkvPrepare, kMixed = kQkv && (ROPE != 0 || NORM);
  auto slot_of = [&](int j, int& head) {
    const int group = nt / 3;
    const int digit = (int)(0xBA7396528410ull >> (4 * (4 * (nt - 3 * group) + j))) & 15;
    head = 4 * group + (digit & 3);
    return digit >> 2;
  };
  auto slot_col = [&](int j) {
    int head;
    const int which = slot_of(j, head);
    return (which * p.num_heads + head) * 64;
  };
  int w_rows[kBN / 64];   // each slot's first row of w, from w_base on
#pragma unroll
  for (int j = 0; j < kBN / 64; ++j) w_rows[j] = kMixed ? slot_col(j) : 64 * j;

  if (blockIdx.y) {   // (a scalar register: nothing is loaded to know)
    lbm_touch(p.touch, lbm_big_threads(BM), false);
    return;
  }

  // ---- staging (as in the kernel above: eight 128-byte rows per wavefront and load)
  constexpr int kPassA = BM / 64, kPassW = kBN / 64;
  const int ld_r = wave * 8 + (lane >> 3);
  const unsigned sw_c = (unsigned)(((lane & 7) ^ ((ld_r >> 1) & 7)) * 8);
  unsigned a_off[kPassA];
#pragma unroll
  for (int j = 0; j < kPassA; ++j) a_off[j] = ((unsigned)min(m0 + ld_r + 64 * j, p.M - 1) * (unsigned)p.K + sw_c) * 2u;
  const unsigned w_off = ((unsigned)ld_r * (unsigned)p.K + sw_c) * 2u;
  const int nk = p.K / kKS;
  const char* a_base = (const char*)p.a;
  const char* w_base = (const char*)(p.w + (kMixed ? 0 : (size_t)n0 * p.K));
  auto dma_row = [&](const char* base, unsigned voff, const unsigned char* lds_dst) {
    const unsigned m0v = (unsigned)(size_t)(__attribute__((address_space(3))) const void*)lds_dst;
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1"
                 :
                 : "v"(voff), "s"(base), "s"(__builtin_amdgcn_readfirstlane(m0v))
                 : "memory", "m0");
  };
  // load j of step ks: the activations' passes first, then the weights'
  auto dma_one = [&](int ks, int stage, int j) {
    unsigned char* st = lds_raw + stage * kStageBytes;
    if (j < kPassA) dma_row(a_base + ks * (kKS * 2), a_off[j], st + (64 * j + 8 * wave) * (kKS * 2));
    else dma_row(w_base + ((size_t)w_rows[j - kPassA] * p.K + (size_t)ks * kKS) * 2, w_off,
                 st + BM * kKS * 2 + (64 * (j - kPassA) + 8 * wave) * (kKS * 2));
  };
  constexpr int kDma = kPassA + kPassW;
  constexpr bool kLoaders = lbm_big_loaders(BM);
  constexpr int kStages = lbm_big_stages(BM);
  if (kLoaders && wave >= kGThreads / 64) {
    // a loading wavefront: every second KB of a step's operands (as in the kernel above)
    const int par = wave - kGThreads / 64, l8 = lane >> 3;
    constexpr int kUnitsA = BM / 16, kLoads = kUnitsA + kBN / 16;
    const unsigned chunk = (unsigned)(((lane & 7) ^ (4 * par + (lane >> 4))) * 8);
    unsigned off[kLoads];
#pragma unroll
    for (int u = 0; u < kLoads; ++u) {
      const int row = u < kUnitsA ? min(m0 + 8 * (2 * u + par) + l8, p.M - 1) : w_rows[(u - kUnitsA) / 4] + (8 * (2 * (u - kUnitsA) + par) + l8) % 64;
      off[u] = ((unsigned)row * (unsigned)p.K + chunk) * 2u;
    }
    const unsigned lds_first = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)&lds_raw[0]) + (unsigned)par * 1024u;
    auto load_step = [&](int s) {
      const unsigned st = lds_first + (unsigned)(s % kStages) * kStageBytes;
#pragma unroll
      for (int u = 0; u < kLoads; ++u) {
        const char* base = (u < kUnitsA ? a_base : w_base) + (size_t)s * (kKS * 2);
        asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off[u]), "s"(base), "s"(st + u * 2048u) : "memory", "m0");
      }
    };
    __builtin_amdgcn_s_setprio(3);
#pragma unroll
    for (int s = 0; s < kStages - 1; ++s)
      if (s < nk) load_step(s);
    for (int s = -1; s < nk; ++s) {    // the barrier of step s hands over the rows of step s + 1 and frees the stage of step s
      if (kStages > 2 && nk - 2 - s >= 1) LBM_DMA_WAIT(kLoads);
      else LBM_DMA_WAIT(0);
      __builtin_amdgcn_s_barrier();
      if (s + kStages < nk) load_step(s + kStages);
    }
    return;
  }

  // the folded LayerNorm's row statistics: two threads per row, each every second partial
  constexpr int kLnHeld = 8;
  f32x2 ln_part[kLnHeld] = {};
  if (LNA) {
    const float* ln_st = p.ln_stats + (size_t)min(m0 + (tid >> 1), p.M - 1) * p.ln_tiles * 2;
#pragma unroll
    for (int i = 0; i < kLnHeld; ++i)
      if ((tid & 1) + 2 * i < p.ln_tiles) ln_part[i] = *(const f32x2*)(ln_st + 2 * ((tid & 1) + 2 * i));
  }
  // per-column vectors of the tile into LDS (read in the epilogue, many barriers from here)
  float cv_bias = 0.f, cv_sum = 0.f, cv_norm = 0.f;
  if (tid < kBN) {
    const int col = kMixed ? slot_col(wave) + lane : n0 + tid;
    if (p.bias) cv_bias = p.bias[col];
    if (LNA) cv_sum = p.ln_colsum[col];
    if (kQkv && NORM) cv_norm = (wave == 0 ? p.q_norm_w : wave == 1 ? p.q_norm_b : wave == 2 ? p.k_norm_w : p.k_norm_b)[lane];
  }
  if (EPI == LBM_LINEAR_BIAS_GELU && tid < kGeluEntries / 8)
    dma_row((const char*)g_gelu_table, (unsigned)tid * 16u, (const unsigned char*)&gelu_tab[wave * 512]);
#pragma unroll
  for (int j = 0; j < (kLoaders ? 0 : kDma); ++j) dma_one(0, 0, j);
  if (tid < kBN) {
    colvec[0][tid] = cv_bias;
    colvec[1][tid] = cv_sum;
    if (kQkv && NORM) qk_norm[wave][lane] = cv_norm;
  }
  if (LNA && (tid >> 1) < BM) {
    const int r = tid >> 1, part = tid & 1;
    const float* ln_st = p.ln_stats + (size_t)min(m0 + r, p.M - 1) * p.ln_tiles * 2;
    float sm = 0.f;
#pragma unroll
    for (int i = 0; i < kLnHeld; ++i)
      if (part + 2 * i < p.ln_tiles) sm += ln_part[i][0];
    for (int i = part + 2 * kLnHeld; i < p.ln_tiles; i += 2) sm += ln_st[2 * i];
    sm += lbm_qkv::lane_xor1(sm);
    const float mean = sm / (float)p.ln_tiles;
    const float n_i = (float)p.K / (float)p.ln_tiles;
    float m2 = 0.f;
#pragma unroll
    for (int i = 0; i < kLnHeld; ++i)
      if (part + 2 * i < p.ln_tiles) {
        const float d = ln_part[i][0] - mean;
        m2 += ln_part[i][1] + n_i * d * d;
      }
    for (int i = part + 2 * kLnHeld; i < p.ln_tiles; i += 2) {
      const float d = ln_st[2 * i] - mean;
      m2 += ln_st[2 * i + 1] + n_i * d * d;
    }
    m2 += lbm_qkv::lane_xor1(m2);
    const float rstd = __builtin_amdgcn_rsqf(m2 / (float)p.K + p.ln_eps);
    if (part == 0) {
      ln_rows[2 * r] = rstd;
      ln_rows[2 * r + 1] = -mean * rstd;
    }
  }

  f32x16 acc[CB][RB];   // [column block of w][row block of a]; element i: column 8 (i / 4) + 4 g + i % 4, row n32
#pragma unroll
  for (int a = 0; a < CB; ++a)
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[a][b][i] = 0.f;

  const int sw_r = (n32 >> 1) & 7;
  // M0 values as integers (no pointer cast inside the loop): this wavefront's KB of every block of 64 rows
  const unsigned m0_wave = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)lds_raw + (unsigned)wave * 1024u);
  unsigned w_offs[kPassW];
#pragma unroll
  for (int j = 0; j < kPassW; ++j) w_offs[j] = w_off + (unsigned)w_rows[j] * (unsigned)p.K * 2u;
  auto dma_at = [&](const char* base, unsigned voff, unsigned m0v) {
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(voff), "s"(base), "s"(m0v) : "memory", "m0");
  };
  auto dma_step = [&](int ks, unsigned stage_bytes) {
    const char* ab = a_base + (size_t)ks * (kKS * 2);
    const char* wb = w_base + (size_t)ks * (kKS * 2);
#pragma unroll
    for (int j = 0; j < kPassA; ++j) dma_at(ab, a_off[j], m0_wave + stage_bytes + (unsigned)(64 * j * kKS * 2));
#pragma unroll
    for (int j = 0; j < kPassW; ++j) dma_at(wb, w_offs[j], m0_wave + stage_bytes + (unsigned)((BM + 64 * j) * kKS * 2));
  };
  bf16x8 wf[2][CB], af[2][RB];
  auto read = [&](unsigned stage_bytes, int kq, bf16x8 (&wfr)[CB], bf16x8 (&afr)[RB]) {
    const unsigned char* la = lds_raw + stage_bytes;
    const unsigned char* lw = la + BM * kKS * 2;
    const int posb = ((kq * 2 + g) ^ sw_r) * 16;
#pragma unroll
    for (int a = 0; a < CB; ++a)
      wfr[a] = __builtin_bit_cast(bf16x8, *(const u32x4*)(lw + (wn + a * 32 + n32) * (kKS * 2) + posb));
#pragma unroll
    for (int b = 0; b < RB; ++b)
      afr[b] = __builtin_bit_cast(bf16x8, *(const u32x4*)(la + (wm + b * 32 + n32) * (kKS * 2) + posb));
  };
  auto mfmas = [&](int kq, int from, int to) {
#pragma unroll
    for (int a = 0; a < CB; ++a)
#pragma unroll
      for (int b = 0; b < RB; ++b)
        if (a * RB + b >= from && a * RB + b < to)
          acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[kq & 1][a], af[kq & 1][b], acc[a][b], 0, 0, 0);
  };
#define LBM_SGB(mask, n) __builtin_amdgcn_sched_group_barrier(mask, n, 0)
  // One 64-wide step on the stage at byte `here`.  The fragment reads of a quarter step are
  // issued one by one in between the MFMAs of the quarter before it (a burst of them fills the
  // LDS queue and stalls the wavefront's MFMAs behind it).  The barrier that hands the other
  // stage over sits in the middle of the last quarter: behind it come the first fragment reads
  // of the next step, covered by the quarter's remaining MFMAs, and at the end of the step the
  // loads of the step after the next one, which have a whole step to land.
  constexpr int kQ = CB * RB, kR = CB + RB, kH = kQ / 2;
  auto step = [&](int s, auto stage_c) {
    constexpr unsigned here = decltype(stage_c)::value * kStageBytes, there = (decltype(stage_c)::value + 1) % kStages * kStageBytes;
#pragma unroll
    for (int kq = 0; kq < 3; ++kq) {
      read(here, kq + 1, wf[(kq + 1) & 1], af[(kq + 1) & 1]);
      mfmas(kq, 0, kQ);
#pragma unroll
      for (int i = 0; i < kR; ++i) { LBM_SGB(0x008, 1); LBM_SGB(0x100, 1); }
      if (kQ > kR) LBM_SGB(0x008, kQ - kR);
      __builtin_amdgcn_sched_barrier(0);
    }
    mfmas(3, 0, kH);
    __builtin_amdgcn_sched_barrier(0);
    if (!kLoaders) LBM_DMA_WAIT(0);
    __syncthreads();   // the other stage has landed everywhere, and everyone has read all of this one
    __builtin_amdgcn_sched_barrier(0);
    read(there, 0, wf[0], af[0]);
    mfmas(3, kH, kQ);
    LBM_SGB(0x100, kR - (kQ - kH) + 1 > 0 ? kR - (kQ - kH) + 1 : 0);
#pragma unroll
    for (int i = 0; i < kQ - kH; ++i) { LBM_SGB(0x008, 1); LBM_SGB(0x100, 1); }
    __builtin_amdgcn_sched_barrier(0);
    if (!kLoaders && s + 2 < nk) dma_step(s + 2, here);
  };
  LBM_DMA_WAIT(0);
  __syncthreads();
  if (!kLoaders) dma_step(1, kStageBytes);
  read(0, 0, wf[0], af[0]);
  for (int s = 0; s < nk; s += kStages) {
    step(s, std::integral_constant<unsigned, 0>{});
    if (kStages == 2 || s + 1 < nk) step(s + 1, std::integral_constant<unsigned, 1>{});
    if (kStages == 3 && s + 2 < nk) step(s + 2, std::integral_constant<unsigned, kStages - 1>{});
  }
#undef LBM_SGB

  // ---- epilogue.  A lane of the producer works on the same eight columns of all four slots of a token: one set of rotary entries,
  // asked for a pass ahead (the first now, it arrives while the tile is staged) and rounded once.
  typedef lbm_qkv::f32x4 qf4;
  constexpr int kTokenPasses = BM / 64;
  const int c8 = lane & 7;
  qf4 cs4[2][4] = {};
  int pool_row[kTokenPasses];
  if (kMixed) {
#pragma unroll
    for (int j = 0; j < kTokenPasses; ++j) {
      const int t = min(m0 + j * 64 + (tid >> 3), p.M - 1);
      if (j == 0) ask_rotary<ROPE>(p, t, c8, cs4[0]);
      pool_row[j] = p.append_rows ? p.append_rows[t] : -1;
    }
  }
  __syncthreads();   // the operand stages are dead: the output tile is staged over them
  // In registers: the folded LayerNorm's scale and correction, + bias, round (the linear's
  // output), GELU, round; then the tile goes through LDS and leaves as whole rows.
  unsigned short* stage = (unsigned short*)lds_raw;
  f32x2 row_f[RB];
#pragma unroll
  for (int b = 0; b < RB; ++b) row_f[b] = LNA ? *(const f32x2*)&ln_rows[2 * (wm + b * 32 + n32)] : f32x2{1.f, 0.f};
#pragma unroll
  for (int a = 0; a < CB; ++a) {
    f32x4 bias4[4], colsum4[4];   // (read once for all row blocks)
#pragma unroll
    for (int c4 = 0; c4 < 4; ++c4) {
      const int col = wn + a * 32 + c4 * 8 + g * 4;
      bias4[c4] = *(const f32x4*)&colvec[0][col];
      if (LNA) colsum4[c4] = *(const f32x4*)&colvec[1][col];
    }
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      f32x4 x[4];
      bf16x4 y[4];
#pragma unroll
      for (int c4 = 0; c4 < 4; ++c4) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float lin = acc[a][b][c4 * 4 + e];
          if (LNA) lin = __builtin_fmaf(lin, row_f[b][0], row_f[b][1] * colsum4[c4][e]);
          x[c4][e] = lin + bias4[c4][e];
        }
        y[c4] = __builtin_convertvector(x[c4], bf16x4);
      }
      if (EPI == LBM_LINEAR_BIAS_GELU) gelu_of<4>(x, gelu_tab, y);
#pragma unroll
      for (int c4 = 0; c4 < 4; ++c4) *(bf16x4*)&stage[(wm + b * 32 + n32) * kBCStride + wn + a * 32 + c4 * 8 + g * 4] = y[c4];
    }
  }
  __syncthreads();
  if (kMixed) {
    // the producer on the staged tile, as in the kernel above
    qf4 w4[2][2] = {}, b4[2][2] = {};   // q's, k's
    if (NORM)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          w4[i][e] = *(const qf4*)&qk_norm[2 * i][c8 * 8 + 4 * e];
          b4[i][e] = *(const qf4*)&qk_norm[2 * i + 1][c8 * 8 + 4 * e];
        }
#pragma unroll
    for (int j = 0; j < kTokenPasses; ++j) {
      const int r = j * 64 + (tid >> 3);
      if (j + 1 < kTokenPasses) ask_rotary<ROPE>(p, min(m0 + r + 64, p.M - 1), c8, cs4[(j + 1) & 1]);
      u32x4 raw[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const u32x2 lo = *(const u32x2*)&stage[r * kBCStride + s * 64 + c8 * 8], hi = *(const u32x2*)&stage[r * kBCStride + s * 64 + c8 * 8 + 4];
        raw[s] = u32x4{lo[0], lo[1], hi[0], hi[1]};
      }
      lbm_qkv::ready_rotary<ROPE>(cs4[j & 1], c8);
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        int head;
        const int which = slot_of(s, head);
        bf16x8 o8;
        if (which == 0) o8 = produce_row<ROPE, NORM, true>(raw[s], 0, c8, w4[0], b4[0], cs4[j & 1], p.eps, p.q_scale);
        else o8 = produce_row<ROPE, NORM, true>(raw[s], which, c8, w4[1], b4[1], cs4[j & 1], p.eps, 1.0f);
        if (m0 + r < p.M) store_produced(p, produced_rows(p, which), o8, which, m0 + r, head, c8, pool_row[j]);
      }
    }
    return;
  }
  constexpr int kPieces = kBN / 8;                    // 16-byte pieces per row of the tile: 32
  constexpr int kRowsPerPass = kGThreads / kPieces;   // 16
  constexpr int kPasses = BM / kRowsPerPass;          // 16 or 12
  const int pr = tid / kPieces, pc = (tid % kPieces) * 8;
  auto piece = [&](int j) {
    const int r = j * kRowsPerPass + pr;
    const u32x2 lo = *(const u32x2*)&stage[r * kBCStride + pc], hi = *(const u32x2*)&stage[r * kBCStride + pc + 4];
    return u32x4{lo[0], lo[1], hi[0], hi[1]};
  };
  if (!kQkv) {
#pragma unroll
    for (int j = 0; j < kPasses; ++j) {
      const int row = m0 + j * kRowsPerPass + pr;
      const u32x4 v = piece(j);
      if (row < p.M) lbm_store_through(p.out + (size_t)row * p.N + n0 + pc, v);
    }
    return;
  }
  // a producer with nothing to do but q's factor (an encoder's): rows of four heads of one kind
  const int dim = p.num_heads * 64, which = n0 / dim, col = n0 + pc - which * dim;   // (dim is a multiple of 256)
  unsigned short* const plain = produced_rows(p, which);
  if (plain) {
#pragma unroll
    for (int j = 0; j < kPasses; ++j) {
      const int row = m0 + j * kRowsPerPass + pr;
      u32x4 v = piece(j);
      const qf4 none[2] = {};
      if (which == 0) v = __builtin_bit_cast(u32x4, produce_row<0, false>(v, 0, 0, none, none, cs4[0], 0.f, p.q_scale));
      if (row < p.M) lbm_store_through(plain + (size_t)row * dim + col, v);
    }
  }
  if (which > 0 && p.append_rows) {
    int to[kPasses];
#pragma unroll
    for (int j = 0; j < kPasses; ++j) to[j] = p.append_rows[min(m0 + j * kRowsPerPass + pr, p.M - 1)];
#pragma unroll
    for (int j = 0; j < kPasses; ++j)
      if (m0 + j * kRowsPerPass + pr < p.M)
        store_produced(p, nullptr, __builtin_bit_cast(bf16x8, piece(j)), which, 0, col >> 6, (col & 63) >> 3, to[j]);
  }
}

}  // namespace

namespace {
// tile width: 64 columns while such tiles are one round of the 256 CUs (N = 1024 at one frame: 128
// workgroups instead of 64), 128 from there on (2,100 rows x 1,024 columns: one round instead of two, 11.4 us
// against 14.6 at K = 1,024, 27 against 38 at 4,096; 700 x 3,072: 10.4 against 13.5)
int lbm_linear_tiles(LinearArgs& p) {
  p.m_tiles = (p.M + kGM - 1) / kGM;
  const long long tiles = (long long)p.m_tiles * (p.N / 128);
  const int tn = p.N % 128 == 0 && tiles > 128 ? 128 : 64;
  p.n_tiles = p.N / tn;
  // (a width of its own, so that the next launch's LayerNorm sums the same values whatever tile made them)
  p.stats_shift = p.N % 128 == 0 && tiles >= 160 ? 7 : 6;
  return tn;
}
// 32, 64 or 96 rows per tile of 64 columns in the place of 128 x tn tiles where they need fewer rounds of the CUs x
// bytes per step (the fill is what bounds either), or 0; sets the row tiles.  With K summed in slices one workgroup
// walks them all: up to K = 4,096 that is the faster way (M x N x K 31 x 1,024 x 4,096: 10.5 -> 10.4 us,
// 1,004 rows 17.3 -> 15.6), from there on several workgroups are (512 x 768 x 6,144: 15.4 against 16.2; 81 x
// 1,024 x 8,192: 13.9 against 18.2); slices of an odd number of 128-wide steps go there too.
int lbm_linear_rows_tiles(LinearArgs& p, int tn, int splits) {
  if (tn != 64 || (splits > 1 && (p.K > 4096 || p.K % (splits * 4 * kKS) != 0))) return 0;
  const int nt = p.N / 64;
  int best = 0;
  long long best_cost = ((long long)p.m_tiles * nt + 255) / 256 * (128 + 64);
  for (int tm : {64, 32, 96}) {
    if (tm == 96 && splits > 1) continue;   // (K is sliced where 64 rows are one round)
    const long long cost = ((long long)((p.M + tm - 1) / tm) * nt + 255) / 256 * (tm + 64);
    if (cost < best_cost) best = tm, best_cost = cost;
  }
  if (best) p.m_tiles = (p.M + best - 1) / best;
  return best;
}
// 256 columns where that halves the rounds of the 256 CUs; sets the tile count.  A round of 128 x 256 tiles
// takes 1.35-1.4 rounds of 128 x 128, so two for one gain (M x N x K 8,040 x 1,024 x 4,096: 61 us against
// 72; 4,100 x 1,024 x 4,096: 44 against 55; 1,200 x 4,096 x 1,024: 21 against 24) and one for one (4,016 x
// 1,024 x 4,096: 48 against 36) or three for two (8,200 x 1,024 x 4,096: 100 against 94) do not.
// The qkv projection between one round of 128 x 128 tiles and the first size of the 192-row ones, us with two rounds and with one: without
// norm and table, interleaved and half-split entries, 16 heads 1,285 rows 18.3, 20.7, 21.3 and 16.2, 19.8, 20.1, 1,900 rows 19.8, 22.5, 23.0 and
// 16.3, 20.1, 20.4; 12 heads 1,800 rows 17.7, 19.4, 19.8 and 14.8, 18.1, 17.8, 2,600 rows 17.2, 21.9, 23.5 and 14.0, 17.7, 18.0.
bool lbm_linear_wider(LinearArgs& p) {
  if (p.N % 256 != 0) return false;
  const long long tiles = (long long)p.m_tiles * (p.N / 256);
  if ((2 * tiles + 255) / 256 < 2 * ((tiles + 255) / 256)) return false;
  p.n_tiles = p.N / 256;
  return true;
}
}  // namespace

namespace {
// Tiles of 256 columns when those of 256 or 192 rows give at least half of the 256 CUs a workgroup
// (several streams' rows into the 3,072 or 4,096 columns of the qkv projection or fc1): the row
// count of the tile (the one that needs the fewest rounds of the CUs times rows, of 128 rows too; as many rows as
// possible among equals), or 0; sets the tile counts
int lbm_linear_big_tiles(LinearArgs& p) {
  if (p.N % kBN != 0) return 0;
  const int nt = p.N / kBN;
  int best = 0;
  long long best_cost = 0;
  for (int bm : {256, 192, 128}) {
    const long long tiles = (long long)((p.M + bm - 1) / bm) * nt;
    if (bm == 128 ? !best : tiles < 128) continue;   // (fewer: the kernel above, whose elements are two sums)
    const long long cost = ((tiles + 255) / 256) * bm;      // rounds of the 256 CUs x rows per tile
    if (!best || cost < best_cost) best = bm, best_cost = cost;
  }
  if (!best) return 0;
  p.m_tiles = (p.M + best - 1) / best;
  p.n_tiles = nt;
  return best;
}
}  // namespace

namespace {
// the kernel addresses a row of either operand with a 32-bit byte offset from a 64-bit base
bool lbm_offsets_fit(int M, int N, int K) {
  return (long long)M * K * 2 < (1LL << 32) && (long long)N * K * 2 < (1LL << 32);
}
}  // namespace

namespace {
// the folded LayerNorm of the activations, checked and copied into the kernel arguments
int lbm_set_row_norm(LinearArgs& p, const lbm_row_norm* ln, const char* who) {
  if (!ln) return LBM_OK;
  if (!ln->w_colsum || !ln->stats || ln->stats_tiles <= 0 || p.K % ln->stats_tiles != 0)
    return lbm_fail(LBM_ERR_INVALID, "%s: standardised rows need w_colsum, stats and a tile count that divides K (got %d for K %d)",
                    who, ln->stats_tiles, p.K);
  p.ln_colsum = ln->w_colsum;
  p.ln_stats = ln->stats;
  p.ln_tiles = ln->stats_tiles;
  p.ln_eps = ln->eps;
  return LBM_OK;
}
}  // namespace

namespace {
// K slices per tile: as many as still leave every workgroup eight k-steps and fit one round of
// the 256 CUs (fc2 of one frame: 128 tiles of 128 x 64, two slices); the residual epilogue only
int lbm_linear_splits(const LinearArgs& p, int epilogue) {
  if (epilogue != LBM_LINEAR_BIAS_RESIDUAL) return 1;
  const int tiles = p.m_tiles * p.n_tiles, nk = p.K / kGK;
  for (int s = 4; s >= 2; s >>= 1)
    if (tiles * s <= 256 && nk % s == 0 && nk / s >= 8) return s;
  return 1;
}
// The counters' part of the workspace has ONE size, whatever the shape (a split launch has at most
// 128 tiles): one workspace serves launches of several shapes, and a counter that lay where another
// shape parks its partial tiles would not be zero.
constexpr size_t kSplitCounterBytes = 512;
static_assert(kSplitCounterBytes >= 256 / 2 * sizeof(unsigned), "two slices per tile at least, 256 workgroups at most");
}  // namespace

size_t lbm_linear_workspace_for(int M, int N, int K, int epilogue) {
  LinearArgs p = {};
  p.M = M; p.N = N; p.K = K;
  const int tn = lbm_linear_tiles(p);
  const int s = lbm_linear_splits(p, epilogue);
  if (s == 1) return 0;
  // (one workgroup for all slices of a tile: nothing is parked, the workspace only says that slices are wanted)
  LinearArgs rows = p;
  if (lbm_linear_rows_tiles(rows, tn, s)) return kSplitCounterBytes;
  return kSplitCounterBytes + (size_t)p.m_tiles * p.n_tiles * s * kGM * tn * 4;
}

int lbm_linear_stats_tiles_for(int M, int N) {
  LinearArgs p = {};
  p.M = M; p.N = N;
  lbm_linear_tiles(p);
  return p.N >> p.stats_shift;
}

namespace {
// what the calling thread's next GEMM launch is to ask for on behalf of launches behind it
thread_local LbmTouch g_prefetch_hint = {};
}  // namespace

void lbm_set_prefetch_hint(const LbmTouch& t) { g_prefetch_hint = t; }
void lbm_take_prefetch_hint(LbmTouch& t) {
  t = g_prefetch_hint;
  g_prefetch_hint = {};
}
dim3 lbm_touch_grid(LbmTouch& t, unsigned wgs) {
  const int idle = lbm_idle_cus(wgs);
  if (!t.lines[0] || idle < kTouchIdle || wgs == 0) return dim3(wgs);
  t.wgs = (unsigned)idle;
  return dim3(wgs, 1 + (t.wgs + wgs - 1) / wgs);
}

namespace {
// Panels of 4 column tiles, not 8: fewer bytes for an XCD's L2 where a launch has few row tiles (us, weights rotating
// through 24 layers, M x N x K 261 x 1,024 x 4,096 11.2 -> 10.1, 261 x 1,024 x 1,024 5.2 -> 4.9, 261 x 3,072 x 1,024
// 6.4 -> 6.2).  64-row tiles whose K is long or whose rows are many are the exception: there
// panels of 8 keep a row of a with two XCDs instead of four (us, M x N x K, weights in HBM, panels of 4 and 8:
// 513 x 1,024 x 4,096 15.7, 15.8, 566 19.6, 19.5, 700 20.3, 19.9, 900 16.6, 16.6, 1,004 19.6, 19.3, at 9 to 16 row tiles, and from
// the last-level cache the same to 1 %; 1,004 x 896 x 3,584 17.9, 17.5; but 673 x 768 x 3,072 11.4, 11.8, 1,280 14.3, 14.4;
// 900 x 640 x 2,560 10.7, 11.1; 1,100 x 512 x 2,048 8.6, 9.0, 1,700 8.8, 9.1, 1,800 9.4, 9.2, 2,048 10.0, 9.5).
void lbm_linear_panels(LinearArgs& p, int rows, int splits) {
  lbm_set_panels(p, rows && !(rows == 64 && splits > 1 && (p.K > 3072 || p.m_tiles >= 28)) ? 2 : 3);
}
}  // namespace

namespace {
// What a launch runs as (and p's tile counts): tiles of `big` rows x 256 columns, of `rows` rows x 64, or of 128 rows x `tn`
// (x 256: wider); `splits` slices of K.  heads: of the qkv projection, whose tiles must not straddle q | k | v.
struct LinearForm { int big, rows, tn, splits; bool wider; };
LinearForm lbm_linear_form(LinearArgs& p, int epilogue, int heads, bool may_split) {
  LinearForm f = {0, 0, 0, 1, false};
  const bool qkv = epilogue == kEpiQkvPrepare;
  // (256 columns: four whole heads each)
  if (qkv ? (heads & 3) == 0 : epilogue != LBM_LINEAR_BIAS_RESIDUAL) f.big = lbm_linear_big_tiles(p);
  if (f.big) {
    lbm_linear_panels(p, 0, 1);
    return f;
  }
  f.tn = lbm_linear_tiles(p);
  if (qkv && f.tn == 128 && (heads & 1)) {   // (128 columns: an even number of heads)
    f.tn = 64;
    p.n_tiles = p.N / 64;
  }
  if (may_split) f.splits = lbm_linear_splits(p, epilogue);
  f.rows = lbm_linear_rows_tiles(p, f.tn, f.splits);
  f.wider = !f.rows && (!qkv || (heads & 3) == 0) && f.splits == 1 && f.tn == 128 && lbm_linear_wider(p);
  lbm_linear_panels(p, f.rows, f.splits);
  return f;
}
}  // namespace

LbmAsks lbm_linear_asks(int M, int N, int K, int epilogue, int heads, bool may_split) {
  LinearArgs p = {};
  p.M = M; p.N = N; p.K = K;
  const LinearForm f = lbm_linear_form(p, heads ? kEpiQkvPrepare : epilogue, heads, may_split);
  if ((f.rows || f.splits == 1) && lbm_idle_cus((long long)p.m_tiles * p.n_tiles) >= kTouchIdle) return f.big || f.wider ? LBM_ASKS_WIDE_IDLE : LBM_ASKS_IDLE;
  return f.big || f.wider ? LBM_ASKS_NOT : LBM_ASKS_WAVES;
}

int lbm_launch_linear(const void* a, const lbm_row_norm* a_norm, const void* w, const float* bias, const float* gamma,
                      const void* residual, void* out, float* out_stats, int M, int N, int K, int epilogue,
                      void* workspace, size_t workspace_bytes, hipStream_t stream) {
  if (M == 0) {
    lbm_set_prefetch_hint({});   // a hint is for the next call, whatever that call does
    return LBM_OK;
  }
  if (K % kGK != 0 || N % 64 != 0)
    return lbm_fail(LBM_ERR_UNSUPPORTED, "lbm_linear: K must be a multiple of 128 and N of 64 (got K %d, N %d)", K, N);
  if (!lbm_offsets_fit(M, N, K))
    return lbm_fail(LBM_ERR_UNSUPPORTED, "lbm_linear: M * K and N * K must stay below 2^31 elements (32-bit byte offsets), got %d x %d x %d", M, N, K);
  if (a_norm && epilogue == LBM_LINEAR_BIAS_RESIDUAL)
    return lbm_fail(LBM_ERR_UNSUPPORTED, "lbm_linear: no row standardisation with the residual epilogue");
  if (out_stats && epilogue != LBM_LINEAR_BIAS_RESIDUAL)
    return lbm_fail(LBM_ERR_UNSUPPORTED, "lbm_linear: row statistics come with the residual epilogue only");
  LinearArgs p = {};
  p.stats_out = out_stats;
  p.a = (const unsigned short*)a;
  p.w = (const unsigned short*)w;
  p.bias = bias;
  p.gamma = gamma;
  p.res = (const unsigned short*)residual;
  p.out = (unsigned short*)out;
  p.M = M; p.N = N; p.K = K;
  lbm_take_prefetch_hint(p.touch);
  if (int rc = lbm_set_row_norm(p, a_norm, "lbm_linear_norm")) return rc;
  const bool lna = a_norm != nullptr;
  const dim3 block(kGThreads), block_s(lbm_linear_threads(128));
  const LinearForm f = lbm_linear_form(p, epilogue, 0, workspace && workspace_bytes >= lbm_linear_workspace_for(M, N, K, epilogue));
  if (epilogue == LBM_LINEAR_BIAS || epilogue == LBM_LINEAR_BIAS_GELU) {
    if (const int bm = f.big) {
      const dim3 grid_b = lbm_touch_grid(p.touch, (unsigned)(p.m_tiles * p.n_tiles));
#define LBM_BIG_LAUNCH(E, L)                                                                                         \
      {                                                                                                              \
        if (bm == 256) hipLaunchKernelGGL((lbm_linear_bf16_big_kernel<256, E, 0, false, L>), grid_b, block, 0, stream, p); \
        else if (bm == 192) hipLaunchKernelGGL((lbm_linear_bf16_big_kernel<192, E, 0, false, L>), grid_b, dim3(lbm_big_threads(192)), 0, stream, p);           \
        else hipLaunchKernelGGL((lbm_linear_bf16_big_kernel<128, E, 0, false, L>), grid_b, dim3(lbm_big_threads(128)), 0, stream, p);           \
      }
      if (epilogue == LBM_LINEAR_BIAS && lna) LBM_BIG_LAUNCH(LBM_LINEAR_BIAS, true)
      else if (epilogue == LBM_LINEAR_BIAS) LBM_BIG_LAUNCH(LBM_LINEAR_BIAS, false)
      else if (lna) LBM_BIG_LAUNCH(LBM_LINEAR_BIAS_GELU, true)
      else LBM_BIG_LAUNCH(LBM_LINEAR_BIAS_GELU, false)
#undef LBM_BIG_LAUNCH
      return lbm_check_launch("lbm_linear_bf16_big_kernel");
    }
  }
  const int splits = f.splits;
  // (where several workgroups share a tile, one that is not its last would see the other's store; one workgroup per tile
  // would not, but what a call with a workspace accepts does not depend on which of the two its sizes give)
  if (splits > 1 && residual == out)
    return lbm_fail(LBM_ERR_INVALID, "lbm_linear_norm: with a workspace the residual may not alias out");
  if (const int tm = f.rows) {
    const dim3 grid_r = lbm_touch_grid(p.touch, (unsigned)(p.m_tiles * p.n_tiles)), block_r(lbm_rows_threads(tm));
#define LBM_ROWS_LAUNCH(E, S, L)                                                                                                \
  {                                                                                                                             \
    if (S == 1 && tm == 96) hipLaunchKernelGGL((lbm_linear_bf16_rows_kernel<E, 96, 1, 0, false, L>), grid_r, block_r, 0, stream, p); \
    else if (tm == 64) hipLaunchKernelGGL((lbm_linear_bf16_rows_kernel<E, 64, S, 0, false, L>), grid_r, block_r, 0, stream, p);       \
    else hipLaunchKernelGGL((lbm_linear_bf16_rows_kernel<E, 32, S, 0, false, L>), grid_r, block_r, 0, stream, p);                \
  }
    if (epilogue == LBM_LINEAR_BIAS && lna) LBM_ROWS_LAUNCH(LBM_LINEAR_BIAS, 1, true)
    else if (epilogue == LBM_LINEAR_BIAS) LBM_ROWS_LAUNCH(LBM_LINEAR_BIAS, 1, false)
    else if (epilogue == LBM_LINEAR_BIAS_GELU && lna) LBM_ROWS_LAUNCH(LBM_LINEAR_BIAS_GELU, 1, true)
    else if (epilogue == LBM_LINEAR_BIAS_GELU) LBM_ROWS_LAUNCH(LBM_LINEAR_BIAS_GELU, 1, false)
    else if (epilogue == LBM_LINEAR_BIAS_RESIDUAL && splits == 1) LBM_ROWS_LAUNCH(LBM_LINEAR_BIAS_RESIDUAL, 1, false)
    else if (epilogue == LBM_LINEAR_BIAS_RESIDUAL && splits == 2) LBM_ROWS_LAUNCH(LBM_LINEAR_BIAS_RESIDUAL, 2, false)
    else if (epilogue == LBM_LINEAR_BIAS_RESIDUAL) LBM_ROWS_LAUNCH(LBM_LINEAR_BIAS_RESIDUAL, 4, false)
    else return lbm_fail(LBM_ERR_INVALID, "lbm_linear: unknown epilogue %d", epilogue);
#undef LBM_ROWS_LAUNCH
    return lbm_check_launch("lbm_linear_bf16_rows_kernel");
  }
  if (splits > 1) {
    p.k_splits = splits;
    p.split_counters = (unsigned*)workspace;
    p.split_part = (float*)((char*)workspace + kSplitCounterBytes);
    const dim3 grid_s((unsigned)(p.m_tiles * p.n_tiles * splits));
    // (128 tiles at most, so they have 64 columns)
    hipLaunchKernelGGL((lbm_linear_bf16_kernel<LBM_LINEAR_BIAS_RESIDUAL, 64, 0, false, false, true>), grid_s, block_s, 0, stream, p);
    return lbm_check_launch("lbm_linear_bf16_kernel<split K>");
  }
  const bool wide = f.tn == 128, wider = f.wider;
  const dim3 grid = lbm_touch_grid(p.touch, (unsigned)(p.m_tiles * p.n_tiles));
#define LBM_LINEAR_LAUNCH(E, L)                                                                                  \
  {                                                                                                              \
    if (wider) hipLaunchKernelGGL((lbm_linear_bf16_kernel<E, 256, 0, false, L>), grid, block, 0, stream, p);     \
    else if (wide) hipLaunchKernelGGL((lbm_linear_bf16_kernel<E, 128, 0, false, L>), grid, block_s, 0, stream, p); \
    else hipLaunchKernelGGL((lbm_linear_bf16_kernel<E, 64, 0, false, L>), grid, block_s, 0, stream, p);          \
  }
  if (epilogue == LBM_LINEAR_BIAS && lna) LBM_LINEAR_LAUNCH(LBM_LINEAR_BIAS, true)
  else if (epilogue == LBM_LINEAR_BIAS) LBM_LINEAR_LAUNCH(LBM_LINEAR_BIAS, false)
  else if (epilogue == LBM_LINEAR_BIAS_GELU && lna) LBM_LINEAR_LAUNCH(LBM_LINEAR_BIAS_GELU, true)
  else if (epilogue == LBM_LINEAR_BIAS_GELU) LBM_LINEAR_LAUNCH(LBM_LINEAR_BIAS_GELU, false)
  else if (epilogue == LBM_LINEAR_BIAS_RESIDUAL) LBM_LINEAR_LAUNCH(LBM_LINEAR_BIAS_RESIDUAL, false)
  else return lbm_fail(LBM_ERR_INVALID, "lbm_linear: unknown epilogue %d", epilogue);
#undef LBM_LINEAR_LAUNCH
  return lbm_check_launch("lbm_linear_bf16_kernel");
}

int lbm_launch_qkv_linear_prepare(const void* a, const lbm_row_norm* a_norm, const void* w, const float* bias, int M, int K,
                                  const float* q_norm_w, const float* q_norm_b, const float* k_norm_w,
                                  const float* k_norm_b, float norm_eps, float q_scale, const float* rope_cs, int rope_layout,
                                  void* q_out, void* k_out, void* v_out, void* pool, const int32_t* append_rows,
                                  int num_heads, int page_size, hipStream_t stream) {
  if (M == 0) return LBM_OK;
  const int N = 3 * num_heads * 64;
  if (K % kGK != 0) return lbm_fail(LBM_ERR_UNSUPPORTED, "lbm_qkv_linear_prepare: K must be a multiple of 128 (got %d)", K);
  if (!lbm_offsets_fit(M, N, K))
    return lbm_fail(LBM_ERR_UNSUPPORTED, "lbm_qkv_linear_prepare: M * K and N * K must stay below 2^31 elements (32-bit byte offsets), got %d x %d x %d", M, N, K);
  LinearArgs p = {};
  p.a = (const unsigned short*)a;
  p.w = (const unsigned short*)w;
  p.bias = bias;
  p.out = (unsigned short*)q_out;
  p.M = M; p.N = N; p.K = K;
  lbm_take_prefetch_hint(p.touch);
  p.q_norm_w = q_norm_w; p.q_norm_b = q_norm_b; p.k_norm_w = k_norm_w; p.k_norm_b = k_norm_b;
  p.rope_cs = rope_cs;
  p.k_out = (unsigned short*)k_out; p.v_out = (unsigned short*)v_out;
  p.pool = (unsigned short*)pool;
  p.append_rows = append_rows;
  p.eps = norm_eps;
  p.q_scale = q_scale;
  p.num_heads = num_heads; p.page_size = page_size;
  if (int rc = lbm_set_row_norm(p, a_norm, "lbm_qkv_linear_prepare_norm")) return rc;
  const bool lna = a_norm != nullptr;
  const int rope = !rope_cs ? 0 : (rope_layout == LBM_ROPE_INTERLEAVED ? 1 : 2);
  const bool norm = q_norm_w != nullptr;
  const LinearForm f = lbm_linear_form(p, kEpiQkvPrepare, num_heads, false);
  if (const int bm = f.big) {
    const dim3 grid_b = lbm_touch_grid(p.touch, (unsigned)(p.m_tiles * p.n_tiles)), block_b(lbm_big_threads(bm));
#define LBM_QKV_BIG_M(BM, R, NRM)                                                                                               \
    {                                                                                                                           \
      if (lna) hipLaunchKernelGGL((lbm_linear_bf16_big_kernel<BM, kEpiQkvPrepare, R, NRM, true>), grid_b, block_b, 0, stream, p);  \
      else hipLaunchKernelGGL((lbm_linear_bf16_big_kernel<BM, kEpiQkvPrepare, R, NRM, false>), grid_b, block_b, 0, stream, p);     \
    }
#define LBM_QKV_BIG(R, NRM)                                                  \
    {                                                                        \
      if (bm == 256) LBM_QKV_BIG_M(256, R, NRM) else if (bm == 192) LBM_QKV_BIG_M(192, R, NRM) else LBM_QKV_BIG_M(128, R, NRM) \
    }
    if (rope == 0 && !norm) LBM_QKV_BIG(0, false)
    else if (rope == 0) LBM_QKV_BIG(0, true)
    else if (rope == 1 && !norm) LBM_QKV_BIG(1, false)
    else if (rope == 1) LBM_QKV_BIG(1, true)
    else if (!norm) LBM_QKV_BIG(2, false)
    else LBM_QKV_BIG(2, true)
#undef LBM_QKV_BIG
#undef LBM_QKV_BIG_M
    return lbm_check_launch("lbm_linear_bf16_big_kernel<qkv prepare>");
  }
  const bool wide = f.tn == 128;
  if (const int tm = f.rows) {
    const dim3 grid_r = lbm_touch_grid(p.touch, (unsigned)(p.m_tiles * p.n_tiles)), block_r(lbm_rows_threads(tm));
#define LBM_QKV_ROWS_T(T, R, NRM)                                                                                                       \
  {                                                                                                                                     \
    if (lna) hipLaunchKernelGGL((lbm_linear_bf16_rows_kernel<kEpiQkvPrepare, T, 1, R, NRM, true>), grid_r, block_r, 0, stream, p);       \
    else hipLaunchKernelGGL((lbm_linear_bf16_rows_kernel<kEpiQkvPrepare, T, 1, R, NRM, false>), grid_r, block_r, 0, stream, p);          \
  }
#define LBM_QKV_ROWS(R, NRM)                                                       \
  {                                                                                \
    if (tm == 96) LBM_QKV_ROWS_T(96, R, NRM) else if (tm == 64) LBM_QKV_ROWS_T(64, R, NRM) else LBM_QKV_ROWS_T(32, R, NRM) \
  }
    if (rope == 0 && !norm) LBM_QKV_ROWS(0, false)
    else if (rope == 0) LBM_QKV_ROWS(0, true)
    else if (rope == 1 && !norm) LBM_QKV_ROWS(1, false)
    else if (rope == 1) LBM_QKV_ROWS(1, true)
    else if (!norm) LBM_QKV_ROWS(2, false)
    else LBM_QKV_ROWS(2, true)
#undef LBM_QKV_ROWS
#undef LBM_QKV_ROWS_T
    return lbm_check_launch("lbm_linear_bf16_rows_kernel<qkv prepare>");
  }
  const dim3 grid = lbm_touch_grid(p.touch, (unsigned)(p.m_tiles * p.n_tiles)), block(lbm_linear_threads(f.wider ? 256 : 128));
#define LBM_QKV_LAUNCH_L(R, NRM, L)                                                                                   \
  {                                                                                                                   \
    if (f.wider) hipLaunchKernelGGL((lbm_linear_bf16_kernel<kEpiQkvPrepare, 256, R, NRM, L>), grid, block, 0, stream, p); \
    else if (wide) hipLaunchKernelGGL((lbm_linear_bf16_kernel<kEpiQkvPrepare, 128, R, NRM, L>), grid, block, 0, stream, p); \
    else hipLaunchKernelGGL((lbm_linear_bf16_kernel<kEpiQkvPrepare, 64, R, NRM, L>), grid, block, 0, stream, p);       \
  }
#define LBM_QKV_LAUNCH(R, NRM)                                                                                        \
  {                                                                                                                   \
    if (lna) LBM_QKV_LAUNCH_L(R, NRM, true) else LBM_QKV_LAUNCH_L(R, NRM, false)                                      \
  }
  if (rope == 0 && !norm) LBM_QKV_LAUNCH(0, false)
  else if (rope == 0) LBM_QKV_LAUNCH(0, true)
  else if (rope == 1 && !norm) LBM_QKV_LAUNCH(1, false)
  else if (rope == 1) LBM_QKV_LAUNCH(1, true)
  else if (!norm) LBM_QKV_LAUNCH(2, false)
  else LBM_QKV_LAUNCH(2, true)
#undef LBM_QKV_LAUNCH_L
#undef LBM_QKV_LAUNCH
  return lbm_check_launch("lbm_linear_bf16_kernel<qkv prepare>");
}
