// fp32 paged attention forward for gfx950 at head_dim 64 (the reference's force_fp32 mode,
// lingbot_map/layers/flashinfer_cache.py:118-127,372-383), on the bf16 matrix instructions.
//
// A float is the exact sum of three bf16 values (8 + 8 + 8 significant bits, same exponent range), so a
// product of two floats is the sum of nine products of bf16 values, each exact in fp32 (Henry, Tang,
// Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype For Higher-Precision Computations",
// ARITH 2019).  Eight of them are computed; the ninth, of the two smallest terms, is below 2^-31 of the
// product.  The leading products and the other seven have accumulators of their own, which meet in one
// fp32 addition: a product alone comes out as fp32 rounds it, and a sum over head dimensions or tokens
// takes a rounding of its full size per 16 or 32 terms.  Six products in one accumulator were a quarter
// faster (29 and 187 us below) but left up to 1.2 x 2^-23 of a product out, and took six roundings per 16
// terms.  Largest error of a score against float64, in units of 2^-24 of its size, for 1 and 64 products,
// v_mfma_f32_16x16x4_f32 / six / eight: 1.1 / 3.6 / 1.1 and 8.5 / 6.3 / 1.0; relative error of the output at
// 4,000 tokens 6.5e-7 / 4.3e-7 / 1.7e-7.
//
// A bf16 instruction does 16 times the work of an fp32 one per cycle; the kernel runs at 1.1 PFLOP/s of
// bf16 products (137 TFLOP/s of fp32 ones).  At 8,032 tokens the matrix pipe works 58 % and the vector ALU (7 splits,
// sums and exponentials per MFMA) 62 % of the cycles, at 1.7 GHz; with six products, fences that spread the
// operand reads and splits over the MFMAs and a tenth fewer vector instructions changed nothing.  Measured,
// 1,004 rows x 16 heads: 1,004 tokens 48 -> 37 us, 8,032 tokens 337 -> 240 us against the fp32 instruction.
// Infinities have a pass of their own at the end of the kernel.
//
// One workgroup = eight wavefronts on 64 query rows of one head, or on 32 where those of 64 would leave CUs idle
// (lbm_f32_row_blocks).  A wavefront takes every eighth
// 32-token tile of the KV list, for all the rows (so that a value of K or V is split once per 64 rows),
// from an LDS buffer of its own: nothing is shared inside the loop and there is no barrier in it.  The
// rows travel global -> LDS directly as fp32 (global_load_lds_dwordx4), the next K tile as soon as this
// one's fragments are read, the next V tile likewise, so either has half an iteration to land and one
// buffer of each suffices.  Fragments are read as fp32 in operand layout and split in registers: K as
// two b128 per 16-wide k-step, V^T as eight dwords of eight rows (no transpose pass).  The eight
// partial results meet through LDS at the end.
//
//   S^T = K Q^T     v_mfma_f32_32x32x16_bf16, A = K rows, B = Q (split once, kept in LDS)
//   P   = exp2(S - m)   m: a reference that is raised only when a score exceeds it by 8 (in log2
//                   units), so the rescale of O is off the common path; numerators stay below 2^8
//   O^T += V^T P^T  B = P^T straight from the registers the split wrote
#include <hip/hip_runtime.h>
#include "lbm_internal.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(8))) float f32x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;

namespace {

constexpr int kWaves = 8, kThreads = kWaves * 64;
constexpr int kAppendPieces = 4;        // 16-byte pieces of K and of V per thread of a workgroup that appends
constexpr int kTile = 32;               // KV tokens per tile
constexpr int kTileBytes = kTile * 64 * 4;
constexpr int kEntryBytes = 256 + kTile * 2 * 8;   // a wavefront's row entries, and the K and V addresses they name
constexpr int kOffEntries = kWaves * 2 * kTileBytes, kOffQ = kOffEntries + kWaves * kEntryBytes;
constexpr int kOStride = 68;            // floats per row of a partial output parked in LDS
constexpr int lbm_f32_lds_bytes(int rows) {
  const int merge = kWaves * (rows * kOStride + 2 * rows) * 4, loop = kOffQ + 3 * rows * 64 * 2;
  return loop > merge ? loop : merge;
}
static_assert(lbm_f32_lds_bytes(64) <= 160 * 1024, "LDS of a CU");
constexpr float kSlack = 8.f;           // a score this far above the reference raises it

// value of the other half-wave's lane beside the own one
__device__ __forceinline__ void swap_halves(float x, float& lo, float& hi) {
  float a = x, b = x;
  asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
  lo = a;
  hi = b;
}

__device__ __forceinline__ unsigned bits(float x) { return __builtin_bit_cast(unsigned, x); }
__device__ __forceinline__ float top16(float x) { return __builtin_bit_cast(float, bits(x) & 0xffff0000u); }

// x = p[0] + p[1] + p[2] exactly, by truncation (K and V)
__device__ __forceinline__ void split_truncated(const f32x8& x, bf16x8 (&p)[3]) {
  u32x4 w[3];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float a = x[2 * i], b = x[2 * i + 1];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      w[k][i] = __builtin_amdgcn_perm(bits(b), bits(a), 0x07060302u);   // {a, b} >> 16
      a -= top16(a);
      b -= top16(b);
    }
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) p[k] = __builtin_bit_cast(bf16x8, w[k]);
}
// the same by rounding to nearest (Q and the numerators: with one operand's remainders of either
// sign, what the left-out product adds has no preferred sign)
__device__ __forceinline__ void split_rounded(f32x8 x, bf16x8 (&p)[3]) {
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    p[k] = __builtin_convertvector(x, bf16x8);
    if (k < 2) {
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] -= (float)p[k][i];
    }
  }
}
// hi[i] += the leading products of a * b[i] over 16 k's, lo[i] += the seven others, small ones first
template <int QB>
__device__ __forceinline__ void mfma_split(const bf16x8 (&a)[3], const bf16x8 (&b)[QB][3], f32x16 (&hi)[QB], f32x16 (&lo)[QB]) {
  constexpr int pa[7] = {2, 1, 2, 0, 1, 1, 0}, pb[7] = {1, 2, 0, 2, 1, 0, 1};
#pragma unroll
  for (int i = 0; i < 7; ++i)
#pragma unroll
    for (int q = 0; q < QB; ++q) lo[q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[pa[i]], b[q][pb[i]], lo[q], 0, 0, 0);
#pragma unroll
  for (int q = 0; q < QB; ++q) hi[q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[q][0], hi[q], 0, 0, 0);
}

// loads of this wavefront still allowed in flight (expcnt and lgkmcnt untouched), and LDS reads done
#define LBM_LOADS_LEFT(N) asm volatile("s_waitcnt vmcnt(%0)" : : "i"(N) : "memory")
#define LBM_LDS_READ() asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory")

}  // namespace

// APPEND: workgroups behind the attention's carry the append; an instance of its own, as asking which a workgroup is costs
// every launch 0.2 to 0.4 us (400 rows over themselves: 18.3, 18.8)
// QB: blocks of 32 query rows per workgroup, 2 or 1
template <int S, bool APPEND, int QB>
__global__ __launch_bounds__(kThreads) void lbm_attn_f32_d64_kernel(AttnArgsF32<S> a) {
  constexpr int kRows = 32 * QB;
  constexpr int kQPlane = kRows * 64;     // bf16 of a Q plane: unpadded rows, chunk c of row r at c ^ ((r >> 1) & 7)
  __shared__ __attribute__((aligned(1024))) unsigned char lds[lbm_f32_lds_bytes(kRows)];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n32 = lane & 31, g = lane >> 5;
  // (what the first loads need of the arguments, the first stream's beside the launch's, in one trip,
  // without integer divisions behind it: 282 own rows of 8 heads 15.1 -> 14.7 us, a block of 148 rows over 740 tokens 26.4 -> 25.6)
  lbm_attn_stream sp = a.s[0];
  asm volatile("" : : "s"(a.q), "s"(a.pool), "s"(a.self_k), "s"(a.self_v), "s"(a.kv_rows), "s"(a.live_kv_tokens), "s"(a.num_heads), "s"(a.page_size), "s"(a.scale_log2),
               "s"(a.n_streams), "s"(a.per_heads), "s"(a.per_eighth), "s"(sp.q_begin), "s"(sp.q_rows), "s"(sp.kv_row_begin), "s"(sp.kv_tokens),
               "s"(APPEND ? a.wg_begin[S] : 0));
  if (APPEND && __builtin_expect((int)blockIdx.x >= a.wg_begin[S], 0)) {
    lbm_append_pieces<kAppendPieces>(a.self_k, a.self_v, const_cast<float*>(a.pool), a.append_rows, a.append_tokens, a.num_heads * 16, a.page_size,
                      (int)blockIdx.x - a.wg_begin[S], kThreads);
    return;
  }
  int b = 0;
  if (S > 1 && a.n_streams > 1) {
#pragma unroll
    for (int i = 1; i < S; ++i) b += (int)((unsigned)(a.wg_begin[i] - 1 - (int)blockIdx.x) >> 31);   // (beyond the streams: more than any workgroup)
    sp = a.s[b];
  }
  const int H = a.num_heads, local = (int)blockIdx.x - a.wg_begin[b];
  int head, qt;
  if ((H & 7) == 0) {   // the query blocks of one head on one XCD (blockIdx mod 8): its L2 serves their K/V
    qt = lbm_divide(local >> 3, H >> 3, a.per_eighth, head);
    head = head * 8 + (local & 7);
  } else {
    qt = lbm_divide(local, H, a.per_heads, head);
  }
  const int q_row0 = qt * kRows;
  if (q_row0 >= sp.q_rows) return;   // padding between streams (whole workgroups)
  const int kv_tokens = max(a.live_kv_tokens ? a.live_kv_tokens[sp.live_at] : sp.kv_tokens, 0);
  const int n_tiles = (kv_tokens + kTile - 1) / kTile, last_token = max(kv_tokens - 1, 0);
  const int out_row = (tid >> 3) % kRows, out_d = (tid & 7) * 8;   // this thread's part of the result
  const bool out_ok = q_row0 + out_row < sp.q_rows && tid < kRows * 8;
  float* out = a.out + ((size_t)(sp.q_begin + q_row0 + out_row) * H + head) * 64 + out_d;
  if (n_tiles == 0) {   // nothing visible: zeros (lingbot_map/layers/flashinfer_cache.py:368-370)
    if (out_ok) ((f32x4*)out)[0] = ((f32x4*)out)[1] = f32x4{0.f, 0.f, 0.f, 0.f};
    return;
  }

  // ---- this wavefront's buffers and where its rows come from
  unsigned char* raw_k = lds + wave * (2 * kTileBytes);
  unsigned char* raw_v = raw_k + kTileBytes;
  int* entries = (int*)(lds + kOffEntries + wave * kEntryBytes);
  unsigned long long* sources = (unsigned long long*)(entries + 64);   // [K | V][row of the tile]
  auto lds_at = [](const void* p) { return __builtin_amdgcn_readfirstlane((unsigned)(size_t)(__attribute__((address_space(3))) const void*)p); };
  const unsigned m0_k = lds_at(raw_k), m0_v = lds_at(raw_v), m0_e = lds_at(entries);
  const unsigned row_bytes = (unsigned)H * 256u;
  // lanes 0-31 work out where the tile's K rows are, lanes 32-63 where its V rows are
  const char* pool_rows = (const char*)(a.pool + (size_t)head * 64) + (g ? (size_t)a.page_size * row_bytes : 0);
  const char* own_rows = (const char*)((g ? a.self_v : a.self_k) + (size_t)head * 64);
  const int32_t* rows = a.kv_rows + sp.kv_row_begin;
  // A load instruction brings four rows of 256 bytes; lane l asks for the 16-byte chunk that belongs
  // at ITS place: chunk c of K row r sits at c ^ (r & 15) (b128 reads of 16 rows x one chunk: all 64
  // banks), chunk c of V row r at c ^ 8 ((r >> 2) & 1) (dword reads of rows r and r + 4: other halves)
  unsigned chunk_k[4], chunk_v[2];
#pragma unroll
  for (int j = 0; j < 4; ++j) chunk_k[j] = (unsigned)(((lane & 15) ^ (4 * j | (lane >> 4))) * 16);
#pragma unroll
  for (int j = 0; j < 2; ++j) chunk_v[j] = (unsigned)(((lane & 15) ^ (8 * j)) * 16);
  auto load_rows = [&](bool v) {
    unsigned long long at[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) at[j] = sources[(v ? kTile : 0) + (lane >> 4) + 4 * j];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const unsigned long long src = at[j] + (v ? chunk_v[j & 1] : chunk_k[j & 3]);
      asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(src), "s"((v ? m0_v : m0_k) + j * 1024u) : "memory", "m0");
    }
  };
  auto load_entries = [&](int t) {   // (tokens past the last re-read it: finite data, masked below)
    const int32_t* src = rows + min(t * kTile + n32, last_token);
    asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dword %0, off" : : "v"(src), "s"(m0_e) : "memory", "m0");
  };
  // (one address per lane instead of sixteen lanes working out the same one, eight times per load)
  auto read_entries = [&]() {
    const int e = entries[n32];   // negative entries name rows of the caller's own K/V
    const char* src = (e < 0 ? own_rows : pool_rows) + (unsigned long long)(unsigned)(e ^ (e >> 31)) * row_bytes;
    sources[lane] = (unsigned long long)src;
  };

  // ---- Q: scaled, split once, parked in LDS as three planes of bf16
  unsigned short* lds_q = (unsigned short*)(lds + kOffQ);
  {
    const int r = min(q_row0 + out_row, sp.q_rows - 1);   // rows past the last one re-read it (never stored)
    const f32x4* qp = (const f32x4*)(a.q + ((size_t)(sp.q_begin + r) * H + head) * 64 + out_d);
    const f32x4 x0 = qp[0] * a.scale_log2, x1 = qp[1] * a.scale_log2;
    bf16x8 p[3];
    split_rounded(f32x8{x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]}, p);
#pragma unroll
    for (int k = 0; k < 3; ++k) *(bf16x8*)&lds_q[k * kQPlane + out_row * 64 + ((tid & 7) ^ ((out_row >> 1) & 7)) * 8] = p[k];
  }
  __syncthreads();

  f32x16 o[QB][2];              // o[qb][db][i]: d = 32 db + 8 (i / 4) + 4 g + i % 4, q = 32 qb + n32
  float m[QB], l[QB];           // reference of the row, this lane's share of its sum
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    m[qb] = -INFINITY;
    l[qb] = 0.f;
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[qb][db][i] = 0.f;
  }

  if (wave < n_tiles) {
    load_entries(wave);
    LBM_LOADS_LEFT(0);
    read_entries();
    load_rows(false);
    load_entries(wave + kWaves);
    load_rows(true);
  }
  // In flight at the top of an iteration, oldest first: K (8 loads), entries of the next tile (1), V (8)
  for (int t = wave; t < n_tiles; t += kWaves) {
    LBM_LOADS_LEFT(9);
    // ---- S^T = K Q^T: s[qb][i] is kv = 8 (i / 4) + 4 g + i % 4, q = 32 qb + n32
    f32x16 s[QB], s_lo[QB];
#pragma unroll
    for (int qb = 0; qb < QB; ++qb)
#pragma unroll
      for (int i = 0; i < 16; ++i) s[qb][i] = s_lo[qb][i] = 0.f;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const int c = ks * 4 + g * 2;
      const f32x4 k0 = *(const f32x4*)(raw_k + n32 * 256 + ((c ^ (n32 & 15)) * 16));
      const f32x4 k1 = *(const f32x4*)(raw_k + n32 * 256 + (((c + 1) ^ (n32 & 15)) * 16));
      bf16x8 kp[3], qp[QB][3];
      split_truncated(f32x8{k0[0], k0[1], k0[2], k0[3], k1[0], k1[1], k1[2], k1[3]}, kp);
#pragma unroll
      for (int qb = 0; qb < QB; ++qb)
#pragma unroll
        for (int k = 0; k < 3; ++k)
          qp[qb][k] = *(const bf16x8*)&lds_q[k * kQPlane + (qb * 32 + n32) * 64 + ((ks * 2 + g) ^ ((n32 >> 1) & 7)) * 8];
      mfma_split<QB>(kp, qp, s, s_lo);
    }
#pragma unroll
    for (int qb = 0; qb < QB; ++qb)
#pragma unroll
      for (int i = 0; i < 16; ++i) s[qb][i] += s_lo[qb][i];
    // ---- the next K tile: its entries have landed, this one's fragments are read
    LBM_LOADS_LEFT(8);
    LBM_LDS_READ();
    read_entries();
    load_rows(false);
    load_entries(t + 2 * kWaves);
    // ---- softmax
    const int n_valid = kv_tokens - t * kTile;
    if (n_valid < kTile) {   // the ragged last tile
#pragma unroll
      for (int qb = 0; qb < QB; ++qb)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (8 * (i >> 2) + 4 * g + (i & 3) >= n_valid) s[qb][i] = -INFINITY;
    }
    float mx[QB];
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      float x = s[qb][0];
#pragma unroll
      for (int i = 1; i < 16; ++i) x = fmaxf(x, s[qb][i]);
      float lo, hi;
      swap_halves(x, lo, hi);
      mx[qb] = fmaxf(lo, hi);
    }
    if (__builtin_amdgcn_ballot_w64(mx[0] > m[0] + kSlack || mx[QB - 1] > m[QB - 1] + kSlack)) {   // (always on the first tile)
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        // (block by block: what a row's sums are rounded against does not depend on how many blocks share its workgroup)
        if (QB > 1 && !__builtin_amdgcn_ballot_w64(mx[qb] > m[qb] + kSlack)) continue;
        const float to = fmaxf(m[qb], mx[qb]);
        const float alpha = __builtin_amdgcn_exp2f(m[qb] - to);
        m[qb] = to;
        l[qb] *= alpha;
#pragma unroll
        for (int db = 0; db < 2; ++db)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[qb][db][i] *= alpha;
      }
    }
    bf16x8 p[2][QB][3];   // [k-step][qb][plane]: element j is kv = 16 kk + 4 g + j % 4 + 8 (j / 4)
#pragma unroll
    for (int qb = 0; qb < QB; ++qb)
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        f32x8 x;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          x[j] = __builtin_amdgcn_exp2f(s[qb][kk * 8 + j] - m[qb]);
        }
        l[qb] += ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
        split_rounded(x, p[kk][qb]);
      }
    // ---- O^T += V^T P^T, the tile's sums in registers that held the scores before they join O
    LBM_LOADS_LEFT(9);
#pragma unroll
    for (int db = 0; db < 2; ++db) {
      f32x16 hi[QB], lo[QB];
#pragma unroll
      for (int qb = 0; qb < QB; ++qb)
#pragma unroll
        for (int i = 0; i < 16; ++i) hi[qb][i] = lo[qb][i] = 0.f;
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        f32x8 x;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int r = kk * 16 + (j & 3) + 8 * (j >> 2);   // + 4 g
          x[j] = *(const float*)(raw_v + (4 * g + r) * 256 + ((db * 8 + (n32 >> 2)) ^ (8 * g)) * 16 + (n32 & 3) * 4);
        }
        bf16x8 vp[3];
        split_truncated(x, vp);
        mfma_split<QB>(vp, p[kk], hi, lo);
      }
#pragma unroll
      for (int qb = 0; qb < QB; ++qb)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[qb][db][i] += hi[qb][i] + lo[qb][i];
    }
    LBM_LDS_READ();
    load_rows(true);
  }
  LBM_LOADS_LEFT(0);   // (the loads past the last tile too: the area is reused)
  __syncthreads();

  // ---- merge the wavefronts' partial results through LDS
  float* so = (float*)lds + wave * (kRows * kOStride);
  float* sl = (float*)lds + kWaves * (kRows * kOStride);   // [wave][row] row sums, then [wave][row] references
  float* sm = sl + kWaves * kRows;
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
      for (int c4 = 0; c4 < 4; ++c4)
        *(f32x4*)&so[(qb * 32 + n32) * kOStride + db * 32 + c4 * 8 + g * 4] =
            f32x4{o[qb][db][c4 * 4], o[qb][db][c4 * 4 + 1], o[qb][db][c4 * 4 + 2], o[qb][db][c4 * 4 + 3]};
    float lo, hi;
    swap_halves(l[qb], lo, hi);
    if (g == 0) {
      sl[wave * kRows + qb * 32 + n32] = lo + hi;
      sm[wave * kRows + qb * 32 + n32] = m[qb];
    }
  }
  __syncthreads();
  float mw[kWaves], mx = -INFINITY;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    mw[w] = sm[w * kRows + out_row];
    mx = fmaxf(mx, mw[w]);
  }
  f32x8 acc = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  float l_tot = 0.f;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    const float wgt = mw[w] > -INFINITY ? __builtin_amdgcn_exp2f(mw[w] - mx) : 0.f;   // no tile: no weight
    l_tot += wgt * sl[w * kRows + out_row];
    const float* src = (const float*)lds + w * (kRows * kOStride) + out_row * kOStride + out_d;
    const f32x4 x0 = *(const f32x4*)src, x1 = *(const f32x4*)(src + 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      acc[i] += wgt * x0[i];
      acc[4 + i] += wgt * x1[i];
    }
  }
  // A term of the split of an infinity is NaN, and so is every result that one had a part in - also where
  // floats give a number (a key at -inf has no weight) or an infinity.  A row that ends with such a
  // value is walked once more, in plain fp32: by its eight lanes, token by token.  (That row alone: the others' bits do not
  // depend on which rows share their workgroup.)  A launch with such a
  // row, or with nothing else, takes 0.44-0.48 ms at 1,004 rows x 1,004 tokens (39 us without) and
  // 4.4-4.6 ms at 8,032 tokens (260 us).
  float inv = l_tot > 0.f ? 1.0f / l_tot : 0.f;
  unsigned top = bits(l_tot) & 0x7fffffffu;
#pragma unroll
  for (int i = 0; i < 8; ++i) top = max(top, bits(acc[i]) & 0x7fffffffu);
#pragma unroll
  for (int x = 1; x < 8; x *= 2) top = max(top, (unsigned)__shfl_xor((int)top, x));
  if (top >= 0x7f800000u) {
    const f32x4* qp = (const f32x4*)(a.q + ((size_t)(sp.q_begin + min(q_row0 + out_row, sp.q_rows - 1)) * H + head) * 64 + out_d);
    const f32x4 q0 = qp[0] * a.scale_log2, q1 = qp[1] * a.scale_log2;
    float m_row = -INFINITY;
    l_tot = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = 0.f;
    for (int t = 0; t < kv_tokens; ++t) {
      const int e = rows[t];
      const size_t at = (size_t)(unsigned)(e ^ (e >> 31)) * (H * 64) + head * 64 + out_d;
      const f32x4* kp = (const f32x4*)((e < 0 ? a.self_k : a.pool) + at);
      const f32x4* vp = (const f32x4*)((e < 0 ? a.self_v : a.pool + (size_t)a.page_size * H * 64) + at);
      const f32x4 k0 = kp[0], k1 = kp[1], v0 = vp[0], v1 = vp[1];
      float s = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) s += q0[i] * k0[i] + q1[i] * k1[i];
#pragma unroll
      for (int x = 1; x < 8; x *= 2) s += __shfl_xor(s, x);
      const float to = fmaxf(m_row, s);
      const float alpha = to > m_row ? __builtin_amdgcn_exp2f(m_row - to) : 1.f;
      const float w = bits(s) == 0xff800000u ? 0.f : __builtin_amdgcn_exp2f(s - to);   // (-inf: also where all so far are)
      m_row = to;
      l_tot = l_tot * alpha + w;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        acc[i] = acc[i] * alpha + w * v0[i];
        acc[4 + i] = acc[4 + i] * alpha + w * v1[i];
      }
    }
    inv = l_tot == 0.f ? 0.f : 1.0f / l_tot;
  }
  if (out_ok) {
    ((f32x4*)out)[0] = f32x4{acc[0], acc[1], acc[2], acc[3]} * inv;
    ((f32x4*)out)[1] = f32x4{acc[4], acc[5], acc[6], acc[7]} * inv;
  }
}

// Blocks of 32 query rows per workgroup: one where all such workgroups are one round of the 256 CUs (a workgroup of two takes half as
// long again: K and V are split into bf16 for either), or where streams of one length take up to three rounds for two.
// us, 16 heads, two blocks and one: 86 rows over 430 tokens 19.4, 13.1; 148 over 740 25.3, 16.5; 200 over 1,800 50.3, 31.4; 377 over 2,639
// 68.6, 44.1; 512 over 4,608 114.6, 86.1; own rows 100 10.3, 7.9, 261 15.7, 10.5, 500 19.9, 14.5; three rounds for two: 1,100 over 5,500
// 290, 267, 1,374 over 6,870 363, 337, two streams of 600 over 3,000 170, 157; two for one, which stay: 600 over 3,000 80, 100,
// 1,004 over 8,032 241, 280, four streams of 148 over 740 28.6, 34.8.
static int lbm_f32_row_blocks(const lbm_attn_stream* s, int n_streams, int num_heads) {
  long long wgs2 = 0, wgs1 = 0;
  bool alike = true;
  for (int i = 0; i < n_streams; ++i) {
    wgs2 += (long long)((s[i].q_rows + 63) / 64) * num_heads;
    wgs1 += (long long)((s[i].q_rows + 31) / 32) * num_heads;
    alike = alike && s[i].kv_tokens == s[0].kv_tokens;
  }
  if (wgs1 <= 256) return 1;
  return alike && 3 * ((wgs1 + 255) / 256) < 5 * ((wgs2 + 255) / 256) ? 1 : 2;
}
template <int S, int QB>
int lbm_launch_attn_f32_d64_rows(AttnArgsF32<S>& a, hipStream_t stream) {
  int wg = 0;
  for (int i = 0; i < S; ++i) {
    if (i < a.n_streams) wg = (wg + 7) & ~7;   // a stream starts on XCD 0, as the kernel's head -> XCD map assumes
    a.wg_begin[i] = wg;
    if (i < a.n_streams) wg += (a.s[i].q_rows + 32 * QB - 1) / (32 * QB) * a.num_heads;
  }
  a.wg_begin[S] = wg;
  for (int i = a.n_streams; i < S; ++i) a.wg_begin[i] = wg;
  if (wg == 0) return LBM_OK;
  wg += (int)(((long long)a.append_tokens * a.num_heads * 16 + kThreads * kAppendPieces - 1) / (kThreads * kAppendPieces));
  if (a.append_tokens > 0) hipLaunchKernelGGL((lbm_attn_f32_d64_kernel<S, true, QB>), dim3(wg), dim3(kThreads), 0, stream, a);
  else hipLaunchKernelGGL((lbm_attn_f32_d64_kernel<S, false, QB>), dim3(wg), dim3(kThreads), 0, stream, a);
  return lbm_check_launch("lbm_attn_f32_d64_kernel");
}
template <int S>
int lbm_launch_attn_f32_d64(AttnArgsF32<S>& a, hipStream_t stream) {
  return lbm_f32_row_blocks(a.s, a.n_streams, a.num_heads) == 1 ? lbm_launch_attn_f32_d64_rows<S, 1>(a, stream) : lbm_launch_attn_f32_d64_rows<S, 2>(a, stream);
}
template int lbm_launch_attn_f32_d64<1>(AttnArgsF32<1>&, hipStream_t);
template int lbm_launch_attn_f32_d64<LBM_MAX_STREAMS>(AttnArgsF32<LBM_MAX_STREAMS>&, hipStream_t);
