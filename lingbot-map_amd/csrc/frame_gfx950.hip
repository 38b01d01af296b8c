// What stands around the blocks of a frame, one launch each: the images' normalisation, the patch convolution's bias with its
// patches as rows, the rotary table of the frame's place in the stream, the groups' outputs side by side.  A few MB each, bound by their launches and a trip to memory;
// as torch operations they are several launches with whole passes over memory between them.
#include <hip/hip_runtime.h>
#include "lbm_internal.h"

namespace {
typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;

constexpr int kThreads = 256;
struct GroupParts {
  const void* part[2 * LBM_MAX_GROUPS];
  void* out[LBM_MAX_GROUPS];
};

// ---------------------------------------------------------------------------- group outputs
// Row r of out[g] is row r of part[2 g], then row r of part[2 g + 1].  blockIdx.y: the part; four 16-byte pieces per thread, their
// loads together.  us, four groups of 1,004 rows of 2 x 1,024 bf16: torch's four concatenations 25.6, their stack for a
// replayed frame 16.4; this 7.2 (33 MB at 4.6 TB/s).
__global__ __launch_bounds__(kThreads) void lbm_group_outputs_kernel(GroupParts parts, unsigned pieces, unsigned row_pieces) {
  constexpr int kEach = 4;
  const int p = blockIdx.y;
  const u32x4* src = (const u32x4*)parts.part[p];
  u32x4* dst = (u32x4*)parts.out[p >> 1] + (p & 1) * row_pieces;
  const unsigned first = blockIdx.x * (kThreads * kEach) + threadIdx.x;
  u32x4 v[kEach];
#pragma unroll
  for (int j = 0; j < kEach; ++j) v[j] = src[min(first + j * kThreads, pieces - 1)];
#pragma unroll
  for (int j = 0; j < kEach; ++j) {
    const unsigned i = first + j * kThreads, row = i / row_pieces;
    if (i < pieces) lbm_store_through(dst + (size_t)row * 2 * row_pieces + (i - row * row_pieces), v[j]);
  }
}

// ---------------------------------------------------------------------------- rotary table of a stream's frames
// out[s][i] = (cos, sin)(angles[i] + first * later[i % pairs]), in float64 up to the result's rounding.  us, 1,004 tokens of
// 32 pairs: torch's sum, polar and conversion 23.4, this 4.9.
__global__ __launch_bounds__(kThreads) void lbm_stream_table_kernel(const double* angles, const double* later, double first,
                                                                    u32x2* out, unsigned n, unsigned pairs, int streams) {
  const unsigned i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= n) return;
  double s, c;
  sincos(angles[i] + first * later[i % pairs], &s, &c);
  const u32x2 v = {__builtin_bit_cast(unsigned, (float)c), __builtin_bit_cast(unsigned, (float)s)};
  for (int b = 0; b < streams; ++b) out[(size_t)b * n + i] = v;
}

// ---------------------------------------------------------------------------- images
// (x - mean[c]) / std[c], rounded to the images' type after each of the two.  Four values of one channel per thread.  us,
// 378 x 518 in bf16: torch's two operations 10.8, this 4.3.
template <bool BF16>
__global__ __launch_bounds__(kThreads) void lbm_normalise_images_kernel(const void* images, const void* mean, const void* std,
                                                                        void* out, unsigned quads, unsigned plane_quads) {
  const unsigned i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= quads) return;
  const unsigned c = i / plane_quads % 3u;
  if (BF16) {
    const float m = (float)((const __bf16*)mean)[c], d = (float)((const __bf16*)std)[c];
    const bf16x4 x = __builtin_bit_cast(bf16x4, ((const u32x2*)images)[i]);
    bf16x4 y;
#pragma unroll
    for (int k = 0; k < 4; ++k) y[k] = (__bf16)((float)(__bf16)((float)x[k] - m) / d);
    ((u32x2*)out)[i] = __builtin_bit_cast(u32x2, y);
  } else {
    const float m = ((const float*)mean)[c], d = ((const float*)std)[c];
    const f32x4 x = ((const f32x4*)images)[i];
    f32x4 y;
#pragma unroll
    for (int k = 0; k < 4; ++k) y[k] = (x[k] - m) / d;
    ((f32x4*)out)[i] = y;
  }
}

// ---------------------------------------------------------------------------- patch tokens
// out[n][p][c] = conv[n][c][p] + bias[c] in bf16: the patch convolution's bias and its channels last.  64 channels x 64
// patches per workgroup through LDS: patches lie side by side on the way in (of any number, so 2 bytes a lane, 128 a
// wavefront's load), channels on the way out (16 bytes a lane).  us, 999 patches of 1,024 channels: torch's sum and copy
// 15.9, this 4.6; of eight images 55, 8.4.
__global__ __launch_bounds__(kThreads) void lbm_patch_tokens_kernel(const unsigned short* conv, const __bf16* bias, unsigned short* out,
                                                                    int patches, int channels) {
  constexpr int kTile = 64, kStride = kTile + 8, kEach = kTile * kTile / kThreads;
  __shared__ __attribute__((aligned(16))) unsigned short tile[kTile * kStride];   // [patch][channel]
  const int tid = threadIdx.x, p0 = blockIdx.x * kTile, c0 = blockIdx.y * kTile;
  const unsigned short* src = conv + ((size_t)blockIdx.z * channels + c0) * patches;
  const int p = tid & 63, last = patches - 1 - p0;
  unsigned short v[kEach];
#pragma unroll
  for (int j = 0; j < kEach; ++j) v[j] = src[(size_t)(j * (kThreads / 64) + (tid >> 6)) * patches + p0 + min(p, last)];
#pragma unroll
  for (int j = 0; j < kEach; ++j) {
    const int c = j * (kThreads / 64) + (tid >> 6);
    const __bf16 sum = (__bf16)((float)__builtin_bit_cast(__bf16, v[j]) + (float)bias[c0 + c]);
    tile[p * kStride + c] = __builtin_bit_cast(unsigned short, sum);
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kTile * kTile / 8 / kThreads; ++j) {
    const int r = j * (kThreads / 8) + (tid >> 3), c = (tid & 7) * 8;
    if (p0 + r < patches)
      lbm_store_through(out + ((size_t)blockIdx.z * patches + p0 + r) * channels + c0 + c, *(const u32x4*)&tile[r * kStride + c]);
  }
}

bool aligned(const void* p, size_t to) { return ((uintptr_t)p & (to - 1)) == 0; }
unsigned blocks_for(unsigned long long n, unsigned per_block) { return (unsigned)((n + per_block - 1) / per_block); }
}  // namespace

extern "C" int lbm_group_outputs(const void* const* parts, void* const* out, int32_t n_groups, int64_t rows, int64_t row_bytes, void* stream) {
  if (!parts || !out) return lbm_fail(LBM_ERR_INVALID, "lbm_group_outputs: null argument");
  if (n_groups < 1 || n_groups > LBM_MAX_GROUPS) return lbm_fail(LBM_ERR_INVALID, "lbm_group_outputs: %d groups, 1 to %d are taken", n_groups, LBM_MAX_GROUPS);
  if (rows < 1 || row_bytes < 16 || row_bytes % 16 || rows > (1LL << 31) / (row_bytes / 16))
    return lbm_fail(LBM_ERR_INVALID, "lbm_group_outputs: %lld rows of %lld bytes (whole 16-byte pieces, fewer than 2^31)", (long long)rows, (long long)row_bytes);
  GroupParts p = {};
  for (int i = 0; i < 2 * n_groups; ++i) {
    p.part[i] = parts[i];
    if (!parts[i] || !aligned(parts[i], 16)) return lbm_fail(LBM_ERR_INVALID, "lbm_group_outputs: part %d is null or not 16-byte aligned", i);
  }
  for (int i = 0; i < n_groups; ++i) {
    p.out[i] = out[i];
    if (!out[i] || !aligned(out[i], 16)) return lbm_fail(LBM_ERR_INVALID, "lbm_group_outputs: output %d is null or not 16-byte aligned", i);
  }
  const unsigned row_pieces = (unsigned)(row_bytes / 16), pieces = (unsigned)rows * row_pieces;
  hipLaunchKernelGGL(lbm_group_outputs_kernel, dim3(blocks_for(pieces, kThreads * 4), 2 * n_groups), dim3(kThreads), 0, (hipStream_t)stream,
                     p, pieces, row_pieces);
  return lbm_check_launch("lbm_group_outputs_kernel");
}

extern "C" int lbm_stream_table(const double* angles, const double* later, int64_t first, float* out, int32_t tokens, int32_t pairs,
                                int32_t n_streams, void* stream) {
  if (!angles || !later || !out) return lbm_fail(LBM_ERR_INVALID, "lbm_stream_table: null argument");
  if (tokens < 1 || pairs < 1 || n_streams < 1 || (long long)tokens * pairs >= (1LL << 31))
    return lbm_fail(LBM_ERR_INVALID, "lbm_stream_table: %d tokens x %d pairs for %d streams", tokens, pairs, n_streams);
  if (!aligned(angles, 8) || !aligned(later, 8) || !aligned(out, 8)) return lbm_fail(LBM_ERR_INVALID, "lbm_stream_table: 8-byte alignment");
  const unsigned n = (unsigned)tokens * (unsigned)pairs;
  hipLaunchKernelGGL(lbm_stream_table_kernel, dim3(blocks_for(n, kThreads)), dim3(kThreads), 0, (hipStream_t)stream, angles, later,
                     (double)first, (u32x2*)out, n, (unsigned)pairs, n_streams);
  return lbm_check_launch("lbm_stream_table_kernel");
}

extern "C" int lbm_normalise_images(const void* images, const void* mean, const void* std, void* out, int32_t dtype, int64_t n_images,
                                    int64_t plane, void* stream) {
  if (!images || !mean || !std || !out) return lbm_fail(LBM_ERR_INVALID, "lbm_normalise_images: null argument");
  if (dtype != LBM_DTYPE_BF16 && dtype != LBM_DTYPE_F32) return lbm_fail(LBM_ERR_INVALID, "lbm_normalise_images: unknown dtype %d", dtype);
  if (n_images < 1 || plane < 4 || plane % 4 || n_images > (1LL << 31) / (3 * (plane / 4)))
    return lbm_fail(LBM_ERR_INVALID, "lbm_normalise_images: %lld images of 3 x %lld values (a multiple of 4)", (long long)n_images, (long long)plane);
  const size_t quad = dtype == LBM_DTYPE_BF16 ? 8 : 16;
  if (!aligned(images, quad) || !aligned(out, quad)) return lbm_fail(LBM_ERR_INVALID, "lbm_normalise_images: %zu-byte alignment", quad);
  const unsigned plane_quads = (unsigned)(plane / 4), quads = (unsigned)n_images * 3u * plane_quads;
  const dim3 grid(blocks_for(quads, kThreads)), block(kThreads);
  if (dtype == LBM_DTYPE_BF16) hipLaunchKernelGGL(lbm_normalise_images_kernel<true>, grid, block, 0, (hipStream_t)stream, images, mean, std, out, quads, plane_quads);
  else hipLaunchKernelGGL(lbm_normalise_images_kernel<false>, grid, block, 0, (hipStream_t)stream, images, mean, std, out, quads, plane_quads);
  return lbm_check_launch("lbm_normalise_images_kernel");
}

extern "C" int lbm_patch_tokens(const void* conv, const void* bias, void* out, int32_t n_images, int32_t channels, int32_t patches, void* stream) {
  if (!conv || !bias || !out) return lbm_fail(LBM_ERR_INVALID, "lbm_patch_tokens: null argument");
  if (n_images < 1 || n_images > 65535 || channels < 64 || channels % 64 || channels > 64 * 65535 || patches < 1)
    return lbm_fail(LBM_ERR_INVALID, "lbm_patch_tokens: %d images of %d channels (a multiple of 64) x %d patches", n_images, channels, patches);
  if (!aligned(conv, 2) || !aligned(bias, 2) || !aligned(out, 16)) return lbm_fail(LBM_ERR_INVALID, "lbm_patch_tokens: alignment");
  hipLaunchKernelGGL(lbm_patch_tokens_kernel, dim3(blocks_for(patches, 64), channels / 64, n_images), dim3(kThreads), 0, (hipStream_t)stream,
                     (const unsigned short*)conv, (const __bf16*)bias, (unsigned short*)out, patches, channels);
  return lbm_check_launch("lbm_patch_tokens_kernel");
}
