// Load-time weight packaging: compressed-tensors INT4 checkpoint -> the
// on-device layout the grouped W4A16 GEMM consumes.
//
// The device layout is the reference's Marlin "uint4b8 no-act-order" layout,
// byte for byte (so packages built by either implementation are
// interchangeable and the reference's own known-answer tests apply):
//
//   weights  [E][K/16][2N] u32: 16(k) x 64(n) tiles of 128 words, tile
//            (kt, nt) at word (kt * N/64 + nt) * 128; word th*4 + w holds the
//            8 nibbles (n0 = nt*64 + w*16 + th/4, n1 = n0 + 8) x
//            (k = kt*16 + 2*(th%4) + {0, 1, 8, 9}) in nibble order
//            (n0,k0) (n0,k8) (n1,k0) (n1,k8) (n0,k1) (n0,k9) (n1,k1) (n1,k9).
//   scales   [E][K/32][N] bf16, every 64-column chunk permuted so that column
//            p of the chunk sits at 8*(p%8) + p/8.
//
// The GEMM kernels (wna16.hip) map MFMA 32x32x16 fragments directly onto
// these words, so no further conversion is needed on MI355X.
//
// Reference: pegainfer-kernels/csrc/kimi_k2/kimi_marlin_int4.cu:21-263;
// Rust ops src/ops/kimi_k2/experts.rs:850-1022.
#include "common.h"
#include "pega_moe.h"

namespace pega {
namespace {

// One output word: columns n0 (words a0, a1 of its checkpoint row) and n0 + 8
// (b0, b1), k pair at bit sh of each word (k 0..7 in a0 / b0, 8..15 in a1 / b1).
__device__ __forceinline__ uint32_t marlin_word(uint32_t a0, uint32_t a1, uint32_t b0, uint32_t b1,
                                                int sh) {
  // byte i: the even-k nibble below the odd-k one, of (n0, k), (n0, k+8), (n0+8, k), (n0+8, k+8)
  const uint32_t t = ((a0 >> sh) & 0xffu) | (((a1 >> sh) & 0xffu) << 8) |
                     (((b0 >> sh) & 0xffu) << 16) | (((b1 >> sh) & 0xffu) << 24);
  uint32_t lo = t & 0x0f0f0f0fu, hi = (t >> 4) & 0x0f0f0f0fu;
  lo = (lo | (lo >> 4)) & 0x00ff00ffu;
  hi = (hi | (hi >> 4)) & 0x00ff00ffu;
  return ((lo | (lo >> 8)) & 0xffffu) | ((hi | (hi >> 8)) << 16);
}

// The weight repack, a transpose bound by HBM: a workgroup takes 64 checkpoint
// rows (one column tile) by up to 512 k.  It reads 256 contiguous bytes of each
// row with 16-byte loads, and from LDS each thread builds whole 16-byte output
// pieces (the four words of one th), so a k-tile's 512 bytes go out contiguous.
// The row pitch of 66 words puts the eight rows a half-wave reads on distinct
// bank pairs.  48 x 2048 x 7168: 426 us with one gathering thread per output
// word (1.65 TB/s), 135 us (5.2 TB/s) here.
constexpr int kRepackK = 512;                      // k per workgroup
constexpr int kRepackPitch = kRepackK / 8 + 2;     // words per LDS row
__global__ __launch_bounds__(256) void reorder_weight_tile_kernel(
    const uint32_t* __restrict__ ckpt, uint32_t* __restrict__ marlin, int size_k, int size_n) {
  __shared__ uint32_t rows[64 * kRepackPitch];
  const int nt = blockIdx.y, n_tiles = size_n >> 6;
  const int k0 = blockIdx.x * kRepackK;
  const int kn = min(kRepackK, size_k - k0);  // a multiple of 32
  const int k_words = size_k >> 3;
  const long long per_expert = static_cast<long long>(size_n) * k_words;
  const uint32_t* src = ckpt + blockIdx.z * per_expert +
                        static_cast<long long>(nt) * 64 * k_words + (k0 >> 3);
  const int quads = kn >> 5;  // 16-byte pieces of a row
  for (int i = threadIdx.x; i < 64 * (kRepackK / 32); i += 256) {
    const int r = i / (kRepackK / 32), q = i % (kRepackK / 32);
    if (q >= quads) continue;
    const uint4 v =
        *reinterpret_cast<const uint4*>(src + static_cast<long long>(r) * k_words + 4 * q);
    uint32_t* d = rows + r * kRepackPitch + 4 * q;
    d[0] = v.x;
    d[1] = v.y;
    d[2] = v.z;
    d[3] = v.w;
  }
  __syncthreads();
  uint4* out = reinterpret_cast<uint4*>(marlin + blockIdx.z * per_expert) +
               (static_cast<long long>(k0 >> 4) * n_tiles + nt) * 32;
  for (int i = threadIdx.x; i < kn * 2; i += 256) {  // 32 pieces per k-tile
    const int kt = i >> 5, th = i & 31;
    const int sh = 8 * (th & 3);
    uint32_t w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t* a = rows + (16 * j + (th >> 2)) * kRepackPitch + 2 * kt;
      const uint32_t* b = a + 8 * kRepackPitch;
      w[j] = marlin_word(a[0], a[1], b[0], b[1], sh);
    }
    out[static_cast<long long>(kt) * n_tiles * 32 + th] = make_uint4(w[0], w[1], w[2], w[3]);
  }
}

// One thread per output word, for buffers that are not 16-byte aligned: gathers
// its 8 nibbles from 4 checkpoint words.
__global__ void reorder_weight_kernel(const uint32_t* __restrict__ ckpt,
                                      uint32_t* __restrict__ marlin, int size_k, int size_n,
                                      long long total_words) {
  const long long idx = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (idx >= total_words) return;
  const long long per_expert = static_cast<long long>(size_n) * (size_k / 8);
  const int e = static_cast<int>(idx / per_expert);
  const long long in_e = idx - e * per_expert;
  const int n_tiles = size_n / 64;
  const int word = static_cast<int>(in_e % 128);
  const long long tile = in_e / 128;
  const int nt = static_cast<int>(tile % n_tiles);
  const int kt = static_cast<int>(tile / n_tiles);
  const int th = word >> 2, w = word & 3;
  const int n0 = nt * 64 + w * 16 + (th >> 2);
  const int k_words = size_k / 8;
  const uint32_t* a = ckpt + e * per_expert + static_cast<long long>(n0) * k_words + 2 * kt;
  const uint32_t* b = a + 8LL * k_words;
  marlin[idx] = marlin_word(a[0], a[1], b[0], b[1], 8 * (th & 3));
}

// The scale repack of whole 64-column tiles, a transpose of 2-byte elements
// through LDS: 64 checkpoint rows by up to 64 groups, read along the groups and
// written along the permuted columns, 128 contiguous bytes a wave either way
// (one element per thread from global memory to global memory: 81 us for
// 48 x 2048 x 224, 1.1 TB/s; 22 us here).
__global__ __launch_bounds__(256) void reorder_scale_tile_kernel(
    const uint16_t* __restrict__ ckpt, uint16_t* __restrict__ marlin, int size_n, int scale_k) {
  __shared__ uint16_t rows[64][66];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n0 = blockIdx.y * 64, g0 = blockIdx.x * 64;
  const long long base = static_cast<long long>(blockIdx.z) * size_n * scale_k;
  const int gn = min(64, scale_k - g0);
  if (lane < gn) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int r = wave * 16 + i;
      rows[r][lane] = ckpt[base + static_cast<long long>(n0 + r) * scale_k + g0 + lane];
    }
  }
  __syncthreads();
  const int p = (lane >> 3) + 8 * (lane & 7);  // the column stored at position `lane`
  for (int g = wave; g < gn; g += 4)
    marlin[base + static_cast<long long>(g0 + g) * size_n + n0 + lane] = rows[p][g];
}

// One thread per element, for widths that are not whole 64-column tiles.
__global__ void reorder_scale_kernel(const uint16_t* __restrict__ ckpt,
                                     uint16_t* __restrict__ marlin, int size_n, int scale_k,
                                     long long total) {
  const long long idx = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (idx >= total) return;
  const long long per_expert = static_cast<long long>(size_n) * scale_k;
  const long long e = idx / per_expert;
  const long long in_e = idx - e * per_expert;
  const int o = static_cast<int>(in_e & 63);
  const long long src_flat = (in_e & ~63LL) + (o >> 3) + 8 * (o & 7);
  const int g = static_cast<int>(src_flat / size_n);
  const int row = static_cast<int>(src_flat - static_cast<long long>(g) * size_n);
  marlin[idx] = ckpt[e * per_expert + static_cast<long long>(row) * scale_k + g];
}

// Row concatenation [rows][2][cols]: gate half then up half, 16-byte copies.
__global__ void concat_rows_kernel(const uint4* __restrict__ a, const uint4* __restrict__ b,
                                   uint4* __restrict__ out, long long rows, int cols16) {
  const long long total = rows * cols16;
  for (long long idx = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
       idx < total; idx += static_cast<long long>(gridDim.x) * blockDim.x) {
    const long long r = idx / cols16;
    const int c = static_cast<int>(idx - r * cols16);
    out[r * 2 * cols16 + c] = a[idx];
    out[r * 2 * cols16 + cols16 + c] = b[idx];
  }
}

__global__ void concat_rows_u16_kernel(const uint16_t* __restrict__ a,
                                       const uint16_t* __restrict__ b,
                                       uint16_t* __restrict__ out, long long rows, int cols) {
  const long long total = rows * cols;
  for (long long idx = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
       idx < total; idx += static_cast<long long>(gridDim.x) * blockDim.x) {
    const long long r = idx / cols;
    const int c = static_cast<int>(idx - r * cols);
    out[r * 2 * cols + c] = a[idx];
    out[r * 2 * cols + cols + c] = b[idx];
  }
}

bool common_shape_ok(int in_dim, int out_dim, int local_experts, int group_size) {
  return in_dim > 0 && out_dim > 0 && local_experts > 0 && group_size == 32 &&
         in_dim % 16 == 0 && out_dim % 64 == 0 && in_dim % group_size == 0;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

unsigned grid_for(long long n, int threads) {
  long long g = (n + threads - 1) / threads;
  return static_cast<unsigned>(g < 1 ? 1 : (g > 0x7fffffffLL ? 0x7fffffffLL : g));
}

}  // namespace

int reorder_weight(const uint8_t* ckpt, uint8_t* marlin, int in_dim, int out_dim,
                   int local_experts, int group_size, hipStream_t stream) {
  if (!ckpt || !marlin) return fail(kInvalidValue, "reorder_weight: null pointer");
  if (!common_shape_ok(in_dim, out_dim, local_experts, group_size))
    return fail(kInvalidValue, "reorder_weight: bad shape in=%d out=%d E=%d group=%d", in_dim,
                out_dim, local_experts, group_size);
  // the tile kernel's grid: k chunks, column tiles (at most 65535), experts (the same)
  if (aligned16(ckpt) && aligned16(marlin) && out_dim / 64 <= 65535 && local_experts <= 65535) {
    const dim3 grid(ceil_div(in_dim, kRepackK), out_dim / 64, local_experts);
    hipLaunchKernelGGL(reorder_weight_tile_kernel, grid, dim3(256), 0, stream,
                       reinterpret_cast<const uint32_t*>(ckpt),
                       reinterpret_cast<uint32_t*>(marlin), in_dim, out_dim);
    return launch_status("reorder_weight");
  }
  const long long total = static_cast<long long>(local_experts) * out_dim * (in_dim / 8);
  hipLaunchKernelGGL(reorder_weight_kernel, dim3(grid_for(total, 256)), dim3(256), 0, stream,
                     reinterpret_cast<const uint32_t*>(ckpt), reinterpret_cast<uint32_t*>(marlin),
                     in_dim, out_dim, total);
  return launch_status("reorder_weight");
}

int reorder_scale(const uint16_t* ckpt, uint16_t* marlin, int in_dim, int out_dim,
                  int local_experts, int group_size, hipStream_t stream) {
  if (!ckpt || !marlin) return fail(kInvalidValue, "reorder_scale: null pointer");
  if (in_dim <= 0 || out_dim <= 0 || local_experts <= 0 || group_size != 32 ||
      in_dim % group_size != 0)
    return fail(kInvalidValue, "reorder_scale: bad shape");
  const int scale_k = in_dim / group_size;
  const long long per_expert = static_cast<long long>(out_dim) * scale_k;
  if (per_expert % 64 != 0)
    return fail(kInvalidValue, "reorder_scale: out*groups (%lld) not a multiple of 64",
                per_expert);
  if (out_dim % 64 == 0 && out_dim / 64 <= 65535 && local_experts <= 65535) {
    const dim3 grid(ceil_div(scale_k, 64), out_dim / 64, local_experts);
    hipLaunchKernelGGL(reorder_scale_tile_kernel, grid, dim3(256), 0, stream, ckpt, marlin,
                       out_dim, scale_k);
    return launch_status("reorder_scale");
  }
  const long long total = per_expert * local_experts;
  hipLaunchKernelGGL(reorder_scale_kernel, dim3(grid_for(total, 256)), dim3(256), 0, stream,
                     ckpt, marlin, out_dim, scale_k, total);
  return launch_status("reorder_scale");
}

int fuse_w13(const uint8_t* gate_w, const uint8_t* up_w, uint8_t* w13_w, const uint16_t* gate_s,
             const uint16_t* up_s, uint16_t* w13_s, int in_dim, int inter, int local_experts,
             int group_size, hipStream_t stream) {
  if (!gate_w || !up_w || !w13_w || !gate_s || !up_s || !w13_s)
    return fail(kInvalidValue, "fuse_w13: null pointer");
  if (!common_shape_ok(in_dim, inter, local_experts, group_size))
    return fail(kInvalidValue, "fuse_w13: bad shape in=%d inter=%d E=%d", in_dim, inter,
                local_experts);
  // Weights: rows = E * K/16, each gate row is 2*inter u32 = inter/2 uint4.
  const long long wrows = static_cast<long long>(local_experts) * (in_dim / 16);
  const int wcols16 = inter / 2;
  hipLaunchKernelGGL(concat_rows_kernel, dim3(grid_for(wrows * wcols16, 256)), dim3(256), 0,
                     stream, reinterpret_cast<const uint4*>(gate_w),
                     reinterpret_cast<const uint4*>(up_w), reinterpret_cast<uint4*>(w13_w),
                     wrows, wcols16);
  int st = launch_status("fuse_w13 weights");
  if (st != kSuccess) return st;
  const long long srows = static_cast<long long>(local_experts) * (in_dim / group_size);
  // 16 bytes a thread where the buffers allow it (inter is a multiple of 64): 48 x 224 rows of
  // 2 x 2048 scales 67 -> 35 us
  if (aligned16(gate_s) && aligned16(up_s) && aligned16(w13_s)) {
    hipLaunchKernelGGL(concat_rows_kernel, dim3(grid_for(srows * (inter / 8), 256)), dim3(256), 0,
                       stream, reinterpret_cast<const uint4*>(gate_s),
                       reinterpret_cast<const uint4*>(up_s), reinterpret_cast<uint4*>(w13_s),
                       srows, inter / 8);
    return launch_status("fuse_w13 scales");
  }
  hipLaunchKernelGGL(concat_rows_u16_kernel, dim3(grid_for(srows * inter, 256)), dim3(256), 0,
                     stream, gate_s, up_s, w13_s, srows, inter);
  return launch_status("fuse_w13 scales");
}

}  // namespace pega

// ---------------------------------------------------------------- C ABI
// Reference declarations: pegainfer-kernels/src/ffi/kimi.rs:68-101; guards
// kimi_marlin_int4.cu:15-19,179-184,201-213,235-242 (local_experts == 48).  The
// reference maps every failure of these calls, a launch failure included, to
// CUDA_ERROR_INVALID_VALUE (kimi_marlin_int4.cu:190,220,254,262), and so do these.
namespace {
int as_invalid_value(int rc) { return rc == pega::kSuccess ? rc : pega::kInvalidValue; }
}  // namespace

PEGA_API int kimi_marlin_int4_reorder_weight_cuda(const uint8_t* weight_packed_checkpoint,
                                                  uint8_t* weight_packed_marlin, int in_dim,
                                                  int out_dim, int local_experts,
                                                  int group_size, hipStream_t stream) {
  if (local_experts != 48)
    return pega::fail(pega::kInvalidValue, "kimi reorder_weight: local_experts must be 48");
  return as_invalid_value(pega::reorder_weight(weight_packed_checkpoint, weight_packed_marlin,
                                               in_dim, out_dim, local_experts, group_size,
                                               stream));
}

PEGA_API int kimi_marlin_int4_reorder_scale_cuda(const uint16_t* weight_scale_checkpoint,
                                                 uint16_t* weight_scale_marlin, int in_dim,
                                                 int out_dim, int local_experts, int group_size,
                                                 hipStream_t stream) {
  if (local_experts != 48)
    return pega::fail(pega::kInvalidValue, "kimi reorder_scale: local_experts must be 48");
  return as_invalid_value(pega::reorder_scale(weight_scale_checkpoint, weight_scale_marlin,
                                              in_dim, out_dim, local_experts, group_size,
                                              stream));
}

PEGA_API int kimi_marlin_int4_fuse_w13_cuda(const uint8_t* gate_weight_packed_marlin,
                                            const uint8_t* up_weight_packed_marlin,
                                            uint8_t* w13_weight_packed_marlin,
                                            const uint16_t* gate_scale_marlin,
                                            const uint16_t* up_scale_marlin,
                                            uint16_t* w13_scale_marlin, int in_dim,
                                            int intermediate_dim, int local_experts,
                                            int group_size, hipStream_t stream) {
  if (local_experts != 48)
    return pega::fail(pega::kInvalidValue, "kimi fuse_w13: local_experts must be 48");
  return as_invalid_value(pega::fuse_w13(gate_weight_packed_marlin, up_weight_packed_marlin,
                                         w13_weight_packed_marlin, gate_scale_marlin,
                                         up_scale_marlin, w13_scale_marlin, in_dim,
                                         intermediate_dim, local_experts, group_size, stream));
}

// Shape-general variants (any expert count; no reference counterpart).
PEGA_API int pega_marlin_int4_reorder_weight(const uint8_t* ckpt, uint8_t* marlin, int in_dim,
                                             int out_dim, int local_experts, int group_size,
                                             hipStream_t stream) {
  return pega::reorder_weight(ckpt, marlin, in_dim, out_dim, local_experts, group_size, stream);
}

PEGA_API int pega_marlin_int4_reorder_scale(const uint16_t* ckpt, uint16_t* marlin, int in_dim,
                                            int out_dim, int local_experts, int group_size,
                                            hipStream_t stream) {
  return pega::reorder_scale(ckpt, marlin, in_dim, out_dim, local_experts, group_size, stream);
}

PEGA_API int pega_marlin_int4_fuse_w13(const uint8_t* gate_w, const uint8_t* up_w,
                                       uint8_t* w13_w, const uint16_t* gate_s,
                                       const uint16_t* up_s, uint16_t* w13_s, int in_dim,
                                       int intermediate_dim, int local_experts, int group_size,
                                       hipStream_t stream) {
  return pega::fuse_w13(gate_w, up_w, w13_w, gate_s, up_s, w13_s, in_dim, intermediate_dim,
                        local_experts, group_size, stream);
}
