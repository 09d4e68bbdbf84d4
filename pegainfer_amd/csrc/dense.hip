// Dense bf16 GEMM of the shared expert on MI355X (gfx950):
//
//   Y[n][m] = bf16( sum_k f(W[m][k]) * f(X[n][k]) ),  fp32 accumulation,
//   W [M][K], X [N][K], Y [N][M], bf16 row-major
//
// Reference: pegainfer-kernels/csrc/shared/linear.cu:321-344
// (gemm_graphsafe_cuda: cublasGemmEx(OP_T, OP_N, M, N, K, W lda K, X ldb K,
// Y ldc M, CUBLAS_COMPUTE_32F)), bound in pegainfer-kernels/src/ffi/shared.rs:220-238
// and called for the Kimi shared expert's gate/up and down projections
// (pegainfer-kimi-k2/src/runner/moe_nccl.rs:107-123).
//
// Load shape: the 16x16x32 fragment layout puts a different W (or X) row in
// each of four neighbouring lanes; loaded that way, every 16-byte-per-lane
// load splits into about 64 cache-line requests and the address unit bounds
// the kernel (78% busy, ~77 cycles per load instruction, 1.6 TB/s of W on the
// Kimi gate/up shape).  So the loads run along k (a lane quad reads 64
// contiguous bytes of one row) and ds_bpermute moves each lane's 16 bytes to
// the lane whose fragment needs them: gate/up 37.3 -> 26.4 us (2.3 TB/s of W).
// A permuted k order that reads 256 contiguous bytes per row per step instead
// quadruples the lines per instruction and ran 2.3x slower.
//
// Order of the sums, the same in both kernels below: K's 32-k steps in 1 to 16 contiguous
// shares (k_shares), each share one chain of v_mfma_f32_16x16x32_bf16 in k order, the shares'
// sums added in order in fp32.  A launch's bits then depend on its sizes alone, not on the
// kernel or tile that a dispatch rule picks.  Lane (c, q) of an MFMA holds row c of the
// tile, k 8q..8q+7 (tokens the A operand, features the B operand).
//
// The first kernel below serves few tokens, where the GEMM is a weight stream: one
// workgroup owns 16 rows of W for 16 RB tokens; its waves take the shares.  Per 32-k step a
// lane issues one 16-byte load of W and one of X per 16-token block; after the lane exchange
// one v_mfma_f32_16x16x32_bf16 runs per token block.  Token rows past N read zeros through an
// out-of-range buffer offset and are never stored.
#include <hipblaslt/hipblaslt.h>

#include <map>
#include <mutex>
#include <tuple>
#include <type_traits>

#include "common.h"
#include "pega_moe.h"

namespace pega {
namespace {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4_t;

constexpr uint32_t kOutOfRange = 0x80000000u;  // voffset that fails every range check
constexpr int kMaxShares = 16;
// First 32-k step of share w of 2^lg (share 2^lg starts where the last one ends).
__device__ __forceinline__ int share_start(int steps, int w, int lg) { return (steps * w) >> lg; }
// W loads are cached too: a step reads 64 bytes of each of 16 rows, so the
// other half of every 128-byte line is the next step's, and a non-temporal
// policy that does not keep the line costs 20% (44.9 against 37.3 us for
// the Kimi gate/up shape).
constexpr int kCached = 0;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), static_cast<short>(0),
                                           static_cast<int>(bytes), 0x00020000);
}

template <int kPolicy>
__device__ __forceinline__ u32x4_t load16(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  return __builtin_amdgcn_raw_buffer_load_b128(r, static_cast<int>(voff), static_cast<int>(soff),
                                               kPolicy);
}

template <int MR, int RB>
struct StepRegs {
  u32x4_t w[MR];  // row l / 4 of the tile, W[..][k0 + 8 (l % 4) .. +7] (lane l)
  u32x4_t x[RB];  // X[n0 + 16 rb + l / 4][k0 + 8 (l % 4) .. +7]
};

// One workgroup per (16 rows of W, 16 RB tokens); wave w of WV takes the shares
// w shares / WV up to the next wave's, one after another, D steps in flight.  SWIGLU: the
// tile holds gate features m0..m0+7 and the matching up features (I rows further on), so a
// tile completes eight outputs by itself; the epilogue rounds both sums to bf16 as the GEMM's
// output would be, applies SwiGLU and writes act[n][m0+c] (Y row stride M = I).  F32: Y is
// fp32 and takes the sums unrounded (the router's logits GEMM, cublasGemmEx with CUDA_R_32F
// output).
//
// A stream of W with few bytes per CU: what counts is that every CU has a workgroup and
// that the first loads are out early.  Kimi's shared expert, 3 tokens, gate/up with SwiGLU
// (58.7 MB) / down (29.4 MB), weights not in cache: 13.6 / 7.3 us, against 21.9 / 8.9 with a
// wave per share on 32-row tiles (128 and 224 workgroups, half the CUs idle in the first); two
// waves and eight steps in flight where there are two shares, 16384 x 4096 at one token, 28.8
// (four steps: 32.4).
template <int WV, int MR, int RB, bool SWIGLU, bool F32>
__global__ __launch_bounds__(64 * WV) void dense_gemm_kernel(const uint16_t* __restrict__ W,
                                                             const uint16_t* __restrict__ X,
                                                             void* __restrict__ Yv, int M,
                                                             int N, int K, int lg_shares) {
  static_assert(!(SWIGLU && F32), "the SwiGLU epilogue writes bf16");
  constexpr int D = WV >= 4 || MR * RB > 3 ? 4 : 8;  // few waves: more loads in flight each
  constexpr bool kOneShare = WV <= 2;                // launched with as many shares as waves
  constexpr int kShares = kOneShare ? WV : kMaxShares;
  __shared__ float s_red[kShares][MR * RB * 4][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, q = lane >> 4;
  constexpr int kOut = SWIGLU ? 8 : 16;  // outputs of a tile
  const int m0 = blockIdx.x * (kOut * MR);
  const int n0 = blockIdx.y * (16 * RB);
  const int steps = K >> 5;
  const int shares = 1 << lg_shares;
  int sh = (shares * wave) / WV;  // this wave's first share, then the one it is in
  const int s0 = share_start(steps, sh, lg_shares);
  const int s1 = share_start(steps, (shares * (wave + 1)) / WV, lg_shares);

  const uint32_t span = SWIGLU ? static_cast<uint32_t>(M) + 8u * MR : 16u * MR;
  const __amdgpu_buffer_rsrc_t wr =
      make_rsrc(W + static_cast<long long>(m0) * K, span * static_cast<uint32_t>(K) * 2u);
  // Loads run along k: lane l fetches row l / 4, k 8 (l % 4) .. +7, so four
  // neighbouring lanes read 64 contiguous bytes of one row (one line request
  // per lane quad, 16 per load); ds_bpermute then hands lane (c, q) the
  // 16 bytes of row c, k 8q .. +7 that its fragment needs, from lane 4c + q.
  const uint32_t lr = static_cast<uint32_t>(lane >> 2), lp = static_cast<uint32_t>(lane & 3);
  const uint32_t w_row = SWIGLU ? (lr & 7u) + (lr >> 3) * static_cast<uint32_t>(M) : lr;
  uint32_t w_voff[MR];
#pragma unroll
  for (int mr = 0; mr < MR; ++mr)
    w_voff[mr] = ((w_row + kOut * mr) * static_cast<uint32_t>(K) + 8u * lp) * 2u;
  const int src_lane_bytes = (4 * c + q) * 4;
  const __amdgpu_buffer_rsrc_t xr =
      make_rsrc(X, static_cast<uint32_t>(N) * static_cast<uint32_t>(K) * 2u);
  uint32_t x_voff[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int n = n0 + 16 * rb + static_cast<int>(lr);
    x_voff[rb] = n < N ? (static_cast<uint32_t>(n) * K + 8u * lp) * 2u : kOutOfRange;
  }
  auto to_fragment = [&](u32x4_t v) {
    u32x4_t f;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      f[e] = static_cast<uint32_t>(
          __builtin_amdgcn_ds_bpermute(src_lane_bytes, static_cast<int>(v[e])));
    return __builtin_bit_cast(bf16x8_t, f);
  };

  auto load_step = [&](StepRegs<MR, RB>& r, int s) {
    s = min(max(s, 0), steps - 1);  // every scalar offset stays inside the rows
    const uint32_t soff = static_cast<uint32_t>(s) * 64u;
#pragma unroll
    for (int mr = 0; mr < MR; ++mr) r.w[mr] = load16<kCached>(wr, w_voff[mr], soff);
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) r.x[rb] = load16<kCached>(xr, x_voff[rb], soff);
  };
  floatx4_t acc[MR][RB];
#pragma unroll
  for (int mr = 0; mr < MR; ++mr)
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) acc[mr][rb] = floatx4_t{};
  // Accumulator element e of (mr, rb) holds token n0 + 16 rb + 4 q + e, row c of tile mr.
  int bound = share_start(steps, sh + 1, lg_shares);
  auto compute_step = [&](const StepRegs<MR, RB>& r) {
    bf16x8_t a[RB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) a[rb] = to_fragment(r.x[rb]);
#pragma unroll
    for (int mr = 0; mr < MR; ++mr) {
      const bf16x8_t b = to_fragment(r.w[mr]);
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
        acc[mr][rb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[rb], b, acc[mr][rb], 0, 0, 0);
    }
  };
  auto flush = [&]() {
#pragma unroll
    for (int mr = 0; mr < MR; ++mr)
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
#pragma unroll
        for (int e = 0; e < 4; ++e) s_red[sh][(mr * RB + rb) * 4 + e][lane] = acc[mr][rb][e];
        acc[mr][rb] = floatx4_t{};
      }
  };
  auto end_step = [&](int s) {
    if (kOneShare || s + 1 != bound) return;  // else the share's last step
    flush();
    bound = share_start(steps, ++sh + 1, lg_shares);
  };

  StepRegs<MR, RB> slot[D];
#pragma unroll
  for (int j = 0; j < D; ++j) {
    load_step(slot[j], s0 + j < s1 ? s0 + j : s1 - 1);
    __builtin_amdgcn_sched_barrier(0);  // one issue order for prologue and loop
  }
  // Whole rounds of D steps; a slot is refilled with the step D ahead right
  // after its compute (pinned there, so each step waits only for its own
  // loads), clamped to the last step of the slice past its end.
  const int rounds = (s1 - s0) / D;
  int s = s0;
  for (int r = 0; r < rounds; ++r, s += D) {
#pragma unroll
    for (int j = 0; j < D; ++j) {
      compute_step(slot[j]);
      load_step(slot[j], min(s + j + D, s1 - 1));
      end_step(s + j);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int j = 0; j < D - 1; ++j)
    if (s + j < s1) {
      compute_step(slot[j]);
      end_step(s + j);
    }

  if (kOneShare) flush();
  // the shares' sums in share order
  __syncthreads();
  constexpr int kJ = MR * RB * 4;
#pragma unroll
  for (int i = 0; i < (kJ + WV - 1) / WV; ++i) {
    const int j = wave + i * WV;
    if (j >= kJ) break;
    float part[kShares], sum = 0.0f;
#pragma unroll
    for (int w = 0; w < kShares; ++w) part[w] = s_red[min(w, shares - 1)][j][lane];
#pragma unroll
    for (int w = 0; w < kShares; ++w) sum = w < shares ? sum + part[w] : sum;
    const int n = n0 + 16 * (j / 4 % RB) + 4 * q + (j & 3);
    const long long o = static_cast<long long>(n) * M + m0 + kOut * (j / (4 * RB)) + c;
    if constexpr (SWIGLU) {
      const float up = __shfl_xor(sum, 8);  // tile rows 8..15
      if (n < N && c < 8)
        static_cast<uint16_t*>(Yv)[o] = swiglu_one(bf2f(f2bf(sum)), bf2f(f2bf(up)));
    } else if (n < N) {
      if constexpr (F32)
        static_cast<float*>(Yv)[o] = sum;
      else
        static_cast<uint16_t*>(Yv)[o] = f2bf(sum);
    }
  }
}

template <int V>
using Int = std::integral_constant<int, V>;

int log2_shares(int shares) { return __builtin_ctz(static_cast<unsigned>(shares)); }

template <int WV, int MR, int RB, bool SWIGLU, bool F32>
void launch_dense(const uint16_t* W, const uint16_t* X, void* Y, int M, int N, int K, int shares,
                  hipStream_t stream) {
  const dim3 grid(M / ((SWIGLU ? 8 : 16) * MR), ceil_div(N, 16 * RB));
  hipLaunchKernelGGL((dense_gemm_kernel<WV, MR, RB, SWIGLU, F32>), grid, dim3(64 * WV), 0, stream,
                     W, X, Y, M, N, K, log2_shares(shares));
}

template <bool SWIGLU, bool F32>
int dense_tile(const uint16_t* W, const uint16_t* X, void* Y, int rows, int M, int N, int K,
               int shares, int cu, hipStream_t stream, const char* name);

// The K shares of a launch (see "Order of the sums" above): 16 where few 32-feature by
// 16..64-token units make up the output, else as many as keep 64 steps in a share.  The
// numbers were chosen for a kernel whose waves took a share each, and are kept because they
// are part of the results' bits; they no longer say how many waves run.
int k_shares(bool swiglu, int M, int N, int K, int cu) {
  const int units = swiglu ? M / 16 : M / (M % 32 == 0 ? 32 : 16);
  int rb = N <= 16 ? 1 : N <= 32 ? 2 : N <= 48 ? 3 : 4;
  if (rb > 1 && static_cast<long long>(units) * ceil_div(N, 16 * rb) < cu) rb = (rb + 1) / 2;
  const long long n = static_cast<long long>(units) * ceil_div(N, 16 * rb);
  const int steps = K / 32;
  int shares = n <= cu ? 16 : (n <= 2LL * cu ? 8 : 4);
  if (n >= cu)
    while (shares > 1 && steps < 64 * shares) shares >>= 1;
  while (shares > 1 && steps < shares) shares >>= 1;
  return shares;
}

// Shared checks and launch.  rows = W rows read (M, or 2 I for SwiGLU),
// M = output features per token row of Y.
template <bool SWIGLU, bool F32 = false>
int dense_launch(const uint16_t* W, const uint16_t* X, void* Y, int rows, int M, int N, int K,
                 hipStream_t stream, const char* name) {
  if (!W || !X || !Y) return fail(kInvalidValue, "%s: null pointer", name);
  if (M <= 0 || N <= 0 || K <= 0)
    return fail(kInvalidValue, "%s: bad shape M=%d N=%d K=%d", name, M, N, K);
  if (M % 16 != 0 || K % 32 != 0)
    return fail(kNotSupported, "%s: M %% 16 and K %% 32 must be 0 (M=%d K=%d)", name, M, K);
  if ((reinterpret_cast<uintptr_t>(W) & 15u) != 0 || (reinterpret_cast<uintptr_t>(X) & 15u) != 0)
    return fail(kNotSupported, "%s: W and X must be 16-byte aligned", name);
  // X is addressed through one 32-bit buffer range that must stay below the
  // out-of-range offset, and so is a streaming workgroup's W span: its 16 or 32 rows, or
  // with SwiGLU its gate rows through its up rows.  The size of W as a whole does not matter.
  const long long w_span = SWIGLU ? static_cast<long long>(M) + 16 : 32;
  if (static_cast<long long>(N) * K * 2 >= static_cast<long long>(kOutOfRange) ||
      w_span * K * 2 >= static_cast<long long>(kOutOfRange))
    return fail(kNotSupported, "%s: operand span over 2 GiB (rows=%d N=%d K=%d)", name, rows, N,
                K);
  const int cu = current_cu_count();
  if (cu <= 0) return fail(kInvalidValue, "%s: no device", name);
  if (ceil_div(N, 64) > 65535)
    return fail(kNotSupported, "%s: too many token blocks (N=%d)", name, N);
  // The streaming kernel while its workgroups fit one per CU, on the smallest token blocks
  // that do; a second workgroup per CU costs more than reading each fragment for two token
  // blocks (2048 x 2816, 24 tokens, 256 workgroups of 16 or 128 of 32 tokens: 4.5 / 5.7 us;
  // 64 tokens, 512 or 256: 7.3 / 6.0).  Blocks of 48 tokens only where the sums are in 16
  // shares, whose short chunks cost the tile kernel most (router logits, 384 tokens, 23.8
  // here / 29.9 there; with two shares, 4096 x 7168, 40 tokens, 23.7 / 17.6).
  // With more workgroups, the LDS-tiled kernel below from 33 tokens on, and from 17 where its
  // own tiles give the CUs a workgroup each; its tiles read X for 32 features at a time, not
  // 16, which also counts for fewer tokens where the weights are many: from 64 MB at 9 to 16
  // tokens, from 128 MB at 5 to 8 (7168 x 18432, 8 tokens 63 here / 53 there; 16384 x 4096, 9
  // tokens 33 / 30; 5120 x 5120, 9 tokens, 19.0 / 20.0).
  // Between the two, two feature tiles a workgroup, which halve the reads of X: at 5 to 16
  // tokens from 32 MB of weights (5120 x 5120, 8 tokens, 21.0 with one / 18.7 with two; 8192 x
  // 8192, 33.4 against 34.9 with the tile kernel), and for narrow outputs that fit the CUs only
  // so (router logits at 512 tokens, 26.5 against 28 with the tile kernel; 1024 x 4096 at 250
  // tokens, 11.2 / 12.9).
  const long long tiles = rows / 16, w_bytes = 2LL * rows * K;
  const int shares = k_shares(SWIGLU, M, N, K, cu);
  const auto fits = [&](int mr, int rb) { return tiles / mr * ceil_div(N, 16 * rb) <= cu; };
  const int rb = N <= 16 || fits(1, 1) ? 1 : (shares == 16 && !fits(1, 2) && fits(1, 3) ? 3 : 2);
  const bool many = N > 16 || (N > 8 && w_bytes >= (64LL << 20)) ||
                    (N > 4 && w_bytes >= (128LL << 20));
  // a tile workgroup reads up to 128 rows of W through one 32-bit range
  const bool tile_fits = 128LL * K * 2 < static_cast<long long>(kOutOfRange);
  bool two = false;
  if (!fits(1, rb) && tiles % 2 == 0) {
    if (rb == 1)
      two = N > 4 && w_bytes >= (32LL << 20) && shares >= 4 &&
            (!many || (shares == 4 && fits(2, 1)));
    else if (rb == 2)
      two = fits(2, 2) && (shares == 16 ? N > 32 : shares >= 2 && N > 128);
  }
  if (tile_fits && !two && !fits(1, rb) && (N > 32 || (many && tiles >= cu * 5LL / 4)))
    return dense_tile<SWIGLU, F32>(W, X, Y, rows, M, N, K, shares, cu, stream, name);
  const auto go = [&](auto wv, auto mr, auto rbc) {
    launch_dense<decltype(wv)::value, decltype(mr)::value, decltype(rbc)::value, SWIGLU, F32>(
        W, X, Y, M, N, K, shares, stream);
  };
  // waves: a share each, at most four (with two tiles eight)
  const auto go_one = [&](auto wv) {
    if (rb == 1) go(wv, Int<1>{}, Int<1>{});
    else if (rb == 2) go(wv, Int<1>{}, Int<2>{});
    else go(wv, Int<1>{}, Int<3>{});
  };
  const auto go_two = [&](auto wv) {
    if (rb == 1) go(wv, Int<2>{}, Int<1>{});
    else go(wv, Int<2>{}, Int<2>{});
  };
  if (two && shares >= 8) go_two(Int<8>{});
  else if (two && shares == 4) go_two(Int<4>{});
  else if (two) go(Int<2>{}, Int<2>{}, Int<2>{});
  else if (shares >= 4) go_one(Int<4>{});
  else if (shares == 2) go_one(Int<2>{});
  else go_one(Int<1>{});
  return launch_status(name);
}

// ---------------------------------------------------------------- many tokens
// The same GEMM for more tokens: a workgroup owns BM features x BN tokens and brings both
// operands straight from memory to a ring of LDS stages of KC k.  Its waves own disjoint
// blocks of the tile (TM x TN of 16 x 16) for all of K, so that the sums keep the order given
// above: at a share's end a wave adds the share's sums to its totals.  One barrier per chunk.
//
// Kimi's shared expert (gate/up with SwiGLU 4096 x 7168, down 7168 x 2048) at 64 / 160 / 250
// tokens: gate/up 20.8 / 32.5 / 35.0 us, down 9.6 / 20.1 / 20.3 us, against 26.4 / 47.0 / 59.8
// and 12.1 / 22.2 / 30.7 us with the streaming kernel, whose fragments cross lanes through
// ds_bpermute; the router's logits (384 x 7168, fp32) at 1000 / 4096 tokens 27.9 / 67.8
// against 41.0 / 90.6 us.
//
// A row's 16-byte pieces are stored at slot piece ^ (row % 16) (% pieces where a row has
// fewer), which spreads the fragment reads (16 rows, one piece) over the banks.  Bound by what
// a CU can bring in from L2 at few tokens, by LDS reads and the matrix pipe at many.
template <int WM_, int WN_, int TM_, int TN_, int KC_, int NS_>
struct TileShape {
  static constexpr int WM = WM_, WN = WN_, TM = TM_, TN = TN_, KC = KC_, NS = NS_;
  static constexpr int kWaves = WM * WN, kThreads = 64 * kWaves;
  static constexpr int kRowBytes = 2 * KC, kPieces = kRowBytes / 16;
  static constexpr int BM = 16 * WM * TM, BN = 16 * WN * TN;
  static constexpr int kStage = (BM + BN) * kRowBytes;
  static constexpr int kSwizzle = kPieces < 16 ? kPieces : 16;
  static constexpr int kRowsPerLoad = 1024 / kRowBytes;
  static constexpr int P = (BM + BN) / kRowsPerLoad / kWaves;  // loads per wave and chunk
  static constexpr int kPitch = BM + 8;                        // floats per row of the epilogue
  static constexpr int kOut = BN * kPitch * 4;
  static constexpr int kLds = NS * kStage > kOut ? NS * kStage : kOut;
  static_assert(P * kWaves * kRowsPerLoad == BM + BN && KC % 32 == 0, "tile shape");
  static_assert(BM / 2 % kRowsPerLoad == 0, "a load's rows are all gate, up or tokens");
  static_assert(kLds <= 160 * 1024 && NS >= 3 && (kPieces & (kPieces - 1)) == 0, "tile shape");
};

// wide: Y is aligned to four of its elements.  M: output features of a token row of Y
// (inter with SWIGLU, whose W has 2 M rows: the tile's first half holds gate features, its
// second half the matching up features).
template <typename S, bool SWIGLU, bool F32>
__global__ __launch_bounds__(S::kThreads) void dense_tile_kernel(const uint16_t* __restrict__ W,
                                                                 const uint16_t* __restrict__ X,
                                                                 void* __restrict__ Yv, int M,
                                                                 int N, int K, int lg_shares,
                                                                 bool wide) {
  constexpr int BM = S::BM, BN = S::BN, NS = S::NS, P = S::P, TM = S::TM, TN = S::TN;
  constexpr int BMO = SWIGLU ? BM / 2 : BM;  // output features of the tile
  constexpr int kSteps = S::KC / 32;         // 32-k steps per chunk
  __shared__ __align__(1024) uint8_t smem[S::kLds];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % S::WM, wn = wave / S::WM;
  const int c = lane & 15, q = lane >> 4;
  const int m0 = blockIdx.x * BMO, n0 = blockIdx.y * BN;
  const int steps = K >> 5;
  const uint32_t row_bytes = static_cast<uint32_t>(K) * 2u;
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(
      (__attribute__((address_space(3))) uint8_t*)smem));

  // This wave's loads of a chunk: each brings kRowsPerLoad rows of the stage, all gate, up
  // or token rows.  Rows past the last feature or token are out of their resource's range.
  u32x4_t rsrc[P];
  uint32_t dst[P], voff[P];
  int piece_k[P];  // the first k of this lane's piece within a chunk
#pragma unroll
  for (int j = 0; j < P; ++j) {
    const int r0 = (wave * P + j) * S::kRowsPerLoad;
    const bool token = r0 >= BM, up = SWIGLU && !token && r0 >= BMO;
    const int part0 = token ? BM : up ? BMO : 0;  // the part's first row of the stage
    const long long first = token ? n0 : up ? M + m0 : m0;
    const int rows = token ? min(BN, N - n0) : min(BMO, M - m0);
    rsrc[j] = rsrc_words((token ? X : W) + first * K,
                         static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(
                             rows * static_cast<int>(row_bytes))));
    const int r = r0 + lane / S::kPieces;
    const int piece = (lane % S::kPieces) ^ (r % S::kSwizzle);
    dst[j] = lds0 + static_cast<uint32_t>(r0 * S::kRowBytes);
    voff[j] = static_cast<uint32_t>(r - part0) * row_bytes + 16u * piece;
    piece_k[j] = 8 * piece;
  }
  // The chunks: whole KC from each share's first step on, the share's last chunk shorter.
  struct Place {
    int share, step, end;  // the chunk's share, first step, and the share's end
  };
  auto advance = [&](Place& p) {
    p.step += kSteps;
    if (p.step >= p.end) {
      p.step = p.end;
      p.end = share_start(steps, ++p.share + 1, lg_shares);
    }
  };
  const Place first{0, 0, share_start(steps, 1, lg_shares)};
  int chunks = 0;
  for (int w = 0; w < 1 << lg_shares; ++w)
    chunks += (share_start(steps, w + 1, lg_shares) - share_start(steps, w, lg_shares) + kSteps - 1) /
              kSteps;
  auto stage_in = [&](const Place& p, int st) {
    const int past_k = (p.end - p.step) * 32;
#pragma unroll
    for (int j = 0; j < P; ++j) {
      // pieces past the share's end bring zeros, in both operands: their products are zeros
      const uint32_t past = piece_k[j] < past_k ? 0u : kOutOfRange;
      dma_b128(rsrc[j], dst[j] + static_cast<uint32_t>(st), voff[j] | past,
               static_cast<uint32_t>(p.step) * 64u);
    }
  };
  struct Frags {  // of a chunk
    bf16x8_t w[kSteps][TM], x[kSteps][TN];
  };
  const uint8_t* w_rd = smem + (wm * TM * 16 + c) * S::kRowBytes;
  const uint8_t* x_rd = smem + (BM + wn * TN * 16 + c) * S::kRowBytes;
  auto read = [&](Frags& f, int st) {
#pragma unroll
    for (int i = 0; i < kSteps; ++i) {
      const int slot = 16 * ((4 * i + q) ^ (c % S::kSwizzle)) + st;
#pragma unroll
      for (int t = 0; t < TM; ++t)
        f.w[i][t] = *reinterpret_cast<const bf16x8_t*>(w_rd + slot + 16 * S::kRowBytes * t);
#pragma unroll
      for (int t = 0; t < TN; ++t)
        f.x[i][t] = *reinterpret_cast<const bf16x8_t*>(x_rd + slot + 16 * S::kRowBytes * t);
    }
  };
  floatx4_t acc[TM][TN], total[TM][TN];  // a share's sums; the sum of the shares before it
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = total[i][j] = floatx4_t{};
  auto products = [&](const Frags& f) {
#pragma unroll
    for (int i = 0; i < kSteps; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int t = 0; t < TM; ++t)
          acc[t][j] =
              __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.x[i][j], f.w[i][t], acc[t][j], 0, 0, 0);
  };
  auto end_share = [&]() {
#pragma unroll
    for (int t = 0; t < TM; ++t)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
#pragma unroll
        for (int e = 0; e < 4; ++e) total[t][j][e] += acc[t][j][e];
        acc[t][j] = floatx4_t{};
      }
  };

  Place in = first, at = first;  // of the next chunk to bring in, and to multiply
#pragma unroll
  for (int i = 0; i < NS - 1; ++i)
    if (i < chunks) {
      stage_in(in, i * S::kStage);
      advance(in);
    }
  if (chunks >= NS - 1) vm_wait<(NS - 2) * P>(); else vm_wait<0>();
  lds_barrier();
  Frags f0, f1;
  read(f0, 0);
  // Chunk ch: the next chunk has landed (each wave waits for its own loads, the barrier for
  // all), every wave has chunk ch - 1's fragments, whose stage chunk ch + NS - 1 then fills,
  // and the next chunk's fragments are read while this chunk's products run.
  int st_rd = S::kStage, st_in = (NS - 1) * S::kStage;
  auto next = [](int st) { return st + S::kStage == NS * S::kStage ? 0 : st + S::kStage; };
  auto chunk = [&](const Frags& cur, Frags& nxt, int ch) {
    if (ch + NS - 2 < chunks) vm_wait<(NS - 3) * P>(); else vm_wait<0>();
    lds_barrier();
    if (ch + NS - 1 < chunks) {
      stage_in(in, st_in);
      advance(in);
    }
    read(nxt, st_rd);  // past the last chunk: a stage whose words are not used
    st_in = next(st_in);
    st_rd = next(st_rd);
    products(cur);
    const int share = at.share;
    advance(at);
    if (at.share != share) end_share();
  };
  for (int ch = 0; ch < chunks; ch += 2) {
    chunk(f0, f1, ch);
    if (ch + 1 < chunks) chunk(f1, f0, ch + 1);
  }

  // The totals through LDS as [token][feature], then four output features per thread.
  float* out = reinterpret_cast<float*>(smem);
  lds_barrier();  // the ring is read
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        out[((wn * TN + j) * 16 + 4 * q + e) * S::kPitch + (wm * TM + i) * 16 + c] = total[i][j][e];
  __syncthreads();
  for (int o = tid; o < BN * (BMO / 4); o += S::kThreads) {
    const int r = o / (BMO / 4), f = (o % (BMO / 4)) * 4;
    const int n = n0 + r;
    if (n >= N || m0 + f >= M) continue;
    const float4 g4 = *reinterpret_cast<const float4*>(out + r * S::kPitch + f);
    const long long at = static_cast<long long>(n) * M + m0 + f;
    if constexpr (F32) {
      float* y = static_cast<float*>(Yv) + at;
      if (wide) {
        *reinterpret_cast<float4*>(y) = g4;
      } else {
        y[0] = g4.x;
        y[1] = g4.y;
        y[2] = g4.z;
        y[3] = g4.w;
      }
    } else {
      uint16_t* y = static_cast<uint16_t*>(Yv) + at;
      const float g[4] = {g4.x, g4.y, g4.z, g4.w};
      uint16_t b[4];
      if constexpr (SWIGLU) {
        const float4 u4 = *reinterpret_cast<const float4*>(out + r * S::kPitch + f + BMO);
        const float u[4] = {u4.x, u4.y, u4.z, u4.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) b[e] = swiglu_one(bf2f(f2bf(g[e])), bf2f(f2bf(u[e])));
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) b[e] = f2bf(g[e]);
      }
      if (wide) {
        *reinterpret_cast<uint2*>(y) = make_uint2(b[0] | (static_cast<uint32_t>(b[1]) << 16),
                                                  b[2] | (static_cast<uint32_t>(b[3]) << 16));
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = b[e];
      }
    }
  }
}

template <typename S, bool SWIGLU, bool F32>
int launch_tile(const uint16_t* W, const uint16_t* X, void* Y, int M, int N, int K, int shares,
                hipStream_t stream, const char* name) {
  const dim3 grid(ceil_div(M, SWIGLU ? S::BM / 2 : S::BM), ceil_div(N, S::BN));
  // four outputs of a row per store where Y's alignment allows it
  const bool wide = (reinterpret_cast<uintptr_t>(Y) & (F32 ? 15u : 7u)) == 0;
  hipLaunchKernelGGL((dense_tile_kernel<S, SWIGLU, F32>), grid, dim3(S::kThreads), 0, stream, W, X,
                     Y, M, N, K, log2_shares(shares), wide);
  return launch_status(name);
}

// The tile shape whose slowest CU brings in the fewest bytes: a CU's workgroups times the
// rows of a stage, since all of these shapes read their operands at about the same rate
// (what bounds them).  On a tie the larger tile.  The 32 x 32 tile has chunks of 256 k: a wave
// has one MFMA per 32-k step there, so that a chunk's barrier and LDS round trip count most
// (4096 x 7168, 40 tokens, weights not in cache, 17.6 us, 20.9 with eight stages of 128 k and 23.8
// with four; 64 tokens, weights in cache, 16.5 / 20.3 with the first two).
template <bool SWIGLU, bool F32>
int dense_tile(const uint16_t* W, const uint16_t* X, void* Y, int rows, int M, int N, int K,
               int shares, int cu, hipStream_t stream, const char* name) {
  // BM, BN in order of preference
  constexpr int kShapes[6][2] = {{128, 128}, {64, 64}, {64, 32}, {32, 64}, {32, 96}, {32, 32}};
  int pick = 0;
  long long best = -1;
  for (int i = 0; i < 6; ++i) {
    const long long wgs = static_cast<long long>(ceil_div(rows, kShapes[i][0])) *
                          ceil_div(N, kShapes[i][1]);
    const long long cost = (wgs + cu - 1) / cu * (kShapes[i][0] + kShapes[i][1]);
    if (best < 0 || cost < best) {
      best = cost;
      pick = i;
    }
  }
  const auto go = [&](auto shape) {
    return launch_tile<decltype(shape), SWIGLU, F32>(W, X, Y, M, N, K, shares, stream, name);
  };
  switch (pick) {
    case 0: return go(TileShape<4, 2, 2, 4, 64, 4>{});
    case 1: return go(TileShape<2, 4, 2, 1, 128, 4>{});
    case 2: return go(TileShape<4, 2, 1, 1, 128, 6>{});
    case 3: return go(TileShape<2, 4, 1, 1, 128, 6>{});
    case 4: return go(TileShape<2, 2, 1, 3, 128, 4>{});
    default: return go(TileShape<2, 2, 1, 1, 256, 4>{});
  }
}

// ---------------------------------------------------------------- prefill sizes
// From kLtMinTokens tokens up the GEMM is compute-bound and a plain library
// GEMM serves it: hipBLASLt's bf16 x bf16 -> bf16 kernel with fp32 accumulation
// (the reference runs cuBLAS there: cublasGemmEx with CUBLAS_COMPUTE_32F,
// linear.cu:321-344).  Column-major, as the reference states the call:
// C (M x N, ld M) = op_T(W: K x M, ld K) . op_N(X: K x N, ld K).  No workspace
// (an algorithm that needs none), so a call allocates nothing on the device; the
// library handle and each shape's descriptors and algorithm are made on the
// shape's first call on a device and reused.
constexpr int kLtMinTokens = 256;

struct LtPlan {
  hipblasLtMatmulDesc_t desc = nullptr;
  hipblasLtMatrixLayout_t a = nullptr, b = nullptr, c = nullptr;
  hipblasLtMatmulAlgo_t algo{};
};

struct LtDevice {
  std::mutex mu;
  hipblasLtHandle_t handle = nullptr;
  std::map<std::tuple<int, int, int>, LtPlan> plans;
};
LtDevice g_lt[64];

int lt_plan(int dev, int M, int N, int K, const char* name, LtDevice** out_d, LtPlan* out) {
  LtDevice& d = g_lt[dev];
  std::lock_guard<std::mutex> lock(d.mu);
  if (d.handle == nullptr && hipblasLtCreate(&d.handle) != HIPBLAS_STATUS_SUCCESS) {
    d.handle = nullptr;
    return fail(kLaunchFailed, "%s: hipblasLtCreate failed", name);
  }
  const auto key = std::make_tuple(M, N, K);
  auto it = d.plans.find(key);
  if (it == d.plans.end()) {
    LtPlan pl;
    const hipblasOperation_t ta = HIPBLAS_OP_T, tb = HIPBLAS_OP_N;
    bool ok = hipblasLtMatmulDescCreate(&pl.desc, HIPBLAS_COMPUTE_32F, HIP_R_32F) ==
                  HIPBLAS_STATUS_SUCCESS &&
              hipblasLtMatmulDescSetAttribute(pl.desc, HIPBLASLT_MATMUL_DESC_TRANSA, &ta,
                                              sizeof(ta)) == HIPBLAS_STATUS_SUCCESS &&
              hipblasLtMatmulDescSetAttribute(pl.desc, HIPBLASLT_MATMUL_DESC_TRANSB, &tb,
                                              sizeof(tb)) == HIPBLAS_STATUS_SUCCESS &&
              hipblasLtMatrixLayoutCreate(&pl.a, HIP_R_16BF, K, M, K) == HIPBLAS_STATUS_SUCCESS &&
              hipblasLtMatrixLayoutCreate(&pl.b, HIP_R_16BF, K, N, K) == HIPBLAS_STATUS_SUCCESS &&
              hipblasLtMatrixLayoutCreate(&pl.c, HIP_R_16BF, M, N, M) == HIPBLAS_STATUS_SUCCESS;
    hipblasLtMatmulPreference_t pref = nullptr;
    hipblasLtMatmulHeuristicResult_t res[1];
    int found = 0;
    if (ok) {
      const uint64_t ws = 0;
      ok = hipblasLtMatmulPreferenceCreate(&pref) == HIPBLAS_STATUS_SUCCESS &&
           hipblasLtMatmulPreferenceSetAttribute(pref, HIPBLASLT_MATMUL_PREF_MAX_WORKSPACE_BYTES,
                                                 &ws, sizeof(ws)) == HIPBLAS_STATUS_SUCCESS &&
           hipblasLtMatmulAlgoGetHeuristic(d.handle, pl.desc, pl.a, pl.b, pl.c, pl.c, pref, 1,
                                           res, &found) == HIPBLAS_STATUS_SUCCESS &&
           found > 0 && res[0].workspaceSize == 0;
    }
    if (pref) hipblasLtMatmulPreferenceDestroy(pref);
    if (!ok) {
      if (pl.a) hipblasLtMatrixLayoutDestroy(pl.a);
      if (pl.b) hipblasLtMatrixLayoutDestroy(pl.b);
      if (pl.c) hipblasLtMatrixLayoutDestroy(pl.c);
      if (pl.desc) hipblasLtMatmulDescDestroy(pl.desc);
      return fail(kNotSupported, "%s: no hipBLASLt algorithm without workspace for M=%d N=%d K=%d",
                  name, M, N, K);
    }
    pl.algo = res[0].algo;
    it = d.plans.emplace(key, pl).first;
  }
  *out_d = &d;
  *out = it->second;
  return kSuccess;
}

int lt_gemm(const uint16_t* W, const uint16_t* X, uint16_t* Y, int M, int N, int K,
            hipStream_t stream, const char* name) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64)
    return fail(kInvalidValue, "%s: no current device", name);
  LtDevice* d = nullptr;
  LtPlan pl;
  const int rc = lt_plan(dev, M, N, K, name, &d, &pl);
  if (rc != kSuccess) return rc;
  const float alpha = 1.0f, beta = 0.0f;
  const hipblasStatus_t st = hipblasLtMatmul(d->handle, pl.desc, &alpha, W, pl.a, X, pl.b, &beta,
                                             Y, pl.c, Y, pl.c, &pl.algo, nullptr, 0, stream);
  if (st != HIPBLAS_STATUS_SUCCESS) return fail(kLaunchFailed, "%s: hipblasLtMatmul failed", name);
  return launch_status(name);
}

// gemm_cuda / gemm_graphsafe_cuda: the checks of dense_launch, then the token
// count picks the kernel.
int dense_gemm_bf16(const uint16_t* W, const uint16_t* X, uint16_t* Y, int M, int N, int K,
                    hipStream_t stream, const char* name) {
  if (N < kLtMinTokens || !W || !X || !Y || M <= 0 || N <= 0 || K <= 0 || M % 16 != 0 ||
      K % 32 != 0 || (reinterpret_cast<uintptr_t>(W) & 15u) != 0 ||
      (reinterpret_cast<uintptr_t>(X) & 15u) != 0 ||
      static_cast<long long>(N) * K * 2 >= static_cast<long long>(kOutOfRange))
    return dense_launch<false>(W, X, Y, M, M, N, K, stream, name);
  return lt_gemm(W, X, Y, M, N, K, stream, name);
}

}  // namespace

// The router's logits GEMM (fp32 output); declared in common.h.
int dense_gemm_f32(const uint16_t* W, const uint16_t* X, float* Y, int M, int N, int K,
                   hipStream_t stream, const char* name) {
  return dense_launch<false, true>(W, X, Y, M, M, N, K, stream, name);
}

}  // namespace pega

using namespace pega;

// Reference: pegainfer-kernels/src/ffi/shared.rs:220-228 (gemm_cuda) and
// :230-238 (gemm_graphsafe_cuda); both compute the same GEMM.  Below 256
// tokens this library's kernels run; from 256 up, hipBLASLt (no workspace).
// Neither allocates device memory per call, so both are graph-safe once a shape has been called outside the capture (its first call
// on a device makes the hipBLASLt handle and plan).
PEGA_API int gemm_cuda(const uint16_t* W, const uint16_t* X, uint16_t* Y, int M, int N, int K,
                       hipStream_t stream) {
  return dense_gemm_bf16(W, X, Y, M, N, K, stream, "gemm_cuda");
}

PEGA_API int gemm_graphsafe_cuda(const uint16_t* W, const uint16_t* X, uint16_t* Y, int M, int N,
                                 int K, hipStream_t stream) {
  return dense_gemm_bf16(W, X, Y, M, N, K, stream, "gemm_graphsafe_cuda");
}

// No reference counterpart as one symbol: the shared expert's gate/up GEMM
// followed by the SwiGLU of its bf16 output.  The reference runs
// gemm_graphsafe_cuda, then silu_mul_fused_cuda (moe_nccl.rs:113-117 via
// silu_mul_hs_fused_into; csrc/shared/fused_proj.cu:11-31): per element
// bf16(f(bf16(g / (1 + e^-g))) * u) over the [N][2I] gate-then-up rows.  That
// is the same arithmetic as kimi_marlin_w13_swiglu_cuda
// (kimi_marlin_wna16.cu:345-361), which is what the epilogue here computes, so
// the result has the same bits as that pair.
PEGA_API int pega_dense_w13_swiglu(const uint16_t* W13, const uint16_t* X, uint16_t* act,
                                   int inter, int N, int K, hipStream_t stream) {
  if (inter > (1 << 29)) return fail(kInvalidValue, "pega_dense_w13_swiglu: bad inter=%d", inter);
  return dense_launch<true>(W13, X, act, 2 * inter, inter, N, K, stream, "pega_dense_w13_swiglu");
}
