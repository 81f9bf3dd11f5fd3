// Projections of a short prompt for gfx950: y = x W^T (+ bias), bf16 with fp32 sums, and with it the gate of a feed-forward,
// y[:, f] = p[:, f] silu(p[:, F + f]), rounded as the gate kernel and the projection in front of it would round.
//
// Some hundred rows against matrices of a few megabytes, which come from memory once a prompt: neither the rate of the matrix unit nor that of the
// memory bounds such a product, but how soon a compute unit has its rows and columns (40 to 50 bytes a cycle reach its LDS) and what a call
// costs the host.  A workgroup takes a tile of BM tokens x BN features on all channels, rounds of 128 channels three to six deep in LDS,
// loaded there directly; four wavefronts of 64 tokens x 32 features each, side by side or, in the smaller tiles, on different channels of
// the same tile, their sums added through LDS in the end.  The tile is the one whose rounds over the chip's 256 compute units bring the fewest rows
// and columns to one of them; tiles that share columns of the matrix run on the same die.  us, weights from memory, the library (and the gate's own
// launch) before: 4096 x 1024 with the gate, 64 / 128 / 512 rows 13.9 / 14.9 / 16.9 -> 7.4 / 7.5 / 11.5; 1024 x 1024 8.5 / 8.1 / 8.4 -> 6.4 / 6.5 /
// 6.6; 1024 x 2048 8.2 / 8.6 / 9.3 -> 8.9 / 8.9 / 9.0; of the host 20 (28) -> 7.5.  Rounds of 64 channels for the tile of 64 x 64: 1024 x 1024, 1000
// rows 9.1 for 8.2.
#include <atomic>

#include "stream_common.hpp"

namespace based {

struct PromptLinearArgs {
  const __bf16* x;  // (M, K)
  const __bf16* w;  // (N, K), gated: (2 N, K)
  const __bf16* bias;
  __bf16* y;  // (M, N)
  long x_sr, w_sr, y_sr;
  int M, N, K, m_tiles, n_tiles;
};

constexpr int kPlDies = 8, kPlUnits = 256;

__device__ __forceinline__ f32x4 pl_mfma(bf16x8 a, bf16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }

// s_waitcnt of a count of vector memory operations, and of LDS operations where LDS is true
template <int VM, bool LDS> __device__ __forceinline__ void wait_for() {
  __builtin_amdgcn_s_waitcnt((VM & 15) | (VM >> 4 << 14) | 0x70 | (LDS ? 0 : 0xf00));
}

// WM x WN wavefronts side by side, WK on different channels.
template <int WM, int WN, int WK> struct PlTile {
  static constexpr int BM = 64 * WM, BN = 32 * WN, ROWS = BM + BN;
  static constexpr int KS = 128, SLAB = ROWS * 64, ROUND = 2 * SLAB;  // a slab: 64 channels of every row, 128 bytes each
  static constexpr int DEPTH = 144 * 1024 / (ROUND * 2), LDS = DEPTH * ROUND * 2;
  static constexpr int LOADS = ROWS / 16;  // of a wavefront, a round; 8 rows each
  static_assert(WM * WN * WK == 4 && DEPTH >= 3 && (DEPTH - 2) * LOADS < 64, "four wavefronts, counted loads");
};

template <int WM, int WN, int WK, bool GATED>
__global__ __launch_bounds__(256, 1) void prompt_linear_kernel(const PromptLinearArgs a) {
  typedef PlTile<WM, WN, WK> P;
  // (an array whose extent the launch gives: in front of every read of a static one the compiler waits for all loads that go to LDS)
  extern __shared__ __attribute__((aligned(16))) __bf16 pl_lds[];
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, quad = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wk = wave % WK, wn = wave / WK % WN, wm = wave / WK / WN;
  // block i is number i / 8 of die i % 8, which has a run of the tiles in the order of the columns
  const int all = a.m_tiles * a.n_tiles, die = blockIdx.x % kPlDies, more = all % kPlDies;
  const int id = die * (all / kPlDies) + (die < more ? die : more) + (int)(blockIdx.x / kPlDies);
  const int m0 = id % a.m_tiles * P::BM, f0 = id / a.m_tiles * (GATED ? P::BN / 2 : P::BN);
  const int rounds = a.K / P::KS;

  // What a lane asks for: 16 bytes of a row; piece p of a row lies at p ^ (row / 2 % 8), so that reads of 16 rows meet every bank once.
  const char* src[P::LOADS];
#pragma unroll
  for (int i = 0; i < P::LOADS; ++i) {
    const int group = wave * P::LOADS + i, slab = group / (P::ROWS / 8), row = group % (P::ROWS / 8) * 8 + (lane >> 3);
    const int piece = (lane & 7) ^ (row >> 1 & 7);
    const __bf16* at;
    if (row < P::BM) {
      const int m = m0 + row;
      at = a.x + (long)(m < a.M ? m : a.M - 1) * a.x_sr;
    } else {
      const int r = row - P::BM, f = f0 + (GATED ? r / 32 * 16 + r % 16 : r);
      at = a.w + ((long)(f < a.N ? f : a.N - 1) + (GATED && r % 32 >= 16 ? a.N : 0)) * a.w_sr;
    }
    src[i] = reinterpret_cast<const char*>(at + slab * 64 + piece * 8);
  }
  auto ask = [&](int round, int place) {
    const int from = round < rounds ? round : 0;  // (asked for and never read: the count of loads stays)
#pragma unroll
    for (int i = 0; i < P::LOADS; ++i)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src[i] + (long)from * P::KS * 2),
                                       (__attribute__((address_space(3))) void*)(pl_lds + place * P::ROUND + (wave * P::LOADS + i) * 512), 16, 0, 0);
  };
  f32x4 acc[2][4];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int r = 0; r < P::DEPTH - 1; ++r) ask(r, r);
  const int turned = l16 >> 1 & 7;
  for (int round = 0, place = 0; round < rounds; ++round) {
    __builtin_amdgcn_sched_barrier(0);
    wait_for<(P::DEPTH - 2) * P::LOADS, true>();  // own reads are done, and all loads but those of the rounds behind this one
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    ask(round + P::DEPTH - 1, place == 0 ? P::DEPTH - 1 : place - 1);
    __builtin_amdgcn_sched_barrier(0);
    const __bf16* at = pl_lds + place * P::ROUND + l16 * 64;
#pragma unroll
    for (int k = 0; k < 4 / WK; ++k) {
      const int step = wk * (4 / WK) + k, p = (step >> 1) * P::SLAB + (((step & 1) * 4 + quad) ^ turned) * 8;
      bf16x8 w[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) w[i] = *reinterpret_cast<const bf16x8*>(at + (P::BM + wn * 32 + i * 16) * 64 + p);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bf16x8 x = *reinterpret_cast<const bf16x8*>(at + (wm * 64 + j * 16) * 64 + p);
#pragma unroll
        for (int i = 0; i < 2; ++i) acc[i][j] = pl_mfma(w[i], x, acc[i][j]);
      }
    }
    place = place == P::DEPTH - 1 ? 0 : place + 1;
  }
  wait_for<0, true>();  // (nothing may come into LDS that is no longer this workgroup's)
  constexpr int MINE = 4 / WK;
  if constexpr (WK > 1) {
    __builtin_amdgcn_s_barrier();
    f32x4* sums = reinterpret_cast<f32x4*>(pl_lds);  // [wm, wn][wk][i][j][lane]
    f32x4* own = sums + ((wave / WK) * WK + wk) * 512;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) own[(i * 4 + j) * 64 + lane] = acc[i][j];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int n = 0; n < MINE; ++n) {
        const f32x4* at = sums + (wave / WK) * WK * 512 + (i * 4 + wk * MINE + n) * 64 + lane;
        f32x4 s = at[0];
#pragma unroll
        for (int k = 1; k < WK; ++k) s += at[k * 512];
        acc[i][n] = s;
      }
  }
  auto biased = [&](const f32x4& s, int row) {
    bf16x4 o;
    bf16x4 b = {};
    if (a.bias) b = *reinterpret_cast<const bf16x4*>(a.bias + row);
#pragma unroll
    for (int m = 0; m < 4; ++m) o[m] = (__bf16)(a.bias ? s[m] + to_f32(b[m]) : s[m]);
    return o;
  };
#pragma unroll
  for (int n = 0; n < MINE; ++n) {
    const int token = m0 + wm * 64 + (WK > 1 ? wk * MINE + n : n) * 16 + l16;
    if (token >= a.M) continue;
    __bf16* y = a.y + (long)token * a.y_sr;
    if constexpr (GATED) {
      const int f = f0 + wn * 16 + quad * 4;
      if (f < a.N) {
        const bf16x4 value = biased(acc[0][n], f), gate = biased(acc[1][n], a.N + f);
        bf16x4 o;
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          const float g = to_f32(gate[m]);
          o[m] = (__bf16)(to_f32(value[m]) * round_to<__bf16>(g / (1.0f + __expf(-g))));
        }
        *reinterpret_cast<bf16x4*>(y + f) = o;
      }
    } else {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int f = f0 + wn * 32 + i * 16 + quad * 4;
        if (f < a.N) *reinterpret_cast<bf16x4*>(y + f) = biased(acc[i][n], f);
      }
    }
  }
}

constexpr int kPlMaxDevices = 64;

template <int WM, int WN, int WK, bool GATED> static int launch_prompt_linear(PromptLinearArgs a, hipStream_t s) {
  typedef PlTile<WM, WN, WK> P;
  static std::atomic<bool> allowed[kPlMaxDevices];
  int dev = 0;
  BASED_REQUIRE(hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < kPlMaxDevices, BASED_ERR_LAUNCH,
                "prompt_linear: cannot identify the current device");
  if (!allowed[dev].load(std::memory_order_acquire)) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(prompt_linear_kernel<WM, WN, WK, GATED>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, P::LDS);
    BASED_REQUIRE(e == hipSuccess, BASED_ERR_LAUNCH, "prompt_linear: %d bytes of LDS refused: %s", P::LDS, hipGetErrorString(e));
    allowed[dev].store(true, std::memory_order_release);
  }
  a.m_tiles = (a.M + P::BM - 1) / P::BM;
  const int cols = GATED ? P::BN / 2 : P::BN;
  a.n_tiles = (a.N + cols - 1) / cols;
  hipLaunchKernelGGL((prompt_linear_kernel<WM, WN, WK, GATED>), dim3((unsigned)a.m_tiles * (unsigned)a.n_tiles), dim3(256), P::LDS, s, a);
  return check_launch("prompt_linear");
}

// Rows and columns that come to a compute unit, in its rounds over the tiles; one workgroup fills its LDS.
template <int WM, int WN, int WK> static int64_t pl_rows(int64_t M, int64_t columns) {
  typedef PlTile<WM, WN, WK> P;
  const int64_t tiles = ((M + P::BM - 1) / P::BM) * ((columns + P::BN - 1) / P::BN);
  return (tiles + kPlUnits - 1) / kPlUnits * P::ROWS;
}

template <bool GATED> static int run_prompt_linear(const PromptLinearArgs& a, hipStream_t s) {
  const int64_t columns = (int64_t)a.N * (GATED ? 2 : 1);
  const int64_t large = pl_rows<2, 2, 1>(a.M, columns), mid = pl_rows<1, 2, 2>(a.M, columns);
  const int64_t small = pl_rows<1, 1, 4>(a.M, columns);
  if (small <= mid && small <= large) return launch_prompt_linear<1, 1, 4, GATED>(a, s);
  return mid <= large ? launch_prompt_linear<1, 2, 2, GATED>(a, s) : launch_prompt_linear<2, 2, 1, GATED>(a, s);
}

}  // namespace based

extern "C" BASED_API int based_prompt_linear(const void* x, int64_t x_row_stride, const void* w, int64_t w_row_stride, const void* bias,
                                             void* y, int64_t y_row_stride, int64_t M, int64_t N, int64_t K, int gated, void* stream) {
  using namespace based;
  BASED_REQUIRE(x && w && y, BASED_ERR_ARG, "prompt_linear: null pointer argument");
  BASED_REQUIRE(M >= 0 && N > 0 && K > 0 && M < (1 << 24) && N < (1 << 24) && K < (1 << 24), BASED_ERR_SHAPE,
                "prompt_linear: bad sizes (%ld, %ld, %ld)", (long)M, (long)N, (long)K);
  BASED_REQUIRE(K % 128 == 0 && N % 4 == 0, BASED_ERR_SHAPE, "prompt_linear: channels in whole 128 and features in whole 4 (%ld, %ld)", (long)K,
                (long)N);
  BASED_REQUIRE(x_row_stride >= K && w_row_stride >= K && y_row_stride >= N, BASED_ERR_ARG, "prompt_linear: rows overlap");
  BASED_REQUIRE(aligned_to(x, 16) && aligned_to(w, 16) && x_row_stride % 8 == 0 && w_row_stride % 8 == 0 && aligned_to(y, 8) &&
                    y_row_stride % 4 == 0 && (!bias || aligned_to(bias, 8)),
                BASED_ERR_ALIGN, "prompt_linear: rows in whole 16-byte pieces");
  if (M == 0) return BASED_OK;
  const PromptLinearArgs a{static_cast<const __bf16*>(x), static_cast<const __bf16*>(w), static_cast<const __bf16*>(bias), static_cast<__bf16*>(y),
                           x_row_stride, w_row_stride, y_row_stride, (int)M, (int)N, (int)K, 0, 0};
  hipStream_t s = static_cast<hipStream_t>(stream);
  return gated ? run_prompt_linear<true>(a, s) : run_prompt_linear<false>(a, s);
}
