// Real-gated linear recurrent unit for gfx950 (Griffin: Mixing Gated Linear Recurrences with Local
// Attention for Efficient Language Models).  Per channel, in fp32:
//   r = sigmoid(ra u + rb),  i = sigmoid(ri u + ib)      ra, ri block-diagonal: n x n per block
//   log a = -c r softplus(lam),   S_t = a S_{t-1} + sqrt(1 - a^2) i u,   out = S * gelu_tanh(y)
//
//   rglru_segment  both gate products of 64 tokens x 64 channels on MFMA (bf16, or fp32 MFMA for fp32
//                tensors), the decay a and the input x = sqrt(1 - a^2) i u formed behind them in fp32, the
//                recurrence over the 64 tokens as S -> P S + X, and, from the (P, X) of the segments in
//                front, the outputs.
//   rglru_step   one token per sequence: the short convolution on its ring of past inputs, the gates,
//                the state update and the output gate.
#include "stream_common.hpp"

namespace based {

constexpr int kSeg = 64;    // tokens per segment
constexpr int kGroup = 64;  // segments whose last one leaves the state behind it

struct RglruArgs {
  const void* u;  // (B, L, W), strides
  const void* y;
  const void* ra;  // (blocks, n, n) [out, in]
  const void* rb;
  const void* ri;
  const void* ib;
  const void* lam;
  unsigned long long* agg;  // (B, segments, W): P below X, kUnset until a segment has them
  int* tickets;  // (B, tiles) ticket_step apart: segments begun
  int ticket_step;
  float* state;  // (B, W)
  void* out;
  int B, L, W, n, segs;
  long u_sb, u_sl, y_sb, y_sl, o_sb, o_sl;
  float c;
  int fresh;
  bool vec_u, vec_y;  // rows of u, ra and ri, and of y and out, in 16-byte pieces
};

template <typename T> struct GateMma;
template <> struct GateMma<__bf16> {
  static constexpr int kK = 32;  // contraction per instruction
  typedef bf16x8 frag_t;
  static constexpr int kPer = 8;
  static __device__ __forceinline__ f32x4 run(frag_t a, frag_t b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};
template <> struct GateMma<float> {
  static constexpr int kK = 4;
  typedef float frag_t;
  static constexpr int kPer = 1;
  static __device__ __forceinline__ f32x4 run(frag_t a, frag_t b, f32x4 c) {
    return mfma_f32(a, b, c);
  }
};

__device__ __forceinline__ void lru_gates(float zr, float zi, float sp, float u, float c, float& a, float& x) {
  const float r = sigmoid_f(zr), i = sigmoid_f(zi);
  const float log_a = -c * r * sp;
  a = exp_f(log_a);
  x = __builtin_amdgcn_sqrtf(one_minus_square(a, log_a)) * i * u;
}

// lru_gates with the products before their biases: nrb, nib = -log2(e) times the bias, k2 = -2 c softplus(lam), kl = log2(e) / 2 times that.
__device__ __forceinline__ void lru_gates_of(float zr, float zi, float nrb, float nib, float k2, float kl, float u, float& a, float& x) {
  constexpr float kL = 1.4426950408889634f;
  const float r = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(__builtin_fmaf(zr, -kL, nrb)));
  const float i = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(__builtin_fmaf(zi, -kL, nib)));
  a = __builtin_amdgcn_exp2f(kl * r);
  x = __builtin_amdgcn_sqrtf(one_minus_square_of(a, k2 * r)) * (i * u);
}

constexpr unsigned long long kUnset = ~0ull;  // P as a NaN that no segment leaves

__global__ __launch_bounds__(256) void rglru_begin_kernel(unsigned long long* agg, long n, int* tickets, int count, int step) {
  const long at = (long)blockIdx.x * 256 + threadIdx.x, all = (long)gridDim.x * 256;
  for (long i = at; i < n; i += all) agg[i] = kUnset;
  for (long i = at; i < count; i += all) tickets[i * step] = 0;
}

// grid: x = segments of the sequence, y = 64-channel tile within its block (ceil(n / 64) per block), z = sequence.
// A workgroup takes the next segment of its tile and sequence, forms the gates of 64 tokens, leaves what they do to any state that enters
// them for the segments behind, and takes the state that enters its own from those in front.  Those were taken before it by workgroups
// that run or have run and that wait for none behind them, so each wait ends.  P and X travel in one 64-bit word, which is its own flag.
// The last of every kGroup segments leaves the state itself (P = 0) instead, once it has it, and nobody reads behind that: at most kGroup
// words a segment whatever the length (all those in front: 1,920 us for the 2,048 segments of B = 1, L = 131072, W = 1024 in bf16; in groups
// 664; at L = 16384 73 and 66).  A fixed place, not the nearest state that is there: the same sums on every run.
// Gates as fp32 pairs through memory for a second kernel, 134 of 184 MB at B = 4, L = 2048, W = 1024, 8 blocks, took 51 us; gates formed
// by two kernels, 43 us: the vector unit is the bound, three exponentials, two reciprocals and a square root an element.  This way 28 us
// with the kernel in front; B = 8, L = 4096: 92 (218).  The products lie with 16 consecutive tokens of a channel in one lane, where the
// recurrence is two instructions an element, and 64 in a wavefront.
// NI: tiles of 16 tokens in a segment, 4 NI tokens to a lane: 4, or as few as hold a short prompt, whose other rows would be products for nothing.
template <typename T, int NI>
__global__ __launch_bounds__(256, sizeof(T) == 4 ? 3 : 4) void rglru_segment_kernel(const RglruArgs a) {
  typedef GateMma<T> M;
  typedef typename Pack<T>::type vec_t;
  constexpr int V = Pack<T>::kN;
  constexpr int KT = 64, KS = KT + 16 / (int)sizeof(T);  // contraction staged at a time
  constexpr int SEG = 16 * NI, TL = 4 * NI;
  __shared__ __attribute__((aligned(16))) T s_u[SEG * KS], s_r[64 * KS], s_i[64 * KS];
  T* s_y = s_r;  // (the output gate, then the output, once the products are done)
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, quad = lane >> 4;
  const int tiles = (a.n + 63) / 64;
  const int blk = blockIdx.y / tiles, c0 = (blockIdx.y % tiles) * 64;  // first output channel within the block
  const int b = blockIdx.z;
  __shared__ int s_seg;
  if (a.segs > 1) {
    if (tid == 0) s_seg = atomicAdd(a.tickets + ((long)b * gridDim.y + blockIdx.y) * a.ticket_step, 1);
    __syncthreads();
  }
  const int seg = a.segs > 1 ? __builtin_amdgcn_readfirstlane(s_seg) : 0, l0 = seg * SEG;
  const T* u = static_cast<const T*>(a.u) + b * a.u_sb + (long)blk * a.n;
  const T* ra = static_cast<const T*>(a.ra) + (long)blk * a.n * a.n;
  const T* ri = static_cast<const T*>(a.ri) + (long)blk * a.n * a.n;
  const int ch = c0 + wave * 16 + l16;  // a channel per column of a wavefront's products
  const int w = blk * a.n + (ch < a.n ? ch : a.n - 1);
  constexpr float kL = 1.4426950408889634f;
  const float nrb = -kL * to_f32(static_cast<const T*>(a.rb)[w]), nib = -kL * to_f32(static_cast<const T*>(a.ib)[w]);
  const float k2 = -2.0f * a.c * softplus_f(to_f32(static_cast<const T*>(a.lam)[w]));
  const float kl = (0.5f * kL) * k2;
  // Token q * TL + i * 4 + j of the segment stands in row i * 16 + q * 4 + j: element j of product i in the lanes of quad q.
  const auto token_of = [](int row) { return (row >> 2 & 3) * TL + (row >> 4) * 4 + (row & 3); };
  // Rows of no whole pieces go element by element: as many columns as are live, rounded up to a power of two (and to `least`).  All 64
  // columns cost fp32 at B = 4, L = 2048, 7 blocks of 143 channels 180 us (124 now) and 1,024 blocks of one channel at L = 777 233 (167).
  const auto columns = [](int live, int least) { return 32 - __builtin_clz((live > least ? live : least) * 2 - 1) - 1; };
  constexpr int YP = (SEG * 64 / V + 255) / 256, YN = SEG * 64 / V;
  vec_t yv[YP];
  const T* y = static_cast<const T*>(a.y) + b * a.y_sb + (long)blk * a.n + c0;
  if (a.vec_y) {
#pragma unroll
    for (int i = 0; i < YP; ++i) {
      const int p = i * 256 + tid, e = p % (64 / V) * V, t = l0 + token_of(p / (64 / V) % SEG);
      yv[i] = *reinterpret_cast<const vec_t*>(y + (t < a.L ? t : a.L - 1) * a.y_sl + (c0 + e < a.n ? e : 0));
    }
  }
  f32x4 zr[NI], zi[NI];  // wavefront: 16 NI tokens (rows) x 16 channels (columns)
#pragma unroll
  for (int i = 0; i < NI; ++i) zr[i] = zi[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  // 64 channels of u and of the gates' rows, asked for one round ahead where the tile is small: a round's products are then shorter than the
  // wait.  A whole segment has other blocks on the unit meanwhile and no registers left (27 spilled, B = 4, L = 2,048 in 40 us for 31).
  constexpr bool AHEAD = NI < 4;
  constexpr int PIECES = 64 * (KT / V) / 256, UN = SEG * (KT / V), UP = (UN + 255) / 256;
  vec_t xu[UP], xr[PIECES], xi[PIECES];
  const auto fetch = [&](int k0) {
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int p = i * 256 + tid, row = p / (KT / V), e = (p % (KT / V)) * V;
      const int c = c0 + row < a.n ? c0 + row : a.n - 1, k = k0 + e < a.n ? k0 + e : 0;
      if (i < UP) {
        const int t = l0 + token_of(row % SEG);
        xu[i] = *reinterpret_cast<const vec_t*>(u + (t < a.L ? t : a.L - 1) * a.u_sl + k);
      }
      xr[i] = *reinterpret_cast<const vec_t*>(ra + (long)c * a.n + k);
      xi[i] = *reinterpret_cast<const vec_t*>(ri + (long)c * a.n + k);
    }
  };
  const auto next = [&](int k0) { return k0 + KT < tiles * KT ? k0 + KT : 0; };
  if (AHEAD && a.vec_u) fetch(next(c0));
  for (int it = 1, k0 = c0; it <= tiles; ++it) {  // the tile's own channels last: their u stays staged
    k0 = next(k0);
    if (it > 1) __syncthreads();
    const int live = a.n - k0 < KT ? a.n - k0 : KT;
    if (a.vec_u) {
      if (!AHEAD) fetch(k0);
#pragma unroll
      for (int i = 0; i < PIECES; ++i) {
        const int p = i * 256 + tid, row = p / (KT / V), e = (p % (KT / V)) * V;
        const bool in = k0 + e < a.n;
        if (i < UP && (UN % 256 == 0 || p < UN)) *reinterpret_cast<vec_t*>(&s_u[row * KS + e]) = in ? xu[i < UP ? i : 0] : vec_t{};
        *reinterpret_cast<vec_t*>(&s_r[row * KS + e]) = in ? xr[i] : vec_t{};
        *reinterpret_cast<vec_t*>(&s_i[row * KS + e]) = in ? xi[i] : vec_t{};
      }
      if (AHEAD && it < tiles) fetch(next(k0));
    } else {
      const int sh = columns(live, M::kK);
#pragma unroll 4
      for (int p = tid; p < 64 << sh; p += 256) {
        const int row = p >> sh, e = p - (row << sh);
        const int t = l0 + token_of(row % SEG), c = c0 + row < a.n ? c0 + row : a.n - 1;
        const bool in = e < live;
        const int k = in ? k0 + e : 0;
        const T xu = u[(t < a.L ? t : a.L - 1) * a.u_sl + k], xr = ra[(long)c * a.n + k], xi = ri[(long)c * a.n + k];
        if (row < SEG) s_u[row * KS + e] = in ? xu : (T)0.0f;
        s_r[row * KS + e] = in ? xr : (T)0.0f;
        s_i[row * KS + e] = in ? xi : (T)0.0f;
      }
    }
    __syncthreads();
    const auto product = [&](int kk) {
      const int e = kk + quad * M::kPer;
      const typename M::frag_t fr = *reinterpret_cast<const typename M::frag_t*>(&s_r[(wave * 16 + l16) * KS + e]);
      const typename M::frag_t fi = *reinterpret_cast<const typename M::frag_t*>(&s_i[(wave * 16 + l16) * KS + e]);
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const typename M::frag_t fu = *reinterpret_cast<const typename M::frag_t*>(&s_u[(i * 16 + l16) * KS + e]);
        zr[i] = M::run(fu, fr, zr[i]);
        zi[i] = M::run(fu, fi, zi[i]);
      }
    };
    if (live == KT) {
#pragma unroll
      for (int kk = 0; kk < KT; kk += M::kK) product(kk);
    } else {
#pragma unroll 1
      for (int kk = 0; kk < live; kk += M::kK) product(kk);
    }
  }
  __syncthreads();
  if (a.vec_y) {
#pragma unroll
    for (int i = 0; i < YP; ++i) {
      const int p = i * 256 + tid;
      if (YN % 256 != 0 && p >= YN) break;
      *reinterpret_cast<vec_t*>(&s_y[p / (64 / V) * KS + p % (64 / V) * V]) = yv[i];
    }
  } else {
    const int sh = columns(a.n - c0 < 64 ? a.n - c0 : 64, 1);
#pragma unroll 4
    for (int p = tid; p < SEG << sh; p += 256) {
      const int row = p >> sh, e = p - (row << sh), t = l0 + token_of(row);
      s_y[row * KS + e] = y[(t < a.L ? t : a.L - 1) * a.y_sl + (c0 + e < a.n ? e : 0)];
    }
  }
  __syncthreads();
  float A[NI][4], I[NI][4];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      lru_gates_of(zr[i][j], zi[i][j], nrb, nib, k2, kl, to_f32(s_u[(i * 16 + quad * 4 + j) * KS + wave * 16 + l16]), A[i][j], I[i][j]);
  if (l0 + SEG > a.L) {  // tokens behind the last one change nothing
    const int live = a.L - l0 - quad * TL;
#pragma unroll
    for (int t = 0; t < TL; ++t) {
      A[t / 4][t % 4] = t < live ? A[t / 4][t % 4] : 1.f;
      I[t / 4][t % 4] = t < live ? I[t / 4][t % 4] : 0.f;
    }
  }
  float P = A[0][0], X = I[0][0];
#pragma unroll
  for (int t = 1; t < TL; ++t) {
    X = __builtin_fmaf(A[t / 4][t % 4], X, I[t / 4][t % 4]);
    P *= A[t / 4][t % 4];
  }
  // Where no decay of the channel is zero (2^kl at the least), no product of them is: the smallest number there is, as near as the format
  // comes, and an infinite state outlives them, as it does token by token.
  const float least = kl > -126.f ? 0x1p-149f : 0.f;
  P = fmaxf(P, least);
  // the quads in front of this one
  float before_p = 1.f, before_x = 0.f;
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    const float p = __shfl(P, q * 16 + l16), x = __shfl(X, q * 16 + l16);
    before_x = q < quad ? __builtin_fmaf(p, before_x, x) : before_x;
    before_p = q < quad ? fmaxf(p * before_p, least) : before_p;
  }
  float S = seg == 0 && !a.fresh ? a.state[(long)b * a.W + w] : 0.f;
  unsigned long long* g = a.agg + (long)b * a.segs * a.W + w;
  const auto leave = [&](float pw, float xw) {
    unsigned int bits = __builtin_bit_cast(unsigned int, pw);
    bits = bits == ~0u ? 0x7fc00000u : bits;
    __hip_atomic_store(g + (long)seg * a.W, (unsigned long long)__builtin_bit_cast(unsigned int, xw) << 32 | bits, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  };
  const bool mine = quad == 3 && ch < a.n, closes = seg % kGroup == kGroup - 1;
  if (seg < a.segs - 1 && mine && !closes) {
    float xw = __builtin_fmaf(P, before_x, X), pw = fmaxf(P * before_p, least);
    if (seg == 0) {  // (what enters the call is part of it: the last segment replaces the state)
      xw = __builtin_fmaf(pw, S, xw);
      pw = 0.f;
    }
    leave(pw, xw);
  }
  if (seg > 0) {
    // a quarter of the segments in front for each quad, from the one that closes the group before on
    const int from = seg < kGroup ? 0 : seg / kGroup * kGroup - 1, count = seg - from;
    const int each = (count + 3) / 4, first = quad * each;
    const unsigned long long* in_front = g + (long)from * a.W;
    float p = 1.f, x = 0.f;
    constexpr int U = 4;
    for (int i0 = 0; i0 < each; i0 += U) {
      unsigned long long v[U];
      bool wait;
      do {
        wait = false;
#pragma unroll
        for (int i = 0; i < U; ++i) {
          const int at = first + i0 + i;
          v[i] = __hip_atomic_load(in_front + (long)(at < count ? at : count - 1) * a.W, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
#pragma unroll
        for (int i = 0; i < U; ++i) wait |= (unsigned int)v[i] == ~0u;
      } while (__any(wait));
#pragma unroll
      for (int i = 0; i < U; ++i) {
        const bool in = i0 + i < each && first + i0 + i < count;
        const float pi = __builtin_bit_cast(float, (unsigned int)v[i]), xi = __builtin_bit_cast(float, (unsigned int)(v[i] >> 32));
        x = in ? __builtin_fmaf(pi, x, xi) : x;
        p = in ? fmaxf(p * pi, least) : p;
      }
    }
    S = __shfl(x, l16);
#pragma unroll
    for (int q = 1; q < 4; ++q) S = __builtin_fmaf(__shfl(p, q * 16 + l16), S, __shfl(x, q * 16 + l16));
  }
  S = __builtin_fmaf(before_p, S, before_x);
  if (seg < a.segs - 1 && mine && closes) leave(0.f, __builtin_fmaf(P, S, X));
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      S = __builtin_fmaf(A[i][j], S, I[i][j]);
      T* at = &s_y[(i * 16 + quad * 4 + j) * KS + wave * 16 + l16];
      *at = from_f32<T>(S * gelu_tanh_f(to_f32(*at)));
    }
  if (seg == a.segs - 1 && mine) a.state[(long)b * a.W + w] = S;
  __syncthreads();
  T* out = static_cast<T*>(a.out) + b * a.o_sb + (long)blk * a.n + c0;
  if (a.vec_y) {
#pragma unroll
    for (int i = 0; i < YP; ++i) {
      const int p = i * 256 + tid, row = p / (64 / V), e = p % (64 / V) * V, t = l0 + token_of(row);
      if (YN % 256 != 0 && p >= YN) break;
      if (t < a.L && c0 + e < a.n) *reinterpret_cast<vec_t*>(out + t * a.o_sl + e) = *reinterpret_cast<const vec_t*>(&s_y[row * KS + e]);
    }
  } else {
    const int sh = columns(a.n - c0 < 64 ? a.n - c0 : 64, 1);
    for (int p = tid; p < SEG << sh; p += 256) {
      const int row = p >> sh, e = p - (row << sh), t = l0 + token_of(row);
      if (t < a.L && c0 + e < a.n) out[t * a.o_sl + e] = s_y[row * KS + e];
    }
  }
}

// Rows from the scratch to an output that shares memory with the input, V elements at a time; 8 rows of a sequence per workgroup.
constexpr int kCopyRows = 8;
template <typename T, int V> __global__ __launch_bounds__(256) void rglru_copy_kernel(const T* src, T* dst, int L, int W, long o_sb, long o_sl) {
  typedef __attribute__((ext_vector_type(V))) T vec_t;
  const int l0 = blockIdx.x * kCopyRows, rows = L - l0 < kCopyRows ? L - l0 : kCopyRows;
  const unsigned pieces = W / V;
  src += ((long)blockIdx.y * L + l0) * W;
  dst += blockIdx.y * o_sb + l0 * o_sl;
  if constexpr (V > 1) {
    for (unsigned p = threadIdx.x; p < rows * pieces; p += 256) {
      const unsigned row = p / pieces, e = (p - row * pieces) * V;
      *reinterpret_cast<vec_t*>(dst + row * o_sl + e) = *reinterpret_cast<const vec_t*>(src + (long)row * W + e);
    }
  } else {  // a row per wavefront, eight loads ahead
    for (int row = threadIdx.x >> 6; row < rows; row += 4)
      for (int e0 = threadIdx.x & 63; e0 < W; e0 += 8 * 64) {
        T x[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = src[(long)row * W + (e0 + i * 64 < W ? e0 + i * 64 : W - 1)];
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (e0 + i * 64 < W) dst[row * o_sl + e0 + i * 64] = x[i];
      }
  }
}

// ---- one token per sequence ----
struct RglruStepArgs {
  const void* x;  // (B, W): input of the short convolution
  const void* y;
  const void* conv_w;  // (taps, W)
  const void* conv_b;
  void* ring;  // (B, taps, W)
  const void* ra;
  const void* rb;
  const void* ri;
  const void* ib;
  const void* lam;
  float* state;
  void* out;
  const int32_t* pos;
  int pos_host;
  int B, W, n, taps;
  long x_sb, y_sb, o_sb, ring_sb;
  float c;
};

constexpr int kLruRows = 8;  // sequences held at a time

// a piece of a gate row: 16 bytes, or one element
template <typename T, bool VEC> struct LruPiece {
  typedef typename Pack<T>::type type;
  static __device__ __forceinline__ float get(type x, int i) { return to_f32(x[i]); }
};
template <typename T> struct LruPiece<T, false> {
  typedef T type;
  static __device__ __forceinline__ float get(type x, int) { return to_f32(x); }
};

// A workgroup takes 32 output channels of one block (a wavefront 8 of them, 8 lanes per channel) and
// up to kLruRows sequences; the convolved inputs of the whole block go through LDS.
template <typename T, bool VEC>
__global__ __launch_bounds__(256) void rglru_step_kernel(const RglruStepArgs a) {
  constexpr int N = VEC ? Pack<T>::kN : 1;
  extern __shared__ __attribute__((aligned(16))) float s_u[];  // [kLruRows][n rounded up to 4]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int tiles = (a.n + 31) / 32;
  const int blk = blockIdx.x / tiles, tile = blockIdx.x % tiles, m0 = blockIdx.y * kLruRows;
  const int rows = a.B - m0 < kLruRows ? a.B - m0 : kLruRows;
  const int ns = (a.n + 3) & ~3;  // rows of whole 16-byte pieces
  const int ch = tile * 32 + wave * 8 + (lane >> 3), part = lane & 7;
  const bool ok = ch < a.n;
  const int cc = ok ? ch : a.n - 1;
  // What does not depend on a position is asked for first: the first pieces of the gate rows, and what the
  // lane needs that finishes sequence m0 + part.
  const T* wr = static_cast<const T*>(a.ra) + ((long)blk * a.n + cc) * a.n;
  const T* wi = static_cast<const T*>(a.ri) + ((long)blk * a.n + cc) * a.n;
  typedef typename LruPiece<T, VEC>::type piece_t;
  piece_t pr[2], pi[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int k = (part + 8 * i) * N;
    pr[i] = *reinterpret_cast<const piece_t*>(wr + (k < a.n ? k : 0));
    pi[i] = *reinterpret_cast<const piece_t*>(wi + (k < a.n ? k : 0));
  }
  const int bp = m0 + (part < rows ? part : 0), wc = blk * a.n + cc;
  const T rb = static_cast<const T*>(a.rb)[wc], ib = static_cast<const T*>(a.ib)[wc], lam = static_cast<const T*>(a.lam)[wc];
  const T yv = static_cast<const T*>(a.y)[bp * a.y_sb + wc];
  const float old = a.state[(long)bp * a.W + wc];
  const int pos_p = row_pos(a.pos, a.pos_host, bp);

  // the convolved inputs of the block: `share` threads per channel, each with every share-th sequence, four of
  // them in flight together
  const int share = a.n >= 256 ? 1 : 256 / a.n;
  for (int k = tid % (256 / share); k < a.n; k += 256 / share) {
    if (tid / (256 / share) >= share) break;
    const int chn = blk * a.n + k;
    const T* cw = static_cast<const T*>(a.conv_w) + chn;
    const float bias = a.conv_b != nullptr ? to_f32(static_cast<const T*>(a.conv_b)[chn]) : 0.f;
    for (int mb = tid / (256 / share); mb < rows; mb += 4 * share) {
      int pos[4];
      T now[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int m = mb + j * share < rows ? mb + j * share : rows - 1;
        pos[j] = row_pos(a.pos, a.pos_host, m0 + m);
        now[j] = static_cast<const T*>(a.x)[(m0 + m) * a.x_sb + chn];
      }
      float acc[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[j] = bias;
      for (int t0 = 0; t0 < a.taps - 1; t0 += 3) {
        T xv[4][3], cv[3];
#pragma unroll
        for (int t = 0; t < 3; ++t) {
          cv[t] = cw[(long)(t0 + t < a.taps - 1 ? t0 + t : 0) * a.W];
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int m = mb + j * share < rows ? mb + j * share : rows - 1;
            const int p = pos[j] - (a.taps - 1) + t0 + t;
            const bool in = t0 + t < a.taps - 1 && p >= 0;
            xv[j][t] = static_cast<const T*>(a.ring)[(m0 + m) * a.ring_sb + (long)(in ? p % a.taps : 0) * a.W + chn];
          }
        }
#pragma unroll
        for (int t = 0; t < 3; ++t)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int p = pos[j] - (a.taps - 1) + t0 + t;
            const bool in = t0 + t < a.taps - 1 && p >= 0;
            acc[j] = in ? __builtin_fmaf(to_f32(cv[t]), to_f32(xv[j][t]), acc[j]) : acc[j];
          }
      }
      const float c_last = to_f32(cw[(long)(a.taps - 1) * a.W]);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int m = mb + j * share;
        if (m < rows) {
          s_u[m * ns + k] = round_to<T>(__builtin_fmaf(c_last, to_f32(now[j]), acc[j]));
          // a slot that no reader of this step looks at; one tile of the block writes it
          if (tile == 0 && pos[j] >= 0) static_cast<T*>(a.ring)[(m0 + m) * a.ring_sb + (long)(pos[j] % a.taps) * a.W + chn] = now[j];
        }
      }
    }
  }
  for (int i = tid; i < (kLruRows - rows) * ns; i += 256) s_u[rows * ns + i] = 0.f;
  __syncthreads();
  float zr[kLruRows], zi[kLruRows];
#pragma unroll
  for (int m = 0; m < kLruRows; ++m) zr[m] = zi[m] = 0.f;
  for (int k = part * N, it = 0; k < a.n; k += 8 * N, ++it) {
    const piece_t rp = it == 0 ? pr[0] : it == 1 ? pr[1] : *reinterpret_cast<const piece_t*>(wr + k);
    const piece_t ip = it == 0 ? pi[0] : it == 1 ? pi[1] : *reinterpret_cast<const piece_t*>(wi + k);
    float r[N], q[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
      r[j] = LruPiece<T, VEC>::get(rp, j);
      q[j] = LruPiece<T, VEC>::get(ip, j);
    }
#pragma unroll
    for (int m = 0; m < kLruRows; ++m) {
      float uv[N];
      if constexpr (VEC)
        load_vec<float, N>(&s_u[m * ns + k], uv);
      else
        uv[0] = s_u[m * ns + k];
#pragma unroll
      for (int j = 0; j < N; ++j) {
        zr[m] = __builtin_fmaf(r[j], uv[j], zr[m]);
        zi[m] = __builtin_fmaf(q[j], uv[j], zi[m]);
      }
    }
  }
  float my_r = 0.f, my_i = 0.f;
#pragma unroll
  for (int m = 0; m < kLruRows; ++m) {
    const float sr = sum8(zr[m]), si = sum8(zi[m]);
    my_r = part == m ? sr : my_r;
    my_i = part == m ? si : my_i;
  }
  // lane `part` finishes sequence m0 + part
  if (ok && part < rows) {
    float av, x;
    lru_gates(my_r + to_f32(rb), my_i + to_f32(ib), softplus_f(to_f32(lam)), s_u[part * ns + ch], a.c, av, x);
    const float S = pos_p > 0 ? __builtin_fmaf(av, old, x) : x;
    a.state[(long)bp * a.W + wc] = S;
    static_cast<T*>(a.out)[bp * a.o_sb + wc] = from_f32<T>(S * gelu_tanh_f(to_f32(yv)));
  }
}

template <typename T> void launch_rglru_prefill(const RglruArgs& a, int tiles, T* apart, hipStream_t s) {
  const dim3 grid((unsigned)a.segs, (unsigned)tiles, (unsigned)a.B), block(256);
  RglruArgs t = a;
  if (apart) {
    t.out = apart;
    t.o_sl = a.W;
    t.o_sb = (long)a.L * a.W;
    t.vec_y = a.vec_y && aligned_to(apart, 16);
  }
  if (a.segs > 1) {
    const long words = (long)a.B * a.segs * a.W;
    const long groups = (words + 1023) / 1024;
    hipLaunchKernelGGL(rglru_begin_kernel, dim3((unsigned)(groups < 2048 ? groups : 2048)), block, 0, s, a.agg, words, a.tickets, a.B * tiles,
                       a.ticket_step);
  }
  // One segment of as few 16-token tiles as hold a short prompt.  bf16, 15 rows of 9 tokens, W = 1536 in 6 blocks: 10.5 us on the whole tile,
  // 6.5 on one of 16; 3 of 20, W = 1024 in 8: 6.9 and 5.3 on one of 32; fp32, 11 of 8 and 2 of 24 of these widths: 25 and 11, 11.3 and 7.7.
  if (a.L <= 16)
    hipLaunchKernelGGL((rglru_segment_kernel<T, 1>), grid, block, 0, s, t);
  else if (a.L <= 32)
    hipLaunchKernelGGL((rglru_segment_kernel<T, 2>), grid, block, 0, s, t);
  else
    hipLaunchKernelGGL((rglru_segment_kernel<T, kSeg / 16>), grid, block, 0, s, t);
  if (apart) {
    constexpr int V = Pack<T>::kN;
    const bool vec = a.W % V == 0 && a.o_sl % V == 0 && a.o_sb % V == 0 && aligned_to(a.out, 16) && aligned_to(apart, 16);
    hipLaunchKernelGGL((vec ? rglru_copy_kernel<T, V> : rglru_copy_kernel<T, 1>), dim3((unsigned)((a.L + kCopyRows - 1) / kCopyRows), (unsigned)a.B),
                       block, 0, s, apart, static_cast<T*>(a.out), a.L, a.W, a.o_sb, a.o_sl);
  }
}

// Whether two (B, L, W) tensors may share elements: their stretches of memory overlap, and they are not the columns of one matrix next
// to each other (rows a whole number of row strides apart, W columns that the other does not reach).
static bool rglru_meet(const void* p, int64_t p_sb, int64_t p_sl, const void* q, int64_t q_sb, int64_t q_sl, int64_t B, int64_t L, int64_t W,
                       int64_t size) {
  const auto edge = [&](const void* base, int64_t sb, int64_t sl, bool high) {
    int64_t e = high ? W : 0;
    for (const int64_t d : {(B - 1) * sb, (L - 1) * sl}) e += (d > 0) == high ? d : 0;
    return (int64_t)(uintptr_t)base + e * size;
  };
  if (edge(p, p_sb, p_sl, false) >= edge(q, q_sb, q_sl, true) || edge(q, q_sb, q_sl, false) >= edge(p, p_sb, p_sl, true)) return false;
  const int64_t row = L > 1 ? p_sl : p_sb, by = (int64_t)(uintptr_t)q - (int64_t)(uintptr_t)p;
  if ((L > 1 && p_sl != q_sl) || (B > 1 && p_sb != q_sb) || row <= 0 || (B > 1 && p_sb % row != 0) || by % size != 0) return true;
  const int64_t col = ((by / size) % row + row) % row;
  return col < W || col + W > row;
}

}  // namespace based

extern "C" BASED_API int64_t based_rglru_prefill_work(const void* u, const void* out, int64_t B, int64_t L, int64_t W, int64_t u_sb,
                                                      int64_t u_sl, int64_t o_sb, int64_t o_sl, int io_dtype) {
  if (B <= 0 || L <= 0 || W <= 0) return 0;
  const int64_t size = io_dtype == BASED_BF16 ? 2 : 4;
  return based::rglru_meet(u, u_sb, u_sl, out, o_sb, o_sl, B, L, W, size) ? (B * L * W * size + 3) / 4 : 0;
}

extern "C" BASED_API int based_rglru_prefill(const void* u, const void* y, const void* ra, const void* rb, const void* ri, const void* ib,
                                             const void* lam, float* work_a, float* work_x, float* work_agg, float* state, void* out,
                                             int64_t B, int64_t L, int64_t W, int64_t blocks, int64_t u_sb, int64_t u_sl, int64_t y_sb,
                                             int64_t y_sl, int64_t o_sb, int64_t o_sl, float c, int fresh, int io_dtype, void* stream) {
  using namespace based;
  BASED_REQUIRE(u && y && ra && rb && ri && ib && lam && work_agg && state && out, BASED_ERR_ARG, "rglru_prefill: null pointer argument");
  BASED_REQUIRE(B >= 0 && L >= 0 && W > 0 && blocks > 0, BASED_ERR_ARG, "rglru_prefill: bad sizes");
  BASED_REQUIRE(W % blocks == 0, BASED_ERR_SHAPE, "rglru_prefill: %ld channels do not divide into %ld blocks", (long)W, (long)blocks);
  BASED_REQUIRE(io_dtype == BASED_BF16 || io_dtype == BASED_F32, BASED_ERR_DTYPE, "rglru_prefill: bad dtype");
  const int64_t n = W / blocks, segs = (L + kSeg - 1) / kSeg, tiles = blocks * ((n + 63) / 64);
  BASED_REQUIRE(B < 65536 && segs < 65536 && tiles < 65536 && L < (1ll << 31), BASED_ERR_SHAPE, "rglru_prefill: grid too large");
  if (B == 0 || L == 0) return BASED_OK;
  const int64_t size = io_dtype == BASED_BF16 ? 2 : 4;
  const int64_t v = 16 / size;
  const auto whole = [&](const void* p, int64_t sb, int64_t sl) { return sl % v == 0 && (B == 1 || sb % v == 0) && aligned_to(p, 16); };
  const bool vec_u = n % v == 0 && whole(u, u_sb, u_sl) && aligned_to(ra, 16) && aligned_to(ri, 16);
  const bool vec_y = n % v == 0 && whole(y, y_sb, y_sl) && whole(out, o_sb, o_sl);
  // 64-bit words of every segment from the first aligned address on; the tickets, at most W of a sequence, in the last entry's 2 W values
  unsigned long long* agg = reinterpret_cast<unsigned long long*>(((uintptr_t)work_agg + 7) & ~(uintptr_t)7);
  const int step = (int)(2 * W / tiles);
  const RglruArgs a{u, y, ra, rb, ri, ib, lam, agg, reinterpret_cast<int*>(agg + B * segs * W), step, state, out, (int)B, (int)L, (int)W, (int)n, (int)segs, u_sb, u_sl, y_sb, y_sl,
                    o_sb, o_sl, c, fresh, vec_u, vec_y};
  // A workgroup reads channels of u that others' outputs would replace.
  const bool apart = rglru_meet(u, u_sb, u_sl, out, o_sb, o_sl, B, L, W, size);
  BASED_REQUIRE(work_x || !apart, BASED_ERR_ARG, "rglru_prefill: no work space for an output that shares memory with the input");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (io_dtype == BASED_BF16)
    launch_rglru_prefill<__bf16>(a, (int)tiles, apart ? reinterpret_cast<__bf16*>(work_x) : nullptr, s);
  else
    launch_rglru_prefill<float>(a, (int)tiles, apart ? work_x : nullptr, s);
  return check_launch("rglru_prefill");
}

extern "C" BASED_API int based_rglru_step(const void* x, const void* y, const void* conv_w, const void* conv_b, void* ring, const void* ra,
                                          const void* rb, const void* ri, const void* ib, const void* lam, float* state, void* out,
                                          const int32_t* pos, int64_t pos_host, int64_t B, int64_t W, int64_t blocks, int taps,
                                          int64_t x_sb, int64_t y_sb, int64_t o_sb, int64_t ring_sb, float c, int io_dtype,
                                          void* stream) {
  using namespace based;
  BASED_REQUIRE(x && y && conv_w && ring && ra && rb && ri && ib && lam && state && out, BASED_ERR_ARG, "rglru_step: null pointer argument");
  BASED_REQUIRE(B >= 0 && W > 0 && blocks > 0 && pos_host >= 0, BASED_ERR_ARG, "rglru_step: bad sizes");
  BASED_REQUIRE(W % blocks == 0, BASED_ERR_SHAPE, "rglru_step: %ld channels do not divide into %ld blocks", (long)W, (long)blocks);
  BASED_REQUIRE(taps >= 1 && taps <= 8, BASED_ERR_SHAPE, "rglru_step: %d taps (1 to 8)", taps);
  BASED_REQUIRE(io_dtype == BASED_BF16 || io_dtype == BASED_F32, BASED_ERR_DTYPE, "rglru_step: bad dtype");
  const int64_t n = W / blocks, tiles = blocks * ((n + 31) / 32), mt = (B + kLruRows - 1) / kLruRows;
  BASED_REQUIRE(n <= 2048, BASED_ERR_SHAPE, "rglru_step: blocks of %ld channels (at most 2048)", (long)n);
  BASED_REQUIRE(tiles < (1ll << 31) && mt < 65536, BASED_ERR_SHAPE, "rglru_step: grid too large");
  if (B == 0) return BASED_OK;
  const RglruStepArgs a{x,  y,  conv_w, conv_b, ring, ra, rb, ri, ib, lam, state, out, pos, (int)pos_host, (int)B, (int)W, (int)n, taps, x_sb,
                        y_sb, o_sb, ring_sb, c};
  const int v = io_dtype == BASED_BF16 ? 8 : 4;
  const bool vec = n % v == 0 && aligned_to(ra, 16) && aligned_to(ri, 16);
  const dim3 grid((unsigned)tiles, (unsigned)mt), block(256);
  const size_t bytes = (size_t)kLruRows * ((n + 3) & ~3) * sizeof(float);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (io_dtype == BASED_BF16) {
    if (vec)
      hipLaunchKernelGGL((rglru_step_kernel<__bf16, true>), grid, block, bytes, s, a);
    else
      hipLaunchKernelGGL((rglru_step_kernel<__bf16, false>), grid, block, bytes, s, a);
  } else {
    if (vec)
      hipLaunchKernelGGL((rglru_step_kernel<float, true>), grid, block, bytes, s, a);
    else
      hipLaunchKernelGGL((rglru_step_kernel<float, false>), grid, block, bytes, s, a);
  }
  return check_launch("rglru_step");
}
