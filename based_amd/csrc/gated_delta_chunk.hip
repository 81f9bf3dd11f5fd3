// Gated delta rule over prompts in chunks of 64 tokens, for gfx950: the recurrence of gated_delta.hip with the serial part made short.
//
// With the decays multiplied up inside a chunk, G_t = g_1 .. g_t, and A_ts = beta_t (k_t . k_s) G_t / G_s for s < t, T = (I + A)^-1,
// the values that enter the state are U = T (beta v) - T (beta G k) S0: an affine function of the state S0 in front of the chunk.
//   delta_chunk_prepare  everything that does not need S0, all chunks at once, a workgroup each: Uv = T (beta v), W = -T (beta G k) and
//                        P_ts = (q_t . k_s) G_t / G_s.  T by forward substitution in the four diagonal blocks of 16 (a power series
//                        would lose digits to cancellation), the others from them block by block.
//   delta_chunk_scan     walks the chunks: U = Uv + W S0, S1 = G_64 S0 + sum_s k_s (G_64 / G_s) u_s^T, and beside the chain
//                        o_t = G_t S0^T q_t + sum_{s <= t} P_ts u_s.  A workgroup of four wavefronts carries 16 value channels of a
//                        head; wavefront w has 16 tokens of every chunk and the state tiles w, w + 4, ..; S0 and U go round
//                        through LDS, two barriers per chunk.
// Products run on bf16 MFMA (16 x 16 x 32, sixteen times the rate of fp32), with 24 bits of every operand: a number of 32 bits enters as
// the sum of three of bf16 (each what the ones before leave, rounded; as in Henry, Tang and Heinecke, "Leveraging the bfloat16 Artificial
// Intelligence Datatype For Higher-Precision Computations"), and of the nine products of two such sums the six that reach 2^-24 of the result
// are taken.  Inputs of bf16 are one part as they are, scaled by row or behind the product, so their products are exact.  Sums are the matrix
// unit's, in 32 bits; the small products have an accumulator of their own.
// The parts hold what they should from 1e-32 to 3.39e38 in size.  Below, the last of them fall among the subnormals and are lost: values of 1e-33,
// 1e-35 and 1e-37 have errors of 3e-7, 3e-5 and 3e-3 (products on fp32 MFMA: 1.4e-7, 1.4e-7, 1.4e-6).  What bf16 rounds to infinity, and infinity
// itself, which leaves no number when it is taken off itself, makes every product that it enters no number.
//
// Operand layout of a lane (l16 = lane % 16, quad = lane / 16): row or column l16, contracted elements 8 quad .. 8 quad + 7; results: column
// l16, rows 4 quad + i.  What a result feeds next is contracted over its rows, so the rows of the tiles 2 n and 2 n + 1 are dealt out in turn:
// row 4 quad + i of tile 2 n + p is element 32 n + 8 quad + 4 p + i, and the four results of a lane in both tiles are one operand.  State
// tiles (channels), U (tokens) and the tiles of W and Uv that make it are dealt so; outputs are not.
//
// Products take 32 tokens at a time and hold zeros where a token does not see another.  What is no finite number stays out of the tiles of 16 tokens
// in front of its own all the same, as in blocks: the first 16 of such 32 are formed a second time without the others, and the outputs'
// wavefronts read zeros in their place (0 to 2 % of a call, 0.7 in the mean of 20 shapes).
//
// Against blocks of 16 (gated_delta_scan_kernel) a chain step takes in four times the tokens with two exchanges instead of one, and
// nothing but W S0 and k^T U stands in the chain.  4 sequences x 8 heads of 2048 tokens, d = 64, dv = 128, bf16: 161 us in blocks, 91 with
// fp32 products (41 of preparation, 55 of scan, 2.0 of whose 4.1 thousand cycles a chunk were products), now 67: preparation 24, bound by
// what it writes (92 MB at 3.8 TB/s), and scan 41, 3.1 thousand cycles a chunk: 2.0 of the chain itself, the rest waits for the chunk's 62 KB
// (without those loads 27 us, with all of them from L2 37).  d = 128: 226 -> 131 us (1 x 4096, 16 heads), fp32 232 -> 188.  Errors against
// 64 bits: 1.9e-7 -> 1.4e-7.
#include <type_traits>

#include "gated_delta.hpp"

namespace based {

constexpr int kDc = 64;        // tokens per chunk
constexpr int kDcRow = 72;     // a row of 64 in LDS, bf16: 16-byte pieces of 16 rows meet every bank once
// Products of a tile of 16 tokens with the tokens up to its end, by 32: a tile and a piece of 32 for each of six
__host__ __device__ constexpr int unit_t(int u) { return (int)(0x332210u >> (4 * u)) & 15; }
__host__ __device__ constexpr int unit_s(int u) { return (int)(0x101000u >> (4 * u)) & 15; }
__host__ __device__ constexpr int unit_of(int t) { return t < 2 ? t : 2 * t - 2; }

struct DeltaChunkArgs {
  const void* q;
  const void* k;
  const void* v;
  const void* a;
  const void* bt;
  const void* a_log;
  const void* dt_bias;
  float* state;  // (B, H, d, dvp)
  float* o;      // (B, L, H, dv)
  float* work;   // (B H, span, per)
  long per;
  int B, L, H, G, d, dv, dvp;
  int c0, span;  // the chunks of this launch
  long x_sb, x_sl;  // strides of q, k, v
  long g_sb, g_sl;  // strides of a, bt
  int fresh, v_vec;
};

// What a chunk leaves in the workspace, in operands of 1 KB (16 bytes a lane): W (token tile, 32 channels, part), q (token tile, 32
// channels; as they are, 8 of bf16 or of fp32 a lane), k transposed (channel tile, 32 tokens, part), P (unit, part), and Uv (value tile,
// token tile) in 32 bits; then, by token, fq G of the queries and what a token's value is multiplied by at the chunk's end, and G_64.  NP: parts of
// an element of q and k.
template <int RB, int NP> struct DcAt {
  static constexpr long kW = 0, kQ = (long)6 * RB * 256, kK = kQ + 2 * RB * (NP == 1 ? 1 : 2) * 256, kP = kK + 2 * RB * NP * 256, kUv = kP + 18 * 256;
};
__host__ __device__ inline long dc_vec_at(int rb, int np, int dv) { return ((long)(np == 1 ? 10 : 16) * rb + 18 + (long)((dv + 15) / 16) * 4) * 256; }
__host__ __device__ inline long dc_floats(int rb, int np, int dv) { return dc_vec_at(rb, np, dv) + 2 * kDc + 4; }

// exp of a sum of log decays held in 64 bits, which as a float would lose |x| 2^-24 of the result
__device__ __forceinline__ float exp_of(double x) {
  const float hi = (float)x, e = expf(hi);
  return __builtin_fmaf(e, (float)(x - (double)hi), e);
}

typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

// Two numbers as three packed pairs of bf16: rounded, what that left rounded, and what is left.
__device__ __forceinline__ void parts2(float a, float b, uint32_t (&o)[3]) {
#pragma unroll
  for (int n = 0; n < 3; ++n) {
    o[n] = pack_bf16(a, b);
    a -= __builtin_bit_cast(float, o[n] << 16);
    b -= __builtin_bit_cast(float, o[n] & 0xffff0000u);
  }
}
__device__ __forceinline__ void parts4(const f32x4& x, u32x2 (&o)[3]) {
  uint32_t a[3], b[3];
  parts2(x[0], x[1], a);
  parts2(x[2], x[3], b);
#pragma unroll
  for (int n = 0; n < 3; ++n) o[n] = u32x2{a[n], b[n]};
}
__device__ __forceinline__ void parts8(const f32x4& x, const f32x4& y, bf16x8 (&o)[3]) {
  u32x2 a[3], b[3];
  parts4(x, a);
  parts4(y, b);
#pragma unroll
  for (int n = 0; n < 3; ++n) o[n] = __builtin_bit_cast(bf16x8, u32x4{a[n][0], a[n][1], b[n][0], b[n][1]});
}

__device__ __forceinline__ f32x4 mfma_bf16(bf16x8 a, bf16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }

// x y added to sum[0], the products that are at most 2^-8 of it to sum[1]: NX and NY parts.
template <int NX, int NY> __device__ __forceinline__ void product(const bf16x8 (&x)[NX], const bf16x8 (&y)[NY], f32x4 (&sum)[2]) {
#pragma unroll
  for (int n = NX + NY - 2 < 2 ? NX + NY - 2 : 2; n > 0; --n)
#pragma unroll
    for (int i = 0; i < NX; ++i)
      if (n - i >= 0 && n - i < NY) sum[1] = mfma_bf16(x[i], y[n - i], sum[1]);
  sum[0] = mfma_bf16(x[0], y[0], sum[0]);
}

// The operand's first 16 of 32 contracted elements.
template <int N> __device__ __forceinline__ void first_half(const bf16x8 (&x)[N], bf16x8 (&y)[N], int quad) {
#pragma unroll
  for (int n = 0; n < N; ++n) y[n] = quad < 2 ? x[n] : bf16x8{};
}

// RB: 16-channel tiles of queries and keys.  LAY as for Four.  Rows go through LDS 64 channels at a time: a lane's operands lie in 16
// rows, and asked for one by one they cost 16 lines of cache per instruction.
template <typename T, int LAY, int RB>
__global__ __launch_bounds__(256, sizeof(T) == 2 ? (RB == 4 ? 4 : 3) : 2) void delta_chunk_prepare_kernel(const DeltaChunkArgs a) {
  constexpr int NP = sizeof(T) == 2 ? 1 : 3, KC = RB / 2, kSlabs = RB / 4;
  constexpr bool kAhead = LAY != 0 && sizeof(T) == 2;  // slabs of queries and keys asked for one ahead (others do not fit the registers)
  typedef DcAt<RB, NP> At;
  typedef __attribute__((ext_vector_type(4))) T t4;
  __shared__ __attribute__((aligned(16))) __bf16 s_x[2][NP][kDc][kDcRow];
  __shared__ __attribute__((aligned(16))) float s_a[kDc][kDc + 4];  // A, then T
  __shared__ double s_lc[kDc];
  // what is no finite number, by the wavefront that saw it: values in either slab, keys
  __shared__ __attribute__((aligned(16))) int s_odd[3][4];
  __shared__ __attribute__((aligned(16))) float s_beta[kDc], s_bg[kDc], s_fq[kDc], s_fk[kDc], s_e1k[kDc], s_e1q[kDc], s_e2[4 * kDc];
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, quad = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int bh = __builtin_amdgcn_readfirstlane(blockIdx.x / a.span), c = a.c0 + (int)(blockIdx.x - bh * a.span);
  const int b = __builtin_amdgcn_readfirstlane(bh / a.H), h = bh - b * a.H;
  const int hk = __builtin_amdgcn_readfirstlane(h / (a.H / a.G));
  const int t0 = c * kDc, left = a.L - t0 < kDc ? a.L - t0 : kDc, x_sl = (int)a.x_sl;
  const T* q = static_cast<const T*>(a.q) + b * a.x_sb + (long)t0 * a.x_sl + (long)hk * a.d;
  const T* k = static_cast<const T*>(a.k) + b * a.x_sb + (long)t0 * a.x_sl + (long)hk * a.d;
  const T* v = static_cast<const T*>(a.v) + b * a.x_sb + (long)t0 * a.x_sl + (long)h * a.dv;
  float* ws = a.work + (long)blockIdx.x * a.per;
  const int dealt = (l16 >> 2) * 8 + (l16 & 3);  // (+ 4 p: row l16 of tile p of a pair)
  const f32x4 none = {0.f, 0.f, 0.f, 0.f};

  // 64 channels from `e0` on of the chunk's rows: thread t has 4 channels of rows t / 16 + 16 j.  Rows past the last token are fetched
  // from it: gates of zero keep them out.
  const int piece = (tid & 15) * 4, row0 = tid >> 4;
  auto keep = [&](int buf, int row, const t4& x) {
    if constexpr (NP == 1) {
      *reinterpret_cast<t4*>(&s_x[buf][0][row][piece]) = x;
    } else {
      u32x2 p[3];
      parts4(f32x4{x[0], x[1], x[2], x[3]}, p);
#pragma unroll
      for (int n = 0; n < 3; ++n) *reinterpret_cast<u32x2*>(&s_x[buf][n][row][piece]) = p[n];
    }
  };
  auto fetch_slab = [&](Four<T, LAY> (&x)[4], const T* src, int e0, int lim) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int t = row0 + j * 16;
      x[j].load(src + (unsigned)((t < left ? t : left - 1) * x_sl), e0 + piece, lim);
    }
  };
  auto store_slab = [&](int buf, const Four<T, LAY> (&x)[4], int e0, int lim) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      t4 r = x[j].r;
#pragma unroll
      for (int i = 0; i < 4; ++i) r[i] = e0 + piece + i < lim ? r[i] : (T)0.0f;
      keep(buf, row0 + j * 16, r);
    }
  };
  // values: any alignment
  auto fetch_v = [&](t4 (&x)[4], int e0) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int t = row0 + j * 16;
      const T* row = v + (unsigned)((t < left ? t : left - 1) * x_sl);
      if (a.v_vec) {
        x[j] = *reinterpret_cast<const t4*>(row + (e0 + piece < a.dv ? e0 + piece : 0));
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) x[j][i] = row[e0 + piece + i < a.dv ? e0 + piece + i : 0];
      }
    }
  };
  auto store_v = [&](int buf, const t4 (&x)[4], int e0) {
    float zero = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      t4 r = x[j];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        r[i] = e0 + piece + i < a.dv ? r[i] : (T)0.0f;
        zero = __builtin_fmaf(to_f32(r[i]), 0.f, zero);
      }
      keep(buf, row0 + j * 16, r);
    }
    const bool odd = __any(!(zero == 0.f));
    if (lane == 0) s_odd[buf][wave] = odd;
  };
  auto any_of = [&](const int (&x)[4]) {
    return __builtin_amdgcn_readfirstlane(x[0] | x[1] | x[2] | x[3]) != 0;
  };
  auto row_operand = [&](int buf, int row, int e, bf16x8 (&x)[NP]) {
#pragma unroll
    for (int n = 0; n < NP; ++n) x[n] = *reinterpret_cast<const bf16x8*>(&s_x[buf][n][row][e]);
  };
  // tokens 32 ks + 8 quad .. of channel l16 of four pieces of 4 channels, EACH channels apart, from `e` on: a transposing read gives lane l16
  // element l16 of the four rows whose 8 bytes each its group of 16 lanes names (24.6 -> 23.9 us)
  auto column_operand = [&](int buf, int ks, int e, int each, bf16x8 (&x)[NP]) {
#pragma unroll
    for (int n = 0; n < NP; ++n) {
      const __bf16* at = &s_x[buf][n][ks * 32 + quad * 8 + (l16 >> 2)][e + (l16 & 3) * each];
      x[n] = __builtin_shufflevector(read_transposed(at), read_transposed(at + 4 * kDcRow), 0, 1, 2, 3, 4, 5, 6, 7);
    }
  };
  auto put = [&](long at, const bf16x8& x) { *reinterpret_cast<bf16x8*>(ws + at * 256 + lane * 4) = x; };
  // Sums over the tokens that a tile of (dealt) tokens sees, 32 at a time: `one` adds 32 of them, its own behind those in front.  Zeros stand for the
  // tokens that a token does not see, and zero times what is no finite number is none: where there is one (ODD), the first 16 of the 32 (`first`:
  // this lane's results are theirs) are formed without the others, by a second pass over what the first has left.
  auto tokens_product = [&](auto odd, int m, bool first, const auto& one) {
    f32x4 sum[2] = {none, none};
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
      if (ks <= m) one(ks, false, sum);
    f32x4 out = sum[0] + sum[1];
    if constexpr (decltype(odd)::value) {
      f32x4 less[2] = {none, none};
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
        if (ks <= m) one(ks, ks == m, less);
      if (first) out = less[0] + less[1];
    }
    return out;
  };

  Four<T, LAY> kr[4], qr[4];
  fetch_slab(kr, k, 0, a.d);
  fetch_slab(qr, q, 0, a.d);
  const long gate = b * a.g_sb + (long)(t0 + (lane < left ? lane : left - 1)) * a.g_sl + h;
  const T gate_a = static_cast<const T*>(a.a)[gate], gate_b = static_cast<const T*>(a.bt)[gate];
  const T a_log = static_cast<const T*>(a.a_log)[h], dt_bias = static_cast<const T*>(a.dt_bias)[h];
  // Products of keys with keys and with queries, transposed (column = token t, rows = the tokens s of a pair of tiles): four of the twelve
  // units for each of wavefronts 1 to 3, while wavefront 0 works the decays out.
  constexpr int kMine = 4;
  f32x4 acc[kMine][2][2];
#pragma unroll
  for (int j = 0; j < kMine; ++j)
#pragma unroll
    for (int p = 0; p < 2; ++p) acc[j][p][0] = acc[j][p][1] = none;
  double sq = 0.0, sk = 0.0;  // (the squares' sums scale whole rows: an error in them does not average out)
#pragma unroll 1
  for (int sl = 0; sl < kSlabs; ++sl) {
    if (sl > 0) {
      if (!kAhead) {
        fetch_slab(kr, k, sl * 64, a.d);
        fetch_slab(qr, q, sl * 64, a.d);
      }
      __syncthreads();
    }
    store_slab(0, kr, sl * 64, a.d);
    store_slab(1, qr, sl * 64, a.d);
    if (kAhead && sl + 1 < kSlabs) {
      fetch_slab(kr, k, (sl + 1) * 64, a.d);
      fetch_slab(qr, q, (sl + 1) * 64, a.d);
    }
    __syncthreads();
    if (wave > 0) {
#pragma unroll
      for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int j = 0; j < kMine; ++j) {
          const int u = (wave - 1) * kMine + j, unit = u < 6 ? u : u - 6;
          bf16x8 y[NP];
          row_operand(u < 6 ? 0 : 1, unit_t(unit) * 16 + l16, r * 32 + quad * 8, y);
#pragma unroll
          for (int p = 0; p < 2; ++p) {
            bf16x8 x[NP];
            row_operand(0, unit_s(unit) * 32 + dealt + 4 * p, r * 32 + quad * 8, x);
            product(x, y, acc[j][p]);
          }
        }
    } else if (sl == 0) {
      // log G in 64 bits: behind a token that forgets nearly everything the differences of these sums still have to carry the
      // ordinary decays
      s_beta[lane] = lane < left ? 1.0f / (1.0f + expf(-to_f32(gate_b))) : 0.f;
      const double z = (double)to_f32(gate_a) + (double)to_f32(dt_bias);
      const double lg = -exp((double)to_f32(a_log)) * (log1p(exp(-fabs(z))) + fmax(z, 0.0));
      double lc = lane < left ? fmax(lg, -200.0) : 0.0;  // exp(-200) is zero in fp32
#pragma unroll
      for (int m = 1; m < 64; m <<= 1) {
        const double up = __shfl_up(lc, m, 64);
        if (lane >= m) lc += up;
      }
      s_lc[lane] = lc;
    }
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      bf16x8 x[2][NP];
#pragma unroll
      for (int n = 0; n < 2; ++n) row_operand(n, wave * 16 + l16, r * 32 + quad * 8, x[n]);
      float f[2][8];
#pragma unroll
      for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int j = 0; j < 8; ++j) f[n][j] = NP == 1 ? to_f32(x[n][0][j]) : to_f32(x[n][0][j]) + (to_f32(x[n][NP > 1][j]) + to_f32(x[n][NP - 1][j]));
#pragma unroll
      for (int j = 0; j < 8; j += 4) {
        sk += (double)(f[0][j] * f[0][j] + f[0][j + 1] * f[0][j + 1]) + (double)(f[0][j + 2] * f[0][j + 2] + f[0][j + 3] * f[0][j + 3]);
        sq += (double)(f[1][j] * f[1][j] + f[1][j + 1] * f[1][j + 1]) + (double)(f[1][j + 2] * f[1][j + 2] + f[1][j + 3] * f[1][j + 3]);
      }
      const long at = At::kQ / 256 + (wave * KC + sl * 2 + r) * (NP == 1 ? 1 : 2);
      if constexpr (NP == 1) {
        put(at, x[1][0]);
      } else {
#pragma unroll
        for (int n = 0; n < 2; ++n)
          *reinterpret_cast<f32x4*>(ws + (at + n) * 256 + lane * 4) =
              f32x4{f[1][4 * n], f[1][4 * n + 1], f[1][4 * n + 2], f[1][4 * n + 3]};
      }
    }
  }
  // the next slab: the first of the keys again, or, where that one is still in LDS, the first of the values
  t4 vr[4];
  if constexpr (kSlabs > 1)
    fetch_slab(kr, k, 0, a.d);
  else
    fetch_v(vr, 0);
  sq += __shfl_xor(sq, 16, 64), sk += __shfl_xor(sk, 16, 64);
  sq += __shfl_xor(sq, 32, 64), sk += __shfl_xor(sk, 32, 64);
  if (quad == 0) {
    const int t = wave * 16 + l16;
    // (times d only in 64 bits: queries of 1e19 and more have no such product in 32)
    s_fq[t] = t < left ? (float)(1.0 / sqrt((sq + (double)kUnitEps) * (double)a.d)) : 0.f;
    s_fk[t] = t < left ? 1.0f / sqrtf((float)(sk + (double)kUnitEps)) : 0.f;
  }
  const bool odd_k = __any(!((float)sk < INFINITY));
  if (lane == 0) s_odd[2][wave] = odd_k;
  __syncthreads();
  // Quotients of decays as products of two, over the token in front of the later tile: a few exponentials a token in place of one for
  // every pair.  Between tiles both are at most one; inside a tile the second is at least one, and is not used where the tile forgets
  // too much for it.
  {
    const double lc = s_lc[lane];
    const float fk = s_fk[lane];
    const int front = (lane & ~15) - 1;
    const double lc_front = front < 0 ? 0.0 : s_lc[front < 0 ? 0 : front];
    if (wave == 0) {
      const double end = s_lc[kDc - 1];
      const float G = exp_of(lc);
      float* vec = ws + dc_vec_at(RB, NP, a.dv);
      s_bg[lane] = -s_beta[lane] * G * fk;
      vec[lane] = s_fq[lane] * G;
      vec[kDc + lane] = fk * exp_of(end - lc < 0.0 ? end - lc : 0.0);
      if (lane == 63) vec[2 * kDc] = G;
      s_e2[lane] = fk * exp_of(lc_front - lc);
    } else {
      const double ref = s_lc[wave * 16 - 1];
      s_e2[wave * kDc + lane] = fk * exp_of(ref - lc < 0.0 ? ref - lc : 0.0);
      if (wave == 1) s_e1k[lane] = s_beta[lane] * fk * exp_of(lc - lc_front);
      if (wave == 2) s_e1q[lane] = s_fq[lane] * exp_of(lc - lc_front);
    }
  }
  __syncthreads();
  if (wave > 0) {
#pragma unroll
    for (int j = 0; j < kMine; ++j) {
      const int u = (wave - 1) * kMine + j;
      const bool keys = u < 6;
      const int unit = keys ? u : u - 6, tt = unit_t(unit), t = tt * 16 + l16, s0 = unit_s(unit) * 32 + quad * 8, ts = s0 >> 4;
      const float e1 = keys ? s_e1k[t] : s_e1q[t];
      const float* e2 = &s_e2[(ts == tt ? 0 : tt) * kDc + s0];
      f32x4 out[2];
#pragma unroll
      for (int p = 0; p < 2; ++p) out[p] = acc[j][p][0] + acc[j][p][1];
      f32x4 f[2] = {*reinterpret_cast<const f32x4*>(e2) * e1, *reinterpret_cast<const f32x4*>(e2 + 4) * e1};
      const double fall = (tt > 0 ? s_lc[tt > 0 ? tt * 16 - 1 : 0] : 0.0) - s_lc[tt * 16 + 15];
      if (fall > 60.0 && ts == tt) {
        const double lc_t = s_lc[t];
        const float ft = keys ? s_fk[t] * s_beta[t] : s_fq[t];
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const double diff = lc_t - s_lc[s0 + 4 * p + i];
            f[p][i] = ft * s_fk[s0 + 4 * p + i] * exp_of(diff < 0.0 ? diff : 0.0);
          }
      }
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int s = s0 + 4 * p + i;
          out[p][i] = s < t || (s == t && !keys) ? out[p][i] * f[p][i] : 0.f;
        }
      if (keys) {
        *reinterpret_cast<f32x4*>(&s_a[t][s0]) = out[0];
        *reinterpret_cast<f32x4*>(&s_a[t][s0 + 4]) = out[1];
      } else {
        bf16x8 x[3];
        parts8(out[0], out[1], x);
#pragma unroll
        for (int n = 0; n < 3; ++n) put(At::kP / 256 + unit * 3 + n, x[n]);
      }
    }
  }
  __syncthreads();
  // T, in the place of A: the diagonal blocks, one per wavefront; column l16: x_t = [t = l16] - sum_{s<t} A_ts x_s
  {
    const int at = wave * 16;
    float x[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      float sum[2] = {t == l16 ? 1.f : 0.f, 0.f};
#pragma unroll
      for (int s4 = 0; s4 < t; s4 += 4) {
        const f32x4 r = *reinterpret_cast<const f32x4*>(&s_a[at + t][at + s4]);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (s4 + j < t) sum[j & 1] = __builtin_fmaf(-r[j], x[s4 + j], sum[j & 1]);
      }
      x[t] = sum[0] + sum[1];
    }
    if (quad == 0) {
#pragma unroll
      for (int t = 0; t < 16; ++t) s_a[at + t][at + l16] = x[t];
    }
  }
  __syncthreads();
  // the blocks below them, a column of blocks per wavefront: T_ij = -T_ii sum_{j <= k < i} A_ik T_kj
  f32x4 col[4] = {none, none, none, none};
  if (wave < 3) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (i == wave) {
#pragma unroll
        for (int x = 0; x < 4; ++x) col[i][x] = s_a[i * 16 + quad * 4 + x][i * 16 + l16];
      } else if (i > wave) {
        f32x4 sum[2] = {none, none};
#pragma unroll
        for (int kb = 0; kb < i; ++kb)
          if (kb >= wave) {
            const f32x4 row = *reinterpret_cast<const f32x4*>(&s_a[i * 16 + l16][kb * 16 + quad * 4]);
#pragma unroll
            for (int x = 0; x < 4; ++x) sum[x & 1] = mfma_f32(row[x], col[kb][x], sum[x & 1]);
          }
        const f32x4 row = *reinterpret_cast<const f32x4*>(&s_a[i * 16 + l16][i * 16 + quad * 4]);
        const f32x4 y = sum[0] + sum[1];
        f32x4 res[2] = {none, none};
#pragma unroll
        for (int x = 0; x < 4; ++x) res[x & 1] = mfma_f32(row[x], y[x], res[x & 1]);
        col[i] = -(res[0] + res[1]);
      }
    }
  }
  if constexpr (kSlabs > 1)
    store_slab(0, kr, 0, a.d);
  else
    store_v(1, vr, 0);
  __syncthreads();  // everybody has read A
  if (wave < 3) {
#pragma unroll
    for (int i = 1; i < 4; ++i)
      if (i > wave) {
#pragma unroll
        for (int x = 0; x < 4; ++x) s_a[i * 16 + quad * 4 + x][wave * 16 + l16] = col[i][x];
      }
  }
  __syncthreads();
  // Every wavefront has two of the four (dealt) token tiles, one of the first 32 tokens and one of the others, and half of the channels.
  const int half = wave & 1, m_of[2] = {wave >> 1, 3 - (wave >> 1)};
  bf16x8 tm[3][3];  // T with its columns scaled: tokens 0 .. 31 for the first tile, then both halves for the second
  auto scaled = [&](const float* by) {
#pragma unroll
    for (int n = 0; n < 3; ++n) {
      const int m = m_of[n > 0], ks = n == 2, t = (m >> 1) * 32 + dealt + 4 * (m & 1), s0 = ks * 32 + quad * 8;
      const f32x4* row = reinterpret_cast<const f32x4*>(&s_a[t][s0]);
      const f32x4* f = reinterpret_cast<const f32x4*>(by + s0);
      const bool unseen = n != 1 && l16 < 8 && quad >= 2;  // (zero, whatever it is scaled by)
      parts8(row[0] * (unseen ? none : f[0]), row[1] * (unseen ? none : f[1]), tm[n]);
    }
  };
  // W (row = token, contracted over channels in the scan: here transposed) and the keys of 32 channels of a slab
  auto keys_tile = [&](auto odd, int buf, int kc) {
    bf16x8 kx[2][2][NP];
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) column_operand(buf, ks, half * 32 + 4 * p, 8, kx[p][ks]);
    const int mine = wave >> 1;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int n = 0; n < NP; ++n) put(At::kK / 256 + ((kc * 2 + mine) * 2 + ks) * NP + n, mine ? kx[1][ks][n] : kx[0][ks][n]);
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      f32x4 out[2];
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        out[p] = tokens_product(odd, m, l16 < 8, [&](int ks, bool half_only, f32x4 (&sum)[2]) {
          if (!half_only) return product(kx[p][ks], tm[m + ks], sum);
          bf16x8 x[NP];
          first_half(kx[p][ks], x, quad);
          product(x, tm[m + ks], sum);
        });
      }
      bf16x8 x[3];
      parts8(out[0], out[1], x);
#pragma unroll
      for (int n = 0; n < 3; ++n) put(At::kW / 256 + (m_of[m] * KC + kc) * 3 + n, x[n]);
    }
  };
  // Uv (rows = tokens, column = channel: the scan's accumulator) of two of a slab's value tiles
  auto values_tile = [&](auto odd, int buf, int tile0) {
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      const int tile = tile0 + half * 2 + x;
      if (tile * 16 >= a.dv) break;  // (uniform)
      bf16x8 vx[2][NP];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) column_operand(buf, ks, (half * 2 + x) * 16, 4, vx[ks]);
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const f32x4 uv = tokens_product(odd, m, quad < 2, [&](int ks, bool half_only, f32x4 (&sum)[2]) {
          if (!half_only) return product(tm[m + ks], vx[ks], sum);
          bf16x8 x[NP];
          first_half(vx[ks], x, quad);
          product(tm[m + ks], x, sum);
        });
        *reinterpret_cast<f32x4*>(ws + At::kUv + ((long)tile * 4 + m_of[m]) * 256 + lane * 4) = uv;
      }
    }
  };
  scaled(s_bg);
  const bool odd_keys = any_of(s_odd[2]);
  int buf = 0;  // the slab in LDS; the next one goes into the other buffer, which everybody has left behind at the barrier before
  if constexpr (kSlabs > 1) {
#pragma unroll 1
    for (int sl = 0; sl < kSlabs; ++sl) {
      auto fetch = [&] {
        if (sl + 1 < kSlabs)
          fetch_slab(kr, k, (sl + 1) * 64, a.d);
        else
          fetch_v(vr, 0);
      };
      if (kAhead) fetch();
      keys_tile(std::false_type(), buf, sl * 2 + half);
      if (odd_keys) keys_tile(std::true_type(), buf, sl * 2 + half);
      if (!kAhead) fetch();
      buf ^= 1;
      if (sl + 1 < kSlabs)
        store_slab(buf, kr, (sl + 1) * 64, a.d);
      else
        store_v(buf, vr, 0);
      __syncthreads();
    }
  } else {
    keys_tile(std::false_type(), 0, half);
    if (odd_keys) keys_tile(std::true_type(), 0, half);
    buf = 1;
  }
  scaled(s_beta);
#pragma unroll 1
  for (int e0 = 0; e0 < a.dv; e0 += 64) {
    const bool more = e0 + 64 < a.dv;
    if (more) fetch_v(vr, e0 + 64);
    values_tile(std::false_type(), buf, e0 / 16);
    if (any_of(s_odd[buf])) values_tile(std::true_type(), buf, e0 / 16);
    if (!more) break;
    buf ^= 1;
    if (kSlabs == 1 && e0 == 0) __syncthreads();  // (a slower wavefront may still read the keys there)
    store_v(buf, vr, e0 + 64);
    __syncthreads();
  }
}

// Whether a workgroup of the scan has more registers than two of them find on a compute unit.
__host__ __device__ constexpr bool dc_lone(int rb) { return rb == 8; }

// A workgroup to a head's 16 value channels.  Wavefronts 0 .. 3 carry the state, 4 .. 7 form the outputs, a chunk behind with the
// products of P: four wavefronts that do both take 44 us for 41 above and 118 for 105 with keys of 128.  Two barriers a chunk:
//   state there   state: U = Uv + W S0, its scaled parts to LDS.  outputs: parts of S0 and of the U before are read, q S0 and P U formed
//   U there       state: S1 = G S0 + k U, its parts to LDS, and those of U.  outputs: stored, the next operands asked for
template <int RB, int NP>
__global__ __launch_bounds__(512, dc_lone(RB) ? 2 : 4) void delta_chunk_scan_kernel(const DeltaChunkArgs a) {
  static_assert(RB % 4 == 0, "every wavefront has state tiles");
  constexpr int RBW = RB / 4, KC = RB / 2;
  typedef DcAt<RB, NP> At;
  // operands of three parts: the state by 32 channels; U by 32 tokens, as the outputs take it and scaled to the chunk's end
  __shared__ __attribute__((aligned(16))) bf16x8 s_s[KC][3][64], s_u[2][3][64], s_us[2][3][64], s_none[3][64];
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, quad = lane >> 4;
  const int role = __builtin_amdgcn_readfirstlane(tid >> 8), wave = __builtin_amdgcn_readfirstlane((tid >> 6) & 3);
  // The workgroups of a head run on one die, whose L2 then has its chunks once.  Workgroup i is number i / 8 of die i % 8: heads in whole eights lie
  // side by side, others one behind the other, tile by tile, a run of them to a die (spread over all dies 61 heads of 40 x 160, 4,677 tokens took 676
  // us for 413, and the blocks 499; runs for whole eights as well: 24 heads of 24 x 256, 4,096 tokens 200 for 184).
  int head = (int)blockIdx.x, ct = (int)blockIdx.y;
  if (gridDim.x % 8 != 0) {
    const int i = ct * (int)gridDim.x + head, n = (int)(gridDim.x * gridDim.y), die = i & 7, more = n & 7;
    const int at = die * (n >> 3) + (die < more ? die : more) + (i >> 3);
    head = __builtin_amdgcn_readfirstlane(at / (int)gridDim.y), ct = __builtin_amdgcn_readfirstlane(at - head * (int)gridDim.y);
  }
  const int bh = head, b = __builtin_amdgcn_readfirstlane(bh / a.H), h = bh - b * a.H, col = ct * 16 + l16;
  const bool col_in = col < a.dv;
  const char* ws = reinterpret_cast<const char*>(a.work + (long)bh * a.span * a.per);
  const long per = a.per * 4, vec_at = dc_vec_at(RB, NP, a.dv) * 4;
  const f32x4 none = {0.f, 0.f, 0.f, 0.f};
  const unsigned at_lane = (unsigned)lane * 16u;
  auto operand_at = [&](const char* p, int n) { return *reinterpret_cast<const bf16x8*>(p + n * 1024 + at_lane); };

  if (role == 0) {
    __builtin_amdgcn_s_setprio(2);
    const int dealt = (wave >> 1) * 32 + quad * 8 + (wave & 1) * 4;  // first of the tokens (channels + 64 x) of this lane's four rows
    // half of a lane's operand, where this wavefront's tile of a pair goes
    auto put = [&](bf16x8 (&to)[3][64], const f32x4& x) {
      u32x2 p[3];
      parts4(x, p);
#pragma unroll
      for (int n = 0; n < 3; ++n) reinterpret_cast<u32x2*>(&to[n][lane])[wave & 1] = p[n];
    };
    float* st = a.state + (long)bh * a.d * a.dvp + (col_in ? col : 0);
    f32x4 S[RBW];  // tiles wave + 4 x
#pragma unroll
    for (int x = 0; x < RBW; ++x) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = x * 64 + dealt + i;
        const bool in = !a.fresh && col_in && row < a.d;
        S[x][i] = in ? st[(long)row * a.dvp] : 0.f;
      }
      put(s_s[(wave >> 1) + 2 * x], S[x]);
    }
    // What a chunk needs from memory: a set of registers, each part asked for anew as soon as its last use has been issued.
    bf16x8 w[KC][3], kt[RBW][2][NP];
    f32x4 uv, tail;
    float last;
    const char *pw = ws + At::kW * 4 + wave * KC * 3072, *pu = ws + At::kUv * 4 + (ct * 4 + wave) * 1024;
    const char *pk = ws + At::kK * 4 + wave * 2 * NP * 1024, *pv = ws + vec_at;
    auto fetch_w = [&] {
#pragma unroll
      for (int r = 0; r < KC; ++r)
#pragma unroll
        for (int j = 0; j < 3; ++j) w[r][j] = operand_at(pw, r * 3 + j);
      uv = *reinterpret_cast<const f32x4*>(pu + at_lane);
      tail = *reinterpret_cast<const f32x4*>(pv + kDc * 4 + (unsigned)dealt * 4u);
    };
    auto fetch_k = [&] {
#pragma unroll
      for (int x = 0; x < RBW; ++x)
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
          for (int j = 0; j < NP; ++j) kt[x][s][j] = operand_at(pk, (x * 8 + s) * NP + j);
      last = *reinterpret_cast<const float*>(pv + kDc * 8);
    };
    fetch_w();
    __builtin_amdgcn_sched_barrier(0);
    fetch_k();
    for (int n = 0; n < a.span; ++n) {
      const long step = n + 1 < a.span ? per : 0;
      pw += step, pu += step, pk += step, pv += step;
      lds_barrier();  // the state is there
      bf16x8 s0[KC][3];
#pragma unroll
      for (int r = 0; r < KC; ++r)
#pragma unroll
        for (int j = 0; j < 3; ++j) s0[r][j] = s_s[r][j][lane];
      // (what is added to a sum that starts from the large term loses its last digits sixteen times: added at the end, once)
      f32x4 u[2][2] = {{none, none}, {none, none}};
#pragma unroll
      for (int r = 0; r < KC; ++r) product(w[r], s0[r], u[r & 1]);
      const f32x4 un = uv + ((u[0][1] + u[1][1]) + (u[0][0] + u[1][0]));
      put(s_us[wave >> 1], un * tail);
      __builtin_amdgcn_sched_barrier(0);
      fetch_w();
      __builtin_amdgcn_sched_barrier(0);
      lds_barrier();  // U is there
      bf16x8 us[2][3];
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int j = 0; j < 3; ++j) us[s][j] = s_us[s][j][lane];
      put(s_u[wave >> 1], un);
#pragma unroll
      for (int x = 0; x < RBW; ++x) {
        f32x4 sum[2][2] = {{none, none}, {none, none}};
#pragma unroll
        for (int s = 0; s < 2; ++s) product(kt[x][s], us[s], sum[s]);
        S[x] = S[x] * last + ((sum[0][1] + sum[1][1]) + (sum[0][0] + sum[1][0]));
        put(s_s[(wave >> 1) + 2 * x], S[x]);
      }
      __builtin_amdgcn_sched_barrier(0);
      fetch_k();
      __builtin_amdgcn_sched_barrier(0);
    }
    lds_barrier();  // the last U is there
#pragma unroll
    for (int x = 0; x < RBW; ++x)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = x * 64 + dealt + i;
        if (col_in && row < a.d) st[(long)row * a.dvp] = S[x][i];
      }
  } else {
    const int o_sl = a.H * a.dv * 4;  // bytes
    char* o = reinterpret_cast<char*>(a.o + ((long)b * a.L * a.H + h) * a.dv) + (long)a.c0 * kDc * o_sl;
    const unsigned mine = (unsigned)((wave * 16 + quad * 4) * o_sl + (col_in ? col : 0) * 4);
    const int pieces = wave >> 1;  // of 32 tokens in front of the last one that the wavefront's own reach
    constexpr int NQ = NP == 1 ? 1 : 2;  // (queries of fp32 are taken apart here: their parts would be half as much again to write and to read)
    bf16x8 p[2][3], qx[KC][NQ];
    f32x4 gq, on = none;  // on: queries' product with the state of the chunk before
    const char *pq = ws + At::kQ * 4 + wave * KC * NQ * 1024, *pp = ws + At::kP * 4 + unit_of(wave) * 3072, *pv = ws + vec_at;
    auto fetch_q = [&] {
#pragma unroll
      for (int r = 0; r < KC; ++r)
#pragma unroll
        for (int j = 0; j < NQ; ++j) qx[r][j] = operand_at(pq, r * NQ + j);
      gq = *reinterpret_cast<const f32x4*>(pv + (unsigned)(wave * 16 + quad * 4) * 4u);
    };
    auto fetch_p = [&] {
#pragma unroll
      for (int s = 0; s < 2; ++s)
        if (s <= pieces) {  // (uniform)
#pragma unroll
          for (int j = 0; j < 3; ++j) p[s][j] = operand_at(pp, s * 3 + j);
        }
    };
    bf16x8 us[2][3];
    // (zeros for those tokens of the last piece that the wavefront's own do not see: what is there may be no finite number)
#pragma unroll
    for (int j = 0; j < 3; ++j) s_none[j][lane] = bf16x8{};
    const bool behind = (wave & 1) == 0 && quad >= 2;
    const bf16x8* from[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) from[s] = behind && s == pieces ? &s_none[0][lane] : &s_u[s][0][lane];
    auto read_u = [&] {
#pragma unroll
      for (int s = 0; s < 2; ++s)
        if (s <= pieces) {  // (uniform)
#pragma unroll
          for (int j = 0; j < 3; ++j) us[s][j] = from[s][j * 64];
        }
    };
    // P U behind `on`
    auto finish = [&] {
      f32x4 sum[2] = {on, none};
      product(p[0], us[0], sum);
      if (pieces > 0) product(p[1], us[1], sum);  // (uniform)
      return sum[0] + sum[1];
    };
    auto store = [&](int n, const f32x4& out) {
      const int left = a.L - (a.c0 + n) * kDc;
      char* ob = o + (long)n * kDc * o_sl;
      if (col_in) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (left >= kDc || wave * 16 + quad * 4 + i < left) *reinterpret_cast<float*>(ob + (long)i * o_sl + mine) = out[i];
      }
    };
    // The workgroups of a head, which share an L2 where the heads are a multiple of the dies, ask together for every line of the chunk after
    // next, a word each: what the registers hold ahead is less than the way from memory takes (fp32, d = 128: 243 -> 206 us).
    const int lines = (int)((per + 127) / 128), first = (ct * 4 + wave) * 64 + lane, every = (int)gridDim.y * 256;
    unsigned seen = 0;
    auto touch = [&](int n) {
      if (n >= a.span) return;  // (uniform)
      const char* chunk = ws + (long)n * per;
      for (int line = first; line < lines; line += every) seen = *reinterpret_cast<const unsigned*>(chunk + (unsigned)line * 128u);
    };
    fetch_q();
    for (int n = 0; n < a.span; ++n) {
      asm volatile("" ::"v"(seen));
      touch(n + 2);
      lds_barrier();  // the state is there, and the U of the chunk before
      bf16x8 s0[KC][3];
#pragma unroll
      for (int r = 0; r < KC; ++r)
#pragma unroll
        for (int j = 0; j < 3; ++j) s0[r][j] = s_s[r][j][lane];
      if (n > 0) read_u();
      f32x4 oo[2] = {none, none};
#pragma unroll
      for (int r = 0; r < KC; ++r) {
        bf16x8 x[NP];
        if constexpr (NP == 1)
          x[0] = qx[r][0];
        else
          parts8(__builtin_bit_cast(f32x4, qx[r][0]), __builtin_bit_cast(f32x4, qx[r][1]), x);
        product(x, s0[r], oo);
      }
      __builtin_amdgcn_sched_barrier(0);
      lds_barrier();  // (the state and U may be written)
      if (n > 0) store(n - 1, finish());
      on = gq * (oo[0] + oo[1]);
      __builtin_amdgcn_sched_barrier(0);
      fetch_p();
      pp += per, pq += n + 1 < a.span ? per : 0, pv += n + 1 < a.span ? per : 0;
      fetch_q();
      __builtin_amdgcn_sched_barrier(0);
    }
    lds_barrier();  // the last U is there
    read_u();
    store(a.span - 1, finish());
  }
}

// Workspace: the chunks of one launch pair.  Long prompts go through it in spans of chunks, the state carried on in between.
// 192 MB, which the last-level cache (256 MB) holds between the two launches beside what they read and write otherwise: work spaces of 224 to 256 MB
// in one launch pair, 1.00; in two of half as much, 0.82 to 0.86 of the time; more pairs of up to 160, 192 and 224 MB in place of 256, in 635 long
// prompts of bf16 0.92, 0.93 and 0.96; 160 MB cost 2 to 3 % where 192 take the call in one pair.
constexpr int64_t kDcWorkFloats = 48ll << 20;

// In bf16 chunks take 0.57 to 0.83 of the times that the rule for fp32, below, was made of.  Three things make them the slower form.  A step of the
// blocks costs by 16 channels of keys, chunks fill 64 or 128: few channels (up to 16, 32, 48), and 65 to 112, whose blocks leave out what chunks
// multiply.  Two workgroups of the scan fit a compute unit (one above 64 channels): beyond 512 to 1,024 of them they take turns, each reads all that
// is formed ahead, and every head adds preparation.  And short prompts pay for two launches.  us, blocks of 16 against chunks, heads, d x dv (in
// 5,658 shapes 0.24 to 1.04 of the blocks' time where the rule takes them, 0.57 in the mean; in 1,500 of any size at most 1.03):
//   24, 34 x 332: L = 700: 160, 45.  32, 64 x 512: L = 1024: 158, 96.  64, 128 x 256: L = 256: 85, 61; L = 1024: 281, 175.
//   Up to 16 channels: 64, 16 x 64: L = 320: 30, 30.  64, 16 x 128: L = 512: 43, 41; L = 1024: 73, 62; L = 2048: 130, 139.  48, 16 x 256: L = 512:
//   44, 55.
//   4, 16 x 512: L = 256: 24, 27; L = 320: 28, 28.
//   Up to 32: 64, 32 x 128: L = 256: 30, 32; L = 320: 37, 35; L = 1024: 90, 63.  48, 32 x 256: L = 1024: 120, 85; L = 4096: 423, 387.  64, 32 x 256:
//   L = 1024: 96, 100.
//   Up to 48: 64, 48 x 256: L = 1024: 120, 102; L = 4096: 411, 493.  80, 48 x 128: L = 2048: 224, 206.  96, 48 x 128: L = 4096: 439, 486.
//   Up to 64: 120, 64 x 128: L = 2048: 310, 309.  128, 64 x 128: L = 512: 86, 73; L = 1024: 158, 172.
//   Up to 96: 80, 96 x 64: L = 4096: 485, 438.  112, 96 x 64: L = 4096: 515, 571.  112, 96 x 16: L = 4096: 530, 392.
//   Up to 112: 112, 112 x 64: L = 4096: 662, 592.  128, 112 x 64: L = 1024: 179, 169; L = 4096: 674, 737.
//   Up to 128: 128, 128 x 128: L = 4096: 1,161, 963.  128, 128 x 32: L = 4096: 479, 496.
//   256 heads: 64 x 64: L = 256: 56, 56; L = 1024: 177, 249.  128 x 128: L = 256: 170, 183.
static bool dc_faster_bf16(int64_t heads, int64_t L, int64_t D, int64_t DV) {
  const int64_t tiles = (DV + 15) / 16, wgs = heads * tiles;
  if (heads > 128 || wgs > 1024 || D > 128 || L < BASED_DELTA_CHUNKS_MIN) return false;
  if (D > 112) return true;
  if (D > 96) return heads <= 112 || L <= 1024;
  if (D > 64) return heads <= 80 || tiles == 1;
  if (D > 48) return heads <= 64 || wgs <= 960 || L <= 512;
  if (D > 32) return heads <= 64 ? wgs <= 768 || L <= 1024 : wgs <= 640;
  if (heads > 64) return false;
  if (D > 16) return wgs <= 768 && L >= (wgs <= 448 ? 4 : tiles <= 16 ? 5 : 6) * kDc;
  return wgs <= (heads <= 48 || L <= 1024 ? 512 : 256) && L >= (wgs > 256 ? 8 : wgs > 128 || heads > 48 || tiles > 16 ? 6 : 4) * kDc;
}

// Where chunks are the faster form in fp32: few heads, and enough chunks.  A chunk step of the scan takes 1.3 us (1.6 with heads of more than 64
// channels, which fill eight tiles whatever their size) where four blocks of 16 take 3.2 to 6.8, by the size of the heads; but both
// launches together start 8 to 10 us later than those of the blocks, values of many tiles read every chunk's rows once each, and every head
// adds 20 to 90 ns of preparation a chunk: 26 times a block's products, and more memory than the cache holds at the far end.  us, blocks
// of 16 against chunks as they were with products on fp32 MFMA (they take 0.8 to 1.02 of that since), heads, d x dv:
//   8, 64 x 64: L = 256: 27.7, 24.0.  32, 64 x 128: L = 256: 29, 28; L = 2048: 161, 91.  64, 64 x 128: L = 256: 33, 35; L = 384: 45, 43.
//   64, 32 x 128: L = 512: 47, 48; L = 2048: 154, 170.  8, 64 x 512: L = 256: 30, 34; L = 384: 39, 38.
//   8, 96 x 96: L = 256: 41, 35.  32, 96 x 256: L = 384: 59, 61; L = 1024: 131, 121.  64, 96 x 128: L = 512: 75, 77; L = 2048: 263, 298.
//   8, 128 x 128: L = 256: 35.0, 35.4; L = 320: 40, 38.  32, 128 x 128: L = 320: 41, 42; L = 384: 47, 45.  16, 128 x 256: L = 384: 45, 47;
//   L = 512: 56, 52.  More heads: 128, 64 x 64, L = 4096: 415, 493; more channels: 16, 256 x 256, L = 300: 62.6, 66.0.
static bool dc_faster(int64_t B, int64_t L, int64_t H, int64_t D, int64_t DV, bool bf16) {
  const int64_t heads = B * H, tiles = (DV + 15) / 16, wgs = heads * tiles;  // (of the scan, two of which a compute unit holds)
  if (bf16 && dc_faster_bf16(heads, L, D, DV)) return true;  // (and what follows: a work space asked for without a type is for either)
  if (heads > 64 || wgs > 512 || D > 128) return false;
  const bool crowded = wgs > 256;
  const int64_t wide = tiles > 16 ? (tiles - 16) / 8 : 0;
  int64_t chunks;
  if (D > 96)
    chunks = 3 + (DV + 127) / 128 + (DV > 128) + (heads > 8 && !crowded);
  else if (crowded && (D <= 16 || (heads > 32 && (D > 64 || D <= 32))))  // (the blocks' steps are cheap here, and there is much to prepare)
    return false;
  else if (D > 64)
    chunks = crowded ? 10 : 4 + wide;
  else if (D > 32)
    chunks = 4 + (D > 48 ? wide : 0) + (wgs > 448) + (wgs > 448 && heads > 32);
  else if (D > 16)
    chunks = crowded ? 12 : 4 + wgs / 100 + wide;
  else
    chunks = 4 + (wgs < 96 ? wgs / 24 : 4) + (tiles > 8) + 2 * wide;
  return L >= chunks * kDc && L >= BASED_DELTA_CHUNKS_MIN;
}

static int dc_tiles(int64_t D) { return D <= 64 ? 4 : 8; }

// parts of an element of queries and keys
static int dc_parts(bool bf16) { return bf16 ? 1 : 3; }

// chunks per span, 0 where blocks of 16 are for the shape
static int64_t dc_span(int64_t B, int64_t L, int64_t H, int64_t D, int64_t DV, bool bf16) {
  if (B <= 0 || L <= 0 || H <= 0 || D <= 0 || DV <= 0 || B >= (1ll << 31) || H >= (1ll << 31) || DV >= (1ll << 20)) return 0;
  if (!dc_faster(B, L, H, D, DV, bf16)) return 0;
  const int64_t chunks = (L + kDc - 1) / kDc, each = B * H * dc_floats(dc_tiles(D), dc_parts(bf16), (int)DV);
  int64_t span = kDcWorkFloats / each;  // (at least 11: a chunk of 128 heads of 128 channels and 8 value tiles takes 4.3 M floats)
  if (span > chunks) span = chunks;
  // spans of about equal length
  const int64_t n = (chunks + span - 1) / span;
  return (chunks + n - 1) / n;
}

static int64_t dc_work(int64_t B, int64_t L, int64_t H, int64_t D, int64_t DV, bool bf16) {
  const int64_t span = dc_span(B, L, H, D, DV, bf16);
  return span == 0 ? 0 : B * H * span * dc_floats(dc_tiles(D), dc_parts(bf16), (int)DV);
}

// Rows of queries and keys whose groups of four channels are one load; chunks of more than 64 channels take no others.
static bool dc_vec(const void* q, const void* k, int64_t B, int64_t D, int64_t x_sb, int64_t x_sl) {
  return D % 4 == 0 && (B == 1 || x_sb % 4 == 0) && x_sl % 4 == 0 && aligned_to(q, 16) && aligned_to(k, 16);
}
static bool dc_near(int64_t H, int64_t DV, int64_t x_sl) { return x_sl >= 0 && x_sl < (1ll << 24) && H * DV < (1ll << 25); }

template <typename T, int RB, int LAY> static int run_delta_chunks(DeltaChunkArgs a, int64_t span, hipStream_t s) {
  constexpr int NP = sizeof(T) == 2 ? 1 : 3;
  const int chunks = (a.L + kDc - 1) / kDc;
  for (int c = 0; c < chunks; c += (int)span) {
    a.c0 = c;
    a.span = chunks - c < span ? chunks - c : (int)span;
    hipLaunchKernelGGL((delta_chunk_prepare_kernel<T, LAY, RB>), dim3((unsigned)((long)a.B * a.H * a.span)), dim3(256), 0, s, a);
    hipLaunchKernelGGL((delta_chunk_scan_kernel<RB, NP>), dim3((unsigned)(a.B * a.H), (unsigned)((a.dv + 15) / 16)), dim3(512), 0, s, a);
    const int rc = check_launch("gated_delta_scan_chunks");
    if (rc) return rc;
    a.fresh = 0;
  }
  return BASED_OK;
}

template <typename T, int RB> static int run_delta_lay(const DeltaChunkArgs& a, bool vec, int64_t span, hipStream_t s) {
  if constexpr (RB == 4)
    if (!vec) return run_delta_chunks<T, RB, 0>(a, span, s);
  return a.d < RB * 16 ? run_delta_chunks<T, RB, 1>(a, span, s) : run_delta_chunks<T, RB, 2>(a, span, s);
}

template <typename T> static int run_delta(const DeltaChunkArgs& a, bool vec, int64_t span, hipStream_t s) {
  return dc_tiles(a.d) == 4 ? run_delta_lay<T, 4>(a, vec, span, s) : run_delta_lay<T, 8>(a, vec, span, s);
}

}  // namespace based

extern "C" BASED_API int64_t based_gated_delta_scan_work(int64_t B, int64_t L, int64_t H, int64_t D, int64_t DV) {
  using namespace based;
  // (a span of bf16 may hold more chunks, and all of them more than fewer of fp32)
  const int64_t wide = dc_work(B, L, H, D, DV, false), narrow = dc_work(B, L, H, D, DV, true);
  return wide == 0 || wide > narrow ? wide : narrow;
}

extern "C" BASED_API int64_t based_gated_delta_scan_work_of(const void* q, const void* k, int64_t B, int64_t L, int64_t H, int64_t D,
                                                            int64_t DV, int64_t x_sb, int64_t x_sl) {
  using namespace based;
  if (!dc_near(H, DV, x_sl) || !(D <= 64 || dc_vec(q, k, B, D, x_sb, x_sl))) return 0;
  return based_gated_delta_scan_work(B, L, H, D, DV);
}

extern "C" BASED_API int64_t based_gated_delta_scan_work_as(const void* q, const void* k, int64_t B, int64_t L, int64_t H, int64_t D,
                                                            int64_t DV, int64_t x_sb, int64_t x_sl, int io_dtype) {
  using namespace based;
  if (!dc_near(H, DV, x_sl) || !(D <= 64 || dc_vec(q, k, B, D, x_sb, x_sl))) return 0;
  return dc_work(B, L, H, D, DV, io_dtype == BASED_BF16);
}

extern "C" BASED_API int based_gated_delta_scan_chunks(const void* q, const void* k, const void* v, const void* a_gate, const void* b_gate,
                                                       const void* a_log, const void* dt_bias, float* state, float* work, float* o,
                                                       int64_t B, int64_t L, int64_t H, int64_t G, int64_t D, int64_t DV, int64_t state_row,
                                                       int64_t x_sb, int64_t x_sl, int64_t g_sb, int64_t g_sl, int fresh, int io_dtype,
                                                       void* stream) {
  using namespace based;
  const char* who = "gated_delta_scan";
  BASED_REQUIRE(q && k && v && a_gate && b_gate && a_log && dt_bias && state && work && o, BASED_ERR_ARG, "%s: null pointer argument", who);
  BASED_REQUIRE(B >= 0 && L >= 0 && H > 0 && G > 0 && D > 0 && DV > 0, BASED_ERR_ARG, "%s: bad sizes", who);
  BASED_REQUIRE(H % G == 0, BASED_ERR_SHAPE, "%s: %ld heads do not divide into %ld query/key heads", who, (long)H, (long)G);
  BASED_REQUIRE(D <= 128, BASED_ERR_SHAPE, "%s: query/key size %ld (at most 128 in chunks)", who, (long)D);
  BASED_REQUIRE(state_row >= DV, BASED_ERR_ARG, "%s: state rows of %ld for a value size of %ld", who, (long)state_row, (long)DV);
  BASED_REQUIRE(io_dtype == BASED_BF16 || io_dtype == BASED_F32, BASED_ERR_DTYPE, "%s: bad dtype", who);
  BASED_REQUIRE(B * H < (1ll << 31) && L < (1ll << 31) - kDc && DV < (1ll << 20), BASED_ERR_SHAPE, "%s: grid too large", who);
  if (B == 0 || L == 0) return BASED_OK;
  BASED_REQUIRE(dc_near(H, DV, x_sl), BASED_ERR_SHAPE, "%s: rows too long", who);
  BASED_REQUIRE(aligned_to(work, 16), BASED_ERR_ALIGN, "%s: the work space must be 16-byte aligned", who);
  const int64_t span = dc_span(B, L, H, D, DV, io_dtype == BASED_BF16);
  BASED_REQUIRE(span > 0 && B * H * span < (1ll << 31), BASED_ERR_SHAPE, "%s: the shape is for blocks of 16", who);
  const bool vec = dc_vec(q, k, B, D, x_sb, x_sl);
  BASED_REQUIRE(vec || D <= 64, BASED_ERR_ALIGN, "%s: chunks of heads of more than 64 channels take rows of whole 16-byte pieces", who);
  const long per = (long)dc_floats(dc_tiles(D), dc_parts(io_dtype == BASED_BF16), (int)DV);
  const int v_vec = DV % 4 == 0 && (B == 1 || x_sb % 4 == 0) && x_sl % 4 == 0 && aligned_to(v, 16);
  const DeltaChunkArgs a{q,      k,      v,       a_gate,         b_gate, a_log, dt_bias, state, o,    work,  per,  (int)B, (int)L, (int)H,
                         (int)G, (int)D, (int)DV, (int)state_row, 0,      0,     x_sb,    x_sl,  g_sb, g_sl, fresh, v_vec};
  hipStream_t s = static_cast<hipStream_t>(stream);
  return io_dtype == BASED_BF16 ? run_delta<__bf16>(a, vec, span, s) : run_delta<float>(a, vec, span, s);
}
