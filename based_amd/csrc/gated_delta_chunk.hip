// Gated delta rule over prompts in chunks of 64 tokens, for gfx950: the recurrence of gated_delta.hip with the serial part made short.
//
// With the decays multiplied up inside a chunk, G_t = g_1 .. g_t, and A_ts = beta_t (k_t . k_s) G_t / G_s for s < t, T = (I + A)^-1,
// the values that enter the state are U = T (beta v) - T (beta G k) S0: an affine function of the state S0 in front of the chunk.
//   delta_chunk_prepare  everything that does not need S0, all chunks at once, a workgroup each: Uv = T (beta v), W = -T (beta G k) and
//                        P_ts = (q_t . k_s) G_t / G_s.  T by forward substitution in the four diagonal blocks of 16 (a power series
//                        would lose digits to cancellation), the others from them block by block.
//   delta_chunk_scan     walks the chunks: U = Uv + W S0, S1 = G_64 S0 + sum_s k_s (G_64 / G_s) u_s^T, and beside the chain
//                        o_t = G_t S0^T q_t + sum_{s <= t} P_ts u_s.  A workgroup of four wavefronts carries 16 value channels of a
//                        head; wavefront w has the 16 tokens w of every chunk and the state rows w, w + 4, ..; S0 and U go round
//                        through LDS, two barriers per chunk.
// Everything is fp32 MFMA (v_mfma_f32_16x16x4_f32).  The accumulator layout (column = lane % 16, row = 4 (lane / 16) + i) is the operand
// of instruction i of a product contracted over rows {i, 4 + i, 8 + i, 12 + i}, so accumulators become operands as they stand, and
// what delta_chunk_prepare leaves lies as the scan's lanes want it: whole wavefronts of 16-byte pieces.
//
// Against blocks of 16 (gated_delta_scan_kernel) a chain step takes in four times the tokens with two exchanges instead of one, and
// nothing but W S0 and k^T U stands in the chain.  Products per 64 tokens, d = 64, dv = 128: 3.9 -> 7.9 M fp32 operations in all, of
// which 3.9 M in the scan.  4 sequences x 8 heads of 2048 tokens: 161 -> 91 us; traced, 41 of preparation (written back at 2.3 TB/s, matrix
// pipe a third busy) and 55 of scan (a lone workgroup per compute unit: 2.0 of 4.1 thousand cycles a chunk are products, the rest waits for
// accumulators, LDS and barriers; eight wavefronts with the outputs apart from the chain take 60).
#include "gated_delta.hpp"

namespace based {

constexpr int kDc = 64;           // tokens per chunk
constexpr int kDcPairs = 10;      // lower-triangular pairs of 16-token tiles
// pairs (0, 0), (1, 0), (1, 1), (2, 0) ..: a digit each, in registers (a table would be read from memory)
__host__ __device__ constexpr int pair_t(int p) { return (int)(0x3333222110ull >> (4 * p)) & 15; }
__host__ __device__ constexpr int pair_s(int p) { return (int)(0x3210210100ull >> (4 * p)) & 15; }
__host__ __device__ constexpr int pair_of(int t, int s) { return t * (t + 1) / 2 + s; }

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

// What a chunk leaves in the workspace, in tiles of 256 floats, a lane's four next to each other: W and q by (token tile, channel
// tile), k G_64 / G_t by (channel tile, token tile), P by pair, Uv by (value tile, token tile); then fq G of every token, and G_64.
// (q and k in bf16 would halve their bytes, and cost the scan a conversion in front of every product: 56 -> 68 us.)
template <int RB> struct DcAt {
  static constexpr long kW = 0, kQ = (long)4 * RB * 256, kK = 2 * kQ, kP = 3 * kQ, kUv = kP + kDcPairs * 256;
};
__host__ __device__ inline long dc_vec_at(int rb, int dv) { return ((long)12 * rb + kDcPairs + (long)((dv + 15) / 16) * 4) * 256; }
__host__ __device__ inline long dc_floats(int rb, int dv) { return dc_vec_at(rb, dv) + kDc + 4; }

// exp of a sum of log decays held in 64 bits, which as a float would lose |x| 2^-24 of the result
__device__ __forceinline__ float exp_of(double x) {
  const float hi = (float)x, e = expf(hi);
  return __builtin_fmaf(e, (float)(x - (double)hi), e);
}

// Four channels of a row in LDS.
template <typename T> __device__ __forceinline__ f32x4 four_at(const T* p) {
  typedef __attribute__((ext_vector_type(4))) T t4;
  const t4 r = *reinterpret_cast<const t4*>(p);
  return f32x4{to_f32(r[0]), to_f32(r[1]), to_f32(r[2]), to_f32(r[3])};
}

// RB: 16-channel tiles of queries and keys.  LAY as for Four.  Rows go through LDS 64 channels at a time: a lane's operands lie in 16
// rows, and asked for one by one they cost 16 lines of cache per instruction (20 of 44 thousand cycles of a lone workgroup).
template <typename T, int LAY, int RB>
__global__ __launch_bounds__(256, 2) void delta_chunk_prepare_kernel(const DeltaChunkArgs a) {
  constexpr int kRow = kDc + 4, kSlabs = RB / 4;
  constexpr bool kAhead = LAY != 0 && sizeof(T) == 2;  // slabs of queries and keys asked for one ahead (others do not fit the registers)
  typedef DcAt<RB> At;
  typedef __attribute__((ext_vector_type(4))) T t4;
  __shared__ __attribute__((aligned(16))) float s_a[kDc][kRow], s_t[kDc][kRow];
  __shared__ __attribute__((aligned(16))) T s_x[2][kDc][kRow];
  __shared__ double s_lc[kDc];
  __shared__ __attribute__((aligned(16))) float s_beta[kDc], s_bg[kDc], s_tail[kDc], s_fq[kDc], s_fk[kDc];
  // (in the place of T, which comes later: three workgroups share a compute unit's LDS for bf16)
  float *s_e1k = &s_t[0][0], *s_e1q = s_e1k + kDc, *s_e2 = s_e1q + kDc;  // s_e2[4][kDc]
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

  // 64 channels from `e0` on of the chunk's rows: thread t has 4 channels of rows t / 16 + 16 j.  Rows past the last token are fetched
  // from it: gates of zero keep them out.
  const int piece = (tid & 15) * 4, row0 = tid >> 4;
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
      *reinterpret_cast<t4*>(&s_x[buf][row0 + j * 16][piece]) = r;
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
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      t4 r = x[j];
#pragma unroll
      for (int i = 0; i < 4; ++i) r[i] = e0 + piece + i < a.dv ? r[i] : (T)0.0f;
      *reinterpret_cast<t4*>(&s_x[buf][row0 + j * 16][piece]) = r;
    }
  };

  Four<T, LAY> kr[4], qr[4];
  fetch_slab(kr, k, 0, a.d);
  fetch_slab(qr, q, 0, a.d);
  const long gate = b * a.g_sb + (long)(t0 + (lane < left ? lane : left - 1)) * a.g_sl + h;
  const T gate_a = static_cast<const T*>(a.a)[gate], gate_b = static_cast<const T*>(a.bt)[gate];
  const T a_log = static_cast<const T*>(a.a_log)[h], dt_bias = static_cast<const T*>(a.dt_bias)[h];
  // Products of keys with keys and with queries, transposed (column = token t, row = token s): seven of the twenty tiles for each of
  // wavefronts 1 to 3, while wavefront 0 works the decays out.
  constexpr int kMine = 7;
  f32x4 acc[kMine][2];
  int ri[kMine], ci[kMine];
#pragma unroll
  for (int j = 0; j < kMine; ++j) {
    const int p = (wave > 0 ? wave - 1 : 0) * kMine + j, pair = p < kDcPairs ? p : p < 2 * kDcPairs ? p - kDcPairs : 0;
    acc[j][0] = acc[j][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    ri[j] = pair_s(pair) * 16 + l16;
    ci[j] = pair_t(pair) * 16 + l16;
  }
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
      for (int r = 0; r < 4; ++r) {
        const int e = r * 16 + quad * 4;
        __builtin_amdgcn_sched_barrier(0);  // (a quarter of the operands in registers at a time)
#pragma unroll
        for (int j = 0; j < kMine; ++j) {
          const int p = (wave - 1) * kMine + j;
          const f32x4 xf = four_at<T>(&s_x[0][ri[j]][e]), yf = four_at<T>(&s_x[p < kDcPairs ? 0 : 1][ci[j]][e]);
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[j][i & 1] = mfma_f32(xf[i], yf[i], acc[j][i & 1]);
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
    for (int r = 0; r < 4; ++r) {
      const int e = r * 16 + quad * 4;
      const f32x4 qf = four_at<T>(&s_x[1][wave * 16 + l16][e]), kf = four_at<T>(&s_x[0][wave * 16 + l16][e]);
      sq += (double)(qf[0] * qf[0] + qf[1] * qf[1]) + (double)(qf[2] * qf[2] + qf[3] * qf[3]);
      sk += (double)(kf[0] * kf[0] + kf[1] * kf[1]) + (double)(kf[2] * kf[2] + kf[3] * kf[3]);
      *reinterpret_cast<f32x4*>(ws + At::kQ + ((long)wave * RB + sl * 4 + r) * 256 + lane * 4) = qf;
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
      s_bg[lane] = -s_beta[lane] * G * fk;
      s_tail[lane] = fk * exp_of(end - lc < 0.0 ? end - lc : 0.0);
      ws[dc_vec_at(RB, a.dv) + lane] = s_fq[lane] * G;
      if (lane == 63) ws[dc_vec_at(RB, a.dv) + kDc] = G;
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
      const int p = (wave - 1) * kMine + j;
      if (p >= 2 * kDcPairs) break;  // (uniform)
      const bool keys = p < kDcPairs;
      const int pair = keys ? p : p - kDcPairs, tt = pair_t(pair), t = ci[j], s0 = pair_s(pair) * 16 + quad * 4;
      f32x4 out = acc[j][0] + acc[j][1];
      const float e1 = keys ? s_e1k[t] : s_e1q[t];
      if (pair_s(pair) != tt) {  // (uniform)
        out *= *reinterpret_cast<const f32x4*>(&s_e2[tt * kDc + s0]) * e1;
      } else {
        const double lc_t = s_lc[t], fall = (tt > 0 ? s_lc[tt > 0 ? tt * 16 - 1 : 0] : 0.0) - s_lc[tt * 16 + 15];
        f32x4 f = *reinterpret_cast<const f32x4*>(&s_e2[s0]) * e1;
        if (fall > 60.0) {
          const float ft = keys ? s_fk[t] * s_beta[t] : s_fq[t];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const double diff = lc_t - s_lc[s0 + i];
            f[i] = ft * s_fk[s0 + i] * exp_of(diff < 0.0 ? diff : 0.0);
          }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) out[i] = s0 + i < t || (s0 + i == t && !keys) ? out[i] * f[i] : 0.f;
      }
      if (keys)
        *reinterpret_cast<f32x4*>(&s_a[t][s0]) = out;
      else
        *reinterpret_cast<f32x4*>(ws + At::kP + pair * 256 + lane * 4) = out;
    }
  }
  __syncthreads();
  // T: the diagonal blocks, one per wavefront; column l16: x_t = [t = l16] - sum_{s<t} A_ts x_s
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
      for (int t = 0; t < 16; ++t) s_t[at + t][at + l16] = x[t];
    }
  }
  __syncthreads();
  // the blocks below them, a column of blocks per wavefront: T_ij = -T_ii sum_{j <= k < i} A_ik T_kj
  const f32x4 none = {0.f, 0.f, 0.f, 0.f};
  if (wave < 3) {
    f32x4 col[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      col[i] = none;
      if (i == wave) {
#pragma unroll
        for (int x = 0; x < 4; ++x) col[i][x] = s_t[i * 16 + quad * 4 + x][i * 16 + l16];
      } else if (i > wave) {
        f32x4 sum[2] = {none, none};
#pragma unroll
        for (int kb = 0; kb < i; ++kb)
          if (kb >= wave) {
            const f32x4 row = *reinterpret_cast<const f32x4*>(&s_a[i * 16 + l16][kb * 16 + quad * 4]);
#pragma unroll
            for (int x = 0; x < 4; ++x) sum[x & 1] = mfma_f32(row[x], col[kb][x], sum[x & 1]);
          }
        const f32x4 row = *reinterpret_cast<const f32x4*>(&s_t[i * 16 + l16][i * 16 + quad * 4]);
        const f32x4 y = sum[0] + sum[1];
        f32x4 res[2] = {none, none};
#pragma unroll
        for (int x = 0; x < 4; ++x) res[x & 1] = mfma_f32(row[x], y[x], res[x & 1]);
        col[i] = -(res[0] + res[1]);
#pragma unroll
        for (int x = 0; x < 4; ++x) s_t[i * 16 + quad * 4 + x][wave * 16 + l16] = col[i][x];
      }
    }
  }
  if constexpr (kSlabs > 1)
    store_slab(0, kr, 0, a.d);
  else
    store_v(1, vr, 0);
  __syncthreads();
  f32x4 tm[kDcPairs];
#pragma unroll
  for (int p = 0; p < kDcPairs; ++p) tm[p] = *reinterpret_cast<const f32x4*>(&s_t[pair_t(p) * 16 + l16][pair_s(p) * 16 + quad * 4]);
  auto column = [&](int buf, int s, int i) { return to_f32(s_x[buf][s * 16 + quad * 4 + i][wave * 16 + l16]); };
  // W^T (row = channel, column = token: the scan's operand) and the scaled keys of a slab's channel tile `wave`
  auto keys_tile = [&](int buf, int tile) {
    f32x4 out[4] = {none, none, none, none};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const f32x4 f = *reinterpret_cast<const f32x4*>(&s_bg[s * 16 + quad * 4]), g = *reinterpret_cast<const f32x4*>(&s_tail[s * 16 + quad * 4]);
      f32x4 kf;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float x = column(buf, s, i), xf = x * f[i];
        kf[i] = x * g[i];
#pragma unroll
        for (int m = s; m < 4; ++m) out[m] = mfma_f32(xf, tm[pair_of(m, s)][i], out[m]);
      }
      *reinterpret_cast<f32x4*>(ws + At::kK + ((long)tile * 4 + s) * 256 + lane * 4) = kf;
    }
#pragma unroll
    for (int m = 0; m < 4; ++m) *reinterpret_cast<f32x4*>(ws + At::kW + ((long)m * RB + tile) * 256 + lane * 4) = out[m];
  };
  // Uv (row = token, column = channel: the scan's accumulator) of a slab's value tile `wave`
  auto values_tile = [&](int buf, int tile) {
    f32x4 out[4] = {none, none, none, none};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const f32x4 f = *reinterpret_cast<const f32x4*>(&s_beta[s * 16 + quad * 4]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float xf = column(buf, s, i) * f[i];
#pragma unroll
        for (int m = s; m < 4; ++m) out[m] = mfma_f32(tm[pair_of(m, s)][i], xf, out[m]);
      }
    }
#pragma unroll
    for (int m = 0; m < 4; ++m) *reinterpret_cast<f32x4*>(ws + At::kUv + ((long)tile * 4 + m) * 256 + lane * 4) = out[m];
  };
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
      keys_tile(buf, sl * 4 + wave);
      if (!kAhead) fetch();
      buf ^= 1;
      if (sl + 1 < kSlabs)
        store_slab(buf, kr, (sl + 1) * 64, a.d);
      else
        store_v(buf, vr, 0);
      __syncthreads();
    }
  } else {
    keys_tile(0, wave);
    buf = 1;
  }
#pragma unroll 1
  for (int e0 = 0; e0 < a.dv; e0 += 64) {
    const bool more = e0 + 64 < a.dv;
    if (more) fetch_v(vr, e0 + 64);
    if (e0 + wave * 16 < a.dv) values_tile(buf, e0 / 16 + wave);
    if (!more) break;
    buf ^= 1;
    if (kSlabs == 1 && e0 == 0) __syncthreads();  // (a slower wavefront may still read the keys there)
    store_v(buf, vr, e0 + 64);
    __syncthreads();
  }
}

// grid: x = (sequence, head), y = 16 value channels
template <int RB>
__global__ __launch_bounds__(256, 2) void delta_chunk_scan_kernel(const DeltaChunkArgs a) {
  static_assert(RB % 4 == 0, "every wavefront has state rows");
  constexpr int RBW = RB / 4;
  typedef DcAt<RB> At;
  __shared__ __attribute__((aligned(16))) f32x4 s_s[RB][64], s_u[2][4][64];
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, quad = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int bh = blockIdx.x, b = __builtin_amdgcn_readfirstlane(bh / a.H), h = bh - b * a.H;
  const int ct = blockIdx.y, col = ct * 16 + l16;
  const bool col_in = col < a.dv;
  const float* ws = a.work + (long)bh * a.span * a.per;
  const long vec_at = dc_vec_at(RB, a.dv);
  float* st = a.state + (long)bh * a.d * a.dvp + (col_in ? col : 0);
  const int o_sl = a.H * a.dv;
  float* o = a.o + ((long)b * a.L * a.H + h) * a.dv + (long)a.c0 * kDc * o_sl;
  const f32x4 none = {0.f, 0.f, 0.f, 0.f};

  f32x4 S[RBW];  // rows 16 (wave + 4 x) ..
#pragma unroll
  for (int x = 0; x < RBW; ++x) {
    const int r = wave + 4 * x;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = r * 16 + quad * 4 + i;
      const bool in = !a.fresh && col_in && row < a.d;
      S[x][i] = in ? st[(long)row * a.dvp] : 0.f;
    }
    s_s[r][lane] = S[x];
  }

  // What a chunk needs from memory: one set of registers, each part asked for anew as soon as its last use has been issued, in the
  // order of the uses, so that a part travels for the rest of the chunk.
  f32x4 w[RB], p[4], uv, gq, qx[RB], kt[RBW][4];
  float last;
  auto tile_at = [&](int n, long at) { return *reinterpret_cast<const f32x4*>(ws + (long)n * a.per + at + lane * 4); };
  auto rows_at = [&](int n, long at) { return *reinterpret_cast<const f32x4*>(ws + (long)n * a.per + at + wave * 16 + quad * 4); };
  auto fetch_w = [&](int n) {
#pragma unroll
    for (int r = 0; r < RB; ++r) w[r] = tile_at(n, At::kW + (wave * RB + r) * 256);
    uv = tile_at(n, At::kUv + (ct * 4 + wave) * 256);
  };
  auto fetch_q = [&](int n) {
#pragma unroll
    for (int r = 0; r < RB; ++r) qx[r] = tile_at(n, At::kQ + (wave * RB + r) * 256);
  };
  auto fetch_k = [&](int n) {
#pragma unroll
    for (int x = 0; x < RBW; ++x)
#pragma unroll
      for (int s = 0; s < 4; ++s) kt[x][s] = tile_at(n, At::kK + ((wave + 4 * x) * 4 + s) * 256);
    last = ws[(long)n * a.per + vec_at + kDc];
  };
  auto fetch_p = [&](int n) {
    gq = rows_at(n, vec_at);
#pragma unroll
    for (int s = 0; s < 4; ++s)  // (tiles behind the wavefront's own tokens: its own again, not used)
      p[s] = tile_at(n, At::kP + (wave * (wave + 1) / 2 + (s <= wave ? s : wave)) * 256);
  };

  fetch_w(0);
  __builtin_amdgcn_sched_barrier(0);
  fetch_q(0);
  __builtin_amdgcn_sched_barrier(0);
  fetch_k(0);
  __builtin_amdgcn_sched_barrier(0);
  fetch_p(0);
  unsigned mine = (unsigned)((wave * 16 + quad * 4) * o_sl + (col_in ? col : 0)) * 4u;
  for (int n = 0; n < a.span; ++n) {
    const int next = n + 1 < a.span ? n + 1 : n, buf = n & 1;
    lds_barrier();  // S0 is there
    f32x4 s0[RB];
#pragma unroll
    for (int r = 0; r < RB; ++r) s0[r] = s_s[r][lane];
    // (what is added to a sum that starts from the large term loses its last digits sixteen times: added at the end, once)
    f32x4 u[4] = {none, none, none, none};
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i) u[i] = mfma_f32(w[r][i], s0[r][i], u[i]);
    s_u[buf][wave][lane] = uv + ((u[0] + u[1]) + (u[2] + u[3]));
    __builtin_amdgcn_sched_barrier(0);
    fetch_w(next);
    __builtin_amdgcn_sched_barrier(0);
    // the queries' product with the state fills the wait for the other wavefronts
    f32x4 oo[2] = {none, none};
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i) oo[i & 1] = mfma_f32(qx[r][i], s0[r][i], oo[i & 1]);
    __builtin_amdgcn_sched_barrier(0);
    fetch_q(next);
    lds_barrier();  // U is there
    f32x4 us[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) us[s] = s_u[buf][s][lane];
#pragma unroll
    for (int x = 0; x < RBW; ++x) {
      f32x4 sum[4] = {none, none, none, none};
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int s = 0; s < 4; ++s) sum[s] = mfma_f32(kt[x][s][i], us[s][i], sum[s]);
      S[x] = S[x] * last + ((sum[0] + sum[1]) + (sum[2] + sum[3]));
      s_s[wave + 4 * x][lane] = S[x];
    }
    __builtin_amdgcn_sched_barrier(0);
    fetch_k(next);
    __builtin_amdgcn_sched_barrier(0);
    oo[0] = gq * (oo[0] + oo[1]);
    oo[1] = none;
#pragma unroll
    for (int s = 0; s < 4; ++s)
      if (s <= wave) {  // (uniform)
#pragma unroll
        for (int i = 0; i < 4; ++i) oo[i & 1] = mfma_f32(p[s][i], us[s][i], oo[i & 1]);
      }
    const f32x4 out = oo[0] + oo[1];
    __builtin_amdgcn_sched_barrier(0);
    fetch_p(next);
    char* ob = reinterpret_cast<char*>(o + (long)n * kDc * o_sl);
    const int left = a.L - (a.c0 + n) * kDc;
    if (col_in) {
      if (left >= kDc) {  // (uniform)
#pragma unroll
        for (int i = 0; i < 4; ++i) *reinterpret_cast<float*>(ob + (long)i * o_sl * 4 + mine) = out[i];
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (wave * 16 + quad * 4 + i < left) *reinterpret_cast<float*>(ob + (long)i * o_sl * 4 + mine) = out[i];
      }
    }
  }
#pragma unroll
  for (int x = 0; x < RBW; ++x)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = (wave + 4 * x) * 16 + quad * 4 + i;
      if (col_in && row < a.d) st[(long)row * a.dvp] = S[x][i];
    }
}

// Workspace: the chunks of one launch pair.  Long prompts go through it in spans of chunks, the state carried on in between.
constexpr int64_t kDcWorkFloats = 64ll << 20;  // 256 MB, which the last-level cache holds between the two launches

// Where chunks are the faster form: few heads, and enough chunks.  A chunk step of the scan takes 1.5 us (2.7 with heads of more than 64
// channels, which fill eight tiles whatever their size) where four blocks of 16 take 3.2 to 6.8, by the size of the heads; but both
// launches together start 8 to 10 us later than those of the blocks, values of many tiles read every chunk's rows once each, and every head
// adds 20 to 90 ns of preparation a chunk: 26 times a block's products, and more memory than the cache holds at the far end.  us, blocks
// of 16 against chunks, heads, d x dv:
//   8, 64 x 64: L = 256: 27.7, 24.0.  32, 64 x 128: L = 256: 29, 28; L = 2048: 161, 91.  64, 64 x 128: L = 256: 33, 35; L = 384: 45, 43.
//   64, 32 x 128: L = 512: 47, 48; L = 2048: 154, 170.  8, 64 x 512: L = 256: 30, 34; L = 384: 39, 38.
//   8, 96 x 96: L = 256: 41, 35.  32, 96 x 256: L = 384: 59, 61; L = 1024: 131, 121.  64, 96 x 128: L = 512: 75, 77; L = 2048: 263, 298.
//   8, 128 x 128: L = 256: 35.0, 35.4; L = 320: 40, 38.  32, 128 x 128: L = 320: 41, 42; L = 384: 47, 45.  16, 128 x 256: L = 384: 45, 47;
//   L = 512: 56, 52.  More heads: 128, 64 x 64, L = 4096: 415, 493; more channels: 16, 256 x 256, L = 300: 62.6, 66.0.
static bool dc_faster(int64_t B, int64_t L, int64_t H, int64_t D, int64_t DV) {
  const int64_t heads = B * H, tiles = (DV + 15) / 16, wgs = heads * tiles;  // (of the scan, two of which a compute unit holds)
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

// chunks per span, 0 where blocks of 16 are for the shape
static int64_t dc_span(int64_t B, int64_t L, int64_t H, int64_t D, int64_t DV) {
  if (B <= 0 || L <= 0 || H <= 0 || D <= 0 || DV <= 0 || B >= (1ll << 31) || H >= (1ll << 31) || DV >= (1ll << 20) || !dc_faster(B, L, H, D, DV))
    return 0;
  const int64_t chunks = (L + kDc - 1) / kDc, each = B * H * dc_floats(dc_tiles(D), (int)DV);
  int64_t span = kDcWorkFloats / each;  // (at least 29: a chunk of 64 heads and 512 value tiles takes 2.3 M floats at most)
  if (span > chunks) span = chunks;
  // spans of about equal length
  const int64_t n = (chunks + span - 1) / span;
  return (chunks + n - 1) / n;
}

// Rows of queries and keys whose groups of four channels are one load; chunks of more than 64 channels take no others.
static bool dc_vec(const void* q, const void* k, int64_t B, int64_t D, int64_t x_sb, int64_t x_sl) {
  return D % 4 == 0 && (B == 1 || x_sb % 4 == 0) && x_sl % 4 == 0 && aligned_to(q, 16) && aligned_to(k, 16);
}
static bool dc_near(int64_t H, int64_t DV, int64_t x_sl) { return x_sl >= 0 && x_sl < (1ll << 24) && H * DV < (1ll << 25); }

template <typename T, int RB, int LAY> static int run_delta_chunks(DeltaChunkArgs a, int64_t span, hipStream_t s) {
  const int chunks = (a.L + kDc - 1) / kDc;
  for (int c = 0; c < chunks; c += (int)span) {
    a.c0 = c;
    a.span = chunks - c < span ? chunks - c : (int)span;
    hipLaunchKernelGGL((delta_chunk_prepare_kernel<T, LAY, RB>), dim3((unsigned)((long)a.B * a.H * a.span)), dim3(256), 0, s, a);
    hipLaunchKernelGGL((delta_chunk_scan_kernel<RB>), dim3((unsigned)(a.B * a.H), (unsigned)((a.dv + 15) / 16)), dim3(256), 0, s, a);
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
  const int64_t span = dc_span(B, L, H, D, DV);
  return span == 0 ? 0 : B * H * span * dc_floats(dc_tiles(D), (int)DV);
}

extern "C" BASED_API int64_t based_gated_delta_scan_work_of(const void* q, const void* k, int64_t B, int64_t L, int64_t H, int64_t D,
                                                            int64_t DV, int64_t x_sb, int64_t x_sl) {
  using namespace based;
  if (!dc_near(H, DV, x_sl) || !(D <= 64 || dc_vec(q, k, B, D, x_sb, x_sl))) return 0;
  return based_gated_delta_scan_work(B, L, H, D, DV);
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
  const int64_t span = dc_span(B, L, H, D, DV);
  BASED_REQUIRE(span > 0 && B * H * span < (1ll << 31), BASED_ERR_SHAPE, "%s: the shape is for blocks of 16", who);
  const bool vec = dc_vec(q, k, B, D, x_sb, x_sl);
  BASED_REQUIRE(vec || D <= 64, BASED_ERR_ALIGN, "%s: chunks of heads of more than 64 channels take rows of whole 16-byte pieces", who);
  const DeltaChunkArgs a{q, k, v, a_gate, b_gate, a_log, dt_bias, state, o, work, (long)dc_floats(dc_tiles(D), (int)DV), (int)B, (int)L, (int)H,
                         (int)G, (int)D, (int)DV, (int)state_row, 0, 0, x_sb, x_sl, g_sb, g_sl, fresh,
                         DV % 4 == 0 && (B == 1 || x_sb % 4 == 0) && x_sl % 4 == 0 && aligned_to(v, 16)};
  hipStream_t s = static_cast<hipStream_t>(stream);
  return io_dtype == BASED_BF16 ? run_delta<__bf16>(a, vec, span, s) : run_delta<float>(a, vec, span, s);
}
