// Causal Taylor linear attention over a whole sequence in fp32 arithmetic, for gfx950: fp32 tensors, and bf16 ones of
// head dims that are no whole 16-channel tiles.
//
// One wavefront carries the state of 16 value channels of one (batch, head) in MFMA accumulators and walks the
// sequence 64 tokens at a time.  All products are v_mfma_f32_16x16x4_f32 (exact fp32 products and sums, twice the
// rate of the vector unit); psi is the 160-slot symmetric packing of linear_attn_prefill.hip with its weights on the
// query side, so that the state holds plain sums of x_i x_j v.
//
//   within the 64     A = tril(1 + s + s^2 / 2), s = q.k / 4;   O += A V
//   across            O += psi(q) S,   z = rowsum(A) + psi(q).Z,   y = O / (z + eps)
//   afterwards        S += psi(k)^T V,   Z += sum psi(k)
//
// A wavefront needs nothing from another one and nothing is staged in LDS, because every operand lies in memory as
// an instruction wants it.  The accumulator layout (column = lane % 16, row = 4 (lane / 16) + i) is the operand of
// instruction i of a product contracted over rows {i, 4 + i, 8 + i, 12 + i}, so S and A go from accumulators into
// operands as they are; the order of a sum over tokens is free, so both products with V contract over
// 16 kt + 4 (lane / 16) + i and share its registers; psi(k)^T is one multiplication with a rotated row of lanes
// per slot tile, psi(q) one of two registers.
//
// Bound: 400 MFMA of 32 cycles per 64 tokens and 16 channels (5.3 us at 2.4 GHz), and about ten instructions around
// each of them, which a lone wavefront cannot issue beside it: B = 16, H = 16, L = 1024, dv = 64 (one wavefront per SIMD)
// takes 196 us, B = 32 (two) 315 us, 60 % of the fp32 MFMA rate.  B = 1 in 16 segments of one chunk: 10.4 + 17.0 us,
// launch and memory round trips for the most part.  (Token by token in vector arithmetic, one workgroup per head:
// 1,700 us from B = 1 to 16.)  The four wavefronts of a workgroup take neighbouring channel tiles of one head and
// read the same q and k rows.
#include <type_traits>
#include <utility>

#include "common.hpp"

namespace based {

constexpr int kF32Chunk = 64;
constexpr int kF32Tiles = 10;                              // slot tiles of 16
constexpr int kF32Slots = 16 * kF32Tiles;
constexpr int kF32SegFloats = kF32Tiles * 256 + kF32Slots;  // a segment's S (as it sits in registers) and Z
constexpr float kPairScale = 0.17677669529663687f;          // 1 / (4 sqrt 2)

struct PrefillF32Args {
  const void* q;
  const void* k;
  const void* v;
  void* y;
  float* kv_state;
  float* k_state;
  float* ws;  // (B H, channel tiles, n_seg, kF32SegFloats)
  int H, L, dv;
  long q_sb, q_sh, q_sl, k_sb, k_sh, k_sl, v_sb, v_sh, v_sl, y_sb, y_sh, y_sl;
  float eps;
  long seg_tokens;
  int n_seg, state_vec;
  int heads, heads_z;  // B H, and those of one blockIdx.z
};

template <int T> __device__ __forceinline__ float row_ror_f32(float x) {  // value of lane (i - T) mod 16 of each 16
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x120 + T, 0xf, 0xf, false));
}

template <typename T, bool VEC> __device__ __forceinline__ f32x4 load_four(const T* p) {
  typedef __attribute__((ext_vector_type(4))) T t4;
  t4 r;
  if constexpr (VEC) {
    r = *reinterpret_cast<const t4*>(p);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = p[i];
  }
  f32x4 x;
#pragma unroll
  for (int i = 0; i < 4; ++i) x[i] = to_f32(r[i]);
  return x;
}

// psi(k) of one token per group of 16 lanes: slot tile t of lane j's entry.
__device__ __forceinline__ void psi_key(float x, int l16, float (&p)[kF32Tiles]) {
  p[0] = x * x;
  p[1] = x * row_ror_f32<1>(x);
  p[2] = x * row_ror_f32<2>(x);
  p[3] = x * row_ror_f32<3>(x);
  p[4] = x * row_ror_f32<4>(x);
  p[5] = x * row_ror_f32<5>(x);
  p[6] = x * row_ror_f32<6>(x);
  p[7] = x * row_ror_f32<7>(x);
  const float far = x * row_ror_f32<8>(x);
  p[8] = l16 < 8 ? far : (l16 == 8 ? 1.f : 0.f);
  p[9] = x;
}

// LDS of one wavefront is its own: its instructions take effect in order, only the compiler has to keep the order.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// What the state needs of a chunk: k by feature (feature = lane % 16, token = 16 kt + 4 (lane / 16) + i) and v likewise by channel.
struct F32Chunk {
  float k[4][4], v[4][4];
};

// DELTA: only the state that the segment adds, to the workspace.  VEC: rows of whole 16-byte (bf16: 8-byte) pieces whose
// offsets within a chunk fit 32 bits.
template <typename T, bool VEC, bool DELTA>
__global__ __launch_bounds__(256, 2) void lin_prefill_f32_kernel(const PrefillF32Args a) {
  __shared__ __attribute__((aligned(16))) float s_z[4][kF32Slots];
  __shared__ __attribute__((aligned(16))) float s_out[DELTA ? 1 : 4][DELTA ? 4 : 16 * kExp];
  const int lane = threadIdx.x & 63, l16 = lane & 15, quad = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tiles = (a.dv + 15) / 16, groups = (tiles + 3) / 4;
  const int head = __builtin_amdgcn_readfirstlane(blockIdx.x / groups);
  const int ct = (blockIdx.x - head * groups) * 4 + wave;
  const int bh = blockIdx.z * a.heads_z + head;
  if (ct >= tiles || bh >= a.heads) return;  // (no barrier in this kernel)
  const int b = __builtin_amdgcn_readfirstlane(bh / a.H), h = bh - b * a.H, seg = blockIdx.y;
  const long begin = seg * a.seg_tokens, end = begin + a.seg_tokens < a.L ? begin + a.seg_tokens : a.L;
  const int ch = ct * 16 + l16;
  const bool ch_in = ch < a.dv;
  const T* q = static_cast<const T*>(a.q) + b * a.q_sb + h * a.q_sh;
  const T* k = static_cast<const T*>(a.k) + b * a.k_sb + h * a.k_sh;
  const T* v = static_cast<const T*>(a.v) + b * a.v_sb + h * a.v_sh;
  T* y = static_cast<T*>(a.y) + b * a.y_sb + h * a.y_sh;
  const unsigned vch = ch_in ? ch : a.dv - 1;
  typedef std::conditional_t<VEC, unsigned, long> off_t;
  // offsets within a chunk, in bytes
  constexpr off_t E = sizeof(T);
  const off_t q_sl = (off_t)a.q_sl * E, k_sl = (off_t)a.k_sl * E, v_sl = (off_t)a.v_sl * E, y_sl = (off_t)a.y_sl * E;
  auto at = [](auto* base, off_t off) {
    typedef std::conditional_t<std::is_const_v<std::remove_pointer_t<decltype(base)>>, const char, char> byte_t;
    return reinterpret_cast<decltype(base)>(reinterpret_cast<byte_t*>(base) + off);
  };
  float* z_run = s_z[wave];  // Z in front of the current chunk

  f32x4 S[kF32Tiles];
#pragma unroll
  for (int t = 0; t < kF32Tiles; ++t) S[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  // A lane's place, hidden from the compiler, which would otherwise form every address of a chunk in front of the loop
  // and keep them all (more than 256 registers)
  auto hidden = [](int x) {
    asm volatile("" : "+v"(x));
    return x;
  };
  auto fetch = [&](F32Chunk& c, long t0) {
    const int left = (int)(a.L - t0 < kF32Chunk ? a.L - t0 : kF32Chunk) - 1;  // rows past the last token are fetched from it
    const T* kb = k + t0 * a.k_sl;
    const T* vb = v + t0 * a.v_sl;
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
      const int l16 = hidden(lane & 15), quad = hidden(lane >> 4);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = kt * 16 + quad * 4 + i;
        const off_t row = t < left ? t : left;
        c.k[kt][i] = to_f32(*at(kb, row * k_sl + (off_t)l16 * E));
        c.v[kt][i] = to_f32(*at(vb, row * v_sl + (off_t)vch * E));
      }
    }
  };
  // a query row, rotated by 4 quad: x[m] = q[(4 quad + m) mod 16]
  auto fetch_q = [&](float (&x)[16], long t0, int m, int left) {
    const int l16 = hidden(lane & 15), quad = hidden(lane >> 4), r = m * 16 + l16;
    const T* qb = q + t0 * a.q_sl;
    const off_t row = (off_t)(r < left ? r : left - 1) * q_sl;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const f32x4 p = load_four<T, VEC>(at(qb, row + (off_t)((quad * 4 + c * 4) & 15) * E));
#pragma unroll
      for (int i = 0; i < 4; ++i) x[c * 4 + i] = p[i];
    }
  };

  const f32x4 none = {0.f, 0.f, 0.f, 0.f};
  F32Chunk c;
  float zsum[kF32Tiles];
  if constexpr (DELTA) {
#pragma unroll
    for (int t = 0; t < kF32Tiles; ++t) zsum[t] = 0.f;
  }
  // S and Z take a chunk of `left` live tokens in
  auto update = [&](const F32Chunk& c, int left) {
    if constexpr (!DELTA) {
#pragma unroll
      for (int t = 0; t < kF32Tiles; ++t) zsum[t] = 0.f;
    }
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (i == 0) __builtin_amdgcn_sched_barrier(0);  // (psi of four steps at a time)
        float p[kF32Tiles];
        psi_key(c.k[kt][i], l16, p);
#pragma unroll
        for (int t = 0; t < kF32Tiles; ++t) {
          S[t] = mfma_f32(p[t], c.v[kt][i], S[t]);
          zsum[t] += p[t];
        }
      }
    if constexpr (!DELTA) {
      wave_lds_fence();
#pragma unroll
      for (int t = 0; t < kF32Tiles; ++t) {
        float s = zsum[t];
        s += __shfl_xor(s, 16, 64);
        s += __shfl_xor(s, 32, 64);
        if (t == 8 && l16 == 8) s -= (float)(kF32Chunk - left);  // rows past the end are zeros but for the constant feature
        if (quad == 0) z_run[t * 16 + l16] += s;
      }
      wave_lds_fence();
    }
  };
  // a sequence in one piece leaves its state here, one in segments from a wavefront that only adds up what they left
  const bool whole = a.n_seg == 1 && a.kv_state != nullptr;
  float* ws = a.ws + ((long)bh * tiles + ct) * a.n_seg * kF32SegFloats;
  if constexpr (!DELTA) {
    f32x4 z0 = {0.f, 0.f, 0.f, 0.f};
    const int zl = lane < kF32Slots / 4 ? lane : 0;
    // four segments' loads in flight at a time (one by one they cost 1.2 us each); past the last one it is read again and dropped
    for (int s0 = 0; s0 < seg; s0 += 4) {
      f32x4 in[4][kF32Tiles + 1];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float* p = ws + (long)(s0 + u < seg ? s0 + u : seg - 1) * kF32SegFloats;
#pragma unroll
        for (int t = 0; t < kF32Tiles; ++t) in[u][t] = *reinterpret_cast<const f32x4*>(p + t * 256 + lane * 4);
        in[u][kF32Tiles] = *reinterpret_cast<const f32x4*>(p + kF32Tiles * 256 + zl * 4);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (s0 + u < seg) {
#pragma unroll
          for (int t = 0; t < kF32Tiles; ++t) S[t] += in[u][t];
          z0 += in[u][kF32Tiles];
        }
    }
    if (lane < kF32Slots / 4) *reinterpret_cast<f32x4*>(z_run + lane * 4) = z0;
    wave_lds_fence();
  }
  if (begin < end) fetch(c, begin);
  for (long t0 = begin; t0 < end; t0 += kF32Chunk) {
    const bool more = t0 + kF32Chunk < end;
    const int left = (int)(a.L - t0 < kF32Chunk ? a.L - t0 : kF32Chunk);  // live tokens of the chunk
    if (left < kF32Chunk) {
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const bool in = kt * 16 + quad * 4 + i < left;
          c.k[kt][i] = in ? c.k[kt][i] : 0.f;
          c.v[kt][i] = in ? c.v[kt][i] : 0.f;
        }
    }
    if constexpr (!DELTA) {
      T* yb = y + t0 * a.y_sl;
      f32x4 rows[4];  // k as operands of the scores: token = lane % 16, features 4 (lane / 16) + i
      const T* kb = k + t0 * a.k_sl;
#pragma unroll
      for (int kt = 0; kt < 4; ++kt) {
        const int l16 = hidden(lane & 15), r = kt * 16 + l16;
        rows[kt] = load_four<T, VEC>(at(kb, (off_t)(r < left ? r : left - 1) * k_sl + (off_t)(hidden(lane >> 4) * 4) * E));
      }
      float qx[2][16];
      fetch_q(qx[0], t0, 0, left);
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        if (m * 16 >= left) break;  // (uniform)
        // (one tile ahead and no more, and Z read anew by every tile: either, kept, would cost 40 registers)
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        const int l16 = hidden(lane & 15), quad = hidden(lane >> 4);
        if (m < 3) fetch_q(qx[(m + 1) & 1], t0, m + 1, left);
        const float(&x)[16] = qx[m & 1];
        f32x4 A[4];
#pragma unroll
        for (int kt = 0; kt <= m; ++kt) A[kt] = none;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int kt = 0; kt <= m; ++kt) A[kt] = mfma_f32(rows[kt][i], x[i], A[kt]);
        float z = 0.f;
#pragma unroll
        for (int kt = 0; kt <= m; ++kt)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float s = A[kt][i] * 0.25f;
            const float w = __builtin_fmaf(s, __builtin_fmaf(s, 0.5f, 1.f), 1.f);
            A[kt][i] = kt < m || quad * 4 + i <= l16 ? w : 0.f;
            z += A[kt][i];
          }
        f32x4 o[2] = {none, none};
        if (t0 > 0) {  // (uniform: nothing lies in front of the first chunk)
          float xs[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) xs[i] = x[i] * 0.0625f;
#pragma unroll
          for (int t = 0; t < kF32Tiles; ++t) {
            const f32x4 zt = *reinterpret_cast<const f32x4*>(z_run + t * 16 + quad * 4);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              float p;
              if (t == 0)
                p = xs[i] * (x[i] * 0.5f);
              else if (t < 8)
                p = xs[i] * x[(i - t) & 15];
              else if (t == 8)
                p = quad < 2 ? xs[i] * x[i + 8] : (quad == 2 && i == 0 ? 1.f : 0.f);
              else
                p = x[i] * 0.25f;
              z = __builtin_fmaf(p, zt[i], z);
              // (slots without a feature hold zero times every value, which an infinity made a NaN)
              const float st = t == 8 ? (quad < 2 || (quad == 2 && i == 0) ? S[t][i] : 0.f) : S[t][i];
              o[i & 1] = mfma_f32(p, st, o[i & 1]);
            }
          }
        }
        // A zero weight takes no part even against a value that is no number: such a tile is summed by itself
        const bool odd = !(__builtin_fabsf(c.v[m][0]) < __builtin_inff() && __builtin_fabsf(c.v[m][1]) < __builtin_inff() &&
                           __builtin_fabsf(c.v[m][2]) < __builtin_inff() && __builtin_fabsf(c.v[m][3]) < __builtin_inff());
        const bool apart = __builtin_amdgcn_ballot_w64(odd) != 0;
#pragma unroll
        for (int kt = 0; kt <= m; ++kt) {
          if (kt == m && apart) {
#pragma unroll 1
            for (int key = 0; key < 16; ++key) {
              const int src = (key >> 2) * 16;
              float av[4], vv[4];
#pragma unroll
              for (int j = 0; j < 4; ++j) vv[j] = __shfl(c.v[m][j], src + l16, 64);
              const float val = (key & 3) == 0 ? vv[0] : (key & 3) == 1 ? vv[1] : (key & 3) == 2 ? vv[2] : vv[3];
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                const int token = quad * 4 + i;
#pragma unroll
                for (int j = 0; j < 4; ++j) av[j] = __shfl(A[m][j], src + token, 64);
                const float w = (key & 3) == 0 ? av[0] : (key & 3) == 1 ? av[1] : (key & 3) == 2 ? av[2] : av[3];
                if (key <= token) o[0][i] = __builtin_fmaf(w, val, o[0][i]);
              }
            }
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i & 1] = mfma_f32(A[kt][i], c.v[kt][i], o[i & 1]);
          }
        }
        z += __shfl_xor(z, 16, 64);
        z += __shfl_xor(z, 32, 64);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int t = m * 16 + quad * 4 + i;
          const float den = __shfl(z, quad * 4 + i, 64) + a.eps;
          const float num = o[0][i] + o[1][i];
          if (ch_in && t < left) *at(yb, (off_t)t * y_sl + (off_t)ch * E) = from_f32<T>(num / den);
        }
      }
    }
    if (!more && !DELTA && !whole) break;
    // the next rows travel while this chunk goes into the state: the outputs above need the registers
    F32Chunk next;
    if (more) fetch(next, t0 + kF32Chunk);
    __builtin_amdgcn_sched_barrier(0);
    update(c, left);
    if (!more) break;
    c = next;
  }

  if constexpr (DELTA) {
    float* p = ws + (long)seg * kF32SegFloats;
#pragma unroll
    for (int t = 0; t < kF32Tiles; ++t) {
      *reinterpret_cast<f32x4*>(p + t * 256 + lane * 4) = S[t];
      float s = zsum[t];
      s += __shfl_xor(s, 16, 64);
      s += __shfl_xor(s, 32, 64);
      if (t == 8 && l16 == 8) s = (float)(end - begin);  // (rows past the end counted as well)
      if (quad == 0) p[kF32Tiles * 256 + t * 16 + l16] = s;
    }
  } else if (whole || seg == a.n_seg) {
    // 16 channels x 273 features, contiguous in the decode state: laid out in LDS, then stored in one go
    float* row = s_out[wave] + l16 * kExp;
#pragma unroll
    for (int t = 0; t < kF32Tiles; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int j = quad * 4 + i;
        const float x = S[t][i];
        if (t == 0) {
          row[1 + kFeat + 17 * j] = x * kPairScale;
        } else if (t < 8) {
          const int pj = (j - t) & 15;
          row[1 + kFeat + 16 * j + pj] = x * kPairScale;
          row[1 + kFeat + 16 * pj + j] = x * kPairScale;
        } else if (t == 8) {
          if (j < 8) {
            row[1 + kFeat + 16 * j + j + 8] = x * kPairScale;
            row[1 + kFeat + 16 * (j + 8) + j] = x * kPairScale;
          } else if (j == 8) {
            row[0] = x;
          }
        } else {
          row[1 + j] = x * 0.5f;
        }
      }
    wave_lds_fence();
    const int n = (a.dv - ct * 16 < 16 ? a.dv - ct * 16 : 16) * kExp;
    float* dst = a.kv_state + ((long)bh * a.dv + ct * 16) * kExp;
    if (a.state_vec) {
      for (int i = lane; i < n / 4; i += 64) reinterpret_cast<f32x4*>(dst)[i] = reinterpret_cast<const f32x4*>(s_out[wave])[i];
    } else {
      for (int i = lane; i < n; i += 64) dst[i] = s_out[wave][i];
    }
    if (ct == 0) {
      float* ks = a.k_state + (long)bh * kExp;
      for (int f = lane; f < kExp; f += 64) {
        float x;
        if (f == 0) {
          x = z_run[8 * 16 + 8];
        } else if (f <= kFeat) {
          x = z_run[9 * 16 + f - 1] * 0.5f;
        } else {
          const int i = (f - 1 - kFeat) >> 4, j = (f - 1 - kFeat) & 15, d = (i - j) & 15;
          const int slot = d < 8 ? d * 16 + i : d > 8 ? (16 - d) * 16 + j : 8 * 16 + (i < j ? i : j);
          x = z_run[slot] * kPairScale;
        }
        ks[f] = x;
      }
    }
  }
}

// Wavefronts that fill the GPU's SIMDs once.  Below, a sequence is cut into segments: a first pass finds what each
// adds to the state, and a second starts every segment from the sum of those before it, which it forms itself (up
// to 15 reads of 11 KB a wavefront, 4 us; more segments would need a pass of their own for the sums).  A segment
// costs a second pass over its keys and values, 160 of 400 products, so two are worth it: (1 + 0.4) / 2 of the time.
// B = 1, H = 16, L = 1024: 176 us in one piece, 28 in sixteen; B = 4, L = 512: 98 against 40 in four.
constexpr int64_t kF32Waves = 1024;
constexpr int64_t kF32MaxSegments = 16;

static int64_t prefill_f32_segments(int64_t B, int64_t H, int64_t L, int64_t dv) {
  if (B <= 0 || H <= 0 || L <= 0 || dv < 1 || dv > 1024 || B * H >= (1ll << 31)) return 1;
  const int64_t waves = B * H * ((dv + 15) / 16), chunks = (L + kF32Chunk - 1) / kF32Chunk;
  int64_t want = kF32Waves / waves;
  if (want > kF32MaxSegments) want = kF32MaxSegments;
  if (want < 2 || chunks < 2) return 1;
  const int64_t per = (chunks + want - 1) / want;
  return (chunks + per - 1) / per;
}

// rows whose offsets within a chunk fit 32 bits of bytes
static bool f32_near(int64_t sl) { return sl >= 0 && sl < (1ll << 32) / (4 * kF32Chunk) - 1024; }

static bool f32_vec_ok(const void* p, int64_t sb, int64_t sh, int64_t sl, int64_t elem) {
  return reinterpret_cast<uintptr_t>(p) % (4 * elem) == 0 && sb % 4 == 0 && sh % 4 == 0 && sl % 4 == 0 && f32_near(sl);
}

template <typename T> static int launch_prefill_f32_as(PrefillF32Args a, int64_t BH, bool vec, hipStream_t s, const char* who) {
  // the groups of four channel tiles of a head are neighbours (a direction of their own: B = 4, H = 16, L = 1000, dv = 128 181 us, not
  // 135); heads beyond what a launch has workgroups for in x go on in z
  const int64_t groups = (a.dv + 63) / 64, most = ((1ll << 24) - 1) / groups;
  a.heads = (int)BH;
  a.heads_z = (int)(BH < most ? BH : most);
  const unsigned wgs = (unsigned)(a.heads_z * groups), more = (unsigned)((BH + a.heads_z - 1) / a.heads_z);
  if (a.n_seg > 1) {
    auto delta = vec ? lin_prefill_f32_kernel<T, true, true> : lin_prefill_f32_kernel<T, false, true>;
    hipLaunchKernelGGL(delta, dim3(wgs, (unsigned)(a.n_seg - (a.kv_state == nullptr)), more), dim3(256), 0, s, a);
    const int rc = check_launch(who);
    if (rc) return rc;
  }
  auto whole = vec ? lin_prefill_f32_kernel<T, true, false> : lin_prefill_f32_kernel<T, false, false>;
  // (one workgroup more per head where the state is wanted: it starts behind the last segment)
  hipLaunchKernelGGL(whole, dim3(wgs, (unsigned)(a.n_seg + (a.n_seg > 1 && a.kv_state != nullptr)), more), dim3(256), 0, s, a);
  return check_launch(who);
}

// The launches behind based_linear_attn_prefill and based_linear_attn_prefill_f32; sizes, pointers and dtype have been checked.
int launch_prefill_f32(const char* who, const void* q, const void* k, const void* v, void* y, float* kv_state, float* k_state, int64_t B,
                       int64_t H, int64_t L, int64_t dv, int64_t q_sb, int64_t q_sh, int64_t q_sl, int64_t k_sb, int64_t k_sh, int64_t k_sl,
                       int64_t v_sb, int64_t v_sh, int64_t v_sl, int64_t y_sb, int64_t y_sh, int64_t y_sl, float eps, int io_dtype,
                       int64_t n_seg, float* ws, hipStream_t s) {
  const int64_t chunks = (L + kF32Chunk - 1) / kF32Chunk, per = chunks > 0 ? (chunks + n_seg - 1) / n_seg : 1;
  const int64_t elem = io_dtype == BASED_BF16 ? 2 : 4;
  const PrefillF32Args a{q, k, v, y, kv_state, k_state, ws, (int)H, (int)L, (int)dv, q_sb, q_sh, q_sl, k_sb, k_sh, k_sl, v_sb, v_sh, v_sl,
                         y_sb, y_sh, y_sl, eps, per * kF32Chunk, (int)n_seg,
                         dv % 4 == 0 && reinterpret_cast<uintptr_t>(kv_state) % 16 == 0};
  const bool vec = f32_vec_ok(q, q_sb, q_sh, q_sl, elem) && f32_vec_ok(k, k_sb, k_sh, k_sl, elem) && f32_near(v_sl) && f32_near(y_sl);
  return io_dtype == BASED_BF16 ? launch_prefill_f32_as<__bf16>(a, B * H, vec, s, who) : launch_prefill_f32_as<float>(a, B * H, vec, s, who);
}

}  // namespace based

extern "C" BASED_API int based_linear_attn_prefill_f32_plan(int64_t B, int64_t H, int64_t L, int64_t dv, int64_t* n_seg,
                                                            int64_t* workspace_bytes) {
  using namespace based;
  BASED_REQUIRE(n_seg && workspace_bytes, BASED_ERR_ARG, "linear_attn_prefill_f32_plan: null output pointer");
  *n_seg = prefill_f32_segments(B, H, L, dv);
  *workspace_bytes = *n_seg > 1 ? B * H * ((dv + 15) / 16) * *n_seg * (int64_t)kF32SegFloats * 4 : 0;
  return BASED_OK;
}

extern "C" BASED_API int based_linear_attn_prefill_f32(
    const void* q, const void* k, const void* v, void* y, float* kv_state, float* k_state, int64_t B, int64_t H, int64_t L, int64_t dv,
    int64_t q_sb, int64_t q_sh, int64_t q_sl, int64_t k_sb, int64_t k_sh, int64_t k_sl, int64_t v_sb, int64_t v_sh, int64_t v_sl,
    int64_t y_sb, int64_t y_sh, int64_t y_sl, float eps, int io_dtype, int64_t n_seg, void* workspace, int64_t workspace_bytes,
    void* stream) {
  using namespace based;
  const char* who = "linear_attn_prefill_f32";
  BASED_REQUIRE(q && k && v && y, BASED_ERR_ARG, "%s: null pointer argument", who);
  BASED_REQUIRE((kv_state == nullptr) == (k_state == nullptr), BASED_ERR_ARG, "%s: kv_state and k_state must both be given or both be NULL", who);
  BASED_REQUIRE(B >= 0 && H > 0 && L >= 0, BASED_ERR_ARG, "%s: bad sizes", who);
  BASED_REQUIRE(io_dtype == BASED_BF16 || io_dtype == BASED_F32, BASED_ERR_DTYPE, "%s: io_dtype %d unsupported", who, io_dtype);
  BASED_REQUIRE(B * H < (1ll << 31) && L < (1ll << 31), BASED_ERR_SHAPE, "%s: sizes too large", who);
  BASED_REQUIRE(dv >= 1 && dv <= 1024, BASED_ERR_SHAPE, "%s: head dim %ld unsupported", who, (long)dv);
  if (B == 0) return BASED_OK;
  const int64_t chunks = (L + kF32Chunk - 1) / kF32Chunk;
  BASED_REQUIRE(n_seg >= 1 && n_seg <= kF32MaxSegments && (n_seg == 1 || n_seg <= chunks), BASED_ERR_ARG, "%s: %ld segments for %ld chunks",
                who, (long)n_seg, (long)chunks);
  if (n_seg > 1) {
    const int64_t per = (chunks + n_seg - 1) / n_seg;
    BASED_REQUIRE((n_seg - 1) * per < chunks, BASED_ERR_ARG, "%s: segment count %ld leaves empty segments (use the plan)", who, (long)n_seg);
    BASED_REQUIRE(workspace != nullptr && workspace_bytes >= B * H * ((dv + 15) / 16) * n_seg * (int64_t)kF32SegFloats * 4, BASED_ERR_ARG,
                  "%s: workspace too small", who);
    BASED_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 15) == 0, BASED_ERR_ALIGN, "%s: workspace must be 16-byte aligned", who);
  }
  return launch_prefill_f32(who, q, k, v, y, kv_state, k_state, B, H, L, dv, q_sb, q_sh, q_sl, k_sb, k_sh, k_sl, v_sb, v_sh, v_sl, y_sb, y_sh,
                            y_sl, eps, io_dtype, n_seg, static_cast<float*>(workspace), static_cast<hipStream_t>(stream));
}
