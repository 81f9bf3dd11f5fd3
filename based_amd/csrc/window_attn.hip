// Causal softmax attention over a sliding window of any size with grouped heads, for gfx950:
// position i attends j with 0 <= i - j < window; query head h reads key/value head h / (H / G);
// key and value sizes may differ.  In the same launches: rotary positions on the leading
// rotary_dim channels of q and k (interleaved pairs (2i, 2i + 1), or half-split pairs
// (i, i + rotary_dim / 2)) and the value norm v / sqrt(mean(v^2) + eps).
//
// The cache holds one row per token and key/value head: dim key channels (rotated), then vdim
// value channels (normalised), (B, S, G, dim + vdim).
//
//   window_kv_write      a portion's keys and values into the cache
//   window_prefill_mfma  bf16: 128 (token, head) rows per workgroup, 32 per wavefront.  The heads of
//                        a group are rows of the same tile, so that a key tile is fetched once for
//                        all of them and a tile of tokens is short against the window.  Scores are
//                        formed transposed (keys x queries), which leaves the weights in the lanes
//                        that the product with the values wants them in.
//   window_prefill_f32   fp32: 64 rows per workgroup, 16 per wavefront, otherwise alike, on fp32 MFMA
//   window_prefill_any   any element type and size: one wavefront per query
//   window_step          one token per sequence: rotation, value norm, cache write and attention,
//                        one workgroup per (sequence, key/value head)
#include "stream_common.hpp"

namespace based {

struct WindowArgs {
  const void* q;
  const void* k;
  const void* v;
  void* kv;
  void* o;
  const float* cos_t;  // (n_pos, rot / 2) or null
  const float* sin_t;
  const int32_t* pos;
  int pos_host, n_pos;
  int B, L, H, G, d, dv, S;
  long q_sb, q_sl, k_sb, k_sl, v_sb, v_sl, o_sb, o_sl;  // heads are contiguous blocks of d / dv
  long kv_sb, kv_st;
  int rot, half_split, window, norm_v;
  float scale, eps, out_scale;
  uint32_t heads_inv;  // 2^32 / (H / G), rounded down (window_prefill_mfma)
};

// partner and sign of channel c in the rotation: x'_c = x_c cos + sgn * x_partner sin
__device__ __forceinline__ void rope_pair(int c, int rot, int half_split, int& pair, int& partner, float& sgn) {
  if (half_split) {
    const int h = rot / 2;
    pair = c < h ? c : c - h;
    partner = c < h ? c + h : c - h;
    sgn = c < h ? -1.f : 1.f;
  } else {
    pair = c >> 1;
    partner = c ^ 1;
    sgn = (c & 1) ? 1.f : -1.f;
  }
}

template <typename T>
__device__ __forceinline__ float rotated(const T* row, int c, int pos, const WindowArgs& a) {
  const float x = to_f32(row[c]);
  if (c >= a.rot) return x;
  int pair, partner;
  float sgn;
  rope_pair(c, a.rot, a.half_split, pair, partner, sgn);
  const long t = (long)pos * (a.rot / 2) + pair;
  return x * a.cos_t[t] + sgn * to_f32(row[partner]) * a.sin_t[t];
}

// What turns 8 channels from c on (c and the rotary size multiples of 8): angles, and for half-split pairs
// the partners.  Loaded without a condition (what is not rotated reads the table's start and its own
// channels) and applied later, so that every load of a row is on its way before the first is waited for.
template <bool HALF> struct Turn8 {
  float cs[HALF ? 8 : 4], sn[HALF ? 8 : 4], partner[8];
  __device__ __forceinline__ void load(const __bf16* row, int c, int pos, const WindowArgs& a) {
    const bool in = c < a.rot;
    const int half = a.rot / 2;
    if constexpr (HALF) {
      const int pair = in ? (c < half ? c : c - half) : 0;
      const long t = in ? (long)pos * half + pair : 0;
      load_vec<float, 8>((a.rot > 0 ? a.cos_t : reinterpret_cast<const float*>(a.kv)) + t, cs);
      load_vec<float, 8>((a.rot > 0 ? a.sin_t : reinterpret_cast<const float*>(a.kv)) + t, sn);
      load_vec<__bf16, 8>(row + (in ? (c < half ? c + half : c - half) : 0), partner);
    } else {
      const long t = in ? (long)pos * half + c / 2 : 0;
      load_vec<float, 4>((a.rot > 0 ? a.cos_t : reinterpret_cast<const float*>(a.kv)) + t, cs);
      load_vec<float, 4>((a.rot > 0 ? a.sin_t : reinterpret_cast<const float*>(a.kv)) + t, sn);
    }
  }
  // (which of the two products is rounded is written out: left to the compiler, kernels differ in it)
  __device__ __forceinline__ void apply(float (&x)[8], int c, const WindowArgs& a) const {
    if (c >= a.rot) return;
    if constexpr (HALF) {
      const float sgn = c < a.rot / 2 ? -1.f : 1.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = __builtin_fmaf(x[j], cs[j], (sgn * partner[j]) * sn[j]);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float u = x[2 * j], v = x[2 * j + 1];
        x[2 * j] = __builtin_fmaf(u, cs[j], -(v * sn[j]));
        x[2 * j + 1] = __builtin_fmaf(v, cs[j], u * sn[j]);
      }
    }
  }
};

// One wavefront per (token, key/value head).
template <typename T>
__global__ __launch_bounds__(256) void window_kv_write_kernel(const WindowArgs a) {
  const long item = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (item >= (long)a.B * a.L * a.G) return;
  const int lane = threadIdx.x & 63;
  const int g = (int)(item % a.G);
  const long bl = item / a.G;
  const int l = (int)(bl % a.L), b = (int)(bl / a.L);
  const int pos = a.pos_host + l;
  const T* k = static_cast<const T*>(a.k) + b * a.k_sb + l * a.k_sl + (long)g * a.d;
  const T* v = static_cast<const T*>(a.v) + b * a.v_sb + l * a.v_sl + (long)g * a.dv;
  T* out = static_cast<T*>(a.kv) + b * a.kv_sb + pos * a.kv_st + (long)g * (a.d + a.dv);
  float ss = 0.f;
  for (int c = lane; c < a.dv; c += 64) ss = __builtin_fmaf(to_f32(v[c]), to_f32(v[c]), ss);
  const float r = a.norm_v ? 1.0f / sqrtf(wave_sum(ss) / (float)a.dv + a.eps) : 1.0f;
  for (int c = lane; c < a.d; c += 64) out[c] = from_f32<T>(rotated(k, c, pos, a));
  for (int c = lane; c < a.dv; c += 64) out[a.d + c] = from_f32<T>(to_f32(v[c]) * r);
}

// The same with 16-byte pieces: LPI (8, 16 or 32) lanes per (token, key/value head), one piece of the key and
// one of the value each.  d, dv and every stride multiples of 8, pointers 16-byte aligned.
template <int LPI, bool HALF>
__global__ __launch_bounds__(256) void window_kv_write_vec_kernel(const WindowArgs a) {
  const long item0 = (long)blockIdx.x * (256 / LPI) + threadIdx.x / LPI;
  const long n_items = (long)a.B * a.L * a.G;
  const bool live = item0 < n_items;
  const long item = live ? item0 : n_items - 1;
  const int c = (threadIdx.x % LPI) * 8;
  const int g = (int)(item % a.G);
  const long bl = item / a.G;
  const int l = (int)(bl % a.L), b = (int)(bl / a.L);
  const int pos = a.pos_host + l;
  const __bf16* k = static_cast<const __bf16*>(a.k) + b * a.k_sb + l * a.k_sl + (long)g * a.d;
  const __bf16* v = static_cast<const __bf16*>(a.v) + b * a.v_sb + l * a.v_sl + (long)g * a.dv;
  __bf16* out = static_cast<__bf16*>(a.kv) + b * a.kv_sb + pos * a.kv_st + (long)g * (a.d + a.dv);
  const int ck = c < a.d ? c : 0, cv = c < a.dv ? c : 0;
  float x[8], y[8];
  Turn8<HALF> turn;
  load_vec<__bf16, 8>(k + ck, x);
  load_vec<__bf16, 8>(v + cv, y);
  turn.load(k, ck, pos, a);
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < 8; ++j) ss = __builtin_fmaf(y[j], y[j], ss);
  ss = c < a.dv ? ss : 0.f;
  ss = LPI == 8 ? sum8(ss) : sum16(ss);
  if (LPI == 32) ss += __shfl_xor(ss, 16, 64);
  const float r = a.norm_v ? 1.0f / sqrtf(ss / (float)a.dv + a.eps) : 1.0f;
  turn.apply(x, ck, a);
#pragma unroll
  for (int j = 0; j < 8; ++j) y[j] *= r;
  if (live && c < a.d) store_vec<__bf16, 8>(out + c, x);
  if (live && c < a.dv) store_vec<__bf16, 8>(out + a.d + c, y);
}

// ---- prefill, bf16, MFMA ----
// KC: 32-channel pieces of the key size; VC: 32-channel pieces of the value size (both rounded up;
// channels past the real sizes are zeros).
constexpr int kTileKeys = 64;
constexpr int kTileRows = 128;  // (token, head) rows per workgroup
constexpr int kDirectTile = kTileKeys * 128;  // elements of a tile of keys and values of 64 channels

// Bound by the vector unit, and in short windows by a workgroup's own start (queries, tables, first tile: 11 of 30 thousand cycles where all
// workgroups run together).  As many wavefronts as fit: sizes up to 64 run in 128 registers, four workgroups to a compute unit (three, with
// 143: 28.9 us where four take 24.8); keys of up to 96 channels with values of 65 to 128 in 256, two (one, with 268, which the compiler takes where
// it may: 16 heads on 4, 96 x 96, 4 x 2048 tokens and 129 keys 62 us for 42).  What a wavefront sees is worked out on the scalar unit, so that only
// tiles at the edges of a window are masked; the lanes of a row look for their largest score together only where one of them has found a larger; and
// rows of 64 channels go straight into LDS.  Kernels alone, 16 heads of 64 channels, with the cache write, without and with these: on 4, 4 x 2048
// tokens and 129 keys 30.8 / 28.6 us; 6 x 2240 and 513 keys 80 / 67.6; on 2, 4 x 4096 and 1,024 keys 138 / 112; on 16, 1 x 2048 and 1,024 keys
// 45.7 / 36.9; on 4, 1 x 700 and 129 keys 12.0 / 10.8.  Weights are summed in 32 bits, as they are before the products take them rounded: sums of the
// rounded ones, by products with ones, take 0.99 of that (4 x 4096 110 for 112) and 1.03 above 64 channels (128 x 128 68.0 for 66.0).

__device__ __forceinline__ f32x4 mfma_bf16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// DIRECT: keys and values of 64 channels each, straight into LDS, the next tile while one is worked on.  Piece p (16 bytes) of row r lies at
// p ^ (r / 2 % 8), of values at p ^ (r / 2 % 4 * 2), so that reads of 16 rows (transposing reads of 8) meet every bank once; one barrier a tile.
// FILL, of such rows: the portion's keys and values are taken as they come, turned and normed on their way to LDS, and left in the cache by the
// workgroups whose tokens they are; nobody reads there what is written.
template <int KC, int VC, bool HALF, bool DIRECT, bool FILL> __device__ __forceinline__ void window_prefill_mfma(const WindowArgs& a) {
  constexpr int D = KC * 32, DV = VC * 32;
  constexpr int KS = D + 8, VS = kTileKeys + 8;  // LDS row strides: 16-lane reads of 16 bytes meet every bank once
  static_assert(!DIRECT || (KC == 2 && VC == 2), "rows of 64 channels");
  static_assert(!FILL || DIRECT, "tiles as DIRECT has them");
  __shared__ __attribute__((aligned(16))) __bf16 lds_k[DIRECT ? 8 : kTileKeys * KS];
  __shared__ __attribute__((aligned(16))) __bf16 lds_v[DIRECT ? 8 : DV * VS];
  // (an array whose extent the launch gives: in front of every read of a static one the compiler waits for all loads that go to LDS)
  extern __shared__ __attribute__((aligned(16))) __bf16 lds_tiles[];
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, quad = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // (what a wavefront sees is worked out once for it, on the scalar unit)
  const int g = blockIdx.y, b = blockIdx.z;
  const int qpk = (int)((uint32_t)a.H / (uint32_t)a.G);
  const int n_rows = a.L * qpk;
  // token of a (token, head) row, and the head: a product with the rounded inverse is the quotient or one less
  const auto token_of = [&](int row, int* head) {
    uint32_t tok = __umulhi((uint32_t)row, a.heads_inv), rest = (uint32_t)row - tok * (uint32_t)qpk;
    if (rest >= (uint32_t)qpk) ++tok, rest -= (uint32_t)qpk;
    if (head) *head = (int)rest;
    return (int)tok;
  };
  const int r0 = blockIdx.x * kTileRows;
  const int r_end = r0 + kTileRows < n_rows ? r0 + kTileRows : n_rows;
  const int row_w = r0 + wave * 32;  // first row of this wavefront
  const __bf16* kv = static_cast<const __bf16*>(a.kv) + b * a.kv_sb + (long)g * (a.d + a.dv);

  const int wave_lo_tok = a.pos_host + token_of(row_w < n_rows ? row_w : n_rows - 1, nullptr);
  const int wave_hi_row = row_w + 31 < n_rows ? row_w + 31 : n_rows - 1;
  const int wave_hi_tok = a.pos_host + token_of(wave_hi_row, nullptr);

  const int first_pos = a.pos_host + token_of(r0, nullptr), last_pos = a.pos_host + token_of(r_end - 1, nullptr);
  const int lo = first_pos - a.window + 1 > 0 ? first_pos - a.window + 1 : 0;

  // staging: keys as 16-byte pieces of rows; values as VK keys x 8 channels, turned on the way
  constexpr int KP = kTileKeys * (D / 8) / 256;  // pieces per thread
  constexpr int VK = VC >= 4 ? 4 : 2, VN = kTileKeys / VK;
  constexpr int VP = VN * (DV / 8) / 256 > 0 ? VN * (DV / 8) / 256 : 1;
  typedef __attribute__((ext_vector_type(VK))) __bf16 bf16xk;
  typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
  u32x4 kbuf[DIRECT ? 1 : KP];
  u32x4 vbuf[DIRECT ? 1 : VP][VK];
  const u32x4 zero4 = {0u, 0u, 0u, 0u};
  // rows past the last key and channels past the sizes are fetched from valid places and cleared in `stage`
  const int st32 = (int)a.kv_st;
  auto ask = [&](int k0, int place) {
    const __bf16* tile = kv + (long)k0 * a.kv_st;
    const int last = last_pos - k0;
    __bf16* to = lds_tiles + place * kDirectTile;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int group = wave * 4 + i, row = (group & 7) * 8 + (lane >> 3);  // 8 rows; keys, then values
      const int piece = group < 8 ? (lane & 7) ^ (row >> 1 & 7) : 8 + ((lane & 7) ^ (row >> 1 & 3) * 2);
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(tile + ((row <= last ? row : last) * st32 + piece * 8)),
                                       (__attribute__((address_space(3))) void*)(to + group * 512), 16, 0, 0);
    }
  };
  auto fetch = [&](int k0) {
    const __bf16* tile = kv + (long)k0 * a.kv_st;
    const int last = last_pos - k0;
#pragma unroll
    for (int i = 0; i < KP; ++i) {
      const int p = i * 256 + tid, key = p / (D / 8), e = (p % (D / 8)) * 8;
      kbuf[i] = *reinterpret_cast<const u32x4*>(tile + ((key <= last ? key : last) * st32 + (e < a.d ? e : 0)));
    }
#pragma unroll
    for (int i = 0; i < VP; ++i) {
      const int p = i * 256 + tid, kv0 = p % VN * VK, e = p / VN * 8;
#pragma unroll
      for (int r = 0; r < VK; ++r) {
        const int key = kv0 + r;
        vbuf[i][r] = *reinterpret_cast<const u32x4*>(tile + ((key <= last ? key : last) * st32 + a.d + (e < a.dv ? e : 0)));
      }
    }
  };
  auto stage = [&]() {
#pragma unroll
    for (int i = 0; i < KP; ++i) {
      const int p = i * 256 + tid, key = p / (D / 8), e = (p % (D / 8)) * 8;
      *reinterpret_cast<u32x4*>(&lds_k[key * KS + e]) = e < a.d ? kbuf[i] : zero4;
    }
#pragma unroll
    for (int i = 0; i < VP; ++i) {
      const int p = i * 256 + tid, kv0 = p % VN * VK, e = p / VN * 8;
      if (e < DV) {
#pragma unroll
        for (int r = 0; r < VK; ++r) vbuf[i][r] = e < a.dv ? vbuf[i][r] : zero4;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          bf16xk col;
#pragma unroll
          for (int r = 0; r < VK; ++r) col[r] = __builtin_bit_cast(bf16x8, vbuf[i][r])[j];
          *reinterpret_cast<bf16xk*>(&lds_v[(e + j) * VS + kv0]) = col;
        }
      }
    }
  };

  // FILL: the same tile by way of registers, eight lanes to a row
  u32x4 fresh_k[FILL ? 2 : 1], fresh_v[FILL ? 2 : 1];
  Turn8<HALF> turn_k[FILL ? 2 : 1];
  auto ask_fresh = [&](int k0) {
    const __bf16* pk = static_cast<const __bf16*>(a.k) + b * a.k_sb + (long)g * a.d;
    const __bf16* pv = static_cast<const __bf16*>(a.v) + b * a.v_sb + (long)g * a.dv;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int row = (i * 256 + tid) >> 3, c = (tid & 7) * 8, key = k0 + row <= last_pos ? k0 + row : last_pos;
      const bool old = key < a.pos_host;
      const __bf16* kr = old ? kv + (long)key * a.kv_st : pk + (long)(key - a.pos_host) * a.k_sl;
      const __bf16* vr = old ? kv + (long)key * a.kv_st + a.d : pv + (long)(key - a.pos_host) * a.v_sl;
      fresh_k[i] = *reinterpret_cast<const u32x4*>(kr + c);
      fresh_v[i] = *reinterpret_cast<const u32x4*>(vr + c);
      turn_k[i].load(kr, c, key, a);
    }
  };
  auto settle = [&](int k0, int to) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int row = (i * 256 + tid) >> 3, piece = tid & 7, key = k0 + row;
      if (key >= a.pos_host) {  // (the same in the eight lanes of a row)
        float x[8], ss = 0.f;
        bf16x8 out;
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = to_f32(__builtin_bit_cast(bf16x8, fresh_k[i])[j]);
        turn_k[i].apply(x, piece * 8, a);
#pragma unroll
        for (int j = 0; j < 8; ++j) out[j] = from_f32<__bf16>(x[j]);
        fresh_k[i] = __builtin_bit_cast(u32x4, out);
        if (a.norm_v) {
#pragma unroll
          for (int j = 0; j < 8; ++j) x[j] = to_f32(__builtin_bit_cast(bf16x8, fresh_v[i])[j]);
#pragma unroll
          for (int j = 0; j < 8; ++j) ss = __builtin_fmaf(x[j], x[j], ss);
          const float by = 1.0f / sqrtf(sum8(ss) / (float)a.dv + a.eps);
#pragma unroll
          for (int j = 0; j < 8; ++j) out[j] = from_f32<__bf16>(x[j] * by);
          fresh_v[i] = __builtin_bit_cast(u32x4, out);
        }
        if (key >= first_pos && key <= last_pos) {
          __bf16* fill = const_cast<__bf16*>(kv) + (long)key * a.kv_st + piece * 8;
          *reinterpret_cast<u32x4*>(fill) = fresh_k[i];
          *reinterpret_cast<u32x4*>(fill + a.d) = fresh_v[i];
        }
      }
      __bf16* tile = lds_tiles + to * kDirectTile + row * 64;
      *reinterpret_cast<u32x4*>(tile + (piece ^ (row >> 1 & 7)) * 8) = fresh_k[i];
      *reinterpret_cast<u32x4*>(tile + kTileKeys * 64 + (piece ^ (row >> 1 & 3) * 2) * 8) = fresh_v[i];
    }
  };

  if constexpr (FILL)
    ask_fresh(lo);
  else if constexpr (DIRECT)
    ask(lo, 0);
  // queries: lane holds channels quad*8 + 32 c .. of row l16 (+16): the MFMA's second operand.  Turned and
  // rounded after the first tile of keys has been asked for.
  bf16x8 qf[2][KC];
  int qpos[2];
  const __bf16* qrow[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int row = row_w + t * 16 + l16;
    const int rr = row < n_rows ? row : n_rows - 1;
    int head;
    const int tok = token_of(rr, &head);
    qpos[t] = a.pos_host + tok;
    qrow[t] = static_cast<const __bf16*>(a.q) + b * a.q_sb + tok * a.q_sl + (long)(g * qpk + head) * a.d;
#pragma unroll
    for (int c = 0; c < KC; ++c) {
      const int e = c * 32 + quad * 8;
      qf[t][c] = *reinterpret_cast<const bf16x8*>(qrow[t] + (e < a.d ? e : 0));
    }
  }
  if constexpr (!DIRECT) fetch(lo);
  if (a.rot > 0) {
    constexpr int CB = KC == 3 || (HALF && KC == 2) ? 1 : KC < 4 ? KC : 4;
#pragma unroll
    for (int c0 = 0; c0 < KC; c0 += CB) {
      Turn8<HALF> turn[2][CB];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int c = 0; c < CB; ++c) turn[t][c].load(qrow[t], (c0 + c) * 32 + quad * 8, qpos[t], a);
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int c = 0; c < CB; ++c) {
          float x[8];
#pragma unroll
          for (int j = 0; j < 8; ++j) x[j] = to_f32(qf[t][c0 + c][j]);
          turn[t][c].apply(x, (c0 + c) * 32 + quad * 8, a);
#pragma unroll
          for (int j = 0; j < 8; ++j) qf[t][c0 + c][j] = (__bf16)x[j];
        }
    }
  }
  if (a.scale < 0.f) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int c = 0; c < KC; ++c)
#pragma unroll
        for (int j = 0; j < 8; ++j) qf[t][c][j] = -qf[t][c][j];
  }
  if (D > a.d) {
#pragma unroll
    for (int c = 0; c < KC; ++c)
      if (c * 32 + quad * 8 >= a.d) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int j = 0; j < 8; ++j) qf[t][c][j] = (__bf16)0.f;
      }
  }
  __builtin_amdgcn_sched_barrier(0);  // (the accumulators take their registers from here on)
  f32x4 acc[2][2 * VC];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int i = 0; i < 2 * VC; ++i) acc[t][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run[2] = {-INFINITY, -INFINITY}, l_run[2] = {0.f, 0.f};
  const float scale2 = fabsf(a.scale) * 1.4426950408889634f;  // scores in powers of two; the sign is the queries'
  int place = 0;
  for (int k0 = lo; k0 <= last_pos; k0 += kTileKeys) {
    if constexpr (FILL) {
      settle(k0, place);
      lds_barrier();  // (the reads of this place two tiles ago lie in front of the barrier of the last one)
      if (k0 + kTileKeys <= last_pos) ask_fresh(k0 + kTileKeys);
      __builtin_amdgcn_sched_barrier(0);
    } else if constexpr (DIRECT) {
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_waitcnt(0x0070);  // own loads are there, own reads of the tile before are done
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      if (k0 + kTileKeys <= last_pos) ask(k0 + kTileKeys, place ^ 1);
      __builtin_amdgcn_sched_barrier(0);
    } else {
      __syncthreads();  // every wavefront is done with the tile before
      stage();
      __syncthreads();
      if (k0 + kTileKeys <= last_pos) fetch(k0 + kTileKeys);
    }
    const __bf16* tile_k = lds_tiles + place * kDirectTile;
    const __bf16* tile_v = tile_k + kTileKeys * 64;
    place ^= 1;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      // 32 keys at a time: does any row of this wavefront see one of them, does every row see all?
      const int kh = k0 + h * 32;
      if (kh > wave_hi_tok || kh + 31 <= wave_lo_tok - a.window) continue;
      const bool late = kh + 31 > wave_lo_tok, early = kh <= wave_hi_tok - a.window;  // (of some row)
      f32x4 s[2][2];
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
        for (int t = 0; t < 2; ++t) s[t][kt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < KC; ++c) {
          const bf16x8 kf = DIRECT ? *reinterpret_cast<const bf16x8*>(&tile_k[(h * 32 + kt * 16 + l16) * 64 + ((c * 4 + quad) ^ (l16 >> 1 & 7)) * 8])
                                   : *reinterpret_cast<const bf16x8*>(&lds_k[(h * 32 + kt * 16 + l16) * KS + c * 32 + quad * 8]);
#pragma unroll
          for (int t = 0; t < 2; ++t) s[t][kt] = mfma_bf16(kf, qf[t][c], s[t][kt]);
        }
      }
      bf16x8 pf[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        // (a score out of sight is minus infinity)
        const int d0 = qpos[t] - kh - quad * 4;
        if (late) {
#pragma unroll
          for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int i = 0; i < 4; ++i) s[t][kt][i] = d0 >= kt * 16 + i ? s[t][kt][i] : -INFINITY;
        }
        if (early) {
          const int w0 = d0 - a.window;
#pragma unroll
          for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int i = 0; i < 4; ++i) s[t][kt][i] = w0 < kt * 16 + i ? s[t][kt][i] : -INFINITY;
        }
        float mx = s[t][0][0];
#pragma unroll
        for (int i = 1; i < 8; ++i) mx = fmaxf(mx, s[t][i >> 2][i & 3]);
        if (__any(mx > m_run[t])) {  // (2^8 of slack would save 3 to 10 % of the time, and round the heaviest weight, which is one, like the others)
          mx = max_quads(mx);
          const float m_new = fmaxf(m_run[t], mx);
          // no key seen yet: every weight is 2^-inf = 0
          const float alpha = __builtin_amdgcn_exp2f((m_run[t] - (m_new == -INFINITY ? 0.f : m_new)) * scale2);
          m_run[t] = m_new;
          l_run[t] *= alpha;
#pragma unroll
          for (int i = 0; i < 2 * VC; ++i) acc[t][i] *= alpha;
        }
        const float m2 = m_run[t] == -INFINITY ? 0.f : m_run[t] * scale2;
        float sum = 0.f;
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[t][kt][i], scale2, -m2));
            sum += p;
            pf[t][kt * 4 + i] = (__bf16)p;
          }
        l_run[t] += sum;  // this lane's keys, their weights in 32 bits; the four lane groups are added at the end
      }
#pragma unroll
      for (int i = 0; i < 2 * VC; ++i) {
        bf16x4 v0, v1;
        if constexpr (DIRECT) {
          // lane l16 receives channel l16 of the four keys whose 8 bytes each its group of 16 lanes names
          const int row = quad * 4 + (l16 >> 2);
          const __bf16* vp = &tile_v[(h * 32 + row) * 64 + ((i * 2 + (l16 >> 1 & 1)) ^ (row >> 1 & 3) * 2) * 8 + (l16 & 1) * 4];
          v0 = read_transposed(vp), v1 = read_transposed(vp + 16 * 64);
        } else {
          const __bf16* vp = &lds_v[(i * 16 + l16) * VS + h * 32 + quad * 4];
          v0 = *reinterpret_cast<const bf16x4*>(vp), v1 = *reinterpret_cast<const bf16x4*>(vp + 16);
        }
        const bf16x8 vf = __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
        for (int t = 0; t < 2; ++t) acc[t][i] = mfma_bf16(vf, pf[t], acc[t][i]);
      }
    }
  }
  int row_end = row_w;
  asm volatile("" : "+v"(row_end));  // (where a row goes is worked out again: kept, it would be a register too many)
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    float l = l_run[t];
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    const float inv = a.out_scale / l;
    const int row = row_end + t * 16 + l16;
    int head;
    const int tok = token_of(row, &head);
    if (row < n_rows) {
      __bf16* op = static_cast<__bf16*>(a.o) + b * a.o_sb + tok * a.o_sl + (long)(g * qpk + head) * a.dv;
#pragma unroll
      for (int i = 0; i < 2 * VC; ++i) {
        const int e = i * 16 + quad * 4;
        if (e < a.dv) {
          bf16x4 o;
#pragma unroll
          for (int j = 0; j < 4; ++j) o[j] = (__bf16)(acc[t][i][j] * inv);
          *reinterpret_cast<bf16x4*>(op + e) = o;
        }
      }
    }
  }
}

template <int KC, int VC, bool HALF, bool DIRECT>
__global__ __launch_bounds__(256, KC <= 2 && VC <= 2 ? 4 : KC <= 3 && VC <= 2 ? 3 : KC <= 3 && VC <= 4 ? 2 : 1)
void window_prefill_mfma_kernel(const WindowArgs a) {
  window_prefill_mfma<KC, VC, HALF, DIRECT, false>(a);
}
template <bool HALF> __global__ __launch_bounds__(256, 2) void window_prefill_fill_kernel(const WindowArgs a) {
  window_prefill_mfma<2, 2, HALF, true, true>(a);
}

// ---- prefill, fp32, fp32 MFMA ----
// KB, VB: 64-channel blocks of the key and value sizes (rounded up; channels past the real sizes are zeros).  64 (token, head) rows
// per workgroup, 16 per wavefront, keys and values 32 at a time in LDS for the four.  As in bf16, scores come transposed: the four
// weights of a lane are what the products with the values take, one each, where product j contracts keys j, 4 + j, 8 + j and 12 + j;
// keys and queries give up their channels in the same order, so that a lane reads 16 bytes for four products.
// Bound by the fp32 matrix rate from some thousand rows on and by the chain of one wavefront below.  16 heads on 4, size 64, 129 keys:
// B = 1, L = 777, with the cache write: 17.7 us (a wavefront per query on the vector unit: 70); B = 4, L = 2048: 77 us (661).
constexpr int kF32Keys = 32, kF32Rows = 64;

// What turns channels c .. c + 3 of a row (as Turn8, for either kind of pairs): loaded without a condition, applied later.
struct Turn4 {
  f32x4 cs, sn, partner;  // (interleaved pairs: two angles)
  __device__ __forceinline__ void load(const float* row, int c, int pos, const WindowArgs& a) {
    const bool in = c < a.rot;
    const int half = a.rot / 2;
    const float *cos_t = a.rot > 0 ? a.cos_t : static_cast<const float*>(a.kv), *sin_t = a.rot > 0 ? a.sin_t : static_cast<const float*>(a.kv);
    if (a.half_split) {  // (uniform)
      const long t = in ? (long)pos * half + (c < half ? c : c - half) : 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) cs[j] = cos_t[t + j], sn[j] = sin_t[t + j];
      partner = *reinterpret_cast<const f32x4*>(row + (in ? (c < half ? c + half : c - half) : 0));
    } else {
      const long t = in ? (long)pos * half + c / 2 : 0;
#pragma unroll
      for (int j = 0; j < 2; ++j) cs[j] = cos_t[t + j], sn[j] = sin_t[t + j];
    }
  }
  __device__ __forceinline__ void apply(f32x4& x, int c, const WindowArgs& a) const {
    if (c >= a.rot) return;
    if (a.half_split) {
      const float sgn = c < a.rot / 2 ? -1.f : 1.f;
#pragma unroll
      for (int j = 0; j < 4; ++j) x[j] = x[j] * cs[j] + sgn * partner[j] * sn[j];
    } else {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const float u = x[2 * j], v = x[2 * j + 1];
        x[2 * j] = u * cs[j] - v * sn[j];
        x[2 * j + 1] = v * cs[j] + u * sn[j];
      }
    }
  }
};

// channels c .. c + 3 of a row, turned; c and the rotary size (its half in half-split pairs) multiples of 4
__device__ __forceinline__ f32x4 turned4(const float* row, int c, int pos, const WindowArgs& a) {
  f32x4 x = *reinterpret_cast<const f32x4*>(row + c);
  if (c < a.rot) {
    const int half = a.rot / 2;
    if (a.half_split) {
      const int pair = c < half ? c : c - half;
      const float sgn = c < half ? -1.f : 1.f;
      const f32x4 y = *reinterpret_cast<const f32x4*>(row + (c < half ? c + half : c - half));
      const float *cs = a.cos_t + (long)pos * half + pair, *sn = a.sin_t + (long)pos * half + pair;
#pragma unroll
      for (int j = 0; j < 4; ++j) x[j] = x[j] * cs[j] + sgn * y[j] * sn[j];
    } else {
      const float *cs = a.cos_t + (long)pos * half + c / 2, *sn = a.sin_t + (long)pos * half + c / 2;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const float u = x[2 * j], v = x[2 * j + 1];
        x[2 * j] = u * cs[j] - v * sn[j];
        x[2 * j + 1] = v * cs[j] + u * sn[j];
      }
    }
  }
  return x;
}

// The cache write of fp32 rows in 16-byte pieces: 16 lanes per (token, key/value head).  Element by element, a wavefront per head, it was
// 19.3 us with the attention at B = 1, L = 777, 4 heads of 64, and 88 at B = 4, L = 2048: 18.9 and 81.
__global__ __launch_bounds__(256) void window_kv_write_f32_kernel(const WindowArgs a) {
  const long n_items = (long)a.B * a.L * a.G, item0 = (long)blockIdx.x * 16 + (threadIdx.x >> 4);
  const bool live = item0 < n_items;
  const long item = live ? item0 : n_items - 1, bl = item / a.G;
  const int c0 = (threadIdx.x & 15) * 4, g = (int)(item % a.G), l = (int)(bl % a.L), b = (int)(bl / a.L), pos = a.pos_host + l;
  const float* k = static_cast<const float*>(a.k) + b * a.k_sb + l * a.k_sl + (long)g * a.d;
  const float* v = static_cast<const float*>(a.v) + b * a.v_sb + l * a.v_sl + (long)g * a.dv;
  float* out = static_cast<float*>(a.kv) + b * a.kv_sb + pos * a.kv_st + (long)g * (a.d + a.dv);
  f32x4 x[2], y[2];  // (sizes up to 128)
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int c = c0 + i * 64;
    x[i] = turned4(k, c < a.d ? c : 0, pos, a);
    y[i] = *reinterpret_cast<const f32x4*>(v + (c < a.dv ? c : 0));
#pragma unroll
    for (int j = 0; j < 4; ++j) ss = c < a.dv ? __builtin_fmaf(y[i][j], y[i][j], ss) : ss;
  }
  const float r = a.norm_v ? 1.0f / sqrtf(sum16(ss) / (float)a.dv + a.eps) : 1.0f;
  if (!live) return;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int c = c0 + i * 64;
    if (c < a.d) *reinterpret_cast<f32x4*>(out + c) = x[i];
    if (c < a.dv) *reinterpret_cast<f32x4*>(out + a.d + c) = y[i] * r;
  }
}

// KH: wavefronts to the same 16 rows, which take 32 keys of a tile each and add up what they have in the end.
// FILL: the portion's keys and values are taken as they come, turned and normed on their way to LDS, and left in the cache by the workgroups
// whose tokens they are; nobody reads there what is written.
template <int KB, int VB, int KH, bool FILL>
__global__ __launch_bounds__(256 * KH) void window_prefill_f32_kernel(const WindowArgs a) {
  constexpr int D = KB * 64, DV = VB * 64, KS = D + 4, VS = DV + 4, NT = 256 * KH, KEYS = kF32Keys * KH;
  __shared__ __attribute__((aligned(16))) float lds[KEYS * (KS + VS)];
  float *lds_k = lds, *lds_v = lds + KEYS * KS;
  __shared__ int s_odd[4 * KH];  // values of this tile that are not finite, by the wavefront that staged them
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, quad = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), part = wave >> 2;
  const int b = blockIdx.y / a.G, g = blockIdx.y % a.G, qpk = a.H / a.G, n_rows = a.L * qpk;
  const int r0 = blockIdx.x * kF32Rows, row_w = r0 + (wave & 3) * 16;
  const auto token_of = [&](int row) { return (row < n_rows ? row : n_rows - 1) / qpk; };
  const float* kv = static_cast<const float*>(a.kv) + b * a.kv_sb + (long)g * (a.d + a.dv);
  const int tok = token_of(row_w + l16), pos = a.pos_host + tok;
  const int head = g * qpk + (row_w + l16 < n_rows ? row_w + l16 : n_rows - 1) % qpk;
  const int first = a.pos_host + token_of(r0), last = a.pos_host + token_of(r0 + kF32Rows - 1);
  const int wave_lo = a.pos_host + token_of(row_w), wave_hi = a.pos_host + token_of(row_w + 15);
  const int lo = first - a.window + 1 > 0 ? first - a.window + 1 : 0;

  f32x4 kbuf[2 * KB], vbuf[2 * VB];
  Turn4 turn[FILL ? 2 * KB : 1];
  const float* fresh_k = static_cast<const float*>(a.k) + b * a.k_sb + (long)g * a.d;
  const float* fresh_v = static_cast<const float*>(a.v) + b * a.v_sb + (long)g * a.dv;
  const auto fetch = [&](int k0) {
#pragma unroll
    for (int i = 0; i < 2 * KB; ++i) {
      const int p = i * NT + tid, e = p % (D / 4) * 4, c = e < a.d ? e : 0;
      const int key = k0 + p / (D / 4) <= last ? k0 + p / (D / 4) : last;
      const float* row = kv + (long)key * a.kv_st;
      if constexpr (FILL) {
        row = key < a.pos_host ? row : fresh_k + (long)(key - a.pos_host) * a.k_sl;
        turn[i].load(row, c, key, a);
      }
      kbuf[i] = *reinterpret_cast<const f32x4*>(row + c);
    }
#pragma unroll
    for (int i = 0; i < 2 * VB; ++i) {
      const int p = i * NT + tid, e = p % (DV / 4) * 4, c = e < a.dv ? e : 0;
      const int key = k0 + p / (DV / 4) <= last ? k0 + p / (DV / 4) : last;
      const float* row = kv + (long)key * a.kv_st + a.d;
      if constexpr (FILL) row = key < a.pos_host ? row : fresh_v + (long)(key - a.pos_host) * a.v_sl;
      vbuf[i] = *reinterpret_cast<const f32x4*>(row + c);
    }
  };
  // what `fetch` brought of the tile at k0, as the cache has it
  const auto settle = [&](int k0) {
    if constexpr (FILL) {
      float* fill = const_cast<float*>(kv);
#pragma unroll
      for (int i = 0; i < 2 * KB; ++i) {
        const int p = i * NT + tid, e = p % (D / 4) * 4, key = k0 + p / (D / 4);
        if (key >= a.pos_host && e < a.d) {
          turn[i].apply(kbuf[i], e, a);
          if (key >= first && key <= last) *reinterpret_cast<f32x4*>(fill + (long)key * a.kv_st + e) = kbuf[i];
        }
      }
#pragma unroll
      for (int i = 0; i < 2 * VB; ++i) {
        const int p = i * NT + tid, e = p % (DV / 4) * 4, key = k0 + p / (DV / 4);
        float ss = 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j) ss = e < a.dv ? __builtin_fmaf(vbuf[i][j], vbuf[i][j], ss) : ss;
        ss = sum16(ss);
        if (VB == 2) ss += __shfl_xor(ss, 16, 64);
        const float r = a.norm_v && key >= a.pos_host ? 1.0f / sqrtf(ss / (float)a.dv + a.eps) : 1.0f;
        vbuf[i] *= r;
        if (key >= first && key <= last && e < a.dv) *reinterpret_cast<f32x4*>(fill + (long)key * a.kv_st + a.d + e) = vbuf[i];
      }
    }
  };
  fetch(lo);
  f32x4 qf[4 * KB];
  const float sign = a.scale < 0.f ? -1.f : a.scale == 0.f ? 0.f : 1.f;
  {
    const float* q = static_cast<const float*>(a.q) + b * a.q_sb + tok * a.q_sl + (long)head * a.d;
#pragma unroll
    for (int c = 0; c < 4 * KB; ++c) {
      const int e = c * 16 + quad * 4;
      qf[c] = turned4(q, e < a.d ? e : 0, pos, a);
#pragma unroll
      for (int j = 0; j < 4; ++j) qf[c][j] = e < a.d ? sign * qf[c][j] : 0.f;
    }
  }
  f32x4 acc[VB][4];  // channels vb * 64 + (quad * 4 + i) * 4 + c of row l16 in [vb][c][i]
#pragma unroll
  for (int vb = 0; vb < VB; ++vb)
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[vb][c] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;
  // Powers of two of the differences, which are exact where they count; the sign is the queries', and so is a scale of zero (a key
  // out of sight stays at minus infinity, an infinite one is no number).
  const float scale2 = a.scale == 0.f ? 1.f : fabsf(a.scale) * 1.4426950408889634f;

  for (int t0 = lo; t0 <= last; t0 += KEYS) {
    settle(t0);
    __syncthreads();  // every wavefront is done with the tile before
    bool odd = false;
#pragma unroll
    for (int i = 0; i < 2 * KB; ++i) {
      const int p = i * NT + tid, key = p / (D / 4), e = p % (D / 4) * 4;
      *reinterpret_cast<f32x4*>(&lds_k[key * KS + e]) = e < a.d ? kbuf[i] : f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int i = 0; i < 2 * VB; ++i) {
      const int p = i * NT + tid, key = p / (DV / 4), e = p % (DV / 4) * 4;
      const f32x4 x = vbuf[i];
      const float zero = (x[0] * 0.f + x[1] * 0.f) + (x[2] * 0.f + x[3] * 0.f);
      odd |= !(zero == 0.f);
      *reinterpret_cast<f32x4*>(&lds_v[key * VS + e]) = e < a.dv ? x : f32x4{0.f, 0.f, 0.f, 0.f};
    }
    odd = __any(odd);
    if (lane == 0) s_odd[wave] = odd;
    __syncthreads();
    if (t0 + KEYS <= last) fetch(t0 + KEYS);
    const int k0 = t0 + part * kF32Keys;
    const float *tile_k = lds_k + part * kF32Keys * KS, *tile_v = lds_v + part * kF32Keys * VS;
    if (k0 > wave_hi || k0 + kF32Keys - 1 <= wave_lo - a.window) continue;
    const bool all = k0 + kF32Keys - 1 <= wave_lo && k0 > wave_hi - a.window;  // does every row see every key?
    const bool kt_in[2] = {k0 + 15 > wave_lo - a.window, k0 + 16 <= wave_hi};  // does any see one of these 16?
    f32x4 s[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
      if (kt_in[kt]) {
        f32x4 half = {0.f, 0.f, 0.f, 0.f};  // (two sums of half the channels each round less than one)
#pragma unroll
        for (int c = 0; c < 4 * KB; c += 2) {
          const f32x4 k0f = *reinterpret_cast<const f32x4*>(&tile_k[(kt * 16 + l16) * KS + c * 16 + quad * 4]);
          const f32x4 k1f = *reinterpret_cast<const f32x4*>(&tile_k[(kt * 16 + l16) * KS + (c + 1) * 16 + quad * 4]);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            s[kt] = mfma_f32(k0f[j], qf[c][j], s[kt]);
            half = mfma_f32(k1f[j], qf[c + 1][j], half);
          }
        }
        s[kt] += half;
      }
    const int d0 = pos - k0 - quad * 4;
    float mx = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float sc = s[kt][i];
        if (!all) sc = (unsigned)(d0 - kt * 16 - i) < (unsigned)a.window ? sc : -INFINITY;
        s[kt][i] = sc;
        mx = fmaxf(mx, sc);
      }
    mx = max_quads(mx);
    if (__any(mx > m_run)) {
      const float m_new = fmaxf(m_run, mx);
      // no key seen yet: every weight is 2^-inf = 0
      const float alpha = __builtin_amdgcn_exp2f((m_run - (m_new == -INFINITY ? 0.f : m_new)) * scale2);
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int vb = 0; vb < VB; ++vb)
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[vb][c] *= alpha;
    }
    const float m2 = m_run == -INFINITY ? 0.f : m_run;
    float sum = 0.f;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[kt][i] = __builtin_amdgcn_exp2f((s[kt][i] - m2) * scale2);
        sum += s[kt][i];
      }
    l_run += sum;  // this lane's keys; the four quads are added at the end
    int odd_any = 0;
#pragma unroll
    for (int w = 0; w < 4 * KH; ++w) odd_any |= s_odd[w];
    if (all || !odd_any) {
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
        if (kt_in[kt]) {
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int vb = 0; vb < VB; ++vb) {
              const f32x4 vf = *reinterpret_cast<const f32x4*>(&tile_v[(kt * 16 + quad * 4 + j) * VS + vb * 64 + l16 * 4]);
#pragma unroll
              for (int c = 0; c < 4; ++c) acc[vb][c] = mfma_f32(vf[c], s[kt][j], acc[vb][c]);
            }
        }
    } else {
      // a weight of zero would not keep an infinity or NaN out of the rows that do not see its key
      for (int key = 0; key < kF32Keys; ++key) {
        float mine = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) mine = (key >> 4) * 4 + (key & 3) == e ? s[e / 4][e % 4] : mine;
        const float p = __shfl(mine, (key >> 2 & 3) * 16 + l16);
        if ((unsigned)(pos - k0 - key) < (unsigned)a.window) {
#pragma unroll
          for (int vb = 0; vb < VB; ++vb)
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
              for (int i = 0; i < 4; ++i)
                acc[vb][c][i] = __builtin_fmaf(p, tile_v[key * VS + vb * 64 + (quad * 4 + i) * 4 + c], acc[vb][c][i]);
        }
      }
    }
  }
  if constexpr (KH > 1) {
    // the other wavefront's sums of the same rows, both taken to the larger of their largest scores
    constexpr int N = 16 * VB + 2;
    static_assert(KH == 2 && N * 256 <= KEYS * (KS + VS), "room for one half");
    __syncthreads();
    float* at = lds + (wave & 3) * 64 + lane;
    if (part == 1) {
      at[0] = m_run, at[256] = l_run;
#pragma unroll
      for (int n = 0; n < 16 * VB; ++n) at[(n + 2) * 256] = acc[n / 16][n / 4 % 4][n % 4];
    }
    __syncthreads();
    if (part == 1) return;
    const float other = at[0], m = fmaxf(m_run, other), m0 = m == -INFINITY ? 0.f : m;
    const float mine = __builtin_amdgcn_exp2f((m_run - m0) * scale2), theirs = __builtin_amdgcn_exp2f((other - m0) * scale2);
    l_run = l_run * mine + at[256] * theirs;
#pragma unroll
    for (int n = 0; n < 16 * VB; ++n) acc[n / 16][n / 4 % 4][n % 4] = acc[n / 16][n / 4 % 4][n % 4] * mine + at[(n + 2) * 256] * theirs;
  }
  float l = l_run;
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  const float inv = a.out_scale / l;
  if (row_w + l16 < n_rows) {
    float* o = static_cast<float*>(a.o) + b * a.o_sb + tok * a.o_sl + (long)head * a.dv;
#pragma unroll
    for (int vb = 0; vb < VB; ++vb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int e = vb * 64 + (quad * 4 + i) * 4;
        if (e < a.dv) *reinterpret_cast<f32x4*>(o + e) = f32x4{acc[vb][0][i], acc[vb][1][i], acc[vb][2][i], acc[vb][3][i]} * inv;
      }
  }
}

// ---- prefill, any element type and any sizes: one wavefront per (token, query head) ----
constexpr int kAnyMaxDim = 512;  // largest key / value size

template <typename T>
__global__ __launch_bounds__(64) void window_prefill_any_kernel(const WindowArgs a) {
  __shared__ float qs[kAnyMaxDim];
  __shared__ float ps[64];
  const int lane = threadIdx.x, l = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int g = h / (a.H / a.G), pos = a.pos_host + l;
  const T* q = static_cast<const T*>(a.q) + b * a.q_sb + l * a.q_sl + (long)h * a.d;
  const T* kv = static_cast<const T*>(a.kv) + b * a.kv_sb + (long)g * (a.d + a.dv);
  for (int c = lane; c < a.d; c += 64) qs[c] = round_to<T>(rotated(q, c, pos, a));
  float acc[kAnyMaxDim / 64];
#pragma unroll
  for (int i = 0; i < kAnyMaxDim / 64; ++i) acc[i] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;
  const int lo = pos - a.window + 1 > 0 ? pos - a.window + 1 : 0;
  __syncthreads();
  for (int k0 = lo; k0 <= pos; k0 += 64) {
    const int key = k0 + lane;
    float s = -INFINITY;
    if (key <= pos) {
      const T* kr = kv + (long)key * a.kv_st;
      float dot = 0.f;
      for (int c = 0; c < a.d; ++c) dot = __builtin_fmaf(qs[c], to_f32(kr[c]), dot);
      s = dot * a.scale;
    }
    float mx = s;
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) mx = fmaxf(mx, __shfl_xor(mx, m, 64));
    const float m_new = fmaxf(m_run, mx);
    const float alpha = expf(m_run - m_new), p = expf(s - m_new);
    m_run = m_new;
    l_run = l_run * alpha + wave_sum(p);
    __syncthreads();
    ps[lane] = p;
    __syncthreads();
    const int n = pos - k0 + 1 < 64 ? pos - k0 + 1 : 64;
#pragma unroll
    for (int i = 0; i < kAnyMaxDim / 64; ++i) {
      const int c = i * 64 + lane;
      if (c < a.dv) {
        float v = acc[i] * alpha;
        for (int j = 0; j < n; ++j) v = __builtin_fmaf(ps[j], to_f32(kv[(long)(k0 + j) * a.kv_st + a.d + c]), v);
        acc[i] = v;
      }
    }
  }
  T* o = static_cast<T*>(a.o) + b * a.o_sb + l * a.o_sl + (long)h * a.dv;
  const float inv = a.out_scale / l_run;
#pragma unroll
  for (int i = 0; i < kAnyMaxDim / 64; ++i) {
    const int c = i * 64 + lane;
    if (c < a.dv) o[c] = from_f32<T>(acc[i] * inv);
  }
}

// ---- one token per sequence ----
constexpr int kStepThreads = 256;
constexpr int kStepKeys = 256;  // keys per round of the running softmax

template <typename T, int N> struct RawPiece {
  typedef typename Pack<T>::type type;
  static __device__ __forceinline__ float get(type x, int i) { return to_f32(x[i]); }
};
template <typename T> struct RawPiece<T, 1> {
  typedef T type;
  static __device__ __forceinline__ float get(type x, int) { return to_f32(x); }
};

// QT: query heads of the group served together (the group is walked QT heads at a time).
// VEC: 16-byte pieces of the rows (sizes and strides multiples of the piece); otherwise element by element.
template <typename T, int QT, bool VEC>
__global__ __launch_bounds__(kStepThreads) void window_step_kernel(const WindowArgs a, int part_floats) {
  constexpr int N = VEC ? Pack<T>::kN : 1;
  extern __shared__ float smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int b = blockIdx.x / a.G, g = blockIdx.x % a.G;
  const int qpk = a.H / a.G;
  const int pos = row_pos(a.pos, a.pos_host, b);
  if (pos < 0 || pos >= a.S || (a.rot > 0 && pos >= a.n_pos)) return;  // a position the cache does not hold
  float* qs = smem;                        // [QT][d]
  float* sc = qs + QT * a.d;               // [QT][kStepKeys]
  float* stat = sc + QT * kStepKeys;       // [3][QT]: running maximum, running sum, rescale of the current keys
  float* part = stat + 3 * QT;             // [QT][parts][vp2 * N], partial outputs
  float* knew = part + part_floats;        // [d] and [dv]: the row of the new token, as the cache holds it
  float* vnew = knew + a.d;
  const T* k = static_cast<const T*>(a.k) + b * a.k_sb + (long)g * a.d;
  const T* v = static_cast<const T*>(a.v) + b * a.v_sb + (long)g * a.dv;
  T* kv = static_cast<T*>(a.kv) + b * a.kv_sb + (long)g * (a.d + a.dv);
  const int lo = pos - a.window + 1 > 0 ? pos - a.window + 1 : 0;
  // lanes per key: the smallest power of two that covers the row in N-element pieces, 64 at most
  const int pieces = (a.d + N - 1) / N;
  int lpk = 1;
  while (lpk < pieces && lpk < 64) lpk <<= 1;
  const int keys_at_once = kStepThreads / lpk, my_key = tid / lpk, my_piece = tid % lpk;
  // lanes per value row, likewise; then the partial sums that are left for LDS
  int vp2 = 1;
  while (vp2 * N < a.dv) vp2 <<= 1;  // <= kStepThreads
  const int v_groups = kStepThreads / vp2, my_vp = tid % vp2, my_vg = tid / vp2;
  const int parts = vp2 < 64 ? kStepThreads / 64 : v_groups, my_part = vp2 < 64 ? wave : my_vg;
  const bool v_in = my_vp * N < a.dv;
  constexpr int KU = 4;  // rows whose loads are in flight together
  typedef typename RawPiece<T, N>::type raw_t;
  auto load_row = [&](int j, int n, int first, int piece, int k0) -> raw_t {
    return *reinterpret_cast<const raw_t*>(kv + (long)(k0 + (j < n ? j : n - 1)) * a.kv_st + first + piece * N);
  };
  // the first rows of the cache are asked for before anything else; the new token's row is not in it yet
  // and is taken from LDS
  const int n_first = pos - lo + 1 < kStepKeys ? pos - lo + 1 : kStepKeys;
  const int kp = my_piece < pieces ? my_piece : 0, vp = v_in ? my_vp : 0;
  raw_t xk[KU], xv[KU];
#pragma unroll
  for (int u = 0; u < KU; ++u) xk[u] = load_row(u * keys_at_once + my_key, n_first, 0, kp, lo);
#pragma unroll
  for (int u = 0; u < KU; ++u) xv[u] = load_row(u * v_groups + my_vg, n_first, a.d, vp, lo);
  {
    T* out = kv + (long)pos * a.kv_st;
    if (wave == 0) {
      float ss = 0.f;
      for (int c = lane; c < a.dv; c += 64) ss = __builtin_fmaf(to_f32(v[c]), to_f32(v[c]), ss);
      const float r = a.norm_v ? 1.0f / sqrtf(wave_sum(ss) / (float)a.dv + a.eps) : 1.0f;
      for (int c = lane; c < a.dv; c += 64) {
        const T x = from_f32<T>(to_f32(v[c]) * r);
        out[a.d + c] = x;
        vnew[c] = to_f32(x);
      }
    } else {
      for (int c = tid - 64; c < a.d; c += kStepThreads - 64) {
        const T x = from_f32<T>(rotated(k, c, pos, a));
        out[c] = x;
        knew[c] = to_f32(x);
      }
    }
  }

  for (int h0 = 0; h0 < qpk; h0 += QT) {
    if (h0 > 0) __syncthreads();  // the round before is done with LDS
    for (int i = tid; i < QT * a.d; i += kStepThreads) {
      const int hh = i / a.d, c = i % a.d;
      const int h = g * qpk + (h0 + hh < qpk ? h0 + hh : h0);
      const T* q = static_cast<const T*>(a.q) + b * a.q_sb + (long)h * a.d;
      qs[i] = round_to<T>(rotated(q, c, pos, a));
    }
    if (tid < QT) {
      stat[tid] = -INFINITY;
      stat[QT + tid] = 0.f;
    }
    __syncthreads();
    float qr[QT][N];  // this lane's piece of every query
#pragma unroll
    for (int hh = 0; hh < QT; ++hh)
#pragma unroll
      for (int i = 0; i < N; ++i) qr[hh][i] = my_piece < pieces ? qs[hh * a.d + (my_piece < pieces ? my_piece : 0) * N + i] : 0.f;
    float acc[QT][N];
#pragma unroll
    for (int hh = 0; hh < QT; ++hh)
#pragma unroll
      for (int i = 0; i < N; ++i) acc[hh][i] = 0.f;
    for (int k0 = lo; k0 <= pos; k0 += kStepKeys) {
      const int n = pos - k0 + 1 < kStepKeys ? pos - k0 + 1 : kStepKeys;
      if (k0 > lo) __syncthreads();
      // the pieces of row j as floats; the last row of all is the new token's
      auto floats = [&](raw_t x, const float* fresh, int piece, int j, float (&f)[N]) {
        const bool is_new = k0 + j == pos;
#pragma unroll
        for (int i = 0; i < N; ++i) {
          const float nv = fresh[piece * N + i], ov = RawPiece<T, N>::get(x, i);
          f[i] = is_new ? nv : ov;
        }
      };
      const bool first = h0 == 0 && k0 == lo;
      for (int j0 = 0; j0 < n; j0 += KU * keys_at_once) {
        if (!first || j0 > 0) {
#pragma unroll
          for (int u = 0; u < KU; ++u) xk[u] = load_row(j0 + u * keys_at_once + my_key, n, 0, kp, k0);
        }
#pragma unroll
        for (int u = 0; u < KU; ++u) {
          const int j = j0 + u * keys_at_once + my_key;
          float f[N];
          floats(xk[u], knew, kp, j, f);
          float dot[QT];
#pragma unroll
          for (int hh = 0; hh < QT; ++hh) {
            dot[hh] = 0.f;
#pragma unroll
            for (int i = 0; i < N; ++i) dot[hh] = __builtin_fmaf(f[i], qr[hh][i], dot[hh]);
          }
          for (int p = my_piece + lpk; p < pieces; p += lpk) {  // rows of more than 64 pieces
            float y[N];
            floats(load_row(j, n, 0, p, k0), knew, p, j, y);
#pragma unroll
            for (int hh = 0; hh < QT; ++hh)
#pragma unroll
              for (int i = 0; i < N; ++i) dot[hh] = __builtin_fmaf(y[i], qs[hh * a.d + p * N + i], dot[hh]);
          }
#pragma unroll
          for (int hh = 0; hh < QT; ++hh) {
            if (lpk == 8) {
              dot[hh] = sum8(dot[hh]);
            } else if (lpk == 16) {
              dot[hh] = sum16(dot[hh]);
            } else {
              for (int m = 1; m < lpk; m <<= 1) dot[hh] += __shfl_xor(dot[hh], m, 64);
            }
            if (my_piece == 0 && j < n) sc[hh * kStepKeys + j] = dot[hh] * a.scale;
          }
        }
      }
      if (!first) {
        // the first value rows are on their way during the softmax
#pragma unroll
        for (int u = 0; u < KU; ++u) xv[u] = load_row(my_vg + u * v_groups, n, a.d, vp, k0);
      }
      __syncthreads();
      for (int hh = wave; hh < QT; hh += kStepThreads / 64) {
        float s[kStepKeys / 64], mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < kStepKeys / 64; ++i) {
          const int j = i * 64 + lane;
          s[i] = j < n ? sc[hh * kStepKeys + j] : -INFINITY;
          mx = fmaxf(mx, s[i]);
        }
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1) mx = fmaxf(mx, __shfl_xor(mx, m, 64));
        const float m_old = stat[hh], m_new = fmaxf(m_old, mx);
        float sum = 0.f;
#pragma unroll
        for (int i = 0; i < kStepKeys / 64; ++i) {
          const float p = expf(s[i] - m_new);
          sc[hh * kStepKeys + i * 64 + lane] = p;
          sum += p;
        }
        sum = wave_sum(sum);
        const float alpha = expf(m_old - m_new);
        if (lane == 0) {
          stat[hh] = m_new;
          stat[QT + hh] = stat[QT + hh] * alpha + sum;
          stat[2 * QT + hh] = alpha;
        }
      }
      __syncthreads();
      if (k0 > lo) {
#pragma unroll
        for (int hh = 0; hh < QT; ++hh)
#pragma unroll
          for (int i = 0; i < N; ++i) acc[hh][i] *= stat[2 * QT + hh];
      }
      for (int j0 = my_vg; j0 < n; j0 += KU * v_groups) {
        if (j0 != my_vg) {
#pragma unroll
          for (int u = 0; u < KU; ++u) xv[u] = load_row(j0 + u * v_groups, n, a.d, vp, k0);
        }
#pragma unroll
        for (int u = 0; u < KU; ++u) {
          const int j = j0 + u * v_groups;
          float f[N];
          floats(xv[u], vnew, vp, j, f);
#pragma unroll
          for (int hh = 0; hh < QT; ++hh) {
            const float p = j < n ? sc[hh * kStepKeys + j] : 0.f;
#pragma unroll
            for (int i = 0; i < N; ++i) acc[hh][i] = j < n ? __builtin_fmaf(p, f[i], acc[hh][i]) : acc[hh][i];
          }
        }
      }
    }
#pragma unroll
    for (int hh = 0; hh < QT; ++hh) {
      for (int m = vp2; m < 64; m <<= 1) {
#pragma unroll
        for (int i = 0; i < N; ++i) acc[hh][i] += __shfl_xor(acc[hh][i], m, 64);
      }
      if (vp2 >= 64 || lane < vp2) {
#pragma unroll
        for (int i = 0; i < N; ++i) part[((hh * parts + my_part) * vp2 + my_vp) * N + i] = acc[hh][i];
      }
    }
    __syncthreads();
    for (int i = tid; i < QT * a.dv; i += kStepThreads) {
      const int hh = i / a.dv, c = i % a.dv;
      if (h0 + hh < qpk) {
        float s = 0.f;
        for (int p = 0; p < parts; ++p) s += part[(hh * parts + p) * vp2 * N + c];
        T* o = static_cast<T*>(a.o) + b * a.o_sb + (long)(g * qpk + h0 + hh) * a.dv;
        o[c] = from_f32<T>(s * (a.out_scale / stat[QT + hh]));
      }
    }
  }
}

// The same for bf16 rows of whole 16-byte pieces: queries, the new key and the new value are turned and
// normalised in the registers of the lanes that use them, the new token starts the running softmax, and the
// cached keys before it follow, so that everything the launch reads is asked for at its start and a window
// of w needs w - 1 rows.  Products of queries and keys are dot-product instructions on bf16 pairs.
// LPK, VP2: lanes per key row and per value row (powers of two), 0: whatever the sizes ask for.
template <int QT, bool HALF, int LPK, int VP2>
__global__ __launch_bounds__(kStepThreads) void window_step_vec_kernel(const WindowArgs a) {
  constexpr int N = 8, KU = 4;
  extern __shared__ float smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int b = blockIdx.x / a.G, g = blockIdx.x % a.G;
  const int qpk = a.H / a.G;
  const int pos = row_pos(a.pos, a.pos_host, b);
  if (pos < 0 || pos >= a.S || (a.rot > 0 && pos >= a.n_pos)) return;  // a position the cache does not hold
  float* sc = smem;                   // [QT][kStepKeys]
  float* stat = sc + QT * kStepKeys;  // [3][QT]: running maximum, running sum, rescale of the current keys
  float* part = stat + 3 * QT;        // [QT][parts][vp2 * 8], partial outputs
  const __bf16* k = static_cast<const __bf16*>(a.k) + b * a.k_sb + (long)g * a.d;
  const __bf16* v = static_cast<const __bf16*>(a.v) + b * a.v_sb + (long)g * a.dv;
  __bf16* kv = static_cast<__bf16*>(a.kv) + b * a.kv_sb + (long)g * (a.d + a.dv);
  const int lo = pos - a.window + 1 > 0 ? pos - a.window + 1 : 0;
  const int old = pos - lo;  // cached keys this token sees
  int lpk = LPK, vp2 = VP2;
  if constexpr (LPK == 0) {
    lpk = 1;
    while (lpk * N < a.d) lpk <<= 1;
  }
  if constexpr (VP2 == 0) {
    vp2 = 1;
    while (vp2 * N < a.dv) vp2 <<= 1;
  }
  const int keys_at_once = kStepThreads / lpk, my_key = tid / lpk, my_piece = tid % lpk;
  const int v_groups = kStepThreads / vp2, my_vp = tid % vp2, my_vg = tid / vp2;
  const int parts = kStepThreads / 64;
  const bool k_in = my_piece * N < a.d, v_in = my_vp * N < a.dv;
  const int ke = k_in ? my_piece * N : 0, ve = v_in ? my_vp * N : 0;
  const int st32 = (int)a.kv_st;
  auto row = [&](int k0, int j, int n) { return kv + (long)k0 * a.kv_st + (n > 0 ? (j < n ? j : n - 1) : 0) * st32; };

  const int n_first = old < kStepKeys ? old : kStepKeys;
  bf16x8 xk[KU], xv[KU], qraw[QT];
#pragma unroll
  for (int u = 0; u < KU; ++u) xk[u] = *reinterpret_cast<const bf16x8*>(row(lo, u * keys_at_once + my_key, n_first) + ke);
#pragma unroll
  for (int u = 0; u < KU; ++u) xv[u] = *reinterpret_cast<const bf16x8*>(row(lo, u * v_groups + my_vg, n_first) + a.d + ve);
  auto q_row = [&](int hh) { return static_cast<const __bf16*>(a.q) + b * a.q_sb + (long)(g * qpk + (hh < qpk ? hh : qpk - 1)) * a.d; };
#pragma unroll
  for (int hh = 0; hh < QT; ++hh) qraw[hh] = *reinterpret_cast<const bf16x8*>(q_row(hh) + ke);
  const bf16x8 knew_raw = *reinterpret_cast<const bf16x8*>(k + ke), vnew_raw = *reinterpret_cast<const bf16x8*>(v + ve);
  Turn8<HALF> turn;
  turn.load(k, ke, pos, a);

  // the new value: normalised by the lanes that share the row
  float vn[N];
  {
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      vn[i] = v_in ? to_f32(vnew_raw[i]) : 0.f;
      ss = __builtin_fmaf(vn[i], vn[i], ss);
    }
    if constexpr (VP2 == 8) {
      ss = sum8(ss);
    } else if constexpr (VP2 == 16) {
      ss = sum16(ss);
    } else {
      for (int m = 1; m < vp2; m <<= 1) ss += __shfl_xor(ss, m, 64);
    }
    const float r = a.norm_v ? 1.0f / sqrtf(ss / (float)a.dv + a.eps) : 1.0f;
    bf16x8 o;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      o[i] = (__bf16)(vn[i] * r);
      vn[i] = to_f32(o[i]);
    }
    if (my_vg == 0 && v_in) *reinterpret_cast<bf16x8*>(kv + (long)pos * a.kv_st + a.d + ve) = o;
  }
  typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
  auto turned = [&](bf16x8 raw, const Turn8<HALF>& t) -> u32x4 {
    float x[N];
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = to_f32(raw[i]);
    t.apply(x, ke, a);
    bf16x8 y;
#pragma unroll
    for (int i = 0; i < N; ++i) y[i] = (__bf16)(k_in ? x[i] : 0.f);
    return __builtin_bit_cast(u32x4, y);
  };
  const u32x4 knew = turned(knew_raw, turn);
  if (my_key == 0 && k_in) *reinterpret_cast<u32x4*>(kv + (long)pos * a.kv_st + ke) = knew;
  auto dot8 = [](u32x4 x, u32x4 y) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t xi = x[i], yi = y[i];  // (a bit cast of a vector's element as such takes element 0)
      s = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, xi), __builtin_bit_cast(bf16x2, yi), s, false);
    }
    return s;
  };
  auto over_pieces = [&](float x) {
    if constexpr (LPK == 8) {
      x = sum8(x);
    } else if constexpr (LPK == 16) {
      x = sum16(x);
    } else {
      for (int m = 1; m < lpk; m <<= 1) x += __shfl_xor(x, m, 64);
    }
    return x;
  };

  for (int h0 = 0; h0 < qpk; h0 += QT) {
    if (h0 > 0) __syncthreads();  // the round before is done with LDS
    u32x4 q[QT];
    Turn8<HALF> tq = turn;
    if (h0 > 0) {
#pragma unroll
      for (int hh = 0; hh < QT; ++hh) qraw[hh] = *reinterpret_cast<const bf16x8*>(q_row(h0 + hh) + ke);
    }
#pragma unroll
    for (int hh = 0; hh < QT; ++hh) {
      if constexpr (HALF)
        load_vec<__bf16, 8>(q_row(h0 + hh) + (ke < a.rot ? (ke < a.rot / 2 ? ke + a.rot / 2 : ke - a.rot / 2) : 0), tq.partner);
      q[hh] = turned(qraw[hh], tq);
    }
    // the new token: maximum = its score, weight 1
    float s_new[QT], acc[QT][N];
#pragma unroll
    for (int hh = 0; hh < QT; ++hh) {
      s_new[hh] = over_pieces(dot8(knew, q[hh])) * a.scale;
#pragma unroll
      for (int i = 0; i < N; ++i) acc[hh][i] = my_vg == 0 ? vn[i] : 0.f;
      if (tid == 0) {
        stat[hh] = s_new[hh];
        stat[QT + hh] = 1.f;
      }
    }
    for (int k0 = lo; k0 < pos; k0 += kStepKeys) {
      const int n = pos - k0 < kStepKeys ? pos - k0 : kStepKeys;
      const bool first = h0 == 0 && k0 == lo;
      if (k0 > lo) __syncthreads();
      for (int j0 = 0; j0 < n; j0 += KU * keys_at_once) {
        if (!first || j0 > 0) {
#pragma unroll
          for (int u = 0; u < KU; ++u) xk[u] = *reinterpret_cast<const bf16x8*>(row(k0, j0 + u * keys_at_once + my_key, n) + ke);
        }
#pragma unroll
        for (int u = 0; u < KU; ++u) {
          const int j = j0 + u * keys_at_once + my_key;
#pragma unroll
          for (int hh = 0; hh < QT; ++hh) {
            const float s = over_pieces(dot8(__builtin_bit_cast(u32x4, xk[u]), q[hh]));
            if (my_piece == 0 && j < n) sc[hh * kStepKeys + j] = s * a.scale;
          }
        }
      }
      if (!first) {
        // the first value rows are on their way during the softmax
#pragma unroll
        for (int u = 0; u < KU; ++u) xv[u] = *reinterpret_cast<const bf16x8*>(row(k0, u * v_groups + my_vg, n) + a.d + ve);
      }
      __syncthreads();
      for (int hh = wave; hh < QT; hh += kStepThreads / 64) {
        float s[kStepKeys / 64], mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < kStepKeys / 64; ++i) {
          const int j = i * 64 + lane;
          const float x = sc[hh * kStepKeys + j];
          s[i] = j < n ? x : -INFINITY;
          mx = fmaxf(mx, s[i]);
        }
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1) mx = fmaxf(mx, __shfl_xor(mx, m, 64));
        const float m_old = stat[hh], m_new = fmaxf(m_old, mx);
        float sum = 0.f;
#pragma unroll
        for (int i = 0; i < kStepKeys / 64; ++i) {
          const float p = exp_f(s[i] - m_new);
          sc[hh * kStepKeys + i * 64 + lane] = p;
          sum += p;
        }
        sum = wave_sum(sum);
        const float alpha = exp_f(m_old - m_new);
        if (lane == 0) {
          stat[hh] = m_new;
          stat[QT + hh] = stat[QT + hh] * alpha + sum;
          stat[2 * QT + hh] = alpha;
        }
      }
      __syncthreads();
#pragma unroll
      for (int hh = 0; hh < QT; ++hh) {
        const float alpha = stat[2 * QT + hh];
#pragma unroll
        for (int i = 0; i < N; ++i) acc[hh][i] *= alpha;
      }
      for (int j0 = my_vg; j0 < n; j0 += KU * v_groups) {
        if (j0 != my_vg) {
#pragma unroll
          for (int u = 0; u < KU; ++u) xv[u] = *reinterpret_cast<const bf16x8*>(row(k0, j0 + u * v_groups, n) + a.d + ve);
        }
#pragma unroll
        for (int u = 0; u < KU; ++u) {
          const int j = j0 + u * v_groups;
#pragma unroll
          for (int hh = 0; hh < QT; ++hh) {
            const float p = j < n ? sc[hh * kStepKeys + (j < n ? j : 0)] : 0.f;
#pragma unroll
            for (int i = 0; i < N; ++i) acc[hh][i] = __builtin_fmaf(p, to_f32(xv[u][i]), acc[hh][i]);
          }
        }
      }
    }
#pragma unroll
    for (int hh = 0; hh < QT; ++hh) {
      if constexpr (VP2 != 0) {
#pragma unroll
        for (int m = VP2; m < 64; m <<= 1)
#pragma unroll
          for (int i = 0; i < N; ++i) acc[hh][i] += __shfl_xor(acc[hh][i], m, 64);
      } else {
        for (int m = vp2; m < 64; m <<= 1) {
#pragma unroll
          for (int i = 0; i < N; ++i) acc[hh][i] += __shfl_xor(acc[hh][i], m, 64);
        }
      }
      if (lane < vp2) {
#pragma unroll
        for (int i = 0; i < N; ++i) part[((hh * parts + wave) * vp2 + my_vp) * N + i] = acc[hh][i];
      }
    }
    __syncthreads();
#pragma unroll
    for (int hh = 0; hh < QT; ++hh) {
      if (h0 + hh < qpk) {
        const float inv = a.out_scale / stat[QT + hh];
        for (int c = tid; c < a.dv; c += kStepThreads) {
          float s = 0.f;
#pragma unroll
          for (int p = 0; p < kStepThreads / 64; ++p) s += part[(hh * parts + p) * vp2 * N + c];
          static_cast<__bf16*>(a.o)[b * a.o_sb + (long)(g * qpk + h0 + hh) * a.dv + c] = (__bf16)(s * inv);
        }
      }
    }
  }
}

template <bool HALF, int LPK, int VP2> void launch_window_step_lanes(const WindowArgs& a, int vp2, hipStream_t s) {
  const int qpk = a.H / a.G;
  const dim3 grid((unsigned)(a.B * a.G)), block(kStepThreads);
  auto bytes = [&](int qt) { return (size_t)qt * (kStepKeys + 3 + kStepThreads / 64 * vp2 * 8) * sizeof(float); };
  if (qpk == 1)
    hipLaunchKernelGGL((window_step_vec_kernel<1, HALF, LPK, VP2>), grid, block, bytes(1), s, a);
  else if (qpk == 2)
    hipLaunchKernelGGL((window_step_vec_kernel<2, HALF, LPK, VP2>), grid, block, bytes(2), s, a);
  else if (qpk <= 4 || bytes(8) > 64 * 1024)
    hipLaunchKernelGGL((window_step_vec_kernel<4, HALF, LPK, VP2>), grid, block, bytes(4), s, a);
  else
    hipLaunchKernelGGL((window_step_vec_kernel<8, HALF, LPK, VP2>), grid, block, bytes(8), s, a);
}

template <bool HALF> void launch_window_step_vec(const WindowArgs& a, hipStream_t s) {
  int lpk = 1, vp2 = 1;
  while (lpk * 8 < a.d) lpk <<= 1;
  while (vp2 * 8 < a.dv) vp2 <<= 1;
  if (lpk == 8 && vp2 == 8)
    launch_window_step_lanes<HALF, 8, 8>(a, vp2, s);
  else if (lpk == 8 && vp2 == 16)
    launch_window_step_lanes<HALF, 8, 16>(a, vp2, s);
  else if (lpk == 16 && vp2 == 16)
    launch_window_step_lanes<HALF, 16, 16>(a, vp2, s);
  else
    launch_window_step_lanes<HALF, 0, 0>(a, vp2, s);
}

template <typename T, bool VEC> void launch_window_step(const WindowArgs& a, hipStream_t s) {
  const int qpk = a.H / a.G;
  const dim3 grid((unsigned)(a.B * a.G)), block(kStepThreads);
  constexpr int N = VEC ? Pack<T>::kN : 1;
  int vp2 = 1;
  while (vp2 * N < a.dv) vp2 <<= 1;
  const int parts = vp2 < 64 ? kStepThreads / 64 : kStepThreads / vp2;
  auto part_floats = [&](int qt) { return qt * parts * vp2 * N; };
  auto bytes = [&](int qt) { return (size_t)(qt * (a.d + kStepKeys + 3) + part_floats(qt) + a.d + a.dv) * sizeof(float); };
  if (qpk == 1)
    hipLaunchKernelGGL((window_step_kernel<T, 1, VEC>), grid, block, bytes(1), s, a, part_floats(1));
  else if (qpk == 2)
    hipLaunchKernelGGL((window_step_kernel<T, 2, VEC>), grid, block, bytes(2), s, a, part_floats(2));
  else if (qpk <= 4 || bytes(8) > 64 * 1024)
    hipLaunchKernelGGL((window_step_kernel<T, 4, VEC>), grid, block, bytes(4), s, a, part_floats(4));
  else
    hipLaunchKernelGGL((window_step_kernel<T, 8, VEC>), grid, block, bytes(8), s, a, part_floats(8));
}

template <int LPI> void launch_kv_write(const WindowArgs& a, hipStream_t s) {
  const long items = (long)a.B * a.L * a.G;
  const dim3 grid((unsigned)((items + 256 / LPI - 1) / (256 / LPI)));
  if (a.half_split)
    hipLaunchKernelGGL((window_kv_write_vec_kernel<LPI, true>), grid, dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL((window_kv_write_vec_kernel<LPI, false>), grid, dim3(256), 0, s, a);
}

template <int KC, int VC, bool DIRECT, bool FILL = false> void launch_window_mfma_pairs(const WindowArgs& a, dim3 grid, hipStream_t s) {
  constexpr unsigned lds = DIRECT ? 2 * kDirectTile * sizeof(__bf16) : 0;
  if constexpr (FILL) {
    static_assert(KC == 2 && VC == 2 && DIRECT, "rows of 64 channels");
    if (a.half_split)
      hipLaunchKernelGGL(window_prefill_fill_kernel<true>, grid, dim3(256), lds, s, a);
    else
      hipLaunchKernelGGL(window_prefill_fill_kernel<false>, grid, dim3(256), lds, s, a);
  } else if (a.half_split) {
    hipLaunchKernelGGL((window_prefill_mfma_kernel<KC, VC, true, DIRECT>), grid, dim3(256), lds, s, a);
  } else {
    hipLaunchKernelGGL((window_prefill_mfma_kernel<KC, VC, false, DIRECT>), grid, dim3(256), lds, s, a);
  }
}

template <int KC> void launch_window_mfma(const WindowArgs& a, dim3 grid, hipStream_t s) {
  const int vc = (a.dv + 31) / 32;
  if (vc <= 1)
    launch_window_mfma_pairs<KC, 1, false>(a, grid, s);
  else if (vc <= 2)
    launch_window_mfma_pairs<KC, 2, false>(a, grid, s);
  else if (vc <= 4)
    launch_window_mfma_pairs<KC, 4, false>(a, grid, s);
  else
    launch_window_mfma_pairs<KC, 8, false>(a, grid, s);
}

static int window_check(const char* who, const WindowArgs& a, int64_t n_rope, int io_dtype, int64_t last) {
  BASED_REQUIRE(a.q && a.k && a.v && a.kv && a.o, BASED_ERR_ARG, "%s: null pointer argument", who);
  BASED_REQUIRE(a.B >= 0 && a.L >= 0 && a.H > 0 && a.G > 0 && a.d > 0 && a.dv > 0 && a.S > 0, BASED_ERR_ARG, "%s: bad sizes", who);
  BASED_REQUIRE(a.H % a.G == 0, BASED_ERR_SHAPE, "%s: %d query heads do not divide into %d key/value heads", who, a.H, a.G);
  BASED_REQUIRE(a.d <= kAnyMaxDim && a.dv <= kAnyMaxDim, BASED_ERR_SHAPE, "%s: head sizes %d / %d (at most %d)", who, a.d, a.dv,
                kAnyMaxDim);
  BASED_REQUIRE(a.window > 0, BASED_ERR_ARG, "%s: window %d", who, a.window);
  BASED_REQUIRE(a.rot >= 0 && a.rot <= a.d && a.rot % 2 == 0, BASED_ERR_SHAPE, "%s: rotary size %d of %d channels", who, a.rot, a.d);
  BASED_REQUIRE(a.rot == 0 || (a.cos_t && a.sin_t), BASED_ERR_ARG, "%s: rotary tables missing", who);
  BASED_REQUIRE(io_dtype == BASED_BF16 || io_dtype == BASED_F32, BASED_ERR_DTYPE, "%s: bad dtype", who);
  BASED_REQUIRE(last < a.S, BASED_ERR_SHAPE, "%s: position %ld does not fit a cache of %d rows", who, (long)last, a.S);
  BASED_REQUIRE(a.rot == 0 || last < n_rope, BASED_ERR_SHAPE, "%s: rotary tables end before position %ld", who, (long)last);
  return BASED_OK;
}

static bool window_vec(const WindowArgs& a, int n) {
  return a.d % n == 0 && a.dv % n == 0 && a.q_sb % n == 0 && a.q_sl % n == 0 && a.k_sb % n == 0 && a.k_sl % n == 0 &&
         a.v_sb % n == 0 && a.v_sl % n == 0 && a.o_sb % n == 0 && a.o_sl % n == 0 && a.kv_sb % n == 0 && a.kv_st % n == 0 &&
         aligned_to(a.q, 16) && aligned_to(a.k, 16) && aligned_to(a.v, 16) && aligned_to(a.kv, 16) && aligned_to(a.o, 16);
}

// fp32 rows in 16-byte pieces that are turned whole; 64 rows to a workgroup of 256 threads, of which a launch takes 2^32.
static bool window_f32(const WindowArgs& a, int io_dtype) {
  return io_dtype == BASED_F32 && (long)a.L * (a.H / a.G) < (1l << 30) - kF32Rows && a.d <= 128 && a.dv <= 128 &&
         a.rot % (a.half_split ? 8 : 4) == 0 && a.d % 4 == 0 && a.dv % 4 == 0 &&
         a.q_sb % 4 == 0 && a.q_sl % 4 == 0 && a.o_sb % 4 == 0 && a.o_sl % 4 == 0 && a.kv_sb % 4 == 0 && a.kv_st % 4 == 0 &&
         aligned_to(a.q, 16) && aligned_to(a.kv, 16) && aligned_to(a.o, 16);
}

// Portions of few rows stay with the general form: a wavefront per query, each on its own way through the keys.  The matrix form takes 68 ns
// a key whatever the rows and the sizes up to 64 (values above 64 channels, keys above: 20 more each), the general one 36 + 0.45 d (values
// above 64 channels: 30 more) as long as an L2 holds the keys that it reads, and more with every thousand rows.  General over matrix form,
// 129 to 2,048 keys, by d x dv: 16 x 16, 300 rows 0.62, 2,600 0.92; 24 x 24, 1,800 0.92; 32 x 32, 300 0.83, 900 0.90, 1,300 0.95, above 4 MB
// of keys and values 1.2 to 1.6; 48 x 48, 600 0.92, 900 0.98; 64 x 64, 300 0.96, 600 1.00; 16 x 128, 300 0.93, 900 0.99; 32 x 128, 300 0.97,
// 600 1.00; 64 x 128, 16 1.08; 80 x 80, 600 0.92; 96 x 32, 600 0.88, 900 1.00; 96 x 96, 160 0.97; 128 x 64, 300 0.95; 128 x 128, 160 1.02.
static bool window_f32_few(const WindowArgs& a) {
  const long rows = (long)a.B * a.L * a.H, end = (long)a.pos_host + a.L, seen = a.window < end ? a.window : end;
  const long keys = seen + a.L - 1 < end ? seen + a.L - 1 : end, bytes = keys * a.B * a.G * (a.d + a.dv) * 4;
  const bool narrow = a.d <= 32 && a.dv <= 32;
  const long room = a.d <= 16 && a.dv <= 16 ? 32 : rows <= 16 ? 12 : narrow && a.L <= 3 ? 8 : 4;
  if (bytes > room << 20) return false;
  if (seen <= 64 && a.d > 64) return rows <= 512;  // (a workgroup's 64 rows span more keys than a row sees: 4 x 96, L = 200, 16 keys: 13.5 us, 15.8)
  if (a.dv > 64) return rows <= (a.d <= 16 ? 500 : a.d <= 32 ? 250 : a.d <= 64 ? 0 : a.d + a.dv <= 160 ? 512 : a.d + a.dv <= 192 ? 256 : 0);
  return rows <= (a.d <= 16 ? 2600 : a.d <= 24 ? 2000 : a.d <= 32 ? 1000 : a.d <= 48 ? 700 : a.d <= 64 ? 400 : a.d <= 96 ? 700 : 350);
}

// Two wavefronts to the same rows where the workgroups are no more than the compute units, or the way through the keys is long; in the first case,
// where that way is short, the cache filled as well (every workgroup turns the keys that it sees: with 1,024 of them 104 us become 158).  us, 16
// heads of 64 channels, one wavefront and a launch for the cache / two / cache filled: on 4, 129 keys, 1 x 777 (196 workgroups) 19.8 / 18.7 / 17.7;
// 1 x 100 13.8 / 12.7 / 11.9; 1 x 2048 (512) 30.5 / 30.4 / -; 4 x 2048 (2,048) 77 / 80 / -; on 16, 1,024 keys, 1 x 2048 (512) 115 / 104 / 158; on 2,
// 513 keys, 2 x 500 (252) 39.2 / 32.5 / 37.7.
// A compute unit holds two workgroups of two wavefronts to a row, and three of one: between 512 and 768 of them the first take a second round that
// the others do not.  Time of two as a part of one's, values of up to 64, by workgroups: 300 keys, 350 0.95, 500 0.96, 600 1.13, 750 1.13, 780 1.08,
// 900 0.87, 1,030 0.84, 1,530 1.01; 1,024 keys, 350 0.92, 500 0.89, 600 0.86, 750 1.16, 900 0.94, 1,030 0.84, 2,040 0.92; 260 keys, 1,300 to 3,000
// 1.00 to 1.05.  Values of 65 to 128, of whose workgroups there is room for one and two: 270 0.80 to 0.87, 350 to 3,000 1.00 to 1.25 with 200 to 513
// keys.  Keys of 65 to 128: never, 50 to 1,000 workgroups 1.00 to 1.08.
static long window_f32_groups(const WindowArgs& a) { return ((long)a.L * (a.H / a.G) + kF32Rows - 1) / kF32Rows * a.B * a.G; }
static bool window_f32_small(const WindowArgs& a) { return window_f32_groups(a) <= 256; }
static long window_f32_keys(const WindowArgs& a) {
  const long end = (long)a.pos_host + a.L;
  return (a.window < end ? a.window : end) + kF32Rows / (a.H / a.G);
}
static bool window_f32_twice(const WindowArgs& a) {
  const long groups = window_f32_groups(a), keys = window_f32_keys(a);
  if (a.dv > 64) return groups <= 300;
  return groups <= 256 || (groups <= 512 ? keys > 256 : groups > 800 && keys > 300);
}

template <int KB, int VB> void launch_window_f32(const WindowArgs& a, dim3 grid, bool fill, hipStream_t s) {
  if constexpr (KB == 1) {
    if (fill) {
      hipLaunchKernelGGL((window_prefill_f32_kernel<KB, VB, 2, true>), grid, dim3(512), 0, s, a);
      return;
    }
    if (window_f32_twice(a)) {
      hipLaunchKernelGGL((window_prefill_f32_kernel<KB, VB, 2, false>), grid, dim3(512), 0, s, a);
      return;
    }
  }
  hipLaunchKernelGGL((window_prefill_f32_kernel<KB, VB, 1, false>), grid, dim3(256), 0, s, a);
}

// Whether memory that rows of `width` elements at these strides span overlaps.
static bool rows_meet(const WindowArgs& a, const void* x, long x_sb, long x_sl, long x_width, const void* y, long y_sb, long y_sl, long y_width, int size) {
  const auto bytes = [&](long sb, long sl, long width) { return ((a.B - 1) * sb + (a.L - 1) * sl + width) * size; };
  const uintptr_t p = reinterpret_cast<uintptr_t>(x), q = reinterpret_cast<uintptr_t>(y);
  return p < q + bytes(y_sb, y_sl, y_width) && q < p + bytes(x_sb, x_sl, x_width);
}

// Whether the attention may fill the cache itself (elements of `size` bytes): keys and values are read by every workgroup that sees them, so that
// nothing else may be written there, and in 16-byte pieces.
static bool window_fresh(const WindowArgs& a, int size) {
  const int n = 16 / size;
  if (a.k_sb % n || a.k_sl % n || a.v_sb % n || a.v_sl % n || !aligned_to(a.k, 16) || !aligned_to(a.v, 16)) return false;
  if (a.k_sb < 0 || a.k_sl < 0 || a.v_sb < 0 || a.v_sl < 0 || a.o_sb < 0 || a.o_sl < 0 || a.kv_sb < 0 || a.kv_st < 0) return false;
  const long kw = (long)a.G * a.d, vw = (long)a.G * a.dv, row = kw + vw;
  const char* cache = static_cast<const char*>(a.kv) + (long)a.pos_host * a.kv_st * size;
  const auto apart = [&](const void* x, long sb, long sl, long width) {
    return !rows_meet(a, x, sb, sl, width, cache, a.kv_sb, a.kv_st, row, size) && !rows_meet(a, x, sb, sl, width, a.o, a.o_sb, a.o_sl, (long)a.H * a.dv, size);
  };
  return apart(a.k, a.k_sb, a.k_sl, kw) && apart(a.v, a.v_sb, a.v_sl, vw);
}
static bool window_f32_fills(const WindowArgs& a) {
  return window_f32_small(a) && window_f32_keys(a) <= 256 && a.d <= 64 && window_fresh(a, 4);
}
// The bf16 form with rows of 64 channels: a launch less for some workgroups turning every key that they see, `before` of them in front of their own
// tokens, by way of registers and with two wavefronts to a SIMD.  Kernel us with a launch for the cache / filled, 16 heads, interleaved pairs, by
// workgroups and `before`: 16 (3 tokens), 0: 6.7 / 5.4; 8, 32: 8.6 / 6.9; 512, 0: 13.9 / 10.4; 512, 68: 15.5 / 13.4; 512, 112: 15.3 / 14.1;
// 128 heads' tokens to a workgroup, 128, 128: 15.3 / 14.2; 256, 128: 14.6 / 13.2; 384, 128: 17.3 / 16.9; 512, 128: 17.4 / 18.2; 1,024, 128: 25.1 /
// 28.6; 28, 168: 11.2 / 12.1; 256, 512: 23.0 / 27.8.  Half-split pairs, which fetch partners and twice the angles: 16 (3 tokens), 0: 6.9 / 5.8; 512,
// 68: 16.4 / 14.8; 98, 128: 12.3 / 12.4; 256, 128: 14.7 / 14.6; 384, 128: 18.1 / 18.8.
static bool window_bf16_fills(const WindowArgs& a) {
  if (a.d != 64 || a.dv != 64) return false;
  const long qpk = a.H / a.G, groups = ((long)a.L * qpk + kTileRows - 1) / kTileRows * a.G * a.B, own = kTileRows / qpk;
  const long front = (long)a.pos_host + a.L - own, before = front < 0 ? 0 : front < a.window - 1 ? front : a.window - 1;
  return before <= 128 && groups <= 768 && groups * before <= 512 * (a.half_split ? 72 : 112) && window_fresh(a, 2);
}

// The attention of a portion whose keys and values are in place (fill: it puts them there itself; `window_f32_fills`, `window_bf16_fills`).
static void launch_window_attend(WindowArgs a, bool vec, int io_dtype, bool fill, hipStream_t s) {
  if (vec) {
    const uint32_t qpk = (uint32_t)(a.H / a.G);
    a.heads_inv = qpk == 1 ? ~0u : (uint32_t)((1ull << 32) / qpk);
    const dim3 grid((unsigned)(((long)a.L * qpk + kTileRows - 1) / kTileRows), (unsigned)a.G, (unsigned)a.B);
    const int kc = (int)((a.d + 31) / 32);
    if (fill)
      launch_window_mfma_pairs<2, 2, true, true>(a, grid, s);
    else if (a.d == 64 && a.dv == 64)
      launch_window_mfma_pairs<2, 2, true>(a, grid, s);
    else if (kc <= 1)
      launch_window_mfma<1>(a, grid, s);
    else if (kc <= 2)
      launch_window_mfma<2>(a, grid, s);
    else if (kc <= 3)
      launch_window_mfma<3>(a, grid, s);
    else if (kc <= 4)
      launch_window_mfma<4>(a, grid, s);
    else
      launch_window_mfma<8>(a, grid, s);
  } else if (window_f32(a, io_dtype) && !window_f32_few(a)) {
    const dim3 grid((unsigned)(((long)a.L * (a.H / a.G) + kF32Rows - 1) / kF32Rows), (unsigned)(a.B * a.G));
    if (a.d <= 64 && a.dv <= 64)
      launch_window_f32<1, 1>(a, grid, fill, s);
    else if (a.d <= 64)
      launch_window_f32<1, 2>(a, grid, fill, s);
    else if (a.dv <= 64)
      launch_window_f32<2, 1>(a, grid, fill, s);
    else
      launch_window_f32<2, 2>(a, grid, fill, s);
  } else {
    const dim3 grid((unsigned)a.L, (unsigned)a.H, (unsigned)a.B);
    if (io_dtype == BASED_BF16)
      hipLaunchKernelGGL(window_prefill_any_kernel<__bf16>, grid, dim3(64), 0, s, a);
    else
      hipLaunchKernelGGL(window_prefill_any_kernel<float>, grid, dim3(64), 0, s, a);
  }
}

}  // namespace based

extern "C" BASED_API int based_window_attn_prefill(
    const void* q, const void* k, const void* v, void* kv_cache, void* o, int64_t start, int64_t B, int64_t L, int64_t H, int64_t G,
    int64_t D, int64_t DV, int64_t S, int64_t q_sb, int64_t q_sl, int64_t k_sb, int64_t k_sl, int64_t v_sb, int64_t v_sl,
    int64_t o_sb, int64_t o_sl, int64_t kv_sb, int64_t kv_st, int64_t window, float scale, int norm_v, float eps, float out_scale,
    const float* rope_cos, const float* rope_sin, int64_t rope_len, int64_t rotary_dim, int half_split, int io_dtype, void* stream) {
  using namespace based;
  BASED_REQUIRE(start >= 0 && start + L < (1ll << 31) && window < (1ll << 31) && L * H < (1ll << 31), BASED_ERR_SHAPE,
                "window_attn_prefill: sequence too long");
  const WindowArgs a{q,       k,       v,      kv_cache, o,        rope_cos, rope_sin, nullptr, (int)start, (int)rope_len,
                     (int)B,  (int)L,  (int)H, (int)G,   (int)D,   (int)DV,  (int)S,   q_sb,    q_sl,       k_sb,
                     k_sl,    v_sb,    v_sl,   o_sb,     o_sl,     kv_sb,    kv_st,    (int)rotary_dim, half_split, (int)window,
                     norm_v,  scale,   eps,    out_scale};
  const int rc = window_check("window_attn_prefill", a, rope_len, io_dtype, start + L - 1);
  if (rc != BASED_OK) return rc;
  BASED_REQUIRE(B * G < 65536 && B < 65536 && H < 65536, BASED_ERR_SHAPE, "window_attn_prefill: grid too large");
  if (B == 0 || L == 0) return BASED_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  // pieces of 8 channels are turned whole: the rotary size is a multiple of 8 (16 in half-split pairs)
  const bool vec = io_dtype == BASED_BF16 && D <= 256 && DV <= 256 && rotary_dim % (half_split ? 16 : 8) == 0 && window_vec(a, 8);
  const int64_t items = B * L * G;
  BASED_REQUIRE(items < (1ll << 32), BASED_ERR_SHAPE, "window_attn_prefill: grid too large");
  const bool fill = vec ? window_bf16_fills(a) : window_f32(a, io_dtype) && !window_f32_few(a) && window_f32_fills(a);
  if (fill)
    ;  // (the attention does it)
  else if (vec) {
    const int64_t widest = D > DV ? D : DV;
    widest <= 64 ? launch_kv_write<8>(a, s) : widest <= 128 ? launch_kv_write<16>(a, s) : launch_kv_write<32>(a, s);
  } else if (io_dtype == BASED_BF16)
    hipLaunchKernelGGL(window_kv_write_kernel<__bf16>, dim3((unsigned)((items + 3) / 4)), dim3(256), 0, s, a);
  else if (window_f32(a, io_dtype) && k_sb % 4 == 0 && k_sl % 4 == 0 && v_sb % 4 == 0 && v_sl % 4 == 0 && aligned_to(k, 16) && aligned_to(v, 16))
    hipLaunchKernelGGL(window_kv_write_f32_kernel, dim3((unsigned)((items + 15) / 16)), dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL(window_kv_write_kernel<float>, dim3((unsigned)((items + 3) / 4)), dim3(256), 0, s, a);
  launch_window_attend(a, vec, io_dtype, fill, s);
  return check_launch("window_attn_prefill");
}

extern "C" BASED_API int based_window_attn_attend(const void* q, const void* kv, void* o, int64_t start, int64_t B, int64_t L, int64_t H,
                                                  int64_t G, int64_t D, int64_t DV, int64_t S, int64_t q_sb, int64_t q_sl, int64_t o_sb,
                                                  int64_t o_sl, int64_t kv_sb, int64_t kv_st, int64_t window, float scale,
                                                  float out_scale, const float* rope_cos, const float* rope_sin, int64_t rope_len,
                                                  int64_t rotary_dim, int half_split, int io_dtype, void* stream) {
  using namespace based;
  BASED_REQUIRE(start >= 0 && start + L < (1ll << 31) && window < (1ll << 31) && L * H < (1ll << 31), BASED_ERR_SHAPE,
                "window_attn_attend: sequence too long");
  // k and v are not read: the rows are there already
  const WindowArgs a{q,      q,      q,      const_cast<void*>(kv), o,       rope_cos, rope_sin, nullptr, (int)start, (int)rope_len,
                     (int)B, (int)L, (int)H, (int)G,                (int)D,  (int)DV,  (int)S,   q_sb,    q_sl,       0,
                     0,      0,      0,      o_sb,                  o_sl,    kv_sb,    kv_st,    (int)rotary_dim, half_split, (int)window,
                     0,      scale,  0.f,    out_scale};
  const int rc = window_check("window_attn_attend", a, rope_len, io_dtype, start + L - 1);
  if (rc != BASED_OK) return rc;
  BASED_REQUIRE(B * G < 65536 && B < 65536 && H < 65536, BASED_ERR_SHAPE, "window_attn_attend: grid too large");
  if (B == 0 || L == 0) return BASED_OK;
  const bool vec = io_dtype == BASED_BF16 && D <= 256 && DV <= 256 && rotary_dim % (half_split ? 16 : 8) == 0 && window_vec(a, 8);
  launch_window_attend(a, vec, io_dtype, false, static_cast<hipStream_t>(stream));
  return check_launch("window_attn_attend");
}

extern "C" BASED_API int based_window_attn_step(
    const void* q, const void* k, const void* v, void* kv_cache, void* o, const int32_t* pos, int64_t pos_host, int64_t B, int64_t H,
    int64_t G, int64_t D, int64_t DV, int64_t S, int64_t q_sb, int64_t k_sb, int64_t v_sb, int64_t o_sb, int64_t kv_sb,
    int64_t kv_st, int64_t window, float scale, int norm_v, float eps, float out_scale, const float* rope_cos,
    const float* rope_sin, int64_t rope_len, int64_t rotary_dim, int half_split, int io_dtype, void* stream) {
  using namespace based;
  BASED_REQUIRE(pos_host >= 0 && pos_host < (1ll << 31) && window < (1ll << 31), BASED_ERR_SHAPE, "window_attn_step: bad position");
  const WindowArgs a{q,      k,      v,      kv_cache, o,       rope_cos, rope_sin, pos,  (int)pos_host, (int)rope_len,
                     (int)B, 1,      (int)H, (int)G,   (int)D,  (int)DV,  (int)S,   q_sb, 0,             k_sb,
                     0,      v_sb,   0,      o_sb,     0,       kv_sb,    kv_st,    (int)rotary_dim, half_split, (int)window,
                     norm_v, scale,  eps,    out_scale};
  const int rc = window_check("window_attn_step", a, rope_len, io_dtype, pos != nullptr ? 0 : pos_host);
  if (rc != BASED_OK) return rc;
  BASED_REQUIRE(B * G < (1ll << 31), BASED_ERR_SHAPE, "window_attn_step: grid too large");
  const int n = io_dtype == BASED_BF16 ? 8 : 4;
  const bool vec = window_vec(a, n);
  BASED_REQUIRE(vec || DV <= kStepThreads, BASED_ERR_SHAPE, "window_attn_step: value size %ld with unaligned rows (at most %d)",
                (long)DV, kStepThreads);
  if (B == 0) return BASED_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (io_dtype == BASED_BF16 && vec && rotary_dim % (half_split ? 16 : 8) == 0)
    half_split ? launch_window_step_vec<true>(a, s) : launch_window_step_vec<false>(a, s);
  else if (io_dtype == BASED_BF16)
    vec ? launch_window_step<__bf16, true>(a, s) : launch_window_step<__bf16, false>(a, s);
  else
    vec ? launch_window_step<float, true>(a, s) : launch_window_step<float, false>(a, s);
  return check_launch("window_attn_step");
}
