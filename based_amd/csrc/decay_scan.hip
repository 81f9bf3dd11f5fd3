// Linear attention with decaying states for gfx950.  Per head (state S: d x dv, fp32), token by token, either
//
//   channel decays (a decay per key channel and token, a bonus for the current token):
//     o_t = (S + diag(u) k_t v_t^T)^T q_t,   then  S <- diag(w_t) S + k_t v_t^T
//   head decays (one constant per head):
//     S <- w_h S + k_t v_t^T,   then  o_t = S^T q_t
//
// with silu on q, k and v first where asked for.  Decays come as base-2 logarithms.  The state lies by
// value channel, (B, H, dv, dp): rows of dp >= d key channels.
//
//   decay_channel, decay_head
//                     bf16: walk 64 tokens at a time with the state in MFMA accumulators, 16 value channels
//                     per wavefront.  Long sequences are cut into segments: a first pass leaves what every
//                     segment adds to the state, `decay_join` turns that into the state at every segment's
//                     start, and the second pass starts there; few segments it puts together itself.
//   decay_scan_any    any element type and size, in segments too: a thread holds some key channels of one value channel.
//   decay_step        one token per sequence; for channel decays with the low-rank decay in front and the
//                     head norm and gate behind.
//   group_norm_gate   o / rms(o) * w * act(g) over groups of a row.
//
// Inside 64 tokens, with P_ts the weight of v_s in o_t, o = P v + (q scaled by the decay since the start) S0.
// All scaling is by decays over tokens that lie in between, never by an inverse, so nothing overflows:
//   * s and t in the same 16 tokens: halves of 2, 4, 8 and 16 tokens meet, k_s decayed to the middle, q_t from there
//     (head decays: a power of the decay, times the product of k_s and q_t);
//   * s in an earlier 16 tokens: k_s decayed to the end of its 16, q_t to the start of its own, and to q
//     also what lies between.
// fp32 numbers enter a bf16 product as pairs (a number rounded to bf16, and the rest rounded to bf16), so
// an operand keeps 16 bits and the sums 24; the weights inside 16 tokens are formed in fp32.
#include <type_traits>

#include "lds_limit.hpp"
#include "stream_common.hpp"

namespace based {

constexpr int kScanTokens = 64;

struct DecayScanArgs {
  const void* q;
  const void* k;
  const void* v;
  const float* lw;       // (B, L, H * d) contiguous: log2 of the channel decays, or null
  const float* head_lw;  // (2, H): log2 of the sizes of the head decays, then the decays, or null
  const void* u;         // (H, d)
  float* state;          // (B, H, dv, dp)
  float* seg;            // (B, H, segs, dv, dp) work, null with one segment
  float* seg_lw;         // (B, H, segs, dp) work: channel decays over a segment
  void* o;               // (B, L, H * dv)
  int B, L, H, d, dv, dp;
  long q_sb, q_sl, k_sb, k_sl, v_sb, v_sl, o_sb, o_sl;
  int segs, seg_chunks;  // segments, and 64-token pieces in each
  int silu, fresh;
  int wide;              // rows of q, k, v and o in whole 16-byte pieces (channel decays, bf16)
  int narrow;            // workgroups of 64 value channels, not of 128 (channel decays, more than 64 key channels)
};

// Products along the 16 lanes of a row, of several independent numbers at once.  A DPP multiplication leaves a lane
// without a source as it is, which is the multiplication by one that is wanted; the compiler has no builtin that
// says so.  A register must not be read through DPP in the two issue slots after it was written: four numbers in turn
// keep that distance by themselves, the first ones are kept from what stands before by the s_nop.
//   suffix[i]: product over lanes l .. 15 of w[i];  after[i] *= suffix of the lane behind (nothing for lane 15)
#define BASED_ROW_STEP(ctrl) \
  "v_mul_f32_dpp %0, %0, %0 " ctrl " row_mask:0xf bank_mask:0xf\n\t" \
  "v_mul_f32_dpp %1, %1, %1 " ctrl " row_mask:0xf bank_mask:0xf\n\t" \
  "v_mul_f32_dpp %2, %2, %2 " ctrl " row_mask:0xf bank_mask:0xf\n\t" \
  "v_mul_f32_dpp %3, %3, %3 " ctrl " row_mask:0xf bank_mask:0xf\n\t"
#define BASED_ROW_LAST(ctrl) \
  "v_mul_f32_dpp %4, %0, %4 " ctrl " row_mask:0xf bank_mask:0xf\n\t" \
  "v_mul_f32_dpp %5, %1, %5 " ctrl " row_mask:0xf bank_mask:0xf\n\t" \
  "v_mul_f32_dpp %6, %2, %6 " ctrl " row_mask:0xf bank_mask:0xf\n\t" \
  "v_mul_f32_dpp %7, %3, %7 " ctrl " row_mask:0xf bank_mask:0xf"
__device__ __forceinline__ void row_suffix4(float* suffix, float* after) {
  asm volatile("s_nop 1\n\t" BASED_ROW_STEP("row_shl:1") BASED_ROW_STEP("row_shl:2") BASED_ROW_STEP("row_shl:4")
               BASED_ROW_STEP("row_shl:8") BASED_ROW_LAST("row_shl:1")
               : "+v"(suffix[0]), "+v"(suffix[1]), "+v"(suffix[2]), "+v"(suffix[3]), "+v"(after[0]), "+v"(after[1]), "+v"(after[2]),
                 "+v"(after[3]));
}
#undef BASED_ROW_STEP
#undef BASED_ROW_LAST

__device__ __forceinline__ f32x4 mfma_16(bf16x8 a, bf16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
// two numbers as packed pairs of bf16: rounded, and what the rounding left
__device__ __forceinline__ void split2(float a, float b, uint32_t& hi, uint32_t& lo) {
  hi = pack_bf16(a, b);
  lo = pack_bf16(a - __builtin_bit_cast(float, hi << 16), b - __builtin_bit_cast(float, hi & 0xffff0000u));
}
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
// eight numbers in the order of an MFMA operand
__device__ __forceinline__ void split8(const float* x, bf16x8& hi, bf16x8& lo) {
  u32x4 h, l;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t a, b;
    split2(x[2 * i], x[2 * i + 1], a, b);
    h[i] = a, l[i] = b;
  }
  hi = __builtin_bit_cast(bf16x8, h);
  lo = __builtin_bit_cast(bf16x8, l);
}
// the halves of a packed pair as they are
__device__ __forceinline__ void store_pair(__bf16* p, __bf16* q, uint32_t x) {
  *reinterpret_cast<uint16_t*>(p) = (uint16_t)x;
  *reinterpret_cast<uint16_t*>(q) = (uint16_t)(x >> 16);
}

// Powers of a head's decay w, without their signs, from the logarithm of its size.  (Nothing is worked out from the two in front of the first
// tokens' loads, which would wait for them.)
struct HeadPowers {
  float l2, w;
  __device__ __forceinline__ HeadPowers(const DecayScanArgs& a, int h) : l2(a.head_lw[h]), w(a.head_lw[a.H + h]) {}
  __device__ __forceinline__ float operator()(int n) const { return __builtin_amdgcn_exp2f(l2 * (float)n); }
  // What a state is multiplied by.  A product of decays that only the format makes zero comes as the smallest number: an infinite state outlives it,
  // as it does token by token.
  __device__ __forceinline__ float of_state(int n) const { return fmaxf((*this)(n), w != 0.f ? 0x1p-149f : 0.f); }
};

// ---- channel decays, bf16 ----
// HALVES groups of four wavefronts (1 or 2) share the key channels, 32 DT each (d <= 32 DT HALVES, d % 4 == 0); a wavefront has 16 of the 64 tokens, a
// lane 8 DT channels of one of them that lie side by side, so that rows come in 16-byte pieces.  In a product the lanes of a 16-lane row bring
// eight channels of a piece of 32 each; every contraction over channels has that order on both sides.
//
// Inside 16 tokens the weights are found by halves: with b = 1, 2, 4, 8, tokens of the second half of each 2 b meet those of its first half, queries
// decayed from the middle to their token, keys from theirs to the middle, so that one operand x (a query or a key, by the lane's half) times itself
// holds all of them; the products of decays double with b on the way.  (Keys passed from token to token on the vector unit were 610 of a
// wavefront's 1,500 instructions to 64 tokens.)  Neighbours are the bf16 that came in; the others are products of fp32 numbers, of four keys with four
// queries at a time, which leaves none of a product unused but the half that lies in front of the key.  Where keys nearly cancel, in two channels
// of opposite sign whose decays differ by 2^-12, the error against 64 bits is 1.667e-3, of which the rounding of o to bf16 is all; with x as pairs of bf16
// it was 5.5e-3.  Calls, us, as pairs / as 16 x 16 products in fp32 / this way: 4 x 2048 tokens, 16 heads of 64 57.9 / 61.5 / 58.7; 20 x 2048 220 / 244 /
// 228; 16 x 1024, 8 heads of 128 114 / 128 / 119; 8 x 2000 144 / 149 / 141; 2 x 768, 16 heads of 64 22.2 / 23.1 / 22.1.
// Across 16 tokens the keys wait in LDS, decayed to the end of theirs, for the queries decayed from the start of their own and what lies between;
// the state takes the same keys, decayed itself by what each 16 tokens leave of it.  Outputs belong to the wavefronts of their tokens, so that neither
// weights nor queries go through LDS, the state's tiles of 16 value channels to a wavefront each: two barriers to 64 tokens, one behind what is written
// of each piece and one behind what is read.
//
// What bounds it: 64 tokens are a chain of instructions, two barriers and products that wait for each other, 10,000 cycles and more.  Heads of 64, us a
// piece of 64 tokens in one chain: 4.5 with one workgroup of eight wavefronts, half of the channels each, to a compute unit; with workgroups of four
// wavefronts 7.4 for two of them, 10.3 for three, so that another wavefront on a SIMD adds some 3 us (a fourth workgroup has to wait: 14.1).  Heads of 128:
// 6.9, workgroups of 128 value channels 9.8.  4 x 2048 tokens, 16 heads of 64, two workgroups to a compute unit: scan 43 us for four pieces and the
// states of up to seven segments, vector unit busy 41 %, matrix unit 15 %, wavefronts waiting for 40 % of their time; state pass 17, 29 %, 9 %, 42 %.
// So channels are dealt to more wavefronts where heads are few, prompts are cut into segments of a piece where that leaves compute units idle
// (decay_channel_segments), and nothing is kept in memory inside the loop: a value fetched back from there waits for the tokens that were asked for
// before it (17 of them: 68.6 us for 62.9).
// us before (tokens passed along, four barriers, segments of four pieces) and now: 4 x 2048 tokens, 16 heads of 64: 75, 58; 2 x 768: 48, 23;
// 30 x 513: 123, 72; 2 x 27, 12 heads: 10.4, 8.2; 4 x 2048, 8 heads of 128: 102, 90; 16 x 1024: 173, 120; 2 x 133: 42.3, 25.7.
template <int DT, int HALVES, int COLS> struct ChannelLds {
  static constexpr int CH = 32 * DT * HALVES, RS = CH + 8, VS = COLS + 8;
  static constexpr int OT = COLS / 16, OF = OT / HALVES;  // tiles of 16 value channels, and those a group of wavefronts finishes
  __bf16 k_hi[kScanTokens * RS], k_lo[kScanTokens * RS];  // k decayed to the end of its 16 tokens, [token][channel as the lanes have them]
  __bf16 v[kScanTokens * VS];
  float total[4][CH];                                     // decay over each 16 tokens, by channel
  // (from here on not in the state pass)
  float u[CH];
  __bf16 s_hi[COLS * RS], s_lo[COLS * RS];                // the state in front of the 64 tokens, [value channel][channel as the lanes have them]
  f32x4 part[HALVES > 1 ? 4 * HALVES * (HALVES - 1) * OF * 64 : 1];  // what the other groups' channels add to an output
};

// q[i] *= decays of the half in front, k[i] *= those of the half behind, t[i] (the decay over a half) over both; two channels at a time.  Lanes without such
// a half meet a one, or keep theirs by the bank mask.  (A register must not be read through DPP in the two issue slots behind its writing: the s_nop.)
#define BASED_HALF_STEP(ctrl, qa, qb, qbank, ka, kb, kbank) \
  "s_nop 1\n\t" \
  "v_mul_f32_dpp %0, " qa ", %0 " ctrl " row_mask:0xf bank_mask:" qbank "\n\t" \
  "v_mul_f32_dpp %1, " qb ", %1 " ctrl " row_mask:0xf bank_mask:" qbank "\n\t" \
  "v_mul_f32_dpp %2, " ka ", %2 " ctrl " row_mask:0xf bank_mask:" kbank "\n\t" \
  "v_mul_f32_dpp %3, " kb ", %3 " ctrl " row_mask:0xf bank_mask:" kbank "\n\t" \
  "v_mul_f32_dpp %4, %4, %4 " ctrl " row_mask:0xf bank_mask:0xf\n\t" \
  "v_mul_f32_dpp %5, %5, %5 " ctrl " row_mask:0xf bank_mask:0xf"
#define BASED_HALF_REGS "+&v"(q[0]), "+&v"(q[1]), "+&v"(k[0]), "+&v"(k[1]), "+&v"(t[0]), "+&v"(t[1])
template <int B> __device__ __forceinline__ void join_halves2(float* q, float* k, float* t, bool second) {
  if constexpr (B < 4) {
    const float f0 = second ? 1.f : t[0], f1 = second ? 1.f : t[1];  // decays of lanes of a first half, a one in the others
    const float s0 = second ? t[0] : 1.f, s1 = second ? t[1] : 1.f;  // of a second half
    if constexpr (B == 1)
      asm(BASED_HALF_STEP("quad_perm:[1,0,3,2]", "%6", "%7", "0xf", "%8", "%9", "0xf") : BASED_HALF_REGS : "v"(f0), "v"(f1), "v"(s0), "v"(s1));
    else
      asm(BASED_HALF_STEP("quad_perm:[2,3,0,1]", "%6", "%7", "0xf", "%8", "%9", "0xf") : BASED_HALF_REGS : "v"(f0), "v"(f1), "v"(s0), "v"(s1));
  } else if constexpr (B == 4) {
    asm(BASED_HALF_STEP("row_half_mirror", "%4", "%5", "0xa", "%4", "%5", "0x5") : BASED_HALF_REGS);
  } else {
    asm(BASED_HALF_STEP("row_mirror", "%4", "%5", "0xc", "%4", "%5", "0x3") : BASED_HALF_REGS);
  }
}
#undef BASED_HALF_STEP
#undef BASED_HALF_REGS

// 16 products of 4 x 4 numbers, each of four lanes: the rows are a's, of the lanes of number ABID of every 2^CBSZ such groups, the columns b's own.
template <int CBSZ, int ABID> __device__ __forceinline__ f32x4 mfma_4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, c, CBSZ, ABID, 0);
}
__device__ __forceinline__ f32x4 mfma_16_half(bf16x4 a, bf16x4 b, f32x4 c) {
  typedef __attribute__((ext_vector_type(4))) short s16x4;
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, a), __builtin_bit_cast(s16x4, b), c, 0, 0, 0);
}
__device__ __forceinline__ void split4(f32x4 x, bf16x4& hi, bf16x4& lo) {
  typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;
  uint32_t h0, h1, l0, l1;
  split2(x[0], x[1], h0, l0);
  split2(x[2], x[3], h1, l1);
  hi = __builtin_bit_cast(bf16x4, u32x2{h0, h1});
  lo = __builtin_bit_cast(bf16x4, u32x2{l0, l1});
}

constexpr int channel_waves(int dt, int halves) { return halves == 1 ? 3 : dt == 1 ? 4 : 2; }  // wavefronts on a SIMD that registers are left for

template <int DT, int HALVES, int COLS, bool STATE_ONLY, bool FOLD>
__global__ __launch_bounds__(256 * HALVES, channel_waves(DT, HALVES)) void decay_channel_kernel(const DecayScanArgs a) {
  typedef ChannelLds<DT, HALVES, COLS> Lds;
  constexpr int RS = Lds::RS, VS = Lds::VS, E = DT * 8, OT = Lds::OT, OF = Lds::OF;
  constexpr int VC = COLS / HALVES / 4;                           // value channels that a lane brings of its token
  constexpr int SP = DT * HALVES * OT / (4 * HALVES);             // 32-channel pieces of the state that a wavefront has of its 16 value channels
  extern __shared__ __attribute__((aligned(16))) char scan_lds[];
  Lds& lds = *reinterpret_cast<Lds*>(scan_lds);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l16 = lane & 15, quad = lane >> 4;
  // This wavefront's key channels, and its 16 tokens of 64: later ones have more in front of them, so that the wavefronts of a SIMD take turns.
  const int half = wave >> 2, ch0 = half * 32 * DT, blk = half & 1 ? 3 - ((wave + blockIdx.x) & 3) : (wave + blockIdx.x) & 3;
  const int tile = wave % OT, piece0 = wave / OT * SP;  // its value channels and pieces of the state
  const int b = blockIdx.x / a.H, h = blockIdx.x % a.H, sg = blockIdx.z;
  const int col_base = blockIdx.y * COLS, dv0 = col_base + tile * 16;
  const bool has_cols = dv0 < a.dv, col_in = dv0 + l16 < a.dv;
  const __bf16* qp = static_cast<const __bf16*>(a.q) + b * a.q_sb + (long)h * a.d;
  const __bf16* kp = static_cast<const __bf16*>(a.k) + b * a.k_sb + (long)h * a.d;
  const __bf16* vp = static_cast<const __bf16*>(a.v) + b * a.v_sb + (long)h * a.dv;
  const float* lwp = a.lw + ((long)b * a.L) * a.H * a.d + (long)h * a.d;
  const long bh = (long)b * a.H + h;
  float* st = a.state + (bh * a.dv + (col_in ? dv0 + l16 : 0)) * a.dp;

  // channel of element 4 f of piece c, and of element i; of the state's tile ct
  auto chan = [&](int c, int f, int quad) { return ch0 + quad * E + c * 8 + f * 4; };
  auto chan_of = [&](int i, int quad) { return ch0 + quad * E + i; };
  auto state_chan = [&](int ct, int quad) { return (piece0 + ct / 2) / DT * 32 * DT + quad * E + (piece0 + ct / 2) % DT * 8 + ct % 2 * 4; };

  struct Stage {
    bf16x4 q[STATE_ONLY ? 1 : 2 * DT], k[2 * DT], v[VC / 4];
    f32x4 lw[2 * DT];
  };
  const int first = sg * a.seg_chunks, chunks = (a.L + kScanTokens - 1) / kScanTokens;
  const int last = first + a.seg_chunks < chunks ? first + a.seg_chunks : chunks;
  // The rows of this wavefront's 16 tokens, unconditionally (places past the end are cleared at use): the place of the 64 tokens is the same for all
  // lanes, and what lies behind it (in front of it, where a stride is below zero) fits 32 bits.
  const int q_back = a.q_sl < 0 ? (int)a.q_sl * (kScanTokens - 1) : 0, k_back = a.k_sl < 0 ? (int)a.k_sl * (kScanTokens - 1) : 0,
            v_back = a.v_sl < 0 ? (int)a.v_sl * (kScanTokens - 1) : 0;
  auto pieces = [](bf16x8 x, bf16x4& lo, bf16x4& hi) {
    lo = __builtin_shufflevector(x, x, 0, 1, 2, 3), hi = __builtin_shufflevector(x, x, 4, 5, 6, 7);
  };
  // (parts: 1 keys, 2 decays, 4 queries, 8 values)
  auto fetch = [&](Stage& s, int chunk, int l16, int quad, auto parts) {
    constexpr int kParts = decltype(parts)::value;
    const int left = a.L - chunk * kScanTokens, mine = blk * 16 + l16, t = mine < left ? mine : left - 1;
    const long t0 = (long)chunk * kScanTokens;
    auto rows = [&](const __bf16* p, long sl, int back, bf16x4* to) {  // key channels
      const char* p0 = reinterpret_cast<const char*>(p + t0 * sl + back);
      const uint32_t at = (uint32_t)(t * (int)sl - back);
      if (a.wide) {  // (uniform)
#pragma unroll
        for (int c = 0; c < DT; ++c)
          pieces(*reinterpret_cast<const bf16x8*>(p0 + (at + (chan(c, 0, quad) < a.d ? chan(c, 0, quad) : 0)) * 2u), to[2 * c], to[2 * c + 1]);
      } else {
#pragma unroll
        for (int g = 0; g < 2 * DT; ++g)
          to[g] = *reinterpret_cast<const bf16x4*>(p0 + (at + (chan(g >> 1, g & 1, quad) < a.d ? chan(g >> 1, g & 1, quad) : 0)) * 2u);
      }
    };
    if constexpr ((kParts & 1) != 0) rows(kp, a.k_sl, k_back, s.k);
    if constexpr ((kParts & 2) != 0) {
      const char* w0 = reinterpret_cast<const char*>(lwp + t0 * a.H * a.d);
      const uint32_t at = (uint32_t)t * (uint32_t)(a.H * a.d);
#pragma unroll
      for (int g = 0; g < 2 * DT; ++g)
        s.lw[g] = *reinterpret_cast<const f32x4*>(w0 + (at + (chan(g >> 1, g & 1, quad) < a.d ? chan(g >> 1, g & 1, quad) : 0)) * 4u);
    }
    if constexpr (!STATE_ONLY && (kParts & 4) != 0) rows(qp, a.q_sl, q_back, s.q);
    if constexpr ((kParts & 8) != 0) {
      const char* v0 = reinterpret_cast<const char*>(vp + t0 * a.v_sl + v_back);
      const uint32_t at = (uint32_t)(t * (int)a.v_sl - v_back);
      const int col = col_base + half * (COLS / HALVES) + quad * VC;
      if (VC >= 8 && a.wide) {
#pragma unroll
        for (int f = 0; f < VC / 8; ++f)
          pieces(*reinterpret_cast<const bf16x8*>(v0 + (at + (uint32_t)(col + f * 8 < a.dv ? col + f * 8 : 0)) * 2u), s.v[2 * f], s.v[2 * f + 1]);
      } else {
#pragma unroll
        for (int f = 0; f < VC / 4; ++f) s.v[f] = *reinterpret_cast<const bf16x4*>(v0 + (at + (uint32_t)(col + f * 4 < a.dv ? col + f * 4 : 0)) * 2u);
      }
    }
  };
  Stage cur;
  if (first < last) fetch(cur, first, l16, quad, std::integral_constant<int, 15>{});
  if constexpr (!STATE_ONLY) {
    const int ch = threadIdx.x;
    if (ch < Lds::CH) lds.u[ch] = ch < a.d ? to_f32(static_cast<const __bf16*>(a.u)[(long)h * a.d + ch]) : 0.f;
  }

  // state: tile ct holds key channels 16 ct + 4 quad + i of value channel dv0 + l16
  f32x4 S[2 * SP];
  {
    const long seg_row = (col_in ? dv0 + l16 : 0), seg_step = (long)a.dv * a.dp;
    const float* segs = a.seg + (bh * a.segs * a.dv + seg_row) * a.dp;
    // FOLD: what the segments in front have added is put together here, the state that enters the call from the last one's place, where
    // the state pass has left it (the last segment replaces it).  Kernels of their own: the others have registers for what they do.
    const bool fold = FOLD && !STATE_ONLY && a.segs > 1;
    const float* from = a.segs > 1 ? segs + (fold ? a.segs - 1 : sg) * seg_step : st;
    const bool zero = STATE_ONLY || ((a.segs == 1 || fold) && a.fresh);
#pragma unroll
    for (int ct = 0; ct < 2 * SP; ++ct) {
      const int ch = state_chan(ct, quad);
      S[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (!zero && col_in && ch < a.d) S[ct] = *reinterpret_cast<const f32x4*>(from + ch);
    }
    if constexpr (STATE_ONLY) {
      if (FOLD && !a.fresh && sg == 0 && col_in) {
        float* keep = a.seg + ((bh * a.segs + a.segs - 1) * a.dv + seg_row) * a.dp;
#pragma unroll
        for (int ct = 0; ct < 2 * SP; ++ct) {
          const int ch = state_chan(ct, quad);
          if (ch < a.d) *reinterpret_cast<f32x4*>(keep + ch) = *reinterpret_cast<const f32x4*>(st + ch);
        }
      }
    } else if (fold) {
      constexpr int U = SP > 2 ? 2 : 4;  // segments asked for together
      for (int s0 = 0; s0 < sg; s0 += U) {
        f32x4 add[U][2 * SP], l[U][2 * SP];
#pragma unroll
        for (int n = 0; n < U; ++n)
#pragma unroll
          for (int ct = 0; ct < 2 * SP; ++ct) {
            const int ch = state_chan(ct, quad) < a.d ? state_chan(ct, quad) : 0, s = s0 + n < sg ? s0 + n : sg - 1;
            add[n][ct] = *reinterpret_cast<const f32x4*>(segs + s * seg_step + ch);
            l[n][ct] = *reinterpret_cast<const f32x4*>(a.seg_lw + (bh * a.segs + s) * a.dp + ch);
          }
#pragma unroll
        for (int n = 0; n < U; ++n) {
          if (s0 + n >= sg) break;  // (uniform)
#pragma unroll
          for (int ct = 0; ct < 2 * SP; ++ct)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const float sum = __builtin_fmaf(S[ct][j], l[n][ct][j], add[n][ct][j]);
              S[ct][j] = col_in && state_chan(ct, quad) < a.d ? sum : 0.f;
            }
        }
      }
    }
  }
  if constexpr (!STATE_ONLY) lds_barrier();  // (the bonus)
  float seg_total = 1.f;  // (state pass) decay of the segment so far, of the channel that is this thread's number

  for (int chunk = first; chunk < last; ++chunk) {
    // (What follows from the lane is worked out anew each time: kept in front of the loop, it went to memory, and every value fetched back waited
    // for the next tokens as well.)
    int here = lane;
    asm volatile("" : "+v"(here));
    const int l16 = here & 15, quad = here >> 4;
    const int tr_row = l16 >> 2, tr_piece = (l16 & 3) * 4;  // what a lane names of a transposed read: a token of four, and four channels of 16
    const int left = a.L - chunk * kScanTokens, n = left < kScanTokens ? left : kScanTokens;
    const int t = blk * 16 + l16;  // this lane's token
    const bool live = t < n;
    float q[STATE_ONLY ? 1 : E], k[E], w[E];
#pragma unroll
    for (int i = 0; i < E; ++i) {
      if constexpr (!STATE_ONLY) q[i] = to_f32(cur.q[i >> 2][i & 3]);
      k[i] = to_f32(cur.k[i >> 2][i & 3]);
      w[i] = __builtin_amdgcn_exp2f(cur.lw[i >> 2][i & 3]);
    }
    if (a.silu) {  // (one branch for all of them)
#pragma unroll
      for (int i = 0; i < E; ++i) {
        if constexpr (!STATE_ONLY) q[i] = round_to<__bf16>(silu_exact(q[i]));
        k[i] = round_to<__bf16>(silu_exact(k[i]));
      }
    }
    if (n < kScanTokens || a.d < Lds::CH) {  // (uniform)
#pragma unroll
      for (int g = 0; g < 2 * DT; ++g) {
        const bool in = live && chan(g >> 1, g & 1, quad) < a.d;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if constexpr (!STATE_ONLY) q[g * 4 + j] = in ? q[g * 4 + j] : 0.f;
          k[g * 4 + j] = in ? k[g * 4 + j] : 0.f;
          w[g * 4 + j] = in ? w[g * 4 + j] : 1.f;
        }
      }
    }
    typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;
    u32x2 vv[VC / 4];
#pragma unroll
    for (int f = 0; f < VC / 4; ++f) vv[f] = __builtin_bit_cast(u32x2, cur.v[f]);
    if (a.silu) {
#pragma unroll
      for (int f = 0; f < VC / 4; ++f)
#pragma unroll
        for (int j = 0; j < 2; ++j) vv[f][j] = pack_bf16(silu_exact(to_f32(cur.v[f][2 * j])), silu_exact(to_f32(cur.v[f][2 * j + 1])));
    }
    if (n < kScanTokens || col_base + COLS > a.dv) {
#pragma unroll
      for (int f = 0; f < VC / 4; ++f)
        if (!(live && col_base + half * (COLS / HALVES) + quad * VC + f * 4 < a.dv)) vv[f] = u32x2{0u, 0u};
    }
#pragma unroll
    for (int f = 0; f < VC / 4; ++f) *reinterpret_cast<u32x2*>(&lds.v[t * VS + half * (COLS / HALVES) + quad * VC + f * 4]) = vv[f];
    const bool more = chunk + 1 < last;
    auto ask = [&](auto parts) {  // (the memory unit takes rows of 16 tokens a lane at a time: a few requests here and there, none of which waits for its turn)
      if (more) fetch(cur, chunk + 1, l16, quad, parts);
      __builtin_amdgcn_sched_barrier(0);
    };

    // the weights inside the 16 tokens: column t, rows s = 4 quad + i
    f32x4 diag = {0.f, 0.f, 0.f, 0.f};
    if constexpr (!STATE_ONLY) {
      float bonus = 0.f;
#pragma unroll
      for (int i = 0; i < E; i += 4) {
        const f32x4 u = *reinterpret_cast<const f32x4*>(&lds.u[chan_of(i, quad)]);
#pragma unroll
        for (int j = 0; j < 4; ++j) bonus = __builtin_fmaf(q[i + j] * u[j], k[i + j], bonus);
      }
      bonus = sum_quads4(bonus, bonus, bonus, bonus);  // (in every lane of the token)
#pragma unroll
      for (int i = 0; i < 4; ++i) diag[i] = quad * 4 + i == l16 ? bonus : 0.f;
      {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < DT; ++c) {  // (neighbours: no decay lies between, the operands are what came in)
          u32x4 x;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            x[e] = pack_bf16(l16 & 1 ? q[c * 8 + 2 * e] : k[c * 8 + 2 * e], l16 & 1 ? q[c * 8 + 2 * e + 1] : k[c * 8 + 2 * e + 1]);
          acc = mfma_16(__builtin_bit_cast(bf16x8, x), __builtin_bit_cast(bf16x8, x), acc);
        }
#pragma unroll
        for (int i = 0; i < E; i += 2) join_halves2<1>(q + i, k + i, w + i, l16 & 1);
#pragma unroll
        for (int i = 0; i < 4; ++i) diag[i] = (l16 & 1) && quad * 4 + i == l16 - 1 ? acc[i] : diag[i];
      }
      // [of four tokens] itself, the four in front, of the first and second four of the eight in front: rows, this lane's token the column
      f32x4 own = {0.f, 0.f, 0.f, 0.f}, front = own, first4 = own, second4 = own;
      auto level = [&](auto half_len) {
        constexpr int HB = decltype(half_len)::value;
#pragma unroll
        for (int i = 0; i < E; ++i) {
          const float x = l16 & HB ? q[i] : k[i];
          if constexpr (HB == 2) own = mfma_4<0, 0>(x, x, own);
          if constexpr (HB == 4) front = mfma_4<1, 0>(x, x, front);
          if constexpr (HB == 8) first4 = mfma_4<2, 0>(x, x, first4), second4 = mfma_4<2, 1>(x, x, second4);
        }
#pragma unroll
        for (int i = 0; i < E; i += 2) join_halves2<HB>(q + i, k + i, w + i, l16 & HB);
      };
      ask(std::integral_constant<int, 1>{});
      level(std::integral_constant<int, 2>{});
      ask(std::integral_constant<int, 2>{});
      level(std::integral_constant<int, 4>{});
      ask(std::integral_constant<int, 4>{});
      level(std::integral_constant<int, 8>{});
      ask(std::integral_constant<int, 8>{});
      const int four = l16 >> 2;
#pragma unroll
      for (int i = 0; i < 4; ++i) {  // added up over the channels' lanes, each where its row is wanted
        const float near = i < 2 && l16 & 2 ? own[i] : 0.f;
        diag[i] += sum_quads4(four == 0 ? near : four == 1 ? front[i] : first4[i], four == 1 ? near : four >= 2 ? second4[i] : 0.f,
                              four == 2 ? near : four == 3 ? front[i] : 0.f, four == 3 ? near : 0.f);
      }
      // q is decayed from the start of the 16 tokens now, k to their end, w the decay over all of them
    } else {
#pragma unroll
      for (int i = 0; i < E; i += 4) row_suffix4(w + i, k + i);  // (the product over all 16 is lane 0's)
      ask(std::integral_constant<int, 15>{});
    }

#pragma unroll
    for (int c = 0; c < DT; ++c) {
      bf16x8 hi, lo;
      split8(k + c * 8, hi, lo);
      *reinterpret_cast<bf16x8*>(&lds.k_hi[t * RS + ch0 + c * 32 + quad * 8]) = hi;
      *reinterpret_cast<bf16x8*>(&lds.k_lo[t * RS + ch0 + c * 32 + quad * 8]) = lo;
    }
    if (l16 == 0) {
#pragma unroll
      for (int i = 0; i < E; i += 4) *reinterpret_cast<f32x4*>(&lds.total[blk][chan_of(i, quad)]) = f32x4{w[i], w[i + 1], w[i + 2], w[i + 3]};
    }
    if constexpr (!STATE_ONLY) {
      if (has_cols) {
        const int s_row = tile / 4 * 64 + (l16 >> 2) * 16 + tile % 4 * 4 + (l16 & 3);  // in the order of the outputs' rows
#pragma unroll
        for (int c = 0; c < SP; ++c) {
          bf16x8 hi, lo;
          const float x[8] = {S[2 * c][0], S[2 * c][1], S[2 * c][2], S[2 * c][3], S[2 * c + 1][0], S[2 * c + 1][1], S[2 * c + 1][2], S[2 * c + 1][3]};
          split8(x, hi, lo);
          *reinterpret_cast<bf16x8*>(&lds.s_hi[s_row * RS + (piece0 + c) * 32 + quad * 8]) = hi;
          *reinterpret_cast<bf16x8*>(&lds.s_lo[s_row * RS + (piece0 + c) * 32 + quad * 8]) = lo;
        }
      }
    }
    lds_barrier();

    f32x4 o[STATE_ONLY ? 1 : OT];  // column t, rows: value channels 16 quad + 4 g + i of each 64
    if constexpr (!STATE_ONLY) {
#pragma unroll
      for (int g = 0; g < OT; ++g) o[g] = f32x4{0.f, 0.f, 0.f, 0.f};
      f32x4 P = diag;  // column t, rows s of 16 tokens j
      for (int j = blk;;) {
        // (all of a round's reads in front of it)
        bf16x4 v4[OT], ph, pl;
        bf16x8 kh[DT], kl[DT], hi[DT], lo[DT];
        const int before = j > 0 ? j - 1 : 0;
#pragma unroll
        for (int g = 0; g < OT; ++g) v4[g] = read_transposed(&lds.v[(j * 16 + quad * 4 + tr_row) * VS + g / 4 * 64 + tr_piece * 4 + g % 4 * 4]);
#pragma unroll
        for (int c = 0; c < DT; ++c) {
          kh[c] = *reinterpret_cast<const bf16x8*>(&lds.k_hi[(before * 16 + l16) * RS + ch0 + c * 32 + quad * 8]);
          kl[c] = *reinterpret_cast<const bf16x8*>(&lds.k_lo[(before * 16 + l16) * RS + ch0 + c * 32 + quad * 8]);
        }
        split4(P, ph, pl);
#pragma unroll
        for (int g = 0; g < OT; ++g) {
          o[g] = mfma_16_half(v4[g], ph, o[g]);
          o[g] = mfma_16_half(v4[g], pl, o[g]);
        }
#pragma unroll
        for (int c = 0; c < DT; ++c) split8(q + c * 8, hi[c], lo[c]);
        if (--j < 0) {  // q is scaled to the start of the 64 tokens
#pragma unroll
          for (int g = 0; g < OT; ++g)
#pragma unroll
            for (int c = 0; c < DT; ++c) {
              const bf16x8 sh = *reinterpret_cast<const bf16x8*>(&lds.s_hi[(g * 16 + l16) * RS + ch0 + c * 32 + quad * 8]);
              const bf16x8 sl = *reinterpret_cast<const bf16x8*>(&lds.s_lo[(g * 16 + l16) * RS + ch0 + c * 32 + quad * 8]);
              o[g] = mfma_16(sh, hi[c], o[g]);
              o[g] = mfma_16(sl, hi[c], o[g]);
              o[g] = mfma_16(sh, lo[c], o[g]);
            }
          break;
        }
        P = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < DT; ++c) {
          P = mfma_16(kh[c], hi[c], P);
          P = mfma_16(kl[c], hi[c], P);
          P = mfma_16(kh[c], lo[c], P);
        }
#pragma unroll
        for (int i = 0; i < E; i += 4) {
          const f32x4 f = *reinterpret_cast<const f32x4*>(&lds.total[j][chan_of(i, quad)]);
#pragma unroll
          for (int e = 0; e < 4; ++e) q[i + e] *= f[e];
        }
      }
    }
    auto store = [&](const f32x4* x) {  // the tiles that this group finishes: 4 OF value channels side by side of each lane
      const int col = col_base + half * OF / 4 * 64 + quad * 16 + half * OF % 4 * 4;
      __bf16* to = static_cast<__bf16*>(a.o) + b * a.o_sb + (long)(chunk * kScanTokens + t) * a.o_sl + (long)h * a.dv + col;
      uint32_t y[2 * OF];
#pragma unroll
      for (int i = 0; i < 2 * OF; ++i) y[i] = pack_bf16(x[i / 2][i % 2 * 2], x[i / 2][i % 2 * 2 + 1]);
      if (!live) return;
      if constexpr (OF > 1) {
        if (a.wide) {
#pragma unroll
          for (int f = 0; f < OF / 2; ++f)
            if (col + f * 8 < a.dv) *reinterpret_cast<u32x4*>(to + f * 8) = u32x4{y[f * 4], y[f * 4 + 1], y[f * 4 + 2], y[f * 4 + 3]};
          return;
        }
      }
#pragma unroll
      for (int f = 0; f < OF; ++f)
        if (col + f * 4 < a.dv) *reinterpret_cast<u32x2*>(to + f * 4) = u32x2{y[f * 2], y[f * 2 + 1]};
    };
    if constexpr (!STATE_ONLY) {
      if constexpr (HALVES == 1) {
        store(o);
      } else {
#pragma unroll
        for (int other = 0; other < HALVES; ++other) {  // (of each group the tiles that it finishes; the others' parts in order of their groups)
          if (other == half) continue;
#pragma unroll
          for (int g = 0; g < OF; ++g)
            lds.part[(((blk * HALVES + other) * (HALVES - 1) + (half < other ? half : half - 1)) * OF + g) * 64 + here] = o[other * OF + g];
        }
      }
    }

    if constexpr (STATE_ONLY) {
      const int ch = threadIdx.x;
      if (ch < Lds::CH) seg_total *= (lds.total[0][ch] * lds.total[1][ch]) * (lds.total[2][ch] * lds.total[3][ch]);
    }
    if (has_cols) {  // the state behind the 64 tokens: what each 16 add, by themselves, and then one behind the other
      bf16x4 v4[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) v4[j] = read_transposed(&lds.v[(j * 16 + quad * 4 + tr_row) * VS + tile * 16 + tr_piece]);
#pragma unroll
      for (int ct = 0; ct < 2 * SP; ++ct) {
        f32x4 add[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int at = (j * 16 + quad * 4 + tr_row) * RS + (piece0 + (ct >> 1)) * 32 + (ct & 1) * 4 + tr_piece * 2;
          add[j] = mfma_16_half(read_transposed(&lds.k_hi[at]), v4[j], f32x4{0.f, 0.f, 0.f, 0.f});
          add[j] = mfma_16_half(read_transposed(&lds.k_lo[at]), v4[j], add[j]);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const f32x4 f = *reinterpret_cast<const f32x4*>(&lds.total[j][state_chan(ct, quad)]);
#pragma unroll
          for (int i = 0; i < 4; ++i) S[ct][i] = __builtin_fmaf(S[ct][i], f[i], add[j][i]);
        }
      }
    }
    lds_barrier();
    if constexpr (!STATE_ONLY && HALVES > 1) {
      f32x4 x[OF];
#pragma unroll
      for (int g = 0; g < OF; ++g) {
        x[g] = o[g];
#pragma unroll
        for (int own = 1; own < HALVES; ++own) x[g] = own == half ? o[own * OF + g] : x[g];
#pragma unroll
        for (int m = 0; m < HALVES - 1; ++m) x[g] += lds.part[(((blk * HALVES + half) * (HALVES - 1) + m) * OF + g) * 64 + here];
      }
      store(x);
    }
  }
  if constexpr (STATE_ONLY) {
    if (blockIdx.y == 0 && threadIdx.x < a.d) a.seg_lw[(bh * a.segs + sg) * a.dp + threadIdx.x] = seg_total;
  }
  if (!has_cols) return;
  float* to = st;
  if constexpr (STATE_ONLY) to = a.seg + ((bh * a.segs + sg) * a.dv + (col_in ? dv0 + l16 : 0)) * a.dp;
  if (STATE_ONLY || sg == a.segs - 1) {
#pragma unroll
    for (int ct = 0; ct < 2 * SP; ++ct) {
      const int ch = state_chan(ct, quad);
      if (col_in && ch < a.d) *reinterpret_cast<f32x4*>(to + ch) = S[ct];
    }
  }
}

// ---- head decays, bf16 ----
// HALVES wavefronts (1 or 2) share the key channels of 16 tokens, DT 32-channel pieces each (d <= 32 DT HALVES, d % 4 == 0), so
// that what a lane holds of a token stays in registers; their parts of P are added through LDS.  Channels of a piece are held by the lanes in the
// order of the accumulators: element e < 4 of a lane in 16-lane row `quad` is channel 4 quad + e, e >= 4
// channel 16 + 4 quad + e - 4; every contraction over channels uses that order on both sides.
template <int DT, int HALVES> struct HeadLds {
  static constexpr int CH = 32 * DT * HALVES, RS = CH + 8, TS = kScanTokens + 8;
  __bf16 q[kScanTokens * RS];
  union {
    __bf16 k[kScanTokens * RS];
    struct {
      __bf16 hi[kScanTokens * TS], lo[kScanTokens * TS];  // P, [t][s]
      f32x4 part[HALVES > 1 ? 4 * 4 * 64 : 1];            // the second half's part of P, as its lanes hold it
    } p;
  };
  __bf16 kt_hi[CH * TS], kt_lo[CH * TS];         // k decayed to the end of the 64 tokens, [channel][token]
  __bf16 vt[64 * HALVES * TS];                            // v, [channel][token]
};

template <int DT, int HALVES, bool STATE_ONLY, bool FOLD>
__global__ __launch_bounds__(256 * HALVES, 2) void decay_head_kernel(const DecayScanArgs a) {
  typedef HeadLds<DT, HALVES> Lds;
  constexpr int RS = Lds::RS, TS = Lds::TS, E = DT * 8, DA = DT * HALVES;
  extern __shared__ __attribute__((aligned(16))) char scan_lds[];
  Lds& lds = *reinterpret_cast<Lds*>(scan_lds);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l16 = lane & 15, quad = lane >> 4;
  const int blk = wave & 3, half = wave >> 2, ch0 = half * 32 * DT;  // this wavefront's 16 tokens of 64, and its key channels
  const int b = blockIdx.x / a.H, h = blockIdx.x % a.H, sg = blockIdx.z;
  const int col_base = blockIdx.y * 64 * HALVES, dv0 = col_base + wave * 16;
  const bool has_cols = dv0 < a.dv, col_in = dv0 + l16 < a.dv;
  const __bf16* qp = static_cast<const __bf16*>(a.q) + b * a.q_sb + (long)h * a.d;
  const __bf16* kp = static_cast<const __bf16*>(a.k) + b * a.k_sb + (long)h * a.d;
  const __bf16* vp = static_cast<const __bf16*>(a.v) + b * a.v_sb + (long)h * a.dv;
  const HeadPowers powers(a, h);
  const long bh = (long)b * a.H + h;
  float* st = a.state + (bh * a.dv + (col_in ? dv0 + l16 : 0)) * a.dp;

  // channel of element e of piece c
  auto chan = [&](int c, int f) { return ch0 + c * 32 + f * 16 + quad * 4; };
  auto chan_of = [&](int i) { return ch0 + (i >> 3) * 32 + ((i >> 2) & 1) * 16 + quad * 4 + (i & 3); };

  // state: tile ct holds key channels 16 ct + 4 quad + i of value channel dv0 + l16
  f32x4 S[2 * DA];
  {
    const long seg_row = (col_in ? dv0 + l16 : 0), seg_step = (long)a.dv * a.dp;
    const float* segs = a.seg + (bh * a.segs * a.dv + seg_row) * a.dp;
    // FOLD: what the segments in front have added is put together here, the state that enters the call from the last one's place, where
    // the state pass has left it (the last segment replaces it).  Kernels of their own: the others have registers for what they do.
    const bool fold = FOLD && !STATE_ONLY && a.segs > 1;
    const float* from = a.segs > 1 ? segs + (fold ? a.segs - 1 : sg) * seg_step : st;
    const bool zero = STATE_ONLY || ((a.segs == 1 || fold) && a.fresh);
#pragma unroll
    for (int ct = 0; ct < 2 * DA; ++ct) {
      const int ch = ct * 16 + quad * 4;
      S[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (!zero && col_in && ch < a.d) S[ct] = *reinterpret_cast<const f32x4*>(from + ch);
    }
    if constexpr (STATE_ONLY) {
      if (FOLD && !a.fresh && sg == 0 && col_in) {
        float* keep = a.seg + ((bh * a.segs + a.segs - 1) * a.dv + seg_row) * a.dp;
#pragma unroll
        for (int ct = 0; ct < 2 * DA; ++ct) {
          const int ch = ct * 16 + quad * 4;
          if (ch < a.d) *reinterpret_cast<f32x4*>(keep + ch) = *reinterpret_cast<const f32x4*>(st + ch);
        }
      }
    } else if (fold) {
      const float seg_decay = powers.of_state(a.seg_chunks * kScanTokens);  // (all in front of the last are of one length)
      constexpr int U = 4;  // segments asked for together
      for (int s0 = 0; s0 < sg; s0 += U) {
        f32x4 add[U][2 * DA];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int ct = 0; ct < 2 * DA; ++ct) {
            const int ch = ct * 16 + quad * 4 < a.d ? ct * 16 + quad * 4 : 0, s = s0 + u < sg ? s0 + u : sg - 1;
            add[u][ct] = *reinterpret_cast<const f32x4*>(segs + s * seg_step + ch);
          }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (s0 + u >= sg) break;  // (uniform)
#pragma unroll
          for (int ct = 0; ct < 2 * DA; ++ct)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const float sum = __builtin_fmaf(S[ct][j], seg_decay, add[u][ct][j]);
              S[ct][j] = col_in && ct * 16 + quad * 4 < a.d ? sum : 0.f;
            }
        }
      }
    }
  }
  struct Stage {
    bf16x4 q[STATE_ONLY ? 1 : 2 * DT], k[2 * DT], v[4];
  };
  const int first = sg * a.seg_chunks, chunks = (a.L + kScanTokens - 1) / kScanTokens;
  const int last = first + a.seg_chunks < chunks ? first + a.seg_chunks : chunks;
  // the rows of this wavefront's 16 tokens, unconditionally (places past the end are cleared at use): the place of the
  // 64 tokens is the same for all lanes, and what lies behind it fits 32 bits
  auto fetch = [&](Stage& s, int chunk) {
    const int left = a.L - chunk * kScanTokens, mine = blk * 16 + l16, t = mine < left ? mine : left - 1;
    const long t0 = (long)chunk * kScanTokens;
    const __bf16* q0 = qp + t0 * a.q_sl;
    const __bf16* k0 = kp + t0 * a.k_sl;
    const __bf16* v0 = vp + t0 * a.v_sl;
    const int tq = t * (int)a.q_sl, tk = t * (int)a.k_sl, tv = t * (int)a.v_sl;
#pragma unroll
    for (int g = 0; g < 2 * DT; ++g) {
      const int ch = chan(g >> 1, g & 1) < a.d ? chan(g >> 1, g & 1) : 0;
      if constexpr (!STATE_ONLY) s.q[g] = *reinterpret_cast<const bf16x4*>(q0 + (tq + ch));
      s.k[g] = *reinterpret_cast<const bf16x4*>(k0 + (tk + ch));
    }
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      const int col = col_base + half * 64 + quad * 16 + f * 4;
      s.v[f] = *reinterpret_cast<const bf16x4*>(v0 + (tv + (col < a.dv ? col : 0)));
    }
  };

  Stage cur;
  if (first < last) fetch(cur, first);
  // A head decay below zero: with w's sign s, s^t v_t in the place of v_t, s S in that of the state and s^t o_t in that of o_t, the powers are
  // those of |w| (4 x 2048 tokens, 16 heads of 64: 43.4 us, without signs at all 43.4; on the weights themselves 44.2, the state turned
  // in front of the first tokens 43.8).
  uint32_t odd_sign = 0u;  // of two halves, where this lane's token has an odd number
  auto turn_state = [&](bool turn) {
#pragma unroll
    for (int ct = 0; ct < 2 * DA; ++ct) S[ct] = turn ? -S[ct] : S[ct];
  };
  odd_sign = powers.w < 0.f && (l16 & 1) ? 0x80008000u : 0u;
  for (int chunk = first; chunk < last; ++chunk) {
    const int left = a.L - chunk * kScanTokens, n = left < kScanTokens ? left : kScanTokens;
    const int t = blk * 16 + l16;  // this lane's token
    const bool live = t < n;
    float q[STATE_ONLY ? 1 : E], k[E];
#pragma unroll
    for (int i = 0; i < E; ++i) {
      if constexpr (!STATE_ONLY) q[i] = to_f32(cur.q[i >> 2][i & 3]);
      k[i] = to_f32(cur.k[i >> 2][i & 3]);
    }
    if (a.silu) {  // (one branch for all of them)
#pragma unroll
      for (int i = 0; i < E; ++i) {
        if constexpr (!STATE_ONLY) q[i] = round_to<__bf16>(silu_exact(q[i]));
        k[i] = round_to<__bf16>(silu_exact(k[i]));
      }
    }
#pragma unroll
    for (int g = 0; g < 2 * DT; ++g) {
      const bool in = live && chan(g >> 1, g & 1) < a.d;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if constexpr (!STATE_ONLY) q[g * 4 + j] = in ? q[g * 4 + j] : 0.f;
        k[g * 4 + j] = in ? k[g * 4 + j] : 0.f;
      }
    }

    __builtin_amdgcn_sched_barrier(0);
    uint32_t vv[8];
    {
      float v[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) v[j] = to_f32(cur.v[j >> 2][j & 3]);
      if (a.silu) {
#pragma unroll
        for (int j = 0; j < 16; ++j) v[j] = silu_exact(v[j]);
      }
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        const bool in = live && col_base + half * 64 + quad * 16 + f * 4 < a.dv;
#pragma unroll
        for (int j = 0; j < 2; ++j) vv[f * 2 + j] = in ? pack_bf16(v[f * 4 + 2 * j], v[f * 4 + 2 * j + 1]) ^ odd_sign : 0u;
      }
    }
    if (chunk + 1 < last) fetch(cur, chunk + 1);
    lds_barrier();  // every wavefront is done with the 64 tokens before
#pragma unroll
    for (int j = 0; j < 8; ++j)
      store_pair(&lds.vt[(half * 64 + quad * 16 + 2 * j) * TS + t], &lds.vt[(half * 64 + quad * 16 + 2 * j + 1) * TS + t], vv[j]);
    {
      const float f = powers(n - 1 - t > 0 ? n - 1 - t : 0);
#pragma unroll
      for (int i = 0; i < E; i += 2) {
        uint32_t hi, lo;
        split2(k[i] * f, k[i + 1] * f, hi, lo);
        store_pair(&lds.kt_hi[chan_of(i) * TS + t], &lds.kt_hi[(chan_of(i) + 1) * TS + t], hi);
        store_pair(&lds.kt_lo[chan_of(i) * TS + t], &lds.kt_lo[(chan_of(i) + 1) * TS + t], lo);
      }
      if constexpr (!STATE_ONLY) {
#pragma unroll
        for (int c = 0; c < DT; ++c) {
          u32x4 q4, k4;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            q4[e] = pack_bf16(q[c * 8 + 2 * e], q[c * 8 + 2 * e + 1]);
            k4[e] = pack_bf16(k[c * 8 + 2 * e], k[c * 8 + 2 * e + 1]);
          }
          *reinterpret_cast<u32x4*>(&lds.k[t * RS + ch0 + c * 32 + quad * 8]) = k4;
          *reinterpret_cast<u32x4*>(&lds.q[t * RS + ch0 + c * 32 + quad * 8]) = q4;
        }
      }
    }
    lds_barrier();

    f32x4 P[STATE_ONLY ? 1 : 4];  // P^T tiles: column t of this wavefront's 16 tokens, rows s of 16 tokens j
    if constexpr (!STATE_ONLY) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        P[j] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (j > blk) continue;
#pragma unroll
        for (int c = 0; c < DT; ++c) {
          const bf16x8 k8 = *reinterpret_cast<const bf16x8*>(&lds.k[(j * 16 + l16) * RS + ch0 + c * 32 + quad * 8]);
          const bf16x8 q8 = *reinterpret_cast<const bf16x8*>(&lds.q[t * RS + ch0 + c * 32 + quad * 8]);
          P[j] = mfma_16(k8, q8, P[j]);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int dist = t - (j * 16 + quad * 4 + i);
          P[j][i] = dist >= 0 ? P[j][i] * powers(dist) : 0.f;
        }
      }
    }
    lds_barrier();  // k is not read any more: P goes into its place
    if constexpr (!STATE_ONLY) {
      if constexpr (HALVES > 1) {
        if (half == 1) {
#pragma unroll
          for (int j = 0; j < 4; ++j) lds.p.part[(blk * 4 + j) * 64 + lane] = P[j];
        }
        lds_barrier();
        if (half == 0) {
#pragma unroll
          for (int j = 0; j < 4; ++j) P[j] += lds.p.part[(blk * 4 + j) * 64 + lane];
        }
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;
        u32x2 hi, lo;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          uint32_t x, y;
          split2(P[j][2 * i], P[j][2 * i + 1], x, y);
          hi[i] = x, lo[i] = y;
        }
        if (half == 0 && j <= (blk | 1)) {
          *reinterpret_cast<u32x2*>(&lds.p.hi[t * TS + j * 16 + quad * 4]) = hi;
          *reinterpret_cast<u32x2*>(&lds.p.lo[t * TS + j * 16 + quad * 4]) = lo;
        }
      }
      lds_barrier();
    }
    if (has_cols) {
      bf16x8 v8[2];
#pragma unroll
      for (int g = 0; g < 2; ++g) v8[g] = *reinterpret_cast<const bf16x8*>(&lds.vt[(wave * 16 + l16) * TS + g * 32 + quad * 8]);
      if constexpr (!STATE_ONLY) {
        if (chunk == first && powers.w < 0.f) turn_state(true);  // (no sooner: the state is on its way until here)
        bf16x8 sh[DA], sl[DA];
#pragma unroll
        for (int c = 0; c < DA; ++c) {
          const float x[8] = {S[2 * c][0], S[2 * c][1], S[2 * c][2], S[2 * c][3], S[2 * c + 1][0], S[2 * c + 1][1], S[2 * c + 1][2], S[2 * c + 1][3]};
          split8(x, sh[c], sl[c]);
        }
        {  // (rounding leaves nothing of an infinity: the difference of two is no number)
          float most = 0.f;
#pragma unroll
          for (int ct = 0; ct < 2 * DA; ++ct)
#pragma unroll
            for (int j = 0; j < 4; ++j) most = fmaxf(most, fabsf(S[ct][j]));
          if (__any(most == INFINITY)) {
#pragma unroll
            for (int ct = 0; ct < 2 * DA; ++ct)
#pragma unroll
              for (int j = 0; j < 4; ++j) sl[ct / 2][ct % 2 * 4 + j] = fabsf(S[ct][j]) == INFINITY ? (__bf16)0.f : sl[ct / 2][ct % 2 * 4 + j];
          }
        }
#pragma unroll
        for (int tb = 0; tb < 4; ++tb) {
          if (tb > 0 && DA > 1) __builtin_amdgcn_sched_barrier(0);  // (one group's operands in registers at a time)
          const int tok = tb * 16 + l16;
          f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int c = 0; c < DA; ++c) {
            const bf16x8 qh = *reinterpret_cast<const bf16x8*>(&lds.q[tok * RS + c * 32 + quad * 8]);
            acc = mfma_16(sh[c], qh, acc);
            acc = mfma_16(sl[c], qh, acc);
          }
          acc *= powers.of_state(tok + 1);
#pragma unroll
          for (int g = 0; g < 2; ++g) {
            if (g * 2 > tb) continue;
            const bf16x8 ph = *reinterpret_cast<const bf16x8*>(&lds.p.hi[tok * TS + g * 32 + quad * 8]);
            const bf16x8 pl = *reinterpret_cast<const bf16x8*>(&lds.p.lo[tok * TS + g * 32 + quad * 8]);
            acc = mfma_16(v8[g], ph, acc);
            acc = mfma_16(v8[g], pl, acc);
          }
          if (tok < n && dv0 + quad * 4 < a.dv) {
            typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;
            const u32x2 out = {pack_bf16(acc[0], acc[1]) ^ odd_sign, pack_bf16(acc[2], acc[3]) ^ odd_sign};
            *reinterpret_cast<u32x2*>(static_cast<__bf16*>(a.o) + b * a.o_sb + (long)(chunk * kScanTokens + tok) * a.o_sl +
                                       (long)h * a.dv + dv0 + quad * 4) = out;
          }
        }
      }
      // the state behind the 64 tokens
#pragma unroll
      for (int ct = 0; ct < 2 * DA; ++ct) {
        if (HALVES > 1 && ct % 2 == 0) __builtin_amdgcn_sched_barrier(0);
        S[ct] *= powers.of_state(n);
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          const bf16x8 kh = *reinterpret_cast<const bf16x8*>(&lds.kt_hi[(ct * 16 + l16) * TS + g * 32 + quad * 8]);
          const bf16x8 kl = *reinterpret_cast<const bf16x8*>(&lds.kt_lo[(ct * 16 + l16) * TS + g * 32 + quad * 8]);
          S[ct] = mfma_16(kh, v8[g], S[ct]);
          S[ct] = mfma_16(kl, v8[g], S[ct]);
        }
      }
    }
  }
  if (!has_cols) return;
  turn_state(powers.w < 0.f && !(last == chunks && (a.L & 1)));  // (of an odd number of tokens the signs are turned already)
  float* to = st;
  if constexpr (STATE_ONLY) to = a.seg + ((bh * a.segs + sg) * a.dv + (col_in ? dv0 + l16 : 0)) * a.dp;
  if (STATE_ONLY || sg == a.segs - 1) {
#pragma unroll
    for (int ct = 0; ct < 2 * DA; ++ct) {
      const int ch = ct * 16 + quad * 4;
      if (col_in && ch < a.d) *reinterpret_cast<f32x4*>(to + ch) = S[ct];
    }
  }
}

// What each segment adds -> the state at its start, four key channels of a value channel per thread.
__global__ __launch_bounds__(256) void decay_join_kernel(const DecayScanArgs a) {
  const int pieces = a.dp / 4;
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= (long)a.B * a.H * a.dv * pieces) return;
  const int ch = (int)(i % pieces) * 4;
  const long row = i / pieces, bh = row / a.dv, col = row % a.dv;
  if (ch >= a.d) return;
  float* st = a.state + (bh * a.dv + col) * a.dp + ch;
  f32x4 S = {0.f, 0.f, 0.f, 0.f};
  if (!a.fresh) S = *reinterpret_cast<const f32x4*>(st);
  const float head = a.lw != nullptr ? 0.f : HeadPowers(a, (int)(bh % a.H)).of_state(a.seg_chunks * kScanTokens);
  for (int s = 0; s < a.segs; ++s) {
    float* p = a.seg + ((bh * a.segs + s) * a.dv + col) * a.dp + ch;
    f32x4 add = {0.f, 0.f, 0.f, 0.f};
    if (s + 1 < a.segs) add = *reinterpret_cast<const f32x4*>(p);
    *reinterpret_cast<f32x4*>(p) = S;
    if (s + 1 == a.segs) return;
    f32x4 l;
    if (a.lw != nullptr) {
      l = *reinterpret_cast<const f32x4*>(a.seg_lw + (bh * a.segs + s) * a.dp + ch);
    } else {
      l = f32x4{head, head, head, head};
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) S[j] = __builtin_fmaf(S[j], l[j], add[j]);
  }
}

// ---- any element type and size ----
// 16 lanes per value channel, groups of four channels of the key each; 16 value channels per workgroup.  Token by token, so what counts is
// the length of the chain and the workgroups beside each other: long portions go in segments, as on MFMA.  fp32, B = 1, H = 16,
// d = dv = 64, channel decays, L = 777: 43 us (one chain: 168); L = 2048: 80 (538).
// A lane's four channels lie side by side: states are read and written in whole pieces (element by element, four accesses of a quarter
// of each line: 32 x 4 heads of 256 x 256, L = 2, head decays, 17.8 us; 13.0 in pieces).
// kTile tokens are staged at once: 16, a barrier pair for each, where all workgroups are on the GPU together anyway, and 8 where keys of
// more than 128 channels would then keep some waiting for LDS, or where there are no more.  fp32, H = 4, d = dv = 256, channel decays, 16
// against 8: B = 64, L = 200: 894 us, 710; B = 16, L = 300: 444, 285; B = 1, L = 300: 72, 78.  64 x 12 heads of 128, L = 1: 18.5, 16.3.
template <typename T, int CPT, bool CHANNEL, bool STATE_ONLY, int kTile>
__global__ __launch_bounds__(256) void decay_scan_any_kernel(const DecayScanArgs a) {
  constexpr int CH = 16 * CPT;
  __shared__ __attribute__((aligned(16))) float sq[STATE_ONLY ? 1 : kTile][CH], sk[kTile][CH], sw[CHANNEL ? kTile : 1][CH];
  __shared__ float sv[kTile][16];
  const int tid = threadIdx.x, l16 = tid & 15, col = tid >> 4;
  const int b = blockIdx.x / a.H, h = blockIdx.x % a.H, dv0 = blockIdx.y * 16, sg = blockIdx.z;
  const bool col_in = dv0 + col < a.dv;
  const T* qp = static_cast<const T*>(a.q) + b * a.q_sb + (long)h * a.d;
  const T* kp = static_cast<const T*>(a.k) + b * a.k_sb + (long)h * a.d;
  const T* vp = static_cast<const T*>(a.v) + b * a.v_sb + (long)h * a.dv;
  const long bh = (long)b * a.H + h, row = col_in ? dv0 + col : 0;
  float* st = a.state + (bh * a.dv + row) * a.dp;
  float* sgp = a.segs > 1 ? a.seg + ((bh * a.segs + sg) * a.dv + row) * a.dp : nullptr;
  const float* from = a.segs > 1 ? sgp : st;
  const bool zero = STATE_ONLY || (a.segs == 1 && a.fresh);
  f32x4 S[CPT / 4], u[CPT / 4];
  float log2_all = 0.f;  // (state pass) what this thread stages of the decay over the segment: always of channel tid % CH
  static_assert(256 % CH == 0, "a thread stages one channel");
  const float head_w = CHANNEL ? 0.f : a.head_lw[a.H + h];
#pragma unroll
  for (int g = 0; g < CPT / 4; ++g) {
    const int c0 = g * 64 + l16 * 4;
    S[g] = !zero && col_in && c0 < a.d ? *reinterpret_cast<const f32x4*>(from + c0) : f32x4{0.f, 0.f, 0.f, 0.f};  // (rows are whole pieces)
#pragma unroll
    for (int j = 0; j < 4; ++j) S[g][j] = c0 + j < a.d ? S[g][j] : 0.f;
  }
  if constexpr (CHANNEL && !STATE_ONLY) {  // (rows of any alignment, through LDS)
    __shared__ __attribute__((aligned(16))) float s_u[CH];
    if (tid < CH) s_u[tid] = tid < a.d ? to_f32(static_cast<const T*>(a.u)[(long)h * a.d + tid]) : 0.f;
    __syncthreads();
#pragma unroll
    for (int g = 0; g < CPT / 4; ++g) u[g] = *reinterpret_cast<const f32x4*>(&s_u[g * 64 + l16 * 4]);
  }
  auto active = [&](T x) { return a.silu ? round_to<T>(silu_exact(to_f32(x))) : to_f32(x); };
  const int begin = sg * a.seg_chunks * kScanTokens;
  const int end = sg < a.segs - 1 ? begin + a.seg_chunks * kScanTokens : a.L;
  for (int t0 = begin; t0 < end; t0 += kTile) {
    const int n = end - t0 < kTile ? end - t0 : kTile;
    __syncthreads();
    for (int i = tid; i < kTile * CH; i += 256) {
      const int t = i / CH, c = i % CH;
      const bool in = t < n && c < a.d;
      if constexpr (!STATE_ONLY) sq[t][c] = in ? active(qp[(t0 + t) * a.q_sl + c]) : 0.f;
      sk[t][c] = in ? active(kp[(t0 + t) * a.k_sl + c]) : 0.f;
      if constexpr (CHANNEL) {
        const float lw = in ? a.lw[(((long)b * a.L + t0 + t) * a.H + h) * a.d + c] : 0.f;
        const float w = exp2f(lw);
        sw[t][c] = w;
        if constexpr (STATE_ONLY) log2_all += w == 0.f ? -INFINITY : lw;
      }
    }
    for (int i = tid; i < kTile * 16; i += 256) {
      const int t = i / 16, c = i % 16;
      sv[t][c] = t < n && dv0 + c < a.dv ? active(vp[(t0 + t) * a.v_sl + dv0 + c]) : 0.f;
    }
    __syncthreads();
    for (int t = 0; t < n; ++t) {
      const float v = sv[t][col];
      float o = 0.f;
#pragma unroll
      for (int g = 0; g < CPT / 4; ++g) {
        const int c = g * 64 + l16 * 4;
        const f32x4 k = *reinterpret_cast<const f32x4*>(&sk[t][c]);
        f32x4 q, w;
        if constexpr (!STATE_ONLY) q = *reinterpret_cast<const f32x4*>(&sq[t][c]);
        if constexpr (CHANNEL) w = *reinterpret_cast<const f32x4*>(&sw[t][c]);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float kv = k[j] * v;
          if constexpr (CHANNEL) {
            if constexpr (!STATE_ONLY) o = __builtin_fmaf(__builtin_fmaf(u[g][j], kv, S[g][j]), q[j], o);
            S[g][j] = __builtin_fmaf(w[j], S[g][j], kv);
          } else {
            S[g][j] = __builtin_fmaf(head_w, S[g][j], kv);
            if constexpr (!STATE_ONLY) o = __builtin_fmaf(S[g][j], q[j], o);
          }
        }
      }
      if constexpr (!STATE_ONLY) {
        o = sum16(o);
        if (l16 == 0 && col_in) static_cast<T*>(a.o)[b * a.o_sb + (t0 + t) * a.o_sl + (long)h * a.dv + dv0 + col] = from_f32<T>(o);
      }
    }
  }
  // (what lies behind the last channel is not written)
  if (STATE_ONLY ? col_in : col_in && sg == a.segs - 1) {
    float* to = STATE_ONLY ? sgp : st;
#pragma unroll
    for (int g = 0; g < CPT / 4; ++g) {
      const int c = g * 64 + l16 * 4;
      if (c + 3 < a.d) {
        *reinterpret_cast<f32x4*>(to + c) = S[g];
      } else {
#pragma unroll
        for (int j = 0; j < 3; ++j)
          if (c + j < a.d) to[c + j] = S[g][j];
      }
    }
  }
  if constexpr (CHANNEL && STATE_ONLY) {
    // the power of a sum of logarithms loses less than a product of decays that were each rounded
    if (blockIdx.y != 0) return;
    __syncthreads();
    float* sum = &sk[0][0];
    sum[tid] = log2_all;
    __syncthreads();
    if (tid >= CH || tid >= a.d) return;
    for (int i = tid + CH; i < 256; i += CH) log2_all += sum[i];
    const float all = exp2f(log2_all);
    a.seg_lw[(bh * a.segs + sg) * a.dp + tid] = all == 0.f && log2_all > -INFINITY ? 0x1p-149f : all;  // (decay_join_kernel)
  }
}

// ---- one token per sequence: one workgroup per (sequence, head) ----
struct DecayStepArgs {
  const void* q;
  const void* k;
  const void* v;
  const float* head_lw;
  const void* u;
  const void* hid;   // (B, R): the low-rank part of the channel decays before tanh
  const void* w2;    // (H * d, R)
  const void* w0;    // (H * d)
  const void* gate;  // (B, H * dv)
  const void* norm_w;
  float* state;
  void* o;
  const int32_t* pos;
  int pos_host;
  int B, H, d, dv, dp, R;
  long q_sb, k_sb, v_sb, h_sb, g_sb, o_sb;
  int silu;
  float eps;
};

// NT threads; LPR lanes per value channel, four key channels each; RPT value channels per thread.
template <typename T, int NT, int LPR, int RPT, bool CHANNEL>
__global__ __launch_bounds__(NT) void decay_step_kernel(const DecayStepArgs a) {
  extern __shared__ float smem[];
  constexpr int kRows = NT / LPR;  // value channels at a time
  const int tid = threadIdx.x, lane = tid & 63;
  const int b = blockIdx.x / a.H, h = blockIdx.x % a.H;
  const int pos = row_pos(a.pos, a.pos_host, b);
  if (pos < 0) return;
  float* sq = smem;             // [4 LPR], zeros behind d
  float* sk = sq + 4 * LPR;     // [4 LPR]
  float* sw = sk + 4 * LPR;     // [4 LPR]
  float* su = sw + 4 * LPR;     // [4 LPR]
  float* sv = su + 4 * LPR;     // [RPT * kRows]
  float* so = sv + RPT * kRows; // [RPT * kRows]
  float* th = so + RPT * kRows; // [R]
  // the state is asked for first
  const int piece = tid % LPR, r0 = tid / LPR, c0 = piece * 4;
  const bool in_c = c0 < a.d;
  float* st = a.state + ((long)b * a.H + h) * a.dv * a.dp;
  f32x4 S[RPT];
#pragma unroll
  for (int i = 0; i < RPT; ++i) {
    const int row = r0 + i * kRows;
    const bool in = in_c && row < a.dv;
    const f32x4 x = *reinterpret_cast<const f32x4*>(st + (in ? (long)row * a.dp + c0 : 0));
#pragma unroll
    for (int j = 0; j < 4; ++j) S[i][j] = in && pos > 0 && c0 + j < a.d ? x[j] : 0.f;
  }
  auto active = [&](T x) { return a.silu ? round_to<T>(silu_exact(to_f32(x))) : to_f32(x); };
  for (int c = tid; c < 4 * LPR; c += NT) {
    const bool in = c < a.d;
    const long at = (long)h * a.d + (in ? c : 0);
    const T xq = static_cast<const T*>(a.q)[b * a.q_sb + at], xk = static_cast<const T*>(a.k)[b * a.k_sb + at];
    sq[c] = in ? active(xq) : 0.f;
    sk[c] = in ? active(xk) : 0.f;
    if constexpr (CHANNEL) su[c] = in ? to_f32(static_cast<const T*>(a.u)[at]) : 0.f;
  }
  for (int c = tid; c < RPT * kRows; c += NT)
    sv[c] = c < a.dv ? active(static_cast<const T*>(a.v)[b * a.v_sb + (long)h * a.dv + c]) : 0.f;
  if constexpr (CHANNEL) {
    for (int j = tid; j < a.R; j += NT) th[j] = tanh_f(to_f32(static_cast<const T*>(a.hid)[b * a.h_sb + j]));
    __syncthreads();
    // four lanes per key channel
    for (int c = tid >> 2; c < 4 * LPR; c += NT / 4) {
      const bool in = c < a.d;
      const long at = (long)h * a.d + (in ? c : 0);
      const T* w = static_cast<const T*>(a.w2) + at * a.R;
      float z = 0.f;
      for (int j = tid & 3; j < a.R; j += 4) z = __builtin_fmaf(to_f32(w[j]), th[j], z);
      z += __shfl_xor(z, 1, 64);
      z += __shfl_xor(z, 2, 64);
      z += to_f32(static_cast<const T*>(a.w0)[at]);
      if ((tid & 3) == 0) sw[c] = in ? expf(-expf(z)) : 0.f;
    }
  }
  __syncthreads();
  float q[4], k[4], w[4], u[4];
  const float head_w = CHANNEL ? 0.f : a.head_lw[a.H + h];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    q[j] = sq[c0 + j], k[j] = sk[c0 + j];
    w[j] = CHANNEL ? sw[c0 + j] : head_w;
    u[j] = CHANNEL ? su[c0 + j] : 0.f;
  }
#pragma unroll
  for (int i = 0; i < RPT; ++i) {
    const int row = r0 + i * kRows;
    const float v = sv[row];
    float o = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float kv = k[j] * v;
      if constexpr (CHANNEL) {
        o = __builtin_fmaf(__builtin_fmaf(u[j], kv, S[i][j]), q[j], o);
        S[i][j] = __builtin_fmaf(w[j], S[i][j], kv);
      } else {
        S[i][j] = __builtin_fmaf(w[j], S[i][j], kv);
        o = __builtin_fmaf(S[i][j], q[j], o);
      }
    }
    if (in_c && row < a.dv) *reinterpret_cast<f32x4*>(st + (long)row * a.dp + c0) = S[i];
    if constexpr (LPR == 8) {
      o = sum8(o);
    } else if constexpr (LPR >= 16) {
      o = sum16(o);
      if constexpr (LPR >= 32) o += __shfl_xor(o, 16, 64);
      if constexpr (LPR >= 64) o += __shfl_xor(o, 32, 64);
    }
    if (piece == 0) so[row] = o;
  }
  __syncthreads();
  T* out = static_cast<T*>(a.o) + b * a.o_sb + (long)h * a.dv;
  if constexpr (CHANNEL) {
    float ss = 0.f;
    for (int c = lane; c < a.dv; c += 64) ss = __builtin_fmaf(so[c], so[c], ss);
    const float r = 1.0f / sqrtf(wave_sum(ss) / (float)a.dv + a.eps);
    const T* gate = static_cast<const T*>(a.gate) + b * a.g_sb + (long)h * a.dv;
    const T* nw = static_cast<const T*>(a.norm_w) + (long)h * a.dv;
    for (int c = tid; c < a.dv; c += NT) out[c] = from_f32<T>(so[c] * r * to_f32(nw[c]) * silu_exact(to_f32(gate[c])));
  } else {
    for (int c = tid; c < a.dv; c += NT) out[c] = from_f32<T>(so[c]);
  }
}

// ---- o / rms(o) * w * act(g) over groups of n elements of a row ----
struct GroupNormArgs {
  const void* o;
  const void* w;     // (G, n)
  const void* gate;
  void* y;
  long rows;         // B L G
  int L, G, n;
  long o_sb, o_sl, g_sb, g_sl, y_sb, y_sl;
  float eps, scale;
  int sigmoid;
};

template <typename T, bool VEC, int LPR>
__global__ __launch_bounds__(256) void group_norm_gate_kernel(const GroupNormArgs a) {
  constexpr int N = VEC ? Pack<T>::kN : 1;
  constexpr int KEEP = LPR == 64 ? 4 : 2;  // pieces of the row a lane keeps between the two passes
  const long row0 = (long)blockIdx.x * (256 / LPR) + threadIdx.x / LPR;
  const bool live = row0 < a.rows;
  const long row = live ? row0 : a.rows - 1;
  const int lane = threadIdx.x % LPR;
  const int g = (int)(row % a.G);
  const long bl = row / a.G, b = bl / a.L, l = bl % a.L;
  const T* o = static_cast<const T*>(a.o) + b * a.o_sb + l * a.o_sl + (long)g * a.n;
  const T* gate = static_cast<const T*>(a.gate) + b * a.g_sb + l * a.g_sl + (long)g * a.n;
  T* y = static_cast<T*>(a.y) + b * a.y_sb + l * a.y_sl + (long)g * a.n;
  const T* w = static_cast<const T*>(a.w) + (long)g * a.n;
  auto load = [&](const T* p, float (&x)[N]) {
    if constexpr (VEC)
      load_vec<T, N>(p, x);
    else
      x[0] = to_f32(*p);
  };
  float keep[KEEP][N], gk[KEEP][N], wk[KEEP][N];
#pragma unroll
  for (int i = 0; i < KEEP; ++i) {
    const int e = (lane + i * LPR) * N;
    load(o + (e < a.n ? e : 0), keep[i]);
    load(gate + (e < a.n ? e : 0), gk[i]);
    load(w + (e < a.n ? e : 0), wk[i]);
  }
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < KEEP; ++i)
#pragma unroll
    for (int j = 0; j < N; ++j) ss = (lane + i * LPR) * N < a.n ? __builtin_fmaf(keep[i][j], keep[i][j], ss) : ss;
  for (int e = (lane + KEEP * LPR) * N; e < a.n; e += LPR * N) {
    float x[N];
    load(o + e, x);
#pragma unroll
    for (int j = 0; j < N; ++j) ss = __builtin_fmaf(x[j], x[j], ss);
  }
  ss = LPR == 8 ? sum8(ss) : LPR == 16 ? sum16(ss) : wave_sum(ss);
  const float r = a.scale / sqrtf(ss / (float)a.n + a.eps);
  auto finish = [&](int e, const float (&x)[N], const float (&gv)[N], const float (&wv)[N]) {
    float out[N];
#pragma unroll
    for (int j = 0; j < N; ++j) out[j] = x[j] * r * wv[j] * (a.sigmoid ? sigmoid_f(gv[j]) : silu_exact(gv[j]));
    if (live) {
      if constexpr (VEC)
        store_vec<T, N>(y + e, out);
      else
        y[e] = from_f32<T>(out[0]);
    }
  };
#pragma unroll
  for (int i = 0; i < KEEP; ++i) {
    const int e = (lane + i * LPR) * N;
    if (e < a.n) finish(e, keep[i], gk[i], wk[i]);
  }
  for (int e = (lane + KEEP * LPR) * N; e < a.n; e += LPR * N) {
    float x[N], gv[N], wv[N];
    load(o + e, x);
    load(gate + e, gv);
    load(w + e, wv);
    finish(e, x, gv, wv);
  }
}

template <typename T, bool VEC> void launch_group_norm(const GroupNormArgs& a, hipStream_t s) {
  const int N = VEC ? Pack<T>::kN : 1;
  const int lpr = a.n <= 8 * N ? 8 : a.n <= 32 * N ? 16 : 64;
  const int per = 256 / lpr;
  const dim3 grid((unsigned)((a.rows + per - 1) / per)), block(256);
  if (lpr == 8)
    hipLaunchKernelGGL((group_norm_gate_kernel<T, VEC, 8>), grid, block, 0, s, a);
  else if (lpr == 16)
    hipLaunchKernelGGL((group_norm_gate_kernel<T, VEC, 16>), grid, block, 0, s, a);
  else
    hipLaunchKernelGGL((group_norm_gate_kernel<T, VEC, 64>), grid, block, 0, s, a);
}

void launch_decay_join(const DecayScanArgs& a, hipStream_t s) {
  const long items = (long)a.B * a.H * a.dv * (a.dp / 4);
  hipLaunchKernelGGL(decay_join_kernel, dim3((unsigned)((items + 255) / 256)), dim3(256), 0, s, a);
}

template <int DT, int HALVES, int COLS, bool CHANNEL, bool FOLD> int launch_decay_mfma(const DecayScanArgs& a, hipStream_t s) {
  void (*scan)(DecayScanArgs);
  void (*states)(DecayScanArgs);
  size_t bytes, state_bytes;
  if constexpr (CHANNEL) {
    typedef ChannelLds<DT, HALVES, COLS> Lds;
    scan = decay_channel_kernel<DT, HALVES, COLS, false, FOLD>, states = decay_channel_kernel<DT, HALVES, COLS, true, FOLD>;
    bytes = sizeof(Lds), state_bytes = offsetof(Lds, u);
  } else {
    static_assert(COLS == 64 * HALVES, "a wavefront has 16 value channels");
    scan = decay_head_kernel<DT, HALVES, false, FOLD>, states = decay_head_kernel<DT, HALVES, true, FOLD>;
    bytes = state_bytes = sizeof(HeadLds<DT, HALVES>);
  }
  static LdsAllowed scan_allowed, states_allowed;
  hipError_t e = allow_lds(reinterpret_cast<const void*>(scan), bytes, scan_allowed);
  if (e == hipSuccess && a.segs > 1) e = allow_lds(reinterpret_cast<const void*>(states), state_bytes, states_allowed);
  BASED_REQUIRE(e == hipSuccess, BASED_ERR_LAUNCH, "decay_scan: %zu bytes of LDS refused: %s", bytes, hipGetErrorString(e));
  dim3 grid((unsigned)(a.B * a.H), (unsigned)((a.dv + COLS - 1) / COLS), (unsigned)a.segs);
  if (a.segs > 1) {
    dim3 all_but_last = grid;
    all_but_last.z -= 1;
    hipLaunchKernelGGL(states, all_but_last, dim3(256 * HALVES), state_bytes, s, a);
    if (!FOLD) launch_decay_join(a, s);
  }
  hipLaunchKernelGGL(scan, grid, dim3(256 * HALVES), bytes, s, a);
  return BASED_OK;
}

// Channel decays.  Up to 64 channels: two wavefronts to the same 16 tokens, half of the channels each, where a SIMD would otherwise have fewer than
// two; beyond that one, which adds nothing up across wavefronts.
static bool channel_split(int64_t B, int64_t H, int64_t DV, int64_t segs, int64_t seg_chunks) {
  return B * H * ((DV + 63) / 64) * segs <= 384 || seg_chunks == 1;
}
// More channels: workgroups of 64 value channels where the 98 KB of each find a compute unit of their own, of 128 beyond that, and where the call has
// work space (by_channel) for twice the segments that way, each so much shorter that decays and keys worked out once for 128 channels count for
// more than the launch that puts segments together and the longer piece.  Calls, us, of 64 / of 128, 8 heads of 128 (pieces of a segment of
// 64): 1 x 4000 (4) 65 / 67; 4 x 1000 (4) 58.6 / 58.7; 6 x 500 (4) 52.3 / 52.0; 2 x 4000 (8) 100 / 88; 6 x 1000 (8) 93 / 80; 4 x 4000 (16) 175 / 141; 6 x
// 2426 (19) 204 / 138; in one, 10 x 700 (11) 83 / 81, 10 x 1472 (23) 166 / 136; 14 x 1100, one of 128 / two, 182 / 151.
static bool channel_narrow(int64_t B, int64_t L, int64_t H, int64_t DV, bool by_channel) {
  const int64_t wgs = B * H * ((DV + 63) / 64), chunks = (L + kScanTokens - 1) / kScanTokens;
  if (wgs > 256) return false;
  if (!by_channel || DV <= 64 || L < BASED_DECAY_SEGMENTS_MIN) return true;
  const int64_t segs = 256 / wgs;
  if (segs > 1) return (chunks + segs - 1) / segs < 7;
  return chunks < 16 || 256 / (B * H * ((DV + 127) / 128)) < 3;
}

// Whether an output may lie in the rows of q, k or v: workgroups of 128 value channels are the only ones of their head, those of 64 would write what
// others of it have yet to read.
static bool decay_rows_meet(const DecayScanArgs& a) {
  const auto span = [&](const void* p, long sb, long sl, long width, uintptr_t& lo, uintptr_t& hi) {
    const long b = (a.B - 1) * sb, l = (a.L - 1) * sl;
    lo = reinterpret_cast<uintptr_t>(p) + ((b < 0 ? b : 0) + (l < 0 ? l : 0)) * 2;
    hi = reinterpret_cast<uintptr_t>(p) + ((b < 0 ? 0 : b) + (l < 0 ? 0 : l) + width) * 2;
  };
  uintptr_t o0, o1;
  span(a.o, a.o_sb, a.o_sl, (long)a.H * a.dv, o0, o1);
  const auto meets = [&](const void* p, long sb, long sl, long width) {
    uintptr_t p0, p1;
    span(p, sb, sl, width, p0, p1);
    return p0 < o1 && o0 < p1;
  };
  return meets(a.q, a.q_sb, a.q_sl, (long)a.H * a.d) || meets(a.k, a.k_sb, a.k_sl, (long)a.H * a.d) || meets(a.v, a.v_sb, a.v_sl, (long)a.H * a.dv);
}

int launch_decay_head(const DecayScanArgs& a, bool fold, hipStream_t s) {
  if (a.d <= 32) return fold ? launch_decay_mfma<1, 1, 64, false, true>(a, s) : launch_decay_mfma<1, 1, 64, false, false>(a, s);
  if (a.d <= 64) return fold ? launch_decay_mfma<2, 1, 64, false, true>(a, s) : launch_decay_mfma<2, 1, 64, false, false>(a, s);
  return launch_decay_mfma<2, 2, 128, false, false>(a, s);
}

int launch_decay_channel(const DecayScanArgs& a, bool fold, hipStream_t s) {
  if (a.d <= 32) return fold ? launch_decay_mfma<1, 1, 64, true, true>(a, s) : launch_decay_mfma<1, 1, 64, true, false>(a, s);
  if (a.d <= 64) {
    if (channel_split(a.B, a.H, a.dv, a.segs, a.seg_chunks))
      return fold ? launch_decay_mfma<1, 2, 64, true, true>(a, s) : launch_decay_mfma<1, 2, 64, true, false>(a, s);
    return fold ? launch_decay_mfma<2, 1, 64, true, true>(a, s) : launch_decay_mfma<2, 1, 64, true, false>(a, s);
  }
  if (a.narrow) return fold ? launch_decay_mfma<2, 2, 64, true, true>(a, s) : launch_decay_mfma<2, 2, 64, true, false>(a, s);
  return launch_decay_mfma<2, 2, 128, true, false>(a, s);
}

template <typename T, int CPT, bool CHANNEL, int TOKENS> void launch_decay_any_tile(const DecayScanArgs& a, hipStream_t s) {
  const unsigned cols = (unsigned)((a.dv + 15) / 16);
  if (a.segs > 1) {
    hipLaunchKernelGGL((decay_scan_any_kernel<T, CPT, CHANNEL, true, TOKENS>), dim3((unsigned)(a.B * a.H), cols, (unsigned)(a.segs - 1)), dim3(256), 0,
                       s, a);
    launch_decay_join(a, s);
  }
  hipLaunchKernelGGL((decay_scan_any_kernel<T, CPT, CHANNEL, false, TOKENS>), dim3((unsigned)(a.B * a.H), cols, (unsigned)a.segs), dim3(256), 0, s, a);
}

template <typename T, int CPT, bool CHANNEL> void launch_decay_any(const DecayScanArgs& a, hipStream_t s) {
  // workgroups that the LDS of 256 compute units holds with 16 tokens: three of 49 KB to one, or four of 33 KB
  const bool many = CPT > 8 && (long)a.B * a.H * ((a.dv + 15) / 16) * a.segs > (CHANNEL ? 768 : 1024);
  if (many || a.L <= 8) return launch_decay_any_tile<T, CPT, CHANNEL, 8>(a, s);
  launch_decay_any_tile<T, CPT, CHANNEL, 16>(a, s);
}

template <typename T, bool CHANNEL> void launch_decay_scan_any(const DecayScanArgs& a, hipStream_t s) {
  if (a.d <= 64)
    launch_decay_any<T, 4, CHANNEL>(a, s);
  else if (a.d <= 128)
    launch_decay_any<T, 8, CHANNEL>(a, s);
  else
    launch_decay_any<T, 16, CHANNEL>(a, s);
}

template <typename T, int NT, int LPR, int RPT, bool CHANNEL> void launch_decay_step_block(const DecayStepArgs& a, hipStream_t s) {
  const size_t bytes = (size_t)(16 * LPR + 2 * RPT * (NT / LPR) + (CHANNEL ? a.R : 0)) * sizeof(float);
  hipLaunchKernelGGL((decay_step_kernel<T, NT, LPR, RPT, CHANNEL>), dim3((unsigned)(a.B * a.H)), dim3(NT), bytes, s, a);
}

// Few rows of the state per thread, so that all of it is in flight at once.
template <typename T, int LPR, bool CHANNEL> void launch_decay_step_rows(const DecayStepArgs& a, hipStream_t s) {
  auto rows = [&](int nt) { return (a.dv + nt / LPR - 1) / (nt / LPR); };
  if (rows(256) <= 2)
    launch_decay_step_block<T, 256, LPR, 2, CHANNEL>(a, s);
  else if (rows(256) <= 4)
    launch_decay_step_block<T, 256, LPR, 4, CHANNEL>(a, s);
  else if (rows(256) <= 8)
    launch_decay_step_block<T, 256, LPR, 8, CHANNEL>(a, s);
  else if (rows(512) <= 8)
    launch_decay_step_block<T, 512, LPR, 8, CHANNEL>(a, s);
  else
    launch_decay_step_block<T, 1024, LPR, 16, CHANNEL>(a, s);
}

template <typename T, bool CHANNEL> void launch_decay_step(const DecayStepArgs& a, hipStream_t s) {
  const int pieces = (a.d + 3) / 4;
  if (pieces <= 8)
    launch_decay_step_rows<T, 8, CHANNEL>(a, s);
  else if (pieces <= 16)
    launch_decay_step_rows<T, 16, CHANNEL>(a, s);
  else if (pieces <= 32)
    launch_decay_step_rows<T, 32, CHANNEL>(a, s);
  else
    launch_decay_step_rows<T, 64, CHANNEL>(a, s);
}

// Segments up to which those of the scan put the ones in front of them together themselves, heads of up to 64 channels, of more with channel decays
// and workgroups of 64 value channels: a launch less, and memory's answer to four (two) segments at a time in front of the scan, with channel decays
// also the segments' decays.  Workgroups of 128 value channels go with the launch always.  us with decay_join_kernel and without.  Channel decays, 16
// heads of 64: 4 x 2048 tokens (8 segments) 61.1, 58.8; 12 x 960 (4) 78.8, 70.4; 1 x 2304 (9) 38.9, 36.7; 2 x 768 (10) 25.9, 22.6; 1 x 2560 (10)
// 39.7, 37.7; beyond ten, 12 40.5, 39.1; 16 42.7, 42.5; 32 48.6, 53.3.  8 heads of 128: 4 x 500 (4) 39.1, 35.1; 2 x 1000 (8) 42.3, 40.0; 1 x 500 (8)
// 26.8, 27.5; 1 x 2000 (10) 57.6, 57.4; 2 x 700, 2 heads (11) 27.3, 30.5; 1 x 2000 (16) 45.4, 48.3; 1 x 4000 (16) 61.8, 66.4.  Head decays: 1 x 2560
// 32.3, 28.7; 1 x 3584 (14) 34.5, 32.5; 1 x 4096 35.3, 34.0.
constexpr int kFoldSegmentsChannel = 10, kFoldSegmentsHead = 16;

// Segments of a scan: enough workgroups to give every SIMD two wavefronts, none shorter than four pieces of 64 tokens.
static int decay_segments(int64_t B, int64_t L, int64_t H, int64_t D, int64_t DV) {
  const int64_t cols = D <= 64 ? 64 : 128, chunks = (L + kScanTokens - 1) / kScanTokens, wgs = B * H * ((DV + cols - 1) / cols);
  int64_t segs = ((D <= 64 ? 512 : 256) + wgs - 1) / wgs;
  if (segs > chunks / 4) segs = chunks / 4;
  if (segs > 64) segs = 64;
  return segs < 2 ? 1 : (int)segs;
}

// Those of a call that has work space by the rule of channel decays.  Where a compute unit has one workgroup, a piece of 64 tokens takes the scan about
// 4.5 us and the state pass 2, a launch and the folding of some segments 3: pieces by themselves pay from four of them on (2 x 440 tokens, 12 heads of
// 64, us in segments of 1, 2 and 4 pieces or in one: 16.8, 19.7, 30.1, 35.5; 5 x 320, 16 heads: 20.6, 20.3, 25.1, 27.0), as long as there are no more of
// them than put themselves together or they are of four pieces anyway (1 x 4096, 16 heads: 42.5 in 16 of four, 48.6 in 32 of two; between the two, 1 x
// 2560, 37.7 in ten of four, 32.3 in 14 of three).  Not where there are workgroups for every compute unit without them: every token but those of
// the last segment is walked twice.  In one / in two, 16 heads, by workgroups, of 300, 960 and 2048 tokens: 480 43.2 / 52.6, 117 / 131, 243 / 282; 448
// 43.6 / 52.0, 113 / 129, 232 / 276; 384 42.0 / 44.6, 112 / 105, 230 / 224; 320 41.7 / 43.5, 107 / 100, 227 / 203; 272 40.9 / 41.7, 107 / 98, 227 / 193:
// from some 500 tokens on two would be the better ones up to 384.
static int decay_channel_segments(int64_t B, int64_t L, int64_t H, int64_t D, int64_t DV) {
  if (L < BASED_DECAY_SEGMENTS_MIN) return 1;
  const int64_t chunks = (L + kScanTokens - 1) / kScanTokens;
  int64_t segs, most = chunks;
  if (D <= 64) {
    const int64_t wgs = B * H * ((DV + 63) / 64);
    segs = wgs <= 256 ? 768 / wgs : 1;
    most = chunks / 4 > kFoldSegmentsChannel ? chunks / 4 : kFoldSegmentsChannel;
  } else {  // (one workgroup to a compute unit.  1 x 2000, 8 heads of 128: 41.9 in 16 of two pieces, 55 in eight of four)
    segs = 256 / (B * H * (channel_narrow(B, L, H, DV, true) ? (DV + 63) / 64 : (DV + 127) / 128));
  }
  if (segs > most) segs = most;
  if (segs > chunks) segs = chunks;
  if (segs > 64) segs = 64;
  return segs < 2 ? 1 : (int)segs;
}

// The same for the general form: eight workgroups to a compute unit.  Every token but those of the last segment is walked twice, so the
// chain is two segments long: three segments ask for a third less at best, and the launches.  Segments where four are wanted, of which
// whole 64-token pieces may leave three, if the two are the shorter chain by more than the launches.  us in segments against one chain,
// channel decays: B = 1, H = 12, L = 250: 31 in four, 57; 8 x 16 heads of 64, in three, L = 257: 75, 73; L = 320: 78, 87; L = 384: 91, 105;
// 16 x 4 heads of 128, in three, L = 290: 121, 123; L = 320: 123, 127; 8 x 4 heads of 256 (head decays), L = 320: 177, 200.
static int decay_any_segments(int64_t B, int64_t L, int64_t H, int64_t DV) {
  const int64_t chunks = (L + kScanTokens - 1) / kScanTokens, wgs = B * H * ((DV + 15) / 16);
  int64_t segs = (2048 + wgs - 1) / wgs;
  if (segs > chunks) segs = chunks;
  if (segs > 64) segs = 64;
  if (segs < 4) return 1;
  const int64_t each = (chunks + segs - 1) / segs;
  if (2 * each * kScanTokens + 16 > L) return 1;
  return (int)((chunks + each - 1) / each);
}

// Whether the MFMA form takes a call: bf16 in whole 8-byte pieces (bits as based_decay_scan_work_of has them).
static bool decay_vec(int64_t bits, int64_t D, int64_t DV, int io_dtype) {
  return io_dtype == BASED_BF16 && D <= 128 && D % 4 == 0 && DV % 4 == 0 && bits % 8 == 0;
}

static int64_t decay_work(int64_t segs, int64_t B, int64_t H, int64_t DV, int64_t state_row) {
  return segs <= 1 ? 0 : B * H * segs * (DV + 1) * state_row;
}

}  // namespace based

extern "C" BASED_API int64_t based_decay_scan_work(int64_t B, int64_t L, int64_t H, int64_t D, int64_t DV, int64_t state_row) {
  if (B <= 0 || L <= 0 || H <= 0 || D <= 0 || DV <= 0) return 0;
  const int64_t mfma = based::decay_segments(B, L, H, D, DV), any = based::decay_any_segments(B, L, H, DV);
  return based::decay_work(mfma > any ? mfma : any, B, H, DV, state_row);
}

extern "C" BASED_API int64_t based_decay_scan_work_of(int64_t bits, int64_t B, int64_t L, int64_t H, int64_t D, int64_t DV, int64_t state_row,
                                                      int io_dtype) {
  using namespace based;
  if (B <= 0 || L < BASED_DECAY_SEGMENTS_MIN || H <= 0 || D <= 0 || DV <= 0) return 0;
  return decay_work(decay_vec(bits, D, DV, io_dtype) ? decay_segments(B, L, H, D, DV) : decay_any_segments(B, L, H, DV), B, H, DV, state_row);
}

// by_channel: the work space is of based_decay_scan_channels_work
static int decay_scan_call(bool by_channel, const void* q, const void* k, const void* v, const float* channel_log2, const float* head_decay,
                           const void* bonus, float* state, float* work, void* o, int64_t B, int64_t L, int64_t H, int64_t D, int64_t DV,
                           int64_t state_row, int64_t q_sb, int64_t q_sl, int64_t k_sb, int64_t k_sl, int64_t v_sb, int64_t v_sl, int64_t o_sb,
                           int64_t o_sl, int activation, int fresh, int io_dtype, void* stream) {
  using namespace based;
  BASED_REQUIRE(q && k && v && state && o, BASED_ERR_ARG, "decay_scan: null pointer argument");
  BASED_REQUIRE((channel_log2 != nullptr) != (head_decay != nullptr), BASED_ERR_ARG, "decay_scan: decays per channel or per head");
  BASED_REQUIRE((channel_log2 != nullptr) == (bonus != nullptr), BASED_ERR_ARG, "decay_scan: the bonus belongs to channel decays");
  BASED_REQUIRE(B >= 0 && L >= 0 && H > 0 && D > 0 && DV > 0, BASED_ERR_ARG, "decay_scan: bad sizes");
  BASED_REQUIRE(D <= 256, BASED_ERR_SHAPE, "decay_scan: key size %ld (at most 256)", (long)D);
  BASED_REQUIRE(state_row >= D && state_row % 4 == 0 && aligned_to(state, 16) && aligned_to(work, 16), BASED_ERR_ALIGN,
                "decay_scan: state rows must be whole 16-byte pieces");
  BASED_REQUIRE(activation == BASED_ACT_NONE || activation == BASED_ACT_SILU, BASED_ERR_ARG, "decay_scan: unknown activation");
  BASED_REQUIRE(io_dtype == BASED_BF16 || io_dtype == BASED_F32, BASED_ERR_DTYPE, "decay_scan: bad dtype");
  BASED_REQUIRE(B * H < (1ll << 31) && L < (1ll << 31) && DV < (1ll << 20), BASED_ERR_SHAPE, "decay_scan: grid too large");
  BASED_REQUIRE(q_sl < (1ll << 24) && k_sl < (1ll << 24) && v_sl < (1ll << 24) && H * D < (1ll << 24), BASED_ERR_SHAPE, "decay_scan: rows too long");
  if (B == 0 || L == 0) return BASED_OK;
  DecayScanArgs a{q,    k,    v,    channel_log2, head_decay, bonus, state, nullptr, nullptr, o,    (int)B, (int)L, (int)H, (int)D, (int)DV,
                  (int)state_row, q_sb, q_sl, k_sb, k_sl, v_sb, v_sl, o_sb, o_sl, 1, (int)((L + kScanTokens - 1) / kScanTokens),
                  activation == BASED_ACT_SILU, fresh, 0, channel_narrow(B, L, H, DV, by_channel)};
  hipStream_t s = static_cast<hipStream_t>(stream);
  const auto at = [](const void* p) { return (int64_t)reinterpret_cast<uintptr_t>(p); };
  const int64_t strides = q_sb | q_sl | k_sb | k_sl | v_sb | v_sl | o_sb | o_sl;
  const int64_t bits = at(q) | at(k) | at(v) | at(bonus) | at(o) | 2 * strides | at(channel_log2) / 2;
  const bool vec = decay_vec(bits, D, DV, io_dtype);
  const int segs = vec ? (by_channel ? decay_channel_segments : decay_segments)(B, L, H, D, DV) : work != nullptr ? decay_any_segments(B, L, H, DV) : 1;
  if (segs > 1) {
    BASED_REQUIRE(work != nullptr, BASED_ERR_ARG, "decay_scan: no work space");
    a.seg_chunks = (a.seg_chunks + segs - 1) / segs;
    a.segs = (int)(((L + kScanTokens - 1) / kScanTokens + a.seg_chunks - 1) / a.seg_chunks);
    a.seg = work;
    a.seg_lw = work + B * H * a.segs * DV * state_row;
  }
  if (a.narrow && DV > 64 && decay_rows_meet(a)) a.narrow = 0;
  const bool fold = vec && (D <= 64 || (channel_log2 != nullptr && a.narrow)) && a.segs > 1 &&
                    a.segs <= (channel_log2 != nullptr ? kFoldSegmentsChannel : kFoldSegmentsHead);
  a.wide = bits % 16 == 0 && D % 8 == 0 && DV % 8 == 0;
  if (vec) {
    const int rc = channel_log2 != nullptr ? launch_decay_channel(a, fold, s) : launch_decay_head(a, fold, s);
    if (rc != BASED_OK) return rc;
  } else if (io_dtype == BASED_BF16) {
    channel_log2 != nullptr ? launch_decay_scan_any<__bf16, true>(a, s) : launch_decay_scan_any<__bf16, false>(a, s);
  } else {
    channel_log2 != nullptr ? launch_decay_scan_any<float, true>(a, s) : launch_decay_scan_any<float, false>(a, s);
  }
  return check_launch("decay_scan");
}

extern "C" BASED_API int based_decay_scan(const void* q, const void* k, const void* v, const float* channel_log2, const float* head_decay,
                                          const void* bonus, float* state, float* work, void* o, int64_t B, int64_t L, int64_t H,
                                          int64_t D, int64_t DV, int64_t state_row, int64_t q_sb, int64_t q_sl, int64_t k_sb,
                                          int64_t k_sl, int64_t v_sb, int64_t v_sl, int64_t o_sb, int64_t o_sl, int activation, int fresh,
                                          int io_dtype, void* stream) {
  return decay_scan_call(false, q, k, v, channel_log2, head_decay, bonus, state, work, o, B, L, H, D, DV, state_row, q_sb, q_sl, k_sb, k_sl, v_sb,
                         v_sl, o_sb, o_sl, activation, fresh, io_dtype, stream);
}

extern "C" BASED_API int64_t based_decay_scan_channels_work(int64_t bits, int64_t B, int64_t L, int64_t H, int64_t D, int64_t DV,
                                                            int64_t state_row, int io_dtype) {
  using namespace based;
  if (B <= 0 || L < BASED_DECAY_SEGMENTS_MIN || H <= 0 || D <= 0 || DV <= 0) return 0;
  return decay_work(decay_vec(bits, D, DV, io_dtype) ? decay_channel_segments(B, L, H, D, DV) : decay_any_segments(B, L, H, DV), B, H, DV, state_row);
}

extern "C" BASED_API int based_decay_scan_channels(const void* q, const void* k, const void* v, const float* channel_log2, const void* bonus,
                                                   float* state, float* work, void* o, int64_t B, int64_t L, int64_t H, int64_t D, int64_t DV,
                                                   int64_t state_row, int64_t q_sb, int64_t q_sl, int64_t k_sb, int64_t k_sl, int64_t v_sb,
                                                   int64_t v_sl, int64_t o_sb, int64_t o_sl, int activation, int fresh, int io_dtype,
                                                   void* stream) {
  return decay_scan_call(true, q, k, v, channel_log2, nullptr, bonus, state, work, o, B, L, H, D, DV, state_row, q_sb, q_sl, k_sb, k_sl, v_sb, v_sl,
                         o_sb, o_sl, activation, fresh, io_dtype, stream);
}

extern "C" BASED_API int based_decay_step(const void* q, const void* k, const void* v, const float* head_decay, const void* bonus,
                                          const void* hidden, const void* w2, const void* w0, const void* gate, const void* norm_w,
                                          float* state, void* o, const int32_t* pos, int64_t pos_host, int64_t B, int64_t H, int64_t D,
                                          int64_t DV, int64_t state_row, int64_t R, int64_t q_sb, int64_t k_sb, int64_t v_sb,
                                          int64_t h_sb, int64_t g_sb, int64_t o_sb, int activation, float eps, int io_dtype,
                                          void* stream) {
  using namespace based;
  const bool channel = hidden != nullptr;
  BASED_REQUIRE(q && k && v && state && o, BASED_ERR_ARG, "decay_step: null pointer argument");
  BASED_REQUIRE(channel ? (bonus && w2 && w0 && gate && norm_w && R > 0) : head_decay != nullptr, BASED_ERR_ARG,
                "decay_step: decays are missing");
  BASED_REQUIRE(B >= 0 && H > 0 && D > 0 && DV > 0 && pos_host >= 0 && pos_host < (1ll << 31), BASED_ERR_ARG, "decay_step: bad sizes");
  BASED_REQUIRE(D <= 256 && DV <= 256 && R <= 1024, BASED_ERR_SHAPE, "decay_step: sizes %ld x %ld, rank %ld (at most 256, 256, 1024)",
                (long)D, (long)DV, (long)R);
  BASED_REQUIRE(state_row >= D && state_row % 4 == 0 && aligned_to(state, 16), BASED_ERR_ALIGN,
                "decay_step: state rows must be whole 16-byte pieces");
  BASED_REQUIRE(activation == BASED_ACT_NONE || activation == BASED_ACT_SILU, BASED_ERR_ARG, "decay_step: unknown activation");
  BASED_REQUIRE(io_dtype == BASED_BF16 || io_dtype == BASED_F32, BASED_ERR_DTYPE, "decay_step: bad dtype");
  BASED_REQUIRE(B * H < (1ll << 31), BASED_ERR_SHAPE, "decay_step: grid too large");
  if (B == 0) return BASED_OK;
  const DecayStepArgs a{q,   k,   v,    head_decay, bonus, hidden, w2, w0, gate, norm_w, state, o, pos, (int)pos_host, (int)B, (int)H,
                        (int)D, (int)DV, (int)state_row, (int)R, q_sb, k_sb, v_sb, h_sb, g_sb, o_sb, activation == BASED_ACT_SILU, eps};
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (io_dtype == BASED_BF16)
    channel ? launch_decay_step<__bf16, true>(a, s) : launch_decay_step<__bf16, false>(a, s);
  else
    channel ? launch_decay_step<float, true>(a, s) : launch_decay_step<float, false>(a, s);
  return check_launch("decay_step");
}

extern "C" BASED_API int based_group_norm_gate(const void* o, const void* weight, const void* gate, void* y, int64_t B, int64_t L,
                                               int64_t G, int64_t n, int64_t o_sb, int64_t o_sl, int64_t g_sb, int64_t g_sl,
                                               int64_t y_sb, int64_t y_sl, float eps, float scale, int activation, int io_dtype,
                                               void* stream) {
  using namespace based;
  BASED_REQUIRE(o && weight && gate && y, BASED_ERR_ARG, "group_norm_gate: null pointer argument");
  BASED_REQUIRE(B >= 0 && L >= 0 && G > 0 && n > 0, BASED_ERR_ARG, "group_norm_gate: bad sizes");
  BASED_REQUIRE(activation == BASED_ACT_SILU || activation == BASED_ACT_SIGMOID, BASED_ERR_ARG, "group_norm_gate: unknown activation");
  BASED_REQUIRE(io_dtype == BASED_BF16 || io_dtype == BASED_F32, BASED_ERR_DTYPE, "group_norm_gate: bad dtype");
  const int64_t rows = B * L * G;
  BASED_REQUIRE(rows < (1ll << 33), BASED_ERR_SHAPE, "group_norm_gate: grid too large");
  if (rows == 0) return BASED_OK;
  const GroupNormArgs a{o,    weight, gate, y,    (long)rows, (int)L, (int)G, (int)n, o_sb, o_sl, g_sb, g_sl, y_sb, y_sl, eps, scale,
                        activation == BASED_ACT_SIGMOID};
  const int p = io_dtype == BASED_BF16 ? 8 : 4;
  const bool vec = n % p == 0 && o_sb % p == 0 && o_sl % p == 0 && g_sb % p == 0 && g_sl % p == 0 && y_sb % p == 0 && y_sl % p == 0 &&
                   aligned_to(o, 16) && aligned_to(weight, 16) && aligned_to(gate, 16) && aligned_to(y, 16);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (io_dtype == BASED_BF16)
    vec ? launch_group_norm<__bf16, true>(a, s) : launch_group_norm<__bf16, false>(a, s);
  else
    vec ? launch_group_norm<float, true>(a, s) : launch_group_norm<float, false>(a, s);
  return check_launch("group_norm_gate");
}
