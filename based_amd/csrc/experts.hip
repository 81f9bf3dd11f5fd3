// Mixture of experts with sigmoid routing for gfx950.  Of E small gated feed-forwards a token takes the `top`
// with the largest scores s = sigmoid(W_router h); each reads s * h, and their outputs are added:
//   y = sum_e down_e(silu(gate_e(s h)) * up_e(s h))
// (s multiplies the sums of gate and up in fp32, which is the same thing.)
//
//   expert_route    scores in fp32, the choice, and for grouped products each choice's place among its
//                   expert's rows; a single workgroup (up to 32 tokens) also does what the next two do
//   expert_place    rows of every expert rounded up to tiles, which expert a tile belongs to, and the choices in
//                   that order
//   expert_gemm     MFMA product of a tile of 32 rows with its expert's matrices, gathered and scattered by that
//                   order: gate and up with the activation behind them, then down; expert_gemm_large: of 256 rows
//   expert_sum      the choices of a token added up (with one choice the product writes the token's row)
//   expert_route_row  the same for few tokens, with the norm in front of the layer
//   expert_f32      fp32: 16 choices of one expert at a time on fp32 MFMA
//   expert_rows     few tokens, or rows that are no whole 16-byte pieces: dot products, one choice at a time
#include "lds_limit.hpp"
#include "stream_common.hpp"

namespace based {

constexpr int kMaxExperts = 256;

struct RouteArgs {
  const void* h;  // (N, D)
  const void* w;  // (E, D)
  int32_t* ids;   // (N, top)
  float* scores;  // (N, top)
  int32_t* rank;  // (N, top) or null
  int32_t* counts;  // (E), with rank; zero on entry unless one workgroup does everything or there is hist
  int32_t* hist;    // choices of each expert in each workgroup's tokens (workgroups, E): ranks stay those among these tokens; or null
  // one workgroup for all tokens: the plan too
  int32_t* tile_first;
  int32_t* tile_expert;
  int32_t* order;
  int tile_rows;
  long n, h_sr;
  int D, E, top;
};

__device__ __forceinline__ f32x4 expert_mfma(bf16x8 a, bf16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }

// scan[e] becomes the sum of own of threads 0 .. e (own 0 from thread E on; up to 256).  By one wavefront where it has a lane for each.
__device__ __forceinline__ void sum_up(uint32_t own, uint32_t* scan, int E) {
  const int e = threadIdx.x;
  if (E <= 64) {
    if (e < 64) {
#pragma unroll
      for (int m = 1; m < 64; m <<= 1) {
        const uint32_t add = __shfl_up(own, m, 64);
        own += e >= m ? add : 0;
      }
      if (e < E) scan[e] = own;
    }
    __syncthreads();
    return;
  }
  if (e < 256) scan[e] = own;
  __syncthreads();
  for (int m = 1; m < 256; m <<= 1) {
    const uint32_t add = e < 256 && e >= m ? scan[e - m] : 0;
    __syncthreads();
    if (e < 256) scan[e] += add;
    __syncthreads();
  }
}

// Tiles of every expert from its count (of each its expert, 8 bits, and its rows), by threads 0 .. 255; scan: 256 ints of LDS.  Called by a whole workgroup.
__device__ __forceinline__ void plan_tiles(const int* counts, uint32_t* scan, int* first_of, int32_t* tile_first, int32_t* tile_expert, int E, int tile_rows) {
  const int e = threadIdx.x;
  const int tiles = e < E ? (counts[e] + tile_rows - 1) / tile_rows : 0;
  sum_up((uint32_t)tiles, scan, E);
  if (e < E) {
    const int first = (int)scan[e] - tiles;
    first_of[e] = first;
    if (tile_first != nullptr) tile_first[e] = first;
    if (tile_expert != nullptr)
      for (int t = 0; t < tiles; ++t) {
        const int left = counts[e] - t * tile_rows;
        tile_expert[first + t] = e | (left < tile_rows ? left : tile_rows) << 8;
      }
  }
  if (e == 0 && tile_first != nullptr) tile_first[E] = (int)scan[E - 1];
  __syncthreads();
}

// A score is no less than zero; less is what stays where all that is left to choose from are no numbers, and the choice is none either.
__device__ __forceinline__ float chosen_score(float best) { return best < 0.f ? __builtin_nanf("") : best; }

// ET: tiles of 16 experts (bf16 MFMA); 0: element by element.  NW wavefronts.  SPLIT: they share 16 TT tokens, a part of the row each;
// otherwise 16 tokens each.
template <typename T, int ET, int NW, bool SPLIT, int TT>
__global__ __launch_bounds__(64 * NW) void expert_route_kernel(const RouteArgs a) {
  constexpr int NT = 64 * NW, TOK = ET == 0 ? 16 : SPLIT ? 16 * TT : 16 * NW;
  extern __shared__ float logits[];  // [NW (SPLIT) or 1][TOK][E]
  __shared__ int hist[kMaxExperts], base[kMaxExperts];
  __shared__ uint32_t scan[256];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, quad = lane >> 4;
  const long n0 = (long)blockIdx.x * TOK;
  const int n = a.n - n0 < TOK ? (int)(a.n - n0) : TOK;
  for (int e = tid; e < a.E; e += NT) hist[e] = 0;
  if constexpr (ET > 0) {
    f32x4 acc[ET][TT];
#pragma unroll
    for (int t = 0; t < ET; ++t)
#pragma unroll
      for (int x = 0; x < TT; ++x) acc[t][x] = f32x4{0.f, 0.f, 0.f, 0.f};
    const __bf16* h[TT];
#pragma unroll
    for (int x = 0; x < TT; ++x) {
      const int tok = (SPLIT ? 0 : wave * 16) + x * 16 + l16;
      h[x] = static_cast<const __bf16*>(a.h) + (n0 + (tok < n ? tok : 0)) * a.h_sr;
    }
    const __bf16* w[ET];
#pragma unroll
    for (int t = 0; t < ET; ++t) {
      const int e = t * 16 + l16;
      w[t] = static_cast<const __bf16*>(a.w) + (long)(e < a.E ? e : 0) * a.D;
    }
    const int pieces = (a.D + 31) / 32, per = SPLIT ? (pieces + NW - 1) / NW : pieces;
    const int p0 = SPLIT ? wave * per : 0, p1 = p0 + per < pieces ? p0 + per : pieces;
    constexpr int PU = ET <= 4 ? 4 : 2;  // pieces whose loads are in flight together
    for (int p = p0; p < p1; p += PU) {
      bf16x8 x8[PU][TT], w8[PU][ET];
#pragma unroll
      for (int u = 0; u < PU; ++u) {
        const int c = (p + u) * 32 + quad * 8;
        const bool in = p + u < p1 && c < a.D;
#pragma unroll
        for (int x = 0; x < TT; ++x) x8[u][x] = *reinterpret_cast<const bf16x8*>(h[x] + (in ? c : 0));
#pragma unroll
        for (int t = 0; t < ET; ++t) w8[u][t] = *reinterpret_cast<const bf16x8*>(w[t] + (in ? c : 0));
      }
#pragma unroll
      for (int u = 0; u < PU; ++u) {
        const bool in = p + u < p1 && (p + u) * 32 + quad * 8 < a.D;
#pragma unroll
        for (int x = 0; x < TT; ++x) {
#pragma unroll
          for (int j = 0; j < 8; ++j) x8[u][x][j] = in ? x8[u][x][j] : (__bf16)0.f;
#pragma unroll
          for (int t = 0; t < ET; ++t) acc[t][x] = expert_mfma(w8[u][t], x8[u][x], acc[t][x]);
        }
      }
    }
    // column = token l16, rows = experts 4 quad + i
#pragma unroll
    for (int t = 0; t < ET; ++t)
#pragma unroll
      for (int x = 0; x < TT; ++x)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int e = t * 16 + quad * 4 + i;
          if (e < a.E) logits[((SPLIT ? wave * TOK : wave * 16) + x * 16 + l16) * a.E + e] = acc[t][x][i];
        }
    __syncthreads();
    for (int i = tid; i < TOK * a.E; i += NT) {
      float z = logits[i];
      if constexpr (SPLIT) {
#pragma unroll
        for (int v = 1; v < NW; ++v) z += logits[v * TOK * a.E + i];
      }
      logits[i] = 1.0f / (1.0f + expf(-z));
    }
  } else {
    for (int i = tid; i < TOK * a.E; i += NT) {
      const int t = i / a.E, e = i % a.E;
      const T* h = static_cast<const T*>(a.h) + (n0 + (t < n ? t : 0)) * a.h_sr;
      const T* w = static_cast<const T*>(a.w) + (long)e * a.D;
      float z = 0.f;
      for (int c = 0; c < a.D; ++c) z = __builtin_fmaf(to_f32(w[c]), to_f32(h[c]), z);
      logits[i] = 1.0f / (1.0f + expf(-z));
    }
  }
  __syncthreads();
  // 16 lanes per token
  const int sub = tid & 15;
  for (int t = tid >> 4; t < TOK; t += NT / 16) {
    float* s = logits + t * a.E;
    for (int j = 0; j < a.top; ++j) {
      float best = -2.f;
      int at = 0;
      for (int e = sub; e < a.E; e += 16)
        if (s[e] > best) best = s[e], at = e;
#pragma unroll
      for (int m = 8; m >= 1; m >>= 1) {
        const float ov = __shfl_xor(best, m, 16);
        const int oa = __shfl_xor(at, m, 16);
        if (ov > best || (ov == best && oa < at)) best = ov, at = oa;
      }
      if (at % 16 == sub) s[at] = -1.f;  // taken
      if (sub == 0 && t < n) {
        const long slot = (n0 + t) * a.top + j;
        a.ids[slot] = at;
        a.scores[slot] = chosen_score(best);
        if (a.rank != nullptr) a.rank[slot] = atomicAdd(&hist[at], 1);
      }
    }
  }
  if (a.rank == nullptr) return;
  __syncthreads();
  if (a.hist != nullptr) {
    for (int e = tid; e < a.E; e += NT) a.hist[(long)blockIdx.x * a.E + e] = hist[e];
    return;
  }
  if (a.order != nullptr) {
    plan_tiles(hist, scan, base, a.tile_first, a.tile_expert, a.E, a.tile_rows);
    for (int e = tid; e < a.E; e += NT) a.counts[e] = hist[e];
  } else {
    for (int e = tid; e < a.E; e += NT) base[e] = hist[e] > 0 ? atomicAdd(&a.counts[e], hist[e]) : 0;
    __syncthreads();
  }
  for (int t = tid >> 4; t < n; t += NT / 16) {
    if (sub != 0) continue;
    for (int j = 0; j < a.top; ++j) {
      const long slot = (n0 + t) * a.top + j;  // (this thread has written it)
      if (a.order != nullptr)
        a.order[(long)base[a.ids[slot]] * a.tile_rows + a.rank[slot]] = (int32_t)slot;
      else
        a.rank[slot] += base[a.ids[slot]];
    }
  }
}

// Few tokens: one workgroup each, router rows as whole lines.  With norm_w (bf16) the token's row is formed first: r = res_in + mult * x
// (fp32, into res_out), h = norm(r) * norm_w (into h_out).
struct RouteRowArgs {
  RouteArgs r;
  const float* res_in;
  float* res_out;
  const __bf16* norm_w;
  __bf16* h_out;
  float mult, eps;
  int kind;
};

constexpr int kRouteRowMax = 4096;  // channels

template <typename T> __global__ __launch_bounds__(512) void expert_route_row_kernel(const RouteRowArgs a) {
  constexpr int N = Pack<T>::kN;
  __shared__ __attribute__((aligned(16))) T row[kRouteRowMax];
  __shared__ float s[kMaxExperts], part[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, D = a.r.D, E = a.r.E;
  const long n = blockIdx.x;
  const T* x = static_cast<const T*>(a.r.h) + n * a.r.h_sr;
  if constexpr (sizeof(T) == 2) {
    const int e8 = tid * 8;
    const bool in = e8 < D;
    float v[8];
    load_vec<__bf16, 8>(x + (in ? e8 : 0), v);
    if (a.norm_w != nullptr) {
      float w8[8], r8[8];
      load_vec<__bf16, 8>(a.norm_w + (in ? e8 : 0), w8);
#pragma unroll
      for (int i = 0; i < 8; ++i) r8[i] = 0.f;
      if (a.res_in != nullptr) load_vec<float, 8>(a.res_in + n * D + (in ? e8 : 0), r8);
      const float mult = a.res_in != nullptr ? a.mult : 1.0f;
      float sum = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        v[i] = in ? __builtin_fmaf(mult, v[i], r8[i]) : 0.f;
        sum += v[i];
      }
      auto all = [&](float q, int at) {
        q = sum16(q);
        q += __shfl_xor(q, 16, 64);
        q += __shfl_xor(q, 32, 64);
        if (lane == 0) part[at + wave] = q;
        __syncthreads();
        float t = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) t += part[at + i];
        return t;
      };
      if (a.res_out != nullptr && in) store_vec<float, 8>(a.res_out + n * D + e8, v);
      const float mean = a.kind == BASED_NORM_LAYER ? all(sum, 0) / (float)D : 0.f;
      float ss = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        v[i] = in ? v[i] - mean : 0.f;
        ss = __builtin_fmaf(v[i], v[i], ss);
      }
      const float rstd = 1.0f / sqrtf(all(ss, 8) / (float)D + a.eps);
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] *= rstd * w8[i];
      if (in) store_vec<__bf16, 8>(a.h_out + n * D + e8, v);
    }
    if (in) store_vec<__bf16, 8>(row + e8, v);
  } else {
    for (int c = tid * N; c < D; c += 512 * N) *reinterpret_cast<f32x4*>(row + c) = *reinterpret_cast<const f32x4*>(x + c);
  }
  __syncthreads();
  constexpr int EU = 4;  // experts whose rows are in flight together
  for (int e0 = wave * EU; e0 < E; e0 += 8 * EU) {
    float acc[EU];
#pragma unroll
    for (int u = 0; u < EU; ++u) acc[u] = 0.f;
#pragma unroll 2
    for (int c = lane * N; c < D; c += 64 * N) {
      float h8[N];
      load_vec<T, N>(row + c, h8);
#pragma unroll
      for (int u = 0; u < EU; ++u) {
        float w8[N];
        load_vec<T, N>(static_cast<const T*>(a.r.w) + (long)(e0 + u < E ? e0 + u : 0) * D + c, w8);
#pragma unroll
        for (int i = 0; i < N; ++i) acc[u] = __builtin_fmaf(w8[i], h8[i], acc[u]);
      }
    }
#pragma unroll
    for (int u = 0; u < EU; ++u) {
      float z = sum16(acc[u]);
      z += __shfl_xor(z, 16, 64);
      z += __shfl_xor(z, 32, 64);
      if (lane == 0 && e0 + u < E) s[e0 + u] = 1.0f / (1.0f + expf(-z));
    }
  }
  __syncthreads();
  if (wave != 0) return;
  float mine[kMaxExperts / 64];
#pragma unroll
  for (int i = 0; i < kMaxExperts / 64; ++i) mine[i] = i * 64 + lane < E ? s[i * 64 + lane] : -4.f;  // (less than any: never chosen)
  for (int j = 0; j < a.r.top; ++j) {
    float best = -3.f;
    int at = 0;
#pragma unroll
    for (int i = 0; i < kMaxExperts / 64; ++i)
      if (mine[i] > best) best = mine[i], at = i * 64 + lane;
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) {
      const float ov = __shfl_xor(best, m, 64);
      const int oa = __shfl_xor(at, m, 64);
      if (ov > best || (ov == best && oa < at)) best = ov, at = oa;
    }
#pragma unroll
    for (int i = 0; i < kMaxExperts / 64; ++i) mine[i] = i * 64 + lane == at ? -2.f : mine[i];
    if (lane == 0) {
      a.r.ids[n * a.r.top + j] = at;
      a.r.scores[n * a.r.top + j] = chosen_score(best);
    }
  }
}

// Tiles of BASED_EXPERT_TILE_ROWS rows: whole ones first, by expert, then what is left of every expert, the most rows first, so that the last to be
// worked on are the smallest.  first_of: an expert's first whole tile; rest_of: the tile of what is left.  tile_first[0] is the number of whole ones.
// Many experts have few tiles each, and what is left of them, by itself and dealt out in columns, reads rows and matrices again that are not in its
// die's cache any more: there all tiles go by expert and count as whole.  Calls, us, rests last / by expert: 1 of 64 of 512, 8192 tokens 101 / 86; 4
// of 64 of 512, 6000 186 / 169; 2 of 64 of 1024, 6000 182 / 168; 4 of 128 of 512, 8192 293 / 262; 2 of 24 of 1024, 6000 126 / 118, 3000 87 / 88; 4 of
// 16 of 512, 8192 159.6 / 158.8, 3000 76 / 74; 2 of 8 of 1024, 8192 138.9 / 140.2, 3000 69 / 68.
constexpr int kManyExperts = 24;

__device__ __forceinline__ void plan_large_tiles(const int* counts, uint32_t* scan, int* first_of, int* rest_of, int32_t* tile_first, int32_t* tile_expert, int E) {
  constexpr int ROWS = BASED_EXPERT_TILE_ROWS;
  const int e = threadIdx.x;
  const int count = e < E ? counts[e] : 0, whole = count / ROWS, rest = count % ROWS;
  sum_up((uint32_t)whole << 9 | (rest > 0), scan, E);  // whole tiles (less than 2^23) and rests (up to 256) at once
  const int wholes = (int)(scan[E - 1] >> 9), rests = (int)(scan[E - 1] & 511);
  if (E >= kManyExperts) {
    if (e < E) {
      const int first = (int)((scan[e] >> 9) + (scan[e] & 511)) - whole - (rest > 0);
      first_of[e] = first;
      rest_of[e] = first + whole;
      if (tile_expert != nullptr) {
        for (int t = 0; t < whole; ++t) tile_expert[first + t] = e | ROWS << 8;
        if (rest > 0) tile_expert[first + whole] = e | rest << 8;
      }
    }
    if (e == 0 && tile_expert != nullptr) tile_first[0] = tile_first[E] = wholes + rests;
    __syncthreads();
    return;
  }
  if (e < E) {
    const int first = (int)(scan[e] >> 9) - whole;
    int rank = 0;
#pragma unroll 8
    for (int o = 0; o < E; ++o) rank += (counts[o] % ROWS << 8 | (255 - o)) > (rest << 8 | (255 - e));
    first_of[e] = first;
    rest_of[e] = wholes + rank;
    if (tile_expert != nullptr) {
      for (int t = 0; t < whole; ++t) tile_expert[first + t] = e | ROWS << 8;
      if (rest > 0) tile_expert[wholes + rank] = e | rest << 8;
    }
  }
  if (e == 0 && tile_expert != nullptr) tile_first[0] = wholes, tile_first[E] = wholes + rests;
  __syncthreads();
}

constexpr int kPlaceThreads = 512, kPlaceGroups = 8;  // of the routing's workgroups, that one places
constexpr long kPlaceHist = 1 << 15;                  // entries of hist up to which every workgroup may read all of it

struct PlaceArgs {
  int32_t* counts;
  const int32_t* hist;  // (groups, E); null: counts are there and ranks are those among all choices
  const int32_t* ids;
  const int32_t* rank;
  int32_t* tile_first;
  int32_t* tile_expert;
  int32_t* order;
  long slots;
  int E, tile_rows, groups, group_slots;
};

// Workgroup i places the choices of groups kPlaceGroups i ..; each of them plans the tiles for itself, which is less than another launch.  Bound by the
// loads that wait for each other, so choices and own counts are asked for in front.  8192 tokens, 2 of 8 experts: 4.7 us; group after
// group, and the tiles summed up by a whole workgroup, 7.2.
__global__ __launch_bounds__(kPlaceThreads) void expert_place_kernel(const PlaceArgs a) {
  __shared__ uint32_t scan[256];
  __shared__ int first_of[kMaxExperts], rest_of[kMaxExperts], total[kMaxExperts], base[kPlaceGroups][kMaxExperts];
  const int tid = threadIdx.x, g0 = blockIdx.x * kPlaceGroups;
  const int mine = a.groups - g0 < kPlaceGroups ? a.groups - g0 : kPlaceGroups;
  const long s0 = (long)g0 * a.group_slots;
  const int n = a.slots - s0 < (long)mine * a.group_slots ? (int)(a.slots - s0) : mine * a.group_slots;
  int id0 = 0, rank0 = 0, own[kPlaceGroups];
  if (tid < n) id0 = a.ids[s0 + tid], rank0 = a.rank[s0 + tid];
  static_assert(kMaxExperts <= kPlaceThreads, "");
#pragma unroll
  for (int g = 0; g < kPlaceGroups; ++g) own[g] = a.hist != nullptr && tid < a.E && g < mine ? a.hist[(long)(g0 + g) * a.E + tid] : 0;
  if (tid < a.E) {
    total[tid] = a.hist != nullptr ? 0 : a.counts[tid];
    base[0][tid] = 0;
  }
  __syncthreads();
  if (a.hist != nullptr) {
    int wide = 1;
    while (wide < a.E) wide <<= 1;
    const int e = tid & (wide - 1), runs = kPlaceThreads / wide;
    if (e < a.E) {
      int before = 0, sum = 0;
#pragma unroll 8
      for (int g = tid / wide; g < a.groups; g += runs) {
        const int c = a.hist[(long)g * a.E + e];
        sum += c;
        before += g < g0 ? c : 0;
      }
      if (sum != 0) atomicAdd(&total[e], sum);
      if (before != 0) atomicAdd(&base[0][e], before);
    }
    __syncthreads();
  }
  if (tid < a.E) {
    int at = base[0][tid];
#pragma unroll
    for (int g = 0; g < kPlaceGroups; ++g) {
      base[g][tid] = at;
      at += own[g];
    }
  }
  const bool large = a.tile_rows == BASED_EXPERT_TILE_ROWS, writes = blockIdx.x == 0;
  if (large)
    plan_large_tiles(total, scan, first_of, rest_of, a.tile_first, writes ? a.tile_expert : nullptr, a.E);
  else
    plan_tiles(total, scan, first_of, writes ? a.tile_first : nullptr, writes ? a.tile_expert : nullptr, a.E, a.tile_rows);
  if (writes && a.hist != nullptr && tid < a.E) a.counts[tid] = total[tid];
  for (int i = tid; i < n; i += kPlaceThreads) {
    const int e = i < kPlaceThreads ? id0 : a.ids[s0 + i], r = base[i / a.group_slots][e] + (i < kPlaceThreads ? rank0 : a.rank[s0 + i]);
    const bool rest = large && r >= total[e] / BASED_EXPERT_TILE_ROWS * BASED_EXPERT_TILE_ROWS;
    a.order[rest ? (long)rest_of[e] * BASED_EXPERT_TILE_ROWS + r % BASED_EXPERT_TILE_ROWS : (long)first_of[e] * a.tile_rows + r] = (int32_t)(s0 + i);
  }
}

__global__ __launch_bounds__(kMaxExperts) void expert_zero_kernel(int32_t* counts, int E) {
  if ((int)threadIdx.x < E) counts[threadIdx.x] = 0;
}

// ---- grouped products ----
struct ExpertGemmArgs {
  const __bf16* x;       // PAIRED: (N, K) rows gathered by order / top; otherwise (tiles * rows, K) in order
  const __bf16* w;       // PAIRED: (E, 2 F, K), up rows then gate rows; otherwise (E, F, K)
  __bf16* y;             // PAIRED: (tiles * rows, F); otherwise (slots, F) scattered by order
  const int32_t* order;
  const int32_t* tile_first;
  const int32_t* tile_expert;  // null: there is one expert (small tiles)
  const int32_t* counts;
  const float* scores;   // (slots), PAIRED
  long x_sr;
  int E, F, K, top, col_tiles, tiles;
};

constexpr int kGemmK = 64;
constexpr int kSmallWeights = 128;
constexpr int kBand = 8;

// Workgroups are dealt to the eight dies in turn: those of one die take neighbouring tiles, which share rows and matrices.
__device__ __forceinline__ int tile_of_block(int i, int n) {
  const int die = i & 7, k = i >> 3, per = n / 8, more = n % 8;
  return die * per + (die < more ? die : more) + k;
}

// 32 rows and 128 rows of the weights (PAIRED: half of them up, half gate) per workgroup, a wavefront 16 rows of each half of the weights; four rounds of
// 64 channels on their way from memory.  They are asked for in front of the products, which the compiler would put between them, with
// 32-bit offsets.
template <bool PAIRED> __global__ __launch_bounds__(256, 2) void expert_gemm_kernel(const ExpertGemmArgs a) {
  // rows of 128 bytes lie side by side, the eight 16-byte pieces of a row turned by half its number: neither the rows that
  // eight lanes write nor the sixteen that a tile reads meet a bank twice
  constexpr int BM = BASED_EXPERT_TILE_ROWS_SMALL, BN = kSmallWeights, AHEAD = 4, KS = kGemmK, MT = BM / 16, HALF = BN / 2;
  auto place = [](int r, int p) { return r * KS + ((p ^ (r >> 1)) & 7) * 8; };
  constexpr int AP = BM / 32, BP = BN / 32;  // 16-byte pieces per thread
  __shared__ __attribute__((aligned(16))) __bf16 xs[BM * KS], ws[BN * KS];
  __shared__ int slot_of[BM];
  // bands of kBand row tiles, walked down the rows first: what is in flight on a die shares its rows and its matrices
  const int id = tile_of_block(blockIdx.x, gridDim.x), band = id / (kBand * a.col_tiles), in_band = id % (kBand * a.col_tiles);
  const int deep = a.tiles - band * kBand < kBand ? a.tiles - band * kBand : kBand;
  const int tile = band * kBand + in_band % deep, f0 = in_band / deep * (PAIRED ? HALF : BN);
  if (tile >= a.tile_first[a.E]) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, quad = lane >> 4;
  int e = 0, rows = a.counts[0] - tile * BM;  // (of one expert)
  if (a.tile_expert != nullptr) {
    const int what = a.tile_expert[tile];
    e = what & 255, rows = what >> 8;
  } else {
    rows = rows < BM ? rows : BM;
  }
  for (int i = tid; i < BM; i += 256) slot_of[i] = a.order[(long)tile * BM + (i < rows ? i : 0)];
  lds_barrier();
  typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
  const int piece = (tid & 7) * 8;  // of the 64 channels of a round
  const __bf16* xrow[AP];
#pragma unroll
  for (int i = 0; i < AP; ++i) {
    const int r = i * 32 + (tid >> 3);
    xrow[i] = a.x + (PAIRED ? (long)(slot_of[r] / a.top) * a.x_sr : ((long)tile * BM + (r < rows ? r : 0)) * a.x_sr);
  }
  const __bf16* wbase = a.w + (long)e * (PAIRED ? 2 * a.F : a.F) * a.K;
  uint32_t wrow[BP];  // bytes
#pragma unroll
  for (int i = 0; i < BP; ++i) {
    const int r = i * 32 + (tid >> 3);
    const int f = PAIRED ? f0 + (r % HALF) : f0 + r;
    wrow[i] = (uint32_t)(((PAIRED && r >= HALF ? a.F : 0) + (f < a.F ? f : a.F - 1)) * a.K) * 2u;
  }
  u32x4 xb[AHEAD][AP], wb[AHEAD][BP];
  const u32x4 zero = {0u, 0u, 0u, 0u};
  auto fetch = [&](int k0, u32x4 (&x)[AP], u32x4 (&w)[BP]) {
    const int c = k0 + piece < a.K ? k0 + piece : 0;
#pragma unroll
    for (int i = 0; i < AP; ++i) x[i] = *reinterpret_cast<const u32x4*>(xrow[i] + c);
#pragma unroll
    for (int i = 0; i < BP; ++i) w[i] = *reinterpret_cast<const u32x4*>(reinterpret_cast<const char*>(wbase) + (wrow[i] + (uint32_t)c * 2u));
    __builtin_amdgcn_sched_barrier(0);  // (the products would otherwise be put in front of most of them)
  };
  f32x4 acc[2][MT];
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[p][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto stage = [&](int k0, const u32x4 (&x)[AP], const u32x4 (&w)[BP]) {
    const bool in = k0 + piece < a.K;
#pragma unroll
    for (int i = 0; i < AP; ++i) *reinterpret_cast<u32x4*>(&xs[place(i * 32 + (tid >> 3), tid & 7)]) = in ? x[i] : zero;
#pragma unroll
    for (int i = 0; i < BP; ++i) *reinterpret_cast<u32x4*>(&ws[place(i * 32 + (tid >> 3), tid & 7)]) = w[i];
  };
  auto multiply = [&]() {
#pragma unroll
    for (int kk = 0; kk < kGemmK; kk += 32) {
      bf16x8 xf[MT];
#pragma unroll
      for (int j = 0; j < MT; ++j) xf[j] = *reinterpret_cast<const bf16x8*>(&xs[place(j * 16 + l16, kk / 8 + quad)]);
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const bf16x8 wf = *reinterpret_cast<const bf16x8*>(&ws[place(p * HALF + wave * 16 + l16, kk / 8 + quad)]);
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[p][j] = expert_mfma(wf, xf[j], acc[p][j]);
      }
    }
  };
#pragma unroll
  for (int s = 0; s < AHEAD; ++s) fetch(s * kGemmK, xb[s], wb[s]);
  // (rounds past the end multiply by zeros: every stage of the loops is the same)
  for (int k00 = 0; k00 < a.K; k00 += AHEAD * kGemmK) {
#pragma unroll
    for (int s = 0; s < AHEAD; ++s) {
      const int k0 = k00 + s * kGemmK;
      lds_barrier();
      stage(k0, xb[s], wb[s]);
      lds_barrier();
      fetch(k0 + AHEAD * kGemmK, xb[s], wb[s]);
      multiply();
    }
  }
  // column = row l16 of the tile's rows, rows = features 4 quad + i
#pragma unroll
  for (int j = 0; j < MT; ++j) {
    const int r = j * 16 + l16;
    if (r >= rows) continue;
    const int slot = slot_of[r];
    if constexpr (PAIRED) {
      const float s = a.scores[slot];
      const int f = f0 + wave * 16 + quad * 4;
      if (f < a.F) {
        bf16x4 o;
#pragma unroll
        for (int m = 0; m < 4; ++m) o[m] = (__bf16)(silu_exact(acc[1][j][m] * s) * (acc[0][j][m] * s));
        *reinterpret_cast<bf16x4*>(a.y + ((long)tile * BM + r) * a.F + f) = o;
      }
    } else {
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const int f = f0 + p * HALF + wave * 16 + quad * 4;
        if (f < a.F) {
          bf16x4 o;
#pragma unroll
          for (int m = 0; m < 4; ++m) o[m] = (__bf16)acc[p][j][m];
          *reinterpret_cast<bf16x4*>(a.y + (long)slot * a.F + f) = o;
        }
      }
    }
  }
}

// ---- the same with tiles of 256 rows and 256 rows of the weights (PAIRED: 128 up, 128 gate), rows and weights straight into LDS ----
// One workgroup of eight wavefronts to a compute unit.  Whole tiles are dealt to the dies in runs, the rests of the experts behind them, the smallest
// last (of many experts each in its place, plan_large_tiles); what is left of a die's tiles after whole rounds of its compute units goes in parts, of
// 64 rows that are there and, where that gives every part a compute unit of its own, of 128 or 64 rows of the weights.  8192 tokens of 1024 channels,
// 2 of 8 experts of 1024: 70 + 43 us (rests in their experts' places, and parts of rows alone: 77 + 48; tiles of 128 x 256 through registers, two
// workgroups to a compute unit: 106 + 70); 2048 rows to every expert, whole rounds alone, 65 + 39.  Calls in a recorded graph, us, before and now, in
// turn: 8192 tokens 150 -> 136, 4096 94 -> 88.5, 1000 51 -> 47, 500 43 -> 36.7; 1 of 8 of 2048, 1000 54 -> 45; 4 of 16 of 512, 2000 71.5 -> 68.5.  A
// whole tile alone takes 29 us: its matrix instructions 22, at the rate that they reach by themselves here (1.6 PFLOP/s), the rest in front of the
// first and behind the last.
constexpr int kLargeRows = BASED_EXPERT_TILE_ROWS;
constexpr int kDies = 8, kDieUnits = 32;
constexpr int kHalf = 128 * kGemmK;  // elements of 128 rows of a round
constexpr int kMaxParts = 16;
constexpr int kPartElements = 9 * kHalf;
constexpr int kLargeLds = kPartElements * 2 + 2 * kLargeRows * 4;  // bytes; whole tiles use 8 kHalf of the elements; choices and their scores behind them

struct ExpertTile {
  const __bf16* w;  // matrices of the tile's expert
  long first;       // first row of the tile among all tiles
  int rows, f0;     // rows that are there, first feature
};

// 16 bytes a lane, side by side from dst on.  TAIL: zeros where the lane's piece (from channel c on) is past the last channel; a row has pieces
// in front of it too, so that the load is always counted.
template <bool TAIL> __device__ __forceinline__ void load_to_lds(const __bf16* src, __bf16* dst, int c, int channels) {
  if (TAIL && c >= channels) {
    *reinterpret_cast<bf16x8*>(dst + (threadIdx.x & 63) * 8) = bf16x8{};
    return;
  }
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src, (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}

// the weights' row (of the expert's matrices) behind row r of CW
template <bool PAIRED, int CW = 256> __device__ __forceinline__ uint32_t large_w_row(const ExpertGemmArgs& a, int f0, int r) {
  const int f = f0 + (PAIRED ? r % (CW / 2) : r);
  return (uint32_t)((PAIRED && r >= CW / 2 ? a.F : 0) + (f < a.F ? f : a.F - 1));
}

template <bool PAIRED> __device__ __forceinline__ const __bf16* large_x_row(const ExpertGemmArgs& a, const ExpertTile& t, const int* slot_of, int r) {
  return a.x + (PAIRED ? (long)(slot_of[r] / a.top) * a.x_sr : (t.first + (r < t.rows ? r : 0)) * a.x_sr);
}

// scores of a tile's rows (PAIRED), in LDS behind their choices
__device__ __forceinline__ const float* large_scores(const int* slot_of) { return reinterpret_cast<const float*>(slot_of + kLargeRows); }

// four features of one row from their sums u (PAIRED: of up, and g of gate)
template <bool PAIRED> __device__ __forceinline__ void large_store(const ExpertGemmArgs& a, __bf16* y, int f, float score, f32x4 u, f32x4 g) {
  if (f >= a.F) return;
  bf16x4 o;
#pragma unroll
  for (int m = 0; m < 4; ++m) o[m] = PAIRED ? (__bf16)(silu_exact(g[m] * score) * (u[m] * score)) : (__bf16)u[m];
  *reinterpret_cast<bf16x4*>(y + f) = o;
}

// A whole tile, two rounds of 64 channels in LDS.  A round is four halves of 128 rows, x0, x1, w0, w1; a wavefront has 64 rows of a half of x
// and 32 of a half of w, and goes through the products of the halves as phases of 16 matrix instructions
//   0: x0 w0    1: x0 w1    2: x1 w1    3: x1 w0
// while it reads from LDS what the next phase multiplies (w1, x1, the next round's x0, its w0) and asks memory for the half whose place
// became free a phase before (w0, w1, x1 of the round after the next, x0 of the one behind it), seven phases ahead of the phase that reads it.
// One barrier a phase; the wait in front of it leaves the loads of six phases on their way.  The compiler, which knows of no distance between
// these loads and reads of LDS, would wait for all of them in front of every read: it does for a static array (148 us where this takes 94), not for one
// whose extent the launch gives.
// TAIL: the last round of channels is no whole one.  It comes by itself behind the others, nothing else on its way any more.  8192 tokens, 2 of 8 experts,
// 1000 channels and features: 159 us a call, everything in parts of 128 or 64 rows 204; 32,768 tokens, 1032 channels, 520 features 363 and 465.
template <bool PAIRED, bool TAIL>
__device__ __forceinline__ void large_whole_tile(const ExpertGemmArgs& a, const ExpertTile& t, __bf16* lds, const int* slot_of) {
  constexpr int KS = kGemmK;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, quad = lane >> 4;
  const int wm = wave & 1, wn = wave >> 1;
  // a wavefront's two loads of a half: rows 16 wave + 8 i + lane / 8, whose eight pieces lie turned by half the row's number
  const int row = wave * 16 + (lane >> 3), piece = (lane ^ (lane >> 4)) & 7;  // (i = 1: the piece's bit 2 the other way round)
  const __bf16* xrow[2][2];
  uint32_t wrow[2][2];  // bytes
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = h * 128 + row + 8 * i;
      int c = (piece ^ (4 * i)) * 8;
      if (TAIL && c >= a.K) c = 0;  // (no whole round: what is asked for in its place lies in the row)
      xrow[h][i] = large_x_row<PAIRED>(a, t, slot_of, r) + c;
      wrow[h][i] = (large_w_row<PAIRED>(a, t.f0, r) * (uint32_t)a.K + (uint32_t)c) * 2u;
    }
  const int rounds = a.K / KS;
  auto ask = [&](int half, int at_round) {  // half 0, 1: x; 2, 3: w
    __bf16* at = lds + (at_round & 1) * 4 * kHalf + half * kHalf + wave * 16 * KS;
    const int round = at_round < rounds ? at_round : 0;  // (asked for and never read)
#pragma unroll
    for (int i = 0; i < 2; ++i)
      load_to_lds<false>(half < 2 ? xrow[half & 1][i] + round * KS
                                 : reinterpret_cast<const __bf16*>(reinterpret_cast<const char*>(t.w + round * KS) + wrow[half & 1][i]),
                        at + i * 8 * KS, 0, 0);
  };
  // fragments: rows l16 of a tile of 16, channels 32 kk + 8 quad ..
  bf16x8 x0[4][2], x1[4][2], wa[2][2], wb[2][2];
  const int turned = (l16 >> 1) & 7, p0 = (quad ^ turned) * 8, p1 = ((4 + quad) ^ turned) * 8;
  auto read_x = [&](int round, int h, bf16x8 (&f)[4][2]) {
    const __bf16* at = lds + (round & 1) * 4 * kHalf + h * kHalf + (wm * 64 + l16) * KS;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f[j][0] = *reinterpret_cast<const bf16x8*>(at + j * 16 * KS + p0);
      f[j][1] = *reinterpret_cast<const bf16x8*>(at + j * 16 * KS + p1);
    }
  };
  auto read_w = [&](int round, int h, bf16x8 (&f)[2][2]) {
    const __bf16* at = lds + (round & 1) * 4 * kHalf + (2 + h) * kHalf + (wn * 32 + l16) * KS;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      f[j][0] = *reinterpret_cast<const bf16x8*>(at + j * 16 * KS + p0);
      f[j][1] = *reinterpret_cast<const bf16x8*>(at + j * 16 * KS + p1);
    }
  };
  f32x4 acc[2][2][2][4];  // [half of x][half of w][16 features][16 rows]
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[h][g][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](const bf16x8 (&x)[4][2], const bf16x8 (&w)[2][2], f32x4 (&c)[2][4], int kk) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) c[i][j] = expert_mfma(w[i][kk], x[j][kk], c[i][j]);
  };
  // 16 products with the loads of a half in the middle; then own reads are done and own loads of all but six phases have landed (lgkmcnt 0,
  // vmcnt 12)
  auto phase = [&](const bf16x8 (&x)[4][2], const bf16x8 (&w)[2][2], f32x4 (&c)[2][4], int half, int round) {
    __builtin_amdgcn_sched_barrier(0);
    multiply(x, w, c, 0);
    __builtin_amdgcn_sched_barrier(0);
    ask(half, round);
    __builtin_amdgcn_sched_barrier(0);
    multiply(x, w, c, 1);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0070 | 12);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  // w0 of the round lies in wu; its w1 comes into wv, and the next round's w0 there again
  auto round_of = [&](int round, bf16x8 (&wu)[2][2], bf16x8 (&wv)[2][2]) {
    read_w(round, 1, wv);
    phase(x0, wu, acc[0][0], 2, round + 2);
    read_x(round, 1, x1);
    phase(x0, wv, acc[0][1], 3, round + 2);
    read_x(round + 1, 0, x0);
    phase(x1, wv, acc[1][1], 1, round + 2);
    read_w(round + 1, 0, wv);
    phase(x1, wu, acc[1][0], 0, round + 3);
  };
  ask(0, 0), ask(2, 0), ask(3, 0), ask(1, 0), ask(0, 1), ask(2, 1), ask(3, 1), ask(1, 1);
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(0x0070 | 10);  // x0, w0 and w1 of round 0
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  read_x(0, 0, x0);
  read_w(0, 0, wa);
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt 0
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  ask(0, 2);
  for (int round = 0; round + 1 < rounds; round += 2) {
    round_of(round, wa, wb);
    round_of(round + 1, wb, wa);
  }
  if (rounds & 1) round_of(rounds - 1, wa, wb);
  __builtin_amdgcn_s_waitcnt(0x0070);  // (nothing may come into LDS that is no longer this workgroup's)
  if constexpr (TAIL) {
    __builtin_amdgcn_s_barrier();  // every wavefront's loads have landed
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int half = 0; half < 4; ++half)
#pragma unroll
      for (int i = 0; i < 2; ++i)
        load_to_lds<true>(half < 2 ? xrow[half & 1][i] + rounds * KS
                                   : reinterpret_cast<const __bf16*>(reinterpret_cast<const char*>(t.w + rounds * KS) + wrow[half & 1][i]),
                          lds + half * kHalf + (wave * 16 + i * 8) * KS, rounds * KS + (piece ^ (4 * i)) * 8, a.K);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0070);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    read_x(0, 0, x0);
    read_w(0, 0, wa);
    read_w(0, 1, wb);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      multiply(x0, wa, acc[0][0], kk);
      multiply(x0, wb, acc[0][1], kk);
    }
    read_x(0, 1, x1);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      multiply(x1, wb, acc[1][1], kk);
      multiply(x1, wa, acc[1][0], kk);
    }
  }
  // column = row l16 of the tile's rows, rows = features 4 quad + i
  int slot[2][4];
  float score[2][4];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int r = h * 128 + wm * 64 + j * 16 + l16;
      slot[h][j] = slot_of[r];
      score[h][j] = PAIRED ? large_scores(slot_of)[r] : 1.f;
    }
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int r = h * 128 + wm * 64 + j * 16 + l16;
      if (r >= t.rows) continue;
      __bf16* y = a.y + (PAIRED ? t.first + r : (long)slot[h][j]) * a.F;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int f = t.f0 + wn * 32 + i * 16 + quad * 4;
        large_store<PAIRED>(a, y, f, score[h][j], acc[h][0][i][j], acc[h][1][i][j]);
        if constexpr (!PAIRED) large_store<PAIRED>(a, y, f + 128, score[h][j], acc[h][1][i][j], acc[h][0][i][j]);
      }
    }
}

// R rows from row r0 of a tile on and part `col` of CW of its 256 rows of the weights, as many rounds of 64 channels on their way as LDS holds; a
// wavefront has 32 rows of the weights and as many of the rows as there are wavefronts to the same weights.
template <int R, int CW, bool PAIRED, bool TAIL>
__device__ __forceinline__ void large_part(const ExpertGemmArgs& a, const ExpertTile& t, __bf16* lds, const int* slot_of, int r0, int col) {
  constexpr int KS = kGemmK, XL = R / 64, WL = CW / 64, WN = CW / 32, RW = R * WN / 8, MT = RW / 16, COLS = PAIRED ? CW / 2 : CW;
  constexpr int SLOT = (CW + R) * KS, DEPTH = kPartElements / SLOT, FLYING = (DEPTH - 2) * (XL + WL);
  static_assert(DEPTH >= 3 && FLYING < 16 && MT >= 1, "");
  if (r0 >= t.rows) {  // (no barrier left)
    __builtin_amdgcn_s_waitcnt(0x0070);  // (scores: nothing may come into LDS that is no longer this workgroup's)
    return;
  }
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, quad = lane >> 4;
  const int wn = wave % WN, wm = wave / WN, f0 = t.f0 + col * COLS;
  const int piece = (lane ^ (lane >> 4)) & 7;  // (rows of an odd group of eight: bit 2 the other way round)
  const __bf16* xrow[XL];
  uint32_t wrow[WL];  // bytes
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int r = (wave * XL + i) * 8 + (lane >> 3);
    xrow[i] = large_x_row<PAIRED>(a, t, slot_of, r0 + r) + (piece ^ (r >> 1 & 4)) * 8;
  }
#pragma unroll
  for (int i = 0; i < WL; ++i) {
    const int r = (wave * WL + i) * 8 + (lane >> 3);
    wrow[i] = (large_w_row<PAIRED, CW>(a, f0, r) * (uint32_t)a.K + (uint32_t)((piece ^ (r >> 1 & 4)) * 8)) * 2u;
  }
  const int rounds = (a.K + KS - 1) / KS;
  auto ask = [&](int at_round, int place) {
    __bf16* at = lds + place * SLOT;  // rows of the weights, then the rows
    const int round = at_round < rounds ? at_round : 0;  // (asked for and never read)
#pragma unroll
    for (int i = 0; i < WL; ++i)
      load_to_lds<TAIL>(reinterpret_cast<const __bf16*>(reinterpret_cast<const char*>(t.w + round * KS) + wrow[i]), at + (wave * WL + i) * 8 * KS,
                        round * KS + (piece ^ ((wave * WL + i) * 4 & 4)) * 8, a.K);
#pragma unroll
    for (int i = 0; i < XL; ++i)
      load_to_lds<TAIL>(xrow[i] + round * KS, at + CW * KS + (wave * XL + i) * 8 * KS, round * KS + (piece ^ ((wave * XL + i) * 4 & 4)) * 8, a.K);
  };
  f32x4 acc[2][MT];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int turned = (l16 >> 1) & 7;
  for (int i = 0; i < DEPTH - 1; ++i) ask(i, i);
  for (int round = 0, place = 0; round < rounds; ++round) {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0070 | FLYING);  // own reads are done, and all loads but those of the rounds behind
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    ask(round + DEPTH - 1, place == 0 ? DEPTH - 1 : place - 1);
    __builtin_amdgcn_sched_barrier(0);
    const __bf16* at = lds + place * SLOT + l16 * KS;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int p = ((kk * 4 + quad) ^ turned) * 8;
      bf16x8 w[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) w[i] = *reinterpret_cast<const bf16x8*>(at + (PAIRED ? i * COLS + wn * 16 : wn * 32 + i * 16) * KS + p);
#pragma unroll
      for (int j = 0; j < MT; ++j) {
        const bf16x8 x = *reinterpret_cast<const bf16x8*>(at + (CW + wm * RW + j * 16) * KS + p);
#pragma unroll
        for (int i = 0; i < 2; ++i) acc[i][j] = expert_mfma(w[i], x, acc[i][j]);
      }
    }
    place = place == DEPTH - 1 ? 0 : place + 1;
  }
  __builtin_amdgcn_s_waitcnt(0x0070);
  int slot[MT];
  float score[MT];
#pragma unroll
  for (int j = 0; j < MT; ++j) {
    const int r = r0 + wm * RW + j * 16 + l16;
    slot[j] = slot_of[r];
    score[j] = PAIRED ? large_scores(slot_of)[r] : 1.f;
  }
#pragma unroll
  for (int j = 0; j < MT; ++j) {
    const int r = r0 + wm * RW + j * 16 + l16;
    if (r >= t.rows) continue;
    __bf16* y = a.y + (PAIRED ? t.first + r : (long)slot[j]) * a.F;
    const int f = f0 + wn * (PAIRED ? 16 : 32) + quad * 4;
    large_store<PAIRED>(a, y, f, score[j], acc[0][j], acc[1][j]);
    if constexpr (!PAIRED) large_store<PAIRED>(a, y, f + 16, score[j], acc[1][j], acc[0][j]);
  }
}

// TAIL: the last round of channels is no whole one.  Block i is number i / 8 of die i % 8.  A die has a run of the whole tiles and, behind it, every
// eighth of the rests, which differ least between the dies that way.
template <bool PAIRED, bool TAIL> __global__ __launch_bounds__(512, 2) void expert_gemm_large_kernel(const ExpertGemmArgs a) {
  extern __shared__ __attribute__((aligned(16))) __bf16 lds[];
  int* slot_of = reinterpret_cast<int*>(lds + kPartElements);
  const int wholes = a.tile_first[0], full = wholes * a.col_tiles, rests = (a.tile_first[a.E] - wholes) * a.col_tiles;
  const int die = blockIdx.x % kDies, k = blockIdx.x / kDies, more = full % kDies, turn = (die - more) & (kDies - 1);
  const int first = die * (full / kDies) + (die < more ? die : more), mine_full = full / kDies + (die < more ? 1 : 0);
  const int mine = mine_full + rests / kDies + (turn < rests % kDies ? 1 : 0);
  const int in_rounds = mine / kDieUnits * kDieUnits, left = mine - in_rounds;
  int parts = 1;
  while (parts < kMaxParts && left * parts * 2 <= kDieUnits) parts *= 2;
  if (k >= in_rounds + left * parts) return;
  const int item = k < in_rounds ? k : in_rounds + (k - in_rounds) / parts, part = k < in_rounds ? 0 : (k - in_rounds) % parts;
  if (k < in_rounds) parts = 1;
  const int tid = threadIdx.x;
  int tile, column;
  if (item < mine_full) {
    // bands of kBand row tiles, walked down the rows first: what is in flight on a die shares its rows and its matrices
    const int id = first + item, band = id / (kBand * a.col_tiles), in_band = id % (kBand * a.col_tiles);
    const int deep = wholes - band * kBand < kBand ? wholes - band * kBand : kBand;
    tile = band * kBand + in_band % deep, column = in_band / deep;
  } else {
    const int id = (item - mine_full) * kDies + turn;
    tile = wholes + id / a.col_tiles, column = id % a.col_tiles;
  }
  ExpertTile t;
  t.first = (long)tile * kLargeRows;
  t.f0 = column * (PAIRED ? 128 : 256);
  // what the tile is and which choices it has, asked for together (one after the other, by way of the expert's count and first tile,
  // 700 tokens, 2 of 8 experts of 1024, 42.5 us a call: 42.0)
  const int what = a.tile_expert[tile];
  if (tid < kLargeRows) slot_of[tid] = a.order[t.first + tid];
  const int e = what & 255;
  t.rows = what >> 8;
  t.w = a.w + (long)e * (PAIRED ? 2 * a.F : a.F) * a.K;
  __syncthreads();
  if (tid >= t.rows && tid < kLargeRows) slot_of[tid] = slot_of[0];  // (rows that nobody has put in order)
  __syncthreads();
  if (PAIRED && tid < kLargeRows)  // (in front of all other loads, so that they are there behind the first wait of the wavefront)
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(a.scores + slot_of[tid]),
                                     (__attribute__((address_space(3))) void*)(slot_of + kLargeRows + (tid & ~63)), 4, 0, 0);
  // blocks of 64 rows first (of 128 where there are no parts for that), then parts of the weights
  const int rows = t.rows <= 64 ? 1 : t.rows <= 128 ? 2 : 4;
  if (parts < rows) {
    if (parts == 2 || rows == 2) return large_part<128, 256, PAIRED, TAIL>(a, t, lds, slot_of, part * 128, 0);
    return large_whole_tile<PAIRED, TAIL>(a, t, lds, slot_of);
  }
  const int r0 = part % rows * 64, col = part / rows;
  if (parts / rows == 1) return large_part<64, 256, PAIRED, TAIL>(a, t, lds, slot_of, r0, 0);
  if (parts / rows == 2) return large_part<64, 128, PAIRED, TAIL>(a, t, lds, slot_of, r0, col);
  large_part<64, 64, PAIRED, TAIL>(a, t, lds, slot_of, col < 4 ? r0 : kLargeRows, col);
}

// The same tiles of 32 rows with 64 rows of the weights (PAIRED: 32 up, 32 gate), rows and weights straight into LDS, rounds of 128 channels three
// deep: a few rows an expert wait for its matrices to come from memory, which asks for many loads on their way and many workgroups.  A wavefront
// takes 32 channels of a round and the whole tile; the four sums of an element are added through LDS in the end.  Channels in whole 128.
constexpr int kDirectWeights = 64, kDirectRows = BASED_EXPERT_TILE_ROWS_SMALL + kDirectWeights;
constexpr int kDirectSlab = kDirectRows * 64, kDirectRound = 2 * kDirectSlab, kDirectDepth = 3;  // elements; a slab: 64 channels of every row
constexpr int kDirectLds = kDirectDepth * kDirectRound * 2 + BASED_EXPERT_TILE_ROWS_SMALL * 4;   // bytes

template <bool PAIRED> __global__ __launch_bounds__(256, 2) void expert_gemm_direct_kernel(const ExpertGemmArgs a) {
  constexpr int BM = BASED_EXPERT_TILE_ROWS_SMALL, BN = kDirectWeights, COLS = PAIRED ? BN / 2 : BN, LOADS = kDirectRows / 16;
  extern __shared__ __attribute__((aligned(16))) __bf16 lds[];
  int* slot_of = reinterpret_cast<int*>(lds + kDirectDepth * kDirectRound);
  const int id = tile_of_block(blockIdx.x, gridDim.x), band = id / (kBand * a.col_tiles), in_band = id % (kBand * a.col_tiles);
  const int deep = a.tiles - band * kBand < kBand ? a.tiles - band * kBand : kBand;
  const int tile = band * kBand + in_band % deep, f0 = in_band / deep * COLS;
  if (tile >= a.tile_first[a.E]) return;
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, quad = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int e = 0, rows = a.counts[0] - tile * BM;  // (of one expert)
  if (a.tile_expert != nullptr) {
    const int what = a.tile_expert[tile];
    e = what & 255, rows = what >> 8;
  } else {
    rows = rows < BM ? rows : BM;
  }
  if (tid < BM) slot_of[tid] = a.order[(long)tile * BM + (tid < rows ? tid : 0)];
  lds_barrier();
  // 8 rows of a slab to a load; piece p (16 bytes) of a row lies at p ^ (row / 2 % 8), so that reads of 16 rows meet every bank once
  const char* src[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int group = wave * LOADS + i, slab = group / (kDirectRows / 8), row = group % (kDirectRows / 8) * 8 + (lane >> 3);
    const __bf16* at;
    if (row < BM) {
      at = a.x + (PAIRED ? (long)(slot_of[row] / a.top) * a.x_sr : ((long)tile * BM + (row < rows ? row : 0)) * a.x_sr);
    } else {
      const int r = row - BM, f = f0 + r % COLS;
      at = a.w + ((long)e * (PAIRED ? 2 * a.F : a.F) + (PAIRED && r >= COLS ? a.F : 0) + (f < a.F ? f : a.F - 1)) * a.K;
    }
    src[i] = reinterpret_cast<const char*>(at + slab * 64 + ((lane & 7) ^ (row >> 1 & 7)) * 8);
  }
  const int rounds = a.K / 128;
  auto ask = [&](int round, int place) {
    const long from = (long)(round < rounds ? round : 0) * 256;  // (past the end: asked for and never read, the count of loads stays)
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src[i] + from),
                                       (__attribute__((address_space(3))) void*)(lds + place * kDirectRound + (wave * LOADS + i) * 512), 16, 0, 0);
  };
  f32x4 acc[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i][0] = acc[i][1] = f32x4{0.f, 0.f, 0.f, 0.f};
  ask(0, 0);
  ask(1, 1);
  const int turned = l16 >> 1 & 7, step = (wave >> 1) * kDirectSlab + (((wave & 1) * 4 + quad) ^ turned) * 8 + l16 * 64;
  for (int round = 0, place = 0; round < rounds; ++round) {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0070 | LOADS);  // own reads are done, and all loads but those of the next round
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    ask(round + 2, place == 0 ? 2 : place - 1);
    __builtin_amdgcn_sched_barrier(0);
    const __bf16* at = lds + place * kDirectRound + step;
    bf16x8 x[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) x[j] = *reinterpret_cast<const bf16x8*>(at + j * 16 * 64);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bf16x8 w = *reinterpret_cast<const bf16x8*>(at + (BM + i * 16) * 64);
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = expert_mfma(w, x[j], acc[i][j]);
    }
    place = place == 2 ? 0 : place + 1;
  }
  __builtin_amdgcn_s_waitcnt(0x0070);  // (nothing may come into LDS that is no longer the loads')
  __builtin_amdgcn_s_barrier();
  f32x4* sums = reinterpret_cast<f32x4*>(lds);  // [wave][feature tile][row tile][lane]
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) sums[((wave * 4 + i) * 2 + j) * 64 + lane] = acc[i][j];
  __syncthreads();
  // two feature tiles (PAIRED: up and gate) of 16 rows to a wavefront
  const int half = wave & 1, r = (wave >> 1) * 16 + l16;
  f32x4 out[2];
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const f32x4* at = sums + ((p * 2 + half) * 2 + (wave >> 1)) * 64 + lane;
    out[p] = (at[0] + at[512]) + (at[1024] + at[1536]);
  }
  if (r >= rows) return;
  const int slot = slot_of[r];
  if constexpr (PAIRED) {
    large_store<true>(a, a.y + ((long)tile * BM + r) * a.F, f0 + half * 16 + quad * 4, a.scores[slot], out[0], out[1]);
  } else {
    __bf16* y = a.y + (long)slot * a.F;
#pragma unroll
    for (int p = 0; p < 2; ++p) large_store<false>(a, y, f0 + (p * 2 + half) * 16 + quad * 4, 1.f, out[p], out[p]);
  }
}

template <bool PAIRED, bool TAIL> int launch_expert_gemm_large(ExpertGemmArgs a, hipStream_t s) {
  static LdsAllowed allowed;
  const hipError_t e = allow_lds(reinterpret_cast<const void*>(expert_gemm_large_kernel<PAIRED, TAIL>), kLargeLds, allowed);
  BASED_REQUIRE(e == hipSuccess, BASED_ERR_LAUNCH, "experts: %d bytes of LDS refused: %s", kLargeLds, hipGetErrorString(e));
  a.col_tiles = PAIRED ? (a.F + 127) / 128 : (a.F + 255) / 256;
  // (parts beyond the first of a tile: less than one for each of the 32 compute units of a die)
  const unsigned per_die = (unsigned)((a.col_tiles * a.tiles + kDies - 1) / kDies + kDieUnits);
  hipLaunchKernelGGL((expert_gemm_large_kernel<PAIRED, TAIL>), dim3(per_die * kDies), dim3(512), kLargeLds, s, a);
  return BASED_OK;
}

// Straight into LDS where tiles of 128 rows of the weights are fewer than half of the compute units and a tile's way is long.  Whole calls, kernels
// alone, us, without and with (both products, the second alone): 2 of 8 experts of 1024, 12 tokens (128 and 64 workgroups) 27.3 / 23.7 / 24.9, 30
// (144, 72) 28.4 / 27.0 / 26.2, 100 (224, 112) 33.9 / 32.7 / 32.5, 164 (288, 144) 37.6 / 36.5 / 38.0; 1 of 8 of 2048, 30 tokens (256, 64) 34.4 / 29.9
// / 29.3, 260 (512, 128) 42.8 / 39.4 / 38.3; 4 of 16 of 512, 30 tokens (152, 152; 512 channels) 29.2 / 30.9 / 30.1.
template <bool PAIRED> int launch_expert_gemm(ExpertGemmArgs a, hipStream_t s) {
  const int before = PAIRED ? kSmallWeights / 2 : kSmallWeights;
  const bool direct = a.K % 128 == 0 && a.K >= 1024 && (long)((a.F + before - 1) / before) * a.tiles <= 128;
  const int weights = direct ? kDirectWeights : kSmallWeights, cols = PAIRED ? weights / 2 : weights;
  a.col_tiles = (a.F + cols - 1) / cols;
  const dim3 grid((unsigned)(a.col_tiles * a.tiles));
  if (!direct) {
    hipLaunchKernelGGL(expert_gemm_kernel<PAIRED>, grid, dim3(256), 0, s, a);
    return BASED_OK;
  }
  static LdsAllowed allowed;
  const hipError_t e = allow_lds(reinterpret_cast<const void*>(expert_gemm_direct_kernel<PAIRED>), kDirectLds, allowed);
  BASED_REQUIRE(e == hipSuccess, BASED_ERR_LAUNCH, "experts: %d bytes of LDS refused: %s", kDirectLds, hipGetErrorString(e));
  hipLaunchKernelGGL(expert_gemm_direct_kernel<PAIRED>, grid, dim3(256), kDirectLds, s, a);
  return BASED_OK;
}

template <bool PAIRED> int launch_expert_product(const ExpertGemmArgs& a, int rows, hipStream_t s) {
  if (rows == BASED_EXPERT_TILE_ROWS)
    return a.K % kGemmK == 0 ? launch_expert_gemm_large<PAIRED, false>(a, s) : launch_expert_gemm_large<PAIRED, true>(a, s);
  return launch_expert_gemm<PAIRED>(a, s);
}

// y[n] = sum of the rows of its choices
template <typename T> __global__ __launch_bounds__(256) void expert_sum_kernel(const T* x, T* y, long n, int D, int top) {
  constexpr int N = Pack<T>::kN;
  const int pieces = D / N;
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n * pieces) return;
  const long row = i / pieces;
  const int c = (int)(i % pieces) * N;
  float s[N];
#pragma unroll
  for (int j = 0; j < N; ++j) s[j] = 0.f;
  for (int t = 0; t < top; ++t) {
    float v[N];
    load_vec<T, N>(x + (row * top + t) * D + c, v);
#pragma unroll
    for (int j = 0; j < N; ++j) s[j] += v[j];
  }
  store_vec<T, N>(y + row * D + c, s);
}

// ---- one choice at a time ----
struct ExpertRowsArgs {
  const void* x;   // first product: (N, K); second: (N * top, K)
  const void* w;   // (E, 2 F, K) / (E, F, K)
  void* y;         // (N * top, F) / (N, F)
  const int32_t* ids;
  const float* scores;
  long n, x_sr;
  int F, K, top;
};

constexpr int kRowsFeatures = 16;  // features per workgroup

template <int LPR> __device__ __forceinline__ float lanes_sum(float v) {
  if constexpr (LPR == 8) return sum8(v);
  v = sum16(v);
  if constexpr (LPR >= 32) v += __shfl_xor(v, 16, 64);
  if constexpr (LPR >= 64) v += __shfl_xor(v, 32, 64);
  return v;
}

// LPR lanes share a dot product; a workgroup takes kRowsFeatures features of one choice (gate and up) or token (down).
template <typename T, int N, int LPR, bool PAIRED>
__global__ __launch_bounds__(256) void expert_rows_kernel(const ExpertRowsArgs a) {
  const int lane = threadIdx.x % LPR, grp = threadIdx.x / LPR;
  constexpr int GROUPS = 256 / LPR;
  const long item = blockIdx.x;  // choice or token
  const int f1 = (int)(blockIdx.y + 1) * kRowsFeatures < a.F ? (int)(blockIdx.y + 1) * kRowsFeatures : a.F;
  constexpr int FU = GROUPS >= kRowsFeatures ? 1 : kRowsFeatures / GROUPS;  // features per group of lanes, in flight together
  int f[FU];
#pragma unroll
  for (int u = 0; u < FU; ++u) f[u] = blockIdx.y * kRowsFeatures + u * GROUPS + grp;
  auto load = [&](const T* p, float (&v)[N]) {
    if constexpr (N == 1)
      v[0] = to_f32(*p);
    else
      load_vec<T, N>(p, v);
  };
  if constexpr (PAIRED) {
    const T* x = static_cast<const T*>(a.x) + item / a.top * a.x_sr;
    const T* w = static_cast<const T*>(a.w) + (long)a.ids[item] * 2 * a.F * a.K;
    float up[FU], gate[FU];
#pragma unroll
    for (int u = 0; u < FU; ++u) up[u] = gate[u] = 0.f;
#pragma unroll 2
    for (int c = lane * N; c < a.K; c += LPR * N) {
      float xv[N];
      load(x + c, xv);
#pragma unroll
      for (int u = 0; u < FU; ++u) {
        const long row = f[u] < f1 ? f[u] : 0;
        float uv[N], gv[N];
        load(w + row * a.K + c, uv);
        load(w + (a.F + row) * a.K + c, gv);
#pragma unroll
        for (int j = 0; j < N; ++j) {
          up[u] = __builtin_fmaf(uv[j], xv[j], up[u]);
          gate[u] = __builtin_fmaf(gv[j], xv[j], gate[u]);
        }
      }
    }
    const float s = a.scores[item];
#pragma unroll
    for (int u = 0; u < FU; ++u) {
      const float uu = lanes_sum<LPR>(up[u]), gg = lanes_sum<LPR>(gate[u]);
      if (lane == 0 && f[u] < f1) static_cast<T*>(a.y)[item * a.F + f[u]] = from_f32<T>(silu_exact(gg * s) * (uu * s));
    }
  } else {
    float acc[FU];
#pragma unroll
    for (int u = 0; u < FU; ++u) acc[u] = 0.f;
    for (int t = 0; t < a.top; ++t) {
      const T* x = static_cast<const T*>(a.x) + (item * a.top + t) * a.x_sr;
      const T* w = static_cast<const T*>(a.w) + (long)a.ids[item * a.top + t] * a.F * a.K;
#pragma unroll 2
      for (int c = lane * N; c < a.K; c += LPR * N) {
        float xv[N];
        load(x + c, xv);
#pragma unroll
        for (int u = 0; u < FU; ++u) {
          float wv[N];
          load(w + (long)(f[u] < f1 ? f[u] : 0) * a.K + c, wv);
#pragma unroll
          for (int j = 0; j < N; ++j) acc[u] = __builtin_fmaf(wv[j], xv[j], acc[u]);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < FU; ++u) {
      const float s = lanes_sum<LPR>(acc[u]);
      if (lane == 0 && f[u] < f1) static_cast<T*>(a.y)[item * a.F + f[u]] = from_f32<T>(s);
    }
  }
}

template <typename T, int N, bool PAIRED> void launch_expert_rows(const ExpertRowsArgs& a, long items, hipStream_t s) {
  const dim3 grid((unsigned)items, (unsigned)((a.F + kRowsFeatures - 1) / kRowsFeatures));
  const int pieces = (a.K + N - 1) / N;
  if (pieces <= 8)
    hipLaunchKernelGGL((expert_rows_kernel<T, N, 8, PAIRED>), grid, dim3(256), 0, s, a);
  else if (pieces <= 16)
    hipLaunchKernelGGL((expert_rows_kernel<T, N, 16, PAIRED>), grid, dim3(256), 0, s, a);
  else if (pieces <= 32)
    hipLaunchKernelGGL((expert_rows_kernel<T, N, 32, PAIRED>), grid, dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL((expert_rows_kernel<T, N, 64, PAIRED>), grid, dim3(256), 0, s, a);
}

template <typename T, bool PAIRED> void launch_expert_rows_vec(const ExpertRowsArgs& a, bool vec, long items, hipStream_t s) {
  if (vec)
    launch_expert_rows<T, Pack<T>::kN, PAIRED>(a, items, s);
  else
    launch_expert_rows<T, 1, PAIRED>(a, items, s);
}

// ---- fp32, rows of one expert on fp32 MFMA ----
// 16 features (PAIRED: of up and of gate) of one expert per workgroup, which looks its choices up among all and takes 16 of them at a time; its
// eight wavefronts share the channels, each with its part of the matrices in registers for all of the choices, and add their sums up at the
// end of each 16.  Bound by reading the matrices, once each, where one choice at a time reads them for every choice: 12 tokens, 4 of 16 experts
// of 512: 49 us by choices, 54 here; 20 tokens 66 and 54; 140 tokens, 1 of 8 of 2048: 250 and 96; 256 tokens, 4 of 16 of 512: 296 and 117.
constexpr int kF32Features = 16, kF32Scan = 1024;

struct ExpertF32Args {
  const float* x;  // PAIRED: (N, K); otherwise (N * top, K)
  const float* w;  // (E, 2 F, K) / (E, F, K)
  float* y;        // (N * top, F)
  const int32_t* ids;
  const float* scores;
  long slots, x_sr;
  int F, K, top;
};

template <bool PAIRED> __global__ __launch_bounds__(512) void expert_f32_kernel(const ExpertF32Args a) {
  constexpr int WT = PAIRED ? 2 : 1, S = 16 / WT;  // pieces of 16 channels in registers
  __shared__ int list[kF32Scan];
  __shared__ int found[8];
  __shared__ __attribute__((aligned(16))) float sums[2][8][WT][256];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, quad = lane >> 4;
  const int e = blockIdx.y, f0 = blockIdx.x * kF32Features;
  const int pieces = (a.K + 15) / 16, per = (pieces + 7) / 8, p_begin = wave * per, p_end = p_begin + per < pieces ? p_begin + per : pieces;
  const float* w = a.w + ((long)e * WT * a.F + (f0 + l16 < a.F ? f0 + l16 : a.F - 1)) * a.K;
  f32x4 wf[WT][S], xf[S];
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  auto channel = [&](int p) { return p * 16 + quad * 4; };
  auto there = [&](int p) { return p < p_end && channel(p) < a.K; };
  auto load_w = [&](int p0) {
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
      for (int t = 0; t < WT; ++t) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(w + (long)t * a.F * a.K + (there(p0 + s) ? channel(p0 + s) : 0));
        wf[t][s] = there(p0 + s) ? v : zero;
      }
  };
  if (per <= S) load_w(p_begin);  // (the caller has several choices for an expert: few of them are not used)
  int parity = 0;
  for (long s0 = 0; s0 < a.slots; s0 += kF32Scan) {
    // this expert's among the next choices, in their order
    int at = 0, n = 0;
    bool mine[kF32Scan / 512];
    int before[kF32Scan / 512];
#pragma unroll
    for (int i = 0; i < kF32Scan / 512; ++i) {
      const long slot = s0 + i * 512 + tid;
      mine[i] = slot < a.slots && a.ids[slot < a.slots ? slot : 0] == e;
    }
#pragma unroll
    for (int i = 0; i < kF32Scan / 512; ++i) {
      const uint64_t b = __ballot(mine[i]);
      before[i] = __popcll(b & ((1ull << lane) - 1));
      if (lane == 0) found[wave] = __popcll(b);
      __syncthreads();
      at = n;
      for (int v = 0; v < 8; ++v) {
        if (v < wave) at += found[v];
        n += found[v];
      }
      if (mine[i]) list[at + before[i]] = (int)(s0 + i * 512 + tid);
      __syncthreads();
    }
    for (int r0 = 0; r0 < n; r0 += 16, parity ^= 1) {
      const int slot = list[r0 + l16 < n ? r0 + l16 : r0];
      const float* x = a.x + (PAIRED ? slot / a.top : slot) * a.x_sr;
      f32x4 acc[WT][S];  // (short chains round less)
#pragma unroll
      for (int t = 0; t < WT; ++t)
#pragma unroll
        for (int s = 0; s < S; ++s) acc[t][s] = zero;
      for (int p0 = p_begin; p0 < p_begin + per; p0 += S) {
#pragma unroll
        for (int s4 = 0; s4 < S; s4 += 4)
          if (p0 + s4 < p_end) {
#pragma unroll
            for (int s = s4; s < s4 + 4; ++s) {
              const f32x4 v = *reinterpret_cast<const f32x4*>(x + (there(p0 + s) ? channel(p0 + s) : 0));
              xf[s] = there(p0 + s) ? v : zero;
            }
          }
        if (per > S) load_w(p0);
#pragma unroll
        for (int s4 = 0; s4 < S; s4 += 4)
          if (p0 + s4 < p_end)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
              for (int s = s4; s < s4 + 4; ++s)
#pragma unroll
                for (int t = 0; t < WT; ++t) acc[t][s] = mfma_f32(wf[t][s][j], xf[s][j], acc[t][s]);
      }
      // column = choice l16, rows = features 4 quad + i
#pragma unroll
      for (int t = 0; t < WT; ++t) {
#pragma unroll
        for (int m = 1; m < S; m <<= 1)
#pragma unroll
          for (int s = 0; s < S; s += 2 * m) acc[t][s] += acc[t][s + m];
        *reinterpret_cast<f32x4*>(&sums[parity][wave][t][lane * 4]) = acc[t][0];
      }
      __syncthreads();  // (the other half of sums is read before this one comes round again)
      const int r = tid >> 4, f = f0 + l16, i = ((l16 >> 2) * 16 + r) * 4 + (l16 & 3);
      if (tid < 256 && r0 + r < n && f < a.F) {
        float z[WT];
#pragma unroll
        for (int t = 0; t < WT; ++t) {
          float q[8];
#pragma unroll
          for (int v = 0; v < 8; ++v) q[v] = sums[parity][v][t][i];
          z[t] = ((q[0] + q[1]) + (q[2] + q[3])) + ((q[4] + q[5]) + (q[6] + q[7]));
        }
        const long out = list[r0 + r];
        if constexpr (PAIRED) {
          const float score = a.scores[out];
          a.y[out * a.F + f] = silu_exact(z[1] * score) * (z[0] * score);
        } else {
          a.y[out * a.F + f] = z[0];
        }
      }
    }
    __syncthreads();  // (the list is written again)
  }
}

constexpr int kRouteOneWg = 32;  // tokens that one workgroup routes, of up to 32 experts (16 of more): it makes the plan too

// Tokens of one workgroup.  Many tokens of few experts: 32, their rows shared out over eight wavefronts (8192 tokens of 1024 channels, 8 experts:
// 7.2 us without the sums of all workgroups' choices, 10 with them; 16 tokens 11.6, a wavefront to 16 tokens 16.9).  So many that every
// wavefront has enough of its own: 64, fewer workgroups whose choices are added up (calls of 16 experts of 16 features, 256 channels: 65,536 tokens
// 113.9 -> 98.8 us, 16,384 49.8 and 49.1, 8192 39.0 and 42.0; 768 channels, 65,536 tokens 232.5 and 234.3, of 4 experts 104.3 and 100.2).
static int route_group(const RouteArgs& a, bool vec) {
  const bool many = vec && a.n >= 4096;
  return !many ? 16 : a.E <= 32 && (a.n < 32768 || a.D > 768) ? 32 : 64;
}

template <int ET> void launch_route_tiles(const RouteArgs& a, hipStream_t s) {
  const size_t one = (size_t)16 * a.E * sizeof(float);
  constexpr int NW = ET <= 4 ? 8 : 4;
  const int group = route_group(a, true);
  if (group == 64) {
    hipLaunchKernelGGL((expert_route_kernel<__bf16, ET, 4, false, 1>), dim3((unsigned)((a.n + 63) / 64)), dim3(256), 4 * one, s, a);
    return;
  }
  if constexpr (ET <= 2) {
    if ((a.n > 16 && a.n <= kRouteOneWg) || group == 32) {
      hipLaunchKernelGGL((expert_route_kernel<__bf16, ET, NW, true, 2>), dim3((unsigned)((a.n + 31) / 32)), dim3(64 * NW), 2 * NW * one, s, a);
      return;
    }
  }
  hipLaunchKernelGGL((expert_route_kernel<__bf16, ET, NW, true, 1>), dim3((unsigned)((a.n + 15) / 16)), dim3(64 * NW), NW * one, s, a);
}

static bool route_is_single(const RouteArgs& a, bool vec) { return a.n <= (vec && a.E <= 32 ? kRouteOneWg : 16); }

template <typename T> void launch_route(RouteArgs a, bool vec, hipStream_t s) {
  const dim3 grid((unsigned)((a.n + 15) / 16));
  if (!route_is_single(a, vec)) a.order = nullptr;
  if constexpr (sizeof(T) == 2) {
    const int et = (a.E + 15) / 16;
    if (vec && et <= 1)
      return launch_route_tiles<1>(a, s);
    if (vec && et <= 2)
      return launch_route_tiles<2>(a, s);
    if (vec && et <= 4)
      return launch_route_tiles<4>(a, s);
    if (vec && et <= 8)
      return launch_route_tiles<8>(a, s);
  }
  hipLaunchKernelGGL((expert_route_kernel<T, 0, 4, false, 1>), grid, dim3(256), (size_t)16 * a.E * sizeof(float), s, a);
}

static bool route_vec(const RouteArgs& a) {
  return a.D % 8 == 0 && a.h_sr % 8 == 0 && a.E <= 128 && aligned_to(a.h, 16) && aligned_to(a.w, 16);
}

static bool route_by_row(const RouteArgs& a, int piece) {
  return a.D % piece == 0 && a.D <= kRouteRowMax && a.h_sr % piece == 0 && aligned_to(a.h, 16) && aligned_to(a.w, 16);
}

// A workgroup to each token, or a score to a thread (element by element: 12 tokens of 1024 channels take 70 us) where the tokens are so many that
// workgroups cost more than channels: calls of 8 experts of ff 64 with 64 channels, 1024 tokens 18.3 us by rows and 19.7 by scores, 4096 tokens 51.6
// and 45.7; 256 channels, 4096 tokens 113 and 117; 64 experts, 32 channels, 1024 tokens 17.0 and 26.4, 4096 tokens 46.9 and 39.1.
static void launch_route_f32(const RouteArgs& r, bool by_row, hipStream_t s) {
  if (by_row && r.n <= (long)16 * r.D * ((r.E + 15) / 16))
    hipLaunchKernelGGL(expert_route_row_kernel<float>, dim3((unsigned)r.n), dim3(512), 0, s,
                       RouteRowArgs{r, nullptr, nullptr, nullptr, nullptr, 1.f, 0.f, BASED_NORM_RMS});
  else
    launch_route<float>(r, false, s);
}

static int route_check(const char* who, const RouteArgs& a) {
  BASED_REQUIRE(a.n >= 0 && a.D > 0 && a.E > 0 && a.top > 0 && a.top <= a.E, BASED_ERR_ARG, "%s: bad sizes", who);
  BASED_REQUIRE(a.E <= kMaxExperts, BASED_ERR_SHAPE, "%s: %d experts (at most %d)", who, a.E, kMaxExperts);
  BASED_REQUIRE(a.n * a.top < (1ll << 31), BASED_ERR_SHAPE, "%s: too many choices", who);
  return BASED_OK;
}

}  // namespace based

/* Tiles of BASED_EXPERT_TILE_ROWS or BASED_EXPERT_TILE_ROWS_SMALL rows. */
// The line: 2 of 8 experts of 1024, 354 tokens (88 choices an expert) 41.2 us with large tiles, 40.1 with small ones, 700 tokens 41.8 and 50.0;
// 1 of 8 of 2048, 900 tokens (112 an expert) 61.8 and 69.2; 4 of 16 of 512, 400 tokens (100) 41.7 and 46.9, 200 tokens (50) 41.5 and 40.7.
static int expert_tile_rows(int64_t slots, int64_t E) { return slots >= 96 * E ? BASED_EXPERT_TILE_ROWS : BASED_EXPERT_TILE_ROWS_SMALL; }

static int64_t expert_tiles(int64_t slots, int64_t E, int64_t rows) { return slots / rows + (E < slots ? E : slots); }

// Few large tiles leave most of the GPU idle: such a call goes in small ones all the same, in the scratch of the large ones.  Choices in all at which both
// take the same time, whether of one expert or of sixteen: 256 x 256 4,000, 512 x 512 2,000, 768 x 768 1,250, 1024 x 1024 900, 2048 x 2048 450, 1024
// channels x 64 2,000, 64 x 1024 1,050, 512 x 2048 1,300, 1024 x 512 1,000, 4096 x 1024 450; 128 x 128 the same at any number.  100 tokens, one
// expert of 1024: 33.2 us in large ones, 27.9 in small ones; 200, 1 of 2 of 2048 x 2048 54.0 and 41.7; 400, 2 of 8 of 1024 42.6 and 46.3.
static bool expert_large_products(int64_t slots, int64_t D, int64_t F) { return D + F <= 256 || (double)slots * (D + F) >= 1.6e6; }

extern "C" BASED_API int64_t based_expert_tiles(int64_t n, int64_t E, int64_t top) {
  if (n <= 0 || E <= 0 || top <= 0) return 0;
  return expert_tiles(n * top, E, expert_tile_rows(n * top, E));
}

extern "C" BASED_API int64_t based_expert_tile_rows(int64_t n, int64_t E, int64_t top) { return expert_tile_rows(n * top, E); }

extern "C" BASED_API int based_expert_grouped(const void* h, const void* router, const void* w1, const void* w2, int32_t* ids, float* scores,
                                              int32_t* rank, int32_t* counts, int32_t* tile_first, int32_t* tile_expert, int32_t* order,
                                              void* work_act, void* work_out, void* y, int64_t n, int64_t D, int64_t F, int64_t E, int64_t top,
                                              int64_t h_sr, void* stream) {
  using namespace based;
  BASED_REQUIRE(h && router && w1 && w2 && ids && scores && rank && counts && tile_first && tile_expert && order && work_act && y,
                BASED_ERR_ARG, "expert_grouped: null pointer argument");
  BASED_REQUIRE(F > 0 && D < (1ll << 28), BASED_ERR_ARG, "expert_grouped: bad sizes");
  BASED_REQUIRE(top == 1 || work_out != nullptr, BASED_ERR_ARG, "expert_grouped: several choices per token need work_out");
  BASED_REQUIRE(D % 8 == 0 && F % 8 == 0 && h_sr % 8 == 0 && 2 * F * D < (1ll << 31), BASED_ERR_SHAPE,
                "expert_grouped: sizes %ld and %ld must be multiples of 8", (long)D, (long)F);
  BASED_REQUIRE(aligned_to(h, 16) && aligned_to(w1, 16) && aligned_to(w2, 16) && aligned_to(work_act, 16) && aligned_to(work_out, 16) &&
                    aligned_to(y, 16),
                BASED_ERR_ALIGN, "expert_grouped: tensors must be 16-byte aligned");
  RouteArgs r{h, router, ids, scores, rank, counts, nullptr, tile_first, nullptr, order, 0, (long)n, (long)h_sr, (int)D, (int)E, (int)top};
  const int rc = route_check("expert_grouped", r);
  if (rc != BASED_OK) return rc;
  if (n == 0) return BASED_OK;
  const int64_t slots = n * top;
  int rows = expert_tile_rows(slots, E);
  if (rows == BASED_EXPERT_TILE_ROWS && !expert_large_products(slots, D, F)) {
    // Rows of all tiles together are no more, less than 32 added to an expert in place of 256; the tiles are, and theirs goes behind the order.
    const int64_t small = expert_tiles(slots, E, BASED_EXPERT_TILE_ROWS_SMALL), at = small * BASED_EXPERT_TILE_ROWS_SMALL;
    const bool room = at + small <= expert_tiles(slots, E, BASED_EXPERT_TILE_ROWS) * BASED_EXPERT_TILE_ROWS;
    if (room || E == 1) {
      rows = BASED_EXPERT_TILE_ROWS_SMALL;
      tile_expert = room ? order + at : nullptr;
    }
  }
  const int64_t tiles = expert_tiles(slots, E, rows);
  BASED_REQUIRE(tiles * ((F > D ? F : D) / 64 + 1) < (1ll << 31), BASED_ERR_SHAPE, "expert_grouped: too many rows");
  hipStream_t s = static_cast<hipStream_t>(stream);
  r.tile_rows = rows, r.tile_expert = tile_expert;
  const bool vec = route_vec(r);
  const int group = route_group(r, vec);
  const int64_t groups = (n + group - 1) / group;
  const bool single = route_is_single(r, vec);
  if (!single) {
    // the workgroups' counts go where the activations come later; where that has no room for them, or they are too many to be read by
    // every workgroup that places choices, the workgroups add theirs up (8192 tokens, 8 experts: clearing the counts and placing in two launches
    // 12.4 us; by the workgroups' counts, in one launch 6.9)
    if (groups * E <= kPlaceHist && groups * E * 4 <= tiles * rows * F * 2)
      r.hist = static_cast<int32_t*>(work_act);
    else
      hipLaunchKernelGGL(expert_zero_kernel, dim3(1), dim3(kMaxExperts), 0, s, counts, (int)E);
  }
  launch_route<__bf16>(r, vec, s);
  if (!single) {
    const PlaceArgs p{counts, r.hist, ids, rank, tile_first, tile_expert, order, (long)slots, (int)E, rows, (int)groups, (int)(group * top)};
    hipLaunchKernelGGL(expert_place_kernel, dim3((unsigned)((groups + kPlaceGroups - 1) / kPlaceGroups)), dim3(kPlaceThreads), 0, s, p);
  }
  const ExpertGemmArgs a{static_cast<const __bf16*>(h), static_cast<const __bf16*>(w1), static_cast<__bf16*>(work_act), order, tile_first,
                         tile_expert, counts, scores, (long)h_sr, (int)E, (int)F, (int)D, (int)top, 0, (int)tiles};
  __bf16* out = static_cast<__bf16*>(top == 1 ? y : work_out);
  const ExpertGemmArgs a2{static_cast<const __bf16*>(work_act), static_cast<const __bf16*>(w2), out, order, tile_first,
                          tile_expert, counts, scores, (long)F, (int)E, (int)D, (int)F, (int)top, 0, (int)tiles};
  int done = launch_expert_product<true>(a, rows, s);
  if (done == BASED_OK) done = launch_expert_product<false>(a2, rows, s);
  if (done != BASED_OK) return done;
  if (top > 1)
    hipLaunchKernelGGL(expert_sum_kernel<__bf16>, dim3((unsigned)((n * (D / 8) + 255) / 256)), dim3(256), 0, s, out, static_cast<__bf16*>(y), (long)n,
                       (int)D, (int)top);
  return check_launch("expert_grouped");
}

extern "C" BASED_API int based_expert_rows(const void* x, const float* residual_in, float* residual_out, const void* norm_weight, void* work_h,
                                           float mult, int norm_kind, float eps, const void* router, const void* w1, const void* w2,
                                           int32_t* ids, float* scores, void* work_act, void* y, int64_t n, int64_t D, int64_t F, int64_t E,
                                           int64_t top, int64_t x_sr, int io_dtype, void* stream) {
  using namespace based;
  BASED_REQUIRE(x && router && w1 && w2 && ids && scores && work_act && y, BASED_ERR_ARG, "expert_rows: null pointer argument");
  BASED_REQUIRE(F > 0 && D < (1 << 20) && F < (1 << 20), BASED_ERR_SHAPE, "expert_rows: grid too large");
  BASED_REQUIRE(io_dtype == BASED_BF16 || io_dtype == BASED_F32, BASED_ERR_DTYPE, "expert_rows: bad dtype");
  RouteArgs r{x, router, ids, scores, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 0, (long)n, (long)x_sr, (int)D, (int)E, (int)top};
  const int rc = route_check("expert_rows", r);
  if (rc != BASED_OK) return rc;
  const bool by_row = route_by_row(r, io_dtype == BASED_BF16 ? 8 : 4);
  if (norm_weight != nullptr) {
    BASED_REQUIRE(by_row && io_dtype == BASED_BF16, BASED_ERR_SHAPE, "expert_rows: the norm takes bf16 rows of a multiple of 8 up to %d channels", kRouteRowMax);
    BASED_REQUIRE(work_h && (norm_kind == BASED_NORM_RMS || norm_kind == BASED_NORM_LAYER) && residual_out != residual_in, BASED_ERR_ARG,
                  "expert_rows: bad norm arguments");
    BASED_REQUIRE(aligned_to(norm_weight, 16) && aligned_to(residual_in, 16) && aligned_to(residual_out, 16) && aligned_to(work_h, 16),
                  BASED_ERR_ALIGN, "expert_rows: tensors must be 16-byte aligned");
  }
  if (n == 0) return BASED_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const void* h = norm_weight != nullptr ? work_h : x;
  const int64_t h_sr = norm_weight != nullptr ? D : x_sr;
  if (norm_weight != nullptr || (by_row && io_dtype == BASED_BF16 && n <= 16)) {
    const RouteRowArgs a{r, residual_in, residual_out, static_cast<const __bf16*>(norm_weight), static_cast<__bf16*>(work_h), mult, eps, norm_kind};
    hipLaunchKernelGGL(expert_route_row_kernel<__bf16>, dim3((unsigned)n), dim3(512), 0, s, a);
  } else if (io_dtype == BASED_BF16) {
    launch_route<__bf16>(r, route_vec(r), s);
  } else {
    launch_route_f32(r, by_row, s);
  }
  const int p = io_dtype == BASED_BF16 ? 8 : 4;
  const bool vec1 = D % p == 0 && h_sr % p == 0 && aligned_to(h, 16) && aligned_to(w1, 16);
  const bool vec2 = F % p == 0 && aligned_to(work_act, 16) && aligned_to(w2, 16);
  const ExpertRowsArgs a1{h, w1, work_act, ids, scores, (long)n, (long)h_sr, (int)F, (int)D, (int)top};
  const ExpertRowsArgs a2{work_act, w2, y, ids, scores, (long)n, (long)F, (int)D, (int)F, (int)top};
  if (io_dtype == BASED_BF16) {
    launch_expert_rows_vec<__bf16, true>(a1, vec1, n * top, s);
    launch_expert_rows_vec<__bf16, false>(a2, vec2, n, s);
  } else {
    launch_expert_rows_vec<float, true>(a1, vec1, n * top, s);
    launch_expert_rows_vec<float, false>(a2, vec2, n, s);
  }
  return check_launch("expert_rows");
}

extern "C" BASED_API int based_expert_grouped_f32(const float* h, const float* router, const float* w1, const float* w2, int32_t* ids, float* scores,
                                                  float* work_act, float* work_out, float* y, int64_t n, int64_t D, int64_t F, int64_t E,
                                                  int64_t top, int64_t h_sr, void* stream) {
  using namespace based;
  BASED_REQUIRE(h && router && w1 && w2 && ids && scores && work_act && y, BASED_ERR_ARG, "expert_grouped_f32: null pointer argument");
  BASED_REQUIRE(F > 0 && D < (1 << 20) && F < (1 << 20), BASED_ERR_SHAPE, "expert_grouped_f32: grid too large");
  BASED_REQUIRE(top == 1 || work_out != nullptr, BASED_ERR_ARG, "expert_grouped_f32: several choices per token need work_out");
  BASED_REQUIRE(D % 4 == 0 && F % 4 == 0 && h_sr % 4 == 0, BASED_ERR_SHAPE, "expert_grouped_f32: sizes %ld and %ld must be multiples of 4", (long)D,
                (long)F);
  BASED_REQUIRE(aligned_to(h, 16) && aligned_to(w1, 16) && aligned_to(w2, 16) && aligned_to(work_act, 16) && aligned_to(work_out, 16) &&
                    aligned_to(y, 16),
                BASED_ERR_ALIGN, "expert_grouped_f32: tensors must be 16-byte aligned");
  const RouteArgs r{h, router, ids, scores, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 0, (long)n, (long)h_sr, (int)D, (int)E, (int)top};
  const int rc = route_check("expert_grouped_f32", r);
  if (rc != BASED_OK) return rc;
  if (n == 0) return BASED_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  launch_route_f32(r, route_by_row(r, 4), s);
  const auto grid = [&](int64_t features) { return dim3((unsigned)((features + kF32Features - 1) / kF32Features), (unsigned)E); };
  float* out = top == 1 ? y : work_out;
  hipLaunchKernelGGL(expert_f32_kernel<true>, grid(F), dim3(512), 0, s,
                     ExpertF32Args{h, w1, work_act, ids, scores, (long)(n * top), (long)h_sr, (int)F, (int)D, (int)top});
  hipLaunchKernelGGL(expert_f32_kernel<false>, grid(D), dim3(512), 0, s,
                     ExpertF32Args{work_act, w2, out, ids, scores, (long)(n * top), (long)F, (int)D, (int)F, (int)top});
  if (top > 1)
    hipLaunchKernelGGL(expert_sum_kernel<float>, dim3((unsigned)((n * (D / 4) + 255) / 256)), dim3(256), 0, s, out, y, (long)n, (int)D, (int)top);
  return check_launch("expert_grouped_f32");
}
