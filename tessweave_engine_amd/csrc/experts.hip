// A feed-forward of routed experts: every token runs the `top` experts with the largest router scores.
//
//   z = W_router h (float32)      s = sigmoid(z)      chosen: the `top` largest (the lowest index wins a tie)
//   out = sum over the chosen experts e of  expert_e(s_e * h)         (the score multiplies the expert's INPUT)
//   expert(y): down( glu(gate y, up y) ), glu as TW_GLU_SWISH_LIMITED with the experts' limit
//
// A second kind of expert and of weighting (`kind` 1 of tw_moe_experts, `mode` 1 of tw_moe_route):
//   z = W_router h + b        chosen: the `top` largest      p = softmax over the chosen logits alone
//   out = sum over the chosen experts e of  p_e * expert_e(h)         (the weight multiplies the expert's OUTPUT)
//   expert(y): down( gelu(up y) ), the exact gelu y Phi(y); no gate matrix
//
// A third (`kind` 2, `mode` 2): gated experts whose weights multiply their outputs, a softmax over ALL logits, and experts
// without matrices:
//   s = softmax(W_router h) over X + identity logits    chosen: the `top` largest of s + correction
//   p = s of the chosen over their sum (+ 1e-20)        expert(y): down( silu(gate y) * up y ); the last `identity`
//   out = sum over the chosen experts e of  p_e * expert_e(h)          experts return h itself
//
// A fourth (`kind` 3, `mode` 0 with groups): plain experts whose weights are scaled scores that multiply their outputs,
//   s = sigmoid(W_router h); the experts stand in `groups` equal groups of neighbours, a group's score is the sum of its two
//   largest s, only experts of the best `keep` groups can be chosen;     p = scale * s of the chosen
//   out = sum over the chosen experts e of  p_e * expert_e(h)         expert(y): down( max(up y, 0)^2 )
//
// A step runs in six launches (four where there are few pairs: see PLAN below) whose shapes depend only on the number
// of rows: route; plan (every expert's rows are laid out one expert after the other, each expert's share padded to whole
// tiles of 16 rows; which expert a tile belongs to is a table on the device, tiles nobody uses say -1); gather (the
// scaled, rounded input rows in that order); two grouped products on the matrix unit, one workgroup a (tile, range of
// columns), whose weights are the tile's expert's; combine (each token adds its experts' rows in the order it chose
// them; a choice of an identity expert adds the input row itself). No launch waits for the
// host, so the whole runs inside a captured graph.
//
// The experts' matrices lie stacked, K padded to a multiple of 32 by zeros and rows to a multiple of 16, in the order the
// matrix unit's fragments are read: [X][rows / 16][K / (4 EPF)][piece 0..3][row 0..15][EPF] (EPF: the elements of 16
// bytes), so that a wave's load of one fragment is 1 KB of consecutive memory (eight cache lines; row-major, its 16 rows
// are 16 lines, and the loads queue for the cache's tag lookups):
//   gate, up [X][Fd][Cd], down [X][C16][Fd]   (Fd, Cd: the inner size and the width rounded up to 32, C16: the width
//   rounded up to 16). The gathered rows and the activations between the two products lie the same way.
#include "gemm_shared.h"

#define TW_MOE_MAX_EXPERTS 1024
#define TW_MOE_TILE 16
#define TW_MOE_WIDE 4                 /* tiles a workgroup takes at once in steps of many rows */
#define TW_MOE_SPLITK_TILES 64        /* up to this many tiles a step, the waves of a workgroup split K */

// ---- route ---------------------------------------------------------------------------------------------------
// Four consecutive elements of a row as floats.
__device__ __forceinline__ f32x4 moe_four(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
__device__ __forceinline__ f32x4 moe_four(const bf16_t* p) {
  const bf16x4 v = *reinterpret_cast<const bf16x4*>(p);
  return f32x4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
}

// A workgroup takes R rows: a wave forms two experts' logits for all of them at a time, four elements a lane and load,
// several loads in flight before the first is used (a logit is a chain of loads from memory, and their latency is all it
// costs: few rows get many waves each, many rows share a read of the router; B pieces of 256 elements go out together, all of 2,048
// where a wave has no more than its two experts). Then a wave a row chooses. (us, four pieces at a time and the choice through LDS / now: 4 rows,
// 20 experts of 2,048, softmax 6.4 / 4.7; 1 row, 16 experts 4.9 / 4.0; 8 rows, 64 experts, eight chosen 14.2 / 9.5; 1,000 rows 9.9 / 6.9.)
// Pieces behind a row's end are not read: a wave has many pairs of more than 64 experts, and each asked for up to seven pieces that it had no use for. Such
// routers have 16 waves a row up to 512 rows, which are all there at once. (us, four waves and four pieces a round with the rest apart / every piece of
// eight read / now: 512 rows of 256, 200 experts 21.9 / 41 / 20.3, 128 experts of 3,072 49 / 60 / 48, 65 rows of 1,024, 200 experts 31 / 42 / 21.)
template <typename T, int R, int WAVES, int B>
__global__ __launch_bounds__(64 * WAVES) void moe_route_kernel(const T* __restrict__ h, long ld_h, const float* __restrict__ router,
                                                               const float* __restrict__ bias, int mode, int n, int C, int X,
                                                               int top, int* __restrict__ ids, float* __restrict__ weights,
                                                               int groups, int keep, float scale) {
  __shared__ float z_s[R][TW_MOE_MAX_EXPERTS];
  __shared__ float score_s[R][TW_MOE_MAX_EXPERTS];   // mode 2: the softmax over all logits (z: what decides the choice); groups: theirs
  const int row0 = blockIdx.x * R, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const T* x[R];
#pragma unroll
  for (int r = 0; r < R; ++r) x[r] = h + (size_t)min(row0 + r, n - 1) * ld_h;
  const bool vec = C % 4 == 0 && ld_h % 4 == 0 && ((uintptr_t)h % 16 == 0) && ((uintptr_t)router % 16 == 0);
  for (int e = 2 * wave; e < X; e += 2 * WAVES) {
    const float* w0 = router + (size_t)e * C;
    const float* w1 = router + (size_t)min(e + 1, X - 1) * C;
    float s0[R], s1[R];
#pragma unroll
    for (int r = 0; r < R; ++r) s0[r] = s1[r] = 0.f;
    if (vec) {
      for (int first = 0; first < C; first += 256 * B) {
        const int c0 = first + 4 * lane;
        f32x4 a[B], b[B], xv[R][B];
#pragma unroll
        for (int j = 0; j < B; ++j) {
          if (first + 256 * j >= C) break;                 // (the same for all lanes: no piece behind the row's end is read)
          const int c = min(c0 + 256 * j, C - 4);
          a[j] = *reinterpret_cast<const f32x4*>(w0 + c);
          b[j] = *reinterpret_cast<const f32x4*>(w1 + c);
#pragma unroll
          for (int r = 0; r < R; ++r) xv[r][j] = moe_four(x[r] + c);
        }
#pragma unroll
        for (int j = 0; j < B; ++j)
          if (c0 + 256 * j < C) {
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                s0[r] = __fmaf_rn(a[j][i], xv[r][j][i], s0[r]);
                s1[r] = __fmaf_rn(b[j][i], xv[r][j][i], s1[r]);
              }
          }
      }
    } else {
      for (int c = lane; c < C; c += 64) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const float xv = tw_to_float(x[r][c]);
          s0[r] = __fmaf_rn(w0[c], xv, s0[r]);
          s1[r] = __fmaf_rn(w1[c], xv, s1[r]);
        }
      }
    }
    const bool biased = bias && mode != 2;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const float t0 = tw_wave_sum(s0[r]), t1 = tw_wave_sum(s1[r]);
      if (lane == 0) {
        z_s[r][e] = t0 + (biased ? bias[e] : 0.f);
        if (e + 1 < X) z_s[r][e + 1] = t1 + (biased ? bias[e + 1] : 0.f);
      }
    }
  }
  __syncthreads();
  if (wave >= R || row0 + wave >= n) return;
  const int row = row0 + wave;
  float* z = z_s[wave];
  float* score = score_s[wave];
  if (X <= 64 && keep == groups) {
    // An expert a lane, everything in registers: the largest of the wave, the lowest lane that holds it, and lane r keeps choice r.
    float v = lane < X ? z[lane] : -INFINITY, share = 0.f;
    if (mode == 2) {
      const float most = tw_wave_max(v);
      share = lane < X ? expf(v - most) : 0.f;
      share /= tw_wave_sum(share);
      v = lane < X ? share + (bias ? bias[lane] : 0.f) : -INFINITY;
    }
    int mine = 0;
    float weight = 0.f;
    for (int r = 0; r < top; ++r) {
      const float best = fmaxf(tw_wave_max(v), -INFINITY);            // (64 logits that are all NaN: no number is the largest)
      const unsigned long long holders = __ballot(v == best);
      const int at = min(holders ? __ffsll((long long)holders) - 1 : X - 1, X - 1);      // (no logit compares as the largest if all are NaN)
      const float chosen = mode == 2 ? share : best;
      const float w = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(chosen), at));
      if (lane == r) {
        mine = at;
        weight = w;
      }
      if (lane == at) v = -INFINITY;
    }
    auto of_choice = [&](float f, int r) { return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(f), r)); };
    if (mode == 0) {
      weight = scale / (1.f + expf(-weight));
    } else {
      // the softmax over the chosen logits (the first is the largest), or the chosen shares', added up in the order of the choices
      if (mode == 1) weight = expf(weight - of_choice(weight, 0));
      float sum = mode == 1 ? 0.f : 1e-20f;
      for (int r = 0; r < top; ++r) sum += of_choice(weight, r);
      weight /= sum;
    }
    if (lane < top) {
      ids[(size_t)row * top + lane] = mine;
      weights[(size_t)row * top + lane] = weight;
    }
    return;
  }
  if (mode == 2) {
    float most = -INFINITY, sum = 0.f;
    for (int e = lane; e < X; e += 64) most = fmaxf(most, z[e]);
    most = tw_wave_max(most);
    for (int e = lane; e < X; e += 64) {
      score[e] = expf(z[e] - most);
      sum += score[e];
    }
    sum = tw_wave_sum(sum);
    for (int e = lane; e < X; e += 64) {             // (a lane reads and writes its own experts only)
      score[e] /= sum;
      z[e] = score[e] + (bias ? bias[e] : 0.f);
    }
    __builtin_amdgcn_wave_barrier();
    __threadfence_block();
  }
  if (keep < groups) {
    // the two largest logits of every group (lanes share a group where there are few), then the groups' ranks
    const int size = X / groups;
    int share = 1;
    while (2 * share * groups <= 64) share *= 2;
    for (int g0 = 0; g0 < groups; g0 += 64 / share) {
      const int grp = g0 + lane / share;
      float b1 = -INFINITY, b2 = -INFINITY;
      if (grp < groups)
        for (int e = lane % share; e < size; e += share) {
          const float v = z[grp * size + e];
          b2 = fmaxf(b2, fminf(b1, v));
          b1 = fmaxf(b1, v);
        }
      for (int o = share / 2; o > 0; o >>= 1) {
        const float o1 = __shfl_xor(b1, o, TW_WAVE), o2 = __shfl_xor(b2, o, TW_WAVE);
        b2 = fmaxf(fminf(b1, o1), fmaxf(b2, o2));
        b1 = fmaxf(b1, o1);
      }
      if (grp < groups && lane % share == 0)
        score[grp] = 1.f / (1.f + expf(-b1)) + (size > 1 ? 1.f / (1.f + expf(-b2)) : 0.f);
    }
    __builtin_amdgcn_wave_barrier();
    __threadfence_block();
    unsigned kept = 0;                               // of groups lane, lane + 64, ..
    for (int i = 0, grp = lane; grp < groups; grp += 64, ++i) {
      const float mine = score[grp];
      int rank = 0;
      for (int j = 0; j < groups; ++j) rank += score[j] > mine || (score[j] == mine && j < grp) ? 1 : 0;
      kept |= rank < keep ? 1u << i : 0u;
    }
    __builtin_amdgcn_wave_barrier();
    __threadfence_block();
    for (int i = 0, grp = lane; grp < groups; grp += 64, ++i) score[grp] = (kept >> i) & 1u ? 1.f : 0.f;
    __builtin_amdgcn_wave_barrier();
    __threadfence_block();
    for (int e = lane; e < X; e += 64)
      if (score[e / size] == 0.f) z[e] = -INFINITY;
    __builtin_amdgcn_wave_barrier();
    __threadfence_block();
  }
  for (int r = 0; r < top; ++r) {
    float best = -INFINITY;
    int at = 0x7fffffff;
    for (int e = lane; e < X; e += 64) {
      const float v = z[e];
      if (v > best || (v == best && e < at)) { best = v; at = e; }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const float ov = __shfl_xor(best, o, TW_WAVE);
      const int oa = __shfl_xor(at, o, TW_WAVE);
      if (ov > best || (ov == best && oa < at)) { best = ov; at = oa; }
    }
    at = min(at, X - 1);                             // (no logit compares as the largest if all are NaN)
    if (lane == 0) {
      ids[(size_t)row * top + r] = at;
      weights[(size_t)row * top + r] = mode == 2 ? score[at] : mode == 1 ? best : scale / (1.f + expf(-best));
      z[at] = -INFINITY;
    }
    __builtin_amdgcn_wave_barrier();
    __threadfence_block();
  }
  if (mode == 1 && lane == 0) {
    // the softmax over the chosen logits alone (the first chosen is the largest), in the order they were chosen
    float* w = weights + (size_t)row * top;
    const float first = w[0];
    float sum = 0.f;
    for (int r = 0; r < top; ++r) {
      w[r] = expf(w[r] - first);
      sum += w[r];
    }
    for (int r = 0; r < top; ++r) w[r] = w[r] / sum;
  }
  if (mode == 2 && lane == 0) {
    float* w = weights + (size_t)row * top;
    float sum = 1e-20f;
    for (int r = 0; r < top; ++r) sum += w[r];
    for (int r = 0; r < top; ++r) w[r] = w[r] / sum;
  }
}

extern "C" int tw_moe_route(int dtype, const void* h, long ld_h, const float* router, const float* bias, int mode, int n, int C,
                            int X, int top, int* ids, float* weights, int groups, int keep, float scale, hipStream_t stream) {
  TW_REQUIRE(h && router && ids && weights && n >= 0 && C > 0 && ld_h >= C && mode >= 0 && mode <= 2);
  TW_REQUIRE(X > 0 && X <= TW_MOE_MAX_EXPERTS && top > 0 && top <= X);
  TW_REQUIRE(groups >= 1 && X % groups == 0 && keep >= 1 && keep <= groups && top <= keep * (X / groups));
  TW_REQUIRE(mode == 0 || (keep == groups && scale == 1.f));
  if (n == 0) return 0;
#define TW_MOE_ROUTE(T)                                                                                                 \
  do {                                                                                                                  \
    if (n <= 64 && X <= 32) moe_route_kernel<T, 1, 16, 8><<<n, 1024, 0, stream>>>((const T*)h, ld_h, router, bias, mode, n, C, X, top, ids, weights, groups, keep, scale); \
    else if (n <= 64 || (n <= 512 && X > 64)) moe_route_kernel<T, 1, 16, 4><<<n, 1024, 0, stream>>>((const T*)h, ld_h, router, bias, mode, n, C, X, top, ids, weights, groups, keep, scale); \
    else if (n <= 512) moe_route_kernel<T, 1, 4, 8><<<n, 256, 0, stream>>>((const T*)h, ld_h, router, bias, mode, n, C, X, top, ids, weights, groups, keep, scale); \
    else moe_route_kernel<T, 4, 8, 2><<<tw_div_up(n, 4), 512, 0, stream>>>((const T*)h, ld_h, router, bias, mode, n, C, X, top, ids, weights, groups, keep, scale); \
  } while (0)
  if (dtype == TW_DTYPE_BF16) TW_MOE_ROUTE(bf16_t);
  else if (dtype == TW_DTYPE_F32) TW_MOE_ROUTE(float);
  else return TW_ERR_BAD_ARGUMENT;
#undef TW_MOE_ROUTE
  return TW_LAUNCH_RESULT();
}

// ---- plan ----------------------------------------------------------------------------------------------------
// items = n * top pairs (token, choice). pos[item]: the pair's row in the experts' order; src_item[row]: the pair of a
// row, -1 for padding (a pair whose expert is number X or above, one without matrices, gets no row: pos -1); tile_expert[tile]: the expert of rows 16 tile .., -1 for a tile behind the last one in use.
// Which of an expert's rows a pair gets depends on the order the atomics arrive in; no result depends on it, since
// every row is computed for itself and a token adds its rows in the order of its choices.
__global__ __launch_bounds__(1024) void moe_plan_kernel(const int* __restrict__ ids, int items, int X, int* __restrict__ pos,
                                                        int* __restrict__ src_item, int* __restrict__ tile_expert,
                                                        int capacity, int tiles, int unit) {
  __shared__ int count[TW_MOE_MAX_EXPERTS];
  __shared__ int offset[TW_MOE_MAX_EXPERTS + 1];
  for (int e = threadIdx.x; e < X; e += blockDim.x) count[e] = 0;
  for (int r = threadIdx.x; r < capacity; r += blockDim.x) src_item[r] = -1;
  for (int t = threadIdx.x; t < tiles; t += blockDim.x) tile_expert[t] = -1;
  __syncthreads();
  for (int i = threadIdx.x; i < items; i += blockDim.x) pos[i] = ids[i] < X ? atomicAdd(&count[ids[i]], 1) : -1;
  __syncthreads();
  if (threadIdx.x == 0) {
    int at = 0;
    for (int e = 0; e < X; ++e) {
      offset[e] = at;
      at += (count[e] + unit - 1) / unit * unit;
    }
    offset[X] = at;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < X; e += blockDim.x)
    for (int t = offset[e] / TW_MOE_TILE; t < offset[e + 1] / TW_MOE_TILE; ++t) tile_expert[t] = e;
  for (int i = threadIdx.x; i < items; i += blockDim.x) {
    if (ids[i] >= X) continue;
    const int row = offset[ids[i]] + pos[i];
    pos[i] = row;
    src_item[row] = i;
  }
}

// The rows an expert's share is padded to: one tile, or, once the experts have a tile's rows each on average, the
// TW_MOE_WIDE tiles that one workgroup of the grouped products then takes against one read of the expert's matrices.
static int moe_unit(long items, int X) { return items >= (long)TW_MOE_TILE * X ? TW_MOE_TILE * TW_MOE_WIDE : TW_MOE_TILE; }

extern "C" long tw_moe_capacity(long items, int X) {
  // rows the experts' order can take: every expert's share rounded up to whole units (never fewer for more items)
  const long unit = moe_unit(items, X);
  return (items + (long)X * (unit - 1) + unit - 1) / unit * unit;
}

extern "C" int tw_moe_plan(const int* ids, int items, int X, int* pos, int* src_item, int* tile_expert, int capacity,
                           hipStream_t stream) {
  TW_REQUIRE(ids && pos && src_item && tile_expert && items >= 0 && X > 0 && X <= TW_MOE_MAX_EXPERTS);
  TW_REQUIRE(capacity >= tw_moe_capacity(items, X) && capacity % TW_MOE_TILE == 0);
  if (items == 0) return 0;
  moe_plan_kernel<<<1, 1024, 0, stream>>>(ids, items, X, pos, src_item, tile_expert, capacity, capacity / TW_MOE_TILE,
                                          moe_unit(items, X));
  return TW_LAUNCH_RESULT();
}

// ---- gather: xs[row] = round(weight * h[token]) in the experts' order, zeros in padding rows and behind C ----------
// A workgroup takes a tile's 16 rows and every gridDim.y-th group of 16 pieces of them: a thread a (row, piece), so that what
// a wave writes is consecutive (xs lies in fragment order).
template <typename T>
__global__ __launch_bounds__(256) void moe_gather_kernel(const T* __restrict__ h, long ld_h, const float* __restrict__ weights,
                                                         const int* __restrict__ src_item, const int* __restrict__ tile_expert,
                                                         T* __restrict__ xs, int C, int Cd, int top) {
  const int tile = blockIdx.x;
  if (tile_expert[tile] < 0) return;
  constexpr int EPF = Elem<T>::kPerFrag;
  const int r = threadIdx.x % TW_MOE_TILE;
  const int item = src_item[tile * TW_MOE_TILE + r];
  const float w = weights && item >= 0 ? weights[item] : 1.f;             // (no weights: they multiply the experts' outputs instead)
  const T* src = h + (item >= 0 ? (size_t)(item / top) * ld_h : 0);
  const bool vec = ld_h % EPF == 0 && (uintptr_t)h % 16 == 0;
  T* dst = xs + (size_t)tile * Cd * TW_MOE_TILE;
#pragma unroll 4
  for (int p = threadIdx.x / TW_MOE_TILE + 16 * blockIdx.y; p < Cd / EPF; p += 16 * gridDim.y) {
    typename Elem<T>::Frag v = Elem<T>::zero();
    const int c = p * EPF;
    if (item >= 0) {
      if (vec && c + EPF <= C) {
        v = tw_load_frag(src + c);
        if (weights) {
#pragma unroll
          for (int e = 0; e < EPF; ++e) v[e] = tw_from_float<T>(w * tw_to_float(v[e]));
        }
      } else {
#pragma unroll
        for (int e = 0; e < EPF; ++e)
          if (c + e < C) v[e] = tw_from_float<T>(w * tw_to_float(src[c + e]));
      }
    }
    *reinterpret_cast<typename Elem<T>::Frag*>(dst + ((size_t)p * TW_MOE_TILE + r) * EPF) = v;
  }
}

// ---- the grouped products ---------------------------------------------------------------------------------------
// One workgroup: a tile of 16 rows against 4 waves x NT x 16 columns of its expert's matrix W[ex] ([N][K], K a multiple
// of 32). GLU: W and W2 are gate and up, the result glu(gate, up) goes out in the compute type; otherwise the float32
// product. Operands go from memory straight into fragments (lane = 16 * piece + row reads 16 bytes).
// SPLITK (steps of few rows, where the tiles in use are too few to fill the chip and every one streams its expert's whole
// matrix; some of many rows, see moe_splits_k): the waves share one range of NT x 16 columns and take every WAVES-th
// step over K each; their sums meet in LDS and are added in the order of the waves. The ranges are the grid's first dimension there:
// workgroups go round the 8 XCDs in that order, and with the tiles first all ranges of a tile met on one XCD, so that five tiles
// kept five eighths of the chip busy and ten one eighth for twice as long (see moe_few_form). With several tiles a workgroup the
// units stay first: nearly all hold rows (float32, 8 experts of 224 x 320, 437 tokens 27.9 / 25.8 us).
// MT > 1 (steps of many rows, whose experts' shares are padded to MT tiles): a workgroup takes MT tiles of one expert
// against every fragment of the expert's matrices it reads.
template <int N> struct MoeCount { static constexpr int value = N; };
// ACT 0: the float32 product; 1: gate and up with the limited swish; 2: one matrix with the exact gelu; 3: gate and up with
// SiLU; 4: one matrix with the square of relu (1 to 4 write the next product's rows in the compute type).
// PLAN (the first product of steps of at most 64 (token, choice) pairs whose weights multiply outputs): there is no plan
// and no gather launch. Every wave finds the tiles itself, lane i holding pair i: a pair whose expert has 16 m pairs before
// it opens a tile, the tiles are numbered in the order of the pairs that open them, and the rows are read where they lie in
// h. The tile's first workgroup writes what the second product and the combination read: tile_expert, pos.
struct MoePairs {
  const int* ids;       // [items]
  int items, top, X;
  long ld_h;
  int* tile_expert;
  int* pos;
};
template <typename T, int ACT, int NT, bool SPLITK = false, int MT = 1, bool PLAN = false, int WAVES = 4, int STEPS = 4, bool AHEAD = false>
__global__ __launch_bounds__(WAVES * 64) void moe_grouped_kernel(const T* __restrict__ A, long lda, const T* __restrict__ W,
                                                          const T* __restrict__ W2, const int* __restrict__ tile_expert,
                                                          void* __restrict__ out, long ldo, int N, int K, float limit,
                                                          MoePairs pairs = {}) {
  constexpr int EPF = Elem<T>::kPerFrag;
  constexpr bool GLU = ACT == 1 || ACT == 3;
  constexpr bool RANGES_FIRST = SPLITK && MT == 1;
  const int tile = (RANGES_FIRST ? blockIdx.y : blockIdx.x) * MT, range = RANGES_FIRST ? blockIdx.x : blockIdx.y;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  int ex, row_of_lane = 0;                           // PLAN: the row of h that lane's row r of the tile is
  if constexpr (PLAN) {
    const int mine = lane < pairs.items ? pairs.ids[lane] : -1;
    const bool real = mine >= 0 && mine < pairs.X;
    int before = 0;                                  // pairs of the same expert before this one
    for (int i = 0; i < pairs.items; ++i) {
      const int other = __builtin_amdgcn_readlane(mine, i);
      before += (i < lane && other == mine) ? 1 : 0;
    }
    const unsigned long long opens = __ballot(real && before % TW_MOE_TILE == 0);
    int opener = -1;                                 // the pair that opens this tile
    {
      unsigned long long left = opens;
      for (int i = 0; i < tile && left; ++i) left &= left - 1;
      if (left) opener = __ffsll((unsigned long long)left) - 1;
    }
    const bool leads = range == 0 && wave == 0;
    if (leads && tile == 0 && lane < pairs.items && !real) pairs.pos[lane] = -1;
    if (opener < 0) {
      if (leads && lane == 0) pairs.tile_expert[tile] = -1;
      return;
    }
    ex = __builtin_amdgcn_readlane(mine, opener);
    const int from = __builtin_amdgcn_readlane(before, opener);
    const bool here = real && mine == ex && before >= from && before < from + TW_MOE_TILE;
    unsigned long long members = __ballot(here);
    if (leads) {
      if (lane == 0) pairs.tile_expert[tile] = ex;
      if (here) pairs.pos[lane] = tile * TW_MOE_TILE + before - from;
    }
    // row j of the tile is its j-th member; rows behind the last repeat the first (nobody reads what they give)
    int pair = opener;
    for (int i = 0; i < TW_MOE_TILE && members; ++i) {
      const int m = __ffsll((unsigned long long)members) - 1;
      members &= members - 1;
      if (i == r) pair = m;
    }
    row_of_lane = pair / pairs.top;
  } else {
    ex = tile_expert[tile];
    if (ex < 0) return;
  }
  const int col0 = (SPLITK ? range : range * 4 + wave) * 16 * NT;
  if (col0 >= N) return;
  constexpr int KSTEP = 4 * EPF;
  constexpr int BLK = 64 * EPF;                      // elements of one step's fragment of a tile: lane l's at l * EPF
  constexpr int k_stride = (SPLITK ? WAVES : 1) * BLK;    // (k counts the elements of a tile's fragments, step after step)
  const int k_first = SPLITK ? wave * BLK : 0;
  const size_t tile_elems = (size_t)K * TW_MOE_TILE;  // all steps of one tile of 16 rows
  const int n_blocks = (N + 15) / 16;
  const T* a_ptr = PLAN ? A + (size_t)row_of_lane * pairs.ld_h + g * EPF : A + (size_t)tile * tile_elems + lane * EPF;
  const T* w_ptr[NT];
  const T* w2_ptr[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const size_t at = ((size_t)ex * n_blocks + min(col0 / 16 + t, n_blocks - 1)) * tile_elems + lane * EPF;
    w_ptr[t] = W + at;
    w2_ptr[t] = GLU ? W2 + at : nullptr;
  }
  f32x4 acc[MT][NT], acc2[MT][NT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[m][t] = acc2[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  // U steps' operands are on their way before the first is used, where waves share columns of many rows (and in AHEAD) those of
  // the U steps behind them too: what bounds this loop is the latency of memory
  constexpr int U = MT > 1 ? 2 : GLU ? STEPS : (NT > 2 ? STEPS : 2 * STEPS);
  struct Operands {
    typename Elem<T>::Frag a[U][MT], b[U][NT], b2[GLU ? U : 1][NT];
  };
  auto load = [&](int k, auto count, Operands& o) {
    constexpr int UN = decltype(count)::value;
#pragma unroll
    for (int u = 0; u < UN; ++u) {
#pragma unroll
      for (int m = 0; m < MT; ++m) o.a[u][m] = tw_load_frag(PLAN ? a_ptr + (k + u * k_stride) / TW_MOE_TILE
                                                                          : a_ptr + (size_t)m * tile_elems + k + u * k_stride);
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        // (few rows: an expert's matrices are read once a step)
        o.b[u][t] = SPLITK ? tw_load_frag_stream(w_ptr[t] + k + u * k_stride) : tw_load_frag(w_ptr[t] + k + u * k_stride);
        if (GLU) o.b2[GLU ? u : 0][t] = SPLITK ? tw_load_frag_stream(w2_ptr[t] + k + u * k_stride) : tw_load_frag(w2_ptr[t] + k + u * k_stride);
      }
    }
    __builtin_amdgcn_sched_barrier(0);               // (the scheduler would put each load in front of its use to save registers)
  };
  auto multiply = [&](auto count, const Operands& o) {
    constexpr int UN = decltype(count)::value;
#pragma unroll
    for (int u = 0; u < UN; ++u)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          tw_mma16(acc[m][t], o.a[u][m], o.b[u][t]);
          if (GLU) tw_mma16(acc2[m][t], o.a[u][m], o.b2[GLU ? u : 0][t]);
        }
    if constexpr (SPLITK && (MT > 1 || AHEAD)) __builtin_amdgcn_sched_barrier(0);
  };
  int k = k_first;
  const int k_end = (int)tile_elems;
  if constexpr (SPLITK && (MT > 1 || AHEAD)) {
    constexpr int BATCH = U * k_stride;
    const int last = k_end - (U - 1) * k_stride;     // a batch that begins before it is whole
    Operands even, odd;
    if (k < last) load(k, MoeCount<U>(), even);
    for (; k < last; k += 2 * BATCH) {
      if (k + BATCH < last) load(k + BATCH, MoeCount<U>(), odd);
      multiply(MoeCount<U>(), even);
      if (k + BATCH >= last) {
        k += BATCH;
        break;
      }
      if (k + 2 * BATCH < last) load(k + 2 * BATCH, MoeCount<U>(), even);
      multiply(MoeCount<U>(), odd);
    }
    for (; k < k_end; k += k_stride) {
      load(k, MoeCount<1>(), even);
      multiply(MoeCount<1>(), even);
    }
  } else if constexpr (sizeof(T) == 4 && !GLU && (SPLITK || ACT != 0)) {
    // (operands that outlive a step: other code, ten registers less than below; faster in float32 without a gate, 8 experts of 4,096 x
    // 2,048, 80 tokens 585 -> 540 us, but in bfloat16, with a gate and in the last product of many rows up to 6 % slower)
    Operands now;
    for (; k + (U - 1) * k_stride < k_end; k += U * k_stride) {
      load(k, MoeCount<U>(), now);
      multiply(MoeCount<U>(), now);
    }
    for (; k < k_end; k += k_stride) {
      load(k, MoeCount<1>(), now);
      multiply(MoeCount<1>(), now);
    }
  } else {
    auto steps = [&](int k, auto count) {
      constexpr int U = decltype(count)::value;
      typename Elem<T>::Frag a[U][MT], b[U][NT], b2[U][NT];
#pragma unroll
      for (int u = 0; u < U; ++u) {
#pragma unroll
        for (int m = 0; m < MT; ++m) a[u][m] = tw_load_frag(PLAN ? a_ptr + (k + u * k_stride) / TW_MOE_TILE
                                                                            : a_ptr + (size_t)m * tile_elems + k + u * k_stride);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          // (few rows: an expert's matrices are read once a step)
          b[u][t] = SPLITK ? tw_load_frag_stream(w_ptr[t] + k + u * k_stride) : tw_load_frag(w_ptr[t] + k + u * k_stride);
          if (GLU) b2[u][t] = SPLITK ? tw_load_frag_stream(w2_ptr[t] + k + u * k_stride) : tw_load_frag(w2_ptr[t] + k + u * k_stride);
        }
      }
      __builtin_amdgcn_sched_barrier(0);               // (the scheduler would put each load in front of its use to save registers)
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int m = 0; m < MT; ++m) {
            tw_mma16(acc[m][t], a[u][m], b[u][t]);
            if (GLU) tw_mma16(acc2[m][t], a[u][m], b2[u][t]);
          }
    };
    for (; k + (U - 1) * k_stride < k_end; k += U * k_stride) steps(k, MoeCount<U>());
    for (; k < k_end; k += k_stride) steps(k, MoeCount<1>());
  }
  if constexpr (SPLITK) {
    __shared__ f32x4 part[GLU ? 2 : 1][WAVES - 1][MT][NT][64];
    if (wave > 0) {
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          part[0][wave - 1][m][t][lane] = acc[m][t];
          if (GLU) part[GLU ? 1 : 0][wave - 1][m][t][lane] = acc2[m][t];
        }
    }
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int w = 0; w < WAVES - 1; ++w)
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          acc[m][t] += part[0][w][m][t][lane];
          if (GLU) acc2[m][t] += part[GLU ? 1 : 0][w][m][t][lane];
        }
  }
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int col = col0 + t * 16 + r;
      if (col >= N) continue;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (ACT != 0) {
          // the activations are the next product's rows: in fragment order too (ldo: the elements of a row)
          const size_t at = (size_t)(tile + m) * ldo * TW_MOE_TILE + ((size_t)(col / EPF) * TW_MOE_TILE + 4 * g + j) * EPF + col % EPF;
          const float z = acc[m][t][j];
          ((T*)out)[at] = tw_from_float<T>(ACT == 1 ? tw_swish_limited(z, acc2[m][t][j], limit)
                                               : ACT == 3 ? tw_silu(z) * acc2[m][t][j]
                                               : ACT == 4 ? fmaxf(z, 0.f) * fmaxf(z, 0.f)
                                               : 0.5f * z * (1.f + erff(z * 0.70710678118654752f)));
        } else {
          ((float*)out)[(size_t)((tile + m) * TW_MOE_TILE + 4 * g + j) * ldo + col] = acc[m][t][j];
        }
      }
    }
}

// float32, steps of many rows: the same products from three bfloat16 parts an operand (gemm_parts_kernel says why and how exact). One
// workgroup: a unit's 64 rows against 64 * WN rows of its expert's matrices (GLU: half of gate, half of up, of the same columns), waves in
// a 2x2 grid, wave tile 32 x (32 * WN). A k-tile is two k-steps; rows and matrices are read in fragment order, split and laid into LDS, two
// k-tiles are on their way (the matrices come from HBM) and three workgroups share a CU. What is not finite, and nothing beside it, is
// formed again from the operands themselves. All launches of the experts, us, the float32 MFMA / this: 16 experts of 2,048 x 1,408, two a token, gated, 128 tokens
// 303 / 198, 478 423 / 266, 2,000 956 / 673; 8 of 4,096 x 2,048, 300 tokens 751 / 497; 64 of 1,024 x 512, four a token, 300 tokens 274 / 154.
// (With six products and one k-tile on its way the first took 181 us against 163; at two workgroups a CU 179, and 478 tokens 257 against 221.)
template <int ACT, int WN>
__global__ __launch_bounds__(256, WN == 2 ? 3 : 4) void moe_parts_kernel(const float* __restrict__ A, const float* __restrict__ W, const float* __restrict__ W2,
                                                           const int* __restrict__ tile_expert, float* __restrict__ out, long ldo, int N, int K,
                                                           float limit) {
  constexpr bool GLU = ACT == 1 || ACT == 3;
  static_assert(!GLU || WN == 2, "a wave holds gate and up");
  constexpr int ROWS = 64 + 64 * WN, PART = ROWS * TW_PART_ROW, COLS = GLU ? 64 : 64 * WN;
  __shared__ __attribute__((aligned(16))) char lds[3 * PART];
  const int tile = blockIdx.x * TW_MOE_WIDE;
  const int ex = tile_expert[tile];
  if (ex < 0) return;
  const int col0 = blockIdx.y * COLS;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 31, g = lane >> 5;
  const int wm0 = (wave >> 1) * 32;
  const size_t tile_elems = (size_t)K * TW_MOE_TILE;
  const int n_blocks = (N + 15) / 16;
  // the matrix row of LDS row `row` behind the unit's 64, and where its block of 16 begins
  auto block_of = [&](int row) {
    const bool second = GLU && row >= 64;
    const int block = min((col0 + (second ? row - 64 : row)) / 16, n_blocks - 1);
    return (second ? W2 : W) + ((size_t)ex * n_blocks + block) * tile_elems;
  };
  auto wave_row = [&](int j) { return GLU ? 64 * j + (wave & 1) * 32 : (wave & 1) * 32 * WN + 32 * j; };

  f32x16 acc[WN], small[WN];
#pragma unroll
  for (int j = 0; j < WN; ++j)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[j][e] = small[j][e] = 0.f;

  const float* src[1 + WN];                                    // a thread's pieces: one of the rows, WN of the matrices
  int at[1 + WN];
  {
    const int row = tid & 15, p = (tid >> 4) & 3, in_block = (p >> 1) * 256 + (p & 1) * 128 + row * 4;
    src[0] = A + (size_t)(tile + wave) * tile_elems + in_block;
    at[0] = tw_part_place(wave * 16 + row, p);
#pragma unroll
    for (int i = 0; i < WN; ++i) {
      src[1 + i] = block_of(i * 64 + wave * 16) + in_block;
      at[1 + i] = tw_part_place(64 + i * 64 + wave * 16 + row, p);
    }
  }
  // (two k-tiles on their way: the experts' matrices come from HBM)
  f32x4 regs[2][1 + WN][2];
  auto load = [&](int kt, f32x4 (&reg)[1 + WN][2]) {
#pragma unroll
    for (int i = 0; i <= WN; ++i) {
      reg[i][0] = tw_load_frag(src[i] + (size_t)kt * 512);
      reg[i][1] = tw_load_frag(src[i] + (size_t)kt * 512 + 64);
    }
  };
  const int swz = (r >> 2) & 3;
  const int k_tiles = K / 32;
  auto k_tile = [&](int kt, f32x4 (&reg)[1 + WN][2]) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i <= WN; ++i) {
      bf16x8 h, m, l;
      tw_three_parts(reg[i][0], reg[i][1], h, m, l);
      *reinterpret_cast<bf16x8*>(lds + at[i]) = h;
      *reinterpret_cast<bf16x8*>(lds + PART + at[i]) = m;
      *reinterpret_cast<bf16x8*>(lds + 2 * PART + at[i]) = l;
    }
    load(min(kt + 2, k_tiles - 1), reg);                       // (unconditional: the last one again behind the end)
    __syncthreads();
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int piece = ((2 * s + g) ^ swz) * 16;
      bf16x8 af[3], wf[3][WN];
#pragma unroll
      for (int p = 2; p >= 0; --p) {
        af[p] = *reinterpret_cast<const bf16x8*>(lds + p * PART + (wm0 + r) * TW_PART_ROW + piece);
#pragma unroll
        for (int j = 0; j < WN; ++j) wf[p][j] = *reinterpret_cast<const bf16x8*>(lds + p * PART + (64 + wave_row(j) + r) * TW_PART_ROW + piece);
      }
      auto product = [&](f32x16 (&sum)[WN], int p, int q) {
#pragma unroll
        for (int j = 0; j < WN; ++j) tw_mma32(sum[j], af[p], wf[q][j]);
      };
      TW_PART_PRODUCTS(product);
    }
  };
  load(0, regs[0]);
  load(min(1, k_tiles - 1), regs[1]);
  int kt = 0;
  for (; kt + 1 < k_tiles; kt += 2) {
    k_tile(kt, regs[0]);
    k_tile(kt + 1, regs[1]);
  }
  if (kt < k_tiles) k_tile(kt, regs[0]);

  float odd = 0.f;                                             // NaN as soon as one of them is not finite
#pragma unroll
  for (int j = 0; j < WN; ++j)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      acc[j][e] += small[j][e];
      odd = __fmaf_rn(acc[j][e], 0.f, odd);
    }
  if (__syncthreads_or(odd != odd)) {
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) small[j][e] = 0.f;
    const int in_block = g * 64 + (r & 15) * 4;
    const float* a = A + (size_t)(tile + (wm0 + r) / 16) * tile_elems + in_block;
    const float* w[WN];
#pragma unroll
    for (int j = 0; j < WN; ++j) w[j] = block_of(wave_row(j) + r) + in_block;
    for (int k = 0; k < K; k += 8)                             // (8 elements of K are 128 floats of a block)
#pragma unroll
      for (int j = 0; j < WN; ++j) tw_mma32(small[j], tw_load_frag(a + (size_t)k * 16), tw_load_frag(w[j] + (size_t)k * 16));
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[j][e] = acc[j][e] * 0.f == 0.f ? acc[j][e] * TW_PART_BACK : small[j][e];
  } else {
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[j][e] *= TW_PART_BACK;
  }

#pragma unroll
  for (int j = 0; j < (GLU ? 1 : WN); ++j) {
    const int col = col0 + (GLU ? (wave & 1) * 32 : wave_row(j)) + r;
    if (col >= N) continue;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int row = wm0 + 8 * (e / 4) + 4 * g + e % 4;
      const float z = acc[j][e];
      if (ACT == 0) {
        out[(size_t)(tile * TW_MOE_TILE + row) * ldo + col] = z;
      } else {
        const float y = ACT == 1 ? tw_swish_limited(z, acc[WN - 1][e], limit) : ACT == 3 ? tw_silu(z) * acc[WN - 1][e]
                        : ACT == 4 ? fmaxf(z, 0.f) * fmaxf(z, 0.f) : 0.5f * z * (1.f + erff(z * 0.70710678118654752f));
        out[(size_t)(tile + row / 16) * ldo * TW_MOE_TILE + ((size_t)(col / 4) * TW_MOE_TILE + row % 16) * 4 + col % 4] = y;
      }
    }
  }
}

// ---- combine: x[token] += its experts' rows, in the order of its choices ------------------------------------------
// A workgroup takes 1,024 columns of a row, four a thread where rows and addresses allow 16-byte accesses.
// weights (or null): a factor on each of the token's rows; accumulate 0: x is written, not added to. more (or null):
// float32 [splits][n][C] partial sums of something else that belongs to the same result (a shared expert's last product
// with its K ranges not yet added up): added here, in index order, before the experts' rows.
// A choice without a row (pos -1) is an expert that returns h itself.
struct MoeCombineArgs {
  float* x; long ld_x;
  const float* ys; long ld_y;
  const int* pos;
  const float* weights;
  const float* more; size_t more_stride;
  const void* h; long ld_h;
  int C, top, splits, accumulate;
};

// Columns c .. c + 3 of a row's sum. Of up to four choices at a time the rows' places go out together, then the rows, and the row itself only where a
// choice has none (2,048 rows of 2,048, two choices of eight experts, all launches 78.4 -> 76 us).
template <typename T>
__device__ __forceinline__ f32x4 moe_combined(const MoeCombineArgs& a, int row, int c) {
  f32x4 sum = {0.f, 0.f, 0.f, 0.f};
  if (a.more)
    for (int s = 0; s < a.splits; ++s) sum += *reinterpret_cast<const f32x4*>(a.more + s * a.more_stride + (size_t)row * a.C + c);
  for (int r0 = 0; r0 < a.top; r0 += 4) {
    int at[4];
    float w[4];
    f32x4 y[4], own = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const size_t item = (size_t)row * a.top + min(r0 + j, a.top - 1);
      at[j] = a.pos[item];
      w[j] = a.weights ? a.weights[item] : 1.f;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) y[j] = *reinterpret_cast<const f32x4*>(a.ys + (size_t)max(at[j], 0) * a.ld_y + c);
    if (min(min(at[0], at[1]), min(at[2], at[3])) < 0) own = moe_four((const T*)a.h + (size_t)row * a.ld_h + c);      // (the same for a row's lanes)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (r0 + j < a.top) sum += w[j] * (at[j] >= 0 ? y[j] : own);
  }
  return sum;
}

template <typename T, bool VEC>
__global__ __launch_bounds__(256) void moe_combine_kernel(MoeCombineArgs a) {
  const int row = blockIdx.x;
  const int c = blockIdx.y * 1024 + threadIdx.x * 4;
  if (c >= a.C) return;
  if constexpr (VEC) {
    f32x4* dst = reinterpret_cast<f32x4*>(a.x + (size_t)row * a.ld_x + c);
    const f32x4 before = a.accumulate ? *dst : f32x4{0.f, 0.f, 0.f, 0.f};
    const f32x4 sum = moe_combined<T>(a, row, c);
    *dst = a.accumulate ? before + sum : sum;
  } else {
    const T* own = (const T*)a.h + (size_t)row * a.ld_h + c;
    for (int j = 0; j < 4 && c + j < a.C; ++j) {
      float sum = 0.f;
      if (a.more)
        for (int s = 0; s < a.splits; ++s) sum += a.more[s * a.more_stride + (size_t)row * a.C + c + j];
      for (int r = 0; r < a.top; ++r) {
        const int at = a.pos[(size_t)row * a.top + r];
        sum += (a.weights ? a.weights[(size_t)row * a.top + r] : 1.f) * (at >= 0 ? a.ys[(size_t)at * a.ld_y + c + j] : tw_to_float(own[j]));
      }
      float* x = a.x + (size_t)row * a.ld_x + c + j;
      *x = a.accumulate ? *x + sum : sum;
    }
  }
}

// The same with the RMS norm of the new rows behind it, out = round(x / sqrt(mean(x^2) + eps) * weight): rows of up to 4,096 elements, a
// workgroup each, so that the stream's next reader needs no launch of its own in front of it (a captured step of float32 layers with
// experts, 4 rows, 469 us with launches of their own and the routers as they were, 445 with both). out may be h.
template <typename T>
__global__ __launch_bounds__(1024) void moe_combine_norm_kernel(MoeCombineArgs a, const float* __restrict__ weight, float eps, T* out) {
  __shared__ float lds[16];
  const int row = blockIdx.x, c = min((int)threadIdx.x * 4, a.C - 4);
  const bool mine = (int)threadIdx.x * 4 < a.C;
  float* x = a.x + (size_t)row * a.ld_x + c;
  const f32x4 before = *reinterpret_cast<const f32x4*>(x), w = *reinterpret_cast<const f32x4*>(weight + c);
  const f32x4 v = before + moe_combined<T>(a, row, c);
  const float ss = mine ? ((v[0] * v[0] + v[1] * v[1]) + v[2] * v[2]) + v[3] * v[3] : 0.f;
  const float rinv = 1.0f / sqrtf(tw_block_sum(ss, lds) / (float)a.C + eps);       // (the barrier: every read of the row, clamped ones too, lies before)
  if (!mine) return;
  *reinterpret_cast<f32x4*>(x) = v;
  T* dst = out + (size_t)row * a.C + c;
#pragma unroll
  for (int e = 0; e < 4; ++e) dst[e] = tw_from_float<T>(v[e] * rinv * w[e]);
}

// Steps of many rows: do the waves of a workgroup better split K than the columns? (float32, 16 experts of 2,048 x 1,408 gated, two a
// token, all launches of the experts, us, columns / K: 134 to 256 tokens 305 / 310, 268 to 440 tokens 473 / 315, 500 tokens 473 / 420; 8
// experts, 300 tokens 298 / 299, 500 tokens 425 / 384; 4 experts, 600 tokens 278 / 355.) A range of columns a wave leaves a CU that
// holds one workgroup a wave a SIMD, 125 us of MFMAs at K = 2,048, so what counts are the rounds of workgroups on the 256 CUs (8
// more are still one: units without rows end at once). With K split there are four times as many, a quarter as long and 1.4
// times as dear, every wave reading rows of its own. Where experts have one unit each, half of the units are empty, which
// costs whole columns' rounds and next to nothing with K split. Of 222 steps of 17 to 32 units (1 to 64 experts, 256 to 4,096 x 96 to
// 5,632) the rule is 0.8 % behind the better of the two in the mean; 6 are 4 to 11 % slower than by columns.
// In bfloat16, whose MFMAs take a tenth of the time, K split is 17 % slower in the mean and up to 2.2 times; there only gated
// products of long sums with one unit an expert have it (16 experts of 2,048 x 1,408, 268 to 440 tokens 121 / 93; of 4,096 x 1,408, 300
// tokens 234 / 154; but of 1,024 x 1,408 53 / 60, and without a gate 70 / 73).
#define TW_MOE_SPLITK_UNITS 32
static bool moe_splits_k(bool f32, int units, long items, int X, int C, int Cd, int Fd, bool gated) {
  if (units > TW_MOE_SPLITK_UNITS) return false;
  const int up = units * tw_div_up(Fd, 4 * 16 * 2), down = units * tw_div_up(C, 4 * 16 * 2);
  if (items <= 60L * X && up > 264 && (f32 || (gated && Cd >= 2048))) return true;
  if (!f32) return false;
  const double first = (gated ? 2.0 : 1.0) * Cd;
  const double columns = first * tw_div_up(up, 264) + (double)Fd * tw_div_up(down, 264);
  const double ranges = first * tw_div_up(units * tw_div_up(Fd, 16 * 2), 256) + (double)Fd * tw_div_up(units * tw_div_up(C, 16 * 2), 256);
  return 1.4 * ranges / 4 < columns;
}

// Steps of few rows: columns a workgroup (NT x 16), waves and k-steps a request, for either product by itself. What bounds few workgroups
// is the tail of the last ones and a wave's chain of requests, so the pieces are small: 16 columns, in float32 (whose MFMAs take as long as the
// loads) 16 waves of 2 steps, in bfloat16 8 waves with 2 steps on their way behind 2. Many fill the chip whatever the pieces are, and what each
// costs by itself counts, the rows that it reads once more and its sums' meeting in LDS: then float32 has 32 columns and 8 waves of 2 steps, or with
// a gate and 17 to 31 tiles 16 and 8 waves of 4, bfloat16 32 columns and 4 waves of 4. Sums too short for the waves have 16 columns and 4 waves of 4.
// Where the lines lie: 156 calls (2 to 128 experts, 96 to 4,096 x 64 to 4,096, 1 to 100 tokens) with either product in each form; the choice is 1.2 to 2.3 %
// behind the fastest form of a product, none more than 14 % of a call (by tiles alone, for both products, 2.3 to 3.6 and 43; 4 experts of 128 x
// 1,632, 31 tokens 24.8 us, now 16.5). All launches of the experts with both products in one form, matrices from HBM,
// us (32 columns and 4 waves / 16 and 16 (bfloat16: 8) / float32: 16 and 8 / 16 and 4 / 32 and 8; C x F, experts, tiles):
//   float32, gated: 2,048 x 1,408, 16, 2 tiles 31.4 / 22.1 / 22.7 / 24.8 / 32.3, 8 61.8 / 51.8 / 52.5 / 53.7 / 60.6, 17 95.3 / 90.8 / 89.7 / 92.0 / 91.8;
//   2,048 x 768, 128, 8 39.6 / 41.7 / 42.0 / 40.5 / 38.9, 64 169 / 190 / 176 / 169 / 166; 1,024 x 512, 64, 4 19.1 / 16.4 / 16.5 / 15.7 / 20.0, 32 42.6 / 46.2 / 43.7
//   / 41.3 / 41.6, 62 57.5 / 76.5 / 63.3 / 54.3 / 58.8; 4,096 x 2,048, 8, 44 514 / 524 / 534 / 535 / 451
//   float32, plain: 2,048 x 1,408, 16, 2 25.0 / 18.5 / 19.1 / 20.7 / 24.5, 8 44.8 / 39.7 / 40.8 / 41.4 / 42.8, 16 55.0 / 54.8 / 55.6 / 55.6 / 52.3; 1,536 x 2,816,
//   16, 18 105 / 119 / 124 / 108 / 98; 2,048 x 768, 128, 64 123 / 151 / 147 / 126 / 118; 1,024 x 512, 64, 16 22.2 / 24.0 / 23.6 / 23.0 / 21.7, 62 44.5 / 68.4 / 59.0 /
//   46.4 / 44.2; 256 x 96, 8, 64 18.4 / 17.9 / 16.7 / 17.5 / 17.3
//   bfloat16, gated: 2,048 x 1,408, 16, 2 19.7 / 14.8, 8 31.8 / 28.7, 16 39.3 / 39.4; 2,048 x 768, 128, 32 56.7 / 60.3, 64 89 / 100
//   bfloat16, plain: 2,048 x 1,408, 16, 2 15.8 / 13.0, 8 24.1 / 24.1, 16 29.8 / 32.9; 768 x 256, 32, 8 12.7 / 10.9, 16 13.9 / 12.6, 32 15.3 / 15.3; 512 x 1,024, 4, 5 11.5 /
//   10.4; 1,536 x 2,816, 16, 8 33.2 / 34.7; 2,048 x 768, 128, 8 19.6 / 20.0
// tiles: of the launch; in_use: the most of them that can hold rows
template <typename T, int ACT, bool PLAN>
static void moe_few_product(const T* rows, const T* W, const T* W2, const int* tile_expert, void* out, int N, int K, float limit, int tiles, int in_use,
                            const MoePairs& pairs, hipStream_t stream) {
  auto run = [&](auto kernel, int nt, int waves) {
    kernel<<<dim3(tw_div_up(N, 16 * nt), tiles), waves * 64, 0, stream>>>(rows, K, W, W2, tile_expert, out, N, N, K, limit, pairs);
  };
#define TW_MOE_FEW(NT, WAVES, STEPS, AHEAD) run(moe_grouped_kernel<T, ACT, NT, true, 1, PLAN, WAVES, STEPS, AHEAD>, NT, WAVES)
  constexpr bool GLU = ACT == 1 || ACT == 3;
  const int pieces = in_use * tw_div_up(N, 16);                // of 16 columns
  if constexpr (sizeof(T) == 4 && GLU) {
    if (K < 448 || (in_use >= 32 && K < 1536)) TW_MOE_FEW(1, 4, 4, false);
    else if (in_use >= 32) TW_MOE_FEW(2, 8, 2, false);
    else if (in_use <= 16) TW_MOE_FEW(1, 16, 2, false);
    else TW_MOE_FEW(1, 8, 4, false);
  } else if constexpr (sizeof(T) == 4) {
    if (K < (ACT == 0 ? 160 : 256)) TW_MOE_FEW(1, 4, 4, false);
    else if (pieces <= 360 || (in_use < 16 && K > 1200)) TW_MOE_FEW(1, 16, 2, false);
    else TW_MOE_FEW(2, 8, 2, false);
  } else if constexpr (GLU) {
    if (K < 256) TW_MOE_FEW(1, 4, 4, false);
    else if (in_use <= 16) TW_MOE_FEW(1, 8, 2, true);
    else TW_MOE_FEW(2, 4, 4, false);
  } else {
    if (pieces <= (ACT == 0 ? 800 : 400)) TW_MOE_FEW(1, 8, 2, true);
    else TW_MOE_FEW(2, 4, 4, false);
  }
#undef TW_MOE_FEW
}

template <typename T, int ACT, bool PLAN>
static void moe_few_products(const T* rows, const T* first, const T* second, const T* down, const int* tile_expert, T* act, float* ys,
                             int C, int Cd, int Fd, float limit, int tiles, int in_use, const MoePairs& pairs, hipStream_t stream) {
  moe_few_product<T, ACT, PLAN>(rows, first, second, tile_expert, act, Fd, Cd, limit, tiles, in_use, pairs, stream);
  moe_few_product<T, 0, false>(act, down, nullptr, tile_expert, ys, C, Fd, 0.f, tiles, in_use, MoePairs{}, stream);
}

// Where moe_parts_kernel takes a float32 step of many rows: where the first product has 140 workgroups of 64 columns and 256 of K. (Fewer
// of either begin and end for longer than they multiply: 8 experts of 2,368 x 320, 848 tokens, 110 workgroups 96 -> 110 us; 16 of 160 x
// 1,440, 128 tokens 41 -> 49.) A tile has 128 columns where they make more than 320 workgroups: 64 for 16 experts of 2,048 x 1,408 without a
// gate, 128 tokens 148 -> 134 us, 1,000 tokens 232 -> 271.
static bool moe_parts_pay(int units, int C, int Fd) { return units * tw_div_up(Fd, 64) > 140 && C >= 256; }
template <int ACT>
static void moe_parts(const float* rows, const float* W, const float* W2, const int* tile_expert, float* out, long ldo, int N, int K, float limit,
                      int units, hipStream_t stream) {
  if constexpr (ACT == 1 || ACT == 3)
    moe_parts_kernel<ACT, 2><<<dim3(units, tw_div_up(N, 64)), 256, 0, stream>>>(rows, W, W2, tile_expert, out, ldo, N, K, limit);
  else if (units * tw_div_up(N, 128) > 320)
    moe_parts_kernel<ACT, 2><<<dim3(units, tw_div_up(N, 128)), 256, 0, stream>>>(rows, W, W2, tile_expert, out, ldo, N, K, limit);
  else
    moe_parts_kernel<ACT, 1><<<dim3(units, tw_div_up(N, 64)), 256, 0, stream>>>(rows, W, W2, tile_expert, out, ldo, N, K, limit);
}

// The two grouped products of a step: kind 0 gated with the limited swish, 1 up alone with gelu, 2 gated with SiLU, 3 up alone
// with the square of relu.
template <typename T, int ACT>
static void moe_products(const T* xs, const T* gate, const T* up, const T* down, const int* tile_expert, T* act, float* ys, int C,
                         int Cd, int Fd, float limit, int tiles, bool wide, long items, int X, hipStream_t stream) {
  constexpr bool PLAIN = ACT == 2 || ACT == 4;
  const T* first = PLAIN ? up : gate;
  const T* second = PLAIN ? nullptr : up;
  if constexpr (sizeof(T) == 4) {
    if (tiles > TW_MOE_SPLITK_TILES && wide && moe_parts_pay(tiles / TW_MOE_WIDE, C, Fd)) {
      moe_parts<ACT>(xs, first, second, tile_expert, act, Fd, Fd, Cd, limit, tiles / TW_MOE_WIDE, stream);
      moe_parts<0>(act, down, nullptr, tile_expert, ys, C, C, Fd, 0.f, tiles / TW_MOE_WIDE, stream);
      return;
    }
  }
  if (tiles <= TW_MOE_SPLITK_TILES) {
    // few rows: most tiles hold one or two rows and each streams its expert's matrices once; the waves then split K
    moe_few_products<T, ACT, false>(xs, first, second, down, tile_expert, act, ys, C, Cd, Fd, limit, tiles,
                                    items < tiles ? (int)items : tiles, MoePairs{}, stream);
  } else if (wide && moe_splits_k(sizeof(T) == 4, tiles / TW_MOE_WIDE, items, X, C, Cd, Fd, !PLAIN)) {
    moe_grouped_kernel<T, ACT, 2, true, TW_MOE_WIDE><<<dim3(tiles / TW_MOE_WIDE, tw_div_up(Fd, 16 * 2)), 256, 0, stream>>>(
        xs, Cd, first, second, tile_expert, act, Fd, Fd, Cd, limit);
    moe_grouped_kernel<T, 0, 2, true, TW_MOE_WIDE><<<dim3(tiles / TW_MOE_WIDE, tw_div_up(C, 16 * 2)), 256, 0, stream>>>(
        act, Fd, down, nullptr, tile_expert, ys, C, C, Fd, 0.f);
  } else if (wide) {
    moe_grouped_kernel<T, ACT, 2, false, TW_MOE_WIDE><<<dim3(tiles / TW_MOE_WIDE, tw_div_up(Fd, 4 * 16 * 2)), 256, 0, stream>>>(
        xs, Cd, first, second, tile_expert, act, Fd, Fd, Cd, limit);
    moe_grouped_kernel<T, 0, 2, false, TW_MOE_WIDE><<<dim3(tiles / TW_MOE_WIDE, tw_div_up(C, 4 * 16 * 2)), 256, 0, stream>>>(
        act, Fd, down, nullptr, tile_expert, ys, C, C, Fd, 0.f);
  } else {
    moe_grouped_kernel<T, ACT, 2><<<dim3(tiles, tw_div_up(Fd, 4 * 16 * 2)), 256, 0, stream>>>(
        xs, Cd, first, second, tile_expert, act, Fd, Fd, Cd, limit);
    moe_grouped_kernel<T, 0, 4><<<dim3(tiles, tw_div_up(C, 4 * 16 * 4)), 256, 0, stream>>>(
        act, Fd, down, nullptr, tile_expert, ys, C, C, Fd, 0.f);
  }
}

struct MoeStep {
  const void *h, *gate, *up, *down;
  long ld_h, ld_x;
  const float* weights;
  const int *ids, *src_item, *tile_expert, *pos;
  void *xs, *act;
  float *ys, *x;
  const float* more;
  int n, top, X, C, Cd, Fd, capacity, kind, accumulate, more_splits;
  float limit;
  bool wide, few;
  const float* norm_weight;
  void* normed;
  float norm_eps;
};

template <typename T, int ACT>
static void moe_products_few(const MoeStep& s, hipStream_t stream) {
  constexpr bool PLAIN = ACT == 2 || ACT == 4;
  // (every tile is opened by a pair of its own, and the tiles in use never exceed what a plan could need)
  const int tiles = s.n * s.top < s.capacity / TW_MOE_TILE ? s.n * s.top : s.capacity / TW_MOE_TILE;
  const MoePairs pairs{s.ids, s.n * s.top, s.top, s.X, s.ld_h, const_cast<int*>(s.tile_expert), const_cast<int*>(s.pos)};
  moe_few_products<T, ACT, true>((const T*)s.h, (const T*)(PLAIN ? s.up : s.gate), (const T*)(PLAIN ? nullptr : s.up), (const T*)s.down,
                                 s.tile_expert, (T*)s.act, s.ys, s.C, s.Cd, s.Fd, s.limit, tiles, tiles, pairs, stream);
}

// Can the first product find its tiles and rows itself? (few pairs, rows of h that are whole fragments)
static bool moe_few(int dtype, const void* h, long ld_h, int n, int top, int C, int Cd, int kind) {
  const int epf = dtype == TW_DTYPE_BF16 ? 8 : 4;
  return kind != 0 && n * top <= 64 && C == Cd && C % (4 * epf) == 0 && ld_h % epf == 0 && (uintptr_t)h % 16 == 0;
}

template <typename T>
static bool moe_combine_wide(const MoeStep& s) {
  return s.C % 4 == 0 && s.ld_x % 4 == 0 && s.ld_h % 4 == 0 && ((((uintptr_t)s.x | (uintptr_t)s.ys | (uintptr_t)s.more) & 15) == 0) && ((uintptr_t)s.h & (4 * sizeof(T) - 1)) == 0;
}

template <typename T>
static void moe_run(const MoeStep& s, hipStream_t stream) {
  if (s.few) {
    if (s.kind == 1) moe_products_few<T, 2>(s, stream);
    else if (s.kind == 2) moe_products_few<T, 3>(s, stream);
    else moe_products_few<T, 4>(s, stream);
  } else {
    const int pieces = tw_div_up(s.Cd, 16 * Elem<T>::kPerFrag);
    moe_gather_kernel<T><<<dim3(s.capacity / TW_MOE_TILE, pieces < 4 ? pieces : 4), 256, 0, stream>>>((const T*)s.h, s.ld_h, s.kind == 0 ? s.weights : nullptr, s.src_item,
                                                         s.tile_expert, (T*)s.xs, s.C, s.Cd, s.top);
    const int tiles = s.capacity / TW_MOE_TILE;
#define TW_MOE_PRODUCTS(ACT)                                                                                            \
    moe_products<T, ACT>((const T*)s.xs, (const T*)s.gate, (const T*)s.up, (const T*)s.down, s.tile_expert, (T*)s.act,    \
                         s.ys, s.C, s.Cd, s.Fd, s.limit, tiles, s.wide, (long)s.n * s.top, s.X, stream)
    if (s.kind == 0) TW_MOE_PRODUCTS(1);
    else if (s.kind == 1) TW_MOE_PRODUCTS(2);
    else if (s.kind == 2) TW_MOE_PRODUCTS(3);
    else TW_MOE_PRODUCTS(4);
#undef TW_MOE_PRODUCTS
  }
  if (!s.x) return;                                  // (whoever reads ys and pos adds them up)
  const MoeCombineArgs a{s.x, s.ld_x, s.ys, s.C, s.pos, s.kind == 0 ? nullptr : s.weights, s.more, (size_t)s.n * s.C, s.h, s.ld_h,
                         s.C, s.top, s.more_splits, s.accumulate};
  const dim3 grid(s.n, tw_div_up(s.C, 1024));
  if (s.norm_weight) moe_combine_norm_kernel<T><<<s.n, tw_div_up(s.C, 256) * 64, 0, stream>>>(a, s.norm_weight, s.norm_eps, (T*)s.normed);
  else if (moe_combine_wide<T>(s)) moe_combine_kernel<T, true><<<grid, 256, 0, stream>>>(a);
  else moe_combine_kernel<T, false><<<grid, 256, 0, stream>>>(a);
}

// h [n][C] (compute type) -> x [n][C] float32 += the routed experts' results. ids, weights [n * top] come from
// tw_moe_route (ids of X and above, where the weights multiply outputs: experts that return h). Scratch: pos [n * top],
// src_item [capacity], tile_expert [capacity / 16] (int32), xs [capacity][Cd], act [capacity][Fd] (compute type),
// ys [capacity][C] (float32), capacity = tw_moe_capacity(n * top, X). x null: the experts' rows stay in ys, unweighted, pair i's
// in row pos[i] (kinds whose weights multiply outputs). norm_weight (or null; with accumulate, aligned rows of up to 4,096 elements): the new rows
// of x behind an RMS norm as well, normed [n][C] in the compute type (h, if it is contiguous, will do).
extern "C" int tw_moe_experts(int dtype, const void* h, long ld_h, const int* ids, const float* weights, int n, int top, int X,
                              const void* gate, const void* up, const void* down, int C, int Cd, int Fd, float limit,
                              int* pos, int* src_item, int* tile_expert, void* xs, void* act, float* ys, int capacity,
                              float* x, long ld_x, int kind, int accumulate, const float* more, int more_splits,
                              const float* norm_weight, float norm_eps, void* normed, hipStream_t stream) {
  TW_REQUIRE(h && ids && weights && up && down && pos && src_item && tile_expert && xs && act && ys && (x || (kind != 0 && !more)));
  TW_REQUIRE(((kind == 0 || kind == 2) && gate) || kind == 1 || kind == 3);
  TW_REQUIRE(more == nullptr || more_splits > 0);
  if (kind == 1 || kind == 3) gate = up;            // (never read: the alignment test below wants a pointer)
  TW_REQUIRE(n >= 0 && top > 0 && C > 0 && Cd >= C && Cd % 32 == 0 && Fd > 0 && Fd % 32 == 0 && ld_h >= C && (!x || ld_x >= C));
  TW_REQUIRE((uintptr_t)xs % 16 == 0 && (uintptr_t)act % 16 == 0 && (uintptr_t)gate % 16 == 0 && (uintptr_t)up % 16 == 0 &&
             (uintptr_t)down % 16 == 0);
  TW_REQUIRE(dtype == TW_DTYPE_BF16 || dtype == TW_DTYPE_F32);
  if (n == 0) return 0;
  const bool few = moe_few(dtype, h, ld_h, n, top, C, Cd, kind);
  if (!few) {
    const int code = tw_moe_plan(ids, n * top, X, pos, src_item, tile_expert, capacity, stream);
    if (code) return code;
  }
  const bool wide = moe_unit((long)n * top, X) == TW_MOE_TILE * TW_MOE_WIDE;
  TW_REQUIRE(!wide || capacity % (TW_MOE_TILE * TW_MOE_WIDE) == 0);
  const MoeStep s{h, gate, up, down, ld_h, ld_x, weights, ids, src_item, tile_expert, pos, xs, act, ys, x, more,
                  n, top, X, C, Cd, Fd, capacity, kind, accumulate, more_splits, limit, wide, few, norm_weight, normed, norm_eps};
  TW_REQUIRE(norm_weight == nullptr || (x && accumulate && normed && norm_eps > 0.f && C <= 4096 && (uintptr_t)norm_weight % 16 == 0 &&
                                        (dtype == TW_DTYPE_BF16 ? moe_combine_wide<bf16_t>(s) : moe_combine_wide<float>(s))));
  if (dtype == TW_DTYPE_BF16) moe_run<bf16_t>(s, stream);
  else moe_run<float>(s, stream);
  return TW_LAUNCH_RESULT();
}
