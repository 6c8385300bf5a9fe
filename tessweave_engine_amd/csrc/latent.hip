// Attention over a cached LATENT: every token leaves one normed vector c (L elements) and one rotated key part
// kr (R elements) that all heads share; head a's key is [W_uk,a c | kr] and its value W_uv,a c. The products with
// W_uk and W_uv are moved to the query side and the output side:
//
//   score_a(i, j) = (W_uk,a^T q_plain,a(i)) . c_j + q_turned,a(i) . kr_j         out_a(i) = W_uv,a sum_j p_a(i, j) c_j
//
// so the attention itself runs over ONE key/value head whose key row is [c | kr] and whose value is c, and only
// c and kr are ever stored. Here: the kernel that finishes a token's projections (norm of c, rotation of kr and
// of the queries' rotated parts, cache write), and the per-head matrix product both sides use.
#include <algorithm>

#include "tw_common.h"

// One rotated pair, products and sums spelled out (a*b - c*d left to the compiler becomes one fused form or the other).
__device__ __forceinline__ void lt_rotate_pair(float lo, float hi, float c, float s, float& out_lo, float& out_hi) {
  out_lo = __fmaf_rn(lo, c, -__fmul_rn(hi, s));
  out_hi = __fmaf_rn(hi, c, __fmul_rn(lo, s));
}

struct LatentFinishArgs {
  const void* proj; long ld;        // a token's projections: the heads' rotated query parts at q_col + a * Rp,
  int q_col, c_col, kr_col;         // the raw latent at c_col (L elements), the raw shared key part at kr_col
  const float* cos_t; const float* sin_t;    // [n][rot / 2]
  const float* norm_w;              // [L]
  void* q_out; long ld_q;           // [n][H][Lp + Rp]: this kernel fills columns Lp .. Lp + Rp of every head
  void* q_full; long ld_full;       // or null. [n][H][hd]: head a = [its D unrotated elements | its rotated part | zeros],
  int D, Dp, hd, full_from;         // for rows from full_from on (queries against keys expanded per head)
  void* keys; void* values;         // keys [pages][1][P][Lp + Rp], values [pages][1][Lp][P]; null: nothing is stored
  const int* slots;
  int H, L, Lp, Rp, rot, P;
  float eps;
};

template <typename T>
__device__ __forceinline__ void latent_finish_token(const LatentFinishArgs& a, int n, float* lds) {
  const T* row = (const T*)a.proj + (size_t)n * a.ld;
  const int half = a.rot / 2;
  const float* cs = a.cos_t + (size_t)n * half;
  const float* sn = a.sin_t + (size_t)n * half;
  const int K = a.Lp + a.Rp;
  // the heads' rotated query parts
  T* q = (T*)a.q_out + (size_t)n * a.ld_q;
  for (int i = threadIdx.x; i < a.H * a.Rp; i += blockDim.x) {
    const int head = i / a.Rp, d = i % a.Rp;
    const T* src = row + a.q_col + head * a.Rp;
    float v;
    if (d < half) {
      float other;
      lt_rotate_pair(tw_to_float(src[d]), tw_to_float(src[d + half]), cs[d], sn[d], v, other);
    } else if (d < a.rot) {
      float other;
      lt_rotate_pair(tw_to_float(src[d - half]), tw_to_float(src[d]), cs[d - half], sn[d - half], other, v);
    } else {
      v = tw_to_float(src[d]);
    }
    q[(size_t)head * K + a.Lp + d] = tw_from_float<T>(v);
  }
  if (a.q_full && n >= a.full_from) {
    __syncthreads();                                                          // the rotated parts above, written by other threads
    T* qf = (T*)a.q_full + (size_t)n * a.ld_full;
    for (int i = threadIdx.x; i < a.H * a.hd; i += blockDim.x) {
      const int head = i / a.hd, d = i % a.hd;
      T v = tw_from_float<T>(0.f);
      if (d < a.D) v = row[head * a.Dp + d];                                   // (the unrotated parts lie first in the row)
      else if (d < a.D + a.Rp) v = q[(size_t)head * K + a.Lp + d - a.D];     // (turned or not; zeros behind the part's own size)
      qf[i] = v;
    }
  }
  if (!a.keys) return;
  const int slot = a.slots[n];
  // the latent's norm (every thread takes part in the sum, stored or not)
  float ss = 0.f;
  for (int i = threadIdx.x; i < a.L; i += blockDim.x) {
    const float v = tw_to_float(row[a.c_col + i]);
    ss = __fmaf_rn(v, v, ss);
  }
  const float total = tw_block_sum(ss, lds);
  if (slot < 0) return;
  const float rinv = 1.f / sqrtf(total / (float)a.L + a.eps);
  const int page = slot / a.P, at = slot % a.P;
  T* key = (T*)a.keys + ((size_t)page * a.P + at) * K;
  T* val = (T*)a.values + (size_t)page * a.Lp * a.P + at;
  for (int i = threadIdx.x; i < a.Lp; i += blockDim.x) {
    const T c = i < a.L ? tw_from_float<T>(tw_to_float(row[a.c_col + i]) * rinv * a.norm_w[i]) : tw_from_float<T>(0.f);
    key[i] = c;
    val[(size_t)i * a.P] = c;
  }
  for (int d = threadIdx.x; d < a.Rp; d += blockDim.x) {
    const T* src = row + a.kr_col;
    float v;
    if (d < half) {
      float other;
      lt_rotate_pair(tw_to_float(src[d]), tw_to_float(src[d + half]), cs[d], sn[d], v, other);
    } else if (d < a.rot) {
      float other;
      lt_rotate_pair(tw_to_float(src[d - half]), tw_to_float(src[d]), cs[d - half], sn[d - half], other, v);
    } else {
      v = tw_to_float(src[d]);                   // what the encoding does not turn passes (the padding behind it is zeros)
    }
    key[a.Lp + d] = tw_from_float<T>(v);
  }
}

// ---- one small matrix per head: out[n][a * so + o] = sum_i x[n][a * sx + i] * w[a][o][i] ------------------------
// x and out hold the heads side by side, sx and so elements apart; w [heads][No][Ni] row-major. A wave takes 16
// rows and 16 output columns of one head; the weights are the A operand, so a lane ends with four consecutive
// output columns of one row. Sums are float32, rounded once to the compute type. Bound by the trips to memory in a row: the
// operands of 8 k-steps are requested together (64 columns a wave, each k-step waiting for its own: 7.6 us of a decode step's
// layer for 16 heads of 128 x 192, 4.4 for 192 x 64).
template <typename T>
struct HeadLinear {
  const T* x; long ldx; int sx;
  const T* w;
  T* out; long ldo; int so;
  int n, heads, Ni, No;
  __host__ __device__ int units() const { return heads * ((No + 15) / 16); }       // of 16 rows each
};

template <typename T>
__device__ __forceinline__ void head_linear_unit(const HeadLinear<T>& a, int unit, int row_tile) {
  typedef typename Elem<T>::Frag Frag;
  constexpr int EPF = Elem<T>::kPerFrag, U = 8;
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int col_tiles = (a.No + 15) / 16;
  const int head = unit / col_tiles, col = unit % col_tiles * 16;
  const int row = row_tile * 16 + r;
  const int chunks = a.Ni / EPF, steps = (chunks + 3) / 4;
  const T* x_row = a.x + (size_t)min(row, a.n - 1) * a.ldx + (size_t)head * a.sx;      // (rows and columns past the last: never stored)
  const T* w_row = a.w + ((size_t)head * a.No + min(col + r, a.No - 1)) * a.Ni;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int st0 = 0; st0 < steps; st0 += U) {
    Frag xf[U], wf[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int chunk = min((st0 + u) * 4 + g, chunks - 1);
      xf[u] = tw_load_frag(x_row + chunk * EPF);
      wf[u] = tw_load_frag(w_row + chunk * EPF);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (st0 + u < steps) {
        const bool in = (st0 + u) * 4 + g < chunks;
        tw_mma16(acc, in ? wf[u] : Elem<T>::zero(), in ? xf[u] : Elem<T>::zero());      // D[output 4g + e][row r]
      }
  }
  const int o = col + 4 * g;
  if (row < a.n && o < a.No) {
    T* dst = a.out + (size_t)row * a.ldo + (size_t)head * a.so + o;
#pragma unroll
    for (int e = 0; e < 4; ++e) dst[e] = tw_from_float<T>(acc[e]);
  }
}

// Workgroups 0 .. n - 1 finish a token each; those behind them form the query side's products W_uk,a^T q_plain,a of the first
// absorb.n rows, which read and write nothing the others write: one launch instead of two.
template <typename T>
__global__ __launch_bounds__(256) void latent_finish_kernel(LatentFinishArgs a, HeadLinear<T> absorb, int n) {
  __shared__ float lds[16];
  if ((int)blockIdx.x < n) {
    latent_finish_token<T>(a, blockIdx.x, lds);
    return;
  }
  const int unit = ((int)blockIdx.x - n) * 4 + (threadIdx.x >> 6), per_tile = absorb.units();
  const int row_tile = unit / per_tile;
  if (row_tile * 16 < absorb.n) head_linear_unit(absorb, unit - row_tile * per_tile, row_tile);
}

extern "C" int tw_latent_finish(int dtype, const void* proj, long ld, int q_col, int c_col, int kr_col,
                                const float* cos_t, const float* sin_t, const float* norm_w, void* q_out, long ld_q,
                                void* q_full, long ld_full, int D, int Dp, int hd, int full_from,
                                void* keys, void* values, const int* slots, int n, int H, int L, int Lp, int Rp, int rot,
                                int page_size, float eps, const void* absorb, int absorb_rows, hipStream_t stream) {
  TW_REQUIRE(proj && cos_t && sin_t && q_out && n >= 0 && H > 0 && Rp > 0 && rot > 0 && rot % 2 == 0 && rot <= Rp);
  if (q_full) TW_REQUIRE(D > 0 && Dp >= D && hd >= D + rot && ld_full >= (long)H * hd && full_from >= 0 && q_col >= H * Dp);
  TW_REQUIRE(q_col >= 0 && ld >= q_col + (long)H * Rp && ld_q >= (long)H * (Lp + Rp) && Lp >= 0);
  if (keys) {
    TW_REQUIRE(values && slots && norm_w && L > 0 && Lp >= L && page_size > 0 && eps > 0.f);
    TW_REQUIRE(c_col >= 0 && kr_col >= 0 && ld >= c_col + (long)L && ld >= kr_col + (long)Rp);
  }
  if (n == 0) return 0;
  LatentFinishArgs a{proj, ld, q_col, c_col, kr_col, cos_t, sin_t, norm_w, q_out, ld_q, q_full, ld_full, D, Dp, hd, full_from,
                     keys, values, slots, H, L, Lp, Rp, rot, page_size, eps};
  if (absorb) {            // [H][Lp][Dp]: the first absorb_rows rows' latent queries too, into columns 0 .. Lp of every head of q_out
    const int epf = dtype == TW_DTYPE_BF16 ? 8 : 4;
    TW_REQUIRE(absorb_rows >= 0 && absorb_rows <= n && Dp > 0 && Dp % epf == 0 && Lp % 4 == 0 && ld % epf == 0 && q_col >= H * Dp);
    TW_REQUIRE((uintptr_t)proj % 16 == 0 && (uintptr_t)absorb % 16 == 0);
  }
  const int rows = absorb ? absorb_rows : 0;
#define TW_LATENT_FINISH(T)                                                                                                    \
  do {                                                                                                                         \
    const HeadLinear<T> hl{(const T*)proj, ld, Dp, (const T*)absorb, (T*)q_out, ld_q, Lp + Rp, rows, H, Dp, Lp};                \
    const int groups = rows ? tw_div_up((long)hl.units() * tw_div_up(rows, 16), 4) : 0;                                         \
    latent_finish_kernel<T><<<n + groups, 256, 0, stream>>>(a, hl, n);                                                         \
  } while (0)
  if (dtype == TW_DTYPE_BF16) TW_LATENT_FINISH(bf16_t);
  else if (dtype == TW_DTYPE_F32) TW_LATENT_FINISH(float);
  else return TW_ERR_BAD_ARGUMENT;
#undef TW_LATENT_FINISH
  return TW_LAUNCH_RESULT();
}

// (the products alone: no token is finished)
extern "C" int tw_head_linear(int dtype, const void* x, long ldx, int sx, const void* w, void* out, long ldo, int so,
                              int n, int heads, int Ni, int No, hipStream_t stream) {
  const int epf = dtype == TW_DTYPE_BF16 ? 8 : 4;
  TW_REQUIRE(x && w && out && n >= 0 && heads > 0 && Ni > 0 && No > 0);
  TW_REQUIRE(dtype == TW_DTYPE_BF16 || dtype == TW_DTYPE_F32);
  TW_REQUIRE(Ni % epf == 0 && No % 4 == 0 && ldx % epf == 0 && sx % epf == 0 && sx >= 0 && so >= No);
  TW_REQUIRE(ldx >= (long)(heads - 1) * sx + Ni && ldo >= (long)(heads - 1) * so + No);
  TW_REQUIRE((uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0);
  if (n == 0) return 0;
#define TW_HEAD_LINEAR(T)                                                                                                      \
  do {                                                                                                                         \
    const HeadLinear<T> hl{(const T*)x, ldx, sx, (const T*)w, (T*)out, ldo, so, n, heads, Ni, No};                              \
    latent_finish_kernel<T><<<tw_div_up((long)hl.units() * tw_div_up(n, 16), 4), 256, 0, stream>>>(LatentFinishArgs{}, hl, 0);    \
  } while (0)
  if (dtype == TW_DTYPE_BF16) TW_HEAD_LINEAR(bf16_t);
  else TW_HEAD_LINEAR(float);
#undef TW_HEAD_LINEAR
  return TW_LAUNCH_RESULT();
}

// ---- prompt portions: keys and values expanded per head for this step ------------------------------------------------
// Against many query rows it is cheaper to expand the cached latents once (k_a = W_uk,a c, v_a = W_uv,a c for every
// cached token of the sequences that bring a portion) and to run ordinary attention with one key/value head per
// query head than to carry the latent's size through every score. Two kernels around one matrix product:
//
//   latent_gather:        the key rows [c | kr] of sequences seq0 .. from their pages into rows of their own, sequence
//                         after sequence, each starting at a multiple of the page size (row = page of its own * P + place),
//                         and the block table of those pages
//   (product)             up[row] = [W_uk ; W_uv] c[row]
//   latent_expand_store:  keys [page][a][place][hd] = [up k-part of head a | kr | zeros], values [page][a][hd][place]
//                         = [up v-part | zeros]: the layout the attention kernels read
struct LatentGatherArgs {
  const void* keys;                  // [pages][1][P][K]
  const int* block_table; int table_stride;
  const int* kv_len; const int* kv_page_start;      // kv_page_start[s]: pages of their own before sequence s (all sequences of the step)
  void* rows;                        // [own pages * P][K]
  int* own_table; int own_stride;    // [>= seq0 + n_seqs][own_stride]
  int seq0, n_seqs, P, K;
};

template <typename T>
__global__ __launch_bounds__(256) void latent_gather_kernel(LatentGatherArgs a) {
  const int base = a.kv_page_start[a.seq0];
  const int pg = blockIdx.x;                                   // page of its own, counted from seq0's first
  int lo = a.seq0, hi = a.seq0 + a.n_seqs - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (a.kv_page_start[mid] - base <= pg) lo = mid; else hi = mid - 1;
  }
  const int s = lo, b = pg - (a.kv_page_start[s] - base);
  if (pg >= a.kv_page_start[a.seq0 + a.n_seqs] - base) return;
  if (threadIdx.x == 0) a.own_table[(size_t)s * a.own_stride + b] = pg;
  const int phys = a.block_table[(size_t)s * a.table_stride + b];
  const int live = min(a.P, a.kv_len[s] - b * a.P);
  const T* src = (const T*)a.keys + (size_t)(phys < 0 ? 0 : phys) * a.P * a.K;
  T* dst = (T*)a.rows + (size_t)pg * a.P * a.K;
  for (int i = threadIdx.x; i < a.P * a.K; i += blockDim.x)
    dst[i] = (phys >= 0 && i / a.K < live) ? src[i] : tw_from_float<T>(0.f);
}

extern "C" int tw_latent_gather(int dtype, const void* keys, const int* block_table, int table_stride, const int* kv_len,
                                const int* kv_page_start, void* rows, int* own_table, int own_stride, int seq0, int n_seqs,
                                int own_pages, int page_size, int K, hipStream_t stream) {
  TW_REQUIRE(keys && block_table && kv_len && kv_page_start && rows && own_table && seq0 >= 0 && n_seqs >= 0 && own_pages >= 0);
  TW_REQUIRE(page_size > 0 && K > 0 && own_stride > 0);
  if (n_seqs == 0 || own_pages == 0) return 0;
  LatentGatherArgs a{keys, block_table, table_stride, kv_len, kv_page_start, rows, own_table, own_stride, seq0, n_seqs, page_size, K};
  if (dtype == TW_DTYPE_BF16) latent_gather_kernel<bf16_t><<<own_pages, 256, 0, stream>>>(a);
  else if (dtype == TW_DTYPE_F32) latent_gather_kernel<float><<<own_pages, 256, 0, stream>>>(a);
  else return TW_ERR_BAD_ARGUMENT;
  return TW_LAUNCH_RESULT();
}

// One workgroup a page: up [rows][H * D + H * E] (the heads' key parts, then their value parts), kr at rows[row][Lp ..].
// VEC (bfloat16, sizes and strides that are multiples of 8): 16 bytes a thread. A key row is copied in groups of 8
// elements; for the transposed values a thread gathers one element of 8 consecutive places (neighbouring threads
// read neighbouring elements of one row) and stores them as one group.
template <typename T, bool VEC>
__global__ __launch_bounds__(256) void latent_expand_store_kernel(const T* __restrict__ up, long ld_up, const T* __restrict__ rows,
                                                                  int K, int Lp, T* __restrict__ keys, T* __restrict__ values,
                                                                  int H, int D, int R, int E, int hd, int P) {
  const int pg = blockIdx.x;
  T* kp = keys + (size_t)pg * H * P * hd;
  T* vp = values + (size_t)pg * H * hd * P;
  if (VEC) {
    const int groups = hd / 8;
    for (int i = threadIdx.x; i < H * P * groups; i += blockDim.x) {
      const int d = (i % groups) * 8, t = (i / groups) % P, a = i / (groups * P);
      const size_t row = (size_t)pg * P + t;
      u32x4 v = {0u, 0u, 0u, 0u};
      if (d < D) v = *reinterpret_cast<const u32x4*>(up + row * ld_up + a * D + d);
      else if (d < D + R) v = *reinterpret_cast<const u32x4*>(rows + row * K + Lp + d - D);
      *reinterpret_cast<u32x4*>(kp + ((size_t)a * P + t) * hd + d) = v;
    }
    const int tgs = P / 8;
    for (int i = threadIdx.x; i < H * tgs * hd; i += blockDim.x) {
      const int e = i % hd, tg = (i / hd) % tgs, a = i / (hd * tgs);
      bf16x8 v;
#pragma unroll
      for (int x = 0; x < 8; ++x) {
        const size_t row = (size_t)pg * P + tg * 8 + x;
        v[x] = e < E ? up[row * ld_up + (size_t)H * D + a * E + e] : (bf16_t)0.f;
      }
      *reinterpret_cast<bf16x8*>(vp + ((size_t)a * hd + e) * P + tg * 8) = v;
    }
    return;
  }
  for (int i = threadIdx.x; i < H * P * hd; i += blockDim.x) {
    const int d = i % hd, t = (i / hd) % P, a = i / (hd * P);
    const size_t row = (size_t)pg * P + t;
    T v = tw_from_float<T>(0.f);
    if (d < D) v = up[row * ld_up + a * D + d];
    else if (d < D + R) v = rows[row * K + Lp + d - D];
    kp[i] = v;
  }
  for (int i = threadIdx.x; i < H * hd * P; i += blockDim.x) {
    const int t = i % P, e = (i / P) % hd, a = i / (P * hd);
    const size_t row = (size_t)pg * P + t;
    vp[i] = e < E ? up[row * ld_up + (size_t)H * D + a * E + e] : tw_from_float<T>(0.f);
  }
}

extern "C" int tw_latent_expand_store(int dtype, const void* up, long ld_up, const void* rows, int K, int Lp, void* keys,
                                      void* values, int own_pages, int H, int D, int R, int E, int hd, int page_size,
                                      hipStream_t stream) {
  TW_REQUIRE(up && rows && keys && values && own_pages >= 0 && H > 0 && D > 0 && R >= 0 && E > 0 && page_size > 0);
  TW_REQUIRE(hd >= D + R && hd >= E && ld_up >= (long)H * (D + E) && K >= Lp + R);
  if (own_pages == 0) return 0;
  const bool vec = dtype == TW_DTYPE_BF16 && D % 8 == 0 && R % 8 == 0 && E % 8 == 0 && hd % 8 == 0 && page_size % 8 == 0 &&
                   ld_up % 8 == 0 && K % 8 == 0 && Lp % 8 == 0 && (uintptr_t)up % 16 == 0 && (uintptr_t)rows % 16 == 0 &&
                   (uintptr_t)keys % 16 == 0 && (uintptr_t)values % 16 == 0;
  if (vec)
    latent_expand_store_kernel<bf16_t, true><<<own_pages, 256, 0, stream>>>((const bf16_t*)up, ld_up, (const bf16_t*)rows, K, Lp,
                                                                            (bf16_t*)keys, (bf16_t*)values, H, D, R, E, hd, page_size);
  else if (dtype == TW_DTYPE_BF16)
    latent_expand_store_kernel<bf16_t, false><<<own_pages, 256, 0, stream>>>((const bf16_t*)up, ld_up, (const bf16_t*)rows, K, Lp,
                                                                             (bf16_t*)keys, (bf16_t*)values, H, D, R, E, hd, page_size);
  else if (dtype == TW_DTYPE_F32)
    latent_expand_store_kernel<float, false><<<own_pages, 256, 0, stream>>>((const float*)up, ld_up, (const float*)rows, K, Lp,
                                                                            (float*)keys, (float*)values, H, D, R, E, hd, page_size);
  else return TW_ERR_BAD_ARGUMENT;
  return TW_LAUNCH_RESULT();
}

// ---- one-token sequences: all heads of a sequence against the one cached head ------------------------------------------
// The query heads are the 16 columns of the matrix unit's tile (a launch has one workgroup row per 16 heads): per 16
// keys a wave forms S^T = K Q^T (keys down, heads across), so every head's probabilities leave the product in the
// layout the next one, O^T += V^T P^T, wants as its operand, and a key row is read once for 16 heads. Values are the
// first Lp elements of the key rows, kept a second time transposed inside a page ([Lp][P]) so that four consecutive
// keys of one element are one 8-byte load. A sequence's keys are cut into `splits` ranges for separate workgroups,
// whose waves take the range's tiles in turn; waves are combined through LDS, ranges by latent_leave_kernel.
//
//   part [seq][head tile][split][16][Lp + 4]: output sums relative to the range's maximum, that maximum, the sum
struct LatentDecodeArgs {
  const void* q; long ldq;            // head a of sequence s at q + row(s) * ldq + a * K
  const void* keys; const void* values;
  const int* block_table; int table_stride;
  const int* q_start; const int* kv_len;
  float* part;
  float scale;
  int H, K, Lp, P, splits;
  int page_shift;                     // log2(P) if P is a power of two, else -1
  const float* sink;                  // [H] or null: exp(sink_a) more in head a's denominator (no key, no value, not scaled)
};

template <typename T> __device__ __forceinline__ float lt_exp(float v);
template <> __device__ __forceinline__ float lt_exp<float>(float v) { return expf(v); }
template <> __device__ __forceinline__ float lt_exp<bf16_t>(float v) { return __expf(v); }

template <typename T> struct LtQuad;
template <> struct LtQuad<float> { typedef f32x4 Type; };
template <> struct LtQuad<bf16_t> { typedef bf16x4 Type; };

// TILES > 0: latents of 16 TILES elements, key rows of up to 64 more (WHOLE: of 64 more), pages of a power of two and at least 16: loops
// have no branches, and a key tile's page and addresses are the whole wave's (scalar). 0: sizes known at run time. With what
// follows in latent_leave_kernel, in a chain of such calls (us, 0 / TILES; bfloat16, then float32): latents of 64 with 32 rotated, 8 requests
// of 190 keys 10.3 / 8.6, 12.2 / 10.9, 64 of 2,000 19.0 / 16.2, 36.2 / 26.5; 128 with 64 11.5 / 9.9, 14.9 / 13.5 and 29.4 / 25.5, 59.7 / 43.9; 192 with 64 12.5 / 11.0, 18.3 / 17.1 and 37.8 / 35.2, 79.9 / 59.9;
// 224 with 32 12.7 / 11.2, 20.0 / 19.6 and 39.7 / 36.5, 83.0 / 80.7.
template <typename T, int TILES, bool WHOLE = false>
__global__ __launch_bounds__(256, TILES ? 2 : 1) void latent_decode_kernel(LatentDecodeArgs a) {
  typedef typename Elem<T>::Frag Frag;
  typedef typename LtQuad<T>::Type Quad;
  constexpr int EPF = Elem<T>::kPerFrag;
  constexpr int STEP = 4 * EPF;                 // key elements one product consumes
  constexpr bool SIZED = TILES > 0;
  constexpr int KC_MAX = ((SIZED && 16 * TILES + 64 < 256 ? 16 * TILES + 64 : 256) + STEP - 1) / STEP;
  constexpr int KC_SURE = WHOLE ? KC_MAX : SIZED ? 16 * TILES / STEP : 0;       // products whose elements are all there, whatever K is
  constexpr int LT_MAX = SIZED ? TILES : 15;    // Lp <= 240
  extern __shared__ float ld_lds[];
  const int s = blockIdx.x, split = blockIdx.y, ht = blockIdx.z;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int K = WHOLE ? 16 * TILES + 64 : a.K, Lp = SIZED ? 16 * TILES : a.Lp, P = a.P;
  const int KC = SIZED ? KC_MAX : (K + STEP - 1) / STEP, LT = SIZED ? LT_MAX : Lp / 16;
  const int len = a.kv_len[s];
  const int row = a.q_start[s];
  const int head = ht * 16 + r;
  const int* table = a.block_table + (size_t)s * a.table_stride;
  const T* keys = (const T*)a.keys;
  const T* values = (const T*)a.values;
  // this lane's query fragments: head r, elements kc * STEP + g * EPF ..
  Frag qf[KC_MAX];
#pragma unroll
  for (int kc = 0; kc < KC_MAX; ++kc) {
    const int col = kc * STEP + g * EPF;
    qf[kc] = (kc < KC && col < K && head < a.H) ? tw_load_frag((const T*)a.q + (size_t)row * a.ldq + (size_t)head * K + col)
                                                 : Elem<T>::zero();
  }
  f32x4 O[LT_MAX];
#pragma unroll
  for (int lt = 0; lt < LT_MAX; ++lt) O[lt] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, sum = 0.f;
  const int tiles = (len + 15) / 16;
  const int per = (tiles + a.splits - 1) / a.splits;
  const int t_begin = split * per, t_end = min(tiles, t_begin + per);
  // What bounds it is the trips to memory in a row: a decode step's wave has one tile or two. Everything a tile reads is
  // requested together (with `col < K ? load : zero` in front of every product each of a tile's eight key loads waited for the
  // one before) and, in bfloat16, the next tile's while this one is worked on: its keys behind the scores, its values behind the
  // products that free their registers, its page numbers a tile earlier still (float32 with sizes known at run time: the most
  // registers that they can need, twice as many, would halve the waves). 8 requests of 150
  // tokens 17.7 -> 12.3 us, one of 2,048 22.6 -> 12.7 (kernel traces).
  // A key past the end is the last one again; masked below.
  constexpr bool AHEAD = EPF == 8 || SIZED;
  auto key_of = [&](int t) { return min(t * 16 + r, len - 1); };
  auto value_of = [&](int t) { return min(t * 16 + 4 * g, (len - 1) / 4 * 4); };      // 4 keys: one page (multiples of 4)
  Frag kf[KC_MAX];
  Quad vq[LT_MAX];
  // (SIZED: places behind the sequence's end in its last page hold anything: masked like them all)
  auto page_of = [&](int t, int key) { return SIZED ? max(0, table[(t * 16) >> a.page_shift]) : table[key / P]; };
  auto key_row = [&](int t, int page) {
    if constexpr (SIZED) return keys + ((uint64_t)(uint32_t)page * (uint32_t)(P * K) + (uint32_t)(((t * 16) & (P - 1)) * K)) + r * K;
    else return keys + ((size_t)page * P + key_of(t) % P) * K;
  };
  auto request_keys = [&](int t, int page) {
    const T* krow = key_row(t, page);
#pragma unroll
    for (int kc = 0; kc < KC_MAX; ++kc)
      if (kc < KC) {                              // (past the row: a copy)
        const int col = kc * STEP + g * EPF;
        kf[kc] = tw_load_frag(krow + (kc < KC_SURE ? col : min(col, K - EPF)));
      }
  };
  auto request_values = [&](int t, int page) {
    if constexpr (SIZED) {
      const T* base = values + ((uint64_t)(uint32_t)page * (uint32_t)(P * Lp) + (uint32_t)((t * 16) & (P - 1)));
#pragma unroll
      for (int lt = 0; lt < LT_MAX; ++lt)
        vq[lt] = *reinterpret_cast<const Quad*>(base + (uint32_t)(lt * 16 * P) + (uint32_t)(r * P + 4 * g));
      return;
    }
    const T* vbase = values + (size_t)page * Lp * P + value_of(t) % P + (size_t)r * P;
#pragma unroll
    for (int lt = 0; lt < LT_MAX; ++lt)
      if (lt < LT) vq[lt] = *reinterpret_cast<const Quad*>(vbase + (size_t)(lt * 16) * P);
  };
  int t = t_begin + wave;
  int k_page = 0, v_page = 0;                     // of the tile to be requested next
  if (t < t_end) {
    k_page = page_of(t, key_of(t));
    v_page = page_of(t, value_of(t));
    if (AHEAD) {
      request_keys(t, k_page);
      request_values(t, v_page);
      if (t + 4 < t_end) {
        k_page = page_of(t + 4, key_of(t + 4));
        v_page = page_of(t + 4, value_of(t + 4));
      }
    }
  }
  for (; t < t_end; t += 4) {
    const bool edge = t * 16 + 16 > len, more = t + 4 < t_end;
    // S^T for 16 keys: this lane holds key t * 16 + r
    f32x4 S = {0.f, 0.f, 0.f, 0.f};
    const T* krow = AHEAD ? nullptr : key_row(t, k_page);
#pragma unroll
    for (int kc = 0; kc < KC_MAX; ++kc)
      if (kc < KC) {
        const int col = kc * STEP + g * EPF;
        if constexpr (AHEAD) {
          if (kc >= KC_SURE && (SIZED || K % STEP != 0) && col >= K) kf[kc] = Elem<T>::zero();
          tw_mma16(S, kf[kc], qf[kc]);            // S[j]: key t * 16 + 4 g + j against head r
        } else {
          const Frag one = col < K ? tw_load_frag(krow + col) : Elem<T>::zero();
          tw_mma16(S, one, qf[kc]);
        }
      }
    if (AHEAD && more) {
      request_keys(t + 4, k_page);
    } else if (!AHEAD) {
      request_values(t, v_page);
      if (more) {
        k_page = page_of(t + 4, key_of(t + 4));
        v_page = page_of(t + 4, value_of(t + 4));
      }
    }
    float top = -INFINITY;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      S[j] = (edge && t * 16 + 4 * g + j >= len) ? -INFINITY : S[j] * a.scale;
      top = fmaxf(top, S[j]);
    }
    top = tw_rows_max(top);                      // over the 16 keys, for head r
    const float m_new = fmaxf(m, top);
    const float alpha = m == -INFINITY ? 0.f : lt_exp<T>(m - m_new);
    f32x4 Pr;
    float part = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      Pr[j] = S[j] == -INFINITY ? 0.f : lt_exp<T>(S[j] - m_new);
      part += Pr[j];
    }
    sum = sum * alpha + tw_rows_sum(part);
    m = m_new;
    const bool rescale = __builtin_amdgcn_ballot_w64(alpha != 1.f) != 0;     // (some head's maximum has moved)
#pragma unroll
    for (int lt = 0; lt < LT_MAX; ++lt) {
      if (lt < LT) {
        Quad v = vq[lt];
        if (edge) {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (t * 16 + 4 * g + j >= len) v[j] = tw_from_float<T>(0.f);     // whatever lies there must not reach a sum
        }
        if (rescale) {
#pragma unroll
          for (int j = 0; j < 4; ++j) O[lt][j] *= alpha;
        }
        tw_mma16_k4(O[lt], v, Pr);               // O[lt][j]: element lt * 16 + 4 g + j of head r
      }
    }
    if (AHEAD && more) {
      request_values(t + 4, v_page);
      if (t + 8 < t_end) {
        k_page = page_of(t + 8, key_of(t + 8));
        v_page = page_of(t + 8, value_of(t + 8));
      }
    }
  }
  // ---- the four waves' results through LDS: [wave][16 heads][Lp + 4] sums, then [wave][16] maxima and sums
  const int OS = Lp + 4;
  float* Ow = ld_lds;
  float* mw = Ow + (size_t)4 * 16 * OS;
  float* sw = mw + 64;
#pragma unroll
  for (int lt = 0; lt < LT_MAX; ++lt)
    if (lt < LT) *reinterpret_cast<f32x4*>(Ow + ((size_t)wave * 16 + r) * OS + lt * 16 + 4 * g) = O[lt];
  if (g == 0) {
    mw[wave * 16 + r] = m;
    sw[wave * 16 + r] = sum;
  }
  __syncthreads();
  const int quads = Lp / 4;
  for (int i = threadIdx.x; i < 16 * quads; i += 256) {
    const int hh = i / quads, l = (i - hh * quads) * 4;
    if (ht * 16 + hh >= a.H) continue;
    const float top = fmaxf(fmaxf(mw[hh], mw[16 + hh]), fmaxf(mw[32 + hh], mw[48 + hh]));
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
    float total = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float f = mw[w * 16 + hh] == -INFINITY ? 0.f : lt_exp<T>(mw[w * 16 + hh] - top);
      const f32x4 v = *reinterpret_cast<const f32x4*>(Ow + ((size_t)w * 16 + hh) * OS + l);
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] += f * v[e];
      total += f * sw[w * 16 + hh];
    }
    float* dst = a.part + ((((size_t)s * gridDim.z + ht) * a.splits + split) * 16 + hh) * (Lp + 4);
    *reinterpret_cast<f32x4*>(dst + l) = o;
    if (l == 0) {
      dst[Lp] = top;
      dst[Lp + 1] = total;
    }
  }
}

// What follows it in a layer: the ranges' results of 16 rows of one head are added up, rounded to the compute type and multiplied
// with the head's W_uv ([No][Lp]; null: they go out as they are); gate (or null): the result times sigmoid(gate). One workgroup a (head, 16 rows). Its
// waves' fragments of W_uv are requested first and the ranges' sums before their weights are known, so that three trips to memory
// lie in a row; with few rows several threads share a row's element and take every P-th range each. From the projections to the
// gated heads, 16 heads, latents of 192, in a chain of such calls (us; five or six launches, 64-column products, run-time sizes and
// ranges of 8 tiles / three launches): 8 requests of 190 keys bfloat16 29.6 / 15.5, float32 48.7 / 21.8; one of 2,050 keys 31.7 / 16.1;
// 64 of 500 36.0 / 25.2; 24 heads, 64 of 4,000 88.2 / 80.2. The results are off by 0.8 times as much against 64 bits (the gate
// multiplies the float32 product).
struct LatentLeave {
  const void* w;                      // [H][No][Lp] or null
  void* out; long ldo; int so;        // head a's results at out + row(s) * ldo + a * so
  const void* gate; long ldg;         // or null: head a's gate at gate + row(s) * ldg + a * so
  int No, n;
};

template <typename T>
__global__ __launch_bounds__(512) void latent_leave_kernel(LatentDecodeArgs a, LatentLeave b) {
  typedef typename Elem<T>::Frag Frag;
  constexpr int EPF = Elem<T>::kPerFrag, U = 8, AHEAD = 4;
  extern __shared__ __attribute__((aligned(16))) unsigned char lt_lds[];
  const int head = blockIdx.x, s0 = blockIdx.y * 16, n = min(16, b.n - s0);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int Lp = a.Lp, S = a.splits, quads = Lp / 4, OS = Lp + 4;
  const int chunks = Lp / EPF, steps = (chunks + 3) / 4;
  const int xrow = Lp + 32 / (int)sizeof(T);
  float* weight = (float*)lt_lds;                            // [16][64]
  float* inv = weight + 16 * 64;                             // [16]
  f32x4* sums = (f32x4*)(inv + 16);                          // [P][items], P x items <= 512
  T* xs = (T*)(sums + 512);                                  // [16][xrow]
  const int ht = head >> 4, hh = head & 15, head_tiles = (a.H + 15) / 16;
  const size_t stride = (size_t)16 * OS;                     // from one range to the next
  auto row_part = [&](int row) { return a.part + ((((size_t)(s0 + row) * head_tiles + ht) * S) * 16 + hh) * OS; };
  // ---- requested first: W_uv's fragments of the wave's first 16 columns, the sums of the thread's first ranges ----------------
  auto load_w = [&](int col, int st0, Frag (&f)[U]) {
    const T* w_row = (const T*)b.w + ((size_t)head * b.No + min(col + r, b.No - 1)) * Lp;
#pragma unroll
    for (int u = 0; u < U; ++u) f[u] = tw_load_frag(w_row + min((st0 + u) * 4 + g, chunks - 1) * EPF);
  };
  Frag wf[U];
  if (b.w && wave * 16 < b.No) load_w(wave * 16, 0, wf);
  const int items = n * quads;
  const int P = items >= 512 ? 1 : min(S, 512 / items);      // threads that share an element
  const int item = P == 1 ? threadIdx.x : threadIdx.x % items, p = P == 1 ? 0 : threadIdx.x / items;
  f32x4 first[AHEAD];
  const bool active = item < items && p < P;
  if (active) {
    const float* base = row_part(item / quads) + item % quads * 4;
#pragma unroll
    for (int k = 0; k < AHEAD; ++k) first[k] = *reinterpret_cast<const f32x4*>(base + min(p + k * P, S - 1) * stride);
  }
  // ---- the ranges' weights, a wave a row, lane s the range s ----------------------------------------------------------------
  for (int row = wave; row < n; row += 8) {
    const float* base = row_part(row) + Lp;
    const float m = lane < S ? base[lane * stride] : -INFINITY;
    const float l = lane < S ? base[lane * stride + 1] : 0.f;
    const float sk = a.sink ? a.sink[head] : -INFINITY;
    const float top = fmaxf(tw_wave_max(m), sk);
    const float f = m == -INFINITY ? 0.f : lt_exp<T>(m - top);
    const float total = tw_wave_sum(f * l);
    weight[row * 64 + lane] = f;
    if (lane == 0) inv[row] = 1.f / (total + (a.sink ? lt_exp<T>(sk - top) : 0.f));
  }
  __syncthreads();
  // ---- the rows, in index order of the ranges within a thread ----------------------------------------------------------------
  auto finish = [&](int i, f32x4 o) {
    const int row = i / quads;
    T* dst = b.w ? xs + row * xrow + i % quads * 4 : (T*)b.out + (size_t)a.q_start[s0 + row] * b.ldo + (size_t)head * b.so + i % quads * 4;
#pragma unroll
    for (int e = 0; e < 4; ++e) dst[e] = tw_from_float<T>(o[e] * inv[row]);
  };
  for (int i = item; i < items; i += 512) {                  // (more than once only where P is 1)
    if (!active) break;
    const int row = i / quads;
    const float* base = row_part(row) + i % quads * 4;
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
    int k = p;
    if (i == item) {
#pragma unroll
      for (int j = 0; j < AHEAD; ++j)
        if (p + j * P < S) {
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] += weight[row * 64 + p + j * P] * first[j][e];
        }
      k = p + AHEAD * P;
    }
    for (; k < S; k += 4 * P) {
      f32x4 v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = *reinterpret_cast<const f32x4*>(base + min(k + j * P, S - 1) * stride);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (k + j * P < S) {
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] += weight[row * 64 + k + j * P] * v[j][e];
        }
    }
    if (P == 1) finish(i, o);
    else sums[p * items + i] = o;
  }
  __syncthreads();
  if (P > 1) {
    if (threadIdx.x < items) {
      f32x4 o = sums[threadIdx.x];
      for (int q = 1; q < P; ++q) o += sums[q * items + threadIdx.x];
      finish(threadIdx.x, o);
    }
    __syncthreads();
  }
  if (!b.w) return;
  // ---- times W_uv: D[output 4g + e][row r] --------------------------------------------------------------------------------------
  const int at_row = a.q_start[s0 + min(r, n - 1)];
  for (int col = wave * 16; col < b.No; col += 128) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int st0 = 0; st0 < steps; st0 += U) {
      if (st0 > 0 || col != wave * 16) load_w(col, st0, wf);
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (st0 + u < steps) {
          const int chunk = (st0 + u) * 4 + g;
          const bool in = chunk < chunks;
          const Frag x = *reinterpret_cast<const Frag*>(xs + min(r, n - 1) * xrow + min(chunk, chunks - 1) * EPF);
          tw_mma16(acc, in ? wf[u] : Elem<T>::zero(), in ? x : Elem<T>::zero());
        }
    }
    const int o = col + 4 * g;
    if (r < n && o < b.No) {
      T* dst = (T*)b.out + (size_t)at_row * b.ldo + (size_t)head * b.so + o;
      const T* gate = (const T*)b.gate + (size_t)at_row * b.ldg + (size_t)head * b.so + o;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        dst[e] = tw_from_float<T>(b.gate ? acc[e] / (1.f + expf(-tw_to_float(gate[e]))) : acc[e]);
    }
  }
}

// Latents of whole 32s from 64 on have an instance each; pages that are no power of two, or rotated parts of more than 64, have none.
static int latent_sized(int K, int Lp, int page_size) {
  return (page_size & (page_size - 1)) == 0 && page_size >= 16 && K <= Lp + 64 && Lp >= 64 && Lp <= 224 && Lp % 32 == 0 ? Lp / 16 : 0;
}

// Key ranges a sequence: the least estimated time, in tiles that a wave takes one after the other: rounds of the workgroups that the CUs
// work on at once, each a begin and its waves' tiles, and the ranges' sums that latent_leave_kernel reads. A CU works on one workgroup where the
// sizes are known at compile time, on two of the general kernel's, which wait longer. Of 150 calls (4 to 32 heads, nine latents, 1 to 174
// sequences of 20 to 5,400 keys, both types) whose ranges were measured beside one another the choice is 1.6 % behind the fastest; 512 workgroups
// with ranges of four tiles or more were 3.8 (192 + 64, 16 heads, 28 sequences of 1,092 keys 18 ranges 23.2 us, 9 17.9; 112 + 48, 10 of 3,651
// 51 ranges 25.7, 25 19.9). (8 requests of 190 keys, latents of 192: with ranges of 8 tiles and sizes known at run time 15.2 us, now 8.0.)
// No call gets more ranges than tw_latent_decode_most_splits.
extern "C" int tw_latent_decode_most_splits(int n_seqs, int heads, int max_kv_len) {
  if (n_seqs <= 0) return 1;
  return std::max(1, std::min({64, tw_div_up(max_kv_len, 16), 1024 / (n_seqs * tw_div_up(heads, 16))}));
}

extern "C" int tw_latent_decode_splits(int n_seqs, int heads, int max_kv_len, int K, int Lp, int page_size) {
  const int tiles = tw_div_up(max_kv_len, 16), most = tw_latent_decode_most_splits(n_seqs, heads, max_kv_len);
  const bool sized = latent_sized(K, Lp, page_size) != 0;
  const int groups = n_seqs * tw_div_up(heads, 16), at_once = sized ? 256 : 512;
  const double begin = sized ? 0.6 : 0.3, sums = sized ? 4e-4 : 1e-4;
  int best = 1;
  double least = 0;
  for (int s = 1; s <= most; ++s) {
    const double t = tw_div_up(groups * s, at_once) * (begin + tw_div_up(tw_div_up(tiles, s), 4)) + sums * n_seqs * heads * s;
    if (s == 1 || t < least) {
      least = t;
      best = s;
    }
  }
  return best;
}

extern "C" long tw_latent_decode_workspace_floats(int n_seqs, int heads, int Lp, int splits) {
  return (long)n_seqs * tw_div_up(heads, 16) * splits * 16 * (Lp + 4);
}

extern "C" int tw_latent_decode(int dtype, const void* q, long ldq, const void* keys, const void* values,
                                const int* block_table, int table_stride, const int* q_start, const int* kv_len,
                                int n_seqs, void* out, long ldo, float* workspace, long workspace_floats, int heads,
                                int K, int Lp, int page_size, float scale, int splits, const float* sink, const void* expand,
                                int expand_out, int out_stride, const void* gate, long ldg, hipStream_t stream) {
  TW_REQUIRE(q && keys && values && block_table && q_start && kv_len && out && n_seqs >= 0 && splits >= 1 && splits <= 64);
  TW_REQUIRE(heads >= 1 && K % 16 == 0 && K <= 256 && Lp % 16 == 0 && Lp >= 16 && Lp <= 240 && Lp <= K);
  TW_REQUIRE(page_size > 0 && page_size % 4 == 0);
  TW_REQUIRE(ldq >= (long)heads * K && (expand || ldo >= (long)heads * Lp));
  const int esize = dtype == TW_DTYPE_BF16 ? 2 : 4;
  TW_REQUIRE((uintptr_t)q % 16 == 0 && (uintptr_t)keys % 16 == 0 && (uintptr_t)values % 16 == 0 && (ldq * esize) % 16 == 0);
  TW_REQUIRE(n_seqs == 0 || (workspace && (uintptr_t)workspace % 16 == 0 && workspace_floats >= tw_latent_decode_workspace_floats(n_seqs, heads, Lp, splits)));
  if (expand) {            // [heads][expand_out][Lp]: out takes the heads' results times their matrices, times sigmoid(gate)
    TW_REQUIRE((uintptr_t)expand % 16 == 0 && expand_out > 0 && expand_out % 4 == 0 && out_stride >= expand_out);
    TW_REQUIRE(ldo >= (long)(heads - 1) * out_stride + expand_out && (!gate || ldg >= (long)(heads - 1) * out_stride + expand_out));
  }
  TW_REQUIRE(expand || !gate);
  if (n_seqs == 0) return 0;
  const bool pow2 = (page_size & (page_size - 1)) == 0;
  LatentDecodeArgs a{q, ldq, keys, values, block_table, table_stride, q_start, kv_len, workspace, scale,
                     heads, K, Lp, page_size, splits, pow2 ? __builtin_ctz(page_size) : -1, sink};
  const LatentLeave b{expand, out, ldo, expand ? out_stride : Lp, gate, ldg, expand_out, n_seqs};
  const int head_tiles = tw_div_up(heads, 16);
  const dim3 grid(n_seqs, splits, head_tiles);
  const size_t lds = ((size_t)4 * 16 * (Lp + 4) + 128) * sizeof(float);
  const int sized = latent_sized(K, Lp, page_size);
  const bool whole = K == Lp + 64;
#define TW_LATENT_DECODE(T)                                                                                                     \
  do {                                                                                                                         \
    auto attend = [&](auto kernel) { kernel<<<grid, 256, lds, stream>>>(a); };                                                  \
    switch (sized) {                                                                                                           \
      case 4: whole ? attend(latent_decode_kernel<T, 4, true>) : attend(latent_decode_kernel<T, 4>); break;                    \
      case 6: whole ? attend(latent_decode_kernel<T, 6, true>) : attend(latent_decode_kernel<T, 6>); break;                    \
      case 8: whole ? attend(latent_decode_kernel<T, 8, true>) : attend(latent_decode_kernel<T, 8>); break;                    \
      case 10: whole ? attend(latent_decode_kernel<T, 10, true>) : attend(latent_decode_kernel<T, 10>); break;                 \
      case 12: whole ? attend(latent_decode_kernel<T, 12, true>) : attend(latent_decode_kernel<T, 12>); break;                 \
      case 14: attend(latent_decode_kernel<T, 14>); break;                                                                     \
      default: attend(latent_decode_kernel<T, 0>);                                                                             \
    }                                                                                                                          \
    const size_t leave = (16 * 64 + 16) * 4 + 512 * 16 + (size_t)16 * (Lp + 32 / sizeof(T)) * sizeof(T);                         \
    latent_leave_kernel<T><<<dim3(heads, tw_div_up(n_seqs, 16)), 512, leave, stream>>>(a, b);                                    \
  } while (0)
  if (dtype == TW_DTYPE_BF16) TW_LATENT_DECODE(bf16_t);
  else if (dtype == TW_DTYPE_F32) TW_LATENT_DECODE(float);
  else return TW_ERR_BAD_ARGUMENT;
#undef TW_LATENT_DECODE
  return TW_LAUNCH_RESULT();
}
