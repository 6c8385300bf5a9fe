// Attention whose scores are mixed across heads before the softmax, over the paged cache.
//
//   keys   [pages][kv_heads][page_size][D]
//   values [pages][kv_heads][E][page_size]     (transposed inside a page; E may differ from D)
//
// For query position i and key position j of one sequence (0 <= i - j < window, or every j <= i
// without a window; with a window, the first `keep` keys of the sequence stay visible to every later query, at
// their true positions):
//   raw_g(i, j)  = scale * q_ig . k_j,kv(g) - slope_g * (i - j)            (slopes optional)
//   s_h(i, j)    = sum_g talk[h][g] * raw_g(i, j)                          (talk optional: s = raw)
//   p_h(i, j)    = exp(s_h(i, j)) / (exp(sink_h) + sum_j' exp(s_h(i, j')))   (sink optional)
//   out_ih       = out_scale * sum_j p_h(i, j) v_j,kv(h)
// Scores, the mixing, the softmax and the output sums are float32.
//
// Because every head's score at (i, j) needs all heads' raw scores there, a workgroup takes 16
// query TOKENS with all their heads. Its waves share the heads out between them (HPW heads a
// wave). Per 16 keys a wave forms S^T = K Q^T for its heads on the matrix unit (accumulator
// element e of lane (r, g) is query row r against key 4g + e, the same place for every head),
// leaves the raw scores in LDS, and after one barrier reads all heads' raw scores of its own lane
// and mixes them for its heads: the mixing needs no exchange between lanes. The probabilities,
// still in accumulator layout, are the B operand of O^T += V^T P^T. The raw-score buffer exists
// twice, so one barrier per key tile is enough.
//
// A tile's keys can be cut into `splits` ranges for separate workgroups (one-token sequences, whose only tile
// would otherwise walk all keys alone; prompt portions with fewer tiles than the chip has CUs); a second kernel
// merges the partial results in index order.
#include <algorithm>

#include "tw_common.h"

template <typename T> __device__ __forceinline__ float mx_exp(float v);
template <> __device__ __forceinline__ float mx_exp<float>(float v) { return expf(v); }
template <> __device__ __forceinline__ float mx_exp<bf16_t>(float v) { return __expf(v); }

template <typename T> struct MxQuad;
template <> struct MxQuad<float> { typedef f32x4 Type; };
template <> struct MxQuad<bf16_t> { typedef bf16x4 Type; };

struct MixedAttnArgs {
  const void* q; long ldq;           // head h of token n at q + n * ldq + h * D
  const void* keys; const void* values;
  const int* block_table; int table_stride;
  const int* q_start; const int* kv_len;
  int seq0;
  void* out; long ldo;               // head h of token n at out + n * ldo + h * E
  const float* talk;                 // [H][H] or null
  const float* sink;                 // [H] or null
  const float* slopes;               // [H] or null
  float* part;                       // splits > 1: [seq - seq0][tile][split][H][rows_kept][E + 2] (output sums, max, sum)
  float scale, out_scale;
  int H, G, D, E, P, window, splits;
  int keep;                          // with a window: keys 0 .. keep - 1 are seen by every later query as well
  int page_shift;                    // log2(P) if P is a power of two, else -1
  int rows_kept;                     // rows of a tile whose partial results are kept: 1 for one-token sequences, else 16
  int q_in_lds;                      // 0: fragments of the tile's queries are read from memory (once, or per key tile where
                                     // they neither fit registers nor LDS beside the raw scores)
};

// Dynamic LDS: q tile [H][16][D + pad] of T (if it is kept there), raw scores [2][H][64] of f32x4, talk [H][H rounded
// up to 4] floats.
template <typename T>
__host__ __device__ inline size_t mx_q_row(int D) { return (size_t)D + 16 / sizeof(T); }

template <typename T>
static size_t mx_lds_bytes(int H, int D, bool q_in_lds) {
  size_t q = q_in_lds ? (size_t)H * 16 * mx_q_row<T>(D) * sizeof(T) : 0;
  q = (q + 15) / 16 * 16;
  return q + (size_t)2 * H * 64 * 16 + (size_t)H * ((H + 3) / 4 * 4) * 4;
}

// HPW heads a wave, VT 16-column tiles of a head's values, WMAX the most waves a workgroup may have (it sets the
// registers a lane may use), AHEAD whether key fragments are requested a tile ahead (it costs registers), SHARE
// whether all heads of a wave read the same key/value head (its fragments are then loaded once for all of them,
// and everything a wave does once a key tile, page lookups, addresses, loads, is paid once for HPW heads).
// EXACT: the key size is exactly what four MFMA steps of fragments hold (128 in bfloat16, 64 in float32) and the
// value size is 16 VT: sizes and loop bounds are then compile-time constants.
// Such an instance whose heads share their keys keeps its query fragments in registers (32 of them), others read them
// from LDS for every key tile.
// Bound by its VALU instructions and the LDS reads of the mixing (16 heads: 128 multiply-adds and 24 LDS reads of 16
// bytes a wave and key tile), two waves a SIMD in step at one barrier a tile. Against queries read through a pointer
// that could mean LDS or memory, every head's raw scores read once per mixed head and masks built per product (2,048
// tokens, window 1,024, 16 heads of 128 on 4, bf16, with the merge): 144 -> 115 us; one token each of 8 sequences of 200:
// 25.4 -> 21.1; float32 436 -> 402.
template <int HPW, bool SHARE, bool EXACT>
struct MxQueries { static constexpr bool kInRegisters = EXACT && (SHARE || HPW == 1); };

template <typename T, int HPW, int VT, int WMAX, bool AHEAD, bool SHARE, bool EXACT>
__global__ __launch_bounds__(WMAX * 64) void attn_mixed_kernel(MixedAttnArgs a) {
  constexpr bool Q_REGS = MxQueries<HPW, SHARE, EXACT>::kInRegisters;
  constexpr int KVN = SHARE ? 1 : HPW;                     // key/value heads a wave loads
  typedef typename Elem<T>::Frag Frag;
  typedef typename MxQuad<T>::Type Quad;
  constexpr int EPF = Elem<T>::kPerFrag;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  const int H = a.H, P = a.P;
  const int D = EXACT ? 16 * Elem<T>::kPerFrag : a.D, E = EXACT ? 16 * VT : a.E;
  const size_t qrow = mx_q_row<T>(D);
  T* lds_q = (T*)lds_raw;
  size_t q_bytes = a.q_in_lds ? (size_t)H * 16 * qrow * sizeof(T) : 0;
  q_bytes = (q_bytes + 15) / 16 * 16;
  f32x4* lds_s = (f32x4*)(lds_raw + q_bytes);
  float* lds_talk = (float*)(lds_raw + q_bytes + (size_t)2 * H * 64 * 16);

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int seq = a.seq0 + blockIdx.y;
  const int q0 = a.q_start[seq], q_len = a.q_start[seq + 1] - q0;
  const int tile = blockIdx.x;
  if (tile * 16 >= q_len) return;
  const int kv_len = a.kv_len[seq];
  const int n_rows = min(16, q_len - tile * 16);
  const int pos0 = kv_len - q_len + tile * 16;              // position of the tile's first row
  const int t_row = r < n_rows ? pos0 + r : -1;
  const int* table = a.block_table + (size_t)seq * a.table_stride;
  const int heads_per_kv = H / a.G;
  const int chunks = EXACT ? 16 : D / EPF, steps = EXACT ? 4 : (chunks + 3) / 4, dts = EXACT ? VT : E / 16;

  // ---- stage the tile's queries and the mixing matrix ------------------------------------------------
  // (rows past the tile's last are row 0 again where they are not staged: their results are never stored)
  const T* q_global = (const T*)a.q + (size_t)(q0 + tile * 16 + (r < n_rows ? r : 0)) * a.ldq;
  Frag q_own[HPW][4];
  if constexpr (Q_REGS) {
#pragma unroll
    for (int i = 0; i < HPW; ++i)
#pragma unroll
      for (int st = 0; st < 4; ++st)
        q_own[i][st] = tw_load_frag(q_global + (size_t)min(wave * HPW + i, H - 1) * D + (st * 4 + g) * EPF);
  }
  for (int i = threadIdx.x; i < (!Q_REGS && a.q_in_lds ? H * 16 * chunks : 0); i += blockDim.x) {
    const int chunk = i % chunks, row = (i / chunks) % 16, head = i / (chunks * 16);
    Frag f = Elem<T>::zero();
    if (row < n_rows)
      f = tw_load_frag((const T*)a.q + (size_t)(q0 + tile * 16 + row) * a.ldq + (size_t)head * D + chunk * EPF);
    *reinterpret_cast<Frag*>(lds_q + ((size_t)head * 16 + row) * qrow + chunk * EPF) = f;
  }
  const int talk_ld = (H + 3) / 4 * 4;                     // (rows of whole 16-byte reads)
  for (int i = threadIdx.x; i < H * talk_ld; i += blockDim.x) {
    const int to = i / talk_ld, from = i % talk_ld;
    lds_talk[i] = from >= H ? 0.f : (a.talk ? a.talk[to * H + from] : (to == from ? 1.f : 0.f));
  }
  __syncthreads();

  // ---- the key tiles of this workgroup ---------------------------------------------------------------------
  const int lo = a.window > 0 ? max(0, pos0 - a.window + 1) : 0;       // first key any row of the tile sees
  const int hi = pos0 + n_rows - 1;                                     // last key (its own position)
  // The key tiles a workgroup walks are numbered without the gap between the kept first keys and the window: tiles
  // 0 .. kept - 1 hold the kept keys that lie before the window's first tile, the tiles behind them are the window's.
  const int keep = a.window > 0 ? a.keep : 0;
  const int win_lo = lo / 16;
  const int kept = min((keep + 15) / 16, win_lo);
  const int skip = win_lo - kept;                                        // key tile of walk index v >= kept: v + skip
  int tile_lo = 0, tile_hi = hi / 16 + 1 - skip;
  if (a.splits > 1) {
    const int per = (tile_hi - tile_lo + a.splits - 1) / a.splits;
    tile_lo = tile_lo + blockIdx.z * per;
    tile_hi = min(tile_hi, tile_lo + per);
  }
  auto key_tile = [&](int v) { return v < kept ? v : v + skip; };
  const bool with_sink = a.sink != nullptr && (a.splits == 1 || blockIdx.z == 0);

  float m[HPW], l[HPW];
  f32x4 acc[HPW][VT];
  float slope[HPW];
#pragma unroll
  for (int i = 0; i < HPW; ++i) {
    const int head = wave * HPW + i;
    m[i] = (with_sink && head < H) ? a.sink[head] : -INFINITY;     // the sink: a key of score sink_h and value zero
    l[i] = (with_sink && head < H) ? 1.f : 0.f;
    slope[i] = (a.slopes && head < H) ? a.slopes[head] : 0.f;
#pragma unroll
    for (int dt = 0; dt < VT; ++dt) acc[i][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const T* keys = (const T*)a.keys;
  const T* values = (const T*)a.values;
  // (the LDS pointer is typed as one: two loads through generic pointers are merged into one load that can reach either
  // memory, which waits for everything in flight)
  typedef const __attribute__((address_space(3))) Frag* LdsFrag;
  // k-steps whose fragments are requested together where they are used (one where registers are short)
  constexpr int QB = (AHEAD || WMAX <= 12) && !(HPW == 2 && VT == 16) ? 4 : 1;
  const bool ragged = !EXACT && chunks % 4 != 0;           // the last k-step ends inside itself
  auto past_zero = [&](int st0, auto& f) {                 // (zeros past the last chunk, in both operands: an infinite key
    if (ragged) {                                          // times the zero of a query would be no number)
#pragma unroll
      for (int o = 0; o < (int)(sizeof(f) / sizeof(Frag)); ++o)
        if ((st0 + o) * 4 + g >= chunks) f[o] = Elem<T>::zero();
    }
  };
  auto q_frags = [&](int head, int st0, auto& f) {         // k-steps st0, st0 + 1, ..., as many as f holds
    constexpr int N = sizeof(f) / sizeof(Frag);
    if (a.q_in_lds) {
#pragma unroll
      for (int o = 0; o < N; ++o)
        f[o] = *(LdsFrag)(lds_q + ((size_t)head * 16 + r) * qrow + min((st0 + o) * 4 + g, chunks - 1) * EPF);
    } else {
#pragma unroll
      for (int o = 0; o < N; ++o)
        f[o] = tw_load_frag(q_global + (size_t)head * D + min((st0 + o) * 4 + g, chunks - 1) * EPF);
    }
    past_zero(st0, f);
  };
  // body(number of k-steps, the first of them) over all k-steps, QB at a time and the rest at once (products for k-steps
  // that are not there: 32 sequences of 1,500, 5 heads of 32, one token each 35.4 -> 44.3 us, now 35.4)
  auto over_steps = [&](auto&& body) {
    int st0 = 0;
    for (; st0 + QB <= steps; st0 += QB) body(std::integral_constant<int, QB>{}, st0);
    if constexpr (QB > 1) {
      const int rest = steps - st0;
      if (rest == 1) body(std::integral_constant<int, 1>{}, st0);
      else if (rest == 2) body(std::integral_constant<int, 2>{}, st0);
      else if (rest == 3) body(std::integral_constant<int, 3>{}, st0);
    }
  };
  int kv_head[KVN];                                        // (SHARE: the wave's first head stands for all)
#pragma unroll
  for (int i = 0; i < KVN; ++i) kv_head[i] = (wave * HPW + i < H ? wave * HPW + i : 0) / heads_per_kv;
  // Loads carry no condition on the page: a key outside the sequence or the window is read from page 0 (every
  // pool has one), its score is selected away and its value set to zero by the masks of the edge tile it lies
  // in (a tile that is not an edge tile has no such key), so whatever that page holds never reaches a result.
  // The K fragments of a key tile are requested one tile ahead (while the tile before is mixed and multiplied
  // with its values), the V quads of a tile before the barrier that publishes its raw scores: a tile then waits
  // for memory once, not twice, and mostly not at all. KP fragments a head fit the registers kept for that
  // (head sizes up to 128 in bfloat16, 64 in float32); longer heads load their fragments where they are used.
  constexpr int KP = AHEAD ? 4 : 1;
  const bool ahead = AHEAD && steps <= KP;
  Frag kpre[KVN][KP];
  // Page numbers are looked up a tile before the loads that need them, so that no load waits for a lookup.
  const int shift = a.page_shift;
  auto page_of = [&](int p) { return shift >= 0 ? p >> shift : p / P; };
  auto in_page = [&](int p) { return shift >= 0 ? p & (P - 1) : p % P; };
  auto key_page = [&](int v) -> int {
    const int p = key_tile(v) * 16 + r;
    return (v < tile_hi && p < kv_len && (p >= lo || p < keep)) ? table[page_of(p)] : -1;
  };
  auto value_page = [&](int v) -> int {
    const int p = key_tile(v) * 16 + 4 * g;
    return (v < tile_hi && p < kv_len && (p + 3 >= lo || p < keep)) ? table[page_of(p)] : -1;
  };
  auto request_keys = [&](int v, int page) {
    if constexpr (!AHEAD) return;
    const int p = key_tile(v) * 16 + r;
#pragma unroll
    for (int i = 0; i < KVN; ++i) {
      const T* k_row = keys + (((size_t)(page < 0 ? 0 : page) * a.G + kv_head[i]) * P + in_page(p)) * D;
#pragma unroll
      for (int st = 0; st < KP; ++st) {
        const int chunk = st * 4 + g;
        kpre[i][st] = chunk < chunks ? tw_load_frag(k_row + chunk * EPF) : Elem<T>::zero();
      }
    }
  };
  int kpage = key_page(tile_lo);
  if (ahead) request_keys(tile_lo, kpage);
  int kpage_next = key_page(tile_lo + 1);
  int vpage = value_page(tile_lo);
  int buf = 0;
  for (int kt = tile_lo; kt < tile_hi; ++kt, buf ^= 1) {
    const int p0 = key_tile(kt) * 16;
    // A tile whose 16 keys every row of the query tile sees (none beyond the first row's position, none before
    // the last row's window) needs no masks; most tiles of a long window are such.
    const bool interior = p0 + 15 <= pos0 && (a.window == 0 || p0 >= pos0 + n_rows - a.window || p0 + 15 < keep);
    // ---- raw scores of this wave's heads ---------------------------------------------------------------
    f32x4 raw_own[HPW];
    {
      const int p = p0 + r;
      const int page = kpage;
#pragma unroll
      for (int i = 0; i < HPW; ++i) {
        const int head = wave * HPW + i;
        raw_own[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (head < H) {
          f32x4 s = {0.f, 0.f, 0.f, 0.f};
          if (AHEAD && ahead) {
            if constexpr (Q_REGS) {
#pragma unroll
              for (int st = 0; st < KP; ++st) tw_mma16(s, kpre[SHARE ? 0 : i][st], q_own[i][st % 4]);
            } else if constexpr (QB == KP) {
              over_steps([&](auto count, int st0) {        // (all k-steps are one group: st0 is 0)
                Frag qf[decltype(count)::value];
                q_frags(head, st0, qf);
#pragma unroll
                for (int o = 0; o < decltype(count)::value; ++o) tw_mma16(s, kpre[SHARE ? 0 : i][o], qf[o]);
              });
            } else {
#pragma unroll
              for (int st = 0; st < KP; ++st)
                if (st < steps) {
                  Frag qf[1];
                  q_frags(head, st, qf);
                  tw_mma16(s, kpre[SHARE ? 0 : i][st], qf[0]);
                }
            }
          } else {
            const T* k_row = keys + (((size_t)(page < 0 ? 0 : page) * a.G + kv_head[SHARE ? 0 : i]) * P + in_page(p)) * D;
            over_steps([&](auto count, int st0) {
              constexpr int N = decltype(count)::value;
              Frag kf[N], qf[N];
#pragma unroll
              for (int o = 0; o < N; ++o) kf[o] = tw_load_frag(k_row + min((st0 + o) * 4 + g, chunks - 1) * EPF);
              q_frags(head, st0, qf);
              past_zero(st0, kf);
#pragma unroll
              for (int o = 0; o < N; ++o) tw_mma16(s, kf[o], qf[o]);
            });
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) s[e] = s[e] * a.scale - slope[i] * (float)(t_row - (p0 + 4 * g + e));
          raw_own[i] = s;
        }
      }
    }
    // ---- this tile's values, then the next tile's keys: both are on their way during the mixing -----------------
    const int pv = p0 + 4 * g;
    Quad vq[KVN][VT];
#pragma unroll
    for (int i = 0; i < KVN; ++i) {
      const T* v_base = values + ((size_t)(vpage < 0 ? 0 : vpage) * a.G + kv_head[i]) * E * P + in_page(pv);
#pragma unroll
      for (int dt = 0; dt < VT; ++dt) {
        if (dt < dts) vq[i][dt] = *reinterpret_cast<const Quad*>(v_base + (size_t)(dt * 16 + r) * P);
      }
    }
    if (ahead) request_keys(kt + 1, kpage_next);
    kpage = kpage_next;
    kpage_next = key_page(kt + 2);
    vpage = value_page(kt + 1);          // (this tile's quads are in registers already)
#pragma unroll
    for (int i = 0; i < HPW; ++i) {
      const int head = wave * HPW + i;
      if (head < H) lds_s[((size_t)buf * H + head) * 64 + lane] = raw_own[i];
    }
    __syncthreads();
    // ---- mix (every head's raw scores are read once for all heads of the wave) ---------------------------------
    // (a sum of four heads at a time: one chain over all 16 is off by 1.5 times as much; the first head's product is the one that
    // is not rounded: distance slopes make its score the largest, and rounding it first cost 2 to 6 % in the results)
    f32x4 mixed[HPW];
    const float* talk_row[HPW];
#pragma unroll
    for (int i = 0; i < HPW; ++i) {
      mixed[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      talk_row[i] = lds_talk + min(wave * HPW + i, H - 1) * talk_ld;
    }
    const f32x4* raw_lane = lds_s + (size_t)buf * H * 64 + lane;
    int other = 0;
    // (two rounds at a time where two heads share them and registers are left: 5 % slower otherwise at 16 heads with values of 256)
#pragma unroll(HPW == 1 || VT == 16 ? 1 : 2)
    for (; other + 4 <= H; other += 4) {                   // four heads' reads in flight at a time
      f32x4 raw[4];
#pragma unroll
      for (int o = 0; o < 4; ++o) raw[o] = raw_lane[(other + o) * 64];
#pragma unroll
      for (int i = 0; i < HPW; ++i) {
        const f32x4 w = *reinterpret_cast<const f32x4*>(talk_row[i] + other);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          mixed[i][e] += fmaf(w[3], raw[3][e], fmaf(w[2], raw[2][e], fmaf(w[0], raw[0][e], w[1] * raw[1][e])));
        }
      }
    }
#pragma unroll 1
    for (; other < H; ++other) {
      const f32x4 raw = raw_lane[other * 64];
#pragma unroll
      for (int i = 0; i < HPW; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) mixed[i][e] = fmaf(talk_row[i][other], raw[e], mixed[i][e]);
    }
    // values of keys outside the sequence or the window are zeros (once a tile, not a product)
    if (!interior) {
      bool seen[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) seen[e] = (pv + e < kv_len) & ((pv + e >= lo) | (pv + e < keep));
#pragma unroll
      for (int i = 0; i < KVN; ++i)
#pragma unroll
        for (int dt = 0; dt < VT; ++dt)
          if (dt < dts) {
#pragma unroll
            for (int e = 0; e < 4; ++e) vq[i][dt][e] = seen[e] ? vq[i][dt][e] : tw_from_float<T>(0.f);
          }
    }
    // ---- mask, online softmax, O^T += V^T P^T -----------------------------------------------------------------
#pragma unroll
    for (int i = 0; i < HPW; ++i) {
      const int head = wave * HPW + i;
      if (head < H) {
        f32x4 s = mixed[i];
        float mx = -INFINITY;
        if (!interior) {
          const int lo_row = a.window > 0 ? t_row - a.window + 1 : 0;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int p = p0 + 4 * g + e;
            const bool ok = (p < kv_len) & (p <= t_row) & ((p >= lo_row) | (p < keep));
            s[e] = ok ? s[e] : -INFINITY;
          }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) mx = fmaxf(mx, s[e]);
        mx = tw_rows_max(mx);
        const float m_new = fmaxf(m[i], mx);
        const float m_use = m_new == -INFINITY ? 0.f : m_new;
        const float alpha = mx_exp<T>(m[i] - m_use);
        f32x4 pr;
        float sum = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          pr[e] = mx_exp<T>(s[e] - m_use);
          sum += pr[e];
        }
        sum = tw_rows_sum(sum);
        l[i] = l[i] * alpha + sum;
        m[i] = m_new;
        // the output sums are rescaled only when some row's maximum has moved (a branch the whole wave takes alike)
        const bool rescale = __builtin_amdgcn_ballot_w64(alpha != 1.f) != 0;
#pragma unroll
        for (int dt = 0; dt < VT; ++dt) {
          if (dt < dts) {
            const Quad v = vq[SHARE ? 0 : i][dt];
            if (rescale) {
#pragma unroll
              for (int e = 0; e < 4; ++e) acc[i][dt][e] *= alpha;
            }
            tw_mma16_k4(acc[i][dt], v, pr);
          }
        }
      }
    }
  }

  // ---- results: lane (r, g) holds out[row r][16 dt + 4 g + e] ------------------------------------------------------
#pragma unroll
  for (int i = 0; i < HPW; ++i) {
    const int head = wave * HPW + i;
    if (head >= H || r >= n_rows) continue;
    if (a.splits == 1) {
      const float inv = l[i] > 0.f ? a.out_scale / l[i] : 0.f;
      T* dst = (T*)a.out + (size_t)(q0 + tile * 16 + r) * a.ldo + (size_t)head * E;
#pragma unroll
      for (int dt = 0; dt < VT; ++dt)
        if (dt < dts)
#pragma unroll
          for (int e = 0; e < 4; ++e) dst[dt * 16 + 4 * g + e] = tw_from_float<T>(acc[i][dt][e] * inv);
    } else if (r < a.rows_kept) {
      float* dst = a.part + (((((size_t)blockIdx.y * gridDim.x + tile) * a.splits + blockIdx.z) * H + head) * a.rows_kept + r) * (E + 2);
#pragma unroll
      for (int dt = 0; dt < VT; ++dt)
        if (dt < dts)
#pragma unroll
          for (int e = 0; e < 4; ++e) dst[dt * 16 + 4 * g + e] = acc[i][dt][e];
      if (g == 0) {
        dst[E] = m[i];
        dst[E + 1] = l[i];
      }
    }
  }
}

// One query token a sequence (a decode step): the query HEADS of a key/value head are the rows of the matrix unit's tile instead
// of 16 tokens of which one is there, and a wave has one key/value head. Per NT key tiles it forms S = Q K^T, leaves its heads'
// raw scores in LDS ([key][head]), and after one barrier reads all heads' scores of a key, four neighbouring heads a lane: the A
// operand of the mixing product S^T talk^T, whose result, its own heads across and keys down, is what the softmax and
// O^T += V^T P^T want. Nothing is shared behind the mixing, so waves keep and store their own heads' sums. Without mixing
// S^T = K Q^T is formed directly and waves never meet. Distance slopes are mixed once (sum_g talk[h][g] slope_g) and come off the
// mixed scores.
// What bounds it is a wave's chain: the trips to memory (everything NT tiles read is requested together and a group ahead) and
// its instructions, about 2 ns each with one wave a SIMD. 16-token tiles whose waves share the heads out walk a range's key
// tiles in turn at 4 us each; one wave with all heads of a key tile (no LDS, the products with other heads' keys thrown away)
// had five times the instructions and was as slow. With the merge, in a chain of such calls, bfloat16, heads of 128 (us, tiles of
// tokens / here): 16 on 4, window 1,024, one sequence 26.6 / 13.4, 32 sequences 45.2 / 25.6; 24 on 4, 2,048 keys 57.0 / 14.7, 64
// sequences of 1,500 208 / 41; without mixing 26.7 / 11.1; float32, 16 on 4, 800 keys 57.7 / 18.6. 8 heads of 64 on 8, 8 sequences
// of 2,050: 29.9 / 21.5. Errors against 64 bits: as before in bfloat16, 0.5 to 1.0 times as large in float32.
template <typename T, int S, int NT, bool TALK>
__global__ __launch_bounds__(512) void attn_mixed_one_kernel(MixedAttnArgs a) {
  typedef typename Elem<T>::Frag Frag;
  typedef typename MxQuad<T>::Type Quad;
  constexpr int EPF = Elem<T>::kPerFrag;
  constexpr int KC = S / (4 * EPF), VT = S / 16;             // k-steps of a key, 16-element tiles of a value
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  const int lane = threadIdx.x & 63, kv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int H = a.H, G = a.G, P = a.P;
  const int seq = a.seq0 + blockIdx.y;
  const int q0 = a.q_start[seq];
  if (a.q_start[seq + 1] <= q0) return;
  const int kv_len = a.kv_len[seq], pos = kv_len - 1;       // the token's own position
  const int* table = a.block_table + (size_t)seq * a.table_stride;
  const int per_kv = H / G, head = kv * per_kv + r;         // lane r's query head, where r < per_kv
  const bool mine = r < per_kv;

  // ---- this workgroup's key tiles, numbered without the gap between the kept first keys and the window (as in attn_mixed_kernel) ----
  const int lo = a.window > 0 ? max(0, pos - a.window + 1) : 0;
  const int keep = a.window > 0 ? a.keep : 0;
  const int win_lo = lo / 16;
  const int kept = min((keep + 15) / 16, win_lo), skip = win_lo - kept;
  int tile_lo = 0, tile_hi = pos / 16 + 1 - skip;
  if (a.splits > 1) {
    const int per = (tile_hi + a.splits - 1) / a.splits;
    tile_lo = blockIdx.z * per;
    tile_hi = min(tile_hi, tile_lo + per);
  }
  auto key_tile = [&](int v) { return v < kept ? v : v + skip; };
  // Page sizes are multiples of 16: a key tile lies in one page, whose number and addresses are the whole wave's (scalar). A
  // tile of the range holds a key that is seen, so its page is held; what else lies in it is masked. Tiles past the range are
  // its last one again, masked whole.
  const uint32_t k_off = r * S + g * EPF, page_size = (uint32_t)G * P * S;
  const uint32_t v_off = r * P + 4 * g;
  Frag kf[NT][KC];
  Quad vq[NT][VT];
  int page[NT];
  auto find_pages = [&](int v0) {
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int p = key_tile(min(v0 + i, tile_hi - 1)) * 16;
      page[i] = max(0, table[p >> a.page_shift]);
    }
  };
  auto place_of = [&](int v) { return (key_tile(min(v, tile_hi - 1)) * 16) & (P - 1); };
  auto request_keys = [&](int v0) {
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const T* base = (const T*)a.keys + ((uint64_t)(uint32_t)page[i] * page_size + (uint32_t)((kv * P + place_of(v0 + i)) * S));
#pragma unroll
      for (int st = 0; st < KC; ++st) kf[i][st] = tw_load_frag(base + k_off + st * 4 * EPF);
    }
  };
  auto request_values = [&](int v0) {
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const T* base = (const T*)a.values + ((uint64_t)(uint32_t)page[i] * page_size + (uint32_t)(kv * S * P + place_of(v0 + i)));
#pragma unroll
      for (int dt = 0; dt < VT; ++dt) vq[i][dt] = *reinterpret_cast<const Quad*>(base + (uint32_t)(dt * 16 * P) + v_off);
    }
  };
  if (tile_lo < tile_hi) {
    find_pages(tile_lo);
    request_keys(tile_lo);
    request_values(tile_lo);
  }
  // ---- the heads' queries, their rows of the mixing matrix, their slopes --------------------------------------------------
  Frag qf[KC];
#pragma unroll
  for (int st = 0; st < KC; ++st) {
    const Frag f = tw_load_frag((const T*)a.q + (size_t)q0 * a.ldq + (size_t)min(head, H - 1) * S + (st * 4 + g) * EPF);
    qf[st] = mine ? f : Elem<T>::zero();
  }
  constexpr int CT = TALK ? 2 : 1;                           // up to 32 heads, 16 a product
  f32x4 talk[CT];
  float slope = 0.f;
  if constexpr (TALK) {
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int from = ct * 16 + 4 * g + e;
        const float w = a.talk[min(head, H - 1) * H + min(from, H - 1)];
        talk[ct][e] = mine && from < H ? w : 0.f;
        if (a.slopes) slope = fmaf(talk[ct][e], a.slopes[min(from, H - 1)], slope);
      }
    if (a.slopes) slope = tw_rows_sum(slope);
  } else if (a.slopes) {
    slope = a.slopes[min(head, H - 1)];
  }
  const bool with_sink = a.sink != nullptr && blockIdx.z == 0;
  float m = with_sink ? a.sink[min(head, H - 1)] : -INFINITY;     // the sink: a key of score sink_h and value zero
  float l = with_sink ? 1.f : 0.f;
  f32x4 acc[VT];
#pragma unroll
  for (int dt = 0; dt < VT; ++dt) acc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int row_floats = (H + 3) / 4 * 4 + 4;                // (rows of whole 16-byte reads)
  float* raw = (float*)lds_raw;

  for (int t = tile_lo; t < tile_hi; t += NT) {
    const bool more = t + NT < tile_hi;
    // ---- scores: lane (r, g) then holds its head r against keys 4g + e of every tile -----------------------------------------
    f32x4 s[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      s[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int st = 0; st < KC; ++st) {
        if constexpr (TALK) tw_mma16(s[i], qf[st], kf[i][st]);
        else tw_mma16(s[i], kf[i][st], qf[st]);
      }
    }
    if (more) {
      find_pages(t + NT);
      request_keys(t + NT);
    }
    if constexpr (TALK) {
      // (here lane (r, g) holds key r against the wave's heads 4g + e)
      if (per_kv % 4 == 0) {
        if (4 * g < per_kv) {
#pragma unroll
          for (int i = 0; i < NT; ++i) *reinterpret_cast<f32x4*>(raw + (i * 16 + r) * row_floats + kv * per_kv + 4 * g) = s[i];
        }
      } else {
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (4 * g + e < per_kv) raw[(i * 16 + r) * row_floats + kv * per_kv + 4 * g + e] = s[i][e];
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        s[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        // (heads 4g + 3 first, 4g last: the first head's product is then added to the others' sum and not rounded by itself)
#pragma unroll
        for (int ct = CT - 1; ct >= 0; --ct)
          if (ct * 16 < H) {
            f32x4 all = *reinterpret_cast<const f32x4*>(raw + (i * 16 + r) * row_floats + min(ct * 16 + 4 * g, (H - 1) / 4 * 4));
#pragma unroll
            for (int e = 3; e >= 0; --e)
              s[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(ct * 16 + 4 * g + e < H ? all[e] : 0.f, talk[ct][e], s[i], 0, 0, 0);
          }
      }
      raw = (float*)lds_raw + (raw == (float*)lds_raw ? NT * 16 * row_floats : 0);
    }
    // ---- mask, softmax ---------------------------------------------------------------------------------------------------------
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int p0 = key_tile(min(t + i, tile_hi - 1)) * 16;
      // (a wave's branch: masks only where a key of the tile is not seen)
      const bool interior = t + i < tile_hi && p0 + 15 <= pos && (p0 >= lo || p0 + 15 < keep);
#pragma unroll
      for (int e = 0; e < 4; ++e) s[i][e] = s[i][e] * a.scale - slope * (float)(pos - (p0 + 4 * g + e));
      if (!interior) {
        bool seen[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int p = p0 + 4 * g + e;
          seen[e] = t + i < tile_hi && p <= pos && (p >= lo || p < keep);
          s[i][e] = seen[e] ? s[i][e] : -INFINITY;
        }
#pragma unroll
        for (int dt = 0; dt < VT; ++dt) {
          if constexpr (EPF == 8) {
            u32x2 bits = __builtin_bit_cast(u32x2, vq[i][dt]);
#pragma unroll
            for (int h = 0; h < 2; ++h) bits[h] &= (seen[2 * h] ? 0x0000ffffu : 0u) | (seen[2 * h + 1] ? 0xffff0000u : 0u);
            vq[i][dt] = __builtin_bit_cast(Quad, bits);
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) vq[i][dt][e] = seen[e] ? vq[i][dt][e] : 0.f;
          }
        }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) mx = fmaxf(mx, s[i][e]);
    }
    mx = tw_rows_max(mx);
    const float m_new = fmaxf(m, mx);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = mx_exp<T>(m - m_use);
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      float part = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[i][e] = mx_exp<T>(s[i][e] - m_use);
        part += s[i][e];
      }
      sum += part;
    }
    l = l * alpha + tw_rows_sum(sum);
    m = m_new;
    if (__builtin_amdgcn_ballot_w64(alpha != 1.f) != 0) {
#pragma unroll
      for (int dt = 0; dt < VT; ++dt)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[dt][e] *= alpha;
    }
    // ---- O^T += V^T P^T ----------------------------------------------------------------------------------------------------------
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int dt = 0; dt < VT; ++dt) tw_mma16_k4(acc[dt], vq[i][dt], s[i]);
    if (more) request_values(t + NT);
  }

  // ---- results: lane (r, g) holds out[head r][16 dt + 4 g + e] -------------------------------------------------------------------
  if (!mine) return;
  if (a.splits == 1) {
    const float inv = l > 0.f ? a.out_scale / l : 0.f;
    T* dst = (T*)a.out + (size_t)q0 * a.ldo + (size_t)head * S + 4 * g;
#pragma unroll
    for (int dt = 0; dt < VT; ++dt)
#pragma unroll
      for (int e = 0; e < 4; ++e) dst[dt * 16 + e] = tw_from_float<T>(acc[dt][e] * inv);
  } else {
    float* dst = a.part + (((size_t)blockIdx.y * a.splits + blockIdx.z) * H + head) * (S + 2);
#pragma unroll
    for (int dt = 0; dt < VT; ++dt)
#pragma unroll
      for (int e = 0; e < 4; ++e) dst[dt * 16 + 4 * g + e] = acc[dt][e];
    if (g == 0) {
      dst[S] = m;
      dst[S + 1] = l;
    }
  }
}

// Merge the partial results of a tile's key ranges, in index order. grid (tiles, n_seqs, H). The ranges' weights are formed
// once a row in LDS (threads side by side: one after the other, every thread for itself, 16 ranges took 9 us of a decode step),
// then eight ranges' sums are in flight a thread. (Ranges past the 64th, which no rule here asks for, are weighted one by one.)
constexpr int MX_MERGE_MOST = 64;                            // weights held a row

template <typename T>
__global__ __launch_bounds__(256) void attn_mixed_merge_kernel(MixedAttnArgs a) {
  __shared__ float weight[16 * MX_MERGE_MOST], top_row[16], inv_row[16];
  const int seq = a.seq0 + blockIdx.y, head = blockIdx.z, tile = blockIdx.x;
  const int q0 = a.q_start[seq], q_len = a.q_start[seq + 1] - q0;
  if (tile * 16 >= q_len) return;
  const int n_rows = min(min(16, q_len - tile * 16), a.rows_kept);
  const int E = a.E, S = a.splits;
  const size_t stride = (size_t)a.H * a.rows_kept * (E + 2);          // between key ranges
  const float* tile_base = a.part + ((((size_t)blockIdx.y * gridDim.x + tile) * S) * a.H + head) * a.rows_kept * (E + 2);
  // a wave a row: lane s the ranges s, s + 64, ...
  const int lane = threadIdx.x & 63;
  for (int row = threadIdx.x >> 6; row < n_rows; row += 4) {
    const float* base = tile_base + (size_t)row * (E + 2) + E;
    float top = -INFINITY, total = 0.f;
    for (int s = lane; s < S; s += 64) top = fmaxf(top, base[s * stride]);
    top = tw_wave_max(top);
    top = top == -INFINITY ? 0.f : top;
    for (int s = lane; s < S; s += 64) {
      const float f = mx_exp<T>(base[s * stride] - top);
      total += base[s * stride + 1] * f;
      if (s < MX_MERGE_MOST) weight[row * MX_MERGE_MOST + s] = f;
    }
    total = tw_wave_sum(total);
    if (lane == 0) {
      top_row[row] = top;
      inv_row[row] = total > 0.f ? a.out_scale / total : 0.f;
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < n_rows * E; i += blockDim.x) {
    const int row = i / E, d = i % E;
    const float* base = tile_base + (size_t)row * (E + 2);
    const float* w = weight + row * MX_MERGE_MOST;
    float o = 0.f;
    int s = 0;
    for (; s + 8 <= min(S, MX_MERGE_MOST); s += 8) {
      float v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = base[(s + k) * stride + d];
#pragma unroll
      for (int k = 0; k < 8; ++k) o += v[k] * w[s + k];
    }
    for (; s < S; ++s) o += base[s * stride + d] * (s < MX_MERGE_MOST ? w[s] : mx_exp<T>(base[s * stride + E] - top_row[row]));
    ((T*)a.out)[(size_t)(q0 + tile * 16 + row) * a.ldo + (size_t)head * E + d] = tw_from_float<T>(o * inv_row[row]);
  }
}

template <typename T, int HPW, int VT, int WMAX, bool AHEAD, bool SHARE, bool EXACT = false>
static int mixed_launch(MixedAttnArgs a, int n_seqs, int tiles, int waves, size_t lds, hipStream_t stream) {
  auto kernel = attn_mixed_kernel<T, HPW, VT, WMAX, AHEAD, SHARE, EXACT>;
  if (MxQueries<HPW, SHARE, EXACT>::kInRegisters) {
    a.q_in_lds = 0;
    lds = mx_lds_bytes<T>(a.H, a.D, false);
  }
  if (lds > 48 * 1024) {
    hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return (int)e;
  }
  kernel<<<dim3(tiles, n_seqs, a.splits), waves * 64, lds, stream>>>(a);
  return TW_LAUNCH_RESULT();
}

// One query token a sequence: sizes that attn_mixed_one_kernel holds (a wave a key/value head, its query heads one tile's rows,
// a key tile in one page).
static bool mixed_one_takes(int max_q_len, int H, int G, int D, int E, int P) {
  return max_q_len == 1 && G <= 8 && H / G <= 16 && D == E && (D == 64 || D == 128) && P >= 16 && (P & (P - 1)) == 0;
}

template <typename T, int S, bool TALK>
static int mixed_one_launch(const MixedAttnArgs& a, int n_seqs, hipStream_t stream) {
  constexpr int NT = Elem<T>::kPerFrag == 8 ? 4 : 2;          // (float32 fragments are twice as many registers)
  const size_t lds = TALK ? (size_t)2 * NT * 16 * ((a.H + 3) / 4 * 4 + 4) * sizeof(float) : 0;
  attn_mixed_one_kernel<T, S, NT, TALK><<<dim3(1, n_seqs, a.splits), a.G * 64, lds, stream>>>(a);
  return TW_LAUNCH_RESULT();
}

template <typename T>
static int mixed_dispatch(const MixedAttnArgs& args, int n_seqs, int max_q_len, hipStream_t stream) {
  const int tiles = tw_div_up(max_q_len, 16);
  // Heads a wave: one up to 8 heads, two above (workgroups of up to 8 waves up to 16 heads). What a wave does once
  // a key tile (page lookups, addresses, loads of keys and values) is paid once for both heads where they share a
  // key/value head, and fewer waves wait at the tile's barrier. The output sums of a wave's heads live in its registers.
  // (measured at 2,048 tokens, heads of 128: 8 heads 164 us with one head a wave, 218 with two; 12 heads 338 and
  // 295; 16 heads 431 and 271; four heads a wave ran out of registers and was slower than two at 16 and 32 heads)
  const int per_kv = args.H / args.G;
  const int hpw = args.H <= 8 ? 1 : 2;
  const int waves = tw_div_up(args.H, hpw);
  const bool share = hpw == 2 && per_kv % 2 == 0;
  MixedAttnArgs a = args;
  a.q_in_lds = mx_lds_bytes<T>(a.H, a.D, true) <= 150 * 1024 ? 1 : 0;
  a.rows_kept = max_q_len == 1 ? 1 : 16;
  a.page_shift = (a.P & (a.P - 1)) == 0 ? __builtin_ctz(a.P) : -1;
  const size_t lds = mx_lds_bytes<T>(a.H, a.D, a.q_in_lds != 0);
  TW_REQUIRE(waves <= 16 && lds <= 150 * 1024);
  int code;
  if (mixed_one_takes(max_q_len, a.H, a.G, a.D, a.E, a.P)) {
    code = a.D == 64 ? (a.talk ? mixed_one_launch<T, 64, true>(a, n_seqs, stream) : mixed_one_launch<T, 64, false>(a, n_seqs, stream))
                     : (a.talk ? mixed_one_launch<T, 128, true>(a, n_seqs, stream) : mixed_one_launch<T, 128, false>(a, n_seqs, stream));
    if (code != 0 || a.splits == 1) return code;
    attn_mixed_merge_kernel<T><<<dim3(1, n_seqs, a.H), 256, 0, stream>>>(a);
    return TW_LAUNCH_RESULT();
  }
  // (the sizes of most models: compile-time instances for values of 128 beside keys of four MFMA steps)
  const bool exact = a.D == 16 * Elem<T>::kPerFrag && a.E == 128;
#define TW_MIXED(HPW_, VT_, WMAX_, AHEAD_)                                                                          \
  (exact && VT_ == 8 && AHEAD_                                                                                      \
     ? (share ? mixed_launch<T, HPW_, VT_, WMAX_, AHEAD_, (HPW_ > 1), (VT_ == 8 && AHEAD_)>(a, n_seqs, tiles, waves, lds, stream)  \
              : mixed_launch<T, HPW_, VT_, WMAX_, AHEAD_, false, (VT_ == 8 && AHEAD_)>(a, n_seqs, tiles, waves, lds, stream))      \
     : (share ? mixed_launch<T, HPW_, VT_, WMAX_, AHEAD_, (HPW_ > 1)>(a, n_seqs, tiles, waves, lds, stream)          \
              : mixed_launch<T, HPW_, VT_, WMAX_, AHEAD_, false>(a, n_seqs, tiles, waves, lds, stream)))
  if (hpw == 1)
    code = a.E <= 64 ? TW_MIXED(1, 4, 8, true) : a.E <= 128 ? TW_MIXED(1, 8, 8, true) : TW_MIXED(1, 16, 8, true);
  else if (waves <= 8)
    code = a.E <= 64 ? TW_MIXED(2, 4, 8, true) : a.E <= 128 ? TW_MIXED(2, 8, 8, true) : TW_MIXED(2, 16, 8, true);
  else if (waves <= 12)         // up to 24 heads: 12 waves, three a SIMD, a third more registers than with room for 16
                                // (24 heads of 128 on 6, 2,048 tokens, window 1,024: 447 -> 336 us, float32 783 -> 662)
    code = a.E <= 64 ? TW_MIXED(2, 4, 12, false) : a.E <= 128 ? TW_MIXED(2, 8, 12, false) : TW_MIXED(2, 16, 12, false);
  else                          // more: up to 16 waves, half the registers each
    code = a.E <= 64 ? TW_MIXED(2, 4, 16, false) : a.E <= 128 ? TW_MIXED(2, 8, 16, false) : TW_MIXED(2, 16, 16, false);
#undef TW_MIXED
  if (code != 0 || a.splits == 1) return code;
  attn_mixed_merge_kernel<T><<<dim3(tiles, n_seqs, a.H), 256, 0, stream>>>(a);
  return TW_LAUNCH_RESULT();
}

// Key ranges for one-token sequences of up to max_kv_len seen keys: the least estimated time, in steps of a workgroup over its key tiles
// (attn_mixed_one_kernel takes 4 tiles a step in bfloat16, 2 in float32, attn_mixed_kernel one): rounds of as many workgroups as the
// CUs work on at once, each a begin and its steps, and for more than one range the merge. A CU works on four of the one's waves (one a SIMD),
// eight of the other's. Of 1,189 calls of 15 forms (1 to 32 heads on 1 to 16, 1 to 300 sequences of 48 to 4,000 keys, both types) whose ranges
// were measured beside one another the choice is 1.4 % behind the fastest, by rules without rounds (256 or 512 workgroups, ranges of four tiles or
// more) 10 and 21 %: bfloat16, 30 heads of 64 on 10, 93 sequences of 645 keys 2 ranges 144 us, 5 132; 20 of 128 on 10, one of 80 keys 2 ranges 1.6
// times as long as 5; 24 on 4, 200 of 100 keys 2 ranges 1.9 times as long as one.
// No call gets more ranges than tw_attn_mixed_most_splits: the merge holds 64, and from 1,024 workgroups on more only cost.
extern "C" int tw_attn_mixed_most_splits(int n_seqs, int max_kv_len) {
  if (n_seqs <= 0) return 1;
  return std::max(1, std::min({MX_MERGE_MOST, tw_div_up(max_kv_len, 16), 1024 / n_seqs}));
}

extern "C" int tw_attn_mixed_splits(int dtype, int n_seqs, int max_kv_len, int H, int G, int D, int E, int page_size) {
  const int tiles = tw_div_up(max_kv_len, 16), most = tw_attn_mixed_most_splits(n_seqs, max_kv_len);
  const bool one = mixed_one_takes(1, H, G, D, E, page_size);
  const int step = !one ? 1 : dtype == TW_DTYPE_BF16 ? 4 : 2, waves = one ? G : H <= 8 ? H : tw_div_up(H, 2);
  const int at_once = 256 * std::max(1, (one ? 4 : 8) / waves);
  int best = 1;
  double least = 0;
  for (int s = 1; s <= most; ++s) {
    const int blocks = n_seqs * s, steps = tw_div_up(tw_div_up(tiles, s), step);
    double t = tw_div_up(blocks, at_once) * ((one ? 0.3 : 0.6) + steps);
    if (s > 1) t += one ? 1.5 + 0.002 * blocks * H / 16 : 0.3 + 0.001 * blocks;
    if (s == 1 || t < least) {
      least = t;
      best = s;
    }
  }
  return best;
}

// Key ranges for prompt portions: only where the row tiles alone would leave most of the chip idle and a tile
// has keys enough to share out (each range at least 8 key tiles).
extern "C" int tw_attn_mixed_prefill_splits(int n_tokens, int n_seqs, int max_kv_len) {
  const int tiles = tw_div_up(n_tokens, 16) + n_seqs;
  const int key_tiles = tw_div_up(max_kv_len, 16);
  int s = 384 / (tiles > 0 ? tiles : 1);
  if (s > key_tiles / 8) s = key_tiles / 8;
  if (s > 8) s = 8;
  return s < 1 ? 1 : s;
}

extern "C" long tw_attn_mixed_workspace_floats(int n_seqs, int max_q_len, int q_heads, int value_dim, int splits) {
  const long tiles = tw_div_up(max_q_len, 16);
  return (long)n_seqs * tiles * splits * q_heads * (max_q_len == 1 ? 1 : 16) * (value_dim + 2);
}

extern "C" int tw_attn_mixed(int dtype, const void* q, long ldq, const void* keys, const void* values,
                             const int* block_table, int table_stride, const int* q_start, const int* kv_len,
                             int seq0, int n_seqs, int max_q_len, void* out, long ldo, const float* talk,
                             const float* sink, const float* slopes, float* workspace, long workspace_floats,
                             int q_heads, int kv_heads, int key_dim, int value_dim, int page_size, int window,
                             int keep_first, float scale, float out_scale, int splits, hipStream_t stream) {
  TW_REQUIRE(q && keys && values && block_table && q_start && kv_len && out);
  TW_REQUIRE(n_seqs >= 0 && seq0 >= 0 && max_q_len >= 1 && splits >= 1 && window >= 0 && keep_first >= 0);
  TW_REQUIRE(q_heads >= 1 && q_heads <= 32 && kv_heads >= 1 && q_heads % kv_heads == 0);
  TW_REQUIRE(key_dim % 16 == 0 && key_dim >= 16 && key_dim <= 256 && value_dim % 16 == 0 && value_dim >= 16 && value_dim <= 256);
  TW_REQUIRE(page_size > 0 && page_size % 4 == 0);
  TW_REQUIRE(ldq >= (long)q_heads * key_dim && ldo >= (long)q_heads * value_dim);
  TW_REQUIRE((uintptr_t)q % 16 == 0 && (uintptr_t)keys % 16 == 0 && (uintptr_t)values % 16 == 0);
  const int esize = dtype == TW_DTYPE_BF16 ? 2 : 4;
  TW_REQUIRE((ldq * esize) % 16 == 0);
  if (splits > 1) {
    TW_REQUIRE(workspace != nullptr);
    TW_REQUIRE(workspace_floats >= tw_attn_mixed_workspace_floats(n_seqs, max_q_len, q_heads, value_dim, splits));
  }
  if (n_seqs == 0) return 0;
  MixedAttnArgs a{q, ldq, keys, values, block_table, table_stride, q_start, kv_len, seq0, out, ldo, talk, sink, slopes,
                  workspace, scale, out_scale, q_heads, kv_heads, key_dim, value_dim, page_size, window, splits, keep_first, -1, 16, 1};
  if (dtype == TW_DTYPE_BF16) return mixed_dispatch<bf16_t>(a, n_seqs, max_q_len, stream);
  if (dtype == TW_DTYPE_F32) return mixed_dispatch<float>(a, n_seqs, max_q_len, stream);
  return TW_ERR_BAD_ARGUMENT;
}

// ---- new keys and values into the pages (no rotation; values transposed inside a page) --------------------------
template <typename T>
__global__ void kv_store_kernel(const T* __restrict__ src, long ld, int k_col, int v_col, const int* __restrict__ slots,
                                T* __restrict__ keys, T* __restrict__ values, int G, int D, int E, int P) {
  const int n = blockIdx.x;
  const int slot = slots[n];
  if (slot < 0) return;
  const int page = slot / P, at = slot % P;
  const T* row = src + (size_t)n * ld;
  for (int i = threadIdx.x; i < G * D; i += blockDim.x) {
    const int kvh = i / D, d = i % D;
    keys[(((size_t)page * G + kvh) * P + at) * D + d] = row[k_col + i];
  }
  for (int i = threadIdx.x; i < G * E; i += blockDim.x) {
    const int kvh = i / E, d = i % E;
    values[(((size_t)page * G + kvh) * E + d) * P + at] = row[v_col + i];
  }
}

extern "C" int tw_kv_store(int dtype, const void* src, long ld, int k_col, int v_col, const int* slots, void* keys,
                           void* values, int n, int kv_heads, int key_dim, int value_dim, int page_size,
                           hipStream_t stream) {
  TW_REQUIRE(src && slots && keys && values && n >= 0 && kv_heads > 0 && key_dim > 0 && value_dim > 0 && page_size > 0);
  TW_REQUIRE(k_col >= 0 && v_col >= 0 && ld >= k_col + (long)kv_heads * key_dim && ld >= v_col + (long)kv_heads * value_dim);
  if (n == 0) return 0;
  if (dtype == TW_DTYPE_BF16)
    kv_store_kernel<bf16_t><<<n, 128, 0, stream>>>((const bf16_t*)src, ld, k_col, v_col, slots, (bf16_t*)keys, (bf16_t*)values,
                                                    kv_heads, key_dim, value_dim, page_size);
  else if (dtype == TW_DTYPE_F32)
    kv_store_kernel<float><<<n, 128, 0, stream>>>((const float*)src, ld, k_col, v_col, slots, (float*)keys, (float*)values,
                                                  kv_heads, key_dim, value_dim, page_size);
  else return TW_ERR_BAD_ARGUMENT;
  return TW_LAUNCH_RESULT();
}
