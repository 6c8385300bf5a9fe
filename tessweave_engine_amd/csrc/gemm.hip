// Linear layers: C[M, N] = A[M, K] * W[N, K]^T (+ bias[N]) (+ residual[M, N]).
// A and W are both contiguous along K (the checkpoint's [out, in] layout), in
// float32 or bfloat16; accumulation is float32 on the MFMA units (true float32
// MFMA for float32 inputs, no reduced-precision matrix mode). The kernels:
//   gemm_tiled      - many rows (prompt portions): LDS-staged 32x32 MFMA tiles
//   gemm_skinny_lds - few rows (decode): weights streamed once from HBM straight
//                     into 16x16 MFMA fragments, split over K when N is small
//   gemm_stream_cu  - 17 to 64 rows: the same with one workgroup per CU
//   gemm_narrow     - up to 16 rows, few columns: a workgroup has the whole of K
//   gemm_generic    - any K (rows not 16-byte aligned): one output per thread
//
// Weight layouts. Row-major [N][K] as in the checkpoint, or SHUFFLED (an exact permutation,
// zero padded): blocks of 16 rows x 4 sixteen-byte chunks stored in the order the MFMA units
// read them, [N/16][K/(4*EPF)][chunk 0..3][row 0..15][EPF]. Element (n, k) is at
//   ((n/16 * k_steps + (k/EPF)/4) * 64 + ((k/EPF)%4) * 16 + n%16) * EPF + k%EPF.
// A wave's load of one block is 1 KB of consecutive memory: the decode kernel streams weights
// as whole cache lines past the caches (non-temporal), the tiled kernel copies blocks.
//
// GLU (gated linear unit) form: the N rows of W are the gate and up projections interleaved in
// blocks of 16 rows (gate rows 16j.., then up rows 16j.., for j = 0, 1, ...). The kernels form
// C[M, N/2][.., 16j + i] = silu(gate_j[i]) * up_j[i] in their epilogues, in float32 from the
// accumulators, so the [M, N] intermediate never reaches memory.
#include <type_traits>
#include <math.h>

#include "tw_common.h"
#include "gemm_shared.h"

// element offset of (row n, 16-byte chunk c) in the shuffled layout
__device__ __forceinline__ size_t tw_shuffled_chunk(int n, int c, int k_steps, int epf) {
  return ((size_t)((size_t)(n >> 4) * k_steps + (c >> 2)) * 64 + (c & 3) * 16 + (n & 15)) * epf;
}

// =====================================================================================
// A norm that travels with its product (decode steps of up to 16 rows). y = W (x rinv w), rinv = 1 / sqrt(mean(x^2) + eps), is
// rinv (W (x w)): whoever forms x last (the epilogue of a product that has the whole of K, EndLeave below) leaves the rows x w
// rounded once, as a norm rounds x rinv w, and of every 16 columns the sum of x^2; whoever multiplies those rows adds the sums up,
// always in one order, while its first weights are on their way, and multiplies its float32 sums by rinv. No norm kernel stands
// between two products then: such a kernel is a few rows' latency and a launch, 3 to 4 us a time.
// =====================================================================================
struct RowNorms {
  const float* sums;          // [M][count]: sums of squares of 16 columns each; count a multiple of 4, up to TW_NORM_MAX_SUMS
  int count;
  float width, eps;
};
struct RowsAsTheyAre {};
struct RowsRounded {};        // A holds float32 rows, rounded to the product's type as they are read
#define TW_NORM_MAX_SUMS 256

// THREADS / 16 lanes a row add its sums up: `request` asks for all of them (clamped, so that no load has a predicate), `finish`
// leaves 1 / sqrt(mean + eps) of row i in rinv[i] (a barrier must lie between it and the readers).
template <int THREADS>
struct RowNormLoads {
  static constexpr int LANES = THREADS / 16, LOADS = TW_NORM_MAX_SUMS / 4 / LANES;
  f32x4 v[LOADS];
  __device__ __forceinline__ void request(const RowNorms& n, int M) {
    const int row = min((int)threadIdx.x / LANES, M - 1), l = threadIdx.x % LANES, last = n.count / 4 - 1;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) v[i] = *reinterpret_cast<const f32x4*>(n.sums + (size_t)row * n.count + min(l + i * LANES, last) * 4);
  }
  __device__ __forceinline__ void finish(const RowNorms& n, float* rinv) const {
    const int l = threadIdx.x % LANES;
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) s += l + i * LANES < n.count / 4 ? (v[i][0] + v[i][1]) + (v[i][2] + v[i][3]) : 0.f;
#pragma unroll
    for (int o = LANES / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, TW_WAVE);
    if (l == 0) rinv[threadIdx.x / LANES] = 1.0f / sqrtf(s / n.width + n.eps);
  }
};

// =====================================================================================
// Skinny kernel (M <= 16*MT rows), workgroup-cooperative. The WAVES (4, or 2) waves of a workgroup own
// neighbouring tiles of 16 output columns and the SAME K range. Per stage of U
// MFMA steps the workgroup copies the activations' K slice [16*MT rows][U*64 B]
// to LDS once (instead of every wave reading it from L2); each wave streams its
// own 16 weight rows from global memory into registers (every weight byte is read by exactly
// one wave). Two stages of weights in flight. splits == 1: the epilogue runs here. splits > 1: float32
// partial sums go to partial[split][M][N] and splitk_reduce_kernel (or the caller's next
// kernel) adds them, always in the same order, so results do not depend on timing.
// =====================================================================================
#define TW_XROW(U) ((U) * 64 + 32)          /* LDS bytes per activation row of a stage, padded: 32 * an odd number (see tw_lds_swz4) */

// PARTIAL: always write float32 partial sums partial[split][M][N] (splits >= 1), no epilogue.
// SHUF: W is in the shuffled layout (ldw = its k_steps): every weight load is 1 KB of consecutive
// memory, needs no predicate (the layout is zero padded) and bypasses the caches.
// GLU (splits == 1 only): the workgroup's tiles are gate, up(, gate, up); C gets half as many columns.
// WAVES = 2 halves the workgroups' size and doubles their number: used where that spreads them more
// evenly over the CUs (the kernel's time is that of the fullest CU).
// In: RowNorms (MT == 1) where A's rows are to be multiplied by their norms' factors, see above.
template <typename T, typename OutT, int MT, int U, int WAVES, bool PARTIAL, bool SHUF, bool GLU, class In = RowsAsTheyAre>
__global__ __launch_bounds__(WAVES * 64) void gemm_skinny_lds_kernel(const T* __restrict__ A, long lda,
                                                              const T* __restrict__ W, long ldw,
                                                              const float* __restrict__ bias,
                                                              const float* residual, long ldr, OutT* C,
                                                              long ldc, float* __restrict__ partial, int M,
                                                              int N, int K, int n_groups, int splits, In norms) {
  typedef typename Elem<T>::Frag Frag;
  constexpr bool NORMED = std::is_same<In, RowNorms>::value;
  static_assert(!NORMED || MT == 1, "norms travel with up to 16 rows");
  constexpr int EPF = Elem<T>::kPerFrag;
  constexpr int XROW = TW_XROW(U);
  constexpr int XSTAGE = MT * 16 * XROW;
  constexpr int THREADS = WAVES * 64;
  constexpr int XLOADS = MT * U / WAVES;               // activation fragments per thread per stage
  static_assert(U % 4 == 0 && (WAVES == 4 || WAVES == 2), "a stage is copied by all threads in whole rounds");
  __shared__ __attribute__((aligned(16))) char lds[2 * XSTAGE];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int group = blockIdx.x % n_groups, split = blockIdx.x / n_groups;
  const int r = lane & 15, g = lane >> 4;
  const int n0 = group * (16 * WAVES) + wave * 16;

  const int chunks = K / EPF;
  const int steps = (chunks + 3) / 4;
  const int steps_per_split = (steps + splits - 1) / splits;
  const int step_begin = split * steps_per_split;
  const int step_end = min(steps, step_begin + steps_per_split);
  const int n_stages = step_end > step_begin ? (step_end - step_begin + U - 1) / U : 0;

  f32x4 acc[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) acc[mt] = f32x4{0.f, 0.f, 0.f, 0.f};

  const T* w_row = SHUF ? W + ((size_t)min(n0 / 16, (N + 15) / 16 - 1) * ldw * 64 + lane) * EPF
                        : W + (size_t)min(n0 + r, N - 1) * ldw;
  // this thread's share of the activation slice: fragment f = i*THREADS + tid -> (row f / (4U), chunk f % (4U))
  const T* x_src[XLOADS];
  int x_dst[XLOADS], x_chunk[XLOADS];
#pragma unroll
  for (int i = 0; i < XLOADS; ++i) {
    const int f = i * THREADS + tid, row = f / (4 * U), c = f % (4 * U);
    x_src[i] = A + (size_t)min(row, M - 1) * lda;
    x_chunk[i] = c;
    x_dst[i] = row * XROW + c * 16;
  }

  // Loads carry no predicate: addresses are clamped to the last valid step or chunk (always inside
  // the matrix), and activation chunks outside this workgroup's K range are replaced by zeros on
  // their way to LDS, so whatever weight was read beside them adds nothing. Without conditional
  // loads the compiler's wait counts are exact, which the order of the pipeline below relies on.
  Frag wf[2][U], xg[XLOADS];
  const int chunk_end = min(step_end * 4, chunks);
  auto load_w = [&](const int buf, int s0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (SHUF)
        wf[buf][u] = tw_load_frag_stream(w_row + (size_t)min(s0 + u, steps - 1) * 64 * EPF);
      else
        wf[buf][u] = tw_load_frag(w_row + (size_t)min((s0 + u) * 4 + g, chunks - 1) * EPF);
    }
  };
  auto load_x = [&](int s0) {
#pragma unroll
    for (int i = 0; i < XLOADS; ++i)
      xg[i] = tw_load_frag(x_src[i] + (size_t)min(s0 * 4 + x_chunk[i], chunks - 1) * EPF);
  };
  auto store_x = [&](int buf, int s0) {
#pragma unroll
    for (int i = 0; i < XLOADS; ++i)
      *reinterpret_cast<Frag*>(lds + buf * XSTAGE + x_dst[i]) = s0 * 4 + x_chunk[i] < chunk_end ? xg[i] : Elem<T>::zero();
  };
  auto multiply = [&](const int buf) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const Frag xf = *reinterpret_cast<const Frag*>(lds + buf * XSTAGE + (mt * 16 + r) * XROW + (u * 4 + g) * 16);
        tw_mma16(acc[mt], wf[buf][u], xf);
      }
  };
  // Two stages i, i + 1 (i even: stage i has its weights in register set 0 and its activations in
  // LDS buffer 0). Per stage: request the next stage's activations, multiply this stage, request
  // the weights of the stage after next into the registers just used, then move the activations to
  // LDS. Loads return in order, so the wait for the activations leaves the newest weight loads in
  // flight: a wave that stalls there has one to two stages of weights on their way.
  auto stage_pair = [&](int i, auto more1, auto more2, auto more3) {
    const int s0 = step_begin + i * U;
    if (more1) load_x(s0 + U);
    __builtin_amdgcn_sched_barrier(0);           // the compiler would sink the loads below the waits
    multiply(0);
    if (more2) load_w(0, s0 + 2 * U);
    __builtin_amdgcn_sched_barrier(0);
    if (more1) store_x(1, s0 + U);
    __syncthreads();
    if (!more1) return;
    if (more2) load_x(s0 + 2 * U);
    __builtin_amdgcn_sched_barrier(0);
    multiply(1);
    if (more3) load_w(1, s0 + 3 * U);
    __builtin_amdgcn_sched_barrier(0);
    if (more2) store_x(0, s0 + 2 * U);
    __syncthreads();
  };

  __shared__ float rinv[16];
  RowNormLoads<THREADS> norm_sums;
  if constexpr (NORMED) norm_sums.request(norms, M);
  if (n_stages > 0) {
    load_x(step_begin);
    load_w(0, step_begin);
    // (of two waves, whose lanes hold 32 registers of sums, the second stage's weights go out behind the sums: with both it takes 138
    // registers, and three waves a SIMD run instead of four)
    if constexpr (NORMED && WAVES == 2) {
      __builtin_amdgcn_sched_barrier(0);
      norm_sums.finish(norms, rinv);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (n_stages > 1) load_w(1, step_begin + U);
    if constexpr (NORMED && WAVES != 2) {
      __builtin_amdgcn_sched_barrier(0);
      norm_sums.finish(norms, rinv);
    }
    store_x(0, step_begin);
    __syncthreads();
    int i = 0;
    for (; i + 3 < n_stages; i += 2) stage_pair(i, std::true_type{}, std::true_type{}, std::true_type{});
    for (; i < n_stages; i += 2) stage_pair(i, i + 1 < n_stages, i + 2 < n_stages, i + 3 < n_stages);
  }

  // acc[mt][j] = sum_k W[n0 + 4g + j][k] * A[16 mt + r][k]
  if constexpr (NORMED) {                                      // (a workgroup without a K range has sums of zero: any factor does)
    const float f = n_stages > 0 ? rinv[r] : 1.f;
    acc[0] = f32x4{acc[0][0] * f, acc[0][1] * f, acc[0][2] * f, acc[0][3] * f};
  }
  if (GLU) {
    // the waves swap their tiles through LDS (every wave is past its last LDS read: the loop
    // ends with a barrier), then each thread forms outputs from a (gate, up) pair
    constexpr int GROW = 17;                                  // floats per staged row, padded
    static_assert(WAVES * MT * 16 * GROW * 4 <= 2 * XSTAGE, "the GLU exchange fits the pipeline's LDS");
    float* ex = reinterpret_cast<float*>(lds);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int col = n0 + 4 * g + j;
        ex[(wave * MT * 16 + mt * 16 + r) * GROW + 4 * g + j] = acc[mt][j] + (bias && col < N ? bias[col] : 0.f);
      }
    __syncthreads();
    constexpr int OUT_COLS = 8 * WAVES;                       // output columns of the workgroup
    for (int o = tid; o < MT * 16 * OUT_COLS; o += THREADS) {
      const int row = o / OUT_COLS, c = o % OUT_COLS, pair = c >> 4, i = c & 15;
      const int col = group * OUT_COLS + c;                   // output column
      if (row >= M || col >= N / 2) continue;
      const float gv = ex[((2 * pair) * MT * 16 + row) * GROW + i];
      const float uv = ex[((2 * pair + 1) * MT * 16 + row) * GROW + i];
      C[(size_t)row * ldc + col] = tw_from_float<OutT>(tw_glu(gv, uv, ldr));
    }
    return;
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int row = mt * 16 + r;
    if (row >= M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int col = n0 + 4 * g + j;
      if (col >= N) continue;
      if (PARTIAL || splits > 1) {
        partial[((size_t)split * M + row) * N + col] = acc[mt][j];
      } else {
        float v = acc[mt][j] + (bias ? bias[col] : 0.f);
        if (residual) v += residual[(size_t)row * ldr + col];
        C[(size_t)row * ldc + col] = tw_from_float<OutT>(v);
      }
    }
  }
}

// =====================================================================================
// Streaming kernel with ONE workgroup per CU (shuffled weights; the launcher uses it above 16 rows).
//
// The kernel above deals whole workgroups of four column tiles to the CUs, a few hundred of them, and every
// workgroup stages its own copy of the activations, which at 64 rows are as many bytes from L2 as the
// weights are from HBM. Here the grid is one workgroup per CU and the 16-column tiles (or gate/up pairs
// of them) are dealt to the workgroups as evenly as whole tiles allow, K ranges first where one range
// would leave CUs idle. A workgroup is TW_CU_WAVES waves: up to TW_CU_MAX_COMPUTE of them take one tile
// each per round (several rounds if the workgroup has more tiles), the others only help with the copies.
// EVERY wave copies its share of the activations' K slice of each stage from global memory straight into
// LDS (`global_load_lds_dwordx4`: no staging registers, no LDS write instructions, one copy per CU instead
// of one per four tiles; the copies of a stage are dealt to all waves because a wave's copies go out one
// after the other). Compute waves stream their own 16 weight rows into registers, TW_CU_NBUF - 1 stages
// ahead, and multiply out of LDS.
//
// LDS layout of a stage: MT * U blocks of 1 KB, block (mt, u) = rows 16 mt .. 16 mt + 15, the four
// 16-byte chunks of k-step u. Slot l of a block holds row l / 4, chunk (l % 4) ^ (row / 4 % 4): four
// neighbouring lanes fetch 64 consecutive bytes, and the 16 lanes that read one chunk of 16 rows meet
// 16 different bank groups. Chunks outside the workgroup's K range are copied from a chunk of zeros,
// so whatever weight is read beside them adds nothing; rows past M are clamped (never stored).
// =====================================================================================
#ifndef TW_CU_NBUF
#define TW_CU_NBUF 4
#endif
#ifndef TW_CU_U
#define TW_CU_U 4
#endif
#ifndef TW_CU_WAVES
#define TW_CU_WAVES 16
#endif
#ifndef TW_CU_MAX_COMPUTE
#define TW_CU_MAX_COMPUTE 14
#endif
/* more than half a CU's LDS (never two of these workgroups on one CU), room for the stages of 64 rows, and 1 KB
   where copies that a wave has no block for are dumped */
#define TW_CU_STAGES_BYTES (TW_CU_NBUF * TW_CU_U * 4 * 1024)
#define TW_CU_LDS_BYTES ((TW_CU_STAGES_BYTES + 1024) > 84 * 1024 ? (TW_CU_STAGES_BYTES + 1024) : 84 * 1024)

__device__ __attribute__((aligned(16))) const uint32_t tw_zero_chunk[4] = {0u, 0u, 0u, 0u};

typedef __attribute__((address_space(3))) void* tw_lds_dst;

// PARTIAL: the K ranges' sums go to `partial` (always so with more than one range), otherwise the finished rows to C. WIDE: 16 bytes at a
// time, to partial or to C, where the launcher finds that columns, strides and addresses allow it. (Forms of their own: with all
// stores in one kernel, chosen as it runs, four row tiles spilled ten registers: 64 rows x 152,064 x 3,584 208 us instead of 185,
// x 3,584 x 18,944 37.9 instead of 34.5, x 2,048 x 2,048 13.0 instead of 10.2.)
template <typename T, typename OutT, int MT, bool PARTIAL, bool GLU, bool WIDE>
__global__ __launch_bounds__(TW_CU_WAVES * 64) void gemm_stream_cu_kernel(
    const T* __restrict__ A, long lda, const T* __restrict__ W, long ldw, const float* __restrict__ bias,
    const float* residual, long ldr, OutT* C, long ldc, float* __restrict__ partial, int M, int N, int K,
    int splits, int wgs_per_split, int compute_waves, int steps_per_split) {
  typedef typename Elem<T>::Frag Frag;
  constexpr int EPF = Elem<T>::kPerFrag, U = TW_CU_U, NBUF = TW_CU_NBUF, WAVES = TW_CU_WAVES;
  constexpr int BLOCKS = MT * U;                       // 1 KB blocks of activations per stage
  constexpr int XSTAGE = BLOCKS * 1024;
  constexpr int XD = (BLOCKS + WAVES - 1) / WAVES;     // copies per wave and stage
  static_assert(NBUF * XSTAGE + 1024 <= TW_CU_LDS_BYTES && NBUF >= 3, "stage layout");
  extern __shared__ __attribute__((aligned(16))) char lds[];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = blockIdx.x % wgs_per_split, split = blockIdx.x / wgs_per_split;
  // this workgroup's tiles of 16 columns: [t0, t1), whole gate/up pairs for GLU
  constexpr int UW = GLU ? 2 : 1;
  const long units = GLU ? N / 32 : (N + 15) / 16;
  const int t0 = (int)(units * j / wgs_per_split) * UW, t1 = (int)(units * (j + 1) / wgs_per_split) * UW;
  const int last_block = (N + 15) / 16 - 1;
  // this workgroup's K range, in k-steps of four 16-byte chunks
  const int chunks = K / EPF, steps = (chunks + 3) / 4;
  const int step_begin = min(steps, split * steps_per_split), step_end = min(steps, step_begin + steps_per_split);
  const int n_stages = (step_end - step_begin + U - 1) / U;
  const int chunk_end = min(step_end * 4, chunks);
  const int r = lane & 15, g = lane >> 4;

#define TW_CU_WAIT(n) asm volatile("s_waitcnt vmcnt(" #n ")" ::: "memory")
#define TW_CU_BARRIER()                   \
  do {                                    \
    __builtin_amdgcn_s_barrier();         \
    asm volatile("" ::: "memory");        \
  } while (0)
  // Wait until at most `n` of this wave's loads and copies are in flight (they finish in the order they
  // were issued). The count is an immediate of the instruction, hence the cases.
  auto wait_for = [&](auto n) {
    constexpr int N_ = decltype(n)::value;
    if constexpr (N_ == 2) TW_CU_WAIT(2);
    else if constexpr (N_ == 4) TW_CU_WAIT(4);
    else if constexpr (N_ == 6) TW_CU_WAIT(6);
    else if constexpr (N_ == 8) TW_CU_WAIT(8);
    else if constexpr (N_ == 10) TW_CU_WAIT(10);
    else if constexpr (N_ == 12) TW_CU_WAIT(12);
    else if constexpr (N_ == 14) TW_CU_WAIT(14);
    else if constexpr (N_ == 16) TW_CU_WAIT(16);
    else if constexpr (N_ == 18) TW_CU_WAIT(18);
    else if constexpr (N_ == 20) TW_CU_WAIT(20);
    else if constexpr (N_ == 24) TW_CU_WAIT(24);
    else TW_CU_WAIT(0);
  };

  // ---- this wave's share of the activation copies: blocks wave, wave + WAVES, ... of every stage ----
  const int row16 = lane >> 2, cswz = (lane & 3) ^ tw_lds_swz4(row16);
  const T* x_row[XD];
  int x_chunk[XD], x_dst[XD];
#pragma unroll
  for (int q = 0; q < XD; ++q) {
    const int b = wave + WAVES * q;
    const bool mine = b < BLOCKS;                          // else: a copy of zeros into the dump area
    const int mt = mine ? b / U : 0, u = mine ? b % U : 0;
    x_row[q] = A + (size_t)min(mt * 16 + row16, M - 1) * lda;
    x_chunk[q] = mine ? u * 4 + cswz : (1 << 28);          // (a chunk far outside every K range)
    x_dst[q] = mine ? b * 1024 : -1;
  }
  auto copy_x = [&](int stage, const int buf) {
    const int c0 = (step_begin + stage * U) * 4;
#pragma unroll
    for (int q = 0; q < XD; ++q) {
      const int c = c0 + x_chunk[q];
      const T* src = c < chunk_end ? x_row[q] + (size_t)c * EPF : reinterpret_cast<const T*>(tw_zero_chunk);
      char* dst = x_dst[q] >= 0 ? lds + buf * XSTAGE + x_dst[q] : lds + NBUF * XSTAGE;
      // (the cast matters: handed a pointer whose type depends on a template parameter, the host pass drops
      // the kernel's definition without a word and the library no longer links)
      __builtin_amdgcn_global_load_lds((const void*)src, (tw_lds_dst)dst, 16, 0, 0);
    }
  };

  for (int first = t0; first < t1; first += compute_waves) {       // rounds: the same for every wave
    const int tile = first + wave;
    if (wave >= compute_waves || tile >= t1) {
      // ---- a wave without a tile in this round: copies only ------------------------------------------
      // stage i's copies have landed once at most the NBUF - 2 newer stages' are in flight
#pragma unroll
      for (int b = 0; b < NBUF - 1; ++b) copy_x(b, b);
      auto stage_h = [&](int i, const int buf) {
        wait_for(std::integral_constant<int, XD * (NBUF - 2)>{});
        TW_CU_BARRIER();                                    // stage i is there for every wave; every wave is past stage i - 1
        copy_x(i + NBUF - 1, (buf + NBUF - 1) % NBUF);      // into the stage that was read last (past the end: zeros)
      };
      int i = 0;
      for (; i + NBUF <= n_stages; i += NBUF) {
#pragma unroll
        for (int b = 0; b < NBUF; ++b) stage_h(i + b, b);
      }
#pragma unroll
      for (int b = 0; b < NBUF; ++b)
        if (i + b < n_stages) stage_h(i + b, b);
      TW_CU_WAIT(0);                                        // no copy lands after the loop
      TW_CU_BARRIER();                                      // (E1)
      if (GLU) {
        TW_CU_BARRIER();                                    // (E2)
        TW_CU_BARRIER();                                    // (E3)
      }
      continue;
    }
    // ---- a wave with a tile of 16 columns --------------------------------------------------------------
    const T* w_row = W + ((size_t)min(tile, last_block) * ldw * 64 + lane) * EPF + (size_t)step_begin * 64 * EPF;
    const int slot = (r * 4 + (g ^ tw_lds_swz4(r))) * 16;
    f32x4 acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
    Frag wf[NBUF][U];
    const int last_step = steps - 1 - step_begin;           // (relative to this workgroup's first k-step)
    auto load_w = [&](int stage, const int buf) {
#pragma unroll
      for (int u = 0; u < U; ++u)
        wf[buf][u] = tw_load_frag_stream(w_row + (size_t)min(stage * U + u, last_step) * (64 * EPF));
    };
    auto multiply = [&](const int buf) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        Frag xf[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          xf[mt] = *reinterpret_cast<const Frag*>(lds + buf * XSTAGE + (mt * U + u) * 1024 + slot);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) tw_mma16(acc[mt], wf[buf][u], xf[mt]);
        // one k-step's fragments at a time: the other waves of the CU cover the LDS latency, and the registers
        // that reading a whole stage ahead would take are what the weights in flight need
        if (MT > 1) __builtin_amdgcn_sched_barrier(0);
      }
    };
    // Stage i: wait for this wave's copies of stage i, meet the others (stage i's activations are in LDS,
    // stage i - 1's are read), ask for the weights and copies of stage i + NBUF - 1, multiply. In the main
    // loop every stage issues U loads and XD copies, so "the NBUF - 2 newer stages may be in flight" is a
    // count; near the end the stages after the last one issue copies (of zeros) but no loads.
    auto stage_c = [&](int i, const int buf, auto main) {
      static_assert(NBUF == 4 || NBUF == 3, "the cases below");
      const int newer = main ? NBUF - 2 : min(max(n_stages - 1 - i, 0), NBUF - 2);   // newer stages with loads
      if (newer == NBUF - 2) wait_for(std::integral_constant<int, (U + XD) * (NBUF - 2)>{});
      else if (newer == 1) wait_for(std::integral_constant<int, U + XD * (NBUF - 2)>{});
      else wait_for(std::integral_constant<int, XD * (NBUF - 2)>{});
      TW_CU_BARRIER();
      if (main || i + NBUF - 1 < n_stages) load_w(i + NBUF - 1, (buf + NBUF - 1) % NBUF);
      copy_x(i + NBUF - 1, (buf + NBUF - 1) % NBUF);
      __builtin_amdgcn_sched_barrier(0);                    // (loads and copies go out before the multiplies, not after)
      multiply(buf);
    };
#pragma unroll
    for (int b = 0; b < NBUF - 1; ++b) {
      if (b < n_stages) load_w(b, b);
      copy_x(b, b);
    }
    int i = 0;
    if (n_stages >= NBUF - 1)                               // (else the prologue issued fewer loads than the counts assume)
      for (; i + 2 * NBUF - 1 <= n_stages; i += NBUF) {     // every load of these stages names a stage that exists
#pragma unroll
        for (int b = 0; b < NBUF; ++b) stage_c(i + b, b, std::true_type{});
      }
    for (; i < n_stages; i += NBUF) {
#pragma unroll
      for (int b = 0; b < NBUF; ++b)
        if (i + b < n_stages) stage_c(i + b, b, std::false_type{});
    }
    TW_CU_WAIT(0);                                          // no copy lands after the loop
    TW_CU_BARRIER();                                        // (E1) every wave is past its last LDS read

    // acc[mt][e] = sum_k W[16 tile + 4g + e][k] * A[16 mt + r][k]
    const int col0 = tile * 16 + 4 * g;
    if (GLU) {
      // the two waves of a gate/up pair swap their tiles through LDS; each thread then forms outputs
      constexpr int GROW = 17;
      float* ex = reinterpret_cast<float*>(lds);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          ex[((wave * MT + mt) * 16 + r) * GROW + 4 * g + e] = acc[mt][e] + (bias && col0 + e < N ? bias[col0 + e] : 0.f);
      TW_CU_BARRIER();                                      // (E2)
      {
        const int gate_wave = wave & ~1;
        const int out0 = ((first + gate_wave) >> 1) * 16;   // first output column of the pair
        for (int o = (wave & 1) * 64 + lane; o < MT * 16 * 16; o += 128) {
          const int row = o >> 4, c = o & 15;
          if (row >= M || out0 + c >= N / 2) continue;
          const float gv = ex[(gate_wave * MT * 16 + row) * GROW + c];
          const float uv = ex[((gate_wave + 1) * MT * 16 + row) * GROW + c];
          C[(size_t)row * ldc + out0 + c] = tw_from_float<OutT>(tw_glu(gv, uv, ldr));
        }
      }
      TW_CU_WAIT(0);
      TW_CU_BARRIER();                                      // (E3) the exchange area is free for the next round's copies
      continue;
    }
    {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const int row = mt * 16 + r;
        if (row >= M || col0 >= N) continue;
        if constexpr (PARTIAL) {
          float* dst = partial + ((size_t)split * M + row) * N + col0;
          if constexpr (WIDE) {
            *reinterpret_cast<f32x4*>(dst) = acc[mt];
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (col0 + e < N) dst[e] = acc[mt][e];
          }
        } else if constexpr (WIDE) {
          // (whole groups of four columns, 64 bytes a row together: the float32 logits of a head of 152,064 x 3,584 at 64 rows
          // 185 us, stored one by one 196; at 32 rows 174 and 177)
          f32x4 v = acc[mt];
          if (bias) v = v + *reinterpret_cast<const f32x4*>(bias + col0);
          if (residual) v = v + *reinterpret_cast<const f32x4*>(residual + (size_t)row * ldr + col0);
          OutT* dst = C + (size_t)row * ldc + col0;
          if (sizeof(OutT) == 4) {
            *reinterpret_cast<f32x4*>(dst) = v;
          } else {
            OutT packed[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) packed[e] = tw_from_float<OutT>(v[e]);
            *reinterpret_cast<uint64_t*>(dst) = *reinterpret_cast<const uint64_t*>(packed);
          }
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if (col0 + e >= N) continue;
            float v = acc[mt][e] + (bias ? bias[col0 + e] : 0.f);
            if (residual) v += residual[(size_t)row * ldr + col0 + e];
            C[(size_t)row * ldc + col0 + e] = tw_from_float<OutT>(v);
          }
        }
      }
    }
    TW_CU_WAIT(0);        // stores and loads are counted together but finish apart: start the next round from zero
  }
#undef TW_CU_WAIT
#undef TW_CU_BARRIER
}

// =====================================================================================
// Few rows against a matrix with few columns (M <= 16, shuffled weights): one workgroup owns 16 output
// columns (GLU: a gate and an up tile of 16) over the WHOLE of K. Its waves take k-steps in turn (wave w:
// steps w, w + WAVES, ..., so that the workgroup reads consecutive kilobytes), weights and activations
// straight into MFMA fragments, two batches of U steps in flight; the waves' float32 sums meet in LDS, are
// added in the waves' order, and the epilogue runs here: no partial sums in memory and no second kernel.
// Bound by the weights' latency and bytes, and by the activations that every workgroup reads from L2 (with K
// above 4096 these cost more than they save).
// =====================================================================================
// HALVES: the gated form with eight gate and eight up rows a workgroup, one fragment of both (each eight weight rows of a fragment are a
// cache line): where pairs of 16 leave CUs idle, or a second round nearly empty (see narrow_halves). The same sums in the same order.
// ACT: the residual's stride names an activation (a form of its own: its code in the plain form cost that 0.15 us a launch).
// In: RowNorms where A's rows are to be multiplied by their norms' factors.
// End: what the epilogue does with a finished element.
//   EndPlain   C = sum (+ bias) (+ residual), or act(sum + bias).
//   EndLeave   C (float32, the residual stream) = sum + bias + residual, and beside it what a norm that travels needs: the rows times
//              the next norm's weight in T (times a second weight too where two norms read the stream), and each 16 columns' sum of
//              squares. AFTER: the stream itself is such a normed row, C = alpha * residual * rinv * before_weight + scale * (sum + bias).
//   EndRotate  the packed product of queries, keys and values: q and k are rotated, q goes to C, k and v to the cache's pages, and what lies behind
//              them (another mixer's columns) to C. A
//              workgroup's 16 columns are then eight of a head's first rotated half and the eight they turn with (each eight weight
//              rows of a fragment are a cache line, so the loads are as wide as before), so that no other kernel has to bring the
//              two halves together: it was 2.5 to 4 us behind every such product.
struct EndPlain {};
template <bool AFTER_NORM>
struct EndLeave {
  static constexpr bool AFTER = AFTER_NORM;
  const float *weight, *weight2;       // [N]; weight2 may be null
  void *rows, *rows2;                  // [M][N] in the input type
  float* sums;                         // [M][N / 16]
  RowNorms before;                     // AFTER: of the residual's rows (sums null: they are as they are)
  const float *before_weight, *scale;  // AFTER: [N]; scale may be null
  float alpha;
};
struct EndRotate {
  const float *cos_t, *sin_t;          // [M][rot / 2]
  const int* slots;
  void *keys, *values;
  int q_heads, kv_heads, head_dim, rot, page_size, write_cache, adjacent;
};
// EndTokenGate  C = gelu_tanh(sum + bias) * table[token of the row][offset + column], as token_gate_kernel: with rows rounded as they are read the
//              launches in front of and behind a layer's small product from the stream to its token input go (128 x 2048, one row, in captured
//              steps: 3.5 us a layer).
template <typename T>
struct EndTokenGate {
  const T* table; long ld;
  const int *ids, *feed;
  int n_feed, vocab, offset;
};
template <class End> struct IsTokenGate { static constexpr bool value = false; };
template <typename T> struct IsTokenGate<EndTokenGate<T>> { static constexpr bool value = true; };
template <class End> struct IsLeave { static constexpr bool value = false, after = false; };
template <bool A> struct IsLeave<EndLeave<A>> { static constexpr bool value = true, after = A; };

template <typename T, typename OutT, int WAVES, bool GATED, bool ACT = false, class In = RowsAsTheyAre, class End = EndPlain, bool HALVES = false>
__global__ __launch_bounds__(WAVES * 64) void gemm_narrow_kernel(const T* __restrict__ A, long lda,
                                                                 const T* __restrict__ W, long ldw,
                                                                 const float* __restrict__ bias,
                                                                 const float* residual, long ldr, OutT* C, long ldc,
                                                                 int M, int N, int K, In norms, End end) {
  typedef typename Elem<T>::Frag Frag;
  constexpr bool NORMED = std::is_same<In, RowNorms>::value, ROTATE = std::is_same<End, EndRotate>::value;
  constexpr bool LEAVE = IsLeave<End>::value, AFTER = IsLeave<End>::after, TOKEN_GATE = IsTokenGate<End>::value;
  constexpr bool ROUND = std::is_same<In, RowsRounded>::value;
  static_assert(!(GATED && (ROTATE || LEAVE)) && (GATED || !HALVES), "the gated form finishes plain outputs");
  constexpr bool GLU = GATED && !HALVES;
  constexpr int EPF = Elem<T>::kPerFrag, U = 4, NT = GLU ? 2 : 1;
  __shared__ float sums[NT * WAVES * 16 * 16];
  __shared__ float rinv[16], rinv_before[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int chunks = K / EPF, steps = (chunks + 3) / 4;
  const int mine = steps > wave ? (steps - wave + WAVES - 1) / WAVES : 0;      // this wave's steps
  // the column of the workgroup's place i (of 16): consecutive, or eight and the eight that turn with them
  int first = blockIdx.x * 16, apart = 0;
  bool turns = false;                                                           // does this workgroup's part of a head turn?
  if constexpr (ROTATE) {
    const int per_head = end.head_dim / 16, head = blockIdx.x / per_head, t = blockIdx.x % per_head;
    turns = head < end.q_heads + end.kv_heads && t < end.rot / 16;
    if (turns && !end.adjacent) {
      first = head * end.head_dim + 8 * t;
      apart = end.rot / 2 - 8;
    }
  }
  auto column = [&](int i) { return first + i + (i >= 8 ? apart : 0); };
  const T* w_base = W + ((size_t)blockIdx.x * NT * ldw * 64 + lane) * EPF;
  if constexpr (ROTATE) {
    const int n = column(r);
    w_base = W + ((size_t)(n >> 4) * ldw * 64 + g * 16 + (n & 15)) * EPF;
  }
  // HALVES: place i of 16 is gate row i, or up row i - 8, of this workgroup's eight
  auto half_row = [&](int i) { return ((blockIdx.x & ~1) + (i >> 3)) * 16 + (blockIdx.x & 1) * 8 + (i & 7); };
  if constexpr (HALVES) {
    const int n = half_row(r);
    w_base = W + ((size_t)(n >> 4) * ldw * 64 + g * 16 + (n & 15)) * EPF;
  }
  const size_t w_tile = (size_t)ldw * 64 * EPF;
  const T* x_base = A + (size_t)min(r, M - 1) * (ROUND ? 0 : lda);               // (rows past M: never stored)
  const float* x_wide = reinterpret_cast<const float*>(A) + (size_t)min(r, M - 1) * lda;     // (ROUND)

  RowNormLoads<WAVES * 64> norm_sums, before_sums;
  if constexpr (NORMED) norm_sums.request(norms, M);
  if constexpr (AFTER) {
    if (end.before.sums) before_sums.request(end.before, M);
  }
  // Loads carry no predicate: steps are clamped to the last one and chunks to the last chunk, and activations
  // past either are replaced by zeros before the product.
  struct Wide { f32x4 part[EPF / 4]; };
  std::conditional_t<ROUND, Wide, Frag> xf[2][U];
  Frag wf[2][NT][U];
  auto load = [&](const int buf, int i0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = wave + (i0 + u) * WAVES;
#pragma unroll
      for (int t = 0; t < NT; ++t)
        wf[buf][t][u] = tw_load_frag_stream(w_base + t * w_tile + (size_t)min(s, steps - 1) * 64 * EPF);
      const size_t at = (size_t)min(s * 4 + g, chunks - 1) * EPF;
      if constexpr (ROUND) {
#pragma unroll
        for (int i = 0; i < EPF / 4; ++i) xf[buf][u].part[i] = *reinterpret_cast<const f32x4*>(x_wide + at + 4 * i);
      } else {
        xf[buf][u] = tw_load_frag(x_base + at);
      }
    }
  };
  auto fragment = [&](const int buf, int u) {
    if constexpr (ROUND) {
      Frag f;
#pragma unroll
      for (int i = 0; i < EPF; ++i) f[i] = tw_from_float<T>(xf[buf][u].part[i / 4][i % 4]);
      return f;
    } else {
      return xf[buf][u];
    }
  };
  f32x4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](const int buf, int i0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = wave + (i0 + u) * WAVES;
      const Frag x = s * 4 + g < chunks ? fragment(buf, u) : Elem<T>::zero();
#pragma unroll
      for (int t = 0; t < NT; ++t) tw_mma16(acc[t], wf[buf][t][u], x);
    }
  };
  load(0, 0);
  load(1, U);
  // what the epilogue adds, requested behind the first weights: thread t < 256 finishes row t / 16, column t % 16
  const int row = tid >> 4, c = tid & 15, col = ROTATE ? column(c) : blockIdx.x * 16 + c;
  const bool store = row < M && col < N / NT;                                   // (HALVES: a row's 16 places, N is a multiple of 32)
  float add[NT], res = 0.f;
#pragma unroll
  for (int t = 0; t < NT; ++t) add[t] = store && bias ? bias[ROTATE ? col : HALVES ? half_row(c) : (blockIdx.x * NT + t) * 16 + c] : 0.f;
  if (!GATED && store && residual) res = residual[(size_t)row * ldr + col];
  float weight = 0.f, weight2 = 0.f, before_weight = 0.f, scale = 1.f;
  if constexpr (LEAVE) {
    if (store) {
      weight = end.weight[col];
      if (end.weight2) weight2 = end.weight2[col];
      if constexpr (AFTER) {
        if (end.before.sums) before_weight = end.before_weight[col];
        if (end.scale) scale = end.scale[col];
      }
    }
  }
  float token_value = 0.f;
  if constexpr (TOKEN_GATE) {
    if (store) {
      int id = end.ids[row];
      if (id < 0) id = (end.feed && -1 - id < end.n_feed) ? end.feed[-1 - id] : 0;
      id = id < 0 ? 0 : (id >= end.vocab ? end.vocab - 1 : id);
      token_value = tw_to_float(end.table[(size_t)id * end.ld + end.offset + col]);
    }
  }
  float turn_cos = 1.f, turn_sin = 0.f;
  int slot = -1;
  if constexpr (ROTATE) {
    if (store) {
      if (end.write_cache) slot = end.slots[row];
      if (turns) {
        const int in_head = (end.adjacent ? col : first + (c & 7)) % end.head_dim;
        const int pair = end.adjacent ? in_head >> 1 : in_head;
        turn_cos = end.cos_t[(size_t)row * (end.rot / 2) + pair];
        turn_sin = end.sin_t[(size_t)row * (end.rot / 2) + pair];
      }
    }
  }
  if constexpr (NORMED || AFTER) __builtin_amdgcn_sched_barrier(0);
  if constexpr (NORMED) norm_sums.finish(norms, rinv);
  if constexpr (AFTER) {
    if (end.before.sums) before_sums.finish(end.before, rinv_before);
  }
  for (int i = 0; i < mine; i += 2 * U) {
    multiply(0, i);
    if (i + 2 * U < mine) load(0, i + 2 * U);
    __builtin_amdgcn_sched_barrier(0);           // the compiler would sink the loads below the waits
    if (i + U < mine) {
      multiply(1, i + U);
      if (i + 3 * U < mine) load(1, i + 3 * U);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // acc[t][j] = sum over this wave's steps of W[16 tile + 4g + j][k] * A[r][k]; columns swapped about by row,
  // so that the 16 rows of a write meet different banks
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int j = 0; j < 4; ++j) sums[((t * WAVES + wave) * 16 + r) * 16 + ((4 * g + j) ^ r)] = acc[t][j];
  __syncthreads();
  if (!store) return;                                          // (LEAVE, ROTATE: N is a multiple of 16, so a row's 16 lanes stay or go together)
  float v[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    v[t] = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) v[t] += sums[((t * WAVES + w) * 16 + row) * 16 + (c ^ row)];
    if constexpr (NORMED) v[t] *= rinv[row];
    v[t] += add[t];
  }
  if constexpr (GLU) {
    C[(size_t)row * ldc + col] = tw_from_float<OutT>(tw_glu(v[0], v[1], ldr));
  } else if constexpr (HALVES) {
    const float up = tw_dpp<TW_ROTATE_8>(v[0]);                // the row's other eight
    if (c < 8) C[(size_t)row * ldc + blockIdx.x * 8 + c] = tw_from_float<OutT>(tw_glu(v[0], up, ldr));
  } else if constexpr (LEAVE) {
    if constexpr (AFTER) {
      v[0] *= scale;
      if (end.before.sums) res = res * rinv_before[row] * before_weight;
      res *= end.alpha;
    }
    const float x = v[0] + res;
    C[(size_t)row * ldc + col] = x;
    static_cast<T*>(end.rows)[(size_t)row * N + col] = tw_from_float<T>(x * weight);
    if (end.weight2) static_cast<T*>(end.rows2)[(size_t)row * N + col] = tw_from_float<T>(x * weight2);
    float sq = x * x;                                          // over the row's 16 lanes
    sq += tw_dpp<TW_ROTATE_8>(sq);
    sq += tw_dpp<TW_ROTATE_4>(sq);
    sq += tw_dpp<TW_SWAP_2>(sq);
    sq += tw_dpp<TW_SWAP_1>(sq);
    if (c == 0) end.sums[(size_t)row * (N / 16) + blockIdx.x] = sq;
  } else if constexpr (ROTATE) {
    T out = tw_from_float<T>(v[0]);                            // what the product would have stored
    if (turns) {
      const float self = tw_to_float(out), other = end.adjacent ? tw_dpp<TW_SWAP_1>(self) : tw_dpp<TW_ROTATE_8>(self);
      const bool high = end.adjacent ? c & 1 : c >= 8;
      // (the products and sums of tw_rotate_pair in elementwise.hip, which round alike)
      const float a = __fmaf_rn(self, turn_cos, -__fmul_rn(other, turn_sin)), b = __fmaf_rn(self, turn_cos, __fmul_rn(other, turn_sin));
      out = tw_from_float<T>(high ? b : a);
    }
    const int head = blockIdx.x / (end.head_dim / 16), d = col - head * end.head_dim;
    if (head < end.q_heads || head >= end.q_heads + 2 * end.kv_heads) {
      C[(size_t)row * ldc + col] = out;
    } else if (slot >= 0) {
      const size_t page = slot / end.page_size;
      const int off = slot % end.page_size, kh = (head - end.q_heads) % end.kv_heads;
      if (head < end.q_heads + end.kv_heads)
        static_cast<T*>(end.keys)[((page * end.kv_heads + kh) * end.page_size + off) * end.head_dim + d] = out;
      else
        static_cast<T*>(end.values)[((page * end.kv_heads + kh) * end.head_dim + d) * end.page_size + off] = out;
    }
  } else if constexpr (TOKEN_GATE) {
    C[(size_t)row * ldc + col] = tw_from_float<OutT>(tw_gelu_tanh(v[0]) * token_value);
  } else {
    if constexpr (ACT) v[0] = tw_act(v[0], ldr);
    else if (residual) v[0] += res;
    C[(size_t)row * ldc + col] = tw_from_float<OutT>(v[0]);
  }
}

// =====================================================================================
// Generic kernel: any K. One thread per output element, float32 accumulation.
// =====================================================================================
template <typename T>
__device__ __forceinline__ float tw_generic_dot(const T* a, const T* W, long ldw, int col, int K, int shuffled) {
  constexpr int EPF = Elem<T>::kPerFrag;
  float v = 0.f;
  if (shuffled) {
    for (int k = 0; k < K; ++k)
      v = fmaf(tw_to_float(a[k]), tw_to_float(W[tw_shuffled_chunk(col, k / EPF, (int)ldw, EPF) + k % EPF]), v);
  } else {
    const T* w = W + (size_t)col * ldw;
    for (int k = 0; k < K; ++k) v = fmaf(tw_to_float(a[k]), tw_to_float(w[k]), v);
  }
  return v;
}

// glu: C has N / 2 columns (see the top of the file)
template <typename T, typename OutT>
__global__ void gemm_generic_kernel(const T* __restrict__ A, long lda, const T* __restrict__ W, long ldw,
                                    const float* __restrict__ bias, const float* residual, long ldr,
                                    OutT* C, long ldc, int M, int N, int K, int shuffled, int glu) {
  const int n_out = glu ? N / 2 : N;
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long)M * n_out) return;
  const int row = (int)(i / n_out), col = (int)(i % n_out);
  const T* a = A + (size_t)row * lda;
  if (glu) {
    const int gate = (col / 16) * 32 + col % 16, up = gate + 16;
    const float gv = tw_generic_dot(a, W, ldw, gate, K, shuffled) + (bias ? bias[gate] : 0.f);
    const float uv = tw_generic_dot(a, W, ldw, up, K, shuffled) + (bias ? bias[up] : 0.f);
    C[(size_t)row * ldc + col] = tw_from_float<OutT>(tw_glu(gv, uv, ldr));
    return;
  }
  float v = tw_generic_dot(a, W, ldw, col, K, shuffled);
  if (bias) v += bias[col];
  if (residual) v += residual[(size_t)row * ldr + col];
  C[(size_t)row * ldc + col] = tw_from_float<OutT>(v);
}

// =====================================================================================
// Host side
// =====================================================================================
// How many K ranges the skinny kernel uses for an [N, K] weight: as many as keep the workgroups at or
// under two for each of the 256 CUs (all resident at once and evenly spread: with 560 workgroups, a few
// over that, some CUs hold three and the kernel takes 10-15 % longer than with 504), each range at
// least 16 MFMA steps long. The choice depends on N and K only, never on the rows of a batch.
static int skinny_lds_splits(int N, int K, int epf) {
  const int groups = tw_div_up(N, 64);
  const int steps = tw_div_up(K / epf, 4);
  int splits = 512 / groups;
  const int max_by_k = steps / 16 > 0 ? steps / 16 : 1;
  if (splits > max_by_k) splits = max_by_k;
  if (splits > 16) splits = 16;
  return splits < 1 ? 1 : splits;
}

// ---- the kernel with one workgroup per CU: how its work is dealt ---------------------------------
static int cu_count() {
  static int cus = 0;                        // (the same for every device of a box)
  if (cus == 0) {
    int device = 0, n = 0;
    if (hipGetDevice(&device) == hipSuccess &&
        hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess && n > 0)
      cus = n;
    else
      cus = 256;
  }
  return cus;
}

struct CuPlan { int splits, wgs_per_split, compute_waves, steps_per_split; };

// K ranges, workgroups per range and compute waves per workgroup for MT row tiles against an [N, K] weight.
// Every candidate number of ranges is priced by the bytes its fullest CU streams (whole tiles, K ranges
// rounded up to whole stages), more where a CU would have few waves to keep loads in flight, plus the
// start of each round and, with more than one range, the partial sums written and read again; the
// cheapest wins. Depends on the row tiles, N and K only, never on the rows of a batch within a tile.
static CuPlan cu_plan(int MT, int N, int K, int epf, bool glu, bool may_split) {
  const int cus = cu_count();
  const int uw = glu ? 2 : 1;
  const long units = glu ? N / 32 : tw_div_up(N, 16);
  const int steps = tw_div_up(K / epf, 4);
  int most = may_split && !glu ? steps / 8 : 1;
  if (most > 16) most = 16;
  if (most < 1) most = 1;
  CuPlan best = {1, 1, 1, steps};
  double best_cost = 0;
  for (int want = 1; want <= most; ++want) {
    const int sps = tw_div_up(tw_div_up(steps, want), TW_CU_U) * TW_CU_U;
    const int splits = tw_div_up(steps, sps);
    if (splits != want && want > 1) continue;                       // (a count that rounding maps onto another one)
    long wgs = cus / splits;
    if (wgs > units) wgs = units;
    if (wgs < 1) wgs = 1;
    const long tiles = tw_div_up(units, wgs) * uw;                  // of the fullest workgroup
    const int rounds = tw_div_up(tiles, TW_CU_MAX_COMPUTE);
    int waves = tw_div_up(tiles, rounds);
    if (glu && waves % 2) ++waves;
    const double stream = (double)tiles * sps * 1024.0 / (waves >= 8 ? 1.0 : waves / 8.0);
    const double partial = splits > 1 || !glu ? 2.0 * splits * (16.0 * MT) * N * 4.0 / cus : 0.0;
    const double cost = stream + rounds * 37000.0 + (splits > 1 ? partial : 0.0);
    if (want == 1 || cost < best_cost) {
      best = {splits, (int)wgs, waves, sps};
      best_cost = cost;
    }
  }
  return best;
}

// Bytes of split-K scratch tw_linear can use for up to max_rows rows (0: none needed).
extern "C" long tw_linear_workspace_bytes(int dtype, int max_rows, int N, int K) {
  const int epf = dtype == TW_DTYPE_F32 ? 4 : 8;
  if (K % epf) return 0;
  const int rows = max_rows < 64 ? max_rows : 64;
  int splits = skinny_lds_splits(N, K, epf);
  for (int mt = 1; mt <= tw_div_up(rows, 16); ++mt) {          // whichever streaming kernel runs for these rows
    const int s = cu_plan(mt, N, K, epf, false, true).splits;
    if (s > splits) splits = s;
  }
  long bytes = splits > 1 ? (long)splits * rows * N * 4 : 0;
  if (max_rows > 64) {
    const long tiled = tw_tiled_workspace_bytes(dtype, max_rows, N, K);
    if (tiled > bytes) bytes = tiled;
  }
  return bytes;
}

// The fullest CU's share of `workgroups` spread over 256 CUs, relative to an even spread.
static double cu_imbalance(long workgroups) {
  return workgroups <= 256 ? 1.0 : (double)tw_div_up(workgroups, 256) * 256.0 / (double)workgroups;
}

template <typename T, typename OutT, int MT, bool PARTIAL, bool SHUF, bool GLU, class In = RowsAsTheyAre>
static int launch_skinny_lds(const T* A, long lda, const T* W, long ldw, const float* bias,
                             const float* residual, long ldr, OutT* C, long ldc, float* partial,
                             long partial_bytes, int M, int N, int K, hipStream_t stream, In norms = In{}) {
  constexpr int EPF = Elem<T>::kPerFrag;
  constexpr int U = MT == 1 ? 8 : 4;
  int splits = GLU ? 1 : skinny_lds_splits(N, K, EPF);
  if (PARTIAL) {
    TW_REQUIRE(partial != nullptr && partial_bytes >= (long)splits * M * N * 4);
  } else if (splits > 1 && (partial == nullptr || partial_bytes < (long)splits * M * N * 4)) {
    splits = 1;
  }
  // One K range and at most 16 rows (the gated projection of a decode step, the head): workgroups of two
  // waves where twice as many of them lie more evenly on the CUs (N = 37,888: 592 workgroups are 2.3 a CU,
  // three on some; 1,184 are 4.6, five on some). With more rows every workgroup stages its own copy of
  // the activations, so the larger workgroups stay.
  if constexpr (MT == 1 && !PARTIAL) {
    if (splits == 1 && cu_imbalance(tw_div_up(N, 32)) < cu_imbalance(tw_div_up(N, 64)) - 0.03) {
      const int groups = tw_div_up(N, 32);
      gemm_skinny_lds_kernel<T, OutT, MT, U, 2, PARTIAL, SHUF, GLU, In><<<groups, 128, 0, stream>>>(
          A, lda, W, ldw, bias, residual, ldr, C, ldc, partial, M, N, K, groups, 1, norms);
      return TW_LAUNCH_RESULT();
    }
  }
  const int groups = tw_div_up(N, 64);
  gemm_skinny_lds_kernel<T, OutT, MT, U, 4, PARTIAL, SHUF, GLU, In><<<groups * splits, 256, 0, stream>>>(
      A, lda, W, ldw, bias, residual, ldr, C, ldc, partial, M, N, K, groups, splits, norms);
  int err = TW_LAUNCH_RESULT();
  if (err || splits == 1 || PARTIAL) return err;
  return launch_splitk_reduce<OutT>(partial, splits, bias, residual, ldr, C, ldc, M, N, stream);
}

template <typename T, typename OutT, int MT, bool PARTIAL, bool GLU>
static int launch_stream_cu_mt(const T* A, long lda, const T* W, long ldw, const float* bias, const float* residual,
                               long ldr, OutT* C, long ldc, float* partial, long partial_bytes, int M, int N, int K,
                               hipStream_t stream) {
  constexpr int EPF = Elem<T>::kPerFrag;
  const bool room = partial != nullptr;
  CuPlan plan = cu_plan(MT, N, K, EPF, GLU, PARTIAL || room);
  if (PARTIAL) {
    TW_REQUIRE(partial != nullptr && partial_bytes >= (long)plan.splits * M * N * 4);
  } else if (plan.splits > 1 && partial_bytes < (long)plan.splits * M * N * 4) {
    plan = cu_plan(MT, N, K, EPF, GLU, false);
  }
  TW_REQUIRE(!GLU || N % 32 == 0);
  auto run = [&](auto sums, auto wide) {
    constexpr bool SUMS = decltype(sums)::value;
    typedef std::conditional_t<SUMS, float, OutT> Out;
    auto kernel = gemm_stream_cu_kernel<T, Out, MT, SUMS, GLU, decltype(wide)::value>;
    static bool attribute_set = false;   // per instantiation
    if (!attribute_set) {
      hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, TW_CU_LDS_BYTES);
      if (e != hipSuccess) return (int)e;
      attribute_set = true;
    }
    kernel<<<plan.splits * plan.wgs_per_split, TW_CU_WAVES * 64, TW_CU_LDS_BYTES, stream>>>(
        A, lda, W, ldw, bias, residual, ldr, (Out*)C, ldc, partial, M, N, K, plan.splits, plan.wgs_per_split, plan.compute_waves,
        plan.steps_per_split);
    return TW_LAUNCH_RESULT();
  };
  if constexpr (GLU) {
    return run(std::false_type{}, std::false_type{});
  } else {
    if (PARTIAL || plan.splits > 1) {
      const bool wide = N % 4 == 0 && (uintptr_t)partial % 16 == 0;
      const int err = wide ? run(std::true_type{}, std::true_type{}) : run(std::true_type{}, std::false_type{});
      if (err || PARTIAL) return err;
      return launch_splitk_reduce<OutT>(partial, plan.splits, bias, residual, ldr, C, ldc, M, N, stream);
    }
    if constexpr (!PARTIAL) {
      const bool wide = N % 4 == 0 && ldc % 4 == 0 && (uintptr_t)C % (4 * sizeof(OutT)) == 0 && (uintptr_t)bias % 16 == 0 &&
                        (residual == nullptr || (ldr % 4 == 0 && (uintptr_t)residual % 16 == 0));
      return wide ? run(std::false_type{}, std::true_type{}) : run(std::false_type{}, std::false_type{});
    }
    return TW_ERR_BAD_ARGUMENT;
  }
}

template <typename T, typename OutT, bool PARTIAL, bool GLU>
static int launch_stream_cu(const T* A, long lda, const T* W, long ldw, const float* bias, const float* residual,
                            long ldr, OutT* C, long ldc, float* partial, long partial_bytes, int M, int N, int K,
                            hipStream_t stream) {
  if (M <= 16) return launch_stream_cu_mt<T, OutT, 1, PARTIAL, GLU>(A, lda, W, ldw, bias, residual, ldr, C, ldc, partial, partial_bytes, M, N, K, stream);
  if (M <= 32) return launch_stream_cu_mt<T, OutT, 2, PARTIAL, GLU>(A, lda, W, ldw, bias, residual, ldr, C, ldc, partial, partial_bytes, M, N, K, stream);
  if (M <= 48) return launch_stream_cu_mt<T, OutT, 3, PARTIAL, GLU>(A, lda, W, ldw, bias, residual, ldr, C, ldc, partial, partial_bytes, M, N, K, stream);
  return launch_stream_cu_mt<T, OutT, 4, PARTIAL, GLU>(A, lda, W, ldw, bias, residual, ldr, C, ldc, partial, partial_bytes, M, N, K, stream);
}

// Above this many rows (and up to 64) the kernel with one workgroup per CU runs for shuffled weights.
#define TW_CU_ABOVE_ROWS 16

template <typename T, typename OutT, bool PARTIAL, bool SHUF, bool GLU>
static int launch_skinny_lds_m(const T* A, long lda, const T* W, long ldw, const float* bias,
                               const float* residual, long ldr, OutT* C, long ldc, float* partial,
                               long partial_bytes, int M, int N, int K, hipStream_t stream) {
  if (M <= 16) return launch_skinny_lds<T, OutT, 1, PARTIAL, SHUF, GLU>(A, lda, W, ldw, bias, residual, ldr, C, ldc, partial, partial_bytes, M, N, K, stream);
  if (M <= 32) return launch_skinny_lds<T, OutT, 2, PARTIAL, SHUF, GLU>(A, lda, W, ldw, bias, residual, ldr, C, ldc, partial, partial_bytes, M, N, K, stream);
  if (M <= 48) return launch_skinny_lds<T, OutT, 3, PARTIAL, SHUF, GLU>(A, lda, W, ldw, bias, residual, ldr, C, ldc, partial, partial_bytes, M, N, K, stream);
  return launch_skinny_lds<T, OutT, 4, PARTIAL, SHUF, GLU>(A, lda, W, ldw, bias, residual, ldr, C, ldc, partial, partial_bytes, M, N, K, stream);
}

// Up to 16 rows of a shuffled weight: is the kernel with 16 output columns (GLU: 16 pairs) over the whole of K a
// workgroup faster than the one with K ranges? Measured with weights from HBM, back to back (us, K ranges and their
// reduction / whole K), at 1, 8 and 16 rows:
//    N x K, bf16       256 x 1024          256 x 3072          256 x 4096         1536 x 4096         4096 x 4096
//      1           4.9 / 2.4           6.0 / 4.3           6.0 / 4.9           7.6 / 5.3          11.2 / 7.4
//      8           5.5 / 3.0           6.5 / 5.3           6.6 / 5.9           7.8 / 6.4          11.5 / 7.8
//     16           6.0 / 3.5           6.9 / 6.6           6.9 / 7.5           8.3 / 8.0          12.4 / 9.0
//                  4608 x 256          4608 x 512         6144 x 1536         8192 x 2048         4608 x 3584
//      1           3.8 / 3.5           4.8 / 3.8           8.5 / 5.6          10.5 / 7.3          10.4 / 9.9
//      8           4.1 / 4.2           5.0 / 4.4           8.8 / 6.5          10.8 / 7.6          10.7 / 11.5
//     16           4.3 / 5.0           5.3 / 5.2           9.6 / 7.7          11.5 / 8.8          11.7 / 13.9
//    gated             2048 x 4096         8192 x 4096         9728 x 896         9728 x 2048         16384 x 2048        22016 x 2048       37888 x 512
//      1          14.4 / 7.4          19.2 / 12.9          6.2 / 5.7          10.0 / 9.4          14.1 / 12.4         17.1 / 16.0        8.7 / 9.7
//      8          14.7 / 8.4          17.5 / 13.4          6.3 / 6.1          10.2 / 10.1         13.6 / 12.2         16.7 / 16.0        9.0 / 10.6
//     16          15.1 / 9.8          17.9 / 16.5          6.6 / 6.8          10.5 / 11.5         13.9 / 12.7         17.3 / 17.1        9.6 / 11.7
//    float32, K halved (the same k-steps): the same signs, but gated 9728 x 768 9.2 / 9.4, 9.3 / 9.8, 9.5 / 10.3 and
//    x 1024 12.1 / 11.0, 11.3 / 11.3, 11.5 / 12.4 (bf16 9728 x 1536 8.3 / 8.0, 8.4 / 8.6, 8.6 / 9.3).
// Up to 256 workgroups (one a CU): as long as a wave's share of K is about what it keeps in flight (8 k-steps of 16
// waves), K <= 4096 in bf16; where few workgroups leave the chip to the K ranges, more than 8 rows end sooner.
// With more workgroups every one reads the activations again: only where the other kernel's waves sit through a chain
// of stages and the weights outweigh the activations. Gated, between one and two a CU, the second round is nearly empty
// and up to 8 rows (in float32 fewer k-steps too) are the most that pays.
// `sums`: float32 sums for the caller's next kernel, no reduction saved: where the other kernel has one range too
// (bf16, 1 and 16 rows: 256 x 512 2.9 / 2.2, 3.2 / 2.9; 4096 x 896 5.4 / 3.4, 6.1 / 4.1; float32 4096 x 448 6.3 / 3.9, 6.9 / 4.4),
// and up to 8 rows with enough columns to fill the chip, where the next kernel reads one sum instead of 3 to 10. In a captured
// graph, with a norm that adds the sums up behind it, cold weights (K ranges / whole K), 1, 8 and 16 rows:
//    bf16 1024 x 2048  6.6 / 6.3, 7.1 / 7.0, 7.2 / 7.6      2048 x 2048  7.1 / 6.4, 7.5 / 7.3, 7.8 / 8.1
//         3072 x 3072  9.7 / 8.0, 10.2 / 9.2, 11.0 / 10.3   3584 x 3584  10.6 / 9.4, 11.2 / 10.4, 12.1 / 11.8
//         4096 x 2048  8.7 / 7.7, 9.1 / 8.1, 9.6 / 8.8      2048 x 4096  8.6 / 8.1, 9.2 / 9.4, 9.6 / 10.9
//    float32 896 x 896  7.7 / 6.6, 8.2 / 7.3, 8.6 / 8.0     2560 x 2048  10.9 / 9.1, 11.7 / 10.3, 12.2 / 11.6
//         2048 x 2048  9.2 / 8.7, 9.7 / 9.8, 10.2 / 11.2    3584 x 3584  17.6 / 15.0, 17.8 / 16.3, 18.8 / 18.9
// Between 2,048 and 3,584 columns the lines are the other kernel's: it gets 1.5 us slower where it has more workgroups than CUs, and
// a microsecond for every 8 k-steps of a range that begin; this one where its 16 waves begin another batch, at 128 and 192 k-steps.
// (8 rows: bf16 2304 x 2560, 180 workgroups of 16 k-steps, 8.3 / 9.0, x 2816, of 17.6, 9.3 / 9.1; 2560 x 3328, 240, 10.1 / 9.8, x 3584, 280, 10.5 / 9.9;
// 2816 x 3328 11.4 / 10.0. float32 2560 x 1536, 240 workgroups, 9.6 / 9.8, x 1792, 280, 11.5 / 10.4, x 2304, 144 k-steps, 12.3 / 12.9; 3072 x 2816, 17.6 k-steps
// a range, 15.1 / 13.7, x 3328, 208, 15.4 / 16.3.)
//
// An eighth and more beyond those lines both are estimated, and this kernel taken where it is expected to be 10 % (float32: 7) faster. What a workgroup reads goes at
// a CU's own rate (its weights, and the activations in whole batches of four k-steps a wave), rounds of workgroups one after the
// other, all together no faster than memory; the other kernel's time is that of its k-steps, of memory and of the reduction. Fitted to
// 3,952 products of 1 to 16 rows (256 to 32,000 x 256 to 11,008, both types, plain with a residual and gated; 3 to 7 % off): plain ones
// come out 3 % faster in the mean than by the lines alone, gated ones 9 % in bfloat16 and 17 in float32, one of them 2 % slower, and are 1
// and 0.4 % behind the better of the two. (us, K ranges or two waves a column / whole K, at 1 and 8 rows: bf16 9216 x 2048 11.3 / 8.2, 11.6 /
// 8.9, 12288 x 2048 13.0 / 9.9, 13.4 / 9.9; 2048 x 5632 with a residual 9.4 / 7.1, 9.7 / 9.0; float32 8192 x 2048 18.8 / 13.9, 19.4 / 14.3, 10304 x
// 2048 21.3 / 18.0, 22.2 / 19.2, 2048 x 4096 13.2 / 11.2, 13.2 / 12.3.)
// Gated: 16 gate and 16 up rows a workgroup, or eight of either in one fragment (HALVES), twice the workgroups that each read the
// activations? What the fullest CU reads decides, in rows of weights (an activation's row counts for as much as below); in bfloat16 only
// where halves are one workgroup a CU at most. (us, back to back, pairs or two waves a column / halves, 1, 4, 8 rows: bf16 2048 x 4096
// 7.3 / 5.9, 7.8 / 6.3, 8.5 / 6.9, 4096 x 2048 5.2 / 4.8, 5.5 / 4.9, 5.8 / 5.2; float32 2048 x 2048 9.1 / 6.3, 9.6 / 6.7, 10.1 / 7.2, 3648 x 2896 15.7 / 10.8,
// 15.3 / 11.6 at 8, 9728 x 896 10.4 / 9.1, 10.4 / 9.6, 10.5 / 10.5, 11264 x 1024 12.5 / 9.8, 12.0 / 10.0, 12.0 / 10.8, x 2048 23.1 / 20.3, 23.0 / 20.7, 23.0 / 21.1. Left
// to pairs: bf16 9728 x 896 5.7 / 5.8, 6.1 / 6.5 at 8 rows, 16384 x 2048 12.1 / 12.5, 12.3 / 13.7; and 11264 x 2048, 10.0 / 9.6, 10.8 / 10.4 back to back,
// but a captured step of four such layers of one row is 4 us slower with halves.)
static double narrow_row_share(int epf, bool glu) { return epf == 8 ? 1.33 : glu ? 0.73 : 0.87; }
static bool narrow_halves(int M, int N, int K, int epf) {
  const int groups = N / 16;
  const double rows = narrow_row_share(epf, true) * M;
  if (groups > 256 && epf == 8) return false;
  return (16 + rows) * tw_div_up(groups, 256) < 0.95 * (32 + rows) * tw_div_up(groups, 512);
}
static double narrow_us(int M, int N, int K, int epf, bool glu) {
  const bool pairs = glu && !narrow_halves(M, N, K, epf);
  const int size = 16 / epf, steps = tw_div_up(K / epf, 4), groups = pairs ? N / 32 : tw_div_up(N, 16);
  const int waves = steps <= 48 ? 4 : steps <= 96 ? 8 : 16;            // (see launch_narrow)
  const double covered = (double)tw_div_up(tw_div_up(steps, waves), 4) * 4 * waves * 64;      // bytes of a row
  const double cu = 1e-3 * (size == 2 ? (glu ? 0.0187 : 0.0195) : 0.0254) * ((pairs ? 32 : 16) + narrow_row_share(epf, glu) * M) * covered * tw_div_up(groups, 256);
  const double memory = 1e-6 * N * (double)K * size / (size == 2 ? 6.57 : 6.14);
  return (size == 2 ? (glu ? 2.66 : 2.80) : glu ? 2.81 : 2.97) + sqrt(sqrt(cu * cu * cu * cu + memory * memory * memory * memory));
}
static double skinny_us(int M, int N, int K, int epf, bool glu, bool reduced = true) {
  const int size = 16 / epf, steps = tw_div_up(K / epf, 4), splits = glu ? 1 : skinny_lds_splits(N, K, epf);
  const double fill = tw_div_up(N, 64) * splits / 512.0;
  const double step = size == 2 ? (glu ? 0.0918 + 0.0005 * M : 0.0715 + 0.0014 * M) : glu ? 0.1101 + 0.0002 * M : 0.0589 + 0.0017 * M;
  const double cu = tw_div_up(steps, splits) * step * (fill > 1 ? fill : 1.0);
  const double memory = 1e-6 * N * (double)K * size / (size == 2 ? 6.57 : 6.4);
  return (size == 2 ? (glu ? 2.99 : 3.62) : glu ? 3.29 : 4.31) + (splits > 1 && reduced ? (size == 2 ? 1.95 + 0.74e-6 * 4 * splits * M * N : 2.22 + 0.67e-6 * 4 * splits * M * N) : 0.0) +
         sqrt(sqrt(cu * cu * cu * cu + memory * memory * memory * memory));
}

static bool narrow_pays(int M, int N, int K, int epf, bool glu, bool sums) {
  const int steps = tw_div_up(K / epf, 4), groups = glu ? N / 32 : tw_div_up(N, 16);
  if (sums) {
    if (groups > 256 || steps < 16) return false;
    if (steps < 32 || (epf == 4 && steps <= 64 && groups >= 48)) return true;
    if (M > 8) return false;
    const int ranges = skinny_lds_splits(N, K, epf), workgroups = tw_div_up(N, 64) * ranges;
    const bool second = workgroups > 256;                                 // more than one of the other kernel's workgroups a CU
    if (epf == 8) return groups >= 128 && steps <= 112 && (steps <= 72 || second || steps > 16 * ranges);
    if (groups < 160) return false;
    return steps <= 128 ? second : steps <= 192 ? groups >= 224 || steps > 16 * ranges : steps <= 224 && (groups >= 240 || steps > 24 * ranges);
  }
  if (groups <= 256 ? steps <= (M > 8 && groups < 96 && !glu ? 96 : 128)
      : glu ? steps >= 28 && steps <= (groups < 512 && epf == 4 ? 32 : 64) && (M <= 8 || groups >= 512)
            : groups <= 512 && steps >= 16 && steps <= 64) return true;
  // (by an eighth: what lies at the lines stays where it is; float32's are those of pairs, halves are estimated from workgroups of eight waves on)
  const bool beyond = groups >= 576 || steps > (groups <= 256 ? 144 : 72) || (glu && epf == 4 && steps > 48 && narrow_halves(M, N, K, epf));
  return beyond && steps >= 28 && narrow_us(M, N, K, epf, glu) < (epf == 4 ? 0.93 : 0.9) * skinny_us(M, N, K, epf, glu);
}

// Whole K a workgroup where its epilogue spares the kernel that would add the K ranges' sums up anyway: a norm (EndLeave) or the
// rotation and cache write (EndRotate), SPARES microseconds as a node of a captured step. (Four layers and a head, captured steps, us:
// neither / norms that travel / rotation too, at 1, 8 and 16 rows: 896 wide with down products of 4,864 174 / 162 / 155, 188 / 180 / 172, 203 / 195 / 187;
// 2,048 wide, 11,008: 318 / 303 / 295, 338 / 326 / 316, 363 / 351 / 342; 3,584 wide, 18,944, 1 and 8 rows: 584 / 559 / 561, 629 / 618 / 618. The
// down products of the last at 8 rows, 3.4 us behind by estimate, gain 6 us a step; those of 2,048 x 11,008 at 4, 3 behind, 2.)
// On either side of the line: of 600 random products of 512 to 4,096 columns and 1 to 16 rows with the product behind them, 470 leave their rows and take
// 0.86 of the time, eleven of them more than 1 % longer, the most 7 %; the others would take 1.08, a tenth of them up to 10 % less.
// The rotation's kernel is 2.5 us, and its epilogue here takes 1 of them. Workgroups of 16 waves have a CU to themselves: further turns of them begin when
// those before end, which the estimate leaves out, and pay for it unless a wave's k-steps are exactly the eight that are on their way from the start. (us, cold
// weights, apart / here, 1 and 6 rows: bf16 7168 x 5120 18.5 / 18.6, 19.1 / 21.6; 10240 x 5120 24.1 / 26.9, 24.6 / 29.5; 10240 x 3584 18.9 / 19.6, 19.2 / 21.0;
// float32 5120 x 3072 17.5 / 19.2, 18.1 / 21.1. One turn, eight waves, eight k-steps a wave: 4096 x 5120 13.8 / 10.9, 14.1 / 12.1; 9216 x 2048 12.7 / 9.8, 13.3 /
// 10.9; 7168 x 4096 18.0 / 14.8, 19.2 / 16.2. Of 900 shapes of 1,152 to 10,240 x 896 to 8,192 and 1 to 16 rows the choice is 0.4 % behind the better of the two;
// six are more than 2 % slower than apart, the most 6 %.)
static bool narrow_end_pays(int M, int N, int K, int epf, double spares) {
  if (M < 1 || M > 16 || N % 64 || K % epf) return false;
  const int steps = tw_div_up(K / epf, 4);
  const double turns = steps > 96 && steps != 128 ? 1.2 * (tw_div_up(N / 16, 256) - 1) : 0.0;
  return narrow_us(M, N, K, epf, false) + turns < skinny_us(M, N, K, epf, false, false) + spares;
}
#define TW_LEAVE_SPARES_US 3.5
#define TW_ROTATE_SPARES_US 1.2

// A plain product with an activation behind it, against the K ranges' sums and a kernel that adds them up and applies it (bf16, in a
// captured graph, cold weights): 4096 x 2048 1 / 8 / 16 rows 7.6 / 4.2, 7.9 / 4.6, 8.5 / 5.2; 5632 x 2048 9.0 / 5.8, 9.5 / 6.6, 10.4 / 7.9;
// 8192 x 3072 12.5 / 9.1, 12.9 / 10.1, 13.6 / 12.3; 11264 x 2048 12.5 / 8.7, 13.1 / 9.3, 14.2 / 11.5.
static bool narrow_act_pays(int M, int N, int K, int epf) {
  return M <= 16 && (narrow_pays(M, N, K, epf, false, false) || (epf == 8 && tw_div_up(N, 16) <= 704 && tw_div_up(K / epf, 4) <= 96));
}

// Waves a workgroup: as few as have a wave's whole share of K in flight at once (8 k-steps), up to 16. (2048 x 1024, 8
// rows: 4 / 8 / 16 waves 3.5 / 4.0 / 5.6 us; 2048 x 2048: 5.2 / 4.4 / 5.9; 2048 x 4096: 8.1 / 6.7 / 6.5)
template <typename T, typename OutT, bool GLU, bool ACT = false, class In = RowsAsTheyAre, class End = EndPlain>
static int launch_narrow(const T* A, long lda, const T* W, long ldw, const float* bias, const float* residual, long ldr,
                         OutT* C, long ldc, int M, int N, int K, hipStream_t stream, In norms = In{}, End end = End{}) {
  const int steps = tw_div_up(K / Elem<T>::kPerFrag, 4);
  auto run = [&](auto halves) {
    constexpr bool H = decltype(halves)::value;
    const int groups = GLU && !H ? N / 32 : tw_div_up(N, 16);
    if (steps <= 48)
      gemm_narrow_kernel<T, OutT, 4, GLU, ACT, In, End, H><<<groups, 256, 0, stream>>>(A, lda, W, ldw, bias, residual, ldr, C, ldc, M, N, K, norms, end);
    else if (steps <= 96)
      gemm_narrow_kernel<T, OutT, 8, GLU, ACT, In, End, H><<<groups, 512, 0, stream>>>(A, lda, W, ldw, bias, residual, ldr, C, ldc, M, N, K, norms, end);
    else
      gemm_narrow_kernel<T, OutT, 16, GLU, ACT, In, End, H><<<groups, 1024, 0, stream>>>(A, lda, W, ldw, bias, residual, ldr, C, ldc, M, N, K, norms, end);
    return TW_LAUNCH_RESULT();
  };
  if constexpr (GLU) {
    if (narrow_halves(M, N, K, Elem<T>::kPerFrag)) return run(std::true_type{});
  }
  return run(std::false_type{});
}

// force: 0 = choose, 1 = generic, 3 = tiled 128x128, 4 = tiled 128x256, 5 = skinny, 6 = tiled 256x256,
// 7 = tiled 256x192, 8 = streaming with one workgroup per CU (shuffled weights, up to 64 rows),
// 9 = whole K per workgroup (shuffled weights, up to 16 rows), 10 to 14 = tiled 192x128, 192x192, 192x256, 192x384, 256x320 (shuffled bfloat16)
template <typename T, typename OutT, bool SHUF, bool GLU>
static int linear_dispatch(const T* A, long lda, const T* W, long ldw, const float* bias,
                           const float* residual, long ldr, OutT* C, long ldc, float* partial,
                           long partial_bytes, int M, int N, int K, int force, hipStream_t stream) {
  constexpr int EPF = Elem<T>::kPerFrag;
  TW_REQUIRE(force == 0 || force == 1 || (force >= 3 && force <= 14));
  // the shuffled layout exists only for K that is a multiple of 16 bytes and is always aligned
  const bool aligned = K % EPF == 0 && lda % EPF == 0 && ((uintptr_t)A % 16 == 0) && ((uintptr_t)W % 16 == 0) &&
                       (SHUF || ldw % EPF == 0);
  if (force == 1 || !aligned) {
    TW_REQUIRE(force <= 1);
    TW_REQUIRE(!SHUF || K % EPF == 0);
    const long outputs = (long)M * (GLU ? N / 2 : N);
    gemm_generic_kernel<T, OutT><<<tw_div_up(outputs, 256), 256, 0, stream>>>(A, lda, W, ldw, bias, residual, ldr, C,
                                                                            ldc, M, N, K, SHUF ? 1 : 0, GLU ? 1 : 0);
    return TW_LAUNCH_RESULT();
  }
  if (force == 8 || (force == 0 && SHUF && M > TW_CU_ABOVE_ROWS && M <= 64)) {
    TW_REQUIRE(M <= 64 && SHUF);
    if constexpr (SHUF)
      return launch_stream_cu<T, OutT, false, GLU>(A, lda, W, ldw, bias, residual, ldr, C, ldc, partial, partial_bytes, M, N, K, stream);
  }
  if constexpr (SHUF) {
    if (force == 9 || (force == 0 && M <= 16 && narrow_pays(M, N, K, EPF, GLU, false))) {
      TW_REQUIRE(M <= 16);
      return launch_narrow<T, OutT, GLU>(A, lda, W, ldw, bias, residual, ldr, C, ldc, M, N, K, stream);
    }
  }
  if (force == 5 || (force == 0 && M <= 64)) {
    TW_REQUIRE(M <= 64);
    return launch_skinny_lds_m<T, OutT, false, SHUF, GLU>(A, lda, W, ldw, bias, residual, ldr, C, ldc, partial, partial_bytes, M, N, K, stream);
  }
  const int shape = force >= 10 ? force - 5 : force == 3 ? 1 : (force == 4 ? 2 : (force == 6 ? 3 : (force == 7 ? 4 : 0)));
  return tw_tiled_linear(sizeof(T) == 4 ? TW_DTYPE_F32 : TW_DTYPE_BF16, sizeof(OutT) == 4 ? 1 : 0, SHUF ? 1 : 0,
                         GLU ? 1 : 0, shape, A, lda, W, ldw, bias, residual, ldr, C, ldc, partial, partial_bytes,
                         M, N, K, stream);
}

template <typename T, typename OutT>
static int linear_layout(int shuffled, const T* A, long lda, const T* W, long ldw, const float* bias,
                         const float* residual, long ldr, OutT* C, long ldc, float* partial,
                         long partial_bytes, int M, int N, int K, int force, hipStream_t stream) {
  if (shuffled)
    return linear_dispatch<T, OutT, true, false>(A, lda, W, ldw, bias, residual, ldr, C, ldc, partial, partial_bytes, M, N, K, force, stream);
  return linear_dispatch<T, OutT, false, false>(A, lda, W, ldw, bias, residual, ldr, C, ldc, partial, partial_bytes, M, N, K, force, stream);
}

static bool weight_layout_ok(int dtype, int shuffled, long ldw, int K) {
  const int epf = dtype == TW_DTYPE_F32 ? 4 : 8;
  return shuffled ? (K % epf == 0 && ldw >= (K / epf + 3) / 4) : ldw >= K;
}

// C = A W^T (+bias) (+residual). out_f32 != 0: C is float32 whatever the input type (residual
// stream, logits); else C has the input type. `residual` may be C itself. `partial` is scratch
// for split-K (tw_linear_workspace_bytes). shuffled != 0: W is in the shuffled layout and ldw
// is the number of k-steps between its row blocks, at least ceil(K / (4 * elements per 16 bytes)).
extern "C" int tw_linear(int dtype, int out_f32, const void* A, long lda, const void* W, long ldw, int shuffled,
                         const float* bias, const float* residual, long ldr, void* C, long ldc,
                         float* partial, long partial_bytes, int M, int N, int K, int force,
                         hipStream_t stream) {
  TW_REQUIRE(M >= 0 && N > 0 && K > 0 && lda >= K && ldc >= N);
  TW_REQUIRE(weight_layout_ok(dtype, shuffled, ldw, K));
  TW_REQUIRE(residual == nullptr || (ldr >= N && out_f32));
  if (M == 0) return 0;
  if (dtype == TW_DTYPE_F32)
    return linear_layout<float, float>(shuffled, (const float*)A, lda, (const float*)W, ldw, bias, residual, ldr,
                                       (float*)C, ldc, partial, partial_bytes, M, N, K, force, stream);
  if (dtype == TW_DTYPE_BF16) {
    if (out_f32)
      return linear_layout<bf16_t, float>(shuffled, (const bf16_t*)A, lda, (const bf16_t*)W, ldw, bias, residual, ldr,
                                          (float*)C, ldc, partial, partial_bytes, M, N, K, force, stream);
    return linear_layout<bf16_t, bf16_t>(shuffled, (const bf16_t*)A, lda, (const bf16_t*)W, ldw, bias, residual, ldr,
                                         (bf16_t*)C, ldc, partial, partial_bytes, M, N, K, force, stream);
  }
  return TW_ERR_BAD_ARGUMENT;
}

// out = act(x @ W.T + bias) for many rows (the tiled kernels, whose epilogue and split-K reduction apply the
// activation before the one rounding): more than 64 rows, K a multiple of 16 bytes, output in the input type.
extern "C" int tw_linear_act(int dtype, const void* A, long lda, const void* W, long ldw, int shuffled, const float* bias,
                             void* C, long ldc, float* partial, long partial_bytes, int M, int N, int K, int act,
                             hipStream_t stream) {
  TW_REQUIRE(act == TW_ACT_RELU_SQUARED || act == TW_ACT_GELU_ERF);
  TW_REQUIRE(M > 64 && N > 0 && K > 0 && lda >= K && ldc >= N && K % (dtype == TW_DTYPE_F32 ? 4 : 8) == 0);
  TW_REQUIRE(dtype == TW_DTYPE_F32 || dtype == TW_DTYPE_BF16);
  TW_REQUIRE(weight_layout_ok(dtype, shuffled, ldw, K));
  return tw_tiled_linear(dtype, dtype == TW_DTYPE_F32 ? 1 : 0, shuffled, 0, 0, A, lda, W, ldw, bias, nullptr, (long)act, C, ldc,
                         partial, partial_bytes, M, N, K, stream);
}

// The same for up to 16 rows of shuffled weights where a workgroup with the whole of K pays (tw_linear_act_few_pays): the
// activation in that kernel's epilogue.
extern "C" int tw_linear_act_few_pays(int dtype, int M, int N, int K) {
  const int epf = dtype == TW_DTYPE_F32 ? 4 : 8;
  return M >= 1 && N > 0 && K > 0 && K % epf == 0 && narrow_act_pays(M, N, K, epf) ? 1 : 0;
}
extern "C" int tw_linear_act_few(int dtype, const void* A, long lda, const void* W, long ldw, const float* bias, void* C, long ldc,
                                 int M, int N, int K, int act, hipStream_t stream) {
  TW_REQUIRE(act == TW_ACT_RELU_SQUARED || act == TW_ACT_GELU_ERF);
  TW_REQUIRE(dtype == TW_DTYPE_F32 || dtype == TW_DTYPE_BF16);
  const int epf = dtype == TW_DTYPE_F32 ? 4 : 8;
  TW_REQUIRE(M >= 1 && M <= 16 && N > 0 && K > 0 && lda >= K && ldc >= N && K % epf == 0 && lda % epf == 0);
  TW_REQUIRE(weight_layout_ok(dtype, 1, ldw, K) && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0);
  if (dtype == TW_DTYPE_F32)
    return launch_narrow<float, float, false, true>((const float*)A, lda, (const float*)W, ldw, bias, nullptr, act, (float*)C, ldc, M, N, K, stream);
  return launch_narrow<bf16_t, bf16_t, false, true>((const bf16_t*)A, lda, (const bf16_t*)W, ldw, bias, nullptr, act, (bf16_t*)C, ldc, M, N, K, stream);
}

template <typename T>
static int glu_layout(int shuffled, const T* A, long lda, const T* W, long ldw, const float* bias, T* C, long ldc,
                      int M, int N, int K, int force, long code, hipStream_t stream) {
  // (no residual in the gated form: its stride carries the activation and the factor, see tw_glu)
  if (shuffled)
    return linear_dispatch<T, T, true, true>(A, lda, W, ldw, bias, nullptr, code, C, ldc, nullptr, 0, M, N, K, force, stream);
  return linear_dispatch<T, T, false, true>(A, lda, W, ldw, bias, nullptr, code, C, ldc, nullptr, 0, M, N, K, force, stream);
}

// Gated linear unit: W [N, K] holds gate and up rows interleaved in blocks of 16 (N a multiple
// of 32); C [M, N / 2] = factor * act(gate) * up in the input type (act: TW_GLU_SILU or TW_GLU_GELU_TANH). bias (may be
// null) is indexed like W's rows.
extern "C" int tw_linear_glu(int dtype, const void* A, long lda, const void* W, long ldw, int shuffled,
                             const float* bias, void* C, long ldc, int M, int N, int K, int force, int act,
                             float factor, hipStream_t stream) {
  TW_REQUIRE(act == TW_GLU_SILU || act == TW_GLU_GELU_TANH || act == TW_GLU_SWISH_LIMITED);
  const long code = tw_glu_code(act, factor);
  TW_REQUIRE(M >= 0 && N > 0 && N % 32 == 0 && K > 0 && lda >= K && ldc >= N / 2);
  TW_REQUIRE(weight_layout_ok(dtype, shuffled, ldw, K));
  if (M == 0) return 0;
  if (dtype == TW_DTYPE_F32)
    return glu_layout<float>(shuffled, (const float*)A, lda, (const float*)W, ldw, bias, (float*)C, ldc, M, N, K, force, code, stream);
  if (dtype == TW_DTYPE_BF16)
    return glu_layout<bf16_t>(shuffled, (const bf16_t*)A, lda, (const bf16_t*)W, ldw, bias, (bf16_t*)C, ldc, M, N, K, force, code, stream);
  return TW_ERR_BAD_ARGUMENT;
}

// ---- decode-path form: few rows, 16-byte aligned K ------------------------------------
// Number of K ranges tw_linear_partials uses for an [N, K] weight (0: shape not supported).
extern "C" int tw_linear_partial_splits(int dtype, int N, int K) {
  const int epf = dtype == TW_DTYPE_F32 ? 4 : 8;
  if (K % epf) return 0;
  return skinny_lds_splits(N, K, epf);
}

// The same for M rows whose stride is LDA elements: up to 64 rows the streaming kernel's ranges; above,
// those of the tiled kernels (0 where they would not split K: the product with its epilogue is then the
// better call). Which tiled kernel runs, and so how it splits, depends on the rows' stride too.
extern "C" int tw_linear_partial_splits_rows(int dtype, int shuffled, int M, int N, int K, long lda) {
  const int epf = dtype == TW_DTYPE_F32 ? 4 : 8;
  if (M <= 64 && shuffled && M > TW_CU_ABOVE_ROWS && K % epf == 0)
    return cu_plan(tw_div_up(M, 16), N, K, epf, false, true).splits;
  if (M <= 16 && shuffled && K % epf == 0 && narrow_pays(M, N, K, epf, false, true)) return 1;
  if (M <= 64) return tw_linear_partial_splits(dtype, N, K);
  if (K % epf || lda < K) return 0;
  const int splits = tw_tiled_partial_splits(dtype, shuffled, lda, M, N, K);
  return splits > 1 ? splits : 0;
}

template <typename T>
static int partials_layout(int shuffled, const T* A, long lda, const T* W, long ldw, float* partial,
                           long partial_bytes, int M, int N, int K, hipStream_t stream) {
  if (shuffled && M > TW_CU_ABOVE_ROWS)
    return launch_stream_cu<T, float, true, false>(A, lda, W, ldw, nullptr, nullptr, 0, (float*)nullptr, N, partial, partial_bytes, M, N, K, stream);
  if (shuffled && M <= 16 && narrow_pays(M, N, K, Elem<T>::kPerFrag, false, true)) {
    TW_REQUIRE(partial != nullptr && partial_bytes >= (long)M * N * 4);
    return launch_narrow<T, float, false>(A, lda, W, ldw, nullptr, nullptr, 0, partial, N, M, N, K, stream);
  }
  if (shuffled)
    return launch_skinny_lds_m<T, float, true, true, false>(A, lda, W, ldw, nullptr, nullptr, 0, (float*)nullptr, N, partial, partial_bytes, M, N, K, stream);
  return launch_skinny_lds_m<T, float, true, false, false>(A, lda, W, ldw, nullptr, nullptr, 0, (float*)nullptr, N, partial, partial_bytes, M, N, K, stream);
}

// partial[split][M][N] (float32) = A[:, K range of split] W[:, same]^T for every split; the caller's
// next kernel adds the splits up (with bias, residual, norm or rotation as it needs). Up to 64 rows the
// streaming kernel runs, above that the tiled kernels.
extern "C" int tw_linear_partials(int dtype, const void* A, long lda, const void* W, long ldw, int shuffled,
                                  float* partial, long partial_bytes, int M, int N, int K, hipStream_t stream) {
  TW_REQUIRE(M >= 1 && N > 0 && K > 0 && lda >= K);
  const int epf = dtype == TW_DTYPE_F32 ? 4 : 8;
  TW_REQUIRE(K % epf == 0 && lda % epf == 0 && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0);
  TW_REQUIRE(weight_layout_ok(dtype, shuffled, ldw, K) && (shuffled || ldw % epf == 0));
  if (M > 64) {
    // the caller sized `partial` for the ranges tw_linear_partial_splits_rows named: they must be the ones used
    const int expect = tw_tiled_partial_splits(dtype, shuffled, lda, M, N, K);
    TW_REQUIRE(expect >= 1 && partial_bytes == (long)expect * M * N * 4);
    int used = 0;
    const int err = tw_tiled_partials(dtype, shuffled, A, lda, W, ldw, partial, partial_bytes, M, N, K, &used, stream);
    if (err) return err;
    return used == expect ? 0 : TW_ERR_BAD_ARGUMENT;
  }
  if (dtype == TW_DTYPE_F32)
    return partials_layout<float>(shuffled, (const float*)A, lda, (const float*)W, ldw, partial, partial_bytes, M, N, K, stream);
  if (dtype == TW_DTYPE_BF16)
    return partials_layout<bf16_t>(shuffled, (const bf16_t*)A, lda, (const bf16_t*)W, ldw, partial, partial_bytes, M, N, K, stream);
  return TW_ERR_BAD_ARGUMENT;
}

// ---- up to 16 rows of shuffled weights, norms that travel ----------------------------------------------------------
static bool few_rows_ok(int dtype, const void* A, long lda, const void* W, long ldw, int M, int N, int K) {
  const int epf = dtype == TW_DTYPE_F32 ? 4 : 8;
  return (dtype == TW_DTYPE_F32 || dtype == TW_DTYPE_BF16) && M >= 1 && M <= 16 && N > 0 && K > 0 && lda >= K && K % epf == 0 && lda % epf == 0 &&
         weight_layout_ok(dtype, 1, ldw, K) && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0;
}
static bool norms_ok(const float* sums, int count, float eps) {
  return sums != nullptr && (uintptr_t)sums % 16 == 0 && count > 0 && count % 4 == 0 && count <= TW_NORM_MAX_SUMS && eps > 0.f;
}

template <typename T>
static int linear_normed(int mode, int out_f32, const T* A, long lda, RowNorms norms, const T* W, long ldw, const float* bias, void* C,
                         long ldc, float* partial, long partial_bytes, int M, int N, int K, long code, hipStream_t stream) {
  constexpr int EPF = Elem<T>::kPerFrag;
  if (mode == 1) {                                             // K ranges' sums, as tw_linear_partials
    if (narrow_pays(M, N, K, EPF, false, true)) {
      TW_REQUIRE(partial != nullptr && partial_bytes >= (long)M * N * 4);
      return launch_narrow<T, float, false, false, RowNorms>(A, lda, W, ldw, nullptr, nullptr, 0, partial, N, M, N, K, stream, norms);
    }
    return launch_skinny_lds<T, float, 1, true, true, false, RowNorms>(A, lda, W, ldw, nullptr, nullptr, 0, (float*)nullptr, N, partial,
                                                                      partial_bytes, M, N, K, stream, norms);
  }
  if (mode == 2) {                                             // gated, as tw_linear_glu
    TW_REQUIRE(N % 32 == 0);
    if (narrow_pays(M, N, K, EPF, true, false))
      return launch_narrow<T, T, true, false, RowNorms>(A, lda, W, ldw, bias, nullptr, code, (T*)C, ldc, M, N, K, stream, norms);
    return launch_skinny_lds<T, T, 1, false, true, true, RowNorms>(A, lda, W, ldw, bias, nullptr, code, (T*)C, ldc, nullptr, 0, M, N, K, stream, norms);
  }
  if (mode == 3)                                               // with an activation, as tw_linear_act_few
    return launch_narrow<T, T, false, true, RowNorms>(A, lda, W, ldw, bias, nullptr, code, (T*)C, ldc, M, N, K, stream, norms);
  const bool narrow = narrow_pays(M, N, K, EPF, false, false);
  auto plain = [&](auto* out) {
    typedef std::remove_reference_t<decltype(*out)> OutT;
    if (narrow) return launch_narrow<T, OutT, false, false, RowNorms>(A, lda, W, ldw, bias, nullptr, 0, out, ldc, M, N, K, stream, norms);
    return launch_skinny_lds<T, OutT, 1, false, true, false, RowNorms>(A, lda, W, ldw, bias, nullptr, 0, out, ldc, partial, partial_bytes, M, N, K,
                                                                      stream, norms);
  };
  return out_f32 ? plain((float*)C) : plain((T*)C);
}

// The products of up to 16 rows whose norms travel (see RowNorms): A holds x * w rounded, sums [M][count] their sums of squares over
// `width` elements. mode 0: C = product (+ bias), float32 or the input type; 1: partial = the K ranges' sums, as tw_linear_partials;
// 2: the gated form, act and factor as tw_linear_glu; 3: C = act(product + bias), as tw_linear_act_few.
extern "C" int tw_linear_normed(int dtype, int mode, int out_f32, const void* A, long lda, const float* sums, int count, int width, float eps,
                                const void* W, long ldw, const float* bias, void* C, long ldc, float* partial, long partial_bytes, int M,
                                int N, int K, int act, float factor, hipStream_t stream) {
  TW_REQUIRE(mode >= 0 && mode <= 3 && few_rows_ok(dtype, A, lda, W, ldw, M, N, K) && norms_ok(sums, count, eps) && width > 0);
  TW_REQUIRE(mode == 1 || (C != nullptr && ldc >= (mode == 2 ? N / 2 : N)));
  TW_REQUIRE(mode != 2 || act == TW_GLU_SILU || act == TW_GLU_GELU_TANH || act == TW_GLU_SWISH_LIMITED);
  TW_REQUIRE(mode != 3 || act == TW_ACT_RELU_SQUARED || act == TW_ACT_GELU_ERF);
  const long code = mode == 2 ? tw_glu_code(act, factor) : act;
  const RowNorms norms = {sums, count, (float)width, eps};
  if (dtype == TW_DTYPE_F32)
    return linear_normed<float>(mode, 1, (const float*)A, lda, norms, (const float*)W, ldw, bias, C, ldc, partial, partial_bytes, M, N, K, code, stream);
  return linear_normed<bf16_t>(mode, out_f32, (const bf16_t*)A, lda, norms, (const bf16_t*)W, ldw, bias, C, ldc, partial, partial_bytes, M, N, K, code, stream);
}

extern "C" int tw_linear_leave_pays(int dtype, int M, int N, int K) {
  const int epf = dtype == TW_DTYPE_F32 ? 4 : 8;
  return N > 0 && K > 0 && N / 16 <= TW_NORM_MAX_SUMS && narrow_end_pays(M, N, K, epf, TW_LEAVE_SPARES_US) ? 1 : 0;
}

// C [M][N] (float32) += A W^T (+ bias), and what a norm of the new rows needs to travel: rows = C * weight (rows2 = C * weight2, or null)
// in the input type, sums [M][N / 16]. after != 0: C <- alpha * (C * rinv * before_weight) + scale * (A W^T + bias), the old rows' rinv from
// before_sums [M][N / 16] over N elements (null: C as it is); these must not be `sums`.
extern "C" int tw_linear_leave(int dtype, const void* A, long lda, const void* W, long ldw, const float* bias, float* C, long ldc, int M, int N,
                               int K, const float* weight, void* rows, const float* weight2, void* rows2, float* sums, int after,
                               const float* before_sums, const float* before_weight, const float* scale, float alpha, float eps,
                               hipStream_t stream) {
  TW_REQUIRE(few_rows_ok(dtype, A, lda, W, ldw, M, N, K) && C != nullptr && ldc >= N && N % 64 == 0 && N / 16 <= TW_NORM_MAX_SUMS);
  TW_REQUIRE(weight && rows && sums && (weight2 == nullptr) == (rows2 == nullptr));
  TW_REQUIRE(before_sums == nullptr || (after && before_weight && before_sums != sums && norms_ok(before_sums, N / 16, eps)));
  auto run = [&](auto t, auto end) {
    typedef decltype(t) T;
    return launch_narrow<T, float, false, false, RowsAsTheyAre>((const T*)A, lda, (const T*)W, ldw, bias, C, ldc, C, ldc, M, N, K, stream,
                                                                RowsAsTheyAre{}, end);
  };
  const RowNorms before = {before_sums, N / 16, (float)N, eps};
  const EndLeave<true> with = {weight, weight2, rows, rows2, sums, before, before_weight, scale, alpha};
  const EndLeave<false> without = {weight, weight2, rows, rows2, sums, before, nullptr, nullptr, 1.f};
  if (dtype == TW_DTYPE_F32) return after ? run(float{}, with) : run(float{}, without);
  return after ? run(bf16_t{}, with) : run(bf16_t{}, without);
}

// C [M][N] (the weight's type) = gelu_tanh(round(A) W^T + bias) * table[token of the row][offset ..] for float32 rows A of the stream; tokens as
// tw_token_gate. Where the product alone takes the kernel with the whole of K a workgroup.
extern "C" int tw_linear_token_gate_pays(int dtype, int M, int N, int K) {
  const int epf = dtype == TW_DTYPE_F32 ? 4 : 8;
  return M >= 1 && M <= 16 && N > 0 && K > 0 && K % epf == 0 && narrow_pays(M, N, K, epf, false, false) ? 1 : 0;
}
extern "C" int tw_linear_token_gate(int dtype, const float* A, long lda, const void* W, long ldw, const float* bias, void* C, long ldc, int M,
                                    int N, int K, const void* table, long ld_table, const int* ids, const int* feed, int n_feed, int vocab,
                                    int offset, hipStream_t stream) {
  TW_REQUIRE(few_rows_ok(dtype, A, lda, W, ldw, M, N, K) && lda % 4 == 0 && C != nullptr && ldc >= N);
  TW_REQUIRE(table && ids && vocab > 0 && offset >= 0 && offset + N <= ld_table);
  if (dtype == TW_DTYPE_F32)
    return launch_narrow<float, float, false>(A, lda, (const float*)W, ldw, bias, nullptr, 0, (float*)C, ldc, M, N, K, stream, RowsAsTheyAre{},
                                              EndTokenGate<float>{(const float*)table, ld_table, ids, feed, n_feed, vocab, offset});
  return launch_narrow<bf16_t, bf16_t, false>((const bf16_t*)A, lda, (const bf16_t*)W, ldw, bias, nullptr, 0, (bf16_t*)C, ldc, M, N, K, stream, RowsRounded{},
                                              EndTokenGate<bf16_t>{(const bf16_t*)table, ld_table, ids, feed, n_feed, vocab, offset});
}

extern "C" int tw_linear_rotate_pays(int dtype, int M, int N, int K) {
  const int epf = dtype == TW_DTYPE_F32 ? 4 : 8;
  return N > 0 && K > 0 && narrow_end_pays(M, N, K, epf, TW_ROTATE_SPARES_US) ? 1 : 0;
}

// The packed product of queries, keys and values of up to 16 rows, finished as tw_rope_kv_write finishes it: qkv [M][ld] = round(A W^T +
// bias), q rotated in place; rotated k and v to the pages of the rows' slots (write_cache; the k and v columns of qkv are not written).
// sums: null, or the rows' norms as tw_linear_normed. rot: a multiple of 16. behind: columns of the product behind the values (a multiple of 16),
// which stay as they are.
extern "C" int tw_linear_rotate(int dtype, const void* A, long lda, const float* sums, int count, int width, float eps, const void* W, long ldw,
                                const float* bias, void* qkv, long ld, int M, int K, const float* cos_t, const float* sin_t, const int* slots,
                                void* keys, void* values, int q_heads, int kv_heads, int head_dim, int rot, int page_size, int write_cache,
                                int adjacent, int behind, hipStream_t stream) {
  TW_REQUIRE(q_heads > 0 && kv_heads > 0 && head_dim > 0 && head_dim % 16 == 0 && page_size > 0 && behind >= 0 && behind % 16 == 0);
  const int N = (q_heads + 2 * kv_heads) * head_dim + behind;
  TW_REQUIRE(few_rows_ok(dtype, A, lda, W, ldw, M, N, K) && qkv != nullptr && ld >= N && rot >= 0 && rot % 16 == 0 && rot <= head_dim);
  TW_REQUIRE(rot == 0 || (cos_t && sin_t));
  TW_REQUIRE(!write_cache || (slots && keys && values));
  TW_REQUIRE(sums == nullptr || (norms_ok(sums, count, eps) && width > 0));
  const EndRotate end = {cos_t, sin_t, slots, keys, values, q_heads, kv_heads, head_dim, rot, page_size, write_cache, adjacent};
  auto run = [&](auto t, auto norms) {
    typedef decltype(t) T;
    return launch_narrow<T, T, false, false, decltype(norms)>((const T*)A, lda, (const T*)W, ldw, bias, nullptr, 0, (T*)qkv, ld, M, N, K, stream,
                                                              norms, end);
  };
  const RowNorms norms = {sums, count, (float)width, eps};
  if (dtype == TW_DTYPE_F32) return sums ? run(float{}, norms) : run(float{}, RowsAsTheyAre{});
  return sums ? run(bf16_t{}, norms) : run(bf16_t{}, RowsAsTheyAre{});
}
