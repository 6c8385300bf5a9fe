// Linear layers for many rows (prompt portions): LDS-staged MFMA tiles. See gemm.hip for the
// weight layouts and the GLU form; this file holds the kernel, its epilogue and its launcher.
#include "gemm_shared.h"
#include <math.h>
#include <algorithm>

// f(integral_constant<int, 0>), ..., f(integral_constant<int, N - 1>): a loop whose index is a constant
// expression in the body (the scheduler's group barriers take constants only)
template <int... Is, typename F>
__device__ __forceinline__ void tw_unroll_impl(std::integer_sequence<int, Is...>, F&& f) {
  (f(std::integral_constant<int, Is>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void tw_unroll(F&& f) {
  tw_unroll_impl(std::make_integer_sequence<int, N>{}, f);
}

// A wave's private use of LDS: its own writes are seen by its own later reads (a wave's LDS operations are executed in
// order), the compiler only has to leave them in that order.
__device__ __forceinline__ void tw_wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Epilogue of the tiled kernels: each wave passes its tile through LDS (32 rows at a time) so
// that a lane stores 8 consecutive columns of one row, whole cache lines instead of 2- or 4-byte
// pieces; bias, residual, the output type and the SiLU-multiply of GLU pairs are applied here.
// `lds` must hold 4 waves x (32 rows x (32 * WN + 4) + 32 * WN) floats and no wave may still read its old contents
// (the __syncthreads below sees to that; afterwards every wave works in its own part).
//
// What bounds it is the instruction cache (64 KB, shared by two CUs). Unrolled over the row blocks, the rounds and the
// eight values of a lane, with every activation inlined at every value, it was 14,000 (gated) to 26,000 instructions, and a
// gated tile also spilled its accumulators: a tile spent a quarter of its time there. Now only the row blocks are written out
// (the copy of the accumulators into LDS must name its registers), a round is a loop of a few hundred instructions, and the
// activation is asked for once a round. 256x256 tiles, K = 3,584, bfloat16: the gated projection of 2,048 rows x 37,888
// columns 653 -> 491 us, of 8,192 rows 2,479 -> 1,832 us (898 -> 1,215 TFLOP/s); plain products 2 to 5 %.
template <typename OutT, int WM, int WN, bool GLU>
__device__ __forceinline__ void tw_tiled_epilogue(f32x16 (&acc)[WM][WN], char* lds, const float* __restrict__ bias,
                                                  const float* residual, long ldr, OutT* C, long ldc, int M, int N,
                                                  int m0, int n0, int wm0, int wn0, int wave, int lane) {
  const int r = lane & 31, g = lane >> 5;
  constexpr int WCOLS = 32 * WN;                             // columns of a wave tile
  constexpr int EROW = WCOLS + 4;                            // floats per staged row, padded
  constexpr int CPR = WCOLS / 8;                             // 8-column groups per row
  const bool vec_ok = (ldc % 8 == 0) && (residual == nullptr || ldr % 4 == 0) &&
                      ((uintptr_t)C % 16 == 0) && ((uintptr_t)residual % 16 == 0);
  // The GLU form reads its staged rows in another pattern: a lane takes 8 gate and 8 up values, 16 columns
  // apart, and the lanes of a row take column groups that are 256 bytes (all 64 banks) apart. With padded
  // rows those reads met 4-way bank conflicts (a quarter of the LDS time of a whole gate_up GEMM). Where a
  // wave tile's row is a multiple of 256 bytes the rows are not padded and the 16-byte pieces of row lr lie
  // at piece ^ (0, 1, 4, 5)[lr % 4]: the 16 lanes that a 16-byte read serves in one pass (four rows, four
  // column groups each) then find 16 different 16-byte columns.
  constexpr bool SWIZZLED = GLU && WCOLS % 64 == 0;
  constexpr int SROW = SWIZZLED ? WCOLS : EROW;
  float* stage = reinterpret_cast<float*>(lds) + wave * 32 * SROW;
  // A plain product's bias: the wave's columns of it go to LDS once, behind all waves' rows (read from memory in front of
  // every store it cost a fifth of a qkv projection's time at 2,048 rows; in registers a lane needs up to three groups of it).
  float* bias_stage = reinterpret_cast<float*>(lds) + 4 * 32 * EROW + wave * WCOLS;
  auto swz = [](int row) { return SWIZZLED ? ((row & 1) | ((row & 2) << 1)) : 0; };

  // A residual that is added to whole rows: all of a row block's values of it are requested in front of the copy into LDS
  // (in the loop every round would wait for its own: C may be the residual, so no load passes a store).
  constexpr int ROUNDS = 32 * CPR / 64;
  auto whole = [&](int i) { return vec_ok && m0 + wm0 + i * 32 + 32 <= M && n0 + wn0 + WCOLS <= N; };   // (row block i of the wave)
  f32x4 res[GLU ? 1 : ROUNDS][2];
  auto request = [&](int i) {
#pragma unroll
    for (int t = 0; t < ROUNDS; ++t) {
      const int q = lane + 64 * t;
      const float* src = residual + (size_t)(m0 + wm0 + i * 32 + q / CPR) * ldr + n0 + wn0 + (q % CPR) * 8;
      res[t][0] = *reinterpret_cast<const f32x4*>(src);
      res[t][1] = *reinterpret_cast<const f32x4*>(src + 4);
    }
  };
  auto finish_ahead = [&](int i) {
#pragma unroll
    for (int t = 0; t < ROUNDS; ++t) {
      const int q = lane + 64 * t;
      const int lr = q / CPR, lc = (q % CPR) * 8;
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = stage[lr * EROW + lc + e];
      if (bias) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] += bias_stage[lc + e];
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) { v[e] += res[t][0][e]; v[4 + e] += res[t][1][e]; }
      OutT* dst = C + (size_t)(m0 + wm0 + i * 32 + lr) * ldc + n0 + wn0 + lc;
      if (sizeof(OutT) == 4) {
        *reinterpret_cast<f32x4*>(dst) = f32x4{v[0], v[1], v[2], v[3]};
        *reinterpret_cast<f32x4*>(dst + 4) = f32x4{v[4], v[5], v[6], v[7]};
      } else {
        bf16x8 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = (bf16_t)v[e];
        *reinterpret_cast<bf16x8*>(dst) = o;
      }
    }
  };
  // The same without a residual or an activation, for 128x128 tiles: their four rounds fit the instruction cache side by side (as a
  // loop each round waits for its own reads of LDS: 1,024 x 4,096 x 896 in bfloat16 15.3 us, so 13.7; with the activations in it,
  // too, the kernel takes so many registers that a CU holds one workgroup instead of two: 20 % slower).
  constexpr bool SMALL = !GLU && WM * WN <= 4;
  const long act = residual == nullptr ? ldr : 0;             // (no residual: the stride names an activation, see tw_act)
  auto finish_at_once = [&](int i) {
    float v[ROUNDS][8];
#pragma unroll
    for (int t = 0; t < ROUNDS; ++t) {
      const int q = lane + 64 * t;
#pragma unroll
      for (int e = 0; e < 8; ++e) v[t][e] = stage[(q / CPR) * EROW + (q % CPR) * 8 + e];
    }
    if (bias) {
#pragma unroll
      for (int t = 0; t < ROUNDS; ++t)
#pragma unroll
        for (int e = 0; e < 8; ++e) v[t][e] += bias_stage[((lane + 64 * t) % CPR) * 8 + e];
    }
#pragma unroll
    for (int t = 0; t < ROUNDS; ++t) {
      const int q = lane + 64 * t;
      OutT* dst = C + (size_t)(m0 + wm0 + i * 32 + q / CPR) * ldc + n0 + wn0 + (q % CPR) * 8;
      if (sizeof(OutT) == 4) {
        *reinterpret_cast<f32x4*>(dst) = f32x4{v[t][0], v[t][1], v[t][2], v[t][3]};
        *reinterpret_cast<f32x4*>(dst + 4) = f32x4{v[t][4], v[t][5], v[t][6], v[t][7]};
      } else {
        bf16x8 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = (bf16_t)v[t][e];
        *reinterpret_cast<bf16x8*>(dst) = o;
      }
    }
  };
  // rows i * 32 .. + 31 of any other plain product
  auto finish = [&](int i) {
#pragma unroll 1
    for (int q = lane; q < 32 * CPR; q += 64) {
      const int lr = q / CPR, lc = (q % CPR) * 8;
      const int row = m0 + wm0 + i * 32 + lr, col = n0 + wn0 + lc;
      if (row >= M || col >= N) continue;
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = stage[lr * EROW + lc + e];
      if (bias) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] += bias_stage[lc + e];
      }
      if (act == TW_ACT_RELU_SQUARED) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = tw_act(v[e], TW_ACT_RELU_SQUARED);
      } else if (act == TW_ACT_GELU_ERF) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = tw_act(v[e], TW_ACT_GELU_ERF);
      }
      if (vec_ok && col + 8 <= N) {
        if (residual) {
          const f32x4 r0 = *reinterpret_cast<const f32x4*>(residual + (size_t)row * ldr + col);
          const f32x4 r1 = *reinterpret_cast<const f32x4*>(residual + (size_t)row * ldr + col + 4);
#pragma unroll
          for (int e = 0; e < 4; ++e) { v[e] += r0[e]; v[4 + e] += r1[e]; }
        }
        OutT* dst = C + (size_t)row * ldc + col;
        if (sizeof(OutT) == 4) {
          *reinterpret_cast<f32x4*>(dst) = f32x4{v[0], v[1], v[2], v[3]};
          *reinterpret_cast<f32x4*>(dst + 4) = f32x4{v[4], v[5], v[6], v[7]};
        } else {
          bf16x8 o;
#pragma unroll
          for (int e = 0; e < 8; ++e) o[e] = (bf16_t)v[e];
          *reinterpret_cast<bf16x8*>(dst) = o;
        }
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (col + e < N) {
            float x = v[e];
            if (residual) x += residual[(size_t)row * ldr + col + e];
            C[(size_t)row * ldc + col + e] = tw_from_float<OutT>(x);
          }
      }
    }
  };
  // the same rows of a gated product: a wave tile's columns are [gate 16 | up 16] pairs, a lane forms 8 outputs of one row
  auto finish_glu = [&](int i) {
    constexpr int GPR = WCOLS / 16;                           // 8-output groups per row
#pragma unroll 1
    for (int q = lane; q < 32 * GPR; q += 64) {
      const int lr = q / GPR, og = q % GPR;
      const int lc = (og >> 1) * 32 + (og & 1) * 8;           // gate columns lc.., up columns lc + 16..
      const int row = m0 + wm0 + i * 32 + lr, col = n0 + wn0 + lc;
      if (row >= M || col + 24 > N) continue;                 // N is a multiple of 32: groups are whole
      float v[8], gv[8], uv[8];
      if (SWIZZLED) {
        const float* base = stage + lr * SROW;
        const int piece = lc >> 2, x = swz(lr);
        const f32x4 g0 = *reinterpret_cast<const f32x4*>(base + ((piece ^ x) << 2));
        const f32x4 g1 = *reinterpret_cast<const f32x4*>(base + (((piece + 1) ^ x) << 2));
        const f32x4 u0 = *reinterpret_cast<const f32x4*>(base + (((piece + 4) ^ x) << 2));
        const f32x4 u1 = *reinterpret_cast<const f32x4*>(base + (((piece + 5) ^ x) << 2));
#pragma unroll
        for (int e = 0; e < 4; ++e) { gv[e] = g0[e]; gv[4 + e] = g1[e]; uv[e] = u0[e]; uv[4 + e] = u1[e]; }
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) { gv[e] = stage[lr * SROW + lc + e]; uv[e] = stage[lr * SROW + lc + 16 + e]; }
      }
      if (bias) {
#pragma unroll
        for (int e = 0; e < 8; ++e) { gv[e] += bias[col + e]; uv[e] += bias[col + 16 + e]; }
      }
      if (ldr == 0) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = tw_glu(gv[e], uv[e], 0);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = tw_glu(gv[e], uv[e], ldr);
      }
      OutT* dst = C + (size_t)row * ldc + (n0 + wn0) / 2 + (og >> 1) * 16 + (og & 1) * 8;
      if (ldc % 8 == 0 && (uintptr_t)C % 16 == 0) {
        if (sizeof(OutT) == 4) {
          *reinterpret_cast<f32x4*>(dst) = f32x4{v[0], v[1], v[2], v[3]};
          *reinterpret_cast<f32x4*>(dst + 4) = f32x4{v[4], v[5], v[6], v[7]};
        } else {
          bf16x8 o;
#pragma unroll
          for (int e = 0; e < 8; ++e) o[e] = (bf16_t)v[e];
          *reinterpret_cast<bf16x8*>(dst) = o;
        }
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) dst[e] = tw_from_float<OutT>(v[e]);
      }
    }
  };

  __syncthreads();                                            // the pipeline's LDS reads are done
  if (!GLU && bias)
    for (int c = lane; c < WCOLS; c += 64) bias_stage[c] = n0 + wn0 + c < N ? bias[n0 + wn0 + c] : 0.f;
#pragma unroll
  for (int i = 0; i < WM; ++i) {
    if constexpr (!GLU) {
      if (residual != nullptr && whole(i)) request(i);
    }
    tw_wave_lds_fence();                                      // (the last round's reads come first)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int srow = 8 * (e / 4) + 4 * g + (e % 4);
        stage[srow * SROW + (((j * 8 + (r >> 2)) ^ swz(srow)) << 2) + (r & 3)] = acc[i][j][e];
      }
    tw_wave_lds_fence();
    if constexpr (GLU) {
      finish_glu(i);
    } else {
      if (residual != nullptr && whole(i)) finish_ahead(i);
      else if (SMALL && residual == nullptr && act == 0 && whole(i)) finish_at_once(i);
      else finish(i);
    }
  }
}

// =====================================================================================
// Tiled kernel. Workgroup = 4 waves in a 2x2 grid, wave tile (32*WM) x (32*WN): tiles of 128x128
// (two workgroups per CU), 128x256 and 256x256 (one per CU, the accumulators in AGPRs). bfloat16; float32: gemm_parts_kernel below.
// One stage holds 128 bytes of K per row (64 elements), rows padded to 144
// bytes in LDS so that 16-byte fragment reads of 8 consecutive lanes hit
// distinct banks. Two stages: the next stage's global loads are in flight
// while the current one is multiplied.
// =====================================================================================
#define TW_LDS_ROW 144

// SHUF: W is in the shuffled layout and ldw is its k_steps. GLU: see the top of the file.
template <typename T, typename OutT, int WM, int WN, bool SHUF, bool GLU>
__global__ __launch_bounds__(256) void gemm_tiled_kernel(const T* __restrict__ A, long lda,
                                                         const T* __restrict__ W, long ldw,
                                                         const float* __restrict__ bias,
                                                         const float* residual, long ldr, OutT* C,
                                                         long ldc, int M, int N, int K, int tiles_m,
                                                         int n_blocks, int splits, float* __restrict__ partial) {
  typedef typename Elem<T>::Frag Frag;
  constexpr int EPF = Elem<T>::kPerFrag;
  constexpr int KCH = 8;                                    // 16-byte chunks of K per row and stage
  constexpr int BK = KCH * EPF;
  constexpr int BM = 64 * WM, BN = 64 * WN;
  constexpr int LROW = KCH * 16 + 16;                       // LDS bytes per row of a stage, padded
  constexpr int A_LOADS = BM * KCH / 256, W_LOADS = BN * KCH / 256;
  constexpr int STAGE = (BM + BN) * LROW;                   // bytes of one stage: A rows then W rows
  extern __shared__ __attribute__((aligned(16))) char lds[];

  // Blocks are dealt to the 8 XCDs round-robin; give each XCD a contiguous run
  // of tiles so that neighbours sharing a weight tile share an L2.
  const int per_xcd = gridDim.x / 8;
  const int logical = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
  if (logical >= n_blocks) return;
  // splits > 1 (few tiles, long K): the k-tiles are dealt to `splits` workgroups per tile, which
  // leave float32 partial sums partial[split][M][N] for splitk_reduce_kernel.
  const int n_tiles = n_blocks / splits;
  const int split = logical / n_tiles, tile = logical % n_tiles;
  // Tiles in bands of 2,048 rows, so that the workgroups an XCD runs at a time share column tiles as
  // well as row tiles (all the row tiles of a tall matrix in one column would share one weight tile
  // and fetch an activation tile each).
  constexpr int BAND = 2048 / BM;
  const int tiles_n = n_tiles / tiles_m;
  const int band = tile / (BAND * tiles_n), in_band = tile - band * BAND * tiles_n;
  const int band_rows = min(BAND, tiles_m - band * BAND);
  const int tile_m = band * BAND + in_band % band_rows, tile_n = in_band / band_rows;
  const int m0 = tile_m * BM, n0 = tile_n * BN;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm0 = (wave >> 1) * 32 * WM, wn0 = (wave & 1) * 32 * WN;
  const int r = lane & 31, g = lane >> 5;

  f32x16 acc[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  // Global addressing: a tile base that is the same for every lane, plus per-thread element
  // offsets fixed for the whole K loop. Rows past the end are clamped to the last valid row
  // (what they produce is never stored), so whole k-tiles need no predicate.
  const T* a_tile = A + (size_t)m0 * lda;
  const T* w_tile = SHUF ? W + (size_t)(n0 / 16) * ldw * 64 * EPF : W + (size_t)n0 * ldw;
  const int k_steps_w = SHUF ? (int)ldw : 0;
  unsigned a_off[A_LOADS], w_off[W_LOADS];
  int st_off[A_LOADS];
#pragma unroll
  for (int i = 0; i < A_LOADS; ++i) {
    const int c = tid + i * 256, row = c / KCH, kc = c % KCH;
    a_off[i] = (unsigned)(min(m0 + row, M - 1) - m0) * (unsigned)lda + kc * EPF;
  }
  constexpr int SPT = KCH / 4;                             // shuffled k-steps per k-tile
  int w_st_off[W_LOADS], w_ks[W_LOADS];
  const int n_blocks_w = (N + 15) / 16;
#pragma unroll
  for (int i = 0; i < W_LOADS; ++i) {
    const int c = tid + i * 256;
    if (SHUF) {
      // piece c of the tile: block (16 rows x 4 chunks) c / 64, lane c % 64 of that block
      const int blk = c >> 6, ln = c & 63, nblk = blk / SPT, ks = blk % SPT;
      const int gblk = min(n0 / 16 + nblk, n_blocks_w - 1);
      w_off[i] = (unsigned)(gblk - n0 / 16) * (unsigned)ldw * 64 * EPF + (ks * 64 + ln) * EPF;
      w_ks[i] = ks;
      w_st_off[i] = (nblk * 16 + (ln & 15)) * LROW + (ks * 4 + (ln >> 4)) * 16;
    } else {
      const int row = c / KCH, kc = c % KCH;
      w_off[i] = (unsigned)(min(n0 + row, N - 1) - n0) * (unsigned)ldw + kc * EPF;
      w_ks[i] = 0;
      w_st_off[i] = row * LROW + kc * 16;
    }
  }
#pragma unroll
  for (int i = 0; i < A_LOADS; ++i) {
    const int c = tid + i * 256, row = c / KCH, kc = c % KCH;
    st_off[i] = row * LROW + kc * 16;
  }
  const int kc_mine = tid % KCH;

  // Two register sets: the global loads of k-tile kt+2 are issued while k-tile kt is multiplied,
  // so two k-tiles per workgroup are on their way from memory at any time.
  Frag a_regs[2][A_LOADS], w_regs[2][W_LOADS];
  const int k_tiles_all = (K + BK - 1) / BK;
  const int per_split = (k_tiles_all + splits - 1) / splits;
  const int kt0 = split * per_split;                          // this workgroup's k-tiles: kt0 .. kt0 + k_tiles - 1
  const int k_tiles = max(0, min(k_tiles_all, kt0 + per_split) - kt0);
  const int whole_tiles = K / BK;

  // whole k-tiles need no predicate at all; the main loop below runs only those
  auto load_whole = [&](int kt, Frag* a_reg, Frag* w_reg) {
    const T* ab = a_tile + (size_t)kt * BK;
    const T* wb = SHUF ? w_tile + (size_t)kt * SPT * 64 * EPF : w_tile + (size_t)kt * BK;
#pragma unroll
    for (int i = 0; i < A_LOADS; ++i) a_reg[i] = tw_load_frag(ab + a_off[i]);
#pragma unroll
    for (int i = 0; i < W_LOADS; ++i) w_reg[i] = tw_load_frag(wb + w_off[i]);
  };
  auto load_global = [&](int kt, Frag* a_reg, Frag* w_reg) {
    if (kt < whole_tiles) {
      load_whole(kt, a_reg, w_reg);
    } else {                                                // the last, partial k-tile: chunks past K are zeros
      const T* ab = a_tile + (size_t)kt * BK;
      const T* wb = SHUF ? w_tile + (size_t)kt * SPT * 64 * EPF : w_tile + (size_t)kt * BK;
      const bool ok = kt * BK + kc_mine * EPF < K;
#pragma unroll
      for (int i = 0; i < A_LOADS; ++i) a_reg[i] = ok ? tw_load_frag(ab + a_off[i]) : Elem<T>::zero();
#pragma unroll
      for (int i = 0; i < W_LOADS; ++i) {
        const bool w_ok = SHUF ? kt * SPT + w_ks[i] < k_steps_w : ok;     // the shuffled layout is zero padded
        w_reg[i] = w_ok ? tw_load_frag(wb + w_off[i]) : Elem<T>::zero();
      }
    }
  };
  auto store_lds = [&](int buf, const Frag* a_reg, const Frag* w_reg) {
    char* base = lds + buf * STAGE;
#pragma unroll
    for (int i = 0; i < A_LOADS; ++i) *reinterpret_cast<Frag*>(base + st_off[i]) = a_reg[i];
#pragma unroll
    for (int i = 0; i < W_LOADS; ++i) *reinterpret_cast<Frag*>(base + BM * LROW + w_st_off[i]) = w_reg[i];
  };

  // this lane's fragment addresses in stage 0 (k-chunk pair cc adds 32 bytes)
  const char* a_frag = lds + (wm0 + r) * LROW + g * 16;
  const char* w_frag = lds + (BM + wn0 + r) * LROW + g * 16;
  auto read_frags = [&](int buf, int cc, Frag* af, Frag* wf) {
#pragma unroll
    for (int i = 0; i < WM; ++i)
      af[i] = *reinterpret_cast<const Frag*>(a_frag + buf * STAGE + i * 32 * LROW + cc * 32);
#pragma unroll
    for (int j = 0; j < WN; ++j)
      wf[j] = *reinterpret_cast<const Frag*>(w_frag + buf * STAGE + j * 32 * LROW + cc * 32);
  };

  auto multiply = [&](int buf) {
    // the fragments of the next k-chunk pair are read from LDS while this one is multiplied
    Frag af[2][WM], wf[2][WN];
    read_frags(buf, 0, af[0], wf[0]);
#pragma unroll
    for (int cc = 0; cc < KCH / 2; ++cc) {
      if (cc + 1 < KCH / 2) read_frags(buf, cc + 1, af[(cc + 1) & 1], wf[(cc + 1) & 1]);
#pragma unroll
      for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j) tw_mma32(acc[i][j], af[cc & 1][i], wf[cc & 1][j]);
    }
  };

  if (k_tiles > 0) {
    load_global(kt0, a_regs[0], w_regs[0]);
    if (k_tiles > 1) load_global(kt0 + 1, a_regs[1], w_regs[1]);
    store_lds(0, a_regs[0], w_regs[0]);
  }
  __syncthreads();
  int j = 0;                                                  // k-tile kt0 + j is in LDS stage j & 1
  // Main loop: two k-tiles per round, every load whole and unconditional, so that the register
  // sets are plain loop-carried values (conditional loads cost a register copy per loaded dword).
  const int whole_here = min(k_tiles, whole_tiles - kt0);
  // The order asked of the scheduler for each k-tile: per k-chunk pair its MFMAs, before them the
  // LDS reads of the next pair, a quarter of the next-but-one k-tile's global loads and a quarter of
  // the next k-tile's LDS writes. Left alone, the compiler puts loads, writes and MFMAs in three
  // clusters, and the memory pipes and the matrix unit take turns instead of working side by side.
#define TW_SGB(mask, n) __builtin_amdgcn_sched_group_barrier(mask, n, 0)
#define TW_TILE_ORDER()                                                                     \
  do {                                                                                      \
    constexpr int MOVES = (A_LOADS + W_LOADS) / 4;                                          \
    TW_SGB(0x100, WM + WN);                                                                 \
    TW_SGB(0x100, WM + WN); TW_SGB(0x020, MOVES); TW_SGB(0x200, MOVES); TW_SGB(0x008, WM * WN); \
    TW_SGB(0x100, WM + WN); TW_SGB(0x020, MOVES); TW_SGB(0x200, MOVES); TW_SGB(0x008, WM * WN); \
    TW_SGB(0x100, WM + WN); TW_SGB(0x020, MOVES); TW_SGB(0x200, MOVES); TW_SGB(0x008, WM * WN); \
    TW_SGB(0x020, MOVES); TW_SGB(0x200, MOVES); TW_SGB(0x008, WM * WN);                     \
  } while (0)
  for (; j + 3 < whole_here; j += 2) {
    load_whole(kt0 + j + 2, a_regs[0], w_regs[0]);           // LDS stage 0, register set 0 is free
    multiply(0);
    store_lds(1, a_regs[1], w_regs[1]);
    TW_TILE_ORDER();
    __syncthreads();
    load_whole(kt0 + j + 3, a_regs[1], w_regs[1]);           // LDS stage 1, register set 1 is free
    multiply(1);
    store_lds(0, a_regs[0], w_regs[0]);
    TW_TILE_ORDER();
    __syncthreads();
  }
#undef TW_TILE_ORDER
#undef TW_SGB
  // The last few k-tiles (j is even here): the same rounds with every step conditional.
  for (; j < k_tiles; j += 2) {
    if (j + 2 < k_tiles) load_global(kt0 + j + 2, a_regs[0], w_regs[0]);
    multiply(0);
    if (j + 1 < k_tiles) store_lds(1, a_regs[1], w_regs[1]);
    __syncthreads();
    if (j + 1 >= k_tiles) break;
    if (j + 3 < k_tiles) load_global(kt0 + j + 3, a_regs[1], w_regs[1]);
    multiply(1);
    if (j + 2 < k_tiles) store_lds(0, a_regs[0], w_regs[0]);
    __syncthreads();
  }

  if (splits > 1) {
    tw_tiled_epilogue<float, WM, WN, false>(acc, lds, nullptr, nullptr, 0, partial + (size_t)split * M * N, (long)N,
                                            M, N, m0, n0, wm0, wn0, wave, lane);
    return;
  }
  tw_tiled_epilogue<OutT, WM, WN, GLU>(acc, lds, bias, residual, ldr, C, ldc, M, N, m0, n0, wm0, wn0, wave, lane);
}

// =====================================================================================
// float32: every operand as the sum of three bfloat16 numbers, on the bfloat16 matrix unit.
//
// x = 2^-24 (h + m + l) exactly (tw_three_parts; a known method), and a product of two parts is exact in the matrix unit, which adds in float32. Of
// the nine products l l alone, below 2^-34 of the whole, is left out; the other eight are added with the smallest first, all but h h into
// sums of their own, which keeps their roundings away from the large sums. So a product by itself is as good as float32's own
// (one element of a row not zero: off by 0.995 x 2^-24 at the most and 0.426 in the mean square, by the float32 MFMA 0.994 and 0.426; with m l and
// l m left out too 1.71 and 0.438, with parts that are cut off instead of rounded as well 6.6 and 1.11, always towards zero), and a sum is
// rounded less often than by the float32 MFMA, which adds two products at a time.
//
// Why: the float32 MFMA takes 64 cycles for 32x32x2, the bfloat16 one 32 for 32x32x16, so eight of these are twice as fast. Workgroup =
// 4 waves in a 2x2 grid, wave tile (32*WM) x (32*WN): 128x128, 64x128 and 64x64. A k-tile is 32 elements of K; it is split once, on its way
// from registers to LDS (6.5 vector instructions an element), while the next one is on its way from memory, and two to five workgroups
// share a CU, so that one splits while another multiplies. A row of a part is 64 bytes of LDS, four pieces of 16, piece p at
// p ^ (row / 4 % 4): the 16 rows that a pass of a fragment read takes, and the 8 lanes of a write, are in different banks.
//
// Against the float32 MFMA (128x128 tiles, two LDS stages, the K ranges of tiled_splits): 478 x 10,432 x 2,048 271 -> 163 us, 478 x 2,048 x
// 4,096 108 -> 67, 4,096 x 32,000 x 2,048 4,314 -> 3,430 (157 TFLOP/s, so 1.25 PFLOP/s in bfloat16, where power is the bound), 65 x 896 x 4,864
// 46 -> 22; 109 random products (65 to 3,000 rows) take 0.55 of the time, the slowest 0.92. (With six products 137, 57, 2,817 and 20;
// 0.49. The factor of 2^24 costs 0 to 4 %.) Their error against 64 bits is 0.35 of what it was in the mean and 0.77 at the most. Rows of 4 to 2,048 elements, of 2^-24 of the sum of
// sizes, largest and mean square (float32 MFMA / this): dense 2.4 to 4.3 and 0.45 to 0.47 / 1.5 to 2.2 and 0.15 to 0.30, all of one sign 58 and
// 11.8 / 18 and 4.2, four elements not zero 2.7 and 0.45 / 2.1 and 0.34, the first element 2^14 times the others 103 and 14.6 / 30 and 5.2.
// What the float32 MFMA does better is a row whose LAST element is 2^14 times the others, 3.0 and 0.42 / 5.0 and 0.95: 16 products meet
// in one instruction, which lines them all up with the largest.
//
// A value of 2^104 and more, an infinity or NaN has no such parts, and every result that it enters is then not finite (nor is a result of 2^79
// and more, 2^48 of whose products are summed). So a tile with such a result is formed again by the float32 MFMA from the operands
// themselves, and infinities, NaN and sums that overflow are what they are there. The tile's other results stay the parts' sums: a row's
// bits do not depend on what its neighbours hold.
// =====================================================================================
template <int WM, int WN, bool SHUF, bool GLU>
__global__ __launch_bounds__(256, WM * WN == 1 ? 5 : 2) void gemm_parts_kernel(const float* __restrict__ A, long lda, const float* __restrict__ W, long ldw,
                                                            const float* __restrict__ bias, const float* residual, long ldr, float* C,
                                                            long ldc, int M, int N, int K, int tiles_m, int n_blocks, int splits,
                                                            float* __restrict__ partial) {
  constexpr int BM = 64 * WM, BN = 64 * WN, BK = 32;
  constexpr int A_PIECES = BM * 4 / 256, W_PIECES = BN * 4 / 256;       // of 8 elements of K, a thread's
  constexpr int PART = (BM + BN) * TW_PART_ROW;
  extern __shared__ __attribute__((aligned(16))) char lds[];

  // (workgroups, K ranges and bands as in gemm_tiled_kernel)
  const int per_xcd = gridDim.x / 8;
  const int logical = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
  if (logical >= n_blocks) return;
  const int n_tiles = n_blocks / splits;
  const int split = logical / n_tiles, tile = logical % n_tiles;
  constexpr int BAND = 2048 / BM;
  const int tiles_n = n_tiles / tiles_m;
  const int band = tile / (BAND * tiles_n), in_band = tile - band * BAND * tiles_n;
  const int band_rows = min(BAND, tiles_m - band * BAND);
  const int tile_m = band * BAND + in_band % band_rows, tile_n = in_band / band_rows;
  const int m0 = tile_m * BM, n0 = tile_n * BN;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm0 = (wave >> 1) * 32 * WM, wn0 = (wave & 1) * 32 * WN;
  const int r = lane & 31, g = lane >> 5;

  f32x16 acc[WM][WN], small[WM][WN];                           // the sums of h h, and of the other products
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = small[i][j][e] = 0.f;

  // A thread's pieces: a base that is the same for every lane and offsets fixed for the whole of K. Rows past the end are clamped to
  // the last one (what they produce is never stored).
  const float* a_tile = A + (size_t)m0 * lda;
  const float* w_tile = SHUF ? W + (size_t)(n0 / 16) * ldw * 256 : W + (size_t)n0 * ldw;
  const int n_blocks_w = (N + 15) / 16;
  unsigned a_off[A_PIECES], w_off[W_PIECES];
  int a_st[A_PIECES], w_st[W_PIECES], w_k[W_PIECES];          // the piece's place in LDS; its first k (chunks of 4 that begin past K are zeros)
#pragma unroll
  for (int i = 0; i < A_PIECES; ++i) {
    const int c = tid + i * 256, row = c >> 2, p = c & 3;
    a_off[i] = (unsigned)(min(m0 + row, M - 1) - m0) * (unsigned)lda + p * 8;
    a_st[i] = tw_part_place(row, p);
  }
#pragma unroll
  for (int i = 0; i < W_PIECES; ++i) {
    const int c = tid + i * 256;
    if (SHUF) {                                                // 16 rows of a block, then the pieces of its two k-steps
      const int row = (c >> 6) * 16 + (c & 15), p = (c >> 4) & 3;
      const int gblk = min(n0 / 16 + (c >> 6), n_blocks_w - 1);
      w_off[i] = (unsigned)(gblk - n0 / 16) * (unsigned)ldw * 256 + (p >> 1) * 256 + (p & 1) * 128 + (c & 15) * 4;
      w_st[i] = BM * TW_PART_ROW + tw_part_place(row, p);
      w_k[i] = p * 8;
    } else {
      const int row = c >> 2, p = c & 3;
      w_off[i] = (unsigned)(min(n0 + row, N - 1) - n0) * (unsigned)ldw + p * 8;
      w_st[i] = BM * TW_PART_ROW + tw_part_place(row, p);
      w_k[i] = p * 8;
    }
  }
  const int a_k = (tid & 3) * 8;
  constexpr int W_NEXT = SHUF ? 64 : 4;                        // floats to the piece's second chunk

  f32x4 a_reg[A_PIECES][2], w_reg[W_PIECES][2];
  const int k_tiles_all = (K + BK - 1) / BK;
  const int per_split = (k_tiles_all + splits - 1) / splits;
  const int kt0 = split * per_split;
  const int k_end = min(k_tiles_all, kt0 + per_split);
  const int whole_tiles = K / BK;

  auto load = [&](int kt) {
    const float* ab = a_tile + (size_t)kt * BK;
    const float* wb = SHUF ? w_tile + (size_t)kt * 512 : w_tile + (size_t)kt * BK;
    if (kt < whole_tiles) {
#pragma unroll
      for (int i = 0; i < A_PIECES; ++i) {
        a_reg[i][0] = tw_load_frag(ab + a_off[i]);
        a_reg[i][1] = tw_load_frag(ab + a_off[i] + 4);
      }
#pragma unroll
      for (int i = 0; i < W_PIECES; ++i) {
        w_reg[i][0] = tw_load_frag(wb + w_off[i]);
        w_reg[i][1] = tw_load_frag(wb + w_off[i] + W_NEXT);
      }
    } else {                                                   // (the shuffled layout ends at a k-step: its chunks past K are zeros)
      const int left = K - kt * BK, w_left = SHUF ? (left + 15) / 16 * 16 : left;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int i = 0; i < A_PIECES; ++i)
          a_reg[i][h] = a_k + 4 * h < left ? tw_load_frag(ab + a_off[i] + 4 * h) : Elem<float>::zero();
#pragma unroll
        for (int i = 0; i < W_PIECES; ++i)
          w_reg[i][h] = w_k[i] + 4 * h < w_left ? tw_load_frag(wb + w_off[i] + W_NEXT * h) : Elem<float>::zero();
      }
    }
  };
  auto split_store = [&]() {
    auto put = [&](int at, const f32x4 (&x)[2]) {
      bf16x8 h, m, l;
      tw_three_parts(x[0], x[1], h, m, l);
      *reinterpret_cast<bf16x8*>(lds + at) = h;
      *reinterpret_cast<bf16x8*>(lds + PART + at) = m;
      *reinterpret_cast<bf16x8*>(lds + 2 * PART + at) = l;
    };
#pragma unroll
    for (int i = 0; i < A_PIECES; ++i) put(a_st[i], a_reg[i]);
#pragma unroll
    for (int i = 0; i < W_PIECES; ++i) put(w_st[i], w_reg[i]);
  };
  const int swz = (r >> 2) & 3;                                // (every fragment's rows begin at a multiple of 16)
  auto multiply = [&]() {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int at = ((2 * s + g) ^ swz) * 16;
      bf16x8 af[3][WM], wf[3][WN];
#pragma unroll
      for (int p = 2; p >= 0; --p) {
#pragma unroll
        for (int i = 0; i < WM; ++i) af[p][i] = *reinterpret_cast<const bf16x8*>(lds + p * PART + (wm0 + i * 32 + r) * TW_PART_ROW + at);
#pragma unroll
        for (int j = 0; j < WN; ++j) wf[p][j] = *reinterpret_cast<const bf16x8*>(lds + p * PART + (BM + wn0 + j * 32 + r) * TW_PART_ROW + at);
      }
      auto product = [&](f32x16 (&sum)[WM][WN], int p, int q) {
#pragma unroll
        for (int i = 0; i < WM; ++i)
#pragma unroll
          for (int j = 0; j < WN; ++j) tw_mma32(sum[i][j], af[p][i], wf[q][j]);
      };
      TW_PART_PRODUCTS(product);
    }
  };

  if (kt0 < k_end) load(kt0);
  for (int kt = kt0; kt < k_end; ++kt) {
    __syncthreads();                                           // (the reads of the k-tile before)
    split_store();
    if (kt + 1 < k_end) load(kt + 1);
    __syncthreads();
    multiply();
  }

  float odd = 0.f;                                             // NaN as soon as one of them is not finite
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        acc[i][j][e] += small[i][j][e];
        odd = __fmaf_rn(acc[i][j][e], 0.f, odd);
      }
  if (__syncthreads_or(odd != odd)) {
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) small[i][j][e] = 0.f;
    const int k_from = kt0 * BK, k_to = min(K, k_end * BK);
    for (int k = k_from; k < k_to; k += 8) {
      f32x4 af[WM], wf[WN];
      const int mine = k + 4 * g;
#pragma unroll
      for (int i = 0; i < WM; ++i) af[i] = mine < K ? tw_load_frag(A + (size_t)min(m0 + wm0 + i * 32 + r, M - 1) * lda + mine) : Elem<float>::zero();
#pragma unroll
      for (int j = 0; j < WN; ++j) {
        const int n = min(n0 + wn0 + j * 32 + r, N - 1);
        const float* w = SHUF ? W + ((size_t)(n >> 4) * ldw + (mine >> 4)) * 256 + ((mine >> 2) & 3) * 64 + (n & 15) * 4 : W + (size_t)n * ldw + mine;
        wf[j] = mine < K ? tw_load_frag(w) : Elem<float>::zero();
      }
#pragma unroll
      for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j) tw_mma32(small[i][j], af[i], wf[j]);
    }
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = acc[i][j][e] * 0.f == 0.f ? acc[i][j][e] * TW_PART_BACK : small[i][j][e];
  } else {
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] *= TW_PART_BACK;
  }

  if (splits > 1)
    tw_tiled_epilogue<float, WM, WN, false>(acc, lds, nullptr, nullptr, 0, partial + (size_t)split * M * N, (long)N, M, N, m0, n0, wm0, wn0,
                                            wave, lane);
  else
    tw_tiled_epilogue<float, WM, WN, GLU>(acc, lds, bias, residual, ldr, C, ldc, M, N, m0, n0, wm0, wn0, wave, lane);
}

// =====================================================================================
// bfloat16, shuffled weights, K a multiple of 32, where gemm_turns_kernel below does not take the product (an odd multiple of 32, rows of
// the result or a residual that are not 16 bytes apart, a bias over a K shorter than the stages: turns_takes) or is the slower
// one (turns_pay): tiles whose operands are copied from global memory straight into LDS (buffer loads of 16 bytes a lane, which land at
// the wave's LDS base + 16 l, from any 32-bit offset the lane names). No staging registers, no LDS write instructions.
// Workgroup = 4 waves in a 2x2 grid, wave tile (32*WM) x (32*WN): 128x256, 256x192, 256x256 (one a CU).
//
// A k-tile is 32 elements of K (one k-step of the shuffled layout). What limits this kernel is the
// number of 128-byte lines a CU's vector cache can have on their way from L2; a copy that takes 64 bytes
// of a row of A brings in the whole line, and by the time the next k-tile wants the other half the line
// is gone again (measured: 1.5 lines fetched per line used). So A is copied in PAIRS of k-tiles, a
// whole line per row: a copy is 8 rows x 128 bytes, and LDS holds TW_DMA_A_SLOTS slots of BM rows x 128
// bytes. In a slot row `row` keeps its 16-byte chunk c (0..3: the even k-tile, 4..7: the odd one) at
// position c ^ (row / 2 % 8), so that the 16 rows one fragment read takes lie in 16 different 16-byte
// columns. W is copied per k-tile into 4 stages; a W block is 16 rows x 4 chunks, [chunk][row], 1 KB,
// which is how W lies in memory (a fragment read takes 256 consecutive bytes per 16 lanes).
//
// Per k-tile and wave: 2 k-chunk pairs of WM*WN MFMAs. The fragments of a pair are read while the
// pair before is multiplied, so the barrier that publishes the next k-tile lies between the two
// pairs of this one and the matrix unit has work queued on both sides of it.
// splits > 1: as in gemm_tiled_kernel (a split's k-tiles begin at an even one).
// =====================================================================================
typedef __attribute__((address_space(3))) void* tw_lds_ptr;
// Copies of 16 bytes a lane from global memory straight into LDS, as BUFFER loads: base + lane's offset + the wave's offset, so
// that a copy takes no address arithmetic (as global loads, with a 64-bit address a lane, they held up the waves that take turns
// below). Offsets within a tile's operands are 32-bit: asked before the kernels are chosen or where they are launched.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t tw_buffer(const void* base) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, 0x7fffffff, 0x00020000);
}
template <int AHEAD = 0>                                     // (bytes further on, in both memories)
__device__ __forceinline__ void tw_copy_to_lds(__amdgpu_buffer_rsrc_t from, char* to, int lane_offset, int wave_offset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(from, (tw_lds_ptr)to, 16, lane_offset, wave_offset, AHEAD, 0);
}
#define TW_DMA_STAGES 4       /* of W, one k-tile each */
#define TW_DMA_A_SLOTS 3      /* of A, a pair of k-tiles each */

template <typename OutT, int WM, int WN, bool GLU>
__global__ __launch_bounds__(256) void gemm_dma_kernel(const bf16_t* __restrict__ A, long lda,
                                                       const bf16_t* __restrict__ W, long k_steps,
                                                       const float* __restrict__ bias, const float* residual,
                                                       long ldr, OutT* C, long ldc, int M, int N, int K,
                                                       int tiles_m, int n_blocks, int splits,
                                                       float* __restrict__ partial) {
  static_assert(WM % 2 == 0, "the tail fix below assumes an even number of A copies per group");
  constexpr int BM = 64 * WM, BN = 64 * WN;
  constexpr int A_SLOT = BM * 128;                      // bytes: a pair of k-tiles of A
  constexpr int W_STAGE = BN * 64;                      // bytes: one k-tile of W
  constexpr int W_RING = TW_DMA_A_SLOTS * A_SLOT;       // the W stages lie behind the A slots
  constexpr int COPIES = WM + WN;                       // 1 KB copies per wave and k-tile
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int per_xcd = gridDim.x / 8;
  const int logical = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;   // neighbours in an XCD share operand tiles
  if (logical >= n_blocks) return;
  const int n_tiles = n_blocks / splits;
  const int split = logical / n_tiles, tile = logical % n_tiles;
  // Tiles in bands of 2,048 rows: the workgroups an XCD runs at a time then share column tiles as well
  // as row tiles (all the row tiles of a tall matrix in one column would fetch an activation tile each).
  constexpr int BAND = 2048 / BM;
  const int tiles_n = n_tiles / tiles_m;
  const int band = tile / (BAND * tiles_n), in_band = tile - band * BAND * tiles_n;
  const int band_rows = min(BAND, tiles_m - band * BAND);
  const int tile_m = band * BAND + in_band % band_rows, tile_n = in_band / band_rows;
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm0 = (wave >> 1) * 32 * WM, wn0 = (wave & 1) * 32 * WN;
  const int r = lane & 31, g = lane >> 5;

  f32x16 acc[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  // this workgroup's k-tiles: kt0 .. kt0 + k_tiles - 1, kt0 even (a pair of k-tiles is never divided)
  const int k_tiles_all = K / 32;
  const int per_split = ((k_tiles_all + splits - 1) / splits + 1) & ~1;
  const int kt0 = split * per_split;
  const int k_tiles = max(0, min(k_tiles_all, kt0 + per_split) - kt0);
  const int pairs = (k_tiles + 1) / 2;
  const bool half_pair = (k_tiles & 1) != 0;               // the last pair has its even k-tile only

  // What this lane copies: per pair of k-tiles its slot of the A blocks (8 rows each) 2 WM wave ..
  // 2 WM wave + 2 WM - 1, in two groups of WM, and per k-tile its slot of the W blocks (16 rows each)
  // WN wave .. WN wave + WN - 1. Rows past M and blocks past N are clamped to the last valid one (their
  // products are never stored).
  const int n_blocks_w = (N + 15) / 16;
  // (A: byte offsets from the tile's first row, for group 0 and from group 0 to group 1; which group a
  // copy belongs to is not known where it is compiled, and a choice between two pointers would put them
  // into memory)
  const auto a_buffer = tw_buffer(A + (size_t)m0 * lda + (size_t)kt0 * 32);
  const auto w_buffer = tw_buffer(W + ((size_t)(n0 / 16) * k_steps + kt0) * 512);
  int a_off[WM], a_step[WM];
  int w_off[WN];
#pragma unroll
  for (int b = 0; b < WM; ++b) {
    int off[2];
#pragma unroll
    for (int grp = 0; grp < 2; ++grp) {
      const int row_in_tile = ((2 * WM) * wave + grp * WM + b) * 8 + (lane >> 3);
      const int chunk = (lane & 7) ^ ((row_in_tile >> 1) & 7);   // slot l % 8 of the row holds this chunk
      off[grp] = min(row_in_tile, M - 1 - m0) * (int)lda * 2 + chunk * 16;
    }
    a_off[b] = off[0];
    a_step[b] = off[1] - off[0];
  }
#pragma unroll
  for (int b = 0; b < WN; ++b) {
    const int block = min(n0 / 16 + WN * wave + b, n_blocks_w - 1) - n0 / 16;
    w_off[b] = block * (int)k_steps * 1024 + lane * 16;
  }
  // In a last pair that has its even k-tile only, the lanes that would fetch chunks 4..7 (past the end of
  // the row, and for the last row perhaps of the matrix) fetch chunks 0..3 again. Whether a lane's chunk
  // is 4..7: bit 2 of l % 8, flipped in every other block of 8 rows.
  const int tail_back[2] = {(lane & 4) ? -64 : 0, (lane & 4) ? 0 : -64};   // bytes
  auto copy_a_one = [&](int pair_v, int grp, int b) {       // (grp, 0 or 1, is the same for the whole wave)
    const int pair = min(pair_v, pairs - 1);               // past the end: a copy nobody reads
    const int tail = (half_pair && pair == pairs - 1) ? -1 : 0;
    char* slot = lds + (pair_v % TW_DMA_A_SLOTS) * A_SLOT;
    const int off = a_off[b] + (a_step[b] & -grp) + (tail_back[b & 1] & tail);
    tw_copy_to_lds(a_buffer, slot + ((2 * WM) * wave + grp * WM + b) * 1024, off, pair * 128);
  };
  auto copy_w_one = [&](int t_v, int b) {
    const int t = min(t_v, k_tiles - 1);
    char* stage = lds + W_RING + (t_v % TW_DMA_STAGES) * W_STAGE;
    tw_copy_to_lds(w_buffer, stage + (WN * wave + b) * 1024, w_off[b], t * 1024);
  };
  // this lane's fragment offsets: A in slot 0 for the k-chunk pairs of an even k-tile (an odd one's
  // chunks are 4 further on: bit 6 of the offset flipped), W in stage 0
  const int a_swz = (r >> 1) & 7;
  const int a_frag[2] = {(wm0 + r) * 128 + ((g ^ a_swz) * 16), (wm0 + r) * 128 + (((2 + g) ^ a_swz) * 16)};
  const char* w_frag = lds + W_RING + (wn0 / 16 + (r >> 4)) * 1024 + g * 256 + (r & 15) * 16;
  // Wait until at most `count` of this wave's copies are in flight (copies finish in order), then meet the
  // other waves. The count is an immediate of the instruction, hence the cases.
#define TW_DMA_WAIT(n) asm volatile("s_waitcnt vmcnt(" #n ") lgkmcnt(0)" ::: "memory")
#define TW_DMA_PUBLISH(count)                                                 \
  do {                                                                        \
    if constexpr ((count) == 6) TW_DMA_WAIT(6);                               \
    else if constexpr ((count) == 8) TW_DMA_WAIT(8);                          \
    else if constexpr ((count) == 10) TW_DMA_WAIT(10);                        \
    else if constexpr ((count) == 12) TW_DMA_WAIT(12);                        \
    else if constexpr ((count) == 14) TW_DMA_WAIT(14);                        \
    else if constexpr ((count) == 16) TW_DMA_WAIT(16);                        \
    else TW_DMA_WAIT(0);                                                      \
    __builtin_amdgcn_s_barrier();                                             \
    asm volatile("" ::: "memory");                                            \
  } while (0)
#define TW_SGB(mask, n) __builtin_amdgcn_sched_group_barrier(mask, n, 0)

  bf16x8 af[2][WM], wf[2][WN];
  // One wave a SIMD issues in order, and the matrix unit takes an MFMA every 32 clocks: whatever else
  // the wave issues between two MFMAs has to fit into that time, or the unit idles. So the other
  // operations of a k-chunk pair follow its MFMAs one by one: first the fragment reads of the next pair
  // (into the other set of registers), then the copies: the W blocks of k-tile t + 3 in the first pair of
  // k-tile t, one group of the A blocks of k-tile pair t / 2 + 2 in the second (the slot those land in
  // held pair t / 2 - 1, last read before the barrier of k-tile 2 (t / 2) - 1). The last MFMAs of a pair
  // have nothing behind them: a copy counts as an access through both memory counters, after which every
  // wait the compiler puts before an MFMA whose operands came from LDS is `lgkmcnt(0)`, and the one before
  // the next pair's first MFMA should find the reads long done. The source is written in the order that
  // is wanted, because a copy writes LDS and the compiler keeps LDS reads on their side of it; the group
  // barriers only pin it.
  auto half = [&](auto copy_is_a, int copy_index, int copy_group, const char* a_read, const char* w_read,
                  bf16x8* af_in, bf16x8* wf_in, bf16x8* af_out, bf16x8* wf_out) {
    constexpr bool IS_A = decltype(copy_is_a)::value;
    constexpr int NCOPY = IS_A ? WM : WN;
    // S slots of one MFMA each; the Q other operations (R fragment reads, then the copies) follow the
    // MFMAs of the first slots one by one (two where there are more operations than slots)
    constexpr int S = WM * WN, R = WM + WN, Q = R + NCOPY;
    tw_unroll<S>([&](auto index) {
      constexpr int slot = decltype(index)::value, i = slot / WN, j = slot % WN;
      tw_mma32(acc[i][j], af_in[i], wf_in[j]);
      constexpr int q0 = Q <= S ? (slot < Q ? slot : Q) : slot * Q / S;
      constexpr int q1 = Q <= S ? (slot + 1 < Q ? slot + 1 : Q) : (slot + 1) * Q / S;
#pragma unroll
      for (int q = q0; q < q1; ++q) {
        if (q < WM) af_out[q] = *reinterpret_cast<const bf16x8*>(a_read + q * 4096);
        else if (q < R) wf_out[q - WM] = *reinterpret_cast<const bf16x8*>(w_read + (q - WM) * 2048);
        else if (IS_A) copy_a_one(copy_index, copy_group, q - R);
        else copy_w_one(copy_index, q - R);
      }
      constexpr int reads_here = (q1 < R ? q1 : R) - (q0 < R ? q0 : R), copies_here = (q1 - q0) - reads_here;
      TW_SGB(0x008, 1);
      if constexpr (reads_here > 0) TW_SGB(0x100, reads_here);
      if constexpr (copies_here > 0) TW_SGB(0x020, copies_here);
    });
  };
  // k-tile t. Its barrier publishes k-tile t + 1. What has to have landed by then and what this wave
  // has issued since: t + 1 odd: W of t + 1 (issued in the first pair of t - 2), since then A, W A, W;
  // t + 1 even: its pair of A, whose second group went out in the second pair of t - 2, since then W A, W.
  // One count for both (the parity of t is not known where the wait is compiled): the smaller.
  auto k_tile = [&](int t) {
    const int odd = t & 1;
    const int a_now = ((t >> 1) % TW_DMA_A_SLOTS) * A_SLOT, a_next = (((t + 1) >> 1) % TW_DMA_A_SLOTS) * A_SLOT;
    const int w_now = (t % TW_DMA_STAGES) * W_STAGE, w_next = ((t + 1) % TW_DMA_STAGES) * W_STAGE;
    half(std::false_type{}, t + TW_DMA_STAGES - 1, 0, lds + ((a_frag[1] ^ (odd << 6)) + a_now), w_frag + w_now + 512,
         af[0], wf[0], af[1], wf[1]);
    __builtin_amdgcn_sched_barrier(0);                     // (nothing of either pair moves across the barrier)
    TW_DMA_PUBLISH(2 * WN + WM);
    __builtin_amdgcn_sched_barrier(0);
    half(std::true_type{}, (t >> 1) + 2, odd, lds + ((a_frag[0] ^ ((odd ^ 1) << 6)) + a_next), w_frag + w_next,
         af[1], wf[1], af[0], wf[0]);                      // (after the last k-tile: read, never used)
    __builtin_amdgcn_sched_barrier(0);                     // (nor into the next k-tile)
  };
  if (k_tiles > 0) {
    // A of pair 0 and W of k-tile 0, then what may still be on its way when k-tile 0 is published:
    // W of k-tile 1, A of pair 1, W of k-tile 2
#pragma unroll
    for (int c = 0; c < 2 * WM; ++c) copy_a_one(0, c / WM, c % WM);
#pragma unroll
    for (int b = 0; b < WN; ++b) copy_w_one(0, b);
#pragma unroll
    for (int b = 0; b < WN; ++b) copy_w_one(1, b);
#pragma unroll
    for (int c = 0; c < 2 * WM; ++c) copy_a_one(1, c / WM, c % WM);
#pragma unroll
    for (int b = 0; b < WN; ++b) copy_w_one(2, b);
    TW_DMA_PUBLISH(2 * COPIES);
#pragma unroll
    for (int i = 0; i < WM; ++i) af[0][i] = *reinterpret_cast<const bf16x8*>(lds + a_frag[0] + i * 4096);
#pragma unroll
    for (int j = 0; j < WN; ++j) wf[0][j] = *reinterpret_cast<const bf16x8*>(w_frag + j * 2048);
    for (int t = 0; t < k_tiles; ++t) k_tile(t);
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");   // no copy may land in the epilogue's staging area
#undef TW_SGB
#undef TW_DMA_PUBLISH
#undef TW_DMA_WAIT
  if (splits > 1) {
    tw_tiled_epilogue<float, WM, WN, false>(acc, lds, nullptr, nullptr, 0, partial + (size_t)split * M * N, (long)N,
                                            M, N, m0, n0, wm0, wn0, wave, lane);
    return;
  }
  tw_tiled_epilogue<OutT, WM, WN, GLU>(acc, lds, bias, residual, ldr, C, ldc, M, N, m0, n0, wm0, wn0, wave, lane);
}

// =====================================================================================
// The same product with EIGHT waves, two a SIMD, that take turns: while one wave of a SIMD multiplies, the other reads its
// next fragments from LDS and issues copies. K a multiple of 64, 16-byte rows of the result.
//
// The waves form a grid of ROWS x 8 / ROWS, each holds 16 RT x 32 Q of the tile: with RT of 4 256 x 64 Q (ROWS 4) or 128 x 128 Q
// (ROWS 2), with 3 192 x 64 Q (for rows that would leave a third of 256 empty).
// A k-tile is 64 elements of K, and a PHASE is 32 columns of a wave's tile in one k-tile: 4 RT MFMAs (256 clocks at 4) between two
// barriers, behind the reads of those columns of W and, in a k-tile's first phase, of the wave's rows of A. Waves 4..7 pass one
// barrier more at the start, so that each wave's reads, copies and waits fall into the time in which the other wave of its
// SIMD multiplies (with one wave a SIMD a copy that misses the vector cache held up the MFMAs behind it: a fifth of the
// matrix unit's time).
//
// LDS holds STAGES k-tiles, filled piece by piece: what phase p read (columns p of W; A, in two halves: p = 0) is replaced by
// the k-tile STAGES further on from phase p + 1 on (A's second half p + 2): a wave waits for its reads of phase p in front of the
// barrier behind which it multiplies, for waves 4..7 the one behind which waves 0..3 issue the first copy of phase p + 1. In
// phase p a wave waits until its copies of what phase p + 1 reads have landed; waves 4..7 do so right before the barrier behind
// which waves 0..3 read it. Copies land in order, so the wait is a count of the younger ones (Turns::wait).
//
// One workgroup a CU takes tile after tile, and the stream of copies runs on from one tile into the next, so that a tile begins
// with its operands in LDS and its result is stored while more arrive. The MFMAs take W as their row operand: a lane then holds
// 4 neighbouring columns of one row of the result, and of a gated product the gate next to its up column, and stores them
// without a trip through LDS (16 bytes a lane of bfloat16 after an exchange with the lane 16 further on). Stores count as
// accesses in flight like copies do, in order: the first phases of a tile allow for the STORES of the one before, which is why
// every wave issues all of them (rows and columns outside the result have an offset outside the buffer, which the memory unit
// drops).
//
// What bounds it, 256x256 tiles: power first. From 8,192 rows on the matrix units are busy for 77 to 84 % of the waves' lifetime, and
// the clock over it is 1.66 to 1.76 GHz of 2.4; at 2,048 rows 73 to 81 % at 1.74 to 1.92 (counters; the rest is the first tile's
// copies, the last one's stores and a last round that is not full). So what costs energy costs time: 16x16x32 MFMAs run 6 % faster
// than 32x32x16 here (they read and write their accumulators half as often). Smaller tiles copy more per MFMA (128x128: 32 KB a
// 512 clocks; 128x256 63 % busy) and are bound by that, so 128x128 tiles issue half of a phase's copies between its MFMAs (2,048 x
// 2,048 x 2,048 23.9 -> 22.1 us; 256x256 tiles get 2 % slower by it).
// bfloat16, the four-wave kernels -> this one, us (one card, weights from HBM; torch's library on another run in parentheses):
//   2,048 x 4,608 x 3,584    75.5 -> 64.4 (66)      2,048 x 37,888 x 3,584 gated    527 -> 455
//   2,048 x 3,584 x 3,584    59.4 -> 54.2 (55)      8,192 x 37,888 x 3,584 gated  1,878 -> 1,571
//   2,048 x 3,584 x 18,944    268 -> 240 (350)        536 x 27,648 x 5,120 gated    217 -> 188
//   2,048 x 2,048 x 2,048    27.4 -> 22.2 (22)      2,048 x 11,264 x 2,048 gated    104 -> 88
//   1,200 x 2,048 x 2,048    30.3 -> 18.4 (20)        536 x 5,120 x 5,120          55.8 -> 46.1
//
// PIECES (tiles of 128 rows, which leave registers for a second set of sums): every `piece` k-tiles a wave adds its sums to the set of
// those before and begins anew, behind a phase's reads and copies. What a float32 sum is off by grows with its additions: see
// choose_turns for where a product needs that. (It costs some 0.8 us a product, whatever the number of pieces: code that runs
// once or twice has to be fetched. More of it costs more: 16 rows at a time, or MFMAs that start from zero, 2 to 4 us.)
// =====================================================================================
__device__ __forceinline__ u32x2 tw_pack4(const float (&v)[4]) {
  const bf16x4 o = {(bf16_t)v[0], (bf16_t)v[1], (bf16_t)v[2], (bf16_t)v[3]};
  return __builtin_bit_cast(u32x2, o);
}
// 16 bytes to the buffer; bytes behind its end are dropped
__device__ __forceinline__ void tw_buffer_store16(u32x4 v, __amdgpu_buffer_rsrc_t to, int offset) {
  __builtin_amdgcn_raw_buffer_store_b128(v, to, offset, 0, 0);
}
__device__ __forceinline__ f32x4 tw_buffer_load16(__amdgpu_buffer_rsrc_t from, int offset) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(from, offset, 0, 0));
}
#define TW_OUTSIDE ((int)0x80000000)   /* an offset that no buffer of tw_buffer holds */

// The shape of a tile and the order of its copies.
template <int ROWS, int Q, int RT = 4>
struct Turns {
  static constexpr int COLS = 8 / ROWS, BM = 16 * RT * ROWS, BN = 32 * Q * COLS;
  static constexpr int A_STAGE = BM * 128, W_STAGE = BN * 128;
  static constexpr int STAGES = 144 * 1024 / (A_STAGE + W_STAGE) > 4 ? 4 : 144 * 1024 / (A_STAGE + W_STAGE);
  static constexpr int LDS = STAGES * (A_STAGE + W_STAGE) + 2 * BN * 4;    // (behind the stages the bias of two tiles)
  static constexpr int A_COPIES = BM / 64, W_COPIES = COLS / 2;            // of 1 KB, a wave's share of A and of a phase's W
  static constexpr int LEAD = STAGES * Q - 1;                              // phases from a copy's to the one that reads it
  static constexpr int A_LATE = Q > 1 ? A_COPIES / 2 : 0;                  // A's copies that go out one phase later
  // phase p's copies: A's late half, A's first half, W, in this order
  static constexpr int piece(int p) { return (p + LEAD) % Q; }             // (the columns of W that it copies)
  static constexpr bool late(int p) { return Q > 1 && piece(p) == 1; }
  static constexpr bool first(int p) { return piece(p) == 0; }
  static constexpr int a_copies(int p) { return (late(p) ? A_LATE : 0) + (first(p) ? A_COPIES - A_LATE : 0); }
  static constexpr int copies(int p) { return a_copies(p) + W_COPIES; }
  static constexpr int behind(int p) { return Q == 1 ? copies(p) / 2 : 0; }              // of them between the phase's MFMAs, behind its wait
  // The wait of phase p: how many copies are younger than the youngest that phase p + 1 needs. Its W went out LEAD - 1 phases
  // ago as that phase's last, A's late half one phase later in front of that phase's W.
  static constexpr int wait(int p) {
    int younger = 0;
    const bool a = (p + 1) % Q == 0 && A_LATE > 0;
    for (int k = 0; k < LEAD - 1 - (a ? 1 : 0); ++k) younger += copies((p - k + 8 * Q) % Q);
    return younger + (a ? W_COPIES : 0) - behind(p);
  }
  static constexpr int CALM = LEAD - 1 - (A_LATE > 0 ? 1 : 0);             // phases of a tile that wait for copies older than the stores
};
template <int N>
__device__ __forceinline__ void tw_wait_accesses() {
  static_assert(N >= 0 && N < 64, "vmcnt has six bits");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

template <typename OutT, int ROWS, int Q, int RT, bool GLU, bool PIECES>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gemm_turns_kernel(const bf16_t* __restrict__ A, long lda, const bf16_t* __restrict__ W, long k_steps, const float* __restrict__ bias,
                       const float* residual, long ldr, OutT* C, long ldc, int M, int N, int k_tiles_all, int tiles_m, int n_blocks,
                       int splits, int per_split, int piece, float* __restrict__ partial) {
  typedef Turns<ROWS, Q, RT> S;
  static_assert(!PIECES || (ROWS == 2 && !GLU));
  constexpr int BM = S::BM, BN = S::BN, BAND = 2048 / BM;            // (bands of rows as above)
  constexpr int STORES = sizeof(OutT) == 4 ? 2 * RT * Q : GLU ? RT * (Q / 2) + Q % 2 * ((RT + 1) / 2) : RT * Q;   // a tile's, of every wave
  constexpr int W_RING = S::STAGES * S::A_STAGE, BIAS = W_RING + S::STAGES * S::W_STAGE;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  // Workgroup x of the 8 XCDs' 32 takes tiles x / 8, x / 8 + 32, ... of its XCD's run of neighbouring tiles.
  const int per_xcd = (n_blocks + 7) / 8;
  const int run_end = min(n_blocks, (int)(blockIdx.x % 8 + 1) * per_xcd);
  int logical = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
  if (logical >= run_end) return;
  const int n_tiles = n_blocks / splits, tiles_n = n_tiles / tiles_m;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / S::COLS, wn = wave % S::COLS;                // (waves 0..3: the upper half of the rows)
  const int turn = wave >> 2;

  f32x4 acc[RT][2 * Q], before[PIECES ? RT : 1][PIECES ? 2 * Q : 1];   // (of this piece of K; of those before it)
  int left;                                                          // k-tiles until a piece ends
  auto clear = [&]() {
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < 2 * Q; ++j) {
        acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        if constexpr (PIECES) before[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
    left = piece;
  };
  auto aim = [&](int block, int& m0, int& n0, int& split) {
    const int tile = block % n_tiles;
    split = block / n_tiles;
    const int band = tile / (BAND * tiles_n), in_band = tile - band * BAND * tiles_n;
    const int band_rows = min(BAND, tiles_m - band * BAND);
    m0 = (band * BAND + in_band % band_rows) * BM;
    n0 = in_band / band_rows * BN;
  };

  // The copies: of k-tile copy_t of block copy_block, into stage copy_stage. A copy of A is 8 rows x 128 bytes, place l % 8 of row
  // u holds the chunk l % 8 ^ (u / 2 % 8) (fragment reads then meet no bank conflict); one of W is half a block of 16 columns x
  // 64 of K, as it lies in memory. Rows past M and blocks past N are clamped to the last valid one (their products are never
  // stored); behind the last tile the copies go on with its operands, which nobody reads.
  __amdgpu_buffer_rsrc_t a_buffer, w_buffer;
  int a_off[S::A_COPIES], copy_block = logical, copy_t = -1, copy_tiles, copy_stage = S::STAGES - 1, w_blocks;
  auto aim_copies = [&]() {
    int m0, n0, split;
    aim(copy_block, m0, n0, split);
    const int kt0 = split * per_split;
    copy_tiles = min(k_tiles_all - kt0, per_split);
    a_buffer = tw_buffer(A + (size_t)m0 * lda + (size_t)kt0 * 64);
    w_buffer = tw_buffer(W + ((size_t)(n0 / 16) * k_steps + (size_t)kt0 * 2) * 512);
    w_blocks = (N + 15) / 16 - n0 / 16;
#pragma unroll
    for (int b = 0; b < S::A_COPIES; ++b) {
      const int row = (wave * S::A_COPIES + b) * 8 + (lane >> 3);
      a_off[b] = min(row, M - 1 - m0) * (int)lda * 2 + ((lane & 7) ^ ((row >> 1) & 7)) * 16;
    }
  };
  auto copy_a = [&](int b) {
    tw_copy_to_lds(a_buffer, lds + copy_stage * S::A_STAGE + (wave * S::A_COPIES + b) * 1024, a_off[b], copy_t * 128);
  };
  auto copy_w = [&](int piece, bool second) {
    // block 2 piece + j of wave column c; a wave copies both halves of one (four wave columns) or one half (two)
    const int c = S::COLS == 4 ? wave >> 1 : wave >> 2, j = S::COLS == 4 ? wave & 1 : (wave >> 1) & 1, half = S::COLS == 4 ? 0 : wave & 1;
    const int block = c * 2 * Q + 2 * piece + j;
    const int at = min(block, w_blocks - 1) * (int)k_steps * 1024 + copy_t * 2048 + half * 1024;
    char* dst = lds + W_RING + copy_stage * S::W_STAGE + block * 2048 + half * 1024;
    if (second) tw_copy_to_lds<1024>(w_buffer, dst, lane * 16, at);
    else tw_copy_to_lds(w_buffer, dst, lane * 16, at);
  };
  auto copy = [&](auto index, auto which) {                          // copy k of phase P
    constexpr int P = decltype(index)::value, k = decltype(which)::value, of_a = S::a_copies(P);
    if constexpr (k == 0 && S::first(P)) {
      copy_stage = copy_stage + 1 == S::STAGES ? 0 : copy_stage + 1;
      if (++copy_t == copy_tiles) {
        if (copy_block + 32 < run_end) copy_block += 32;
        aim_copies();
        copy_t = 0;
      }
    }
    if constexpr (k < of_a) copy_a(S::late(P) ? S::A_COPIES - S::A_LATE + k : k);
    else copy_w(S::piece(P), k > of_a);
  };

  // this lane's fragments in a stage: of A chunk 4 c + g of row 16 RT wm + 16 i + r, of W the same chunk of column 16 j + r of a block
  bf16x8 af[RT][2], wf[2][2];
  const int r0 = lane & 15, g0 = lane >> 4;
  int a_frag[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) a_frag[c] = (wm * 16 * RT + r0) * 128 + (((4 * c + g0) ^ ((r0 >> 1) & 7)) * 16);
  const int w_frag = W_RING + wn * 4096 * Q + lane * 16;
  int stage = 0, phases = 0;                                         // the k-tile's stage; the tile's phases before it
  bool behind_stores = false;                                        // a tile was stored before this one
  auto phase = [&](auto index) {
    constexpr int P = decltype(index)::value;
    if constexpr (P == 0) {
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int i = 0; i < RT; ++i) af[i][c] = *reinterpret_cast<const bf16x8*>(lds + a_frag[c] + stage * S::A_STAGE + i * 2048);
    }
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int j = 0; j < 2; ++j) wf[j][c] = *reinterpret_cast<const bf16x8*>(lds + w_frag + stage * S::W_STAGE + P * 4096 + j * 2048 + c * 1024);
    __builtin_amdgcn_sched_barrier(0);
    tw_unroll<S::copies(P) - S::behind(P)>([&](auto which) { copy(index, which); });
    if constexpr (PIECES && P == 0) {
      if (left == 0) {
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
          for (int j = 0; j < 2 * Q; ++j) {
            before[i][j] = before[i][j] + acc[i][j];
            acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
          }
        left = piece;
      }
      --left;
    }
    if (behind_stores && phases + P < S::CALM) tw_wait_accesses<S::wait(P) + STORES>();
    else tw_wait_accesses<S::wait(P)>();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    tw_unroll<4 * RT>([&](auto which) {
      constexpr int m = decltype(which)::value, c = m / (2 * RT), i = m / 2 % RT, j = m % 2;
      tw_mma16(acc[i][2 * P + j], wf[j][c], af[i][c]);
      constexpr int b = S::behind(P), gap = 4 * RT / (b + 1);
      if constexpr (b > 0 && (m + 1) % gap == 0 && (m + 1) / gap <= b) {
        __builtin_amdgcn_sched_barrier(0);
        copy(index, std::integral_constant<int, S::copies(P) - b + (m + 1) / gap - 1>{});
        __builtin_amdgcn_sched_barrier(0);
      }
    });
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  // The result of a tile. Element e of acc[i][j] is row 16 i + r, column 16 j + 4 g + e of the wave's tile.
  // (r and g pass through an empty asm in front of a tile's stores: the compiler would else work the stores' offsets out in front
  // of the tile loop and keep them in registers that the loop does not have)
  int bias_at = 0;
  auto bias_of = [&](int j, int g) { return *reinterpret_cast<const f32x4*>(lds + BIAS + bias_at + (wn * 32 * Q + j * 16 + 4 * g) * 4); };
  auto store_f32 = [&](auto adds_residual, __amdgpu_buffer_rsrc_t to, int ld, __amdgpu_buffer_rsrc_t add, int ld_add, bool biased,
                       int m0, int n0, auto act_of, int r, int g) {
    constexpr bool adds = decltype(adds_residual)::value;
    // the residual of AT row tiles of 16 at a time (all four where the sums leave registers for it)
    constexpr int AT = ROWS == 2 ? 4 : 1;
    f32x4 res[AT][2 * Q];
    tw_unroll<RT>([&](auto index) {
      constexpr int i = decltype(index)::value;
      if constexpr (adds && i % AT == 0) {
#pragma unroll
        for (int k = 0; k < AT; ++k)
#pragma unroll
          for (int j = 0; j < 2 * Q; ++j) {
            const int row = wm * 16 * RT + (i + k) * 16 + r, col = wn * 32 * Q + j * 16 + 4 * g;
            res[k][j] = tw_buffer_load16(add, row < M - m0 && col < N - n0 ? row * ld_add * 4 + col * 4 : TW_OUTSIDE);
          }
      }
      const int row = wm * 16 * RT + i * 16 + r;
#pragma unroll
      for (int j = 0; j < 2 * Q; ++j) {
        const int col = wn * 32 * Q + j * 16 + 4 * g;
        f32x4 v = acc[i][j];
        if (biased) v = v + bias_of(j, g);
        if constexpr (adds) v = v + res[i % AT][j];
        else {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = tw_act(v[e], act_of());
        }
        tw_buffer_store16(__builtin_bit_cast(u32x4, v), to, row < M - m0 && col < N - n0 ? row * ld * 4 + col * 4 : TW_OUTSIDE);
      }
    });
  };
  // (an activation is asked for once a tile)
  auto with_act = [&](auto&& store) {
    const long act = residual == nullptr ? ldr : 0;          // (no residual: the stride names an activation, see tw_act)
    if (act == 0) store([]() { return 0L; });
    else if (act == TW_ACT_RELU_SQUARED) store([]() { return (long)TW_ACT_RELU_SQUARED; });
    else store([]() { return (long)TW_ACT_GELU_ERF; });
  };
  // 16 bytes a lane from two tiles a and b of 16 x 16 in bfloat16: after the exchange between rows of 16 lanes the lanes of
  // g = 0, 1, 2, 3 hold columns 0..7 of a, 0..7 of b, 8..15 of a, 8..15 of b
  auto store_pair = [&](__amdgpu_buffer_rsrc_t to, u32x2 a, u32x2 b, int offset) {
    const auto x = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
    const auto y = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
    tw_buffer_store16(u32x4{x[0], y[0], x[1], y[1]}, to, offset);
  };
  auto store_tile = [&](int m0, int n0, int split) {
    int r = lane & 15, g = lane >> 4;
    asm volatile("" : "+v"(r), "+v"(g));
    if constexpr (!GLU) {
      if (splits > 1) {
        store_f32(std::false_type{}, tw_buffer(partial + ((size_t)split * M + m0) * N + n0), N, a_buffer, 0, false, m0, n0, []() { return 0L; }, r, g);
        return;
      }
    }
    if constexpr (sizeof(OutT) == 4) {
      const auto to = tw_buffer(C + (size_t)m0 * ldc + n0);
      if (residual) store_f32(std::true_type{}, to, (int)ldc, tw_buffer(residual + (size_t)m0 * ldr + n0), (int)ldr, bias != nullptr, m0, n0, []() { return 0L; }, r, g);
      else with_act([&](auto act_of) { store_f32(std::false_type{}, to, (int)ldc, a_buffer, 0, bias != nullptr, m0, n0, act_of, r, g); });
    } else if constexpr (GLU) {
      const auto to = tw_buffer(C + (size_t)m0 * ldc + n0 / 2);
      auto gated = [&](auto code_of) {
        auto form = [&](int i, int p) {                      // column tiles 2 p and 2 p + 1: gate and up of 16 columns
          f32x4 gate = acc[i][2 * p], up = acc[i][2 * p + 1];
          if (bias) {
            gate = gate + bias_of(2 * p, g);
            up = up + bias_of(2 * p + 1, g);
          }
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = tw_glu(gate[e], up[e], code_of());
          return tw_pack4(v);
        };
        auto offset = [&](int row, int col) {                // (columns of the result)
          return row < M - m0 && 2 * col < N - n0 ? row * (int)ldc * 2 + col * 2 : TW_OUTSIDE;
        };
        tw_unroll<RT>([&](auto index) {                      // two neighbouring column groups of a row tile together
          constexpr int i = decltype(index)::value;
#pragma unroll
          for (int p = 0; p + 1 < Q; p += 2)
            store_pair(to, form(i, p), form(i, p + 1), offset(wm * 16 * RT + i * 16 + r, wn * 16 * Q + p * 16 + (g & 1) * 16 + (g >> 1) * 8));
          if constexpr (Q % 2 == 1 && i % 2 == 0) {          // the last of an odd number: two row tiles, or the last one alone
            const u32x2 first = form(i, Q - 1);
            const int at = offset(wm * 16 * RT + (i + (g & 1)) * 16 + r, wn * 16 * Q + (Q - 1) * 16 + (g >> 1) * 8);
            if constexpr (i + 1 < RT) store_pair(to, first, form(i + 1, Q - 1), at);
            else store_pair(to, first, first, g & 1 ? TW_OUTSIDE : at);
          }
        });
      };
      if (ldr == 0) gated([]() { return 0L; });
      else gated([&]() { return ldr; });
    } else {
      const auto to = tw_buffer(C + (size_t)m0 * ldc + n0);
      with_act([&](auto act_of) {
        tw_unroll<RT>([&](auto index) {
          constexpr int i = decltype(index)::value;
          const int row = wm * 16 * RT + i * 16 + r;
#pragma unroll
          for (int p = 0; p < Q; ++p) {
            u32x2 half[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
              f32x4 x = acc[i][2 * p + j];
              if (bias) x = x + bias_of(2 * p + j, g);
              float v[4];
#pragma unroll
              for (int e = 0; e < 4; ++e) v[e] = tw_act(x[e], act_of());
              half[j] = tw_pack4(v);
            }
            const int col = wn * 32 * Q + p * 32 + (g & 1) * 16 + (g >> 1) * 8;
            store_pair(to, half[0], half[1], row < M - m0 && col < N - n0 ? row * (int)ldc * 2 + col * 2 : TW_OUTSIDE);
          }
        });
      });
    }
  };

  // what the phases before the first would have copied, then the wait of the last of them
  aim_copies();
  tw_unroll<S::LEAD>([&](auto index) {
    constexpr int T = decltype(index)::value - S::LEAD;
    constexpr int P = (T + 8 * S::LEAD * Q) % Q;
    tw_unroll<S::copies(P)>([&](auto which) { copy(std::integral_constant<int, P>{}, which); });
  });
  clear();
  tw_wait_accesses<S::wait(Q - 1) + S::behind(Q - 1)>();
  __builtin_amdgcn_s_barrier();
  if (turn == 1) __builtin_amdgcn_s_barrier();                       // waves 4..7: half a phase behind
  asm volatile("" ::: "memory");
  for (;;) {
    int m0, n0, split;
    aim(logical, m0, n0, split);
    if (bias && wave * 64 < BN) {
      // this tile's bias, 64 columns a wave: read behind its last phase, by when it has long landed. (Two places in turn: waves
      // 4..7 may still be at the tile before.)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(tw_buffer(bias + n0), (tw_lds_ptr)(lds + BIAS + bias_at + wave * 256), 4,
                                               min(wave * 64 + lane, N - 1 - n0) * 4, 0, 0, 0);
    }
    const int k_tiles = min(k_tiles_all - split * per_split, per_split);
    for (phases = 0; phases < k_tiles * Q; phases += Q) {
      tw_unroll<Q>(phase);
      stage = stage + 1 == S::STAGES ? 0 : stage + 1;
    }
    if constexpr (PIECES) {
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < 2 * Q; ++j) acc[i][j] = before[i][j] + acc[i][j];
    }
    store_tile(m0, n0, split);
    logical += 32;
    if (logical >= run_end) break;
    behind_stores = true;
    bias_at = BN * 4 - bias_at;
    clear();
  }
  if (turn == 0) __builtin_amdgcn_s_barrier();
  tw_wait_accesses<0>();                                             // (no copy may land behind the workgroup's end)
}

// =====================================================================================
// Host side
// =====================================================================================
// How many K ranges the tiled kernel uses: with fewer tiles than the chip has room for (a prompt
// portion of a few hundred rows against a square or tall matrix) the k-tiles of a tile are dealt
// to several workgroups. Depends on the shape only.
// How a launch may deviate from "compute C": `leave` keeps the float32 sums of the K ranges in `partial`
// for the caller's next kernel (no reduction kernel; the caller passes C = partial as float32 without
// bias or residual, so that with a single range the product itself is partial[0]); `dry` launches
// nothing and only reports, in `splits`, the number of K ranges the launch would use.
struct TiledMode {
  bool leave = false, dry = false;
  int splits = 0;
};

static int tiled_splits(int M, int N, int K, int epf, int bm, int bn) {
  const long tiles = (long)tw_div_up(M, bm) * tw_div_up(N, bn);
  if (tiles >= 192) return 1;
  const int k_tiles = tw_div_up(K, 8 * epf);
  long splits = tw_div_up(384, tiles);
  const long resident = (long)bm * bn <= 128 * 128 ? 512 : 256;   // workgroups the chip holds at once
  if (splits > resident / tiles) splits = resident / tiles;       // never a few more than that: a second round
  if (splits > k_tiles / 8) splits = k_tiles / 8;
  if (splits > 8) splits = 8;
  return splits < 1 ? 1 : (int)splits;
}

template <typename T, typename OutT, int WM, int WN, bool SHUF, bool GLU>
static int launch_tiled(const T* A, long lda, const T* W, long ldw, const float* bias,
                        const float* residual, long ldr, OutT* C, long ldc, float* partial,
                        long partial_bytes, int M, int N, int K, int want_splits, hipStream_t stream,
                        TiledMode* mode = nullptr) {
  constexpr int BM = 64 * WM, BN = 64 * WN, KCH = 8;
  constexpr int EPF = Elem<T>::kPerFrag;
  const int tiles_m = tw_div_up(M, BM), tiles_n = tw_div_up(N, BN);
  int splits = GLU ? 1 : (want_splits > 0 ? want_splits : tiled_splits(M, N, K, EPF, BM, BN));
  if (mode && mode->dry) {
    mode->splits = splits;
    return 0;
  }
  if (splits > 1 && (partial == nullptr || partial_bytes < (long)splits * M * N * 4 || (uintptr_t)partial % 16 != 0)) splits = 1;
  if (mode) mode->splits = splits;
  const long n_blocks = (long)tiles_m * tiles_n * splits;
  TW_REQUIRE(n_blocks < (1L << 30));
  // per-tile offsets are 32-bit
  TW_REQUIRE((long)BM * lda < (1L << 31));
  TW_REQUIRE(SHUF ? (long)(BN / 16) * ldw * 64 * EPF < (1L << 31) : (long)BN * ldw < (1L << 31));
  const int grid = (int)((n_blocks + 7) / 8 * 8);
  const size_t pipeline_bytes = sizeof(T) == 4 ? 3 * (size_t)(BM + BN) * TW_PART_ROW : 2 * (size_t)(BM + BN) * (KCH * 16 + 16);
  const size_t epilogue_bytes = 4 * (32 * (size_t)(32 * WN + 4) + 32 * WN) * 4;
  const size_t lds_bytes = pipeline_bytes > epilogue_bytes ? pipeline_bytes : epilogue_bytes;
  auto kernel = [] {
    if constexpr (sizeof(T) == 4) return gemm_parts_kernel<WM, WN, SHUF, GLU>;
    else return gemm_tiled_kernel<T, OutT, WM, WN, SHUF, GLU>;
  }();
  static bool attribute_set = false;   // per instantiation
  if (!attribute_set) {
    hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)lds_bytes);
    if (e != hipSuccess) return (int)e;
    attribute_set = true;
  }
  kernel<<<grid, 256, lds_bytes, stream>>>(A, lda, W, ldw, bias, residual, ldr, C, ldc, M, N, K, tiles_m,
                                           (int)n_blocks, splits, partial);
  int err = TW_LAUNCH_RESULT();
  if (err || splits == 1 || (mode && mode->leave)) return err;
  return launch_splitk_reduce<OutT>(partial, splits, bias, residual, ldr, C, ldc, M, N, stream);
}


// Does gemm_turns_kernel take this product in tiles of S? No K range is empty; a tile's bias lands within the tile, so that K is as long
// as its stages; operands are copied and results stored 16 bytes at a time; offsets within a tile are 32-bit.
static int turns_per_split(int K, int splits) { return tw_div_up(K / 64, splits); }
template <typename S>
static bool turns_takes(int out_bytes, const void* A, long lda, long ldw, const float* bias, const float* residual, long ldr, const void* C,
                        long ldc, int N, int K) {
  return K % 64 == 0 && K >= 64 && (bias == nullptr || K / 64 >= S::STAGES) && lda % 8 == 0 && (uintptr_t)A % 16 == 0 && N % 8 == 0 &&
         ldc % (16 / out_bytes) == 0 && (uintptr_t)C % 16 == 0 && (residual == nullptr || (ldr % 4 == 0 && (uintptr_t)residual % 16 == 0)) &&
         S::BM * lda * 2 < (1L << 31) && S::BN / 16 * ldw * 1024 < (1L << 31) && S::BM * ldc * out_bytes < (1L << 31) &&
         (residual == nullptr || S::BM * ldr * 4 < (1L << 31)) && (long)S::BM * N * 4 < (1L << 31);
}

template <typename OutT, int ROWS, int Q, int RT, bool GLU>
static int launch_turns(const bf16_t* A, long lda, const bf16_t* W, long ldw, const float* bias, const float* residual, long ldr,
                        OutT* C, long ldc, float* partial, long partial_bytes, int M, int N, int K, int want_splits, int piece,
                        hipStream_t stream, TiledMode* mode = nullptr) {
  typedef Turns<ROWS, Q, RT> S;
  const int tiles_m = tw_div_up(M, S::BM), tiles_n = tw_div_up(N, S::BN);
  int splits = GLU ? 1 : (want_splits > 0 ? want_splits : tiled_splits(M, N, K, 8, S::BM, S::BN));
  while ((splits - 1) * turns_per_split(K, splits) >= K / 64) --splits;
  if (mode && mode->dry) {
    mode->splits = splits;
    return 0;
  }
  if (splits > 1 && (partial == nullptr || partial_bytes < (long)splits * M * N * 4 || (uintptr_t)partial % 16 != 0)) splits = 1;
  if (mode) mode->splits = splits;
  const long n_blocks = (long)tiles_m * tiles_n * splits;
  TW_REQUIRE(n_blocks < (1L << 30));
  const int grid = (int)(n_blocks > 256 ? 256 : (n_blocks + 7) / 8 * 8);
  const int per_split = turns_per_split(K, splits);
  auto run = [&](auto in_pieces) {
    auto kernel = gemm_turns_kernel<OutT, ROWS, Q, RT, GLU, decltype(in_pieces)::value>;
    static bool attribute_set = false;   // per instantiation
    if (!attribute_set) {
      hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, S::LDS);
      if (e != hipSuccess) return (int)e;
      attribute_set = true;
    }
    kernel<<<grid, 512, S::LDS, stream>>>(A, lda, W, ldw, bias, residual, ldr, C, ldc, M, N, K / 64, tiles_m, (int)n_blocks, splits,
                                          per_split, piece, partial);
    return TW_LAUNCH_RESULT();
  };
  int err;
  if constexpr (ROWS == 2 && !GLU) err = piece > 0 && piece < per_split ? run(std::true_type{}) : run(std::false_type{});
  else err = run(std::false_type{});
  if (err || splits == 1 || (mode && mode->leave)) return err;
  return launch_splitk_reduce<OutT>(partial, splits, bias, residual, ldr, C, ldc, M, N, stream);
}

template <typename OutT, int WM, int WN, bool GLU>
static int launch_dma(const bf16_t* A, long lda, const bf16_t* W, long ldw, const float* bias,
                      const float* residual, long ldr, OutT* C, long ldc, float* partial, long partial_bytes,
                      int M, int N, int K, int want_splits, hipStream_t stream, TiledMode* mode = nullptr) {
  constexpr int BM = 64 * WM, BN = 64 * WN;
  TW_REQUIRE(K % 32 == 0 && K >= 32 && lda % 8 == 0);
  const int tiles_m = tw_div_up(M, BM), tiles_n = tw_div_up(N, BN);
  int splits = GLU ? 1 : (want_splits > 0 ? want_splits : tiled_splits(M, N, K, 8, BM, BN));
  if (mode && mode->dry) {
    mode->splits = splits;
    return 0;
  }
  if (splits > 1 && (partial == nullptr || partial_bytes < (long)splits * M * N * 4 || (uintptr_t)partial % 16 != 0)) splits = 1;
  if (mode) mode->splits = splits;
  const long n_blocks = (long)tiles_m * tiles_n * splits;
  TW_REQUIRE(n_blocks < (1L << 30));
  // offsets within a tile's operands are 32-bit
  TW_REQUIRE((long)BM * lda * 2 < (1L << 31) && (long)(BN / 16) * ldw * 1024 < (1L << 31));
  const int grid = (int)((n_blocks + 7) / 8 * 8);
  const size_t pipeline_bytes = TW_DMA_A_SLOTS * (size_t)BM * 128 + TW_DMA_STAGES * (size_t)BN * 64;
  static_assert(TW_DMA_A_SLOTS * BM * 128 + TW_DMA_STAGES * BN * 64 <= 160 * 1024, "a workgroup has 160 KB of LDS");
  const size_t epilogue_bytes = 4 * (32 * (size_t)(32 * WN + 4) + 32 * WN) * 4;
  const size_t lds_bytes = pipeline_bytes > epilogue_bytes ? pipeline_bytes : epilogue_bytes;
  auto kernel = gemm_dma_kernel<OutT, WM, WN, GLU>;
  static bool attribute_set = false;   // per instantiation
  if (!attribute_set) {
    hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)lds_bytes);
    if (e != hipSuccess) return (int)e;
    attribute_set = true;
  }
  kernel<<<grid, 256, lds_bytes, stream>>>(A, lda, W, ldw, bias, residual, ldr, C, ldc, M, N, K, tiles_m,
                                           (int)n_blocks, splits, partial);
  int err = TW_LAUNCH_RESULT();
  if (err || splits == 1 || (mode && mode->leave)) return err;
  return launch_splitk_reduce<OutT>(partial, splits, bias, residual, ldr, C, ldc, M, N, stream);
}

// Which tile (1: 128x128, 2: 128x256, 3: 256x256, 4: 256x192): the one with the least estimated time,
// rounds of tiles over 256 CUs (128x128: two to a CU, so half rounds) x tile area / the rate a tile of
// that shape reaches when the chip is full (measured, relative). The estimate ranks the shapes as
// measured on the projections of 7B-class models from 256 to 16,384 rows. Larger tiles move fewer
// bytes per MFMA through the 64 B/clk vector-memory path and LDS; smaller ones waste less in the
// last round.
// (with the present epilogue, 8,192 x 37,888 x 3,584 in bfloat16, TFLOP/s plain / gated: 128x128 906 / 891, 128x256
// 1,027 / 1,037, 256x256 1,195 / 1,179, 256x192 1,146 / 1,121)
// (1 to 4: of every kernel; 5 to 9: of gemm_turns_kernel alone)
static const int kTileM[10] = {0, 128, 128, 256, 256, 192, 192, 192, 192, 256}, kTileN[10] = {0, 128, 256, 256, 192, 128, 192, 256, 384, 320};
static const double kTileRate[5] = {0, 0.76, 0.90, 1.05, 1.00};

static int choose_shape(bool big_ok, int M, int N) {
  if (!big_ok) return 1;
  int best = 1;
  double best_cost = 0;
  for (int shape = 1; shape <= 4; ++shape) {
    const long tiles = (long)tw_div_up(M, kTileM[shape]) * tw_div_up(N, kTileN[shape]);
    const double cost = (double)tw_div_up(tiles, 256) * kTileM[shape] * kTileN[shape] / kTileRate[shape];
    if (shape == 1 || cost < best_cost) {
      best = shape;
      best_cost = cost;
    }
  }
  return best;
}

// Estimated seconds of `shape` with K dealt to `splits` workgroups per tile: the rounds of workgroups
// over 256 CUs at the shape's relative rate (4.42e-13 s per unit of tile area and element of K: a
// 128x256 tile over K = 18,944 takes 295 us), plus, with splits, what splitk_reduce moves: the partial
// sums written and read, the residual and the result, at the 6.5 TB/s such just-written data streams at.
static double plan_seconds(int shape, int splits, int M, int N, int K) {
  const long tiles = (long)tw_div_up(M, kTileM[shape]) * tw_div_up(N, kTileN[shape]);
  double t = (double)tw_div_up(tiles * splits, 256) * kTileM[shape] * kTileN[shape] / kTileRate[shape] *
             ((double)K / splits) * 4.42e-13;
  if (splits > 1) t += (2.0 * splits + 2.0) * M * N * 4.0 / 6.5e12;
  return t;
}

// Shape and K ranges of a product (splits 0: the launcher's own rule for few tiles). Beside the choice
// above, 128x256 or 256x256 tiles with 2 to 8 K ranges are taken where they fill one round of CUs that whole tiles
// leave partly idle and K is long enough to pay for the reduction: the down projection of a 2,048-token
// prompt (N = 3,584, K = 18,944) has 224 tiles of 128x256 or 112 of 256x256; two K ranges of the latter
// run at the large tile's rate on 224 CUs (295 -> 265 us with the reduction).
struct TilePlan { int shape, splits, piece; };        // piece: of gemm_turns_kernel, 0: the whole of K

static TilePlan choose_staged(bool big_ok, bool glu, int M, int N, int K, int epf) {
  TilePlan plan = {choose_shape(big_ok, M, N), 0, 0};
  if (!big_ok || glu || K % 32 != 0) return plan;
  const int own = tiled_splits(M, N, K, epf, kTileM[plan.shape], kTileN[plan.shape]);
  double best = plan_seconds(plan.shape, own, M, N, K) * 0.95;
  for (int shape = 2; shape <= 3; ++shape) {               // 128x256 and 256x256: one workgroup a CU
    const long tiles = (long)tw_div_up(M, kTileM[shape]) * tw_div_up(N, kTileN[shape]);
    for (int splits = 2; splits <= 8; ++splits) {
      if (tiles * splits > 256 || K / splits < 2048) continue;
      const double t = plan_seconds(shape, splits, M, N, K);
      if (t < best) {
        best = t;
        plan = {shape, splits, 0};
      }
    }
  }
  return plan;
}

// The same for gemm_turns_kernel, in microseconds: a launch, then rounds of tiles over 256 CUs, each with the tile's begin and end and
// its k-tiles. A k-tile takes `alone` where the chip is mostly idle (copies and barriers) and rounds x `full` x the share of the
// chip in use where it is not (power: the clock falls with the matrix units in use); between the two the fourth powers add up.
// Fitted to 126 products (100 to 8,192 rows, 512 to 11,264 columns, K 512 to 5,632, each at all four shapes: 4 to 6 % off, root mean
// square), and K ranges to 280 with 2 or 4: the choice was the fastest of all shapes and ranges or, in the mean, 0.2 % behind it (one of
// 126 more than 4 %). Asked about 764 more (65 to 5,800 rows, 256 to 152,064 columns, K 64 to 15,040; plain, float32 with a residual
// and gated) it is 0.4 % behind, 27 of them more than 5 %, if a round counts whole for few rows of a matrix that comes from HBM
// (its workgroups wait for memory however few they are: 384 x 32,000 x 4,096 by 128x256 124 us, by 256x256 99).
// Its sums are no longer than those of the kernels above: where these would take more K ranges, tiles of 128 rows add up K in
// pieces as long as those ranges, in the ranges' order, and larger tiles, whose registers are full, take as many ranges. (1,200 x
// 2,048 x 2,048 in one sum instead of three ranges was off by 2.7e-7 of the result instead of 1.5e-7.)
struct TurnsCost { double launch, tile, alone, full; };
static const TurnsCost kTurnsCost[5] = {{}, {3.8, 1.45, 0.351, 0.482}, {4.3, 2.27, 0.589, 0.815}, {3.5, 5.29, 0.960, 1.363}, {3.2, 4.42, 0.759, 1.060}};
// Tiles of 192 rows, and of 320 columns, come after: they take a product where they are expected to be 3 % faster than the choice among
// the four, all nine estimated from another 402 products in one sum (65 to 4,700 rows, 896 to 37,888 columns, K 512 to 8,192; 5 to 7 %
// off). Over these the choice is then 1.8 % faster in the mean than among the four, none more than 1 % slower, and 0.4 % behind the
// best of the nine. (With K ranges, which no product of that fit had, 8 %: products of 129 to 167 rows were 3 to 7 % slower at 3.) They fill what 128 and 256 rows leave (536 x 27,648 x 5,120 183 -> 145 us by 192x384, 521 x 22,016 x 2,048 59 -> 49 by 192x256,
// 536 x 7,168 x 5,120 58.6 -> 54.8 by 192x128), and 256x320 has a tenth less to copy and to read a product than 256x256
// (37,888 x 3,584, gated: 2,048 rows 416 to 434 -> 405 to 410, 8,192 rows 1,535 -> 1,502 to 1,519).
static const TurnsCost kNineCost[10] = {{}, {4.1, 1.71, 0.361, 0.504}, {4.5, 2.95, 0.596, 0.819}, {1.0, 8.67, 0.982, 1.136}, {2.7, 5.83, 0.776, 0.955},
                                        {4.2, 2.50, 0.535, 0.608}, {4.1, 3.97, 0.663, 0.808}, {3.1, 5.44, 0.843, 0.989}, {1.0, 9.36, 1.179, 1.298}, {1.0, 9.78, 1.194, 1.316}};
static double turns_us(const TurnsCost& c, int shape, int splits, int M, int N, int K) {
  const long blocks = (long)tw_div_up(M, kTileM[shape]) * tw_div_up(N, kTileN[shape]) * splits;
  const double rounds = tw_div_up(blocks, 256), alone = rounds * c.alone;
  const double full = (M <= 512 && (double)N * K >= 5e7 ? rounds : blocks / 256.0) * c.full;
  double t = c.launch + rounds * c.tile + tw_div_up(K / 64, splits) * sqrt(sqrt(alone * alone * alone * alone + full * full * full * full));
  if (splits > 1) t += 3.5 + 0.24e-6 * 4.0 * splits * M * N;       // the ranges' sums written and added up
  return t;
}
// (A product asks for its plan up to three times, for its scratch, its ranges and its launch, and a model's steps ask for the
// same few: the last 64 are kept, a thread's own. Estimating 32 candidates takes a microsecond, which a step that is issued launch by
// launch, a prompt's portion, would spend in front of each product.)
static TilePlan choose_turns(bool glu, int M, int N, int K) {
  struct Known {
    int M, N, K, glu;
    TilePlan plan;
  };
  static thread_local Known known[64] = {};                  // (M = 0: none)
  Known& at = known[((unsigned)M * 2654435761u ^ (unsigned)N * 40503u ^ (unsigned)K * 2246822519u ^ (glu ? 0x80000000u : 0u)) >> 26];
  if (at.M == M && at.N == N && at.K == K && at.glu == (int)glu) return at.plan;
  TilePlan plan = {1, 1, 0};
  const TilePlan staged = choose_staged(true, glu, M, N, K, 8);
  const int ranges = glu ? 1 : staged.splits > 0 ? staged.splits : tiled_splits(M, N, K, 8, kTileM[staged.shape], kTileN[staged.shape]);
  double best = 0;
  auto ask = [&](const TurnsCost& cost, int shape, double of_ranges) {
    for (int splits = kTileM[shape] > 128 ? ranges : 1; splits <= (glu ? 1 : 8); ++splits) {
      if (splits > 1 && splits > ranges && K / splits < 512) break;
      // (pieces against as many ranges, 23 products of 8 to 128 tiles: level at 30 to 50 tiles and 1,024 of K, 10 % behind at 10
      // tiles and 20 to 40 % ahead at 80 and more)
      const double t = turns_us(cost, shape, splits, M, N, K) * (splits > 1 ? of_ranges : 1.0) + (splits < ranges ? 1.2 : 0.0);
      if (best == 0 || t < best) {
        best = t;
        plan = {shape, splits, splits < ranges ? turns_per_split(K, ranges) : 0};
      }
    }
  };
  for (int shape = 1; shape <= 4; ++shape) ask(kTurnsCost[shape], shape, 1.0);
  best = 0.97 * turns_us(kNineCost[plan.shape], plan.shape, plan.splits, M, N, K) + (plan.piece ? 1.2 : 0.0);
  for (int shape = 5; shape <= 9; ++shape) ask(kNineCost[shape], shape, 1.05);
  at = {M, N, K, (int)glu, plan};
  return plan;
}

// Where gemm_turns_kernel takes a product: is it the faster one? Its workgroup of 144 KB begins and ends more slowly, alone on its CU,
// than two small ones, which shows where there is little between: up to 256 tiles of 128x128, K of 64 and 128. It ends most slowly
// with a residual, which arrives while nothing else runs. (The others / this one, us; with a residual: 100 x 1,024 x 64 5.7 / 7.7, x 256
// 7.5 / 7.8, 300 x 2,048 x 64 6.1 / 8.3, x 256 7.9 / 8.7, 2,048 x 2,048 x 128 8.6 / 7.4, 300 x 11,264 x 128 10.9 / 14.7, x 512 15.0 / 18.1,
// x 1,024 20.5 / 22.8, 536 x 11,264 x 512 18.8 / 19.9, 1,024 x 11,264 x 128 17.9 / 14.6; without: 300 x 2,048 x 64 5.4 / 6.3,
// 1,024 x 2,048 x 128 6.4 / 6.7, 2,048 x 4,096 x 64 9.0 / 7.5; gated 300 x 2,048 x 64 7.0 / 7.3. Tiles that N does not fill are where the
// others end slowly: 320 x 344 x 128 7.1 / 6.1, with a residual 7,450 x 608 x 128 16.3 / 13.7.)
static bool turns_pay(bool glu, bool adds, int M, int N, int K) {
  if (N % 64 != 0) return true;
  const long tiles = (long)tw_div_up(M, 128) * tw_div_up(N, 128);
  if (adds) return K > (tiles <= 128 ? 320 : tiles <= 256 ? 64 : tiles <= 600 ? 512 : 0);
  return tiles > 256 || K > (glu ? 64 : 128);
}

// float32 (gemm_parts_kernel): 1 is 128x128, 2 64x128, 3 64x64, with K ranges, the least estimated time in microseconds. A launch, rounds of
// the workgroups that a CU holds, and k-tiles of 32, which take `alone` a round where a CU has little else and n x `full` where its n
// workgroups share the matrix unit; the fourth powers of the two add up. Fitted to 1,586 forms of 142 products (65 to 3,000 rows, 512 to
// 32,000 columns, K 256 to 4,864, 1 to 8 ranges) when the kernel formed six products of parts: 5 to 6 % off, the choice 0.4 % behind the
// fastest of all. With eight every form takes some 15 % longer and the choice stays good: of 159 other products it is 0.6 % behind the fastest form,
// 8 of them more than 5 %, the same as by constants fitted anew to their 1,327 forms. (An estimate takes 0.3 us: it is not kept.)
static const struct { int m, n, held; double launch, tile, alone, full, sums; } kParts[4] = {
    {}, {128, 128, 2, 3.1, 1.73, 1.429, 1.170, 0.32}, {64, 128, 3, 4.2, 0.0, 0.966, 0.723, 0.30}, {64, 64, 5, 3.1, 0.0, 0.686, 0.426, 0.34}};
static TilePlan choose_parts(bool glu, int M, int N, int K) {
  static const int kRanges[6] = {1, 2, 3, 4, 6, 8};
  TilePlan plan = {1, 1, 0};
  double best = 0;
  for (int shape = 1; shape <= 3; ++shape) {
    const auto& c = kParts[shape];
    const long tiles = (long)tw_div_up(M, c.m) * tw_div_up(N, c.n);
    for (int splits : kRanges) {
      if (splits > 1 && (glu || tiles >= 512 || tiles * splits > 1536 || K / splits < 128)) break;
      const long blocks = tiles * splits, n = (blocks + 255) / 256, rounds = (n + c.held - 1) / c.held;
      const double alone = rounds * c.alone, full = (n <= 2 * c.held ? n : blocks / 256.0 + 0.5) * c.full;
      double t = c.launch + rounds * c.tile + tw_div_up(tw_div_up(K, 32), splits) * sqrt(sqrt(alone * alone * alone * alone + full * full * full * full));
      if (splits > 1) t += 3.0 + c.sums * 4e-6 * splits * M * N;
      if (best == 0 || t < best) {
        best = t;
        plan = {shape, splits, 0};
      }
    }
  }
  return plan;
}

template <typename T, typename OutT, bool SHUF, bool GLU>
static std::enable_if_t<sizeof(T) == 4, int> tiled_by_shape(int shape, const T* A, long lda, const T* W, long ldw, const float* bias,
                          const float* residual, long ldr, OutT* C, long ldc, float* partial,
                          long partial_bytes, int M, int N, int K, hipStream_t stream, TiledMode* mode = nullptr) {
  if (shape >= 3) return TW_ERR_BAD_ARGUMENT;      // (forced shapes 1 and 2: float32's first and second)
  const TilePlan plan = shape ? TilePlan{shape, 0, 0} : choose_parts(GLU, M, N, K);
  auto run = [&](auto wm, auto wn) {
    return launch_tiled<T, OutT, wm.value, wn.value, SHUF, GLU>(A, lda, W, ldw, bias, residual, ldr, C, ldc, partial, partial_bytes, M, N, K, plan.splits, stream, mode);
  };
  constexpr std::integral_constant<int, 1> one;
  constexpr std::integral_constant<int, 2> two;
  return plan.shape == 1 ? run(two, two) : plan.shape == 2 ? run(one, two) : run(one, one);
}

template <typename T, typename OutT, bool SHUF, bool GLU>
static std::enable_if_t<sizeof(T) == 2, int> tiled_by_shape(int shape, const T* A, long lda, const T* W, long ldw, const float* bias,
                          const float* residual, long ldr, OutT* C, long ldc, float* partial,
                          long partial_bytes, int M, int N, int K, hipStream_t stream, TiledMode* mode = nullptr) {
  constexpr bool BIG = SHUF;
  auto takes = [&](auto tile) { return turns_takes<decltype(tile)>(sizeof(OutT), A, lda, ldw, bias, residual, ldr, C, ldc, N, K); };
  TilePlan plan = {shape, 0, 0};                    // a forced shape keeps the launcher's own rule
  bool turns = BIG;                                 // (each plan is for its own kernels: choose_turns for a product all of whose tiles they take)
  if (shape == 0) {
    turns = BIG && turns_pay(GLU, residual != nullptr, M, N, K) && takes(Turns<4, 3>{}) && takes(Turns<4, 4>{}) && takes(Turns<2, 2>{}) && takes(Turns<2, 1>{}) && takes(Turns<4, 6, 3>{}) && takes(Turns<4, 5, 4>{});
    plan = turns ? choose_turns(GLU, M, N, K) : choose_staged(BIG, GLU, M, N, K, Elem<T>::kPerFrag);
  }
  shape = plan.shape;
  const int splits = plan.splits;
  if constexpr (BIG) {
    // bfloat16 and shuffled weights: the kernels that copy straight into LDS, if K and the strides allow
#define TW_TURNS(SHAPE, ROWS, Q, RT)                                                                                              \
    if (turns && shape == SHAPE && takes(Turns<ROWS, Q, RT>{}))                                                                     \
      return launch_turns<OutT, ROWS, Q, RT, GLU>(A, lda, W, ldw, bias, residual, ldr, C, ldc, partial, partial_bytes, M, N, K, splits, plan.piece, stream, mode)
    TW_TURNS(1, 2, 1, 4);
    TW_TURNS(2, 2, 2, 4);
    TW_TURNS(3, 4, 4, 4);
    TW_TURNS(4, 4, 3, 4);
    TW_TURNS(5, 4, 2, 3);
    TW_TURNS(6, 4, 3, 3);
    TW_TURNS(7, 4, 4, 3);
    TW_TURNS(8, 4, 6, 3);
    TW_TURNS(9, 4, 5, 4);
#undef TW_TURNS
    if (K % 32 == 0 && K >= 32 && lda % 8 == 0) {
      if (shape == 4) return launch_dma<OutT, 4, 3, GLU>(A, lda, W, ldw, bias, residual, ldr, C, ldc, partial, partial_bytes, M, N, K, splits, stream, mode);
      if (shape == 3) return launch_dma<OutT, 4, 4, GLU>(A, lda, W, ldw, bias, residual, ldr, C, ldc, partial, partial_bytes, M, N, K, splits, stream, mode);
      if (shape == 2) return launch_dma<OutT, 2, 4, GLU>(A, lda, W, ldw, bias, residual, ldr, C, ldc, partial, partial_bytes, M, N, K, splits, stream, mode);
    }
    if (shape == 3 || shape == 4)             // (K no multiple of 32: the register-staged 256x256 tile for both)
      return launch_tiled<T, OutT, 4, 4, SHUF, GLU>(A, lda, W, ldw, bias, residual, ldr, C, ldc, partial, partial_bytes, M, N, K, splits, stream, mode);
  }
  if (shape >= 3) return TW_ERR_BAD_ARGUMENT;
  if (shape == 2)
    return launch_tiled<T, OutT, 2, 4, SHUF, GLU>(A, lda, W, ldw, bias, residual, ldr, C, ldc, partial, partial_bytes, M, N, K, splits, stream, mode);
  return launch_tiled<T, OutT, 2, 2, SHUF, GLU>(A, lda, W, ldw, bias, residual, ldr, C, ldc, partial, partial_bytes, M, N, K, splits, stream, mode);
}

template <typename T, typename OutT>
static int tiled_by_layout(int shuffled, int glu, int shape, const void* A, long lda, const void* W, long ldw,
                           const float* bias, const float* residual, long ldr, void* C, long ldc, float* partial,
                           long partial_bytes, int M, int N, int K, hipStream_t stream,
                           TiledMode* mode = nullptr) {
  const T* a = (const T*)A;
  const T* w = (const T*)W;
  OutT* c = (OutT*)C;
  if (glu) {
    if constexpr (sizeof(T) == sizeof(OutT)) {
      if (shuffled) return tiled_by_shape<T, OutT, true, true>(shape, a, lda, w, ldw, bias, residual, ldr, c, ldc, partial, partial_bytes, M, N, K, stream, mode);
      return tiled_by_shape<T, OutT, false, true>(shape, a, lda, w, ldw, bias, residual, ldr, c, ldc, partial, partial_bytes, M, N, K, stream, mode);
    }
    return TW_ERR_BAD_ARGUMENT;          // the GLU form writes the input type
  }
  if (shuffled) return tiled_by_shape<T, OutT, true, false>(shape, a, lda, w, ldw, bias, residual, ldr, c, ldc, partial, partial_bytes, M, N, K, stream, mode);
  return tiled_by_shape<T, OutT, false, false>(shape, a, lda, w, ldw, bias, residual, ldr, c, ldc, partial, partial_bytes, M, N, K, stream, mode);
}

int tw_tiled_linear(int dtype, int out_f32, int shuffled, int glu, int shape, const void* A, long lda,
                    const void* W, long ldw, const float* bias, const float* residual, long ldr, void* C,
                    long ldc, float* partial, long partial_bytes, int M, int N, int K, hipStream_t stream) {
  TW_REQUIRE(shape >= 0 && shape <= 9);
  if (dtype == TW_DTYPE_F32)
    return tiled_by_layout<float, float>(shuffled, glu, shape, A, lda, W, ldw, bias, residual, ldr, C, ldc, partial, partial_bytes, M, N, K, stream);
  if (dtype != TW_DTYPE_BF16) return TW_ERR_BAD_ARGUMENT;
  if (out_f32)
    return tiled_by_layout<bf16_t, float>(shuffled, glu, shape, A, lda, W, ldw, bias, residual, ldr, C, ldc, partial, partial_bytes, M, N, K, stream);
  return tiled_by_layout<bf16_t, bf16_t>(shuffled, glu, shape, A, lda, W, ldw, bias, residual, ldr, C, ldc, partial, partial_bytes, M, N, K, stream);
}

// K ranges the tiled kernels would use for this product (1: no split).
int tw_tiled_partial_splits(int dtype, int shuffled, long lda, int M, int N, int K) {
  TiledMode mode;
  mode.dry = true;
  int err;
  const long ldw = shuffled ? tw_div_up(K, dtype == TW_DTYPE_F32 ? 16 : 32) : K;
  if (dtype == TW_DTYPE_F32)
    err = tiled_by_layout<float, float>(shuffled, 0, 0, nullptr, lda, nullptr, ldw, nullptr, nullptr, 0, nullptr, N, nullptr, 0, M, N, K, nullptr, &mode);
  else if (dtype == TW_DTYPE_BF16)
    err = tiled_by_layout<bf16_t, float>(shuffled, 0, 0, nullptr, lda, nullptr, ldw, nullptr, nullptr, 0, nullptr, N, nullptr, 0, M, N, K, nullptr, &mode);
  else
    return 0;
  return err ? 0 : mode.splits;
}

// partial[s][M][N] (float32) = A[:, K range s] W[:, K range s]^T for the ranges the tiled kernels choose;
// no reduction. *splits_used tells how many ranges there are (1: partial[0] is the product itself).
int tw_tiled_partials(int dtype, int shuffled, const void* A, long lda, const void* W, long ldw, float* partial,
                      long partial_bytes, int M, int N, int K, int* splits_used, hipStream_t stream) {
  TW_REQUIRE(partial != nullptr && (uintptr_t)partial % 16 == 0 && partial_bytes >= (long)M * N * 4);
  TiledMode mode;
  mode.leave = true;
  int err;
  if (dtype == TW_DTYPE_F32)
    err = tiled_by_layout<float, float>(shuffled, 0, 0, A, lda, W, ldw, nullptr, nullptr, 0, partial, N, partial, partial_bytes, M, N, K, stream, &mode);
  else if (dtype == TW_DTYPE_BF16)
    err = tiled_by_layout<bf16_t, float>(shuffled, 0, 0, A, lda, W, ldw, nullptr, nullptr, 0, partial, N, partial, partial_bytes, M, N, K, stream, &mode);
  else
    return TW_ERR_BAD_ARGUMENT;
  if (splits_used) *splits_used = mode.splits;
  return err;
}

long tw_tiled_workspace_bytes(int dtype, int rows, int N, int K) {
  const int epf = dtype == TW_DTYPE_F32 ? 4 : 8;
  // enough for whichever kernel runs: the 128x128 tiles' own rule, float32's plan, or either plan for shuffled bfloat16 weights
  int most = tiled_splits(rows, N, K, epf, 128, 128);
  if (dtype == TW_DTYPE_F32) most = std::max(most, choose_parts(false, rows, N, K).splits);
  auto ask = [&](const TilePlan& plan) {
    const int s = plan.splits > 0 ? plan.splits : tiled_splits(rows, N, K, epf, kTileM[plan.shape], kTileN[plan.shape]);
    if (s > most) most = s;
  };
  if (dtype == TW_DTYPE_BF16) {
    ask(choose_staged(true, false, rows, N, K, epf));
    if (K % 64 == 0) ask(choose_turns(false, rows, N, K));
  }
  return most > 1 ? (long)most * rows * N * 4 : 0;
}
