// The gated delta rule: a recurrent mixer whose state is corrected towards each new value before it is read.
//
//   per value head h (its query/key head is h / (H / G)), S: [D][E] float32, carried from step to step:
//     q~ = q / sqrt(sum q^2 + 1e-6) * q_scale        k~ = k / sqrt(sum k^2 + 1e-6)
//     beta = sigmoid(b)      g = exp(-exp(A_log_h) * softplus(a + dt_bias_h))
//     S <- g S;   u = beta (v - S^T k~);   S <- S + k~ u^T;   o = S^T q~          (the read-out sees the token's write)
//
// q, k, v arrive in float32 (a short convolution's result), b and a are columns of a float32 projection; the unit
// norms, the gates, the state and every product with it are float32. A step's rows of one sequence are walked in
// order from the request's state, which the same lanes read at the start and write at the end: nothing depends on
// how a prompt was cut.
//
// A workgroup owns 256 / KS value columns of one (sequence, head). A wave holds 64 / KS of them: lane = KS * column +
// slice, and a lane keeps part `slice` of its column of S in registers (DPL elements), so both products of a token are
// DPL multiply-adds and a sum over KS neighbouring lanes (DPP: inside a quad, or rotations of a row of 16). What a token
// costs is the length of that dependent chain, so keys longer than 16 are cut into 16 slices: 8 multiply-adds a
// product at a key size of 128, and a head's columns spread over eight workgroups. The state lies in memory as
// [H][E][Dk] (a column of S is contiguous), Dk <= KS * DPL. Tokens are staged in LDS in chunks: the waves share a
// chunk's tokens out, norm q and k, form beta and g, then all walk the chunk.
#include "tw_common.h"
#include "norm_gate.h"

#define TW_DELTA_CHUNK 16             /* tokens the walk stages at a time */
#define TW_DELTA_WALK_MOST 4          /* up to this many tokens a sequence, a step walks them one by one */

struct DeltaArgs {
  const float* qkv; long ld_qkv;      // q of key head j at q_col + j * D, k at k_col + j * D, v of head h at v_col + h * E
  int q_col, k_col, v_col;
  const float* ab; long ld_ab;        // b of head h at b_col + h, a at a_col + h
  int b_col, a_col;
  const float* A_log; const float* dt_bias;   // [H]
  float* state;                       // [requests][H][E][Dk]
  const int* q_start; const int* state_slots;
  float* out; long ld_out;            // float32 [n][>= H * E]: head h at h * E
  int H, G, D, E, Dk;
  float q_scale;
  int row0, row1;                     // chunks of 32: of the launch's rows, those that this pair of launches takes
};

template <int CTRL>
__device__ __forceinline__ float delta_quad_swap(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}
// sum over KS neighbouring lanes (4: a quad; 16: a row); every lane gets it
template <int KS>
__device__ __forceinline__ float delta_group_sum(float v) {
  if constexpr (KS == 4) {
    v += delta_quad_swap<0xB1>(v);    // lanes 1 0 3 2
    v += delta_quad_swap<0x4E>(v);    // lanes 2 3 0 1
  } else {
    v += delta_quad_swap<0x128>(v);   // the row rotated by 8 lanes, then by 4, 2, 1
    v += delta_quad_swap<0x124>(v);
    v += delta_quad_swap<0x122>(v);
    v += delta_quad_swap<0x121>(v);
  }
  return v;
}

__device__ __forceinline__ float delta_softplus(float x) { return x > 20.f ? x : log1pf(expf(x)); }

template <int DPL, int KS>
__global__ __launch_bounds__(256) void delta_walk_kernel(DeltaArgs a, int seq0) {
  constexpr int SL = DPL + 4;                        // a slice's stride in LDS: the slices a read meets lie in different banks
  constexpr int ROW = KS * SL;
  constexpr int CW = 256 / KS, CV = 64 / KS;         // value columns a workgroup, a wave
  __shared__ __attribute__((aligned(16))) float q_s[TW_DELTA_CHUNK][ROW];
  __shared__ __attribute__((aligned(16))) float k_s[TW_DELTA_CHUNK][ROW];
  __shared__ float v_s[TW_DELTA_CHUNK][CW];
  __shared__ float gate_s[TW_DELTA_CHUNK][2];        // beta, g
  const int blocks_e = (a.E + CW - 1) / CW;
  const int eb = blockIdx.x % blocks_e, head = blockIdx.x / blocks_e;
  const int s = seq0 + blockIdx.y;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int slice = lane & (KS - 1);
  const int e = eb * CW + wave * CV + lane / KS;
  const bool live = e < a.E;
  const int kh = head / (a.H / a.G);
  const int first = a.q_start[s], last = a.q_start[s + 1];
  float* S_mem = a.state + (((size_t)a.state_slots[s] * a.H + head) * a.E + (live ? e : 0)) * a.Dk + slice * DPL;
  const bool held = live && slice * DPL < a.Dk;      // (Dk may be shorter than 4 * DPL: the last slices then hold nothing)
  float S[DPL];
#pragma unroll
  for (int i = 0; i < DPL; i += 4) {
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (held && slice * DPL + i < a.Dk) v = *reinterpret_cast<const f32x4*>(S_mem + i);
    S[i] = v[0]; S[i + 1] = v[1]; S[i + 2] = v[2]; S[i + 3] = v[3];
  }
  const float rate = -expf(a.A_log[head]);
  const float dt_bias = a.dt_bias[head];
  for (int t0 = first; t0 < last; t0 += TW_DELTA_CHUNK) {
    const int nt = min(TW_DELTA_CHUNK, last - t0);
    __syncthreads();                                 // the chunk before has been walked by every wave
    for (int i = wave; i < nt; i += 4) {
      const float* row = a.qkv + (size_t)(t0 + i) * a.ld_qkv;
      const float* qr = row + a.q_col + (size_t)kh * a.D;
      const float* kr = row + a.k_col + (size_t)kh * a.D;
      float qv[4], kv[4], qq = 0.f, kk = 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int d = lane + 64 * j;
        qv[j] = d < a.D ? qr[d] : 0.f;
        kv[j] = d < a.D ? kr[d] : 0.f;
        qq = __fmaf_rn(qv[j], qv[j], qq);
        kk = __fmaf_rn(kv[j], kv[j], kk);
      }
      qq = tw_wave_sum(qq);
      kk = tw_wave_sum(kk);
      const float qn = a.q_scale / sqrtf(qq + 1e-6f), kn = 1.f / sqrtf(kk + 1e-6f);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int d = lane + 64 * j;
        if (d < KS * DPL) {
          q_s[i][(d / DPL) * SL + d % DPL] = qv[j] * qn;
          k_s[i][(d / DPL) * SL + d % DPL] = kv[j] * kn;
        }
      }
      const int ev = eb * CW + lane;
      if (lane < CW) v_s[i][lane] = ev < a.E ? row[a.v_col + (size_t)head * a.E + ev] : 0.f;
      if (lane == 0) {
        const float* ab = a.ab + (size_t)(t0 + i) * a.ld_ab;
        const float b = ab[a.b_col + head], x = ab[a.a_col + head];
        gate_s[i][0] = 1.f / (1.f + expf(-b));
        gate_s[i][1] = expf(rate * delta_softplus(x + dt_bias));
      }
    }
    __syncthreads();
    for (int i = 0; i < nt; ++i) {
      const float* kp = &k_s[i][slice * SL];
      const float* qp = &q_s[i][slice * SL];
      const float beta = gate_s[i][0], g = gate_s[i][1];
      float d0 = 0.f, d1 = 0.f, d2 = 0.f, d3 = 0.f;
#pragma unroll
      for (int j = 0; j < DPL; j += 4) {
        const f32x4 kq = *reinterpret_cast<const f32x4*>(kp + j);
        d0 = __fmaf_rn(S[j], kq[0], d0);
        d1 = __fmaf_rn(S[j + 1], kq[1], d1);
        d2 = __fmaf_rn(S[j + 2], kq[2], d2);
        d3 = __fmaf_rn(S[j + 3], kq[3], d3);
      }
      const float dot = delta_group_sum<KS>((d0 + d1) + (d2 + d3));
      const float u = beta * (v_s[i][wave * CV + lane / KS] - g * dot);
      float o0 = 0.f, o1 = 0.f, o2 = 0.f, o3 = 0.f;
#pragma unroll
      for (int j = 0; j < DPL; j += 4) {
        const f32x4 kq = *reinterpret_cast<const f32x4*>(kp + j);
        const f32x4 qq = *reinterpret_cast<const f32x4*>(qp + j);
        S[j] = __fmaf_rn(kq[0], u, g * S[j]);
        S[j + 1] = __fmaf_rn(kq[1], u, g * S[j + 1]);
        S[j + 2] = __fmaf_rn(kq[2], u, g * S[j + 2]);
        S[j + 3] = __fmaf_rn(kq[3], u, g * S[j + 3]);
        o0 = __fmaf_rn(S[j], qq[0], o0);
        o1 = __fmaf_rn(S[j + 1], qq[1], o1);
        o2 = __fmaf_rn(S[j + 2], qq[2], o2);
        o3 = __fmaf_rn(S[j + 3], qq[3], o3);
      }
      const float o = delta_group_sum<KS>((o0 + o1) + (o2 + o3));
      if (live && slice == 0) a.out[(size_t)(t0 + i) * a.ld_out + (size_t)head * a.E + e] = o;
    }
  }
#pragma unroll
  for (int i = 0; i < DPL; i += 4)
    if (held && slice * DPL + i < a.Dk) *reinterpret_cast<f32x4*>(S_mem + i) = f32x4{S[i], S[i + 1], S[i + 2], S[i + 3]};
}

// The waves of a workgroup meet once each one's LDS traffic is done. (Unlike __syncthreads() this does not wait for loads
// from memory: the next chunk's rows stay on their way across it.)
__device__ __forceinline__ void delta_lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// ---- many tokens a sequence: chunks of 32 tokens, solved side by side, then walked ----------------------------------
// Inside a chunk with state S0 at its start, L_i = sum_{m <= i} log g_m (so that G_i = exp(L_i) and every quotient
// G_i / G_j, j <= i, is an exponential of a sum of logarithms that are at most 0):
//   u_i = beta_i (v_i - G_i S0^T k_i) - sum_{j < i} A_ij u_j,      A_ij = beta_i (G_i / G_j) (k_i . k_j)
//   o_i = G_i S0^T q_i + sum_{j <= i} M_ij u_j,                    M_ij = (G_i / G_j) (q_i . k_j)
//   S   = G_last S0 + sum_j (G_last / G_j) k_j u_j^T
// which is the token-by-token rule written out. All of it but the products with S0 is the same whatever the state is: with
// T = (I + A)^-1, W = T (beta G K) and U0 = T (beta V)
//   U = U0 - W S0,    O = M U0 + (G Q - M W) S0,    S = G_last S0 + K'^T U.
// delta_prepare forms W, Q' = G Q - M W, K', U0 and O0 = M U0 for every (chunk, head) at once; delta_chunk then goes through a
// sequence's chunks with three products each. Everything is float32, the products on the matrix unit (16x16x4). T comes from
// substitution, a column a lane, in blocks of 16 tokens (a series in powers of A would lose digits where keys are alike). For
// the same reason the products of keys are sums of eight elements added in 64 bits, and a chunk's change of the state is summed
// before it meets the state. Errors against 64 bits (400 tokens, heads of 128), outputs and state: 1.9e-7 and 1.5e-7, with keys
// that share half of their length 3.0e-7 and 2.8e-7 (with one float32 chain each 2.6e-7 and 2.2e-7, 7.4e-7 and 6.9e-7; chunks
// of 16 solved in the chain of tokens 2.3e-7 and 2.2e-7, 3.6e-7 and 3.4e-7). The time is the same.
//
// What bounds them: delta_chunk the chain from chunk to chunk and the 48 KB of operands a chunk that each of its workgroups
// reads (2 us a chunk, 30 GB/s a CU), delta_prepare its own length: written out over the 32 tokens with a thread a column it
// was 4,000 instructions, executed once, and took 32 us for one chunk. Solved inside the chain (chunks of 16 tokens, four
// barriers each) a chunk took 4.5 us. 16 heads of 128, the two launches
// together: one sequence of 2,048 tokens 579 -> 170 us, two of 800 and 1,200 tokens 340 -> 120 us, 100 tokens 34 -> 24 us.
#define TW_DELTA_PREP 32              /* tokens a chunk */

struct DeltaPrepared {                // per (chunk, head), all in the order the walk's lanes read them, 16 bytes a lane
  float* W;                           // [4 waves][NT][2][64][4]: A operands, row = token, reduction = the wave's key elements
  float* Q;                           // the same of Q'
  float* K;                           // [4][NT][2][64][4]: A operands of K'^T, row = key element, reduction = token
  float* U;                           // [value tiles][2][64][4]: accumulators, row = token, column = value
  float* O;                           // the same of O0
  float* G;                           // [1]: G_last
};

// A sequence's rows among those that a pair of launches takes (none: first == last).
__device__ __forceinline__ void delta_rows(const DeltaArgs& a, int seq0, int s, int& first, int& last) {
  const int lo = a.q_start[seq0] + a.row0, hi = a.q_start[seq0] + a.row1;
  first = min(max(a.q_start[s], lo), hi);
  last = min(max(a.q_start[s + 1], lo), hi);
}

// The number of a sequence's first chunk: chunks of sequences never overlap whatever their lengths, and there are at most
// rows / 32 + sequences of them.
__device__ __forceinline__ int delta_first_chunk(const DeltaArgs& a, int seq0, int s) {
  int first, last;
  delta_rows(a, seq0, s, first, last);
  return (first - a.q_start[seq0] - a.row0) / TW_DELTA_PREP + (s - seq0);
}

// grid (chunk numbers, H), 256 threads
template <int NT>
__global__ __launch_bounds__(256) void delta_prepare_kernel(DeltaArgs a, DeltaPrepared out, int seq0, int n_seqs) {
  constexpr int C = TW_DELTA_PREP, DP = 64 * NT, ROW = DP + 4, PW = C + 4;
  __shared__ __attribute__((aligned(16))) float q_s[C][ROW];
  __shared__ __attribute__((aligned(16))) float k_s[C][ROW];
  __shared__ __attribute__((aligned(16))) float at_s[C][PW];     // k_j . k_i, then A_ij at [j][i] (0 unless j < i)
  __shared__ __attribute__((aligned(16))) float m_s[C][PW];      // q_i . k_j, then M_ij at [i][j] (0 unless j <= i)
  __shared__ __attribute__((aligned(16))) float t_s[C][PW];      // T (its block above the diagonal is never read)
  __shared__ __attribute__((aligned(16))) float mt_s[C][PW];     // M T
  __shared__ float beta_s[C], lg_s[C], g_s[C], kn_s[C], qn_s[C], tail_s[C];
  const int chunk = blockIdx.x, head = blockIdx.y;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // the sequence this chunk number belongs to: the last one whose first chunk is not behind it
  int s = -1;
  for (int s0 = 0; s0 < n_seqs; s0 += 64) {
    const bool in = s0 + lane < n_seqs && delta_first_chunk(a, seq0, seq0 + s0 + lane) <= chunk;
    const int n = __popcll(__ballot(in));
    s = n ? s0 + n - 1 : s;
    if (n < 64) break;
  }
  s += seq0;
  int first, last;
  delta_rows(a, seq0, s, first, last);
  const int t0 = first + (chunk - delta_first_chunk(a, seq0, s)) * C;
  if (t0 >= last) return;                            // (a number that no chunk has)
  const int kh = head / (a.H / a.G);

  // ---- rows and gates into LDS (tokens behind the sequence's end: zeros, beta = 0, g = 1) -----------------------------
  // (Loads are whole, from clamped places, and issued together: a load behind a condition waits for the one before.)
  const int r = lane & 15, g = lane >> 4;
  const int value_tiles = (a.E + 15) / 16;
  auto values = [&](int x, f32x4* vf) {              // value tile x: the B operands of a product over tokens
    const float* v = a.qkv + a.v_col + (size_t)head * a.E + min(16 * x + r, a.E - 1);
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
      for (int j = 0; j < 4; ++j) vf[tt][j] = v[(size_t)min(t0 + 16 * tt + 4 * g + j, last - 1) * a.ld_qkv];
  };
  f32x4 vf[2];
  values(min(wave, value_tiles - 1), vf);            // (needed at the end only)
  const bool vec = a.D % 4 == 0 && a.ld_qkv % 4 == 0 && a.q_col % 4 == 0 && a.k_col % 4 == 0 && (uintptr_t)a.qkv % 16 == 0;
  if (vec) {
    constexpr int N = C * DP / 4 / 256;
    f32x4 qv[N], kv[N];
#pragma unroll
    for (int n = 0; n < N; ++n) {
      const int x = threadIdx.x + 256 * n, t = x / (DP / 4), d = (x % (DP / 4)) * 4;
      const float* row = a.qkv + (size_t)min(t0 + t, last - 1) * a.ld_qkv + (size_t)kh * a.D + min(d, a.D - 4);
      qv[n] = *reinterpret_cast<const f32x4*>(row + a.q_col);
      kv[n] = *reinterpret_cast<const f32x4*>(row + a.k_col);
    }
#pragma unroll
    for (int n = 0; n < N; ++n) {
      const int x = threadIdx.x + 256 * n, t = x / (DP / 4), d = (x % (DP / 4)) * 4;
      const bool in = t0 + t < last && d < a.D;
#pragma unroll
      for (int j = 0; j < 4; ++j) { qv[n][j] = in ? qv[n][j] : 0.f; kv[n][j] = in ? kv[n][j] : 0.f; }
      *reinterpret_cast<f32x4*>(&q_s[t][d]) = qv[n];
      *reinterpret_cast<f32x4*>(&k_s[t][d]) = kv[n];
    }
  } else {
    for (int x = threadIdx.x; x < C * DP; x += 256) {
      const int t = x / DP, d = x % DP;
      const bool in = t0 + t < last && d < a.D;
      const float* row = a.qkv + (size_t)min(t0 + t, last - 1) * a.ld_qkv + (size_t)kh * a.D + min(d, a.D - 1);
      const float qv = row[a.q_col], kv = row[a.k_col];
      q_s[t][d] = in ? qv : 0.f;
      k_s[t][d] = in ? kv : 0.f;
    }
  }
  if (threadIdx.x < C) {
    const bool in = t0 + threadIdx.x < last;
    const float* ab = a.ab + (size_t)(in ? t0 + threadIdx.x : t0) * a.ld_ab;
    beta_s[threadIdx.x] = in ? 1.f / (1.f + expf(-ab[a.b_col + head])) : 0.f;
    lg_s[threadIdx.x] = in ? -expf(a.A_log[head]) * delta_softplus(ab[a.a_col + head] + a.dt_bias[head]) : 0.f;
  }
  __syncthreads();

  // ---- K K^T and Q K^T, the three tiles on and below the diagonal by a wave each; the fourth wave: squared lengths ------
  if (wave < 3) {
    const int ti = wave ? 1 : 0, tj = wave == 2 ? 1 : 0;
    // (sums of eight elements, added in 64 bits: where keys are alike, rounding here doubled the error of the results)
    double kk[4] = {0., 0., 0., 0.}, qk[4] = {0., 0., 0., 0.};
#pragma unroll
    for (int x = 0; x < 4 * NT; ++x) {
      const f32x4 kj = *reinterpret_cast<const f32x4*>(&k_s[16 * tj + r][16 * x + 4 * g]);
      const f32x4 ki = *reinterpret_cast<const f32x4*>(&k_s[16 * ti + r][16 * x + 4 * g]);
      const f32x4 qi = *reinterpret_cast<const f32x4*>(&q_s[16 * ti + r][16 * x + 4 * g]);
#pragma unroll
      for (int h = 0; h < 4; h += 2) {
        f32x4 kp = {0.f, 0.f, 0.f, 0.f}, qp = kp;
#pragma unroll
        for (int e = h; e < h + 2; ++e) {
          kp = __builtin_amdgcn_mfma_f32_16x16x4f32(ki[e], kj[e], kp, 0, 0, 0);
          qp = __builtin_amdgcn_mfma_f32_16x16x4f32(qi[e], kj[e], qp, 0, 0, 0);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) { kk[j] += kp[j]; qk[j] += qp[j]; }
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      at_s[16 * tj + r][16 * ti + 4 * g + j] = (float)kk[j];
      m_s[16 * ti + 4 * g + j][16 * tj + r] = (float)qk[j];
    }
  } else {
    const int t = lane >> 1;
    float qq = 0.f, kk = 0.f;
#pragma unroll 1
    for (int y = 0; y < NT; ++y) {                   // (sums of eight squares, added in pairs)
      f32x4 qp = {0.f, 0.f, 0.f, 0.f}, kp = qp;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int d = 64 * y + 8 * i + (lane & 1) * 4;
        const f32x4 qv = *reinterpret_cast<const f32x4*>(&q_s[t][d]), kv = *reinterpret_cast<const f32x4*>(&k_s[t][d]);
#pragma unroll
        for (int j = 0; j < 4; ++j) { qp[j] = __fmaf_rn(qv[j], qv[j], qp[j]); kp[j] = __fmaf_rn(kv[j], kv[j], kp[j]); }
      }
      qq += (qp[0] + qp[1]) + (qp[2] + qp[3]);
      kk += (kp[0] + kp[1]) + (kp[2] + kp[3]);
    }
    qq += __shfl_xor(qq, 1, TW_WAVE);
    kk += __shfl_xor(kk, 1, TW_WAVE);
    if (!(lane & 1)) {
      kn_s[t] = 1.f / sqrtf(kk + 1e-6f);
      qn_s[t] = a.q_scale / sqrtf(qq + 1e-6f);
    }
  }
  __syncthreads();

  // ---- the decay between tokens, beta and the unit norms put on them ----------------------------------------------------
  {
    const int j = threadIdx.x % C, i0 = threadIdx.x / C;         // this thread's pairs: (i0 + 8 p, j)
    float between[4] = {0.f, 0.f, 0.f, 0.f};         // logs of G_i / G_j (j <= i), summed over the tokens in between
#pragma unroll 8
    for (int m = 0; m < C; ++m) {
      const float lg = m > j ? lg_s[m] : 0.f;
#pragma unroll
      for (int p = 0; p < 4; ++p) between[p] += m <= i0 + 8 * p ? lg : 0.f;
    }
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int i = i0 + 8 * p;
      const float decay = expf(between[p]);
      // (one rounding each)
      const double unit = (double)decay * kn_s[j];
      at_s[j][i] = j < i ? (float)(beta_s[i] * unit * kn_s[i] * at_s[j][i]) : 0.f;
      m_s[i][j] = j <= i ? (float)(unit * qn_s[i] * m_s[i][j]) : 0.f;
      if (i == C - 1) tail_s[j] = (float)unit;
      if (j == 0) g_s[i] = expf(between[p] + lg_s[0]);
    }
  }
  __syncthreads();

  // ---- T = (I + A)^-1, by the first wave: the two diagonal blocks by substitution (a lane a column), then the block below ---
  if (wave == 0) {
    if (lane < 32) {
      const int b = lane & 16;                       // the block's first token
      float x[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) x[i] = i == r ? 1.f : 0.f;
#pragma unroll
      for (int j = 0; j < 15; ++j)
#pragma unroll
        for (int i4 = (j + 1) / 4 * 4; i4 < 16; i4 += 4) {
          const f32x4 v = *reinterpret_cast<const f32x4*>(&at_s[b + j][b + i4]);
#pragma unroll
          for (int y = 0; y < 4; ++y)
            if (i4 + y > j) x[i4 + y] = __fmaf_rn(-v[y], x[j], x[i4 + y]);
        }
#pragma unroll
      for (int i = 0; i < 16; ++i) t_s[b + i][b + r] = x[i];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    f32x4 below, left, p = {0.f, 0.f, 0.f, 0.f}, t21 = p;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      below[j] = at_s[4 * g + j][16 + r];            // A of the lower tokens on the upper ones, row r
      left[j] = t_s[4 * g + j][r];
    }
    tw_mma16(p, below, left);                        // an accumulator, and the next product's B operand
    tw_mma16(t21, *reinterpret_cast<const f32x4*>(&t_s[16 + r][16 + 4 * g]), p);
#pragma unroll
    for (int j = 0; j < 4; ++j) t_s[16 + 4 * g + j][r] = -t21[j];
  }
  __syncthreads();

  // ---- M T, its three tiles on and below the diagonal by a wave each --------------------------------------------------------
  if (wave < 3) {
    const int ti = wave ? 1 : 0, tj = wave == 2 ? 1 : 0;
    f32x4 mt = {0.f, 0.f, 0.f, 0.f};
    for (int tk = tj; tk <= ti; ++tk) {
      f32x4 tf;
#pragma unroll
      for (int j = 0; j < 4; ++j) tf[j] = t_s[16 * tk + 4 * g + j][16 * tj + r];
      tw_mma16(mt, *reinterpret_cast<const f32x4*>(&m_s[16 * ti + r][16 * tk + 4 * g]), tf);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) mt_s[16 * ti + 4 * g + j][16 * tj + r] = mt[j];
  }
  __syncthreads();

  // ---- the five results -----------------------------------------------------------------------------------------------------
  const size_t unit = (size_t)chunk * a.H + head;
  if (threadIdx.x == 0) out.G[unit] = g_s[C - 1];
  // rows of T and M T (tiles 00, 10, 11), their columns times beta G / |k| for the keys and times beta for the values
  f32x4 tk[3], mk[3], tv[3], mv[3];
#pragma unroll
  for (int t = 0; t < 3; ++t) {
    const int row = (t ? 16 : 0) + r, col = (t == 2 ? 16 : 0) + 4 * g;
    const f32x4 tr = *reinterpret_cast<const f32x4*>(&t_s[row][col]), mr = *reinterpret_cast<const f32x4*>(&mt_s[row][col]);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float bv = beta_s[col + j], bk = bv * g_s[col + j] * kn_s[col + j];
      tk[t][j] = tr[j] * bk;
      mk[t][j] = mr[j] * bk;
      tv[t][j] = tr[j] * bv;
      mv[t][j] = mr[j] * bv;
    }
  }
  // keys, a tile of 16 a wave and round: K^T is the A operand, so that a lane ends with four key elements of one token, which
  // is how the walk takes W and Q', and K' is K^T itself
  float* W = out.W + unit * C * DP + lane * 4;
  float* Q = out.Q + unit * C * DP + lane * 4;
  float* K = out.K + unit * C * DP + lane * 4;
#pragma unroll 1
  for (int x = wave; x < 4 * NT; x += 4) {
    f32x4 kf[2], w[2], q[2];
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      f32x4 tail;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        kf[tt][j] = k_s[16 * tt + 4 * g + j][16 * x + r];
        tail[j] = kf[tt][j] * tail_s[16 * tt + 4 * g + j];
      }
      *reinterpret_cast<f32x4*>(K + (x * 2 + tt) * 256) = tail;
      w[tt] = q[tt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    tw_mma16(w[0], kf[0], tk[0]);
    tw_mma16(q[0], kf[0], mk[0]);
    tw_mma16(w[1], kf[0], tk[1]);
    tw_mma16(q[1], kf[0], mk[1]);
    tw_mma16(w[1], kf[1], tk[2]);
    tw_mma16(q[1], kf[1], mk[2]);
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      const float gq = g_s[16 * tt + r] * qn_s[16 * tt + r];
      const f32x4 qv = *reinterpret_cast<const f32x4*>(&q_s[16 * tt + r][16 * x + 4 * g]);
#pragma unroll
      for (int j = 0; j < 4; ++j) q[tt][j] = __fmaf_rn(gq, qv[j], -q[tt][j]);
      *reinterpret_cast<f32x4*>(W + (x * 2 + tt) * 256) = w[tt];
      *reinterpret_cast<f32x4*>(Q + (x * 2 + tt) * 256) = q[tt];
    }
  }
  // values, a tile of 16 columns a wave and round (columns behind the last one: the last one's, which nobody reads)
  float* U = out.U + unit * C * 16 * value_tiles + lane * 4;
  float* O = out.O + unit * C * 16 * value_tiles + lane * 4;
#pragma unroll 1
  for (int x = wave; x < value_tiles; x += 4) {
    f32x4 u[2], o[2], next[2];
    values(min(x + 4, value_tiles - 1), next);
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) u[tt] = o[tt] = f32x4{0.f, 0.f, 0.f, 0.f};
    tw_mma16(u[0], tv[0], vf[0]);
    tw_mma16(o[0], mv[0], vf[0]);
    tw_mma16(u[1], tv[1], vf[0]);
    tw_mma16(o[1], mv[1], vf[0]);
    tw_mma16(u[1], tv[2], vf[1]);
    tw_mma16(o[1], mv[2], vf[1]);
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      *reinterpret_cast<f32x4*>(U + (x * 2 + tt) * 256) = u[tt];
      *reinterpret_cast<f32x4*>(O + (x * 2 + tt) * 256) = o[tt];
      vf[tt] = next[tt];
    }
  }
}

// grid (H * value tiles, n_seqs). A workgroup owns 16 value columns of one (sequence, head); its four waves own a quarter of
// the key elements each (NT tiles of 16), and a wave's part of S stays in registers in the layout that is both the B operand of
// W S and Q' S and the accumulator of K'^T U: lane (c, g) holds S[16 tile + 4 g + j][c]. Per chunk the waves' parts of the two
// products meet in LDS (twice, so that one barrier a chunk is enough), every wave adds them up and updates its part of S, two
// waves write the outputs. A chunk's operands are requested two chunks ahead.
template <int NT>
__global__ __launch_bounds__(256) void delta_chunk_kernel(DeltaArgs a, DeltaPrepared in, int seq0) {
  constexpr int C = TW_DELTA_PREP, DP = 64 * NT;
  __shared__ __attribute__((aligned(16))) f32x4 part_s[2][4][4][64];   // [copy][wave][W S of two token tiles, Q' S of two][lane]
  const int value_tiles = (a.E + 15) / 16;
  const int eb = blockIdx.x % value_tiles, head = blockIdx.x / value_tiles;
  const int s = seq0 + blockIdx.y;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int e = eb * 16 + r;                         // this lane's value column
  const bool live = e < a.E;
  int first, last;
  delta_rows(a, seq0, s, first, last);
  if (first >= last) return;
  const int chunks = (last - first + C - 1) / C;
  const size_t unit0 = (size_t)delta_first_chunk(a, seq0, s) * a.H + head;
  const int d_wave = 16 * NT * wave;                 // the wave's first key element
  float* S_mem = a.state + (((size_t)a.state_slots[s] * a.H + head) * a.E + (live ? e : 0)) * a.Dk;
  f32x4 S[NT];
#pragma unroll
  for (int mm = 0; mm < NT; ++mm) {
    const int d0 = d_wave + 16 * mm + 4 * g;
    S[mm] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (live && d0 < a.Dk) S[mm] = *reinterpret_cast<const f32x4*>(S_mem + d0);
  }
  struct Operands {
    f32x4 w[NT][2], q[NT][2], k[NT][2], u[2], o;
    float G;
  };
  auto request = [&](int chunk, Operands& x) __attribute__((always_inline)) {
    const size_t unit = unit0 + (size_t)chunk * a.H;
    const size_t keys = unit * C * DP + (size_t)wave * NT * 512 + lane * 4;
    const size_t values = (unit * value_tiles + eb) * 512 + lane * 4;
#pragma unroll
    for (int mm = 0; mm < NT; ++mm)
#pragma unroll
      for (int tt = 0; tt < 2; ++tt) {
        x.w[mm][tt] = *reinterpret_cast<const f32x4*>(in.W + keys + (mm * 2 + tt) * 256);
        x.q[mm][tt] = *reinterpret_cast<const f32x4*>(in.Q + keys + (mm * 2 + tt) * 256);
        x.k[mm][tt] = *reinterpret_cast<const f32x4*>(in.K + keys + (mm * 2 + tt) * 256);
      }
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) x.u[tt] = *reinterpret_cast<const f32x4*>(in.U + values + tt * 256);
    x.o = *reinterpret_cast<const f32x4*>(in.O + values + (wave & 1) * 256);
    x.G = in.G[unit];
  };
  auto link = [&](int chunk, int copy, Operands& x) __attribute__((always_inline)) {
    f32x4 pw[2], pq[2];
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) pw[tt] = pq[tt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int mm = 0; mm < NT; ++mm)
#pragma unroll
      for (int tt = 0; tt < 2; ++tt) {
        tw_mma16(pw[tt], x.w[mm][tt], S[mm]);        // [token][column]
        tw_mma16(pq[tt], x.q[mm][tt], S[mm]);
      }
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      part_s[copy][wave][tt][lane] = pw[tt];
      part_s[copy][wave][2 + tt][lane] = pq[tt];
    }
    delta_lds_barrier();
    // U of tokens 16 tt + 4 g .. + 3: an accumulator, and the B operand of the product over tokens
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
      x.u[tt] -= (part_s[copy][0][tt][lane] + part_s[copy][1][tt][lane]) + (part_s[copy][2][tt][lane] + part_s[copy][3][tt][lane]);
#pragma unroll
    for (int mm = 0; mm < NT; ++mm) {
      // (the chunk's change is summed by itself: summed onto the state, every one of its products rounds at the state's size)
      f32x4 change = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int tt = 0; tt < 2; ++tt) tw_mma16(change, x.k[mm][tt], x.u[tt]);
#pragma unroll
      for (int j = 0; j < 4; ++j) S[mm][j] = __fmaf_rn(x.G, S[mm][j], change[j]);
    }
    if (wave < 2) {
      const f32x4 o = x.o + ((part_s[copy][0][2 + wave][lane] + part_s[copy][1][2 + wave][lane]) +
                             (part_s[copy][2][2 + wave][lane] + part_s[copy][3][2 + wave][lane]));
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int t = first + chunk * C + 16 * wave + 4 * g + j;
        if (live && t < last) a.out[(size_t)t * a.ld_out + (size_t)head * a.E + e] = o[j];
      }
    }
    if (chunk + 2 < chunks) request(chunk + 2, x);   // (its registers are free again)
  };
  Operands even, odd;
  request(0, even);
  if (chunks > 1) request(1, odd);
  for (int c = 0; c < chunks; c += 2) {
    link(c, 0, even);
    if (c + 1 < chunks) link(c + 1, 1, odd);
  }
#pragma unroll
  for (int mm = 0; mm < NT; ++mm) {
    const int d0 = d_wave + 16 * mm + 4 * g;
    if (live && d0 < a.Dk) *reinterpret_cast<f32x4*>(S_mem + d0) = S[mm];
  }
}

// ---- portions of a few dozen tokens: chunks of 16 tokens, each solved inside the chain --------------------------------
// One launch instead of two (see delta_in_chunks): a few chunks of 4.5 us behind 2.5 us of start end before delta_prepare and
// delta_chunk would (13 + 7 us at 33 tokens, 16 heads of 128). A workgroup owns 16 value columns of one (sequence, head) and its
// waves a quarter of the key elements each, as above. Per chunk: the waves form their parts of K S0, Q S0, K K^T and Q K^T from
// the same fragments, the parts meet in LDS and thread 16 i + j adds them up for the pair (i, j) and puts decay, beta and the
// unit norms on (q and k are multiplied as they come; their squared lengths are the diagonals of K K^T and of one more product,
// Q Q^T); every lane solves the triangular system of its column by substitution; one wave reads the chunk's outputs out, every
// wave updates its part of S. Tokens behind a sequence's end are staged as zeros with beta = 0 and g = 1: they change nothing.
// The next chunk's rows are on their way from memory while this one is worked on.
template <int NT>
__global__ __launch_bounds__(256) void delta_short_kernel(DeltaArgs a, int seq0) {
  constexpr int C = 16, DP = 64 * NT;                // key elements, rounded up: 16 NT a wave
  constexpr int ROW = DP + 4;                        // (+ 4: the four token rows a transposed read meets lie 16 banks apart)
  constexpr int PW = C + 4;
  __shared__ __attribute__((aligned(16))) float q_s[C][ROW];
  __shared__ __attribute__((aligned(16))) float k_s[C][ROW];
  __shared__ __attribute__((aligned(16))) float part_s[4][5][C][C];   // [wave][K S0, Q S0, K K^T, Q K^T, Q Q^T][row][column]
  __shared__ __attribute__((aligned(16))) float v_s[C][C];
  __shared__ __attribute__((aligned(16))) float pk_s[C][C];      // (S0^T k_i)[column]
  __shared__ __attribute__((aligned(16))) float pq_s[C][C];
  __shared__ __attribute__((aligned(16))) float at_s[C][PW];     // at_s[j][i] = A_ij (0 unless j < i)
  __shared__ __attribute__((aligned(16))) float qk_s[C][PW];     // qk_s[i][j] = (G_i / G_j) (q_i . k_j) (0 unless j <= i)
  __shared__ float beta_s[C], lg_s[C], g_s[C], tail_s[C];        // beta_i, log g_i, G_i, G_last / G_i * (1 / |k_i|)
  const int blocks_e = (a.E + 15) / 16;
  const int eb = blockIdx.x % blocks_e, head = blockIdx.x / blocks_e;
  const int s = seq0 + blockIdx.y;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int e = eb * 16 + r;                         // this lane's value column
  const bool live = e < a.E;
  const int kh = head / (a.H / a.G);
  const int first = a.q_start[s], last = a.q_start[s + 1];
  if (first >= last) return;
  const int d_wave = 16 * NT * wave;                 // the wave's first key element
  float* S_mem = a.state + (((size_t)a.state_slots[s] * a.H + head) * a.E + (live ? e : 0)) * a.Dk;
  f32x4 S[NT];
#pragma unroll
  for (int mm = 0; mm < NT; ++mm) {
    const int d0 = d_wave + 16 * mm + 4 * g;
    S[mm] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (live && d0 < a.Dk) S[mm] = *reinterpret_cast<const f32x4*>(S_mem + d0);
  }
  const float rate = -expf(a.A_log[head]);
  const float dt_bias = a.dt_bias[head];

  // a wave stages tokens wave, wave + 4, wave + 8, wave + 12 of a chunk: their raw rows, in registers
  float rq[4][NT], rk[4][NT], rv[4], rb[4], ra[4];
  auto fetch = [&](int t0) {
#pragma unroll
    for (int ii = 0; ii < 4; ++ii) {
      const int t = t0 + wave + 4 * ii;
      const bool in = t < last;
      const float* row = a.qkv + (size_t)(in ? t : first) * a.ld_qkv;
      const float* qr = row + a.q_col + (size_t)kh * a.D;
      const float* kr = row + a.k_col + (size_t)kh * a.D;
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const int d = lane + 64 * j;
        const bool ok = in && d < a.D;
        rq[ii][j] = ok ? qr[d] : 0.f;
        rk[ii][j] = ok ? kr[d] : 0.f;
      }
      const int ev = eb * 16 + r;
      rv[ii] = in && ev < a.E ? row[a.v_col + (size_t)head * a.E + ev] : 0.f;
      const float* ab = a.ab + (size_t)(in ? t : first) * a.ld_ab;
      rb[ii] = ab[a.b_col + head];
      ra[ii] = ab[a.a_col + head];
    }
  };
  auto stage = [&](int t0) {
#pragma unroll
    for (int ii = 0; ii < 4; ++ii) {
      const int i = wave + 4 * ii;
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        q_s[i][lane + 64 * j] = rq[ii][j];           // (as they come: the unit norms are put on the products)
        k_s[i][lane + 64 * j] = rk[ii][j];
      }
      if (lane < 16) v_s[i][lane] = rv[ii];
    }
    // the gates of the wave's four tokens, one lane a token (every lane holds all four tokens' b and a)
    const int mine = lane & 3;
    const float b = mine == 0 ? rb[0] : mine == 1 ? rb[1] : mine == 2 ? rb[2] : rb[3];
    const float x = mine == 0 ? ra[0] : mine == 1 ? ra[1] : mine == 2 ? ra[2] : ra[3];
    if (lane < 4) {
      const int i = wave + 4 * mine;
      const bool in = t0 + i < last;
      beta_s[i] = in ? 1.f / (1.f + expf(-b)) : 0.f;
      lg_s[i] = in ? rate * delta_softplus(x + dt_bias) : 0.f;
    }
  };

  fetch(first);
  for (int t0 = first; t0 < last; t0 += C) {
    delta_lds_barrier();                             // the chunk before has been worked on by every wave
    stage(t0);
    if (t0 + C < last) fetch(t0 + C);
    delta_lds_barrier();

    // ---- this wave's parts of the four products -----------------------------------------------------------------------
    {
      f32x4 pk = {0.f, 0.f, 0.f, 0.f}, pq = pk, kk = pk, qk = pk, qq = pk;
#pragma unroll
      for (int mm = 0; mm < NT; ++mm) {
        const f32x4 kf = *reinterpret_cast<const f32x4*>(&k_s[r][d_wave + 16 * mm + 4 * g]);
        const f32x4 qf = *reinterpret_cast<const f32x4*>(&q_s[r][d_wave + 16 * mm + 4 * g]);
        tw_mma16(pk, kf, S[mm]);                     // [token][column]
        tw_mma16(pq, qf, S[mm]);
        tw_mma16(kk, kf, kf);                        // [token i][token j]
        tw_mma16(qk, qf, kf);
        tw_mma16(qq, qf, qf);                        // (its diagonal: the queries' squared lengths, as K K^T's are the keys')
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        part_s[wave][0][4 * g + j][r] = pk[j];
        part_s[wave][1][4 * g + j][r] = pq[j];
        part_s[wave][2][4 * g + j][r] = kk[j];
        part_s[wave][3][4 * g + j][r] = qk[j];
        part_s[wave][4][4 * g + j][r] = qq[j];
      }
    }
    delta_lds_barrier();

    // ---- thread 16 i + j adds the waves' parts up (in their order) and puts the decay between tokens i and j on -----
    {
      const int i = threadIdx.x >> 4, j = threadIdx.x & 15;
      auto whole = [&](int t, int row, int column) {
        return (part_s[0][t][row][column] + part_s[1][t][row][column]) + (part_s[2][t][row][column] + part_s[3][t][row][column]);
      };
      float sum[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) sum[t] = whole(t, i, j);
      // q and k were multiplied as they came: 1 / |k_i|, 1 / |k_j| and q_scale / |q_i| from the diagonals
      const float kn_i = 1.f / sqrtf(whole(2, i, i) + 1e-6f), kn_j = 1.f / sqrtf(whole(2, j, j) + 1e-6f);
      const float qn_i = a.q_scale / sqrtf(whole(4, i, i) + 1e-6f);
      float between = 0.f, upto = 0.f;               // log of G_i / G_j (j <= i), and L_i
#pragma unroll
      for (int m = 0; m < C; ++m) {
        const float lg = lg_s[m];
        if (m > j && m <= i) between += lg;
        if (m <= i) upto += lg;
      }
      const float decay = expf(between);
      pk_s[i][j] = kn_i * sum[0];
      pq_s[i][j] = qn_i * sum[1];
      at_s[j][i] = j < i ? beta_s[i] * decay * (kn_i * kn_j) * sum[2] : 0.f;
      qk_s[i][j] = j <= i ? decay * (qn_i * kn_j) * sum[3] : 0.f;
      if (j == 0) g_s[i] = expf(upto);
      if (i == C - 1) tail_s[j] = decay * kn_j;
    }
    delta_lds_barrier();

    // ---- the triangular system of this lane's column (the lanes of a column, in every wave, all solve it) -----------
    float u[C];
#pragma unroll
    for (int i = 0; i < C; ++i) u[i] = beta_s[i] * (v_s[i][r] - g_s[i] * pk_s[i][r]);
#pragma unroll
    for (int j = 0; j < C - 1; ++j) {
      float arow[C];
#pragma unroll
      for (int x = 0; x < C; x += 4) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(&at_s[j][x]);
        arow[x] = v[0]; arow[x + 1] = v[1]; arow[x + 2] = v[2]; arow[x + 3] = v[3];
      }
#pragma unroll
      for (int i = j + 1; i < C; ++i) u[i] = __fmaf_rn(-arow[i], u[j], u[i]);
    }
    // u of tokens 4 g .. 4 g + 3: the B operand of the two products over tokens
    f32x4 ub;
#pragma unroll
    for (int j = 0; j < 4; ++j) ub[j] = g == 0 ? u[j] : g == 1 ? u[4 + j] : g == 2 ? u[8 + j] : u[12 + j];

    // ---- the read-out: o_i = G_i (S0^T q_i) + sum_j qk[i][j] u_j, by the chunk's wave in turn -------------------------
    if (wave == ((t0 - first) / C & 3)) {
      f32x4 o = {0.f, 0.f, 0.f, 0.f};
      const f32x4 w = *reinterpret_cast<const f32x4*>(&qk_s[r][4 * g]);
      tw_mma16(o, w, ub);                            // [token i][column]
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int i = 4 * g + j;
        const float out = __fmaf_rn(g_s[i], pq_s[i][r], o[j]);
        if (live && t0 + i < last) a.out[(size_t)(t0 + i) * a.ld_out + (size_t)head * a.E + e] = out;
      }
    }

    // ---- the state behind the chunk: S <- G_last S + K^T diag(G_last / G_j) U ----------------------------------------
    const float G_last = g_s[C - 1];
    f32x4 wb;
#pragma unroll
    for (int j = 0; j < 4; ++j) wb[j] = tail_s[4 * g + j] * ub[j];
#pragma unroll
    for (int mm = 0; mm < NT; ++mm) {
      f32x4 kt;                                      // A operand: row = key element 16 tile + r, reduction = token 4 g + j
#pragma unroll
      for (int j = 0; j < 4; ++j) kt[j] = k_s[4 * g + j][d_wave + 16 * mm + r];
#pragma unroll
      for (int j = 0; j < 4; ++j) S[mm][j] *= G_last;
      tw_mma16(S[mm], kt, wb);
    }
  }
#pragma unroll
  for (int mm = 0; mm < NT; ++mm) {
    const int d0 = d_wave + 16 * mm + 4 * g;
    if (live && d0 < a.Dk) *reinterpret_cast<f32x4*>(S_mem + d0) = S[mm];
  }
}

// Chunks of 32 tokens in two launches (or of 16 in one)? Two launches start later but their chain is less than half as long;
// where workgroups queue, a sequence of a few tokens costs a whole chunk either way, one of 32 more than one of 16.
// Measured, one launch / two, us:                 one portion of 49    64          80          96          128
//   16 heads of 128 (128 workgroups of the chain)   22.5 / 21.3   23.0 / 21.1   27.4 / 23.4   31.7 / 24.6   41.4 / 28.1
//   32 heads of 128 (256)                           21.5 / 24.0   22.1 / 25.0   26.7 / 29.4   31.2 / 28.9   40.1 / 31.8
//   16 heads of 256 (256)                           25.7 / 30.8   26.4 / 31.4   31.6 / 35.9   37.1 / 37.8   47.9 / 39.7
//   32 heads of 256 (512)                           34.5 / 44.1   35.9 / 42.8   43.6 / 48.4   50.5 / 49.7   64.6 / 54.3
// 60 portions of 5 and one of 64: 16 heads of 128 119 / 111, 32 heads 215 / 222, 16 heads of 256 269 / 421; 30 of 17 and one of
// 64: 108 / 66, 196 / 118, 250 / 208; 30 of 40 and one of 64: 148 / 107, 279 / 203, 363 / 374; 16 of 60: 97 / 69, 188 / 119,
// 243 / 196.
static bool delta_in_chunks(int rows, int n_seqs, int max_q_len, int H, int E, int Dk) {
  const long groups = (long)n_seqs * H * tw_div_up(E, 16);
  return max_q_len > (groups > 128 && groups <= 512 ? 88 : 48) && rows >= (Dk <= 128 ? 8L : 48L) * n_seqs;
}

// Chunks of 32: the scratch of a chunk of one head, and how many rows a pair of launches takes. A step's rows go through in
// pieces (a sequence's state passes from one to the next through its memory, as from step to step), so that the scratch stays
// below 512 MB unless 512 rows and the sequences alone need more: 9,200 rows of 16 heads of 128, 3,200 of 32 heads of 256, whose
// 8,192 rows take 1.4 GB at once. What pieces cost is the sequences that wait for the ones before them: one of 8,192 or 16,384
// tokens is as fast either way (32 heads of 256 2.7 and 2.8 ms, 5.4 and 5.6), four of 4,096 lose at 16 heads of 128
// (734 us in one piece, 933 in two, 1,138 in four), less at 32 heads of 256 (5.4 and 5.6 ms), so pieces are no smaller than they
// have to be.
static long delta_unit_floats(int E, int Dk) {
  const long DP = Dk <= 64 ? 64 : Dk <= 128 ? 128 : 256;
  return TW_DELTA_PREP * (3 * DP + 2L * tw_div_up(E, 16) * 16) + 4;
}
static int delta_piece_rows(int rows, int n_seqs, int H, int E, int Dk) {
  long chunks = (128L << 20) / (delta_unit_floats(E, Dk) * H) - n_seqs;
  if (chunks < 16) chunks = 16;
  return chunks * TW_DELTA_PREP < rows ? (int)chunks * TW_DELTA_PREP : rows;
}

// float32 scratch of a launch over n_seqs sequences of up to `rows` rows together (0: it needs none)
extern "C" long tw_delta_workspace_floats(int rows, int n_seqs, int max_q_len, int H, int E, int Dk) {
  if (n_seqs <= 0 || rows <= 0 || H <= 0 || E <= 0 || Dk <= 0 || !delta_in_chunks(rows, n_seqs, max_q_len, H, E, Dk)) return 0;
  return ((long)delta_piece_rows(rows, n_seqs, H, E, Dk) / TW_DELTA_PREP + n_seqs) * H * delta_unit_floats(E, Dk);
}

template <int NT>
static int delta_chunks(DeltaArgs a, int seq0, int n_seqs, int rows, float* workspace, hipStream_t stream) {
  const int piece = delta_piece_rows(rows, n_seqs, a.H, a.E, a.Dk);
  const size_t chunks = (size_t)piece / TW_DELTA_PREP + n_seqs, units = chunks * a.H;
  const size_t keys = units * TW_DELTA_PREP * 64 * NT, values = units * TW_DELTA_PREP * 16 * tw_div_up(a.E, 16);
  DeltaPrepared p;
  p.W = workspace;
  p.Q = p.W + keys;
  p.K = p.Q + keys;
  p.U = p.K + keys;
  p.O = p.U + values;
  p.G = p.O + values;
  for (a.row0 = 0; a.row0 < rows; a.row0 += piece) {
    a.row1 = min(rows, a.row0 + piece);
    delta_prepare_kernel<NT><<<dim3((unsigned)chunks, a.H), 256, 0, stream>>>(a, p, seq0, n_seqs);
    delta_chunk_kernel<NT><<<dim3(a.H * tw_div_up(a.E, 16), n_seqs), 256, 0, stream>>>(a, p, seq0);
  }
  return TW_LAUNCH_RESULT();
}

extern "C" int tw_delta_rule(const float* qkv, long ld_qkv, int q_col, int k_col, int v_col, const float* ab, long ld_ab,
                             int b_col, int a_col, const float* A_log, const float* dt_bias, float* state,
                             const int* q_start, const int* state_slots, float* out, long ld_out, int seq0, int n_seqs,
                             int max_q_len, int H, int G, int D, int E, int Dk, float q_scale, int rows, float* workspace,
                             long workspace_floats, hipStream_t stream) {
  TW_REQUIRE(qkv && ab && A_log && dt_bias && state && q_start && state_slots && out);
  TW_REQUIRE(H > 0 && G > 0 && H % G == 0 && D > 0 && D <= 256 && E > 0 && Dk >= D && Dk % 4 == 0 && Dk <= 256);
  TW_REQUIRE(max_q_len >= 1);
  TW_REQUIRE(seq0 >= 0 && n_seqs >= 0 && ld_out >= (long)H * E && (uintptr_t)state % 16 == 0);
  TW_REQUIRE(q_col >= 0 && k_col >= 0 && v_col >= 0 && b_col >= 0 && a_col >= 0);
  TW_REQUIRE(ld_qkv >= (long)max(q_col, k_col) + (long)G * D && ld_qkv >= (long)v_col + (long)H * E);
  TW_REQUIRE(ld_ab >= (long)max(a_col, b_col) + H);
  if (n_seqs == 0) return 0;
  DeltaArgs a{qkv, ld_qkv, q_col, k_col, v_col, ab, ld_ab, b_col, a_col, A_log, dt_bias, state, q_start, state_slots,
              out, ld_out, H, G, D, E, Dk, q_scale, 0, 0};
  if (rows > 0 && H <= 65535 && delta_in_chunks(rows, n_seqs, max_q_len, H, E, Dk)) {
    TW_REQUIRE(workspace != nullptr && (uintptr_t)workspace % 16 == 0 &&
               workspace_floats >= tw_delta_workspace_floats(rows, n_seqs, max_q_len, H, E, Dk));
    if (Dk <= 64) return delta_chunks<1>(a, seq0, n_seqs, rows, workspace, stream);
    if (Dk <= 128) return delta_chunks<2>(a, seq0, n_seqs, rows, workspace, stream);
    return delta_chunks<4>(a, seq0, n_seqs, rows, workspace, stream);
  } else if (max_q_len > TW_DELTA_WALK_MOST) {
    const dim3 grid(H * tw_div_up(E, 16), n_seqs);
    if (Dk <= 64) delta_short_kernel<1><<<grid, 256, 0, stream>>>(a, seq0);
    else if (Dk <= 128) delta_short_kernel<2><<<grid, 256, 0, stream>>>(a, seq0);
    else delta_short_kernel<4><<<grid, 256, 0, stream>>>(a, seq0);
  } else if (Dk <= 16) {
    delta_walk_kernel<4, 4><<<dim3(H * tw_div_up(E, 64), n_seqs), 256, 0, stream>>>(a, seq0);
  } else {
    const dim3 grid(H * tw_div_up(E, 16), n_seqs);
    if (Dk <= 64) delta_walk_kernel<4, 16><<<grid, 256, 0, stream>>>(a, seq0);
    else if (Dk <= 128) delta_walk_kernel<8, 16><<<grid, 256, 0, stream>>>(a, seq0);
    else delta_walk_kernel<16, 16><<<grid, 256, 0, stream>>>(a, seq0);
  }
  return TW_LAUNCH_RESULT();
}

// out[n][h * E + e] = o[n][h * E + e] / sqrt(mean_e(o^2) + eps) * weight[e] * silu(gate[n][h * E + e]), rounded to the
// compute type: a unit norm per head with one weight vector shared by the heads, times a gate. One wave a (token, head), element by
// element: heads of whole groups of four are norm_gate_kernel's.
template <typename T>
__global__ __launch_bounds__(256) void head_norm_gate_kernel(const float* __restrict__ o, long ld_o, const float* __restrict__ gate,
                                                             long ld_g, const float* __restrict__ weight, T* __restrict__ out,
                                                             long ld_out, int n, int H, int E, float eps, int weight_stride,
                                                             int gate_kind) {
  const int unit = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (unit >= n * H) return;
  const int lane = threadIdx.x & 63;
  const int row = unit / H, head = unit % H;
  const float* src = o + (size_t)row * ld_o + (size_t)head * E;
  float ss = 0.f;
  for (int e = lane; e < E; e += 64) ss = __fmaf_rn(src[e], src[e], ss);
  ss = tw_wave_sum(ss);
  const float rinv = 1.f / sqrtf(ss / (float)E + eps);
  const float* g = gate + (size_t)row * ld_g + (size_t)head * E;
  T* dst = out + (size_t)row * ld_out + (size_t)head * E;
  for (int e = lane; e < E; e += 64) {
    const float z = g[e];
    const float sig = 1.f / (1.f + expf(-z));
    // weight_stride: 0 for one weight vector for all heads, E for one a head; gate_kind 0: SiLU of the gate, 1: its sigmoid
    dst[e] = tw_from_float<T>(src[e] * rinv * weight[(size_t)head * weight_stride + e] * (gate_kind == 1 ? sig : z * sig));
  }
}

extern "C" int tw_head_norm_gate(int dtype, const float* o, long ld_o, const float* gate, long ld_g, const float* weight,
                                 void* out, long ld_out, int n, int H, int E, float eps, int weight_per_head, int gate_kind,
                                 hipStream_t stream) {
  TW_REQUIRE(o && gate && weight && out && n >= 0 && H > 0 && E > 0 && eps > 0.f && (gate_kind == 0 || gate_kind == 1));
  const int weight_stride = weight_per_head ? E : 0;
  TW_REQUIRE(ld_o >= (long)H * E && ld_g >= (long)H * E && ld_out >= (long)H * E);
  if (n == 0) return 0;
  const NormGateArgs a{o, ld_o, gate, ld_g, weight, out, ld_out, n, H, E, E, weight_stride, eps, 1.f};
  auto fast = [&](auto t) {
    typedef decltype(t) T;
    return gate_kind == 1 ? norm_gate_launch<T, float, TW_GATE_SIGMOID_BEHIND>(a, stream) : norm_gate_launch<T, float, TW_GATE_SILU_BEHIND>(a, stream);
  };
  if (dtype == TW_DTYPE_BF16 ? fast(bf16_t{}) : dtype == TW_DTYPE_F32 && fast(float{})) return TW_LAUNCH_RESULT();
  const int blocks = tw_div_up((long)n * H, 4);
  if (dtype == TW_DTYPE_BF16)
    head_norm_gate_kernel<bf16_t><<<blocks, 256, 0, stream>>>(o, ld_o, gate, ld_g, weight, (bf16_t*)out, ld_out, n, H, E, eps, weight_stride, gate_kind);
  else if (dtype == TW_DTYPE_F32)
    head_norm_gate_kernel<float><<<blocks, 256, 0, stream>>>(o, ld_o, gate, ld_g, weight, (float*)out, ld_out, n, H, E, eps, weight_stride, gate_kind);
  else return TW_ERR_BAD_ARGUMENT;
  return TW_LAUNCH_RESULT();
}
