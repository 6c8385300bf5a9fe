// Rows normed in equal units (a head, a group of heads) and gated, for retention, the delta rule, the mLSTM and the linear states: rows whose
// units are whole groups of four aligned elements. (Other rows keep the kernels that go element by element.)
#pragma once
#include "tw_common.h"

// How the gate g meets a unit u: the unit times SiLU(g) or sigmoid(g) behind the norm, or SiLU(g) in front of it.
#define TW_GATE_SILU_BEHIND 0
#define TW_GATE_SIGMOID_BEHIND 1
#define TW_GATE_SILU_BEFORE 2

struct NormGateArgs {
  const float* y; long ld_y;
  const void* gate; long ld_g;         // the compute type or float
  const float* weight;                 // null: none
  void* out; long ld_out;              // the compute type
  int n, parts, size, pitch;           // units of `size` elements `pitch` apart, the places between them zero (weight and y lie alike)
  int weight_stride;                   // the weights of a unit behind those of the one before (0: one unit's for all)
  float eps, scale;                    // scale: behind everything
};

__device__ __forceinline__ float ng_half_wave_sum(float v) {    // over a lane's half of a wave, in every lane of it
  auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(b[0]) + __uint_as_float(b[1]);
  v += tw_dpp<TW_ROTATE_8>(v);
  v += tw_dpp<TW_ROTATE_4>(v);
  v += tw_dpp<TW_SWAP_2>(v);
  return v + tw_dpp<TW_SWAP_1>(v);
}

// THREADS threads a unit (half a wave, a wave, or the workgroup), PER groups of four elements a thread. A unit is a chain of one trip to memory
// and a reduction: y, gate and weight are all requested before the first is used, and stay in registers. Element by element, with weight and
// gate asked for behind the reduction, it was two or three trips.
// (us in a captured graph, before / now: 8 rows of 8 heads of 256 3.3 / 2.4; 4 rows of 8 groups of 512 4.5 / 2.8; 4 rows
// of 2,048 12.2 and 4.7 / 3.0; 2,048 rows of 16 heads of 128 13.1 / 9.3, 3,000 of 2,048 15.0 / 12.0. With a whole wave a unit of 128 half the
// lanes had nothing: 14.2. Many units of 516 to 768, of which a workgroup's threads have up to half too many: 8,192 of 640 element by element / a workgroup /
// a wave a unit 14.3 / 15.7 / 10.5, 32,768 42 / 48 / 31; of up to 512 units the workgroup's chain is the shorter one, 2.7 and a wave's 3.1.)
template <typename T, typename G, int THREADS, int PER, int KIND>
__global__ __launch_bounds__(256) void norm_gate_kernel(NormGateArgs a) {
  typedef G Gate4 __attribute__((ext_vector_type(4)));
  typedef T Out4 __attribute__((ext_vector_type(4)));
  __shared__ float lds[16];
  const long unit = (long)blockIdx.x * (256 / THREADS) + threadIdx.x / THREADS;
  if (unit >= (long)a.n * a.parts) return;                     // (half a wave, a whole one or a whole workgroup)
  const int lane = threadIdx.x % THREADS, row = (int)(unit / a.parts), part = (int)(unit % a.parts);
  const size_t at = (size_t)part * a.pitch;
  const float* y = a.y + (size_t)row * a.ld_y + at;
  const G* gate = (const G*)a.gate + (size_t)row * a.ld_g + at;
  const float* weight = a.weight ? a.weight + (size_t)part * a.weight_stride : nullptr;
  const int last = a.size / 4 - 1;
  f32x4 v[PER], w[PER], g[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int c = min(lane + i * THREADS, last) * 4;
    v[i] = *reinterpret_cast<const f32x4*>(y + c);
    const Gate4 q = *reinterpret_cast<const Gate4*>(gate + c);
    g[i] = f32x4{tw_to_float(q[0]), tw_to_float(q[1]), tw_to_float(q[2]), tw_to_float(q[3])};
    w[i] = weight ? *reinterpret_cast<const f32x4*>(weight + c) : f32x4{1.f, 1.f, 1.f, 1.f};
  }
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const bool mine = lane + i * THREADS <= last;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float sig = 1.f / (1.f + expf(-g[i][e]));
      const float f = KIND == TW_GATE_SIGMOID_BEHIND ? sig : g[i][e] * sig;
      if (KIND == TW_GATE_SILU_BEFORE) v[i][e] *= f;
      else g[i][e] = f;
      ss = mine ? __fmaf_rn(v[i][e], v[i][e], ss) : ss;      // (0 times an infinity read again would be a NaN)
    }
  }
  const float sum = THREADS == 32 ? ng_half_wave_sum(ss) : THREADS == 64 ? tw_wave_sum(ss) : tw_block_sum(ss, lds);
  const float rinv = 1.f / sqrtf(sum / (float)a.size + a.eps);
  T* out = (T*)a.out + (size_t)row * a.ld_out + at;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int c = (lane + i * THREADS) * 4;
    if (c >= a.size) continue;
    Out4 r;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float u = v[i][e] * rinv * w[i][e];
      r[e] = tw_from_float<T>(KIND == TW_GATE_SILU_BEFORE ? u * a.scale : u * (g[i][e] * a.scale));
    }
    *reinterpret_cast<Out4*>(out + c) = r;
  }
  for (int c = a.size + lane * 4; c < a.pitch; c += THREADS * 4) *reinterpret_cast<Out4*>(out + c) = Out4{};
}

// Runs the kernel above where it takes the operands; false (and nothing done) where it does not.
template <typename T, typename G, int KIND>
static bool norm_gate_launch(const NormGateArgs& a, hipStream_t stream) {
  if (a.size % 4 || a.pitch % 4 || a.ld_y % 4 || a.ld_g % 4 || a.ld_out % 4 || a.weight_stride % 4 || a.size > 2048 ||
      (((uintptr_t)a.y | (uintptr_t)a.weight) & 15) || ((uintptr_t)a.gate & (4 * sizeof(G) - 1)) || ((uintptr_t)a.out & (4 * sizeof(T) - 1))) return false;
  const long units = (long)a.n * a.parts;
  if (a.size <= 128) norm_gate_kernel<T, G, 32, 1, KIND><<<tw_div_up(units, 8), 256, 0, stream>>>(a);
  else if (a.size <= 256) norm_gate_kernel<T, G, 64, 1, KIND><<<tw_div_up(units, 4), 256, 0, stream>>>(a);
  else if (a.size <= 512) norm_gate_kernel<T, G, 64, 2, KIND><<<tw_div_up(units, 4), 256, 0, stream>>>(a);
  else if (a.size <= 768 && units >= 1024) norm_gate_kernel<T, G, 64, 3, KIND><<<tw_div_up(units, 4), 256, 0, stream>>>(a);
  else if (a.size <= 1024) norm_gate_kernel<T, G, 256, 1, KIND><<<(unsigned)units, 256, 0, stream>>>(a);
  else norm_gate_kernel<T, G, 256, 2, KIND><<<(unsigned)units, 256, 0, stream>>>(a);
  return true;
}
