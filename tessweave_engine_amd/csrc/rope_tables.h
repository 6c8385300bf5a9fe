// Rotary tables: cos/sin[t, j] of angle = float(position[t]) * inv_freq[j], times `magnitude`, for the kernel that forms one table and for
// those that form a step's tables beside something else that a step begins with.
#pragma once
#include "tw_common.h"

// (1 for the plain encoding; encodings that stretch their frequencies for longer contexts also scale both tables)
// rest (or null): what float32 rounded off the frequencies; the angle then carries the product's rounding error and this
// one beside it (at position 1,000 a float32 product alone is off by up to 3e-5).
struct RopeTable {
  const float *inv_freq, *rest;
  float *cos_out, *sin_out;
  int half;
  float magnitude;
};

__device__ __forceinline__ void tw_rope_entry(const RopeTable& a, const int* __restrict__ positions, int i) {
  const int t = i / a.half, j = i % a.half;
  const float p = (float)positions[t], f = a.inv_freq[j];
  const float angle = __fmul_rn(p, f);
  float c = cosf(angle), s = sinf(angle);
  if (a.rest) {
    const float off = __fmaf_rn(p, a.rest[j], __fmaf_rn(p, f, -angle));      // (a few hundredths at most)
    const float off2 = off * off;
    const float so = off * __fmaf_rn(-off2, 1.f / 6.f, 1.f), co = -0.5f * off2;
    const float sine = __fmaf_rn(so, c, __fmaf_rn(co, s, s));
    c = __fmaf_rn(-so, s, __fmaf_rn(co, c, c));
    s = sine;
  }
  a.cos_out[i] = c * a.magnitude;
  a.sin_out[i] = s * a.magnitude;
}

// Up to four tables of n tokens, entry after entry: workgroups of 256 threads, `block` of tw_rope_blocks. (Handed over by the caller as it lies here.)
#define TW_ROPE_TABLES 4
struct RopeTables {
  RopeTable table[TW_ROPE_TABLES];
  const int* positions;
  int count, n;
};
__device__ __forceinline__ void tw_rope_block(const RopeTables& a, int block) {
  int i = block * 256 + threadIdx.x;
#pragma unroll
  for (int k = 0; k < TW_ROPE_TABLES; ++k) {
    if (k >= a.count) return;
    const int entries = a.n * a.table[k].half;
    if (i < entries) return tw_rope_entry(a.table[k], a.positions, i);
    i -= entries;
  }
}
static inline int tw_rope_blocks(const RopeTables& a) {
  long entries = 0;
  for (int k = 0; k < a.count; ++k) entries += (long)a.n * a.table[k].half;
  return tw_div_up(entries, 256);
}
static inline bool tw_rope_tables_ok(const RopeTables& a, int n) {
  if (a.count < 0 || a.count > TW_ROPE_TABLES || (a.count > 0 && (!a.positions || a.n != n))) return false;
  for (int k = 0; k < a.count; ++k)
    if (!a.table[k].inv_freq || !a.table[k].cos_out || !a.table[k].sin_out || a.table[k].half <= 0) return false;
  return true;
}
