// Writing a step's values into the cache's 8-token groups [NB, G, BS / 8, Dv, 8].
//
// A token contributes one element to each 16-byte entry of its group, so a workgroup per token would
// write every entry in eight parts from eight workgroups, on eight XCDs with an L2 each.  Here a
// thread takes 8 dimensions of `vrows` neighbouring rows (8; 1 for small steps, whose rows are mostly
// sequences of their own): 8 rows that fill one group are transposed in registers and leave as whole
// entries, at whichever of a thread's rows the group begins.  Where it begins is told by the slot of the
// first of the 8 rows, so the first group of a sequence that begins among them is written element by
// element, by two threads (its later groups leave whole), as are rows of a group that is not whole.
#pragma once

#include "../kernels/common.h"

namespace akap_stream {

template <typename T>
struct ValueGroups {
  const T* src;             // element of the step's first row, value head 0, dimension 0
  int stride;               // of the rows
  T* cache;
  const int64_t* slots;
  int64_t num_slots;
  int T_, G, Dv, BS, vrows;
  float eps;
  bool norm;                // each head's values divided by their root mean square
  const float* bias;        // [G Dv] added first, or null
  const T* bias_t;          // the same in the rows' type, or null
};

__host__ __device__ __forceinline__ int64_t value_group_threads(int T, int G, int Dv, int vrows) {
  return (int64_t)((T + vrows - 1) / vrows) * G * (Dv >> 3);
}

namespace vg {
__device__ __forceinline__ void ld8(const float* p, float (&v)[8]) {
  const float4 a = *(const float4*)p, b = *(const float4*)(p + 4);
  v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
  v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}
__device__ __forceinline__ void ld8(const akap::bf16* p, float (&v)[8]) {
  const akap::bf16x8 a = *(const akap::bf16x8*)p;
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = (float)a[i];
}
__device__ __forceinline__ void st8(float* p, const float (&v)[8]) {
  *(float4*)p = make_float4(v[0], v[1], v[2], v[3]);
  *(float4*)(p + 4) = make_float4(v[4], v[5], v[6], v[7]);
}
__device__ __forceinline__ void st8(akap::bf16* p, const float (&v)[8]) {
  akap::bf16x8 o;
#pragma unroll
  for (int i = 0; i < 8; ++i) o[i] = (akap::bf16)v[i];
  *(akap::bf16x8*)p = o;
}
}  // namespace vg

// `item` of value_group_threads(); with norm, Dv / 8 is a power of two up to 64 and the lanes of a
// head are neighbours (whole waves call this, items in lane order)
template <typename T>
__device__ __forceinline__ void write_values(const ValueGroups<T>& a, int64_t item) {
  const int lph = a.Dv >> 3, per = a.G * lph;
  const int t0 = (int)(item / per) * a.vrows;
  const bool live = t0 < a.T_;
  const int e = (int)(item % per), g = e / lph, c = (e - g * lph) * 8;
  const int n = live ? min(a.vrows, a.T_ - t0) : 0;
  const int64_t s0 = live ? a.slots[t0] : -1;
  // the 8 rows that fill the first group which begins at or after row t (its slot s)
  auto group = [&](int t, int64_t s, int& first) {
    first = t + (int)((8 - (s & 7)) & 7);
    const int64_t f = (s + 7) & ~(int64_t)7;
    bool whole = s >= 0 && first + 8 <= a.T_ && f + 7 < a.num_slots;
#pragma unroll
    for (int i = 0; i < 8; ++i)     // (all eight requested together)
      whole &= a.slots[min(first + i, a.T_ - 1)] == f + i;
    return whole;
  };
  float add[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (a.bias) vg::ld8(a.bias + g * a.Dv + c, add);
  if (a.bias_t) vg::ld8(a.bias_t + g * a.Dv + c, add);
  auto row = [&](int t, float (&v)[8]) {      // (every lane of a head, rows clamped)
    vg::ld8(a.src + (size_t)t * a.stride + g * a.Dv + c, v);
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] += add[k];
    if (a.norm) {
      float ss = 0.f;
#pragma unroll
      for (int k = 0; k < 8; ++k) ss += v[k] * v[k];
      for (int o = lph >> 1; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);
      const float inv = 1.0f / sqrtf(ss / (float)a.Dv + a.eps);
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] *= inv;
    }
  };
  auto dst = [&](int64_t slot) {
    return a.cache + (((size_t)(slot / a.BS * a.G + g) * (a.BS >> 3) + (slot % a.BS >> 3)) * a.Dv +
                      c) * 8 + (slot & 7);
  };
  if (a.vrows == 8) {
    if (!live) return;
    // the group that begins among my rows, and the one that began among the 8 before and may end here
    int mine, prev = 0;
    const bool whole = group(t0, s0, mine);
    const bool before = t0 > 0 && group(t0 - 8, a.slots[t0 - 8], prev);
    if (whole) {
      float v[8][8];
#pragma unroll
      for (int i = 0; i < 8; ++i) row(mine + i, v[i]);
      T* o = dst(a.slots[mine]);
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const float r[8] = {v[0][k], v[1][k], v[2][k], v[3][k], v[4][k], v[5][k], v[6][k], v[7][k]};
        vg::st8(o + k * 8, r);
      }
    }
    for (int t = t0; t < t0 + n; ++t) {       // what is in neither
      if ((whole && t >= mine) || (before && t >= prev && t < prev + 8)) continue;
      float v[8];
      row(t, v);
      const int64_t slot = a.slots[t];
      if (slot < 0 || slot >= a.num_slots) continue;
      T* o = dst(slot);
#pragma unroll
      for (int k = 0; k < 8; ++k) o[k * 8] = (T)v[k];
    }
    return;
  }
  float v[8];
  row(live ? t0 : 0, v);
  if (s0 < 0 || s0 >= a.num_slots) return;
  T* o = dst(s0);
#pragma unroll
  for (int k = 0; k < 8; ++k) o[k * 8] = (T)v[k];
}

}  // namespace akap_stream
