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

// page of a slot and place in it, by a shift where the page is a power of two and by 32-bit division
// otherwise: the 64-bit one of a few slots was a third of a cache write's instructions
__device__ __forceinline__ void slot_at(int64_t slot, int64_t num_slots, int BS, size_t& page,
                                        int& off) {
  if (num_slots > 0x7fffffff) {
    page = (size_t)(slot / BS);
    off = (int)(slot - (int64_t)page * BS);
  } else if ((BS & (BS - 1)) == 0) {
    page = (uint32_t)slot >> (31 - __clz(BS));
    off = (uint32_t)slot & (BS - 1);
  } else {
    const uint32_t pg = (uint32_t)slot / (uint32_t)BS;
    page = pg;
    off = (int)((uint32_t)slot - pg * BS);
  }
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
__device__ __forceinline__ void write_values(const ValueGroups<T>& a, uint32_t item) {
  typedef T Piece __attribute__((ext_vector_type(8)));
  const uint32_t lph = a.Dv >> 3, per = a.G * lph, block = item / per;
  const uint32_t e = item - block * per, g = e / lph, c = (e - g * lph) * 8;
  const int t0 = (int)block * a.vrows;
  const bool live = t0 < a.T_;
  const T* src = a.src + g * a.Dv + c;
  float add[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (a.bias) vg::ld8(a.bias + g * a.Dv + c, add);
  if (a.bias_t) vg::ld8(a.bias_t + g * a.Dv + c, add);
  auto load = [&](int t) { return *(const Piece*)(src + (size_t)t * a.stride); };
  auto row = [&](const Piece& x, float (&v)[8]) {      // (every lane of a head)
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = (float)x[k] + add[k];
    if (a.norm) {
      float ss = 0.f;
#pragma unroll
      for (int k = 0; k < 8; ++k) ss += v[k] * v[k];
      for (int o = (int)lph >> 1; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);
      const float inv = 1.0f / sqrtf(ss / (float)a.Dv + a.eps);
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] *= inv;
    }
  };
  auto dst = [&](int64_t slot) {
    size_t page;
    int off;
    slot_at(slot, a.num_slots, a.BS, page, off);
    return a.cache + (((page * a.G + g) * (a.BS >> 3) + (off >> 3)) * a.Dv + c) * 8 + (off & 7);
  };
  auto single = [&](int t, int64_t slot) {
    float v[8];
    row(load(t), v);
    if (slot < 0 || slot >= a.num_slots) return;
    T* o = dst(slot);
#pragma unroll
    for (int k = 0; k < 8; ++k) o[k * 8] = (T)v[k];
  };
  if (a.vrows != 8) {
    single(live ? t0 : 0, live ? a.slots[t0] : -1);
    return;
  }
  if (!live) return;
  // the group that begins among my rows (at the first multiple of 8 among the slots), and the one that
  // began among the 8 before and may end here; the rows' loads are under way before either is known to
  // be whole
  const int n = min(8, a.T_ - t0), tb = max(t0 - 8, 0);
  const int64_t s0 = a.slots[t0], sb = a.slots[tb];
  const int mine = t0 + (int)((8 - (s0 & 7)) & 7), prev = tb + (int)((8 - (sb & 7)) & 7);
  const int64_t fm = (s0 + 7) & ~(int64_t)7, fp = (sb + 7) & ~(int64_t)7;
  Piece x[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) x[i] = load(min(mine + i, a.T_ - 1));
  bool whole = s0 >= 0 && mine + 8 <= a.T_ && fm + 7 < a.num_slots;
  bool before = t0 > 0 && sb >= 0 && prev + 8 <= a.T_ && fp + 7 < a.num_slots;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    whole &= a.slots[min(mine + i, a.T_ - 1)] == fm + i;
    before &= a.slots[min(prev + i, a.T_ - 1)] == fp + i;
  }
  if (whole) {
    float v[8][8];
#pragma unroll
    for (int i = 0; i < 8; ++i) row(x[i], v[i]);
    T* o = dst(fm);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float r[8] = {v[0][k], v[1][k], v[2][k], v[3][k], v[4][k], v[5][k], v[6][k], v[7][k]};
      vg::st8(o + k * 8, r);
    }
  }
  for (int t = t0; t < t0 + n; ++t)           // what is in neither
    if (!(whole && t >= mine) && !(before && t >= prev && t < prev + 8)) single(t, a.slots[t]);
}

}  // namespace akap_stream
