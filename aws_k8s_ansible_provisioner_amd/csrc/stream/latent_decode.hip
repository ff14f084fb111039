// Latent attention of decode rows on the matrix cores at R = 512, r = 64 (bf16): the heads of a token
// against a partition of its cached rows, each row read from memory ONCE.
//
// A cached row [c (R) | k_rot (r)] is both key and value.  The grouped copy of the latents exists
// because a value operand wants 8 keys of one dimension beside each other; read from it, a key costs
// 2176 bytes.  Here 8 NW rows at a time arrive in LDS by DMA, the next step's while this one's are
// computed, their 16-byte pieces turned by XOR, and the value operands are read out of the same rows with
// ds_read_b64_tr_b16: 16 lanes give 4 keys x 16 dimensions and receive 4 keys of one dimension each.
//
// Wave w of NW scores the keys 16 (w >> 1) .. of the step for the queries (heads) 16 (w & 1) .. (S^T =
// K Q^T, v_mfma_f32_16x16x32_bf16, the queries in registers), the waves of the same queries agree on the
// maximum, weights go to LDS; then every wave sums ITS part of the latent dimensions over all keys of the
// step (O^T = C^T P^T, v_mfma_f32_32x32x16_bf16).
//
// Bound by reading the rows: 32 us for 64 sequences of ~2010 keys (148 MB at 4.6 TB/s), 93 for 150 of ~2120
// under 32 heads (3.9), 108 for 200 of ~2250 (4.8); 39, 116 and 121 where a wait for the queries stood in
// the loop and every step asked whether it is masked; the kernel that read rows and groups took 51 for the
// first.  With eight waves and steps of 64 keys, as four waves' chain of barriers, fragment reads and
// exponentials takes longer per 32 keys (48 for 39 us, four slots ahead).  Grids that do not fit one
// workgroup to a CU run two of four waves there.
#include <type_traits>

#include "../kernels/common.h"
#include "stream.h"

namespace akap_stream {

using akap::bf16;
using akap::bf16x4;
using akap::bf16x8;
using akap::f32x16;
using akap::f32x4;

namespace {

constexpr int kR = 512, kRot = 64, kRowBytes = (kR + kRot) * 2;
constexpr int kBlk = 32;                          // keys that lie side by side in a page
constexpr int kDma = kBlk * kRowBytes / 1024 / 4; // 1-KB pieces per wave (four waves a block)
constexpr int kKs = (kR + kRot) / 32;             // contraction steps of a score

typedef short s16x4 __attribute__((ext_vector_type(4)));

// 16-byte piece c of row k lies at c ^ turn(k): the rows 0 .. 15 of a score operand and the 4 x 4 pieces
// of a value operand's 4 keys then fall on different banks (a row is 9 x 128 bytes)
__device__ __forceinline__ int turn(int k) {
  return ((k >> 1) & 1) * 4 + ((k >> 3) & 1) * 2 + ((k >> 2) & 1);
}
__device__ __forceinline__ float rows_max(float x) {      // over the four lanes l, l ^ 16, l ^ 32, l ^ 48
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float rows_sum(float x) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}
__device__ __forceinline__ void lds_barrier() {           // LDS alone: rows stay in flight
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// NW waves, steps of 8 NW keys
template <int NW>
__global__ __launch_bounds__(64 * NW, 2) void latent_decode_rows_kernel(LatentAttnParams p) {
  constexpr int kStep = 8 * NW, kSlot = kStep * kRowBytes, KQ = NW / 2, DT = 16 / NW;
  constexpr int kPp = kStep + 8;                          // pitch of the weights in LDS (elements)
  __shared__ __align__(16) unsigned char smem[2 * kSlot + 32 * kPp * 2 + (2 * KQ + 1) * 32 * 4];
  bf16* ps = (bf16*)(smem + 2 * kSlot);                   // [32 queries][kPp]
  float* mx_s = (float*)(smem + 2 * kSlot + 32 * kPp * 2);   // [key quarters][32]
  float* sum_s = mx_s + 32 * KQ;                          // [key quarters][32]
  float* alpha_s = sum_s + 32 * KQ;                       // [32]
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = blockIdx.x, part = blockIdx.z, c0 = blockIdx.y * 32;
  const int kv = p.seq_lens[b];
  if (kv <= 0) return;                                    // (the workgroup's) a padding row
  int per = (kv + p.num_parts - 1) / p.num_parts;
  per = (per + kBlk - 1) / kBlk * kBlk;
  const int jb = part * per, end = min(kv, jb + per);
  if (jb >= end) return;                                  // (the merge reads partitions with keys alone)
  const int steps = (end - jb + kStep - 1) / kStep, blocks = (end - jb + kBlk - 1) / kBlk;
  const int32_t* bt = p.block_tables + (size_t)b * p.max_blocks;

  // lane i holds the first row of block (batch of 64) + i; entries outside the table or the cache: page 0
  int rows = 0;
  auto look = [&](int n0) {
    const int j = jb + min(n0 + lane, blocks - 1) * kBlk, idx = j / p.BS;
    int page = idx < p.max_blocks ? bt[idx] : 0;
    if (page < 0 || page >= p.NB) page = 0;
    rows = page * p.BS + (j - idx * p.BS);
  };
  look(0);
  unsigned off[kDma];                                     // a lane's source bytes in the block's rows
#pragma unroll
  for (int i = 0; i < kDma; ++i) {
    const int s = ((w & 3) * kDma + i) * 64 + lane, row = s / (kRowBytes / 16), c = s % (kRowBytes / 16);
    off[i] = row * kRowBytes + (c ^ turn(row)) * 16;
  }
  auto stage = [&](int t) {
    const int n = t * (kStep / kBlk) + (w >> 2);
    if (n >= blocks) return;            // (what lies in the slot is masked like any key past the end)
    if (n >= 64 && (n & 63) < kStep / kBlk) look(n & ~63);
    const char* src = (const char*)p.cache +
                      (size_t)__builtin_amdgcn_readlane(rows, n & 63) * kRowBytes;
    unsigned char* dst = smem + (t & 1) * kSlot + w * kDma * 1024;
#pragma unroll
    for (int i = 0; i < kDma; ++i)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src + off[i]),
                                       (__attribute__((address_space(3))) void*)(dst + i * 1024), 16, 0, 0);
  };
  stage(0);
  // the wave's 16 queries, whole
  const int kq = w >> 1, qh = w & 1, n16 = lane & 15, g = lane >> 4;
  bf16x8 qf[kKs];
  {
    const int h = c0 + 16 * qh + n16 < p.H ? c0 + 16 * qh + n16 : c0;
    const bf16* ql = (const bf16*)p.q_lat + ((size_t)h * p.T + b) * kR + 8 * g;
    const bf16* qr = (const bf16*)p.q + (size_t)b * p.q_stride + (size_t)h * p.q_head + p.rot_off + 8 * g;
#pragma unroll
    for (int c = 0; c < kKs; ++c)
      qf[c] = *(const bf16x8*)(c < kR / 32 ? ql + 32 * c : qr + 32 * (c - kR / 32));
    // arrived here, once: a wait at the first product would stand in the loop, where it waits for the
    // rows of the next step as well
#pragma unroll
    for (int c = 0; c < kKs; ++c) asm volatile("" : "+v"(qf[c]));
  }
  const float sc2 = p.scale * 1.44269504088896f;
  float m = -INFINITY, l = 0.f;                           // of query 16 qh + n16; l: this lane's keys
  f32x16 o[DT];                                           // [dimensions 32 (DT w + dt)][query lane & 31]
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[dt][i] = 0.f;
  // byte offsets in a slot: score operand (row 16 kq + n16, piece 4 c + g), even c; value operand (key
  // 8 hf + jr of 16, dimensions 16 (g & 1) + 4 (lane & 3) of 32), first four keys, even tiles
  const int krow = 16 * kq + n16, hf = lane >> 5, jr = n16 >> 2;
  const unsigned ka = krow * kRowBytes + (g ^ turn(krow)) * 16;
  const unsigned va = (8 * hf + jr) * kRowBytes + w * DT * 64 +
                      ((2 * (g & 1) + ((lane & 3) >> 1)) ^ turn(8 * hf + jr)) * 16 + (lane & 1) * 8;

  // (masked: the last step, whose rows may lie past the partition's end; without the question the
  // others' reads of value operands run ahead of their products)
  auto step = [&](int t, auto masked) __attribute__((always_inline)) {
    // the step's rows have landed for this wave; every wave is through with the step before
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();
    if (t + 1 < steps) stage(t + 1);
    const unsigned char* slot = smem + (t & 1) * kSlot;
    const int j0 = jb + t * kStep;
    f32x4 s[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int c = 0; c < kKs; ++c) {
      const bf16x8 kf = *(const bf16x8*)(slot + (ka ^ (c & 1) * 64) + (c >> 1) * 128);
      s[c & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[c], s[c & 1], 0, 0, 0);
    }
    float sv[4], mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < 4; ++i) {                         // key j0 + 16 kq + 4 g + i
      sv[i] = s[0][i] + s[1][i];
      if (masked() && j0 + 16 * kq + 4 * g + i >= end) sv[i] = -INFINITY;
      mx = fmaxf(mx, sv[i]);
    }
    mx = rows_max(mx);
    if (g == 0) mx_s[kq * 32 + 16 * qh + n16] = mx;
    lds_barrier();
#pragma unroll
    for (int k = 0; k < KQ; ++k) mx = fmaxf(mx, mx_s[k * 32 + 16 * qh + n16]);
    const float mn = fmaxf(m, mx * sc2);
    const float ms = mn == -INFINITY ? 0.f : mn;          // nothing finite yet: every weight below is 0
    const float alpha = __builtin_amdgcn_exp2f(m - ms);
    m = mn;
    bf16x4 pb;
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float e = __builtin_amdgcn_exp2f(fmaf(sv[i], sc2, -ms));
      sum += e;
      pb[i] = (bf16)e;
    }
    l = l * alpha + sum;
    *(bf16x4*)(ps + (16 * qh + n16) * kPp + 16 * kq + 4 * g) = pb;
    if (kq == 0 && g == 0) alpha_s[16 * qh + n16] = alpha;
    lds_barrier();
    const float a = alpha_s[lane & 31];
    if (__any(a != 1.0f)) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[dt][i] *= a;
    }
#pragma unroll
    for (int sl = 0; sl < kStep / 16; ++sl) {
      const bf16x8 pf = *(const bf16x8*)(ps + (lane & 31) * kPp + 16 * sl + 8 * hf);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        bf16x8 vf;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const unsigned at = (va ^ (i * 16 + (dt & 1) * 64)) + (16 * sl + 4 * i) * kRowBytes + (dt >> 1) * 128;
          const s16x4 x = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (__attribute__((address_space(3))) s16x4*)(slot + at));
          const bf16x4 v = __builtin_bit_cast(bf16x4, x);
#pragma unroll
          for (int e = 0; e < 4; ++e) vf[4 * i + e] = v[e];
        }
        if (masked()) {    // what lies behind the partition's end may hold values that are not finite
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (j0 + 16 * sl + 8 * hf + e >= end) vf[e] = (bf16)0.f;
        }
        o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pf, o[dt], 0, 0, 0);
      }
    }
  };
  for (int t = 0; t + 1 < steps; ++t) step(t, std::false_type{});
  step(steps - 1, std::true_type{});
  l = rows_sum(l);
  if (g == 0) sum_s[kq * 32 + 16 * qh + n16] = l;
  lds_barrier();
  auto total = [&](int q) {
    float x = sum_s[q];
#pragma unroll
    for (int k = 1; k < KQ; ++k) x += sum_s[32 * k + q];
    return x;
  };
  // accumulator register i of o[dt]: dimension 32 (DT w + dt) + 8 (i >> 2) + 4 hf + (i & 3)
  const int h = c0 + (lane & 31), d0 = 32 * DT * w + 4 * hf;
  if (p.num_parts == 1) {
    if (h >= p.H) return;
    const float lq = total(lane & 31);
    const float f = lq > 0.f ? 1.0f / lq : 0.f;
    bf16* to = (bf16*)p.out + ((size_t)h * p.T + b) * kR + d0;
    const bool wide = ((uintptr_t)p.out & 7) == 0;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int i = 0; i < 16; i += 4) {
        const bf16x4 v = {(bf16)(o[dt][i] * f), (bf16)(o[dt][i + 1] * f), (bf16)(o[dt][i + 2] * f),
                          (bf16)(o[dt][i + 3] * f)};
        bf16* at = to + 32 * dt + 2 * i;
        if (wide) {
          *(bf16x4*)at = v;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) at[e] = v[e];
        }
      }
    return;
  }
  if (kq == 0 && g == 0 && c0 + 16 * qh + n16 < p.H) {
    const int q = 16 * qh + n16;
    float* ml = p.ws_ml + (((size_t)b * p.H + c0 + q) * p.num_parts + part) * 2;
    ml[0] = m;
    ml[1] = total(q);
  }
  if (h >= p.H) return;
  float* wo = p.ws_o + (((size_t)b * p.H + h) * p.num_parts + part) * kR + d0;
  const bool wide = ((uintptr_t)p.ws_o & 15) == 0;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 16; i += 4) {
      float* at = wo + 32 * dt + 2 * i;
      if (wide) {
        *(float4*)at = make_float4(o[dt][i], o[dt][i + 1], o[dt][i + 2], o[dt][i + 3]);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) at[e] = o[dt][i + e];
      }
    }
}

}  // namespace

void launch_latent_decode_rows(const LatentAttnParams& p, hipStream_t s) {
  const dim3 grid(p.B, (p.H + 31) / 32, p.num_parts);
  // one workgroup of eight waves per CU, or two of four where the grid is larger: eight waves' LDS would
  // have it run in rounds
  const int64_t wgs = (int64_t)grid.x * grid.y * grid.z;
  if (wgs <= 256) latent_decode_rows_kernel<8><<<grid, 512, 0, s>>>(p);
  else latent_decode_rows_kernel<4><<<grid, 256, 0, s>>>(p);
}

}  // namespace akap_stream
