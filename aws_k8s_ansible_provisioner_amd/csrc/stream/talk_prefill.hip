// Head-mixed attention of prompt chunks on the matrix cores, 128 queries of one query head against
// all value heads at a time (bf16 caches K [NB, G, BS, D], V [NB, G, BS / 8, Dv, 8], D = 64 or 128,
// pages of whole 32-token pieces), and the launch that mixes the heads and gates.
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

constexpr int kKeys = 64;              // keys per step
constexpr int kQ = 128;                // queries of a workgroup
constexpr float kLog2e = 1.44269504088896f;
constexpr float kLowest = -3.402823466e38f;   // a running maximum over no keys

__device__ __forceinline__ void dma16(const void* g, void* l) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)g,
                                   (__attribute__((address_space(3))) void*)l, 16, 0, 0);
}
__device__ __forceinline__ float both_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float both_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// key of row r of a 32-key tile: a lane's weights then are whole 8-key value groups
__device__ __forceinline__ int row_key(int r) {
  return 16 * (r >> 4) + 8 * ((r >> 2) & 1) + 4 * ((r >> 3) & 1) + (r & 3);
}
template <int D>
__device__ __forceinline__ int swz(int key, int c) {
  return D == 128 ? c ^ (key & 15) : c ^ ((key >> 1) & 7);
}

__device__ __forceinline__ int sequence_of(const int32_t* q_start, int B, int t) {
  int lo = 0, hi = B - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (q_start[mid] <= t) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// The sums of a 32-token block of the step in the workspace: [H][G Dv / 4][tokens of the block][4],
// so that a wave's lanes (a token each) store and read neighbouring 16-byte pieces.
__device__ __forceinline__ size_t ws_at(const TalkParams& p, int t, int g, int e4) {
  const int blk = t >> 5, nr = min(32, p.T - 32 * blk), GV = p.G * p.Dv;
  return (size_t)blk * 32 * p.H * GV + ((size_t)(g * (GV >> 2) + e4) * nr + (t & 31)) * 4;
}

// Eight waves; a step takes 64 keys.  Wave w scores the 32 queries w & 3 against the 32 keys w >> 2
// (S^T = K Q^T; a query is a lane column), agrees on the maximum with the wave of the other keys and
// puts its weights into LDS as operands; then every wave multiplies the weights of all 128 queries
// with ITS 32 TPW value entries (O^T = V^T P^T), whose fragments it takes straight from the cache: a
// value is read once per 128 queries.  Keys arrive in LDS by DMA, two steps ahead (three buffers).  The
// scores of step i + 1 are formed beside the first half of step i's products, its weights beside the
// second half.  The running maximum is exact, so the largest weight is 1 and not rounded.
//
// Bound by the chain of a step (score products, maximum, barrier, exponentials, barrier: half of the time
// alone) beside the products (116 us of the matrix units' time): 8 chunks of 1000 tokens behind 1000
// cached, 16 / 4 heads of 128 330 us; 64 queries per workgroup with every fragment from the caches
// took 919.  Opposite order of matrix and vector work in a SIMD's two waves gained nothing (24 us
// more).  The steps that all four query tiles see whole have a body of their own, without a branch per
// tile; with one body for all 352 us, and 290 for 4 chunks of 700 behind 300 of 32 / 8 heads, now 273.
template <int D, int TPW>
__global__ __launch_bounds__(512, 2) void talk_staged_kernel(TalkParams p, const int32_t* tile_seq,
                                                             const int32_t* tile_row, int num_tiles,
                                                             int tile_rows) {
  constexpr int KS = D / 16;
  constexpr int PW = kKeys * D * 2 / 1024 / 8;          // 1-KB pieces of the keys per wave
  constexpr int kK = kKeys * D * 2, kP = kQ * kKeys * 2;   // bytes of a buffer of keys, of weights
  __shared__ __align__(16) unsigned char lds[3 * kK + 2 * kP + 3 * kQ * 4];
  bf16* kl0 = (bf16*)lds;
  bf16x8* ps0 = (bf16x8*)(lds + 3 * kK);
  float* m_loc = (float*)(lds + 3 * kK + 2 * kP);       // [2][kQ]
  float* alpha_s = m_loc + 2 * kQ;                      // [kQ]

  // the heads of a tile run side by side on one XCD (they read the same values), longest tiles first
  const int subs = tile_rows / kQ, units = num_tiles * subs;
  const int per = (int)blockIdx.x >> 3, g = per % p.H;
  const int unit = units - 1 - (per / p.H * 8 + ((int)blockIdx.x & 7));
  if (unit < 0) return;
  const int tile = unit / subs;
  const int b = __builtin_amdgcn_readfirstlane(tile_seq[tile]);
  const int r_first = tile_row[tile] + kQ * (unit - tile * subs);
  const int q0 = p.q_start[b], chunk = p.q_start[b + 1] - q0;
  if (r_first >= chunk) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, hf = lane >> 5, qt = w & 3, kb = w >> 2;
  const int ctx = (int)p.positions[q0];
  const int last = ctx + min(r_first + kQ, chunk) - 1;  // last key that any query sees
  const int steps = last / kKeys + 1;
  auto last_of = [&](int q) { return ctx + min(r_first + 32 * q + 32, chunk) - 1; };   // of a query tile
  const int kvh = g / (p.H / p.G), BS = p.BS, G = p.G, Dv = p.Dv;
  const __attribute__((address_space(4))) int* bt =
      (const __attribute__((address_space(4))) int*)(p.block_tables + (size_t)b * p.max_blocks);
  const int last_piece = last >> 5;

  // a lane's element of the wave's first piece of a step's keys; the second's, 4 rows on, has another bit of
  // the turned column as well (formed in the loop: it lacks the register)
  static_assert(PW == 1 || (PW == 2 && D == 128), "pieces");
  const int koff = ((w * PW * 64 + lane) / (D / 8) & 31) * D +
                   swz<D>((w * PW * 64 + lane) / (D / 8), (w * PW * 64 + lane) % (D / 8)) * 8;
  // page and row in it of the 32-key piece a walk stands at; past the last piece it stays there
  struct Walk {
    int piece, idx, row;
  };
  auto advance = [&](Walk& c) {
    if (c.piece >= last_piece) return;
    ++c.piece;
    c.row += 32;
    if (c.row == BS) { c.row = 0; ++c.idx; }
  };
  Walk kw = {0, 0, 0}, vw = {0, 0, 0};
  if (w >> 2) advance(kw);
  auto stage = [&](int buf) {                            // the keys of the next step
    const bf16* kc = (const bf16*)p.k_cache +
                     (((size_t)bt[kw.idx] * G + kvh) * BS + kw.row) * D;
    bf16* kl = kl0 + buf * (kK / 2);
    int off = koff;
    asm volatile("" : "+v"(off));
    dma16(kc + off, kl + w * PW * 512);
    if (PW > 1) dma16(kc + ((off ^ 32) + 4 * D), kl + (w * PW + 1) * 512);
    advance(kw);
    advance(kw);
  };
  // value fragments of the next half step (32 keys); 8-key groups past the last key repeat the last
  const int NT = G * (Dv >> 5), DVT = Dv >> 5;
  const int ti0 = ((int)blockIdx.y * 8 + w) * TPW;
  bf16x8 vf[2][TPW][2];
  int cvk[TPW], dvk[TPW];
#pragma unroll
  for (int k = 0; k < TPW; ++k) {
    const int ti = min(ti0 + k, NT - 1);
    cvk[k] = ti / DVT;
    dvk[k] = (ti - cvk[k] * DVT) * 256;
  }
  auto values = [&](int half) {
    const size_t page = (size_t)bt[vw.idx] * G;
    const int lim = (last >> 3) - 4 * vw.piece;
    const unsigned off0 = (unsigned)((min(hf, lim) * Dv + r) * 8);
    const unsigned off1 = (unsigned)((min(2 + hf, lim) * Dv + r) * 8);
#pragma unroll
    for (int k = 0; k < TPW; ++k) {
      const bf16* vc = (const bf16*)p.v_cache +
                       ((page + cvk[k]) * (BS >> 3) + (vw.row >> 3)) * Dv * 8 + dvk[k];
      vf[half][k][0] = *(const bf16x8*)(vc + off0);
      vf[half][k][1] = *(const bf16x8*)(vc + off1);
    }
    advance(vw);
  };

  stage(0);
  stage(1);
  stage(2);
  bf16x8 qf[KS];
  const int tok = r_first + 32 * qt + r;
  {
    const bool valid = tok < chunk;
    const bf16* q = (const bf16*)p.q + ((size_t)(q0 + (valid ? tok : 0)) * p.H + g) * D + 8 * hf;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const bf16x8 z = {0, 0, 0, 0, 0, 0, 0, 0};
      const bf16x8 v = *(const bf16x8*)(q + 16 * s);
      qf[s] = valid ? v : z;
    }
  }
  const int limit = tok < chunk ? ctx + tok : -1;
  const int w_first = r_first + 32 * qt + 31 < chunk ? ctx + r_first + 32 * qt : -1;
  const float sc2 = p.scale * kLog2e;
  // (the maximum of the scores themselves: differences to it are exact however large they are)
  float m_run = kLowest, l_run = 0.f, mx = -INFINITY;
  f32x16 acc[TPW][4], s;
#pragma unroll
  for (int k = 0; k < TPW; ++k)
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[k][q][i] = 0.f;

  auto scores = [&](int buf) {
    const bf16* kl = kl0 + buf * (kK / 2);
    const int key = 32 * kb + row_key(r);
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.f;
#pragma unroll
    for (int c = 0; c < KS; ++c) {
      const bf16x8 kf = *(const bf16x8*)(kl + key * D + swz<D>(key, 2 * c + hf) * 8);
      s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[c], s, 0, 0, 0);
    }
  };
  auto maximum = [&](int t) {
    const int first = t * kKeys + 32 * kb;
    if (first + 31 > w_first) {
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (first + 16 * (i >> 3) + 8 * hf + (i & 7) > limit) s[i] = -INFINITY;
    }
    mx = s[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) mx = fmaxf(mx, s[i]);
    mx = both_max(mx);
    m_loc[kb * kQ + 32 * qt + r] = mx;      // (both halves' lanes hold the same)
  };
  auto weights = [&](int t) {
    const float m_new = fmaxf(fmaxf(m_run, mx), m_loc[(kb ^ 1) * kQ + 32 * qt + r]);
    const float alpha = __builtin_amdgcn_exp2f((m_run - m_new) * sc2);
    float sum[2] = {0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      s[i] = __builtin_amdgcn_exp2f((s[i] - m_new) * sc2);
      sum[i & 1] += s[i];
    }
    l_run = l_run * alpha + (sum[0] + sum[1]);
    m_run = m_new;
    bf16x8* ps = ps0 + (t & 1) * (kP / 16);
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      bf16x8 pb;
#pragma unroll
      for (int j = 0; j < 8; ++j) pb[j] = (bf16)s[8 * e + j];
      ps[(4 * qt + 2 * kb + e) * 64 + lane] = pb;
    }
    alpha_s[32 * qt + r] = alpha;           // (as both key halves' waves do)
  };
  auto products = [&](int t, int half, auto whole) __attribute__((always_inline)) {
    const bf16x8* ps = ps0 + (t & 1) * (kP / 16);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      // keys past a query tile's last take no part: a weight of 0 would not hide a value that is not
      // finite
      if (!whole() && t * kKeys + 32 * half > last_of(q)) continue;
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const bf16x8 pf = ps[(4 * q + 2 * half + e) * 64 + lane];
#pragma unroll
        for (int k = 0; k < TPW; ++k)
          acc[k][q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[half][k][e], pf, acc[k][q], 0, 0, 0);
      }
    }
  };

  values(0);
  asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  scores(0);
  maximum(0);
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  weights(0);
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  int t = 0, b1 = 1, b0 = 0;
  auto step = [&](auto whole) __attribute__((always_inline)) {
    {
      float a[4];
      bool moved = false;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        a[q] = alpha_s[32 * q + r];
        moved |= a[q] != 1.0f;
      }
      if (__any(moved)) {
#pragma unroll
        for (int k = 0; k < TPW; ++k)
#pragma unroll
          for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[k][q][i] *= a[q];
      }
    }
    const bool ahead = whole() || t + 1 < steps;
    if (ahead) scores(b1);
    // (beside DMA in flight the compiler waits for every load where it needs one: the first half's values
    // arrive here, and only then the second half's are asked for, which have the first products' time)
#pragma unroll
    for (int k = 0; k < TPW; ++k) asm volatile("" : "+v"(vf[0][k][0]), "+v"(vf[0][k][1]));
    values(1);
    __builtin_amdgcn_sched_barrier(0);
    products(t, 0, whole);
    if (ahead) maximum(t + 1);
    // the keys of step t + 2 have landed, those of step t were last read before the barrier before
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (ahead) {
      values(0);
      stage(b0);
      weights(t + 1);
    }
    products(t, 1, whole);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    b0 = b0 == 2 ? 0 : b0 + 1;
    b1 = b1 == 2 ? 0 : b1 + 1;
  };
  // (whole: step t's second half starts no later than the first query tile's last key; that may be key 31)
  const int all = min(steps - 1, (last_of(0) + 32) / kKeys);
  for (; t < all; ++t) step(std::true_type{});
  for (; t < steps; ++t) step(std::false_type{});
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // (nothing may land after the end)
  // both key halves' sums; the normalised sums of the wave's value entries
  l_run = both_sum(l_run);
  if (hf == 0) m_loc[kb * kQ + 32 * qt + r] = l_run;
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int tq = r_first + 32 * q + r;
    if (tq >= chunk) continue;
    const float inv = 1.0f / (m_loc[32 * q + r] + m_loc[kQ + 32 * q + r]);
#pragma unroll
    for (int k = 0; k < TPW; ++k)
      if (ti0 + k < NT) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          *(float4*)(p.ws_o + ws_at(p, q0 + tq, g, 8 * (ti0 + k) + 2 * j + hf)) =
              make_float4(acc[k][q][4 * j] * inv, acc[k][q][4 * j + 1] * inv,
                          acc[k][q][4 * j + 2] * inv, acc[k][q][4 * j + 3] * inv);
      }
  }
}

// out = talk x the heads' normalised sums, times the gate.  A lane takes 4 value entries of a token,
// all heads' sums of them in flight together, past the caches: they are read once, and lines that the
// attention just wrote need not make room for them.  Bound by reading the sums: 60 us for 7300 rows of
// 16 x 512 fp32 (240 MB), their gates and outputs, 81 us for 2500 rows of 32 x 1024 (328 MB); through the
// caches 67 and 109.  No branch, coefficient or gate stands between a head's loads: with one of each per
// head 91 and 142 us, and 10.1 for 6.6 where the step is 200 rows.
template <int HM>
__global__ __launch_bounds__(256) void talk_mix_kernel(TalkParams p) {
  const int t = ((p.row0 >> 5) + blockIdx.x) * 32 + (threadIdx.x & 31);
  const int e4 = blockIdx.y * 8 + (threadIdx.x >> 5), GV = p.G * p.Dv;
  if (e4 * 4 >= GV || t < p.row0 || t >= p.T) return;
  const int c = __builtin_amdgcn_readfirstlane(e4 * 4 / p.Dv);   // (a wave's: Dv is whole 32s)
  const int dv = e4 * 4 - c * p.Dv, rep = p.H / p.G;
  f32x4 o[HM];
#pragma unroll
  for (int g = 0; g < HM; ++g)
    o[g] = akap::ld_nt((const f32x4*)(p.ws_o + ws_at(p, t, min(g, p.H - 1), e4)));
  const bool wide = ((p.gate_stride & 3) | ((uintptr_t)p.gate & 7) | (p.out_stride & 3) |
                     ((uintptr_t)p.out & 7)) == 0;
  const __attribute__((address_space(4))) float* talk =
      (const __attribute__((address_space(4))) float*)p.talk;
  bf16x4 next = {};
  auto gates = [&](int i) __attribute__((always_inline)) {
    if (!p.gate || i >= rep) return;
    const bf16* gp = (const bf16*)p.gate + (size_t)t * p.gate_stride + (c * rep + i) * p.Dv + dv;
    if (wide) {
      next = *(const bf16x4*)gp;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) next[e] = gp[e];
    }
  };
  gates(0);
  if (p.seq_lens[sequence_of(p.q_start, p.B, t)] <= 0) return;
#pragma unroll
  for (int g = 0; g < HM; ++g)
    if (g >= p.H) o[g] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int i = 0; i < rep; ++i) {
    const int h = c * rep + i;
    const bf16x4 z = next;
    gates(i + 1);                         // (asked for before the stores that it could alias)
    float v[4] = {0.f, 0.f, 0.f, 0.f};
    if (p.talk) {
      float f[HM];
#pragma unroll
      for (int g = 0; g < HM; ++g) f[g] = talk[(size_t)h * p.H + min(g, p.H - 1)];
#pragma unroll
      for (int g = 0; g < HM; ++g) {
        const float fg = g < p.H ? f[g] : 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = fmaf(fg, o[g][e], v[e]);
      }
    } else {
#pragma unroll
      for (int g = 0; g < HM; ++g)
        if (g == h) {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] += o[g][e];
        }
    }
    if (p.gate) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] *= 1.0f / (1.0f + __expf(-(float)z[e]));
    }
    bf16* at = (bf16*)p.out + (size_t)t * p.out_stride + h * p.Dv + dv;
    const bf16x4 ob = {(bf16)v[0], (bf16)v[1], (bf16)v[2], (bf16)v[3]};
    if (wide) {
      *(bf16x4*)at = ob;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) at[e] = ob[e];
    }
  }
}

}  // namespace

bool launch_talk_staged(const TalkParams& p, const int32_t* tile_seq, const int32_t* tile_row,
                        int num_tiles, int tile_rows, hipStream_t s) {
  if ((p.D != 64 && p.D != 128) || p.Dv % 32 || p.BS % 32 || tile_rows % kQ || !(p.scale > 0.f) ||
      p.H > 32 || ((uintptr_t)p.ws_o & 15))
    return false;
  const int NT = p.G * (p.Dv / 32), units = num_tiles * (tile_rows / kQ);
  if (units > 0) {
    // 8 value tiles of 32 per grid row with one per wave, 16 with two
    const int tpw = NT <= 8 ? 1 : 2;
    const dim3 grid((units + 7) / 8 * 8 * p.H, (NT + 8 * tpw - 1) / (8 * tpw));
#define AKAP_TS(DD, TP) \
  talk_staged_kernel<DD, TP><<<grid, 512, 0, s>>>(p, tile_seq, tile_row, num_tiles, tile_rows)
    if (p.D == 64) {
      if (tpw == 1) AKAP_TS(64, 1); else AKAP_TS(64, 2);
    } else {
      if (tpw == 1) AKAP_TS(128, 1); else AKAP_TS(128, 2);
    }
#undef AKAP_TS
  }
  if (p.T > p.row0) {
    const dim3 grid((p.T + 31) / 32 - (p.row0 >> 5), (p.G * p.Dv / 4 + 7) / 8);
    if (p.H <= 8) talk_mix_kernel<8><<<grid, 256, 0, s>>>(p);
    else if (p.H <= 16) talk_mix_kernel<16><<<grid, 256, 0, s>>>(p);
    else talk_mix_kernel<32><<<grid, 256, 0, s>>>(p);
  }
  return true;
}

}  // namespace akap_stream
