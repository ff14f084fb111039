// Latent attention of prompt chunks for wide latents (R = 512 dimensions, r rotated ones, bf16): 32
// tokens x 2 heads per workgroup of 8 waves in two roles, one of each on every SIMD.
//
// Waves 0-3 score: wave w holds one head's 32 queries (R + r dimensions, 144 registers) and takes the
// 32 keys w >> 1 of a 64-key step (S^T = K Q^T, a query is a lane column); the two waves of a head
// agree on the maximum through LDS and put their weights there as operands.  The cached rows arrive
// by LDS-DMA, a step and a half ahead.  Waves 4-7 multiply: wave w holds 128 of the R output dimensions
// of all 64 queries (128 registers) and takes its value fragments straight from the grouped copy, each
// read once per workgroup.  So the exponentials of one step run under the products of the step
// before, and no product is computed twice.  Two barriers per step.
//
// Bound by what a wave issues in order: a step's rows and groups are 138 KB, 2200 cycles of a CU's
// load path, its products 2176 cycles of a SIMD; the step takes about 3600, and a workgroup 5 us to
// start.  5 prompts of up to 2047 tokens (odd lengths), 16 heads: 296 us, 0.78 PFLOP/s; four waves on
// one head's 32 queries with every fragment from the caches took 650.  One wave per head's whole
// output (512 registers) spilled (1509 us); workgroups that take several units in turn lost more to
// their imbalance than they gained at their start (388); either role at a higher wave priority 350.
#include "../kernels/common.h"
#include "stream.h"

namespace akap_stream {

using akap::bf16;
using akap::bf16x4;
using akap::bf16x8;
using akap::f32x16;
using akap::u32x4;

namespace {

constexpr int kKeys = 64;
constexpr float kLog2e = 1.44269504088896f;
constexpr float kLowest = -3.402823466e38f;   // a running maximum over no keys
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

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

template <int NV, int NKR>
__global__ __launch_bounds__(512, 2) void latent_prefill_wide_kernel(LatentAttnParams p) {
  constexpr int R = 32 * NV, DK = R + 16 * NKR, KS = DK / 16, CH = DK / 8, ND = NV / 4;
  static_assert(CH % 16 == 8, "the row swizzle");
  constexpr int KI = CH / 8;                     // 1-KB pieces of 8 staged rows
  constexpr int kK = kKeys * DK * 2;             // bytes of a step's rows
  __shared__ __align__(16) unsigned char lds[2 * kK + 64 * kKeys * 2 + 3 * 64 * 4];
  bf16* kl0 = (bf16*)lds;
  bf16x8* ps = (bf16x8*)(lds + 2 * kK);          // weights [2 heads][4 operands of 16 keys][64]
  float* m_loc = (float*)(lds + 2 * kK + 64 * kKeys * 2);   // [2 key halves][64]
  float* alpha_s = m_loc + 2 * 64;               // [64]
  // units (32 tokens, longest first) are dealt over the XCDs, the head pairs of one side by side on
  // one XCD; every exit before the loop is the workgroup's
  const int hblocks = (p.H + 1) / 2, sub = p.tile_rows / 32;
  const int jx = (int)blockIdx.x >> 3, unit = jx / hblocks * 8 + ((int)blockIdx.x & 7);
  if (unit >= p.num_tiles * sub) return;
  const int tile = p.num_tiles - 1 - unit / sub, si = sub - 1 - unit % sub;
  const int b = __builtin_amdgcn_readfirstlane(p.tile_seq[tile]);
  if (b < 0 || b >= p.B) return;
  const int qs0 = p.q_start[b], qlen = p.q_start[b + 1] - qs0, kv = p.seq_lens[b];
  const int rend = min(p.tile_row[tile] + p.tile_rows, qlen), r0 = p.tile_row[tile] + 32 * si;
  if (r0 >= rend || kv < qlen) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, hf = lane >> 5, h0 = jx % hblocks * 2;
  const bool valid = r0 + r < rend;
  const int t = qs0 + (valid ? r0 + r : r0);
  const int ctx = kv - qlen;
  const int pos_last = ctx + min(r0 + 31, rend - 1);
  const int steps = pos_last / kKeys + 1, last_piece = pos_last >> 5;
  const __attribute__((address_space(4))) int* bt =
      (const __attribute__((address_space(4))) int*)(p.block_tables + (size_t)b * p.max_blocks);

  // the walk over 32-key pieces (pages are whole pieces), the page after the current one requested
  // ahead; past the last piece it stays there
  auto page_of = [&](int idx) {
    const int blk = idx < p.max_blocks ? bt[idx] : 0;
    return blk >= 0 && blk < p.NB ? blk : 0;
  };
  int piece = 0, page_idx = 0, page_row = 0, page = page_of(0), page_ahead = page_of(1);
  auto cache_row = [&]() -> size_t { return (size_t)(page * p.BS + page_row); };
  auto advance = [&]() {
    if (piece >= last_piece) return;
    ++piece;
    page_row += 32;
    if (page_row == p.BS) {
      page_row = 0;
      ++page_idx;
      page = page_ahead;
      page_ahead = page_of(page_idx + 1);
    }
  };

  if (w < 4) {
    const int head = w & 1, kb = w >> 1;
    // staged rows: 16-byte piece c of row k lies at c ^ ((k >> 1) & 7), which with the rows' stride of
    // an odd number of 128 bytes spreads 16 neighbouring rows over all banks
    int koff[KI];
#pragma unroll
    for (int i = 0; i < KI; ++i) {
      const int s = i * 64 + lane, k = 8 * w + s / CH;
      koff[i] = (s / CH) * DK + ((s % CH) ^ ((k >> 1) & 7)) * 8;
    }
    // wave w stages rows 8 w .. of both 32-key pieces of a step, 1 KB at a time
    const bf16* src[2];
    auto next = [&]() {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        src[u] = (const bf16*)p.cache + (cache_row() + 8 * w) * DK;
        advance();
      }
    };
    auto stage = [&](int buf, int from, int to) {
      bf16* dst = kl0 + buf * (kK / 2) + 8 * w * DK;
#pragma unroll
      for (int i = from; i < to; ++i)
        dma16(src[i / KI] + koff[i % KI], dst + i / KI * 32 * DK + i % KI * 512);
    };
    next();
    stage(0, 0, 2 * KI);
    // The queries pass through the second buffer, as rows like the keys': loaded as operands, 16
    // bytes of 32 rows at a time, they took 9000 cycles.
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int hu = min(h0 + u, p.H - 1);
      bf16* dst = kl0 + kK / 2 + (32 * u + 8 * w) * DK;
#pragma unroll
      for (int i = 0; i < KI; ++i) {
        const int s = i * 64 + lane, k = 8 * w + s / CH, c = (s % CH) ^ ((k >> 1) & 7);
        const int tq = qs0 + min(r0 + k, rend - 1);
        const bf16* src_q = c * 8 < R
            ? (const bf16*)p.q_lat + ((size_t)hu * p.T + tq) * R + c * 8
            : (const bf16*)p.q + (size_t)tq * p.q_stride + (size_t)hu * p.q_head + p.rot_off + c * 8 - R;
        dma16(src_q, dst + i * 512);
      }
    }
    next();
    bf16x8 qf[KS];
    const int pos = valid ? ctx + r0 + r : -1, pos_first = r0 + 31 < rend ? ctx + r0 : -1;
    const float sc2 = p.scale * kLog2e;
    float m_run = kLowest, l_run = 0.f, mx;
    f32x16 s;
    // a lane's fragments: four row addresses, the rest are immediate offsets
    const bf16* kp[4];
#pragma unroll
    for (int c = 0; c < 4; ++c)
      kp[c] = kl0 + (32 * kb + row_key(r)) * DK + ((2 * c + hf) ^ ((row_key(r) >> 1) & 7)) * 8;
    auto scores = [&](int st, bool ahead) {      // ahead: stages the step after st meanwhile
      const int at = (st & 1) * (kK / 2);
      // fragments are read kB ahead of their products, which form two chains (a product waits for
      // the one before it in a chain twice as long as it occupies the unit)
      constexpr int kB = 4;
      static_assert(KS % kB == 0 && kB % 2 == 0, "batches");
      f32x16 s2;
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = s2[i] = 0.f;
      bf16x8 kf[2][kB];
      auto read = [&](int g) {
#pragma unroll
        for (int i = 0; i < kB; ++i) {
          const int c = g * kB + i;
          kf[g & 1][i] = *(const bf16x8*)(kp[c & 3] + at + (c >> 2) * 64);
        }
      };
      read(0);
#pragma unroll
      for (int g = 0; g < KS / kB; ++g) {
        if (g + 1 < KS / kB) read(g + 1);
        if (ahead) {
          stage((st + 1) & 1, g * 2 * KI / (KS / kB), (g + 1) * 2 * KI / (KS / kB));
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < kB; i += 2) {
          s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[g & 1][i], qf[g * kB + i], s, 0, 0, 0);
          s2 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[g & 1][i + 1], qf[g * kB + i + 1], s2, 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] += s2[i];
      // register i: key 64 st + 32 kb + 16 (i >> 3) + 8 hf + (i & 7), column r
      const int first = st * kKeys + 32 * kb;
      if (first + 31 > pos_first) {
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (first + 16 * (i >> 3) + 8 * hf + (i & 7) > pos) s[i] = -INFINITY;
      }
      mx = s[0];
#pragma unroll
      for (int i = 1; i < 16; ++i) mx = fmaxf(mx, s[i]);
      mx = both_max(mx) * sc2;
      m_loc[kb * 64 + 32 * head + r] = mx;       // (both halves' lanes hold the same)
    };
    auto weights = [&]() {
      const float m_new = fmaxf(fmaxf(m_run, mx), m_loc[(kb ^ 1) * 64 + 32 * head + r]);
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
      float sum[2] = {0.f, 0.f};
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        bf16x8 pb;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float x = __builtin_amdgcn_exp2f(fmaf(s[8 * e + j], sc2, -m_new));
          sum[j & 1] += x;
          pb[j] = (bf16)x;
        }
        ps[(4 * head + 2 * kb + e) * 64 + lane] = pb;
      }
      l_run = l_run * alpha + (sum[0] + sum[1]);
      m_run = m_new;
      alpha_s[32 * head + r] = alpha;            // (as both key halves' waves do)
    };
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    {
      const bf16* ql = kl0 + kK / 2 + (32 * head + r) * DK;
#pragma unroll
      for (int c = 0; c < KS; ++c) qf[c] = *(const bf16x8*)(ql + ((2 * c + hf) ^ ((r >> 1) & 7)) * 8);
    }
    scores(0, false);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (steps > 1) {
      stage(1, 0, 2 * KI);
      next();
    }
    weights();
    for (int st = 0; st < steps; ++st) {
      // rows of step st + 1 have landed, weights are written
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      if (st + 1 < steps) scores(st + 1, true);
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      if (st + 1 < steps) {
        next();
        weights();
      }
    }
    l_run = both_sum(l_run);
    m_loc[kb * 64 + 32 * head + r] = l_run;
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    return;
  }

  const int c = w - 4, dv0 = 32 * ND * c;
  bf16x8 vf[4][ND];
  const unsigned voff = (unsigned)((hf * R + dv0 + r) * 8);
  auto values = [&](int f) {                     // operand f (16 keys) of the next step
    const bf16* src = (const bf16*)p.vgroups + ((cache_row() >> 3) + 2 * (f & 1)) * R * 8;
#pragma unroll
    for (int d = 0; d < ND; ++d) vf[f][d] = *(const bf16x8*)(src + voff + 32 * d * 8);
    if (f & 1) advance();
  };
#pragma unroll
  for (int f = 0; f < 4; ++f) values(f);
  f32x16 o[2][ND];
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[q][d][i] = 0.f;
  asm volatile("s_barrier" ::: "memory");
  asm volatile("s_barrier" ::: "memory");
  for (int st = 0; st < steps; ++st) {
    asm volatile("s_barrier" ::: "memory");
    bf16x8 pf[2][2];
    auto operands = [&](int half) {
#pragma unroll
      for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int q = 0; q < 2; ++q) pf[q][f] = ps[(4 * q + 2 * half + f) * 64 + lane];
    };
    operands(0);
    const float a0 = alpha_s[r], a1 = alpha_s[32 + r];
    if (__any(a0 != 1.f || a1 != 1.f)) {
#pragma unroll
      for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          o[0][d][i] *= a0;
          o[1][d][i] *= a1;
        }
    }
    auto product = [&](int f) {
#pragma unroll
      for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int q = 0; q < 2; ++q)
          o[q][d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[f][d], pf[q][f & 1], o[q][d], 0, 0, 0);
      values(f);
    };
    product(0);
    product(1);
    operands(1);
    // this step's weights are in registers
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    product(2);
    product(3);
  }
  asm volatile("s_barrier" ::: "memory");
  // a lane holds entries 32 d + 8 j + 4 hf + (0..3) of its token; the halves exchange, so that each
  // stores 8 neighbouring entries
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    if (h0 + q >= p.H) break;
    const float l = m_loc[32 * q + r] + m_loc[64 + 32 * q + r], inv = l > 0.f ? 1.f / l : 0.f;
    bf16* out = (bf16*)p.out + ((size_t)(h0 + q) * p.T + t) * R + dv0;
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
      for (int kp = 0; kp < 2; ++kp) {
        bf16x4 oa, ob;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          oa[i] = (bf16)(o[q][d][8 * kp + i] * inv);
          ob[i] = (bf16)(o[q][d][8 * kp + 4 + i] * inv);
        }
        const u32x2 a = __builtin_bit_cast(u32x2, oa), e = __builtin_bit_cast(u32x2, ob);
        const auto x0 = __builtin_amdgcn_permlane32_swap(a[0], e[0], false, false);
        const auto x1 = __builtin_amdgcn_permlane32_swap(a[1], e[1], false, false);
        const u32x4 v = {x0[0], x1[0], x0[1], x1[1]};
        if (valid) *(u32x4*)(out + 32 * d + 16 * kp + 8 * hf) = v;
      }
  }
}

}  // namespace

void launch_latent_prefill_wide(const LatentAttnParams& p, hipStream_t s) {
  const int units = p.num_tiles * (p.tile_rows / 32);
  latent_prefill_wide_kernel<16, 4><<<(units + 7) / 8 * 8 * ((p.H + 1) / 2), 512, 0, s>>>(p);
}

}  // namespace akap_stream
