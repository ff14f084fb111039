// Softmax attention of prompt chunks on the matrix cores with the keys and values staged through
// LDS (bf16 caches K [NB, G, BS, D], V [NB, G, BS / 8, D, 8], D = 64 or 128, pages of whole 32-token
// pieces): causal, with a lower bound of visible keys from chunks counted from position 0 and / or a
// window, pooled entries before the window, a sink in the softmax's denominator, a gate per head.
//
// Four waves, a team, take 4 units of (32 tokens, query head) of one key/value head: with 4 heads to a
// group the heads of 32 tokens; a workgroup is one team, or in small grids two that take the steps in turn
// and add up their sums at the end.  64 keys and values at a time arrive by LDS-DMA while the 64 before are
// computed (two buffers, one barrier per step); each staged byte feeds 4 waves, where fragments taken
// straight from the caches cost every wave its own loads.  Two workgroups of 4 waves on a CU instead of
// one of 8 stage twice the bytes, but one starts or ends under the other's steps and a tile's masked
// steps are fewer: 64 prompts of 256 tokens 81 -> 64 us, 8 of 2048 196 -> 187, the pooled prompts below
// 172 -> 165.  S^T = K Q^T and O^T = V^T P^T with v_mfma_f32_32x32x16_bf16: the key rows in the
// order that makes a lane's weights whole 8-key value groups, so they become the next operand
// without lane traffic.  The K rows are XOR-swizzled by the DMA's source address, the fragment
// reads are free of bank conflicts.
//
// The running maximum is exact and moves by 32 keys, so every weight that is the largest so far is 1
// and not rounded: letting it lag by up to 8 log2 units cost 1 to 7 % more error, one maximum per 64
// keys 0.25 % (and took 196 and 149 us).  It is a maximum over keys alone: a head's sink enters the
// finished sums in fp32 (as the start of the maximum, a sink above the scores would have every weight
// rounded: 1.1 to 1.4 times the error); only the sink of score 0 starts maximum and sum.
//
// Bound by what a SIMD can issue: per 64 keys and wave about 280 vector instructions at 2.4 to 4
// cycles, 32 exponentials at 8.5, 32 products that take 10 of issue each, 32 fragment reads at 8; two
// waves together 5000 cycles where their products alone are 2112.  A wave's products interleaved by hand
// with the weights of the step before, or the two halves of the waves in opposite phases between
// barriers, cost 5 to 15 % instead of gaining; without the rescaling of the sums 8 % less, without the
// exponentials 5 %.  8 x 2048 tokens, 16 / 4 heads of 128, causal: 187 us (0.73 PFLOP/s; fragments
// straight from the caches took 331), 5 prompts of up to 3001 tokens through a window of 1024 and pooled
// blocks of 64: 161 us (553).  Tried for the pooled form's small weights: the minimum of a step's scores and a branch to a full exponential 16 us
// more, the step's body twice 170 us more (spills); roots and squares cost 4.
#include <type_traits>

#include "../kernels/common.h"
#include "stream.h"

namespace akap_stream {

using akap::bf16;
using akap::bf16x4;
using akap::bf16x8;
using akap::f32x16;
using akap::u32x4;

namespace {

constexpr int kKeys = 64;              // keys per step
constexpr int NW = 4;                  // waves of a team
// Steps up to which one team takes them all: a prompt of 128 tokens of 16 / 4 heads, the layer, 15.0 us with
// 0, 14.3 with 4, 14.2 with 8; 64 behind 450 22.5, 22.8, 22.8 (24.2 with 16), 700 behind 300 34.6, 35.1, 35.3
// (39.4)
constexpr int kTeamSteps = 4;
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
// key of row r of a 32-key tile
__device__ __forceinline__ int row_key(int r) {
  return 16 * (r >> 4) + 8 * ((r >> 2) & 1) + 4 * ((r >> 3) & 1) + (r & 3);
}
// 16-byte piece of a staged key row that holds the row's piece c: 16 neighbouring rows of a fragment
// read fall on different banks (rows of 256 resp. 128 bytes)
template <int D>
__device__ __forceinline__ int swz(int key, int c) {
  return D == 128 ? c ^ (key & 15) : c ^ ((key >> 1) & 7);
}

// POOL: the pooled form (positions given, pooled entries before the window if there are any)
// TEAMS: of four waves, which take the steps in turn
template <int D, bool POOL, int TEAMS>
__global__ __launch_bounds__(64 * NW * TEAMS, 2) void flash_prefill_kernel(const FlashParams p) {
  constexpr int KS = D / 16, DT = D / 32;       // contraction steps of a score, tiles of an output
  constexpr int PIECES = kKeys * D * 2 / 1024;  // 1-KB pieces of the keys (and of the values)
  constexpr int PW = PIECES / NW;               // of a wave
  static_assert(PIECES % NW == 0 && PW >= 1, "pieces");
  constexpr int kBuf = 2 * kKeys * D;           // elements of a buffer: keys, values
  __shared__ __align__(16) bf16 lds_all[TEAMS * 2 * kBuf];
  const int rep = p.H / p.G;
  const int subs = p.tile_rows / 32;            // 32-token pieces of a tile
  const int parts = subs * rep / NW;
  // longest tiles first (the map is sorted by rising work); the workgroups of a tile side by side,
  // a head's on one XCD where the heads times parts divide among the eight
  const int flat = (int)gridDim.x - 1 - (int)blockIdx.x;
  const int tile = flat / (p.G * parts), rest = flat - tile * (p.G * parts);
  const int part = rest / p.G, g = rest - part * p.G;
  const int tid = threadIdx.x & (64 * NW - 1), lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);      // in its team
  const int team = TEAMS > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x / (64 * NW)) : 0;
  bf16* const lds = lds_all + team * 2 * kBuf;
  const int r = lane & 31, hf = lane >> 5;
  const int b = __builtin_amdgcn_readfirstlane(p.tile_seq[tile]);
  if (b < 0 || b >= p.B) return;                        // (the workgroup's exits, but for a team's below)
  const int q0 = p.q_start[b], q_len = p.q_start[b + 1] - q0;
  if (q_len <= 0) return;
  const int ctx = p.positions ? (int)p.positions[q0] : p.seq_lens[b] - q_len;
  if (ctx < 0 && !p.positions) return;                  // fewer keys than rows
  const int kv_len = ctx + q_len;
  const int item = part * NW + w, sub = item / rep, h = g * rep + item - sub * rep;
  const int tok0 = p.tile_row[tile] + 32 * sub;        // the wave's first token of the chunk
  const int tok = tok0 + r;
  const bool valid = tok < q_len, active = tok0 < q_len;
  const int pos = ctx + tok;
  auto lower = [&](int i) {
    int lo = p.chunk > 0 ? i / p.chunk * p.chunk : 0;
    if (p.window > 0) lo = max(lo, i - p.window + 1);
    return lo;
  };
  const int limit = valid ? pos : -1, lo_l = lower(pos);
  // the wave's and the workgroup's ranges
  const int w_first = ctx + tok0, w_last = ctx + min(tok0 + 31, q_len - 1);
  const int g_tok0 = p.tile_row[tile] + 32 * (part * NW / rep);
  const int g_tok1 = p.tile_row[tile] + 32 * ((part * NW + NW - 1) / rep) + 31;
  if (g_tok0 >= q_len) return;                          // (the whole workgroup)
  const int g_last = ctx + min(g_tok1, q_len - 1);
  const int key_first = lower(ctx + g_tok0) & ~31;      // staging starts at a 32-key piece
  const int w_lo0 = lower(w_first), w_lo1 = lower(w_last);
  const int steps = max((g_last - key_first) / kKeys + 1, 1);
  // teams at work: few steps are not worth the second's sums.  (Where one works the other's waves end here,
  // and the barriers count the waves that have not ended.)
  const int teams = TEAMS > 1 && steps > kTeamSteps ? 2 : 1;
  if (team >= teams) return;
  const int32_t* bt = p.block_tables + (size_t)b * p.max_blocks;
  const int BS = p.BS, G = p.G;
  const int last_piece = max(kv_len - 1, 0) >> 5;

  // staging of step t: a wave's pieces lie in one 32-key piece of it, so page and row are uniform
  int koff[PW], voff[PW];
#pragma unroll
  for (int i = 0; i < PW; ++i) {
    const int s = (w * PW + i) * 64 + lane, key = s / (D / 8), c = swz<D>(key, s % (D / 8));
    koff[i] = (key & 31) * D + c * 8;
    voff[i] = (s % (D * 4)) * 8;
  }
  auto piece_of = [&](int t) {
    return __builtin_amdgcn_readfirstlane(
        min((key_first >> 5) + t * 2 + (w * PW) / (PIECES / 2), last_piece));
  };
  const __attribute__((address_space(4))) int* btc = (const __attribute__((address_space(4))) int*)bt;
  auto page_of = [&](int t) {       // entries outside the cache or the table: page 0
    const int idx = piece_of(t) * 32 / BS, page = idx < p.max_blocks ? btc[idx] : 0;
    return page >= 0 && page < p.NB ? page : 0;
  };
  auto stage = [&](int t, int buf, int page) {
    bf16* kl = lds + buf * kBuf;
    bf16* vl = kl + kKeys * D;
    const size_t base = ((size_t)page * G + g) * BS * D + (size_t)(piece_of(t) * 32 % BS) * D;
    const bf16* kb = (const bf16*)p.k_cache + base;
    const bf16* vb = (const bf16*)p.v_cache + base;
#pragma unroll
    for (int i = 0; i < PW; ++i) dma16(kb + koff[i], kl + (w * PW + i) * 512);
#pragma unroll
    for (int i = 0; i < PW; ++i) dma16(vb + voff[i], vl + (w * PW + i) * 512);
  };
  stage(team, 0, page_of(team));
  int page_next = page_of(team + teams);

  bf16x8 qf[KS];
  {
    const bf16* q = (const bf16*)p.q + ((size_t)(q0 + (valid ? tok : 0)) * p.H + h) * D + 8 * hf;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const bf16x8 z = {0, 0, 0, 0, 0, 0, 0, 0};
      const bf16x8 v = *(const bf16x8*)(q + 16 * s);
      qf[s] = valid ? v : z;
    }
  }
  const float sc2 = p.scale * kLog2e;
  // The maximum in log2 units of the scaled scores; POOL: of the scores themselves, so that the
  // difference is exact however large they are, and a weight is the square of its root, as the
  // exponential gives nothing below 2^-126 where a bf16 holds weights down to 2^-133
  auto weight = [&](float below) {
    const float root = __builtin_amdgcn_exp2f(below * (0.5f * sc2));
    return root * root;
  };
  const bool unit = p.unit_sink && team == 0;
  float m_run = unit ? 0.f : kLowest;
  float l_run = unit && hf == 0 ? 1.f : 0.f;   // (a lane's own keys; the halves meet at the end)
  f32x16 o[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[d][i] = 0.f;

  // one step of 64 keys: scores against the staged keys, weights of those from lo to hi, a lane's own
  // (masked: not all of them; low: some are before lo).  Keys before klo or past khi are seen by no query of
  // the wave (later tokens, and what a page's last owner left behind the sequence's end); a weight of 0
  // would not hide values that are not finite, so their groups are read as the nearest that the wave sees,
  // and pooled entries, which every wave's queries see to another end, are cleared one by one.
  auto compute = [&](const bf16* kl, const bf16* vl, bool masked, int klo, int khi, auto pooled,
                     bool low, int lo, int hi) {
    f32x16 s[2];
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int i = 0; i < 16; ++i) s[k][i] = 0.f;
    bf16x8 kf[KS][2];
#pragma unroll
    for (int c = 0; c < KS; ++c)
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int key = 32 * k + row_key(r);
        kf[c][k] = *(const bf16x8*)(kl + key * D + swz<D>(key, 2 * c + hf) * 8);
      }
#pragma unroll
    for (int c = 0; c < KS; ++c)
#pragma unroll
      for (int k = 0; k < 2; ++k)
        s[k] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[c][k], qf[c], s[k], 0, 0, 0);
    // the value fragments are requested now: they arrive under the softmax
    bf16x8 vf[2][2][DT];
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int n = min(max(4 * k + 2 * e + hf, klo >> 3), khi >> 3);
#pragma unroll
        for (int d = 0; d < DT; ++d) vf[k][e][d] = *(const bf16x8*)(vl + (n * D + 32 * d + r) * 8);
      }
    // maximum, weights and products of 32 keys at a time
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      if (masked) {
        if (32 * k > khi || 32 * k + 31 < klo) continue;   // (no lane sees any of them)
        const int last = hi - 8 * hf, first = lo - 8 * hf;
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (32 * k + 16 * (i >> 3) + (i & 7) > last) s[k][i] = -INFINITY;
        if (low) {
#pragma unroll
          for (int i = 0; i < 16; ++i)
            if (32 * k + 16 * (i >> 3) + (i & 7) < first) s[k][i] = -INFINITY;
        }
      }
      float mx = -INFINITY;
#pragma unroll
      for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[k][i]);
      mx = both_max(mx);
      const float m_new = fmaxf(m_run, POOL ? mx : mx * sc2);
      float sum[2] = {0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float e = POOL ? weight(s[k][i] - m_new)
                             : __builtin_amdgcn_exp2f(fmaf(s[k][i], sc2, -m_new));
        s[k][i] = e;
        sum[i & 1] += e;
      }
      if (__any(m_new != m_run)) {
        const float alpha = POOL ? weight(m_run - m_new) : __builtin_amdgcn_exp2f(m_run - m_new);
        l_run *= alpha;
#pragma unroll
        for (int d = 0; d < DT; ++d)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[d][i] *= alpha;
      }
      m_run = m_new;
      l_run += sum[0] + sum[1];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        bf16x8 pb;
#pragma unroll
        for (int j = 0; j < 8; ++j) pb[j] = (bf16)s[k][8 * e + j];
        if (pooled() && masked) {
#pragma unroll
          for (int d = 0; d < DT; ++d)
#pragma unroll
            for (int j = 0; j < 8; ++j)
              if (32 * k + 16 * e + 8 * hf + j > khi) vf[k][e][d][j] = (bf16)0.f;
        }
#pragma unroll
        for (int d = 0; d < DT; ++d)
          o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[k][e][d], pb, o[d], 0, 0, 0);
      }
    }
  };

  if (POOL) {
    // pooled entries 0 .. nb - 1 (what the workgroup's last token sees), 64 at a time through the
    // second buffer: fp32 rows, rounded to bf16 operands on the way
    const int W = p.window, P = p.pool;
    auto before = [&](int i) { return P > 0 && i - W + 1 > 0 ? (i - W + 1) / P : 0; };
    const int nb = before(g_last), w_nb = before(w_last), w_all = before(w_first);
    const int mine = valid ? before(pos) : 0;          // (the wave's last and first token above)
    bf16* kl = lds + kBuf;
    bf16* vl = kl + kKeys * D;
    for (int ca = 0; ca < nb; ca += teams * kKeys) {
      const int c0 = ca + team * kKeys;
      constexpr int F4 = D / 4, NE = kKeys * F4 / (64 * NW);   // float4 pieces of a row, per thread
      float4 kk[NE], vv[NE];
#pragma unroll
      for (int u = 0; u < NE; ++u) {
        const int e = u * 64 * NW + tid, key = e / F4, d = (e % F4) * 4, c = min(c0 + key, nb - 1);
        const int page = bt[c * P / BS], idx = c * P % BS / P;
        const size_t at = ((size_t)(page * G + g) * p.PS + idx) * D + d;
        kk[u] = *(const float4*)(p.k_pool + at);
        vv[u] = *(const float4*)(p.v_pool + at);
        if (c0 + key >= nb) vv[u] = make_float4(0.f, 0.f, 0.f, 0.f);
      }
      if (ca > 0) __syncthreads();            // every wave has read the 64 before
#pragma unroll
      for (int u = 0; u < NE; ++u) {
        const int e = u * 64 * NW + tid, key = e / F4, d = (e % F4) * 4;
        const bf16x4 k4 = {(bf16)kk[u].x, (bf16)kk[u].y, (bf16)kk[u].z, (bf16)kk[u].w};
        *(bf16x4*)(kl + key * D + swz<D>(key, d >> 3) * 8 + (d & 7)) = k4;
        bf16* vp = vl + ((key >> 3) * D + d) * 8 + (key & 7);
        vp[0] = (bf16)vv[u].x; vp[8] = (bf16)vv[u].y;
        vp[16] = (bf16)vv[u].z; vp[24] = (bf16)vv[u].w;
      }
      __syncthreads();
      if (active && c0 < w_nb)
        compute(kl, vl, c0 + kKeys > w_all, 0, min(w_nb - 1 - c0, kKeys - 1), std::true_type{},
                false, 0, mine - 1 - c0);
    }
  }

  for (int u = 0; u * teams < steps; ++u) {
    const int t = u * teams + team;
    // step t has landed for this wave; every wave has read the buffer that step t + 1 goes to
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    if (t + teams < steps) {
      stage(t + teams, (u + 1) & 1, page_next);
      page_next = page_of(t + 2 * teams);
    }
    const int key0 = key_first + t * kKeys;
    if (t < steps && active && key0 <= w_last && key0 + kKeys > w_lo0) {
      const bf16* kl = lds + (u & 1) * kBuf;
      compute(kl, kl + kKeys * D, key0 + kKeys - 1 > w_first || key0 < w_lo1, max(w_lo0 - key0, 0),
              min(w_last - key0, kKeys - 1), std::false_type{}, key0 < w_lo1, lo_l - key0, limit - key0);
    }
  }

  l_run = both_sum(l_run);
  if (TEAMS > 1 && teams > 1) {
    // the second team's maxima and sums into the first's, through the buffers
    float* to = (float*)lds_all + w * (16 * DT + 2) * 64 + lane;
    __syncthreads();
    if (team == 1) {
      to[0] = m_run;
      to[64] = l_run;
#pragma unroll
      for (int d = 0; d < DT; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) to[(2 + 16 * d + i) * 64] = o[d][i];
    }
    __syncthreads();
    if (team == 1) return;
    const float m1 = to[0], m = fmaxf(m_run, m1);
    const float fa = POOL ? weight(m_run - m) : __builtin_amdgcn_exp2f(m_run - m);
    const float fb = POOL ? weight(m1 - m) : __builtin_amdgcn_exp2f(m1 - m);
    l_run = l_run * fa + to[64] * fb;
    m_run = m;
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[d][i] = o[d][i] * fa + to[(2 + 16 * d + i) * 64] * fb;
  }
  if (!active) return;
  float corr = 1.f;
  if (p.sink) {
    const float sk = p.sink[h], mk = m_run * 0.693147180559945f;   // back from log2 units
    const float m = fmaxf(mk, sk);
    corr = expf(mk - m);
    l_run = l_run * corr + expf(sk - m);
  }
  float inv = l_run > 0.f ? corr / l_run : 0.f;
  const int t_out = q0 + (valid ? tok : 0);
  if (p.gate) {
    const float z = (float)((const bf16*)p.gate)[(size_t)t_out * p.gate_stride + h];
    inv *= 1.0f / (1.0f + expf(-z));
  }
  // a lane holds entries 32 d + 8 j + 4 hf + (0..3) of its token; the halves exchange, so that each
  // stores 8 neighbouring entries
  bf16* out = (bf16*)p.out + (size_t)t_out * p.out_stride + (size_t)h * D;
  const bool wide = ((p.out_stride & 7) | ((uintptr_t)p.out & 15)) == 0;
#pragma unroll
  for (int d = 0; d < DT; ++d)
#pragma unroll
    for (int kp = 0; kp < 2; ++kp) {
      bf16x4 oa, ob;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        oa[i] = (bf16)(o[d][8 * kp + i] * inv);
        ob[i] = (bf16)(o[d][8 * kp + 4 + i] * inv);
      }
      const u32x2 a = __builtin_bit_cast(u32x2, oa), c = __builtin_bit_cast(u32x2, ob);
      const auto r0 = __builtin_amdgcn_permlane32_swap(a[0], c[0], false, false);
      const auto r1 = __builtin_amdgcn_permlane32_swap(a[1], c[1], false, false);
      const u32x4 v = {r0[0], r1[0], r0[1], r1[1]};
      if (valid) {
        bf16* at = out + 32 * d + 16 * kp + 8 * hf;
        if (wide) {
          *(u32x4*)at = v;
        } else {
          const bf16x8 e = __builtin_bit_cast(bf16x8, v);
#pragma unroll
          for (int i = 0; i < 8; ++i) at[i] = e[i];
        }
      }
    }
}

}  // namespace

bool flash_prefill_sizes(int H, int G, int D, int Dv, int BS, int tile_rows, float scale) {
  return D == Dv && (D == 64 || D == 128) && BS % 32 == 0 && G > 0 && H % G == 0 && scale > 0.f &&
         tile_rows % 128 == 0;
}

void launch_flash_prefill(const FlashParams& p, hipStream_t s) {
  if (p.num_tiles <= 0) return;
  const dim3 grid((unsigned)p.num_tiles * p.G * (p.tile_rows / 32 * (p.H / p.G) / NW));
  // Two teams of four waves, which take the steps in turn, where the grid leaves CUs to one team each: a
  // prompt of 700 tokens behind 300, 16 / 4 heads of 128, the layer 39.5 -> 35.2 us, one of 2000 67.5 ->
  // 59.2, the pooled form's 45.1 -> 41.3 and 57.1 -> 54.6.  At up to 512 workgroups 32 / 8 heads lost (8
  // prompts of 150 30.8 -> 36.6, 4 of 500 behind 600 66.4 -> 72.0).
  const bool two = grid.x <= 256;
#define AKAP_FP(DD, PL)                                                             \
  do {                                                                              \
    if (two) flash_prefill_kernel<DD, PL, 2><<<grid, 128 * NW, 0, s>>>(p);          \
    else flash_prefill_kernel<DD, PL, 1><<<grid, 64 * NW, 0, s>>>(p);               \
  } while (0)
  if (p.positions) {
    if (p.D == 64) AKAP_FP(64, true); else AKAP_FP(128, true);
  } else {
    if (p.D == 64) AKAP_FP(64, false); else AKAP_FP(128, false);
  }
#undef AKAP_FP
}

}  // namespace akap_stream
