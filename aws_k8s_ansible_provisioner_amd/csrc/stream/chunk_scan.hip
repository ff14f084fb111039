// Prompt chunks of the two recurrences with a matrix state and one decay per head and token, on
// the matrix instructions, with fp32 operands in three bf16 parts:
//   selective scan   S <- a_t S + dt_t B_t x_t^T,  y_t = S^T C_t + d x_t     (a_t from dt_t)
//   retention        S <- a S + k_t v_t^T,         o_t = S^T q_t, normed and gated per head
// A sequence's rows go in chunks of 32.  With c_i the sum of the log2 decays from the chunk's
// start through row i, S0 the state before it, k / q / v the rows (k times dt for the scan):
//   o_i   = 2^(c_i) q_i S0 + sum_{j <= i} 2^(c_i - c_j) (q_i . k_j) v_j
//   S_end = 2^(c_end) S0 + sum_j k_j (2^(c_end - c_j) v_j)^T
// Values, states and sums are fp32, the decays' sums fp64: differences of sums of the size of 30 in fp32
// would lose two digits.  The products with the state, which are most of the work, take their operands
// apart, x = h + m + l with 8 bits each, and sum the six largest of the nine products in fp32 (h h, the
// others' sums apart where there are registers for it): 2^-26 of a product is left out, and a sum of 16
// products is rounded once per instruction, where v_mfma_f32_32x32x2_f32 rounds every two.  Against 64 bits,
// 8 x 2048 rows: scan outputs 1.03e-7 and states 1.12e-7 (in fp32 products 1.04e-7 and 1.14e-7), retention
// states 1.7e-7 (2.7e-7).  Operands that do not split (not finite, past bf16's range, or one so small that
// a part would be denormal, which the matrix units take as zero) go through the fp32 products.
//
// chunk_prep_kernel prepares every (chunk, key head) side by side: the parts of q and k (rotated and
// scaled for the retention) as operand fragments and the 32 x 32 products q_i . k_j in fp32; the scan's
// keys belong to a group, so its heads share them.  It also sums the scan's decays.
// chunk_walk_kernel then walks the chunks of a (sequence, head): a wave owns 32 state columns in
// accumulators.  An accumulator lane holds column l & 31 and rows 8 g + 4 (l >> 5) + r in
// register 4 g + r: with the fragments' entries in that order (lane (i, hh) of step j: entries
// 16 j + 4 hh + 0..3 and 16 j + 8 + 4 hh + 0..3) eight neighbouring registers are an operand of the next
// product, so the state, the values and the outputs feed each other without lane traffic.
//
// Bound by vector work (900 instructions per chunk, half of them the state's parts) and products (4100 cycles per
// chunk); the next step's parts are formed between a step's products.  Of the 11200 cycles a chunk takes (8
// sequences of 64 heads, a wave per SIMD) 5100 issue, 4000 wait to issue, most of them behind products with nothing
// beside them (the state's own), 2000 wait for LDS, memory and barriers, of which fragments asked for a chunk
// earlier took none away.  16384 rows of 8 sequences, 64 heads x 128 x 64 states: 351 us, 377 on average
// under a profiler, where the fp32 products took 409 and the row-by-row scan 1420; 64 sequences of 26 rows
// 86 -> 65; 8 heads x 128 x 128 (segments) 78 + 34 for the pass before it, and 58 for the fragments: all
// three wait much for memory, and with entries of one part (HALF) 148 MB of fragments are written and 215
// read, of 215 and 316 where all have three (walks 3 + 4 us more, fragments 67).
//
// A walk alone is a serial chain of about 4 us per chunk (128 x 32 state entries per wave), so
// where the (sequence, head, 32 columns) triples of the long sequences leave SIMDs idle, these run in
// segments of rows: the same walk without outputs leaves every segment's own state,
// chunk_join_kernel turns these into the state before each segment, and the full walk starts
// from there.  Only the device knows the sequences' lengths: each workgroup counts the long ones.
#include <type_traits>

#include "../kernels/common.h"
#include "stream.h"

namespace akap_stream {

using akap::bf16;
using akap::bf16x8;
using akap::f32x16;

namespace {

constexpr int kL = 32;      // rows of a chunk
constexpr int kScal = 256;  // floats of the scan's scalars per (chunk, head): 5 x 32, and room

__device__ __forceinline__ float ldv(const float* p) { return *p; }
__device__ __forceinline__ float ldv(const bf16* p) { return (float)*p; }
__device__ __forceinline__ void ld4(const float* p, float (&v)[4]) {
  const float4 a = *(const float4*)p;
  v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
}
__device__ __forceinline__ void ld4(const bf16* p, float (&v)[4]) {
  const akap::bf16x4 a = *(const akap::bf16x4*)p;
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = (float)a[i];
}

// Rows of a chunk through a buffer descriptor: reads past `bytes` give zeros.
using Rsrc = __amdgpu_buffer_rsrc_t;
__device__ __forceinline__ Rsrc rows_of(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, bytes, 0x00020000);
}
__device__ __forceinline__ float rd(Rsrc r, uint32_t off, float) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}
__device__ __forceinline__ bf16 rd(Rsrc r, uint32_t off, bf16) {
  return __builtin_bit_cast(bf16, (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0));
}
__device__ __forceinline__ void st4(float* p, float a, float b, float c, float d) {
  *(float4*)p = make_float4(a, b, c, d);
}
__device__ __forceinline__ void st4(bf16* p, float a, float b, float c, float d) {
  const akap::bf16x4 o = {(bf16)a, (bf16)b, (bf16)c, (bf16)d};
  *(akap::bf16x4*)p = o;
}

// a value that all lanes hold, as a scalar
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// the same value, as one the compiler knows nothing about: what is derived from it is formed anew
// in every round of a loop instead of being kept in registers across it
__device__ __forceinline__ uint32_t fresh(uint32_t v) {
  asm volatile("" : "+v"(v));
  return v;
}

// 16 bytes per lane from global memory to LDS (a lane's place: the wave's address + 16 lane)
__device__ __forceinline__ void dma16(const void* g, void* l) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)g,
                                   (__attribute__((address_space(3))) void*)l, 16, 0, 0);
}

__device__ __forceinline__ f32x16 mfma(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ f32x16 mfma16(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
// Two values rounded to bf16, as a word: where entries of a vector are used again the compiler converts them one
// by one and packs them afterwards (a third of all vector work here).
__device__ __forceinline__ uint32_t pair(float a, float b) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, akap::bf16x2));
}
__device__ __forceinline__ float lower(uint32_t two) { return __uint_as_float(two << 16); }
__device__ __forceinline__ float upper(uint32_t two) { return __uint_as_float(two & 0xffff0000u); }

// v = h + m + l exactly (8 bits each, rounded to nearest) unless v is too large for bf16 or not finite
__device__ __forceinline__ void split8(const float (&v)[8], bf16x8& h, bf16x8& m, bf16x8& l) {
  u32x4 a, b, c;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    a[i] = pair(v[2 * i], v[2 * i + 1]);
    const float r = v[2 * i] - lower(a[i]), s = v[2 * i + 1] - upper(a[i]);
    b[i] = pair(r, s);
    c[i] = pair(r - lower(b[i]), s - upper(b[i]));
  }
  h = __builtin_bit_cast(bf16x8, a);
  m = __builtin_bit_cast(bf16x8, b);
  l = __builtin_bit_cast(bf16x8, c);
}
// Zeros and magnitudes in [kSmall, kSplits) split into three parts that the matrix units take as they are:
// they take a denormal part as zero, and the last bit of 2^-101 is 2^-124.  One value outside, whatever
// lies beside it, and the product is formed in fp32: against a large partner it may be what counts.
constexpr float kSplits = 3.38e38f, kSmall = 0x1p-101f;

// The scan's weights of a chunk's rows in the state after it come this much larger and the keys' parts this
// much smaller: the largest power that takes every weighted value, however far it decayed, to kSmall.
constexpr float kUp = 0x1p48f, kDown = 0x1p-48f;

// extremes of magnitudes; a NaN among them makes both NaN
struct Range {
  float lo = INFINITY, hi = 0.f;
  __device__ __forceinline__ void add(float v) {
    lo = __builtin_elementwise_minimum(lo, fabsf(v));
    hi = __builtin_elementwise_maximum(hi, fabsf(v));
  }
};
// below `limit` without being zero (zeros are ordinary, so this is asked where the range says so)
__device__ __forceinline__ bool below(float v, float limit) {
  return (__float_as_uint(v) << 1) - 1u < (__float_as_uint(limit) << 1) - 1u;
}

// Products of split operands: the largest go to `big`, the five next to `small`; what is left out is
// 2^-26 of the product.
__device__ __forceinline__ void mfma_split(const bf16x8 (&a)[3], const bf16x8 (&b)[3], f32x16& big,
                                           f32x16& small) {
  small = mfma16(a[2], b[0], small);
  big = mfma16(a[0], b[0], big);
  small = mfma16(a[0], b[2], small);
  small = mfma16(a[1], b[1], small);
  small = mfma16(a[1], b[0], small);
  small = mfma16(a[0], b[1], small);
}

// N times one matrix product and V vector instructions, in this order: the next step's vector work runs
// while a step's products do
template <int N, int V>
__device__ __forceinline__ void interleave() {
#pragma unroll
  for (int i = 0; i < N; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x002, V, 0);
  }
}

// A retention's decay below 0.41 per token takes the weight of a chunk's first key below 2^-40, and keys times
// weights to where they do not split.  They then come kLift larger and the values kSink smaller (8 x 2048
// rows, 8 heads x 128 x 128, decays of 0.003 to 0.07: 215 us as at other decays, 700 with the fp32 products).
constexpr float kLift = 0x1p80f, kSink = 0x1p-80f;
__device__ __forceinline__ bool lifted(float l2) { return l2 * (kL - 1) < -40.f; }

// decay^k for a decay given by its log2 (-inf: a decay of zero)
__device__ __forceinline__ float decay_pow(float l2, int k) {
  return k == 0 ? 1.0f : exp2f(l2 * (float)k);
}

// Keys in one bf16 part take the power of two in their weight, exactly, and values the rest of it, 1 to 2 times
// key_scale(), so that both split however small the weight is.  Keys come kEven smaller and values kEven larger:
// the power that takes every value of FLT_MIN and more to kSmall.
// (They are looked over times kFirst, as far from infinity and from zero as keys times whole weights.)
constexpr float kEven = 0x1p29f, kFirst = 0x1p-4f;
__device__ __forceinline__ int decay_exponent(float l2, int k) {
  return k == 0 ? 0 : (int)fmaxf(floorf(l2 * (float)k), -512.f);
}

// a retention's keys times this
template <int N>
constexpr float key_scale() { return N == 64 ? 0.125f : 0.08838834764831845f; }

// the sequence that owns an entry (the same in all lanes), and the rows [r0, r1) of the entry (r1 <= r0:
// none): a chain of scalar loads
typedef const __attribute__((address_space(4))) int32_t* ScalarInts;

// entries of the per-chunk buffers: sequence b (the same in all lanes) owns those from base(b) on
__device__ __forceinline__ int base_of(const int32_t* q_start, int b, int rows) {
  return ((ScalarInts)q_start)[b] / rows + b;
}

__device__ __forceinline__ int locate(const ChunkScanParams& p, int entry, int rows, int& r0, int& r1) {
  const ScalarInts q_start = (ScalarInts)p.q_start;
  entry = uniform(entry);
  int lo = 0, hi = p.B - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (q_start[mid] / rows + mid <= entry) lo = mid; else hi = mid - 1;
  }
  const int first = q_start[lo], end = q_start[lo + 1];
  r0 = first + (entry - (first / rows + lo)) * rows;
  r1 = min(r0 + rows, end);
  if (r0 < first) r1 = r0;
  return lo;
}

// Is a sequence of n rows walked whole?  Cut are those longer than a segment, unless they are so many
// that whole they fill the chip: from 768 waves on the second pass over the keys costs more than
// idle SIMDs (8 x 2048 rows, 8 heads x 128 x 128, 256 waves otherwise: 264 us in segments; 64 heads x
// 128 x 64, 1024 waves: 452 us whole).
constexpr int kFill = 768;
constexpr int kScanWaves = 2048, kRetentionWaves = 1024;   // see chunk_scan_piece()

// are the long sequences of the step cut?
__device__ __forceinline__ bool long_ones_cut(const ChunkScanParams& p) {
  const int per = p.H * (p.V / 32);
  if (p.B * per < kFill) return true;
  int count = 0;
#pragma unroll 4
  for (int b0 = 0; b0 < p.B; b0 += 64) {
    const int b = b0 + (int)(threadIdx.x & 63);
    count += __popcll(__ballot(p.q_start[min(b + 1, p.B)] - p.q_start[min(b, p.B)] > p.SEG));
  }
  return count > 0 && count * per < kFill;
}
__device__ __forceinline__ bool walked_whole(const ChunkScanParams& p, int n) {
  return n <= p.SEG || !long_ones_cut(p);
}

// The step's item-th walk: of the sequences that are not cut (WHOLE: else none of these) first, then of the cut
// ones' segments, without gaps.  True: there is one, of rows [r0, r1) of sequence b.  A lane looks at a
// sequence.  Of more sequences than lanes the item-th is looked at itself, and a cut one is a gap: so many are
// mostly short, and a walk of few rows would take less time than to find it (500 sequences of 30 rows, 16 heads x
// 128 x 128: 606 us by counting, 518 so; 64 heads x 128 x 64 with its convolution 1014 and 846).
constexpr int kCounted = 64;
template <bool WHOLE>
__device__ __forceinline__ bool walk_of(const ChunkScanParams& p, int item, int& b, int& r0, int& r1, bool& cut) {
  const int lane = threadIdx.x & 63;
  if (WHOLE && p.B > kCounted) {
    if (item < p.B) {
      b = uniform(item);
      r0 = ((ScalarInts)p.q_start)[b];
      r1 = ((ScalarInts)p.q_start)[b + 1];
      return r1 > r0 && walked_whole(p, r1 - r0);
    }
    item -= p.B;
  }
  const bool cuts = long_ones_cut(p);
  if (p.B == 1) {
    const ScalarInts q_start = (ScalarInts)p.q_start;
    const int first = q_start[0], end = q_start[1];
    cut = cuts && end - first > p.SEG;
    b = 0;
    r0 = first + (cut ? item * p.PIECE : 0);
    r1 = cut ? min(r0 + p.PIECE, end) : end;
    return r1 > r0 && (cut || (WHOLE && item == 0));
  }
  if (!cuts && (!WHOLE || p.B > kCounted)) return false;
  for (int turn = WHOLE && p.B <= kCounted ? 0 : 1; turn < 2; ++turn)
    for (int b0 = 0; b0 < p.B; b0 += 64) {
      const int from = p.q_start[min(b0 + lane, p.B)], n = p.q_start[min(b0 + lane + 1, p.B)] - from;
      const bool long_one = cuts && n > p.SEG;
      const int walks = n <= 0 ? 0 : turn == 0 ? !long_one : long_one ? (n + p.PIECE - 1) / p.PIECE : 0;
      // sums up to a lane: within rows of 16, then the last lane of one row or two to the next
      int upto = walks;
      upto += __builtin_amdgcn_update_dpp(0, upto, 0x111, 0xf, 0xf, false);
      upto += __builtin_amdgcn_update_dpp(0, upto, 0x112, 0xf, 0xf, false);
      upto += __builtin_amdgcn_update_dpp(0, upto, 0x114, 0xf, 0xf, false);
      upto += __builtin_amdgcn_update_dpp(0, upto, 0x118, 0xf, 0xf, false);
      upto += __builtin_amdgcn_update_dpp(0, upto, 0x142, 0xa, 0xf, false);
      upto += __builtin_amdgcn_update_dpp(0, upto, 0x143, 0xc, 0xf, false);
      const int total = __builtin_amdgcn_readlane(upto, 63);
      if (item < total) {
        const int at = __ffsll((unsigned long long)__ballot(upto > item)) - 1;
        const int first = __builtin_amdgcn_readlane(from, at), end = first + __builtin_amdgcn_readlane(n, at);
        const int k = item - __builtin_amdgcn_readlane(upto - walks, at);
        cut = turn == 1;
        b = b0 + at;
        r0 = first + (cut ? k * p.PIECE : 0);
        r1 = cut ? min(r0 + p.PIECE, end) : end;
        return true;
      }
      item -= total;
    }
  return false;
}

// first segment of sequence b in the buffers (long sequences alone have any): counted like the
// entries, or, where most sequences are short, from 2 q_start[b] / PIECE on (a long one of n rows has
// at most 2 n / PIECE of them)
__host__ __device__ __forceinline__ bool few_long(int T, int B, int PIECE) { return B > T / PIECE + 2; }

__device__ __forceinline__ size_t seg_base(const ChunkScanParams& p, int b) {
  return few_long(p.T, p.B, p.PIECE) ? (size_t)(2 * (int64_t)((ScalarInts)p.q_start)[b] / p.PIECE)
                                     : (size_t)base_of(p.q_start, b, p.PIECE);
}

// does a sequence whose first row is t (the same in all lanes) go on from its slot's state?  (The scan's row
// form starts anew at positions below 0 too.)
__device__ __forceinline__ bool goes_on(const ChunkScanParams& p, int t) {
  typedef const __attribute__((address_space(4))) int64_t* ScalarLongs;
  const int64_t pos = ((ScalarLongs)p.positions)[t];
  return p.mode == 0 ? pos > 0 : pos != 0;
}

// the slot of the sequence with first row t
__device__ __forceinline__ int slot_of(const ChunkScanParams& p, int t) { return ((ScalarInts)p.seq_slot)[t]; }

__device__ __forceinline__ bool live_slot(const ChunkScanParams& p, int slot) {
  return slot >= 0 && slot < p.num_slots;
}

// ------------------------------------------------------------------ fragments of q and k
// HALF: bf16 rows of a retention of which at most half the entries turn.  The other half of the queries' and keys'
// are bf16 numbers, one part instead of three: 36 of a chunk's 52 KB are written here and read by the walk, 16 of
// 24 by the pass before it.  These keys come times the powers of two in their weights (see kEven; if a value of the
// chunk does not split, as they are) and what is left of the weights goes to the values, in three parts.
//
// One workgroup per (chunk, key head).  Buffer of an entry, in pieces of 64 lanes x 16 bytes: [q: 3 parts
// of N / 16 pieces][k transposed: the same, the scan's times kDown, the retention's times their weights
// in the new state (see lifted())][q . k in fp32: 4][1 if a value does not split: then the parts are the
// fp32 values' upper and lower halves, without kDown, and those of a lifted() head without weights]; rows
// past the chunk's end are zero.
template <int MODE, int NT, typename TY, bool HALF>
__device__ __forceinline__ void fragments(const ChunkScanParams& p, const int entry, const int kh) {
  constexpr int N = NT * 32, LS = N + 4;   // rows 4 banks apart: 16-byte reads of 32 rows are free
  // q and k, then (once every wave has read them) the waves' shares of the products
  using TR = typename std::conditional<MODE == 0, double, float>::type;
  constexpr int kRed = 4096 * sizeof(TR) / 4;
  __shared__ __align__(16) float rows[2 * kL * LS > kRed ? 2 * kL * LS : kRed];
  __shared__ float wt[kL];     // retention: the rows' weights in the state after the chunk
  __shared__ float wp[HALF ? kL : 1];   // of keys in one part
  float *qs = rows, *ks = rows + kL * LS;
  TR* red = (TR*)rows;
  int r0, r1;
  const int b = locate(p, entry, kL, r0, r1);
  if (r1 <= r0) return;
  // (looked at once the rows are on their way; the positions of a sequence without a slot are not used)
  const bool live = live_slot(p, slot_of(p, ((ScalarInts)p.q_start)[b]));
  const int n = r1 - r0, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int half = p.rot_dims / 2;
  // a thread keeps to four columns; its rows' loads are in flight together
  const int d = (tid % (N / 4)) * 4, i0 = tid / (N / 4);
  constexpr int RS = 256 / (N / 4), RN = kL / RS;   // rows per turn, turns
  float q4[RN][4], k4[RN][4], q2[MODE == 1 ? RN : 1][4], k2[MODE == 1 ? RN : 1][4];
  int64_t pos[MODE == 1 ? RN : 1];
  const bool rot = MODE == 1 && d < p.rot_dims, low = d < half;
#pragma unroll
  for (int u = 0; u < RN; ++u) {
    const int t = r0 + min(i0 + u * RS, n - 1);
    if (MODE == 0) {
      const float* row = p.xbc + (size_t)t * p.x_stride + p.H * p.V + kh * N + d;
      ld4(row, k4[u]);
      ld4(row + p.KH * N, q4[u]);
    } else {
      const TY* row = (const TY*)p.proj + (size_t)t * p.proj_stride + kh * N;
      ld4(row + p.q_off + d, q4[u]);
      ld4(row + p.k_off + d, k4[u]);
      if (rot) {
        const int d2 = low ? d + half : d - half;
        pos[u] = p.positions[t];
        ld4(row + p.q_off + d2, q2[u]);
        ld4(row + p.k_off + d2, k2[u]);
      }
    }
  }
  if (rot) {
    const int a = low ? d : d - half;
#pragma unroll
    for (int u = 0; u < RN; ++u) {
      const float* cs = p.cos_sin + (size_t)(live ? pos[u] : 0) * p.rot_dims + a;
      float c4[4], s4[4];
      ld4(cs, c4);
      ld4(cs + half, s4);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float sn = low ? -s4[j] : s4[j];
        q4[u][j] = q4[u][j] * c4[j] + q2[u][j] * sn;
        k4[u][j] = k4[u][j] * c4[j] + k2[u][j] * sn;
      }
    }
  }
  // (keys of one part are needed without it)
  constexpr float staged = MODE == 1 && !HALF ? key_scale<N>() : 1.0f, kscale = HALF ? key_scale<N>() : 1.0f;
#pragma unroll
  for (int u = 0; u < RN; ++u) {
    const int i = i0 + u * RS;
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f), b4 = a;
    if (i < n) {
      a = make_float4(q4[u][0], q4[u][1], q4[u][2], q4[u][3]);
      b4 = make_float4(k4[u][0] * staged, k4[u][1] * staged, k4[u][2] * staged, k4[u][3] * staged);
    }
    *(float4*)(qs + i * LS + d) = a;
    *(float4*)(ks + i * LS + d) = b4;
  }
  const bool lift = MODE == 1 && lifted(p.log2_decay[kh]);
  if (MODE == 1 && tid < kL) {
    const float l2 = p.log2_decay[kh], by = lift ? kLift : 1.f;
    const float w = tid < n ? decay_pow(l2, n - 1 - tid) * by : 0.f;
    wt[tid] = w;
    if (HALF) wp[tid] = w != 0.f ? __builtin_ldexpf(by * kFirst, decay_exponent(l2, n - 1 - tid)) : 0.f;
  }
  __syncthreads();
  const int li = lane & 31, hh = lane >> 5;
  constexpr int NQ = N / 16, XQ = HALF ? NQ / 2 : NQ;
  float* buf = p.frag + ((size_t)entry * p.KH + kh) * p.frag_floats;
  // piece f: contraction step f of q (entries 16 f + 4 hh + 0..3 and 8 on), rows 32 (f / 2) of the state
  // and tokens 16 (f % 2) + 4 hh + 0..3 and 8 on of k
  float v[2][NQ / 4][8];
  Range range[2];
#pragma unroll
  for (int u = 0; u < NQ / 4; ++u) {
    const int f = wave + 4 * u, j0 = 16 * (f & 1) + 4 * hh;
    *(float4*)v[0][u] = *(const float4*)(qs + li * LS + 16 * f + 4 * hh);
    *(float4*)(v[0][u] + 4) = *(const float4*)(qs + li * LS + 16 * f + 8 + 4 * hh);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int j = j0 + (i & 3) + 8 * (i >> 2);
      const float k = ks[j * LS + 32 * (f >> 1) + li];
      v[1][u][i] = MODE == 0 ? k : !HALF || f < XQ ? k * kscale * wt[j] : k * wp[HALF ? j : 0];
    }
#pragma unroll
    for (int w = 0; w < 2; ++w)
#pragma unroll
      for (int i = 0; i < 8; ++i) range[w].add(v[w][u][i]);
  }
  // (fragment f's parts are of the values times scale, those of one part are asked for FLT_MIN alone)
  constexpr float scale[2] = {1.f, MODE == 0 ? kDown : 1.f}, scale1[2] = {1.f, 1.f / (kEven * kFirst)};
  constexpr float few = HALF ? __FLT_MIN__ / scale1[1] : kSmall / scale[1];
  bool bad = !(range[0].hi < kSplits) || !(range[1].hi < kSplits);
  if (range[0].lo < kSmall || range[1].lo < few) {
#pragma unroll
    for (int w = 0; w < 2; ++w)
#pragma unroll
      for (int u = 0; u < NQ / 4; ++u)
#pragma unroll
        for (int i = 0; i < 8; ++i)
          bad |= below(v[w][u][i], !HALF || wave + 4 * u < XQ ? kSmall / scale[w] : __FLT_MIN__ / scale1[w]);
  }
  bad = __syncthreads_or(bad);
  if (!live) return;
#pragma unroll
  for (int w = 0; w < 2; ++w)
#pragma unroll
    for (int u = 0; u < NQ / 4; ++u) {
      bf16x8 part[3];
      float e[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) e[i] = v[w][u][i] * (!HALF || wave + 4 * u < XQ ? scale[w] : scale1[w]);
      split8(e, part[0], part[1], part[2]);
      if (__builtin_expect(bad, 0)) {      // as they are, in two halves
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          uint32_t bits = __float_as_uint(v[w][u][i]);
          const int f = wave + 4 * u;
          if (w == 1 && (lift || (HALF && f >= XQ))) {
            const int j = 16 * (f & 1) + 4 * hh + (i & 3) + 8 * (i >> 2);
            bits = __float_as_uint(ks[j * LS + 32 * (f >> 1) + li] * (HALF && f >= XQ ? 1.f : kscale));
          }
          part[0][i] = __builtin_bit_cast(bf16, (uint16_t)(bits >> 16));
          part[1][i] = __builtin_bit_cast(bf16, (uint16_t)bits);
        }
      }
#pragma unroll
      for (int i = 0; i < 3; ++i)
        if (!HALF || i == 0 || wave + 4 * u < XQ)
          ((bf16x8*)buf)[(3 * NQ * w + wave + 4 * u + i * NQ) * 64 + lane] = part[i];
    }
  // q . k with the keys as rows: lane (i, hh) register 4 g + r is q_i . k_(8 g + 4 hh + r), the
  // operand the walk needs; the waves contract a part of the entries each.  The scan's in four chains
  // that meet in fp64: the products have mostly one sign, and the error of one long fp32 sum of them
  // was most of the outputs' (8.7e-8 against 64 bits, row by row 7.4e-8, so 7.0e-8)
  constexpr int NC = MODE == 0 ? 4 : 1;
  f32x16 acc[NC];
#pragma unroll
  for (int n = 0; n < NC; ++n)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[n][i] = 0.f;
  for (int f = wave; f < NT * 4; f += 4) {
    const float4 a = *(const float4*)(ks + li * LS + 8 * f + 4 * hh);
    const float4 c = *(const float4*)(qs + li * LS + 8 * f + 4 * hh);
    acc[0] = mfma(a.x * kscale, c.x, acc[0]);
    acc[1 % NC] = mfma(a.y * kscale, c.y, acc[1 % NC]);
    acc[2 % NC] = mfma(a.z * kscale, c.z, acc[2 % NC]);
    acc[3 % NC] = mfma(a.w * kscale, c.w, acc[3 % NC]);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    TR sum = acc[0][i];
#pragma unroll
    for (int n = 1; n < NC; ++n) sum += acc[n][i];
    red[wave * 1024 + ((i >> 2) * 64 + lane) * 4 + (i & 3)] = sum;
  }
  __syncthreads();
  TR s[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    s[r] = red[tid * 4 + r];
#pragma unroll
    for (int w = 1; w < 4; ++w) s[r] += red[w * 1024 + tid * 4 + r];
  }
  ((float4*)buf)[6 * NQ * 64 + tid] = make_float4((float)s[0], (float)s[1], (float)s[2], (float)s[3]);
  if (tid == 0) ((int*)buf)[6 * NQ * 256 + 1024] = bad;
}

// ------------------------------------------------------------------ step sizes and decays
// Half a wave per (chunk, head) of the selective scan, a lane per row.  With c the sums of the log2
// decays (formed in fp64): [32] dt, [32] 2^c, [32] kUp dt 2^(c_end - c), [32] c, [32] what c lost when
// it was rounded.  Rows past the end: dt 0, decay 1.
template <typename TY>
__device__ __forceinline__ void scalars(const ChunkScanParams& p, const int entry, const int heads) {
  const int i = threadIdx.x & 31;
  int r0, r1;
  const int b = locate(p, entry, kL, r0, r1);
  if (r1 <= r0 || !live_slot(p, slot_of(p, ((ScalarInts)p.q_start)[b]))) return;
  const int n = r1 - r0;
  const TY* src = (const TY*)p.proj + (size_t)(r0 + min(i, n - 1)) * p.proj_stride + p.dt_off;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int h = heads * 32 + u * 8 + (threadIdx.x >> 5);
    if (h >= p.H) return;   // (all lanes of a half wave share h)
    const float v = ldv(src + h) + p.dt_bias[h];
    const float dt = i < n ? (v > 20.f ? v : log1pf(expf(v))) : 0.f;
    double l = i < n ? -(double)expf(p.a_log[h]) * 1.4426950408889634 * (double)dt : 0.0;
    if (l < -4096.0) l = -4096.0;  // 2^l is zero long before; keeps the sums finite
#pragma unroll
    for (int o = 1; o < 32; o <<= 1) {
      const double up = __shfl_up(l, o, 32);
      if (i >= o) l += up;
    }
    const double end = __shfl(l, 31, 32);
    float* sc = p.scal + ((size_t)entry * p.H + h) * kScal;
    const float hi = (float)l;
    sc[i] = dt;
    sc[kL + i] = exp2f(hi);
    sc[2 * kL + i] = i < n ? kUp * (dt * exp2f((float)(end - l))) : 0.f;
    sc[3 * kL + i] = hi;
    sc[4 * kL + i] = (float)(l - (double)hi);
  }
}

// Both wait for chains of loads (8 x 2048 rows, 64 heads x 128 x 64: 13 us each, one launch after the other), so
// they run side by side in one, 21 us: the key heads' workgroups first, then those of 32 heads (in turns 23).
// Short steps gain the launch: a prompt of 200 rows 61 -> 55 us with its convolution, 64 of 26 106 -> 100.
template <int MODE, int NT, typename TY, bool HALF>
__global__ __launch_bounds__(256) void chunk_prep_kernel(const ChunkScanParams p) {
  if (MODE == 1 || (int)blockIdx.y < p.KH) fragments<MODE, NT, TY, HALF>(p, blockIdx.x, blockIdx.y);
  else scalars<TY>(p, blockIdx.x, blockIdx.y - p.KH);
}

// ------------------------------------------------------------------ the walk
// HW heads (of one key head) of V / 32 waves each, a wave per 32 state columns; FULL: outputs,
// from the state in the slot (or, SEGM and the sequence is cut, from the segment buffer); else the
// segment's own state from zeros.  Fragments and scalars arrive by LDS-DMA: those of q while the state
// of the chunk before is formed (a retention's segments ask for them once the outputs of the chunk before
// have used its own, see hand_on()), those of k (in time for the chunk's state) while its outputs are, so
// that one buffer of each does and two workgroups share a CU; the values in registers a chunk ahead.
template <int MODE, int NT, int V, int HW, typename TY, bool HALF, bool FULL, bool SEGM>
__global__ __launch_bounds__(2 * V * HW, 2) void chunk_walk_kernel(const ChunkScanParams p) {
  constexpr int N = NT * 32, NQ = NT * 2, VW = V / 32, NW = VW * HW;
  constexpr bool kNorm = MODE == 1 && FULL;
  constexpr int XP = MODE == 1 && sizeof(TY) == 2 ? 1 : 3;   // parts of a value (of bf16 rows: itself)
  // pieces of 1 KB: [q parts][q . k][scalars of the heads (scan)] and [k parts]; without outputs
  // twice [k parts][scalars]
  // (HALF: of the pieces from XQ on the first part alone)
  constexpr int XQ = HALF ? NQ / 2 : NQ;
  constexpr int KU = 3 * NQ, SU = MODE == 0 ? HW : 0, G0 = 3 * NQ, C0 = FULL ? G0 + 4 : KU;
  constexpr int QB = C0 + SU;
  __shared__ __align__(16) float4 qbuf[QB * 64];
  __shared__ __align__(16) float4 kbuf[(FULL ? KU : QB) * 64];
  __shared__ __align__(16) float tab[MODE == 1 ? NW * 2 * kL : 4];   // per wave, see below
  __shared__ __align__(16) float wtab[HALF ? NW * 2 * kL : 4];       // per wave, see below
  __shared__ __align__(16) float pd[kNorm ? 1024 : 4];       // retention: 2^(c_i - c_j), by lane
  __shared__ __align__(16) float ssq[kNorm ? 2 * NW * kL : 4];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 31, hh = lane >> 5;
  // SEGM: a workgroup per head and segment of a cut sequence (FULL: or sequence that is not cut), those that
  // find none last.  One that leaves at once shifts the turns in which the next ones are dealt out to the
  // CUs, and some then wait behind a full one: with such between them a tenth of the waves of 8 x 2048 rows,
  // 8 heads x 128 x 128 began when others had ended (passes of 48 and 111 us, now 36 and 87).  Heads of eight
  // walks side by side: heads that share their keys walk on one XCD, whose cache then holds these (24
  // sequences of 100 rows, 8 heads: 45.6 us, heads side by side 49.3).  Other keys' heads, and the next eight walks,
  // start at another XCD: walks are long and short by turns, or fewer than eight (2 prompts of 500 rows, 128 heads
  // of 8 keys x 64 x 128: 158 us, all heads of a walk on one XCD 162, turned 130; 8 of 300, 32 heads x 64 x 64 81,
  // 86, 76).
  const int heads = p.H / HW;
  int b, r0, r1, h0;
  bool cut = false;
  if (SEGM) {
    constexpr int kSide = 8;
    const int round = blockIdx.x / (kSide * heads), at = blockIdx.x % (kSide * heads);
    h0 = at / kSide * HW;
    const int turned = (at + round + (MODE == 0 ? h0 / (p.H / p.KH) : h0)) % kSide;
    if (!walk_of<FULL>(p, round * kSide + turned, b, r0, r1, cut)) return;
  } else {
    h0 = (int)blockIdx.x / p.B * HW;
    b = blockIdx.x % p.B;
    r0 = ((ScalarInts)p.q_start)[b];
    r1 = ((ScalarInts)p.q_start)[b + 1];
    if (r1 <= r0) return;
  }
  const int hw = wave / VW, h = h0 + hw;
  const int first = ((ScalarInts)p.q_start)[b];
  const size_t seg = cut ? (size_t)((int)seg_base(p, b) + (r0 - first) / p.PIECE) : 0;
  const int slot = slot_of(p, first);
  if (!live_slot(p, slot)) return;
  const int kh = MODE == 0 ? h0 / (p.H / p.KH) : h;
  const int col = (wave % VW) * 32 + li;
  const int c0 = (r0 - first) / kL, chunks = (r1 - r0 + kL - 1) / kL;
  const size_t cb = (size_t)(base_of(p.q_start, b, kL) + c0);
  const uint32_t l16 = lane * 16;
  auto frag_of = [&](int c) { return (const char*)(p.frag + ((cb + c) * p.KH + kh) * p.frag_floats); };
  auto pieces = [&](const char* src, float4* to, auto count) {
    constexpr int n = decltype(count)::value;
#pragma unroll
    for (int u = 0; u < (n + NW - 1) / NW; ++u)
      if ((u + 1) * NW <= n || u * NW + wave < n)
        dma16(src + (u * NW + wave) * 1024 + l16, to + (u * NW + wave) * 64);
  };
  auto stage_scalars = [&](int c, float4* to) {
    if (MODE == 0 && wave < HW)
      dma16((const char*)(p.scal + ((cb + c) * p.H + h0 + wave) * kScal) + l16, to + wave * 64);
  };
  auto parts_of = [&](const char* src, float4* to) {
    if (!HALF) {
      pieces(src, to, std::integral_constant<int, 3 * NQ>{});
      return;
    }
    pieces(src, to, std::integral_constant<int, NQ>{});
    pieces(src + NQ * 1024, to + NQ * 64, std::integral_constant<int, XQ>{});
    pieces(src + 2 * NQ * 1024, to + 2 * NQ * 64, std::integral_constant<int, XQ>{});
  };
  auto stage_q = [&](int c) {
    parts_of(frag_of(c), qbuf);
    pieces(frag_of(c) + 6 * NQ * 1024, qbuf + G0 * 64, std::integral_constant<int, 4>{});
    stage_scalars(c, qbuf + C0 * 64);
  };
  auto stage_k = [&](int c, float4* to) { parts_of(frag_of(c) + 3 * NQ * 1024, to); };
  // values of a chunk's rows 8 g + 4 hh + r at a lane's column
  const int ld = MODE == 0 ? p.x_stride : p.proj_stride;
  constexpr int es = MODE == 0 ? 4 : sizeof(TY);
  using TX = typename std::conditional<MODE == 0, float, TY>::type;
  const uint32_t lx = (uint32_t)(4 * hh * ld + (MODE == 0 ? 0 : p.v_off) + h * V + col) * es;
  TX xn[16];
  int odd_n;          // does a key or query of the chunk not split?
  auto values = [&](int c) {
    odd_n = *(const int*)(frag_of(c) + (6 * NQ + 4) * 1024);
    const int t0 = r0 + c * kL, n = min(kL, r1 - t0);
    const Rsrc rs = rows_of((MODE == 0 ? (const char*)p.xbc : (const char*)p.proj) + (size_t)t0 * ld * es,
                            (uint32_t)(n * ld * es));
    const uint32_t step = (uint32_t)ld * es;
    uint32_t o = fresh(lx);
#pragma unroll
    for (int s = 0; s < 16; ++s) {
      xn[s] = rd(rs, o, TX{});
      o += (s & 3) == 3 ? 5 * step : step;
    }
  };
  auto stage = [&](int c, float4* to) {
    stage_k(c, to);
    stage_scalars(c, to + C0 * 64);
  };
  // The first chunk's are on their way while the state is asked for.  (Not of a retention in fp32, but with outputs in
  // segments: its values' parts leave no registers for it.  14 spilled where now 9 do, without outputs 34 and 24; a
  // prompt of 100 rows, 8 heads x 128 x 128, 34.3 us and 31.9.)
  constexpr bool kFull32 = MODE == 1 && sizeof(TY) == 4 && !(FULL && SEGM);
  auto begin = [&] {
    values(0);
    if (FULL) stage_q(0); else stage(0, qbuf);
  };
  if (!kFull32) begin();
  const float l2 = MODE == 1 ? p.log2_decay[h] : 0.f;
  const bool lift = MODE == 1 && uniform(lifted(l2));
  // retention: decay^k and decay^(k + 1)
  float* tb = tab + (MODE == 1 ? wave * 2 * kL : 0);
  // HALF: what the values of a chunk's rows take of their weights in the state after it, and zeros
  float* wb = wtab + (HALF ? wave * 2 * kL : 0);
  if (MODE == 1) {
    if (lane < kL) {
      tb[lane] = decay_pow(l2, lane);
      tb[kL + lane] = decay_pow(l2, lane + 1);
    }
    if (HALF) {
      const float rest = __builtin_ldexpf(decay_pow(l2, kL - 1 - lane), -decay_exponent(l2, kL - 1 - lane));
      wb[lane] = lane < kL ? rest * (key_scale<N>() * kEven * (lift ? kSink : 1.f)) : 0.f;
    }
    if (kNorm) {
      for (int e = tid; e < 1024; e += 64 * NW) {
        const int ln = (e >> 2) & 63, j = 8 * (e >> 8) + 4 * (ln >> 5) + (e & 3), i = ln & 31;
        pd[e] = j <= i ? decay_pow(l2, i - j) : 0.f;
      }
    }
  }
  // entry (row, column) of the state: the scan keeps [N, V], the retention [V, N]
  float* sp = cut ? p.seg + (seg * p.H + h) * N * V
                  : p.state + ((size_t)slot * p.H + h) * N * V;
  f32x16 S[NT];
  const bool load = FULL && (cut || goes_on(p, first));
  const bool anew = FULL && (cut ? r0 == first && !goes_on(p, first) : !load);   // a state of zeros
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int row = 32 * t + 8 * g + 4 * hh;
      if (!load) {
#pragma unroll
        for (int r = 0; r < 4; ++r) S[t][4 * g + r] = 0.f;
      } else if (MODE == 0) {
#pragma unroll
        for (int r = 0; r < 4; ++r) S[t][4 * g + r] = sp[(size_t)(row + r) * V + col];
      } else {
        const float4 v = *(const float4*)(sp + (size_t)col * N + row);
        S[t][4 * g] = v.x; S[t][4 * g + 1] = v.y; S[t][4 * g + 2] = v.z; S[t][4 * g + 3] = v.w;
      }
    }
  const float dsk = MODE == 0 ? p.d_skip[h] : 0.f;
  float total = 0.f;   // log2 decay of the segment
  // outputs transposed: row 8 g + 4 hh + r of the accumulator is a column of the state, lane li the
  // token.  They are written after the next chunk's wait, which would otherwise wait for them.
  f32x16 O;
  auto write = [&](int c) {
    const int t = r0 + c * kL + li;
    if (t >= r1) return;
    const int at = h * V + (wave % VW) * 32 + 4 * hh;
    if (MODE == 0) {
      float* o = p.y + (size_t)t * p.H * V + at;
#pragma unroll
      for (int g = 0; g < 4; ++g)
        st4(o + 8 * g, O[4 * g], O[4 * g + 1], O[4 * g + 2], O[4 * g + 3]);
    } else {
      TY* o = (TY*)p.out + (size_t)t * p.out_stride + at;
#pragma unroll
      for (int g = 0; g < 4; ++g)
        st4(o + 8 * g, O[4 * g], O[4 * g + 1], O[4 * g + 2], O[4 * g + 3]);
    }
  };
  float x[16];
  bool odd, apart;    // the chunk's keys or queries, its weighted values do not split
  auto arrive = [&] {                 // what this wave requested, then every wave
    // (vmcnt 0, lgkmcnt 0, as a builtin: the compiler then knows that the values have arrived)
    __builtin_amdgcn_s_waitcnt(0x0070);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  auto take = [&](int c) {            // the chunk's values; the next one's are requested
#pragma unroll
    for (int s = 0; s < 16; ++s) x[s] = (float)xn[s];
    odd = __builtin_amdgcn_readfirstlane(odd_n) != 0;
    if (c + 1 < chunks) values(c + 1);
  };
  // the fp32 entries 4 (f & 1) .. + 3 of a piece's parts
  auto joined = [&](const bf16x8* parts, int f) {
    typedef uint32_t Words __attribute__((ext_vector_type(2)));   // two entries each
    const Words* at = (const Words*)(parts + (f >> 1) * 64) + (f & 1);
    const Words a = at[0];
    if (f >> 1 >= XQ)
      return make_float4(lower(a[0]), upper(a[0]), lower(a[1]), upper(a[1]));
    const Words b = at[NQ * 128], d = at[NQ * 256];
    float v[4];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint32_t top = 0xffff0000u;
      const float lo = (__uint_as_float(a[i] << 16) + __uint_as_float(b[i] << 16)) +
                       __uint_as_float(d[i] << 16);
      const float hi = (__uint_as_float(a[i] & top) + __uint_as_float(b[i] & top)) +
                       __uint_as_float(d[i] & top);
      v[2 * i] = odd ? __uint_as_float(a[i] << 16 | (b[i] & ~top)) : lo;
      v[2 * i + 1] = odd ? __uint_as_float((a[i] & top) | b[i] >> 16) : hi;
    }
    return make_float4(v[0], v[1], v[2], v[3]);
  };
  auto part8 = [&](const float* v, bf16x8 (&to)[3]) {
    const float e[8] = {v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7]};
    split8(e, to[0], to[1], to[2]);
  };
  // the values times their weights in the state after the chunk (the scan's times kUp; the retention's are
  // in k), and their parts
  float xw[16];
  bf16x8 w[2][3], wh[HALF ? 2 : 1][3];       // (wh: of values times wb, for keys in one part)
  Range wr;
  float4 w4[MODE == 0 || HALF ? 4 : 1];
  auto fetch_weights = [&](const float* sc, int n) {
    if (MODE == 0) {
#pragma unroll
      for (int g = 0; g < 4; ++g) w4[g] = *(const float4*)(sc + 2 * kL + 8 * g + 4 * hh);
    } else if (HALF) {
      const float* at = wb + (kL - n) + 4 * hh;
#pragma unroll
      for (int g = 0; g < 4; ++g) w4[g] = make_float4(at[8 * g], at[8 * g + 1], at[8 * g + 2], at[8 * g + 3]);
    }
  };
  // values s and s + 1 times their weights, in parts (of the unrounded products)
  auto weigh_two = [&](int s, uint32_t (&part)[3]) {
    const float f0 = (&w4[s >> 2].x)[s & 3], f1 = (&w4[s >> 2].x)[(s & 3) + 1];
    part[0] = pair(x[s] * f0, x[s + 1] * f1);
    const float r0 = fmaf(x[s], f0, -lower(part[0])), r1 = fmaf(x[s + 1], f1, -upper(part[0]));
    part[1] = pair(r0, r1);
    part[2] = pair(r0 - lower(part[1]), r1 - upper(part[1]));
  };
  // (in twelve pieces, which stand between products)
  auto weigh_four = [&](int g) __attribute__((always_inline)) {
    if (g == 0) wr = Range{};
    const float f[4] = {w4[MODE == 0 ? g : 0].x, w4[MODE == 0 ? g : 0].y, w4[MODE == 0 ? g : 0].z,
                        w4[MODE == 0 ? g : 0].w};
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float v = MODE == 0 ? x[4 * g + r] * f[r] : x[4 * g + r];
      xw[4 * g + r] = v;
      if (MODE == 0) wr.hi = __builtin_elementwise_maximum(wr.hi, fabsf(v));
      else wr.add(v);
    }
  };
  u32x4 wp[3];
  auto weigh_pair = [&](int m, int i) __attribute__((always_inline)) {
    // (parts of the unrounded product)
    const int at = 8 * m + 2 * i;
    const float* f = MODE == 0 ? &w4[MODE == 0 ? at >> 2 : 0].x + (at & 3) : nullptr;
    wp[0][i] = pair(xw[at], xw[at + 1]);
    if (XP == 3) {
      const float r = fmaf(x[at], MODE == 0 ? f[0] : 1.f, -lower(wp[0][i]));
      const float s = fmaf(x[at + 1], MODE == 0 ? f[1] : 1.f, -upper(wp[0][i]));
      wp[1][i] = pair(r, s);
      wp[2][i] = pair(r - lower(wp[1][i]), s - upper(wp[1][i]));
    }
    if (i < 3) return;
#pragma unroll
    for (int u = 0; u < XP; ++u) w[m][u] = __builtin_bit_cast(bf16x8, wp[u]);
#pragma unroll
    for (int u = 0; u < XP; ++u) asm volatile("" : "+v"(w[m][u]));   // (formed here, beside products)
  };
  auto weigh = [&] {
#pragma unroll
    for (int g = 0; g < 4; ++g) weigh_four(g);
#pragma unroll
    for (int i = 0; i < 8; ++i) weigh_pair(i >> 2, i & 3);
    if constexpr (HALF) {
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        u32x4 part[3];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          uint32_t two[3];
          weigh_two(8 * m + 2 * i, two);
#pragma unroll
          for (int u = 0; u < 3; ++u) part[u][i] = two[u];
        }
#pragma unroll
        for (int u = 0; u < 3; ++u) {
          wh[m][u] = __builtin_bit_cast(bf16x8, part[u]);
          asm volatile("" : "+v"(wh[m][u]));
        }
      }
    }
  };
  // do the weighted values split (a value of one part: is it one that the matrix units take)?
  auto judge = [&] {
    // Of one part they also meet pair weights that may be too small to split, see outputs(): what these
    // lose, 2^-125, stays far below the normed rows' roundings while the values are no larger.
    apart = __any(!(wr.hi < (XP == 3 ? kSplits : 0x1p40f)));
    const float least = (XP == 3 ? kSmall : __FLT_MIN__) * (lift ? kLift : 1.f);
    if (MODE == 1 && __builtin_expect(__any(wr.lo < least), 0)) {     // (kUp: none of the scan's)
      bool few = false;
#pragma unroll
      for (int s = 0; s < 16; ++s) few |= below(x[s], least);
      apart |= __any(few);
    }
    if (MODE == 0 && __builtin_expect(apart, 0)) {
#pragma unroll
      for (int s = 0; s < 16; ++s) xw[s] = x[s] * ((&w4[MODE == 0 ? s >> 2 : 0].x)[s & 3] * kDown);
    }
  };
  // the state after the chunk of n rows: dend S + k^T xw
  auto advance = [&](const float4* kb, float dend, int n) {
    const bf16x8* kp = (const bf16x8*)kb + fresh(lane);
    if (__builtin_expect(odd || apart, 0)) {
      if (MODE == 0 && !apart) {       // (judge() did it for others)
#pragma unroll
        for (int s = 0; s < 16; ++s) xw[s] *= kDown;
      }
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) S[t][i] *= dend;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        float up[4];       // undoes the scaling of a key; a lifted() head's values take its weight's exponent
        float upe[4];      // the same of a key in one part, which takes its own weight's rest besides
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          up[r] = MODE == 0 && !odd ? kUp : 1.f;
          if (HALF) {
            const float f = lift ? 1.f : tb[max(n - 1 - (8 * g + 4 * hh + r), 0)];
            upe[r] = odd ? key_scale<N>() * f : wb[kL - n + 8 * g + 4 * hh + r];
          }
          if (lift) {
            const float f = tb[max(n - 1 - (8 * g + 4 * hh + r), 0)];
            const int e = __builtin_amdgcn_frexp_expf(f);
            xw[4 * g + r] = odd ? xw[4 * g + r] * f : __builtin_ldexpf(xw[4 * g + r], e);
            if (!odd) {
              up[r] = __builtin_ldexpf(kSink, -e);
              if (HALF) upe[r] = __builtin_ldexpf(upe[r], -e);
            }
          }
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const float4 a = joined(kp, 4 * t + g);
          const bool one = HALF && t >= NT / 2;
          S[t] = mfma(a.x * (one ? upe[0] : up[0]), xw[4 * g], S[t]);
          S[t] = mfma(a.y * (one ? upe[1] : up[1]), xw[4 * g + 1], S[t]);
          S[t] = mfma(a.z * (one ? upe[2] : up[2]), xw[4 * g + 2], S[t]);
          S[t] = mfma(a.w * (one ? upe[3] : up[3]), xw[4 * g + 3], S[t]);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      return;
    }
    if (lift) {          // (parts anew: scaled where they are formed they would be for every head)
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = xw[8 * m + i] * kSink;
        split8(v, w[m][0], w[m][1], w[m][2]);
#pragma unroll
        for (int u = 0; u < XP; ++u) asm volatile("" : "+v"(w[m][u]));
      }
    }
    // piece u: rows 32 (u / 2) of the state, tokens 16 (u % 2) on; the next one's fragments are on
    // their way while a piece's products run, the smallest first
    bf16x8 k[2][3];
    auto fetch = [&](int u) {
#pragma unroll
      for (int i = 0; i < 3; ++i)
        if (i == 0 || u < XQ) k[u & 1][i] = kp[(u + i * NQ) * 64];
    };
    // (of a factor that the compiler knows nothing about: else all of them, common to both ways through here,
    // stand ahead of the branch and not between the products)
    float by = dend;
    asm volatile("" : "+v"(by));
    auto decay = [&](int t) {
#pragma unroll
      for (int i = 0; i < 16; ++i) S[t][i] *= by;
    };
    fetch(0);
    decay(0);
#pragma unroll
    for (int u = 0; u < NQ; ++u) {
      const int t = u >> 1, m = u & 1;
      if (u + 1 < NQ) fetch(u + 1);
      __builtin_amdgcn_sched_barrier(0);
      constexpr int ka[6] = {2, 0, 1, 1, 0, 0}, wa[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
      for (int i = 0; i < 6; ++i)
        if (HALF && t >= NT / 2) {
          if (ka[i] == 0) S[t] = mfma16(k[m][0], wh[m][wa[i]], S[t]);
        } else if (wa[i] < XP) {
          S[t] = mfma16(k[m][ka[i]], w[m][wa[i]], S[t]);
        }
      if (m == 0 && t + 1 < NT) {
        decay(t + 1);
        interleave<XP == 3 ? 6 : 3, XP == 3 ? 3 : 6>();
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // hand_on() lets the next chunk's queries into the buffer.  A retention's segments do so as soon as the queries
  // were used and norm a chunk's outputs when the next one's keys were asked for: what follows the queries'
  // products is short (walk of 8 x 2048 rows, 8 heads x 128 x 128 84 -> 76 us, 40 prompts of 300 rows 139 -> 129).
  // The scan has more to do there (half a per cent slower so), and a few heads alone wait for each step and not
  // for memory (a retention's prompt of 100 rows 28.9 us, so 29.9).
  constexpr bool kEarly = MODE == 1 && SEGM;
  float dend;
  auto outputs = [&](int c, auto hand_on) {
    const int t0 = r0 + c * kL, n = min(kL, r1 - t0);
    const int lane_ = (int)fresh(lane), li = lane_ & 31, hh = lane_ >> 5;
    const bf16x8* qp = (const bf16x8*)qbuf + lane_;
    const float* sc = MODE == 0 ? (const float*)(qbuf + (C0 + hw) * 64) : nullptr;
    bf16x8 q[2][3];                   // (the next fragments are on their way while a step's products run)
    auto fetch = [&](int j) {
#pragma unroll
      for (int u = 0; u < 3; ++u)
        if (u == 0 || j < XQ) q[j & 1][u] = qp[(j + u * NQ) * 64];
    };
    fetch(0);
    float P[16];
    const float ch_i = MODE == 0 ? sc[3 * kL + li] : 0.f, cl_i = MODE == 0 ? sc[4 * kL + li] : 0.f;
    const float e = MODE == 0 ? sc[kL + li] : tb[kL + li];
    // q_i . k_j times the decay between the tokens (the scan's: and dt_j), for j = 8 g + 4 hh + 0..3
    float4 pl[4];
    auto fetch_pairs = [&](int g) {
      pl[0] = qbuf[(G0 + g) * 64 + lane_];
      if (MODE == 0) {
        pl[1] = *(const float4*)(sc + 8 * g + 4 * hh);
        pl[2] = *(const float4*)(sc + 3 * kL + 8 * g + 4 * hh);
        pl[3] = *(const float4*)(sc + 4 * kL + 8 * g + 4 * hh);
      } else {
        pl[1] = *(const float4*)(pd + (g * 64 + lane_) * 4);
      }
    };
    auto pair_weights = [&](int g) {
      const float gv[4] = {pl[0].x, pl[0].y, pl[0].z, pl[0].w};
      const float dt[4] = {pl[1].x, pl[1].y, pl[1].z, pl[1].w};
      if (MODE == 0) {
        // the sums as float pairs: a difference of sums then has the error of its own size
        const float ch[4] = {pl[2].x, pl[2].y, pl[2].z, pl[2].w};
        const float cl[4] = {pl[3].x, pl[3].y, pl[3].z, pl[3].w};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int j = 8 * g + 4 * hh + r;
          const float d = (ch_i - ch[r]) + (cl_i - cl[r]);
          float f = gv[r] * (dt[r] * __builtin_amdgcn_exp2f(d));
          // (d_skip x is the diagonal's share of the same product)
          f += j == li ? dsk : 0.f;
          asm("" : "+v"(f));     // a select, no branch
          P[4 * g + r] = j <= li ? f : 0.f;
        }
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float f = gv[r] * dt[r];
          asm("" : "+v"(f));
          P[4 * g + r] = 8 * g + 4 * hh + r <= li ? f : 0.f;
        }
      }
    };
    f32x16 O2;
#pragma unroll
    for (int i = 0; i < 16; ++i) O[i] = O2[i] = 0.f;
    bf16x8 a[2][3];
    float least = INFINITY;           // of the lane's part of the state
    auto state_parts = [&](int j) {
      float v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        v[i] = S[j >> 1][8 * (j & 1) + i];
        least = __builtin_elementwise_minimum(least, fabsf(v[i]));
      }
      split8(v, a[j & 1][0], a[j & 1][1], a[j & 1][2]);
    };
    constexpr int PG = NQ / 4;        // steps per group of pairs
    constexpr bool kEarlyWeights = XP == 3 && PG > 1;
    fetch_pairs(0);
    state_parts(0);
#pragma unroll
    for (int j = 0; j < NQ; ++j) {
      if (j + 1 < NQ) fetch(j + 1);
      if (PG == 1 ? j > 0 : j % PG == 1 && j + 1 < NQ) fetch_pairs(PG == 1 ? j : j / PG + 1);
      if (kEarlyWeights && j + 2 == NQ) fetch_weights(sc, n);
      __builtin_amdgcn_sched_barrier(0);
      if (j < XQ) {
        mfma_split(a[j & 1], q[j & 1], O, O2);
      } else {
        O2 = mfma16(a[j & 1][2], q[j & 1][0], O2);
        O = mfma16(a[j & 1][0], q[j & 1][0], O);
        O2 = mfma16(a[j & 1][1], q[j & 1][0], O2);
      }
      if (j + 1 < NQ) state_parts(j + 1);
      if (kEarlyWeights && j + 1 == NQ) {   // (their factors were asked for a step before)
#pragma unroll
        for (int g = 0; g < 4; ++g) weigh_four(g);
        interleave<6, 6>();
      } else if (j % PG == 0) {
        pair_weights(j / PG);
        if (j < XQ) interleave<6, MODE == 0 ? 18 : 12>(); else interleave<3, 24>();
      } else {
        if (j < XQ) interleave<6, 9>(); else interleave<3, 18>();
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (!kEarlyWeights) fetch_weights(sc, n);
    if (!kFull32) dend = MODE == 0 ? sc[2 * kL - 1] : tb[kL + n - 1];
#pragma unroll
    for (int s = 0; s < 16; ++s) O[s] = (O[s] + O2[s]) * e;
    __builtin_amdgcn_sched_barrier(0);
    if (kEarly) {
      hand_on();
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (XP == 3) {
      // (Values and weights would take as long to split.  The pieces are set between the products by hand: asked
      // to, the compiler left all of them behind the last, 8 x 2048 rows, 64 heads 525 -> 520 us with the decays.)
#pragma unroll
      for (int s = 0; s < 16; ++s) {
        O = mfma(x[s], P[s], O);
        if (s < 4 && !kEarlyWeights) weigh_four(s);
        if (s >= 4 && s < 12) weigh_pair((s - 4) >> 2, s & 3);
        __builtin_amdgcn_sched_barrier(0);
      }
      judge();
    } else {
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        bf16x8 v, b[3];
        part8(P + 8 * m, b);
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = (bf16)x[8 * m + i];
#pragma unroll
        for (int u = 2; u >= 0; --u) O = mfma16(v, b[u], O);
      }
      weigh();
      judge();
    }
    float fin = 0.f;
#pragma unroll
    for (int s = 0; s < 16; ++s) fin = fmaf(O[s], 0.f, fin);
    bool few = false;
    if (__builtin_expect((c > 0 || !anew) && __any(!(least >= kSmall)), 0)) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) few |= below(S[t][i], kSmall);
    }
    if (__builtin_expect(odd || (XP == 1 && apart) || __any(fin != 0.f || few), 0)) {
      // an operand that does not split, or is not finite: the fp32 products (queries from memory, or still here)
      const bf16x8* qg = kFull32 ? qp : (const bf16x8*)frag_of(c) + fresh(lane);
#pragma unroll
      for (int i = 0; i < 16; ++i) O[i] = 0.f;
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const float4 a = joined(qg, 4 * t + g);
          O = mfma(S[t][4 * g], a.x, O);
          O = mfma(S[t][4 * g + 1], a.y, O);
          O = mfma(S[t][4 * g + 2], a.z, O);
          O = mfma(S[t][4 * g + 3], a.w, O);
        }
#pragma unroll
      for (int s = 0; s < 16; ++s) O[s] *= e;
      float inf = 0.f;
#pragma unroll
      for (int s = 0; s < 16; ++s) inf = fmaf(x[s], 0.f, inf);
      if (__any(inf != 0.f)) {
        // a value that is not finite must not reach the rows before its own (0 x inf)
#pragma unroll 1
        for (int i = 0; i < kL; ++i) {
          f32x16 one = O;
#pragma unroll
          for (int s = 0; s < 16; ++s)
            one = mfma(8 * (s >> 2) + 4 * hh + (s & 3) <= i ? x[s] : 0.f, P[s], one);
#pragma unroll
          for (int s = 0; s < 16; ++s) O[s] = li == i ? one[s] : O[s];
        }
      } else {
#pragma unroll
        for (int s = 0; s < 16; ++s) O = mfma(x[s], P[s], O);
      }
    }
  };
  if (kFull32) begin();
  if constexpr (FULL) {
    akap::bf16x4 zb[kNorm ? 4 : 1];
    float4 zf[kNorm ? 4 : 1];
    // the head's root mean square: a lane's columns, the other half's, the other waves'
    auto finish = [&](int c) {
      if (kNorm) {
        const float* sq = ssq + (c & 1) * NW * kL;
        float ss = 0.f;
#pragma unroll
        for (int w = 0; w < VW; ++w) ss += sq[(hw * VW + w) * kL + li];
        const float inv = 1.0f / sqrtf(ss / (float)V + p.eps);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          float zv[4];
          if (sizeof(TY) == 2) {
#pragma unroll
            for (int r = 0; r < 4; ++r) zv[r] = (float)zb[g][r];
          } else {
            zv[0] = zf[g].x; zv[1] = zf[g].y; zv[2] = zf[g].z; zv[3] = zf[g].w;
          }
#pragma unroll
          for (int r = 0; r < 4; ++r)
            O[4 * g + r] = O[4 * g + r] * inv * zv[r] * (1.0f / (1.0f + __expf(-zv[r])));
        }
      }
    };
#pragma unroll 1
    for (int c = 0; c < chunks; ++c) {
      const int t0 = r0 + c * kL, n = min(kL, r1 - t0);
      arrive();                       // the queries are there, the keys before were used
      take(c);
      stage_k(c, kbuf);
      if (c > 0) {
        if (kEarly) finish(c - 1);
        write(c - 1);
      }
      if (kNorm) {
        const TY* zr = (const TY*)p.proj + (size_t)(t0 + min(li, n - 1)) * p.proj_stride + p.g_off +
                       h * V + (wave % VW) * 32 + 4 * hh;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          if (sizeof(TY) == 2) zb[g] = *(const akap::bf16x4*)(zr + 8 * g);
          else zf[g] = *(const float4*)(zr + 8 * g);
        }
      }
      auto hand_on = [&] {
        arrive();                     // the keys are there, the queries were used
        if (c + 1 < chunks) stage_q(c + 1);
      };
      outputs(c, hand_on);
      if (kFull32) dend = tb[kL + n - 1];
      if (kNorm) {
        float ss = 0.f;
#pragma unroll
        for (int s = 0; s < 16; ++s) ss = fmaf(O[s], O[s], ss);
        ss += __shfl_xor(ss, 32, 64);
        if (hh == 0) ssq[(c & 1) * NW * kL + wave * kL + li] = ss;
      }
      if (!kEarly) hand_on();
      advance(kbuf, dend, n);
      if (!kEarly) finish(c);
    }
    if (kEarly) {
      arrive();
      finish(chunks - 1);
    }
    write(chunks - 1);
  } else {
    // (now and next are restrict so that the reads of one buffer are known not to touch the other:
    // else every read would wait for the DMA under way)
    auto step = [&](int c, const float4* __restrict__ now, float4* __restrict__ next) {
      const int n = min(kL, r1 - (r0 + c * kL));
      arrive();
      take(c);
      if (c + 1 < chunks) stage(c + 1, next);
      const float* sc = MODE == 0 ? (const float*)(now + (C0 + hw) * 64) : nullptr;
      const float dend = MODE == 0 ? sc[2 * kL - 1] : tb[kL + n - 1];
      if (MODE == 0) total += sc[4 * kL - 1];
      fetch_weights(sc, n);
      weigh();
      judge();
      advance(now, dend, n);
    };
#pragma unroll 1
    for (int c = 0; c < chunks; c += 2) {
      step(c, qbuf, kbuf);
      if (c + 1 < chunks) step(c + 1, kbuf, qbuf);
    }
  }
  if (FULL && cut) return;   // the slots were written when the segments were joined
  // (addresses formed anew: kept since the state was read they would take the loop's registers)
  const uint32_t first_at = fresh(MODE == 0 ? 4 * hh * V + col : col * N + 4 * hh);
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int row = 32 * t + 8 * g;
      if (MODE == 0) {
#pragma unroll
        for (int r = 0; r < 4; ++r) sp[first_at + (row + r) * V] = S[t][4 * g + r];
      } else {
        *(float4*)(sp + first_at + row) = make_float4(S[t][4 * g], S[t][4 * g + 1],
                                                             S[t][4 * g + 2], S[t][4 * g + 3]);
      }
    }
  if (SEGM && !FULL && lane == 0 && wave % VW == 0)
    p.seg_decay[seg * p.H + h] = MODE == 0 ? exp2f(total) : decay_pow(l2, r1 - r0);
}

// the state before each segment from the segments' own states, and the sequence's final state
// into its slot: a thread per four entries, the loads of eight segments in flight together
__global__ __launch_bounds__(256) void chunk_join_kernel(const ChunkScanParams p) {
  const int b = blockIdx.x, h = blockIdx.y;
  const size_t hs = (size_t)p.V * p.N;
  const size_t e = ((size_t)blockIdx.z * 256 + threadIdx.x) * 4;
  const int r0 = ((ScalarInts)p.q_start)[b], r1 = ((ScalarInts)p.q_start)[b + 1];
  if (r1 <= r0 || walked_whole(p, r1 - r0) || e >= hs) return;
  const int slot = slot_of(p, r0);
  if (!live_slot(p, slot)) return;
  const int nseg = (r1 - r0 + p.PIECE - 1) / p.PIECE;
  const size_t sb = seg_base(p, b);
  float4* st = (float4*)(p.state + ((size_t)slot * p.H + h) * hs + e);
  float4 prev = goes_on(p, r0) ? *st : make_float4(0.f, 0.f, 0.f, 0.f);
  for (int s0 = 0; s0 < nseg; s0 += 8) {
    float4 own[8];
    float dec[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const size_t at = (sb + min(s0 + u, nseg - 1)) * p.H + h;
      own[u] = *(const float4*)(p.seg + at * hs + e);
      dec[u] = p.seg_decay[at];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      if (s0 + u >= nseg) break;
      *(float4*)(p.seg + ((sb + s0 + u) * p.H + h) * hs + e) = prev;
      prev.x = fmaf(dec[u], prev.x, own[u].x);
      prev.y = fmaf(dec[u], prev.y, own[u].y);
      prev.z = fmaf(dec[u], prev.z, own[u].z);
      prev.w = fmaf(dec[u], prev.w, own[u].w);
    }
  }
  *st = prev;
}

template <int MODE, int NT, int V, int HW, typename TY, bool HALF = false>
void run(const ChunkScanParams& p, hipStream_t s) {
  const int chunks = p.T / kL + p.B;
  chunk_prep_kernel<MODE, NT, TY, HALF>
      <<<dim3(chunks, p.KH + (MODE == 0 ? (p.H + 31) / 32 : 0)), 256, 0, s>>>(p);
  constexpr int nt = 2 * V * HW;
  if (p.SEG == 0) {
    chunk_walk_kernel<MODE, NT, V, HW, TY, HALF, true, false><<<p.B * (p.H / HW), nt, 0, s>>>(p);
    return;
  }
  // at most so many sequences are cut, and so many segments theirs; whole multiples of eight walks
  const int cut = min(p.B, p.T / p.SEG), segs = p.T / p.PIECE + cut;
  auto grid = [&](int walks) { return (walks + 7) / 8 * 8 * (p.H / HW); };
  chunk_walk_kernel<MODE, NT, V, HW, TY, HALF, false, true><<<grid(segs), nt, 0, s>>>(p);
  chunk_join_kernel<<<dim3(p.B, p.H, (p.V * p.N + 1023) / 1024), 256, 0, s>>>(p);
  chunk_walk_kernel<MODE, NT, V, HW, TY, HALF, true, true>
      <<<grid(p.B > kCounted ? p.B + segs : p.T / p.PIECE + p.B), nt, 0, s>>>(p);
}

// two heads of 64 columns that share their keys go through one workgroup: the keys' fragments
// are staged once for both
template <int MODE, int NT, typename TY>
void pick_v(const ChunkScanParams& p, hipStream_t s) {
  if constexpr (MODE == 1 && sizeof(TY) == 2) {
    // (which pieces have one part is fixed when the kernels are built: half of them, as the models turn half
    // of the entries or fewer; 8 x 2048 rows, 8 heads x 128 x 128: 176 us, 197 where all have three)
    if (p.rot_dims * 2 <= p.N) {
      if (p.V == 128) run<MODE, NT, 128, 1, TY, true>(p, s);
      else run<MODE, NT, 64, 1, TY, true>(p, s);
      return;
    }
  }
  if (p.V == 128) run<MODE, NT, 128, 1, TY>(p, s);
  else if (MODE == 0 && (p.H / p.KH) % 2 == 0) run<MODE, NT, 64, MODE == 0 ? 2 : 1, TY>(p, s);
  else run<MODE, NT, 64, 1, TY>(p, s);
}

template <int MODE, typename TY>
void pick(const ChunkScanParams& p, hipStream_t s) {
  if (p.N == 128) pick_v<MODE, 4, TY>(p, s);
  else pick_v<MODE, 2, TY>(p, s);
}

}  // namespace

bool chunk_scan_sizes(int V, int N) {
  return (V == 64 || V == 128) && (N == 64 || N == 128);
}

int chunk_scan_segment(int mode, int T, int B, int H, int V) {
  // Only the rows of all sequences are known here; which are long enough to be cut, and whether they
  // are, walked_whole() says.  Below kFill waves in all, long ones are cut.  Above, a step may be one
  // long prompt beside many short sequences or running rows (8 heads x 128 x 128: 64 rows and a prompt
  // of 2048 178 us in segments, 433 whole; 23 prompts of 100 and one of 5000 186, 998); where nothing
  // is cut, the two launches more take 5 us (24 prompts of 600: 187 -> 193; 40 of 900: 467 -> 476).  The
  // scan, whose many heads fill the chip with a few prompts, takes them only where the mean length
  // says that most sequences are short (64 heads x 128 x 64, 64 rows and a prompt of 2048: 263 us, 441
  // whole).
  const int64_t waves = (int64_t)B * H * (V / 32);
  if (waves < kFill) {
    if (T >= 1024 || T >= 384 * (int64_t)B) return 256;
    // Few short prompts, whose segments are of 64 rows, are cut from 129 rows on: the retention's from a mean
    // of 160 (8 heads x 128 x 128: a prompt of 160 rows 33 us either way, of 200 41.6 whole and 33.7 cut, of 350
    // 59.8 and 34.6; three of 256 50 and 41, four of 250 55 and 42), the scan's, whose two launches more weigh
    // more, of one or two prompts (64 heads x 128 x 64: one of 200 60.9 and 63, of 240 67.5 and 62.3, of 300 76
    // and 62.5, two of 256 73.4 and 68.3, three of 256 74.5 and 84; 128 heads: one of 256 71.7 and 79.8, of 350
    // 85.5 and 82).
    const bool longer = mode == 1 ? T >= 160 * (int64_t)B
                                  : waves <= 256 && T >= (waves <= 128 ? 240 : 320) * (int64_t)B;
    return longer && chunk_scan_piece(mode, T, B, H, V) == 64 ? 128 : 0;
  }
  return T - B >= 1024 && (mode == 1 || T < 256 * (int64_t)B) ? 256 : 0;
}

int chunk_scan_piece(int mode, int T, int B, int H, int V) {
  // A segment's chunks are a serial chain, 256 rows of them 40 us; where the step's segments would leave
  // SIMDs idle they are shorter.  Up to 1024 waves of the retention, one per SIMD (8 heads x 128 x 128:
  // a prompt of 400 rows 66 us in segments of 256, 36 of 64; of 2000 76 and 51 of 128; four of 1000 84
  // and 64 of 128, 69 of 64), 2048 of the scan, whose many heads make the steps coarse (64 heads x 128 x
  // 64: a prompt of 400 rows 74 and 47; two of 1000 113 and 87 of 128; one of 2000 86 and 90).
  const int64_t most = mode == 0 ? kScanWaves : kRetentionWaves;
  for (int piece = 64; piece < 256; piece *= 2)
    if (chunk_scan_segments(T, B, piece) * H * (V / 32) <= most) return piece;
  return 256;
}

int64_t chunk_scan_segments(int T, int B, int PIECE) {
  return few_long(T, B, PIECE) ? 2 * (int64_t)T / PIECE + 2 : (int64_t)T / PIECE + B;
}

void launch_chunk_scan(const ChunkScanParams& p, bool f32, hipStream_t s) {
  if (p.T <= 0 || p.B <= 0) return;
  if (p.mode == 0) {
    if (f32) pick<0, float>(p, s); else pick<0, bf16>(p, s);
  } else {
    if (f32) pick<1, float>(p, s); else pick<1, bf16>(p, s);
  }
}

}  // namespace akap_stream
