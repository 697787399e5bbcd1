// Varlen prefill attention on gfx950: the prompt run of vLLM 0.5.1's
// FlashAttention backend, flash_attn_varlen_func(q, k, v, cu_seqlens,
// cu_seqlens, max_seqlen, max_seqlen, scale, causal=True) (EXT), reached from
// aegaeon/aegaeon/worker.py:517-523 with the metadata of worker.py:652-711.
//
// Layout: q [T, Hq, D], k and v [T, Hkv, D], out [T, Hq, D] in 16-bit
// elements, any token stride, the heads of a token contiguous.  Sequence b
// holds tokens [cu_seqlens[b], cu_seqlens[b+1]); query i of a sequence attends
// to keys j <= i of the same sequence (all of them when not causal).
//
// Per 64-key tile and 32-query block of a wave:
//   S^T[64 keys x 32 queries] = K[64 x D] . Q^T[D x 32]   2 x D/16 MFMA 32x32x16
//     (A = K rows from LDS, B = the wave's queries, held in registers);
//   online softmax in fp32 in the exp2 domain: lane l holds query l & 31 and
//     16 of the 32 keys of a block (keys 8(i/4) + 4(l/32) + i%4 of
//     accumulator element i), its partner lane l ^ 32 the other 16;
//   O^T[D x 32] += V^T[D x 64] . P^T[64 x 32]             D/32 x 4 MFMA 32x32x16
//     with P rounded to 16 bits (as FlashAttention does) and taken straight
//     from the S^T accumulators: elements 8j .. 8j+7 of a lane are the keys of
//     k-step j, which are keys {4 hh .. 4 hh + 3, 8 + 4 hh .. 8 + 4 hh + 3} of
//     the step's 16 (hh = l / 32), so V^T's A operand holds those keys.
// Lazy rescaling as in the decode kernel: the reference max moves only when a
// tile's max exceeds it by more than 8 (log2 units).
//
// Two kernels share that arithmetic (their outputs are bit-identical); the
// host picks one by the batch's longest prompt:
//
// Long prompts (max_seqlen > kLongPrompt): ping-pong.  A workgroup of eight
// waves takes eight units of 32 queries and fills a CU; waves w and w + 4 share
// a SIMD, and the two halves of the workgroup run opposite phases between
// workgroup barriers.  Per key tile j a wave runs a matrix phase (S_j and the
// previous tile's O += V_{j-1}^T . P_{j-1}, 32 MFMAs at D = 128) and then a
// softmax phase (the VALU work that turns S_j into P_j); waves 4-7 start one
// phase later than waves 0-3, so on every SIMD one wave feeds the matrix core
// while the other runs its softmax.  K and V go from HBM straight into LDS
// (buffer loads with the LDS bit, no registers), V untransposed, and the
// P.V operands are read with gfx950's transposing LDS reads.
//
// Short prompts: three workgroups of four waves per CU that overlap each
// other's latencies, softmax and matrix work unordered; K and V reach LDS the
// same way.  (With short prompts the ping-pong workgroup's start-up costs more
// than the phase overlap gains, four-wave against ping-pong: 16 x 512 54.4 and
// 63.9 us, 8 x 1024 78.9 and 83.2; from 2048 tokens on the overlap wins: 4 x
// 2048 131.6 and 130.1, 2 x 4096 270 and 252, 1 x 8192 464 and 423.)
//
// Wave units, both kernels: the work of a (sequence, kv head) pair is cut into
// units of 32 queries of one query head, unit u = query block u / G of the
// head u % G of the kv head's G; a workgroup's waves take consecutive units.
// They share the pair's K and V tiles, and since the heads of one query block
// are neighbours, a causal workgroup's waves need (almost) the same keys and a
// short or ragged prompt leaves no wave without queries but its last.  (A
// workgroup of 128 or 256 queries of one head idled its early waves on the
// diagonal tiles and its late ones past the end: 48 prompts of 25-766 tokens
// 111.1 -> 94.0 us, 4 x 2048 of 28/4 heads 151.5 -> 142.4.)
//
// Work order, both kernels: a job is a tile of a pair's units, and the jobs
// run with the tile index slowest, in decreasing order, so the most expensive
// tiles (the last of each sequence) are dispatched first; within a tile index
// the pairs follow each other, kv heads fastest.  The hardware deals workgroup
// i to XCD i % 8: with a multiple of 8 pairs of one length, XCD x runs every
// tile of the x-th eighth of the pairs, whose K and V its L2 keeps (1 x 4096
// tokens of 40 heads: 193.5 us against 197.4 with the pairs dealt in turn), and
// fewer pairs spread evenly over the XCDs.  Prompts of different lengths: each
// wave finds job i among the tiles that exist (pick_job), so no workgroup is
// launched for an empty tile (48 prompts of 25-766 tokens: 5900 of 9200
// workgroups were).  More of them than a wave searches, and fewer tokens than
// 90% of the bound: the pairs are dealt in turn, as an eighth of them could be
// all the long ones (320 prompts of 16-1024 tokens sorted by length, 32/4
// heads: eighths 1189 us, in turn 418; unsorted 472 and 429; of one length 341
// and 349).
//
// Times in this file's comments are before and after in one process on one GPU;
// GPUs differ by up to 4%, and the first 20 ms after a pause run slower.
#include <algorithm>
#include <cmath>

#include "aegkv_internal.h"

namespace aegkv {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
typedef __attribute__((address_space(3))) void lds_void;

constexpr int kXcds = 8;                     // XCDs of an MI355X (gfx950)
constexpr int kPfKTile = 64;                 // keys per step
constexpr float kPfRescaleSlack = 8.f;
constexpr int kLongPrompt = 1536;            // longer prompts take the ping-pong kernel
// short-prompt kernel: four waves
constexpr int kShortThreads = 256;
constexpr int kShortWaves = kShortThreads / 64;
// ping-pong kernel: eight waves
constexpr int kLongWaves = 8;
constexpr int kLongThreads = 64 * kLongWaves;
constexpr int kUnitQ = 32;       // queries of a wave unit
constexpr int kCompactSets = 4;  // 64-sequence sets a wave searches for its job

template <int DT>
struct PfOps;

template <>
struct PfOps<AEGKV_DTYPE_BF16> {
  static __device__ __forceinline__ f32x16 mfma(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
  // two floats to two 16-bit values, round to nearest even (one instruction)
  static __device__ __forceinline__ uint32_t pack(float x, float y) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{x, y}, bf16x2));
  }
};

template <>
struct PfOps<AEGKV_DTYPE_FP16> {
  static __device__ __forceinline__ f32x16 mfma(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint32_t pack(float x, float y) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{x, y}, f16x2));
  }
};

// max(a, b, c) through the compiler's own max, never inline asm.  The
// scores are MFMA results, and a VALU read of an MFMA result needs wait states
// that only the compiler's hazard tracking inserts: it does not see the
// operands of an inline-asm v_max3_f32.  That form read unfinished scores on
// unmasked key tiles whenever the matrix core ran late, which showed as
// run-to-run output differences (one ulp, in ~7% of rows) once the four-wave
// kernel's workgroups were dealt to CUs in another order.  The compiler's max
// costs a few canonicalising v_max_f32 (0-3% per call).
__device__ __forceinline__ float max3(float a, float b, float c) {
  return __builtin_fmaxf(__builtin_fmaxf(a, b), c);
}

// floor(n / d) for 0 <= n < 2^31 by a multiplication (mul = floor(2^(31 + shift)
// / d) + 1, shift = ceil(log2 d): 2^(31 + shift) < mul * d <= 2^(31 + shift) +
// 2^shift).  A division by a number the compiler does not know is some twenty
// vector instructions; a workgroup's start has half a dozen of them.
struct FastDiv {
  uint32_t mul, shift;
  __device__ __forceinline__ int div(int n) const {
    return (int)(__umulhi(2u * (uint32_t)n, mul) >> shift);
  }
};
inline FastDiv fast_div(int32_t d) {  // 1 <= d < 2^31
  FastDiv f;
  f.shift = 0;
  while ((1ll << f.shift) < d) ++f.shift;
  f.mul = (uint32_t)((((uint64_t)1 << (31 + f.shift)) / (uint64_t)d) + 1);
  return f;
}

struct PrefillArgs {
  const uint8_t* q;
  const uint8_t* k;
  const uint8_t* v;
  uint8_t* out;
  int64_t q_tok_b, k_tok_b, v_tok_b, o_tok_b;  // byte strides per token
  const int32_t* cu_seqlens;                   // [batch + 1], device
  int32_t token_bound;                         // min(total tokens, INT32_MAX)
  int32_t batch, n_kv_heads, group, max_seqlen, causal;
  FastDiv by_heads, by_group, by_pairs;        // n_kv_heads, group, n_pairs
  int32_t n_pairs;                             // batch * n_kv_heads
  int32_t n_tiles;                             // tiles of a pair of max_seqlen tokens
  int32_t compact;                             // jobs numbered over existing tiles only
  int32_t per_xcd;                             // else: pairs per XCD (0: dealt in turn)
  float scale_log2;                            // |softmax scale| * log2(e), > 0 (1 for 0)
  int32_t scale_sign;                          // of the scale: 1, -1 or 0
};

// The wave's state for its 32 queries: lane (col = l & 31, hh = l / 32) holds
// query q0 + col and, of the O^T accumulators, head dims 32 db + 8 g + 4 hh ..
// + 3 in element 4 g .. 4 g + 3 of o[db].
template <int DT, int D>
struct WaveState {
  static constexpr int KS = D / 16;  // k-steps of K.Q^T
  static constexpr int DB = D / 32;  // 32-row blocks of O^T
  u32x4 qv[KS];                      // Q^T operand: dims 16 ks + 8 hh .. +7
  f32x16 o[DB];
  float m, lsum;

  __device__ __forceinline__ void init(const PrefillArgs& a, int h, int64_t s0, int len, int qi,
                                       int hh) {
    const uint8_t* qp =
        a.q + (s0 + min(qi, len - 1)) * a.q_tok_b + ((int64_t)h * D + 8 * hh) * 2;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)  // queries past the end: 0
      qv[ks] = qi < len ? *reinterpret_cast<const u32x4*>(qp + 32 * ks) : u32x4{0, 0, 0, 0};
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[db][i] = 0.f;
    m = -INFINITY;
    lsum = 0.f;
  }

  // The softmax takes a maximum of raw scores and masks them with -inf, so its
  // scale is positive; another one's sign goes into the loaded queries, where
  // it is exact (scale 0: no query, every score 0).  Kernels of their own
  // (SIGNED) do that: a test of the scale here had the compiler wait for the
  // queries as they are loaded.
  __device__ __forceinline__ void sign_queries(const PrefillArgs& a) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        qv[ks][i] = a.scale_sign < 0 ? qv[ks][i] ^ 0x80008000u : 0u;
  }

  // S^T of a 64-key tile from K rows at kp (pitch KPITCH bytes, this lane's
  // row and 16-byte column already added); the two 32-key blocks alternate so
  // that neighbouring MFMAs are independent.  `ahead` LDS reads are kept in
  // flight ahead of the MFMA that uses them.
  template <int KPITCH, int AHEAD>
  __device__ __forceinline__ void qk(const uint8_t* kp, f32x16 (&s)[2]) const {
#pragma unroll
    for (int sb = 0; sb < 2; ++sb)
#pragma unroll
      for (int i = 0; i < 16; ++i) s[sb][i] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int sb = 0; sb < 2; ++sb)
        s[sb] = PfOps<DT>::mfma(*reinterpret_cast<const u32x4*>(kp + 32 * sb * KPITCH + 32 * ks),
                                qv[ks], s[sb]);
    if (AHEAD > 0) {
      __builtin_amdgcn_sched_group_barrier(0x100, AHEAD, 0);  // LDS reads
#pragma unroll
      for (int i = 0; i < 2 * KS - AHEAD; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);    // one MFMA
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);    // the next read
      }
      __builtin_amdgcn_sched_group_barrier(0x008, AHEAD, 0);
    }
  }

  // -inf where a key of the tile at k0 is past the end or (causal) after the
  // query; only the tiles that reach past the wave's first query wq0 or the
  // end need it.  One comparison with a constant per score: the lane's last key
  // is counted from its first score's.  (Two comparisons of a key number per
  // score, and a first tile that rescaled its zero sums: 48 prompts of 25-766
  // tokens 69.9 us, so 68.8; 4 x 2048 133.2 and 129.0; 1 x 8192 436 and 433.)
  __device__ __forceinline__ void mask(f32x16 (&s)[2], int k0, int wq0, int qi, int len,
                                       int causal, int hh) const {
    if ((causal && k0 + kPfKTile - 1 > wq0) || k0 + kPfKTile > len) {
      const int last = (causal ? min(qi, len - 1) : len - 1) - k0 - 4 * hh;
#pragma unroll
      for (int sb = 0; sb < 2; ++sb)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          s[sb][i] = last >= 32 * sb + 8 * (i >> 2) + (i & 3) ? s[sb][i] : -INFINITY;
    }
  }

  // online softmax of a masked S^T tile into the P^T operands of its four
  // 16-key steps
  // (`first`: the wave's first tile, whose sums are still zero)
  __device__ __forceinline__ void softmax(f32x16 (&s)[2], u32x4 (&pb)[4], float scale_log2,
                                          bool first) {
    // raw-score max (the scale is positive) over four chains of triples: a lone
    // pair of scores would be canonicalised first (28 instructions, now 16:
    // 1 x 8192 435.5 -> 427.0 us, 4 x 2048 131.3 -> 128.9)
    float c4[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const f32x16& x = s[c >> 1];
      const int e = 8 * (c & 1);
      c4[c] = max3(x[e], x[e + 1], x[e + 2]);
    }
#pragma unroll
    for (int k = 3; k < 7; k += 2)
#pragma unroll
      for (int c = 0; c < 4; ++c)
        c4[c] = max3(c4[c], s[c >> 1][8 * (c & 1) + k], s[c >> 1][8 * (c & 1) + k + 1]);
    const float d0 = max3(c4[0], s[0][7], s[0][15]), d1 = max3(c4[1], s[1][7], s[1][15]);
    float bm = fmaxf(max3(d0, c4[2], c4[3]), d1);
    // the partner lane's max (same query), exchanged between the wave's
    // halves in registers: one v_permlane32_swap instead of the LDS round trip
    // of a shuffle.  (Both kernels, 20 repeated calls each, also with two
    // unsynchronised workgroups per CU: bit-identical outputs, and bit-identical
    // to the shuffle; the four-wave kernel 0-2% faster with it.)
    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(bm), __float_as_uint(bm),
                                                     false, false);
    bm = fmaxf(fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1])), bm) * scale_log2;
    if (first) {
      m = fmaxf(m, bm);
    } else if (__builtin_amdgcn_ballot_w64(bm > m + kPfRescaleSlack)) {
      const float mn = fmaxf(m, bm);
      const float alpha = __builtin_amdgcn_exp2f(m - mn);  // 0 while m = -inf
      lsum *= alpha;
#pragma unroll
      for (int db = 0; db < DB; ++db) o[db] *= alpha;
      m = mn;
    }
    const float nms = m == -INFINITY ? 0.f : -m;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      const int sb = kk >> 1, base = 8 * (kk & 1);
      uint32_t pw[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float p0 =
            __builtin_amdgcn_exp2f(__builtin_fmaf(s[sb][base + 2 * j], scale_log2, nms));
        const float p1 =
            __builtin_amdgcn_exp2f(__builtin_fmaf(s[sb][base + 2 * j + 1], scale_log2, nms));
        lsum += p0 + p1;
        pw[j] = PfOps<DT>::pack(p0, p1);
      }
      pb[kk] = u32x4{pw[0], pw[1], pw[2], pw[3]};
    }
  }

  // normalise and store the wave's outputs (queries past the end: none).  A
  // lane holds 8-byte pieces of one row, so they go through LDS at `x` (the
  // wave's own 32 rows of D, 16-byte chunk c of row r at c ^ r % chunks, which
  // keeps both sides off each other's banks) and leave as whole rows.  (Straight from the
  // registers, 32 rows x 16 bytes per store, a wave's stores took 2.2 us of a
  // 20 us job: 48 prompts of 25-766 tokens 82.0 us, so 70.1; 4 x 2048 141.7
  // and 131.3; 1 x 8192 452 and 435.)
  __device__ __forceinline__ void store(const PrefillArgs& a, uint8_t* x, int h, int64_t s0,
                                        int len, int wq0) {
    constexpr int RB = D * 2, CPR = D / 8, RPI = 64 / CPR;  // bytes, chunks per row; rows per store
    const int lane = threadIdx.x & 63, col = lane & 31, hh = lane >> 5;
    const float lt = lsum + __shfl_xor(lsum, 32);
    const float inv = 1.f / lt;
    uint8_t* xw = x + col * RB + 8 * hh;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x16& r = o[db];
        *reinterpret_cast<u32x2*>(xw + ((4 * db + g) ^ (col % CPR)) * 16) =
            u32x2{PfOps<DT>::pack(r[4 * g] * inv, r[4 * g + 1] * inv),
                  PfOps<DT>::pack(r[4 * g + 2] * inv, r[4 * g + 3] * inv)};
      }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the wave's own writes
    const int row = lane / CPR, pos = lane % CPR;
    uint8_t* op = a.out + (s0 + wq0) * a.o_tok_b + (int64_t)h * RB;
#pragma unroll
    for (int i = 0; i < 32 / RPI; ++i) {
      const int r = RPI * i + row;
      const u32x4 v = *reinterpret_cast<const u32x4*>(x + 1024 * i + 16 * lane);
      if (wq0 + r < len)
        *reinterpret_cast<u32x4*>(op + r * a.o_tok_b + (pos ^ (r % CPR)) * 16) = v;
    }
  }
};

// The clamped token range of sequence b.
__device__ __forceinline__ void seq_range(const PrefillArgs& a, int b, int& s0, int& len) {
  const int c0 = a.cu_seqlens[b], c1 = a.cu_seqlens[b + 1];
  s0 = min(max(c0, 0), a.token_bound);
  len = min(min(max(c1, s0), a.token_bound) - s0, a.max_seqlen);
}

// Sum over the wave's lanes, uniform.
__device__ __forceinline__ int wave_sum(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);  // row_shr 1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);  // row_shr 2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);  // row_shr 4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);  // row_shr 8
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, true);  // row_bcast 15, rows 1 and 3
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, true);  // row_bcast 31, rows 2 and 3
  return __builtin_amdgcn_readlane(x, 63);
}

// Tiles of W units of a sequence of n tokens.
template <int W>
__device__ __forceinline__ int tiles_of(const PrefillArgs& a, int n) {
  return ((n + kUnitQ - 1) / kUnitQ * a.group + W - 1) / W;
}

// Job i among the tiles that exist, for up to 64 * SETS sequences (see
// pick_job): a binary search for its tile index, then its rank among the
// sequences that have that tile.
template <int W, int SETS>
__device__ __forceinline__ bool pick_compact(const PrefillArgs& a, uint32_t i, int& kvh, int& s0,
                                             int& len, int& u0) {
  const int lane = threadIdx.x & 63;
  int st[SETS], ln[SETS], t[SETS];
#pragma unroll
  for (int k = 0; k < SETS; ++k) {
    const int b = 64 * k + lane;
    seq_range(a, min(b, a.batch - 1), st[k], ln[k]);
    t[k] = b < a.batch ? tiles_of<W>(a, ln[k]) : 0;
  }
  auto jobs_from = [&](int tile) -> uint32_t {  // jobs of tile index >= tile
    int x = 0;
#pragma unroll
    for (int k = 0; k < SETS; ++k) x += max(t[k] - tile, 0);
    return (uint32_t)wave_sum(x) * (uint32_t)a.n_kv_heads;
  };
  if (jobs_from(0) <= i) return false;
  int lo = 0, hi = a.n_tiles;  // jobs_from(lo) > i >= jobs_from(hi)
  uint32_t after = 0;          // jobs_from(hi)
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    const uint32_t n = jobs_from(mid);
    if (n > i) lo = mid;
    else { hi = mid; after = n; }
  }
  int rank = a.by_heads.div((int)(i - after));
  kvh = (int)(i - after) - rank * a.n_kv_heads;
  u0 = lo * W;
  // the rank-th sequence with a tile `lo`
  s0 = len = 0;
#pragma unroll
  for (int k = 0; k < SETS; ++k) {
    const uint64_t mask = __builtin_amdgcn_ballot_w64(t[k] > lo);
    const int c = __builtin_popcountll(mask);
    if (rank >= 0 && rank < c) {
      const int at = (int)__builtin_amdgcn_mbcnt_hi(
          (uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
      const uint64_t hit = __builtin_amdgcn_ballot_w64(t[k] > lo && at == rank);
      const int src = __builtin_ctzll(hit);
      s0 = __builtin_amdgcn_readlane(st[k], src);
      len = __builtin_amdgcn_readlane(ln[k], src);
    }
    rank -= c;
  }
  return true;
}

// The job of workgroup blockIdx.x of W waves (uniform): sequence range, kv
// head and first unit.  Returns false when the tile is empty or there are
// fewer jobs.  What bounds a short prompt's start is the number of
// instructions every wave spends here: one set of sequences is searched when one
// holds them, lengths stay in 32 bits, and nothing is divided by the hardware's
// reciprocal (200 prompts of 4-300 tokens 64.0 -> 62.1 us, 16 x 512 57.2 ->
// 55.5, 48 prompts of 25-766 tokens 70.6 -> 69.5).
template <int W>
__device__ __forceinline__ bool pick_job(const PrefillArgs& a, int& kvh, int& s0, int& len,
                                         int& u0) {
  const uint32_t i = blockIdx.x;
  if (a.compact)
    return a.batch <= 64 ? pick_compact<W, 1>(a, i, kvh, s0, len, u0)
                         : pick_compact<W, kCompactSets>(a, i, kvh, s0, len, u0);
  // every tile of the bound: tile n_tiles - 1 of each pair first
  const int k = a.by_pairs.div((int)i);
  int r = (int)i - k * a.n_pairs;
  if (a.per_xcd) r = r % kXcds * a.per_xcd + r / kXcds;
  const int b = a.by_heads.div(r);
  kvh = r - b * a.n_kv_heads;
  seq_range(a, b, s0, len);
  const int tile = a.n_tiles - 1 - k;
  u0 = tile * W;
  return tile < tiles_of<W>(a, len);
}

// ---------------------------------------------------------------- short prompts
// Units [u0, u0 + 4) of kv head kvh of the sequence at token s0 with len
// tokens.  K and V tiles go from HBM straight into LDS (loads with the LDS bit)
// and V's operands are read with the transposing LDS reads, so a workgroup
// holds 48 KiB of LDS (two K stages, one V stage) and no staging registers,
// and three of them share a CU: a prompt of a few key tiles is a chain of
// latencies (job, first tiles, stores), which only other workgroups hide.
// (Two per CU with K and V staged through registers and V transposed on the way
// into LDS: 48 prompts of 25-766 tokens 94.0 us, 8 x 1024 95.5, 16 x 512 69.0;
// this 84.5, 87.6, 62.8.)
// Rows are stored unpadded with their 16-byte chunks permuted by the row
// (the loads pick the chunk, the LDS position is the lane's): K chunk c of row
// r at c ^ (r % 16) at D = 128, V chunk c at c ^ 4 (r % 4), so the 16 rows of a
// K read and the 4 rows of a transposing V read hit distinct banks.
template <int DT, int D, bool SIGNED>
__device__ __forceinline__ void attend_short(const PrefillArgs& a, uint8_t* lds, int kvh,
                                             int64_t s0, int len, int u0) {
  using E = PfOps<DT>;
  using W = WaveState<DT, D>;
  constexpr int RB = D * 2;                     // bytes per row
  constexpr int T_BYTES = kPfKTile * RB;        // bytes per tile
  constexpr int DB = W::DB;
  constexpr int CPR = D / 8;                    // 16-byte chunks per row
  constexpr int RPI = 64 / CPR;                 // rows per load instruction
  constexpr int NI = kPfKTile / (RPI * kShortWaves);  // load instructions per wave and tile
  const int kv_end = a.causal ? min(len, a.by_group.div(u0 + kShortWaves - 1) * kUnitQ + kUnitQ) : len;
  const int n_kt = (kv_end + kPfKTile - 1) / kPfKTile;

  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);  // uniform: the tile tests below branch
  const int col = lane & 31, hh = lane >> 5;
  const int wb = a.by_group.div(u0 + w);        // the wave's query block
  const int h = kvh * a.group + (u0 + w - wb * a.group);
  const int wq0 = wb * kUnitQ;                  // the wave's first query
  const int qi = wq0 + col;                     // this lane's query, relative to the sequence

  // Load instruction ii of wave w covers rows RPI (w + 4 ii) .. of a tile, lane
  // l the chunk stored at byte 16 l of them; the permutations depend on the
  // lane and wave only (rows 4 RPI apart permute alike).
  const int lrow = RPI * w + lane / CPR, lpos = lane % CPR;
  const int kch = D == 128 ? lpos ^ (lrow & 15) : lpos ^ ((lrow >> 1) & 7);
  const int vch = D == 128 ? lpos ^ ((lrow & 3) << 2) : lpos ^ (((lrow >> 1) & 1) << 2);
  const uint8_t* kbase = a.k + s0 * a.k_tok_b + (int64_t)kvh * RB + kch * 16;
  const uint8_t* vbase = a.v + s0 * a.v_tok_b + (int64_t)kvh * RB + vch * 16;
  auto dma = [&](const uint8_t* base, int64_t tok_b, int kt, uint8_t* stage) {
#pragma unroll
    for (int ii = 0; ii < NI; ++ii) {
      // rows past the sequence re-read its last one: their scores are masked,
      // their weights 0
      const int row = min(kt * kPfKTile + lrow + kShortWaves * RPI * ii, len - 1);
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)(base + row * tok_b),
          (lds_void*)(stage + (w + kShortWaves * ii) * 1024), 16, 0, 0);
    }
  };
  auto dma_k = [&](int kt) { dma(kbase, a.k_tok_b, kt, lds + (kt & 1) * T_BYTES); };
  auto dma_v = [&](int kt) { dma(vbase, a.v_tok_b, kt, lds + 2 * T_BYTES); };
  dma_k(0);
  W st;
  st.init(a, h, s0, len, qi, hh);
  dma_v(0);

  // K operand: row col (+ 32 sb), chunk 2 ks + hh
  const int kx = D == 128 ? (hh ^ (col & 15)) * 16 : (hh ^ ((col >> 1) & 7)) * 16;
  auto qk = [&](int kt, f32x16 (&s)[2]) {
    const uint8_t* kp = lds + (kt & 1) * T_BYTES + col * RB;
#pragma unroll
    for (int sb = 0; sb < 2; ++sb)
#pragma unroll
      for (int i = 0; i < 16; ++i) s[sb][i] = 0.f;
#pragma unroll
    for (int ks = 0; ks < W::KS; ++ks)
#pragma unroll
      for (int sb = 0; sb < 2; ++sb)
        s[sb] = E::mfma(*reinterpret_cast<const u32x4*>(kp + (kx ^ (32 * ks)) + 32 * sb * RB),
                        st.qv[ks], s[sb]);
  };
  // V operand (see the long kernel's transposing reads): lane (G, s) reads 4
  // dims 32 db + 16 (G & 1) + 4 (s % 4) .. + 3 of key 4 (G >> 1) + s / 4
  // (+ 16 kk, + 8), whose chunk's bit 2 (and 3) are permuted
  const int vG = lane >> 4, vs = lane & 15;
  const int vkey = 4 * (vG >> 1) + (vs >> 2);
  const int vx = 64 * (D == 128 ? vkey & 3 : (vkey >> 1) & 1);
  const uint8_t* vp =
      lds + 2 * T_BYTES + vkey * RB + (2 * (vG & 1) + ((vs & 3) >> 1)) * 16 + 8 * (vs & 1);
  auto pv = [&](const u32x4 (&pb)[4]) {
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        const uint8_t* x = vp + (vx ^ (64 * db)) + 16 * kk * RB;
        const u32x2 lo = __builtin_bit_cast(
            u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)x));
        const u32x2 hi = __builtin_bit_cast(
            u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(x + 8 * RB)));
        st.o[db] = E::mfma(u32x4{lo[0], lo[1], hi[0], hi[1]}, pb[kk], st.o[db]);
      }
  };
  auto mine = [&](int kt) {  // the wave has queries that need tile kt (uniform)
    return wq0 < len && (!a.causal || kt * kPfKTile <= wq0 + kUnitQ - 1);
  };

  // Tile kt: K_{kt+1} and V_kt are loaded while S_kt and its softmax are
  // computed; they are waited for before the barrier that starts P.V.  V_kt's
  // stage is free once every wave is past the P.V of tile kt - 1 (the barrier at
  // the top), K_{kt+1}'s since the S of tile kt - 1.
  // K_0 (the loads before V_0's), for every wave's reads after the barrier.  The
  // queries' own wait is the compiler's, in front of their first MFMA; they are
  // loaded under a condition, so it is for every load in flight, V_0's and
  // K_1's too.  (Queries used right here, which put that wait before K_1's
  // loads: 64 x 128 36.6 -> 46.0 us, 200 prompts of 4-300 tokens 60.2 -> 68.6,
  // others 0-2% slower.)
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NI) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  if constexpr (SIGNED) st.sign_queries(a);
  for (int kt = 0; kt < n_kt; ++kt) {
    if (kt > 0) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this wave's V reads
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      dma_v(kt);
    }
    if (kt + 1 < n_kt) dma_k(kt + 1);
    u32x4 pb[4];
    if (mine(kt)) {
      f32x16 sc[2];
      qk(kt, sc);
      st.mask(sc, kt * kPfKTile, wq0, qi, len, a.causal, hh);
      st.softmax(sc, pb, a.scale_log2, kt == 0);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (mine(kt)) pv(pb);
  }
  // the K stages: every wave is past its last read of them
  static_assert(kShortWaves * kUnitQ <= 2 * kPfKTile, "the outputs fit the K stages");
  st.store(a, lds + w * (kUnitQ * RB), h, s0, len, wq0);
}

template <int DT, int D, bool SIGNED>
__global__ __launch_bounds__(kShortThreads, 3) void prefill_short_kernel(PrefillArgs a) {
  // two K stages, then one V stage
  __shared__ __align__(16) uint8_t lds[3 * kPfKTile * D * 2];
  int kvh, s0, len, u0;
  if (!pick_job<kShortWaves>(a, kvh, s0, len, u0)) return;  // uniform, before any barrier
  attend_short<DT, D, SIGNED>(a, lds, kvh, s0, len, u0);
}

// ----------------------------------------------------------------- long prompts
// Units [u0, u0 + 8) of kv head kvh of the sequence at token s0 with len
// tokens, ping-pong between the workgroup's halves.
template <int DT, int D, bool SIGNED>
__device__ __forceinline__ void attend_long(const PrefillArgs& a, uint8_t* lds, int kvh,
                                            int64_t s0, int len, int u0) {
  using E = PfOps<DT>;
  using W = WaveState<DT, D>;
  constexpr int KPITCH = D * 2 + 16;            // bytes per K row in LDS
  constexpr int K_BYTES = kPfKTile * KPITCH;
  // V rows stay untransposed at 2D + 64 bytes: the transposing reads of four
  // consecutive keys (64 bytes of each) then hit distinct banks
  constexpr int VPITCH = D * 2 + 64;
  constexpr int V_BYTES = kPfKTile * VPITCH;
  constexpr int DB = W::DB;
  constexpr int CPR = D / 8;                    // 16-byte chunks of a row's data
  constexpr int CK = KPITCH / 16, CV = VPITCH / 16;  // chunks per stored row
  constexpr int NK = (CK + kLongWaves - 1) / kLongWaves;
  constexpr int NV = (CV + kLongWaves - 1) / kLongWaves;
  constexpr uint32_t kPad = 0xFFFFFFF0u;        // an offset out of every range
  const int kv_end = a.causal ? min(len, a.by_group.div(u0 + kLongWaves - 1) * kUnitQ + kUnitQ) : len;
  const int n_kt = (kv_end + kPfKTile - 1) / kPfKTile;

  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);  // uniform: the tile tests below branch
  const int half = w >> 2;           // 0: waves 0-3, 1: waves 4-7 (one phase later)
  const int col = lane & 31, hh = lane >> 5;
  const int wb = a.by_group.div(u0 + w);        // the wave's query block
  const int h = kvh * a.group + (u0 + w - wb * a.group);
  const int wq0 = wb * kUnitQ;                  // the wave's first query
  const int qi = wq0 + col;                     // this lane's query, relative to the sequence
  // the wave's last key tile: causal waves stop at their last query's tile; a
  // wave past the end of the sequence attends to nothing (-1)
  const int jw = wq0 >= len ? -1
                 : a.causal ? min(n_kt - 1, min(wq0 + 31, len - 1) / kPfKTile)
                            : n_kt - 1;
  W st;
  st.init(a, h, s0, len, qi, hh);

  // Direct HBM -> LDS staging through raw buffer ranges over the sequence's K
  // and V rows of kv head kvh, ending at the last row's last byte.  Lane l of
  // a load instruction writes LDS bytes [16 l, 16 l + 16) after the
  // instruction's base, so instruction i of a tile covers stored chunks
  // [64 i, 64 i + 64); a row's pad chunks and rows past the sequence end get
  // an out-of-range offset, for which the hardware writes zeros and reads
  // nothing (zero V keeps P.V finite; those keys' scores are masked).
  const __amdgpu_buffer_rsrc_t krs =
      byte_range(a.k + s0 * a.k_tok_b + (int64_t)kvh * D * 2,
                 (uint32_t)((int64_t)(len - 1) * a.k_tok_b + D * 2));
  const __amdgpu_buffer_rsrc_t vrs =
      byte_range(a.v + s0 * a.v_tok_b + (int64_t)kvh * D * 2,
                 (uint32_t)((int64_t)(len - 1) * a.v_tok_b + D * 2));
  const uint32_t k_tok = (uint32_t)a.k_tok_b, v_tok = (uint32_t)a.v_tok_b;
  // instruction ii of wave w: K instruction w + 8 ii, V instruction
  // (w + 7) % 8 + 8 ii (the spare ones of a tile go to different waves); the
  // lane's byte offset within a tile
  uint32_t koffs[NK], voffs[NV];
#pragma unroll
  for (int ii = 0; ii < NK; ++ii) {
    const int c = (w + kLongWaves * ii) * 64 + lane, row = c / CK, ch = c % CK;
    koffs[ii] = ch < CPR ? row * k_tok + ch * 16 : kPad;
  }
#pragma unroll
  for (int ii = 0; ii < NV; ++ii) {
    const int c = (((w + kLongWaves - 1) % kLongWaves) + kLongWaves * ii) * 64 + lane;
    const int row = c / CV, ch = c % CV;
    voffs[ii] = ch < CPR ? row * v_tok + ch * 16 : kPad;
  }
  auto dma_k = [&](int kt) {
    const uint32_t t0 = kt * kPfKTile * k_tok;
#pragma unroll
    for (int ii = 0; ii < NK; ++ii) {
      const int i = w + kLongWaves * ii;  // uniform
      if (i < CK)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            krs, (lds_void*)(lds + (kt & 1) * K_BYTES + i * 1024), 16,
            koffs[ii] == kPad ? kPad : koffs[ii] + t0, 0, 0, 0);
    }
  };
  auto dma_v = [&](int kt) {
    const uint32_t t0 = kt * kPfKTile * v_tok;
#pragma unroll
    for (int ii = 0; ii < NV; ++ii) {
      const int i = (w + kLongWaves - 1) % kLongWaves + kLongWaves * ii;  // uniform
      if (i < CV)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            vrs, (lds_void*)(lds + 2 * K_BYTES + (kt & 1) * V_BYTES + i * 1024), 16,
            voffs[ii] == kPad ? kPad : voffs[ii] + t0, 0, 0, 0);
    }
  };
  // Transposing V reads (ds_read_b64_tr_b16: in each 16-lane group, result
  // lane j element k is element j % 4 of source lane 4k + j / 4).  Lane
  // (group G = lane / 16, s = lane % 16) reads 4 dims 16 (G & 1) + 4 (s % 4)
  // .. + 3 of key 4 (G >> 1) + s / 4; after the transpose it holds dim
  // 16 (G & 1) + s of keys 4 (G >> 1) .. + 3 (+ 16 kk, + 8 for elements 4-7,
  // + 32 db for the dims): the A operand of O^T = V^T . P^T.
  const int vG = lane >> 4, vs = lane & 15;
  const int vtr_off = (4 * (vG >> 1) + (vs >> 2)) * VPITCH + (16 * (vG & 1) + 4 * (vs & 3)) * 2;
  auto pv = [&](int kt, const u32x4 (&pb)[4]) {
    const uint8_t* vb = lds + 2 * K_BYTES + (kt & 1) * V_BYTES + vtr_off;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_s16x4*)(vb + 16 * kk * VPITCH + 64 * db)));
        const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_s16x4*)(vb + (16 * kk + 8) * VPITCH + 64 * db)));
        st.o[db] = E::mfma(u32x4{lo[0], lo[1], hi[0], hi[1]}, pb[kk], st.o[db]);
      }
    // two reads per MFMA, four MFMAs ahead
    __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
    for (int i = 0; i < 4 * DB - 2; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
  };
  auto qk = [&](int kt, f32x16 (&s)[2]) {
    st.template qk<KPITCH, 2>(lds + (kt & 1) * K_BYTES + col * KPITCH + 16 * hh, s);
  };
  auto softmax = [&](int kt, f32x16 (&s)[2], u32x4 (&pb)[4]) {
    st.mask(s, kt * kPfKTile, wq0, qi, len, a.causal, hh);
    st.softmax(s, pb, a.scale_log2, kt == 0);
  };
  // K_{j+1} and V_j (read from slot 2j + 2 on) are loaded in slot 2j, whose
  // stages were last read in slot 2j - 1
  auto stage = [&](int j) {
    if (j + 1 < n_kt) dma_k(j + 1);
    if (j < n_kt) dma_v(j);
  };

  // Slots between workgroup barriers.  Phase p of a wave runs in slot
  // p + half: even p = 2j is the matrix phase of tile j (S_j, then the P.V of
  // tile j - 1; p = 2 n_kt only the last P.V), odd p = 2j + 1 its softmax.
  // Tile j's K is read in slots 2j and 2j + 1, its V in slots 2j + 2 and
  // 2j + 3.  Each half runs its own loop, so S_j lives within one iteration and
  // only P and O are carried; both halves pass 2 n_kt + 2 barriers after the
  // prologue's.  The barriers are plain s_barrier: a slot's LDS reads are
  // consumed by its own MFMAs before its barrier, and the direct loads issued
  // at the end of slot 2j are waited for (vmcnt) only before the barrier that
  // ends slot 2j + 1, so they land while slot 2j + 1 computes.
#define PF_BARRIER() \
  do { asm volatile("" ::: "memory"); __builtin_amdgcn_s_barrier(); asm volatile("" ::: "memory"); } while (0)
#define PF_BARRIER_LOADED()                              \
  do {                                                   \
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     \
    __builtin_amdgcn_s_barrier();                        \
    asm volatile("" ::: "memory");                       \
  } while (0)
  u32x4 pb[4];
  dma_k(0);
  __syncthreads();  // waits for K_0 and the queries
  if constexpr (SIGNED) st.sign_queries(a);
  if (half == 0) {
    for (int j = 0; j < n_kt; ++j) {
      f32x16 sc[2];  // slot 2j
      if (j <= jw) qk(j, sc);
      if (j >= 1 && j - 1 <= jw) pv(j - 1, pb);
      stage(j);
      PF_BARRIER();
      if (j <= jw) softmax(j, sc, pb);  // slot 2j + 1
      PF_BARRIER_LOADED();
    }
    if (n_kt - 1 <= jw) pv(n_kt - 1, pb);  // slot 2 n_kt
    PF_BARRIER();
    static_assert(kLongWaves / 2 * kUnitQ * D * 2 <= 2 * K_BYTES, "a half's outputs fit");
    // slot 2 n_kt + 1: the outputs, through the K stages (last read in slot
    // 2 n_kt - 1), while the other half runs its last P.V
    st.store(a, lds + w * (kUnitQ * D * 2), h, s0, len, wq0);
    PF_BARRIER();
  } else {
    stage(0);  // slot 0: idle
    PF_BARRIER();
    for (int j = 0; j < n_kt; ++j) {
      f32x16 sc[2];  // slot 2j + 1
      if (j <= jw) qk(j, sc);
      if (j >= 1 && j - 1 <= jw) pv(j - 1, pb);
      PF_BARRIER_LOADED();
      if (j <= jw) softmax(j, sc, pb);  // slot 2j + 2
      stage(j + 1);
      PF_BARRIER();
    }
    if (n_kt - 1 <= jw) pv(n_kt - 1, pb);  // slot 2 n_kt + 1
    PF_BARRIER();
    // through the V stages, whose last reads were this half's
    st.store(a, lds + 2 * K_BYTES + (w - 4) * (kUnitQ * D * 2), h, s0, len, wq0);
  }
#undef PF_BARRIER
#undef PF_BARRIER_LOADED
}

template <int DT, int D, bool SIGNED>
__global__ __launch_bounds__(kLongThreads) void prefill_long_kernel(PrefillArgs a) {
  constexpr int K_BYTES = kPfKTile * (D * 2 + 16);
  constexpr int V_BYTES = kPfKTile * (D * 2 + 64);
  // two K stages, then two V stages
  __shared__ __align__(16) uint8_t lds[2 * K_BYTES + 2 * V_BYTES];
  int kvh, s0, len, u0;
  if (!pick_job<kLongWaves>(a, kvh, s0, len, u0)) return;  // uniform, before any barrier
  attend_long<DT, D, SIGNED>(a, lds, kvh, s0, len, u0);
}

template <int DT, int D, bool SIGNED>
void launch_kernel(const PrefillArgs& a, bool long_prompts, uint32_t grid, hipStream_t stream) {
  if (long_prompts)
    hipLaunchKernelGGL((prefill_long_kernel<DT, D, SIGNED>), dim3(grid), dim3(kLongThreads), 0,
                       stream, a);
  else
    hipLaunchKernelGGL((prefill_short_kernel<DT, D, SIGNED>), dim3(grid), dim3(kShortThreads), 0,
                       stream, a);
}
template <int DT, int D>
void launch_prefill(const PrefillArgs& a, bool long_prompts, uint32_t grid, hipStream_t stream) {
  if (a.scale_sign > 0) launch_kernel<DT, D, false>(a, long_prompts, grid, stream);
  else launch_kernel<DT, D, true>(a, long_prompts, grid, stream);
}

}  // namespace
}  // namespace aegkv

using namespace aegkv;

extern "C" {

int aegkv_varlen_prefill_attention(void* out, int64_t out_token_stride, const void* q,
                                   int64_t q_token_stride, const void* k, int64_t k_token_stride,
                                   const void* v, int64_t v_token_stride,
                                   const int32_t* cu_seqlens, int32_t batch, int32_t max_seqlen,
                                   int64_t total_tokens, int32_t n_q_heads, int32_t n_kv_heads,
                                   int32_t head_dim, float scale, int32_t causal, int32_t dtype,
                                   aegkv_stream_t stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  if (batch < 0 || max_seqlen < 0 || total_tokens < 0 || n_q_heads <= 0 || n_kv_heads <= 0)
    return AEGKV_ERR_INVALID_ARG;
  if (n_q_heads % n_kv_heads != 0) return AEGKV_ERR_INVALID_ARG;
  if (dtype != AEGKV_DTYPE_BF16 && dtype != AEGKV_DTYPE_FP16) return AEGKV_ERR_UNSUPPORTED;
  if (head_dim != 64 && head_dim != 128) return AEGKV_ERR_UNSUPPORTED;
  if (!std::isfinite(scale)) return AEGKV_ERR_INVALID_ARG;
  if (batch == 0 || max_seqlen == 0 || total_tokens == 0) return AEGKV_OK;
  if (!out || !q || !k || !v || !cu_seqlens) return AEGKV_ERR_INVALID_ARG;
  if (q_token_stride < (int64_t)n_q_heads * head_dim ||
      out_token_stride < (int64_t)n_q_heads * head_dim ||
      k_token_stride < (int64_t)n_kv_heads * head_dim ||
      v_token_stride < (int64_t)n_kv_heads * head_dim)
    return AEGKV_ERR_INVALID_ARG;
  if (!aligned16(out) || !aligned16(q) || !aligned16(k) || !aligned16(v) ||
      q_token_stride % 8 || k_token_stride % 8 || v_token_stride % 8 || out_token_stride % 8)
    return AEGKV_ERR_MISALIGNED;
  const bool long_prompts = max_seqlen > kLongPrompt;
  const int waves = long_prompts ? kLongWaves : kShortWaves;
  const int group = n_q_heads / n_kv_heads;
  const int64_t n_pairs = (int64_t)n_kv_heads * batch;
  const int64_t max_units = ((int64_t)max_seqlen + kUnitQ - 1) / kUnitQ * group;
  const int64_t n_tiles = (max_units + waves - 1) / waves;
  // a bound of the jobs (8 x query heads x whole tiles), well below 2^31
  const int64_t q_tiles = (max_units / group + waves - 1) / waves;
  if (8 * (int64_t)n_q_heads * batch * q_tiles > INT32_MAX) return AEGKV_ERR_UNSUPPORTED;
  // the long kernel addresses K and V rows by 32-bit byte offsets within a
  // sequence, up to one key tile past its end
  if (long_prompts && ((int64_t)max_seqlen + kPfKTile) *
                              std::max(k_token_stride, v_token_stride) * 2 >
                          (int64_t)UINT32_MAX)
    return AEGKV_ERR_UNSUPPORTED;
  // Job numbers over the existing tiles only, unless the lengths are all the
  // bound (nothing to skip) or there are more than a wave searches.  The sum of
  // the tiles is bounded by the tokens, plus a part-filled unit and tile per
  // sequence.
  const bool compact = total_tokens < (int64_t)batch * max_seqlen && batch <= 64 * kCompactSets;
  int64_t grid = n_pairs * n_tiles;
  if (compact) {
    const int64_t units = (total_tokens / kUnitQ + batch) * group;
    grid = std::min(grid, (units / waves + batch) * n_kv_heads);
  }

  PrefillArgs a;
  a.q = static_cast<const uint8_t*>(q);
  a.k = static_cast<const uint8_t*>(k);
  a.v = static_cast<const uint8_t*>(v);
  a.out = static_cast<uint8_t*>(out);
  a.q_tok_b = q_token_stride * 2;
  a.k_tok_b = k_token_stride * 2;
  a.v_tok_b = v_token_stride * 2;
  a.o_tok_b = out_token_stride * 2;
  a.cu_seqlens = cu_seqlens;
  a.token_bound = (int32_t)std::min<int64_t>(total_tokens, INT32_MAX);
  a.batch = batch;
  a.n_kv_heads = n_kv_heads;
  a.group = group;
  a.max_seqlen = max_seqlen;
  a.n_pairs = (int32_t)n_pairs;
  a.by_heads = fast_div(n_kv_heads);
  a.by_group = fast_div(group);
  a.by_pairs = fast_div((int32_t)n_pairs);
  a.n_tiles = (int32_t)n_tiles;
  a.compact = compact ? 1 : 0;
  const bool in_turn =
      n_pairs % kXcds != 0 || total_tokens * 10 < (int64_t)batch * max_seqlen * 9;
  a.per_xcd = in_turn ? 0 : (int32_t)(n_pairs / kXcds);
  a.causal = causal ? 1 : 0;
  a.scale_sign = scale > 0 ? 1 : scale < 0 ? -1 : 0;
  a.scale_log2 = scale == 0 ? 1.f : std::fabs(scale) * 1.4426950408889634f;
  const uint32_t g32 = (uint32_t)grid;
  if (dtype == AEGKV_DTYPE_BF16) {
    if (head_dim == 64) launch_prefill<AEGKV_DTYPE_BF16, 64>(a, long_prompts, g32, stream);
    else launch_prefill<AEGKV_DTYPE_BF16, 128>(a, long_prompts, g32, stream);
  } else {
    if (head_dim == 64) launch_prefill<AEGKV_DTYPE_FP16, 64>(a, long_prompts, g32, stream);
    else launch_prefill<AEGKV_DTYPE_FP16, 128>(a, long_prompts, g32, stream);
  }
  AEGKV_HIP_TRY(hipGetLastError());
  return AEGKV_OK;
}

}  // extern "C"
