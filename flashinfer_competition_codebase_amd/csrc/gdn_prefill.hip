// gdn_prefill.hip - Gated Delta Net prefill (variable-length sequences) for
// gfx950 (MI355X), chunkwise with MFMA.
//
// Semantics: the reference's prefill (solution/triton/prefill_kernel.py:
// 85-183) -- per sequence of cu_seqlens, the decode step applied token after
// token to the running fp32 state (k-last [HV, V, K] per sequence), output
// per token, the final state per sequence.  The recurrence is evaluated in
// chunks of C = 64 tokens (the chunkwise form of the gated delta rule): with
// gamma_i the cumulative log-decay inside a chunk and S_0 the state ([K, V])
// at its start,
//   A     = strict_lower(beta_i e^(gamma_i - gamma_j) k_i . k_j)
//   T     = (I + A)^-1                                 (unit lower triangular)
//   X     = V - diag(e^gamma) K S_0        (what the decayed state misses)
//   Delta = T diag(beta) X                 (the per-token delta-rule corrections;
//                                           = U - W S_0 of the WY form)
//   O     = scale [diag(e^gamma) Q S_0 + (Q K^T (.) M) Delta],
//           M_ij = e^(gamma_i - gamma_j) for j <= i
//   S_C   = e^(gamma_C) S_0 + (diag(e^(gamma_C - gamma)) K)^T Delta
// Every exponent is <= 0.  With the q/k L2-norm on, the row norms enter as
// per-row scale factors of the same products.
//
// Prefills of at most kSmallTokens (56) tokens in all (so every sequence is
// that short) skip the chunkwise machinery: one launch of the decode kernel's
// variable-length mode (gdn_decode_kernel.h) applies the recurrence token by
// token with the state in registers, one workgroup per (sequence, v-head,
// row tile), reading each sequence's token range from cu_seqlens on the
// device.  Prefills of 57 to 64 tokens in all (every sequence one chunk)
// with at most 128 (sequence, v-head) pairs run one launch of the one-chunk
// kernel: each workgroup prepares its sequence's chunk in its own LDS (kernel
// 2's code) and scans it (kernel 3's), so the slot never goes through the
// workspace.  Larger prefills run the chunkwise kernels -- after
// the token kernel's launch, for 2..64 sequences that may all be at most 56
// tokens long (the host knows only the total): it runs only if every sequence
// is, and the chunkwise kernels then return at once.
//
// Kernels (one stream, in order):
//   1. chunk_offsets: one workgroup turns cu_seqlens into the first chunk
//      slot of every sequence (token ranges clamped to [0, L]) by a scan,
//      and writes each slot's sequence, first token and token count.  With
//      one sequence, or a few (their slots found in the kernels), it is not
//      launched.
//   2. prep, one wave per (chunk slot, q/k head) -- or (chunk slot, v-head)
//      when there are few of those: what does not depend on the
//      state, for all chunks at once -- K K^T (bf16 MFMA: the inputs are bf16,
//      once per wave), then per v-head the gates and gamma and T by block
//      recursion (fp32 MFMA) -- into a 14 KiB workspace slot per (chunk,
//      v-head): the lower blocks of T diag(beta), split into bf16 hi + lo in
//      the order the scan's MFMAs read them, and the row scales.
//   3. scan, one workgroup per (sequence, v-head), XCD-aware order: the
//      sequential part chunk after chunk.  Four main waves, one a SIMD, hold
//      the whole 128 x 128 state in registers (32 columns each); four helper
//      waves beside them bring the next chunk's K, Q rows and slot to LDS by
//      DMA, into the other of two buffers, and make the K^T and Q K^T tiles
//      of the current one.  Products with fp32 operands run as bf16 MFMA on
//      hi/lo splits.  Each workgroup reads its chunks' inputs once, so the
//      workspace is the only HBM traffic beyond the algorithmic bytes.
//   One long sequence at few v-heads is cut into segments, since its scan
//   alone would occupy HV workgroups for the whole run: a first scan launch
//   runs, without outputs, segment 0 from the sequence's state and, from
//   each later segment's start, the transition columns (an identity start,
//   no values) and the zero-start end state; a combine kernel chains the
//   segment starts; a second scan launch runs every segment from its start
//   with the outputs.
//
// MFMA lane layouts.  16 x 16 (v_mfma_f32_16x16x4_f32, _16x16x32_bf16):
// A[i][k] from lane i + 16 g, B[k][j] from lane j + 16 g (k = g for fp32; for
// bf16 the lane's 8 items cover the 32-long k block), D[i][j] in lane j + 16
// (i / 4), register i % 4.  32 x 32 (_32x32x16_bf16): A[i][k] from lane i +
// 32 g, B[k][j] from lane j + 32 g (8 items of the 16-long k block), D row 8 q
// + 4 g + e, column j in lane j + 32 g, register 4 q + e.  A bf16 product sums
// over its k block in any order both operands share.  Where the contracted
// index is a token, item e of lane group g of a 16-long block stands for
//   k = 8 (e / 4) + 4 g + e % 4,
// so a lane's 8 items are the 4-element runs at k = 4 g and 8 + 4 g, the runs
// a 32 x 32 result holds per lane -- results become operands without
// exchanging data between lanes.  Where it is a key (K and Q rows read from
// LDS against the state), item e of lane group g is key 8 g + e of the block:
// one 16-byte read per operand.  The state's registers hold its keys in that
// order.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <mutex>

#include "gdn_decode_kernel.h"
#include "gdn_prefill.h"
#include "gdn_prefill_segments.h"

namespace gdn_pf {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef int32_t i32x4 __attribute__((ext_vector_type(4)));

constexpr int kDim = 128;            // K == V == 128
constexpr int kChunk = 64;           // tokens per chunk
constexpr int kThreads = 256;        // 4 wavefronts
// Batches whose chunk slots the kernels find themselves, without the offsets
// kernel: at most kFewSeqs sequences (one a lane) and kFewPrepGroups (slot,
// v-head) pairs.  Each preparation wave and scan workgroup then scans the batch's
// lengths itself, which is always the faster up to there and not always past it
// (captured calls, in the kernels against the offsets kernel, us: 3 sequences of
// 40 tokens at 4/8 heads 19.3 / 20.7, 16 x 512 there 49.2 / 51.2, 64 x 128, 1536
// pairs, 49.4 / 51.1; past it 16 x 1024, 2176 pairs, 74.8 / 77.4, 8 x 1024 at 16/32,
// 4352, 108.6 / 110.1, but 64 x 64 there, 4096, 126.7 / 124.4 and 64 x 512, 18432, 452.6
// / 449.5).
constexpr int kFewSeqs = 64;
constexpr long long kFewPrepGroups = 2048;

// Chunk slots the workspace holds for L tokens in N sequences: every chunk
// of a well-formed batch fits, sum(ceil(len_i / 64)) <= ceil(L / 64) + N, and
// every chunk holds at least one token, so there are at most L of them.
// For malformed cu_seqlens the kernels cap the slots they use at this count.
long long max_slots(long long L, long long N) {
  const long long by_seqs = (L + kChunk - 1) / kChunk + N;
  return by_seqs < L ? by_seqs : L;
}

bool few_seqs(long long L, long long N, long long HV) {
  return N > 1 && N <= kFewSeqs && max_slots(L, N) * HV <= kFewPrepGroups;
}
// Total tokens up to which the token-by-token kernel runs the prefill (so no
// sequence is longer).  The line is where it met the two chunkwise kernels on one
// sequence; several short ones favour it more (captured calls: 4 x 14 tokens at
// 4/8 heads 7.7 us, one chunk 12.4).  On one sequence the one-chunk kernel, 12.2 us
// whatever the tokens, is now faster from 33 tokens at 4/8 heads (56: 19.3 us) and
// from 25 at 16/32 (56: 25.3 against 12.6): not used there, as the entry points
// publish the line.
constexpr int kSmallTokens = 56;

// Batches of 2..kFewSeqs sequences with at most kSmallTokens tokens a
// sequence on average may have no longer sequence, which only cu_seqlens on
// the device tells: they launch the token-by-token kernel first (it runs
// only if every sequence is that short) and then the chunkwise kernels
// (which return at once in that case).  4 sequences of 20 tokens at qk4_v8
// then take the token kernel's time instead of the chunkwise kernels'.
bool maybe_all_short(long long L, long long N) {
  return L > kSmallTokens && N >= 2 && N <= kFewSeqs && L <= N * kSmallTokens;
}
constexpr float kL2Eps = 1e-6f;
// A preparation wave takes a whole GVA group of v-heads (K K^T made once for
// all of them, the v-heads one after another) unless there are at most
// kPrepSplitMaxWaves (slot, v-head) pairs, 16 a CU: then each wave takes one
// v-head, and the chain of one wave -- the preparation's time on a grid that
// small -- is one v-head's.  Twelve waves fit a CU at once, and past them the
// shorter chain still pays for the second round and for K K^T (captured calls, by
// v-head against by group, us: 16 x 384 tokens at 16/32 heads, 3584 pairs, 88.5 /
// 91.9; 4096 pairs: 16 x 448 there 110.3 / 111.2, at 8/32 103.4 / 108.1, 64 x 448 at 4/8
// 108.2 / 109.7; 16 x 640 at 16/32, 5632 pairs, 147.8 / 143.4).
constexpr long long kPrepSplitMaxWaves = 4096;
constexpr long long kPrepSpreadMaxWaves = 1024;     // a wave a workgroup up to 4 a CU (kernel 2)
inline bool prep_split(long long slots, int HV) { return slots * HV <= kPrepSplitMaxWaves; }
constexpr float kSoftplusThreshold = 20.0f;
constexpr float kLog2e = 1.44269504088896341f;
constexpr float kLn2 = 0.693147180559945309f;

// Workspace slot of one (chunk, v-head), offsets in floats.  The scan's MFMA
// operand T diag(beta) is stored in operand order: a 32 x 16 block is 64
// lanes x 8 bf16 contiguous (lane = row + 32 g, items in the k order above),
// so a wave reads one with a single 1 KiB access.  It is lower triangular
// 64 x 64, so only the blocks (row block rb, token block kb) with kb < 2 rb +
// 2 are kept, six of eight, split into a bf16 high and low part (x ~ hi + lo
// to ~2^-16 relative).  Then rows of 64 per-token scales.
constexpr int kBlk = 512;                             // bf16 per operand block
constexpr int kBlkF = kBlk / 2;                       // the same in floats
constexpr int kTriBlocks = 6;
__host__ __device__ constexpr int tri_blk(int rb, int kb) { return 2 * rb + kb; }
constexpr int kSlotScales = 2 * kTriBlocks * kBlkF;   // after T diag(beta), hi then lo
// rows of the scales
constexpr int kRowXg = 0;                             // rk_i e^gamma_i [64]
constexpr int kRowEg = kRowXg + kChunk;               // scale e^gamma_i [64]
constexpr int kRowKs = kRowEg + kChunk;               // rk_i e^(gamma_C - gamma_i) [64]
constexpr int kRowGl = kRowKs + kChunk;               // e^gamma_C [64 copies]
constexpr int kRowGa = kRowGl + kChunk;               // gamma_i log2(e) [64], hi
constexpr int kRowGaLo = kRowGa + kChunk;             //   lo
constexpr int kRowRk = kRowGaLo + kChunk;             // scale rk_i [64]
constexpr int kScaleFloats = kRowRk + 2 * kChunk;     // padded to whole 1 KiB DMA pieces
constexpr int kSlotFloats = kSlotScales + kScaleFloats;
static_assert(kSlotScales % 256 == 0 && kScaleFloats % 256 == 0, "whole 1 KiB DMA pieces");
static_assert(tri_blk(1, 3) == kTriBlocks - 1, "six lower blocks");

// The combine's key order: first of the 4 keys that row tile t holds in lane
// group g (items e = 0..3 are that key + e): tiles 2 kb and 2 kb + 1 together
// are keys 32 kb + 8 g .. + 7, the combine's operand.  Row i of tile t is
// thus key state_key(t, i / 4) + i % 4.
__host__ __device__ constexpr int state_key(int t, int g) {
  return 32 * (t >> 1) + 8 * g + 4 * (t & 1);
}

__device__ __forceinline__ float bf16_to_f32(uint16_t h) {
  return __uint_as_float(static_cast<uint32_t>(h) << 16);
}

// Two floats to a packed bf16 pair (round to nearest even), element 0 in
// the low half.  split4: x ~ hi + lo with hi = bf16(x), lo = bf16(x - hi).
__device__ __forceinline__ uint32_t pack_bf16x2(float a, float b) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}

__device__ __forceinline__ void split4(const f32x4& x, s16x4& hi, s16x4& lo) {
  u32x2 h, l;
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const float x0 = x[2 * e], x1 = x[2 * e + 1];
    h[e] = pack_bf16x2(x0, x1);
    l[e] = pack_bf16x2(x0 - __uint_as_float(h[e] << 16), x1 - __uint_as_float(h[e] & 0xffff0000u));
  }
  hi = __builtin_bit_cast(s16x4, h);
  lo = __builtin_bit_cast(s16x4, l);
}

// The wavefront's index in its workgroup, as a value the compiler knows is
// the same in every lane (a scalar register): branches on it are scalar
// branches and LDS bases derived from it need no per-lane waterfall.
__device__ __forceinline__ int wave_index() {
  return __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
}

// Workgroup barrier that orders LDS only.  The waves of these kernels
// exchange data through LDS alone, so global loads issued ahead of a barrier
// stay in flight across it instead of being drained as __syncthreads'
// all-memory fence would.
__device__ __forceinline__ void block_sync_lds() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Workgroup barrier after this wave's LDS reads and writes (s_waitcnt
// lgkmcnt(0)) but not its global loads in flight.  The empty asm statements
// keep the compiler from moving memory accesses across.
__device__ __forceinline__ void barrier_lds_no_dma() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xC07F);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Ordering among the lanes of one wave, whose LDS accesses are carried out in
// program order: no instruction, but the fences keep the compiler from moving
// an access across (the barrier alone is no memory operation, and what one
// lane stores and another loads looks unrelated in each lane's own view).
__device__ __forceinline__ void wave_sync_lds() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

__device__ __forceinline__ f32x4 mfma_f32(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma_bf16(s16x8 a, s16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

__device__ __forceinline__ f32x16 mfma32_bf16(s16x8 a, s16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

__device__ __forceinline__ s16x8 cat(s16x4 a, s16x4 b) {
  return s16x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
}

struct Params {
  const uint16_t* q;         // [L, H, 128] bf16
  const uint16_t* k;         // [L, H, 128] bf16
  const uint16_t* v;         // [L, HV, 128] bf16
  const float* state;        // [N, HV, 128, 128] fp32 k-last, or null (zeros)
  const float* A_log;        // [HV]
  const uint16_t* a;         // [L, HV] bf16
  const float* dt_bias;      // [HV]
  const uint16_t* b;         // [L, HV] bf16
  const int32_t* cu_seqlens; // [N + 1]
  uint16_t* out;             // [L, HV, 128] bf16
  float* new_state;          // [N, HV, 128, 128] fp32 k-last
  const int32_t* offs;       // [N + 1] first chunk slot of each sequence (workspace)
  const i32x4* slot_info;    // [max_slots] per chunk slot: sequence, first token, tokens
                             // (0 past the last slot) (workspace)
  float* slots;              // [max_slots, HV, kSlotFloats] (workspace)
  float scale;
  int L;
  int N;
  int H;
  int HV;
  int ratio;                 // HV / H
  int l2norm;
  int single;                // one sequence: chunk c is slot c (no offsets kernel)
  int few;                   // 2..kFewSeqs sequences: the kernels compute the chunk
                             // slots from cu_seqlens (no offsets kernel)
  long long max_slots;       // slots the workspace holds
  // Segments (seg_chunks > 0): segment j of a sequence is its chunks
  // [j seg_chunks, (j + 1) seg_chunks), and the segments of all sequences are
  // numbered in sequence order (at most nseg); per (segment, v-head) 128 x 128 fp32
  // blocks in k-last order (element (k, c) at c * 128 + k).
  int seg_chunks;            // chunks per segment, 0: no segments
  int nseg;                  // segments
  float* seg_S;              // [nseg, HV] state at each segment's start (1 .. nseg-1;
                             // in place 0 too)
  float* seg_B;              // [nseg, HV] state at its end from a zero start
  float* seg_M;              // [nseg, HV] its transition: end = M start + B (M[k][k'])
  // > 0: the token-by-token kernel was launched first with this limit (at
  // most kFewSeqs sequences); if every sequence has at most this many tokens
  // it ran the whole prefill and these kernels return at once.
  int short_limit;
  int prep_heads;            // v-heads per preparation wave: ratio, or 1
  int prep_waves;            // waves per preparation workgroup: kPrepWaves, or 1
};

// Token range [start, end) of sequence s, clamped to [0, L] so that no
// cu_seqlens content makes a kernel read outside the inputs.
__device__ __forceinline__ void seq_range(const Params& p, int s, int& start, int& end) {
  int s0 = p.cu_seqlens[s];
  int s1 = p.cu_seqlens[s + 1];
  s0 = s0 < 0 ? 0 : (s0 > p.L ? p.L : s0);
  s1 = s1 < s0 ? s0 : (s1 > p.L ? p.L : s1);
  start = s0;
  end = s1;
}

// A value the caller knows is the same in every lane, in a scalar register
// (the compiler loads what it cannot tell is constant into vector registers,
// and addresses formed from it stay there).
__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }

// Whether every sequence of a batch of at most 64 has at most `limit`
// tokens (one read per lane, the clamping of seq_range; uniform).
__device__ __forceinline__ bool all_within(const Params& p, int limit) {
  const int lane = threadIdx.x & 63;
  int len = 0;
  if (lane < p.N) {
    int s0, s1;
    seq_range(p, lane, s0, s1);
    len = s1 - s0;
  }
  return __ballot(len > limit) == 0;
}

// Chunk slots of a batch of at most 64 sequences, from cu_seqlens in one
// wave (lane s: sequence s): the prefix the offsets kernel writes, held in
// registers.  excl = slots of the sequences before s, incl = excl + its own,
// both capped at the workspace's slots as there.  A sequence's chunk count
// is at most 2^25 (ranges are clamped to [0, L], L < 2^31), so 64 of them
// sum without overflow in 32 bits.
struct FewSlots {
  int start, end;          // this lane's sequence's token range (0, 0 past N)
  long long excl, incl;
};

__device__ __forceinline__ FewSlots few_slots(const Params& p) {
  const int lane = threadIdx.x & 63;
  FewSlots f{0, 0, 0, 0};
  unsigned cnt = 0;
  if (lane < p.N) {
    seq_range(p, lane, f.start, f.end);
    cnt = static_cast<unsigned>(f.end - f.start + kChunk - 1) / kChunk;
  }
  unsigned x = cnt;                                // inclusive scan over the wave
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const unsigned y = __shfl_up(x, d, 64);
    if (lane >= d) x += y;
  }
  const long long incl = x, excl = static_cast<long long>(x) - cnt;
  f.incl = incl < p.max_slots ? incl : p.max_slots;
  f.excl = excl < p.max_slots ? excl : p.max_slots;
  return f;
}

// Segments of a batch of at most 64 sequences, in one wave (lane s: sequence
// s): its token range, its segment count (seg_chunks chunks a segment; one
// for an empty sequence), the segments of the sequences before it, and its
// units of a segment launch (OUT: one a segment; else 2 nseg - 3: segment 0
// from the sequence's state, the middle ones from a zero start and from the
// identity; none for a sequence of one segment).
struct SegSeqs {
  int start, end;
  int nseg, seg_excl;
  int u_excl, u_incl;
};

// Units of the first segment launch for nseg segments in all: one sequence
// has 2 nseg - 3, several at most 2 nseg.
__host__ __device__ inline long long seg_units1(long long nseg, long long N) {
  return N == 1 ? 2 * nseg - 3 : 2 * nseg;
}

template <bool OUT>
__device__ __forceinline__ SegSeqs seg_seqs(const Params& p) {
  const int lane = threadIdx.x & 63;
  SegSeqs f{0, 0, 0, 0, 0, 0};
  int units = 0;
  if (lane < p.N) {
    seq_range(p, lane, f.start, f.end);
    const int nch = (f.end - f.start + kChunk - 1) / kChunk;
    f.nseg = nch > p.seg_chunks ? (nch + p.seg_chunks - 1) / p.seg_chunks : 1;
    units = OUT ? f.nseg : (f.nseg >= 2 ? 2 * f.nseg - 3 : 0);
  }
  if (p.N == 1) {                                  // uniform: nothing to scan
    f.u_incl = units;
    return f;
  }
  int xs = f.nseg, xu = units;                     // inclusive scans over the wave
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int ys = __shfl_up(xs, d, 64);
    const int yu = __shfl_up(xu, d, 64);
    if (lane >= d) {
      xs += ys;
      xu += yu;
    }
  }
  f.seg_excl = xs - f.nseg;
  f.u_excl = xu - units;
  f.u_incl = xu;
  // A malformed batch (overlapping ranges) may need more segments than the
  // workspace holds: then every sequence is one segment (a plain scan in the
  // second launch), so each one's state is still written.
  if (__builtin_amdgcn_readlane(xs, 63) > p.nseg) {
    f.nseg = lane < p.N ? 1 : 0;
    f.seg_excl = lane;
    f.u_excl = OUT ? lane : 0;
    f.u_incl = OUT && lane < p.N ? lane + 1 : f.u_excl;
  }
  return f;
}

// ---------------------------------------------------------------------------
// 1. chunk slots per sequence
// ---------------------------------------------------------------------------
// One workgroup of 256 threads: each thread counts one sequence's chunks, a
// block-wide inclusive scan (wave scans through LDS) turns 256 counts into
// offsets, and a running total carries from one group of 256 sequences to
// the next.  The group's offsets and token ranges then go to LDS, and the
// threads fill the group's slots of the slot table, each finding its slot's
// sequence by binary search there.  Slots past the last one get zero tokens.
__global__ __launch_bounds__(kThreads) void chunk_offsets_kernel(Params p, int32_t* offs,
                                                                 i32x4* slot_info) {
  __shared__ long long wave_sum[kThreads / 64];
  __shared__ int32_t grp_offs[kThreads + 1];   // offs[base .. base + 256]
  __shared__ int32_t grp_start[kThreads];
  __shared__ int32_t grp_end[kThreads];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  if (p.short_limit > 0 && all_within(p, p.short_limit)) return;    // uniform
  long long carry = 0;
  if (threadIdx.x == 0) offs[0] = 0;
  for (int base = 0; base < p.N; base += kThreads) {
    const int s = base + threadIdx.x;
    long long cnt = 0;
    int start = 0, end = 0;
    if (s < p.N) {
      seq_range(p, s, start, end);
      cnt = (end - start + kChunk - 1) / kChunk;
    }
    long long x = cnt;                         // inclusive scan within the wave
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const long long y = __shfl_up(x, d, 64);
      if (lane >= d) x += y;
    }
    if (lane == 63) wave_sum[wave] = x;
    __syncthreads();
    long long before = carry;
    for (int w = 0; w < wave; ++w) before += wave_sum[w];
    long long total = carry;
    for (int w = 0; w < kThreads / 64; ++w) total += wave_sum[w];
    long long v = before + x;
    if (v > p.max_slots) v = p.max_slots;      // only for overlapping ranges
    if (total > p.max_slots) total = p.max_slots;
    if (s < p.N) offs[s + 1] = static_cast<int32_t>(v);
    grp_offs[threadIdx.x + 1] = static_cast<int32_t>(v);
    if (threadIdx.x == 0) grp_offs[0] = static_cast<int32_t>(carry);
    grp_start[threadIdx.x] = start;
    grp_end[threadIdx.x] = end;
    carry = total;
    __syncthreads();
    // slots [grp_offs[0], grp_offs[256]) belong to this group's sequences;
    // slot c's sequence is the largest j with grp_offs[j] <= c
    for (int c = grp_offs[0] + threadIdx.x; c < grp_offs[kThreads]; c += kThreads) {
      int lo = 0, hi = kThreads - 1;
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (grp_offs[mid] <= c) lo = mid; else hi = mid - 1;
      }
      const int t0 = grp_start[lo] + (c - grp_offs[lo]) * kChunk;
      const int n = min(kChunk, grp_end[lo] - t0);
      slot_info[c] = i32x4{base + lo, t0, n, 0};
    }
    __syncthreads();                           // LDS is rewritten next round
  }
  for (long long c = carry + threadIdx.x; c < p.max_slots; c += kThreads)
    slot_info[c] = i32x4{0, 0, 0, 0};
}

// Gates of token t, v-head hv: the decay's log2 and beta
// (g = exp(-exp(A_log) softplus(a + dt_bias)), beta = sigmoid(b)).  The decays
// stay in log2 units: each later exponential is one v_exp_f32.  A decay below
// 2^kForgetLog2 is zero with or without the tokens beside it, so the log2 stops
// there: the cumulative sums stay finite (a difference of two -inf is NaN) and
// keep the other tokens' decays however large this one's is.  NaN passes.
constexpr float kForgetLog2 = -1024.0f;
__device__ __forceinline__ void gates_of(uint16_t a_raw, uint16_t b_raw, float dt_bias,
                                         float A_log, float& log2g, float& beta) {
  const float x = bf16_to_f32(a_raw) + dt_bias;
  const float sp = x > kSoftplusThreshold ? x * kLog2e : __builtin_amdgcn_logf(1.0f + __expf(x));
  log2g = -__expf(A_log) * sp;
  log2g = log2g < kForgetLog2 ? kForgetLog2 : log2g;
  beta = __builtin_amdgcn_rcpf(1.0f + __expf(-bf16_to_f32(b_raw)));
}

// One DPP step of a wave scan: x from the lane CTRL names (0 where it names
// none, or in rows ROW_MASK leaves out).
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ double dpp_add_src(double x) {
  const u32x2 w = __builtin_bit_cast(u32x2, x);
  u32x2 r;
#pragma unroll
  for (int i = 0; i < 2; ++i)
    r[i] = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(w[i]), CTRL,
                                                             ROW_MASK, 0xf, false));
  return __builtin_bit_cast(double, r);
}

// Inclusive prefix sum over the 64 lanes of a wave: shifts by 1, 2, 4 and 8
// within each row of 16 lanes (row_shr), then lane 15's total added to rows
// 1 and 3 and lane 31's to rows 2 and 3 (row_bcast:15, row_bcast:31).  In 64
// bits: a head that forgets fast reaches gamma ~ -1000 within a chunk, where
// an fp32 sum is only good to 1e-4 and so are the decays e^(gamma_i - gamma_j)
// of its last tokens; as hi + lo pairs the differences are good to 2^-24 of
// themselves (state error against 64 bits on short sequences: up to 1.5e-5
// with fp32 sums, 3-5e-6 -- the products' hi/lo splits -- with these).
__device__ __forceinline__ double wave_prefix_sum(double x) {
  x += dpp_add_src<0x111, 0xf>(x);
  x += dpp_add_src<0x112, 0xf>(x);
  x += dpp_add_src<0x114, 0xf>(x);
  x += dpp_add_src<0x118, 0xf>(x);
  x += dpp_add_src<0x142, 0xa>(x);
  x += dpp_add_src<0x143, 0xc>(x);
  return x;
}

// 2^((xh + xl) - (yh + yl)), for x <= y; the clamp keeps what a mask discards
// (x > y) finite.
__device__ __forceinline__ float decay(float xh, float xl, float yh, float yl) {
  return __builtin_amdgcn_exp2f(fminf((xh - yh) + (xl - yl), 0.0f));
}

// ---------------------------------------------------------------------------
// 2. per-chunk preparation
// ---------------------------------------------------------------------------
// One wave per chunk and q/k head (its v-heads one after another) or v-head.
// The chain of one chunk -- K K^T, gates, A, the triangular inverse by 16 x 16
// blocks -- has little work in each step, so what bounds it is latency: four
// waves sharing it waited 53% of their cycles on ten barriers and on LDS round
// trips, 12 KiB of K rows and two 64 x 64 matrices there limited a CU to four
// such chains, and each diagonal block's substitution used 16 of 64 lanes.  A
// wave of its own needs no barrier, keeps K K^T's operands and every block in
// registers in the two layouts the products read (6 KiB of LDS and 155
// registers: twelve chains a CU), and runs the four substitutions at once.  Kernel
// trace, before and after: 64 x 512 tokens at 16/32 heads 112-119 -> 82 us (4.5
// TB/s of K rows in and slots out), 12 ragged sequences there 43 -> 28 us, 16 x
// 1024 at 4/8 18.3 -> 14.6 us.
//
// 16 x 16 blocks in registers, lane (i, g) = (lane % 16, lane / 16), item e:
//   column layout  [4 g + e][i]   (an MFMA result; the B operand)
//   row layout     [i][4 g + e]   (the A operand)
// with the contracted index taken as 4 g + (step) on both sides.  A result of
// swapped operands is the product's transpose, i.e. the row layout:
// (L X)^T = X^T L^T, where X's column layout reads as X^T's A operand and L's
// row layout as L^T's B operand.

constexpr int kPrepWaves = 4;       // a workgroup
constexpr int kBlkStride = 20;      // floats of a 16-long row or column: 16-byte aligned,
                                    // and reads down a column spread over the banks

struct __attribute__((aligned(16))) PrepLds {
  float blk[4][16 * kBlkStride];    // the diagonal blocks of A by rows, then of T by columns
  float gamma[kChunk];              // hi and lo
  float gamma_lo[kChunk];
  float beta[kChunk];
  float rk[kChunk];
};

// A B (contracted over 16, fp32 MFMA) added to acc: rows of A in row layout,
// B in column layout.
__device__ __forceinline__ f32x4 mm16(const f32x4& a, const f32x4& b, f32x4 acc) {
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) acc = mfma_f32(a[ks], b[ks], acc);
  return acc;
}

__device__ __forceinline__ f32x4 lds4(const float* ptr) {
  return *reinterpret_cast<const f32x4*>(ptr);
}

// One chunk's preparation, tokens t0 .. t0 + n - 1 (n: 1..64) of q/k head h,
// for v-heads hv0 .. hv0 + prep_heads - 1, by the calling wave: the slots go
// to the workspace (slot c), or with LDS_SLOT (one v-head) to lds_T and
// lds_scales in the calling workgroup's LDS -- whose other waves' first barrier,
// that the chunk's rows are in LDS, it joins once its own loads have come.
template <bool LDS_SLOT>
__device__ __forceinline__ void prep_chunk(const Params& p, int c, int t0, int n, int hv0, int h,
                                           int prep_heads, PrepLds& lds, uint16_t* lds_T,
                                           float* lds_scales) {
  const int lane = threadIdx.x & 63;
  const int i = lane & 15;
  const int g = lane >> 4;
  const f32x4 zero = {0, 0, 0, 0};

  // K K^T's lower blocks, in row layout: kk[r (r + 1) / 2 + cb] is rows 16 r
  // + i, columns 16 cb + 4 g + e.  The operands (row 16 r + i, keys 32 m + 8 g
  // .. + 7) come straight from memory, rows >= n as zeros; the first v-head's
  // gate inputs are in flight with them.
  const int tok = t0 + (lane < n ? lane : n - 1);
  uint16_t a_raw = p.a[static_cast<size_t>(tok) * p.HV + hv0];
  uint16_t b_raw = p.b[static_cast<size_t>(tok) * p.HV + hv0];
  float dtb = p.dt_bias[hv0], alog = p.A_log[hv0];
  f32x4 kk[10];
  {
    s16x8 kf[4][4];
    const uint16_t* base = p.k + (static_cast<size_t>(t0) * p.H + h) * kDim + 8 * g;
    const size_t step = static_cast<size_t>(p.H) * kDim;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = min(16 * r + i, n - 1);
#pragma unroll
      for (int m = 0; m < 4; ++m)
        kf[r][m] = *reinterpret_cast<const s16x8*>(base + row * step + 32 * m);
    }
    if (n < kChunk) {                                // uniform
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int m = 0; m < 4; ++m)
          if (16 * r + i >= n) kf[r][m] = s16x8{0, 0, 0, 0, 0, 0, 0, 0};
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int cb = 0; cb <= r; ++cb) {
        f32x4 acc = zero;
#pragma unroll
        for (int m = 0; m < 4; ++m) acc = mfma_bf16(kf[cb][m], kf[r][m], acc);
        kk[r * (r + 1) / 2 + cb] = acc;
      }
  }

  if constexpr (LDS_SLOT) barrier_lds_no_dma();

  // K row scales of the L2-norm (1 when off), |k|^2 from K K^T's diagonal
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const f32x4 d = kk[r * (r + 1) / 2 + r];
    const float k2 = (i & 2) ? ((i & 1) ? d[3] : d[2]) : ((i & 1) ? d[1] : d[0]);
    if (g == (i >> 2)) lds.rk[16 * r + i] = p.l2norm ? __builtin_amdgcn_rsqf(k2 + kL2Eps) : 1.0f;
  }

  for (int j = 0; j < prep_heads; ++j) {
    const int hv = hv0 + j;
    float* const slot = LDS_SLOT ? nullptr
                                 : p.slots + (static_cast<size_t>(c) * p.HV + hv) * kSlotFloats;
    uint16_t* const T16 = LDS_SLOT ? lds_T : reinterpret_cast<uint16_t*>(slot);
    float* const scales = LDS_SLOT ? lds_scales : slot + kSlotScales;

    // gates of token t0 + lane (padded rows: no decay, no update), and the
    // inclusive scan of the log-decay over the chunk
    float log2g, beta;
    gates_of(a_raw, b_raw, dtb, alog, log2g, beta);
    if (j + 1 < prep_heads) {                        // the next v-head's inputs
      a_raw = p.a[static_cast<size_t>(tok) * p.HV + hv + 1];
      b_raw = p.b[static_cast<size_t>(tok) * p.HV + hv + 1];
      dtb = p.dt_bias[hv + 1];
      alog = p.A_log[hv + 1];
    }
    if (lane >= n) log2g = beta = 0.0f;
    const double gamma64 = wave_prefix_sum(static_cast<double>(log2g));
    const float gamma = static_cast<float>(gamma64);
    const float gamma_lo = static_cast<float>(gamma64 - static_cast<double>(gamma));
    wave_sync_lds();
    lds.gamma[lane] = gamma;
    lds.gamma_lo[lane] = gamma_lo;
    lds.beta[lane] = beta;
    wave_sync_lds();

    // A's blocks below the diagonal, row layout; the diagonal ones (strictly
    // lower) by rows to LDS.  The decays are computed for every element with
    // the exponent clamped to <= 0 (it is <= 0 wherever the element is kept:
    // gamma does not increase) and the masks are selects.
    f32x4 gj[4], gjl[4], rkj[4];
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) {
      gj[cb] = lds4(&lds.gamma[16 * cb + 4 * g]);
      gjl[cb] = lds4(&lds.gamma_lo[16 * cb + 4 * g]);
      rkj[cb] = lds4(&lds.rk[16 * cb + 4 * g]);
    }
    f32x4 A[10];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float gi = lds.gamma[16 * r + i], gil = lds.gamma_lo[16 * r + i];
      const float bri = lds.beta[16 * r + i] * lds.rk[16 * r + i];
#pragma unroll
      for (int cb = 0; cb <= r; ++cb) {
        const int at = r * (r + 1) / 2 + cb;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float dec = decay(gi, gil, gj[cb][e], gjl[cb][e]);
          const float x = bri * rkj[cb][e] * dec * kk[at][e];
          A[at][e] = cb < r || 4 * g + e < i ? x : 0.0f;
        }
      }
      *reinterpret_cast<f32x4*>(&lds.blk[r][i * kBlkStride + 4 * g]) = A[r * (r + 1) / 2 + r];
    }
    wave_sync_lds();

    // T = (I + A)^-1 by block recursion on 16 x 16 blocks (A is strictly lower
    // triangular, so T is unit lower triangular):
    // 1. lane (i, g) solves for column i of diagonal block g by forward
    //    substitution, two partial sums per dot product; row r's entries of A
    //    are read a row ahead of their use;
    f32x4 TD[4], TR[4];                              // column, row layout
    {
      const float* arow = lds.blk[g];
      float t[16];
      f32x4 ar[16][4];
      auto read_row = [&](int r) {
#pragma unroll
        for (int q = 0; q < (r + 3) / 4; ++q) ar[r][q] = lds4(&arow[r * kBlkStride + 4 * q]);
      };
      read_row(1);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        if (r + 1 < 16) read_row(r + 1);
        float s0 = (r == i) ? 1.0f : 0.0f, s1 = 0.0f;
#pragma unroll
        for (int q = 0; q < r; ++q) {
          const float aij = ar[r][q >> 2][q & 3];
          if (q & 1) s1 = fmaf(-aij, t[q], s1); else s0 = fmaf(-aij, t[q], s0);
        }
        t[r] = s0 + s1;
      }
      wave_sync_lds();
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<f32x4*>(&lds.blk[g][i * kBlkStride + 4 * q]) =
            f32x4{t[4 * q], t[4 * q + 1], t[4 * q + 2], t[4 * q + 3]};
      wave_sync_lds();
    }
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      TD[b] = lds4(&lds.blk[b][i * kBlkStride + 4 * g]);
#pragma unroll
      for (int e = 0; e < 4; ++e) TR[b][e] = lds.blk[b][(4 * g + e) * kBlkStride + i];
    }
    // 2. the 32 x 32 diagonal halves: T_10 = -T_11 A_10 T_00, T_32 = -T_33
    //    A_32 T_22;
    const f32x4 x10 = mm16(A[1], TD[0], zero);
    const f32x4 x32 = mm16(A[8], TD[2], zero);
    const f32x4 T10D = -mm16(TR[1], x10, zero);
    const f32x4 T10 = -mm16(x10, TR[1], zero);
    const f32x4 T32 = -mm16(x32, TR[3], zero);
    // 3. the lower-left 32 x 32 quarter: T_BA = -T_B (A_BA T_A).
    f32x4 T[10];                                     // row layout, as A
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) {
      f32x4 x[2];
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) {
        const int at = (2 + rb) * (3 + rb) / 2;
        x[rb] = cb == 0 ? mm16(A[at + 1], T10D, mm16(A[at], TD[0], zero))
                        : mm16(A[at + 1], TD[1], zero);
      }
      T[3 + cb] = -mm16(x[0], TR[2], zero);
      T[6 + cb] = -mm16(x[1], TR[3], mm16(x[0], T32, zero));
    }
    T[0] = TR[0];
    T[1] = T10;
    T[2] = TR[1];
    T[5] = TR[2];
    T[8] = T32;
    T[9] = TR[3];

    // T diag(beta) in operand order, split into hi + lo: row 16 r + i, tokens
    // 16 cb + 4 g .. + 3 are items 4 (g / 2) .. + 3 of lane 16 (r % 2) + i +
    // 32 (g % 2) of block (r / 2, cb).  Blocks (0, 1) and (2, 3), above the
    // diagonal inside an operand block, are zero.
    uint16_t* const dst0 = T16 + (i + 32 * (g & 1)) * 8 + 4 * (g >> 1);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
#pragma unroll
      for (int cb = 0; cb <= (r | 1); ++cb) {
        s16x4 hi = {0, 0, 0, 0}, lo = {0, 0, 0, 0};
        if (cb <= r) split4(T[r * (r + 1) / 2 + cb] * lds4(&lds.beta[16 * cb + 4 * g]), hi, lo);
        uint16_t* const dst = dst0 + tri_blk(r >> 1, cb) * kBlk + 128 * (r & 1);
        *reinterpret_cast<s16x4*>(dst) = hi;
        *reinterpret_cast<s16x4*>(dst + kTriBlocks * kBlk) = lo;
      }
    }

    // Row scales for the scan: the decayed K rows of X, the decay of the
    // output's rows (times the scale), the K rows of the state update, the
    // chunk decay, and gamma and the K row scales (times the scale) for its P.
    {
      // padded rows carry gamma forward
      auto last = [](float x) {
        return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), kChunk - 1));
      };
      const float rki = lds.rk[lane];
      const float e0 = __builtin_amdgcn_exp2f(gamma);
      const float egi = fmaf(e0, gamma_lo * kLn2, e0);
      scales[kRowXg + lane] = rki * egi;
      scales[kRowEg + lane] = p.scale * egi;
      scales[kRowKs + lane] = rki * decay(last(gamma), last(gamma_lo), gamma, gamma_lo);
      scales[kRowGl + lane] = last(egi);
      scales[kRowGa + lane] = gamma;
      scales[kRowGaLo + lane] = gamma_lo;
      scales[kRowRk + lane] = p.scale * rki;
    }
  }
}

// FEW: the batch's chunk slots come from cu_seqlens in the kernel (few
// sequences, no offsets kernel); a template flag, so that the kernels of the
// other modes are compiled without that code.
// Four independent waves a workgroup: four jobs (v-head groups, or v-heads) of
// one slot, whose K rows they share, or with fewer jobs a slot one job of four
// slots.  With at most four waves a CU in all, one wave a workgroup, so that
// they spread over the CUs (160 jobs, 4 ragged sequences at 4/8 heads: 9.4 ->
// 7.3 us; 2176 jobs, 16 x 1024 tokens there: 15.5 us so, 14.6 us by four).
template <bool FEW>
__global__ __launch_bounds__(64 * kPrepWaves) __attribute__((amdgpu_waves_per_eu(3)))
void prep_kernel(Params p) {
  __shared__ PrepLds lds_all[kPrepWaves];
  const int wave = wave_index();
  const int jobs = p.HV / p.prep_heads;
  const bool by_job = jobs >= p.prep_waves;
  const long long c64 = by_job ? static_cast<long long>(blockIdx.x)
                               : static_cast<long long>(blockIdx.x) * p.prep_waves + wave;
  const int job = static_cast<int>(by_job ? blockIdx.y * p.prep_waves + wave : blockIdx.y);
  if (c64 >= p.max_slots || job >= jobs) return;   // uniform per wave; no barriers below
  const int c = static_cast<int>(c64);
  // v-heads hv0 .. hv0 + prep_heads - 1, all of q/k head h
  const int hv0 = job * p.prep_heads;
  const int h = hv0 / p.ratio;
  if (p.short_limit > 0 && all_within(p, p.short_limit)) return;    // uniform
  int t0, n;                                       // n: 1..64, 0 past the last slot
  if (p.single) {
    int start, end;
    seq_range(p, 0, start, end);
    t0 = start + c * kChunk;
    n = min(kChunk, end - t0);
  } else if (FEW) {
    // slot c belongs to the sequence whose slots [excl, incl) hold it
    const FewSlots f = few_slots(p);
    const unsigned long long own = __ballot(f.excl <= c && c < f.incl);
    t0 = 0;
    n = 0;
    if (own != 0) {
      const int s = __builtin_ctzll(own);
      const long long first = __shfl(f.excl, s, 64);
      t0 = __shfl(f.start, s, 64) + static_cast<int>(c - first) * kChunk;
      n = min(kChunk, __shfl(f.end, s, 64) - t0);
    }
  } else {
    const i32x4 info = p.slot_info[c];
    t0 = info.y;
    n = info.z;
  }
  t0 = uniform(t0);
  n = uniform(n);
  if (n <= 0) return;                              // uniform per wave
  prep_chunk<false>(p, c, t0, n, hv0, h, p.prep_heads, lds_all[wave], nullptr, nullptr);
}

// ---------------------------------------------------------------------------
// 3. the scan: one workgroup per (sequence, v-head) and the whole state
// ---------------------------------------------------------------------------
// Four main waves, one per SIMD, and four helper waves, one beside each.
// Main wave w keeps 32 columns of the state in registers (all 128 keys: st[t]
// is the 32 x 32 tile of keys 32 t ..); its lane (m, g) = (lane % 32, lane /
// 32) holds column 32 w + perm32(m), register r of tile t the key 32 t + 16
// (r / 8) + 8 g + r % 8.  Registers 8 h .. 8 h + 7 of a tile are thus 8
// consecutive keys: the state's operand of a product over keys in either role
// (B of K S, A of S^T Q^T) against 16-byte pieces of K and Q rows, and every
// per-chunk result is the next product's operand in place.  Per chunk, with S
// its start state:
//   X      = V - diag(rk e^gamma) K S
//   Delta  = T diag(beta) X
//   O^T    = S^T Q^T diag(scale rq e^gamma) + Delta^T P^T
//   S     <- e^gamma_C S + K^T diag(rk e^(gamma_C - gamma)) Delta
// as bf16 MFMA (32x32x16): K, Q, V are bf16; S, X, Delta, T diag(beta) and
// P enter split into hi + lo, and a product x y is hi_x hi_y + hi_x lo_y +
// lo_x hi_y (the lo lo term is ~2^-16 relative and dropped).
//
// What bounds it is issue: on a SIMD an MFMA takes ~8 cycles of issue
// whatever its size and a VALU instruction ~4 (measured: two fp32 FMAs a wave
// fit under a 16x16x32 for free, six under a 32x32x16), and one wave alone
// issues an instruction every ~5.5 cycles.  So the larger product (half the
// instructions, half the LDS reads a column of the 16-column waves before
// it), and everything the chain over the chunks does not need off the main
// waves: their DMA (~1.7 k cycles a chunk held at the issue), K^T and P' tiles
// (~2.2 k) and Q norms (~0.4 k) take the helpers' issue slots.  Measured
// against eight 16-column waves that each did a share of everything, kernel
// trace: 64 x 512 tokens at 16/32 heads 429-463 -> 365-405 us, 12 ragged
// sequences of 7-2048 tokens there 191 -> 152 us, 16 x 1024 at 4/8 76
// (two workgroups of half a state each, on twice the CUs) -> 66 us; ~9.4 k cycles a
// chunk step.  With all CUs at it the clock falls under the MFMA load (64 x 512: 0.87
// PFLOP/s of bf16 products, where a plain 8192^3 product reaches 1.26).
//
// The waves share the chunk's K rows, Q rows and workspace slot, which the
// LDS DMA (global_load_lds_dwordx4: each lane's 16 bytes land at the wave's
// LDS base + 16 lane, no registers) brings into one of two LDS buffers while
// the chunk before runs on the other.  The operands with tokens as the
// contracted index come from products with a selector (a 32 x 32
// permutation), which moves a 32 x 32 tile's columns into the result layout
// exactly: V^T tiles (each main wave's own 32 columns of V, loaded into
// registers) and K^T tiles (helper w makes key tile w from the K rows in LDS
// and shares it through LDS).  Two barriers a chunk: the helpers' tiles made
// and the buffer's last reads before the second half; the next chunk landed.
constexpr int kScanWaves = 4;
constexpr int kScanThreads = 2 * 64 * kScanWaves;
constexpr int kTriDma = 2 * kTriBlocks * kBlk / 8 / 64;   // T diag(beta), hi and lo (12)
constexpr int kScaleDma = kScaleFloats / 4 / 64;  // row scales (2)
// K^T operand blocks of a chunk: (key tile t, token block kb), 64 lanes x 8 bf16
constexpr int kKtElems = 4 * 4 * kBlk;
// P' operand blocks (the six lower (row block, token block) ones), hi then lo
constexpr int kPElems = 2 * kTriBlocks * kBlk;

// A chunk's K and Q rows (256 bytes each) and T diag(beta).  The 16-byte
// piece p of row r is at position p ^ (r % 16) of the row: the 8 lanes the
// LDS serves together read one piece of 8 rows, on disjoint banks.
template <bool OUT> struct ScanIn;
template <> struct __attribute__((aligned(16))) ScanIn<true> {
  uint16_t Kr[kChunk * kDim];
  uint16_t Qr[kChunk * kDim];
  uint16_t T[2 * kTriBlocks * kBlk];
};
template <> struct __attribute__((aligned(16))) ScanIn<false> {  // without outputs: no Q
  uint16_t Kr[kChunk * kDim];
  uint16_t T[2 * kTriBlocks * kBlk];
};
struct __attribute__((aligned(16))) ScanScales {
  float row[kScaleFloats];
};
static_assert(2 * sizeof(ScanIn<true>) + 2 * sizeof(ScanScales) + 2 * (kKtElems + kPElems) +
                  4 * kChunk + 4 * kBlk <= 160 * 1024,
              "one scan workgroup per CU");

typedef __attribute__((address_space(1))) void global_void;
typedef __attribute__((address_space(3))) void lds_void;

// One wave's DMA instruction: lane l's 16 bytes from base + byte_off (the
// base the same for the whole workgroup, in scalar registers) to dst + 16 l
// (dst the same for the whole wave).
__device__ __forceinline__ void dma16_at(const void* base, unsigned byte_off, void* dst) {
  __builtin_amdgcn_global_load_lds((global_void*)(static_cast<const char*>(base) + byte_off),
                                   (lds_void*)dst, 16, 0, 0);
}

// Byte offset of element `item` of token row `row` (< 64) of a bf16 matrix
// whose rows are `step` (< 2^24) elements apart: a 24-bit product, one
// full-rate instruction where a 32-bit one takes four.
__device__ __forceinline__ unsigned row_bytes(int row, unsigned step, unsigned item) {
  return 2u * (__umul24(static_cast<unsigned>(row), step) + item);
}

// Wait for this wave's outstanding vector memory operations (its DMA among
// them): s_waitcnt vmcnt(0), the other counters left alone.
__device__ __forceinline__ void wait_vmem() { __builtin_amdgcn_s_waitcnt(0x0F70); }

// Operand label m (0..31) of a 32 x 32 result's row or column as the key (or
// state column) it stands for: result row 8 q + 4 g + e, register 4 q + e of
// lane group g, is key 16 (q / 2) + 8 g + 4 (q % 2) + e, so that a lane's
// registers 8 h .. 8 h + 7 are the keys 16 h + 8 g .. + 7.
__device__ __forceinline__ int perm32(int m) {
  return (m & 0x13) | ((m & 4) << 1) | ((m & 8) >> 1);
}

__device__ __forceinline__ s16x8 ld_op(const void* ptr) {
  return *reinterpret_cast<const s16x8*>(ptr);
}

// Registers 8 H .. 8 H + 7 of a result tile as hi and lo operand items.
template <int H>
__device__ __forceinline__ s16x8 split8(const f32x16& x, s16x8& lo) {
  s16x4 ha, la, hb, lb;
  split4(f32x4{x[8 * H], x[8 * H + 1], x[8 * H + 2], x[8 * H + 3]}, ha, la);
  split4(f32x4{x[8 * H + 4], x[8 * H + 5], x[8 * H + 6], x[8 * H + 7]}, hb, lb);
  lo = cat(la, lb);
  return cat(ha, hb);
}

// Registers 8 H .. 8 H + 7 as bf16 (rounded to nearest even; exact for
// values that came from bf16).
template <int H>
__device__ __forceinline__ s16x8 to_bf16x8(const f32x16& x) {
  const u32x4 w = {pack_bf16x2(x[8 * H], x[8 * H + 1]), pack_bf16x2(x[8 * H + 2], x[8 * H + 3]),
                   pack_bf16x2(x[8 * H + 4], x[8 * H + 5]), pack_bf16x2(x[8 * H + 6], x[8 * H + 7])};
  return __builtin_bit_cast(s16x8, w);
}

// Four 4-row runs of a result tile's rows (8 q + 4 g, q = 0..3) of a row of
// per-token scales: token 32 R + 8 q + 4 g + e in item 4 q + e.
__device__ __forceinline__ f32x16 row_scales(const float* row, int R, int g) {
  f32x16 s;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(row + 32 * R + 8 * q + 4 * g);
#pragma unroll
    for (int e = 0; e < 4; ++e) s[4 * q + e] = v[e];
  }
  return s;
}

// The Q rows' space where there is one.
__device__ __forceinline__ uint16_t* q_rows(ScanIn<true>& in) { return in.Qr; }
__device__ __forceinline__ uint16_t* q_rows(ScanIn<false>& in) { return in.Kr; }

// The per-workgroup constants of a scan.
struct ScanCtx {
  const uint16_t* k;
  const uint16_t* q;
  const uint16_t* v;
  uint16_t* out;
  const float* slot_base;      // the first chunk's slot
  size_t slot_step;            // floats from one chunk's slot to the next
  unsigned kstep, vstep;       // elements from one token's K / Q row (V row) to the next
  int start, end, nchunks;     // token range and chunks
  int H, HV, h, hv;
  bool values;
};

// Where chunk c's inputs come from (rows >= n repeat row n - 1).
struct ChunkSrc {
  const uint16_t* kbase;
  const uint16_t* qbase;
  const uint16_t* vbase;
  const float* slot;
  int n;
};

__device__ __forceinline__ ChunkSrc chunk_src(const ScanCtx& cx, int c) {
  const int tc = cx.start + c * kChunk;
  ChunkSrc s;
  s.kbase = cx.k + (static_cast<size_t>(tc) * cx.H + cx.h) * kDim;
  s.qbase = cx.q + (static_cast<size_t>(tc) * cx.H + cx.h) * kDim;
  s.vbase = cx.v + (static_cast<size_t>(tc) * cx.HV + cx.hv) * kDim;
  s.slot = cx.slot_base + c * cx.slot_step;
  s.n = min(kChunk, cx.end - tc);
  return s;
}

// Instruction j (0..3) of this wave's share of a K or Q chunk's 16: rows
// 4 i .. 4 i + 3, i = wave + 4 j, one 16-byte piece a lane (rows >= n repeat
// row n - 1).
__device__ __forceinline__ void dma_rows(const uint16_t* base, unsigned step, int n, int j,
                                         int wave, int lane, uint16_t* dst) {
  const int i = wave + kScanWaves * j;
  const unsigned piece = static_cast<unsigned>((lane & 15) ^ (lane >> 4) ^ (4 * (i & 3)));
  dma16_at(base, row_bytes(min(4 * i + (lane >> 4), n - 1), step, piece * 8), dst + i * 512);
}

// Part `part` (0..3) of wave `wave`'s (0..3) share of a chunk's DMA into In
// and Sc (SLOT: its slot too): a K and a Q row instruction, and one of the
// slot's.
template <bool OUT, bool SLOT = true>
__device__ __forceinline__ void issue_part(ScanIn<OUT>* __restrict__ In,
                                           ScanScales* __restrict__ Sc, const ScanCtx& cx,
                                           const ChunkSrc& s, int part, int wave, int lane) {
  dma_rows(s.kbase, cx.kstep, s.n, part, wave, lane, In->Kr);
  if constexpr (OUT) dma_rows(s.qbase, cx.kstep, s.n, part, wave, lane, In->Qr);
  if constexpr (SLOT) {
    static_assert(kTriDma == 3 * kScanWaves && kScaleDma <= kScanWaves, "T in parts 0..2");
    const int i = wave + kScanWaves * part;
    const unsigned off = static_cast<unsigned>(lane) * 16u;
    if (part < 3)
      dma16_at(s.slot + i * 256, off, In->T + i * 512);
    else if (wave < kScaleDma)                                // uniform per wave
      dma16_at(s.slot + i * 256, off, Sc->row + wave * 256);
  }
}

// The chunk's V for this wave's 32 columns, as the A operands of the selector products:
// vf[2 R + b2] is token 32 R + m, columns 32 w + 16 b2 + 8 g .. + 7 (rows
// >= n repeat row n - 1).
__device__ __forceinline__ void load_v(u32x4 (&vf)[4], const ScanCtx& cx, const ChunkSrc& s,
                                       int lane) {
  const int wave = wave_index();
  const int m = lane & 31, g = lane >> 5;
#pragma unroll
  for (int R = 0; R < 2; ++R) {
    const int row = 32 * R + m;
    const unsigned off = row_bytes(min(row, s.n - 1), cx.vstep, 32 * wave + 8 * g);
#pragma unroll
    for (int b2 = 0; b2 < 2; ++b2)
      vf[2 * R + b2] = *reinterpret_cast<const u32x4*>(
          reinterpret_cast<const char*>(s.vbase) + off + 32 * b2);
  }
}

// P' (the B operand blocks of Delta^T P'^T, hi then lo) from the chunk's K
// and Q rows.  Tile (it, jt): rows i = 16 it + c, tokens j = 16 jt + 4 g4 + e
// in lane (c, g4) = (lane % 16, lane / 16): items 4 (g4 / 2) + e of lane
// (i % 32, g4 % 2) of block (it / 2, jt).  Wave w makes tiles w, w + 4 and
// w + 8 of the ten lower ones and the two above the diagonal inside a block:
//   it = 0 1 2 3 | 1 3 2 3 | 2 3 0 2, jt = 0 1 2 3 | 0 0 0 1 | 1 2 1 3.
struct PTile {
  int it, jt;
  __device__ __forceinline__ PTile(int wave, int u) {
    constexpr unsigned kIt = 0x8eede4u, kJt = 0xd940e4u;      // 2 bits a tile
    it = (kIt >> (2 * (wave + 4 * u))) & 3;
    jt = (kJt >> (2 * (wave + 4 * u))) & 3;
  }
};

// Key block kb's product of a tile: operands from the rows' 16-byte pieces
// 4 kb + g4 (row r's at position piece ^ (r % 16)).
__device__ __forceinline__ void p_tile_ops(const uint16_t* Kr, const uint16_t* Qr, PTile pt,
                                           int kb, int lane, s16x8& ka, s16x8& qb) {
  const int c = lane & 15, g4 = lane >> 4;
  const unsigned at = (static_cast<unsigned>(c) * kDim + 8u * (g4 ^ c)) ^ (32u * kb);
  ka = ld_op(Kr + pt.jt * 16 * kDim + at);
  qb = ld_op(Qr + pt.it * 16 * kDim + at);
}

// A finished (K Q^T) tile, scaled and masked, into its blocks.
__device__ __forceinline__ void p_tile_store(const f32x4& acc, const ScanScales* Sc, PTile pt,
                                             int lane, uint16_t* Pb) {
  const int c = lane & 15, g4 = lane >> 4;
  const float gi = Sc->row[kRowGa + 16 * pt.it + c], gil = Sc->row[kRowGaLo + 16 * pt.it + c];
  const f32x4 gj = lds4(&Sc->row[kRowGa + 16 * pt.jt + 4 * g4]);
  const f32x4 gjl = lds4(&Sc->row[kRowGaLo + 16 * pt.jt + 4 * g4]);
  const f32x4 rkj = lds4(&Sc->row[kRowRk + 16 * pt.jt + 4 * g4]);
  const int lim = 16 * (pt.it - pt.jt) + c - 4 * g4;          // j <= i: e <= lim
  f32x4 pv;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float y = rkj[e] * decay(gi, gil, gj[e], gjl[e]) * acc[e];
    pv[e] = e <= lim ? y : 0.0f;
  }
  s16x4 hi, lo;
  split4(pv, hi, lo);
  uint16_t* const dst = Pb + tri_blk(pt.it >> 1, pt.jt) * kBlk +
                        (16 * (pt.it & 1) + c + 32 * (g4 & 1)) * 8 + 4 * (g4 >> 1);
  *reinterpret_cast<s16x4*>(dst) = hi;
  *reinterpret_cast<s16x4*>(dst + kTriBlocks * kBlk) = lo;
}

// What a chunk's second half needs of its K and Q rows, share w (0..3) of
// four.  First what the rows alone give: key tile w of K^T (lane (m, g): tokens
// 32 R + 8 q + 4 g + e of key 32 w + perm32(m), operand blocks (w, 2 R) and (w,
// 2 R + 1) of Kt), the products of the share's three P' tiles, and with the
// L2-norm 1 / |q_i| of Q rows 16 w .. + 15 into Qn.
template <bool OUT, bool L2>
__device__ __forceinline__ void side_products(const ScanIn<OUT>* __restrict__ In, uint16_t* Kt,
                                              float* Qn, const uint16_t* __restrict__ Sel, int w,
                                              int lane, f32x4 (&acc)[3]) {
  const int m = lane & 31, g = lane >> 5;
  const unsigned row0 = static_cast<unsigned>(m) * kDim + 8u * (g ^ (m & 15));
#pragma unroll
  for (int R = 0; R < 2; ++R) {
    f32x16 kt;
#pragma unroll
    for (int r = 0; r < 16; ++r) kt[r] = 0.0f;
#pragma unroll
    for (int h = 0; h < 2; ++h)
      kt = mfma32_bf16(ld_op(&In->Kr[(row0 ^ (16u * (2 * w + h))) + R * 32 * kDim]),
                       ld_op(&Sel[h * kBlk + lane * 8]), kt);
    uint16_t* const dst = Kt + (w * 4 + 2 * R) * kBlk + lane * 8;
    *reinterpret_cast<s16x8*>(dst) = to_bf16x8<0>(kt);
    *reinterpret_cast<s16x8*>(dst + kBlk) = to_bf16x8<1>(kt);
  }
  if constexpr (OUT) {
#pragma unroll
    for (int u = 0; u < 3; ++u) {
      acc[u] = f32x4{0, 0, 0, 0};
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        s16x8 ka, qb;
        p_tile_ops(In->Kr, In->Qr, PTile(w, u), kb, lane, ka, qb);
        acc[u] = mfma_bf16(ka, qb, acc[u]);
      }
    }
  }
  if constexpr (L2) {
    // four lanes a row (pieces 4 j + lane % 4: the lanes the LDS serves
    // together on disjoint banks)
    const int r = lane >> 2;
    const uint16_t* const qr = &In->Qr[(16 * w + r) * kDim];
    float q2 = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const u32x4 x = *reinterpret_cast<const u32x4*>(qr + 8 * ((4 * j + (lane & 3)) ^ r));
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float lo = __uint_as_float(x[i] << 16);
        const float hi = __uint_as_float(x[i] & 0xffff0000u);
        q2 = fmaf(hi, hi, fmaf(lo, lo, q2));
      }
    }
    q2 += __shfl_xor(q2, 1, 64);
    q2 += __shfl_xor(q2, 2, 64);
    if ((lane & 3) == 0) Qn[16 * w + r] = __builtin_amdgcn_rsqf(q2 + kL2Eps);
  }
}

// Then, with the chunk's scales, the share's P' tiles into Pb.
template <bool OUT>
__device__ __forceinline__ void side_store(const ScanScales* Sc, uint16_t* Pb, int w, int lane,
                                           const f32x4 (&acc)[3]) {
  if constexpr (OUT) {
#pragma unroll
    for (int u = 0; u < 3; ++u) p_tile_store(acc[u], Sc, PTile(w, u), lane, Pb);
  }
}

// Chunk ci of a helper wave: the side tiles from In and Sc, then the next
// chunk's DMA into InN and ScN (their last reads were in the chunk before).
// The pointers to the chunks' inputs are restrict: the compiler then knows
// that the DMA never writes what is read meanwhile, and waits for it only at
// the end.  Kt, Pb and Qn are not: the other waves access them within the
// call, on the other side of its barriers.
template <bool OUT, bool L2>
__device__ __forceinline__ void help_chunk(const ScanIn<OUT>* __restrict__ In,
                                           const ScanScales* __restrict__ Sc,
                                           ScanIn<OUT>* __restrict__ InN,
                                           ScanScales* __restrict__ ScN,
                                           uint16_t* Kt, uint16_t* Pb, float* Qn,
                                           const ScanCtx& cx,
                                           const uint16_t* __restrict__ Sel, int ci) {
  const int lane = threadIdx.x & 63;
  const int w = wave_index() - kScanWaves;
  f32x4 acc[3];
  side_products<OUT, L2>(In, Kt, Qn, Sel, w, lane, acc);
  side_store<OUT>(Sc, Pb, w, lane, acc);
  if (ci + 1 < cx.nchunks) {                                  // uniform
    // issued while the main waves finish their first half
    const ChunkSrc nsrc = chunk_src(cx, ci + 1);
    issue_part<OUT>(InN, ScN, cx, nsrc, 0, w, lane);
    issue_part<OUT>(InN, ScN, cx, nsrc, 1, w, lane);
    barrier_lds_no_dma();
    issue_part<OUT>(InN, ScN, cx, nsrc, 2, w, lane);
    issue_part<OUT>(InN, ScN, cx, nsrc, 3, w, lane);
    wait_vmem();                     // the next chunk's DMA has landed
  }
  barrier_lds_no_dma();
}

// Chunk ci of a main wave, from In and Sc (LAST: the last chunk, which may be
// a partial one); Kt: the K^T operand blocks; Pb: the P' operand blocks
// (OUT); Qn: the Q row scales (L2) -- written by the helper waves within the
// call, before the barrier ahead of their use, so not restrict; nor are In and
// Sc, whose slot another wave of the one-chunk kernel (SLOT_LATE) writes until a
// barrier behind the products that do not need it.  OUT: the outputs too (else
// only the state).  L2: the L2-norm.
//
// The output's intra-chunk term uses P = diag(rq) P' with
//   P'_ij = scale rk_j e^(gamma_i - gamma_j) (Q K^T)_ij,  j <= i,
// made by the helper waves from the chunk's K and Q rows: a (K Q^T) tile on
// bf16 MFMA (16x16x32) leaves each lane 4 consecutive j of one row i, half
// the 8 items of a lane of P' as the B operand of Delta^T P'^T.  The Q row
// scales rq = 1 / |q_i| (L2-norm) scale the output row:
// O = diag(rq) (diag(scale e^gamma) Q S + P' Delta).
template <bool OUT, bool L2, bool LAST, bool SLOT_LATE = false>
__device__ __forceinline__ void scan_chunk(const ScanIn<OUT>* In, const ScanScales* Sc,
                                           const uint16_t* Kt, const uint16_t* Pb,
                                           const float* Qn, const ScanCtx& cx,
                                           f32x16 (&st)[4], const uint16_t* __restrict__ Sel,
                                           int ci) {
  // The lane index, opaque to the compiler: it would keep every LDS and
  // global offset derived from it in a register across the chunks, more than
  // there are.
  int lane = threadIdx.x & 63;
  asm volatile("" : "+v"(lane));
  const int wave = wave_index();
  const int m = lane & 31;
  const int g = lane >> 5;

  // piece 2 b + g of row 32 R + m, at position (2 b + g) ^ (m % 16)
  const unsigned row0 = static_cast<unsigned>(m) * kDim + 8u * (g ^ (m & 15));
  auto k_op = [&](int b, int R) { return ld_op(&In->Kr[(row0 ^ (16u * b)) + R * 32 * kDim]); };

  // K S (token rows) and S^T Q^T (the output's first term, transposed), one
  // 16-key block of the state at a time; block b + 1's operands are read
  // while block b's products run.
  f32x16 x[2], o[2];
#pragma unroll
  for (int r = 0; r < 16; ++r) x[0][r] = x[1][r] = o[0][r] = o[1][r] = 0.0f;
  s16x8 ak[2][2], bq[2][2];
  auto read_ops = [&](int b, int set) {
#pragma unroll
    for (int R = 0; R < 2; ++R) {
      ak[set][R] = k_op(b, R);
      if constexpr (OUT) bq[set][R] = ld_op(&In->Qr[(row0 ^ (16u * b)) + R * 32 * kDim]);
    }
  };
  read_ops(0, 0);
  // V, ~3 k cycles ahead of its use (a chunk ahead, it holds registers through
  // the second half, where the most are live), issued behind the first LDS
  // reads and not where the compiler would, right before the use
  u32x4 vf[4];
  load_v(vf, cx, chunk_src(cx, ci), lane);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    const int set = b & 1;
    if (b < 7) read_ops(b + 1, set ^ 1);
    s16x8 sl;
    const s16x8 sh = (b & 1) ? split8<1>(st[b >> 1], sl) : split8<0>(st[b >> 1], sl);
#pragma unroll
    for (int R = 0; R < 2; ++R) {
      x[R] = mfma32_bf16(ak[set][R], sh, x[R]);
      if constexpr (OUT) o[R] = mfma32_bf16(sh, bq[set][R], o[R]);
    }
#pragma unroll
    for (int R = 0; R < 2; ++R) {
      x[R] = mfma32_bf16(ak[set][R], sl, x[R]);
      if constexpr (OUT) o[R] = mfma32_bf16(sl, bq[set][R], o[R]);
    }
  }

  if constexpr (SLOT_LATE) barrier_lds_no_dma();   // the slot is in LDS

  // X = V - diag(rk e^gamma) K S, V^T from the selector products; split
  s16x8 xh[4], xl[4];
#pragma unroll
  for (int R = 0; R < 2; ++R) {
    f32x16 v;
#pragma unroll
    for (int r = 0; r < 16; ++r) v[r] = 0.0f;
    if (cx.values) {                                          // uniform
      v = mfma32_bf16(__builtin_bit_cast(s16x8, vf[2 * R]), ld_op(&Sel[lane * 8]), v);
      v = mfma32_bf16(__builtin_bit_cast(s16x8, vf[2 * R + 1]), ld_op(&Sel[kBlk + lane * 8]), v);
    }
    const f32x16 xg = row_scales(Sc->row + kRowXg, R, g);
#pragma unroll
    for (int r = 0; r < 16; ++r) x[R][r] = v[r] - xg[r] * x[R][r];
    xh[2 * R] = split8<0>(x[R], xl[2 * R]);
    xh[2 * R + 1] = split8<1>(x[R], xl[2 * R + 1]);
  }

  // The state's decay of the second half, beside Delta's chains of products
  // (which leave the vector unit idle), where no output accumulators take the
  // registers (first segment launch of 1 x 16384 tokens at 4/8 heads 59.5 ->
  // 54.6 us; with outputs it spills).  The segment scan with outputs of a single
  // sequence spills all the same, 12-16 registers around the loop, and the plain one
  // behind the offsets kernel with the L2-norm 3.
  const float gl = Sc->row[kRowGl];
  if constexpr (!OUT) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) st[t][r] *= gl;
  }

  // Delta = T diag(beta) X (T lower triangular: token blocks kb < 2 R + 2)
  f32x16 d[2];
#pragma unroll
  for (int R = 0; R < 2; ++R) {
#pragma unroll
    for (int r = 0; r < 16; ++r) d[R][r] = 0.0f;
#pragma unroll
    for (int kb = 0; kb < 2 * R + 2; ++kb) {
      const s16x8 th = ld_op(&In->T[tri_blk(R, kb) * kBlk + lane * 8]);
      const s16x8 tl = ld_op(&In->T[(kTriBlocks + tri_blk(R, kb)) * kBlk + lane * 8]);
      d[R] = mfma32_bf16(th, xh[kb], d[R]);
      d[R] = mfma32_bf16(th, xl[kb], d[R]);
      d[R] = mfma32_bf16(tl, xh[kb], d[R]);
    }
  }

  // Delta as operand: A of Delta^T P^T and, scaled by ks, B of the update
  s16x8 dh[4], dl[4], eh[4], el[4];
#pragma unroll
  for (int R = 0; R < 2; ++R) {
    if constexpr (OUT) {
      dh[2 * R] = split8<0>(d[R], dl[2 * R]);
      dh[2 * R + 1] = split8<1>(d[R], dl[2 * R + 1]);
    }
    const f32x16 ks = row_scales(Sc->row + kRowKs, R, g);
#pragma unroll
    for (int r = 0; r < 16; ++r) d[R][r] *= ks[r];
    eh[2 * R] = split8<0>(d[R], el[2 * R]);
    eh[2 * R + 1] = split8<1>(d[R], el[2 * R + 1]);
  }

  barrier_lds_no_dma();              // the helpers' K^T and P' tiles are in LDS

  // S <- e^gamma_C S + K^T (ks (.) Delta), key tile t, and
  // O^T = rq (.) (qs (.) S^T Q^T + Delta^T P'^T): lane (m, g) ends with
  // columns 32 w + 16 h + 8 g .. + 7 of token 32 R + m, a 16-byte store each.
  // Eight groups of products, each two key tiles' of one token block and one
  // of O's six lower blocks (three independent chains), their operands read a
  // group ahead.
  float qs[2], rq[2];
  if constexpr (OUT) {
#pragma unroll
    for (int R = 0; R < 2; ++R) {
      qs[R] = Sc->row[kRowEg + 32 * R + m];
      if constexpr (L2) rq[R] = Qn[32 * R + m];
    }
  }
  // O's blocks in the order of the groups: (R, kb)
  constexpr int kOR[6] = {0, 1, 0, 1, 1, 1}, kOKb[6] = {0, 0, 1, 1, 2, 3};
  s16x8 ktop[2][2], pop[2][2];
  auto read_group = [&](int i, int set) {
#pragma unroll
    for (int u = 0; u < 2; ++u)
      ktop[set][u] = ld_op(&Kt[((2 * (i >> 2) + u) * 4 + (i & 3)) * kBlk + lane * 8]);
    if constexpr (OUT) {
      if (i < 6) {
        const int blk = tri_blk(kOR[i], kOKb[i]);
        pop[set][0] = ld_op(&Pb[blk * kBlk + lane * 8]);
        pop[set][1] = ld_op(&Pb[(kTriBlocks + blk) * kBlk + lane * 8]);
      }
    }
  };
  auto store_o = [&](int R) {
    const int c0 = cx.start + ci * kChunk;
    const int tok = 32 * R + m;
    if constexpr (L2) {
#pragma unroll
      for (int r = 0; r < 16; ++r) o[R][r] *= rq[R];
    }
    if (!LAST || tok < cx.end - c0) {
      char* const dst = reinterpret_cast<char*>(
                            cx.out + (static_cast<size_t>(c0) * cx.HV + cx.hv) * kDim) +
                        row_bytes(tok, cx.vstep, 32 * wave + 8 * g);
      *reinterpret_cast<s16x8*>(dst) = to_bf16x8<0>(o[R]);
      *reinterpret_cast<s16x8*>(dst + 32) = to_bf16x8<1>(o[R]);
    }
  };
  read_group(0, 0);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int set = i & 1, t = 2 * (i >> 2), kb = i & 3;
    if (i < 7) read_group(i + 1, set ^ 1);
    if (OUT && kb == 0) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int r = 0; r < 16; ++r) st[t + u][r] *= gl;
    }
    if constexpr (OUT) {
      if (i < 2) {
#pragma unroll
        for (int r = 0; r < 16; ++r) o[i][r] *= qs[i];
      }
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) st[t + u] = mfma32_bf16(ktop[set][u], eh[kb], st[t + u]);
    if constexpr (OUT) {
      if (i < 6) o[kOR[i]] = mfma32_bf16(dh[kOKb[i]], pop[set][0], o[kOR[i]]);
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) st[t + u] = mfma32_bf16(ktop[set][u], el[kb], st[t + u]);
    if constexpr (OUT) {
      if (i < 6) {
        o[kOR[i]] = mfma32_bf16(dh[kOKb[i]], pop[set][1], o[kOR[i]]);
        o[kOR[i]] = mfma32_bf16(dl[kOKb[i]], pop[set][0], o[kOR[i]]);
      }
      if (i == 4) store_o(0);
      if (i == 6) store_o(1);
    }
    __builtin_amdgcn_sched_barrier(0);
  }

  if constexpr (!LAST) barrier_lds_no_dma();   // the next chunk's inputs have landed; this
}                                              // one's LDS reads are done

// The state between memory and the main waves' registers, through LDS.  A lane's
// register runs are 16 bytes of a column of its own: straight from or to memory
// an instruction touches 32 columns, in 64 pieces of 16 bytes.  So the
// instructions move two whole columns each (512 bytes, 32 lanes), and the layouts
// are exchanged in 16 KiB of LDS a wave, the 16-byte piece p of column r at
// position p ^ perm32(r): the lanes that the LDS serves together are on disjoint
// banks both ways.  Columns 24 .. 31 may lie apart.  Captured calls, GPU time: 4 x
// 64 tokens at 4/8 heads 17.1 -> 16.2 us (16.4 with two workgroups of half a state
// each), without a start state 16.0 -> 15.0; 64 x 64 at 16/32 126 -> 115.
struct StateRows {
  char* lo;                    // columns 0 .. 23
  char* hi;                    // columns 24 .. 31
  __device__ __forceinline__ char* at(int r, int pos) const {
    return (r < 24 ? lo + r * 512 : hi + (r - 24) * 512) + pos * 16;
  }
};

// src, dst: the wave's first column (k-last: 128 consecutive keys a column).
__device__ __forceinline__ void load_state(f32x16 (&st)[4], const float* src, const StateRows& rows,
                                           int lane) {
  const int half = lane >> 5, pos = lane & 31;
  f32x4 v[16];
#pragma unroll
  for (int i = 0; i < 16; ++i)
    v[i] = *reinterpret_cast<const f32x4*>(src + (2 * i + half) * kDim + 4 * pos);
#pragma unroll
  for (int i = 0; i < 16; ++i)
    *reinterpret_cast<f32x4*>(rows.at(2 * i + half, pos ^ perm32(2 * i + half))) = v[i];
  wave_sync_lds();
  const int m = lane & 31, g = lane >> 5;
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(
          rows.at(perm32(m), (8 * t + 4 * (q >> 1) + 2 * g + (q & 1)) ^ m));
#pragma unroll
      for (int e = 0; e < 4; ++e) st[t][4 * q + e] = x[e];
    }
}

__device__ __forceinline__ void store_state(float* dst, const f32x16 (&st)[4],
                                            const StateRows& rows) {
  int lane = threadIdx.x & 63;
  asm volatile("" : "+v"(lane));      // as in scan_chunk
  const int m = lane & 31, g = lane >> 5;
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *reinterpret_cast<f32x4*>(
          rows.at(perm32(m), (8 * t + 4 * (q >> 1) + 2 * g + (q & 1)) ^ m)) =
          f32x4{st[t][4 * q], st[t][4 * q + 1], st[t][4 * q + 2], st[t][4 * q + 3]};
  wave_sync_lds();
  const int half = lane >> 5, pos = lane & 31;
#pragma unroll
  for (int i = 0; i < 16; ++i)
    *reinterpret_cast<f32x4*>(dst + (2 * i + half) * kDim + 4 * pos) =
        *reinterpret_cast<const f32x4*>(rows.at(2 * i + half, pos ^ perm32(2 * i + half)));
}

// The end state of a scan: k-last fp32 (element (k, c) at c * 128 + k), or,
// for a transition M (identity start), as the A operand blocks of the
// combine's product M S (16x16x32): for row tile t and column block kb, 64
// lanes x 8 bf16, hi then lo (block ((t * 4 + kb) * 2 + hl) * 512).  Wave w's
// columns are block kb = w: the selector products of its state read as an
// operand with the columns as rows give lane (m, g) the columns 32 w + 16 h +
// 8 g .. + 7 of key 32 t2 + perm32(m), the 8 items (lane group 2 h + g) of the
// combine's row i of tile t, 32 (t / 2) + 8 (i / 4) + 4 (t % 2) + i % 4 being
// that key (state_key).
__device__ __forceinline__ void store_end(float* st_out, bool transition, const f32x16 (&st)[4],
                                          const s16x8 (&sel)[2]) {
  int lane = threadIdx.x & 63;
  asm volatile("" : "+v"(lane));      // as in scan_chunk
  const int wave = wave_index();
  const int m = lane & 31;
  const int g = lane >> 5;
  if (!transition) {
    float* const dst = st_out + static_cast<size_t>(32 * wave + perm32(m)) * kDim + 8 * g;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<f32x4*>(dst + 32 * t + 16 * (q >> 1) + 4 * (q & 1)) =
            f32x4{st[t][4 * q], st[t][4 * q + 1], st[t][4 * q + 2], st[t][4 * q + 3]};
    return;
  }
  uint16_t* ma = reinterpret_cast<uint16_t*>(st_out);
  const int key = perm32(m);
  const int tb = (key >> 2) & 1, i = 4 * (key >> 3) + (key & 3);
#pragma unroll
  for (int t2 = 0; t2 < 4; ++t2) {
    s16x8 hi[2], lo[2];
    hi[0] = split8<0>(st[t2], lo[0]);
    hi[1] = split8<1>(st[t2], lo[1]);
    f32x16 mh, ml;
#pragma unroll
    for (int r = 0; r < 16; ++r) mh[r] = ml[r] = 0.0f;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      mh = mfma32_bf16(hi[h], sel[h], mh);
      ml = mfma32_bf16(lo[h], sel[h], ml);
    }
    uint16_t* const blk = ma + ((2 * t2 + tb) * 4 + wave) * 2 * kBlk;
    uint16_t* const d0 = blk + (i + 16 * g) * 8;
    uint16_t* const d1 = blk + (i + 16 * (2 + g)) * 8;
    *reinterpret_cast<s16x8*>(d0) = to_bf16x8<0>(mh);
    *reinterpret_cast<s16x8*>(d1) = to_bf16x8<1>(mh);
    *reinterpret_cast<s16x8*>(d0 + kBlk) = to_bf16x8<0>(ml);
    *reinterpret_cast<s16x8*>(d1 + kBlk) = to_bf16x8<1>(ml);
  }
}

// Grid: (unit, q/k head) pairs in groups of 8 times the GVA ratio.  Workgroup
// b serves pair 8 (b / (8 ratio)) + b % 8 and v-head (b / 8) % ratio of its
// q/k head: the workgroups that read the same K and Q are dispatched 8 apart,
// all to XCD b % 8 (workgroups go to the XCDs round-robin), and share its L2
// copy.  A unit is a sequence, or with SEG a role of one segment of a
// sequence.  The first segment launch (OUT false, no outputs) runs
// segment 0 from the sequence's state (end: seg_S[1]) and segments
// 1 .. nseg-2 from a zero start (end: seg_B) and from the identity without
// values (end: seg_M, as the combine's operand); the second (OUT) runs every
// segment from its start (segment 0: the sequence's state -- in place, seg_S[0],
// the first launch's copy of it -- then seg_S) with the outputs, the last one's
// end being the new state (seg_unit).
template <bool FEW, bool SEG, bool OUT, bool L2, bool FUSE>
__device__ __forceinline__ void scan_body(Params p) {
  static_assert(OUT || SEG, "only segments run without outputs");
  static_assert(!FUSE || (!FEW && !SEG && OUT), "the one-chunk kernel runs plain scans");
  static_assert(OUT || !L2, "the L2-norm scales outputs only");
  // separate LDS objects, so that the compiler sees that the DMA into one
  // never writes what the chunk reads from another
  __shared__ ScanIn<OUT> In0, In1;
  __shared__ ScanScales S0, S1;
  __shared__ __attribute__((aligned(16))) uint16_t Kt[kKtElems];
  __shared__ __attribute__((aligned(16))) uint16_t Pb[OUT ? kPElems : 8];
  __shared__ float Qn[L2 ? kChunk : 1];    // 1 / |q_i| of the chunk's Q rows (L2-norm)
  __shared__ __attribute__((aligned(16))) uint16_t Sel[2 * kBlk];   // the selectors
  const long long b = blockIdx.x;
  const int ratio = p.ratio;
  const long long pair = (b / (8LL * ratio)) * 8 + (b & 7);
  const int jr = static_cast<int>((b >> 3) % ratio);
  // units the grid covers: with SEG the launch's bound, each workgroup
  // finding its sequence's segment below (those past the batch's exit)
  const long long units = SEG ? (OUT ? p.nseg : seg_units1(p.nseg, p.N))
                              : static_cast<long long>(p.N);
  if (pair >= units * p.H) return;                              // uniform per workgroup
  if (p.short_limit > 0 && all_within(p, p.short_limit)) return;  // uniform
  const int unit = static_cast<int>(pair / p.H);
  const int h = static_cast<int>(pair % p.H);
  const int hv = h * ratio + jr;
  const int lane = threadIdx.x & 63;
  const int wave = wave_index();
  const int m = lane & 31;
  const int g = lane >> 5;
  const size_t blk = static_cast<size_t>(kDim) * kDim;

  // State registers; k-last storage: 8 consecutive keys are two 16-byte
  // vectors.
  f32x16 st[4];
  const int c = 32 * wave + perm32(m);
  auto load_st = [&](const float* src) {           // null: zeros
#pragma unroll
    for (int t = 0; t < 4; ++t) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int key = 32 * t + 16 * (q >> 1) + 8 * g + 4 * (q & 1);
        const f32x4 v = src != nullptr ? *reinterpret_cast<const f32x4*>(
                                             src + static_cast<size_t>(c) * kDim + key)
                                       : f32x4{0, 0, 0, 0};
#pragma unroll
        for (int e = 0; e < 4; ++e) st[t][4 * q + e] = v[e];
      }
    }
  };
  // role: start state, values, where the end state goes
  const float* st_in = nullptr;       // null: zeros (or the identity)
  bool identity = false, values = true, pass_through = false;
  float* st_out;
  float* st_keep = nullptr;           // where the start is copied to
  int s = 0, start, end, slot0 = 0, nchunks = 0;
  // the sequence's chunk slots (never more than its range holds, and never
  // more slots than the workspace has, whatever cu_seqlens contains)
  auto seq_slots = [&](int sq, int& base, int& count) {
    if (p.single) {
      base = 0;
      count = (end - start + kChunk - 1) / kChunk;
    } else if (FEW) {
      const FewSlots f = few_slots(p);
      base = static_cast<int>(__shfl(f.excl, sq, 64));
      count = static_cast<int>(__shfl(f.incl, sq, 64)) - base;
    } else {
      base = p.offs[sq];
      count = p.offs[sq + 1] - base;
    }
  };
  if (SEG) {
    const SegSeqs f = seg_seqs<OUT>(p);
    const unsigned long long own = __ballot(lane < p.N && f.u_excl <= unit && unit < f.u_incl);
    if (own == 0) return;                         // past the batch's units (uniform)
    s = __builtin_ctzll(own);                     // uniform: lane reads, no shuffles
    const int nseg = __builtin_amdgcn_readlane(f.nseg, s);
    const int g0 = __builtin_amdgcn_readlane(f.seg_excl, s);   // the sequence's first segment
    if (g0 + nseg > p.nseg) return;               // past the workspace's (a malformed batch)
    const int u = unit - __builtin_amdgcn_readlane(f.u_excl, s);
    start = __builtin_amdgcn_readlane(f.start, s);
    end = __builtin_amdgcn_readlane(f.end, s);
    const size_t sh = static_cast<size_t>(s) * p.HV + hv;        // the sequence's state
    auto seg_blk = [&](float* base, int sg) {
      return base + (static_cast<size_t>(sg) * p.HV + hv) * blk;
    };
    const SegUnit un = seg_unit(OUT, nseg, u, p.state != nullptr && p.state == p.new_state);
    const int j = un.seg;
    if (un.from == SegBlock::kState)
      st_in = p.state ? p.state + sh * blk : nullptr;
    else if (un.from == SegBlock::kStart)
      st_in = seg_blk(p.seg_S, g0 + j);
    if constexpr (OUT) {
      st_out = un.to == SegBlock::kNewState ? p.new_state + sh * blk : nullptr;
      pass_through = j > 0;
    } else {
      identity = un.from == SegBlock::kIdentity;
      values = !identity;
      st_out = seg_blk(un.to == SegBlock::kStart     ? p.seg_S
                       : un.to == SegBlock::kZeroEnd ? p.seg_B
                                                     : p.seg_M,
                       g0 + un.to_seg);
      if (un.keep_start) st_keep = seg_blk(p.seg_S, g0 + j);
    }
    int base, count;
    seq_slots(s, base, count);
    const int first = j * p.seg_chunks;
    slot0 = base + first;
    // the last segment takes the rest (at most seg_chunks, but the whole
    // sequence when a malformed batch runs every sequence as one segment)
    nchunks = j == nseg - 1 ? count - first : min(p.seg_chunks, count - first);
    start = min(end, start + first * kChunk);
    if (nchunks > 0) end = min(end, start + nchunks * kChunk);
  } else {
    s = unit;
    seq_range(p, s, start, end);
    st_in = p.state ? p.state + (static_cast<size_t>(s) * p.HV + hv) * blk : nullptr;
    st_out = p.new_state + (static_cast<size_t>(s) * p.HV + hv) * blk;
    if constexpr (FUSE)
      nchunks = end > start ? 1 : 0;    // every sequence is one chunk (at most 64 tokens in all)
    else
      seq_slots(s, slot0, nchunks);
  }

  // The identity start of a transition gives column c the unit vector of key c,
  // so that its end column is that start key's column of M.
  const float* const src = st_in != nullptr && (end > start || pass_through) && wave < kScanWaves
                               ? st_in : nullptr;  // helper waves hold no columns
  if constexpr (OUT && !FUSE) {
    load_st(nullptr);
    // LDS that nothing else uses before the scan's first barrier
    const StateRows rows = {reinterpret_cast<char*>(wave == 0   ? In1.Kr
                                                    : wave == 1 ? q_rows(In1)
                                                    : wave == 2 ? Kt
                                                                : In1.T),
                            reinterpret_cast<char*>(wave == 0   ? In1.Kr + 24 * 256
                                                    : wave == 1 ? q_rows(In1) + 24 * 256
                                                    : wave == 2 ? Kt + 24 * 256
                                                                : Pb)};
    if (src != nullptr) load_state(st, src + 32 * wave * kDim, rows, lane);   // uniform
  } else {
    load_st(src);
  }
  if constexpr (!OUT) {
    if (identity) {
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          st[t][r] = 32 * t + 16 * (r >> 3) + 8 * g + (r & 7) == c ? 1.0f : 0.0f;
    }
  }
  // selector operands: Sel_h[k][j] = (16 h + k == perm32(j)) over a 16-long k
  // block
  s16x8 sel[2];
#pragma unroll
  for (int h2 = 0; h2 < 2; ++h2)
#pragma unroll
    for (int e = 0; e < 8; ++e) sel[h2][e] = perm32(m) == 16 * h2 + 8 * g + e ? 0x3f80 : 0;

  if constexpr (SEG && !OUT) {
    if (st_keep != nullptr && wave < kScanWaves) store_end(st_keep, false, st, sel);
  }

  // No tokens: a sequence ends in zeros, as the reference; a segment with no
  // chunk slots (a malformed batch whose slots ran past the workspace's)
  // passes its start through (transition: the identity, zero-start end:
  // zeros), and so does the sequence's end state.
  if (nchunks <= 0) {
    if (st_out != nullptr && wave < kScanWaves) {
      if (!SEG) {
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r) st[t][r] = 0.0f;
      }
      store_end(st_out, identity, st, sel);
    }
    return;
  }
  start = uniform(start);
  end = uniform(end);
  nchunks = uniform(nchunks);
  slot0 = uniform(slot0);
  ScanCtx cx;
  cx.k = p.k;
  cx.q = p.q;
  cx.v = p.v;
  cx.out = p.out;
  cx.slot_base = p.slots + (static_cast<size_t>(slot0) * p.HV + hv) * kSlotFloats;
  cx.slot_step = static_cast<size_t>(p.HV) * kSlotFloats;
  cx.kstep = static_cast<unsigned>(p.H) * kDim;
  cx.vstep = static_cast<unsigned>(p.HV) * kDim;
  cx.start = start;
  cx.end = end;
  cx.nchunks = nchunks;
  cx.H = p.H;
  cx.HV = p.HV;
  cx.h = h;
  cx.hv = hv;
  cx.values = values;

  // The end state behind the last chunk step, whose middle barrier was the last
  // use of the K and Q rows.
  auto store_last = [&]() {
    if (st_out == nullptr) return;                             // uniform
    if constexpr (OUT) {
      uint16_t* const base = wave == 0   ? In0.Kr
                             : wave == 1 ? In0.Qr
                             : wave == 2 ? In1.Kr
                                         : In1.Qr;
      const StateRows rows = {reinterpret_cast<char*>(base),
                              reinterpret_cast<char*>(base + 24 * 256)};
      store_state(st_out + 32 * wave * kDim, st, rows);
    } else {
      store_end(st_out, identity, st, sel);
    }
  };

  const ChunkSrc first_src = chunk_src(cx, 0);
  if (wave < 2) *reinterpret_cast<s16x8*>(&Sel[wave * kBlk + lane * 8]) = sel[wave];
  if constexpr (FUSE) {
    // Main waves bring the chunk's K and Q rows by DMA; helper wave 0 prepares
    // its slot in LDS, and beside it the other helpers make the K^T and Q K^T
    // tiles and the main waves their products of the rows and the state.
    static_assert(sizeof(PrepLds) <= sizeof(ScanIn<OUT>), "the preparation fits a buffer");
    if (wave == kScanWaves) {                                                  // uniform
      prep_chunk<true>(p, 0, start, end - start, hv, h, 1, *reinterpret_cast<PrepLds*>(&In1),
                       In0.T, S0.row);             // with the first barrier
      barrier_lds_no_dma();
      barrier_lds_no_dma();
      return;
    }
    if (wave > kScanWaves) {                                                   // uniform
      constexpr int kSide = kScanWaves - 1;        // three waves, share 3 the first one's too
      const int w = wave - kScanWaves - 1;
      f32x4 acc[3], acc3[3];
      barrier_lds_no_dma();
      side_products<OUT, L2>(&In0, Kt, Qn, Sel, w, lane, acc);
      if (w == 0) side_products<OUT, L2>(&In0, Kt, Qn, Sel, kSide, lane, acc3);
      barrier_lds_no_dma();
      side_store<OUT>(&S0, Pb, w, lane, acc);
      if (w == 0) side_store<OUT>(&S0, Pb, kSide, lane, acc3);
      barrier_lds_no_dma();
      return;
    }
#pragma unroll
    for (int part = 0; part < 4; ++part)
      issue_part<OUT, false>(&In0, &S0, cx, first_src, part, wave, lane);
    wait_vmem();
    barrier_lds_no_dma();
    scan_chunk<OUT, L2, true, true>(&In0, &S0, Kt, Pb, Qn, cx, st, Sel, 0);
    store_last();
    return;
  }
  if (wave >= kScanWaves) {                                                    // uniform
#pragma unroll
    for (int part = 0; part < 4; ++part)
      issue_part<OUT>(&In0, &S0, cx, first_src, part, wave - kScanWaves, lane);
    // With the L2-norm the helpers' first half is the longer one: their
    // instructions first (12 ragged sequences at 16/32 heads with it 173.5 ->
    // 165.0 us a call; without the norm the main waves' chain is, 1-2% slower
    // so).
    if constexpr (L2) __builtin_amdgcn_s_setprio(2);
    wait_vmem();
    barrier_lds_no_dma();
    for (int ci = 0; ci < nchunks; ci += 2) {
      help_chunk<OUT, L2>(&In0, &S0, &In1, &S1, Kt, Pb, Qn, cx, Sel, ci);
      if (ci + 1 < nchunks)                                                    // uniform
        help_chunk<OUT, L2>(&In1, &S1, &In0, &S0, Kt, Pb, Qn, cx, Sel, ci + 1);
    }
    return;
  }
  wait_vmem();                       // the state, here rather than in each chunk step
  barrier_lds_no_dma();
  for (int ci = 0; ci < nchunks - 1; ++ci)
    scan_chunk<OUT, L2, false>((ci & 1) ? &In1 : &In0, (ci & 1) ? &S1 : &S0, Kt, Pb, Qn, cx, st,
                               Sel, ci);
  scan_chunk<OUT, L2, true>((nchunks & 1) ? &In0 : &In1, (nchunks & 1) ? &S0 : &S1, Kt, Pb, Qn,
                            cx, st, Sel, nchunks - 1);
  store_last();
}

template <bool FEW, bool SEG, bool OUT, bool L2>
__global__ __launch_bounds__(kScanThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
void scan_kernel(Params p) {
  scan_body<FEW, SEG, OUT, L2, false>(p);
}

// Prefills whose tokens all fit one chunk: each (sequence, v-head)
// workgroup prepares its sequence's chunk in LDS and scans it, in one launch.
// Its time is a chain: the loads, one wave's preparation, and the chunk step's
// rest; the step's first half and its tiles run beside the preparation (64
// tokens in a graph, 4/8 heads 14.2 -> 13.1 us, 16/32 with the L2-norm 14.9 -> 13.4;
// 13.3 and 14.2 with two workgroups of half a state and four waves preparing).
template <bool L2>
__global__ __launch_bounds__(kScanThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
void one_chunk_kernel(Params p) {
  scan_body<false, false, true, L2, true>(p);
}

// ---------------------------------------------------------------------------
// 4. segments: chain each sequence's segment starts
// ---------------------------------------------------------------------------
// The first segment launch leaves, per (sequence, v-head), S_1 and for each
// middle segment j its transition M_j (as the A operand blocks of M S, bf16
// hi/lo) and zero-start end B_j.  Combine: S_{j+1} = M_j S_j + B_j for j = 1
// .. nseg-2, segment after segment, as bf16 MFMA with S_j split into hi + lo.
// One workgroup per (sequence, v-head, 16 state columns); wave w computes row
// tile w (rows state_key(w, i / 4) + i % 4, the rows
// of M's tile w) and hands its rows of S_j to the other waves as half of the
// B operand's k block w / 2 through LDS (two buffers: one barrier a step).  A step is short (12 MFMAs a wave), so each wave's M
// blocks and B tile are loaded three steps ahead, into three register sets
// used in turn.  Every workgroup reads all of M_j: the eight of a (sequence,
// v-head) are numbered hv + 8k within the sequence's (HV rounded up to 8
// between them), so all of them run on XCD hv % 8 (workgroups go to the XCDs
// round-robin) and read M_j from its L2 after the first.
constexpr int kCombWaves = 8;

struct CombStage {
  s16x8 ma[4][2];                             // [k block][hi, lo] of row tile w
  f32x4 bt;                                   // B_j rows of row tile w
};

__global__ __launch_bounds__(64 * kCombWaves) void seg_combine_kernel(Params p) {
  __shared__ s16x8 Sop[2][4][2][64];          // [buffer][k block][hi, lo][lane]
  const int hv_pad = (p.HV + 7) & ~7;
  const int per_seq = hv_pad * 8;
  const int sq = static_cast<int>(blockIdx.x) / per_seq;
  const int hv = static_cast<int>(blockIdx.x) % hv_pad;
  const int c0 = static_cast<int>(blockIdx.x) % per_seq / hv_pad * 16;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int col = lane & 15;
  const int g4 = lane >> 4;
  const size_t blk = static_cast<size_t>(kDim) * kDim;
  if (sq >= p.N || hv >= p.HV) return;        // padding (uniform)
  // the sequence's segments: one sequence has the workspace's (its chain
  // starts without reading cu_seqlens; steps past a shorter sequence's last
  // segment chain values nothing reads); several count theirs
  int nseg = p.nseg, g0 = 0;
  if (p.N > 1) {
    const SegSeqs f = seg_seqs<true>(p);
    nseg = __builtin_amdgcn_readlane(f.nseg, sq);
    g0 = __builtin_amdgcn_readlane(f.seg_excl, sq);
  }
  if (nseg < 3 || g0 + nseg > p.nseg) return; // nothing to chain; past the workspace's
  const int last = nseg - 2;                  // steps j = 1 .. last
  const size_t tile = static_cast<size_t>(c0 + col) * kDim + state_key(wave, g4);
  auto seg_blk = [&](const float* base, int j) {
    return base + (static_cast<size_t>(g0 + j) * p.HV + hv) * blk;
  };
  // S_1, this wave's row tile in the MFMA result layout
  f32x4 S = *reinterpret_cast<const f32x4*>(seg_blk(p.seg_S, 1) + tile);
  auto load = [&](int j, CombStage& cs) {     // past the last step: the last one's again
    j = j < last ? j : last;
    const uint16_t* M = reinterpret_cast<const uint16_t*>(seg_blk(p.seg_M, j));
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int hl = 0; hl < 2; ++hl)
        cs.ma[kb][hl] =
            *reinterpret_cast<const s16x8*>(M + (((wave * 4 + kb) * 2 + hl) * kBlk + lane * 8));
    cs.bt = *reinterpret_cast<const f32x4*>(seg_blk(p.seg_B, j) + tile);
  };
  auto step = [&](int j, CombStage& cs) {
    const int buf = j & 1;
    s16x4 hi, lo;
    split4(S, hi, lo);
    const int item = (wave & 1) * 4;
    uint16_t* sh16 = reinterpret_cast<uint16_t*>(&Sop[buf][wave >> 1][0][lane]);
    uint16_t* sl16 = reinterpret_cast<uint16_t*>(&Sop[buf][wave >> 1][1][lane]);
    *reinterpret_cast<s16x4*>(sh16 + item) = hi;
    *reinterpret_cast<s16x4*>(sl16 + item) = lo;
    block_sync_lds();
    f32x4 acc = cs.bt;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      const s16x8 bh = Sop[buf][kb][0][lane];
      const s16x8 bl = Sop[buf][kb][1][lane];
      acc = mfma_bf16(cs.ma[kb][0], bh, acc);
      acc = mfma_bf16(cs.ma[kb][0], bl, acc);
      acc = mfma_bf16(cs.ma[kb][1], bh, acc);
    }
    S = acc;
    *reinterpret_cast<f32x4*>(const_cast<float*>(seg_blk(p.seg_S, j + 1)) + tile) = S;
    load(j + 3, cs);                          // this set's next use: three steps on
  };
  CombStage s0, s1, s2;
  load(1, s0);
  load(2, s1);
  load(3, s2);
  for (int j = 1; j <= last; j += 3) {        // uniform
    step(j, s0);
    if (j + 1 <= last) step(j + 1, s1);
    if (j + 2 <= last) step(j + 2, s2);
  }
}

bool aligned(const void* ptr, uintptr_t a) {
  return (reinterpret_cast<uintptr_t>(ptr) & (a - 1)) == 0;
}

size_t align256(size_t x) { return (x + 255) & ~static_cast<size_t>(255); }

// Workspace: chunk offsets [N + 1] int32, slot table [max_slots] x 16 bytes,
// the v-head slots [max_slots, HV, kSlotFloats] fp32, then with segments
// their S, B and M blocks; each part 256-byte aligned.
size_t offsets_bytes(long long N) { return align256(static_cast<size_t>(N + 1) * sizeof(int32_t)); }

size_t slot_info_bytes(long long L, long long N) {
  return align256(static_cast<size_t>(max_slots(L, N)) * sizeof(i32x4));
}

size_t slots_bytes(long long L, long long N, long long HV) {
  return align256(static_cast<size_t>(max_slots(L, N)) * HV * kSlotFloats * sizeof(float));
}

// Segments.  A sequence's plain scan is a chain of chunk steps on HV
// workgroups; with few sequences and v-heads that leaves most of the GPU idle
// (16384 tokens at 8 v-heads: 256 steps on 8 CUs), so each sequence is cut
// into segments of len chunks scanned at once: the first launch runs 2 nseg
// - 3 units of a sequence of nseg segments (HV workgroups each), the second
// nseg, one workgroup per CU, each of len chunk steps, and the combine nseg -
// 2 small steps.  The host knows only the total tokens and the sequence
// count, so it plans for sequences of the mean length: the length is the one
// that minimises the estimated critical path, (rounds of the first launch +
// rounds of the second) x len chunk steps + (nseg - 2) combine steps + the
// two more launches, with a round of kCUs workgroups and a chunk step
// costing kStepPerCombine combine steps; the batch is cut when that beats its
// plain scan, (rounds of N HV workgroups) x chunks x kStepPerCombine: from 6
// chunks a sequence at N HV = 8.  A chunk step takes 3.2-3.5 us and a combine step
// 1.2, a ratio of 3; 5 gives the better lengths (captured calls with 5 / 3 / no
// segments, us: 2048 tokens at 4/8 heads 56.2 / 57.2 / 116.6, 16384 there 145.4 /
// 150.1 / 841.5, 8192 at 16/32 213.1 / 218.6 / 454.0) but cuts sequences of 6 and 7
// chunks, and some batches, that the plain scan takes faster (384 tokens at 4/8
// 36.2 / 31.5 / 31.5, 448 36.7 / 34.9 / 34.8, 4 x 448 46.4 / 37.0 / 36.6, 8 x 1024 87.5 /
// 87.0 / 73.7; from 512 tokens on one sequence gains by it).  The kernels count each sequence's
// segments from cu_seqlens (so sequences shorter or longer than the mean get as
// many as they need), in one wave: at most kFewSeqs sequences.
constexpr long long kSegMaxHeads = 256;  // N HV workgroups that fill the GPU unsegmented
constexpr long long kSegMinLen = 2;
constexpr long long kCUs = 256;
constexpr long long kStepPerCombine = 5;
constexpr long long kSegLaunches = 8;    // the segment path's two more launches

struct SegPlan {
  long long len;    // chunks a segment (the mean sequence if not cut)
  long long cost;   // estimated critical path, combine steps; -1: cannot be cut
};

SegPlan seg_plan(long long L, long long N, long long HV) {
  const long long chunks = ((L + kChunk - 1) / kChunk + N - 1) / N;   // a sequence, mean
  SegPlan best{chunks, -1};
  for (long long len = kSegMinLen; 3 * len <= chunks; ++len) {
    const long long n = (chunks + len - 1) / len;
    const long long rounds =
        (N * (2 * n - 3) * HV + kCUs - 1) / kCUs + (N * n * HV + kCUs - 1) / kCUs;
    const long long cost = rounds * len * kStepPerCombine + (n - 2) + kSegLaunches;
    if (best.cost < 0 || cost < best.cost) best = SegPlan{len, cost};
  }
  return best;
}

// Prefills past the token path whose tokens all fit one chunk (so every
// sequence is one chunk), with at most 128 (sequence, v-head) workgroups: one
// launch in which each prepares its chunk in LDS and scans it -- no workspace
// round trip and one launch instead of two or three (captured calls against
// those: 64 tokens at 4/8 heads 12.3 / 14.9 us, 4 x 16 at 16/32 13.3 / 22.1).  Past 128
// it depends on the lengths, which the host does not know: 5 x 12 tokens at 16/32
// 14.0 / 21.0 us, but 30 x 2 at 4/8, which the token kernel takes, 15.3 / 13.9.
bool fused_prefill(long long L, long long N, long long HV) {
  return L > kSmallTokens && L <= kChunk && N >= 1 && 2 * N * HV <= kCUs;
}

bool use_segments(long long L, long long N, long long HV) {
  if (N < 1 || N > kFewSeqs || N * HV > kSegMaxHeads) return false;
  const SegPlan plan = seg_plan(L, N, HV);
  const long long chunks = ((L + kChunk - 1) / kChunk + N - 1) / N;
  const long long whole = (N * HV + kCUs - 1) / kCUs * chunks * kStepPerCombine;
  return plan.cost >= 0 && plan.cost < whole;
}

long long seg_chunks(long long L, long long N, long long HV) { return seg_plan(L, N, HV).len; }

// Segments the workspace holds: one sequence's exactly; for several, the most
// a well-formed batch can have, sum(ceil(chunks_i / len)) <= (chunks + N
// (len - 1)) / len with chunks <= max_slots.  The kernels skip the segments of
// a (malformed) batch past this count.
long long num_segments(long long L, long long N, long long HV) {
  const long long len = seg_chunks(L, N, HV);
  if (N == 1) return ((L + kChunk - 1) / kChunk + len - 1) / len;
  return (max_slots(L, N) + N * (len - 1)) / len;
}

// Per segment and v-head one 128 x 128 fp32 block (S, B and M each).
size_t seg_blocks_bytes(long long L, long long N, long long HV) {
  return align256(static_cast<size_t>(num_segments(L, N, HV)) * HV * kDim * kDim * sizeof(float));
}

size_t workspace_bytes(long long L, long long N, long long H, long long HV) {
  (void)H;
  size_t bytes = offsets_bytes(N) + slot_info_bytes(L, N) + slots_bytes(L, N, HV);
  if (use_segments(L, N, HV)) bytes += 3 * seg_blocks_bytes(L, N, HV);
  return bytes;
}

}  // namespace gdn_pf

using namespace gdn_pf;

// One launch of the decode kernel's variable-length mode over the prefill's
// packed inputs: grid (row tiles x v-heads of a q/k head, q/k heads,
// sequences), one row per 16-lane group and one wave per workgroup for a few
// heads, four waves for more.
static hipError_t small_prefill(const void* q, const void* k, const void* v, const float* state,
                                const float* A_log, const void* a, const float* dt_bias,
                                const void* b, const int32_t* cu_seqlens, float scale,
                                void* output, float* new_state, int L, int N, int H, int HV,
                                bool l2, int short_limit, hipStream_t stream) {
  constexpr int kNs = 1;
  constexpr int kPolicy = gdn::kPolicyDefault;   // the next decode step re-reads the state
  const unsigned ratio = static_cast<unsigned>(HV / H);
  const unsigned h_ratio = static_cast<unsigned>(H) | (ratio << 16);
  const auto* q16 = static_cast<const uint16_t*>(q);
  const auto* k16 = static_cast<const uint16_t*>(k);
  const auto* v16 = static_cast<const uint16_t*>(v);
  const auto* a16 = static_cast<const uint16_t*>(a);
  const auto* b16 = static_cast<const uint16_t*>(b);
  auto* out16 = static_cast<uint16_t*>(output);
  if (static_cast<long long>(N) * HV <= 16) {
    constexpr int kW = 1;
    const dim3 grid(ratio * (kDim / (gdn::kLaneGroups * kNs * kW)), H, N);
    auto* kern = l2 ? gdn::gdn_decode_k128<kNs, kW, true, kPolicy, false, true, true>
                    : gdn::gdn_decode_k128<kNs, kW, false, kPolicy, false, true, true>;
    hipLaunchKernelGGL(kern, grid, dim3(64 * kW), 0, stream, state, q16, k16, v16, a16, b16,
                       h_ratio, 0, A_log, dt_bias, out16, new_state, scale, cu_seqlens, L,
                       short_limit);
  } else {
    constexpr int kW = 4;
    const dim3 grid(ratio * (kDim / (gdn::kLaneGroups * kNs * kW)), H, N);
    auto* kern = l2 ? gdn::gdn_decode_k128<kNs, kW, true, kPolicy, false, true, true>
                    : gdn::gdn_decode_k128<kNs, kW, false, kPolicy, false, true, true>;
    hipLaunchKernelGGL(kern, grid, dim3(64 * kW), 0, stream, state, q16, k16, v16, a16, b16,
                       h_ratio, 0, A_log, dt_bias, out16, new_state, scale, cu_seqlens, L,
                       short_limit);
  }
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Fixed workspace of gdn_prefill_noalloc: a file-scope device array, so each
// GPU holds its own copy, at its own address, from the library's load on
// that GPU until the process ends.  Host code never passes the array's name
// to a kernel (on the host it is only a stand-in for the symbol): the
// device address comes from hipGetSymbolAddress, once per device, with that
// device current, and is cached per device.
// ---------------------------------------------------------------------------
constexpr size_t kScratchBytes = GDN_PREFILL_NOALLOC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
static std::atomic<void*> g_scratch_ptr[kMaxDevices];
static std::mutex g_scratch_mutex;

// Device address of the current device's scratch array.
static hipError_t current_scratch(void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  void* ptr = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (ptr == nullptr) {
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    ptr = g_scratch_ptr[dev].load(std::memory_order_relaxed);
    if (ptr == nullptr) {
      e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
      if (e != hipSuccess) return e;
      if (ptr == nullptr) return hipErrorInvalidSymbol;
      g_scratch_ptr[dev].store(ptr, std::memory_order_release);
    }
  }
  *out = ptr;
  return hipSuccess;
}

// fixed_scratch: the workspace is the current device's scratch array
// (workspace / workspace_size are ignored); sizes whose workspace exceeds it
// return hipErrorOutOfMemory before anything is launched.
static int prefill_impl(const void* q, const void* k, const void* v, const float* state,
                const float* A_log, const void* a, const float* dt_bias, const void* b,
                const int32_t* cu_seqlens, float scale, void* output, float* new_state,
                int total_seq_len, int num_seqs, int H, int HV, int K, int V,
                int use_qk_l2norm, void* workspace, size_t workspace_size,
                void* hip_stream, void* const* events, bool fixed_scratch = false) {
  if (total_seq_len < 0 || num_seqs < 0 || H <= 0 || HV <= 0 || HV % H != 0)
    return hipErrorInvalidValue;
  if (K != kDim || V != kDim) return hipErrorInvalidValue;
  if (HV > 65535) return hipErrorInvalidValue;      // grid y
  if (H > 32767) return hipErrorInvalidValue;       // packed in 15 bits for the token kernel
  if (num_seqs == 0) return hipSuccess;
  if (!cu_seqlens || !A_log || !dt_bias || !new_state || (!workspace && !fixed_scratch))
    return hipErrorInvalidValue;
  if (total_seq_len > 0 && (!q || !k || !v || !a || !b || !output))
    return hipErrorInvalidValue;
  const size_t need = workspace_bytes(total_seq_len, num_seqs, H, HV);
  if (fixed_scratch) {
    if (need > kScratchBytes) return hipErrorOutOfMemory;
    workspace = nullptr;                               // set once validation has passed
  } else if (workspace_size < need) {
    return hipErrorInvalidValue;
  }
  if (!aligned(q, 16) || !aligned(k, 16) || !aligned(v, 16) || !aligned(output, 16) ||
      !aligned(new_state, 16) || !aligned(state, 16) || !aligned(workspace, 256) ||
      !aligned(A_log, 4) || !aligned(dt_bias, 4) || !aligned(cu_seqlens, 4) ||
      !aligned(a, 2) || !aligned(b, 2))
    return hipErrorInvalidValue;
  if (state != nullptr && state == new_state) {
    // in place is fine: a workgroup of the token path and of the plain scan
    // reads its state slice before writing it, and no two workgroups share a
    // slice; in segments, whose first and last are scanned by different
    // workgroups of one launch, the first starts from a copy that the launch
    // before made
  } else if (state != nullptr) {
    const uintptr_t s0 = reinterpret_cast<uintptr_t>(state);
    const uintptr_t d0 = reinterpret_cast<uintptr_t>(new_state);
    const size_t bytes = static_cast<size_t>(num_seqs) * HV * kDim * kDim * sizeof(float);
    if (s0 < d0 + bytes && d0 < s0 + bytes) return hipErrorInvalidValue;
  }
  const long long slots = max_slots(total_seq_len, num_seqs);
  if (slots > 0x7fffffffLL || num_seqs > 0x7fffffff - 1) return hipErrorInvalidValue;
  if ((static_cast<long long>(num_seqs) * H + 7) / 8 * 8 * (HV / H) > 0x7fffffffLL)  // scan grid
    return hipErrorInvalidValue;
  if (fixed_scratch) {
    const hipError_t e = current_scratch(&workspace);
    if (e != hipSuccess) return e;
  }

  Params p;
  p.q = static_cast<const uint16_t*>(q);
  p.k = static_cast<const uint16_t*>(k);
  p.v = static_cast<const uint16_t*>(v);
  p.state = state;
  p.A_log = A_log;
  p.a = static_cast<const uint16_t*>(a);
  p.dt_bias = dt_bias;
  p.b = static_cast<const uint16_t*>(b);
  p.cu_seqlens = cu_seqlens;
  p.out = static_cast<uint16_t*>(output);
  p.new_state = new_state;
  char* ws = static_cast<char*>(workspace);
  int32_t* offs = reinterpret_cast<int32_t*>(ws);
  i32x4* slot_info = reinterpret_cast<i32x4*>(ws + offsets_bytes(num_seqs));
  p.offs = offs;
  p.slot_info = slot_info;
  p.slots = reinterpret_cast<float*>(ws + offsets_bytes(num_seqs) +
                                     slot_info_bytes(total_seq_len, num_seqs));
  p.seg_chunks = 0;
  p.nseg = 0;
  p.seg_S = p.seg_B = p.seg_M = nullptr;
  if (use_segments(total_seq_len, num_seqs, HV)) {
    char* sg = reinterpret_cast<char*>(p.slots) + slots_bytes(total_seq_len, num_seqs, HV);
    const size_t blocks = seg_blocks_bytes(total_seq_len, num_seqs, HV);
    p.seg_chunks = static_cast<int>(seg_chunks(total_seq_len, num_seqs, HV));
    p.nseg = static_cast<int>(num_segments(total_seq_len, num_seqs, HV));
    p.seg_S = reinterpret_cast<float*>(sg);
    p.seg_B = reinterpret_cast<float*>(sg + blocks);
    p.seg_M = reinterpret_cast<float*>(sg + 2 * blocks);
  }
  p.scale = scale;
  p.L = total_seq_len;
  p.N = num_seqs;
  p.H = H;
  p.HV = HV;
  p.ratio = HV / H;
  p.l2norm = use_qk_l2norm != 0;
  p.single = num_seqs == 1;
  p.few = few_seqs(total_seq_len, num_seqs, HV);
  p.max_slots = slots;
  p.short_limit = maybe_all_short(total_seq_len, num_seqs) ? kSmallTokens : 0;
  p.prep_heads = prep_split(slots, HV) ? 1 : p.ratio;
  p.prep_waves = slots * (HV / p.prep_heads) <= kPrepSpreadMaxWaves ? 1 : kPrepWaves;

  hipStream_t stream = static_cast<hipStream_t>(hip_stream);
  // events[i] (optional) is recorded before launch i and events[3] after the last
  auto mark = [&](int i) -> hipError_t {
    return events ? hipEventRecord(static_cast<hipEvent_t>(events[i]), stream) : hipSuccess;
  };
  if (total_seq_len <= kSmallTokens && num_seqs <= 65535) {   // grid z
    // token-by-token path: the three intervals of the timed form are the
    // (empty) offsets and preparation steps and the one launch
    hipError_t e = mark(0);
    if (e == hipSuccess) e = mark(1);
    if (e == hipSuccess) e = mark(2);
    if (e != hipSuccess) return e;
    e = small_prefill(q, k, v, state, A_log, a, dt_bias, b, cu_seqlens, scale, output,
                      new_state, total_seq_len, num_seqs, H, HV, use_qk_l2norm != 0, 0, stream);
    if (e == hipSuccess) e = mark(3);
    return e;
  }
  // One workgroup per (sequence or segment role, v-head), in groups of 8
  // (unit, q/k head) pairs times the GVA ratio.
  auto scan_grid = [&](long long units) {
    return dim3(static_cast<unsigned>((units * H + 7) / 8 * 8 * p.ratio));
  };
  if (fused_prefill(total_seq_len, num_seqs, HV)) {
    // one launch (the timed form's intervals as on the token path)
    hipError_t e = mark(0);
    if (e == hipSuccess) e = mark(1);
    if (e == hipSuccess) e = mark(2);
    if (e != hipSuccess) return e;
    p.short_limit = 0;
    auto* fused = p.l2norm ? one_chunk_kernel<true> : one_chunk_kernel<false>;
    hipLaunchKernelGGL(fused, scan_grid(num_seqs), dim3(kScanThreads), 0, stream, p);
    e = hipGetLastError();
    if (e == hipSuccess) e = mark(3);
    return e;
  }
  hipError_t e = mark(0);
  if (e != hipSuccess) return e;
  if (p.short_limit > 0) {
    // A batch whose sequences may all be short: the token-by-token kernel
    // first, running only if every sequence has at most kSmallTokens tokens
    // (decided on the device from cu_seqlens); the chunkwise kernels after it
    // return at once in that case and run the whole batch otherwise.
    e = small_prefill(q, k, v, state, A_log, a, dt_bias, b, cu_seqlens, scale, output,
                      new_state, total_seq_len, num_seqs, H, HV, use_qk_l2norm != 0,
                      p.short_limit, stream);
    if (e != hipSuccess) return e;
  }
  if (!p.single && !p.few)
    hipLaunchKernelGGL(chunk_offsets_kernel, dim3(1), dim3(kThreads), 0, stream, p, offs,
                       slot_info);
  e = hipGetLastError();
  if (e == hipSuccess) e = mark(1);
  if (e != hipSuccess) return e;
  if (slots > 0) {
    auto* prep = p.few ? prep_kernel<true> : prep_kernel<false>;
    const int jobs = HV / p.prep_heads;
    const int w = p.prep_waves;
    const dim3 grid = jobs >= w ? dim3(static_cast<unsigned>(slots), (jobs + w - 1) / w)
                                : dim3(static_cast<unsigned>((slots + w - 1) / w), jobs);
    hipLaunchKernelGGL(prep, grid, dim3(64 * w), 0, stream, p);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  e = mark(2);
  if (e != hipSuccess) return e;
  if (p.seg_chunks > 0) {
    // segments: transitions and zero-start ends, the starts, then every
    // segment with its outputs (grids: the workspace's segments bound the
    // batch's units; workgroups past them exit)
    auto* scan1 = p.few ? scan_kernel<true, true, false, false>
                        : scan_kernel<false, true, false, false>;
    hipLaunchKernelGGL(scan1, scan_grid(seg_units1(p.nseg, num_seqs)), dim3(kScanThreads), 0,
                       stream, p);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(seg_combine_kernel,
                       dim3(static_cast<unsigned>(num_seqs * ((HV + 7) & ~7) * 8)),
                       dim3(64 * kCombWaves), 0, stream, p);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    auto* scan = p.few ? (p.l2norm ? scan_kernel<true, true, true, true>
                                   : scan_kernel<true, true, true, false>)
                       : (p.l2norm ? scan_kernel<false, true, true, true>
                                   : scan_kernel<false, true, true, false>);
    hipLaunchKernelGGL(scan, scan_grid(p.nseg), dim3(kScanThreads), 0, stream, p);
  } else {
    auto* scan = p.few ? (p.l2norm ? scan_kernel<true, false, true, true>
                                   : scan_kernel<true, false, true, false>)
                       : (p.l2norm ? scan_kernel<false, false, true, true>
                                   : scan_kernel<false, false, true, false>);
    hipLaunchKernelGGL(scan, scan_grid(num_seqs), dim3(kScanThreads), 0, stream, p);
  }
  e = hipGetLastError();
  if (e == hipSuccess) e = mark(3);
  return e;
}

extern "C" {

size_t gdn_prefill_workspace_bytes(int total_seq_len, int num_seqs, int H, int HV) {
  if (total_seq_len < 0 || num_seqs < 0 || H <= 0 || HV <= 0 || HV % H != 0) return 0;
  return workspace_bytes(total_seq_len, num_seqs, H, HV);
}

int gdn_prefill(const void* q, const void* k, const void* v, const float* state,
                const float* A_log, const void* a, const float* dt_bias, const void* b,
                const int32_t* cu_seqlens, float scale, void* output, float* new_state,
                int total_seq_len, int num_seqs, int H, int HV, int K, int V,
                int use_qk_l2norm, void* workspace, size_t workspace_size,
                void* hip_stream) {
  return prefill_impl(q, k, v, state, A_log, a, dt_bias, b, cu_seqlens, scale, output,
                      new_state, total_seq_len, num_seqs, H, HV, K, V, use_qk_l2norm, workspace,
                      workspace_size, hip_stream, nullptr);
}

int gdn_prefill_timed(const void* q, const void* k, const void* v, const float* state,
                      const float* A_log, const void* a, const float* dt_bias, const void* b,
                      const int32_t* cu_seqlens, float scale, void* output, float* new_state,
                      int total_seq_len, int num_seqs, int H, int HV, int K, int V,
                      int use_qk_l2norm, void* workspace, size_t workspace_size,
                      void* hip_stream, void* const* events) {
  if (events == nullptr) return hipErrorInvalidValue;
  for (int i = 0; i < 4; ++i)
    if (events[i] == nullptr) return hipErrorInvalidValue;
  return prefill_impl(q, k, v, state, A_log, a, dt_bias, b, cu_seqlens, scale, output,
                      new_state, total_seq_len, num_seqs, H, HV, K, V, use_qk_l2norm, workspace,
                      workspace_size, hip_stream, events);
}

int gdn_prefill_noalloc(const void* q, const void* k, const void* v, const float* state,
                        const float* A_log, const void* a, const float* dt_bias, const void* b,
                        const int32_t* cu_seqlens, float scale, void* output, float* new_state,
                        int total_seq_len, int num_seqs, int H, int HV, int K, int V,
                        int use_qk_l2norm, void* hip_stream) {
  return prefill_impl(q, k, v, state, A_log, a, dt_bias, b, cu_seqlens, scale, output,
                      new_state, total_seq_len, num_seqs, H, HV, K, V, use_qk_l2norm, nullptr,
                      0, hip_stream, nullptr, true);
}

int gdn_prefill_token_path_max_tokens(void) { return kSmallTokens; }

int gdn_prefill_dispatches(int total_seq_len, int num_seqs, int HV) {
  if (num_seqs <= 0 || total_seq_len < 0 || HV <= 0) return 0;
  if (total_seq_len <= kSmallTokens && num_seqs <= 65535) return 1;
  if (fused_prefill(total_seq_len, num_seqs, HV)) return 1;
  const int offsets = num_seqs == 1 || few_seqs(total_seq_len, num_seqs, HV) ? 0 : 1;
  const int token = maybe_all_short(total_seq_len, num_seqs) ? 1 : 0;
  if (use_segments(total_seq_len, num_seqs, HV)) return token + offsets + 4;
  return token + offsets + 2;
}

int gdn_prefill_abi_version(void) { return 6; }

}  // extern "C"
