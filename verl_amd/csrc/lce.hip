// Fused vocab-projection log-prob / entropy head for gfx950.
//
// Forward : logits tiles are produced by the MFMA tile engine and consumed in registers by an
//           online-softmax epilogue (running max, sum exp, sum z*exp, label logit and, on request,
//           sum exp^2 per token).  The [tokens, vocab] logits are not needed afterwards; on request
//           they are also written out in fp32 as a cache for the backward pass.
// Backward: per vocabulary chunk, d_logits is formed as one bf16 [tokens, vocab_chunk] panel,
//           either from the cached logits (a streaming pass) or from logits tiles recomputed by
//           the tile engine; the same engine then forms
//           d_hidden (+)= panel . W[chunk]  and  d_weight[chunk] = panel^T . hidden  in one launch.
//
// Arithmetic follows LinearCrossEntropy (verl/utils/kernel/linear_cross_entropy.py:40-116) /
// efficient_entropy_forward+backward (verl/utils/kernel/kernels.py:563-753, :1512-1723): bf16
// products, fp32 accumulation, logits scaled by 1/temperature in fp32, fp32 softmax state.
#include <stdlib.h>

#include <atomic>
#include <mutex>
#include <vector>

#include "common.h"
#include "gemm_core.h"

namespace vamd {

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;
constexpr float kNegBig = -1.0e30f;  // stands in for -inf so that (x - x) and 0 * x stay finite
// What a column past the end of the vocabulary holds in place of its product.  Times any sensible
// log2(e) / temperature it stays below kNegBig, the running maximum's start value (or overflows to -inf, which the
// maximum ignores as well): the maximum is never taken from it, so its exponent is hugely negative against every
// maximum there can be and it contributes exactly 0 to the sums (0 times a finite number).
constexpr float kNoColumn = -3.0e38f;

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Optional per-kernel timing for benchmarks: when enabled, every head kernel launch (from any
// thread: autograd runs backward on its own) is bracketed by a pair of HIP events on the launch
// stream.
enum : int { kTagForward = 0, kTagMerge = 1, kTagRecompute = 2, kTagDGrad = 3, kTagDLogits = 4, kNumTags = 5 };
struct TimedLaunch {
  int tag;
  hipEvent_t start, stop;
};
static std::atomic<bool> g_timing_on{false};
static std::mutex g_timed_mu;
static std::vector<TimedLaunch> g_timed;

struct ScopedTiming {
  hipStream_t s;
  TimedLaunch t;
  bool on;
  ScopedTiming(int tag, hipStream_t stream) : s(stream), on(g_timing_on.load()) {
    if (!on) return;
    t.tag = tag;
    if (hipEventCreate(&t.start) != hipSuccess || hipEventCreate(&t.stop) != hipSuccess) {
      on = false;
      return;
    }
    (void)hipEventRecord(t.start, s);
  }
  ~ScopedTiming() {
    if (!on) return;
    (void)hipEventRecord(t.stop, s);
    std::lock_guard<std::mutex> lock(g_timed_mu);
    g_timed.push_back(t);
  }
};

// =============================================================================================
// Forward
// =============================================================================================
// How the logits tiles (token tile x vocabulary tile) of a forward launch are shared out over the workgroups.
//
// splits: one round of workgroups, each with one token tile and one of `splits` equal ranges of the vocabulary.  Right when
//   token tiles x splits comes close to the CU count; 45 token tiles (5 splits) leave 31 of 256 CUs idle, 86 tiles
//   (2 splits) leave 84, and 129 tiles run at half rate.
// bands: the token tiles are cut into bands of 8 (then 4, 2, 1 for what is left), and a band of R tiles is walked by the
//   P workgroups of an XCD together: R token tiles x P / R vocabulary tiles per round, so that they share operand slabs
//   through that XCD's L2 as they do with splits.  Bands go to the XCDs eight at a time while there are eight (a wave);
//   the rounds of what is left form one sequence, of which each XCD takes an equal share.  A workgroup whose share crosses
//   into another band writes out its softmax state and starts afresh.  Within a share the part of the later band, which
//   begins at the start of the vocabulary, comes first: then all XCDs walk the vocabulary together, in two groups that are
//   a fixed distance apart, and the weight comes out of HBM about twice per wave instead of once per band (in order of
//   the sequence 21503 x 3584 x 152064 took 16.95 instead of 16.41 ms: on a board at its power limit traffic is time).
constexpr int kXcds = 8;
struct FwdPlan {
  int tok_tiles, voc_tiles;
  int splits;     // 0: bands
  int group;      // bands: P, workgroups per XCD (a multiple of 8)
  int waves;      // bands: eight full bands each, one per XCD
  int count[4];   // bands: rounds of a band of 1, 2, 4, 8 token tiles
  int rounds;     // bands: rounds of all bands after the waves together, below 2^27
  int few_cols;   // not 0: lce_forward_few_kernel, `splits` workgroups of this many columns each

  // Everything a workgroup asks of the plan is additions, shifts and comparisons of uniform 32-bit values: it is asked
  // with a tile's accumulators in registers, where a division would spill them.
  struct Band {
    // place among the bands after the waves, first token tile, log2 of its token tiles, rounds, first round
    int index, first, log2_rows, count, start;
    __host__ __device__ __forceinline__ int rows() const { return 1 << log2_rows; }
  };
  __host__ __device__ __forceinline__ int bands() const {  // after the waves
    const int left = tok_tiles - 64 * waves;
    return (left >> 3) + ((left >> 2) & 1) + ((left >> 1) & 1) + (left & 1);
  }
  __host__ __device__ __forceinline__ Band first_band() const {
    Band b{0, 64 * waves, 3, count[3], 0};
    shrink(b);
    return b;
  }
  // the band after b; past the last one its count is 0 and its start is `rounds`
  __host__ __device__ __forceinline__ void next(Band& b) const {
    b.first += b.rows();
    b.start += b.count;
    ++b.index;
    shrink(b);
  }
  __host__ __device__ __forceinline__ void shrink(Band& b) const {
    const int left = tok_tiles - b.first;
    if (left >= 8) return;
    b.log2_rows = left >= 4 ? 2 : left >= 2 ? 1 : 0;
    b.count = left <= 0 ? 0 : left >= 4 ? count[2] : left >= 2 ? count[1] : count[0];
  }
  // the first band that ends after round q
  __device__ __forceinline__ Band band_of_round(int q) const {
    Band b = first_band();
    while (b.count > 0 && q >= b.start + b.count) next(b);
    return b;
  }
  __device__ __forceinline__ int share_begin(int xcd) const { return (rounds * xcd) >> 3; }
  // Where the state of (band, XCD, workgroup of the XCD) goes, in rows of 256 tokens: first the bands of the waves, then
  // the others.  Those and the XCDs are walked in order, so index + xcd is different for every pair that meets.
  __device__ __forceinline__ int64_t wave_slot(int wave, int xcd, int member) const {
    return (int64_t)(kXcds * wave + xcd) * group + member;
  }
  __device__ __forceinline__ int64_t slot(int band_index, int xcd, int member) const {
    return (int64_t)(kXcds * waves + band_index + xcd) * group + member;
  }
  __host__ __device__ __forceinline__ int64_t slots() const {
    return splits ? (int64_t)splits * tok_tiles : (int64_t)(kXcds * waves + bands() + kXcds) * group;
  }
};
static_assert(kXcds == 8, "share_begin() divides by shifting, a wave is 64 token tiles");

struct FwdArgs {
  Operand hidden;  // R operand: [n_tokens][H]
  Operand weight;  // C operand: [vocab][H]
  const int64_t* labels;
  int n_tokens, vocab, k_slabs;
  FwdPlan plan;
  float scale2;      // log2(e) / temperature
  float rcp_t;       // 1 / temperature
  float4* partials;  // [plan.slots()][256] : (max in the log2 domain, sum e, sum e x with x = hidden . weight, label logit)
  float* z_cache;    // optional [n_tokens][vocab] fp32 logits / temperature, kept for the backward
  float* pi2_partials;  // optional [plan.slots()][256] : sum of e^2 relative to the same max
  int stream_from;      // lce_forward_few_kernel: stream_from()
};

// The tiles of one workgroup.  The ways of sharing out are kernels of their own: with both in one kernel the split
// walk, whose token tile never changes, carried the bands' lookups and the state's write-out through its tile loop, with 41
// scalar registers spilled (16384 x 3584 x 152064 12.50 ms, apart 12.47; 3300 x 896 x 151936, in bands, 706 and 699 us).
// Splits whose last token tile leaves wavefronts without rows, which skip the products, are a third: with that in the kernel,
// launches without such wavefronts took 0.4 to 0.6 % longer (us: 2048 x 896 x 151936 439.6, apart 437.5; 21503 x 4096 x
// 128256 15738, apart 15601).
enum Walk { kSplits, kSplitsIdle, kBands, kWalks };

// splits: one range of the vocabulary for one token tile
template <Walk WALK>
struct FwdSched {
  int k_slabs, tn, vt_begin, ntiles;
  int64_t slot;  // where the state goes

  __device__ __forceinline__ void init(const FwdPlan& p, int slabs, int wg) {
    k_slabs = slabs;
    // bands of 8 token tiles x all splits per XCD
    const int band = 8 * p.splits, b = wg / band, first = b * 8, w = wg - b * band;
    const int rows = (p.tok_tiles - first) < 8 ? (p.tok_tiles - first) : 8;
    const int sp = w / rows;
    tn = first + w % rows;
    vt_begin = (int)(((int64_t)sp * p.voc_tiles) / p.splits);
    ntiles = (int)(((int64_t)(sp + 1) * p.voc_tiles) / p.splits) - vt_begin;
    slot = (int64_t)sp * p.tok_tiles + tn;
  }
  __device__ __forceinline__ int count() const { return ntiles; }
  __device__ __forceinline__ void tile(int i, int& r0, int& c0) const {
    r0 = tn * kTile;
    c0 = (vt_begin + i) * kTile;
  }
  __device__ __forceinline__ int slab0(int) const { return 0; }
  __device__ __forceinline__ int slabs(int) const { return k_slabs; }
  __device__ __forceinline__ bool rows_outside(int row, int extent) const {
    return WALK == kSplitsIdle && tn * kTile + row >= extent;
  }
};

// bands: the workgroup's column of every band its XCD's share of the rounds touches
template <>
struct FwdSched<kBands> {
  const FwdPlan* plan;
  int k_slabs, ntiles;
  int xcd, member, wave_count;  // this XCD, workgroup within it, its tiles of a wave
  FwdPlan::Band band0;          // the band its share starts in

  struct Place {
    int tn, vt;    // token tile, vocabulary tile
    int64_t slot;  // where the state goes
  };
  struct Column {
    int first, count;  // first vocabulary tile, and how many; they are group >> log2_rows apart
  };
  __device__ __forceinline__ Column column(const FwdPlan::Band& b) const {
    const int q0 = plan->share_begin(xcd) - b.start, q1 = plan->share_begin(xcd + 1) - b.start;
    const int lo = q0 > 0 ? q0 : 0, hi = q1 < b.count ? q1 : b.count, cols = plan->group >> b.log2_rows;
    const int first = (member >> b.log2_rows) + cols * lo;
    int n = hi > lo ? hi - lo : 0;  // the last round of a band may have fewer columns than workgroups
    if (n > 0 && first + cols * (n - 1) >= plan->voc_tiles) --n;
    return Column{first, n};
  }
  __device__ __forceinline__ void init(const FwdPlan& p, int slabs, int wg) {
    plan = &p;
    k_slabs = slabs;
    xcd = wg / p.group;
    member = wg % p.group;
    band0 = p.band_of_round(p.share_begin(xcd));
    const int cols = p.group >> 3;
    wave_count = p.voc_tiles > (member >> 3) ? (p.voc_tiles - (member >> 3) + cols - 1) / cols : 0;
    ntiles = p.waves * wave_count;
    for (FwdPlan::Band b = band0; b.start < p.share_begin(xcd + 1); p.next(b)) ntiles += column(b).count;
  }
  __device__ __forceinline__ int count() const { return ntiles; }
  __device__ __forceinline__ Place at(int i) const {
    int left = ntiles;
    for (int w = 0; w < plan->waves; ++w, i -= wave_count, left -= wave_count)
      if (i < wave_count)
        return Place{8 * (kXcds * w + xcd) + (member & 7), (member >> 3) + (plan->group >> 3) * i,
                     plan->wave_slot(w, xcd, member)};
    // the bands of the share from the last to the first
    FwdPlan::Band b = band0;
    Column c = column(b);
    while (i < left - c.count) {
      left -= c.count;
      plan->next(b);
      c = column(b);
    }
    return Place{b.first + (member & (b.rows() - 1)), c.first + (plan->group >> b.log2_rows) * (i - (left - c.count)),
                 plan->slot(b.index, xcd, member)};
  }
  __device__ __forceinline__ void tile(int i, int& r0, int& c0) const {
    const Place p = at(i);
    r0 = p.tn * kTile;
    c0 = p.vt * kTile;
  }
  __device__ __forceinline__ int slab0(int) const { return 0; }
  __device__ __forceinline__ int slabs(int) const { return k_slabs; }
  __device__ __forceinline__ bool rows_outside(int, int) const { return false; }
};

// The epilogues that write matrices hand the accumulators through an LDS patch private to the
// wavefront (in the 32 KB the pipeline leaves free), ROWS x 32 values at a time (ROWS / 16 x 2 MFMA blocks), so that
// global accesses are whole 128-byte rows of fp32 (64-byte rows of bf16) touched by 8 consecutive
// lanes instead of 16-byte pieces of 16 different rows.  After the exchange lane L holds columns
// 4 (L % 8) .. + 3 of rows 8 i + L / 8 (i < ROWS / 8) of the patch.  LDS operations of one wavefront
// execute in issue order, so the patch needs no barrier, only the waits that order its writes and reads.
constexpr int kNB2 = kNB / 2, kMB2 = kMB / 2;  // 32 x 32 patches per wavefront along r and c
template <int ROWS>
struct BlockExchange {
  static constexpr int kRB = ROWS / kBlk, kPatchBytes = ROWS * 128;
  char* stage;  // this wavefront's patch
  int lx, lq, rd_row, rd_chunk;
  __device__ __forceinline__ void init(char* patches, const LanePos& p) {
    stage = patches + (threadIdx.x >> 6) * kPatchBytes;
    lx = p.lx;
    lq = p.lq;
    rd_row = (threadIdx.x & 63) >> 3;
    rd_chunk = threadIdx.x & 7;
  }
  // blk[cb][rb]: the 16 x 16 blocks of the patch, cb along c, rb along r
  __device__ __forceinline__ void run(const f32x4 (&blk)[2][kRB], f32x4 (&out)[ROWS / 8]) const {
#pragma unroll
    for (int cb = 0; cb < 2; ++cb)
#pragma unroll
      for (int rb = 0; rb < kRB; ++rb) {
        const int row = 16 * rb + lx;
        *reinterpret_cast<f32x4*>(stage + row * 128 + (((4 * cb + lq) ^ ((row >> 1) & 7)) << 4)) = blk[cb][rb];
      }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int i = 0; i < ROWS / 8; ++i) {
      const int row = 8 * i + rd_row;
      out[i] = *reinterpret_cast<const f32x4*>(stage + row * 128 + ((rd_chunk ^ ((row >> 1) & 7)) << 4));
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
};
using GradExchange = BlockExchange<32>;
// the patch (mb2, nb2) of an accumulator
__device__ __forceinline__ void exchange_patch(const GradExchange& ex, const Accum& acc, int mb2, int nb2, f32x4 (&out)[4]) {
  const f32x4 blk[2][2] = {{acc.a[2 * mb2][2 * nb2], acc.a[2 * mb2][2 * nb2 + 1]},
                           {acc.a[2 * mb2 + 1][2 * nb2], acc.a[2 * mb2 + 1][2 * nb2 + 1]}};
  ex.run(blk, out);
}

constexpr int kGradStageBytes = kWaves * GradExchange::kPatchBytes;
// forward: two sets of labels, label-logit sums, states of one half of the wavefronts (and squared sums); with a logits
// cache, behind them, patches of 16 rows
static_assert(kLdsBytes % (2 * kTile * 4) == 0, "the sets of labels are told apart by one address bit");
constexpr int kFwdTokenLds = 2 * kTile * 4 + kThreads * kNB * 4 + kTile * (16 + 4);
using CacheExchange = BlockExchange<16>;
constexpr int kFwdCacheLds = kFwdTokenLds + kWaves * CacheExchange::kPatchBytes;
static_assert(kLdsBytes + kFwdCacheLds <= 160 * 1024 && kFwdTokenLds % 128 == 0, "LDS of a CU");

__device__ __forceinline__ void merge_state(float& m, float& s, float& sy, float m2, float s2, float sy2) {
  const float mm = fmaxf(m, m2);
  const float a = fast_exp2(m - mm), b = fast_exp2(m2 - mm);
  s = s * a + s2 * b;
  sy = sy * a + sy2 * b;
  m = mm;
}
// the same with the squared sums q
__device__ __forceinline__ void merge_state(float& m, float& s, float& sy, float& q, float m2, float s2, float sy2,
                                            float q2) {
  const float mm = fmaxf(m, m2);
  const float a = fast_exp2(m - mm), b = fast_exp2(m2 - mm);
  s = s * a + s2 * b;
  sy = sy * a + sy2 * b;
  q = q * a * a + q2 * b * b;
  m = mm;
}

// Per-lane online-softmax state for the kNB token slots (nb) the lane owns.  With CACHE the
// scaled logits of every valid (token, vocabulary column) are also written out in fp32, so the
// backward pass can form d_logits without repeating the GEMM.
// With PI2 a fifth running sum, sum_j e_j^2, is carried, from which sum_j softmax(z)_j^2 follows
// (calculate_sum_pi_squared_from_logits, verl/utils/torch_functional.py:680-694).
template <bool CACHE, bool PI2, Walk WALK>
struct FwdEpi {
  LanePos p;
  float scale2;
  int vocab;
  // vectors and not arrays: an array here ends up in scratch memory, whose set-up alone is 1 to 2 us of a launch (129 x 896 x
  // 151936 68.4 -> 70.9 us, 400 x 1024 x 32000 32.1 -> 33.2)
  f32x4 m, s, sy, s2;
  // The labels of the lane's token rows and the label-logit sums live in LDS behind the pipeline's stages: with them in
  // registers the kernel spilled, and every reload of a spilled value waits out the slab transfers in flight (one
  // counter counts both).
  unsigned lab_lds, zl_lds, red_lds;  // LDS byte addresses: labels [256] by row, in the set in use of two; sums
                                      // [kThreads][kNB]; states [256] float4, then squared sums [256]
  char* patches;  // CACHE: the wavefronts' exchange patches
  const FwdArgs* args;
  FwdSched<WALK> sched;
  int64_t slot;  // where the state of the token tile at hand goes
  float rcp_t;

  // When the token tile changes: the low dwords of its 256 labels, 64 per wavefront of the first four, straight into LDS;
  // a token past the end reads as label 0, whose sums nobody looks at.  They go into the set that is not in use: other
  // wavefronts may still be in the epilogue that reads this one.
  __device__ __forceinline__ void prefetch(int tile, int r0, int) {
    if constexpr (WALK == kBands) {
      const auto here = sched.at(tile);
      if (here.slot == slot) return;
      if (tile > 0) write_state();  // (here no accumulators are alive)
      slot = here.slot;
      lab_lds ^= kTile * 4;
    } else if (tile > 0) {
      return;
    }
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    if (w < 4) {
      const u32x4 rs = span_rsrc(args->labels, (int64_t)args->n_tokens * 8);
      load_to_lds_4(rs, ((unsigned)r0 + 64u * w + (threadIdx.x & 63u)) * 8u, lab_lds + 64u * w * 4u);
    }
  }

  __device__ __forceinline__ void reset() {
#pragma unroll
    for (int nb = 0; nb < kNB; ++nb) {
      m[nb] = kNegBig;
      s[nb] = 0.f;
      sy[nb] = 0.f;
      s2[nb] = 0.f;
    }
  }

  // merge the four lane quarters (they hold disjoint vocabulary columns of the same token)
  __device__ __forceinline__ void merge_lanes(f32x4& z, int thread) {
    merge_with_peer(z, ((thread & 63) ^ 16) << 2);
    merge_with_peer(z, ((thread & 63) ^ 32) << 2);
  }
  static __device__ __forceinline__ float from_peer(int peer, float x) {
    return __int_as_float(__builtin_amdgcn_ds_bpermute(peer, __float_as_int(x)));
  }
  __device__ __forceinline__ void merge_with_peer(f32x4& z, int peer) {
#pragma unroll
    for (int nb = 0; nb < kNB; ++nb) {
      merge_into(nb, from_peer(peer, m[nb]), from_peer(peer, s[nb]), from_peer(peer, sy[nb]),
                 PI2 ? from_peer(peer, s2[nb]) : 0.f);
      z[nb] += from_peer(peer, z[nb]);
    }
  }
  __device__ __forceinline__ void merge_into(int nb, float m2, float sm2, float sy2, float q2) {
    float a = m[nb], b = s[nb], c = sy[nb], q = s2[nb];
    if (PI2) merge_state(a, b, c, q, m2, sm2, sy2, q2);
    else merge_state(a, b, c, m2, sm2, sy2);
    m[nb] = a;
    s[nb] = b;
    sy[nb] = c;
    s2[nb] = q;
  }

  // The token tile is done for this workgroup: combine the lanes, then the two wavefronts that share a token quarter
  // (wc = 0 / 1, through LDS), write the state out and start afresh.
  __device__ __forceinline__ void write_state() {
    typedef float __attribute__((address_space(3))) * lds_f32_t;
    typedef f32x4 __attribute__((address_space(3))) * lds_f32x4_t;
    // The thread's number as a value made here: everything addressed with it is then computed here too.  From threadIdx.x
    // the compiler computes the lot ahead of the tile loop and, with the accumulators in the way, spills 110 registers.
    int thread = threadIdx.x;
    asm volatile("" : "+v"(thread));
    const int row0 = ((thread >> 6) % kWavesR) * (kNB * kBlk) + (thread & 15);  // acc_row(p, 0)
    f32x4 z;
    const lds_f32_t sums = (lds_f32_t)(uintptr_t)(zl_lds + 4u * (unsigned)(thread * kNB));
#pragma unroll
    for (int nb = 0; nb < kNB; ++nb) {
      z[nb] = sums[nb];
      sums[nb] = 0.f;
    }
    merge_lanes(z, thread);
    const lds_f32x4_t red = (lds_f32x4_t)(uintptr_t)red_lds;
    const lds_f32_t redq = (lds_f32_t)(uintptr_t)(red_lds + kTile * 16);
    const bool lq0 = (thread & 48) == 0;
    if (thread >= 64 * kWavesR && lq0) {  // wc = 1
#pragma unroll
      for (int nb = 0; nb < kNB; ++nb) {
        red[row0 + kBlk * nb] = f32x4{m[nb], s[nb], sy[nb], z[nb]};
        if (PI2) redq[row0 + kBlk * nb] = s2[nb];
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (thread < 64 * kWavesR && lq0) {
#pragma unroll
      for (int nb = 0; nb < kNB; ++nb) {
        const int row = row0 + kBlk * nb;
        const f32x4 o = red[row];
        merge_into(nb, o[0], o[1], o[2], PI2 ? redq[row] : 0.f);
        if (PI2) args->pi2_partials[slot * kTile + row] = s2[nb];
        args->partials[slot * kTile + row] = make_float4(m[nb], s[nb], sy[nb], z[nb] + o[3]);
      }
    }
    reset();
  }

  // The scaled logits of the tile's valid tokens and columns, in whole 128-byte rows.
  __device__ __forceinline__ void store_logits(const Accum& acc, int r0, int c0) {
    const int tok0 = r0 + p.wr * (kNB * kBlk), n_tokens = args->n_tokens;
    float* const z_cache = args->z_cache;
    CacheExchange ex;
    ex.init(patches, p);
#pragma unroll
    for (int nb = 0; nb < kNB; ++nb)
#pragma unroll
      for (int mb2 = 0; mb2 < kMB2; ++mb2) {
        const f32x4 blk[2][1] = {{acc.a[2 * mb2][nb] * rcp_t}, {acc.a[2 * mb2 + 1][nb] * rcp_t}};
        f32x4 out[2];
        ex.run(blk, out);
        const int col = c0 + p.wc * 128 + mb2 * 32 + 4 * ex.rd_chunk;
        if (col < vocab) {
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            const int tok = tok0 + nb * kBlk + 8 * i + ex.rd_row;
            if (tok < n_tokens)
              __builtin_nontemporal_store(out[i], reinterpret_cast<f32x4*>(z_cache + (int64_t)tok * vocab + col));
          }
        }
      }
  }

  __device__ __forceinline__ void operator()(Accum& acc, int /*tile*/, int r0, int c0) {
    const bool ragged = c0 + kTile > vocab;
    // element (mb, v) of the lane is column 16 mb + v of this: comparing immediates with one register, where a column
    // number per element would be computed ahead of the tile loop and held (or spilled) through it
    const int cols_left = vocab - c0 - p.wc * 128 - 4 * p.lq;
    if constexpr (CACHE) store_logits(acc, r0, c0);
#pragma unroll
    for (int nb = 0; nb < kNB; ++nb) {
      // pass 1: tile maximum of the raw products (the vocabulary tail of the last tile replaced in place)
      float xmax = kNegBig;
      if (ragged) {
#pragma unroll
        for (int mb = 0; mb < kMB; ++mb)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const float x = mb * kBlk + v < cols_left ? acc.a[mb][nb][v] : kNoColumn;
            acc.a[mb][nb][v] = x;
            xmax = fmaxf(xmax, x);
          }
      } else {
#pragma unroll
        for (int mb = 0; mb < kMB; ++mb)
#pragma unroll
          for (int v = 0; v < 4; ++v) xmax = fmaxf(xmax, acc.a[mb][nb][v]);
      }
      // label logit: only when some lane's label falls in this wavefront's 128 columns
      typedef int __attribute__((address_space(3))) * lds_i32_t;
      typedef float __attribute__((address_space(3))) * lds_f32_t;
      const int label = *(lds_i32_t)(uintptr_t)(lab_lds + 4u * (unsigned)acc_row(p, nb));
      const int rel = label - c0 - p.wc * 128;
      if (__any(rel >= 0 && rel < 128)) {
        float add = 0.f;
        // a label past the vocabulary but inside its ragged last tile matches nothing: those columns hold kNoColumn
        const int mine = rel - 4 * p.lq < cols_left ? rel - 4 * p.lq : -1;
#pragma unroll
        for (int mb = 0; mb < kMB; ++mb)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            add += mb * kBlk + v == mine ? acc.a[mb][nb][v] * rcp_t : 0.f;
          }
        const lds_f32_t slot = (lds_f32_t)(uintptr_t)(zl_lds + 4u * (threadIdx.x * kNB + nb));
        *slot += add;
      }
      // pass 2: the running state in the log2 domain, three operations and an exponential per element:
      // e = 2^(x scale2 - m), s += e, sy += e x (the raw product: the 1 / temperature goes on at the very end)
      const float m_new = fmaxf(m[nb], xmax * scale2);
      const float resc = fast_exp2(m[nb] - m_new);
      float s_ = s[nb] * resc, sy_ = sy[nb] * resc, s2_ = PI2 ? s2[nb] * resc * resc : 0.f;
#pragma unroll
      for (int mb = 0; mb < kMB; ++mb)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const float x = acc.a[mb][nb][v];
          const float e = fast_exp2(fmaf(x, scale2, -m_new));
          s_ += e;
          sy_ = fmaf(e, x, sy_);
          if (PI2) s2_ = fmaf(e, e, s2_);
        }
      m[nb] = m_new;
      s[nb] = s_;
      sy[nb] = sy_;
      if (PI2) s2[nb] = s2_;
    }
  }
};

template <bool CACHE, bool PI2, Walk WALK>
__global__ __launch_bounds__(kThreads) void lce_forward_kernel(FwdArgs a) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  FwdSched<WALK> sched;
  sched.init(a.plan, a.k_slabs, xcd_regroup(blockIdx.x, gridDim.x));

  FwdEpi<CACHE, PI2, WALK> epi;
  epi.p = lane_pos();
  epi.scale2 = a.scale2;
  epi.vocab = a.vocab;
  epi.rcp_t = a.rcp_t;
  epi.args = &a;
  epi.sched = sched;
  if constexpr (WALK == kBands) epi.slot = -1;
  else epi.slot = sched.slot;
  epi.reset();
  typedef float __attribute__((address_space(3))) * lds_f32_t;
  epi.lab_lds = lds_address(lds + kLdsBytes);
  epi.zl_lds = epi.lab_lds + 2 * kTile * 4;
  epi.red_lds = epi.zl_lds + kThreads * kNB * 4;
#pragma unroll
  for (int nb = 0; nb < kNB; ++nb) *(lds_f32_t)(uintptr_t)(epi.zl_lds + 4u * (threadIdx.x * kNB + nb)) = 0.f;
  epi.patches = lds + kLdsBytes + kFwdTokenLds;

  run_tiles<false, false>(a.hidden, a.weight, sched, epi, lds);

  if (sched.count() > 0) epi.write_state();
}

// The forward pass over at most kFewTokens tokens.  It is bound by reading the weight: with a 256-token tile the matrix cores
// spend most of their time on padding (93 tokens x 896 x 151936: 68 us, 4 TB/s), with 128 tokens the MFMAs of a 256-row slab
// of the weight take about half as long as the slab takes out of HBM.  Every workgroup streams an equal range of weight rows,
// cut into tiles of equal height up to 256 whose rows only are fetched, through three LDS stages, so that two slabs (up to
// 16 MB over the chip) are in flight while one is multiplied; one barrier per slab: 53.6 us, 5.1 TB/s; whole pass 76 -> 60 us;
// 93 x 3584 x 152064 5.4 TB/s, 93 x 4096 x 128256 5.7 TB/s.  From 129 tokens on the 256-token tile's padding is less than half.  A wavefront owns 64 tokens
// x 64 columns (2 x 4 wavefronts) and keeps the softmax state of its tokens in registers to the end.
constexpr int kFewTokens = 128;
// The few-token kernels read every piece of the weight in one workgroup, and the backward pass reads it again.  A weight that about
// fits the 256 MB memory-side cache is read with plain loads; of a larger one the workgroups on the first 200 MB, and the others
// with the non-temporal hint, which leaves those there for the backward pass.  Everything with plain loads, everything with the hint
// and so, us, 64 tokens:
//                        the cache full of other data, read       the same, written            pass after pass
//                        forward          and backward            forward        and backward  forward        and backward
//   1536 x 151936        98   94   95     318  311  304           156   94  144  375  315  355   96   90   84  309  305  290
//   2048 x 151936       140  134  134     402  408  392           197  135  191  461  413  447  138  130  103  388  402  355
//   3584 x 152064       191  178  178     619  609  605           251  179  260  681  629  696  191  179  177  617  607  593
//   4096 x 128256       191  166  167     586  557  550           243  167  249  644  560  632  187  162  157  570  551  538
//   896 (272 MB, plain)  61   59   61     210  208  208           113   60  113  264  213  261   53   53   53  201  201  200
// (runs differ by 1 to 2 %).  The last two columns find the weight of the pass before in the cache, which no update does.  Where
// the cache is full of what was just written, as behind a trunk's forward pass, plain loads wait for that to be written back,
// and everything with the hint is quicker at every size: what the rule gains is the backward pass on a cache without such data.
constexpr int64_t kFittingWeightBytes = 320ll << 20, kCachedWeightBytes = 200ll << 20;
constexpr int kFewStageBytes = (kFewTokens + kTile) * kBK * 2;
constexpr int kFewStages = 3;
constexpr int kFewLds = kFewStages * kFewStageBytes;
constexpr int kFewCacheLds = kFewLds + kWaves * CacheExchange::kPatchBytes;  // with a logits cache
static_assert(kFewCacheLds <= 160 * 1024, "LDS of a CU");
constexpr int kFewWavesR = 2, kFewWavesC = 4, kFewMB = kTile / kBlk / kFewWavesC;
constexpr int kFewLoadsR = kFewTokens * 8 / kThreads;  // transfers per lane of one slab of hidden (2)
static_assert(kFewLoadsR + kLoads == 6, "the s_waitcnt vmcnt(6) of lce_forward_few_kernel counts the transfers of one slab");
static_assert(kFewTokens == kFewWavesR * kNB * kBlk, "a wavefront owns kNB blocks of tokens");

// the weight's slab of a stage; `stream` is the same for the whole workgroup
template <bool KMAJOR>
__device__ __forceinline__ void few_fetch_weight(const SlabDma<KMAJOR>& dma, const SlabSrc& src, unsigned slab_lds, int stream) {
  if (stream) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) dma.template issue_one<true>(i, src, slab_lds);
  } else {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) dma.template issue_one<false>(i, src, slab_lds);
  }
}

template <bool CACHE, bool PI2>
__global__ __launch_bounds__(kThreads) void lce_forward_few_kernel(FwdArgs a) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int split = xcd_regroup(blockIdx.x, gridDim.x);
  const int c_begin = split * a.plan.few_cols;
  const int c_end = c_begin + a.plan.few_cols < a.vocab ? c_begin + a.plan.few_cols : a.vocab;  // > c_begin
  const int w = threadIdx.x >> 6, lx = threadIdx.x & 15, lq = (threadIdx.x >> 4) & 3;
  const int wr = w % kFewWavesR, wc = w / kFewWavesR;

  // tiles of equal height, rows past a tile's read as zero without being fetched
  const int tiles = (c_end - c_begin + kTile - 1) / kTile, slabs = tiles * a.k_slabs;
  const int tile_cols = ((c_end - c_begin + tiles - 1) / tiles + kBlk - 1) / kBlk * kBlk;
  auto tile_end = [&](int t) {
    const int end = c_begin + (t + 1) * tile_cols;
    return end < c_end ? end : c_end;
  };
  auto weight_rsrc = [&](int t) {
    Operand weight = a.weight;
    weight.x_extent = tile_end(t);
    return tile_rsrc<false>(weight, c_begin + t * tile_cols);
  };
  SlabDma<false> dma;       // the same for both operands: their rows are the same distance apart
  dma.init(a.hidden);
  FragAddr<false> fr, fc;
  fr.init(wr * kNB, kNB);
  fc.init(wc * kFewMB, kFewMB);

  int label[kNB];
  float m[kNB], s[kNB], sy[kNB], s2[kNB], zl[kNB];
#pragma unroll
  for (int nb = 0; nb < kNB; ++nb) {
    const int tok = wr * (kNB * kBlk) + nb * kBlk + lx;
    label[nb] = tok < a.n_tokens ? (int)a.labels[tok] : -1;
    m[nb] = kNegBig;
    s[nb] = sy[nb] = s2[nb] = zl[nb] = 0.f;
  }

  // fetch cursor; past the end it stays on the last slab
  const u32x4 rs_r = tile_rsrc<false>(a.hidden, 0);
  u32x4 rs_c = weight_rsrc(0);
  int t2 = 0, k2 = 0, fill = 0;
  auto fetch = [&]() {
    const SlabSrc r{rs_r, slab_soff<false>(a.hidden, k2 * kBK)}, c{rs_c, slab_soff<false>(a.weight, k2 * kBK)};
    const unsigned base = lds_address(lds) + (unsigned)fill * kFewStageBytes;
#pragma unroll
    for (int i = 0; i < kFewLoadsR; ++i) dma.issue_one(i, r, base);
    few_fetch_weight(dma, c, base + kFewTokens * kBK * 2, c_begin >= a.stream_from);
    fill = fill == kFewStages - 1 ? 0 : fill + 1;
    if (t2 == tiles - 1 && k2 == a.k_slabs - 1) return;
    if (++k2 == a.k_slabs) {
      k2 = 0;
      ++t2;
      rs_c = weight_rsrc(t2);
    }
  };
  fetch();
  fetch();

  f32x4 acc[kFewMB][kNB];
  int kt = 0, tile = 0, stage = 0;
  for (int it = 0; it < slabs; ++it) {
    if (kt == 0) {
#pragma unroll
      for (int mb = 0; mb < kFewMB; ++mb)
#pragma unroll
        for (int nb = 0; nb < kNB; ++nb) acc[mb][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    // slab `it` has landed (all but the six transfers of the next one), and nobody reads the stage before it any more:
    // that one takes slab it + 2
    asm volatile("s_waitcnt vmcnt(6) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    fetch();
    const char* cur = lds + stage * kFewStageBytes;
    stage = stage == kFewStages - 1 ? 0 : stage + 1;
    bf16x8 r[kSteps][kNB], c[kSteps][kFewMB];
#pragma unroll
    for (int ks = 0; ks < kSteps; ++ks) {
#pragma unroll
      for (int nb = 0; nb < kNB; ++nb) r[ks][nb] = fr.read(cur, ks, nb);
#pragma unroll
      for (int mb = 0; mb < kFewMB; ++mb) c[ks][mb] = fc.read(cur + kFewTokens * kBK * 2, ks, mb);
    }
#pragma unroll
    for (int ks = 0; ks < kSteps; ++ks)
#pragma unroll
      for (int mb = 0; mb < kFewMB; ++mb)
#pragma unroll
        for (int nb = 0; nb < kNB; ++nb)
          acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c[ks][mb], r[ks][nb], acc[mb][nb], 0, 0, 0);
    if (++kt < a.k_slabs) continue;
    kt = 0;
    // the tile is done: online softmax over its columns, as in FwdEpi
    const int col0 = c_begin + tile * tile_cols + wc * (kFewMB * kBlk) + 4 * lq;  // column of element (0, 0) of the lane
    const int cols_left = tile_end(tile) - col0;
    if constexpr (CACHE) {
      LanePos pos{};
      pos.lx = lx;
      pos.lq = lq;
      CacheExchange ex;
      ex.init(lds + kFewLds, pos);
#pragma unroll
      for (int nb = 0; nb < kNB; ++nb)
#pragma unroll
        for (int mb2 = 0; mb2 < kFewMB / 2; ++mb2) {
          const f32x4 blk[2][1] = {{acc[2 * mb2][nb] * a.rcp_t}, {acc[2 * mb2 + 1][nb] * a.rcp_t}};
          f32x4 out[2];
          ex.run(blk, out);
          // 4 columns that exist or do not: vocab % 8 == 0, and tiles end at multiples of kBlk or at the vocabulary
          const int col = col0 - 4 * lq + 32 * mb2 + 4 * ex.rd_chunk;
          if (col < tile_end(tile)) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
              const int tok = wr * (kNB * kBlk) + nb * kBlk + 8 * i + ex.rd_row;
              if (tok < a.n_tokens)
                __builtin_nontemporal_store(out[i], reinterpret_cast<f32x4*>(a.z_cache + (int64_t)tok * a.vocab + col));
            }
          }
        }
    }
    ++tile;
#pragma unroll
    for (int nb = 0; nb < kNB; ++nb) {
      float xmax = kNegBig, add = 0.f;
      const int mine = label[nb] - col0;
#pragma unroll
      for (int mb = 0; mb < kFewMB; ++mb)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const float x = mb * kBlk + v < cols_left ? acc[mb][nb][v] : kNoColumn;
          acc[mb][nb][v] = x;
          xmax = fmaxf(xmax, x);
          add += mb * kBlk + v == mine && mine < cols_left ? x * a.rcp_t : 0.f;
        }
      zl[nb] += add;
      const float m_new = fmaxf(m[nb], xmax * a.scale2);
      const float resc = fast_exp2(m[nb] - m_new);
      float s_ = s[nb] * resc, sy_ = sy[nb] * resc, s2_ = PI2 ? s2[nb] * resc * resc : 0.f;
#pragma unroll
      for (int mb = 0; mb < kFewMB; ++mb)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const float x = acc[mb][nb][v];
          const float e = fast_exp2(fmaf(x, a.scale2, -m_new));
          s_ += e;
          sy_ = fmaf(e, x, sy_);
          if (PI2) s2_ = fmaf(e, e, s2_);
        }
      m[nb] = m_new;
      s[nb] = s_;
      sy[nb] = sy_;
      if (PI2) s2[nb] = s2_;
    }
  }

  // the four lane quarters, then the four wavefronts that share 64 tokens, hold disjoint columns
#pragma unroll
  for (int step = 16; step <= 32; step <<= 1)
#pragma unroll
    for (int nb = 0; nb < kNB; ++nb) {
      zl[nb] += __shfl_xor(zl[nb], step, 64);
      const float m2 = __shfl_xor(m[nb], step, 64), b2 = __shfl_xor(s[nb], step, 64), y2 = __shfl_xor(sy[nb], step, 64);
      if (PI2) merge_state(m[nb], s[nb], sy[nb], s2[nb], m2, b2, y2, __shfl_xor(s2[nb], step, 64));
      else merge_state(m[nb], s[nb], sy[nb], m2, b2, y2);
    }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");  // the stages are free
  float4* red = reinterpret_cast<float4*>(lds);                                          // [4][128]
  float* redq = reinterpret_cast<float*>(lds + kFewWavesC * kFewTokens * sizeof(float4));  // [4][128] squared sums
  if (lq == 0) {
#pragma unroll
    for (int nb = 0; nb < kNB; ++nb) {
      const int row = wr * (kNB * kBlk) + nb * kBlk + lx;
      red[wc * kFewTokens + row] = make_float4(m[nb], s[nb], sy[nb], zl[nb]);
      if (PI2) redq[wc * kFewTokens + row] = s2[nb];
    }
  }
  __syncthreads();
  if (threadIdx.x < kFewTokens) {
    const int row = threadIdx.x;
    float4 x = red[row];
    float q = PI2 ? redq[row] : 0.f;
#pragma unroll
    for (int j = 1; j < kFewWavesC; ++j) {
      const float4 y = red[j * kFewTokens + row];
      if (PI2) merge_state(x.x, x.y, x.z, q, y.x, y.y, y.z, redq[j * kFewTokens + row]);
      else merge_state(x.x, x.y, x.z, y.x, y.y, y.z);
      x.w += y.w;
    }
    a.partials[(int64_t)split * kTile + row] = x;
    if (PI2) a.pi2_partials[(int64_t)split * kTile + row] = q;
  }
}

struct MergeArgs {
  const float4* partials;
  const float* pi2_partials;  // null unless sum_pi_squared is wanted
  FwdPlan plan;
  int n_tokens;
  int lanes_log2;  // lanes that share a token, as a power of two
  float rcp_t;  // the partial sums of e * (hidden . weight) carry no 1 / temperature yet
  float* logprobs;
  float* entropy;
  float* lse;
  float* mean_z;
  float* sum_pi_squared;
};

// Combines the partial states of a token.  `1 << lanes_log2` consecutive lanes share a token: each walks every
// (1 << lanes_log2)-th split, then the lanes' states meet by lane exchanges.  A launch over few tokens has up to 256 splits
// per token, and one thread walking them is a chain of 256 dependent merges behind as many exposed loads (93 tokens:
// 78 us, longer than the forward GEMM in front of it; 64 lanes per token: about 5 us).
__global__ __launch_bounds__(256) void lce_merge_kernel(MergeArgs a) {
  const int lanes = 1 << a.lanes_log2;
  const int64_t tok = ((int64_t)blockIdx.x * 256 + threadIdx.x) >> a.lanes_log2;
  const bool exists = tok < a.n_tokens;
  float m = kNegBig, s = 0.f, sy = 0.f, zl = 0.f, q = 0.f;
  if (exists) {
    const int tn = (int)(tok / kTile), row = (int)(tok % kTile), mine = threadIdx.x & (lanes - 1);
    auto add = [&](int64_t slot) {
      const float4 x = a.partials[slot * kTile + row];
      if (a.pi2_partials) merge_state(m, s, sy, q, x.x, x.y, x.z, a.pi2_partials[slot * kTile + row]);
      else merge_state(m, s, sy, x.x, x.y, x.z);
      zl += x.w;
    };
    if (a.plan.splits) {
      for (int sp = mine; sp < a.plan.splits; sp += lanes) add((int64_t)sp * a.plan.tok_tiles + tn);
    } else {  // every workgroup column of every XCD whose share of the rounds touches the token tile's band
      const bool in_wave = tn < 64 * a.plan.waves;
      FwdPlan::Band b = a.plan.first_band();
      while (!in_wave && tn >= b.first + b.rows()) a.plan.next(b);
      const int cols = a.plan.group >> (in_wave ? 3 : b.log2_rows);
      if (in_wave)
        for (int col = mine; col < cols && col < a.plan.voc_tiles; col += lanes)
          add(a.plan.wave_slot(tn / 64, tn / 8 % kXcds, col * 8 + tn % 8));
      int x0 = 0, x1;  // the XCDs whose shares touch the band
      while (!in_wave && a.plan.share_begin(x0 + 1) <= b.start) ++x0;
      for (x1 = x0; x1 + 1 < kXcds && a.plan.share_begin(x1 + 1) < b.start + b.count;) ++x1;
      for (int j = mine; !in_wave && j < (x1 - x0 + 1) * cols; j += lanes) {
        const int xcd = x0 + j / cols, col = j % cols;
        const int q0 = a.plan.share_begin(xcd), q1 = a.plan.share_begin(xcd + 1);
        const int lo = q0 > b.start ? q0 - b.start : 0;
        if (q1 > b.start + lo && col + cols * lo < a.plan.voc_tiles)  // it had a tile to do
          add(a.plan.slot(b.index, xcd, col * b.rows() + (tn - b.first)));
      }
    }
  }
  for (int step = 1; step < lanes; step <<= 1) {
    const float m2 = __shfl_xor(m, step, 64), s2 = __shfl_xor(s, step, 64), sy2 = __shfl_xor(sy, step, 64);
    zl += __shfl_xor(zl, step, 64);
    merge_state(m, s, sy, q, m2, s2, sy2, __shfl_xor(q, step, 64));
  }
  if (!exists || (threadIdx.x & (lanes - 1)) != 0) return;
  if (a.pi2_partials) a.sum_pi_squared[tok] = q / (s * s);
  const float lse = (m + log2f(s)) * kLn2;
  const float mz = (sy / s) * a.rcp_t;
  a.lse[tok] = lse;
  a.mean_z[tok] = mz;
  a.entropy[tok] = lse - mz;
  a.logprobs[tok] = zl - lse;
}

// =============================================================================================
// Backward
// =============================================================================================
__device__ __forceinline__ u32x2 pack_bf16x4(float a, float b, float c, float d) {
  bf16x4 o;
  o[0] = (__bf16)a;
  o[1] = (__bf16)b;
  o[2] = (__bf16)c;
  o[3] = (__bf16)d;
  return __builtin_bit_cast(u32x2, o);
}

__device__ __forceinline__ float bf16_bits_to_float(unsigned h) { return __uint_as_float(h << 16); }

struct RecomputeArgs {
  Operand hidden;  // R: [n_tokens][H]
  Operand weight;  // C: rows of this vocabulary chunk, x_extent = vocab - chunk_c0
  const int64_t* labels;
  const float* lse;
  const float* mean_z;
  const float* g_lp;   // may be null
  const float* g_ent;  // may be null -> g_ent_scalar
  float g_ent_scalar;
  int n_tokens, vocab_left;  // vocab_left = vocab - chunk_c0
  int chunk_c0;
  int k_slabs, tok_tiles, chunk_tiles;
  float rcp_t;
  uint16_t* dz;  // [tok_tiles*256][dz_ld] bf16
  int dz_ld;
};

// The same hand-over for a bf16 result: the wavefront's patch holds 32 rows x 32 columns of bf16 (2 KB), rounded
// before the exchange, so the LDS traffic is half that of the fp32 patch and the global stores are 16 bytes per
// lane: a store instruction covers 16 rows x 64 bytes.  16-byte chunk c of row r lives at position c ^ ((r >> 2) & 3)
// so that the 8-byte writes of 16 rows at one column spread over the banks.  After the exchange lane L holds columns
// 8 (L % 4) .. + 7 of rows 16 i + L / 4 (i = 0, 1).
struct BlockExchangeBf16 {
  char* stage;
  int lx, lq, rd_row, rd_chunk;
  __device__ __forceinline__ void init(char* area, const LanePos& p) {
    stage = area + (threadIdx.x >> 6) * 2048;
    lx = p.lx;
    lq = p.lq;
    rd_row = (threadIdx.x & 63) >> 2;
    rd_chunk = threadIdx.x & 3;
  }
  __device__ __forceinline__ void run(const f32x4 (&blk)[2][2], u32x4 (&out)[2]) const {
#pragma unroll
    for (int cb = 0; cb < 2; ++cb)
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) {
        const int row = 16 * rb + lx;
        const int chunk = (2 * cb + (lq >> 1)) ^ ((row >> 2) & 3);
        *reinterpret_cast<u32x2*>(stage + row * 64 + chunk * 16 + (lq & 1) * 8) =
            pack_bf16x4(blk[cb][rb][0], blk[cb][rb][1], blk[cb][rb][2], blk[cb][rb][3]);
      }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int row = 16 * i + rd_row;
      out[i] = *reinterpret_cast<const u32x4*>(stage + row * 64 + ((rd_chunk ^ ((row >> 2) & 3)) << 4));
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
};
constexpr int kBf16StageBytes = (kThreads / 64) * 2048;  // one 32 x 32 bf16 patch per wavefront

// Per-token inputs of the d_logits epilogue (lse, mean_z, g_lp, label, g_ent) for the 256 tokens of a tile, staged
// in LDS by memory -> LDS transfers issued when the tile's first slab starts (prefetch): five arrays of 256 dwords,
// two sets used in turn so that a tile's transfers never land in what the previous tile's epilogue still reads.
constexpr int kTokArrays = 5, kTokSetBytes = kTokArrays * kTile * 4;
constexpr int kRecomputeExtraLds = kBf16StageBytes + 2 * kTokSetBytes;
static_assert(kLdsBytes + kRecomputeExtraLds <= 160 * 1024, "LDS of a CU");

struct RecomputeEpi {
  LanePos p;
  const RecomputeArgs* a;
  BlockExchangeBf16 ex;
  char* tok_stage;  // [2][kTokArrays][256] dwords
  int parity;       // set of the tile whose epilogue runs next

  __device__ __forceinline__ void init(char* lds_after_pipeline, const LanePos& pos, const RecomputeArgs* args) {
    p = pos;
    a = args;
    ex.init(lds_after_pipeline, pos);
    tok_stage = lds_after_pipeline + kBf16StageBytes;
    parity = 0;
  }

  // wavefront w brings in half (w & 1) of array (w >> 1): 0 lse, 1 mean_z, 2 g_lp, 3 labels (low dwords); the
  // wavefronts 0 and 1 also bring in g_ent when it is a tensor
  __device__ __forceinline__ void prefetch(int tile, int r0, int /*c0*/) {
    const RecomputeArgs& A = *a;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const unsigned lane = threadIdx.x & 63u;
    const int arr = w >> 1, half = w & 1;
    const unsigned set_lds = lds_address(tok_stage) + (unsigned)(tile & 1) * kTokSetBytes;
    const void* src = arr == 0 ? (const void*)A.lse : arr == 1 ? (const void*)A.mean_z
                      : arr == 2 ? (const void*)A.g_lp : (const void*)A.labels;
    const unsigned elt = arr == 3 ? 8u : 4u;
    if (src) {  // uniform over the wavefront
      const u32x4 rs = span_rsrc(src, (int64_t)A.n_tokens * elt);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const unsigned tok = (unsigned)r0 + half * 128u + i * 64u + lane;
        load_to_lds_4(rs, tok * elt, set_lds + arr * (kTile * 4) + (half * 128u + i * 64u) * 4u);
      }
    }
    if (A.g_ent && w < 2) {
      const u32x4 rs = span_rsrc(A.g_ent, (int64_t)A.n_tokens * 4);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const unsigned tok = (unsigned)r0 + half * 128u + i * 64u + lane;
        load_to_lds_4(rs, tok * 4u, set_lds + 4 * (kTile * 4) + (half * 128u + i * 64u) * 4u);
      }
    }
  }

  // d_logits of the two token rows (rb) x 128 columns the lane holds of 32-row patch nb2, rounded, handed over and
  // stored.  PLAIN: a tile inside the matrix with no label in the wavefront's 128 columns -- nothing but the
  // arithmetic, four multiply-adds and an exponential per element; otherwise the one-hot term and the zeros for
  // padding rows and columns come in through two comparisons per element (no branches).
  // The accumulators hold logits, z = x / T in fp32: the expressions are lce_dlogits_kernel's, bit for bit.
  //   code[rb]: 4 mb + v of the element of row rb that holds the label's column, or -1
  //   lim[rb] : columns of the wavefront's 128 that exist for row rb (0 for a padding row), minus 4 lq
  template <bool PLAIN>
  __device__ __forceinline__ void patch_rows(Accum& acc, int nb2, int r0, int c0, const float (&lse2)[2],
                                             const float (&u1)[2], const float (&u0)[2], const float (&glp)[2],
                                             const int (&code)[2], const int (&lim)[2]) {
    const RecomputeArgs& A = *a;
#pragma unroll
    for (int mb2 = 0; mb2 < kMB2; ++mb2) {
      f32x4 d[2][2];
#pragma unroll
      for (int cb = 0; cb < 2; ++cb)
#pragma unroll
        for (int rb = 0; rb < 2; ++rb)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const int mb = 2 * mb2 + cb;
            const float z = acc.a[mb][2 * nb2 + rb][v];
            const float prob = fast_exp2(fmaf(z, kLog2e, -lse2[rb]));
            const float u = fmaf(u1[rb], z, u0[rb]);  // g_lp/T + g_ent/T * (z - mean_z)
            if constexpr (PLAIN) {
              d[cb][rb][v] = -prob * u;
            } else {
              const float onehot = code[rb] == 4 * mb + v ? glp[rb] : 0.f;
              const float dzv = fmaf(-prob, u, onehot);
              d[cb][rb][v] = (mb * kBlk + v) < lim[rb] ? dzv : 0.f;  // every row of the panel is written, padding as zeros
            }
          }
      u32x4 o[2];
      ex.run(d, o);
      const int col0 = c0 + p.wc * 128 + mb2 * 32 + 8 * ex.rd_chunk;
      const int64_t row0 = r0 + p.wr * (kNB * kBlk) + nb2 * 32 + ex.rd_row;
#pragma unroll
      for (int i = 0; i < 2; ++i) *reinterpret_cast<u32x4*>(A.dz + (row0 + 16 * i) * A.dz_ld + col0) = o[i];
    }
  }

  __device__ __forceinline__ void operator()(Accum& acc, int /*tile*/, int r0, int c0) {
    const RecomputeArgs& A = *a;
    // read through LDS-typed pointers: as generic pointers some of these became flat loads, whose wait also
    // waits out every slab transfer in flight
    typedef const float __attribute__((address_space(3))) * lds_f32_t;
    typedef const int __attribute__((address_space(3))) * lds_i32_t;
    const lds_f32_t tokf = (lds_f32_t)(uintptr_t)(lds_address(tok_stage) + (unsigned)parity * kTokSetBytes);
    const lds_i32_t toki = (lds_i32_t)tokf;
    parity ^= 1;
    const bool inside = r0 + kTile <= A.n_tokens && c0 + kTile <= A.vocab_left;  // uniform over the workgroup
    const int cols_left = A.vocab_left - c0 - p.wc * 128 - 4 * p.lq;
    // Rounded to z first, as the logits cache holds it, so that the gradients are the same bits with and without a cache,
    // which is kept or not by what memory there is (with the scale folded into the exponent they differed in the last bit
    // of some at T = 0.7).
    if (A.rcp_t != 1.f) {
#pragma unroll
      for (int mb = 0; mb < kMB; ++mb)
#pragma unroll
        for (int nb = 0; nb < kNB; ++nb) acc.a[mb][nb] = acc.a[mb][nb] * A.rcp_t;
    }
#pragma unroll
    for (int nb2 = 0; nb2 < kNB2; ++nb2) {
      // the lane's two token rows of this 32-row patch
      // u = u1 z + u0 with u1 = g_ent / T and u0 = g_lp / T - g_ent / T * mean_z: one multiply-add per element
      float lse2[2], u1[2], u0[2], glp[2];
      int code[2], lim[2];
      bool hit = false;
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) {
        const int t = acc_row(p, 2 * nb2 + rb);  // row inside the tile
        lse2[rb] = tokf[t] * kLog2e;
        glp[rb] = (A.g_lp ? tokf[2 * kTile + t] : 0.f) * A.rcp_t;
        u1[rb] = (A.g_ent ? tokf[4 * kTile + t] : A.g_ent_scalar) * A.rcp_t;
        u0[rb] = fmaf(-u1[rb], tokf[kTile + t], glp[rb]);
        const int rel = toki[3 * kTile + t] - A.chunk_c0 - c0 - p.wc * 128;  // label's column among the wavefront's 128
        const bool here = rel >= 0 && rel < 128;
        hit = hit || here;
        // the lane holds columns 16 mb + 4 lq + v: the label's is one of them when its 4-column group is lq
        code[rb] = (here && ((rel >> 2) & 3) == p.lq) ? 4 * (rel >> 4) + (rel & 3) : -1;
        lim[rb] = r0 + t < A.n_tokens ? cols_left : 0;
      }
      if (inside && !__any(hit)) patch_rows<true>(acc, nb2, r0, c0, lse2, u1, u0, glp, code, lim);
      else patch_rows<false>(acc, nb2, r0, c0, lse2, u1, u0, glp, code, lim);
    }
  }
};

__global__ __launch_bounds__(kThreads) void lce_recompute_kernel(RecomputeArgs a) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  GroupedSched sched;
  sched.grid = TileGrid{a.tok_tiles, a.chunk_tiles};
  sched.k_slabs = a.k_slabs;
  sched.nwg = gridDim.x;
  sched.wg = xcd_regroup(blockIdx.x, gridDim.x);
  RecomputeEpi epi;
  epi.init(lds + kLdsBytes, lane_pos(), &a);
  run_tiles<false, false>(a.hidden, a.weight, sched, epi, lds);
}

// d_logits panel of one vocabulary chunk from cached logits, to the bits of RecomputeEpi.  Bound by memory.
// A workgroup takes kPanelCols columns of a token, two groups of 4 per thread, each group's loads and stores contiguous across the
// wavefront; workgroups walk along a row.  With 8 consecutive columns per thread an instruction touched half of every line,
// and tokens as the fast index made neighbouring workgroups a row of the cache apart: 16384 x 152064 2695 -> 2470 us (6.1 TB/s),
// 4096 x 151936 717 -> 600, 777 x 151936 127 -> 115.  One group per thread 2913, four 2549, cached instead of non-temporal loads
// 2682, non-temporal stores 2499.
// Rows of the panel past the last token are not written: the gradient products read them as zero without fetching them
// (filling the last 256-token tile took 64 x 151936 from 15.5 to 22.4 us).
constexpr int kPanelCols = 2048;
struct DLogitsArgs {
  const float* z_cache;  // [cache_rows][vocab]
  const int64_t* rows;   // the row of each token, or null: token i has row i
  int64_t cache_rows;
  const int64_t* labels;
  const float* lse;
  const float* mean_z;
  const float* g_lp;
  const float* g_ent;
  float g_ent_scalar, rcp_t;
  int n_tokens, vocab, chunk_c0, chunk_cols;  // chunk_cols: panel columns to fill (multiple of 256)
  uint16_t* dz;
  int dz_ld;
};

__global__ __launch_bounds__(256) void lce_dlogits_kernel(DLogitsArgs a) {
  const int blocks = (a.chunk_cols + kPanelCols - 1) / kPanelCols, tok = blockIdx.x / blocks;
  const int j0 = (int)(blockIdx.x % blocks) * kPanelCols + threadIdx.x * 4;  // column inside the chunk
  const int64_t row = a.rows ? a.rows[tok] : tok;
  const int cols = row >= 0 && row < a.cache_rows ? a.vocab - a.chunk_c0 : 0;  // columns that exist
  const float lse2 = a.lse[tok] * kLog2e;
  const float glp = (a.g_lp ? a.g_lp[tok] : 0.f) * a.rcp_t;
  const float gent = (a.g_ent ? a.g_ent[tok] : a.g_ent_scalar) * a.rcp_t;
  const float u0 = fmaf(-gent, a.mean_z[tok], glp);
  const int label = (int)a.labels[tok] - a.chunk_c0;
  f32x4 z[2];
#pragma unroll
  for (int g = 0; g < 2; ++g) {
    const int j = j0 + g * (kPanelCols / 2);
    z[g] = f32x4{0.f, 0.f, 0.f, 0.f};
    // vocab % 8 == 0: the 4 columns are all in or all out
    if (j < a.chunk_cols && j < cols)
      z[g] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(a.z_cache + row * a.vocab + a.chunk_c0 + j));
  }
  u32x2 out[2];
#pragma unroll
  for (int g = 0; g < 2; ++g) {
    const int j = j0 + g * (kPanelCols / 2);
    float d[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float prob = fast_exp2(fmaf(z[g][e], kLog2e, -lse2));
      const float u = fmaf(gent, z[g][e], u0);
      d[e] = fmaf(-prob, u, (j + e == label) ? glp : 0.f);
    }
    out[g] = j < cols ? pack_bf16x4(d[0], d[1], d[2], d[3]) : u32x2{0u, 0u};
  }
#pragma unroll
  for (int g = 0; g < 2; ++g) {
    const int j = j0 + g * (kPanelCols / 2);
    if (j < a.chunk_cols) *reinterpret_cast<u32x2*>(a.dz + (int64_t)tok * a.dz_ld + j) = out[g];
  }
}

// ---------------------------------------------------------------------------------------------
// d_hidden (+)= dz_panel . W[chunk]          R = dz (direct), C = W (kmajor, k = vocab)
// d_weight[chunk] (+)= dz_panel^T . hidden    R = dz (kmajor, k = token), C = hidden (kmajor)
enum : int { kStoreF32 = 0, kAddF32 = 1, kFinalBf16 = 2, kFinalBf16AddPrev = 3 };

// How the gradient GEMMs of one vocabulary chunk are shared out over the workgroups: plan_gradients().
struct GradPlan {
  int splits = 1, split_slabs = 1;  // d_hidden: SplitKSched; each piece is summed into its own fp32 accumulator
  int extra = 0, late = 0;          // d_weight: LateStartSched
};

struct GemmOutArgs {
  Operand R, C;
  int k_slabs, r_tiles, c_tiles;
  int r_valid, c_valid;  // rows / cols of the output that exist
  int mode;              // d_hidden: one of the enum above; d_weight: a VAMD_DW_* value
  float* acc32;          // fp32 accumulator [r_valid][ld_out], of d_hidden one per piece
  uint16_t* out;         // bf16 output
  int64_t ld_out;
};

struct DHiddenEpi {
  LanePos p;
  const GemmOutArgs* a;
  SplitKSched sched;
  GradExchange ex;
  __device__ __forceinline__ void prefetch(int, int, int) {}
  __device__ __forceinline__ void operator()(Accum& acc, int tile, int r0, int c0) {
    const GemmOutArgs& A = *a;
    float* const acc32 = A.acc32 + (int64_t)sched.piece(tile) * A.r_valid * A.ld_out;
    const bool read_prev = A.mode == kAddF32 || A.mode == kFinalBf16AddPrev;
    const bool to_f32 = A.mode == kStoreF32 || A.mode == kAddF32;
#pragma unroll
    for (int nb = 0; nb < kNB2; ++nb)
#pragma unroll
      for (int mb = 0; mb < kMB2; ++mb) {
        f32x4 v[4];
        exchange_patch(ex, acc, mb, nb, v);
        const int col = c0 + p.wc * 128 + mb * 32 + 4 * ex.rd_chunk;
        if (col >= A.c_valid) continue;
        const int row0 = r0 + p.wr * (kNB * kBlk) + nb * 32 + ex.rd_row;
        f32x4 prev[4];
        if (read_prev) {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            prev[i] = (row0 + 8 * i < A.r_valid)
                          ? *reinterpret_cast<const f32x4*>(acc32 + (int64_t)(row0 + 8 * i) * A.ld_out + col)
                          : f32x4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int row = row0 + 8 * i;
          if (row >= A.r_valid) continue;
          f32x4 x = v[i];
          if (read_prev) x = x + prev[i];
          const int64_t off = (int64_t)row * A.ld_out + col;
          if (to_f32) *reinterpret_cast<f32x4*>(acc32 + off) = x;
          else *reinterpret_cast<u32x2*>(A.out + off) = pack_bf16x4(x[0], x[1], x[2], x[3]);
        }
      }
  }
};

// Hand-over of a result that is stored as bf16 and not added to anything: 32 rows x 64 columns, rounded before the exchange, so
// that a wavefront's store instruction covers 8 whole 128-byte lines (as 8 bytes per lane of 32-column patches it covered the
// halves of 8).  Gradient products 777 x 896 x 151936 467 -> 453 us, 777 x 3584 x 152064 1625 -> 1497, 64 tokens 562 -> 475,
// 16384 tokens 25.82 -> 25.69 ms.  16-byte chunk c of row r lives at position c ^ ((r >> 1) & 7) of the wavefront's patch,
// which is that of GradExchange.
typedef unsigned u32x4_at8 __attribute__((ext_vector_type(4), aligned(8)));  // d_weight's alignment is the caller's
struct LineExchange {
  char* stage;
  int lx, lq, rd_row, rd_chunk;
  __device__ __forceinline__ explicit LineExchange(const GradExchange& e)
      : stage(e.stage), lx(e.lx), lq(e.lq), rd_row(e.rd_row), rd_chunk(e.rd_chunk) {}
  // the patch (mb4, nb2) of an accumulator; lane L gets columns 8 (L % 8) .. + 7 of rows 8 i + L / 8
  __device__ __forceinline__ void run(const Accum& acc, int mb4, int nb2, u32x4 (&out)[4]) const {
#pragma unroll
    for (int cb = 0; cb < 4; ++cb)
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) {
        const f32x4& v = acc.a[4 * mb4 + cb][2 * nb2 + rb];
        const int row = 16 * rb + lx, chunk = (2 * cb + (lq >> 1)) ^ ((row >> 1) & 7);
        *reinterpret_cast<u32x2*>(stage + row * 128 + chunk * 16 + (lq & 1) * 8) = pack_bf16x4(v[0], v[1], v[2], v[3]);
      }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 8 * i + rd_row;
      out[i] = *reinterpret_cast<const u32x4*>(stage + row * 128 + ((rd_chunk ^ ((row >> 1) & 7)) << 4));
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
};

// STREAM: a d_weight stored in bf16 goes past the caches.  One that does not fit the memory-side cache is written back while
// whatever comes next reads; of one that fits, the next reader (accumulation, norm, optimizer) finds it there.  The line lies at
// the 200 MB that the cache holds beside other data (kCachedWeightBytes).  Forward and backward and then a norm of d_weight, after a
// pass that fills the cache with other data, plain and STREAM, us: 300 x 1024 x 32000 (66 MB) 155 and 177, 300 x 1024 x 64000
// (131 MB) 282 and 297, 300 x 1024 x 96000 (197 MB) 407 and 411, 64 tokens 277 and 297; 300 x 1024 x 128000 (262 MB) 543 and 524,
// 64 x 2048 x 64000 398 and 372, 300 x 896 x 151936 (272 MB) 566 and 554, 128 tokens 472 and 439, 2048 tokens 2018 and 2012,
// 128 x 3584 x 152064 (1.09 GB) 1335 and 1236; with an addition to another gradient in the norm's place 156 and 175, 274 and 287,
// 399 and 400, 292 and 285; 534 and 512, 386 and 367, 556 and 544, 460 and 430, 2014 and 2004, 1379 and 1277.  Without a reader
// 300 x 1024 x 32000 to 96000 within 2 %, the larger ones 324 and 308 (128 x 896), 807 and 732 (128 x 3584), 1346 and 1331 (300);
// only 64 x 3584 x 152064 loses (682 and 695, and gains with either reader).
template <bool STREAM>
struct DWeightEpi {
  LanePos p;
  const GemmOutArgs* a;
  GradExchange ex;
  __device__ __forceinline__ void prefetch(int, int, int) {}
  __device__ __forceinline__ void operator()(Accum& acc, int /*tile*/, int r0, int c0) {
    const GemmOutArgs& A = *a;
    if (A.mode == VAMD_DW_STORE) {
      const LineExchange line(ex);
#pragma unroll
      for (int nb = 0; nb < kNB2; ++nb)
#pragma unroll
        for (int mb = 0; mb < kMB / 4; ++mb) {
          u32x4 v[4];
          line.run(acc, mb, nb, v);
          const int col = c0 + p.wc * 128 + mb * 64 + 8 * line.rd_chunk;  // c_valid % 128 == 0: 8 columns are all in or all out
          const int row0 = r0 + p.wr * (kNB * kBlk) + nb * 32 + line.rd_row;
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (col < A.c_valid && row0 + 8 * i < A.r_valid) {
              auto* const dst = reinterpret_cast<u32x4_at8*>(A.out + (int64_t)(row0 + 8 * i) * A.ld_out + col);
              if constexpr (STREAM) __builtin_nontemporal_store(v[i], dst);
              else *dst = v[i];
            }
        }
      return;
    }
#pragma unroll
    for (int nb = 0; nb < kNB2; ++nb)
#pragma unroll
      for (int mb = 0; mb < kMB2; ++mb) {
        f32x4 v[4];
        exchange_patch(ex, acc, mb, nb, v);
        const int col = c0 + p.wc * 128 + mb * 32 + 4 * ex.rd_chunk;
        if (col >= A.c_valid) continue;
        const int row0 = r0 + p.wr * (kNB * kBlk) + nb * 32 + ex.rd_row;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int row = row0 + 8 * i;
          if (row >= A.r_valid) continue;
          f32x4 x = v[i];
          const int64_t off = (int64_t)row * A.ld_out + col;
          u32x2* dst = reinterpret_cast<u32x2*>(A.out + off);
          if (A.mode == VAMD_DW_ADD_BF16) {
            const u32x2 o = *dst;
            x[0] += bf16_bits_to_float(o[0] & 0xffffu);
            x[1] += bf16_bits_to_float(o[0] >> 16);
            x[2] += bf16_bits_to_float(o[1] & 0xffffu);
            x[3] += bf16_bits_to_float(o[1] >> 16);
          } else if (A.mode >= VAMD_DW_F32_STORE) {
            f32x4* acc = reinterpret_cast<f32x4*>(A.acc32 + off);
            if (A.mode != VAMD_DW_F32_STORE) x = x + *acc;
            *acc = x;
            if (A.mode != VAMD_DW_F32_ADD_FINISH) continue;
          }
          *dst = pack_bf16x4(x[0], x[1], x[2], x[3]);
        }
      }
  }
};

// Both gradient GEMMs of one vocabulary chunk in a single launch: a workgroup first walks its share of the d_hidden
// units, then its share of the d_weight tiles, shared out by plan_gradients() so that all workgroups finish together.
template <bool STREAM>
__global__ __launch_bounds__(kThreads) void lce_dgrad_kernel(GemmOutArgs gh, GemmOutArgs gw, GradPlan plan) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int nwg = gridDim.x;
  const int wg = xcd_regroup(blockIdx.x, nwg);
  const LanePos pos = lane_pos();
  if (gh.r_tiles > 0) {
    SplitKSched sched{TileGrid{gh.r_tiles, gh.c_tiles}, plan.splits, plan.split_slabs, gh.k_slabs, nwg, wg};
    DHiddenEpi epi;
    epi.p = pos;
    epi.a = &gh;
    epi.sched = sched;
    epi.ex.init(lds + kLdsBytes, pos);
    run_tiles<false, true>(gh.R, gh.C, sched, epi, lds);
  }
  __syncthreads();
  {
    LateStartSched sched{TileGrid{gw.r_tiles, gw.c_tiles}, gw.k_slabs, nwg, wg, plan.extra, plan.late};
    DWeightEpi<STREAM> epi;
    epi.p = pos;
    epi.a = &gw;
    epi.ex.init(lds + kLdsBytes, pos);
    run_tiles<true, true>(gw.R, gw.C, sched, epi, lds);
  }
}

// d_hidden over at most kFewTokens tokens: the k range (the vocabulary) is cut into pieces, each summed into an fp32
// accumulator of its own by one workgroup per 256 hidden columns.  Bound by reading the weight, as the forward pass over few
// tokens is, and built like it: 128 token rows, so that the MFMAs of a slab of the weight take half as long as the slab takes
// out of HBM, and three LDS stages, so that two slabs are in flight while one is multiplied.  As pieces of 256-token tiles
// in lce_dgrad_kernel, with one slab in flight and half of the MFMAs on padding, and as here (with the launch that sums the
// pieces): 64 x 896 x 151936 125 -> 75 us, 64 x 3584 x 152064 247 -> 202 (5.6 TB/s), 128 x 3584 x 152064 340 -> 230,
// 128 x 1024 x 8192 51 -> 25.
struct FewHiddenArgs {
  Operand dz;      // R: [n_tokens][panel pitch], k = panel column
  Operand weight;  // C: K-major, [vocab][hidden]
  int k_slabs, split_slabs, col_tiles;
  int stream_from;  // stream_from()
  float* acc32;     // [pieces][n_tokens][hidden]
  int n_tokens, hidden;
};

__global__ __launch_bounds__(kThreads) void lce_dhidden_few_kernel(FewHiddenArgs a) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  // the workgroups of a piece are neighbours: they read the same columns of the panel
  const int wg = xcd_regroup(blockIdx.x, gridDim.x), piece = wg / a.col_tiles, c0 = (wg - piece * a.col_tiles) * kTile;
  const int k_begin = piece * a.split_slabs, left = a.k_slabs - k_begin;
  const int slabs = left < a.split_slabs ? left : a.split_slabs;  // > 0
  const int w = threadIdx.x >> 6, lx = threadIdx.x & 15, lq = (threadIdx.x >> 4) & 3;
  const int wr = w % kFewWavesR, wc = w / kFewWavesR;

  SlabDma<false> dma_r;
  SlabDma<true> dma_c;
  dma_r.init(a.dz);
  dma_c.init(a.weight);
  dma_c.set_tile(a.weight, c0);
  FragAddr<false> fr;
  FragAddr<true> fc;
  fr.init(wr * kNB, kNB);
  fc.init(wc * kFewMB, kFewMB);

  // fetch cursor; past the end it stays on the last slab
  const u32x4 rs_r = tile_rsrc<false>(a.dz, 0), rs_c = tile_rsrc<true>(a.weight, c0);
  int k2 = 0, fill = 0;
  auto fetch = [&]() {
    const int k0 = (k_begin + k2) * kBK;
    const SlabSrc r{rs_r, slab_soff<false>(a.dz, k0)}, c{rs_c, slab_soff<true>(a.weight, k0)};
    const unsigned base = lds_address(lds) + (unsigned)fill * kFewStageBytes;
#pragma unroll
    for (int i = 0; i < kFewLoadsR; ++i) dma_r.issue_one(i, r, base);
    few_fetch_weight(dma_c, c, base + kFewTokens * kBK * 2, k_begin * kBK >= a.stream_from);
    fill = fill == kFewStages - 1 ? 0 : fill + 1;
    if (k2 < slabs - 1) ++k2;
  };
  fetch();
  fetch();

  f32x4 acc[kFewMB][kNB];
#pragma unroll
  for (int mb = 0; mb < kFewMB; ++mb)
#pragma unroll
    for (int nb = 0; nb < kNB; ++nb) acc[mb][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
  int stage = 0;
  for (int it = 0; it < slabs; ++it) {
    // as in lce_forward_few_kernel: slab `it` has landed, and the stage before it takes slab it + 2
    asm volatile("s_waitcnt vmcnt(6) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    fetch();
    const char* cur = lds + stage * kFewStageBytes;
    stage = stage == kFewStages - 1 ? 0 : stage + 1;
    bf16x8 r[kSteps][kNB], c[kSteps][kFewMB];
#pragma unroll
    for (int ks = 0; ks < kSteps; ++ks) {
#pragma unroll
      for (int nb = 0; nb < kNB; ++nb) r[ks][nb] = fr.read(cur, ks, nb);
#pragma unroll
      for (int mb = 0; mb < kFewMB; ++mb) c[ks][mb] = fc.read(cur + kFewTokens * kBK * 2, ks, mb);
    }
#pragma unroll
    for (int ks = 0; ks < kSteps; ++ks)
#pragma unroll
      for (int mb = 0; mb < kFewMB; ++mb)
#pragma unroll
        for (int nb = 0; nb < kNB; ++nb)
          acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c[ks][mb], r[ks][nb], acc[mb][nb], 0, 0, 0);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no transfer into LDS is left when the workgroup ends

  float* const out = a.acc32 + (int64_t)piece * a.n_tokens * a.hidden;
#pragma unroll
  for (int nb = 0; nb < kNB; ++nb) {
    const int tok = wr * (kNB * kBlk) + nb * kBlk + lx;
#pragma unroll
    for (int mb = 0; mb < kFewMB; ++mb) {
      const int col = c0 + wc * (kFewMB * kBlk) + mb * kBlk + 4 * lq;  // hidden % 128 == 0: 4 columns are all in or all out
      if (tok < a.n_tokens && col < a.hidden)
        *reinterpret_cast<f32x4*>(out + (int64_t)tok * a.hidden + col) = acc[mb][nb];
    }
  }
}

// d_hidden = sum of the pieces' fp32 accumulators, rounded once.
__global__ __launch_bounds__(256) void lce_dhidden_sum_kernel(const float* acc32, int pieces, int64_t elements,
                                                              uint16_t* out) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= elements) return;
  f32x4 s = *reinterpret_cast<const f32x4*>(acc32 + i);
#pragma unroll 16
  for (int k = 1; k < pieces; ++k) s = s + *reinterpret_cast<const f32x4*>(acc32 + (int64_t)k * elements + i);
  *reinterpret_cast<u32x2*>(out + i) = pack_bf16x4(s[0], s[1], s[2], s[3]);
}

// =============================================================================================
// Host side
// =============================================================================================
template <class K>
static int allow_big_lds(K kernel, int bytes = kLdsBytes) {
  VAMD_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                               bytes));
  return VAMD_OK;
}

typedef void (*ForwardKernel)(FwdArgs);
// [walk, or few tokens][logits kept][squared sums]
static const ForwardKernel kForwardKernels[kWalks + 1][2][2] = {
    {{lce_forward_kernel<false, false, kSplits>, lce_forward_kernel<false, true, kSplits>},
     {lce_forward_kernel<true, false, kSplits>, lce_forward_kernel<true, true, kSplits>}},
    {{lce_forward_kernel<false, false, kSplitsIdle>, lce_forward_kernel<false, true, kSplitsIdle>},
     {lce_forward_kernel<true, false, kSplitsIdle>, lce_forward_kernel<true, true, kSplitsIdle>}},
    {{lce_forward_kernel<false, false, kBands>, lce_forward_kernel<false, true, kBands>},
     {lce_forward_kernel<true, false, kBands>, lce_forward_kernel<true, true, kBands>}},
    {{lce_forward_few_kernel<false, false>, lce_forward_few_kernel<false, true>},
     {lce_forward_few_kernel<true, false>, lce_forward_few_kernel<true, true>}}};

// The kernels use more LDS than the default launch limit; the limit is a per-device function
// attribute, so it is raised once on every device the library is used on.
static int ensure_lds_attributes() {
  static std::mutex mu;
  static bool done[64];
  int dev = 0;
  VAMD_HIP(hipGetDevice(&dev));
  VAMD_REQUIRE(dev >= 0 && dev < 64, "lce: device index %d out of range", dev);
  std::lock_guard<std::mutex> lock(mu);
  if (done[dev]) return VAMD_OK;
  int s;
  for (int w = 0; w < kWalks; ++w)
    for (int pi2 = 0; pi2 < 2; ++pi2) {
      if ((s = allow_big_lds(kForwardKernels[w][0][pi2], kLdsBytes + kFwdTokenLds)) != VAMD_OK) return s;
      if ((s = allow_big_lds(kForwardKernels[w][1][pi2], kLdsBytes + kFwdCacheLds)) != VAMD_OK) return s;
    }
  if ((s = allow_big_lds(lce_forward_few_kernel<false, false>, kFewLds)) != VAMD_OK) return s;
  if ((s = allow_big_lds(lce_forward_few_kernel<false, true>, kFewLds)) != VAMD_OK) return s;
  if ((s = allow_big_lds(lce_forward_few_kernel<true, false>, kFewCacheLds)) != VAMD_OK) return s;
  if ((s = allow_big_lds(lce_forward_few_kernel<true, true>, kFewCacheLds)) != VAMD_OK) return s;
  if ((s = allow_big_lds(lce_recompute_kernel, kLdsBytes + kRecomputeExtraLds)) != VAMD_OK) return s;
  if ((s = allow_big_lds(lce_dhidden_few_kernel, kFewLds)) != VAMD_OK) return s;
  if ((s = allow_big_lds(lce_dgrad_kernel<false>, kLdsBytes + kGradStageBytes)) != VAMD_OK) return s;
  if ((s = allow_big_lds(lce_dgrad_kernel<true>, kLdsBytes + kGradStageBytes)) != VAMD_OK) return s;
  done[dev] = true;
  return VAMD_OK;
}

static inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Row pitch of the staged d_logits panel: the chunk width plus 256 bytes, so that the rows a
// wavefront touches together (32 .. 64 consecutive tokens at one column) spread over the memory
// channels instead of landing on a power-of-two stride.
static inline int64_t dz_pitch(int64_t cv) { return cv + 128; }

// max_slots: most partial states (of 256 tokens each) the caller's buffer holds; the built-in buffer of the entry point that
// allocates nothing is sized for 256 CUs and must serve a part with more of them too.
static FwdPlan plan_forward(int64_t n_tokens, int64_t vocab, int64_t max_slots = INT64_MAX) {
  const int64_t cus = device_cu_count(), tok_tiles = ceil_div(n_tokens, kTile), voc_tiles = ceil_div(vocab, kTile);
  FwdPlan p{};
  p.tok_tiles = (int)tok_tiles;
  p.voc_tiles = (int)voc_tiles;
  int64_t sp = cus / tok_tiles;  // as many workgroups as fit in one round over the CUs
  if (sp > max_slots / tok_tiles) sp = max_slots / tok_tiles;
  if (sp < 1) sp = 1;
  if (sp > voc_tiles) sp = voc_tiles;
  p.splits = (int)sp;
  if (n_tokens <= kFewTokens) {
    // equal ranges of weight rows; 64 rows are the least that is worth a workgroup
    const int64_t even = ceil_div(ceil_div(vocab, cus < max_slots ? cus : max_slots), kBlk) * kBlk;
    p.few_cols = (int)(even < 64 ? 64 : even);
    p.splits = (int)ceil_div(vocab, p.few_cols);
    return p;
  }
  if (cus % (8 * kXcds) != 0) return p;
  const int64_t split_rounds = ceil_div(tok_tiles * sp, cus) * ceil_div(voc_tiles, sp);
  FwdPlan b = p;
  b.splits = 0;
  b.group = (int)(cus / kXcds);
  for (int k = 0; k < 4; ++k) b.count[k] = (int)ceil_div(voc_tiles, b.group >> k);
  b.waves = (int)(tok_tiles / 64);
  int64_t rounds = tok_tiles % 64 / 8 * b.count[3];
  for (int k = 0; k < 3; ++k) rounds += (tok_tiles >> k & 1) * b.count[k];
  b.rounds = (int)rounds;
  const int64_t band_rounds = (int64_t)b.waves * b.count[3] + ceil_div(rounds, kXcds);
  // Bands cost what 1 - 2 % more rounds would (more of the weight's traffic, states written more than once): 9000 tokens x
  // 3584 x 152064, 84 rounds in bands and 85 in splits, 7.07 and 6.97 ms; 3300 x 896 x 151936, 31 and 32, 0.710 and
  // 0.736; 11290 x 3584 x 152064, 105 and 119, 8.81 and 9.24; 22000 tokens, 200 and 297, 16.9 and 19.9.
  return rounds < (1 << 27) && 34 * band_rounds <= 33 * split_rounds && b.slots() <= max_slots ? b : p;
}

// Any vocabulary size is served; only the fp32 logits cache, whose rows are read and written 32 bytes at a time,
// needs a multiple of 8.
static int check_head_shapes(int64_t n, int64_t h, int64_t v, const void* logits_cache) {
  VAMD_REQUIRE(n > 0 && h > 0 && v > 0, "lce: empty problem n=%lld h=%lld v=%lld", (long long)n, (long long)h,
               (long long)v);
  VAMD_REQUIRE(h % 128 == 0, "lce: hidden_size %lld must be a multiple of 128", (long long)h);
  VAMD_REQUIRE(!logits_cache || v % 8 == 0, "lce: a logits cache needs a vocab that is a multiple of 8, got %lld",
               (long long)v);
  VAMD_REQUIRE(n < (1ll << 30) && v < (1ll << 30), "lce: n_tokens / vocab too large");
  VAMD_REQUIRE(reinterpret_cast<uintptr_t>(logits_cache) % 16 == 0, "lce: logits_cache must be 16-byte aligned");
  return VAMD_OK;
}

static int64_t default_vocab_chunk(int64_t n_tokens, int64_t hidden_size, int64_t vocab, int64_t requested) {
  const int64_t n_pad = ceil_div(n_tokens, kTile) * kTile;
  const int64_t v_pad = ceil_div(vocab, kTile) * kTile;
  int64_t cv = requested;
  if (cv <= 0) {
    int64_t budget = 512ll << 20;  // bytes of bf16 d_logits staged at a time
    if (const char* e = getenv("VAMD_LCE_DZ_BUDGET_MB")) {
      const long mb = strtol(e, nullptr, 10);
      if (mb > 0) budget = (int64_t)mb << 20;
    }
    cv = budget / (n_pad * 2) / kTile * kTile;
  }
  cv = ceil_div(cv, kTile) * kTile;
  // the weight rows of a chunk are walked with 32-bit byte offsets from the chunk's first row
  const int64_t cap = ((1ll << 32) - 1) / (hidden_size * 2) / kTile * kTile;
  if (cv > cap) cv = cap;
  if (cv < kTile) cv = kTile;
  if (cv > v_pad) cv = v_pad;
  return cv;
}

// d_hidden has few tiles with a long k range (the chunk's vocabulary), d_weight many tiles with a short one (the tokens),
// and both sum up to the same number of slabs.  Whole d_hidden tiles only balance when there are several per CU: 777
// tokens x 896 have 16 tiles of 2374 slabs, which kept 16 CUs busy while 240 waited (2983 us; cut into 11 pieces 463 us),
// 7339 x 3584 have 406 on 256 CUs (87 % of the launch busy).  So a tile's k range is cut into pieces of equal length,
// each summed in fp32 into an accumulator of its own, and the d_weight tiles are shared out so that the workgroups
// with a piece more get correspondingly fewer tiles.  The number of pieces is the one whose slowest workgroup is
// quickest, counting in slabs (1.4 us each): an epilogue about 2, and a d_weight tile of up to 3 slabs 7 in all: with every CU
// storing, its 128 KB take 6 us, and a slab or three more hardly show.  It decides over 129 to 192 tokens (three slabs; up to 128
// tokens d_hidden has a kernel of its own, but for vocabularies below kFewMinVocab, where it makes no difference, 64 x 1024 x 512
// 20.1 us and 64 x 2048 x 768 24.4, and for several chunks, which are not measured).  Backward pass with 2 for every epilogue, and as it is, us: 130 x 896 x 151936 193 and 190, 130 x 3584 x 152064 692
// and 615, 130 x 4096 x 128256 630 and 545; 160 tokens 200 and 198, 712 and 616; 192 tokens 207 and 209, 726 and 637, 643 and
// 582; 160 x 1024 x 8192 52 both.  The 7 and where it ends are a fit, not a law: four slabs stay at 4 + 2 = 6, below three,
// because 7 is slower there (256 tokens, with 6 and 7, us: 896 192 and 201, 3584 646 and 675, 4096 585 and 613).  Results in fp32
// or added to what is there, which move two to four times the bytes, are counted alike: not measured.
constexpr int kEpilogueSlabs = 2, kFewTileSlabs = 3, kFewTileCost = 7, kMaxSplits = 64, kMinPieceSlabs = 32;
constexpr int64_t kMaxPieceBytes = 256ll << 20;  // bound on the pieces' accumulators
static GradPlan plan_gradients(int64_t n_tokens, int64_t hidden_size, int64_t cols, bool want_dh, bool want_dw,
                               int cus, int fixed_pieces = 0) {
  const int64_t h_tiles = ceil_div(hidden_size, kTile);
  const int64_t th = want_dh ? ceil_div(n_tokens, kTile) * h_tiles : 0, kh = ceil_div(cols, kBK);
  const int64_t tw = want_dw ? ceil_div(cols, kTile) * h_tiles : 0, tile_slabs = ceil_div(n_tokens, kBK);
  const int64_t cost_w = tile_slabs <= kFewTileSlabs ? kFewTileCost : tile_slabs + kEpilogueSlabs;
  const int64_t piece_bytes = n_tokens * hidden_size * 4;
  GradPlan best;
  best.split_slabs = (int)kh;
  double best_cost = 0;
  bool first = true;
  for (int64_t want = fixed_pieces ? fixed_pieces : 1; want <= (fixed_pieces ? fixed_pieces : want_dh ? kMaxSplits : 1);
       ++want) {
    const int64_t len = ceil_div(kh, want), pieces = ceil_div(kh, len);
    if (pieces != want && !fixed_pieces) continue;  // the same cut as for a smaller count
    if (want > 1 && len < kMinPieceSlabs && !fixed_pieces) break;  // nothing to gain that pays for the summing launch
    if (pieces > 1 && pieces * piece_bytes > kMaxPieceBytes && !fixed_pieces) break;
    const int64_t units = th * pieces, cost_h = len + kEpilogueSlabs;
    const int64_t extra = units % cus, few = units / cus * cost_h, many = few + (extra ? cost_h : 0);
    // least time in which all d_weight tiles fit behind the d_hidden units
    int64_t lo = many, hi = many + (ceil_div(tw, cus) + 1) * cost_w;
    while (lo < hi) {
      const int64_t t = (lo + hi) / 2;
      const int64_t fit = extra * ((t - many) / cost_w) + (cus - extra) * ((t - few) / cost_w);
      if (fit >= tw) hi = t;
      else lo = t + 1;
    }
    const double cost = (double)lo + (pieces > 1 ? 4.0 + (double)(2 * pieces * piece_bytes) / 7.0e6 : 0.0);  // a launch, 5 TB/s
    if (first || cost < best_cost) {
      first = false;
      best_cost = cost;
      best.splits = (int)pieces;
      best.split_slabs = (int)len;
      best.extra = (int)extra;
      best.late = (int)((lo - few) / cost_w - (lo - many) / cost_w);
    }
  }
  return best;
}

// Whether d_hidden is formed by lce_dhidden_few_kernel: over few tokens, in one vocabulary chunk (it starts its accumulators
// afresh).  It gains at every vocabulary measured (64 x 1024 x 2048, both gradients: 44 -> 29 us); below two pieces of
// kFewMinSlabs slabs there is nothing to share out.
constexpr int kFewMinSlabs = 8, kFewMinVocab = 2 * kFewMinSlabs * kBK;
static bool few_hidden(int64_t planned_tokens, int64_t chunk, int64_t vocab) {
  return planned_tokens <= kFewTokens && vocab >= kFewMinVocab && chunk >= vocab;
}

// Its workgroups: as many pieces as fill one round over the CUs.
static GradPlan plan_few_hidden(int64_t hidden_size, int64_t vocab, int cus) {
  const int64_t slabs = ceil_div(vocab, kBK), pieces = cus / ceil_div(hidden_size, kTile);
  GradPlan p;
  p.split_slabs = (int)ceil_div(slabs, pieces < 1 ? 1 : pieces);
  if (p.split_slabs < kFewMinSlabs) p.split_slabs = kFewMinSlabs;
  p.splits = (int)ceil_div(slabs, p.split_slabs);
  return p;
}

// The first weight row that the few-token kernels read past the caches.
static int stream_from(int64_t hidden_size, int64_t vocab) {
  const int64_t row_bytes = hidden_size * 2;
  return (int)(vocab * row_bytes <= kFittingWeightBytes ? vocab : kCachedWeightBytes / row_bytes);
}

}  // namespace vamd

using namespace vamd;

extern "C" int vamd_lce_timing_enable(int on) {
  g_timing_on.store(on != 0);
  return VAMD_OK;
}

extern "C" int vamd_lce_timing_collect(double* ms_by_kernel, int64_t* launches_by_kernel) {
  VAMD_REQUIRE(ms_by_kernel && launches_by_kernel, "timing_collect: null pointer");
  for (int i = 0; i < kNumTags; ++i) {
    ms_by_kernel[i] = 0;
    launches_by_kernel[i] = 0;
  }
  int status = VAMD_OK;
  std::lock_guard<std::mutex> lock(g_timed_mu);
  for (TimedLaunch& t : g_timed) {
    float ms = 0.f;
    if (hipEventSynchronize(t.stop) != hipSuccess || hipEventElapsedTime(&ms, t.start, t.stop) != hipSuccess) {
      set_error("timing_collect: event query failed");
      status = VAMD_EHIP;
    } else {
      ms_by_kernel[t.tag] += ms;
      launches_by_kernel[t.tag] += 1;
    }
    (void)hipEventDestroy(t.start);
    (void)hipEventDestroy(t.stop);
  }
  g_timed.clear();
  return status;
}

extern "C" size_t vamd_lce_forward_workspace_bytes(int64_t n_tokens, int64_t hidden_size, int64_t vocab) {
  (void)hidden_size;
  if (n_tokens <= 0 || vocab <= 0) return 0;
  return (size_t)plan_forward(n_tokens, vocab).slots() * kTile * (sizeof(float4) + sizeof(float));  // state + squared sums
}

// Forward launches shared by the two entry points; `workspace` holds at least
// vamd_lce_forward_workspace_bytes() bytes and the arguments have been checked.
static int lce_forward_launch(const void* hidden, const void* weight, const int64_t* labels, int64_t n_tokens,
                              int64_t hidden_size, int64_t vocab, float rcp_temperature, float* logprobs,
                              float* entropy, float* lse, float* mean_z, float* logits_cache, float* sum_pi_squared,
                              void* workspace, void* stream, int64_t max_slots = INT64_MAX) {

  FwdArgs a;
  a.hidden = Operand{static_cast<const uint16_t*>(hidden), hidden_size, (int)n_tokens, (int)hidden_size};
  a.weight = Operand{static_cast<const uint16_t*>(weight), hidden_size, (int)vocab, (int)hidden_size};
  a.labels = labels;
  a.n_tokens = (int)n_tokens;
  a.vocab = (int)vocab;
  a.k_slabs = (int)(hidden_size / kBK);
  a.plan = plan_forward(n_tokens, vocab, max_slots);
  a.scale2 = rcp_temperature * kLog2e;
  a.rcp_t = rcp_temperature;
  a.partials = static_cast<float4*>(workspace);
  a.pi2_partials = sum_pi_squared
                       ? reinterpret_cast<float*>(static_cast<char*>(workspace) +
                                                  (size_t)a.plan.slots() * kTile * sizeof(float4))
                       : nullptr;
  a.z_cache = logits_cache;
  a.stream_from = stream_from(hidden_size, vocab);
  hipStream_t s = static_cast<hipStream_t>(stream);
  {
    ScopedTiming tm(kTagForward, s);
    const dim3 grid(a.plan.splits ? a.plan.tok_tiles * a.plan.splits : a.plan.group * kXcds), block(kThreads);
    const bool pi2 = sum_pi_squared != nullptr, cache = logits_cache != nullptr;
    const int lds_bytes = a.plan.few_cols ? (cache ? kFewCacheLds : kFewLds) : kLdsBytes + (cache ? kFwdCacheLds : kFwdTokenLds);
    const bool idle = ceil_div(n_tokens, kNB * kBlk) % (kTile / (kNB * kBlk)) != 0;  // a wavefront owns kNB blocks of tokens
    const int walk = a.plan.few_cols ? kWalks : !a.plan.splits ? kBands : idle ? kSplitsIdle : kSplits;
    hipLaunchKernelGGL(kForwardKernels[walk][cache][pi2], grid, block, lds_bytes, s, a);
  }
  VAMD_LAUNCH_CHECK();

  MergeArgs m;
  m.partials = a.partials;
  m.pi2_partials = a.pi2_partials;
  m.sum_pi_squared = sum_pi_squared;
  m.plan = a.plan;
  // a lane per state up to a wavefront per token: fewer states than lanes would leave lanes idle
  const int states = a.plan.splits ? a.plan.splits : (int)(a.plan.slots() / a.plan.tok_tiles);
  m.lanes_log2 = 0;
  while (m.lanes_log2 < 6 && (2 << m.lanes_log2) <= states) ++m.lanes_log2;
  m.n_tokens = (int)n_tokens;
  m.rcp_t = rcp_temperature;
  m.logprobs = logprobs;
  m.entropy = entropy;
  m.lse = lse;
  m.mean_z = mean_z;
  {
    ScopedTiming tm(kTagMerge, s);
    hipLaunchKernelGGL(lce_merge_kernel, dim3((unsigned)ceil_div(n_tokens << m.lanes_log2, 256)), dim3(256), 0, s, m);
  }
  VAMD_LAUNCH_CHECK();
  return VAMD_OK;
}

static int check_forward_args(const void* hidden, const void* weight, const int64_t* labels, int64_t n_tokens,
                              int64_t hidden_size, int64_t vocab, float rcp_temperature, const float* logprobs,
                              const float* entropy, const float* lse, const float* mean_z, const float* logits_cache) {
  int st = check_head_shapes(n_tokens, hidden_size, vocab, logits_cache);
  if (st != VAMD_OK) return st;
  VAMD_REQUIRE(hidden && weight && labels && logprobs && entropy && lse && mean_z, "lce_forward: null pointer");
  VAMD_REQUIRE(rcp_temperature > 0.f, "lce_forward: temperature must be positive");
  return VAMD_OK;
}

extern "C" int vamd_lce_forward(const void* hidden, const void* weight, const int64_t* labels, int64_t n_tokens,
                                int64_t hidden_size, int64_t vocab, float rcp_temperature, float* logprobs,
                                float* entropy, float* lse, float* mean_z, float* logits_cache,
                                float* sum_pi_squared, void* workspace, size_t workspace_bytes, void* stream) {
  int st = check_forward_args(hidden, weight, labels, n_tokens, hidden_size, vocab, rcp_temperature, logprobs, entropy,
                              lse, mean_z, logits_cache);
  if (st != VAMD_OK) return st;
  const size_t need = vamd_lce_forward_workspace_bytes(n_tokens, hidden_size, vocab);
  if (!workspace || workspace_bytes < need) {
    set_error("lce_forward: workspace %zu bytes, need %zu", workspace_bytes, need);
    return VAMD_EWORKSPACE;
  }
  if ((st = ensure_lds_attributes()) != VAMD_OK) return st;
  return lce_forward_launch(hidden, weight, labels, n_tokens, hidden_size, vocab, rcp_temperature, logprobs, entropy,
                            lse, mean_z, logits_cache, sum_pi_squared, workspace, stream);
}

// ---------------------------------------------------------------------------------------------
// The forward pass for callers that cannot allocate: the per-(token tile, vocabulary split)
// softmax partials live in a file-scope device array instead of a caller workspace.  Every GPU
// holds its own copy of the array at its own address; the address is looked up once per device.
// The array's name is only a host-side handle for that lookup: launches and copies use the
// looked-up pointer.
namespace vamd {
// up to 65536 tokens in bands: (34 bands + 8 XCDs) x 32 workgroups x 256 tokens
constexpr int64_t kStaticSlots = (VAMD_LCE_STATIC_MAX_TOKENS / (8 * kTile) + 2 + kXcds) * 32;
constexpr size_t kStaticScratchBytes = (size_t)kStaticSlots * kTile * (sizeof(float4) + sizeof(float)) + 512;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

static int static_scratch_pointer(void** out) {
  static std::mutex mu;
  static void* ptr_by_device[64];
  int dev = 0;
  VAMD_HIP(hipGetDevice(&dev));
  VAMD_REQUIRE(dev >= 0 && dev < 64, "lce: device index %d out of range", dev);
  std::lock_guard<std::mutex> lock(mu);
  if (!ptr_by_device[dev]) {
    void* p = nullptr;
    VAMD_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    VAMD_REQUIRE(p != nullptr, "lce: the static scratch array has no device address");
    ptr_by_device[dev] = p;
  }
  *out = ptr_by_device[dev];
  return VAMD_OK;
}
}  // namespace vamd

extern "C" int vamd_lce_forward_static(const void* hidden, const void* weight, const int64_t* labels,
                                       int64_t n_tokens, int64_t hidden_size, int64_t vocab, float rcp_temperature,
                                       float* logprobs, float* entropy, float* lse, float* mean_z,
                                       float* sum_pi_squared, void* stream) {
  int st = check_forward_args(hidden, weight, labels, n_tokens, hidden_size, vocab, rcp_temperature, logprobs, entropy,
                              lse, mean_z, nullptr);
  if (st != VAMD_OK) return st;
  VAMD_REQUIRE(n_tokens <= VAMD_LCE_STATIC_MAX_TOKENS,
               "lce_forward_static: %lld tokens; the built-in buffer serves at most %d tokens per call: use "
               "vamd_lce_forward with a caller workspace",
               (long long)n_tokens, (int)VAMD_LCE_STATIC_MAX_TOKENS);
  if ((st = ensure_lds_attributes()) != VAMD_OK) return st;
  void* ws = nullptr;
  if ((st = static_scratch_pointer(&ws)) != VAMD_OK) return st;
  // Every partial the merge kernel reads is written by the forward kernel of the same call, so
  // nothing in the buffer has to start at zero and a previous call's contents do not matter.
  // the plan is made so that its states fit the buffer whatever the CU count
  return lce_forward_launch(hidden, weight, labels, n_tokens, hidden_size, vocab, rcp_temperature, logprobs, entropy,
                            lse, mean_z, nullptr, sum_pi_squared, ws, stream, kStaticSlots);
}

namespace vamd {
// How d_hidden is formed: the pieces of its k range.  Decided as if both gradients were asked for, whichever are, so that
// d_hidden is the same bits either way; the first (widest) vocabulary chunk decides for all chunks.  For some of the tokens of
// a larger call it is that call's way, so that its bits come out, where it has one vocabulary chunk.  With several chunks it sums
// over other ranges anyway: there the tokens at hand decide (1000 of 11290 x 3584 x 152064 would run as 56 whole tiles).
struct HiddenPlan {
  bool few;         // lce_dhidden_few_kernel
  int pieces;
  int split_slabs;  // few: slabs of a piece
  int accumulators(int64_t chunk, int64_t vocab) const {  // fp32 [n_tokens][hidden] each
    return few || pieces > 1 || chunk < vocab ? pieces : 0;
  }
};
static HiddenPlan plan_hidden(int64_t n_tokens, int64_t planned_tokens, int64_t hidden_size, int64_t vocab,
                              int64_t vocab_chunk) {
  const int64_t cv = default_vocab_chunk(n_tokens, hidden_size, vocab, vocab_chunk);
  const bool same_ranges =
      planned_tokens > n_tokens && default_vocab_chunk(planned_tokens, hidden_size, vocab, vocab_chunk) >= vocab;
  const int64_t planned = same_ranges ? planned_tokens : n_tokens;
  const bool few = few_hidden(planned, cv, vocab);
  const GradPlan p = few ? plan_few_hidden(hidden_size, vocab, device_cu_count())
                         : plan_gradients(planned, hidden_size, cv < vocab ? cv : vocab, true, true, device_cu_count());
  return HiddenPlan{few, p.splits, p.split_slabs};
}
}  // namespace vamd

extern "C" size_t vamd_lce_backward_subset_workspace_bytes(int64_t n_tokens, int64_t planned_tokens,
                                                           int64_t hidden_size, int64_t vocab, int64_t vocab_chunk) {
  if (n_tokens <= 0 || vocab <= 0 || hidden_size <= 0) return 0;
  const int64_t n_pad = ceil_div(n_tokens, kTile) * kTile;
  const int64_t cv = default_vocab_chunk(n_tokens, hidden_size, vocab, vocab_chunk);
  const int accumulators =
      plan_hidden(n_tokens, planned_tokens, hidden_size, vocab, vocab_chunk).accumulators(cv, vocab);
  return align_up((size_t)n_pad * dz_pitch(cv) * 2, 256) + align_up((size_t)accumulators * n_tokens * hidden_size * 4, 256);
}

extern "C" size_t vamd_lce_backward_workspace_bytes(int64_t n_tokens, int64_t hidden_size, int64_t vocab,
                                                    int64_t vocab_chunk) {
  return vamd_lce_backward_subset_workspace_bytes(n_tokens, n_tokens, hidden_size, vocab, vocab_chunk);
}

extern "C" int vamd_lce_backward(const void* hidden, const void* weight, const int64_t* labels, int64_t n_tokens,
                                 int64_t hidden_size, int64_t vocab, float rcp_temperature, const float* lse,
                                 const float* mean_z, const float* d_logprobs, const float* d_entropy,
                                 float d_entropy_scalar, const float* logits_cache, void* d_hidden, void* d_weight,
                                 int d_weight_mode, float* d_weight_acc32, int64_t vocab_chunk, void* workspace,
                                 size_t workspace_bytes, void* stream) {
  return vamd_lce_backward_subset(hidden, weight, labels, n_tokens, n_tokens, hidden_size, vocab, rcp_temperature, lse,
                                  mean_z, d_logprobs, d_entropy, d_entropy_scalar, logits_cache, d_hidden, d_weight,
                                  d_weight_mode, d_weight_acc32, vocab_chunk, workspace, workspace_bytes, stream);
}

extern "C" int vamd_lce_backward_subset(const void* hidden, const void* weight, const int64_t* labels,
                                        int64_t n_tokens, int64_t planned_tokens, int64_t hidden_size, int64_t vocab,
                                        float rcp_temperature, const float* lse, const float* mean_z,
                                        const float* d_logprobs, const float* d_entropy, float d_entropy_scalar,
                                        const float* logits_cache, void* d_hidden, void* d_weight, int d_weight_mode,
                                        float* d_weight_acc32, int64_t vocab_chunk, void* workspace,
                                        size_t workspace_bytes, void* stream) {
  return vamd_lce_backward_subset_rows(hidden, weight, labels, n_tokens, planned_tokens, hidden_size, vocab,
                                       rcp_temperature, lse, mean_z, d_logprobs, d_entropy, d_entropy_scalar,
                                       logits_cache, nullptr, d_hidden, d_weight, d_weight_mode, d_weight_acc32,
                                       vocab_chunk, workspace, workspace_bytes, stream);
}

extern "C" int vamd_lce_backward_subset_rows(const void* hidden, const void* weight, const int64_t* labels,
                                             int64_t n_tokens, int64_t planned_tokens, int64_t hidden_size,
                                             int64_t vocab, float rcp_temperature, const float* lse,
                                             const float* mean_z, const float* d_logprobs, const float* d_entropy,
                                             float d_entropy_scalar, const float* logits_cache,
                                             const int64_t* logits_rows, void* d_hidden, void* d_weight,
                                             int d_weight_mode, float* d_weight_acc32, int64_t vocab_chunk,
                                             void* workspace, size_t workspace_bytes, void* stream) {
  int st = check_head_shapes(n_tokens, hidden_size, vocab, logits_cache);
  if (st != VAMD_OK) return st;
  VAMD_REQUIRE(hidden && weight && labels && lse && mean_z, "lce_backward: null pointer");
  VAMD_REQUIRE(rcp_temperature > 0.f, "lce_backward: temperature must be positive");
  VAMD_REQUIRE(d_weight_mode >= VAMD_DW_STORE && d_weight_mode <= VAMD_DW_NONE,
               "lce_backward: unknown d_weight_mode %d", d_weight_mode);
  const bool want_dw = d_weight_mode != VAMD_DW_NONE;
  VAMD_REQUIRE(d_hidden || want_dw, "lce_backward: neither d_hidden nor a weight gradient is asked for");
  {
    const bool writes_bf16 = d_weight_mode <= VAMD_DW_ADD_BF16 || d_weight_mode == VAMD_DW_F32_ADD_FINISH;
    const bool uses_f32 = want_dw && d_weight_mode >= VAMD_DW_F32_STORE;
    VAMD_REQUIRE(!writes_bf16 || d_weight, "lce_backward: d_weight_mode %d writes d_weight, which is null", d_weight_mode);
    VAMD_REQUIRE(!uses_f32 || (d_weight_acc32 && reinterpret_cast<uintptr_t>(d_weight_acc32) % 16 == 0),
                 "lce_backward: d_weight_mode %d needs a 16-byte aligned d_weight_acc32", d_weight_mode);
  }
  {  // K-major operands are addressed with 32-bit byte offsets from their tile origin
    const int64_t rows_padded = ceil_div(n_tokens, kTile) * kTile;
    const int64_t row_pitch = dz_pitch(default_vocab_chunk(n_tokens, hidden_size, vocab, vocab_chunk));
    VAMD_REQUIRE(n_tokens * hidden_size * 2 < (1ll << 32) && rows_padded * row_pitch * 2 < (1ll << 32),
                 "lce_backward: hidden states (%lld x %lld) or the d_logits panel exceed 4 GiB; split the tokens into "
                 "chunks and accumulate d_weight", (long long)n_tokens, (long long)hidden_size);
  }
  VAMD_REQUIRE(planned_tokens >= n_tokens, "lce_backward: %lld tokens are no part of %lld", (long long)n_tokens,
               (long long)planned_tokens);
  const size_t need =
      vamd_lce_backward_subset_workspace_bytes(n_tokens, planned_tokens, hidden_size, vocab, vocab_chunk);
  if (!workspace || workspace_bytes < need) {
    set_error("lce_backward: workspace %zu bytes, need %zu", workspace_bytes, need);
    return VAMD_EWORKSPACE;
  }
  if ((st = ensure_lds_attributes()) != VAMD_OK) return st;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int cus = device_cu_count();

  const int tok_tiles = (int)ceil_div(n_tokens, kTile);
  const int64_t n_pad = (int64_t)tok_tiles * kTile;
  const int64_t cv = default_vocab_chunk(n_tokens, hidden_size, vocab, vocab_chunk);
  const int n_chunks = (int)ceil_div(vocab, cv);
  Carver carve(workspace);
  const int64_t pitch = dz_pitch(cv);
  uint16_t* dz = carve.take<uint16_t>((size_t)n_pad * pitch);
  // (a narrower last chunk may fill fewer pieces than the first)
  const HiddenPlan hp = plan_hidden(n_tokens, planned_tokens, hidden_size, vocab, vocab_chunk);
  const int pieces = d_hidden ? hp.pieces : 1, accumulators = d_hidden ? hp.accumulators(cv, vocab) : 0;
  const bool few = d_hidden && hp.few;
  float* acc32 = accumulators ? carve.take<float>((size_t)accumulators * n_tokens * hidden_size) : nullptr;
  const uint16_t* hid = static_cast<const uint16_t*>(hidden);
  const uint16_t* wgt = static_cast<const uint16_t*>(weight);
  const int h_tiles = (int)ceil_div(hidden_size, kTile);
  // Columns past the hidden size are not fetched (SlabDma::set_tile), except over 129 to 256 tokens, where the products wait for
  // memory and tiles that fetch less are no quicker but come out of step with the others.  Backward pass with them and without, us
  // (runs differ by 0.5 to 1 %): 130 x 896 x 151936 184.5 and 184.6, 160 tokens 195 and 197, 200 tokens 206 and 214, 256 tokens
  // 226 and 234; 200 x 1664 x 151936 333 and 352, 256 tokens 352 and 368; 256 x 384 x 151936 141 and 146; 200 x 1152 x 65536 121.5
  // and 122.5; 200 x 640 x 32000 63.9 and 62.9.
  const int col_extent = tok_tiles > 1 || few ? (int)hidden_size : h_tiles * kTile;

  for (int ci = 0; ci < n_chunks; ++ci) {
    const int64_t c0 = (int64_t)ci * cv;
    const int64_t left = vocab - c0;                   // vocabulary rows from c0 on
    const int64_t cols = left < cv ? left : cv;        // valid columns in this chunk
    const int chunk_tiles = (int)ceil_div(cols, kTile);

    if (logits_cache) {
      DLogitsArgs d;
      d.z_cache = logits_cache;
      d.rows = logits_rows;
      d.cache_rows = logits_rows ? planned_tokens : n_tokens;
      d.labels = labels;
      d.lse = lse;
      d.mean_z = mean_z;
      d.g_lp = d_logprobs;
      d.g_ent = d_entropy;
      d.g_ent_scalar = d_entropy_scalar;
      d.rcp_t = rcp_temperature;
      d.n_tokens = (int)n_tokens;
      d.vocab = (int)vocab;
      d.chunk_c0 = (int)c0;
      d.chunk_cols = chunk_tiles * kTile;
      d.dz = dz;
      d.dz_ld = (int)pitch;
      {
        ScopedTiming tm(kTagDLogits, s);
        hipLaunchKernelGGL(lce_dlogits_kernel, dim3((unsigned)(n_tokens * ceil_div(d.chunk_cols, kPanelCols))), dim3(256),
                           0, s, d);
      }
      VAMD_LAUNCH_CHECK();
    } else {
      RecomputeArgs r;
      r.hidden = Operand{hid, hidden_size, (int)n_tokens, (int)hidden_size};
      r.weight = Operand{wgt + c0 * hidden_size, hidden_size, (int)left, (int)hidden_size};
      r.labels = labels;
      r.lse = lse;
      r.mean_z = mean_z;
      r.g_lp = d_logprobs;
      r.g_ent = d_entropy;
      r.g_ent_scalar = d_entropy_scalar;
      r.n_tokens = (int)n_tokens;
      r.vocab_left = (int)left;
      r.chunk_c0 = (int)c0;
      r.k_slabs = (int)(hidden_size / kBK);
      r.tok_tiles = tok_tiles;
      r.chunk_tiles = chunk_tiles;
      r.rcp_t = rcp_temperature;
      r.dz = dz;
      r.dz_ld = (int)pitch;
      {
        const int tiles = tok_tiles * chunk_tiles;
        const int grid = tiles < cus ? tiles : cus;
        {
          ScopedTiming tm(kTagRecompute, s);
          hipLaunchKernelGGL(lce_recompute_kernel, dim3(grid), dim3(kThreads), kLdsBytes + kRecomputeExtraLds, s, r);
        }
        VAMD_LAUNCH_CHECK();
      }
    }

    // d_hidden: k runs over the chunk's vocabulary columns (staged zeros beyond `cols`)
    GemmOutArgs gh;
    // (the panel has no rows past n_tokens: they read as zero through the operand's bounds)
    gh.R = Operand{dz, pitch, (int)n_tokens, (int)cv};
    gh.C = Operand{wgt + c0 * hidden_size, hidden_size, col_extent, (int)left};
    gh.k_slabs = (int)ceil_div(cols, kBK);
    gh.r_tiles = d_hidden && !few ? tok_tiles : 0;  // an input that needs no gradient leaves its GEMM an empty tile list
    gh.c_tiles = h_tiles;
    gh.r_valid = (int)n_tokens;
    gh.c_valid = (int)hidden_size;
    // No more workgroups than pieces and tiles: with one on every CU, idle or not, and the tiles planned for all of them,
    // the backward of small heads took 85 instead of 73 us (2239 x 896 x 2000: 68 tiles), 44.5 instead of 42.1 (1209 x 128 x 1000).
    const int64_t units = (int64_t)h_tiles * ((gh.r_tiles ? (int64_t)tok_tiles * pieces : 0) + (want_dw ? chunk_tiles : 0));
    const int workgroups = (int)(units < cus ? units : cus);
    if (n_chunks == 1 && pieces == 1) gh.mode = kFinalBf16;
    else if (ci == 0) gh.mode = kStoreF32;
    else if (ci == n_chunks - 1 && pieces == 1) gh.mode = kFinalBf16AddPrev;
    else gh.mode = kAddF32;
    gh.acc32 = acc32;
    gh.out = static_cast<uint16_t*>(d_hidden);
    gh.ld_out = hidden_size;
    // d_weight rows of this chunk: k runs over tokens (staged zeros beyond n_tokens)
    GemmOutArgs gw;
    gw.R = Operand{dz, pitch, (int)(ceil_div(cols, 8) * 8), (int)n_tokens};
    gw.C = Operand{hid, hidden_size, col_extent, (int)n_tokens};
    gw.k_slabs = (int)ceil_div(n_tokens, kBK);
    gw.r_tiles = want_dw ? chunk_tiles : 0;
    gw.c_tiles = h_tiles;
    gw.r_valid = (int)cols;
    gw.c_valid = (int)hidden_size;
    gw.mode = d_weight_mode;
    gw.acc32 = d_weight_acc32 ? d_weight_acc32 + c0 * hidden_size : nullptr;
    gw.out = d_weight ? static_cast<uint16_t*>(d_weight) + c0 * hidden_size : nullptr;
    gw.ld_out = hidden_size;
    if (few) {
      const FewHiddenArgs f{gh.R, gh.C, gh.k_slabs, hp.split_slabs, h_tiles,
                            stream_from(hidden_size, vocab), acc32, (int)n_tokens, (int)hidden_size};
      {
        ScopedTiming tm(kTagDGrad, s);
        hipLaunchKernelGGL(lce_dhidden_few_kernel, dim3(h_tiles * pieces), dim3(kThreads), kFewLds, s, f);
      }
      VAMD_LAUNCH_CHECK();
    }
    if (workgroups > 0) {
      const GradPlan plan = plan_gradients(n_tokens, hidden_size, cols, gh.r_tiles > 0, want_dw, workgroups, few ? 1 : pieces);
      {
        ScopedTiming tm(kTagDGrad, s);
        const bool stream_dw = vocab * hidden_size * 2 > kCachedWeightBytes;
        hipLaunchKernelGGL(stream_dw ? lce_dgrad_kernel<true> : lce_dgrad_kernel<false>, dim3(workgroups), dim3(kThreads),
                           kLdsBytes + kGradStageBytes, s, gh, gw, plan);
      }
      VAMD_LAUNCH_CHECK();
    }
  }
  if (pieces > 1 || few) {
    const int64_t elements = n_tokens * hidden_size;
    {
      ScopedTiming tm(kTagDGrad, s);
      hipLaunchKernelGGL(lce_dhidden_sum_kernel, dim3((unsigned)ceil_div(elements, 1024)), dim3(256), 0, s, acc32, pieces,
                         elements, static_cast<uint16_t*>(d_hidden));
    }
    VAMD_LAUNCH_CHECK();
  }
  return VAMD_OK;
}
