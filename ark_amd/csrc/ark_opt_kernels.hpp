// ark_opt_kernels.hpp -- gfx950 kernels of the optimizer step.
//
// Two stream-ordered kernels per step, no host round trip:
//   1. sumsq_kernel   : reads every gradient once (2 B/param for fp16), forms
//                       the f64 sum of squares of the unscaled gradients along
//                       the canonical pairwise tree and the inf/NaN flag, one
//                       partial per block of SPB segments.  Its first block is
//                       the finalizer: it takes the partials as they appear,
//                       finishes the tree, runs the AMP skip / growth state
//                       machine, the clip decision and the bias corrections,
//                       and writes the step scalars.
//   2. adamw_kernel   : the fused streaming update (22 B/param): unscale, clip
//                       coefficient, AdamW with decoupled weight decay, fp16
//                      coefficient, AdamW with decoupled weight decay, fp16
//                      weight requantisation; exits at once on a skipped step.
//                      Its first waves clear the slots the partials went through.
//
// Every tensor is cut into ARK_OPT_NORM_SEGMENT-element segments, listed in
// table order, each with a 48-byte descriptor holding its four pointers
// already offset to the segment start, so a block finds its data with one
// scalar load and no dependent lookups.
//
// sumsq_kernel: a 256-lane block covers a segment as two halves of 256 x 8
// elements, lane l owning elements [h*2048 + 8l, h*2048 + 8l + 8) of half h
// (one 16-byte load per half).  That layout is what the canonical tree needs:
// lane groups of 8 in index order.
// adamw_kernel: one wave per 256-element row, lane l owning elements
// [4l, 4l + 4): every load and store instruction of every array covers one
// contiguous span (512 B of fp16, 1 KiB of fp32).  Blocks of four waves on
// rows kAdamStride apart measured fastest on MI355X for this mix of four read
// streams and three write streams (adamw_kernel).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "ark_opt.h"

namespace ark {

constexpr int kSeg = ARK_OPT_NORM_SEGMENT;  // elements per segment
constexpr int kBlock = 256;                 // lanes per sumsq block (4 waves)
constexpr int kVec = 8;                     // sumsq elements per lane group
constexpr int kHalfSeg = kBlock * kVec;     // 2048
static_assert(kSeg == 2 * kHalfSeg, "segment = two halves of 256 x 8");
constexpr int kRow = 256;                   // adamw elements per wave
constexpr int kRowsPerSeg = kSeg / kRow;    // 16
constexpr uint32_t kAdamWaves = 4;          // adamw waves per block, one row each
constexpr uint32_t kAdamStride = 32;        // rows between a block's waves
constexpr uint32_t kAdamGroup = kAdamWaves * kAdamStride;  // rows of kAdamStride blocks

// Segment descriptor flags.
constexpr uint32_t kSegNoUnscale = 1u;  // ARK_OPT_TENSOR_NO_UNSCALE
constexpr uint32_t kSegVec = 2u;        // w, g, m, v all 16-byte aligned

struct SegDesc {
  uint16_t* w;      // pointers to the segment's first element
  const void* g;
  float* m;
  float* v;
  uint32_t n;       // valid elements in this segment, 1..kSeg
  float wd;         // weight decay of the tensor
  uint32_t flags;   // kSeg*
  uint32_t tensor;  // index in the caller's table
};
static_assert(sizeof(SegDesc) == 48, "48-byte descriptor");

// Scalars of one step, written by the norm pass's finalizer, read by adamw_kernel.
struct StepScalars {
  uint32_t applied;
  uint32_t clipped;
  float inv;     // 1 / loss_scale
  float coef;    // clip coefficient (1 when not clipped)
  float lr;
  float lr_eff;  // sqrtf(bc2) / bc1 * lr
  float c1;      // 1 - beta1
  float c2;      // 1 - beta2
};

// The norm pass's slots, one per partial, lie behind the scalars in memory.
constexpr size_t kSlotsOffset = 256;
inline double* slots_of(StepScalars* scal) {
  return reinterpret_cast<double*>(reinterpret_cast<char*>(scal) + kSlotsOffset);
}

// beta^t by binary exponentiation, then lr_eff = (sqrt(bc2) / bc1) * lr, one
// IEEE binary32 operation per step as in opti.s:223-258.  Compiled for host
// and device; both round every operation to nearest even.
__host__ __device__ inline float pow_binary(float beta, uint32_t t) {
  float res = 1.0f;
  float base = beta;
  while (t != 0u) {
    if (t & 1u) res = res * base;
    base = base * base;
    t >>= 1;
  }
  return res;
}

__host__ __device__ inline float lr_eff_of(float lr, float beta1, float beta2,
                                           uint32_t t) {
  if (t == 0u) t = 1u;  // opti.s:211-212
  const float bc1 = 1.0f - pow_binary(beta1, t);
  const float bc2 = 1.0f - pow_binary(beta2, t);
  float r = sqrtf(bc2);
  r = r / bc1;
  return r * lr;
}

// Segments per norm block: 2 for fp16 gradients, 8 for fp32 (4 or 8 past
// kMaxParts partials); halved while fewer than 2048 blocks would cover the
// table.
int sumsq_spb(uint64_t nseg, uint32_t grad_dtype);
// Group sums the norm pass's finalizer holds, and the most partials it takes
// (64 lanes of 8 per group).
constexpr uint32_t kFinGroups = 1024;
constexpr uint32_t kMaxParts = kFinGroups * 64u * 8u;

// How often a finalizer wave looks for the partials of one group (1024 at
// most) before it gives the step up: each look is a round trip past the L2s and
// a sleep, 0.7 us or more together on MI355X, so the wait lasts over ten seconds.
// The norm pass of 1.2B parameters takes at most 13 looks at a group; what the
// bound leaves room for is other work on the GPU that holds the pass back.
constexpr uint32_t kFinMaxPolls = 1u << 24;

// What the finalizer needs (block 0 of the norm pass).  part: the slots, every
// byte 0xFF before the first step; a step's AdamW pass leaves them so.
struct FinalizeArgs {
  double* part;
  uint32_t nparts;
  uint32_t max_polls;  // kFinMaxPolls
  float lr;
  const float* lr_ptr;  // NULL, or a device scalar this step's lr is read from
  ark_opt_state* state;
  StepScalars* scal;
  ark_opt_step_info* host_info;  // NULL, or pinned host memory that gets the step's info
  ark_opt_hparams hp;
};

// The clip's partials (launch_grad_clip): up to kFinTarget are taken as they
// are, more are first folded in aligned groups of kFoldGroup.
constexpr uint32_t kFinTarget = 8192u;
constexpr uint32_t kFoldGroup = 64u;
// adamw: one wave per row, 16 rows per segment; rows and work-items must stay
// below 2^32 work-items.
constexpr uint64_t kMaxSegments = (1ull << 32) / (64ull * kRowsPerSeg) - 1;
// An AdamW pass launches whole groups of rows: first one row for every 64 slots
// of the norm pass, which it puts back to unset (kUnset), then the table's,
// whose descriptors are padded with empty ones.
inline uint32_t slot_rows(uint32_t nparts) {
  return ((nparts + 63u) / 64u + kAdamGroup - 1u) / kAdamGroup * kAdamGroup;
}
inline uint32_t norm_slots(uint32_t nparts) { return slot_rows(nparts) * 64u; }
// Most rows of one launch, whose work-items stay below 2^32: the largest tables
// take two.
constexpr uint32_t kAdamMaxRows = (1u << 26) - kAdamGroup;
static_assert(kAdamGroup % kRowsPerSeg == 0, "a group covers whole segments");
inline uint32_t padded_segs(uint32_t nseg) {
  constexpr uint32_t kSegs = kAdamGroup / kRowsPerSeg;
  return (nseg + kSegs - 1u) / kSegs * kSegs;
}
static_assert((kMaxSegments + 7) / 8 <= kMaxParts, "8 segments per norm block cover every table");

// ---------------------------------------------------------------------------
// Launch helpers (ark_opt_kernels.hip); each returns hipSuccess or the error.
// ---------------------------------------------------------------------------

// The norm pass, fin.nparts blocks of spb segments and the finalizer: the step's
// scalars, state and info.  A batch of segments whose segments all exist, hold
// kSeg elements and carry kSegVec takes 16-byte loads.  Blocks b >= nt_from read
// with non-temporal loads (see sumsq_nt_from).  lds_bytes of dynamic LDS per
// block (unused by the kernel) bound how many blocks a CU holds at once
// (sumsq_lds_for).
hipError_t launch_sumsq(uint32_t grad_dtype, int spb, const SegDesc* segs, uint32_t nseg,
                        uint32_t nt_from, const FinalizeArgs& fin, uint32_t lds_bytes,
                        hipStream_t stream);

// Resident norm blocks per CU for fp16 gradients.  Their fast path (squares
// straight from the fp16 bits under a power-of-two loss scale) has so little
// arithmetic per byte that 8 blocks per CU, the wave-slot limit, issue loads
// faster than HBM returns them: on MI355X the pass over EKO-237M's 474 MB
// takes 79.0-79.5 us at 8 blocks per CU, 77.2-77.5 at 7 and 78.9-79.1 at 6,
// and over the 1.3B set's 2.56 GB 372.6 us at 7 against 379.1 at 8.  0 = no
// cap (fp32 gradients).
constexpr int kSumsqBlocksPerCuF16 = 7;
// The dynamic LDS that holds the norm kernel for (grad_dtype, spb) at
// `blocks` per CU (resident_lds_bytes; 0 = no cap).
uint32_t sumsq_lds_for(uint32_t grad_dtype, int spb, int blocks);
// Resident AdamW waves per CU for a table of nseg segments, held by a
// dynamic-LDS reservation: more waves hide the latency of what the norm pass
// left in the Infinity Cache and of a skipped step's one load, but over-issue
// the seven streams that come from HBM, so the fewer the larger the uncached
// share; a step from units finds nothing cached.  Measured on MI355X over
// models' tables, step in us (two to five tables in turn, 9 rounds in a random
// order, whose 10th and 90th percentiles lie within 0.4 % of the median; a
// skipped step behind the bar):
//   waves                     12       16       20       24   |  12   16   20   24
//   fp16 gradients     7M     33.74    33.08    33.36    32.62
//                      21M    85.0     83.2     82.8     81.6
//                      39M   147.5    141.6    141.4    141.0 |  35   32   30   29
//                      60M   223.9    215.3    214.9    215.2 |  49   45   42   40
//                      82M   303.1    291.1    291.8    289.6 |  68   62   58   56
//                      110M  395.1    378.1    379.2    378.4 |  85   77   72   69
//                      159M  579.3    570.1    576.7    579.7 | 120  109  101   97
//                      237M  862.6    840.5    843.5    846.3 | 173  156  144  138
//                      334M 1232.0   1219.5   1240.8   1249.5 | 245  219  202  194
//   fp32 gradients     7M     37.00    36.34    35.64    35.78
//                      21M    96.6     94.0     92.3     91.8
//                      39M   171.6    166.0    164.1    162.7
//                      82M   355.3    347.7    345.6    343.8
//                      110M  468.5    460.4    458.1    458.2
//                      159M  692.4    694.5    697.7    697.4
//                      180M  782.7    776.5    778.1    783.3
//                      237M 1015.9   1013.5   1009.3   1009.8
//                      273M 1192.5   1204.0   1209.6   1213.8
//                      334M 1464.4   1478.1   1488.0   1491.1
//   from units         10M    64.65    64.73    64.25    64.37  (with the
//                      45M   253.2    253.5    253.9    254.6   accumulation)
//                      237M 1280.9   1291.5   1300.4   1303.3
inline int adamw_waves(uint64_t nseg, uint32_t grad_dtype, bool from_units) {
  if (from_units) return 12;
  if (nseg <= (1u << 15)) return 24;  // 134M parameters
  if (grad_dtype == ARK_OPT_GRAD_F16) return 16;
  return nseg <= (1u << 16) ? 20 : 12;  // 268M
}
// The dynamic LDS that holds the AdamW kernel for grad_dtype at `waves` per
// CU, rounded up to whole blocks (resident_lds_bytes; 0 = no cap).
uint32_t adamw_lds_for(uint32_t grad_dtype, int waves);

// The norm pass leaves the last kNormCachedBytes it reads (its lowest
// blocks, where the AdamW pass starts) in the Infinity Cache and streams the
// rest past it.  Measured on MI355X over 128-320 MiB and all-streaming:
// 256 MiB (the cache's size) is fastest, the step 0.5 % faster at EKO-237M
// and 0.9 % at 1.3B than with every load cache-allocating.
constexpr uint64_t kNormCachedBytes = 256ull << 20;
inline uint32_t sumsq_nt_from(int spb, uint64_t grad_bytes) {
  const uint64_t per_block = (uint64_t)spb * kSeg * grad_bytes;
  const uint64_t b = kNormCachedBytes / per_block;
  return b > 0xFFFFFFFFull ? 0xFFFFFFFFu : (uint32_t)b;
}

// lds_bytes: dynamic LDS per block, the residency cap (adamw_lds_for).
// max_rows: rows per launch, a multiple of kAdamGroup.
hipError_t launch_adamw(uint32_t grad_dtype, const SegDesc* segs,
                        uint32_t nseg, uint32_t nparts, StepScalars* scal, float beta1,
                        float beta2, float eps, uint32_t lds_bytes, uint32_t max_rows,
                        hipStream_t stream);

// One tensor given by value (fp32 gradients used as given, no unscale or
// clip) with host-computed scalars: the drop-in of one
// ark_asm_adam_step_f16 call.  n may exceed one segment.
hipError_t launch_adamw_single(uint16_t* w, const float* g, float* m, float* v,
                               uint64_t n, float wd, bool vec,
                               const StepScalars& sc, float beta1, float beta2,
                               float eps, hipStream_t stream);

// The same for an fp32-weight tensor: the drop-in of one ark_asm_adam_step
// call (opti.s:20-177).
hipError_t launch_adamw_single_w32(float* w, const float* g, float* m, float* v, uint64_t n,
                                   float wd, bool vec, const StepScalars& sc, float beta1,
                                   float beta2, float eps, hipStream_t stream);

// The single-tensor clip (ark_asm_grad_clip, opti.s:369-432): the
// canonical tree's sum of squares of one fp32 array (one partial per block of
// two segments, folded past kFinTarget partials), then the norm, the clip
// decision and the in-place scaling.
//
// Elements one call takes: the partials stay within what one fold leaves
// kFinTarget of (2^19 blocks of 2 segments).
constexpr uint64_t kClipMaxElements = (uint64_t)kFinTarget * kFoldGroup * 2u * kSeg;
inline uint32_t clip_parts(uint64_t n) { return (uint32_t)((n + 2u * kSeg - 1) / (2u * kSeg)); }
// Most blocks of the scaling launch, each of which forms the decision: eight a
// CU, as many as are resident at once up to 4096 leaves (past them a block's 71
// registers leave seven).
constexpr uint64_t kClipBlocks = 2048;
// parts: clip_parts(n) doubles; folded: ceil(clip_parts(n) / kFoldGroup)
// doubles (used past kFinTarget partials); norm: device-visible, gets the
// pre-clip norm.  n >= 1.
hipError_t launch_grad_clip(float* g, uint64_t n, float threshold, double* parts,
                            double* folded, float* norm, hipStream_t stream);

hipError_t launch_record_overflow(const ark_opt_hparams& hp,
                                  ark_opt_state* state,
                                  ark_opt_step_info* host_info, hipStream_t stream);

}  // namespace ark
