// Time estimates of the prefill planner, in plain C++ (no HIP header), so that
// the choices they lead to can be checked on the host.
//
// A batch at one candidate segment length, sums over its sequences of at least
// two chunks ("long"):
#pragma once

#ifdef __HIP__
#define GDN_HD __host__ __device__ inline
#else
#define GDN_HD inline
#endif

namespace gdn {

struct PlanStats {
  float chunks;      // chunks of the long sequences
  float first;       // chunks of their first segments
  float segments;    // segments
  float longs;       // long sequences
  float shorts;      // sequences of at most one chunk
  float mfrac;       // share of a segment an M-run forms before its map is negligible (mean over the v-heads)
  int longest;       // chunks of the longest sequence
  int L;             // segment length in chunks
  int nseg;          // segments of the longest sequence
  float warmup;      // warm-up chunks of a later segment's run (warm-up scheme)
  bool many;         // more than 32 sequences: the wide consumer is weighed too
};

GDN_HD float plan_max(float a, float b) { return a > b ? a : b; }
GDN_HD float plan_min(float a, float b) { return a < b ? a : b; }

// Batches of single-chunk sequences alone, on either consumer.  The full-head
// consumer takes 32 at a time and so runs in rounds; the wide one fills the CUs'
// second groups from 33 on and then claims items one by one.  us per call, split
// / wide: 33 sequences of 40 tokens 29.9 / 25.7, 64 31.3 / 29.7, 65 39.7 / 35.7,
// 94 40.4 / 44.2, 100 48.9 / 44.7, 128 49.0 / 50.1, 129 58.9 / 52.3, 256 94.7 /
// 80.5, 500 167 / 139.
GDN_HD float plan_shorts_split_us(float n) { return 9.5f * static_cast<float>((static_cast<int>(n) + 31) / 32); }
GDN_HD float plan_shorts_wide_us(float n) { return n <= 64.0f ? 9.8f + 0.137f * n : 9.0f + 0.237f * n; }

// Single-chunk sequences beside runs on the split consumer, in batches of more
// than 32 sequences: their groups start where a CU is free, so with few runs
// (fewer than the 16 machines) the groups that found none start a round later.
// Runs of two chunks or more take at least ceil(runs / 16) rounds of two: 16 runs
// of two and three chunks among 32 to 47 sequences 37 to 40 us per call, 17 to 30
// of them 44 to 45, which the balanced load alone puts at 39 (wide consumer 39).
GDN_HD float plan_rounds(float runs) { return static_cast<float>((static_cast<int>(runs) + 15) / 16); }
GDN_HD float plan_beside_runs_us(float shorts_us, float runs, float run_us, float balanced_us, float late) {
  const float again = plan_min(late * shorts_us, run_us);
  return shorts_us + (runs >= 16.0f ? balanced_us : plan_max(balanced_us, again));
}

// Split consumer, M-run scheme, in us without the parts that do not depend on
// the segment length or the consumer.  A run's 16 items are taken together by 16 of 256 groups,
// so the runs are scheduled on 16 machines: the longest run, or the balanced
// load plus a fifth of an average run for the last round.  Single-chunk
// sequences share the CUs (one group of eight v-heads each, 32 at a time).
// Having segments costs the finish, every segment of the longest sequence
// after its second a step of the scan (a group reads 80 KB of maps and states
// per step), every chunk of an M-run its corrections.
//
// Fitted to 348 batches timed at every segment length (1 to 191 sequences of 13
// to 512 chunks, uniform and with one to 16 long ones among short ones, mixed
// and near-1 gates): the length chosen is 0.5% slower than the best on average,
// 9.5% at worst.  The estimate before, which priced a scan step at 0.75 us,
// cut 1 x 2000 tokens into 8 segments: 61.9 us per call, now 52.7 with 4
// (unsegmented 82.3); one of 1,900 among 31 single tokens 68.0 -> 61.6;
// 2 x 1000 52.5 -> 46.5; 4 x 1000 56.5 -> 52.0.
GDN_HD float plan_split_mrun_us(const PlanStats& b) {
  constexpr float kStep = 1.84f, kItem = 2.8f, kTail = 0.2f, kMachines = 16.0f, kShort = 9.4f;
  constexpr float kFinish = 7.0f, kScanStep = 3.6f, kCorr = 0.13f;
  if (b.longs == 0.0f) return plan_shorts_split_us(b.shorts);
  const float runs = 2.0f * b.segments - b.longs;
  const float mwork = (b.chunks - b.first) * b.mfrac;
  const float work = b.chunks + mwork;
  const float longest = static_cast<float>(b.L < b.longest ? b.L : b.longest);
  const float run = work / runs + kItem;   // an average run
  const float tail = runs > kMachines ? kTail * run : 0.0f;
  float balanced = ((work + kItem * runs) / kMachines + tail) * kStep;
  if (b.many && runs > 16.0f) balanced = plan_max(balanced, plan_rounds(runs) * (2.0f + kItem) * kStep);
  if (!b.many)
    balanced += b.shorts * (kShort / 32.0f);
  else if (b.shorts > 0.0f)
    balanced = 3.3f + plan_beside_runs_us(b.shorts * (7.7f / 32.0f), runs, run * kStep, balanced, 0.6f);
  const float body = plan_max(b.longs > 0.0f ? (longest + kItem) * kStep : 0.0f, balanced);
  return body + (b.nseg > 1 ? kFinish + kScanStep * static_cast<float>(b.nseg - 2) + kCorr * mwork : 0.0f);
}

// Split consumer, warm-up scheme: one run per segment, each later segment's
// `warmup` chunks longer, scheduled as above; item overhead (descriptor, warm-up
// bounds, first copies, final stores) 1.5 chunk steps, a quarter of an average
// run for the last round, 0.75 steps for having segments (measured batches: 16
// sequences of 16,384 tokens in all L = 18, 2 x 8192 tokens 16, 4 x 16384 64).
GDN_HD float plan_split_warm_us(const PlanStats& b) {
  constexpr float kStep = 1.87f, kItem = 1.5f, kTail = 0.25f, kSegmented = 0.75f, kMachines = 16.0f;
  if (b.longs == 0.0f) return plan_shorts_split_us(b.shorts);
  const float work = b.chunks + b.warmup * (b.segments - b.longs);
  const float longest = static_cast<float>(b.longest > b.L ? b.L + b.warmup : b.longest);
  const float run = work / b.segments + kItem;   // an average run
  const float tail = b.segments > kMachines ? kTail * run : 0.0f;
  float balanced = ((work + kItem * b.segments) / kMachines + tail) * kStep;
  if (b.many && b.segments > 16.0f) balanced = plan_max(balanced, plan_rounds(b.segments) * (2.0f + kItem) * kStep);
  if (b.many && b.shorts > 0.0f)
    balanced = 8.2f + plan_beside_runs_us(b.shorts * (6.9f / 32.0f), b.segments, run * kStep, balanced, 0.48f);
  else if (b.many)
    balanced += 4.0f;
  return plan_max((longest + kItem) * kStep, balanced) + (b.longest > b.L ? kSegmented * kStep : 0.0f);
}

// Wide consumer.  A run's 8 items take 8 of 256 CUs, two halves to a CU: a chunk
// step takes kLone while the other half has no work or little (the longest
// run's end) and kStep of a CU's time when both are busy, so the longest run and
// the balanced load have steps of their own.
//
// Fitted together with the split consumer's estimate to 1,355 batches of 33 to
// 700 sequences timed on both consumers at every segment length (one to 16
// sequences of 150 to 16,000 tokens among short ones; uniform; log-uniform over
// a factor of 4 to 36): consumer and length chosen are 0.6% slower than the best
// on average under mixed and near-1 gates, 1.0% under fast ones,
// 19% at worst.  The rule before, by number of sequences and mean length, took
// the wide consumer for skewed batches under mixed and slow gates: one of 256
// tokens among 33 45.9 us (split 30.9), one of 4,000 among 64 92.4 (66.5), 66
// of 549 on average over a factor of 16 224 (166).
GDN_HD float plan_wide_mrun_us(const PlanStats& b) {
  constexpr float kLone = 4.43f, kStep = 2.78f, kItem = 1.64f, kTail = 0.46f, kMachines = 32.0f, kShort = 6.0f, kMix = 0.1f;
  constexpr float kFinish = 8.8f, kScanStep = 2.8f, kCorr = 0.146f;
  if (b.longs == 0.0f) return plan_shorts_wide_us(b.shorts);
  const float runs = 2.0f * b.segments - b.longs;
  const float mwork = (b.chunks - b.first) * b.mfrac;
  const float work = b.chunks + mwork;
  const float longest = static_cast<float>(b.L < b.longest ? b.L : b.longest);
  const float tail = runs > kMachines ? kTail * work / runs : 0.0f;
  const float balanced = ((work + kItem * runs) / kMachines + tail) * kStep + b.shorts * (kShort / 32.0f);
  const float lone = (longest + kItem) * kLone;
  return plan_max(lone, balanced) + kMix * plan_min(lone, balanced) +
         (b.nseg > 1 ? kFinish + kScanStep * static_cast<float>(b.nseg - 2) + kCorr * mwork : 0.0f);
}

GDN_HD float plan_wide_warm_us(const PlanStats& b) {
  constexpr float kLone = 3.66f, kStep = 2.05f, kItem = 2.4f, kTail = 0.76f, kMachines = 32.0f, kShort = 6.1f;
  if (b.longs == 0.0f) return plan_shorts_wide_us(b.shorts);
  const float work = b.chunks + b.warmup * (b.segments - b.longs);
  const float longest = static_cast<float>(b.longest > b.L ? b.L + b.warmup : b.longest);
  const float tail = b.segments > kMachines ? kTail * work / b.segments : 0.0f;
  const float balanced = ((work + kItem * b.segments) / kMachines + tail) * kStep + b.shorts * (kShort / 32.0f);
  return plan_max((longest + kItem) * kLone, balanced);
}

}  // namespace gdn
