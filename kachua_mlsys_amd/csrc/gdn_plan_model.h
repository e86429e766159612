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
};

GDN_HD float plan_max(float a, float b) { return a > b ? a : b; }

// Split consumer, M-run scheme, in us without the parts that do not depend on
// the segment length.  A run's 16 items are taken together by 16 of 256 groups,
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
  const float runs = 2.0f * b.segments - b.longs;
  const float mwork = (b.chunks - b.first) * b.mfrac;
  const float work = b.chunks + mwork;
  const float longest = static_cast<float>(b.L < b.longest ? b.L : b.longest);
  const int nseg = b.longest > 0 ? (b.longest - 1) / b.L + 1 : 0;
  const float tail = runs > kMachines ? kTail * (work / runs + kItem) : 0.0f;
  const float balanced = ((work + kItem * runs) / kMachines + tail) * kStep + b.shorts * (kShort / 32.0f);
  const float body = plan_max(b.longs > 0.0f ? (longest + kItem) * kStep : 0.0f, balanced);
  return body + (nseg > 1 ? kFinish + kScanStep * static_cast<float>(nseg - 2) + kCorr * mwork : 0.0f);
}

}  // namespace gdn
