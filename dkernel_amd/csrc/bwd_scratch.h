// Scratch of a backward call and what it is used for: partial dK / dV per q head (several q heads per kv
// head), then the partial sums of rows and columns that are cut into segments (SegView).
#pragma once

#include <algorithm>

#include "device_common.h"

namespace dk {


enum class SegRows { kKeys, kQueries, kQueryPairs };  // what the rows of a launch's segments are

struct BwdScratch {
  size_t group = 0;  // bytes of the per-q-head partials of dK / dV, 0: the pass works per kv head
  SegView dq, kv;    // the two passes run one after the other and use the same bytes behind them
  size_t bytes = 0;  // all of it
};

// Several q heads per kv head: whether a workgroup of the dK/dV pass walks a column for all of them, long columns cut into
// segments, instead of one workgroup per q head into fp32 partials that are summed.  The walk saves those partials (twice
// their bytes of traffic), but its pieces are longer by the group's size: below some hundred steps per resident workgroup
// it needs so many segments to even them out that their sums cost as much.  Per q head / walk, us, training, 32 / 8 heads of
// 128: 4000 tokens (68 steps) 394 / 418, 2 x 3000 of 96 dims (92) 474 / 496, 9000 of 16 / 4 heads (101) 600 / 619, 4 x 2048
// (110) 661 / 610, 3 x 3000 (138) 808 / 742, 8000 (171) 937 / 872, 10000 (236) 1261 / 1186, 10000, local 8, vertical 16 (128)
// 773 / 684; blocks of 32, 3 x 3000 (110) 675 / 614; 24 / 8 heads of 64, 6 x 2000 (85) 444 / 416.
constexpr double kWalkFrom = 105;

// What cutting the columns of a 16-bit call with one head a workgroup must gain, in steps: the kernel that adds the sums takes 5 us and
// more, and the longest column, once it is left alone on its compute unit, runs faster than the average one.  Fit over 70 training
// calls of 64 - 256 dims (backward, us of 128 dims): 1.1 a step, - 0.022 a partial sum, - 2.  Below the line, not cut / cut: 16
// heads, 2 x 1831 121 / 129, 8 heads of 256 dims, 2 x 1826 165 / 178, 32 heads, 1 x 1377 85 / 90, 8 heads, 2 x 1464 80 / 84; just above it 16
// / 4 heads, 3 x 1358 106 / 93, 12 heads, 2 x 2057 127 / 136, 16 heads of 64, 3 x 2006 106 / 93.  Not for global columns, which stand
// out of short ones (8 heads, 4 x 2553, longest column 1.04 times the average: 206 / 184), nor for masked tiles, whose average is overestimated.
constexpr double kLeastGain = 3.5;
inline bool walk_groups(const BwdParams &p, size_t group, int kv_slots, double from) {
  const int ratio = p.Hq / p.Hkv;
  const bool one_table = p.csc.num_heads != p.Hq || p.csc.group % ratio == 0;  // for all q heads of a kv head
  if (ratio == 1 || !one_table || !p.csc.row_lengths || !kv_slots) return false;
  return group == 0 || average_steps(p.csc.row_lengths, p.csc.num_rows, 1, (int64_t)p.seqs.batch * p.Hkv, kv_slots, ratio) >= from;
}

// group: bytes of the per-q-head partials if the pass uses them; dq_slots, kv_slots: workgroups of the two passes that the
// chip holds at once (0: its rows are not cut); dq_pairs: the dQ pass takes pairs of rows; walk_from: steps per resident
// workgroup from which on the dK/dV pass walks whole groups although it could use partials (< 0: it does not walk them);
// kv_gain: steps that cutting columns of one head must gain (plan_segments), where they fall off gradually.
inline BwdScratch plan_bwd_scratch(const BwdParams &p, size_t group, int dq_slots, bool dq_pairs, int kv_slots, double walk_from,
                                   double kv_gain) {
  constexpr size_t kMost = (size_t)4 << 30;
  const bool walk = walk_from >= 0 && walk_groups(p, group, kv_slots, walk_from);
  BwdScratch s;
  s.group = s.bytes = !walk && group <= kMost ? group : 0;
  const int64_t copies = (int64_t)p.seqs.batch * p.Hq;
  // limit: longest row : average per slot from which on rows are cut; share: segment : average.  Both lower with masked
  // tiles, whose average is overestimated (long rows are mostly whole tiles, short ones mostly parts of them): 12 heads
  // of 64, 4 x 3000 tokens, global blocks of 32, training, us: not cut 310, limit 0.8 and share 0.4 251, 0.6 275, limit 1
  // 277.  Other tables, share 0.4 / 0.6 / 0.8: 16 heads x 4000 tokens 212 / 207 / 207 (not cut 232), 8 x 9000 322 / 316 /
  // 316 (426), 12 x 6000, vertical 4 235 / 228 / 239 (291).  dK / dV by q heads: a higher limit, as the sums pass
  // through memory once more (not cut / cut: 24 / 8 heads x 3000 tokens, ratio 1.2, 227 / 235; 16 / 4 heads of 256
  // dims, 0.9, 386 / 395; 16 / 4 x 5000, 1.5, 331 / 309).
  const double limit = p.csr.sub_block ? 0.8 : 1.0, kv_limit = s.group ? 1.3 : limit, share = p.csr.sub_block ? 0.4 : 0.6;
  SegView dq, kv;
  if (dq_slots)
    dq = dq_pairs ? plan_segments(p.csr.pair_lengths, (p.csr.num_rows + 1) / 2, 2, copies, dq_slots, limit, share)
                  : plan_segments(p.csr.row_lengths, p.csr.num_rows, 1, copies, dq_slots, limit, share);
  // (walks: columns of one length that is a good part of the average are the rule, so they are cut finer: 3 x 4000 tokens, 24
  // / 8 heads, share 0.6 / 0.5 / 0.4 884 / 854 / 822, 4 x 2048, 32 / 8 625 / - / 610)
  if (walk)
    kv = plan_segments(p.csc.row_lengths, p.csc.num_rows, 1, (int64_t)p.seqs.batch * p.Hkv, kv_slots, limit, 0.4, p.Hq / p.Hkv);
  else if (kv_slots && (p.Hq == p.Hkv || s.group))
    kv = plan_segments(p.csc.row_lengths, p.csc.num_rows, 1, copies, kv_slots, kv_limit, share, 1,
                       p.csr.order || p.csr.sub_block ? -1 : kv_gain);
  const size_t at = (s.group + 255) / 256 * 256;
  const int64_t dq_slots_all = dq.slots * copies, kv_slots_all = kv.slots * (walk ? copies / (p.Hq / p.Hkv) : copies);
  const double partials = (double)std::max(dq_slots_all, kv_slots_all) * 128 * p.D * sizeof(float);  // (no number of slots overflows)
  const size_t need = partials > (double)kMost ? kMost + 1 : at + (size_t)partials;
  if (walk && need > kMost && group) return plan_bwd_scratch(p, group, dq_slots, dq_pairs, kv_slots, -1, kv_gain);
  if (need > at && need <= kMost && p.D % 4 == 0) s.dq = dq, s.kv = kv, s.bytes = need;
  return s;
}

// The scratch as the caller's workspace allows it: all of it, the per-q-head partials only, or none.  plan(walk) plans it,
// with or without walks of whole groups.
template <typename Plan>
inline BwdScratch usable_bwd_scratch(Plan plan, void *workspace, size_t bytes) {
  BwdScratch s = plan(true);
  if (bytes < s.bytes) s = plan(false);
  const bool ok = workspace && ((uintptr_t)workspace % 16) == 0;
  if (!ok || bytes < s.group) return BwdScratch{};
  if (bytes < s.bytes) s.dq = s.kv = SegView{}, s.bytes = s.group;
  float *partial = (float *)((char *)workspace + (s.group + 255) / 256 * 256);
  s.dq.partial = s.kv.partial = partial;
  return s;
}

// Work items of a launch along grid.y: `rows` and the segments beyond the first of each cut one.
inline int64_t segment_items(const SegView &s, int rows) {
  int64_t items = rows;
  for (int i = 1; i < kMaxSegments; ++i) items += s.n[i];
  return items;
}

}  // namespace dk
