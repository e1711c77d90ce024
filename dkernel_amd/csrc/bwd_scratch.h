// Scratch of a backward call and what it is used for: partial dK / dV per q head (several q heads per kv
// head), then the partial sums of rows and columns that are cut into segments (SegView).
#pragma once

#include <algorithm>

#include "device_common.h"

namespace dk {

enum class SegRows { kKeys, kQueries, kQueryPairs };  // what the rows of a launch's segments are

struct BwdScratch {
  size_t group = 0;  // bytes of the per-q-head partials, 0: the pass works per kv head
  SegView dq, kv;    // the two passes run one after the other and use the same bytes behind them
  size_t bytes = 0;  // all of it
};

// dq_slots, kv_slots: workgroups of the two passes that the chip holds at once (0: its rows are not cut);
// dq_pairs: the dQ pass takes pairs of rows.
inline BwdScratch plan_bwd_scratch(const BwdParams &p, size_t group, int dq_slots, bool dq_pairs, int kv_slots) {
  constexpr size_t kMost = (size_t)4 << 30;
  BwdScratch s;
  s.group = s.bytes = group <= kMost ? group : 0;
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
  // (columns only where a workgroup serves one q head)
  if (kv_slots && (p.Hq == p.Hkv || s.group)) kv = plan_segments(p.csc.row_lengths, p.csc.num_rows, 1, copies, kv_slots, kv_limit, share);
  const size_t at = (s.group + 255) / 256 * 256;
  const size_t need = at + (size_t)std::max(dq.slots, kv.slots) * copies * 128 * p.D * sizeof(float);
  if (need > at && need <= kMost && p.D % 4 == 0) s.dq = dq, s.kv = kv, s.bytes = need;
  return s;
}

// The scratch as the caller's workspace allows it: all of it, the per-q-head partials only, or none.
inline BwdScratch usable_bwd_scratch(BwdScratch s, void *workspace, size_t bytes) {
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
