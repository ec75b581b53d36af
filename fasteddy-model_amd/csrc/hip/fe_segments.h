/*
 * fe_segments.h -- z segments of the stage launches: shapes, and an ensemble's common length.
 */
#ifndef FE_SEGMENTS_H
#define FE_SEGMENTS_H

#include <algorithm>
#include <functional>
#include <map>
#include <vector>

namespace {

/* Even segment length for n segments of Nz levels, and the segment count it gives. */
inline void seg_shape(int Nz, int n, int &len, int &nseg) {
  len = (Nz + n - 1) / n;
  len += len & 1;
  nseg = (Nz + len - 1) / len;
}

/* Levels' worth of a work item: its levels and about two for loading its window and filling the
 * pipeline. */
inline int ens_item_cost(int levels) { return levels + 2; }

/* A member's tiles and levels, and its segment length where one is set (0: none). */
struct SegMember {
  long tiles;
  int Nz, zseg;
};

/* Segment length of the members that have none set: of all even lengths >= 4, the one whose
 * work items end earliest when the work-groups of the persistent grid (slots) take them longest first
 * (longest length on ties).  A lone run's own choice spreads one member over the whole chip; here
 * the members fill it together, and segments as short as a lone 64 x 64 x 48 member's (4 levels)
 * spend a third of their items on set-up.  Measured in ms a step, lone-run choice -> this one: 16 of
 * 64 x 64 x 48 0.399 (12 segments) -> 0.335 (2); 40 of them 0.928 -> 0.765 (4); eight of 96^2 x 64 to
 * 192^2 x 96 within 1% of the best length of 8, 12, 16, 24, 32, 48, 64 levels, 48 of them within 3%. */
inline int ens_segment_length(const std::vector<SegMember> &mem, int slots) {
  int mz = 0;
  for (auto &m : mem)
    if (m.zseg <= 0) mz = std::max(mz, m.Nz);
  long best = -1;
  int blen = 0;
  for (int len = 4; len == 4 || len < mz + 2; len += 2) {   /* members lower than 4 levels: one segment each */
    std::map<int, long, std::greater<int>> items;      /* item cost -> items */
    for (auto &m : mem) {
      int zseg = m.zseg, nseg;
      if (zseg <= 0) seg_shape(m.Nz, (m.Nz + len - 1) / len, zseg, nseg);
      nseg = (m.Nz + zseg - 1) / zseg;
      items[ens_item_cost(std::min(zseg, m.Nz))] += m.tiles * (nseg - 1);
      items[ens_item_cost(m.Nz - (nseg - 1) * zseg)] += m.tiles;
    }
    std::map<long, long> load{{0, slots}};              /* work taken -> work-groups */
    for (auto &it : items)
      for (long left = it.second; left > 0;) {
        const auto lo = load.begin();
        const long at = lo->first, n = std::min(left, lo->second);
        if ((lo->second -= n) == 0) load.erase(lo);
        load[at + it.first] += n;
        left -= n;
      }
    const long end = load.rbegin()->first;
    if (best < 0 || end <= best) { best = end; blen = len; }
  }
  return blen;
}

}  // namespace

#endif
