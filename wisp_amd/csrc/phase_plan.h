// The order in which a paged call of several token groups moves and uses its
// experts (host only).
//
// The pager decides such a call group by group, as the reference does: a
// group's experts are made resident, least recently used ones leave, and an
// expert that a later group needs again is loaded again.  Those decisions
// fix what the call leaves behind (slots, ticks, counters, record).  They do
// not fix the copies: an expert's product with all the tokens routed to it
// in the whole call can be taken while it is in HBM once.  The plan works
// through the call's experts instead of its groups:
//   phase 0    the experts resident at the start (those evicted later from
//              their old slot), no copies;
//   middle     the experts that are gone at the end, as many at a time as
//              there are slots that the call fills anew;
//   last       the experts that the call leaves in those slots.
// Each expert's weights cross the host link once; by groups, a chunk of 96
// tokens at 24 of 128 slots loads 6 times as many (79 ms, against 17 ms).
// Nothing here allocates: the plan is made inside C entry points.
#pragma once

#include <stdint.h>

#include "common.h"
#include "pager_core.h"

namespace wisp {

struct PhaseLoad {
  int16_t expert, slot;
  bool use;  // its tokens' products are taken in this phase
};

struct PhasePlan {
  PhaseTable first;  // phase 0
  // where phase 0 finds each expert: its slot before the call, kDecided for
  // the slot that the pager decided, kNone where a later phase has it
  int16_t place[kMaxExperts];
  // the copies of phase i + 1: load[start[i]] to load[start[i + 1]]
  int nphases = 0;
  int start[kMaxExperts + 2];
  PhaseLoad load[kMaxExperts];
  int loads = 0;     // copies of the plan
  int recorded = 0;  // copies of the decision record
};

// The plan of a decision record whose groups are all decided; false when a
// word of the record is out of range (E and cap are at most kMaxExperts).
inline bool plan_phases(const int32_t* rec, int T, int K, int E, int cap, PhasePlan* p) {
  const RecordLayout RL(T, K);
  int16_t home[kMaxExperts], fin[kMaxExperts];
  bool loaded[kMaxExperts], touched[kMaxExperts], last[kMaxExperts];
  for (int i = 0; i < kMaxExperts; ++i) {
    home[i] = fin[i] = -1;
    loaded[i] = touched[i] = last[i] = false;
  }
  p->nphases = p->loads = p->recorded = 0;
  // n pairs from pair `off` of a list that starts at word `base`
  auto each = [&](int base, int off, int n, auto&& f) {
    if (off < 0 || n < 0 || off > RL.max_pairs || n > RL.max_pairs - off) return false;
    for (const int32_t *w = rec + base + 2 * off, *end = w + 2 * n; w < end; w += 2) {
      if (w[0] < 0 || w[0] >= E || w[1] < 0 || w[1] >= cap) return false;
      f(w[0], w[1]);
    }
    return true;
  };
  if (rec[kRecGroupsDone] < 0 || rec[kRecGroupsDone] > RL.max_groups) return false;
  for (int g = 0; g < rec[kRecGroupsDone]; ++g) {
    const int32_t* G = rec + RL.group_base(g);
    if (!each(RL.evicted_base(), G[4], G[5],
              [&](int e, int s) {
                if (!loaded[e] && home[e] < 0) home[e] = s;  // there since before the call
                touched[s] = true;
                fin[s] = -1;
              }) ||
        !each(RL.loaded_base(), G[6], G[7], [&](int e, int s) {
          loaded[e] = touched[s] = true;
          fin[s] = e;
          ++p->recorded;
        }))
      return false;
  }
  for (int s = 0; s < kMaxExperts; ++s)
    p->first.expert[s] = s < cap && !touched[s] ? PhaseTable::kDecided : PhaseTable::kNone;
  for (int e = 0; e < E; ++e) {
    if (home[e] >= 0) p->first.expert[home[e]] = (int16_t)e;
    p->place[e] = home[e] >= 0 ? home[e] : loaded[e] ? PhaseTable::kNone : PhaseTable::kDecided;
  }
  // Slots whose old expert is also their last keep it throughout, unless no
  // other slot is there for the experts that come and go.
  auto kept = [&](int s) { return fin[s] >= 0 && home[fin[s]] == s; };
  int nroom = 0, npassing = 0;
  int16_t room[kMaxExperts], passing[kMaxExperts];
  for (int s = 0; s < cap; ++s) {
    if (!touched[s] || kept(s)) continue;
    room[nroom++] = (int16_t)s;
    if (fin[s] >= 0) last[fin[s]] = true;
  }
  for (int e = 0; e < E; ++e)
    if (loaded[e] && home[e] < 0 && !last[e]) passing[npassing++] = (int16_t)e;
  const bool reuse = nroom == 0 && npassing > 0;
  if (reuse)
    for (int s = 0; s < cap; ++s)
      if (touched[s]) room[nroom++] = (int16_t)s;
  auto add = [&](int16_t e, int16_t s, bool use) {
    if (p->loads == kMaxExperts) return false;
    p->load[p->loads++] = {e, s, use};
    return true;
  };
  for (int i = 0; i < npassing; ++i) {
    if (i % nroom == 0) p->start[p->nphases++] = p->loads;
    if (!add(passing[i], room[i % nroom], true)) return false;
  }
  p->start[p->nphases++] = p->loads;
  for (int i = 0; i < nroom; ++i) {
    const int16_t s = room[i], e = fin[s];
    if (e >= 0 && !add(e, s, !reuse && home[e] < 0)) return false;
  }
  p->start[p->nphases] = p->loads;
  return true;
}

}  // namespace wisp
