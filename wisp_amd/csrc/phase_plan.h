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
// tokens at 24 of 128 slots loads 6 times as many (77 ms, against 17 ms).
#pragma once

#include <stdint.h>

#include <vector>

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
  std::vector<int16_t> place;
  std::vector<std::vector<PhaseLoad>> phases;
  int loads = 0;     // copies of the plan
  int recorded = 0;  // copies of the decision record
};

// The plan of a decision record whose groups are all decided.
inline PhasePlan plan_phases(const int32_t* rec, int T, int K, int E, int cap) {
  const RecordLayout RL(T, K);
  PhasePlan p;
  std::vector<int> home(E, -1), fin(cap, -1);
  std::vector<char> loaded(E, 0), touched(cap, 0), last(E, 0);
  for (int g = 0; g < rec[kRecGroupsDone]; ++g) {
    const int32_t* G = rec + RL.group_base(g);
    const int32_t* ev = rec + RL.evicted_base() + 2 * G[4];
    for (int i = 0; i < G[5]; ++i) {
      const int e = ev[2 * i], s = ev[2 * i + 1];
      if (!loaded[e] && home[e] < 0) home[e] = s;  // there since before the call
      touched[s] = 1;
      fin[s] = -1;
    }
    const int32_t* ld = rec + RL.loaded_base() + 2 * G[6];
    for (int i = 0; i < G[7]; ++i) {
      const int e = ld[2 * i], s = ld[2 * i + 1];
      loaded[e] = 1;
      touched[s] = 1;
      fin[s] = e;
      ++p.recorded;
    }
  }
  for (int s = 0; s < kMaxExperts; ++s)
    p.first.expert[s] = s < cap && !touched[s] ? PhaseTable::kDecided : PhaseTable::kNone;
  for (int e = 0; e < E; ++e) {
    if (home[e] >= 0) p.first.expert[home[e]] = (int16_t)e;
    p.place.push_back(home[e] >= 0 ? (int16_t)home[e]
                      : loaded[e]  ? PhaseTable::kNone
                                   : PhaseTable::kDecided);
  }
  // slots whose old expert is also their last keep it throughout, unless no
  // other slot is there for the experts that come and go
  std::vector<PhaseLoad> finals, kept;
  std::vector<int16_t> room;
  for (int s = 0; s < cap; ++s) {
    if (!touched[s]) continue;
    const int e = fin[s];
    if (e >= 0 && home[e] == s) {
      kept.push_back({(int16_t)e, (int16_t)s, false});
      continue;
    }
    room.push_back((int16_t)s);
    if (e >= 0) {
      finals.push_back({(int16_t)e, (int16_t)s, home[e] < 0});
      last[e] = 1;
    }
  }
  std::vector<int16_t> passing;
  for (int e = 0; e < E; ++e)
    if (loaded[e] && home[e] < 0 && !last[e]) passing.push_back((int16_t)e);
  if (room.empty() && !passing.empty()) {
    for (const PhaseLoad& k : kept) room.push_back(k.slot);
    finals = kept;
  }
  for (size_t i = 0; i < passing.size(); i += room.size()) {
    std::vector<PhaseLoad> ph;
    for (size_t j = 0; j < room.size() && i + j < passing.size(); ++j)
      ph.push_back({passing[i + j], room[j], true});
    p.phases.push_back(ph);
  }
  p.phases.push_back(finals);
  p.loads = (int)(passing.size() + finals.size());
  return p;
}

}  // namespace wisp
