// Planner of the multi-layer passes (qg_sweep.hpp): which window of bits each
// pass holds and which rotations and bonds it runs there.  Host only; a
// function of the circuit's shape, never of its angles.
#pragma once
#include <algorithm>
#include <array>
#include <cstdint>
#include <list>
#include <mutex>
#include <utility>
#include <vector>

#include "qg_internal.h"

namespace qg {

// One round of a pass: a rotation per register bit (bit -1: none).  The bonds
// in b1 and b2 (bond k couples global bits k and k + 1; b1 the group that acts
// first in a layer) run before it.
struct PlanRound {
  int lo;
  int bit[4], layer[4];
  uint32_t b1 = 0, b2 = 0;
};

struct PlanPass {
  int lo, hi;  // the window: global bits [lo, hi)
  int c;       // contiguous low local bits (the window itself when lo = 0)
  std::vector<PlanRound> rounds;
};

// A bound on the rounds of all passes of a circuit on its default tile (a round
// holds four rotations; at most 1.52 slots go to each, at 29 qubits).  It grows
// with n and L, while a larger shape's own rounds can be fewer than a smaller's.
inline int sweep_round_bound(int n, int L) { return (25 * n * L / 16 + 3) / 4; }

// The circuit as three events per bit and layer: the bond of the first group,
// the bond of the second (passed over where the end bits have none), the
// rotation.  Bond k belongs to qubits n-2-k and n-1-k; the odd bonds act first
// (state.py:229-241).  CZ bonds commute, and keep the same order here.
class SweepPlanner {
 public:
  SweepPlanner(int n, int L, bool cz, int K, int c) : n_(n), L_(L), cz_(cz), K_(std::min(K, n)), c_(c) {
    for (int l = K_ - 4;; l = std::max(0, l - 4)) {
      los_[nl_++] = l;
      if (l == 0) break;
    }
  }

  // A beam of a few states (progress of every bit): each step extends every
  // state by every window and keeps those that have run the most rotations,
  // fewer rounds first among equals.  The passes grow with the layers only.
  // Host time 0.14 ms at 19 qubits and 20 layers, 0.35 ms at 24 and 40.
  std::vector<PlanPass> plan(int steps) const {
    std::vector<std::pair<int, int>> win{{0, K_}};
    for (int lo = c_; K_ < n_ && lo + K_ - c_ <= n_; ++lo) win.push_back({lo, lo + K_ - c_});
    struct Node {
      State at;
      int rots, rounds, parent, window;
    };
    std::vector<Node> all{{start(), 0, 0, -1, -1}};  // every kept node, a level after the other
    size_t first = 0;                                // of the last level
    std::vector<Node> next;
    const int total = n_ * L_;
    constexpr size_t kBeam = 3;
    while (all[first].rots < total) {
      const size_t last = all.size();
      next.clear();
      for (size_t i = first; i < last; ++i)
        for (int w = 0; w < (int)win.size(); ++w) {
          next.push_back(all[i]);
          Node& nd = next.back();
          int rots = 0, rounds = 0;
          run(nd.at, win[w].first, win[w].second, steps, &rots, &rounds, nullptr);
          nd.rots += rots;
          nd.rounds += rounds;
          nd.parent = (int)i;
          nd.window = w;
          if (!rots) next.pop_back();
        }
      while (all.size() - last < kBeam) {
        const Node* best = nullptr;
        for (const Node& nd : next) {
          if (best && (nd.rots != best->rots ? nd.rots < best->rots : nd.rounds >= best->rounds)) continue;
          bool same = false;
          for (size_t k = last; k < all.size(); ++k)
            same |= std::equal(nd.at.prog, nd.at.prog + n_, all[k].at.prog);
          if (!same) best = &nd;
        }
        if (!best) break;
        all.push_back(*best);
      }
      if (all.size() == last) return {};  // cannot happen: some window always has a ready rotation
      first = last;
    }
    std::vector<int> order;
    for (int i = (int)first; all[i].parent >= 0; i = all[i].parent) order.push_back(all[i].window);
    std::vector<PlanPass> out;
    State at = start();
    for (int k = (int)order.size() - 1; k >= 0; --k) {
      PlanPass p;
      p.lo = win[order[k]].first;
      p.hi = win[order[k]].second;
      p.c = p.lo == 0 ? p.hi : c_;
      int rots = 0, rounds = 0;
      run(at, p.lo, p.hi, steps, &rots, &rounds, &p.rounds);
      out.push_back(std::move(p));
    }
    return out;
  }

 private:
  struct State {
    int32_t prog[kMaxQubits];  // 3 * layer + the event the bit waits for (2: its rotation)
    int8_t event[kMaxQubits];  // prog % 3
  };
  int n_, L_;
  bool cz_;
  int K_, c_;
  int los_[4], nl_ = 0;  // register windows: local bits [los, los + 4)

  int group(int bond) const { return (n_ - 2 - bond) % 2 == 1 ? 0 : 1; }
  // Moves bit b to its next event, past the bond that an end bit does not have.
  void advance(State& s, int b) const {
    do {
      s.prog[b]++;
      s.event[b] = s.event[b] == 2 ? 0 : s.event[b] + 1;
    } while (missing(s, b));
  }
  bool missing(const State& s, int b) const {
    const int e = s.event[b];
    if (e == 2) return false;
    return !(b + 1 < n_ && group(b) == e) && !(b > 0 && group(b - 1) == e);
  }
  State start() const {
    State s;
    for (int b = 0; b < n_; ++b) {
      s.prog[b] = 0;
      s.event[b] = 0;
      while (missing(s, b)) {
        s.prog[b]++;
        s.event[b]++;
      }
    }
    return s;
  }

  // Runs up to `steps` steps (bonds, then at most one rotation per bit) on the
  // window [lo, hi), within kMaxRounds rounds.  Bonds that no rotation of the
  // pass follows are left for a later pass.
  void run(State& s, int lo, int hi, int steps, int* rots, int* rounds, std::vector<PlanRound>* out) const {
    const int c = lo == 0 ? 0 : c_, end = 3 * L_;
    int cur = 0;  // the layout of the last round
    // bonds inside the window, or with their control above it (a CZ bond: either side)
    const int k0 = cz_ && lo > 0 ? lo - 1 : lo, k1 = hi < n_ ? hi : hi - 1;
    State q = s;
    for (int step = 0; step < steps; ++step) {
      uint32_t bonds[2] = {0, 0};
      for (int g = 0; g < 2; ++g)
        for (int k = group(k0) == g ? k0 : k0 + 1; k < k1; k += 2)
          if (q.event[k] == g && q.prog[k] == q.prog[k + 1] && q.prog[k] < end) {
            advance(q, k);
            advance(q, k + 1);
            bonds[g] |= 1u << k;
          }
      uint32_t ready = 0;
      for (int b = lo; b < hi; ++b)
        if (q.event[b] == 2 && q.prog[b] < end) ready |= 1u << b;
      if (!ready) break;
      // register windows, the current one first, then from the end of the
      // list that it is nearer to
      const uint32_t local = c == 0 ? ready >> lo : (ready >> lo) << c;
      int order[4], no = 0, used[4], nu = 0;
      order[no++] = cur;
      for (int i = 0; i < nl_; ++i) {
        const int j = cur * 2 < nl_ ? i : nl_ - 1 - i;
        if (j != cur) order[no++] = j;
      }
      uint32_t left = local, held[4];
      for (int i = 0; i < no; ++i) {
        const uint32_t m = left & (15u << los_[order[i]]);
        if (!m) continue;
        held[nu] = m;
        used[nu++] = order[i];
        left &= ~m;
      }
      if (*rounds + nu > kMaxRounds) break;
      if (out)
        for (int i = 0; i < nu; ++i) {
          PlanRound r;
          r.lo = los_[used[i]];
          for (int k = 0; k < 4; ++k) {
            const bool on = (held[i] >> (r.lo + k)) & 1u;
            r.bit[k] = on ? lo + r.lo + k - c : -1;
            r.layer[k] = on ? q.prog[r.bit[k]] / 3 : -1;
          }
          if (i == 0) {
            r.b1 = bonds[0];
            r.b2 = bonds[1];
          }
          out->push_back(r);
        }
      cur = used[nu - 1];
      for (int b = lo; b < hi; ++b)
        if ((ready >> b) & 1u) {
          advance(q, b);
          ++*rots;
        }
      *rounds += nu;
      s = q;
    }
  }
};

// What a planned circuit depends on: qubits, layers, CZ ladder (else CNOT), local
// bits, contiguous bits, steps.
typedef std::array<int, 6> SweepKey;

// The plans last asked for, shared by the plans of a context: a plan that is laid
// out for the shapes of a request stream, or made anew for a circuit of a known
// shape, does not plan again (30 qubits, 100 layers 0.63 ms a layout, 24 qubits,
// 40 layers 0.15 ms, against 0.02 ms without planning).  Holds at most kPlans
// plans and kRounds rounds (4 MiB); safe to use from several threads.
class SweepPlans {
 public:
  static constexpr size_t kPlans = 64, kRounds = 65536;

  std::vector<PlanPass> get(const SweepKey& k) {
    {
      std::lock_guard<std::mutex> lock(m_);
      for (auto it = held_.begin(); it != held_.end(); ++it)
        if (it->first == k) {
          held_.splice(held_.begin(), held_, it);
          return it->second;
        }
    }
    std::vector<PlanPass> p = SweepPlanner(k[0], k[1], k[2] != 0, k[3], k[4]).plan(k[5]);
    std::lock_guard<std::mutex> lock(m_);
    held_.emplace_front(k, p);
    rounds_ += rounds_of(p);
    while (held_.size() > kPlans || rounds_ > kRounds) {
      rounds_ -= rounds_of(held_.back().second);
      held_.pop_back();
    }
    return p;
  }
  size_t plans() const { return held_.size(); }
  size_t rounds() const { return rounds_; }

 private:
  static size_t rounds_of(const std::vector<PlanPass>& p) {
    size_t r = 0;
    for (const PlanPass& s : p) r += s.rounds.size();
    return r;
  }
  std::mutex m_;
  std::list<std::pair<SweepKey, std::vector<PlanPass>>> held_;  // the last asked for first
  size_t rounds_ = 0;
};

}  // namespace qg
