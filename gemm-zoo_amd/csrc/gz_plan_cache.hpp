// The plans of the last few sizes that a thread has called with: host code alone, no HIP.
#pragma once

namespace gz {

// What a plan of the launcher's own choice depends on.
struct PlanKey {
  int M, N, K, layoutA, layoutB, num_cus;
  bool operator==(const PlanKey& o) const {
    return M == o.M && N == o.N && K == o.K && layoutA == o.layoutA && layoutB == o.layoutB && num_cus == o.num_cus;
  }
};

// SLOTS plans, found by comparing every key (the sizes of a network share their low bits, and often two of three extents, so
// a slot computed from them is one slot for most of them: with such a table every call of a thread that took two sizes in
// turn planned anew).  The one that was planned longest ago makes room for a new size.  A plan outlives the call of of()
// that returned it until SLOTS other sizes have been asked for.
template <class Plan, int SLOTS> class RecentPlans {
 public:
  // the plan kept for `key`, or a fresh Plan(key)
  Plan& of(const PlanKey& key) {
    if (last_ < used_ && keys_[last_] == key) return plans_[last_];
    for (int i = 0; i < used_; i++)
      if (keys_[i] == key) return plans_[last_ = i];
    last_ = next_;
    next_ = (next_ + 1) % SLOTS;
    if (used_ < SLOTS) used_++;
    keys_[last_] = key;
    return plans_[last_] = Plan(key);
  }

 private:
  PlanKey keys_[SLOTS];
  Plan plans_[SLOTS];
  int used_ = 0, next_ = 0, last_ = 0;
};

}  // namespace gz
