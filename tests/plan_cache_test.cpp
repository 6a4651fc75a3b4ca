// Host test of gz_plan_cache.hpp: counts how often a size's plan is made.  Run by test_plan_cache_host.py.
#include <cstdio>
#include <vector>

#include "gz_plan_cache.hpp"

static thread_local int made;
struct Plan {
  gz::PlanKey key{};
  Plan() = default;
  explicit Plan(const gz::PlanKey& k) : key(k) { made++; }
};
static bool same(const gz::PlanKey& a, const gz::PlanKey& b) {
  return a.M == b.M && a.N == b.N && a.K == b.K && a.layoutA == b.layoutA && a.layoutB == b.layoutB && a.num_cus == b.num_cus;
}
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)

// `rounds` calls of each of the keys in turn: every call gets its own plan; how many were made
static int in_turn(const std::vector<gz::PlanKey>& keys, int rounds) {
  gz::RecentPlans<Plan, 16> plans;
  made = 0;
  for (int r = 0; r < rounds; r++)
    for (const auto& k : keys)
      if (!same(plans.of(k).key, k)) return -1;
  return made;
}

int main() {
  // the layers of a network on one number of tokens: all multiples of 128, two extents shared
  std::vector<gz::PlanKey> layers;
  for (int i = 1; i <= 16; i++) layers.push_back({256, 1024 * i, 4096, 0, 1, 256});
  for (int n : {1, 2, 4, 8, 16}) CHECK(in_turn({layers.begin(), layers.begin() + n}, 20) == n);
  // more sizes than slots: right plans all the same
  layers.push_back({512, 4096, 4096, 0, 1, 256});
  CHECK(in_turn(layers, 3) == 3 * 17);
  // every part of the key counts
  const gz::PlanKey k{64, 128, 256, 0, 1, 256};
  std::vector<gz::PlanKey> near{k, k, k, k, k, k, k};
  near[1].M++; near[2].N++; near[3].K++; near[4].layoutA = 1; near[5].layoutB = 0; near[6].num_cus = 304;
  CHECK(in_turn(near, 5) == 7);
  // the size that was planned longest ago makes room, the others stay
  gz::RecentPlans<Plan, 16> plans;
  for (int i = 0; i < 17; i++) plans.of(layers[i]);
  made = 0;
  for (int i = 1; i < 17; i++) plans.of(layers[i]);
  CHECK(made == 0);
  plans.of(layers[0]);
  CHECK(made == 1);
  std::puts("ok");
  return 0;
}
