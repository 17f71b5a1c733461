// The gate of resident launches with streams of this file's own: a launch has
// ended when the test says so.
#include <chrono>
#include <set>
#include <string>
#include <thread>

#include "cvf_gate.h"

using namespace cvf;

namespace {
std::set<int> g_idle;        // streams whose launches have ended
std::vector<int> g_waited;   // streams that others were made to wait for
struct Fake {
  using Event = int;
  using Stream = int;
  static bool idle(int st) { return g_idle.count(st) != 0; }
  static int after(int, int other, int) { return g_waited.push_back(other), 0; }
};
using Gate = ResidentGate<Fake>;
}  // namespace

// n handles of `groups` workgroups, `per_cu` to a CU, launch one after the
// other, none of which ends: how many of them run before one is made to wait
extern "C" int probe_together(int n, int groups, int per_cu, int cus) {
  g_idle.clear();
  g_waited.clear();
  Gate gate;
  std::vector<Gate::User> u((size_t)n);
  for (int i = 0; i < n; ++i) {
    u[i].plan = ResidentPlan{0, (uint32_t)groups, (uint32_t)per_cu, (uint32_t)cus};
    u[i].stream = i;
    gate.add(&u[i]);
  }
  for (int i = 0; i < n; ++i) {
    gate.enter(&u[i]);
    if (!g_waited.empty()) return i;
    gate.leave(&u[i]);
  }
  return n;
}

// Two whole-card handles, the first of which launches on and on: whether the
// second, which came while the first was launching, gets in before the first
// one's next launch
extern "C" int probe_order() {
  using namespace std::chrono;
  g_idle = {0, 1};
  Gate gate;
  Gate::User a, b;
  a.plan = b.plan = ResidentPlan{0, 256, 1, 256};
  b.stream = 1;
  gate.add(&a);
  gate.add(&b);
  std::string order;  // (written between enter and leave: one handle at a time)
  gate.enter(&a);
  std::thread t([&] {
    gate.enter(&b);
    order += 'b';
    gate.leave(&b);
  });
  std::this_thread::sleep_for(milliseconds(200));  // b waits
  for (int i = 0; i < 3; ++i) {
    order += 'a';
    gate.leave(&a);
    gate.enter(&a);
  }
  gate.leave(&a);
  t.join();
  return order == "abaa";
}
