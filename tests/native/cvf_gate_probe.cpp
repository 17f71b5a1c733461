// The gate of resident launches with events of this file's own: a launch is
// done when the test says so.
#include <chrono>
#include <set>
#include <string>
#include <thread>

#include "cvf_gate.h"

using namespace cvf;

namespace {
std::set<int> g_done;        // launches that have ended
std::vector<int> g_waited;   // events that the streams were made to wait for
struct Fake {
  using Event = int;
  using Stream = int;
  static bool done(int e) { return g_done.count(e) != 0; }
  static int wait(int, int e) { return g_waited.push_back(e), 0; }
  static int record(int, int) { return 0; }
};
using Gate = ResidentGate<Fake>;
}  // namespace

// n handles of `groups` workgroups, `per_cu` to a CU, launch one after the
// other, none of which ends: how many of them run before one is made to wait
extern "C" int probe_together(int n, int groups, int per_cu, int cus) {
  g_done.clear();
  g_waited.clear();
  Gate gate;
  std::vector<Gate::User> u((size_t)n);
  for (int i = 0; i < n; ++i) {
    u[i].plan = ResidentPlan{0, (uint32_t)groups, (uint32_t)per_cu, (uint32_t)cus};
    u[i].done = i;
    gate.add(&u[i]);
  }
  for (int i = 0; i < n; ++i) {
    gate.enter(&u[i], 0);
    if (!g_waited.empty()) return i;
    gate.leave(&u[i], 0);
  }
  return n;
}

// Two whole-card handles, the first of which launches on and on: whether the
// second, which came while the first was launching, gets in before the first
// one's next launch
extern "C" int probe_order() {
  using namespace std::chrono;
  g_done = {0, 1};
  Gate gate;
  Gate::User a, b;
  a.plan = b.plan = ResidentPlan{0, 256, 1, 256};
  b.done = 1;
  gate.add(&a);
  gate.add(&b);
  std::string order;  // (written between enter and leave: one handle at a time)
  gate.enter(&a, 0);
  std::thread t([&] {
    gate.enter(&b, 0);
    order += 'b';
    gate.leave(&b, 0);
  });
  std::this_thread::sleep_for(milliseconds(200));  // b waits
  for (int i = 0; i < 3; ++i) {
    order += 'a';
    gate.leave(&a, 0);
    gate.enter(&a, 0);
  }
  gate.leave(&a, 0);
  t.join();
  return order == "abaa";
}
