// Turns of the resident launches of several handles of a process (host only).
#pragma once

#include <stdint.h>

#include <algorithm>
#include <condition_variable>
#include <mutex>
#include <vector>

namespace cvf {

// Engines of workgroups on a card, 8 XCDs of 4: a launch's workgroups go round
// them in turn.
constexpr uint32_t kEngines = 32;

// What a resident plan asks of its device: workgroups, how many of them a CU
// holds at once, and the CUs.
struct ResidentPlan {
  int device = 0;
  uint32_t groups = 0, per_cu = 1, cus = 1;
  // workgroups on the busiest engine, times the engines
  uint32_t spread() const { return (groups + kEngines - 1) / kEngines * kEngines; }
};

// Launches that are on one device at the same time.
struct ResidentLoad {
  uint32_t groups = 0;  // spread
  double room = 0;      // share of the room for workgroups such as each plan's
  bool large = false;   // some plan has one workgroup per CU
  void add(const ResidentPlan& p) {
    groups += p.spread();
    room += (double)p.spread() / ((double)p.per_cu * p.cus);
    large = large || p.per_cu < 2;
  }
  // Whether all their workgroups surely are on the card at once, wherever the
  // dispatcher puts them: with no more workgroups than CUs on any engine there
  // is an empty CU for the next one; with workgroups of at most half a CU, half
  // of the room is free CUs or free halves of CUs.
  bool fits(uint32_t cus) const { return groups <= cus || (!large && room <= 0.5); }
};

// A resident kernel's workgroups wait for each other, so each launch needs all
// of its own on the card at once, and two launches of which each has a part
// would wait until their limit.  Handles of a process whose plans are resident
// therefore enter() before they enqueue one such launch (a sequence of at most
// graph_steps steps) and leave() after it: those that surely fit together run
// side by side, any other one waits on the device for those before it.  They
// get in in the order in which they came, so that a handle that steps on and on
// lets the others in between its launches.  A handle that does not have to wait
// only takes the lock and looks whether the others' streams are idle; one that
// does records its event on theirs.  (An event recorded by every launch while
// there was another handle took 6 us of a sample's 350.)
// Streams: idle(stream); after(stream, other, event): the first goes on after
// what is on the other now, by that event; an error code, 0 for none.
template <class Streams>
struct ResidentGate {
  using Event = typename Streams::Event;
  using Stream = typename Streams::Stream;
  struct User {
    ResidentPlan plan;
    Stream stream = {};  // of its launches: on no other, and nothing is captured on it
    Event event = {};
    bool launching = false, pending = false;  // pending: its last launch may not have ended
  };
  std::mutex mu;
  std::condition_variable changed;
  uint64_t came = 0, in = 0;  // calls of enter(), and those of them that have returned
  std::vector<User*> users;

  void add(User* u) {
    std::lock_guard<std::mutex> lock(mu);
    if (std::find(users.begin(), users.end(), u) == users.end()) users.push_back(u);
  }
  void remove(User* u) {
    std::lock_guard<std::mutex> lock(mu);
    users.erase(std::remove(users.begin(), users.end(), u), users.end());
  }
  int enter(User* u) {
    std::unique_lock<std::mutex> lock(mu);
    const uint64_t me = came++;
    std::vector<User*> before;
    for (;;) {
      bool launching = false;
      if (in == me) {
        // with all that may be running, then (if need be) with what is
        bool fits = false;
        for (int look = 0; look < 2 && !fits; ++look) {
          ResidentLoad load;
          load.add(u->plan);
          before.clear();
          launching = false;
          for (User* o : users) {
            if (o == u || o->plan.device != u->plan.device) continue;
            if (look && !o->launching && o->pending && Streams::idle(o->stream)) o->pending = false;
            if (!o->launching && !o->pending) continue;
            before.push_back(o);
            load.add(o->plan);
            launching = launching || o->launching;
          }
          fits = before.empty() || load.fits(u->plan.cus);
        }
        if (fits) before.clear();
        if (fits || !launching) break;
      }
      // someone came earlier, or has not enqueued its launch yet
      changed.wait(lock);
    }
    int e = 0;
    for (User* o : before)
      if (!e) e = Streams::after(u->stream, o->stream, o->event);
    u->launching = e == 0;
    ++in;
    changed.notify_all();
    return e;
  }
  void leave(User* u) {
    std::lock_guard<std::mutex> lock(mu);
    u->launching = false;
    u->pending = true;
    changed.notify_all();
  }
};

}  // namespace cvf
