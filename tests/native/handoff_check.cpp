// The hand-off of instances to a team's blocks (cuopo_amd/csrc/opo_handoff.h)
// under every interleaving of the blocks' operations on shared memory.  Each
// block is a coroutine that gives way before every such operation; a search
// over the choices of who goes next visits every state that some order reaches
// (a state met before is not followed again).  A wait is a step that is
// possible once its condition holds, so a block that misses its word shows as
// a state in which nobody can go on.
#include <ucontext.h>

#include <cstdio>
#include <memory>
#include <set>
#include <string>
#include <vector>

#include "../../cuopo_amd/csrc/opo_handoff.h"

namespace {

struct World;

struct Block {
  ucontext_t ctx;
  std::unique_ptr<char[]> stack{new char[kStack]};
  static constexpr size_t kStack = 64 * 1024;
  World *w = nullptr;
  int team = 0, rank = 0;
  bool done = false;
  bool (*ready)(World &, const Block &) = nullptr;  // null: may go on
  unsigned want = 0;                                 // what `ready` waits for
  unsigned steps = 0, taken = 0;
  std::vector<unsigned> ran;                         // instances, in order
};

struct Case {
  int teams, blocks, nz;  // blocks per team
  std::vector<int> runs;  // per instance: 1 it runs, 0 it has finished
};

struct World {
  const Case &c;
  unsigned next = 0;
  std::vector<unsigned long long> cur;
  std::vector<unsigned> arrivals;            // per team
  std::vector<std::vector<unsigned>> stage;  // per instance and block of its team: stages done
  std::vector<Block> b;
  ucontext_t back;
  std::string wrong;

  explicit World(const Case &k) : c(k), cur(k.teams, 0), arrivals(k.teams, 0), b(k.teams * k.blocks) {
    stage.assign(k.runs.size(), std::vector<unsigned>(k.blocks, 0));
  }
  void give_way(Block &x) {
    ++x.steps;
    swapcontext(&x.ctx, &back);
  }
  // a block's local state follows from its step, its last index and the instances it was given
  std::vector<unsigned long long> state() const {
    std::vector<unsigned long long> k(cur.begin(), cur.end());
    k.push_back(next);
    k.insert(k.end(), arrivals.begin(), arrivals.end());
    for (const auto &s : stage) k.insert(k.end(), s.begin(), s.end());
    for (const auto &x : b) {
      k.push_back(x.steps * 2ull + x.done);
      k.push_back(x.taken);
      k.push_back(x.ran.size());
      k.insert(k.end(), x.ran.begin(), x.ran.end());
    }
    return k;
  }
};

struct Queue {
  World &w;
  Block &me;
  unsigned take() {
    w.give_way(me);
    return me.taken = w.next++;
  }
  void publish(unsigned long long v) {
    w.give_way(me);
    w.cur[me.team] = v;
  }
  bool await(unsigned turn, unsigned long long *v) {
    me.want = turn;
    me.ready = [](World &k, const Block &x) { return opo::is_turn(k.cur[x.team], x.want); };
    w.give_way(me);
    me.ready = nullptr;
    *v = w.cur[me.team];
    return true;
  }
};

// What a block of resident_pass does, stages reduced to their waits and arrivals.
void pass(World &w, Block &me) {
  const unsigned total = (unsigned)w.c.runs.size();
  Queue q{w, me};
  unsigned arrived = 0;
  auto wait_team = [&] {
    me.want = arrived * (unsigned)w.c.blocks;
    me.ready = [](World &k, const Block &x) { return k.arrivals[x.team] >= x.want; };
    w.give_way(me);
    me.ready = nullptr;
  };
  for (unsigned turn = 1;; ++turn) {
    unsigned i = ~0u;
    if (me.rank == 0) i = opo::hand_out(q, turn, total, [&](unsigned k) { return w.c.runs[k] != 0; });
    else opo::hand_in(q, turn, &i);
    if (i >= total) return;
    if (!w.c.runs[i]) w.wrong = "a finished instance was handed out";
    me.ran.push_back(i);
    for (int s = 0; s < 2 * w.c.nz - 1; ++s) {
      if (s > 0) {
        wait_team();
        for (unsigned d : w.stage[i])
          if (d < (unsigned)s) w.wrong = "a stage began before the one before it had ended";
      }
      ++w.stage[i][me.rank];
      w.give_way(me);
      ++w.arrivals[me.team];
      ++arrived;
    }
    if (opo::ends_with_wait(w.c.nz)) wait_team();
  }
}

void enter(unsigned lo, unsigned hi) {
  Block *me = reinterpret_cast<Block *>(((unsigned long long)hi << 32) | lo);
  pass(*me->w, *me);
  me->done = true;
}

using States = std::set<std::vector<unsigned long long>>;

// One order of steps: the choices given, then the first possible block each
// time, up to a state met before; the number of possible blocks at every step
// goes to `wide`.
std::string run(const Case &c, std::vector<int> &choice, std::vector<int> &wide, States &met) {
  World w(c);
  for (int t = 0; t < c.teams; ++t)
    for (int r = 0; r < c.blocks; ++r) {
      Block &x = w.b[t * c.blocks + r];
      x.w = &w;
      x.team = t;
      x.rank = r;
      getcontext(&x.ctx);
      x.ctx.uc_stack.ss_sp = x.stack.get();
      x.ctx.uc_stack.ss_size = Block::kStack;
      x.ctx.uc_link = &w.back;
      const unsigned long long p = reinterpret_cast<unsigned long long>(&x);
      makecontext(&x.ctx, reinterpret_cast<void (*)()>(enter), 2, (unsigned)p, (unsigned)(p >> 32));
    }
  wide.clear();
  for (size_t step = 0;; ++step) {
    std::vector<Block *> can;
    bool all_done = true;
    for (auto &x : w.b) {
      all_done = all_done && x.done;
      if (!x.done && (!x.ready || x.ready(w, x))) can.push_back(&x);
    }
    if (all_done) break;
    if (can.empty()) return "a block waits for a word that will not come";
    if (step == choice.size()) {
      if (!met.insert(w.state()).second) return "";
      choice.push_back(0);
    }
    wide.push_back((int)can.size());
    Block &x = *can[choice[step]];
    swapcontext(&w.back, &x.ctx);
    if (!w.wrong.empty()) return w.wrong;
  }
  for (auto &x : w.b)
    if (x.ran != w.b[x.team * c.blocks].ran) return "the blocks of a team ran different instances";
  for (size_t i = 0; i < c.runs.size(); ++i)
    for (unsigned d : w.stage[i])
      if (d != (c.runs[i] ? 2u * c.nz - 1 : 0u)) return "an instance was not run exactly once";
  return "";
}

// All orders, depth first.
std::string all_orders(const Case &c, States &met) {
  std::vector<int> choice, wide;
  for (;;) {
    const std::string e = run(c, choice, wide, met);
    if (!e.empty()) return e;
    choice.resize(wide.size());
    while (!choice.empty() && choice.back() + 1 == wide[choice.size() - 1]) choice.pop_back();
    if (choice.empty()) return "";
    ++choice.back();
  }
}

}  // namespace

int main() {
  const Case cases[] = {
      {1, 2, 2, {0, 1, 1}}, {1, 2, 2, {1, 0, 0, 1}}, {1, 2, 3, {1, 1, 0}}, {1, 2, 1, {1, 1, 1}},
      {1, 2, 1, {0, 1, 0, 1}}, {1, 2, 1, {0, 0}}, {1, 3, 1, {1, 1}}, {1, 3, 2, {0, 1, 1}}, {2, 2, 1, {1, 0, 1, 1}},
      {2, 2, 2, {1, 0, 1, 1}}, {1, 4, 2, {1, 0, 1}},
  };
  int bad = 0;
  for (const Case &c : cases) {
    States met;
    const std::string e = all_orders(c, met);
    std::printf("teams %d, blocks %d, slices %d, instances", c.teams, c.blocks, c.nz);
    for (int r : c.runs) std::printf(" %d", r);
    std::printf(": %s (%zu states)\n", e.empty() ? "ok" : e.c_str(), met.size());
    std::fflush(stdout);
    bad += !e.empty();
  }
  return bad ? 1 : 0;
}
