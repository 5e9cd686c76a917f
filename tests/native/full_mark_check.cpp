// Runs the full-mark protocol (halloc_amd/csrc/ha_mark.h) through every
// interleaving of small sets of concurrent adds, frees, adds taken back, head
// searches and a reuse of the slab by another class.  Each operation on the
// slab is a step of its own, and a store takes effect when its step runs, so a
// store that is held back behind other groups' steps is among them.  Once all
// are done, a slab whose count is at its class's threshold has to be marked; a
// needless mark has to be gone after one more head search.  So has a mark that
// is missing because a group of another class with the same chunk size, which
// compares with its own threshold, added to the slab.
#include <ucontext.h>

#include <cstdio>
#include <functional>
#include <string>
#include <vector>

#include "../../halloc_amd/csrc/ha_mark.h"

using ha::u32;

namespace {

constexpr size_t STACK = 64 << 10;
constexpr u32 THR_REUSED = 40;  // the class that takes the emptied slab over

struct Slab {
  u32 count, mark, thr;
};
Slab slab;

struct Actor {
  ucontext_t ctx;
  std::vector<char> stack = std::vector<char>(STACK);
  std::function<void()> body;
  bool done, wants_empty;
};
ucontext_t sched;
Actor* cur;
std::vector<Actor> actors(4);

void step() { swapcontext(&cur->ctx, &sched); }  // back when this actor is next
void entry() {
  cur->body();
  cur->done = true;
  swapcontext(&cur->ctx, &sched);
}

struct M {
  void set(u32 v) const { step(); slab.mark = v; }
  u32 get() const { step(); return slab.mark; }
  void settle() const {}  // a store is in place once its step has run
  bool full() const {
    step();
    const u32 thr = slab.thr;
    step();
    return slab.count >= thr;
  }
};

u32 add(u32 n) { step(); slab.count += n; return slab.count - n; }
u32 sub(u32 n) { step(); slab.count -= n; return slab.count + n; }

void a_add(u32 n, u32 thr) {
  const u32 oc = add(n);
  ha::mark_added(M(), oc, oc + n, thr);
}
void a_free(u32 n, u32 thr) {
  const u32 oc = sub(n);
  ha::mark_freed(M(), oc, oc - n, thr);
}
void a_taken_back(u32 n) {
  (void)add(n);
  const u32 oc = sub(n);
  ha::mark_taken_back(M(), oc, oc - n, slab.thr);
}
void a_search(u32 thr) {
  step();
  const u32 c = slab.count;
  ha::mark_checked(M(), c, thr);
}
void a_reuse(u32 n) {  // takes the empty slab for its class, then fills it
  cur->wants_empty = true;
  step();
  cur->wants_empty = false;
  slab.thr = THR_REUSED;
  a_add(n, THR_REUSED);
}

struct Kind {
  const char* name;
  char k;
  u32 n;
};

long runs = 0;

// one run: follows `path` (choices among the actors that can go on), then the
// first; returns the choices that were open at each step
bool run(const std::vector<Kind>& ks, u32 start, u32 thr, std::vector<u32>& path, std::vector<u32>& open) {
  slab = Slab{start, start >= thr ? 1u : 0u, thr};
  for (size_t i = 0; i < ks.size(); ++i) {
    Actor& a = actors[i];
    a.done = a.wants_empty = false;
    const Kind k = ks[i];
    a.body = [k, thr] {
      if (k.k == 'a') a_add(k.n, thr);
      else if (k.k == 'o') a_add(k.n, thr + 5);
      else if (k.k == 'f') a_free(k.n, thr);
      else if (k.k == 'b') a_taken_back(k.n);
      else if (k.k == 's') a_search(thr);
      else a_reuse(k.n);
    };
    getcontext(&a.ctx);
    a.ctx.uc_stack.ss_sp = a.stack.data();
    a.ctx.uc_stack.ss_size = a.stack.size();
    a.ctx.uc_link = nullptr;
    makecontext(&a.ctx, entry, 0);
    cur = &a;
    swapcontext(&sched, &a.ctx);  // up to its first step
  }
  open.clear();
  for (size_t d = 0;; ++d) {
    std::vector<Actor*> can;
    for (size_t i = 0; i < ks.size(); ++i) {
      Actor& a = actors[i];
      if (!a.done && !(a.wants_empty && slab.count)) can.push_back(&a);
    }
    if (can.empty()) break;
    if (d == path.size()) path.push_back(0);
    open.push_back((u32)can.size());
    cur = can[path[d]];
    swapcontext(&sched, &cur->ctx);
  }
  ++runs;
  bool other = false;
  for (const Kind& k : ks) other |= k.k == 'o';
  if (slab.count >= slab.thr && !slab.mark && !other) return false;
  // one search by itself (its steps must not wait) leaves the mark right
  const bool was_full = slab.count >= slab.thr;
  struct Direct {
    void set(u32 v) const { slab.mark = v; }
    u32 get() const { return slab.mark; }
    void settle() const {}
    bool full() const { return slab.count >= slab.thr; }
  };
  ha::mark_checked(Direct(), slab.count, slab.thr);
  return slab.mark == (was_full ? 1u : 0u);
}

bool all(const std::vector<Kind>& ks, u32 start, u32 thr) {
  std::vector<u32> path, open;
  for (;;) {
    if (!run(ks, start, thr, path, open)) {
      std::printf("count %u, threshold %u:", start, thr);
      for (const Kind& k : ks) std::printf(" %s(%u)", k.name, k.n);
      std::printf(", order");
      for (size_t d = 0; d < open.size(); ++d) std::printf(" %u", path[d]);
      std::printf(": count %u mark %u\n", slab.count, slab.mark);
      return false;
    }
    path.resize(open.size());
    while (!path.empty() && path.back() + 1 == open[path.size() - 1]) path.pop_back();
    if (path.empty()) return true;
    ++path.back();
  }
}

}  // namespace

int main() {
  const u32 thr = 100;
  const Kind A{"add", 'a', 10}, A2{"add", 'a', 3}, F{"free", 'f', 10}, F2{"free", 'f', 4}, B{"taken back", 'b', 12},
      B2{"taken back", 'b', 7}, S{"search", 's', 0}, O{"add of another class", 'o', 8}, R{"reuse", 'r', 50};
  const std::vector<std::vector<Kind>> sets = {{A, F},    {F, S},    {A, F, S}, {A, A2, F}, {F, F2, A},  {B, A},
                                               {B, F},    {B, A, F}, {B, B2, A}, {B, S, A}, {B2, F2, A2}, {B, B2, F}, {O, A2, F2}, {O, S}};
  for (const auto& ks : sets)
    for (u32 start = 76; start <= 120; ++start)
      if (!all(ks, start, thr)) return 1;
  for (u32 extra : {0u, 1u})  // emptied while a free that crossed the threshold holds its store back
    if (!all({F, Kind{"free", 'f', 95 + extra}, R}, 105 + extra, thr)) return 1;
  std::printf("ok\n");
  return 0;
}
