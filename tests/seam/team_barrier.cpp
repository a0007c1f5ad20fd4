// Every order of the steps of a few workgroups that go through a chain of team barriers with the flag
// words of ptyk_team.h: announcing one barrier, and reading the words one by one (again from the first
// after a pass that missed someone), are the single steps.  Prints the number of states; fails where a
// barrier hands out anything but the largest value announced for it, or if no order reaches the end.
// ONE_WORD: the same with one word a workgroup and any epoch from the awaited one on, the form in which
// a slow reader meets the next barrier's value.
#include <cstdint>
#include <cstdio>
#include <unordered_set>
#include <vector>

#include "ptyk_team.h"

#ifdef ONE_WORD
static int word(int w, unsigned) { return ptyk::team_word(w, 0); }
static bool here(unsigned long long f, unsigned e) { return (int)((unsigned)(f >> 32) - e) >= 0; }
#else
static int word(int w, unsigned e) { return ptyk::team_word(w, e); }
static bool here(unsigned long long f, unsigned e) { return ptyk::team_here(f, e); }
#endif

constexpr int W = 3, BARRIERS = 5;

static unsigned value(int w, unsigned e) { return 1 + (w * 7 + e * 5) % 11; }
static unsigned largest(unsigned e) {
  unsigned v = 0;
  for (int w = 0; w < W; ++w) v = value(w, e) > v ? value(w, e) : v;
  return v;
}

// one workgroup: barrier (1..BARRIERS, then BARRIERS + 1: past the last), next step (0: announce,
// 1 + i: read word i), the pass's largest value and whether all were there so far
struct Wg {
  unsigned barrier = 1, step = 0, most = 0, ok = 1;
};
struct State {
  Wg g[W];
  uint64_t key() const {
    uint64_t k = 0;
    for (const Wg& x : g) k = (k << 16) | (x.barrier << 12) | (x.step << 9) | (x.most << 1) | x.ok;
    return k;
  }
};

// The words as the announcements so far leave them, started from first (the barrier numbers run on from
// one iteration to the next, so both parities come first).
static unsigned long long read_word(const State& s, int w, unsigned first, unsigned e) {
  std::vector<unsigned long long> words(W * ptyk::PTYK_EPIE_FLAG_STRIDE, ptyk::team_flag(first, 0));
  const unsigned announced = s.g[w].barrier - (s.g[w].step == 0);
  for (unsigned k = 1; k <= announced && k <= BARRIERS; ++k)
    words[word(w, first + k)] = ptyk::team_flag(first + k, value(w, k));
  return words[word(w, e)];
}

int main() {
  long states = 0;
  for (unsigned first : {6u, 7u}) {
    std::unordered_set<uint64_t> seen;
    std::vector<State> todo(1);
    seen.insert(todo[0].key());
    bool end = false;
    while (!todo.empty()) {
      const State s = todo.back();
      todo.pop_back();
      bool past = true;
      for (int w = 0; w < W; ++w) {
        if (s.g[w].barrier > BARRIERS) continue;
        past = false;
        State t = s;
        Wg& x = t.g[w];
        if (x.step == 0) {
          x.step = 1;
        } else {
          const unsigned long long f = read_word(s, x.step - 1, first, first + x.barrier);
          x.ok = x.ok && here(f, first + x.barrier);
          if (ptyk::team_value(f) > x.most) x.most = ptyk::team_value(f);
          if (x.step < W) {
            ++x.step;
          } else if (x.ok) {
            if (x.most != largest(x.barrier)) {
              std::printf("barrier %u gives %u for %u\n", x.barrier, x.most, largest(x.barrier));
              return 1;
            }
            x = Wg{x.barrier + 1, 0, 0, 1};
          } else {
            x = Wg{x.barrier, 1, 0, 1};
          }
        }
        if (seen.insert(t.key()).second) todo.push_back(t);
      }
      end = end || past;
    }
    if (!end) {
      std::printf("no order reaches the end\n");
      return 1;
    }
    states += (long)seen.size();
  }
  std::printf("%ld states\n", states);
  return 0;
}
