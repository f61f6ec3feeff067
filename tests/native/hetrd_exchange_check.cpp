// Host model of the tridiagonalisation's exchange over the rules that its kernel
// uses (csrc/hip/tridiag_exchange.hpp): which workgroup publishes, reads and refills
// which words, without the arithmetic.
#include <vector>

#include "../../sparse-dft_amd/csrc/hip/tridiag_exchange.hpp"

using namespace sdft_hip;

namespace {
constexpr int kEmpty = -1;  // a word that has not been published

struct Group {
  int g = 0, step = 0, row = 0;  // reading row `row` of step `step`
  bool done = false;
};

struct Model {
  int n, groups;
  std::vector<int> word;  // [buffer][row]: the step whose value it holds
  std::vector<Group> group;
  bool wrong = false;
  int& at(int step, int row) { return word[std::size_t(step % kHetrdBuffers) * n + row]; }
  void publish(int g, int step) {
    for (int r = hetrd_first_row(groups, g, step + 1); g + r * groups < n; ++r) at(step, g + r * groups) = step;
  }
  void enter(Group& w, int step) {
    w.step = step;
    w.row = step + 1;
    w.done = step + 1 >= n || !hetrd_reads(n, groups, w.g, step);
  }
  Model(int n_, int groups_) : n(n_), groups(groups_), word(std::size_t(kHetrdBuffers) * n_, kEmpty) {
    for (int g = 0; g < groups; ++g) {
      group.push_back({});
      group.back().g = g;
      publish(g, 0);
    }
    for (Group& w : group) enter(w, 0);
  }
  // Reads one word, or ends the step behind the last; false when it waits.
  bool advance(Group& w) {
    if (w.done) return false;
    const int k = w.step;
    if (w.row < n) {
      const int have = at(k, w.row);
      if (have == kEmpty) return false;
      wrong |= have != k;
      ++w.row;
      return true;
    }
    if (k > 0)
      for (int r = 0; w.g + r * groups < n; ++r)
        if (w.g + r * groups >= k) at(k + 2, w.g + r * groups) = kEmpty;
    if (k + 2 < n) publish(w.g, k + 1);
    enter(w, k + 1);
    return true;
  }
};
}  // namespace

extern "C" {

// Workgroups that read a step, do not publish the next and may find the buffer
// refilled: a refill of step k - 1's buffer waits for the publishers of step k only.
int hetrd_unguarded_readers(int n, int groups) {
  int count = 0;
  for (int k = 1; k + 1 < n; ++k)
    for (int g = 0; g < groups; ++g) {
      const bool publishes = g + hetrd_first_row(groups, g, k + 1) * groups < n;
      bool refilled = false;
      for (int h = 0; h < groups; ++h) refilled |= h != g && hetrd_reads(n, groups, h, k);
      count += hetrd_reads(n, groups, g, k - 1) && !publishes && refilled;
    }
  return count;
}

// The reduction with workgroup `late` moving only when no other can: 0 when every
// workgroup ends with the values of its own steps, 1 when one waits for a word that
// never comes, 2 when one takes another step's value.
int hetrd_with_late_group(int n, int groups, int late) {
  Model m(n, groups);
  for (;;) {
    bool moved = false;
    for (Group& w : m.group)
      while (w.g != late && m.advance(w)) moved = true;
    if (!moved) moved = m.advance(m.group[std::size_t(late)]);
    if (!moved) break;
  }
  for (const Group& w : m.group)
    if (!w.done) return 1;
  return m.wrong ? 2 : 0;
}

}  // extern "C"
