// The last few answers of a planner, per thread: a launch asks its kernel's planner several times (does it
// take the shape, with what grid), a training step the same few shapes over and over, and a search
// over strip heights is a microsecond of host time that a small layer's launch would wait for.
#ifndef CP4_PLAN_MEMO_H
#define CP4_PLAN_MEMO_H

#include <array>

namespace cp4 {

// Key: what the answer depends on, a std::array of integers (compute units of the device included).  make()
// may ask the same memo for something else, as the workspace of a layer on padded channels does: the answer is
// put away, and given out as a copy, only when there is one.
template <class Key, class Answer, int kEntries = 4>
struct PlanMemo {
  Key keys[kEntries];
  Answer answers[kEntries];
  int used = 0, next = 0;
  template <class Make>
  Answer get(const Key& key, Make make) {
    for (int i = 0; i < used; ++i)
      if (keys[i] == key) return answers[i];
    const Answer answer = make();
    answers[next] = answer;
    keys[next] = key;
    next = (next + 1) % kEntries;
    if (used < kEntries) ++used;
    return answer;
  }
};

}  // namespace cp4
#endif
