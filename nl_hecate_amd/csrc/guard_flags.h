// Flags of the tests in chunkwise_guard.hip: pairs of words in pinned host memory, handed out in turn.
#pragma once
#include <mutex>

namespace nlh {

// Both lowered before the launch.  A kernel raises `reached` in any case, `fired` if a coupling may fire.
struct GuardFlag { int fired, reached; };

// Lowered flags read "may fire": only a kernel that ran can say that nothing does.
inline bool guard_clear(const volatile GuardFlag *f) { return f->reached != 0 && f->fired == 0; }

// N places of one allocation, so that tests of several threads do not share one.
template <int N>
class GuardFlags {
  public:
    // alloc(bytes) -> memory, or null; not called again once it has given some.
    template <class Alloc>
    GuardFlag *lowered(Alloc alloc) {
        const std::lock_guard<std::mutex> lock(mutex_);
        if (!flags_) flags_ = static_cast<GuardFlag *>(alloc(N * sizeof(GuardFlag)));
        if (!flags_) return nullptr;
        volatile GuardFlag *f = flags_ + next_++ % N;
        f->fired = f->reached = 0;
        return const_cast<GuardFlag *>(f);
    }

  private:
    std::mutex mutex_;
    GuardFlag *flags_ = nullptr;
    unsigned next_ = 0;
};

}  // namespace nlh
