// Error words in pinned host memory: a word that a call's kernel writes on an
// error and the host reads once it has waited for the call's stream. No device
// allocation, clearing launch or copy back per call (rn_attend_heads with a handful
// of heads: 42 -> 14 us a call).
#pragma once
#include <cstddef>
#include <cstdint>
#include <mutex>

namespace rn {

// One call's word, from Memory::take() or left over from an earlier call. Calls
// from several threads hold different words; at most kSpare wait for the next
// calls, words past that go back to Memory. A word is passed on only after
// settle(): until a wait has shown the kernel done, a late store may still land
// in it, so a call whose launch or wait failed keeps its word for good.
template <class Memory>
class ErrorFlag {
public:
    static constexpr size_t kSpare = 16;

    ErrorFlag() {
        {
            std::lock_guard<std::mutex> lock(mu_);
            if (spares_ > 0) word_ = spare_[--spares_];
        }
        if (!word_) word_ = Memory::take();
        if (word_) *word_ = 0;
    }
    ~ErrorFlag() {
        if (!word_ || !settled_) return;
        {
            std::lock_guard<std::mutex> lock(mu_);
            if (spares_ < kSpare) {
                spare_[spares_++] = word_;
                return;
            }
        }
        Memory::give(word_);
    }
    ErrorFlag(const ErrorFlag&) = delete;
    ErrorFlag& operator=(const ErrorFlag&) = delete;

    // null when there was no memory
    int32_t* word() const { return word_; }
    // what the kernel left, after a wait for its stream that succeeded
    int32_t settle() {
        settled_ = true;
        return *const_cast<volatile int32_t*>(word_);
    }

private:
    static inline std::mutex mu_;
    static inline int32_t* spare_[kSpare] = {};
    static inline size_t spares_ = 0;
    int32_t* word_ = nullptr;
    bool settled_ = false;
};

}  // namespace rn
