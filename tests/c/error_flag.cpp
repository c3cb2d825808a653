// The error words of calls whose wait succeeded, failed, or never came, with heap
// memory in place of pinned memory. Prints what goes wrong; exits with 1 then.
#include <cstdio>
#include <set>

#include "rn_flags.hpp"

namespace {
std::set<int32_t*> held;
struct Heap {
    static int32_t* take() { return *held.insert(new int32_t(7)).first; }
    static void give(int32_t* w) {
        held.erase(w);
        delete w;
    }
};
using Flag = rn::ErrorFlag<Heap>;
int wrong = 0;
void expect(bool ok, const char* what) {
    if (!ok) std::printf("wrong: %s\n", what), wrong = 1;
}
}  // namespace

int main() {
    int32_t* first = nullptr;
    {
        Flag f;
        first = f.word();
        expect(*first == 0, "a new word is clear");
        *first = 4;  // the kernel's store
        expect(f.settle() == 4, "the word after the wait");
    }
    {
        Flag f;
        expect(f.word() == first && *f.word() == 0, "a settled word is used again, clear");
    }  // its wait failed: the kernel may still run
    {
        Flag f;
        *first = 4;  // the store of the call before
        expect(f.settle() == 0, "a late store reaches another call");
    }
    expect(held.count(first) == 1, "the word of a failed wait stays allocated");
    {
        std::set<int32_t*> words;
        Flag flags[40];
        for (Flag& f : flags) words.insert(f.word()), f.settle();
        expect(words.size() == 40, "calls at one time hold different words");
    }
    expect(held.size() == Flag::kSpare + 1, "the spare words are bounded");
    return wrong;
}
