// The builder's pinned count words (csrc/pinned_words.hpp): a set that kernels
// write is never handed out again nor copied over before it is given back.
#include <cstdio>

#include "pinned_words.hpp"

int main() {
    int bad = 0;
    auto expect = [&](bool ok, const char *what) {
        if (!ok) std::printf("wrong: %s\n", what);
        bad += !ok;
    };
    uint64_t mem[svo::PinnedWords::kWords], other[1];
    svo::PinnedWords none;
    expect(!none.take(1) && !none.land(1) && !none.give(nullptr), "nothing without pinned memory");
    svo::PinnedWords w;
    w.mem = mem;
    expect(!w.take(svo::PinnedWords::kWords + 1) && !w.land(svo::PinnedWords::kWords + 1), "more words than there are");
    expect(w.land(svo::PinnedWords::kWords) == mem, "a copy lands while no set is out");
    expect(!w.give(mem), "nothing to give back yet");
    expect(w.take(2) == mem, "the set is free");
    expect(!w.take(1) && !w.land(1), "neither a second set nor a copy while it is out");
    expect(!w.give(other) && !w.take(1), "another array does not free it");
    expect(w.give(mem) && !w.give(mem), "given back once");
    expect(w.take(1) == mem, "free again");
    w.reset();
    expect(w.land(1) == mem, "free after a build that failed");
    std::printf("%s\n", bad ? "bad" : "ok");
    return bad;
}
