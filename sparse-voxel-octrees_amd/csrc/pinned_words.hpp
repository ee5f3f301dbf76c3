// The pinned words in which a build's host side receives counts: one set that
// kernels write is out at a time, and copies land there only while none is. What
// gets null goes through device or pageable memory instead. The caller owns the
// memory.
#pragma once

#include <cstdint>

namespace svo {

class PinnedWords {
public:
    static constexpr int kWords = 256;
    uint64_t *mem = nullptr;  // kWords words; null if there was no memory to pin

    // `count` words for kernels to write, out until given back
    uint64_t *take(int count) {
        if (!land(count)) return nullptr;
        out_ = true;
        return mem;
    }
    // where a copy of `count` words that is waited for at once may land
    uint64_t *land(int count) const { return mem && !out_ && count <= kWords ? mem : nullptr; }
    // gives `w` back; false if it is not the set that is out
    bool give(const uint64_t *w) {
        if (!out_ || w != mem) return false;
        out_ = false;
        return true;
    }
    void reset() { out_ = false; }  // a build that failed with a set out has ended

private:
    bool out_ = false;
};

}  // namespace svo
