// Flags that kernels store into pinned host memory and the host polls while the
// work behind them is still queued.
#pragma once

namespace arapgs {

// A stored word is tag | flag. Tags are even, differ from one to the next and
// name what the flag belongs to, so a word that earlier work left behind is never
// taken for the awaited one; tag 0 stands for none.
class TaggedFlags {
public:
    // words: n ints as the allocator gave them. They may be memory that an earlier
    // owner's kernels stored equal tags into, so they are cleared here.
    void attach(int* words, int n) {
        for (int i = 0; i < n; i++) __atomic_store_n(words + i, 0, __ATOMIC_SEQ_CST);
    }
    int next_tag() {
        do seq_ = (seq_ + 1) & 0x1fffffffu;
        while (seq_ == 0);
        return (int)(seq_ << 1);
    }
    // The flag stored with this tag, or -1 while the word holds another.
    static int read(const int* word, int tag) {
        const int v = __atomic_load_n(word, __ATOMIC_ACQUIRE);
        return (v & ~1) == tag ? v & 1 : -1;
    }
    // Whether the word holds a set flag of any tag from `first` to `last`, in the order in which they were given.
    static bool set_within(const int* word, int first, int last) {
        const int v = __atomic_load_n(word, __ATOMIC_ACQUIRE);
        const unsigned at = ((unsigned)(v >> 1) - (unsigned)(first >> 1)) & 0x1fffffffu;
        return (v & 1) && at <= (((unsigned)(last >> 1) - (unsigned)(first >> 1)) & 0x1fffffffu);
    }

private:
    unsigned seq_ = 0;
};

}  // namespace arapgs
