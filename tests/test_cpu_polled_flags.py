"""The tagged flags that a solve polls in pinned memory (csrc/polled_flags.hpp): memory
that still holds an earlier owner's words, equal tags among them, is never taken for a
flag of the new owner's kernels."""
import glob
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include "polled_flags.hpp"
#include <cstdio>
#include <set>
using arapgs::TaggedFlags;
#define CHECK(x) do { if (!(x)) { std::printf("%s, line %d\n", #x, __LINE__); return 1; } } while (0)
int main() {
    int words[32], first_tags[64];
    {
        TaggedFlags earlier;
        for (int i = 0; i < 64; i++) first_tags[i] = earlier.next_tag();
    }
    for (int t = 0; t < 64; t++) {  // every word as the kernels of the earlier owner left it: done, under its tag
        for (int& w : words) w = first_tags[t] | 1;
        TaggedFlags f;
        f.attach(words, 32);
        for (int i = 0; i < 64; i++) {
            const int tag = f.next_tag();
            CHECK(tag != 0 && (tag & 1) == 0);
            for (int& w : words) CHECK(TaggedFlags::read(&w, tag) == -1);
        }
    }
    TaggedFlags f;
    f.attach(words, 32);
    std::set<int> seen;
    for (int i = 0; i < 5000; i++) {
        const int tag = f.next_tag();
        CHECK(seen.insert(tag).second);
        int& w = words[i % 32];
        CHECK(TaggedFlags::read(&w, tag) == -1);
        w = tag;
        CHECK(TaggedFlags::read(&w, tag) == 0);
        w = tag | 1;
        CHECK(TaggedFlags::read(&w, tag) == 1);
    }
    // a word that has moved on within, or outside, a run of tags; also across the end of the numbers
    for (unsigned start : {1u, 77u, 0x1ffffffdu}) {
        auto tag = [&](unsigned i) { return (int)(((start + i) & 0x1fffffffu) << 1); };
        int w = 0;
        CHECK(!TaggedFlags::set_within(&w, tag(0), tag(5)));
        for (unsigned i = 0; i <= 5; i++) {
            w = tag(i) | 1;
            CHECK(TaggedFlags::set_within(&w, tag(0), tag(5)));
            w = tag(i);
            CHECK(!TaggedFlags::set_within(&w, tag(0), tag(5)));
        }
        w = tag(6) | 1;
        CHECK(!TaggedFlags::set_within(&w, tag(0), tag(5)));
        w = (int)(((start - 1) & 0x1fffffffu) << 1) | 1;
        CHECK(!TaggedFlags::set_within(&w, tag(0), tag(5)));
    }
    return 0;
}
"""


def test_words_of_an_earlier_owner(tmp_path):
    src = glob.glob(os.path.join(ROOT, "arap*_amd", "csrc"))[0]
    (tmp_path / "t.cpp").write_text(PROGRAM)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-I", src, str(tmp_path / "t.cpp"), "-o", str(tmp_path / "t")])
    r = subprocess.run([str(tmp_path / "t")], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
