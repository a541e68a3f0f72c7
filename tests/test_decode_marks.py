"""What the merge inside the split-KV decode kernels takes for an arrival (floneum_amd/csrc/decode_marks.h): a mark shares the workspace
with other calls' partial results, which nothing clears, so every bit but the four of the XCC id has to tell it from them, and no two
calls of a handle may share a tag (20 compared bits of tag came round again after 2^20 calls)."""
import os
import subprocess

HEADERS = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "floneum_amd", "csrc")

PROGRAM = r"""
#include <algorithm>
#include <cstdio>
#include <vector>
#include "decode_marks.h"
using namespace fhip;
int main() {
    std::vector<uint64_t> tags;
    for (uint64_t n = 1; n <= 3000000; n++) tags.push_back(mark_tag(0x5eed0001u + n));
    for (uint64_t i = 0; i < 1000; i++) {
        const uint64_t tag = tags[i * 2999];
        if (tag & ~MARK_TAG) return printf("tag %llx\n", (unsigned long long)tag), 1;
        for (uint32_t xcc = 0; xcc < 16; xcc++) {
            const uint64_t mark = mark_of(tag, xcc, 1);
            if (!mark_is(mark, tag, 1) || !mark_is_of(mark, tag) || mark_arrivals(mark) != 1) return puts("a mark is not seen"), 1;
            for (uint32_t other = 0; other < 16; other++)
                if (mark_same_xcc(mark, other) != (other == xcc)) return puts("xcc"), 1;
            for (int bit = 0; bit < 64; bit++)
                if (mark_is(mark ^ (uint64_t)1 << bit, tag, 1) != (bit >= 8 && bit < 12)) return printf("bit %d\n", bit), 1;
            if (mark_is(mark & 0xffffffffu, tag, 1) || mark_is(mark >> 32, tag, 1)) return puts("half a mark"), 1;
        }
        if (mark_is(0, tag, 1) || mark_is(tags[i * 2999 + 1] | 1, tag, 1)) return puts("cleared, or the next call's"), 1;
    }
    std::sort(tags.begin(), tags.end());
    if (tags[0] == 0 || std::adjacent_find(tags.begin(), tags.end()) != tags.end()) return puts("two calls share a tag"), 1;
    return 0;
}
"""


def test_marks(tmp_path):
    source, program = tmp_path / "marks.cpp", tmp_path / "marks"
    source.write_text(PROGRAM)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-I", HEADERS, str(source), "-o", str(program)])
    done = subprocess.run([str(program)], capture_output=True, text=True)
    assert done.returncode == 0, done.stdout
