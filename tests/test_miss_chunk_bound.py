"""The chunks that a launch with miss records may need: the host's bound
against the kernels' rule, in a C++ program on the CPU.  A single launch has
no later one to finish what a pause leaves, so the bound must hold for any
numbers of records per iteration, those that fill chunks badly among them."""

import os
import subprocess

from conftest import PKG

PROGRAM = r"""
#include "util_kernels.hpp"
#include <cstdio>
#include <random>
using namespace ffr;

// a run of a wave: `n` records per iteration, as next_chunk takes chunks
template <typename F> static void run(int words, uint64_t iterations, F &&n, uint64_t &chunks,
                                      uint64_t &records)
{
    const unsigned size = miss_chunk(words);
    bool have = false;
    unsigned pos = 0;
    for (uint64_t i = 0; i < iterations; ++i) {
        const unsigned k = n(i);
        if (!k)
            continue;
        if (!have || pos + k > size) {
            ++chunks;
            have = true;
            pos = 0;
        }
        pos += k;
        records += k;
    }
}

int main()
{
    std::mt19937 rng(1);
    int tighter = 0;
    for (int words : {1, 4, 8, 12})
        for (int kind = 0; kind < 8; ++kind)
            for (uint64_t runs : {1ull, 16ull, 512ull})
                for (uint64_t iterations : {1ull, 63ull, 4097ull, 200000ull / runs}) {
                    uint64_t chunks = 0, records = 0;
                    for (uint64_t w = 0; w < runs; ++w)
                        run(words, iterations, [&](uint64_t i) -> unsigned {
                            switch (kind) {
                            case 0: return 64;
                            case 1: return 63;
                            case 2: return i % 65 ? 64 : 1; // 4096 = 1 + 63.98 * 64
                            case 3: return i & 1 ? 64 : 63;
                            case 4: return rng() % 65;
                            case 5: return 1;
                            case 6: return i % 257 ? 64 : 1;
                            default: return 40 + rng() % 25;
                            }
                        }, chunks, records);
                    const uint64_t most = miss_chunks_most(records, runs, words);
                    if (chunks > most) {
                        std::printf("words %d kind %d runs %llu: %llu chunks, bound %llu\n", words,
                                    kind, (unsigned long long)runs, (unsigned long long)chunks,
                                    (unsigned long long)most);
                        return 1;
                    }
                    // (whole chunks, and one begun per run, are not enough)
                    tighter += chunks > records / miss_chunk(words) + runs;
                }
    std::printf("%d\n", tighter);
    return tighter ? 0 : 2;
}
"""


def test_bound_holds_for_any_fill(tmp_path):
    src, exe = tmp_path / "bound.cpp", tmp_path / "bound"
    src.write_text(PROGRAM)
    rocm = os.environ.get("ROCM", "/opt/rocm")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-w",
                           f"-I{rocm}/include", f"-I{PKG}/csrc", str(src), "-o", str(exe)])
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
