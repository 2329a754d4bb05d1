"""How a bucket is cut into token blocks and in which order a launch lists them (csrc/token_blocks.h), compiled for the host."""
import os
import random
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
# arguments: by_size, then the experts' row counts; prints a line "expert rows-per-full-tile full-tiles remainder" and the positions of the
# first full and of the last tile, as the bucketing kernel adds them up
PROGRAM = """
#include <stdio.h>
#include <stdlib.h>
#include <vector>
#include "token_blocks.h"
int main(int argc, char** v) {
    constexpr int even = EVEN, tokens = TOKENS;
    std::vector<moe::TokenBlocks> b;
    for (int i = 2; i < argc; ++i) b.push_back(moe::token_blocks<even>(tokens, atoi(v[i])));
    const moe::TileOrder<even> order{tokens, atoi(v[1])};
    const int E = (int)b.size();
    for (int e = 0; e < E; ++e) {
        int full = 0, last = 0;
        for (int i = 0; i < E; ++i) {
            full += order.ahead_of_full(b[i], i, b[e], e);
            last += order.ahead_of_last(b[i], i, b[e], e);
        }
        printf("%d %d %d %d %d\\n", b[e].rows, b[e].full, b[e].rem, full, last);
    }
}
"""
CUTS = [(64, "0", 1), (128, "moe::kPrefillStep", 16), (256, "moe::kPrefillStepBf16", 64)]


@pytest.fixture(params=CUTS, ids=["decode", "mxfp4", "bf16"])
def cut(request, tmp_path):
    tokens, even, step = request.param
    src, exe = tmp_path / "cut.cpp", str(tmp_path / "cut")
    src.write_text(PROGRAM.replace("EVEN", even).replace("TOKENS", str(tokens)))
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include"),
                    "-I" + os.path.join(ROOT, "gpt-oss-amd_amd", "csrc"), str(src), "-o", exe], check=True, capture_output=True)

    def run(by_size, counts):
        out = subprocess.run([exe, str(by_size)] + [str(c) for c in counts], check=True, capture_output=True, text=True).stdout
        return [tuple(int(v) for v in line.split()) for line in out.splitlines()]
    return run, tokens, step


def test_cut_costs_no_more_than_whole_blocks(cut):
    """No more blocks and no more matrix work, in the steps that the kernel rounds up to, than whole blocks and a remainder take."""
    run, tokens, step = cut
    steps = lambda n: -(-n // step)  # noqa: E731
    counts = list(range(1, 4000))
    for count, (rows, full, rem, _, _) in zip(counts, run(1, counts)):
        n = -(-count // tokens)
        assert rows * full + rem == count and full + (rem > 0) == n and 0 <= rem < rows <= tokens, count
        assert full * steps(rows) + steps(rem) <= (n - 1) * steps(tokens) + steps(count - (n - 1) * tokens), count
        if n > 1 and step > 1 and not (step == 16 and n > 2):  # cut evenly: within a step for each block
            assert rows - (-(-count // n)) < step, count
        else:
            assert rows == tokens, count


@pytest.mark.parametrize("by_size", [0, 1])
def test_every_tile_has_a_place_of_its_own(cut, by_size):
    """The places are 0 .. tiles - 1, each once, and they go down by size (by_size), or the last tiles by size after all the others."""
    run, tokens, step = cut
    rng = random.Random(tokens + by_size)
    for experts in (1, 2, 7, 40, 130):
        for _ in range(6):
            counts = [rng.choice([0, 1, tokens, tokens + 1, 2 * tokens, 3 * tokens - 1, rng.randrange(3 * tokens), rng.randrange(20 * tokens)])
                      for _ in range(experts)]
            place = {}
            for rows, full, rem, at_full, at_last in run(by_size, counts):
                for j in range(full):
                    assert at_full + j not in place
                    place[at_full + j] = (1 if not by_size else 0, -(-rows // step))
                if rem:
                    assert at_last not in place
                    place[at_last] = (0, -(-rem // step))
            assert sorted(place) == list(range(len(place))), counts
            order = [place[i] for i in range(len(place))]
            if by_size:
                assert order == sorted(order, reverse=True), counts
            else:
                last = [s for kind, s in order if kind == 0]
                assert [k for k, _ in order] == sorted((k for k, _ in order), reverse=True) and last == sorted(last, reverse=True), counts
