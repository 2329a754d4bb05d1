"""How a bucket is cut into token blocks (even_tile_rows of csrc/kernels.h), compiled for the host: for every bucket length of both prefill
kernels, no more blocks and no more matrix work than whole blocks and a remainder take, in the steps that the kernel rounds up to."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = """
#include <stdio.h>
#include <stdlib.h>
#include "kernels.h"
int main(int, char** v) {
    const int tokens = atoi(v[1]), step = atoi(v[2]);
    for (int count = 1; count <= 6000; ++count) printf("%d\\n", moe::even_tile_rows(count, tokens, step));
}
"""


@pytest.mark.parametrize("tokens,step", [(128, "kPrefillStep"), (256, "kPrefillStepBf16")])
def test_even_cut_costs_no_more_than_whole_blocks(tmp_path, tokens, step):
    src, exe = tmp_path / "cut.cpp", str(tmp_path / "cut")
    src.write_text(PROGRAM.replace("atoi(v[2])", "moe::" + step))
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include"),
                    "-I" + os.path.join(ROOT, "gpt-oss-amd_amd", "csrc"), str(src), "-o", exe], check=True, capture_output=True)
    rows = [int(v) for v in subprocess.run([exe, str(tokens)], check=True, capture_output=True, text=True).stdout.split()]
    unit = {128: 16, 256: 64}[tokens]  # MFMA tiles of 16 tokens; four of them in the bf16 kernel's full row blocks
    steps = lambda n: -(-n // unit)  # noqa: E731
    for count, full in enumerate(rows, 1):
        n = -(-count // tokens)
        last = count - (n - 1) * full
        assert 0 < last <= full <= tokens, (count, full)
        whole = (n - 1) * steps(tokens) + steps(count - (n - 1) * tokens)
        assert (n - 1) * steps(full) + steps(last) <= whole, (count, full)
    assert rows[tokens] < tokens  # one row past a whole block: cut
    if tokens == 128:  # longer MXFP4 buckets are left whole
        assert all(r == tokens for r in rows[2 * tokens:])
