"""The flags by which the host takes a call's results chunk by chunk (frk_stage.hpp): a call's number is never what a chunk's flag
holds already, around the end of 32 bits too, where small results (few flags written) come before larger ones."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = """
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "frink_amd/csrc/frk_stage.hpp"
int main(int argc, char **argv) {  // the chunks of each call, "=N": N is the last call's number
    uint32_t epoch = 0;
    std::vector<uint32_t> flags(128, 0);
    for (int i = 1; i < argc; i++) {
        if (argv[i][0] == '=') {
            epoch = (uint32_t)strtoul(argv[i] + 1, nullptr, 10);
            continue;
        }
        epoch = frk::next_epoch(epoch, flags.data(), flags.size());
        const size_t chunks = (size_t)atoi(argv[i]);
        size_t early = 0;
        for (size_t c = 0; c < chunks; c++) early += flags[c] == epoch;
        printf("%zu ", early);
        for (size_t c = 0; c < chunks; c++) flags[c] = epoch;  // (as the kernel raises them)
    }
}
"""


@pytest.fixture(scope="module")
def early(tmp_path_factory):
    d = tmp_path_factory.mktemp("stage")
    (d / "stage.cpp").write_text(SOURCE)
    subprocess.check_call(["g++", "-std=c++17", "-Wall", "-fsanitize=address,undefined", "-I", ROOT, str(d / "stage.cpp"), "-o", str(d / "stage")])
    return lambda *args: [int(v) for v in subprocess.check_output([str(d / "stage")] + [str(a) for a in args]).split()]


@pytest.mark.parametrize("last", [0, 1, 2 ** 31 - 1, 2 ** 32 - 3, 2 ** 32 - 2, 2 ** 32 - 1])
def test_no_chunk_is_ready_before_its_flag_is_raised(early, last):
    assert early("=%d" % last, 1, 128, 2, 128, 1, 1, 128) == [0] * 7


def test_a_flag_of_the_first_round_of_numbers_is_not_mistaken(early):
    """A call with many chunks, small results until the numbers are used up and have begun again, many chunks."""
    assert early(128, "=%d" % (2 ** 32 - 2), 1, 1, 128, 128) == [0] * 5
