"""The stop word of the solver's iterations, compiled for the host from the
header that the kernels include."""
import ctypes as C
import itertools
import subprocess

import pytest

from fastipc_amd import build as B

SOURCE = r'''
#include "fipc_ctx.h"
extern "C" int past(int it, int stop) { return pcg_past(it, stop); }
extern "C" int stop_word(int it) { return pcg_stop(it); }
extern "C" int running() { return PCG_RUNNING; }
extern "C" int at_start() { return PCG_AT_START; }
'''


@pytest.fixture(scope="module")
def word(tmp_path_factory):
    d = tmp_path_factory.mktemp("stop")
    src, so = d / "stop.hip", d / "stop.so"
    src.write_text(SOURCE)
    subprocess.run([B.HIPCC, "--offload-host-only", "-O1", "-std=c++17", "-fPIC", "-shared", "-I", B.CSRC, str(src),
                    "-o", str(so)], check=True, capture_output=True)
    return C.CDLL(str(so))


@pytest.mark.parametrize("it", [0, 1, 2, 63, 1000, 2 ** 31 - 2])
def test_waves_of_the_launch_that_stops_the_solve_decide_alike(word, it):
    """Block 0 stores the word while waves of other blocks may not have read it
    yet: every interleaving of four waves' reads with the store leaves them all
    in the launch, and all launches after it end at their start."""
    words = (word.running(), word.stop_word(it))
    for reads in itertools.product(words, repeat=4):
        assert [word.past(it, w) for w in reads] == [0, 0, 0, 0]
    assert word.past(it + 1, word.stop_word(it))
    assert word.stop_word(it) not in (word.running(), word.at_start())


def test_no_iteration_runs_after_a_start_that_passes(word):
    assert word.past(0, word.at_start()) and not word.past(2 ** 31 - 2, word.running())
