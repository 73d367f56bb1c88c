"""The rule that links a seed to an earlier one of its run (spaced_link,
csrc/extend.hpp), compiled for the host: against a plain search over small
tables of seeds, and at the largest genome the matcher takes (2^31 - 1 bases),
where one seed length past a reversed seed of the last window lies the word of
an empty position.  No GPU test can hold that genome."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mauve-py_amd", "csrc")
EMPTY, REV = 0xFFFFFFFF, 0x80000000

SRC = r"""
#include "extend.hpp"
// the words of positions [lo, lo + n)
extern "C" uint32_t link_of(uint32_t p, uint32_t S, const uint32_t *words, uint32_t lo, uint32_t n)
{
    return mh::spaced_link(p, S, [=](uint32_t x) { return x - lo < n ? words[x - lo] : 0xDEADBEEFu; });
}
"""


@pytest.fixture(scope="module")
def link(tmp_path_factory):
    d = tmp_path_factory.mktemp("link")
    (d / "link.cpp").write_text(SRC)
    so = str(d / "link.so")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", CSRC, str(d / "link.cpp"), "-o", so])
    f = ctypes.CDLL(so).link_of
    f.restype = ctypes.c_uint32
    f.argtypes = [ctypes.c_uint32, ctypes.c_uint32, ctypes.c_void_p, ctypes.c_uint32, ctypes.c_uint32]
    return lambda p, S, words, lo=0: f(p, S, words.ctypes.data, lo, len(words))


@pytest.mark.parametrize("S", [1, 5, 19])
def test_link_is_the_furthest_seed_of_the_diagonal(link, S):
    rng = np.random.default_rng(S)
    for rev in (0, REV):
        L = 60
        words = np.full(L, EMPTY, np.uint32)
        for p in np.nonzero(rng.random(L) < 0.6)[0]:
            d = int(rng.integers(0, 3))          # one of three diagonals
            words[p] = (100 - p + d if rev else p + d) | rev
        for p in np.nonzero(words != EMPTY)[0]:
            q = int(words[p]) & 0x7FFFFFFF
            want = int(p)
            for t in range(1, min(S, int(p)) + 1):
                w = q + t if rev else q - t
                if w >= 0 and words[p - t] == (w | rev):
                    want = int(p) - t
            assert link(int(p), S, words) == want


@pytest.mark.parametrize("S", [11, 23, 31])
def test_last_window_of_the_largest_genome_links_to_no_empty_position(link, S):
    q = (1 << 31) - 1 - S                     # the last window of 2^31 - 1 bases
    words = np.full(S + 1, EMPTY, np.uint32)
    words[S] = q | REV
    assert link(S, S, words) == S
    words[1] = (q + S - 1) | REV              # the furthest window there can be
    assert link(S, S, words) == 1
    # and far into genome 0
    lo = (1 << 31) - 200
    assert link(lo + S, S, words, lo) == lo + 1
