"""Work of more workgroups than one launch takes goes in runs: each workgroup
once, in order, fewer than 2^32 threads a launch, starting at multiples of 8."""
import ctypes as C

import pytest

from hostlib import host_lib

CODE = """
#include "common.hpp"
extern "C" int runs(unsigned long long blocks, unsigned threads, int cap, unsigned* first, unsigned* count) {
  int k = 0;
  hcg::launch_runs(blocks, threads, [&](uint32_t f, uint32_t c) {
    if (k < cap) first[k] = f, count[k] = c;
    ++k;
  });
  return k;
}
"""


@pytest.mark.parametrize("threads", [64, 256, 512, 1024])
def test_runs_cover_the_blocks(tmp_path, threads):
    lib = host_lib(tmp_path, CODE)
    most = (2 ** 32 - 1) // threads // 8 * 8
    cells = [32768, 46341, 65535]
    counts = [0, 1, 7, 1000, most - 1, most, most + 1, most + 8, 3 * most + 5, 2 ** 31 - 2]
    counts += [((s + 15) // 16) * ((s + r - 1) // r) for s in cells for r in (1, 2, 4)]
    for blocks in counts:
        first, count = (C.c_uint * 4096)(), (C.c_uint * 4096)()
        k = lib.runs(C.c_uint64(blocks), threads, 4096, first, count)
        assert k == -(-blocks // most)
        at = 0
        for f, c in zip(first[:k], count[:k]):
            assert f == at and f % 8 == 0 and 0 < c and c * threads < 2 ** 32
            at += c
        assert at == blocks
