"""The contraction kernels read whole 16-channel blocks of the sorted channel
values.  For every channel count and kind of weight, the rows that they read from
the last sample's block on have to lie within the padded buffer."""
import ctypes as C

import pytest

from hcgrid_amd import capi
from hostlib import host_lib

CODE = """
#include "mfma_job.hpp"
extern "C" unsigned long long rows_read(unsigned nchan, unsigned kind) { return hcg::value_rows_read(nchan, kind); }
extern "C" unsigned nb_of(unsigned nchan, unsigned kind) { return hcg::kFormNb[hcg::mfma_form(nchan, kind)]; }
"""


@pytest.mark.parametrize("kind", range(6))
def test_rows_read_are_in_the_buffer(tmp_path, kind):
    lib = host_lib(tmp_path, CODE)
    lib.rows_read.restype = C.c_uint64
    padded = capi.load().hcg_channels_padded_len
    for nchan in list(range(1, 1200)) + [4095, 4096, 4097, 65535]:
        nb, rows = lib.nb_of(nchan, kind), lib.rows_read(nchan, kind)
        assert rows >= nchan and (nb == 0 or 16 * nb >= nchan)
        for n in (1, 8, 31, 32, 33, 1000, 1024):
            held = (padded(n) // 8 - (n - 1) // 8) * nchan
            assert rows <= held, (nchan, n, nb, rows, held)
