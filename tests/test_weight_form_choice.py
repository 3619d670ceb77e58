"""Which form of a weight a product takes, by a weight that is kept laid out and by one that is laid out for every product."""
import ctypes

import pytest

from intrasm_engine_amd import _lib

EACH_CALL = 0x10
NO_SPILL = (0, 0, 0)


def _choose(kinds, m, k, n, density, phases):
    return _lib.load().iex_form_choose(kinds, m, k, n, int(m * k * density), (ctypes.c_int * 3)(*phases))


# (phases of spill as measured on uniformly random patterns of that density)
@pytest.mark.parametrize("m,k,n,density,phases,kept,each_call", [
    (2752, 1024, 64, 0.5, NO_SPILL, 0, -1),                       # 14 us laid out and multiplied, 10 from the CSR arrays
    (4096, 11008, 64, 0.1, (1283, 1233, 1186), 0, -1),            # 45, 24.5
    (2752, 1024, 256, 0.1, (86, 86, 86), 0, -1),                  # 14.2, 12.0
    (11008, 4096, 512, 0.5, NO_SPILL, 128, 0),                    # two-of-four 94, dense 80
    (11008, 4096, 1024, 0.5, NO_SPILL, 192, 0),                   # 111, 106
    (11008, 4096, 2048, 0.5, NO_SPILL, 192, 192),                 # 167, 187
    (4096, 4096, 8192, 0.5, NO_SPILL, 256, 256),                  # 171, 208
    (4096, 4096, 16, 0.5, NO_SPILL, 0, 0),                        # dense 27, CSR 38
    (256, 512, 1024, 0.2, (8, 8, 8), 0, 0),                       # so small a weight keeps a call's kind, and bits
    (257, 512, 1024, 0.2, (8, 8, 8), 0, -1),
])
def test_laying_out_counts_where_it_happens_in_every_call(m, k, n, density, phases, kept, each_call):
    assert _choose(15, m, k, n, density, phases) == kept
    assert _choose(15 | EACH_CALL, m, k, n, density, phases) == each_call


def test_only_the_kinds_that_are_offered():
    assert _choose(EACH_CALL, 4096, 4096, 8192, 0.5, NO_SPILL) == -1
    assert _choose(4 | EACH_CALL, 4096, 4096, 8192, 0.5, NO_SPILL) == 192
    assert _choose(1 | EACH_CALL, 4096, 4096, 8192, 0.5, NO_SPILL) == 0
