"""Sizes that follow from the tile size and the tables' limits (anuga_core_amd/
csrc/de_shape.h), compiled for the host."""

import ctypes as C
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "anuga_core_amd", "csrc")
SOURCE = r"""
#include "de_shape.h"
extern "C" int hash_slots(int n) { return de_hash_slots(n); }
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("shape")
    src, so = tmp / "shape.cpp", tmp / "libshape.so"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I" + CSRC, "-o", str(so),
                    str(src)], check=True)
    return C.CDLL(str(so))


def test_a_probe_reaches_a_free_slot(lib):
    """Limits of 510 cells (512-triangle tiles), 384 and 520 nodes among them:
    four times these are no powers of two, and of 4 x 520 slots a mask reaches
    64, fewer than the keys, so that a probe would not end."""
    for n in range(1, 1023):
        s = lib.hash_slots(n)
        reached = {i & (s - 1) for i in range(s)}
        assert len(reached) == s and 2 * n <= s <= max(4 * n, 2)
