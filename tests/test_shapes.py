"""Sizes that follow from the tile size and the tables' limits (anuga_core_amd/
csrc/de_shape.h), compiled for the host."""

import ctypes as C
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "anuga_core_amd", "csrc")
SOURCE = r"""
#include "de_shape.h"
extern "C" int hash_slots(int n) { return de_hash_slots(n); }
extern "C" uint64_t hash_bits(uint64_t a, uint64_t b) { return de_hash_bits(a, b); }
extern "C" int edge_lds(int b, int h, int n) { return de_edge_lds(b, h, n); }
extern "C" int edge_lds_static(int b) { return de_edge_lds_static(b); }
extern "C" int tables_fit(int b, int h, int n) { return de_tables_fit(b, h, n); }
extern "C" int wave_passes(int w, int n) { return de_wave_passes(w, n); }
extern "C" int wave_chunk(int v, int j, int w, int n) { return de_wave_chunk(v, j, w, n); }
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("shape")
    src, so = tmp / "shape.cpp", tmp / "libshape.so"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I" + CSRC, "-o", str(so),
                    str(src)], check=True)
    lib = C.CDLL(str(so))
    lib.hash_bits.restype = C.c_uint64
    return lib


def test_a_probe_reaches_a_free_slot(lib):
    """Limits of 510 cells (512-triangle tiles), 384 and 520 nodes among them:
    four times these are no powers of two, and of 4 x 520 slots a mask reaches
    64, fewer than the keys, so that a probe would not end."""
    for n in range(1, 1023):
        s = lib.hash_slots(n)
        reached = {i & (s - 1) for i in range(s)}
        assert len(reached) == s and 2 * n <= s <= max(4 * n, 2)


def test_every_chunk_is_formed_once(lib):
    """Workgroups of any number of waves, three, five and six (192, 320 and 384
    threads) among them, which do not divide the reduction's 32 chunks."""
    for chunks in (1, 31, 32, 33):
        for waves in range(1, 17):
            got = [lib.wave_chunk(v, j, waves, chunks) for v in range(waves)
                   for j in range(lib.wave_passes(waves, chunks))]
            assert sorted(c for c in got if c >= 0) == list(range(chunks))


@pytest.mark.parametrize("block", [128, 192, 256, 320, 384, 512])
def test_tables_whose_lds_does_not_fit_are_left_out(lib, block):
    """Tiles of 512 triangles with 64 halo edges and 330 nodes would take 66
    KB; the default tiles fit at every limit of the tables."""
    for hecap in range(16, 257, 16):
        for ncap in range(0, 385, 2):
            fit = lib.tables_fit(block, hecap, ncap)
            both, bare = (lib.edge_lds(block, hecap, n) + lib.edge_lds_static(block)
                          for n in (ncap, 0))
            if ncap and both <= 65536:
                assert fit == 2
            else:
                assert fit == (bare <= 65536)
            if block <= 256:
                assert fit == (2 if ncap else 1)
    assert lib.tables_fit(512, 64, 330) == 1 and lib.tables_fit(512, 256, 0) == 0
    # the LDS that the kernel lays out: cells under the edge values, halo edge
    # values, depths and beds; nodes on 16 B and the triangles' node words
    assert lib.edge_lds(256, 64, 0) == 8 * (12 * 256 + 4 * 64 + 2 * 256)
    assert lib.edge_lds(256, 64, 180) == lib.edge_lds(256, 64, 0) + 16 * 180 + 4 * 256


@pytest.mark.parametrize("x0,dx", [(0.0, 1.0), (0.0, 10.0), (0.0, 0.1), (-3.0, 2.0 ** -7),
                                   (500000.0, 25.0), (0.0, 1.0 / 3.0)])
def test_hashes_of_grid_points_spread(lib, x0, dx):
    """384 points of a grid, round coordinates among them, over 1024 slots
    occupy about as many as random ones (320 expected, 9 the deviation)."""
    x = x0 + dx * np.arange(16.0)
    y = 2.0 * x0 + dx * np.arange(24.0)
    p = np.stack(np.meshgrid(x, y), axis=-1).reshape(-1, 2).view(np.uint64).tolist()
    slots = {(lib.hash_bits(C.c_uint64(a), C.c_uint64(b)) >> 32) & 1023 for a, b in p}
    assert len(slots) > 320 - 6 * 9
