// Sizes that follow from the tile size and the tables' limits, for the
// kernels, the host and CPU tests.
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#define DE_SHAPE_FN __host__ __device__ constexpr
#else
#define DE_SHAPE_FN constexpr
#endif

// Slots of an open-addressing table of at most n keys: a power of two, so that
// a mask reaches every slot, and at least 2 n, so that a probe meets a free one.
DE_SHAPE_FN int de_hash_slots(int n)
{
    int s = 2;
    while (s < 2 * n) s *= 2;
    return s;
}

// Hash of two doubles' bits, to be used from bit 32 up. Round coordinates
// differ in a few high bits only, and a product carries bits upwards: without
// the shifts, those of a grid have the low bits of their products in common
// and crowd into few slots.
DE_SHAPE_FN uint64_t de_hash_bits(uint64_t a, uint64_t b)
{
    uint64_t h = (a ^ (a >> 32)) * 0x9e3779b97f4a7c15ull + (b ^ (b >> 29)) * 0xc2b2ae3d27d4eb4full;
    h ^= h >> 32;
    return h * 0x9e3779b97f4a7c15ull;
}

// A workgroup of `waves` waves forms `chunks` chunks in de_wave_passes passes:
// the chunk of a wave in pass j, or -1 in the last pass where there is none.
DE_SHAPE_FN int de_wave_passes(int waves, int chunks) { return (chunks + waves - 1) / waves; }
DE_SHAPE_FN int de_wave_chunk(int wave, int j, int waves, int chunks)
{
    const int c = wave + j * waves;
    return chunks % waves == 0 || c < chunks ? c : -1;
}

// LDS of a workgroup of a fused kernel: at most 64 KB.
#define DE_LDS_MAX 65536

// Bytes of LDS that de_xflux_e asks for at its launch, with tiles of `block`
// triangles, at most hecap halo edges and ncap nodes a tile (0: no nodes), and
// those that it has of its own (three values of each wave).
DE_SHAPE_FN int de_edge_lds(int block, int hecap, int ncap)
{
    return 8 * (14 * block + 4 * hecap) + (ncap ? 16 * ncap + 4 * block : 0);
}
DE_SHAPE_FN int de_edge_lds_static(int block) { return 3 * 8 * (block / 64); }

// What of the tables fits: 2 with the nodes, 1 without them, 0 nothing.
DE_SHAPE_FN int de_tables_fit(int block, int hecap, int ncap)
{
    const int most = DE_LDS_MAX - de_edge_lds_static(block);
    return ncap && de_edge_lds(block, hecap, ncap) <= most ? 2
           : de_edge_lds(block, hecap, 0) <= most          ? 1
                                                           : 0;
}
