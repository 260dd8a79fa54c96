// Sizes that follow from the tile size and the tables' limits, for the
// kernels, the host and CPU tests.
#pragma once

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

// A workgroup of `waves` waves forms `chunks` chunks in de_wave_passes passes:
// the chunk of a wave in pass j, or -1 in the last pass where there is none.
DE_SHAPE_FN int de_wave_passes(int waves, int chunks) { return (chunks + waves - 1) / waves; }
DE_SHAPE_FN int de_wave_chunk(int wave, int j, int waves, int chunks)
{
    const int c = wave + j * waves;
    return chunks % waves == 0 || c < chunks ? c : -1;
}
