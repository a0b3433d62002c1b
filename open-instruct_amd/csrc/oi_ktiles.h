// Where a loader of a tile product stands along k.  Kept apart and free of device code so that k ranges past 32 bits
// can be checked on the host: one workgroup walks through such a range for most of a minute.
#pragma once
#include <cstdint>

#ifdef __HIP_DEVICE_COMPILE__
#define OI_KTILES_FN __device__ __forceinline__
#elif defined(__HIPCC__)
#define OI_KTILES_FN __host__ __device__ __forceinline__
#else
#define OI_KTILES_FN inline
#endif

// k-tiles of DEPTH rows each; counts of tiles fit 32 bits where counts of rows do not.
template <int DEPTH>
struct KTiles {
    int left;      // from this k-tile on, negated: -1 at the last one, 0 and up past it
    int live;      // all ones, or 0 past the last k-tile
    int last_row;  // of the last k-tile: rows behind it do not exist

    OI_KTILES_FN KTiles(int ktiles, int64_t k_valid) : left(-ktiles), live(-1) {
        const int64_t rows = k_valid - (int64_t)(ktiles - 1) * DEPTH;
        last_row = (int)(rows >= DEPTH ? DEPTH : rows > 1 ? rows : 1) - 1;
    }
    OI_KTILES_FN void next() {
        ++left;
#ifdef __HIP_DEVICE_COMPILE__
        // in assembly, or the compiler makes a compare of it whose result it puts into a vector register
        asm("s_ashr_i32 %0, %1, 31" : "=s"(live) : "s"(left) : "scc");
#else
        live = left < 0 ? -1 : 0;
#endif
    }
    // bytes to this k-tile from the one before, which is this one too past the last
    OI_KTILES_FN int64_t step(int64_t bytes) const { return bytes & (int64_t)live; }
    // the last k-tile, whose rows may end early, and what follows
    OI_KTILES_FN bool ending() const { return left >= -1; }
    OI_KTILES_FN int end_row() const { return left == -1 ? last_row : DEPTH - 1; }
};
