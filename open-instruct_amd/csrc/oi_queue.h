// Which tile ids a launch of resident workgroups hands out, and whose they are.  Kept apart and free of device code so that
// every id's being handed out once can be checked on the host.
#pragma once
#include <cstdint>

#ifdef __HIPCC__
#define OI_QUEUE_FN __host__ __device__ __forceinline__
#else
#define OI_QUEUE_FN inline
#endif

// XCD-aware tile order.  Consecutive workgroup ids go round-robin to the 8 XCDs, each with its own
// L2.  The tiles of a launch are numbered in bands of 8 rows, n outermost inside a band, so that 32
// consecutive numbers are an 8 (m) x 4 (n) super-tile (wider where there are fewer than 8 rows); the ids
// of an XCD come in runs of 32 such numbers, which its 32 workgroups share operand slabs of in that L2,
// and the 8 XCDs take neighbouring runs along n.  The sweep over n completes before m advances: the chip
// as a whole then works on one slab of A (the larger operand: lm_head rows, dZ rows) at a time, which
// stays in the memory-side cache while every n tile passes over it, instead of streaming all of A from
// HBM once per n super-tile.  Measured: +4 to +7 % on every shape of the lm_head path (the kernel runs at
// the chip's power limit, and HBM traffic costs power).  Every number is a tile, whatever the counts, and the
// numbers past the last whole 256 are dealt out evenly: runs of 32 would leave whole XCDs to take tiles from
// the others' queues, out of the runs that share slabs.  d_hidden of 7648 rows (480 tiles, 4096 x 128256): 7.03 ms in
// runs of 32, 6.61 evenly; scoring pass of 1432 rows 1.258 -> 1.223 ms.  Ids without a number give one >= items.
OI_QUEUE_FN uint32_t item_of_pid(uint32_t pid, uint32_t items) {
    const uint32_t xcd = pid & 7, local = pid >> 3, first = (local >> 5) * 256, at = local & 31;
    const uint32_t left = first < items ? items - first : 0, run = left >= 256 ? 32 : (left + 7) / 8;
    return at < run ? first + xcd * run + at : 0xffffffffu;
}
OI_QUEUE_FN void tile_of_item(uint32_t item, uint32_t tiles_m, uint32_t tiles_n, int64_t* tm, int64_t* tn) {
    const uint32_t band = item / (8 * tiles_n), in_band = item - band * 8 * tiles_n;
    const uint32_t left = tiles_m - band * 8, rows = left < 8 ? left : 8;
    const uint32_t col = in_band / rows;
    *tm = band * 8 + (in_band - col * rows);
    *tn = col;
}
// number of ids to enumerate (whole runs for every XCD, a multiple of 256), and those of an XCD that may have an item
OI_QUEUE_FN int64_t pids_for_items(int64_t items) { return (items + 255) / 256 * 256; }
OI_QUEUE_FN uint32_t locals_for_items(uint32_t items) { return items / 256 * 32 + (items % 256 + 7) / 8; }
// Workgroups of a queue-driven launch on a device of `cus` CUs: one per CU (each takes a whole CU's LDS), at most `per_xcd`
// (0: any number) on an XCD, no more than there are ids, and always whole eighths, so that every XCD gets the same number.
inline uint32_t resident_workgroups(int64_t items, int64_t cus, uint32_t per_xcd) {
    int64_t most = (cus + 7) / 8;
    if (per_xcd && per_xcd < most) most = per_xcd;
    const int64_t ids = pids_for_items(items) >> 3;
    return (uint32_t)((ids < most ? ids : most) * 8);
}
// ids of every queue that the workgroups of such a launch begin with, each with that of its own number.  One number for all
// queues: counted queue by queue, for launches of any number of workgroups, steps and passes of 1400 rows and more take 0.2
// to 0.4 % longer (22942 rows x 4096 x 128256 53.10 ms, 53.30).
OI_QUEUE_FN uint32_t ids_begun(uint32_t workgroups) { return workgroups >> 3; }
