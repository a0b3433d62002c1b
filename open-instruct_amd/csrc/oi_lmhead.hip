// Fused lm_head projection + per-token logprob / entropy for gfx950.  The logits stay on the chip, except where the
// forward leaves them for its backward (lmhead_dz_kept_kernel).
//
// One bf16 MFMA main loop, C[m, n] = sum_k a(m, k) * b(n, k), serves four kernels that differ in
// what they do with the fp32 tile and in the memory order of their operands (k-contiguous: the k
// values of a row lie together; k-major: the rows of a k value lie together):
//
//   forward   a = W [V, H],  b = hidden [N, H]   both k-contiguous -> online (max, sum-exp,
//             sum exp*z) per token, merged over the vocabulary tiles of a work item
//   dz        a = W,         b = hidden          -> dZ = g * (onehot - softmax), bf16 [N, Vc]
//   d_hidden  a = W [Vc, H] k-major,      b = dZ [N, Vc] k-contiguous -> fp32 accumulate over chunks
//   d_weight  a = hidden [N, H] k-major,  b = dZ [N, Vc] k-major      -> bf16 rows of dW
//
// so the backward reads W, hidden and dZ where they lie: no transposed copies.
//
// Tile: 256 x 256 x 64 per 512-thread workgroup, 8 waves as 4 (m) x 2 (n), each wave 64 x 128 =
// 4 x 8 MFMA 16x16x32 accumulators.  With vocabulary as the m dim a lane's accumulators of a
// column of tiles belong to ONE token, so the softmax statistics reduce inside the lane.  LDS: a ring of five 32 KB
// operand slots (k-tiles of A and of B) filled by direct global->LDS loads of whole 128-byte line segments; the 16-byte chunks of a row are
// XOR-permuted so that fragment reads (16-byte reads of a k-contiguous image, transposing 8-byte
// reads of a k-major image) stay free of bank conflicts.  A launch is one resident workgroup per
// CU that draws tile ids from per-XCD counters.
#include "oi_common.h"
#include "oi_grpo_math.h"
#include "oi_ktiles.h"
#include "oi_queue.h"

#include <type_traits>

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int BM = 256, BN = 256, BK = 64;
constexpr int NTHREADS = 512;
constexpr int TILE_ELEMS = BM * BK;             // one operand tile in LDS, rows of 128 B, unpadded
constexpr int STAGE_STRIDE = 256 + 8;           // bf16 per row of the dZ staging tile
constexpr int LDS_ELEMS = 5 * TILE_ELEMS;       // 163840 B: the five-slot operand ring, all of a CU's LDS
static_assert(256 * STAGE_STRIDE <= LDS_ELEMS, "the dZ staging tile must fit");

// A workgroup's tile is 256 (m) x 32 NJ (n): each wave 64 x 16 NJ, NJ column tiles.  NJ is 8, or less for token rows: for the
// last tile of a forward (tile_width), for all tiles of a forward or a d_hidden product of few rows (fwd_tiles, plan_rows:
// 6) and for a forward's last round (4).
constexpr int WIDE = 8;
template <int NJ = WIDE>
using AccTile = f32x4[4][NJ];

// Work queue.  A launch of the tile kernels is one workgroup per CU (the LDS ring leaves room for
// no second one) that stays for the whole launch and draws tile ids from a counter, rather than
// one short-lived workgroup per tile.  There is one counter per XCD (workgroup b is taken to run
// on XCD b mod 8, as the tile order assumes), so the ids an XCD draws are the ones item_of_pid
// maps onto shared operand slabs; a wrong guess costs cache hits, never correctness.  The XCDs do
// not finish their shares together (measured on the forward: 1.7 ms apart in an 18 ms launch), so
// a workgroup whose own queue has run dry goes on with the queues of the other XCDs: the launch then ends within one work
// item for all of them.  The next id is requested
// before the current tile is computed and handed to the other waves through one LDS word
// afterwards.  `counters` are 8 zeroed words; every workgroup leaves each of them raised past the
// number of ids at most once.
//
// A draw takes about 3 us when many workgroups draw at once.  So a workgroup begins with the id of its own number, without
// a draw (the counters count from behind those), a launch without items draws none, and a workgroup whose queue is empty
// looks at the other counters side by side instead of drawing from one after the other to find them empty as well (at
// the end of every launch).  A forward that finds no rows 49 -> 5 us; 4096 x 100352, us before and after: forward of 100
// rows 202, 188, of 256 240, 218, of 268 332, 306; d_hidden of 100 rows 182, 175; steps of 22942 rows 0.5 % shorter.
constexpr int QUEUE_WORDS = 8;
constexpr int FWD_QUEUE_WORDS = 2 * QUEUE_WORDS;  // the forward hands out its long and its short items from two sets of queues
// threadIdx.x as a value the optimiser cannot trace: everything derived from it (fragment and
// epilogue addresses) is then recomputed per tile instead of being hoisted out of the tile loop,
// where it would stay live through the main loop and push accumulators into scratch
__device__ __forceinline__ int opaque_tid() {
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
}
__device__ __forceinline__ void lds_barrier();
struct ItemQueue {
    static constexpr uint32_t NONE = 0xffffffffu;
    uint32_t* counters;
    // the word sits in the fifth ring slot, which the main loop first writes after its first barrier
    volatile uint32_t* mailbox;
    uint32_t items, locals, xcd, begun;
    // thread 0 only: the queues of XCDs xcd .. xcd + dry - 1 (mod 8) are known to be empty, `drawn` came from
    // the queue of XCD xcd + dry, `next` is the id it stands for
    uint32_t dry, drawn, next;

    // begins: the workgroups take the ids of their own numbers first
    __device__ __forceinline__ ItemQueue(uint32_t* counters_, uint32_t items_, uint32_t locals_, uint16_t* lds, bool begins)
        : counters(counters_),
          mailbox(reinterpret_cast<volatile uint32_t*>(lds + 4 * BM * BK)),
          items(items_),
          locals(locals_),  // ids per queue
          xcd(blockIdx.x & 7),
          begun(begins ? ids_begun(gridDim.x) : 0),
          dry(counters_ ? 0 : 8),  // without counters there is nothing to draw
          drawn(0),
          next(NONE) {
        // a kernel may run several queues one after the other over the same word: every wave must have
        // read the previous one's last value before thread 0 writes this one's first
        __syncthreads();
    }
    // asks for an id.  (The addition waits for the counter.  Left to settle(), with the draw in flight until then, it changes
    // nothing: steps of 268 and 2400 rows 1.001x, frozen-head DPO of 2950 rows 0.990 to 0.994x.)
    __device__ __forceinline__ void request() {
        if (threadIdx.x == 0 && dry < 8) drawn = draw();
    }
    __device__ __forceinline__ uint32_t draw() { return begun + atomicAdd(&counters[(xcd + dry) & 7], 1u); }
    __device__ __forceinline__ void settle() {
        if (threadIdx.x != 0) return;
        next = NONE;
        while (dry < 8) {
            if (drawn < locals) {
                next = drawn * 8 + ((xcd + dry) & 7);
                return;
            }
            // counters only grow: one that reads past its ids is empty
            uint32_t at[8];
#pragma unroll
            for (int q = 0; q < 8; ++q)
                at[q] = __hip_atomic_load(&counters[(xcd + q) & 7], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            uint32_t with_ids = 8;
#pragma unroll
            for (int q = 7; q > 0; --q)
                if ((uint32_t)q > dry && begun + at[q] < locals) with_ids = q;
            dry = with_ids;
            if (dry < 8) drawn = draw();
        }
    }
    // the settled id, for every thread.  The LDS must be free.
    __device__ __forceinline__ uint32_t take() {
        lds_barrier();
        if (threadIdx.x == 0) *mailbox = next;
        lds_barrier();
        return __builtin_amdgcn_readfirstlane(*mailbox);
    }
    // its item; ids without one are passed over
    __device__ __forceinline__ uint32_t take_item() {
        for (;;) {
            const uint32_t pid = take();
            if (pid == NONE) return NONE;
            const uint32_t item = item_of_pid(pid, items);
            if (item < items) return item;
            request();
            settle();
        }
    }
};
// begins: these are the kernel's first items.  (Items that are to fill the end of others' launch time must be drawn: a
// workgroup that is late would have its own left to do.)
template <class Body>
__device__ __forceinline__ void for_each_id(uint32_t* __restrict__ counters, uint32_t locals, uint16_t* lds, bool begins,
                                            Body&& body) {
    if (locals == 0) return;
    ItemQueue queue(counters, 0, locals, lds, begins);
    uint32_t pid = blockIdx.x;
    if (!begins) {
        queue.request();
        queue.settle();
        pid = queue.take();
    }
    while (pid != ItemQueue::NONE) {
        queue.request();
        body(pid);
        queue.settle();
        pid = queue.take();
    }
}
template <class Body>
__device__ __forceinline__ void for_each_tile(uint32_t* __restrict__ counters, int64_t tiles_m, int64_t tiles_n,
                                              uint16_t* lds, Body&& body) {
    const uint32_t items = (uint32_t)(tiles_m * tiles_n);
    for_each_id(counters, locals_for_items(items), lds, true, [&](uint32_t pid) {
        const uint32_t item = item_of_pid(pid, items);
        if (item >= items) return;
        int64_t tm, tn;
        tile_of_item(item, (uint32_t)tiles_m, (uint32_t)tiles_n, &tm, &tn);
        body(tm, tn);
    });
}
// stand-alone products have no workspace for counters: one workgroup per id
inline unsigned grid_for_tiles(int64_t tiles_m, int64_t tiles_n) { return (unsigned)pids_for_items(tiles_m * tiles_n); }

// LDS tile layout: row r of an operand tile holds its 64 k-values as eight 16-byte chunks; chunk c
// is stored at position c ^ swz(r).  With that permutation the 16-byte fragment reads of 16
// consecutive rows at one logical chunk fall on distinct banks, and the rows stay unpadded, which
// the direct global->LDS loads need (a wave's 64 lanes fill 1 KB of consecutive LDS).
__device__ __forceinline__ int swz(int row) { return (row >> 1) & 7; }

#define OI_LDS_PTR(p) ((__attribute__((address_space(3))) void*)(p))
#define OI_GLOBAL_PTR(p) ((const __attribute__((address_space(1))) void*)(p))

// Wait until at most PENDING of this wave's global->LDS loads are still in flight, then meet the
// other waves.  A bare s_barrier (no fence) keeps the compiler from draining the loads that were
// issued for later k-tiles.
template <int PENDING>
__device__ __forceinline__ void wait_loads_and_barrier() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PENDING) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// Meets the other waves once this wave's LDS accesses are done.  __syncthreads() also waits for every global
// store and load of the wave, which in an epilogue is the round trip of its stores at each barrier.
// No pointer to a region that is handed over at a barrier is `__restrict__`: nothing but its own accesses would
// touch the region then, and a read whose value is first used in a branch behind the barrier is moved there.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// A count in device memory, in a scalar register: sizes and base addresses that follow from it then take no vector
// registers and no vector instructions in the main loops.
__device__ __forceinline__ int device_count(const int32_t* p) { return __builtin_amdgcn_readfirstlane(*p); }
// The same for 64-bit values that every lane holds alike
__device__ __forceinline__ int64_t scalar(int64_t v) {
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)((uint64_t)v >> 32));
    return (int64_t)(((uint64_t)hi << 32) | lo);
}
template <class T>
__device__ __forceinline__ const T* scalar(const T* p) {
    return reinterpret_cast<const T*>(scalar((int64_t)reinterpret_cast<uint64_t>(p)));
}

constexpr int SLOT_BYTES = TILE_ELEMS * 2;
constexpr int64_t MAX_LD = (int64_t)1 << 22;  // 255 rows * ld * 2 bytes must fit 32 bits

// One operand of a tile product, in either of two memory layouts.
//   k-contiguous (KM = false): element (row, k) at p[row * ld + k]; the tile takes rows
//     [r0, r0 + 256), rows at or past `extent` are clamped onto the last valid one.
//   k-major (KM = true): element (row, k) at p[k * ld + row]; the tile takes columns
//     [r0, r0 + 256) of every k row, 16-byte column chunks past `extent` (a multiple of 8) are
//     clamped onto the last valid chunk, k rows at or past `k_valid` onto the last valid row (the
//     other operand must hold zeros there).  This is the layout in which a matrix is its own
//     transpose operand: W [V, H] as the B operand of dZ * W, hidden [N, H] and dZ [N, V] as the
//     operands of dZ^T * hidden, with no transposed copies in memory.
// In both cases the results of clamped rows / columns are garbage that the epilogues discard.
struct Operand {
    const uint16_t* p;
    int64_t ld, r0, extent, k_valid;
};
__device__ __forceinline__ Operand scalar(const Operand& o) {
    return {scalar(o.p), o.ld, scalar(o.r0), scalar(o.extent), scalar(o.k_valid)};
}

typedef short v4i16 __attribute__((ext_vector_type(4)));

// acc = A_tile * B_tile^T over k in [0, K), K a multiple of 64.
//
// What bounds it is power: the chip runs these loops at its limit, so the clock follows the energy of an operation.
// Hence v_mfma_f32_16x16x32_bf16 and not 32x32x16, whose accumulators are read and written twice as often per
// operation: MFMAs alone on random data, eight waves per CU, sustain 2.01 against 1.74 PFLOP/s.  Products of
// 16384 x 8192 x 4096 in the four layouts, 1.31 -> 1.40 to 1.45 PFLOP/s; the vendor's kernel 1.38 to 1.42 (all on
// one box); policy-loss step of 22942 rows, 4096 x 128256: 55.8 -> 50.9 ms.
//
// Operand tiles reach the LDS by direct global->LDS loads (no VGPR staging, no LDS store
// instructions), whole 128-byte cache-line segments per 8 lanes.  The path from L2 into the LDS
// delivers a 64 KB k-tile to a CU in about the time the matrix pipe needs to multiply it, so the
// loads must be in flight all the time: issued in one burst per k-tile they back up in the load
// unit and hold the issuing waves (and their MFMAs) for twice the MFMA time of that k-step.
// Spreading them needs a free destination throughout the k-tile, which two full stages cannot give
// (the stage being read is the only candidate), hence a ring of FIVE operand slots of 32 KB, all
// of a CU's 160 KB: k-tile t reads A_t and B_t from two slots, A_(t+1) and B_(t+1) are landing in
// two more, A_(t+2) goes into the fifth at any time, and B_(t+2) takes A_t's slot once the barrier
// near the end of k-tile t has passed.  Every wave issues 4 + 4 loads of 1 KB per k-tile.
//
// LDS image of a k-contiguous operand tile: [256 rows][64 k], the eight 16-byte chunks of a row
// stored at c ^ swz(row); wave w loads rows [32 w, 32 w + 32); fragments are 16-byte reads.
// LDS image of a k-major operand tile: [64 k][256 columns], the 32 chunks of a k row stored at
// c ^ 4 (k & 3) ^ 2 (k / 8 & 1); wave w loads k rows [8 w, 8 w + 8); fragments come through the transposing read
// ds_read_b64_tr_b16: in a group of 16 lanes, lane s points at (k0 + s / 4, 4 columns from
// 4 (s % 4)) and lane i receives column i at k0 .. k0 + 3, which is the MFMA operand layout (row
// per lane, consecutive k per register).  The permutation puts the k rows that 32 lanes read together on
// different banks.
//
// The product comes in two halves: begin_loads requests the first two k-tiles into slots 0 .. 3 (all but the
// last block), gemm_loop waits for them and does the rest.  A caller may do other work in between that
// touches slot 4 only.
//
// Loader side: direct global->LDS loads in their buffer form, which takes a uniform 64-bit base (that of a k-tile) and
// a uniform byte offset in scalar registers and 32 bits per lane in one vector register.  (With 64-bit lane addresses
// the loads of a k-tile held 32 vector registers, and the compiler waited for every LDS access in flight before it used
// any fragment, because it counts such a load among them.)  Lanes clamp their offsets onto valid rows and columns, so
// no bounds are set.
//
// A loader stands at one k-tile and moves on to the next with advance().  Past the last one it stays there and all lanes
// fetch the same 16 bytes, into slots that nobody reads: the waits of the loop count loads, so one has to be issued and
// has to come back in its turn.  (A load outside the bounds of its buffer does not: it is counted off at once, ahead of
// older loads that are still under way.)  WALK: how it moves.  A k range that goes ROUND begins at k-tile `start`; a FAR
// one may be longer than a row pitch (stand-alone products whose rows are all one).
enum Walk { NEAR, ROUND, FAR };
template <bool KM, int LOADS, Walk WALK = NEAR>
struct Loader {
    static_assert(!KM || WALK != ROUND, "the others begin at the first k-tile");
    static_assert(LOADS == 4 || !KM, "k-major operands are whole tiles");
    static constexpr bool MOVES_BASE = KM || WALK == FAR;  // by more than 32 bits in all
    const char* base;   // of the operand, or of the k-tile
    uint32_t plus;      // bytes from there to the k-tile
    uint32_t plus_end;  // and to the end of the last one (ROUND)
    uint32_t off[LOADS];  // per-lane byte offsets of the loads
    int lds_wave;       // bytes to this wave's first load inside a slot
    KTiles<BK> k;
    static constexpr int LDS_BLOCK = KM ? 2 * 256 * 2 : 8 * BK * 2;  // bytes between the LDS destinations of loads

    __device__ __forceinline__ Loader(const Operand& op, int ktiles, int start, int lane, int wave) : k(ktiles, op.k_valid) {
        plus = WALK == ROUND ? (uint32_t)start * (BK * 2) : 0;
        plus_end = (uint32_t)ktiles * (BK * 2);
        if constexpr (!KM) {
            base = reinterpret_cast<const char*>(op.p + op.r0 * op.ld);
            const int last_row = (int)((op.extent - 1 - op.r0) < 255 ? (op.extent - 1 - op.r0) : 255);
#pragma unroll
            for (int b = 0; b < LOADS; ++b) {
                const int r = (wave * LOADS + b) * 8 + (lane >> 3);
                const int c = (lane & 7) ^ swz(r);
                off[b] = __umul24(r < last_row ? r : last_row, pitch(op)) + c * 16;
            }
            lds_wave = wave * LOADS * LDS_BLOCK;
        } else {
            base = reinterpret_cast<const char*>(op.p);
            set_rows(op, lane, wave);
            lds_wave = wave * LOADS * LDS_BLOCK;
        }
    }
    // at most 2^23; rows inside a tile are at most 255
    static __device__ __forceinline__ uint32_t pitch(const Operand& op) { return (uint32_t)(op.ld * 2); }
    // k-major: this k-tile's k rows, which may end inside it
    __device__ __forceinline__ void set_rows(const Operand& op, int lane, int wave) {
        const int last_k = k.end_row();
        const int r0 = (int)op.r0, extent = (int)op.extent;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int kk = wave * 8 + b * 2 + (lane >> 5);
            const int c = r0 + ((lane & 31) ^ (4 * (kk & 3)) ^ (2 * ((kk >> 3) & 1))) * 8;
            off[b] = (__umul24(kk < last_k ? kk : last_k, pitch(op)) + (uint32_t)((c + 8 <= extent ? c : extent - 8) * 2)) & k.live;
        }
    }
    __device__ __forceinline__ void advance(const Operand& op, int lane, int wave) {
        k.next();
        if constexpr (MOVES_BASE) base += k.step(KM ? BK * 2 * op.ld : BK * 2);
        else plus += BK * 2 & k.live;
        if constexpr (WALK == ROUND) plus = plus == plus_end ? 0 : plus;
        if constexpr (KM) {
            if (k.ending()) set_rows(op, lane, wave);
        } else if (!k.live) {
#pragma unroll
            for (int b = 0; b < LOADS; ++b) off[b] = 0;
        }
    }
};
// 16 bytes per lane from base + off (lane) + plus, 1 KB of consecutive LDS per wave
__device__ __forceinline__ void load_to_lds(const char* base, uint32_t off, uint32_t plus, char* to) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(__builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base), 0, -1, 0x00027000),
                                             OI_LDS_PTR(to), 16, off, plus, 0, 0);
}
// one 1 KB load: block b of this wave's share of an operand k-tile into the ring slot at byte offset `slot`
template <bool KM, int LOADS, Walk WALK>
__device__ __forceinline__ void load_block(const Loader<KM, LOADS, WALK>& L, int slot, int b, uint16_t* lds) {
    load_to_lds(L.base, L.off[b], L.plus, reinterpret_cast<char*>(lds) + slot + L.lds_wave + b * L.LDS_BLOCK);
}
// ring slots: A_t -> (2 t) mod 5, B_t -> (2 t + 1) mod 5
template <bool A_KM, bool B_KM, int NJ = WIDE, Walk WALK = NEAR>
__device__ __forceinline__ void begin_loads(const Operand& A_, const Operand& B_, int64_t K, uint16_t* lds,
                                            int start = 0) {
    const Operand A = scalar(A_), B = scalar(B_);
    const int tid = opaque_tid();
    // the wave index as a scalar: the LDS destinations of the loads (M0) then take no VALU work
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ktiles = __builtin_amdgcn_readfirstlane((int)(K / BK));
    constexpr int B_LOADS = NJ / 2;
    Loader<A_KM, 4, WALK> la(A, ktiles, start, lane, wave);
    Loader<B_KM, B_LOADS, WALK> lb(B, ktiles, start, lane, wave);
#pragma unroll
    for (int b = 0; b < 4; ++b) load_block(la, 0, b, lds);
#pragma unroll
    for (int b = 0; b < B_LOADS; ++b) load_block(lb, SLOT_BYTES, b, lds);
    la.advance(A, lane, wave);
    lb.advance(B, lane, wave);
#pragma unroll
    for (int b = 0; b < 4; ++b) load_block(la, 2 * SLOT_BYTES, b, lds);
#pragma unroll
    for (int b = 0; b < B_LOADS - 1; ++b) load_block(lb, 3 * SLOT_BYTES, b, lds);
}

// `__restrict__` here and in store_tile is what tells the compiler that the LDS accesses of these functions carry
// alias information; without any it waits for every global->LDS load in flight before each LDS access
// (d_weight of 3072 rows: 2.7 -> 4.9 ms).
template <bool A_KM, bool B_KM, Walk WALK = NEAR, int NJ>
__device__ __forceinline__ void gemm_loop(AccTile<NJ>& __restrict__ acc, const Operand& A_, const Operand& B_, int64_t K,
                                          uint16_t* lds, int start = 0) {
    const Operand A = scalar(A_), B = scalar(B_);
    const int tid = opaque_tid();
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave & 3, wn = wave >> 2;
    const int ktiles = __builtin_amdgcn_readfirstlane((int)(K / BK));
    constexpr int B_LOADS = NJ / 2;
    Loader<A_KM, 4, WALK> la(A, ktiles, start, lane, wave);        // at k-tile kt+2
    Loader<B_KM, B_LOADS, WALK> lb(B, ktiles, start, lane, wave);  // at k-tile kt+1 in group 0, kt+2 behind the barrier
    la.advance(A, lane, wave);
    la.advance(A, lane, wave);
    lb.advance(B, lane, wave);

#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    // consumer side: byte offsets of this lane's fragments inside a slot; a lane holds row lr of a 16-row
    // fragment at the k values 8 g .. 8 g + 7 of a k-step
    const int lr = lane & 15, g = lane >> 4;
    // k-contiguous image: the second k-step flips bit 2 of the stored chunk; rows 16 apart share the same
    // permutation
    const int pg = (g ^ swz(lr)) * 16;
    const int a_base = (wm * 64 + lr) * (BK * 2) + pg, b_base = (wn * 16 * NJ + lr) * (BK * 2) + pg;
    // k-major image: source lane lr of a 16-lane group points at k row (lr >> 2) of the group's 8 and at 4
    // columns from 4 (lr & 3) of the fragment's 16; fragments are two chunks apart, which flips the chunk bits
    // that the permutation reaches
    const int e4 = lr >> 2, km_row = (g * 8 + e4) * 512 + 8 * (lr & 1), km_perm = (4 * e4) ^ (2 * (g & 1));
    const int a_km = km_row + ((wm * 8 + ((lr & 3) >> 1)) ^ km_perm) * 16;
    const int b_km = km_row + ((wn * 16 + ((lr & 3) >> 1)) ^ km_perm) * 16;
    const char* ring = reinterpret_cast<const char*>(lds);
    auto read_tr = [&](int at) {
        // k rows 0 .. 3 and 4 .. 7 of the lane's 8
        const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) v4i16*)OI_LDS_PTR(const_cast<char*>(ring + at)));
        const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) v4i16*)OI_LDS_PTR(const_cast<char*>(ring + at + 4 * 512)));
        const short __attribute__((ext_vector_type(8))) both = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        return __builtin_bit_cast(bf16x8, both);
    };
    auto read_a = [&](int slot, int ks, int i) {
        if constexpr (A_KM) return read_tr(((slot + a_km) ^ (i * 32)) + ks * 32 * 512);
        else return *reinterpret_cast<const bf16x8*>(ring + slot + (a_base ^ (ks * 64)) + i * 16 * (BK * 2));
    };
    auto read_b = [&](int slot, int ks, int j) {
        if constexpr (B_KM) return read_tr(((slot + b_km) ^ (j * 32)) + ks * 32 * 512);
        else return *reinterpret_cast<const bf16x8*>(ring + slot + (b_base ^ (ks * 64)) + j * 16 * (BK * 2));
    };

    // A k-tile is two k-steps of 32, each NJ groups of four MFMAs: group u of the 2 NJ multiplies B fragment
    // u (u mod NJ of its k-step) with the four A fragments, up and down in turn, so that one operand of an MFMA is
    // always that of the one before (power is what limits the loop).  The fragment reads and the global->LDS loads (24
    // and 8 of a wide tile) stand one by one between the MFMAs.  Nothing may move across the scheduling barriers: loads
    // issued back to back hold up the wave's MFMA issue, and a fragment read issued ahead of the MFMAs before it would
    // be waited for together with the current fragments (a full LDS round trip with the matrix pipe idle).
    constexpr int GROUPS = 2 * NJ, BARRIER = NJ == 2 ? 2 : GROUPS * 3 / 4;
    bf16x8 a[2][4], b[GROUPS];
    // A_0 and B_0 must have landed.  The wait is for everything in flight: one that leaves the 7 younger loads and the
    // previous tile's stores under way measured the same (full batch within 0.3 %).
    wait_loads_and_barrier<0>();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        a[0][i] = read_a(0, 0, i);
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        b[j] = read_b(SLOT_BYTES, j / NJ, j % NJ);
        __builtin_amdgcn_sched_barrier(0);
    }

    // Fragments: at the start of a k-tile the A fragments of the first k-step and B fragments 0 .. 3 are there or under
    // way; the groups ahead of the barrier read the rest.  At the barrier k-tile kt+1 must have landed (its last load was
    // issued in group 0; the 4 younger ones may stay in flight) and this wave's reads of k-tile kt must be complete:
    // behind it A_kt's slot is overwritten with B_(kt+2), and the last quarter of the groups reads the first fragments of
    // k-tile kt+1 (past the last k-tile: of slots that hold nothing of use, for nobody).
    // The scalar work of a k-tile (loaders, slots) is spread as well: in one place it is a gap between MFMAs.
    // slots of A_kt, B_kt (being read), A_(kt+1), B_(kt+1), and the one that is free all along: takes A_(kt+2)
    int s_a = 0, s_b = SLOT_BYTES, s_a1 = 2 * SLOT_BYTES, s_b1 = 3 * SLOT_BYTES, s_a2 = 4 * SLOT_BYTES;
#pragma unroll 1
    for (int left = ktiles; left > 0; --left) {
#pragma unroll
        for (int u = 0; u < GROUPS; ++u) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int i = (u & 1) ? 3 - q : q, j = u % NJ;
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u / NJ][i], b[u], acc[i][j], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                if (u == BARRIER && q == 1) {
                    asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)" ::: "memory");
                    __builtin_amdgcn_s_barrier();
                    asm volatile("" ::: "memory");
                }
                // one of the loads, as evenly spread as the slot hand-over allows
                if (u == 0 && q == 1) load_block(lb, s_b1, B_LOADS - 1, lds);
                if constexpr (NJ == 8) {
                    if ((u == 2 || u == 5 || u == 7 || u == 10) && q == 1) load_block(la, s_a2, u == 2 ? 0 : u == 5 ? 1 : u == 7 ? 2 : 3, lds);
                    if ((u == 12 || u == 13) && q == 3) load_block(lb, s_a, u - 12, lds);
                    if (u == 15 && q == 1) load_block(lb, s_a, 2, lds);
                } else if constexpr (NJ == 6) {
                    if (u < 8 && u % 2 == 1 && q == 1) load_block(la, s_a2, u / 2, lds);
                    if (u >= 10 && q == 1) load_block(lb, s_a, u - 10, lds);
                } else if constexpr (NJ == 4) {
                    if (u >= 1 && u <= 4 && q == 1) load_block(la, s_a2, u - 1, lds);
                    if (u == 7 && q == 0) load_block(lb, s_a, 0, lds);
                } else {
                    if (u == 0 && q >= 2) load_block(la, s_a2, q - 2, lds);
                    if (u == 1 && (q == 0 || q == 2)) load_block(la, s_a2, 2 + q / 2, lds);
                }
                if (u == (NJ == 2 ? 2 : BARRIER - 1) && q == 2) la.advance(A, lane, wave);
                if (u == (NJ == 2 ? 1 : BARRIER - 2) && q == 2) lb.advance(B, lane, wave);
                // fragments
                if (u < BARRIER && u + 4 < GROUPS && q == 0) b[u + 4] = read_b(s_b, (u + 4) / NJ, (u + 4) % NJ);
                if constexpr (NJ >= 6) {
                    if (u >= NJ / 4 && u < NJ / 4 + 4 && q == 2) a[1][u - NJ / 4] = read_a(s_a, 1, u - NJ / 4);
                } else if constexpr (NJ == 4) {
                    if (u < 2 && q >= 2) a[1][2 * u + q - 2] = read_a(s_a, 1, 2 * u + q - 2);
                } else {
                    if (u == 0) a[1][q] = read_a(s_a, 1, q);
                }
                if constexpr (NJ == 2) {
                    if (u == 2 && q >= 1) a[0][q - 1] = read_a(s_a1, 0, q - 1);
                    if (u == 3 && q == 0) a[0][3] = read_a(s_a1, 0, 3);
                    if (u == 3 && q >= 1) b[q - 1] = read_b(s_b1, (q - 1) / NJ, (q - 1) % NJ);
                    if (u == 3 && q == 3) b[3] = read_b(s_b1, 1, 1);
                } else {
                    if (u == BARRIER && q >= 1) a[0][q - 1] = read_a(s_a1, 0, q - 1);
                    if (u == BARRIER + 1 && q == 0) a[0][3] = read_a(s_a1, 0, 3);
                    if (u == BARRIER + 1 && q >= 1 && q <= 2) b[q - 1] = read_b(s_b1, 0, q - 1);
                    if (u == (NJ >= 6 ? BARRIER + 2 : BARRIER + 1) && q == (NJ >= 6 ? 1 : 3)) b[2] = read_b(s_b1, 0, 2);
                    if (u == GROUPS - 1 && q == (NJ == 8 ? 0 : 3)) b[3] = read_b(s_b1, 0, 3);
                }
                if (u == GROUPS - 1 && q == 3) {
                    const int was_a = s_a, was_b = s_b;
                    s_a = s_a1;
                    s_b = s_b1;
                    s_a1 = s_a2;
                    s_b1 = was_a;
                    s_a2 = was_b;
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    // every wave is done reading before the caller reuses the LDS (epilogue staging, next tile)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
template <bool A_KM, bool B_KM, Walk WALK = NEAR>
__device__ __forceinline__ void gemm_tile(AccTile<>& acc, const Operand& A, const Operand& B, int64_t K, uint16_t* lds) {
    begin_loads<A_KM, B_KM, WIDE, WALK>(A, B, K, lds);
    gemm_loop<A_KM, B_KM, WALK>(acc, A, B, K, lds);
}
// both operands k-contiguous: C[m, n] = sum_k A[m0 + m, k] * B[n0 + n, k]
template <Walk WALK>
__device__ __forceinline__ void gemm_tile(AccTile<>& acc, const uint16_t* __restrict__ A, int64_t lda, int64_t m0,
                                          int64_t M, const uint16_t* __restrict__ B, int64_t ldb, int64_t n0,
                                          int64_t N, int64_t K, uint16_t* lds, int start) {
    const Operand a = {A, lda, m0, M, K}, b = {B, ldb, n0, N, K};
    begin_loads<false, false, WIDE, WALK>(a, b, K, lds, start);
    gemm_loop<false, false, WALK>(acc, a, b, K, lds, start);
}

// An MFMA leaves lane l with rows 4 (l / 16) .. + 3 of column l % 16 of a 16 x 16 tile (acc[i][j]: rows 16 i, columns
// 16 j of the wave's 64 x 16 NJ).  The epilogues take column groups of 32: swapping the odd quarters of the lanes of one
// column tile with the even ones of the next gives a lane one column and eight consecutive rows of every 16.
// Element (i, r) of lane `lane` of column group j is then
//   m (row, vocabulary in the logits kernels) = wm*64 + i*32 + (r/8)*16 + (lane/32)*8 + r%8
//   n (column, token in the logits kernels)   = wn*16*NJ + j*32 + lane%32
__device__ __forceinline__ void swap_quarters(const f32x4& x, const f32x4& y, f32x16& z, int r0) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const auto w = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, (float)x[e]),
                                                        __builtin_bit_cast(uint32_t, (float)y[e]), false, false);
        z[r0 + e] = __builtin_bit_cast(float, (uint32_t)w[0]);
        z[r0 + 4 + e] = __builtin_bit_cast(float, (uint32_t)w[1]);
    }
}
struct Columns {
    f32x16 z[2];  // not an array of floats: the search for the label's register would put that into memory
};
template <int NJ>
__device__ __forceinline__ Columns tile_columns(const AccTile<NJ>& acc, int j) {
    Columns c;
#pragma unroll
    for (int i = 0; i < 4; ++i) swap_quarters(acc[i][2 * j], acc[i][2 * j + 1], c.z[i >> 1], (i & 1) * 8);
    return c;
}
__device__ __forceinline__ int acc_row(int wm, int i, int r, int lane) {
    return wm * 64 + i * 32 + (r >> 3) * 16 + (lane >> 5) * 8 + (r & 7);
}
template <int NJ = WIDE>
__device__ __forceinline__ int acc_col(int wn, int j, int lane) { return wn * 16 * NJ + j * 32 + (lane & 31); }
// Width of the forward's tile of token rows from row0.  Where tiles may be narrow, the last one is as wide as the rows
// that are left need, in groups of 64: the loop is bound by the matrix cores, so products of rows that do not exist
// cost what others do.  The line between: a narrow tile gets ahead of the tiles that multiply the same W rows, and is
// worth that while an XCD's 4 MB L2 holds the 512 hidden_dim bytes of those rows and more, and while it is not one of
// too many (vocabulary 128256, kept logits, us with whole and with narrow tiles: 300 rows x 2048 276, 234; 300 x 4096
// 455, 386; 1900 x 3584 1513, 1477; 2940 x 4096 2445, 2387; 3900 x 6144 4666, 4590; across the line 900 x 8192 1691,
// 1719; 2940 x 8192 4605, 4675; 5000 x 4096 4003, 4024, exponentials; 5000 x 8192 7652, 7983).  With up to two tiles
// of rows there is little to be shared (300 x 8192 874, 851).  `rows` is all that the call has, selected or not: a
// choice on the device keeps the other widths' code in every call's kernel (2940 x 8192 0.5 % longer for it).
//
// The products behind it have tiles of one height only (plan_rows): among whole ones narrow ones gain nothing, as the
// pieces that tiles are cut into stop being alike (d_hidden of 268 rows 312, so 322).
inline bool narrow_tiles(int64_t rows, int64_t hdim) { return rows <= 2 * BN || (rows <= 16 * BN && hdim <= 6144); }
// What a narrow tile leaves in memory ends with it.  d_weight's k-tiles, the only reader of rows past the last one, do so
// at the same row or before.
static_assert(32 * 2 % BK == 0, "rows past the end are written to the end of the last k-tile");
__device__ __forceinline__ int tile_width(int64_t rows, int64_t row0, bool narrow) {
    const int64_t left = rows - row0;
    if (!narrow || left > 192) return WIDE;
    return left > 128 ? 6 : left > 64 ? 4 : 2;
}
// What a call has of token rows: up to one tile (narrow too), tiles of which the last may be narrow, whole tiles.  As
// forward kernels, NARROW_LAST and TWO_TILES, of up to two tiles whose exponentials are kept, have code for all widths
// (fwd_tiles).
enum RowTiles { ONE_TILE, TWO_TILES, NARROW_LAST, WHOLE_TILES };
inline RowTiles row_tiles(int64_t rows, int64_t hdim) {
    return rows <= BN ? ONE_TILE : narrow_tiles(rows, hdim) ? NARROW_LAST : WHOLE_TILES;
}
// The k-tile at which the product of vocabulary tile vt with ONE_TILE or TWO_TILES begins.  Such a call reads W once and
// little else, 128 bytes of 256 rows at a time: with all workgroups at the same k-tile those lie hidden_dim * 2 bytes
// apart, on few of the memory channels.  So each run of 2^run vocabulary tiles, the ones that an XCD works on together
// and that share hidden's k-tiles in its L2, begins at another eighth.  One tile (vocabulary 128256, us before and after):
// 100 rows x 2048 160, 134; 100 x 4096 260, 212; 256 x 4096 311, 247; 256 x 8192 560, 444; 30 x 8192 378, 382.  Two tiles
// of 192 rows, whose workgroups keep step: steps of 268 rows (4096 x 100352) 979, 967 and on another card 821, 795 (forward 318,
// 303), of 300 (8192 x 128256) 2244, 2220, frozen-head DPO of 355 rows (8192 x 128256) 1429, 1404.  Two of 256, steps of 500
// rows: 4096 x 100352 1231, 1221; 8192 x 128256 2850, 2832; 3584 x 151665 1582, 1584; 2048 x 151936 988, 992.  Scoring passes,
// whose workgroups take several vocabulary tiles one after the other, lose by it (268 rows, 4096 x 128256: 397, 409).  With
// more tiles of rows W's k-tiles are shared as well and nothing is gained (4096 x 100352 520 rows 418, 420; 2940 x 4096 2205,
// 2195), while going round costs 0.4 % (scoring pass of 1432 rows).
__device__ __forceinline__ int first_k_tile(int64_t vt, int run, int64_t hdim) {
    return __builtin_amdgcn_readfirstlane((int)(vt >> run & 7) * (int)(hdim / BK) / 8);
}
template <class Body>
__device__ __forceinline__ void with_width(int nj, Body&& body) {
    if (nj == WIDE) body(std::integral_constant<int, WIDE>{});
    else if (nj == 6) body(std::integral_constant<int, 6>{});
    else if (nj == 4) body(std::integral_constant<int, 4>{});
    else body(std::integral_constant<int, 2>{});
}

// A fp32 tile that another kernel picks up: in the order in which its column groups lie in the registers
// (16 bytes per lane, consecutive lanes together, groups of PART_GROUP floats), so that neither side
// rearranges anything.
constexpr int PART_FLOATS = BM * BN, PART_GROUP = NTHREADS * 4;
__device__ __forceinline__ int part_group(int i, int j, int q) { return (i * 4 + j) * 4 + q; }
__device__ __forceinline__ void store_part(const Columns& c, float* part, int j, int tid) {
    asm volatile("" : "+v"(tid));
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q)
            *reinterpret_cast<oi_f32x4*>(part + part_group(i, j, q) * PART_GROUP + tid * 4) =
                oi_f32x4{c.z[i][q * 4], c.z[i][q * 4 + 1], c.z[i][q * 4 + 2], c.z[i][q * 4 + 3]};
}
__device__ __forceinline__ Columns load_part(const float* part, int j, int tid) {
    oi_f32x4 v[2][4];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q)
            v[i][q] = *reinterpret_cast<const oi_f32x4*>(part + part_group(i, j, q) * PART_GROUP + tid * 4);
    Columns c;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) c.z[i][r] = v[i][r >> 2][r & 3];
    return c;
}

// Online softmax statistics in the log2 domain of the scaled logits x = z * c:
//   m = max x,  s = sum 2^(x - m),  t = sum 2^(x - m) * (x - m)
// (entropy = ln2 * (log2 s - t / s), logsumexp = ln2 * (m + log2 s)).
__device__ __forceinline__ void merge_stats(float ma, float sa, float ta, float mb, float sb, float tb, float* m,
                                            float* s, float* t) {
    const float mn = fmaxf(ma, mb);
    const float da = ma - mn, db = mb - mn;
    const float fa = __builtin_amdgcn_exp2f(da), fb = __builtin_amdgcn_exp2f(db);
    *s = sa * fa + sb * fb;
    *t = fa * fmaf(da, sa, ta) + fb * fmaf(db, sb, tb);
    *m = mn;
}

// Fold the 32 logits that one lane holds for token column j of a finished tile into the running
// statistics.  PARTIAL handles the last vocabulary tile: rows past the vocabulary are skipped by
// predicate (weight exactly 0) instead of through a sentinel value.
// KEEP leaves 2^(x - ref) in place of every logit (0 for rows past the vocabulary): the exponentials
// of the statistics times 2^(max - ref), which the backward products can use in place of a
// recomputation.  `ref` is the token's reference exponent (the scaled logit of its own label, known
// before the tile is computed): relative to it the kept numbers stay inside the bf16 range whatever
// the magnitude of the logits, as long as the token's largest logit is less than KEEP_MAX_LOG2
// binary orders above its label's (tokens beyond that are flagged by the merge kernel and take the
// recomputing backward).
template <bool PARTIAL, bool KEEP>
__device__ __forceinline__ void stats_update(f32x16 (&z)[2], int wm, int lane, int64_t m0, int64_t vocab, float c,
                                             float ref, float& st_m, float& st_s, float& st_t) {
    // the maximum is taken over the unscaled logits (c > 0) and every exponent is one fma: the new
    // maximum is the rounded product max(z) * c while the exponents are rounded once, so the largest
    // term is 2^(a few ulp) rather than exactly 1, far below the accuracy of the sums
    float zmax = OI_NEG_BIG;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r)
            if (!PARTIAL || m0 + acc_row(wm, i, r, lane) < vocab) zmax = fmaxf(zmax, z[i][r]);
    const float mn = fmaxf(st_m, fmaxf(zmax * c, OI_NEG_BIG));
    const float shift = st_m - mn;
    const float alpha = __builtin_amdgcn_exp2f(shift);
    float s = st_s * alpha;
    float t = alpha * fmaf(shift, st_s, st_t);
    const float pow2_max = KEEP ? __builtin_amdgcn_exp2f(fminf(mn - ref, 126.f)) : 0.f;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            float d = fmaf(z[i][r], c, -mn);
            float e = __builtin_amdgcn_exp2f(d);
            if (PARTIAL && m0 + acc_row(wm, i, r, lane) >= vocab) {
                d = 0.f;
                e = 0.f;
            }
            s += e;
            t = fmaf(e, d, t);
            if (KEEP) z[i][r] = e * pow2_max;
        }
    st_m = mn;
    st_s = s;
    st_t = t;
}

// A finished tile leaves as bf16 rows of 256 columns one column group at a time: group j holds the 64 rows
// (tokens, or rows of a product) wn * 16 NJ + j * 32 + (0..31) of both wn halves with all 256 columns (every m-wave
// contributes its 64).  A lane holds groups of eight consecutive columns of one row; a wave's meet in its share of one
// ring slot and go to global memory as whole 128-byte lines, eight rows at a time.  The waves do not wait for each
// other: with rows of 512 bytes that all waves fill there were two barriers per group (d_weight of 268 rows x 100352
// 370 us, now 356, of 2340 rows x 128256 1983, now 1960; step of 268 rows 985, now 969).
//
// A share: 32 rows of 128 bytes, unpadded; the 16-byte pieces of a row at c ^ piece_perm(row), which spreads the
// 16-byte accesses of 16 rows, and those of a row pair, over all 64 banks.  Counters still show 1000 conflict cycles per
// tile of 256 x 256, four for each access; under 1 % of a tile of 64 k-tiles.
__device__ __forceinline__ int piece_perm(int row) { return row >> 1 & 7; }
constexpr int GROUP_ROWS = 64;
constexpr int GROUP_BF16_AT = 4 * TILE_ELEMS;  // ring slot 4: slots 0 .. 3 may be filling for the next tile
static_assert(GROUP_ROWS * BM <= TILE_ELEMS, "a bf16 group fits one ring slot");
template <int NJ = WIDE>
__device__ __forceinline__ int64_t group_row(int64_t row0, int j, int r) { return row0 + (r >> 5) * 16 * NJ + j * 32 + (r & 31); }
// One wave's share: 32 rows of 64 columns (128 bytes), row lane % 32 from each lane.  Columns acc_row(wm, i, 8 p .. 8 p + 7,
// lane) of the lane's row, which value(r) gives
constexpr int SHARE_COLS = 64, SHARE_ELEMS = 32 * SHARE_COLS;
template <class Value>
__device__ __forceinline__ void stage_bf16x8(uint16_t* share, int lane, int i, int p, Value&& value) {
    const int srow = lane & 31, piece = (i * 4 + p * 2 + (lane >> 5)) ^ piece_perm(srow);
    *reinterpret_cast<oi_u32x4*>(share + srow * SHARE_COLS + piece * 8) =
        oi_u32x4{oi_pack_bf16x2(value(p * 8), value(p * 8 + 1)), oi_pack_bf16x2(value(p * 8 + 2), value(p * 8 + 3)),
                 oi_pack_bf16x2(value(p * 8 + 4), value(p * 8 + 5)), oi_pack_bf16x2(value(p * 8 + 6), value(p * 8 + 7))};
}
// between a wave's writes to its share and its reads: the LDS serves a wave in order, so this only holds the compiler
__device__ __forceinline__ void share_staged() { asm volatile("" ::: "memory"); }
// piece it of a lane: row it * 8 + lane / 8, columns 8 (lane % 8) ..
constexpr int GROUP_PIECES = SHARE_ELEMS / 8 / OI_WAVE;
__device__ __forceinline__ int piece_row(int lane, int it) { return it * 8 + (lane >> 3); }
__device__ __forceinline__ oi_u32x4 staged_piece(const uint16_t* share, int lane, int it) {
    const int r = piece_row(lane, it);
    return *reinterpret_cast<const oi_u32x4*>(share + r * SHARE_COLS + ((lane & 7) ^ piece_perm(r)) * 8);
}

// ---------------------------------------------------------------------------------------------
// forward: per-token softmax statistics over the vocabulary tiles of one split
// ---------------------------------------------------------------------------------------------
// CACHE: the vocabulary tiles [cache_tile0, cache_tile0 + cache_tiles) also leave 2^(z c - xref[n])
// behind as bf16, token-major [n_pad, cache_ld]; rows of tokens past the end are zero up to the next multiple of 64 and
// not written behind it, where the last tile is narrow.
// LOGITS: every tile leaves its fp32 logits behind (store_part), tile (vt, tt) at logits +
// (vt * logits_tiles + tt) * PART_FLOATS.
// What a forward launch covers and where its exponentials go.  Splits [0, long_splits) take
// tiles_per_split vocabulary tiles each, the others one.  A launch hands out the long splits
// [first, first + n_first) from one set of queues and then the short splits
// [long_splits, long_splits + n_second) from a second set.
// The cache takes the vocabulary tiles [cache_tile0, cache_tile0 + cache_tiles) as columns from 0 on;
// with skip_label the label's own entry is stored as 0 (the caller adds that term itself).
struct FwdLaunch {
    int64_t tiles_per_split, long_splits, first, n_first, n_second;
    uint16_t* ecache;
    int64_t cache_ld, cache_tile0, cache_tiles;
    int skip_label;
    const float* xref;  // per token: the exponent that the kept exponentials are relative to (null: 0)
    float* logits;
    int64_t logits_tiles;
    bool narrow, either;  // the last tile of rows may be narrow; tiles may have either height (see FwdTiles)
};
enum FwdKeep { FWD_PLAIN, FWD_EXPONENTIALS, FWD_LOGITS };

// what a forward tile is folded into, and from
struct FwdArgs {
    const uint16_t *W, *hidden;
    const int64_t* labels;
    int64_t n_tokens, hdim, vocab;
    float c;
    int64_t n_pad;
    float4* partial;
    float* zy;
};
// running statistics of one token column of a lane, its reference exponent and its label (vocabulary ids fit
// 32 bits: vocab <= 2^22)
struct FwdColumn {
    float m, s, t, ref;
    int lab;
};
__device__ __forceinline__ FwdColumn fwd_column(const FwdArgs& a, const float* xref, int64_t n) {
    FwdColumn col = {OI_NEG_BIG, 0.f, 0.f, (xref && n < a.n_tokens) ? xref[n] : 0.f, 0};
    const int64_t y = n < a.n_tokens ? a.labels[n] : 0;
    col.lab = (int)(y < 0 ? 0 : (y >= a.vocab ? a.vocab - 1 : y));
    // in a register now: a wait for these loads later on would also wait for whatever was requested since
    asm volatile("" : "+v"(col.lab), "+v"(col.ref));
    return col;
}
// Column group j of vocabulary tile vt: the label's logit, the statistics and, where they are kept, the
// exponentials (through the wave's share of `stage`; every lane of the wave takes part).
template <FwdKeep KEEP, int NJ>
__device__ __forceinline__ void fwd_fold(f32x16 (&__restrict__ z)[2], FwdColumn& col, const FwdArgs& a, const FwdLaunch& fl,
                                         int64_t vt, int64_t n0, int j, int tid, uint16_t* stage) {
    constexpr bool CACHE = KEEP == FWD_EXPONENTIALS;
    asm volatile("" : "+v"(tid));  // addresses are formed here, not ahead of the tile's main loop
    const int lane = tid & 63, wave = tid >> 6, wm = wave & 3, wn = wave >> 2;
    uint16_t* share = stage + wave * SHARE_ELEMS;
    const int64_t m0 = vt * BM;
    // the target logit, when its row falls into this wave's 64 rows
    const int rel = col.lab - ((int)m0 + wm * 64);
    // register of this lane that holds the label's row, -1 when another lane or wave does
    int label_reg = -1;
    if (rel >= 0 && rel < 64) {
        const int rr = rel & 31;
        if (((rr >> 3) & 1) == (lane >> 5)) label_reg = (rel >> 5) * 16 + (rr >> 4) * 8 + (rr & 7);
    }
    if (label_reg >= 0) {
        float v = 0.f;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if (i * 16 + r == label_reg) v = z[i][r];
        const int64_t n = n0 + acc_col<NJ>(wn, j, lane);
        if (n < a.n_tokens) a.zy[n] = v;
    }
    if (m0 + BM > a.vocab)
        stats_update<true, CACHE>(z, wm, lane, m0, a.vocab, a.c, col.ref, col.m, col.s, col.t);
    else
        stats_update<false, CACHE>(z, wm, lane, m0, a.vocab, a.c, col.ref, col.m, col.s, col.t);
    if constexpr (CACHE) {
        if (fl.skip_label && label_reg >= 0) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (i * 16 + r == label_reg) z[i][r] = 0.f;
        }
        if (vt < fl.cache_tile0 || vt >= fl.cache_tile0 + fl.cache_tiles) return;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int p = 0; p < 2; ++p) stage_bf16x8(share, lane, i, p, [&](int r) { return z[i][r]; });
        share_staged();
        uint16_t* dst = fl.ecache + n0 * fl.cache_ld + (vt - fl.cache_tile0) * BM + wm * SHARE_COLS + (lane & 7) * 8;
#pragma unroll 1
        for (int it = 0; it < GROUP_PIECES; ++it) {
            const int64_t row = group_row<NJ>(0, j, wn * 32 + piece_row(lane, it));  // token of the tile
            const oi_u32x4 v = staged_piece(share, lane, it);
            *reinterpret_cast<oi_u32x4*>(dst + row * fl.cache_ld) = n0 + row < a.n_tokens ? v : oi_u32x4{0u, 0u, 0u, 0u};
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}
// the statistics of the lane's column meet those of the other lane half (same token, other rows), which leaves
// them in lanes 0 .. 31
__device__ __forceinline__ void fwd_merge_halves(FwdColumn& col) {
    const float om = __shfl_xor(col.m, 32, OI_WAVE), os = __shfl_xor(col.s, 32, OI_WAVE), ot = __shfl_xor(col.t, 32, OI_WAVE);
    float m, s, t;
    merge_stats(col.m, col.s, col.t, om, os, ot, &m, &s, &t);
    col.m = m;
    col.s = s;
    col.t = t;
}
// of `columns` tokens, red [4 m-waves][columns][3] to the partial statistics of a split (tid < columns)
__device__ __forceinline__ float4 fwd_merge_waves(const float* red, int columns, int tid) {
    float m = red[tid * 3], s = red[tid * 3 + 1], t = red[tid * 3 + 2];
#pragma unroll
    for (int w = 1; w < 4; ++w) {
        const float* p = red + (w * columns + tid) * 3;
        merge_stats(m, s, t, p[0], p[1], p[2], &m, &s, &t);
    }
    return make_float4(m, s, t, 0.f);
}

// RUN: of first_k_tile, or none
constexpr int FROM_ZERO = -1;
template <FwdKeep KEEP, int RUN, int NJ>
__device__ __forceinline__ void lmhead_fwd_item(const FwdArgs& a, const FwdLaunch& fl, int64_t split, int64_t tt, int64_t n0,
                                                uint16_t* lds) {
    const int64_t vocab_tiles = (a.vocab + BM - 1) / BM;
    // the first long_splits splits take tiles_per_split vocabulary tiles each, the others one
    const bool long_item = split < fl.long_splits;
    const int64_t vt_begin =
        long_item ? split * fl.tiles_per_split : fl.long_splits * fl.tiles_per_split + (split - fl.long_splits);
    int64_t vt_end = vt_begin + (long_item ? fl.tiles_per_split : 1);
    vt_end = vt_end < vocab_tiles ? vt_end : vocab_tiles;

    const int tid = opaque_tid(), lane = tid & 63, wave = tid >> 6, wm = wave & 3, wn = wave >> 2;
    const Operand tokens = {a.hidden, a.hdim, n0, a.n_tokens, a.hdim};
    Operand rows = {a.W, a.hdim, vt_begin * BM, a.vocab, a.hdim};

    FwdColumn col[NJ / 2];
#pragma unroll
    for (int j = 0; j < NJ / 2; ++j)
        col[j] = fwd_column(a, KEEP == FWD_EXPONENTIALS ? fl.xref : nullptr, n0 + acc_col<NJ>(wn, j, lane));

    constexpr Walk WALK = RUN == FROM_ZERO ? NEAR : ROUND;
    auto start_of = [&](int64_t vt) { return WALK == ROUND ? first_k_tile(vt, RUN, a.hdim) : 0; };
    begin_loads<false, false, NJ, WALK>(rows, tokens, a.hdim, lds, start_of(vt_begin));
    for (int64_t vt = vt_begin; vt < vt_end; ++vt) {
        AccTile<NJ> acc;
        gemm_loop<false, false, WALK>(acc, rows, tokens, a.hdim, lds, start_of(vt));
        // the next tile's first loads run beside this tile's statistics, which leave slots 0 .. 3 alone (scoring
        // pass of 1432 rows, 4096 x 128256: 1.435 -> 1.40 ms; steps 0.2 to 0.6 %)
        rows.r0 += BM;
        if (vt + 1 < vt_end) begin_loads<false, false, NJ, WALK>(rows, tokens, a.hdim, lds, start_of(vt + 1));
#pragma unroll
        for (int j = 0; j < NJ / 2; ++j) {
            Columns c = tile_columns<NJ>(acc, j);
            // leaves while the statistics are computed
            if (KEEP == FWD_LOGITS) store_part(c, fl.logits + (vt * fl.logits_tiles + tt) * PART_FLOATS, j, tid);
            fwd_fold<KEEP, NJ>(c.z, col[j], a, fl, vt, n0, j, tid, lds + GROUP_BF16_AT);
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    constexpr int COLUMNS = 32 * NJ;
    float* red = reinterpret_cast<float*>(lds);  // [4 wm][COLUMNS tokens][3]
#pragma unroll
    for (int j = 0; j < NJ / 2; ++j) {
        fwd_merge_halves(col[j]);
        if (lane < 32) {
            float* p = red + (wm * COLUMNS + acc_col<NJ>(wn, j, lane)) * 3;
            p[0] = col[j].m;
            p[1] = col[j].s;
            p[2] = col[j].t;
        }
    }
    lds_barrier();
    if (tid < COLUMNS && n0 + tid < a.n_tokens) a.partial[split * a.n_pad + n0 + tid] = fwd_merge_waves(red, COLUMNS, tid);
}

// Calls of up to 8 tiles of rows may cut them into tiles of 256 or of 192 rows.
inline bool either_height(int64_t row_tiles) { return row_tiles <= 8; }
// How a forward of up to 8 tiles of rows cuts them.  A narrow tile among whole ones does not keep step with them, so W's
// k-tiles come from memory for it once more; tiles that all have 192 rows do.  And a last round that only some workgroups
// have a tile for is as long as any: where few have, its vocabulary tiles are handed out in tiles of 128 rows, which
// take about half the time (an XCD's worth of tiles of 4096 with nothing else running: 256 rows 78 us, 192 62, 128 48, 64
// 50: below 128 the loop waits for its loads).  The estimate takes what its parts take, in 32nds of a whole tile in a
// full chip.  us before and after: 4096 x 100352 268 rows 335, 312; 384 330, 318; 512 397, 366; 520 471, 424; 1300 893, 865;
// 4096 x 128256 268 rows 389, 341; 576 569, 542; 8192 x 128256 268 rows 746, 660; 520 1145, 961; 3584 x 151665 384 rows 430,
// 400.  In alike tiles but without cutting the last round 384 rows take 348 (4096 x 100352, 3.06 rounds).  Where the
// estimate stays with whole tiles nothing changes (700 rows 494, 492).  The logits that a forward keeps for its backward lie
// in whole tiles; it takes none of this.
struct FwdTiles {
    int height;         // rows of a tile
    uint32_t row_tiles;
    uint32_t tail, tail_row_tiles;  // the last `tail` of the short splits come in tiles of TAIL_ROWS
};
constexpr int FEWER = 6, FEWER_ROWS = 32 * FEWER, TAIL = 4, TAIL_ROWS = 32 * TAIL;
// what a k-tile of tiles of the widths 8, 6 and less takes, in 32nds of a whole one's time
constexpr uint32_t WHOLE_COST = 32, FEWER_COST = 26, TAIL_COST = 18;
__host__ __device__ inline uint32_t fewer_tiles(int64_t rows) { return (uint32_t)((rows + FEWER_ROWS - 1) / FEWER_ROWS); }
__device__ __forceinline__ FwdTiles fwd_tiles(int64_t rows, uint32_t vocab_tiles, uint32_t short_splits, bool narrow) {
    // what a narrow one among whole ones costs the others, which read the same k-tiles of W
    constexpr uint32_t APART = 8;
    FwdTiles t = {BN, (uint32_t)((rows + BN - 1) / BN), 0, 0};
    if (t.row_tiles == 0) return t;
    const int last = tile_width(rows, (int64_t)(t.row_tiles - 1) * BN, narrow);
    uint32_t cost = t.row_tiles * WHOLE_COST;
    if (last != WIDE) cost += (last == FEWER ? FEWER_COST : TAIL_COST) - WHOLE_COST + (t.row_tiles > 1 ? APART : 0);
    uint32_t one = last == WIDE ? WHOLE_COST : 0;
    // no rows past those of whole tiles, which is what the buffers hold
    if (fewer_tiles(rows) * FEWER_COST < cost && fewer_tiles(rows) * FEWER_ROWS <= t.row_tiles * BN) {
        one = FEWER_COST;
        t.height = FEWER_ROWS;
        t.row_tiles = fewer_tiles(rows);
    }
    const uint32_t rest = vocab_tiles * t.row_tiles % gridDim.x, tail = (rest + t.row_tiles - 1) / t.row_tiles;
    const uint32_t tail_row_tiles = (uint32_t)((rows + TAIL_ROWS - 1) / TAIL_ROWS);
    const uint32_t rounds = (tail * tail_row_tiles + gridDim.x - 1) / gridDim.x;
    if (tail <= short_splits && rounds * TAIL_COST < one) {
        t.tail = tail;
        t.tail_row_tiles = tail_row_tiles;
    }
    return t;
}

template <FwdKeep KEEP, RowTiles TILES>
__global__ void __launch_bounds__(NTHREADS)
    lmhead_fwd_kernel(FwdArgs a, const int32_t* __restrict__ n_dev, FwdLaunch fl, uint32_t* __restrict__ queue) {
    __shared__ __align__(16) uint16_t lds[LDS_ELEMS];
    if (n_dev) a.n_tokens = device_count(n_dev);  // rows selected on the device: the host only knows an upper bound
    constexpr bool ALL_WIDTHS = TILES == TWO_TILES || TILES == NARROW_LAST;
    constexpr int RUN = TILES == ONE_TILE ? 5 : TILES == TWO_TILES ? 4 : FROM_ZERO;
    FwdTiles ft = {BN, (uint32_t)((a.n_tokens + BN - 1) / BN), 0, 0};
    if (ALL_WIDTHS && KEEP != FWD_LOGITS && fl.either)
        ft = fwd_tiles(a.n_tokens, (uint32_t)(fl.n_first * fl.tiles_per_split + fl.n_second), (uint32_t)fl.n_second, fl.narrow);
    // every long item of every XCD's queue is taken before the first short one: the short items are
    // there to fill the end of the launch
#pragma unroll 1
    for (int pass = 0; pass < 2; ++pass) {
        const int64_t first = pass ? fl.long_splits : fl.first, splits = pass ? fl.n_second : fl.n_first;
        const uint32_t tail = pass ? ft.tail : 0, head = (uint32_t)splits - tail;
        const uint32_t items = head * ft.row_tiles, tail_items = tail * ft.tail_row_tiles;
        const uint32_t locals = locals_for_items(items);
        for_each_id(queue + pass * QUEUE_WORDS, locals + locals_for_items(tail_items), lds, pass == 0 || fl.n_first == 0,
                    [&](uint32_t pid) {
            int64_t split, tt, n0;
            int width = WIDE;
            if (ALL_WIDTHS && pid >= locals * 8) {
                const uint32_t item = item_of_pid(pid - locals * 8, tail_items);
                if (item >= tail_items) return;
                tile_of_item(item, tail, ft.tail_row_tiles, &split, &tt);
                split += head;
                n0 = tt * TAIL_ROWS;
                width = TAIL;
            } else {
                const uint32_t item = item_of_pid(pid, items);
                if (item >= items) return;
                tile_of_item(item, head, ft.row_tiles, &split, &tt);
                n0 = tt * ft.height;
                if (ALL_WIDTHS && ft.height != BN) width = FEWER;
                else if (TILES != WHOLE_TILES) width = tile_width(a.n_tokens, n0, fl.narrow);
            }
            auto item = [&](auto nj) {
                lmhead_fwd_item<KEEP, RUN, decltype(nj)::value>(a, fl, first + split, tt, n0, lds);
            };
            if constexpr (TILES != WHOLE_TILES) with_width(width, item);
            else item(std::integral_constant<int, WIDE>{});
        });
    }
}

// A token whose largest scaled logit lies more than this many binary orders above its reference
// exponent is not served from kept exponentials (they would leave the bf16 range, or the factor
// that undoes the reference would): 2^64 leaves room for the fp32 sums over the vocabulary above it
// and for the per-token factor 2^(ref - lse2) >= 2^-(64 + 22) below it.
constexpr float KEEP_MAX_LOG2 = 64.f;

// Merges the partial statistics of token n over the vocabulary splits.  With a row selection
// (`rows` non-null) token n of the compacted batch is row rows[n] of the caller's tensors, the count
// comes from the device, and the rows that were left out are written as zeros: the grid covers
// n_total rows, thread i handles compacted token i and caller row i.
// `unsafe` (one byte per caller row, optional, cleared by the caller beforehand): set for a token
// whose kept exponentials cannot be trusted (its maximum is too far above xref[n], or is not a
// number); never cleared here, so marks that the caller has put there survive.
// Launch: a workgroup handles 64 tokens (lane = token, so the 16-byte partials of a split are read as one
// contiguous piece per wave), wave w merges the splits w, w + 16, ... and the results meet in the LDS.
// Bound by the latency of the reads, since a call has few workgroups: hence 16 waves with four reads each in
// flight.  One wave in four with one read in flight took 50 us for 268 tokens x 392 splits (10 us now),
// 30 us for 1432 x 275 (9 us).
constexpr int COMBINE_TOKENS = 64, COMBINE_WAVES = 16, COMBINE_THREADS = COMBINE_WAVES * OI_WAVE;
__global__ void __launch_bounds__(COMBINE_THREADS)
    lmhead_fwd_combine_kernel(const float4* __restrict__ partial, const float* __restrict__ zy, int64_t n_tokens,
                              const int32_t* __restrict__ n_dev, const int32_t* __restrict__ rows,
                              const uint8_t* __restrict__ row_mask, int64_t n_total, int64_t n_splits, int64_t n_pad,
                              float inv_t, float c, float* __restrict__ logprob, float* __restrict__ entropy,
                              float* __restrict__ lse_out, const float* __restrict__ xref,
                              uint8_t* __restrict__ unsafe) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t first = (int64_t)blockIdx.x * COMBINE_TOKENS, n = first + lane;
    if (n_dev) n_tokens = *n_dev;
    if (wave == 0 && row_mask && n < n_total && !row_mask[n]) {
        logprob[n] = 0.f;
        if (entropy) entropy[n] = 0.f;
        if (lse_out) lse_out[n] = 0.f;
    }
    if (first >= n_tokens) return;
    float m = OI_NEG_BIG, s = 0.f, t = 0.f;
    if (n < n_tokens) {
        const float4* p = partial + n;
        int64_t sp = wave;
        for (; sp + 3 * COMBINE_WAVES < n_splits; sp += 4 * COMBINE_WAVES) {
            float4 q[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) q[u] = p[(sp + u * COMBINE_WAVES) * n_pad];
#pragma unroll
            for (int u = 0; u < 4; ++u) merge_stats(m, s, t, q[u].x, q[u].y, q[u].z, &m, &s, &t);
        }
        for (; sp < n_splits; sp += COMBINE_WAVES) {
            const float4 q = p[sp * n_pad];
            merge_stats(m, s, t, q.x, q.y, q.z, &m, &s, &t);
        }
    }
    __shared__ float red[COMBINE_WAVES - 1][3][COMBINE_TOKENS];
    if (wave > 0) {
        red[wave - 1][0][lane] = m;
        red[wave - 1][1][lane] = s;
        red[wave - 1][2][lane] = t;
    }
    __syncthreads();
    if (wave != 0 || n >= n_tokens) return;
    const int merged = n_splits < COMBINE_WAVES ? (int)n_splits : COMBINE_WAVES;
    for (int w = 0; w < merged - 1; ++w) merge_stats(m, s, t, red[w][0][lane], red[w][1][lane], red[w][2][lane], &m, &s, &t);
    const double ln2 = 0.69314718055994530942;
    const double log2s = log2((double)s);
    // the statistics are in units of x = z * c with the fp32 constant c the tile kernel multiplied by:
    // back to nats through that very constant (inv_t / c, not the literal ln 2), so that the logprob of
    // a token whose label holds all of the probability comes out as 0 at any size of the logits
    const double lse = ((double)m + log2s) * ((double)inv_t / (double)c);
    const int64_t o = rows ? rows[n] : n;
    logprob[o] = (float)((double)zy[n] * (double)inv_t - lse);
    if (entropy) entropy[o] = (float)((log2s - (double)t / (double)s) * ln2);
    if (lse_out) lse_out[o] = (float)lse;
    if (unsafe && !(m - (xref ? xref[n] : 0.f) <= KEEP_MAX_LOG2)) unsafe[o] = 1;  // a NaN maximum is flagged too
}

// ---------------------------------------------------------------------------------------------
// backward step 1: dZ tile = g * inv_T * (onehot - softmax), bf16
// ---------------------------------------------------------------------------------------------
// What a dZ tile is made from besides its logits (per-token vectors in the order of the multiplied rows)
struct DzInputs {
    const int64_t* labels;
    const float *lse, *grad, *logprob;
    int64_t n_tokens, vocab;
    float c, inv_t;
};
// One lane's 32 logits z0, z1 (rows acc_row(wm, 0 / 1, r, lane) of the tile's 256 vocabulary rows from m0)
// of token n to bf16 entries of dZ in the staging row srow.
//
// stage[row][v]: rows = tokens, 256 (+8 pad) vocabulary columns.  A lane stores 16 bytes (8 vocabulary entries of
// one token) and consecutive lanes store to consecutive rows, 132 words apart: 16 of them meet all 64 banks.
__device__ __forceinline__ void dz_column(const f32x16& z0, const f32x16& z1, const DzInputs& in, int64_t n, int64_t m0,
                                          int wm, int lane, uint16_t* srow) {
    const int rows_left = (int)(in.vocab - m0 < BM ? in.vocab - m0 : BM);  // real vocabulary rows of the tile
    const int wave_row0 = wm * 64;
    const bool live = n < in.n_tokens;
    const float g = live ? in.grad[n] * in.inv_t : 0.f;
    // a token without gradient gets an exponent of -huge: every entry becomes -0 * 0
    const float l2 = g != 0.f ? in.lse[n] * OI_LOG2E : 3.0e38f;
    int64_t y = live ? in.labels[n] : -1;
    if (live) y = y < 0 ? 0 : (y >= in.vocab ? in.vocab - 1 : y);
    // The label's entry is g (1 - p_label) = - g expm1(logprob), taken from the forward's result
    // (exact also where p_label is close to 1) and written over the entry that the sweep below
    // leaves there: the sweep itself then treats all entries alike.
    const int rel = (live && y >= m0 && y < m0 + BM) ? (int)(y - m0) - wave_row0 : -1;
    const bool mine = rel >= 0 && rel < 64 && (((rel & 31) >> 3) & 1) == (lane >> 5);
    const float ng = -g;
    auto sweep = [&](auto last_tile_tag) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                float d[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int r = p * 8 + e;
                    float val = ng * __builtin_amdgcn_exp2f(fmaf(i == 0 ? z0[r] : z1[r], in.c, -l2));
                    if (decltype(last_tile_tag)::value && acc_row(wm, i, r, lane) >= rows_left) val = 0.f;
                    d[e] = val;
                }
                *reinterpret_cast<oi_u32x4*>(srow + acc_row(wm, i, p * 8, lane)) =
                    oi_u32x4{oi_pack_bf16x2(d[0], d[1]), oi_pack_bf16x2(d[2], d[3]), oi_pack_bf16x2(d[4], d[5]),
                             oi_pack_bf16x2(d[6], d[7])};
            }
    };
    if (rows_left < BM) sweep(std::true_type{});  // the last vocabulary tile: rows past the vocabulary hold 0
    else sweep(std::false_type{});
    if (mine) {
        // same lane, same LDS piece as the store above: program order keeps them apart
        const float val = ng * expm1f(in.logprob[n]);
        srow[wave_row0 + rel] = (uint16_t)oi_f32_to_bf16_bits(val);
    }
}

template <Walk WALK>
__device__ __forceinline__ void lmhead_dz_tile(const uint16_t* __restrict__ W, const uint16_t* __restrict__ hidden,
                                               const DzInputs& in, int64_t hdim, int64_t v_begin, int64_t chunk_cols,
                                               uint16_t* __restrict__ dz, int64_t vt, int64_t tt, uint16_t* lds) {
    const int tid = opaque_tid(), lane = tid & 63, wave = tid >> 6, wm = wave & 3, wn = wave >> 2;
    const int64_t n0 = tt * BN, m0 = v_begin + vt * BM;

    AccTile<> acc;
    // As the forward, so that the logits are its to the bit.  (Not where a step of 257 to 512 rows left exponentials, whose
    // forward may begin elsewhere along k: for the rows that it flagged the logits are its up to the order of their sums.)
    gemm_tile<WALK>(acc, W, hdim, m0, in.vocab, hidden, hdim, n0, in.n_tokens, hdim, lds,
                    WALK == ROUND ? first_k_tile(m0 / BM, 5, hdim) : 0);

    uint16_t* stage = lds;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int nl = acc_col(wn, j, lane);
        const Columns c = tile_columns(acc, j);
        dz_column(c.z[0], c.z[1], in, n0 + nl, m0, wm, lane, stage + nl * STAGE_STRIDE);
    }
    __syncthreads();
    const int64_t vcol0 = vt * BM;  // column of this tile inside the chunk
    // [token, vocab] order: 32 16-byte pieces per token row
#pragma unroll 4
    for (int it = 0; it < 16; ++it) {
        const int cidx = tid + it * NTHREADS;
        const int row = cidx >> 5, ch = cidx & 31;
        *reinterpret_cast<oi_u32x4*>(dz + (n0 + row) * chunk_cols + vcol0 + ch * 8) =
            *reinterpret_cast<const oi_u32x4*>(stage + row * STAGE_STRIDE + ch * 8);
    }
}

template <Walk WALK>
__global__ void __launch_bounds__(NTHREADS)
    lmhead_dz_kernel(const uint16_t* __restrict__ W, const uint16_t* __restrict__ hidden, DzInputs in,
                     const int32_t* __restrict__ n_dev, int64_t hdim, int64_t v_begin, int64_t chunk_cols, int64_t n_pad,
                     uint16_t* __restrict__ dz, uint32_t* __restrict__ queue) {
    __shared__ __align__(16) uint16_t lds[LDS_ELEMS];
    if (n_dev) {
        in.n_tokens = device_count(n_dev);
        n_pad = (in.n_tokens + BN - 1) / BN * BN;
    }
    for_each_tile(queue, chunk_cols / BM, n_pad / BN, lds, [&](int64_t vt, int64_t tt) {
        lmhead_dz_tile<WALK>(W, hidden, in, hdim, v_begin, chunk_cols, dz, vt, tt, lds);
    });
}

// The same dZ (to the bit) from the logits that the forward left behind as fp32 tiles, whole vocabulary at
// once.  Workgroup (j, tt, vt) takes column group j of tile (vt, tt): 64 tokens (j * 32 + 0..31 of both halves of the
// tile's width, which is the forward's) x 256 vocabulary columns, 64 KB in and 32 KB out.  A quarter of a whole tile per
// workgroup so that four of them share a CU and one's stores run beside another's loads.
constexpr int KEPT_ROWS = 64;
__global__ void __launch_bounds__(NTHREADS)
    lmhead_dz_kept_kernel(const float* __restrict__ logits, int64_t logits_tiles, DzInputs in,
                          const int32_t* __restrict__ n_dev, bool narrow, int64_t cols, uint16_t* __restrict__ dz) {
    __shared__ __align__(16) uint16_t stage[KEPT_ROWS * STAGE_STRIDE];
    if (n_dev) in.n_tokens = *n_dev;
    const int j = blockIdx.x & 3;
    const int64_t tt = blockIdx.x >> 2, vt = blockIdx.y, n0 = tt * BN;
    const int nj = tile_width(in.n_tokens, n0, narrow), half = 16 * nj;  // a group's rows: 32 at j * 32 of both halves
    if (n0 >= in.n_tokens || j >= nj / 2) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wm = wave & 3, wn = wave >> 2;
    const float* tile = logits + (vt * logits_tiles + tt) * PART_FLOATS;
    const Columns c = load_part(tile, j, tid);
    const int row = wn * 32 + (lane & 31);
    dz_column(c.z[0], c.z[1], in, n0 + wn * half + j * 32 + (lane & 31), vt * BM, wm, lane,
              stage + row * STAGE_STRIDE);
    __syncthreads();
#pragma unroll
    for (int it = 0; it < KEPT_ROWS * (BM / 8) / NTHREADS; ++it) {
        const int cidx = tid + it * NTHREADS;
        const int r = cidx >> 5, ch = cidx & 31;
        const int64_t n = n0 + (r >> 5) * half + j * 32 + (r & 31);
        *reinterpret_cast<oi_u32x4*>(dz + n * cols + vt * BM + ch * 8) =
            *reinterpret_cast<const oi_u32x4*>(stage + r * STAGE_STRIDE + ch * 8);
    }
}

// ---------------------------------------------------------------------------------------------
// backward steps 2 and 3: plain tile products with a store epilogue
// ---------------------------------------------------------------------------------------------
// Where a tile product goes.
// mode 0: out_f32  = acc          mode 1: out_f32 += acc
// mode 2: out_bf16 = acc          mode 3: out_bf16 = out_f32 + acc   (last chunk of d_hidden)
// Rows below m_valid and columns below N are stored.  With `out_rows`, row r of a bf16 result goes to row
// out_rows[r] of out_bf16 (the fp32 accumulator stays compact).  scale_a / scale_b: factors of row r, see
// DynRows.  Every element has one writer per launch and the launches follow each other on the stream, so the
// sums of modes 1 and 3 are plain loads and stores.
struct StoreTo {
    int mode;
    float* out_f32;
    uint16_t* out_bf16;
    int64_t ldo, N, m_valid;
    const int32_t* out_rows;
    const float *scale_a, *scale_b;
};
// Whole 16-byte pieces (8 bytes for the bf16 results of mode 3) can be stored and loaded.  Rows are whole pieces here
// (products that are not have gemm_any_kernel) and fp32 buffers are aligned; bf16 rows may lie on 4-byte boundaries.
__device__ __forceinline__ bool stores_in_pieces(const StoreTo& st) {
    return st.mode <= 1 || (reinterpret_cast<uintptr_t>(st.out_bf16) & 15) == 0;
}

// Column group j of a finished tile (products have whole ones) is its rows row0 + wn * 128 + j * 32 + (0..31) of both wn
// halves with all 256 columns from col0.  z0, z1: the lane's accumulators, row acc_col(wn, j, lane), columns acc_row(wm,
// 0 / 1, r, lane), i.e. groups of eight consecutive columns of one row.  bf16 goes through the wave's share of the LDS and
// leaves 128 bytes of a row at a time; fp32 meets in the LDS region `stage` (64 rows) and leaves as whole rows of 1 KB,
// every thread of the workgroup taking part.
//
// What bounds the epilogue is that nothing is multiplied meanwhile (one workgroup per CU), so few instructions
// and whole lines.  Registers transposed in quads of lanes and stored from there in 64-byte pieces, with a wait
// for the stores of the tile before the next tile's first load: d_weight of 268 rows (100352 x 4096, 6272
// tiles of 5 k-tiles) 606 us; through the LDS 544; without waiting for stores at its barriers 504; with the next tile's
// first loads ahead of it 478.  On a faster box that form took 417; without waiting for each store before the next (and
// with the tile engine's other changes) 370; without barriers 356.
constexpr int STAGE_F32 = BM + 4;                            // floats per row: rows 4 banks apart
constexpr int GROUP_F32 = GROUP_ROWS * STAGE_F32 * 2;        // LDS elements of an fp32 region
static_assert(2 * GROUP_F32 <= LDS_ELEMS, "the epilogue's regions fit the ring");
//
// A wave's loads and stores leave its counter in the order in which they were issued, so a load behind a group's stores
// is not there before those have reached memory.  PLAIN products (no factors of rows, no row index) therefore have no
// such loads in their code (behind a branch, their waits stand in everybody's way: each store of d_weight waited for the
// one before: an eighth of d_weight of 268 rows, 3 % of that of 3072).  What a product is added to is read group by
// group all the same: requested one group ahead, reads meet the stores of the group before, and sums of few k-tiles lose
// what those of many do not gain (100352 x 4096, us so and one group ahead: K = 320 791, 843; K = 1024 1156, 1196;
// 128256 x 4096, K = 7680 6000, 6005).
//
// Rows and columns past the end read what the last valid ones do, and store nothing.
template <bool PLAIN, int PIECES, int NJ = WIDE>
struct GroupRows {
    float a, b;       // factors of the lane's accumulator row
    int dst[PIECES];  // result rows of the thread's pieces

    // srow: group row of the lane's accumulators; r_first: that of the thread's piece 0, the others `step` apart
    __device__ __forceinline__ void request(const StoreTo& st, int64_t row0, int j, int srow, int r_first, int step) {
        if constexpr (!PLAIN) {
            const int64_t last = st.m_valid - 1;
            if (st.scale_a) {
                const int64_t row = group_row<NJ>(row0, j, srow);
                a = st.scale_a[row < last ? row : last];
                b = st.scale_b[row < last ? row : last];
            }
#pragma unroll
            for (int it = 0; it < PIECES; ++it) {
                const int64_t row = group_row<NJ>(row0, j, r_first + it * step);
                dst[it] = (int)row;
                if (st.mode >= 2 && st.out_rows) dst[it] = st.out_rows[row < last ? row : last];
            }
        }
    }
    // a row whose factor is exactly 0 is 0 whatever its sum holds (the sums of rows that were taken out may
    // have left the fp32 range)
    __device__ __forceinline__ float scale(const StoreTo& st, float v) const {
        return !PLAIN && st.scale_a ? (b == 0.f ? 0.f : v * a * b) : v;
    }
    // element offset of column col of piece it, group row r
    __device__ __forceinline__ int64_t at(const StoreTo& st, int64_t row0, int64_t col, int j, int r, int it) const {
        return (PLAIN ? group_row<NJ>(row0, j, r) : (int64_t)dst[it]) * st.ldo + col;
    }
};
// mode 2 in whole pieces.  PLAIN results (d_weight) are as large as the head, and who reads them next does so long after
// they would have left the caches: past those, which keep the operands, and W for the pass that follows (ordinary stores
// wait in the memory-side cache and are written back while the next forward streams W).  100352 x 4096, us before and
// after: d_weight of 100 rows 271, 240, of 268 rows 362, 335, of 1024 738, 710; the next step's forward 245, 202; 362, 331;
// 709, 687; from 1400 rows on both within 1 %.  Step of 268 rows 1100 -> 1048.  Pieces of 128 bytes are whole lines: past
// the caches, half lines go at 3.3 TB/s where whole ones go at 5.2.
template <bool PLAIN>
__device__ __forceinline__ void store_group_bf16(const f32x16& z0, const f32x16& z1, const StoreTo& st, int64_t row0,
                                                 int64_t col0, int j, uint16_t* stage, int tid) {
    asm volatile("" : "+v"(tid));  // addresses are formed here, not ahead of the tile's main loop
    const int lane = tid & 63, wave = tid >> 6, wm = wave & 3, wn = wave >> 2;
    uint16_t* share = stage + wave * SHARE_ELEMS;
    GroupRows<PLAIN, GROUP_PIECES> rows;
    rows.request(st, row0, j, wn * 32 + (lane & 31), wn * 32 + (lane >> 3), 8);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const f32x16& z = i == 0 ? z0 : z1;
            stage_bf16x8(share, lane, i, p, [&](int r) { return rows.scale(st, z[r]); });
        }
    share_staged();
    const int64_t col = col0 + wm * SHARE_COLS + (lane & 7) * 8;
#pragma unroll
    for (int it = 0; it < GROUP_PIECES; ++it) {
        const oi_u32x4 v = staged_piece(share, lane, it);
        const int r = wn * 32 + piece_row(lane, it);
        if (group_row(row0, j, r) >= st.m_valid || col >= st.N) continue;
        oi_u32x4* to = reinterpret_cast<oi_u32x4*>(st.out_bf16 + rows.at(st, row0, col, j, r, it));
        if constexpr (PLAIN) __builtin_nontemporal_store(v, to);
        else *to = v;
    }
}

// Every other mode, any pitch, any alignment of the element type.  ADDS: modes 1 and 3 in whole pieces.
// Piece `it` of a thread is row (thread / 64) + 8 it of the group, columns 4 (thread mod 64) ..
constexpr int F32_PIECES = GROUP_ROWS * (BM / 4) / NTHREADS;
template <bool PLAIN, bool ADDS, int NJ = WIDE>
struct F32Rows {
    GroupRows<PLAIN, F32_PIECES, NJ> rows;
    oi_f32x4 sum[F32_PIECES];

    __device__ __forceinline__ void request(const StoreTo& st, int64_t row0, int64_t col0, int j, int tid) {
        asm volatile("" : "+v"(tid));
        rows.request(st, row0, j, (tid >> 8) * 32 + (tid & 31), tid >> 6, NTHREADS / 64);
        if constexpr (ADDS) {
            // a wave reads one row at a time, whose address is scalar; results have any pitch, so it is formed in 64 bits
            const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
            const int64_t last = st.m_valid - 1;
            const int c = (tid & 63) * 4, last_c = (int)(st.N - 4 - col0 < BM - 4 ? st.N - 4 - col0 : BM - 4);
            const uint32_t col = c < last_c ? c : last_c;
#pragma unroll
            for (int it = 0; it < F32_PIECES; ++it) {
                const int64_t row = group_row<NJ>(row0, j, wave + it * (NTHREADS / 64));
                sum[it] = *reinterpret_cast<const oi_f32x4*>(st.out_f32 + (row < last ? row : last) * st.ldo + col0 + col);
            }
        }
    }
};
template <bool PLAIN, bool ADDS, int NJ = WIDE>
__device__ __forceinline__ void store_group_f32(const f32x16& z0, const f32x16& z1, const StoreTo& st, bool pieces,
                                                const F32Rows<PLAIN, ADDS, NJ>& in, int64_t row0, int64_t col0, int j,
                                                uint16_t* stage, int tid) {
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63, wave = tid >> 6, wm = wave & 3, wn = wave >> 2;
    const int mode = st.mode, srow = wn * 32 + (lane & 31);
    float* stage32 = reinterpret_cast<float*>(stage);
    const int ch = tid & 63, r_first = tid >> 6;
    const int64_t col = col0 + ch * 4;
    const auto& rows = in.rows;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const f32x16& z = i == 0 ? z0 : z1;
            *reinterpret_cast<oi_f32x4*>(stage32 + srow * STAGE_F32 + acc_row(wm, i, q * 4, lane)) =
                oi_f32x4{rows.scale(st, z[q * 4]), rows.scale(st, z[q * 4 + 1]), rows.scale(st, z[q * 4 + 2]),
                         rows.scale(st, z[q * 4 + 3])};
        }
    lds_barrier();
    const float* from = stage32 + r_first * STAGE_F32 + ch * 4;
    auto piece = [&](int it) {
        oi_f32x4 v = *reinterpret_cast<const oi_f32x4*>(from + it * 8 * STAGE_F32);
        if constexpr (ADDS) v += in.sum[it];
        return v;
    };
    if (mode <= 1 && (ADDS || pieces)) {
#pragma unroll
        for (int it = 0; it < F32_PIECES; ++it) {
            const int64_t row = group_row<NJ>(row0, j, r_first + it * 8);
            const oi_f32x4 v = piece(it);
            if (row < st.m_valid && col < st.N) *reinterpret_cast<oi_f32x4*>(st.out_f32 + row * st.ldo + col) = v;
        }
        return;
    }
    if (ADDS) {
#pragma unroll
        for (int it = 0; it < F32_PIECES; ++it) {
            const int r = r_first + it * 8;
            const oi_f32x4 v = piece(it);
            if (group_row<NJ>(row0, j, r) >= st.m_valid || col >= st.N) continue;
            *reinterpret_cast<uint2*>(st.out_bf16 + rows.at(st, row0, col, j, r, it)) =
                make_uint2(oi_pack_bf16x2(v.x, v.y), oi_pack_bf16x2(v.z, v.w));
        }
        return;
    }
    // bf16 in 4-byte words: rows off 16-byte boundaries, and every row of mode 2 that comes here (added pieces of tiles)
    if (col >= st.N) return;
#pragma unroll 1
    for (int it = 0; it < F32_PIECES; ++it) {
        const int64_t row = group_row<NJ>(row0, j, r_first + it * 8);
        if (row >= st.m_valid) break;
        oi_f32x4 v = *reinterpret_cast<const oi_f32x4*>(from + it * 8 * STAGE_F32);
        if (mode == 3) v += *reinterpret_cast<const oi_f32x4*>(st.out_f32 + row * st.ldo + col);
        uint32_t* b = reinterpret_cast<uint32_t*>(st.out_bf16 + (st.out_rows ? (int64_t)st.out_rows[row] : row) * st.ldo + col);
        b[0] = oi_pack_bf16x2(v.x, v.y);
        b[1] = oi_pack_bf16x2(v.z, v.w);
    }
}
__device__ __forceinline__ bool plain_rows(const StoreTo& st) { return !st.scale_a && !(st.mode >= 2 && st.out_rows); }
__device__ __forceinline__ bool adds_in_pieces(const StoreTo& st, bool pieces) { return pieces && (st.mode == 1 || st.mode == 3); }

// out[row, col] = sum_k R(row, k) * C(col, k).  R's rows (token or vocabulary rows of the result) are the tile
// product's n dimension and C's (the result's columns) its m dimension, because a lane's consecutive
// accumulators are consecutive in m: after the swap of lane quarters eight columns of one row, which the epilogue
// stores without a transpose.
// One tile, or with `part` a piece of one along k whose fp32 tile goes there and nowhere else.
struct ProductTile {
    Operand R, C;
    int64_t K;
    float* part;
};
// all but mode 2 in whole pieces: two regions in turn; one is written again only after the barrier of the group in
// between, by which every wave has read it out
template <bool PLAIN, bool ADDS>
__device__ __forceinline__ void store_tile_f32(const AccTile<>& acc, const ProductTile& t, const StoreTo& st, bool pieces,
                                               uint16_t* lds, int tid) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        __builtin_amdgcn_sched_barrier(0);
        F32Rows<PLAIN, ADDS> in;
        in.request(st, t.R.r0, t.C.r0, j, tid);
        const Columns c = tile_columns(acc, j);
        store_group_f32<PLAIN, ADDS>(c.z[0], c.z[1], st, pieces, in, t.R.r0, t.C.r0, j, lds + (j & 1) * GROUP_F32, tid);
        __builtin_amdgcn_sched_barrier(0);
    }
}
template <bool PLAIN>
__device__ __forceinline__ void store_tile_as(const AccTile<>& acc, const ProductTile& t, const StoreTo& st, bool pieces,
                                              uint16_t* lds, int tid) {
    if (st.mode == 2 && pieces) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            __builtin_amdgcn_sched_barrier(0);
            const Columns c = tile_columns(acc, j);
            store_group_bf16<PLAIN>(c.z[0], c.z[1], st, t.R.r0, t.C.r0, j, lds + GROUP_BF16_AT, tid);
            __builtin_amdgcn_sched_barrier(0);
        }
    } else if (adds_in_pieces(st, pieces)) {
        store_tile_f32<PLAIN, true>(acc, t, st, pieces, lds, tid);
    } else {
        store_tile_f32<PLAIN, false>(acc, t, st, pieces, lds, tid);
    }
}
// In mode 2 with whole pieces this leaves the ring slots 0 .. 3 alone.
__device__ __forceinline__ void store_tile(const AccTile<>& __restrict__ acc, const ProductTile& t, const StoreTo& st, bool pieces,
                                           uint16_t* lds) {
    const int tid = opaque_tid();
    if (t.part) {
#pragma unroll
        for (int j = 0; j < 4; ++j) store_part(tile_columns(acc, j), t.part, j, tid);
    } else if (plain_rows(st)) {
        store_tile_as<true>(acc, t, st, pieces, lds, tid);
    } else {
        store_tile_as<false>(acc, t, st, pieces, lds, tid);
    }
}
// a product without terms (no rows selected): zeros, or what the earlier launches summed up
__device__ __forceinline__ void store_no_terms(const StoreTo& st) {
    if (st.mode == 1) return;
    for (int64_t row = blockIdx.x; row < st.m_valid; row += gridDim.x) {
        const int64_t dst = (st.mode >= 2 && st.out_rows) ? (int64_t)st.out_rows[row] : row;
        for (int64_t col = threadIdx.x; col < st.N; col += NTHREADS) {
            if (st.mode == 0) st.out_f32[row * st.ldo + col] = 0.f;
            else st.out_bf16[dst * st.ldo + col] =
                st.mode == 3 ? (uint16_t)oi_f32_to_bf16_bits(st.out_f32[row * st.ldo + col]) : (uint16_t)0;
        }
    }
}

// Sizes that depend on a row count which only the device knows (rows selected by a mask).
//   role 1 (d_hidden = dZ * W, rows of the product are tokens):  M, m_valid and A's extent follow n
//   role 2 (d_weight = dZ^T * hidden, the k dimension is tokens): K and the operands' k extents follow n
struct DynRows {
    const int32_t* n_dev;
    int role;
    const int32_t* out_rows;
    // optional factors of row r of the product, applied as (acc * scale_a[r]) * scale_b[r] before it
    // is stored or accumulated (two factors so that neither has to leave the fp32 range)
    const float *scale_a, *scale_b;
    // optional: the store mode comes from device memory (a negative value: the launch does nothing)
    const int32_t* mode_dev;
    // role 1: pieces of tiles that the scratch holds, where tiles may have either height (plan_rows)
    uint32_t pieces = 0;
};

// A launch of resident workgroups computes its tiles in rounds of one per workgroup, and a last round
// that is half empty takes as long as a full one; with fewer tiles than workgroups most of the chip idles
// from the start (200 token rows at a hidden size of 4096 are 16 tiles of the d_hidden product for 256 CUs,
// each running over the whole vocabulary).  The tiles past the last whole round are therefore cut along
// k into `parts` pieces each, which fill the workgroups evenly; a piece leaves its fp32 tile in scratch and
// gemm_reduce_kernel adds the pieces of a tile in order (the result does not depend on who ran when).
// The number of parts is the one with the lowest estimate, in k-tiles of 64 (about 1.5 us): rounds of
// pieces, 4 k-tiles of prologue and drain per piece, and 3/32 of a k-tile for writing and reading back the
// 256 KB of a piece.  Pieces are at least 16 k-tiles long.  All from sizes, on the device, where the row
// count lives; the reduce kernel comes to the same numbers.
// Measured (whole policy-loss step, before -> after): 268 rows, hidden 4096, vocabulary 100352 (32 tiles):
// 2.94 -> 1.55 ms; 2400 rows, 3584, 151665 (140 tiles): 8.85 -> 7.46 ms; 22942 rows in three slabs of 480
// tiles, 4096, 128256: unchanged (a last round that is 7/8 full is left alone).
struct TailSplit {
    uint32_t whole, rest, parts;  // tiles [0, whole) in one piece, the `rest` after them in `parts` pieces
    uint32_t cost;                // of the last round, in 32nds of a k-tile
};
constexpr uint32_t SPLIT_MIN_KTILES = 16, SPLIT_MAX_PARTS = 32, SPLIT_MAX_ITEMS = 1024;
// cost of `parts` pieces for each tile, in 32nds of a k-tile (`per_ktile`: what one takes), `most` in all; SPLIT_NEVER: not
// to be had
constexpr uint32_t SPLIT_NEVER = 0x3ffffffu;  // costs are below, 32 * 2^16 k-tiles and less than half of that besides
__host__ __device__ inline uint32_t split_cost(uint32_t rest, uint32_t grid, uint32_t ktiles, uint32_t per_ktile, uint32_t most,
                                               uint32_t parts) {
    if (parts == 1) return per_ktile * ktiles + 32 * 4;
    if (parts > SPLIT_MAX_PARTS || rest * parts > most || ktiles < SPLIT_MIN_KTILES * parts) return SPLIT_NEVER;
    const uint32_t rounds = (rest * parts + grid - 1) / grid;
    return rounds * (per_ktile * ktiles / parts + 32 * 4) + 3 * rest * parts;
}
// Every lane of a wave weighs one number of parts on the device: one after the other, in all waves of a launch, they
// took as long as two k-tiles.
__host__ __device__ inline TailSplit plan_tail(uint32_t tiles, uint32_t grid, uint32_t ktiles, uint32_t per_ktile = 32,
                                               uint32_t most = SPLIT_MAX_ITEMS) {
    const uint32_t rest = tiles % grid;
    if (rest == 0) return {tiles, 0, 1, split_cost(grid, grid, ktiles, per_ktile, most, 1)};
#ifdef __HIP_DEVICE_COMPILE__
    const uint32_t mine = 1 + __lane_id();
    uint32_t best = split_cost(rest, grid, ktiles, per_ktile, most, mine) * 64 + (mine & 63);
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) {
        const uint32_t other = __shfl_xor(best, d, OI_WAVE);
        best = other < best ? other : best;
    }
    best = __builtin_amdgcn_readfirstlane(best);
#else
    uint32_t best = ~0u;
    for (uint32_t parts = 1; parts <= SPLIT_MAX_PARTS; ++parts) {
        const uint32_t cost = split_cost(rest, grid, ktiles, per_ktile, most, parts) * 64 + parts;
        best = cost < best ? cost : best;
    }
#endif
    const uint32_t parts = best & 63;
    if (parts == 1) return {tiles, 0, 1, best >> 6};
    return {tiles - rest, rest, parts, best >> 6};
}

// Rows products of few rows also come in tiles of 192 rows, all of them: 268 rows are then 384 instead of 512 that are
// multiplied.  (One narrow tile among wide ones has pieces of another length, falls out of step with those that read the
// same k-tiles of W, and gains nothing.)  What takes less by the estimate
// (FEWER_COST) is chosen, where that leaves all tiles in one round and in pieces.  d_hidden, us in tiles of 256 and of 192:
// 4096 x 100352 268 rows 295, 235; 384 299, 246; 520 448, 365; 1152 743, 735; 8192 x 128256 268 rows 728, 596; 520 1109, 898;
// 3584 x 151665 268 rows 426, 347; 2048 x 151936 268 rows 266, 211.  Counts in between stay with 256 (4096 x 100352 400
// rows 294, 600 441).  Kernels of calls with more than 8 tiles of rows have no code for it: their gain would be 6 % at most.
struct RowsPlan {
    TailSplit split;
    bool fewer;
};
// M: the rows of whole tiles, `rows` what there is of them; `pieces`: what the scratch holds (that of tiles of 256 rows at
// any count up to the call's), 0 for tiles of 256 only
__device__ __forceinline__ RowsPlan plan_rows(int64_t M, int64_t rows, uint32_t tiles_c, uint32_t grid, uint32_t ktiles,
                                              uint32_t pieces) {
    RowsPlan p = {plan_tail((uint32_t)((M + BN - 1) / BN) * tiles_c, grid, ktiles), false};
    if (pieces == 0 || p.split.whole) return p;
    const uint32_t tiles = fewer_tiles(rows) * tiles_c;
    const TailSplit t = plan_tail(tiles, grid, ktiles, FEWER_COST, pieces);
    if (tiles < grid && t.whole == 0 && t.cost < p.split.cost) p = {t, true};
    return p;
}

// The sizes of a product that only the device knows, filled in from dyn
struct ProductSizes {
    int64_t M, K, m_valid;
};
__device__ __forceinline__ ProductSizes product_sizes(int64_t M, int64_t K, int64_t m_valid, const DynRows& dyn) {
    ProductSizes z = {M, K, m_valid};
    if (dyn.n_dev) {
        const int64_t n = device_count(dyn.n_dev);
        if (dyn.role == 1) {
            z.M = (n + BM - 1) / BM * BM;
            z.m_valid = n;
        } else if (dyn.role == 2) {
            z.K = (n + BK - 1) / BK * BK;
        }
    }
    return z;
}

// `queue` null: one workgroup per tile id (blockIdx); otherwise a launch of resident workgroups
// that draw their tiles from the queue.  `parts` (with a queue only): scratch for the pieces of split tiles.
// WIDTHS: rows products (role 1) in tiles of one of two heights, see plan_rows.
template <bool R_KM, bool C_KM, bool WIDTHS = false>
__global__ void __launch_bounds__(NTHREADS)
    gemm_store_kernel(Operand R, int64_t M, Operand C, int64_t N, int64_t K, int mode, float* out_f32,
                      uint16_t* out_bf16, int64_t ldo, int64_t m_valid, DynRows dyn, uint32_t* __restrict__ queue,
                      float* __restrict__ parts) {
    __shared__ __align__(16) uint16_t lds[LDS_ELEMS];
    if (dyn.mode_dev) {
        mode = device_count(dyn.mode_dev);
        if (mode < 0) return;
    }
    const ProductSizes z = product_sizes(M, K, m_valid, dyn);
    if (dyn.n_dev && dyn.role == 1) R.extent = z.M;
    if (dyn.n_dev && dyn.role == 2) {
        const int64_t n = device_count(dyn.n_dev);
        R.k_valid = z.K;  // rows of dZ behind these are not defined
        C.k_valid = n;
    }
    K = z.K;
    const StoreTo st = {mode, out_f32, out_bf16, ldo, N, z.m_valid, dyn.out_rows, dyn.scale_a, dyn.scale_b};
    const bool pieces = stores_in_pieces(st);
    if (K <= 0) {
        store_no_terms(st);
        return;
    }
    const uint32_t tiles_c = (uint32_t)((N + BM - 1) / BM), ktiles = (uint32_t)(K / BK);
    RowsPlan rp = {{0, 0, 1, 0}, false};
    if (parts) rp = plan_rows(z.M, z.m_valid, tiles_c, gridDim.x, ktiles, WIDTHS ? dyn.pieces : 0);
    const uint32_t height = WIDTHS && rp.fewer ? FEWER_ROWS : BN;
    const uint32_t tiles_r = WIDTHS && rp.fewer ? fewer_tiles(z.m_valid) : (uint32_t)((z.M + BN - 1) / BN);
    const uint32_t tiles = tiles_r * tiles_c;
    TailSplit ts = rp.split;
    if (!parts) ts.whole = tiles;
    auto tile_at = [&](uint32_t any_item) {
        const uint32_t item = __builtin_amdgcn_readfirstlane(any_item);
        ProductTile t = {R, C, K, nullptr};
        uint32_t tile = item;
        if (item >= ts.whole) {
            const uint32_t r = item - ts.whole, p = r / ts.rest;
            tile = ts.whole + (r - p * ts.rest);
            const uint32_t k0 = ktiles * p / ts.parts, k1 = ktiles * (p + 1) / ts.parts;
            const int64_t k_begin = (int64_t)k0 * BK;
            t.R.p += R_KM ? k_begin * R.ld : k_begin;
            t.C.p += C_KM ? k_begin * C.ld : k_begin;
            t.R.k_valid -= k_begin;
            t.C.k_valid -= k_begin;
            t.K = (int64_t)(k1 - k0) * BK;
            t.part = parts + (int64_t)r * PART_FLOATS;
        }
        int64_t tr, tc;
        tile_of_item(tile, tiles_r, tiles_c, &tr, &tc);
        t.R.r0 = tr * height;
        t.C.r0 = tc * BM;
        return t;
    };
    // Whole bf16 pieces leave through slot 4 while the next tile's first loads go to slots 0 .. 3: a tile of
    // few k-tiles (d_weight of a short batch) otherwise spends more time between its main loops than in them.
    // The fp32 modes need more LDS than one slot and belong to batches of several slabs, whose tiles are long.
    const bool ahead = mode == 2 && pieces;
    if (tiles == 0) return;
    const uint32_t items = ts.whole + ts.rest * ts.parts;
    // ids without an item among them: the exact number changes the main loop's code, and large d_hidden products take 1.2 %
    // longer (2950 rows x 8192 4388 us, 4448)
    ItemQueue q(queue, items, (uint32_t)(pids_for_items(items) >> 3), lds, true);
    uint32_t item = item_of_pid(blockIdx.x, q.items);
    if (item >= q.items && queue) {  // an id without an item
        q.request();
        q.settle();
        item = q.take_item();
    }
    if (item >= q.items) return;
    ProductTile t = tile_at(item);
    if constexpr (WIDTHS) {
        if (rp.fewer) {  // all of them in pieces, which leave without the LDS
            begin_loads<C_KM, R_KM, FEWER>(t.C, t.R, t.K, lds);
            for (;;) {
                AccTile<FEWER> acc;
                q.request();
                gemm_loop<C_KM, R_KM>(acc, t.C, t.R, t.K, lds);
                q.settle();
                item = q.take_item();
                float* part = t.part;
                if (item != ItemQueue::NONE) {
                    t = tile_at(item);
                    begin_loads<C_KM, R_KM, FEWER>(t.C, t.R, t.K, lds);
                }
                const int tid = opaque_tid();
#pragma unroll
                for (int j = 0; j < FEWER / 2; ++j) store_part(tile_columns<FEWER>(acc, j), part, j, tid);
                if (item == ItemQueue::NONE) return;
                lds_barrier();  // every wave has read the queue's word, which lies in slot 4
            }
        }
    }
    begin_loads<C_KM, R_KM>(t.C, t.R, t.K, lds);
    for (;;) {
        AccTile<> acc;
        q.request();
        gemm_loop<C_KM, R_KM>(acc, t.C, t.R, t.K, lds);
        q.settle();
        item = q.take_item();
        const ProductTile done = t;
        if (item != ItemQueue::NONE) {
            t = tile_at(item);
            if (ahead) begin_loads<C_KM, R_KM>(t.C, t.R, t.K, lds);
        }
        lds_barrier();  // every wave has read the queue's word, which lies in slot 4
        store_tile(acc, done, st, pieces, lds);
        if (item == ItemQueue::NONE) return;
        if (!ahead) {
            lds_barrier();
            begin_loads<C_KM, R_KM>(t.C, t.R, t.K, lds);
        }
    }
}

// ---- products whose rows are not whole 16-byte pieces --------------------------------------------------------
// The stand-alone products take any pitch and any alignment of the element type (modes 0, 1 and 2, no row index, no
// factors); the others' rows are hidden_dim (a multiple of 64) columns.  Kept out of gemm_store_kernel, whose main
// loop comes out 0.3 % slower with this code in it.
//
// Widest access of a row: 8 columns (16 bytes of bf16), 4 (16 bytes of fp32, 8 of bf16), 2 (4 bytes of bf16) or 1;
// `out` is the buffer that the mode touches
__host__ __device__ inline int store_width(int mode, const void* out, int64_t N, int64_t ldo) {
    const uintptr_t p = reinterpret_cast<uintptr_t>(out), element = mode <= 1 ? 4 : 2;
    if (((N | ldo) & 7) == 0 && (p & 15) == 0) return 8;
    if (((N | ldo) & 3) == 0 && (p & (4 * element - 1)) == 0) return 4;
    return mode == 2 && (ldo & 1) == 0 && (p & 3) == 0 ? 2 : 1;
}

// A staged group whose rows cannot be stored four columns at a time: a lane takes W columns every 64 W, so that a
// wave's access is one run of a row; four rows at a time, whose sums so far (clamped onto valid entries) and LDS
// reads are all under way before the first is used.
// Four neighbouring columns per lane, stored one by one, against this: bf16 [8192, 8190] x 256 113 -> 76 us, fp32 130
// -> 91, added to fp32 243 -> 135; added to fp32 [300, 1001] x 512 49 -> 25.
template <int W>
__device__ __forceinline__ void store_group_by_columns(const StoreTo& st, int64_t row0, int64_t col0, int j, const float* stage32,
                                                       int tid) {
    constexpr int PER = BM / (64 * W), ROWS = 4;
    const int mode = st.mode, lane = tid & 63, left = (int)(st.N - col0 < BM ? st.N - col0 : BM);
#pragma unroll 1
    for (int r0 = tid >> 6; r0 < GROUP_ROWS; r0 += 8 * ROWS) {
        float v[ROWS][PER][W];
        int64_t row[ROWS], dst[ROWS];
#pragma unroll
        for (int u = 0; u < ROWS; ++u) {
            row[u] = group_row(row0, j, r0 + 8 * u);
            const int64_t r = row[u] < st.m_valid ? row[u] : st.m_valid - 1;
            dst[u] = (mode >= 2 && st.out_rows ? (int64_t)st.out_rows[r] : r) * st.ldo + col0;
        }
        if (mode == 1) {
#pragma unroll
            for (int u = 0; u < ROWS; ++u)
#pragma unroll
                for (int k = 0; k < PER; ++k)
#pragma unroll
                    for (int w = 0; w < W; ++w) {
                        const int c = (lane + 64 * k) * W + w;
                        v[u][k][w] = st.out_f32[dst[u] + (c < left ? c : left - 1)];
                    }
        }
#pragma unroll
        for (int u = 0; u < ROWS; ++u)
#pragma unroll
            for (int k = 0; k < PER; ++k)
#pragma unroll
                for (int w = 0; w < W; ++w) {
                    const float z = stage32[(r0 + 8 * u) * STAGE_F32 + (lane + 64 * k) * W + w];
                    v[u][k][w] = mode == 1 ? v[u][k][w] + z : z;
                }
#pragma unroll
        for (int u = 0; u < ROWS; ++u) {
            if (row[u] >= st.m_valid) return;
#pragma unroll
            for (int k = 0; k < PER; ++k) {
                const int c = (lane + 64 * k) * W;
                if (c >= left) continue;
                if (W == 2 && c + 1 < left) {
                    *reinterpret_cast<uint32_t*>(st.out_bf16 + dst[u] + c) = oi_pack_bf16x2(v[u][k][0], v[u][k][W - 1]);
                } else if (mode <= 1) {
                    st.out_f32[dst[u] + c] = v[u][k][0];
                } else {
                    st.out_bf16[dst[u] + c] = (uint16_t)oi_f32_to_bf16_bits(v[u][k][0]);
                }
            }
        }
    }
}

// Column group j of a tile through the LDS region `stage`, as store_group_f32
__device__ __forceinline__ void store_group_any(const f32x16& z0, const f32x16& z1, const StoreTo& st, int width, int64_t row0,
                                                int64_t col0, int j, uint16_t* stage, int tid) {
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63, wave = tid >> 6, wm = wave & 3, wn = wave >> 2;
    const int mode = st.mode, srow = wn * 32 + (lane & 31);
    float* stage32 = reinterpret_cast<float*>(stage);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const f32x16& z = i == 0 ? z0 : z1;
            *reinterpret_cast<oi_f32x4*>(stage32 + srow * STAGE_F32 + acc_row(wm, i, q * 4, lane)) =
                oi_f32x4{z[q * 4], z[q * 4 + 1], z[q * 4 + 2], z[q * 4 + 3]};
        }
    lds_barrier();
    if (width == 2) return store_group_by_columns<2>(st, row0, col0, j, stage32, tid);
    if (width == 1) return store_group_by_columns<1>(st, row0, col0, j, stage32, tid);
    // four columns at once (added to fp32 [128256, 4092] x 256: one by one 1857 us, so 945; bf16 901 -> 561)
    constexpr int ITERS = GROUP_ROWS * (BM / 4) / NTHREADS;
    const int ch = tid & 63, r_first = tid >> 6;
    const int64_t col = col0 + ch * 4;
    if (col >= st.N) return;
    oi_f32x4 v[ITERS];
    if (mode == 1) {
#pragma unroll
        for (int it = 0; it < ITERS; ++it) {
            int64_t row = group_row(row0, j, r_first + it * 8);
            row = row < st.m_valid ? row : st.m_valid - 1;
            v[it] = *reinterpret_cast<const oi_f32x4*>(st.out_f32 + row * st.ldo + col);
        }
    }
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
        const oi_f32x4 z = *reinterpret_cast<const oi_f32x4*>(stage32 + (r_first + it * 8) * STAGE_F32 + ch * 4);
        v[it] = mode == 1 ? v[it] + z : z;
    }
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
        const int64_t row = group_row(row0, j, r_first + it * 8);
        if (row >= st.m_valid) return;
        if (mode <= 1)
            *reinterpret_cast<oi_f32x4*>(st.out_f32 + row * st.ldo + col) = v[it];
        else
            *reinterpret_cast<uint2*>(st.out_bf16 + row * st.ldo + col) =
                make_uint2(oi_pack_bf16x2(v[it].x, v[it].y), oi_pack_bf16x2(v[it].z, v[it].w));
    }
}

// one workgroup per tile id, any width
template <bool R_KM, bool C_KM>
__global__ void __launch_bounds__(NTHREADS)
    gemm_any_kernel(Operand R, int64_t M, Operand C, int64_t N, int64_t K, int mode, float* out_f32, uint16_t* out_bf16,
                    int64_t ldo, int width) {
    __shared__ __align__(16) uint16_t lds[LDS_ELEMS];
    const StoreTo st = {mode, out_f32, out_bf16, ldo, N, M, nullptr, nullptr, nullptr};
    const uint32_t tiles_r = (uint32_t)((M + BN - 1) / BN), tiles_c = (uint32_t)((N + BM - 1) / BM);
    const uint32_t item = item_of_pid(blockIdx.x, tiles_r * tiles_c);
    if (item >= tiles_r * tiles_c) return;
    int64_t tr, tc;
    tile_of_item(item, tiles_r, tiles_c, &tr, &tc);
    R.r0 = tr * BN;
    C.r0 = tc * BM;
    AccTile<> acc;
    gemm_tile<C_KM, R_KM, FAR>(acc, C, R, K, lds);
    const int tid = opaque_tid();
    // two regions in turn, as in store_tile
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        __builtin_amdgcn_sched_barrier(0);
        const Columns c = tile_columns(acc, j);
        store_group_any(c.z[0], c.z[1], st, width, R.r0, C.r0, j, lds + (j & 1) * GROUP_F32, tid);
        __builtin_amdgcn_sched_barrier(0);
    }
}

template <bool R_KM, bool C_KM>
int launch_product(const Operand& a, int64_t M, const Operand& b, int64_t N, int64_t K, float* out_f32, void* out_bf16, int64_t ldo,
                   int accumulate, hipStream_t s) {
    const int mode = out_f32 ? (accumulate ? 1 : 0) : 2;
    const int width = store_width(mode, out_f32 ? static_cast<void*>(out_f32) : out_bf16, N, ldo);
    const dim3 grid(grid_for_tiles((M + BM - 1) / BM, (N + BN - 1) / BN));
    uint16_t* o16 = static_cast<uint16_t*>(out_bf16);
    // both operands one row each (pitch 0): the only k-contiguous ones that can be longer than a pitch
    const bool far = !R_KM && !C_KM && K > MAX_LD;
    if (width == 8 && !far)
        hipLaunchKernelGGL((gemm_store_kernel<R_KM, C_KM>), grid, dim3(NTHREADS), 0, s, a, M, b, N, K, mode, out_f32, o16, ldo, M,
                           DynRows{}, static_cast<uint32_t*>(nullptr), static_cast<float*>(nullptr));
    else
        hipLaunchKernelGGL((gemm_any_kernel<R_KM, C_KM>), grid, dim3(NTHREADS), 0, s, a, M, b, N, K, mode, out_f32, o16, ldo,
                           width);
    return oi_launch_status();
}

// A product added to bf16 rows that are there already: out[row, col] += sum over the n selected tokens (n on the
// device; none: nothing happens).  It serves the d_weight of flagged rows, of which there are normally none, so it is
// kept out of gemm_store_kernel's main loop; the few k-tiles of a call that has some leave it bound by reading and
// writing d_weight.  Policy-loss step of 3000 rows, 4096 x 128256, one of them flagged: 22.8 ms with the entries read
// and added one by one, 15.5 ms so.
__global__ void __launch_bounds__(NTHREADS)
    gemm_add_kernel(Operand R, int64_t M, Operand C, int64_t N, uint16_t* out, int64_t ldo, const int32_t* __restrict__ n_dev,
                    uint32_t* __restrict__ queue) {
    __shared__ __align__(16) uint16_t lds[LDS_ELEMS];
    const int64_t n = device_count(n_dev);
    if (n <= 0) return;
    const int64_t K = (n + BK - 1) / BK * BK;
    R.k_valid = K;
    C.k_valid = n;
    for_each_tile(queue, (M + BN - 1) / BN, (N + BM - 1) / BM, lds, [&](int64_t tr, int64_t tc) {
        R.r0 = tr * BN;
        C.r0 = tc * BM;
        AccTile<> acc;
        gemm_tile<true, true>(acc, C, R, K, lds);
        const int tid = opaque_tid(), lane = tid & 63, wave = tid >> 6, wm = wave & 3, wn = wave >> 2;
        constexpr int ITERS = GROUP_ROWS * (BM / 4) / NTHREADS;
        const int ch = tid & 63, r_first = tid >> 6, srow = wn * 32 + (lane & 31);
        const int64_t col = C.r0 + ch * 4;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            __builtin_amdgcn_sched_barrier(0);
            // what is there already is requested before the tile goes through the LDS; rows and columns past the
            // end read the last valid entries and store nothing.  N and ldo are multiples of 64, out is 4-byte aligned.
            uint32_t there[ITERS][2];
            const int64_t from = col < N ? col : N - 4;
#pragma unroll
            for (int it = 0; it < ITERS; ++it) {
                int64_t row = group_row(R.r0, j, r_first + it * 8);
                row = row < M ? row : M - 1;
                const uint32_t* b = reinterpret_cast<const uint32_t*>(out + row * ldo + from);
                there[it][0] = b[0];
                there[it][1] = b[1];
            }
            // two regions in turn, as in store_tile
            float* stage32 = reinterpret_cast<float*>(lds + (j & 1) * GROUP_F32);
            const Columns c = tile_columns(acc, j);
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    *reinterpret_cast<oi_f32x4*>(stage32 + srow * STAGE_F32 + acc_row(wm, i, q * 4, lane)) =
                        oi_f32x4{c.z[i][q * 4], c.z[i][q * 4 + 1], c.z[i][q * 4 + 2], c.z[i][q * 4 + 3]};
            lds_barrier();
#pragma unroll
            for (int it = 0; it < ITERS; ++it) {
                const int64_t row = group_row(R.r0, j, r_first + it * 8);
                oi_f32x4 v = *reinterpret_cast<const oi_f32x4*>(stage32 + (r_first + it * 8) * STAGE_F32 + ch * 4);
                v += oi_f32x4{oi_bf16lo_to_f32(there[it][0]), oi_bf16hi_to_f32(there[it][0]), oi_bf16lo_to_f32(there[it][1]),
                              oi_bf16hi_to_f32(there[it][1])};
                if (row >= M || col >= N) continue;
                uint32_t* b = reinterpret_cast<uint32_t*>(out + row * ldo + col);
                b[0] = oi_pack_bf16x2(v.x, v.y);
                b[1] = oi_pack_bf16x2(v.z, v.w);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    });
}

// Adds the pieces of the split tiles of a gemm_store_kernel launch over `grid` workgroups and stores the
// sums as that kernel stores a tile.  One workgroup per column group of a tile (as in lmhead_dz_kept_kernel);
// bound by reading the pieces once.
__global__ void __launch_bounds__(NTHREADS)
    gemm_reduce_kernel(const float* __restrict__ parts, uint32_t grid, int64_t M, int64_t N, int64_t K, int mode,
                       float* out_f32, uint16_t* out_bf16, int64_t ldo, int64_t m_valid, DynRows dyn) {
    __shared__ __align__(16) uint16_t stage[GROUP_F32];
    const ProductSizes z = product_sizes(M, K, m_valid, dyn);
    const StoreTo st = {mode, out_f32, out_bf16, ldo, N, z.m_valid, dyn.out_rows, dyn.scale_a, dyn.scale_b};
    const int64_t tiles_c = (N + BM - 1) / BM;
    const RowsPlan rp = plan_rows(z.M, z.m_valid, (uint32_t)tiles_c, grid, (uint32_t)(z.K / BK), dyn.pieces);
    const TailSplit ts = rp.split;
    const int64_t height = rp.fewer ? FEWER_ROWS : BN, tiles_r = rp.fewer ? fewer_tiles(z.m_valid) : (z.M + BN - 1) / BN;
    const uint32_t tile = blockIdx.x >> 2;
    const int j = blockIdx.x & 3, tid = threadIdx.x;
    if (tile >= ts.rest || j * 2 >= (rp.fewer ? FEWER : WIDE)) return;
    const float* src = parts + (int64_t)tile * PART_FLOATS;
    Columns c = load_part(src, j, tid);
    for (uint32_t p = 1; p < ts.parts; ++p) {
        src += (int64_t)ts.rest * PART_FLOATS;
        const Columns more = load_part(src, j, tid);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) c.z[i][r] += more.z[i][r];
    }
    int64_t tr, tc;
    tile_of_item(ts.whole + tile, (uint32_t)tiles_r, (uint32_t)tiles_c, &tr, &tc);
    const bool pieces = stores_in_pieces(st);
    const int64_t row0 = tr * height, col0 = tc * BM;
    auto store = [&](auto adds, auto nj) {
        F32Rows<false, decltype(adds)::value, decltype(nj)::value> in;
        in.request(st, row0, col0, j, tid);
        store_group_f32<false, decltype(adds)::value, decltype(nj)::value>(c.z[0], c.z[1], st, pieces, in, row0, col0, j, stage, tid);
    };
    auto store_rows = [&](auto nj) {
        if (adds_in_pieces(st, pieces)) store(std::true_type{}, nj);
        else store(std::false_type{}, nj);
    };
    if (rp.fewer) store_rows(std::integral_constant<int, FEWER>{});
    else store_rows(std::integral_constant<int, WIDE>{});
}

inline int64_t round_up(int64_t x, int64_t m) { return (x + m - 1) / m * m; }

__global__ void zero_words_kernel(uint32_t* __restrict__ p, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}
__global__ void zero_bytes_kernel(uint8_t* __restrict__ p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

// ---------------------------------------------------------------------------------------------
// row selection: which token rows are multiplied at all
// ---------------------------------------------------------------------------------------------
// Row i takes part when its mask byte is set (no mask: every row) and, in the backward pass when
// asked for, when its upstream gradient is not exactly zero.  The selection is made on the device
// and stays there: the host sizes grids and buffers for all n rows and every kernel reads the
// selected count from memory, so no call ever waits for the GPU.
__device__ __forceinline__ bool row_selected(const uint8_t* __restrict__ mask, const float* __restrict__ grad,
                                             int64_t i) {
    return (!mask || mask[i] != 0) && (!grad || grad[i] != 0.f);
}

constexpr int SELECT_THREADS = 1024;
// Of one workgroup: rows[0 .. count) = positions of the selected rows in ascending order (a stable
// compaction: count per thread segment, block scan, write).  Returns the count to every thread.
__device__ __forceinline__ int select_rows(const uint8_t* __restrict__ mask, const float* __restrict__ grad, int64_t n,
                                           int32_t* __restrict__ rows) {
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int64_t per = (n + SELECT_THREADS - 1) / SELECT_THREADS;
    const int64_t b = t * per, e = b + per < n ? b + per : n;
    // up to 64 rows of a thread: their bits, read once
    const bool few = per <= 64;
    uint64_t bits = 0;
    int c = 0;
    if (few) {
#pragma unroll 8
        for (int k = 0; k < per; ++k) {
            const int64_t i = b + k < e ? b + k : n - 1;
            const bool set = row_selected(mask, grad, i);
            bits |= (uint64_t)(set && b + k < e) << k;
        }
        c = __popcll(bits);
    } else {
        for (int64_t i = b; i < e; ++i) c += row_selected(mask, grad, i) ? 1 : 0;
    }
    int incl = c;
#pragma unroll
    for (int off = 1; off < OI_WAVE; off <<= 1) {
        const int o = __shfl_up(incl, off, OI_WAVE);
        if (lane >= off) incl += o;
    }
    __shared__ int wave_total[SELECT_THREADS / OI_WAVE];
    if (lane == OI_WAVE - 1) wave_total[wave] = incl;
    __syncthreads();
    int base = 0, total = 0;
#pragma unroll
    for (int w = 0; w < SELECT_THREADS / OI_WAVE; ++w) {
        base += w < wave ? wave_total[w] : 0;
        total += wave_total[w];
    }
    int pos = base + incl - c;
    if (few) {
        for (; bits; bits &= bits - 1) rows[pos++] = (int32_t)(b + __ffsll((unsigned long long)bits) - 1);
    } else {
        for (int64_t i = b; i < e; ++i)
            if (row_selected(mask, grad, i)) rows[pos++] = (int32_t)i;
    }
    return total;
}
// One workgroup.  Also clears `n_zero` (<= 1024) queue words for the launches that follow.
__global__ void __launch_bounds__(SELECT_THREADS)
    select_rows_kernel(const uint8_t* __restrict__ mask, const float* __restrict__ grad, int64_t n,
                       int32_t* __restrict__ rows, int32_t* __restrict__ count, uint32_t* __restrict__ zero_words,
                       int n_zero) {
    const int total = select_rows(mask, grad, n, rows);
    if (threadIdx.x == 0) *count = total;
    if ((int)threadIdx.x < n_zero) zero_words[threadIdx.x] = 0u;
}

// Workgroup j copies selected row j: the hidden-state row (hdim bf16, 16-byte pieces), its label
// and, for the backward pass, its logsumexp and upstream gradient.
__global__ void __launch_bounds__(256)
    gather_rows_kernel(const uint16_t* __restrict__ hidden, const int64_t* __restrict__ labels,
                       const float* __restrict__ lse, const float* __restrict__ grad,
                       const float* __restrict__ logprob, const int32_t* __restrict__ rows,
                       const int32_t* __restrict__ count, int64_t hdim, uint16_t* __restrict__ hidden_c,
                       int64_t* __restrict__ labels_c, float* __restrict__ lse_c, float* __restrict__ grad_c,
                       float* __restrict__ logprob_c) {
    const int64_t j = blockIdx.x;
    if (j >= *count) return;
    const int64_t src = rows[j];
    const oi_u32x4* from = reinterpret_cast<const oi_u32x4*>(hidden + src * hdim);
    oi_u32x4* to = reinterpret_cast<oi_u32x4*>(hidden_c + j * hdim);
    for (int64_t c = threadIdx.x; c < hdim / 8; c += blockDim.x) to[c] = from[c];
    if (threadIdx.x == 0) {
        labels_c[j] = labels[src];
        if (lse_c) lse_c[j] = lse[src];
        if (grad_c) grad_c[j] = grad[src];
        if (logprob_c) logprob_c[j] = logprob[src];
    }
}

__device__ __forceinline__ float dot_bf16x8(const oi_u32x4& a, const oi_u32x4& b, float acc) {
    const uint32_t aw[4] = {a.x, a.y, a.z, a.w}, bw[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        acc = fmaf(oi_bf16lo_to_f32(aw[k]), oi_bf16lo_to_f32(bw[k]), acc);
        acc = fmaf(oi_bf16hi_to_f32(aw[k]), oi_bf16hi_to_f32(bw[k]), acc);
    }
    return acc;
}

// xref[j] = c * <hidden[j, :], W[label_j, :]>: the scaled logit of token j's own label, the exponent
// that the token's kept exponentials are relative to.  It needs to be close to the token's largest
// scaled logit, not equal to it (the same number is taken out again wherever the exponentials are
// used), so the summation order of this dot product does not matter.  One wave per token.
__global__ void __launch_bounds__(256)
    label_ref_kernel(const uint16_t* __restrict__ hidden, const uint16_t* __restrict__ W,
                     const int64_t* __restrict__ labels, const int32_t* __restrict__ n_dev, int64_t n_tokens,
                     int64_t hdim, int64_t vocab, float c, float* __restrict__ xref) {
    const int lane = threadIdx.x & 63;
    const int64_t j = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (n_dev) n_tokens = *n_dev;
    if (j >= n_tokens) return;
    int64_t y = labels[j];
    y = y < 0 ? 0 : (y >= vocab ? vocab - 1 : y);
    const oi_u32x4* a = reinterpret_cast<const oi_u32x4*>(hidden + j * hdim);
    const oi_u32x4* b = reinterpret_cast<const oi_u32x4*>(W + y * hdim);
    float acc = 0.f;
    for (int64_t p = lane; p < hdim / 8; p += OI_WAVE) {  // hdim is a multiple of 64
        acc = dot_bf16x8(a[p], b[p], acc);
    }
    acc = oi_wave_sum(acc);
    if (lane == 0) xref[j] = acc * c;
}

// Selection without a launch of its own.  Of up to SELECT_AT_ONCE rows every workgroup counts the mask's bytes in front of
// its rows for itself (8 of a lane at a time, from L2), which tells where those go; it then does what was to be done with
// them, a wave for each row.  A launch that only makes the row index, and another one each for what goes by it, take 4.6 us
// of a busy stream whatever they do, and one workgroup takes 18 us for the index of 32768 rows.  Rows selected, gathered and
// marked, and those left out cleared: 2 launches, 4 with the reference exponents, before; 435 rows x 4096, four 19 us, one
// 6; 2950 rows x 8192, four 48, one 29.
//
// The bytes counted grow with the square of the rows, so there is a limit, which is as far as the tests go on both sides; it is
// not where the two ways meet.  Scores, us, at once and by an index: 65600 rows x 2048 157, 206; x 4096 277, 325; x 8192 522,
// 575; 131072 x 2048 319, 473; x 4096 549, 717.
constexpr int64_t SELECT_AT_ONCE = 65536;
constexpr int AT_ONCE_WAVES = 4, AT_ONCE_THREADS = AT_ONCE_WAVES * OI_WAVE;
// Rows of a wave: more where there are many workgroups anyway, so that the mask is not read by too many, and the more the
// shorter they are.  Forward with the sum and backward, us, one row, two and four: 24576 rows x 2048 155 77, 150 76, 149 75;
// 32768 x 4096 346 156, 341 158, 341 171; x 8192 614 281, 624 291, 638 318; 65536 x 2048 342 204, 320 174, 314 168; x 4096
// 561 308, 544 292, 549 298; x 8192 1037 551, 1038 555, 1055 577.
inline int rows_per_wave(int64_t n, int64_t hdim) { return n <= 16384 ? 1 : hdim <= 2048 ? 4 : 2; }
inline unsigned at_once_grid(int64_t n, int64_t hdim) {
    const int64_t rows = AT_ONCE_WAVES * rows_per_wave(n, hdim);
    return (unsigned)((n + rows - 1) / rows);
}
__device__ __forceinline__ int nonzero_bytes(uint64_t x) {
    constexpr uint64_t low = 0x7f7f7f7f7f7f7f7full;
    return __popcll((((x & low) + low) | x) & ~low);
}
// selected rows among [0, b), for every thread of the workgroup
__device__ __forceinline__ int rows_before(const uint8_t* __restrict__ mask, int64_t b) {
    const int tid = threadIdx.x;
    const int64_t to_word = (8 - (reinterpret_cast<uintptr_t>(mask) & 7)) & 7, head = to_word < b ? to_word : b;
    const int64_t words = (b - head) / 8, tail = head + words * 8;
    const uint64_t* w = reinterpret_cast<const uint64_t*>(mask + head);
    int c = 0;
#pragma unroll 4
    for (int64_t i = tid; i < words; i += AT_ONCE_THREADS) c += nonzero_bytes(w[i]);
    if (tid < head) c += mask[tid] != 0;
    if (tail + tid < b) c += mask[tail + tid] != 0;
    __shared__ int sum[AT_ONCE_WAVES];
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) c += __shfl_xor(c, d, OI_WAVE);
    if ((tid & 63) == 0) sum[tid >> 6] = c;
    __syncthreads();
    int total = 0;
#pragma unroll
    for (int k = 0; k < AT_ONCE_WAVES; ++k) total += sum[k];
    return total;
}
// each(row, selected, rank among the selected) for the wave's rows; last(count) for the workgroup that has the last row.
template <class Each, class Last>
__device__ __forceinline__ void for_selected_rows(const uint8_t* __restrict__ mask, int64_t n, int per_wave, Each&& each,
                                                  Last&& last) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int of_group = AT_ONCE_WAVES * per_wave;  // at most 64
    const int64_t b = (int64_t)blockIdx.x * of_group;
    const uint64_t set = __ballot(lane < of_group && b + lane < n && mask[b + lane] != 0);
    const int before = rows_before(mask, b);
#pragma unroll 1
    for (int k = 0; k < per_wave; ++k) {
        const int at = wave * per_wave + k;
        if (b + at >= n) return;
        const int rank = before + __popcll(set & ((1ull << at) - 1));
        const bool selected = set >> at & 1;
        each(b + at, selected, (int64_t)rank);
        if (b + at == n - 1) last(rank + (selected ? 1 : 0));
    }
}
// What is gathered, and on the way: `zero_words` cleared; with `xref`, the reference exponents (as label_ref_kernel);
// with `clear`, a byte of every row, selected or not; with `zero_rows`, its rows that were not selected.
struct GatherRows {
    const uint16_t* hidden;
    const int64_t* labels;
    const float *lse, *grad, *logprob;
    int64_t hdim;
    int32_t *rows, *count;
    uint16_t* hidden_c;
    int64_t* labels_c;
    float *lse_c, *grad_c, *logprob_c;
    uint32_t* zero_words;
    int n_zero;
    const uint16_t* W;
    int64_t vocab;
    float c;
    float* xref;
    uint8_t* clear;
    uint16_t* zero_rows;
};
__global__ void __launch_bounds__(AT_ONCE_THREADS)
    select_gather_kernel(const uint8_t* __restrict__ mask, int64_t n, int per_wave, GatherRows g) {
    const int lane = threadIdx.x & 63;
    if (blockIdx.x == 0)
        for (int i = threadIdx.x; i < g.n_zero; i += AT_ONCE_THREADS) g.zero_words[i] = 0u;
    for_selected_rows(
        mask, n, per_wave,
        [&](int64_t src, bool selected, int64_t j) {
            if (g.clear && lane == 0) g.clear[src] = 0;
            if (!selected) {
                if (!g.zero_rows) return;
                uint16_t* row = g.zero_rows + src * g.hdim;  // hdim is a multiple of 64; rows may lie on 4-byte boundaries
                if ((reinterpret_cast<uintptr_t>(row) & 15) == 0)
                    for (int64_t p = lane; p < g.hdim / 8; p += OI_WAVE) reinterpret_cast<oi_u32x4*>(row)[p] = oi_u32x4{0u, 0u, 0u, 0u};
                else
                    for (int64_t p = lane; p < g.hdim / 2; p += OI_WAVE) reinterpret_cast<uint32_t*>(row)[p] = 0u;
                return;
            }
            const int64_t label = g.labels[src];
            const oi_u32x4* from = reinterpret_cast<const oi_u32x4*>(g.hidden + src * g.hdim);
            oi_u32x4* to = reinterpret_cast<oi_u32x4*>(g.hidden_c + j * g.hdim);
            if (g.xref) {
                const int64_t y = label < 0 ? 0 : (label >= g.vocab ? g.vocab - 1 : label);
                const oi_u32x4* wy = reinterpret_cast<const oi_u32x4*>(g.W + y * g.hdim);
                float acc = 0.f;
#pragma unroll 8
                for (int64_t p = lane; p < g.hdim / 8; p += OI_WAVE) {
                    const oi_u32x4 a = from[p], b = wy[p];
                    to[p] = a;
                    acc = dot_bf16x8(a, b, acc);
                }
                acc = oi_wave_sum(acc);
                if (lane == 0) g.xref[j] = acc * g.c;
            } else {
#pragma unroll 8
                for (int64_t p = lane; p < g.hdim / 8; p += OI_WAVE) to[p] = from[p];
            }
            if (lane != 0) return;
            g.rows[j] = (int32_t)src;
            g.labels_c[j] = label;
            if (g.lse_c) g.lse_c[j] = g.lse[src];
            if (g.grad_c) g.grad_c[j] = g.grad[src];
            if (g.logprob_c) g.logprob_c[j] = g.logprob[src];
        },
        [&](int count) {
            if (lane == 0) *g.count = count;
        });
}

// Which rows a slab pass works on: rows order[offset .. offset + count) of a row index that lives
// on the device.  Written by a planning kernel, read by every kernel of the pass.
struct SlabMeta {
    int32_t offset, count;
    // how the slab's d_weight product is stored (the modes of StoreTo): the only slab writes
    // bf16 rows (2); of several, the first stores fp32 (0), the middle ones add to it (1) and the last
    // one adds the fp32 sum to its own product and writes bf16 rows (3); a pass without rows: -1
    int32_t dw_mode, reserved;
};

// Workgroup j copies row order[meta->offset + j] into the slab's own buffers: the hidden-state row
// (hdim bf16, 16-byte pieces), its label and its row number, and leaves the token's reference exponent
// (see label_ref_kernel) on the way.
__global__ void __launch_bounds__(256)
    gather_slab_kernel(const uint16_t* __restrict__ hidden, const uint16_t* __restrict__ W,
                       const int64_t* __restrict__ labels, const int32_t* __restrict__ order,
                       const SlabMeta* __restrict__ meta, int64_t hdim, int64_t vocab, float c,
                       uint16_t* __restrict__ hidden_s, int64_t* __restrict__ labels_s, int32_t* __restrict__ rows_s,
                       float* __restrict__ xref_s) {
    const int64_t j = blockIdx.x;
    if (j >= meta->count) return;
    const int64_t src = order[meta->offset + j], label = labels[src];
    const int64_t y = label < 0 ? 0 : (label >= vocab ? vocab - 1 : label);
    const oi_u32x4* from = reinterpret_cast<const oi_u32x4*>(hidden + src * hdim);
    const oi_u32x4* wy = reinterpret_cast<const oi_u32x4*>(W + y * hdim);
    oi_u32x4* to = reinterpret_cast<oi_u32x4*>(hidden_s + j * hdim);
    float acc = 0.f;
    for (int64_t p = threadIdx.x; p < hdim / 8; p += blockDim.x) {
        const oi_u32x4 a = from[p], b = wy[p];
        to[p] = a;
        acc = dot_bf16x8(a, b, acc);
    }
    __shared__ float scratch[16];
    acc = oi_block_sum(acc, scratch);
    if (threadIdx.x == 0) {
        labels_s[j] = label;
        rows_s[j] = (int32_t)src;
        xref_s[j] = acc * c;
    }
}

// Backward products straight from the kept exponentials e'[n, v] = 2^(x_nv - ref_n), x = z c:
//   dZ[n, v] = g_n inv_T (1[v = y_n] - 2^(x_nv - lse2_n)) = s_n (e'[n, v] - 1[v = y_n] 2^(lse2_n - ref_n)),
//   s_n = -g_n inv_T 2^(ref_n - lse2_n).
// The per-token factor leaves the products: d_hidden[n] = s_n (e'[n, :] W) (a row factor in the
// store epilogue) and d_weight = e'^T (s h) (the hidden rows are scaled once).  Workgroup j prepares
// token j of a slab (caller row rows_s[j]): the two halves of s_n (so that neither leaves the fp32
// range), the label's entry of the slab's exponentials, replaced by
// 2^(x_y - ref) - 2^(lse2 - ref) = 2^(lse2 - ref) expm1(logprob) from the forward's fp32 logprob
// (exact where the label's probability is close to 1), and, when d_weight is wanted, the scaled
// hidden row.  A token flagged in `unsafe` gets factors of exactly 0: it adds nothing to either
// product here and takes the recomputing backward afterwards.
// `upstream`: d loss / d logprob of a caller row, which GrpoUpstream derives here (a launch of its own for it took 5 us of
// every slab) and leaves in `grad` for the flagged rows, and StoredUpstream reads there.
struct StoredUpstream {
    __device__ __forceinline__ float operator()(int64_t row, float* grad) const { return grad[row]; }
};
struct GrpoUpstream {  // as grpo_fused_bwd_kernel, without an upstream gradient of the loss
    const float *logprob, *old, *ref, *adv, *rho, *row_denoms;
    int64_t cols;
    GrpoCfg cfg;
    float beta, scale;
    __device__ __forceinline__ float operator()(int64_t row, float* grad) const {
        const float x = logprob[row], ratio = old ? expf(x - old[row]) : 1.f;
        const float d = grpo_token_dnew(x, ratio, adv[row], ref != nullptr, ref ? ref[row] : 0.f, rho ? rho[row] : 1.f, cfg, beta);
        const float g = scale * row_denoms[(uint32_t)row / (uint32_t)cols] * d;  // rows are at most 2^22
        if (threadIdx.x == 0) grad[row] = g;
        return g;
    }
};
template <class Upstream>
__global__ void __launch_bounds__(256)
    slab_prepare_kernel(Upstream upstream, const float* __restrict__ lse, float* __restrict__ grad,
                        const float* __restrict__ logprob, const uint8_t* __restrict__ unsafe,
                        const int32_t* __restrict__ rows_s, const int64_t* __restrict__ labels_s,
                        const float* __restrict__ xref_s, const SlabMeta* __restrict__ meta, float inv_t,
                        int64_t vocab, int64_t hdim, uint16_t* __restrict__ ecache, int64_t cache_ld,
                        const uint16_t* __restrict__ hidden_s, float* __restrict__ scale_a,
                        float* __restrict__ scale_b, uint16_t* __restrict__ scaled_hidden) {
    const int64_t j = blockIdx.x;
    if (j >= meta->count) return;
    const int64_t src = rows_s[j];
    const bool dead = unsafe[src] != 0;
    const float l2 = lse[src] * OI_LOG2E - xref_s[j];  // log2 of the sum of the kept numbers of this token
    const float half = dead ? 0.f : __builtin_amdgcn_exp2f(-0.5f * l2);
    const float a = half, b = -upstream(src, grad) * inv_t * half;
    if (threadIdx.x == 0) {
        scale_a[j] = a;
        scale_b[j] = b;
        int64_t y = labels_s[j];
        y = y < 0 ? 0 : (y >= vocab ? vocab - 1 : y);
        ecache[j * cache_ld + y] =
            (uint16_t)oi_f32_to_bf16_bits(__builtin_amdgcn_exp2f(fminf(l2, 126.f)) * expm1f(logprob[src]));
    }
    if (!scaled_hidden) return;
    const oi_u32x4* from = reinterpret_cast<const oi_u32x4*>(hidden_s + j * hdim);
    oi_u32x4* to = reinterpret_cast<oi_u32x4*>(scaled_hidden + j * hdim);
    for (int64_t c = threadIdx.x; c < hdim / 8; c += blockDim.x) {
        const oi_u32x4 v = from[c];
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
        uint32_t o[4];
#pragma unroll
        for (int k = 0; k < 4; ++k)
            o[k] = dead ? 0u : oi_pack_bf16x2(oi_bf16lo_to_f32(w[k]) * a * b, oi_bf16hi_to_f32(w[k]) * a * b);
        to[c] = oi_u32x4{o[0], o[1], o[2], o[3]};
    }
}

// d_hidden rows of tokens that took no part are zero
__global__ void __launch_bounds__(256)
    zero_unselected_rows_kernel(const uint8_t* __restrict__ mask, const float* __restrict__ grad, int64_t hdim,
                                uint16_t* __restrict__ out) {
    const int64_t i = blockIdx.x;
    if (row_selected(mask, grad, i)) return;
    uint32_t* row = reinterpret_cast<uint32_t*>(out + i * hdim);  // hdim is a multiple of 64
    for (int64_t c = threadIdx.x; c < hdim / 2; c += blockDim.x) row[c] = 0u;
}

// Timing probe for the measurement harness: while armed, the slab-wise entry points record a pair
// of HIP events around one of their three products in every pass (which one is chosen when the probe is
// armed; d_hidden: the tile kernel and the launch that adds the pieces of its cut tiles, which finds none where no tile
// is cut), on the stream of the call.  Off by default and between arm / read; not meant for
// calls that are being captured into a graph.
struct Probe {
    int kernel = -1;  // 0 forward with kept exponentials, 1 d_hidden product, 2 d_weight product; -1 = off
    int used = 0;
    static constexpr int MAX_LAUNCHES = 1024;
    hipEvent_t ev[2 * MAX_LAUNCHES];
};
Probe g_probe;
struct ProbeScope {
    bool on;
    hipStream_t s;
    ProbeScope(int kernel, hipStream_t stream) : on(g_probe.kernel == kernel && g_probe.used < Probe::MAX_LAUNCHES), s(stream) {
        if (on) (void)hipEventRecord(g_probe.ev[2 * g_probe.used], s);
    }
    ~ProbeScope() {
        if (on) (void)hipEventRecord(g_probe.ev[2 * g_probe.used++ + 1], s);
    }
};

// Workgroups of a queue-driven launch on the current device
unsigned resident_grid(int64_t tiles_m, int64_t tiles_n, unsigned per_xcd = 0) {
    return resident_workgroups(tiles_m * tiles_n, oi_cu_count(), per_xcd);
}

// Scratch for the pieces of the rows products of a call, as launch_rows_product starts them: at most `row_tiles` x
// `h_tiles` tiles, the vocabulary in chunks of `chunk` columns.  The row count is known on the device only, so it is
// the most that plan_tail asks for at any count up to there: 256 pieces of 256 KB for one or two row tiles of 4096
// columns, 1008 for seven and more.
size_t split_bytes(int64_t row_tiles, int64_t h_tiles, int64_t chunk, int64_t vocab) {
    const uint32_t grid = resident_grid(row_tiles, h_tiles);
    const int64_t columns[2] = {chunk < vocab ? chunk : vocab, (vocab - 1) % chunk + 1};  // of the first and last chunk
    uint32_t most = 0;
    for (int64_t c : columns) {
        const uint32_t ktiles = (uint32_t)(round_up(c, BK) / BK);
        // what is left of whole rounds repeats after `grid` row tiles
        for (int64_t r = 1; r <= row_tiles && r <= (int64_t)grid && ktiles >= 2 * SPLIT_MIN_KTILES; ++r) {
            const TailSplit t = plan_tail((uint32_t)(r * h_tiles), grid, ktiles);
            if (t.rest * t.parts > most) most = t.rest * t.parts;
        }
        if (columns[0] == columns[1]) break;
    }
    return (size_t)most * PART_FLOATS * sizeof(float);
}

// Vocabulary columns that the recomputing backward takes at a time.  At 32768 token rows 32768, 65536 and
// the whole vocabulary measured the same and 16384 columns 1.3-2.5 % slower, so the scratch (2 bytes per
// token row and column) decides; fewer rows take as many more columns as the same scratch holds, up to the
// whole vocabulary at once, because every chunk is three launches with ragged ends: cross-entropy step of
// 3072 rows, hidden 4096, vocabulary 128256: 11.6 ms in four chunks, 11.2 ms in one; policy-loss step of
// 268 rows (whose launches over flagged rows find none): 1.55 -> 1.35 ms.
constexpr int64_t BWD_VOCAB_CHUNK = 32768;
constexpr int64_t CHUNK_BUDGET = (int64_t)32768 * 32768;  // token rows x columns
inline int64_t vocab_chunk(int64_t n_pad, int64_t v_pad, int64_t at_least) {
    const int64_t fits = CHUNK_BUDGET / n_pad / 1024 * 1024;
    const int64_t most = fits > at_least ? fits : at_least;
    if (v_pad <= most) return v_pad;
    // equal chunks, whole groups of four vocabulary tiles
    const int64_t n = (v_pad + most - 1) / most;
    return round_up((v_pad + n - 1) / n, 1024);
}
// chunk of the forward that also accumulates the weighted sum of weight rows: fewer, longer launches
// (measured on the 70B head shape: 16384 columns 79.2 ms, 32768 77.3, 65536 75.4 per step)
constexpr int64_t WSUM_VOCAB_CHUNK = 65536;

struct Carver {
    size_t off = 0;
    size_t take(size_t bytes) {
        const size_t o = off;
        off += (bytes + 255) / 256 * 256;
        return o;
    }
};

// buffers of a row selection: the row index, the selected count and the compacted per-row inputs
struct SelectionPlan {
    size_t off_rows, off_count, off_hidden, off_labels, off_lse, off_grad, off_logprob;
};
SelectionPlan plan_selection(Carver& cv, int64_t n_pad, int64_t hdim, bool backward) {
    SelectionPlan p;
    p.off_rows = cv.take((size_t)n_pad * sizeof(int32_t));
    p.off_count = cv.take(sizeof(int32_t));
    p.off_hidden = cv.take((size_t)n_pad * hdim * 2);
    p.off_labels = cv.take((size_t)n_pad * sizeof(int64_t));
    p.off_lse = backward ? cv.take((size_t)n_pad * sizeof(float)) : 0;
    p.off_grad = backward ? cv.take((size_t)n_pad * sizeof(float)) : 0;
    p.off_logprob = backward ? cv.take((size_t)n_pad * sizeof(float)) : 0;
    return p;
}

// Where the forward leaves the exponentials it computes anyway, or its logits (all null / 0: nowhere)
struct KeepPlan {
    uint16_t* buf;        // bf16 [n_pad, ld], token-major
    int64_t ld, tiles;    // columns of the buffer, and as vocabulary tiles
    const float* xref;    // per token: the exponent the kept numbers are relative to
    uint8_t* unsafe;      // per caller row: set when the kept numbers of that token cannot be used
    float* logits;        // or the fp32 logits themselves, tile by tile (buf null)
};

struct FwdPlan {
    int64_t token_tiles, vocab_tiles, n_splits, tiles_per_split, long_splits, n_pad;
    int64_t chunk, n_chunks;  // chunked flavour only
    size_t off_partial, off_zy, off_queue, off_chunk, off_parts, total;
    size_t parts_bytes;  // chunked flavour: scratch for the pieces of the products
    SelectionPlan sel;
};
// `chunked`: the launch covers one backward-sized vocabulary chunk at a time (the forward that also
// accumulates the weighted sum of weight rows): every split is a long one, so that a chunk is a whole
// number of splits, and there is one set of queues per chunk for the forward and one for the product.
FwdPlan plan_fwd(int64_t n_tokens, int64_t hdim, int64_t vocab, bool with_selection, bool chunked = false) {
    FwdPlan p;
    p.token_tiles = (n_tokens + BN - 1) / BN;
    p.vocab_tiles = (vocab + BM - 1) / BM;
    p.n_pad = p.token_tiles * BN;
    // Work items of 4 vocabulary tiles (8 tiles measured 1.6 % slower, 2 tiles no faster: every
    // item also writes and later merges a set of partial statistics).  Fewer tiles per split only
    // when the problem is too small to give every CU work otherwise.
    int64_t tps = 4;
    while (tps > 1 && ((p.vocab_tiles + tps - 1) / tps) * p.token_tiles < 512) tps /= 2;
    p.tiles_per_split = tps;
    // The ids are handed out with the vocabulary split as the slow index, so the last splits are
    // the last work of the launch: they are single tiles, about four per CU, which the workgroups
    // that run out of long items pick up (the launch then ends within one tile, not one item).
    const int64_t short_wanted = (4 * 256 + p.token_tiles - 1) / p.token_tiles;
    // whole groups of 8 long splits: the ids of a group of 8 splits are handed out together, and a
    // long item among the last short ones would be the new ragged end
    p.long_splits = tps > 1 && p.vocab_tiles > short_wanted ? (p.vocab_tiles - short_wanted) / tps / 8 * 8 : 0;
    p.n_splits = p.long_splits + (p.vocab_tiles - p.long_splits * tps);
    p.chunk = p.n_chunks = 0;
    if (chunked) {
        p.n_splits = p.long_splits = (p.vocab_tiles + tps - 1) / tps;
        const int64_t v_pad = p.vocab_tiles * BM;
        p.chunk = vocab_chunk(p.n_pad, v_pad, WSUM_VOCAB_CHUNK);
        p.n_chunks = (v_pad + p.chunk - 1) / p.chunk;
    }
    Carver cv;
    p.off_partial = cv.take((size_t)p.n_splits * p.n_pad * sizeof(float4));
    p.off_zy = cv.take((size_t)p.n_pad * sizeof(float));
    p.off_queue = cv.take((chunked ? (size_t)p.n_chunks * (FWD_QUEUE_WORDS + QUEUE_WORDS) : (size_t)FWD_QUEUE_WORDS) *
                          sizeof(uint32_t));
    p.off_chunk = chunked ? cv.take((size_t)p.n_pad * p.chunk * 2) : 0;
    p.parts_bytes = chunked ? split_bytes(p.token_tiles, (hdim + BN - 1) / BN, p.chunk, vocab) : 0;
    p.off_parts = cv.take(p.parts_bytes);
    if (with_selection) p.sel = plan_selection(cv, p.n_pad, hdim, false);
    p.total = cv.off;
    return p;
}

// Bytes of the forward's logits, tile by tile, for a backward that reads them instead of computing them
// again; 0 where they are not to be kept.  Keeping them takes the recomputation (a quarter of the matrix
// work of a step with a trained head) out of the step and costs 4 bytes per row and column between the passes:
// cross-entropy of 3072 rows, hidden 4096, vocabulary 128256: dZ 2460 -> 430 us (5.5 TB/s), forward 2350 -> 2770 us
// with its stores, step 10.9 -> 8.65 ms.  The line is 4 GiB, twice the scratch of the backward's dZ at the same sizes:
// a larger batch would hold a large part of a card's memory, and its step is better made slab by slab.
size_t kept_bytes(int64_t n_tokens, int64_t vocab) {
    const int64_t n_pad = round_up(n_tokens, BN), v_pad = round_up(vocab, BM);
    if (v_pad > CHUNK_BUDGET / n_pad / 1024 * 1024) return 0;
    return (size_t)n_pad * v_pad * sizeof(float);
}

struct BwdPlan {
    int64_t n_pad, v_pad, chunk, n_chunks;
    size_t off_dz, off_dh32, off_queues, off_parts, total;
    size_t parts_bytes;
    SelectionPlan sel;
};
// `few_rows`: for a call that normally finds no rows (its products are not split)
BwdPlan plan_bwd(int64_t n_tokens, int64_t hdim, int64_t vocab, bool with_selection, bool few_rows = false) {
    BwdPlan p;
    p.n_pad = round_up(n_tokens, 256);
    p.v_pad = round_up(vocab, 256);
    p.chunk = vocab_chunk(p.n_pad, p.v_pad, BWD_VOCAB_CHUNK);
    p.n_chunks = (p.v_pad + p.chunk - 1) / p.chunk;
    Carver cv;
    p.off_dz = cv.take((size_t)p.n_pad * p.chunk * 2);
    p.off_dh32 = cv.take((size_t)n_tokens * hdim * 4);
    // one set of work-queue counters per tile-kernel launch (three per vocabulary chunk)
    p.off_queues = cv.take((size_t)(3 * p.n_chunks) * QUEUE_WORDS * sizeof(uint32_t));
    p.parts_bytes = few_rows ? 0 : split_bytes(p.n_pad / BM, (hdim + BN - 1) / BN, p.chunk, vocab);
    p.off_parts = cv.take(p.parts_bytes);
    if (with_selection) p.sel = plan_selection(cv, p.n_pad, hdim, true);
    p.total = cv.off;
    return p;
}

int check_lmhead(const void* hidden, const void* weight, const int64_t* labels, int64_t n_tokens, int64_t hdim,
                 int64_t vocab, float inv_t) {
    OI_RETURN_IF(n_tokens < 0 || hdim <= 0 || vocab <= 0, OI_EINVAL);
    OI_RETURN_IF(hdim % 64 != 0, OI_EINVAL);
    OI_RETURN_IF(!(inv_t >= 1.0e-6f) || !(inv_t <= 1.0e6f), OI_EINVAL);
    // row strides of every operand (hidden_dim, padded vocabulary, padded token count) are folded
    // into 32-bit byte offsets inside a 256-row tile
    OI_RETURN_IF(n_tokens > MAX_LD || vocab > MAX_LD || hdim > MAX_LD, OI_EINVAL);
    if (n_tokens == 0) return OI_OK;
    OI_RETURN_IF(!hidden || !weight || !labels, OI_ENULL);
    OI_RETURN_IF(!oi_aligned(hidden, 16) || !oi_aligned(weight, 16), OI_EALIGN);
    return OI_OK;
}

// The per-row inputs the tile kernels read: the caller's own, or their compacted copies
struct RowInputs {
    const uint16_t* hidden;
    const int64_t* labels;
    const float *lse, *grad;
    const int32_t *rows, *n_dev;  // null without a selection
    const float* logprob;         // the forward's result: the label's entry of dZ is rebuilt from it
};

// What else a selection does for its rows, all optional: reference exponents of the selected ones (weight, c, xref), a byte
// of every row cleared, rows of a result that were not selected zeroed.
struct SelectionExtras {
    const void* weight;
    int64_t vocab;
    float c;
    float* xref;
    uint8_t* clear;
    void* zero_rows;
};
// select + gather on `s`; clears `n_zero` queue words on the way
RowInputs launch_selection(const SelectionPlan& sp, char* ws, const void* hidden, const int64_t* labels,
                           const float* lse, const float* grad, const uint8_t* row_mask, bool skip_zero_grad,
                           int64_t n_tokens, int64_t hdim, uint32_t* zero_words, int n_zero, hipStream_t s,
                           const float* logprob = nullptr, const SelectionExtras& extra = {}) {
    int32_t* rows = reinterpret_cast<int32_t*>(ws + sp.off_rows);
    int32_t* count = reinterpret_cast<int32_t*>(ws + sp.off_count);
    uint16_t* hidden_c = reinterpret_cast<uint16_t*>(ws + sp.off_hidden);
    int64_t* labels_c = reinterpret_cast<int64_t*>(ws + sp.off_labels);
    float* lse_c = lse ? reinterpret_cast<float*>(ws + sp.off_lse) : nullptr;
    float* grad_c = grad ? reinterpret_cast<float*>(ws + sp.off_grad) : nullptr;
    float* logprob_c = logprob ? reinterpret_cast<float*>(ws + sp.off_logprob) : nullptr;
    const RowInputs in = {hidden_c, labels_c, lse_c, grad_c, rows, count, logprob_c};
    // rows that a gradient of 0 leaves out have four more bytes each to be counted by everyone
    if (n_tokens <= SELECT_AT_ONCE && !skip_zero_grad) {
        const GatherRows g = {static_cast<const uint16_t*>(hidden), labels, lse, grad, logprob, hdim, rows, count, hidden_c,
                              labels_c, lse_c, grad_c, logprob_c, zero_words, n_zero,
                              static_cast<const uint16_t*>(extra.weight), extra.vocab, extra.c, extra.xref, extra.clear,
                              static_cast<uint16_t*>(extra.zero_rows)};
        hipLaunchKernelGGL(select_gather_kernel, dim3(at_once_grid(n_tokens, hdim)), dim3(AT_ONCE_THREADS), 0, s, row_mask,
                           n_tokens, rows_per_wave(n_tokens, hdim), g);
        return in;
    }
    const float* zero_grads = skip_zero_grad ? grad : nullptr;
    hipLaunchKernelGGL(select_rows_kernel, dim3(1), dim3(SELECT_THREADS), 0, s, row_mask, zero_grads, n_tokens, rows, count,
                       zero_words, n_zero);
    hipLaunchKernelGGL(gather_rows_kernel, dim3((unsigned)n_tokens), dim3(256), 0, s,
                       static_cast<const uint16_t*>(hidden), labels, lse, grad, logprob, rows, count, hdim, hidden_c,
                       labels_c, lse_c, grad_c, logprob_c);
    if (extra.clear)
        hipLaunchKernelGGL(zero_bytes_kernel, dim3((unsigned)((n_tokens + 255) / 256)), dim3(256), 0, s, extra.clear, n_tokens);
    if (extra.xref)
        hipLaunchKernelGGL(label_ref_kernel, dim3((unsigned)((n_tokens + 3) / 4)), dim3(256), 0, s, in.hidden,
                           static_cast<const uint16_t*>(extra.weight), in.labels, in.n_dev, n_tokens, hdim, extra.vocab, extra.c,
                           extra.xref);
    if (extra.zero_rows)
        hipLaunchKernelGGL(zero_unselected_rows_kernel, dim3((unsigned)n_tokens), dim3(256), 0, s, row_mask, zero_grads, hdim,
                           static_cast<uint16_t*>(extra.zero_rows));
    return in;
}

// lse, upstream gradient and logprob of the selected rows (the rows were selected and gathered earlier)
__global__ void gather_f32_kernel(const float* __restrict__ lse, const float* __restrict__ grad,
                                  const float* __restrict__ logprob, const int32_t* __restrict__ rows,
                                  const int32_t* __restrict__ count, float* __restrict__ lse_c,
                                  float* __restrict__ grad_c, float* __restrict__ logprob_c) {
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= *count) return;
    const int64_t src = rows[j];
    lse_c[j] = lse[src];
    grad_c[j] = grad[src];
    logprob_c[j] = logprob[src];
}

template <FwdKeep KEEP>
auto fwd_kernel(int64_t n_tokens, const FwdLaunch& fl) {
    if constexpr (KEEP == FWD_EXPONENTIALS)
        if (n_tokens > BN && n_tokens <= 2 * BN) return lmhead_fwd_kernel<KEEP, TWO_TILES>;
    return n_tokens <= BN            ? lmhead_fwd_kernel<KEEP, ONE_TILE>
           : fl.narrow || fl.either ? lmhead_fwd_kernel<KEEP, NARROW_LAST>
                                    : lmhead_fwd_kernel<KEEP, WHOLE_TILES>;
}

// forward launches: tile kernel + merge of the partial statistics.  `queue` must be zeroed.
// `keep`: where the exponentials of every vocabulary tile go as well (buf null: nowhere).
void enqueue_fwd(const FwdPlan& p, char* ws, const RowInputs& in, const uint8_t* row_mask, const void* weight,
                 int64_t n_tokens, int64_t hidden_dim, int64_t vocab, float inv_temperature, float* logprob,
                 float* entropy, float* lse, const KeepPlan& keep, hipStream_t s) {
    float4* partial = reinterpret_cast<float4*>(ws + p.off_partial);
    float* zy = reinterpret_cast<float*>(ws + p.off_zy);
    uint32_t* queue = reinterpret_cast<uint32_t*>(ws + p.off_queue);
    const float c = inv_temperature * OI_LOG2E;
    const dim3 grid(resident_grid(p.n_splits, p.token_tiles));
    const FwdArgs fa = {static_cast<const uint16_t*>(weight), in.hidden, in.labels, n_tokens, hidden_dim, vocab, c,
                        p.n_pad, partial, zy};
    const FwdLaunch fl = {p.tiles_per_split, p.long_splits, 0, p.long_splits, p.n_splits - p.long_splits,
                          keep.buf, keep.ld, 0, keep.buf ? keep.tiles : 0, 0, keep.xref, keep.logits, p.token_tiles,
                          row_tiles(n_tokens, hidden_dim) != WHOLE_TILES, !keep.logits && either_height(p.token_tiles)};
    auto launch = [&](auto keep_as) {
        hipLaunchKernelGGL(fwd_kernel<decltype(keep_as)::value>(n_tokens, fl), grid, dim3(NTHREADS), 0, s, fa, in.n_dev,
                           fl, queue);
    };
    if (keep.buf) {
        const ProbeScope probe(0, s);
        launch(std::integral_constant<FwdKeep, FWD_EXPONENTIALS>{});
    } else if (keep.logits)
        launch(std::integral_constant<FwdKeep, FWD_LOGITS>{});
    else
        launch(std::integral_constant<FwdKeep, FWD_PLAIN>{});
    hipLaunchKernelGGL(lmhead_fwd_combine_kernel, dim3((unsigned)((n_tokens + COMBINE_TOKENS - 1) / COMBINE_TOKENS)),
                       dim3(COMBINE_THREADS), 0, s, partial,
                       zy, n_tokens, in.n_dev, in.rows, row_mask, n_tokens, p.n_splits, p.n_pad, inv_temperature, c, logprob,
                       entropy, lse, keep.buf ? keep.xref : static_cast<const float*>(nullptr),
                       keep.buf ? keep.unsafe : static_cast<uint8_t*>(nullptr));
}

// scratch for pieces of tiles (none: tiles are not cut)
struct Pieces {
    float* at;
    uint32_t most;
};
Pieces pieces_at(char* at, size_t bytes) {
    return {bytes ? reinterpret_cast<float*>(at) : nullptr, (uint32_t)(bytes / (PART_FLOATS * sizeof(float)))};
}

// A product of token rows with W (k-contiguous x k-major, rows counted on the device): the tile kernel and,
// where its tiles may be split along k, the addition of their pieces.
void launch_rows_product(unsigned grid, const Operand& a, int64_t M, const Operand& b, int64_t N, int64_t K, int mode,
                         float* out_f32, void* out_bf16, int64_t ldo, int64_t m_valid, DynRows dyn, uint32_t* queue,
                         const Pieces& parts, hipStream_t s) {
    uint16_t* o16 = static_cast<uint16_t*>(out_bf16);
    const bool either = parts.at && either_height(M / BM);
    dyn.pieces = either ? parts.most : 0;
    auto* kernel = either ? gemm_store_kernel<false, true, true> : gemm_store_kernel<false, true, false>;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(NTHREADS), 0, s, a, M, b, N, K, mode, out_f32, o16, ldo, m_valid, dyn, queue,
                       parts.at);
    if (!parts.at) return;
    const int64_t tiles = (either ? fewer_tiles(M) : M / BM) * ((N + BN - 1) / BN);
    const int64_t most = tiles < (int64_t)grid ? tiles : (int64_t)grid - 1;  // tiles past the last whole round
    hipLaunchKernelGGL(gemm_reduce_kernel, dim3((unsigned)(most * 4)), dim3(NTHREADS), 0, s, parts.at, grid, M, N, K, mode,
                       out_f32, o16, ldo, m_valid, dyn);
}

// The forward that also prepares d_hidden.  With x = z c in the log2 domain and a per-token
// reference exponent ref_n (the scaled logit of the token's own label),
//   d_hidden[n] = sum_v dZ[n, v] W[v]
//               = s_n sum_{v != y} 2^(x_nv - ref_n) W[v] - g_n inv_T expm1(logprob_n) W[y_n],
//   s_n = -g_n inv_T 2^(ref_n - lse2_n),
// and the sum does not depend on the upstream gradient: it is accumulated while the logits exist,
// one vocabulary chunk at a time (the exponentials of the chunk as bf16 in a chunk-sized buffer,
// with the label's own entry left out; then wsum (+)= E_chunk * W_chunk in fp32).  A backward pass
// that only needs d_hidden is then one pass over [tokens, hidden]: 4 N H V matrix work for forward +
// backward instead of 6 N H V, and nothing is recomputed.  Tokens whose largest logit is too far
// above their label's are flagged in `unsafe`; their sums are not used (the backward recomputes them).
void enqueue_fwd_wsum(const FwdPlan& p, char* ws, const RowInputs& in, const uint8_t* row_mask, const void* weight,
                      int64_t n_tokens, int64_t hidden_dim, int64_t vocab, float inv_temperature, float* logprob,
                      float* entropy, float* lse, float* wsum, float* xref, uint8_t* unsafe, hipStream_t s) {
    float4* partial = reinterpret_cast<float4*>(ws + p.off_partial);
    float* zy = reinterpret_cast<float*>(ws + p.off_zy);
    uint32_t* queues = reinterpret_cast<uint32_t*>(ws + p.off_queue);
    uint16_t* chunk_buf = reinterpret_cast<uint16_t*>(ws + p.off_chunk);
    const Pieces parts = pieces_at(ws + p.off_parts, p.parts_bytes);
    const float c = inv_temperature * OI_LOG2E;
    const uint16_t* Wp = static_cast<const uint16_t*>(weight);
    const int64_t h_tiles = (hidden_dim + BN - 1) / BN;
    const int64_t v_pad = p.vocab_tiles * BM;
    const int64_t splits_per_chunk = (p.chunk / BM + p.tiles_per_split - 1) / p.tiles_per_split;
    const FwdArgs fa = {Wp, in.hidden, in.labels, n_tokens, hidden_dim, vocab, c, p.n_pad, partial, zy};
    for (int64_t ci = 0; ci < p.n_chunks; ++ci) {
        const int64_t v_begin = ci * p.chunk;
        const int64_t v_end = v_begin + p.chunk < v_pad ? v_begin + p.chunk : v_pad;
        const int64_t cols = v_end - v_begin;                                   // multiple of 256
        const int64_t valid = vocab - v_begin < cols ? vocab - v_begin : cols;  // real rows of W
        const int64_t first = ci * splits_per_chunk;
        const int64_t n_first = p.n_splits - first < splits_per_chunk ? p.n_splits - first : splits_per_chunk;
        uint32_t* q = queues + ci * (FWD_QUEUE_WORDS + QUEUE_WORDS);
        const FwdLaunch fl = {p.tiles_per_split, p.long_splits, first, n_first, 0, chunk_buf, cols, v_begin / BM,
                              cols / BM, 1, xref, nullptr, 0, row_tiles(n_tokens, hidden_dim) != WHOLE_TILES,
                              either_height(p.token_tiles)};
        hipLaunchKernelGGL(fwd_kernel<FWD_EXPONENTIALS>(n_tokens, fl),
                           dim3(resident_grid(n_first, p.token_tiles)), dim3(NTHREADS), 0, s, fa,
                           in.n_dev, fl, q);
        const Operand a = {chunk_buf, cols, 0, p.n_pad, cols};
        const Operand b = {Wp + v_begin * hidden_dim, hidden_dim, 0, hidden_dim, valid};
        const DynRows dyn = {in.n_dev, 1, nullptr, nullptr, nullptr, nullptr};
        launch_rows_product(resident_grid(p.n_pad / BM, h_tiles), a, p.n_pad, b, hidden_dim, round_up(valid, BK),
                            ci == 0 ? 0 : 1, wsum, nullptr, hidden_dim, n_tokens, dyn, q + FWD_QUEUE_WORDS, parts, s);
    }
    hipLaunchKernelGGL(lmhead_fwd_combine_kernel, dim3((unsigned)((n_tokens + COMBINE_TOKENS - 1) / COMBINE_TOKENS)),
                       dim3(COMBINE_THREADS), 0, s, partial,
                       zy, n_tokens, in.n_dev, in.rows, row_mask, n_tokens, p.n_splits, p.n_pad, inv_temperature, c, logprob,
                       entropy, lse, static_cast<const float*>(xref), unsafe);
}

// d_hidden row of token n from the weighted sum that the forward left behind for it, row j among the selected; zero where it
// was not selected.  THREADS threads for each row.  The factor s is applied in two halves so that neither leaves the fp32
// range.  Rows flagged in `unsafe` are left alone (the recomputing backward writes them).
struct WsumInputs {
    const float *wsum, *xref;
    const uint8_t* unsafe;
    const uint16_t* W;
    const int64_t* labels;
    const float *lse, *logprob, *grad;
    int64_t hdim, vocab;
    float inv_t;
    uint16_t* d_hidden;
};
template <int THREADS>
__device__ __forceinline__ void dh_row_from_wsum(const WsumInputs& a, int64_t n, bool selected, int64_t j) {
    constexpr int UNROLL = 8 * OI_WAVE / THREADS;
    const int lane = threadIdx.x & (THREADS - 1);
    uint2* dst = reinterpret_cast<uint2*>(a.d_hidden + n * a.hdim);
    if (!selected) {
        for (int64_t c = lane; c < a.hdim / 4; c += THREADS) dst[c] = make_uint2(0u, 0u);
        return;
    }
    if (a.unsafe[n]) return;
    const float g = a.grad[n] * a.inv_t;
    const float half = __builtin_amdgcn_exp2f(0.5f * (a.xref[j] - a.lse[n] * OI_LOG2E));
    const float sb = -g * half;
    const float tl = -g * expm1f(a.logprob[n]);
    int64_t y = a.labels[n];
    y = y < 0 ? 0 : (y >= a.vocab ? a.vocab - 1 : y);
    const float4* src = reinterpret_cast<const float4*>(a.wsum + j * a.hdim);
    const uint2* wy = reinterpret_cast<const uint2*>(a.W + y * a.hdim);
#pragma unroll UNROLL
    for (int64_t c = lane; c < a.hdim / 4; c += THREADS) {  // hdim is a multiple of 64
        const float4 o = src[c];
        const uint2 w = wy[c];
        const float r0 = o.x * half * sb + tl * oi_bf16lo_to_f32(w.x), r1 = o.y * half * sb + tl * oi_bf16hi_to_f32(w.x);
        const float r2 = o.z * half * sb + tl * oi_bf16lo_to_f32(w.y), r3 = o.w * half * sb + tl * oi_bf16hi_to_f32(w.y);
        dst[c] = make_uint2(oi_pack_bf16x2(r0, r1), oi_pack_bf16x2(r2, r3));
    }
}
__global__ void __launch_bounds__(AT_ONCE_THREADS)
    dh_from_wsum_kernel(const uint8_t* __restrict__ mask, int64_t n, int per_wave, WsumInputs a) {
    for_selected_rows(
        mask, n, per_wave, [&](int64_t row, bool selected, int64_t j) { dh_row_from_wsum<OI_WAVE>(a, row, selected, j); }, [](int) {});
}
// The same where there is nothing to count: all rows, or those of a row index where there are more than are counted at once.
// A workgroup for each row: bytes alone bound it then, and a wave for each row (four in turn past 16384) keeps too few under
// way.  Backward, us, waves and workgroups: all of 32768 rows x 8192 386, 304; of 32768 x 4096 198, 157; of 65600 x 8192 735,
// 635; of 65600 rows by an index 762, 727, x 4096 443, 419, of 131072 x 2048 678, 710 (70 % of them 597, 615).
constexpr int ROW_THREADS = 256;
__global__ void __launch_bounds__(ROW_THREADS)
    dh_from_wsum_rows_kernel(const int32_t* __restrict__ rows, const int32_t* __restrict__ count, WsumInputs a) {
    const int64_t j = blockIdx.x;
    if (count && j >= *count) return;
    dh_row_from_wsum<ROW_THREADS>(a, rows ? (int64_t)rows[j] : j, true, j);
}

// The recomputing backward.  Per vocabulary chunk: dZ [n_pad, cols] (token-major, bf16, zero in padded
// columns and in padded rows up to the next k-tile; rows behind it may never have been written), then both
// products straight from W and the (selected) hidden rows, which enter as k-major operands:
//   d_hidden[n, h] (+)= sum_v dZ[n, v] * W[v_begin + v, h]      A k-contiguous, B k-major
//   d_weight[v_begin + v, h] = sum_n dZ[n, v] * hidden[n, h]    A k-major,      B k-major
// The sums stop at the last real vocabulary row / token (rounded up to a k-tile, whose missing
// rows are read from the last real one and meet zeros of dZ).  The queue words must be zeroed.
// dw_adds: the product is added to the bf16 rows of d_weight that an earlier call wrote, instead of stored there; a call
// without tokens then changes nothing and costs nothing (the rows must be selected on the device).
// logits: the forward's logits (kept_bytes), read instead of recomputed.
// per_xcd > 0 caps the resident workgroups of every launch on each XCD: the launches that serve flagged rows normally find
// none, and a launch over a few CUs that finds nothing costs a fraction of one over all of them.
constexpr unsigned REPAIR_PER_XCD = 4;
void enqueue_bwd(const BwdPlan& p, char* ws, const RowInputs& in, const void* weight, int64_t n_tokens,
                 int64_t hidden_dim, int64_t vocab, float inv_temperature, void* d_hidden, void* d_weight,
                 hipStream_t s, bool dw_adds = false, unsigned per_xcd = 0,
                 const float* logits = nullptr) {
    auto grid_of = [&](int64_t tiles_m, int64_t tiles_n) { return dim3(resident_grid(tiles_m, tiles_n, per_xcd)); };
    uint16_t* dz = reinterpret_cast<uint16_t*>(ws + p.off_dz);
    float* dh32 = reinterpret_cast<float*>(ws + p.off_dh32);
    const Pieces parts = pieces_at(ws + p.off_parts, p.parts_bytes);
    uint32_t* queues = reinterpret_cast<uint32_t*>(ws + p.off_queues);
    const uint16_t* Wp = static_cast<const uint16_t*>(weight);
    const float c = inv_temperature * OI_LOG2E;
    const int64_t h_tiles = (hidden_dim + BN - 1) / BN;
    for (int64_t ci = 0; ci < p.n_chunks; ++ci) {
        const int64_t v_begin = ci * p.chunk;
        const int64_t v_end = (ci + 1) * p.chunk < p.v_pad ? (ci + 1) * p.chunk : p.v_pad;
        const int64_t cols = v_end - v_begin;                                   // multiple of 256
        const int64_t valid = vocab - v_begin < cols ? vocab - v_begin : cols;  // real rows of W
        uint32_t* q = queues + ci * 3 * QUEUE_WORDS;
        const DzInputs di = {in.labels, in.lse, in.grad, in.logprob, n_tokens, vocab, c, inv_temperature};
        if (logits)
            hipLaunchKernelGGL(lmhead_dz_kept_kernel, dim3((unsigned)(p.n_pad / BN * 4), (unsigned)(cols / BM)),
                               dim3(NTHREADS), 0, s, logits, p.n_pad / BN, di, in.n_dev,
                               row_tiles(n_tokens, hidden_dim) != WHOLE_TILES, cols, dz);
        else
            hipLaunchKernelGGL((row_tiles(n_tokens, hidden_dim) == ONE_TILE ? lmhead_dz_kernel<ROUND> : lmhead_dz_kernel<NEAR>),
                               grid_of(cols / BM, p.n_pad / BN), dim3(NTHREADS), 0, s, Wp, in.hidden, di, in.n_dev, hidden_dim, v_begin, cols, p.n_pad, dz, q);
        const bool first = ci == 0, last = ci == p.n_chunks - 1;
        const int mode = last ? (first ? 2 : 3) : (first ? 0 : 1);
        {
            const Operand a = {dz, cols, 0, p.n_pad, cols};
            const Operand b = {Wp + v_begin * hidden_dim, hidden_dim, 0, hidden_dim, valid};
            const DynRows dyn = {in.n_dev, 1, in.rows, nullptr, nullptr, nullptr};
            launch_rows_product(grid_of(p.n_pad / BM, h_tiles).x, a, p.n_pad, b, hidden_dim, round_up(valid, BK), mode,
                                dh32, d_hidden, hidden_dim, n_tokens, dyn, q + QUEUE_WORDS, parts, s);
        }
        if (d_weight) {
            const Operand a = {dz, cols, 0, cols, round_up(n_tokens, BK)};
            const Operand b = {in.hidden, hidden_dim, 0, hidden_dim, n_tokens};
            uint16_t* dw = static_cast<uint16_t*>(d_weight) + v_begin * hidden_dim;
            const dim3 grid = grid_of(cols / BM, h_tiles);
            if (dw_adds)
                hipLaunchKernelGGL(gemm_add_kernel, grid, dim3(NTHREADS), 0, s, a, valid, b, hidden_dim, dw, hidden_dim, in.n_dev,
                                   q + 2 * QUEUE_WORDS);
            else
                hipLaunchKernelGGL((gemm_store_kernel<true, true>), grid, dim3(NTHREADS), 0, s, a, cols, b, hidden_dim,
                                   round_up(n_tokens, BK), 2, static_cast<float*>(nullptr), dw, hidden_dim, valid,
                                   DynRows{in.n_dev, 2, nullptr, nullptr, nullptr, nullptr}, q + 2 * QUEUE_WORDS,
                                   static_cast<float*>(nullptr));
        }
    }
}

// Both backward products of a slab from its kept exponentials (see slab_prepare_kernel): the whole
// vocabulary as one chunk, d_hidden rows stored once through the slab's row numbers, d_weight
// stored / accumulated as *dw_mode_dev says (the slab's place among the slabs of the call is known
// on the device only: the first one stores, the last one rounds to bf16, see SlabMeta).
// `queues`: 2 * QUEUE_WORDS zeroed words.
void enqueue_products_from_exponentials(const uint16_t* ecache, int64_t cache_ld, int64_t slab_pad,
                                        const int32_t* count, const int32_t* rows_s, const float* scale_a,
                                        const float* scale_b, const uint16_t* scaled_hidden, const void* weight,
                                        int64_t hidden_dim, int64_t vocab, void* d_hidden, void* d_weight,
                                        const int32_t* dw_mode_dev, float* dw32, uint32_t* queues, const Pieces& parts,
                                        hipStream_t s) {
    const uint16_t* Wp = static_cast<const uint16_t*>(weight);
    const int64_t h_tiles = (hidden_dim + BN - 1) / BN;
    {
        const ProbeScope probe(1, s);
        const Operand a = {ecache, cache_ld, 0, slab_pad, cache_ld};
        const Operand b = {Wp, hidden_dim, 0, hidden_dim, vocab};
        const DynRows dyn = {count, 1, rows_s, scale_a, scale_b, nullptr};
        launch_rows_product(resident_grid(slab_pad / BM, h_tiles), a, slab_pad, b, hidden_dim, round_up(vocab, BK), 2,
                            nullptr, d_hidden, hidden_dim, slab_pad, dyn, queues, parts, s);
    }
    if (d_weight) {
        const ProbeScope probe(2, s);
        const Operand a = {ecache, cache_ld, 0, cache_ld, slab_pad};
        const Operand b = {scaled_hidden, hidden_dim, 0, hidden_dim, slab_pad};
        const DynRows dyn = {count, 2, nullptr, nullptr, nullptr, dw_mode_dev};
        hipLaunchKernelGGL((gemm_store_kernel<true, true>), dim3(resident_grid(cache_ld / BM, h_tiles)),
                           dim3(NTHREADS), 0, s, a, cache_ld, b, hidden_dim, round_up(slab_pad, BK), 2, dw32,
                           static_cast<uint16_t*>(d_weight), hidden_dim, vocab, dyn, queues + QUEUE_WORDS,
                           static_cast<float*>(nullptr));
    }
}

// workspace of the whole-step entry point: forward and backward regions side by side (they share
// one row selection), the statistics partials, and the per-token vectors that connect the stages
struct StepPlan {
    FwdPlan fwd;
    BwdPlan bwd;
    size_t off_fwd, off_bwd, off_stats, off_lse, off_grad, off_denoms, total;
};
StepPlan plan_step(int64_t rows, int64_t cols, int64_t hdim, int64_t vocab) {
    StepPlan p;
    const int64_t n = rows * cols;
    p.fwd = plan_fwd(n, hdim, vocab, false);
    p.bwd = plan_bwd(n, hdim, vocab, true);
    Carver cv;
    p.off_fwd = cv.take(p.fwd.total);
    p.off_bwd = cv.take(p.bwd.total);
    p.off_stats = cv.take(oi_grpo_fused_workspace_bytes(rows, cols));
    p.off_lse = cv.take((size_t)n * sizeof(float));
    p.off_grad = cv.take((size_t)n * sizeof(float));
    p.off_denoms = cv.take((size_t)rows * sizeof(float));
    p.total = cv.off;
    return p;
}

// ---------------------------------------------------------------------------------------------
// The whole step in slabs of tokens, with nothing recomputed
// ---------------------------------------------------------------------------------------------
// The selected rows are taken a slab at a time (at most `cap` rows; the slabs of a call are made
// equal on the device, where the selected count lives).  A slab's forward leaves its exponentials
// (every vocabulary column, bf16, relative to each token's own reference exponent) in a slab-sized
// buffer, the slab's tokens get their upstream gradient at once (the caller of run_slab_passes says
// how: for the GRPO loss it depends only on the token's own logprob and on denominators that come
// from the mask), and both products read the buffer before the next slab overwrites it: d_hidden
// rows are final, d_weight accumulates in fp32 over the slabs.  6 N H V of matrix work instead of
// 8 N H V; the buffer holds [slab, vocabulary], never [tokens, vocabulary].  Tokens that the
// forward flags (largest logit too far above the label's) add nothing in their slab and are served
// by one recomputing backward over the flagged rows after the last slab, so the results do not
// depend on the size of the logits.  Every slab costs a pass over the fp32 d_weight and leaves the
// ends of its launches ragged.
constexpr int64_t SLAB_UNIT = 256;  // a slab capacity is a multiple of this many rows (a token tile)
constexpr int SLAB_QUEUE_WORDS = FWD_QUEUE_WORDS + 2 * QUEUE_WORDS;
struct SlabPlan {
    int64_t cap, n_passes, n_pad, v_pad;
    FwdPlan fwd;     // of one slab
    BwdPlan repair;  // the recomputing backward over all rows (for the flagged ones)
    size_t off_fwd, off_order, off_count, off_meta, off_unsafe, off_keep, off_repair, off_hidden_s, off_labels_s,
        off_rows_s, off_xref_s, off_scale_a, off_scale_b, off_scaled_hidden, off_queues, off_dw32, off_stats, off_lse,
        off_grad, off_denoms, off_parts, total;
    size_t parts_bytes;
};
SlabPlan plan_slabs(int64_t n, int64_t stats_rows, int64_t stats_cols, int64_t hdim, int64_t vocab, bool want_dw,
                    int64_t slab_tokens, int64_t n_passes_override = 0) {
    SlabPlan p;
    p.n_pad = round_up(n, 256);
    p.v_pad = round_up(vocab, 256);
    const int64_t cap = round_up(slab_tokens < SLAB_UNIT ? SLAB_UNIT : slab_tokens, SLAB_UNIT);
    p.cap = p.n_pad < cap ? p.n_pad : cap;
    p.n_passes = n_passes_override > 0 ? n_passes_override : (p.n_pad + p.cap - 1) / p.cap;
    p.fwd = plan_fwd(p.cap, hdim, vocab, false);
    p.repair = plan_bwd(n, hdim, vocab, true, true);
    Carver cv;
    p.off_fwd = cv.take(p.fwd.total);
    p.off_order = cv.take((size_t)p.n_pad * sizeof(int32_t));
    p.off_count = cv.take(sizeof(int32_t));
    p.off_meta = cv.take((size_t)p.n_passes * sizeof(SlabMeta));
    p.off_unsafe = cv.take((size_t)p.n_pad);
    // the slab's exponentials and, after the last slab, the workspace of the repair share one region
    const size_t keep_bytes = (size_t)p.cap * p.v_pad * 2;
    p.off_keep = p.off_repair = cv.take(keep_bytes > p.repair.total ? keep_bytes : p.repair.total);
    p.off_hidden_s = cv.take((size_t)p.cap * hdim * 2);
    p.off_labels_s = cv.take((size_t)p.cap * sizeof(int64_t));
    p.off_rows_s = cv.take((size_t)p.cap * sizeof(int32_t));
    p.off_xref_s = cv.take((size_t)p.cap * sizeof(float));
    p.off_scale_a = cv.take((size_t)p.cap * sizeof(float));
    p.off_scale_b = cv.take((size_t)p.cap * sizeof(float));
    p.off_scaled_hidden = cv.take(want_dw ? (size_t)p.cap * hdim * 2 : 0);
    p.off_queues = cv.take((size_t)p.n_passes * SLAB_QUEUE_WORDS * sizeof(uint32_t));
    p.off_dw32 = cv.take(want_dw && p.n_passes > 1 ? (size_t)vocab * hdim * sizeof(float) : 0);
    p.off_stats = cv.take(oi_grpo_fused_workspace_bytes(stats_rows, stats_cols));
    p.off_lse = cv.take((size_t)n * sizeof(float));
    p.off_grad = cv.take((size_t)n * sizeof(float));
    p.off_denoms = cv.take((size_t)stats_rows * sizeof(float));
    p.parts_bytes = split_bytes(p.cap / BM, (hdim + BN - 1) / BN, p.v_pad, vocab);
    p.off_parts = cv.take(p.parts_bytes);
    p.total = cv.off;
    return p;
}

// The selected rows split into the fewest slabs of at most `cap` rows: all of the same size (a multiple of
// 256 rows, the last one takes what is left), or, when that takes fewer rounds of tiles, full slabs of
// `cap` rows and a last one with the remainder.  What is counted is the slab's d_hidden product, the one
// tile kernel whose work items are long (a tile runs over the whole vocabulary): it has
// ceil(rows / 256) * h_tiles tiles for `grid` resident workgroups, in whole rounds.  A last round that is
// mostly empty is cut along the vocabulary (plan_tail) and costs less than that, so the choice matters little:
// steps at 4096 x 128256, full slabs of 8192 against equal ones, 8500 rows 21.6 to 21.8 against 22.0 ms, 9472 rows 24.6
// against 24.6, 12288 rows 30.5 to 31.3 against 30.6 to 31.4, 16640 rows 43.2 against 43.1.  Passes past the last slab
// are empty.
struct SlabPlanning {
    int cap, n_passes, h_tiles, grid;
    SlabMeta* meta;
};
// of n selected rows, pass i
__device__ __forceinline__ void plan_slab(const SlabPlanning& p, int n, int i) {
    const int cap = p.cap, h_tiles = p.h_tiles, grid = p.grid;
    SlabMeta* meta = p.meta;
    const int k = n > 0 ? (n + cap - 1) / cap : 1;
    int equal = ((n + k - 1) / k + 255) / 256 * 256;
    equal = equal > cap ? cap : equal;
    auto rounds = [&](int size) {
        int total = 0;
        for (int j = 0; j < k; ++j) {
            const int left = n - j * size;
            const int rows = left < 0 ? 0 : (left > size ? size : left);
            total += ((rows + 255) / 256 * h_tiles + grid - 1) / grid;
        }
        return total;
    };
    const int size = rounds(cap) < rounds(equal) ? cap : equal;
    const int left = n - i * size;
    meta[i].offset = i * size;
    meta[i].count = left < 0 ? 0 : (left > size ? size : left);
    const bool first = i == 0, last = i == k - 1;
    meta[i].dw_mode = i >= k ? -1 : (last ? (first ? 2 : 3) : (first ? 0 : 1));
    meta[i].reserved = 0;
}

// What a step starts from: the queue words of every pass and the marks of the rows (n_pad bytes) are
// cleared, and the per-token outputs are zero: rows that take no part stay there, and the passes that look
// at every row before its own slab has run (the upstream gradient of a slab's pairs) read zeros rather than whatever the
// caller's buffers held.  d_hidden rows of tokens that take no part are zero.
struct SlabSetup {
    const uint8_t* mask;
    int64_t n, n_pad, queue_words, hdim;
    float *logprob, *entropy, *lse;
    uint32_t *unsafe, *queues;
    uint16_t* d_hidden;
};
// The share of workgroup `block` of `blocks` of 1024 threads, four rows of d_hidden at a time
constexpr int SETUP_THREADS = 1024, SETUP_ROWS = 4;
__device__ __forceinline__ void slab_setup(const SlabSetup& a, int64_t block, int64_t blocks) {
    const int64_t first = block * SETUP_THREADS + threadIdx.x, stride = blocks * SETUP_THREADS;
    for (int64_t i = first; i < a.n; i += stride) {
        a.logprob[i] = 0.f;
        if (a.entropy) a.entropy[i] = 0.f;
        a.lse[i] = 0.f;
    }
    for (int64_t i = first; i < a.n_pad / 4; i += stride) a.unsafe[i] = 0u;
    for (int64_t i = first; i < a.queue_words; i += stride) a.queues[i] = 0u;
    const int64_t row = block * SETUP_ROWS + (threadIdx.x >> 8);
    if (row >= a.n || row_selected(a.mask, nullptr, row)) return;
    uint32_t* out = reinterpret_cast<uint32_t*>(a.d_hidden + row * a.hdim);  // hdim is a multiple of 64
    for (int64_t c = threadIdx.x & 255; c < a.hdim / 2; c += 256) out[c] = 0u;
}
inline int64_t setup_blocks(int64_t n) { return (n + SETUP_ROWS - 1) / SETUP_ROWS; }
__global__ void __launch_bounds__(SETUP_THREADS) slab_setup_kernel(SlabSetup a) { slab_setup(a, blockIdx.x, gridDim.x); }

// The start of a GRPO step in one launch: workgroup 0 selects the rows, plans the slabs and, where one denominator serves
// all rows, leaves it in row_denoms; the others set up.  A small launch is 5 us of the stream, and a step of few rows is
// three products and small launches: as five launches this took 23 us of the 1050 of a step of 268 rows.
struct GrpoStart {
    int32_t *order, *count;
    SlabPlanning planning;
    float* row_denoms;  // null: the denominators are the rows' own
    int64_t rows;
    float denominator;
};
static_assert(SETUP_THREADS == SELECT_THREADS, "one launch");
__global__ void __launch_bounds__(SETUP_THREADS) grpo_start_kernel(SlabSetup a, GrpoStart g) {
    if (blockIdx.x > 0) return slab_setup(a, blockIdx.x - 1, gridDim.x - 1);
    const int n = select_rows(a.mask, nullptr, a.n, g.order);
    if (threadIdx.x == 0) *g.count = n;
    for (int i = threadIdx.x; i < g.planning.n_passes; i += SETUP_THREADS) plan_slab(g.planning, n, i);
    if (!g.row_denoms) return;
    const double den = g.denominator > 0.f ? (double)g.denominator : (double)n;
    const float inv = (float)(den > 0.0 ? 1.0 / den : 0.0);  // as grpo_stats_final_kernel leaves it
    for (int64_t r = threadIdx.x; r < g.rows; r += SETUP_THREADS) g.row_denoms[r] = inv;
}

// What a slab-wise step is made of besides the passes themselves
struct SlabStep {
    const void *hidden, *weight;
    const int64_t* labels;       // per caller row, as the kernels score them
    const uint8_t* mask;         // per caller row: the rows that are multiplied
    int64_t n_tokens, hidden_dim, vocab;
    float inv_temperature;
    float *logprob, *entropy;    // per caller row (entropy may be null)
    void *d_hidden, *d_weight;   // d_weight may be null
};

// Runs the slab passes of `st` over the row index order[0 .. *count) that `start` leaves in the
// workspace together with the passes' SlabMeta, once it has set up what SlabSetup says (it returns a status: reading one
// clears it).  `upstream()` may enqueue kernels and returns, by reference, a status and the upstream gradient as
// slab_prepare_kernel takes it, given the logprobs computed so far (the rows of the slabs up to the current one; in the
// last pass, all rows).
template <class Start, class Upstream>
int run_slab_passes(const SlabPlan& p, char* ws, const SlabStep& st, hipStream_t s, Start&& start, Upstream&& upstream) {
    const int64_t n = st.n_tokens, hdim = st.hidden_dim, vocab = st.vocab;
    char* ws_fwd = ws + p.off_fwd;
    int32_t* order = reinterpret_cast<int32_t*>(ws + p.off_order);
    int32_t* count = reinterpret_cast<int32_t*>(ws + p.off_count);
    SlabMeta* meta = reinterpret_cast<SlabMeta*>(ws + p.off_meta);
    uint8_t* unsafe = reinterpret_cast<uint8_t*>(ws + p.off_unsafe);
    uint16_t* keep_buf = reinterpret_cast<uint16_t*>(ws + p.off_keep);
    uint16_t* hidden_s = reinterpret_cast<uint16_t*>(ws + p.off_hidden_s);
    int64_t* labels_s = reinterpret_cast<int64_t*>(ws + p.off_labels_s);
    int32_t* rows_s = reinterpret_cast<int32_t*>(ws + p.off_rows_s);
    float* xref_s = reinterpret_cast<float*>(ws + p.off_xref_s);
    float* scale_a = reinterpret_cast<float*>(ws + p.off_scale_a);
    float* scale_b = reinterpret_cast<float*>(ws + p.off_scale_b);
    uint16_t* scaled_hidden = st.d_weight ? reinterpret_cast<uint16_t*>(ws + p.off_scaled_hidden) : nullptr;
    uint32_t* queues = reinterpret_cast<uint32_t*>(ws + p.off_queues);
    float* dw32 = st.d_weight && p.n_passes > 1 ? reinterpret_cast<float*>(ws + p.off_dw32) : nullptr;
    float* lse = reinterpret_cast<float*>(ws + p.off_lse);
    float* grad = reinterpret_cast<float*>(ws + p.off_grad);
    const Pieces parts = pieces_at(ws + p.off_parts, p.parts_bytes);
    const uint16_t* hid = static_cast<const uint16_t*>(st.hidden);

    const SlabSetup setup = {st.mask, n, p.n_pad, p.n_passes * SLAB_QUEUE_WORDS, hdim, st.logprob, st.entropy, lse,
                             reinterpret_cast<uint32_t*>(unsafe), queues, static_cast<uint16_t*>(st.d_hidden)};
    const int started = start(setup, order, count, meta);
    if (started != OI_OK) return started;
    for (int64_t i = 0; i < p.n_passes; ++i) {
        const int32_t* cnt = &meta[i].count;
        uint32_t* pass_queues = queues + i * SLAB_QUEUE_WORDS;
        hipLaunchKernelGGL(gather_slab_kernel, dim3((unsigned)p.cap), dim3(256), 0, s, hid,
                           static_cast<const uint16_t*>(st.weight), st.labels, order, meta + i, hdim, vocab,
                           st.inv_temperature * OI_LOG2E, hidden_s, labels_s, rows_s, xref_s);
        const RowInputs in = {hidden_s, labels_s, nullptr, nullptr, rows_s, cnt, nullptr};
        const KeepPlan keep = {keep_buf, p.v_pad, p.v_pad / BM, xref_s, unsafe, nullptr};
        // the forward's own queue words are the first FWD_QUEUE_WORDS of the pass
        FwdPlan fp = p.fwd;
        fp.off_queue = (size_t)(reinterpret_cast<char*>(pass_queues) - ws_fwd);
        enqueue_fwd(fp, ws_fwd, in, nullptr, st.weight, p.cap, hdim, vocab, st.inv_temperature, st.logprob, st.entropy,
                    lse, keep, s);
        int rc = OI_OK;
        const auto gradient = upstream(rc);
        if (rc != OI_OK) return rc;
        hipLaunchKernelGGL(slab_prepare_kernel, dim3((unsigned)p.cap), dim3(256), 0, s, gradient, lse, grad, st.logprob, unsafe,
                           rows_s, labels_s, xref_s, meta + i, st.inv_temperature, vocab, hdim, keep_buf, p.v_pad,
                           hidden_s, scale_a, scale_b, scaled_hidden);
        enqueue_products_from_exponentials(keep_buf, p.v_pad, p.cap, cnt, rows_s, scale_a, scale_b, scaled_hidden,
                                           st.weight, hdim, vocab, st.d_hidden, st.d_weight, &meta[i].dw_mode, dw32,
                                           pass_queues + FWD_QUEUE_WORDS, parts, s);
    }
    // the flagged rows, if any: one recomputing backward over them (its workspace takes the place of
    // the exponentials), added to what the slabs left in d_weight; the upstream gradients are those of the last
    // pass, which saw every logprob
    {
        char* ws_rep = ws + p.off_repair;
        uint32_t* rq = reinterpret_cast<uint32_t*>(ws_rep + p.repair.off_queues);
        const int n_words = (int)(3 * p.repair.n_chunks * QUEUE_WORDS);
        const bool select_clears = n_words <= SELECT_THREADS;
        if (!select_clears)
            hipLaunchKernelGGL(zero_words_kernel, dim3((unsigned)((n_words + 255) / 256)), dim3(256), 0, s, rq, n_words);
        const RowInputs in = launch_selection(p.repair.sel, ws_rep, st.hidden, st.labels, lse, grad, unsafe, false, n,
                                              hdim, rq, select_clears ? n_words : 0, s, st.logprob);
        enqueue_bwd(p.repair, ws_rep, in, st.weight, n, hdim, vocab, st.inv_temperature, st.d_hidden, st.d_weight, s, true,
                    REPAIR_PER_XCD);
    }
    return oi_launch_status();
}

}  // namespace

extern "C" size_t oi_lmhead_fwd_workspace_bytes(int64_t n_tokens, int64_t hidden_dim, int64_t vocab,
                                                int with_row_mask) {
    if (n_tokens <= 0 || vocab <= 0 || hidden_dim <= 0) return 0;
    return plan_fwd(n_tokens, hidden_dim, vocab, with_row_mask != 0).total;
}

namespace {
// `logits`: null, or kept_bytes of memory for the backward that follows
int lmhead_forward(const void* hidden, const void* weight, const int64_t* labels, const uint8_t* row_mask,
                   int64_t n_tokens, int64_t hidden_dim, int64_t vocab, float inv_temperature, float* logprob,
                   float* entropy, float* lse, float* logits, void* workspace, size_t workspace_bytes, void* stream) {
    const FwdPlan p = plan_fwd(n_tokens, hidden_dim, vocab, row_mask != nullptr);
    OI_RETURN_IF(workspace_bytes < p.total, OI_EWORKSPACE);
    char* ws = static_cast<char*>(workspace);
    uint32_t* queue = reinterpret_cast<uint32_t*>(ws + p.off_queue);
    hipStream_t s = static_cast<hipStream_t>(stream);
    RowInputs in = {static_cast<const uint16_t*>(hidden), labels, nullptr, nullptr, nullptr, nullptr, nullptr};
    if (row_mask)
        in = launch_selection(p.sel, ws, hidden, labels, nullptr, nullptr, row_mask, false, n_tokens, hidden_dim, queue,
                              FWD_QUEUE_WORDS, s);
    else
        hipLaunchKernelGGL(zero_words_kernel, dim3(1), dim3(64), 0, s, queue, FWD_QUEUE_WORDS);
    KeepPlan keep = {};
    keep.logits = logits;
    enqueue_fwd(p, ws, in, row_mask, weight, n_tokens, hidden_dim, vocab, inv_temperature, logprob, entropy, lse, keep, s);
    return oi_launch_status();
}
}  // namespace

extern "C" int oi_lmhead_logp_fwd(const void* hidden, const void* weight, const int64_t* labels,
                                  const uint8_t* row_mask, int64_t n_tokens, int64_t hidden_dim, int64_t vocab,
                                  float inv_temperature, float* logprob, float* entropy, float* lse, void* workspace,
                                  size_t workspace_bytes, void* stream) {
    int rc = check_lmhead(hidden, weight, labels, n_tokens, hidden_dim, vocab, inv_temperature);
    if (rc != OI_OK) return rc;
    if (n_tokens == 0) return OI_OK;
    OI_RETURN_IF(!logprob || !workspace, OI_ENULL);
    OI_RETURN_IF(!oi_aligned(workspace, 256), OI_EALIGN);
    return lmhead_forward(hidden, weight, labels, row_mask, n_tokens, hidden_dim, vocab, inv_temperature, logprob, entropy,
                          lse, nullptr, workspace, workspace_bytes, stream);
}

extern "C" size_t oi_lmhead_kept_bytes(int64_t n_tokens, int64_t vocab) {
    if (n_tokens <= 0 || vocab <= 0 || n_tokens > MAX_LD || vocab > MAX_LD) return 0;
    return kept_bytes(n_tokens, vocab);
}

extern "C" int oi_lmhead_logp_fwd_kept(const void* hidden, const void* weight, const int64_t* labels,
                                       const uint8_t* row_mask, int64_t n_tokens, int64_t hidden_dim, int64_t vocab,
                                       float inv_temperature, float* logprob, float* entropy, float* lse, float* logits,
                                       size_t logits_bytes, void* workspace, size_t workspace_bytes, void* stream) {
    int rc = check_lmhead(hidden, weight, labels, n_tokens, hidden_dim, vocab, inv_temperature);
    if (rc != OI_OK) return rc;
    if (n_tokens == 0) return OI_OK;
    OI_RETURN_IF(!logprob || !lse || !logits || !workspace, OI_ENULL);
    OI_RETURN_IF(!oi_aligned(workspace, 256) || !oi_aligned(logits, 16), OI_EALIGN);
    const size_t need = kept_bytes(n_tokens, vocab);
    OI_RETURN_IF(need == 0 || logits_bytes < need, OI_EWORKSPACE);
    return lmhead_forward(hidden, weight, labels, row_mask, n_tokens, hidden_dim, vocab, inv_temperature, logprob, entropy,
                          lse, logits, workspace, workspace_bytes, stream);
}

extern "C" size_t oi_lmhead_fwd_wsum_workspace_bytes(int64_t n_tokens, int64_t hidden_dim, int64_t vocab,
                                                     int with_row_mask) {
    if (n_tokens <= 0 || vocab <= 0 || hidden_dim <= 0) return 0;
    return plan_fwd(n_tokens, hidden_dim, vocab, with_row_mask != 0, true).total;
}

extern "C" int oi_lmhead_logp_fwd_wsum(const void* hidden, const void* weight, const int64_t* labels,
                                       const uint8_t* row_mask, int64_t n_tokens, int64_t hidden_dim, int64_t vocab,
                                       float inv_temperature, float* logprob, float* entropy, float* lse, float* wsum,
                                       float* xref, uint8_t* unsafe, void* workspace, size_t workspace_bytes,
                                       void* stream) {
    int rc = check_lmhead(hidden, weight, labels, n_tokens, hidden_dim, vocab, inv_temperature);
    if (rc != OI_OK) return rc;
    if (n_tokens == 0) return OI_OK;
    OI_RETURN_IF(!logprob || !lse || !wsum || !xref || !unsafe || !workspace, OI_ENULL);
    OI_RETURN_IF(!oi_aligned(workspace, 256) || !oi_aligned(wsum, 16) || !oi_aligned(xref, 4), OI_EALIGN);
    const FwdPlan p = plan_fwd(n_tokens, hidden_dim, vocab, row_mask != nullptr, true);
    OI_RETURN_IF(workspace_bytes < p.total, OI_EWORKSPACE);
    char* ws = static_cast<char*>(workspace);
    uint32_t* queues = reinterpret_cast<uint32_t*>(ws + p.off_queue);
    const int n_queue_words = (int)(p.n_chunks * (FWD_QUEUE_WORDS + QUEUE_WORDS));
    hipStream_t s = static_cast<hipStream_t>(stream);
    RowInputs in = {static_cast<const uint16_t*>(hidden), labels, nullptr, nullptr, nullptr, nullptr, nullptr};
    const bool select_clears_queues = row_mask && n_queue_words <= SELECT_THREADS;
    if (!select_clears_queues)
        hipLaunchKernelGGL(zero_words_kernel, dim3((unsigned)((n_queue_words + 255) / 256)), dim3(256), 0, s, queues,
                           n_queue_words);
    if (row_mask) {
        const SelectionExtras extra = {weight, vocab, inv_temperature * OI_LOG2E, xref, unsafe, nullptr};
        in = launch_selection(p.sel, ws, hidden, labels, nullptr, nullptr, row_mask, false, n_tokens, hidden_dim, queues,
                              select_clears_queues ? n_queue_words : 0, s, nullptr, extra);
    } else {
        hipLaunchKernelGGL(zero_bytes_kernel, dim3((unsigned)((n_tokens + 255) / 256)), dim3(256), 0, s, unsafe, n_tokens);
        hipLaunchKernelGGL(label_ref_kernel, dim3((unsigned)((n_tokens + 3) / 4)), dim3(256), 0, s, in.hidden,
                           static_cast<const uint16_t*>(weight), in.labels, in.n_dev, n_tokens, hidden_dim, vocab,
                           inv_temperature * OI_LOG2E, xref);
    }
    enqueue_fwd_wsum(p, ws, in, row_mask, weight, n_tokens, hidden_dim, vocab, inv_temperature, logprob, entropy, lse,
                     wsum, xref, unsafe, s);
    return oi_launch_status();
}

namespace {
// workspace of oi_lmhead_dh_from_wsum: the row index of the mask, and the recomputing backward for
// the rows that the forward flagged
struct DhPlan {
    BwdPlan repair;
    size_t off_rows, off_count, off_repair, total;
};
DhPlan plan_dh(int64_t n_tokens, int64_t hdim, int64_t vocab) {
    DhPlan p;
    p.repair = plan_bwd(n_tokens, hdim, vocab, true, true);
    Carver cv;
    p.off_rows = cv.take((size_t)round_up(n_tokens, 256) * sizeof(int32_t));
    p.off_count = cv.take(sizeof(int32_t));
    p.off_repair = cv.take(p.repair.total);
    p.total = cv.off;
    return p;
}
}  // namespace

extern "C" size_t oi_lmhead_dh_workspace_bytes(int64_t n_tokens, int64_t hidden_dim, int64_t vocab) {
    if (n_tokens <= 0 || hidden_dim <= 0 || vocab <= 0) return 0;
    return plan_dh(n_tokens, hidden_dim, vocab).total;
}

extern "C" int oi_lmhead_dh_from_wsum(const void* hidden, const void* weight, const int64_t* labels, const float* lse,
                                      const float* logprob, const float* grad_logprob, const uint8_t* row_mask,
                                      const float* wsum, const float* xref, const uint8_t* unsafe, int64_t n_tokens,
                                      int64_t hidden_dim, int64_t vocab, float inv_temperature, void* d_hidden,
                                      void* workspace, size_t workspace_bytes, void* stream) {
    int rc = check_lmhead(hidden, weight, labels, n_tokens, hidden_dim, vocab, inv_temperature);
    if (rc != OI_OK) return rc;
    if (n_tokens == 0) return OI_OK;
    OI_RETURN_IF(!lse || !logprob || !grad_logprob || !wsum || !xref || !unsafe || !d_hidden || !workspace, OI_ENULL);
    OI_RETURN_IF(!oi_aligned(wsum, 16) || !oi_aligned(d_hidden, 8) || !oi_aligned(workspace, 256), OI_EALIGN);
    const DhPlan p = plan_dh(n_tokens, hidden_dim, vocab);
    OI_RETURN_IF(workspace_bytes < p.total, OI_EWORKSPACE);
    hipStream_t s = static_cast<hipStream_t>(stream);
    char* ws = static_cast<char*>(workspace);
    // the same ascending selection as in the forward pass, from the same mask
    const WsumInputs wi = {wsum, xref, unsafe, static_cast<const uint16_t*>(weight), labels, lse, logprob, grad_logprob, hidden_dim,
                           vocab, inv_temperature, static_cast<uint16_t*>(d_hidden)};
    if (row_mask && n_tokens <= SELECT_AT_ONCE) {
        hipLaunchKernelGGL(dh_from_wsum_kernel, dim3(at_once_grid(n_tokens, hidden_dim)), dim3(AT_ONCE_THREADS), 0, s,
                           row_mask, n_tokens, rows_per_wave(n_tokens, hidden_dim), wi);
    } else {
        const int32_t *rows = nullptr, *count = nullptr;
        if (row_mask) {
            int32_t* r = reinterpret_cast<int32_t*>(ws + p.off_rows);
            int32_t* c = reinterpret_cast<int32_t*>(ws + p.off_count);
            hipLaunchKernelGGL(select_rows_kernel, dim3(1), dim3(SELECT_THREADS), 0, s, row_mask,
                               static_cast<const float*>(nullptr), n_tokens, r, c, static_cast<uint32_t*>(nullptr), 0);
            hipLaunchKernelGGL(zero_unselected_rows_kernel, dim3((unsigned)n_tokens), dim3(256), 0, s, row_mask,
                               static_cast<const float*>(nullptr), hidden_dim, static_cast<uint16_t*>(d_hidden));
            rows = r;
            count = c;
        }
        hipLaunchKernelGGL(dh_from_wsum_rows_kernel, dim3((unsigned)n_tokens), dim3(ROW_THREADS), 0, s, rows, count, wi);
    }
    // the flagged rows (a subset of the mask's), recomputed; normally none
    char* ws_rep = ws + p.off_repair;
    uint32_t* rq = reinterpret_cast<uint32_t*>(ws_rep + p.repair.off_queues);
    const int n_words = (int)(3 * p.repair.n_chunks * QUEUE_WORDS);
    const bool select_clears = n_words <= SELECT_THREADS;
    if (!select_clears)
        hipLaunchKernelGGL(zero_words_kernel, dim3((unsigned)((n_words + 255) / 256)), dim3(256), 0, s, rq, n_words);
    const RowInputs in = launch_selection(p.repair.sel, ws_rep, hidden, labels, lse, grad_logprob, unsafe, false,
                                          n_tokens, hidden_dim, rq, select_clears ? n_words : 0, s, logprob);
    enqueue_bwd(p.repair, ws_rep, in, weight, n_tokens, hidden_dim, vocab, inv_temperature, d_hidden, nullptr, s, false,
                REPAIR_PER_XCD);
    return oi_launch_status();
}

extern "C" size_t oi_lmhead_bwd_workspace_bytes(int64_t n_tokens, int64_t hidden_dim, int64_t vocab,
                                                int want_d_weight, int with_row_selection) {
    if (n_tokens <= 0 || hidden_dim <= 0 || vocab <= 0) return 0;
    (void)want_d_weight;
    return plan_bwd(n_tokens, hidden_dim, vocab, with_row_selection != 0).total;
}

namespace {
// `logits`: null, or what the forward over the same rows (the same mask, no rows skipped) left behind
int lmhead_backward(const void* hidden, const void* weight, const int64_t* labels, const float* lse,
                    const float* grad_logprob, const uint8_t* row_mask, int skip_zero_grad_rows, int64_t n_tokens,
                    int64_t hidden_dim, int64_t vocab, float inv_temperature, const float* logprob, const float* logits,
                    void* d_hidden, void* d_weight, void* workspace, size_t workspace_bytes, void* stream) {
    int rc = check_lmhead(hidden, weight, labels, n_tokens, hidden_dim, vocab, inv_temperature);
    if (rc != OI_OK) return rc;
    if (n_tokens == 0) return OI_OK;
    OI_RETURN_IF(!lse || !grad_logprob || !logprob || !d_hidden || !workspace, OI_ENULL);
    // bf16 results are stored as pairs (4-byte words)
    OI_RETURN_IF(!oi_aligned(workspace, 256) || !oi_aligned(d_hidden, 4) || !oi_aligned(d_weight, 4), OI_EALIGN);
    const bool selecting = row_mask != nullptr || skip_zero_grad_rows != 0;
    const BwdPlan p = plan_bwd(n_tokens, hidden_dim, vocab, selecting);
    OI_RETURN_IF(workspace_bytes < p.total, OI_EWORKSPACE);
    hipStream_t s = static_cast<hipStream_t>(stream);
    char* ws = static_cast<char*>(workspace);
    uint32_t* queues = reinterpret_cast<uint32_t*>(ws + p.off_queues);
    const int n_queue_words = (int)(3 * p.n_chunks * QUEUE_WORDS);
    RowInputs in = {static_cast<const uint16_t*>(hidden), labels, lse, grad_logprob, nullptr, nullptr, logprob};
    const bool select_clears_queues = selecting && n_queue_words <= SELECT_THREADS;
    if (!select_clears_queues)
        hipLaunchKernelGGL(zero_words_kernel, dim3((unsigned)((n_queue_words + 255) / 256)), dim3(256), 0, s, queues,
                           n_queue_words);
    if (selecting)
        in = launch_selection(p.sel, ws, hidden, labels, lse, grad_logprob, row_mask, skip_zero_grad_rows != 0, n_tokens,
                              hidden_dim, queues, select_clears_queues ? n_queue_words : 0, s, logprob,
                              SelectionExtras{nullptr, 0, 0.f, nullptr, nullptr, d_hidden});
    enqueue_bwd(p, ws, in, weight, n_tokens, hidden_dim, vocab, inv_temperature, d_hidden, d_weight, s, false,
                0, logits);
    return oi_launch_status();
}
}  // namespace

extern "C" int oi_lmhead_logp_bwd(const void* hidden, const void* weight, const int64_t* labels, const float* lse,
                                  const float* grad_logprob, const uint8_t* row_mask, int skip_zero_grad_rows,
                                  int64_t n_tokens, int64_t hidden_dim, int64_t vocab, float inv_temperature,
                                  const float* logprob, void* d_hidden, void* d_weight, void* workspace,
                                  size_t workspace_bytes, void* stream) {
    return lmhead_backward(hidden, weight, labels, lse, grad_logprob, row_mask, skip_zero_grad_rows, n_tokens, hidden_dim,
                           vocab, inv_temperature, logprob, nullptr, d_hidden, d_weight, workspace, workspace_bytes,
                           stream);
}

extern "C" int oi_lmhead_logp_bwd_kept(const void* hidden, const void* weight, const int64_t* labels, const float* lse,
                                       const float* grad_logprob, const uint8_t* row_mask, int64_t n_tokens,
                                       int64_t hidden_dim, int64_t vocab, float inv_temperature, const float* logprob,
                                       const float* logits, size_t logits_bytes, void* d_hidden, void* d_weight,
                                       void* workspace, size_t workspace_bytes, void* stream) {
    if (n_tokens > 0) {
        OI_RETURN_IF(!logits, OI_ENULL);
        OI_RETURN_IF(!oi_aligned(logits, 16), OI_EALIGN);
        const size_t need = oi_lmhead_kept_bytes(n_tokens, vocab);
        OI_RETURN_IF(need == 0 || logits_bytes < need, OI_EWORKSPACE);
    }
    return lmhead_backward(hidden, weight, labels, lse, grad_logprob, row_mask, 0, n_tokens, hidden_dim, vocab,
                           inv_temperature, logprob, logits, d_hidden, d_weight, workspace, workspace_bytes, stream);
}


extern "C" size_t oi_lmhead_grpo_workspace_bytes(int64_t rows, int64_t cols, int64_t hidden_dim, int64_t vocab,
                                                 int want_d_weight, int64_t slab_tokens) {
    if (rows <= 0 || cols <= 0 || hidden_dim <= 0 || vocab <= 0) return 0;
    if (slab_tokens > 0) return plan_slabs(rows * cols, rows, cols, hidden_dim, vocab, want_d_weight != 0, slab_tokens).total;
    return plan_step(rows, cols, hidden_dim, vocab).total;
}

namespace {
// oi_lmhead_grpo_fwd_bwd in slabs of tokens (slab_tokens > 0); arguments as checked by the entry point
int grpo_step_in_slabs(const void* hidden, const void* weight, const int64_t* labels, const uint8_t* mask,
                       const float* old_logprobs, const float* ref_logprobs, const float* advantages,
                       const float* rho_weights, int64_t rows, int64_t cols, int64_t hidden_dim, int64_t vocab,
                       float inv_temperature, int loss_fn, float ratio_lo, float ratio_hi, int kl_estimator, float beta,
                       int axis_mode, float denominator, float scale, float* logprob, float* entropy, float* out_stats,
                       void* d_hidden, void* d_weight, int64_t slab_tokens, void* workspace, size_t workspace_bytes,
                       void* stream) {
    const int64_t n_tokens = rows * cols;
    const SlabPlan p = plan_slabs(n_tokens, rows, cols, hidden_dim, vocab, d_weight != nullptr, slab_tokens);
    OI_RETURN_IF(workspace_bytes < p.total, OI_EWORKSPACE);
    hipStream_t s = static_cast<hipStream_t>(stream);
    char* ws = static_cast<char*>(workspace);
    float* grad = reinterpret_cast<float*>(ws + p.off_grad);
    float* row_denoms = reinterpret_cast<float*>(ws + p.off_denoms);
    int rc = oi_check_grpo(rows, cols, axis_mode, loss_fn, kl_estimator);
    if (rc != OI_OK) return rc;
    const SlabStep st = {hidden, weight, labels, mask, n_tokens, hidden_dim, vocab, inv_temperature, logprob, entropy,
                         d_hidden, d_weight};
    rc = run_slab_passes(
        p, ws, st, s,
        [&](const SlabSetup& setup, int32_t* order, int32_t* count, SlabMeta* meta) {
            const int64_t h_tiles = (hidden_dim + BN - 1) / BN;
            const SlabPlanning planning = {(int)p.cap, (int)p.n_passes, (int)h_tiles, (int)resident_grid(p.cap / BM, h_tiles), meta};
            const GrpoStart g = {order, count, planning, axis_mode == 0 ? row_denoms : nullptr, rows, denominator};
            hipLaunchKernelGGL(grpo_start_kernel, dim3((unsigned)(1 + setup_blocks(n_tokens))), dim3(SETUP_THREADS), 0, s, setup, g);
            // the denominators come from the mask alone
            return axis_mode == 0 ? oi_launch_status()
                                  : oi_launch_grpo_denoms(mask, rows, cols, denominator, row_denoms, s);
        },
        // every token's d loss / d logprob from its own logprob
        [&](int&) {
            return GrpoUpstream{logprob, old_logprobs, ref_logprobs, advantages, rho_weights, row_denoms, cols,
                                GrpoCfg{loss_fn, ratio_lo, ratio_hi, kl_estimator}, beta, scale};
        });
    if (rc != OI_OK) return rc;
    // loss and statistics from all logprobs
    return oi_grpo_fused_fwd(logprob, old_logprobs, ref_logprobs, advantages, mask, rho_weights, entropy, nullptr, nullptr,
                             nullptr, nullptr, rows, cols, loss_fn, ratio_lo, ratio_hi, kl_estimator, beta, axis_mode,
                             denominator, scale, out_stats, row_denoms, ws + p.off_stats,
                             oi_grpo_fused_workspace_bytes(rows, cols), stream);
}
}  // namespace

extern "C" int oi_lmhead_grpo_fwd_bwd(const void* hidden, const void* weight, const int64_t* labels,
                                      const uint8_t* mask, const float* old_logprobs, const float* ref_logprobs,
                                      const float* advantages, const float* rho_weights, int64_t rows, int64_t cols,
                                      int64_t hidden_dim, int64_t vocab, float inv_temperature, int loss_fn,
                                      float ratio_lo, float ratio_hi, int kl_estimator, float beta, int axis_mode,
                                      float denominator, float scale, float* logprob, float* entropy, float* out_stats,
                                      void* d_hidden, void* d_weight, int64_t slab_tokens, void* workspace,
                                      size_t workspace_bytes, void* stream) {
    OI_RETURN_IF(rows <= 0 || cols <= 0 || rows > MAX_LD || cols > MAX_LD || slab_tokens < 0, OI_EINVAL);
    const int64_t n_tokens = rows * cols;
    int rc = check_lmhead(hidden, weight, labels, n_tokens, hidden_dim, vocab, inv_temperature);
    if (rc != OI_OK) return rc;
    OI_RETURN_IF(!mask || !advantages || !logprob || !out_stats || !d_hidden || !workspace, OI_ENULL);
    OI_RETURN_IF(!oi_aligned(workspace, 256) || !oi_aligned(d_hidden, 4) || !oi_aligned(d_weight, 4), OI_EALIGN);
    if (slab_tokens > 0)
        return grpo_step_in_slabs(hidden, weight, labels, mask, old_logprobs, ref_logprobs, advantages, rho_weights, rows,
                                  cols, hidden_dim, vocab, inv_temperature, loss_fn, ratio_lo, ratio_hi, kl_estimator,
                                  beta, axis_mode, denominator, scale, logprob, entropy, out_stats, d_hidden, d_weight,
                                  slab_tokens, workspace, workspace_bytes, stream);
    const StepPlan p = plan_step(rows, cols, hidden_dim, vocab);
    OI_RETURN_IF(workspace_bytes < p.total, OI_EWORKSPACE);
    hipStream_t s = static_cast<hipStream_t>(stream);
    char* ws = static_cast<char*>(workspace);
    char* ws_fwd = ws + p.off_fwd;
    char* ws_bwd = ws + p.off_bwd;
    float* lse = reinterpret_cast<float*>(ws + p.off_lse);
    float* grad = reinterpret_cast<float*>(ws + p.off_grad);
    float* row_denoms = reinterpret_cast<float*>(ws + p.off_denoms);

    // one selection for both passes: it lives in the backward region; the select kernel also clears
    // the backward queues, the forward queue gets the small fill kernel
    uint32_t* fwd_queue = reinterpret_cast<uint32_t*>(ws_fwd + p.fwd.off_queue);
    uint32_t* bwd_queues = reinterpret_cast<uint32_t*>(ws_bwd + p.bwd.off_queues);
    const int n_queue_words = (int)(3 * p.bwd.n_chunks * QUEUE_WORDS);
    const bool select_clears_queues = n_queue_words <= SELECT_THREADS;
    hipLaunchKernelGGL(zero_words_kernel, dim3(1), dim3(64), 0, s, fwd_queue, FWD_QUEUE_WORDS);
    if (!select_clears_queues)
        hipLaunchKernelGGL(zero_words_kernel, dim3((unsigned)((n_queue_words + 255) / 256)), dim3(256), 0, s,
                           bwd_queues, n_queue_words);
    RowInputs in = launch_selection(p.bwd.sel, ws_bwd, hidden, labels, nullptr, nullptr, mask, false, n_tokens,
                                    hidden_dim, bwd_queues, select_clears_queues ? n_queue_words : 0, s, nullptr,
                                    SelectionExtras{nullptr, 0, 0.f, nullptr, nullptr, d_hidden});
    enqueue_fwd(p.fwd, ws_fwd, in, mask, weight, n_tokens, hidden_dim, vocab, inv_temperature, logprob, entropy, lse,
                KeepPlan{}, s);

    // loss and statistics from the logprobs, then every token's d loss / d logprob (upstream gradient 1)
    rc = oi_grpo_fused_fwd(logprob, old_logprobs, ref_logprobs, advantages, mask, rho_weights, entropy, nullptr, nullptr,
                           nullptr, nullptr, rows, cols, loss_fn, ratio_lo, ratio_hi, kl_estimator, beta, axis_mode,
                           denominator, scale, out_stats, row_denoms, ws + p.off_stats,
                           oi_grpo_fused_workspace_bytes(rows, cols), stream);
    if (rc != OI_OK) return rc;
    rc = oi_grpo_fused_bwd(logprob, old_logprobs, ref_logprobs, advantages, mask, rho_weights, rows, cols, loss_fn,
                           ratio_lo, ratio_hi, kl_estimator, beta, scale, row_denoms, nullptr, grad, stream);
    if (rc != OI_OK) return rc;

    float* lse_c = reinterpret_cast<float*>(ws_bwd + p.bwd.sel.off_lse);
    float* grad_c = reinterpret_cast<float*>(ws_bwd + p.bwd.sel.off_grad);
    float* logprob_c = reinterpret_cast<float*>(ws_bwd + p.bwd.sel.off_logprob);
    hipLaunchKernelGGL(gather_f32_kernel, dim3((unsigned)((n_tokens + 255) / 256)), dim3(256), 0, s, lse, grad, logprob,
                       in.rows, in.n_dev, lse_c, grad_c, logprob_c);
    in.lse = lse_c;
    in.grad = grad_c;
    in.logprob = logprob_c;
    enqueue_bwd(p.bwd, ws_bwd, in, weight, n_tokens, hidden_dim, vocab, inv_temperature, d_hidden, d_weight, s);
    return oi_launch_status();
}

// ---------------------------------------------------------------------------------------------
// The whole DPO step on hidden states, in slabs of whole chosen / rejected pairs
// ---------------------------------------------------------------------------------------------
namespace {
// Workgroup s handles sequence s: every position t of its range gets the label it is scored against
// (labels[t + 1]) and a mask byte (that label is not -100); the number of scored positions goes to
// cnt[s].  The positions that belong to no range (the last one of a padded row, of the packed row)
// are masked out.
__global__ void __launch_bounds__(256)
    dpo_rows_kernel(const int64_t* __restrict__ labels, const int32_t* __restrict__ cu, int64_t n_seqs, int64_t total,
                    int64_t* __restrict__ labels_eff, uint8_t* __restrict__ mask, int32_t* __restrict__ cnt) {
    const int64_t s = blockIdx.x;
    int64_t a, b;
    oi_seq_range(cu, s, n_seqs, total, &a, &b);
    float c = 0.f;
    for (int64_t t = a + threadIdx.x; t < b; t += blockDim.x) {
        const int64_t y = labels[t + 1];
        labels_eff[t] = y;
        const bool keep = y != -100;
        mask[t] = keep ? 1 : 0;
        c += keep ? 1.f : 0.f;
    }
    __shared__ float scratch[16];
    c = oi_block_sum(c, scratch);  // exact: at most 2^22 positions per sequence
    if (threadIdx.x == 0) {
        cnt[s] = (int32_t)c;
        const int64_t last = cu ? (s == n_seqs - 1 ? total - 1 : -1) : s * total + total - 1;
        if (last >= 0) {
            labels_eff[last] = -100;
            mask[last] = 0;
        }
    }
}

// One thread.  The scored rows are taken pair by pair (pair p = sequences p and n_seqs / 2 + p, the
// chosen and the rejected answer to one prompt: open_instruct/dpo_utils.py:734-763, 876-877): off[s]
// is where sequence s starts in the row index, and the slabs are filled with whole pairs in that order
// (a pair that does not fit the current slab starts the next one), because the upstream gradient of a
// token depends on the logprob sums of both sequences of its pair and must be known when the slab's
// exponentials are multiplied.  A pair with more rows than a slab holds is cut across slabs and its
// sequences are marked (seq_unsafe): their tokens take the recomputing backward after the last slab.
// Two consecutive slabs always hold more than `cap` rows together, so 2 ceil(rows / cap) + 1 passes
// are enough.
__global__ void dpo_plan_kernel(const int32_t* __restrict__ cnt, int n_seqs, int cap, int n_passes,
                                int32_t* __restrict__ off, uint8_t* __restrict__ seq_unsafe, int32_t* __restrict__ count,
                                SlabMeta* __restrict__ meta) {
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    const int bs = n_seqs / 2;
    int run = 0;
    for (int p = 0; p < bs; ++p) {
        off[p] = run;
        run += cnt[p];
        off[bs + p] = run;
        run += cnt[bs + p];
    }
    *count = run;
    int i = 0, start = 0, fill = 0;
    auto close = [&]() {
        if (i < n_passes) {
            meta[i].offset = start;
            meta[i].count = fill;
        }
        ++i;
        start += fill;
        fill = 0;
    };
    for (int p = 0; p < bs; ++p) {
        int rows = cnt[p] + cnt[bs + p];
        const bool oversize = rows > cap;
        seq_unsafe[p] = seq_unsafe[bs + p] = oversize ? 1 : 0;
        if (oversize) {
            while (rows > 0) {
                const int take = rows < cap - fill ? rows : cap - fill;
                fill += take;
                rows -= take;
                if (fill == cap) close();
            }
        } else {
            if (fill + rows > cap) close();
            fill += rows;
        }
    }
    if (fill > 0) close();
    const int k = i < n_passes ? i : n_passes;  // slabs with rows (at least the one that stores zeros)
    for (int j = k; j < n_passes; ++j) {
        meta[j].offset = start;
        meta[j].count = 0;
    }
    const int kk = k > 0 ? k : 1;
    for (int j = 0; j < n_passes; ++j) {
        const bool first = j == 0, last = j == kk - 1;
        meta[j].dw_mode = j >= kk ? -1 : (last ? (first ? 2 : 3) : (first ? 0 : 1));
        meta[j].reserved = 0;
    }
}

// Workgroup s writes the scored positions of sequence s, in ascending order, to
// order[off[s] .. off[s] + cnt[s]) and marks them in `unsafe` when the sequence is marked.
__global__ void __launch_bounds__(256)
    dpo_order_kernel(const uint8_t* __restrict__ mask, const int32_t* __restrict__ cu, int64_t n_seqs, int64_t total,
                     const int32_t* __restrict__ off, const uint8_t* __restrict__ seq_unsafe,
                     int32_t* __restrict__ order, uint8_t* __restrict__ unsafe) {
    const int64_t s = blockIdx.x;
    int64_t a, b;
    oi_seq_range(cu, s, n_seqs, total, &a, &b);
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int64_t per = (b - a + 255) / 256;
    const int64_t lo = a + t * per, hi = lo + per < b ? lo + per : b;
    int c = 0;
    for (int64_t i = lo; i < hi; ++i) c += mask[i] ? 1 : 0;
    int incl = c;
#pragma unroll
    for (int o = 1; o < OI_WAVE; o <<= 1) {
        const int up = __shfl_up(incl, o, OI_WAVE);
        if (lane >= o) incl += up;
    }
    __shared__ int wave_total[4];
    if (lane == OI_WAVE - 1) wave_total[wave] = incl;
    __syncthreads();
    int base = 0;
    for (int w = 0; w < wave; ++w) base += wave_total[w];
    int pos = off[s] + base + incl - c;
    const bool flag = seq_unsafe[s] != 0;
    for (int64_t i = lo; i < hi; ++i)
        if (mask[i]) {
            order[pos++] = (int32_t)i;
            if (flag) unsafe[i] = 1;
        }
}

__global__ void fill_f32_kernel(float* __restrict__ p, int64_t n, float v) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

struct DpoPlan {
    SlabPlan slabs;
    int64_t n, bs;
    size_t off_slabs, off_labels_eff, off_mask, off_cnt, off_off, off_seq_unsafe, off_counts, off_dseq, off_gl, total;
};
DpoPlan plan_dpo(int64_t n_seqs, int64_t total, bool packed, int64_t hdim, int64_t vocab, bool want_dw,
                 int64_t slab_tokens) {
    DpoPlan p;
    p.n = packed ? total : n_seqs * total;
    p.bs = n_seqs / 2;
    const int64_t n_pad = round_up(p.n, 256);
    const int64_t cap = round_up(slab_tokens < SLAB_UNIT ? SLAB_UNIT : slab_tokens, SLAB_UNIT);
    const int64_t cap_eff = n_pad < cap ? n_pad : cap;
    // everything fits one slab when the batch does; otherwise see dpo_plan_kernel
    const int64_t n_passes = n_pad <= cap ? 1 : 2 * ((n_pad + cap_eff - 1) / cap_eff) + 1;
    p.slabs = plan_slabs(p.n, 1, 1, hdim, vocab, want_dw, slab_tokens, n_passes);
    Carver cv;
    p.off_slabs = cv.take(p.slabs.total);
    p.off_labels_eff = cv.take((size_t)p.n * sizeof(int64_t));
    p.off_mask = cv.take((size_t)p.n);
    p.off_cnt = cv.take((size_t)n_seqs * sizeof(int32_t));
    p.off_off = cv.take((size_t)n_seqs * sizeof(int32_t));
    p.off_seq_unsafe = cv.take((size_t)n_seqs);
    p.off_counts = cv.take((size_t)n_seqs * sizeof(float));
    p.off_dseq = cv.take((size_t)n_seqs * sizeof(float));
    p.off_gl = cv.take((size_t)p.bs * sizeof(float));
    p.total = cv.off;
    return p;
}
}  // namespace

extern "C" size_t oi_lmhead_dpo_workspace_bytes(int64_t n_seqs, int64_t total, int packed, int64_t hidden_dim,
                                                int64_t vocab, int want_d_weight, int64_t slab_tokens) {
    if (n_seqs <= 0 || total <= 0 || hidden_dim <= 0 || vocab <= 0 || slab_tokens <= 0) return 0;
    return plan_dpo(n_seqs, total, packed != 0, hidden_dim, vocab, want_d_weight != 0, slab_tokens).total;
}

extern "C" int oi_lmhead_dpo_fwd_bwd(const void* hidden, const void* weight, const int64_t* labels,
                                     const int32_t* cu_seq_lens, int64_t n_seqs, int64_t total, int64_t hidden_dim,
                                     int64_t vocab, float inv_temperature, const float* ref_chosen,
                                     const float* ref_rejected, float beta, float label_smoothing, float margin,
                                     int average_log_prob, float grad_scale, float* per_token_logps, float* seq_logps,
                                     float* losses, float* chosen_rewards, float* rejected_rewards, void* d_hidden,
                                     void* d_weight, int64_t slab_tokens, void* workspace, size_t workspace_bytes,
                                     void* stream) {
    OI_RETURN_IF(n_seqs < 2 || n_seqs % 2 != 0 || total < 1 || slab_tokens <= 0, OI_EINVAL);
    OI_RETURN_IF(n_seqs > MAX_LD || total > MAX_LD, OI_EINVAL);
    const bool packed = cu_seq_lens != nullptr;
    const int64_t n_tokens = packed ? total : n_seqs * total;
    int rc = check_lmhead(hidden, weight, labels, n_tokens, hidden_dim, vocab, inv_temperature);
    if (rc != OI_OK) return rc;
    OI_RETURN_IF((ref_chosen == nullptr) != (ref_rejected == nullptr), OI_EINVAL);
    OI_RETURN_IF(!per_token_logps || !seq_logps || !losses || !d_hidden || !workspace, OI_ENULL);
    OI_RETURN_IF(!oi_aligned(workspace, 256) || !oi_aligned(d_hidden, 4) || !oi_aligned(d_weight, 4), OI_EALIGN);
    const DpoPlan p = plan_dpo(n_seqs, total, packed, hidden_dim, vocab, d_weight != nullptr, slab_tokens);
    OI_RETURN_IF(workspace_bytes < p.total, OI_EWORKSPACE);
    hipStream_t s = static_cast<hipStream_t>(stream);
    char* ws = static_cast<char*>(workspace);
    char* ws_slabs = ws + p.off_slabs;
    int64_t* labels_eff = reinterpret_cast<int64_t*>(ws + p.off_labels_eff);
    uint8_t* mask = reinterpret_cast<uint8_t*>(ws + p.off_mask);
    int32_t* cnt = reinterpret_cast<int32_t*>(ws + p.off_cnt);
    int32_t* off = reinterpret_cast<int32_t*>(ws + p.off_off);
    uint8_t* seq_unsafe = reinterpret_cast<uint8_t*>(ws + p.off_seq_unsafe);
    float* counts = reinterpret_cast<float*>(ws + p.off_counts);
    float* d_seq = reinterpret_cast<float*>(ws + p.off_dseq);
    float* grad_losses = reinterpret_cast<float*>(ws + p.off_gl);
    float* grad = reinterpret_cast<float*>(ws_slabs + p.slabs.off_grad);
    uint8_t* unsafe = reinterpret_cast<uint8_t*>(ws_slabs + p.slabs.off_unsafe);
    const int64_t bs = p.bs;

    hipLaunchKernelGGL(dpo_rows_kernel, dim3((unsigned)n_seqs), dim3(256), 0, s, labels, cu_seq_lens, n_seqs, total,
                       labels_eff, mask, cnt);
    hipLaunchKernelGGL(fill_f32_kernel, dim3((unsigned)((bs + 63) / 64)), dim3(64), 0, s, grad_losses, bs, grad_scale);
    const SlabStep st = {hidden, weight, labels_eff, mask, n_tokens, hidden_dim, vocab, inv_temperature, per_token_logps,
                         nullptr, d_hidden, d_weight};
    // per-sequence sums of the logprobs computed so far, the loss derivative of every pair, and from it
    // every token's d loss / d logprob (right for the pairs whose tokens are all there)
    auto upstream = [&](int& r) {
        r = oi_seq_logp_fwd(per_token_logps, labels, cu_seq_lens, n_seqs, total, average_log_prob, seq_logps, counts, stream);
        if (r == OI_OK)
            r = oi_dpo_sigmoid_bwd(seq_logps, seq_logps + bs, ref_chosen, ref_rejected, nullptr, grad_losses, bs, beta,
                                   label_smoothing, margin, d_seq, d_seq + bs, stream);
        if (r == OI_OK)
            r = oi_seq_logp_bwd(d_seq, labels, cu_seq_lens, counts, n_seqs, total, average_log_prob, grad, stream);
        return StoredUpstream{};
    };
    rc = run_slab_passes(
        p.slabs, ws_slabs, st, s,
        [&](const SlabSetup& setup, int32_t* order, int32_t* count, SlabMeta* meta) {
            hipLaunchKernelGGL(slab_setup_kernel, dim3((unsigned)setup_blocks(n_tokens)), dim3(SETUP_THREADS), 0, s, setup);
            hipLaunchKernelGGL(dpo_plan_kernel, dim3(1), dim3(1), 0, s, cnt, (int)n_seqs, (int)p.slabs.cap,
                               (int)p.slabs.n_passes, off, seq_unsafe, count, meta);
            hipLaunchKernelGGL(dpo_order_kernel, dim3((unsigned)n_seqs), dim3(256), 0, s, mask, cu_seq_lens, n_seqs, total,
                               off, seq_unsafe, order, unsafe);
            return oi_launch_status();
        },
        upstream);
    if (rc != OI_OK) return rc;
    // the sums are those of the last upstream pass (every logprob was there); losses and rewards from them
    return oi_dpo_sigmoid_fwd(seq_logps, seq_logps + bs, ref_chosen, ref_rejected, nullptr, bs, beta, label_smoothing,
                              margin, losses, chosen_rewards, rejected_rewards, stream);
}

extern "C" int oi_lmhead_probe_arm(int kernel) {
    OI_RETURN_IF(kernel < 0 || kernel > 2 || g_probe.kernel >= 0, OI_EINVAL);
    for (int i = 0; i < 2 * Probe::MAX_LAUNCHES; ++i) {
        const hipError_t e = hipEventCreate(&g_probe.ev[i]);
        if (e != hipSuccess) {
            for (int j = 0; j < i; ++j) (void)hipEventDestroy(g_probe.ev[j]);
            return (int)e;
        }
    }
    g_probe.used = 0;
    g_probe.kernel = kernel;
    return OI_OK;
}

extern "C" int oi_lmhead_probe_read(float* ms, int capacity, int* n_launches) {
    OI_RETURN_IF(g_probe.kernel < 0 || capacity < 0, OI_EINVAL);
    OI_RETURN_IF(!n_launches || (capacity > 0 && !ms), OI_ENULL);
    const int n = g_probe.used < capacity ? g_probe.used : capacity;
    int rc = OI_OK;
    for (int i = 0; i < n && rc == OI_OK; ++i) {
        hipError_t e = hipEventSynchronize(g_probe.ev[2 * i + 1]);
        if (e == hipSuccess) e = hipEventElapsedTime(&ms[i], g_probe.ev[2 * i], g_probe.ev[2 * i + 1]);
        if (e != hipSuccess) rc = (int)e;
    }
    *n_launches = g_probe.used;
    for (int i = 0; i < 2 * Probe::MAX_LAUNCHES; ++i) (void)hipEventDestroy(g_probe.ev[i]);
    g_probe.kernel = -1;
    g_probe.used = 0;
    return rc;
}

extern "C" int oi_gemm_bf16_tn(const void* A, int64_t lda, int64_t M, const void* B, int64_t ldb, int64_t N, int64_t K,
                               float* out_f32, void* out_bf16, int64_t ldo, int accumulate, void* stream) {
    OI_RETURN_IF(M <= 0 || N <= 0 || K <= 0 || K % 64 != 0 || ldo < N, OI_EINVAL);
    OI_RETURN_IF(lda < 0 || ldb < 0 || lda % 8 != 0 || ldb % 8 != 0, OI_EINVAL);
    OI_RETURN_IF((lda != 0 && lda < K) || (ldb != 0 && ldb < K), OI_EINVAL);
    OI_RETURN_IF(lda > MAX_LD || ldb > MAX_LD, OI_EINVAL);
    OI_RETURN_IF(!A || !B || (!out_f32 && !out_bf16) || (out_f32 && out_bf16), OI_ENULL);
    OI_RETURN_IF(accumulate && !out_f32, OI_EINVAL);
    OI_RETURN_IF(!oi_aligned(A, 16) || !oi_aligned(B, 16), OI_EALIGN);
    // bf16 rows of even pitch are written as pairs (4-byte words), fp32 results as single words
    OI_RETURN_IF(!oi_aligned(out_f32, 4) || !oi_aligned(out_bf16, (ldo & 1) ? 2 : 4), OI_EALIGN);
    const Operand a = {static_cast<const uint16_t*>(A), lda, 0, M, K};
    const Operand b = {static_cast<const uint16_t*>(B), ldb, 0, N, K};
    return launch_product<false, false>(a, M, b, N, K, out_f32, out_bf16, ldo, accumulate, static_cast<hipStream_t>(stream));
}

extern "C" int oi_gemm_bf16_layouts(const void* A, int64_t lda, int a_k_major, const void* B, int64_t ldb,
                                    int b_k_major, int64_t M, int64_t N, int64_t K, float* out_f32, void* out_bf16,
                                    int64_t ldo, int accumulate, void* stream) {
    OI_RETURN_IF(M <= 0 || N <= 0 || K <= 0 || K % 64 != 0 || ldo < N, OI_EINVAL);
    OI_RETURN_IF(lda <= 0 || ldb <= 0 || lda % 8 != 0 || ldb % 8 != 0 || lda > MAX_LD || ldb > MAX_LD, OI_EINVAL);
    // a k-major operand is read in 16-byte column chunks: whole chunks only
    OI_RETURN_IF(lda < (a_k_major ? M : K) || ldb < (b_k_major ? N : K), OI_EINVAL);
    OI_RETURN_IF((a_k_major && M % 8 != 0) || (b_k_major && N % 8 != 0), OI_EINVAL);
    OI_RETURN_IF(!A || !B || (!out_f32 && !out_bf16) || (out_f32 && out_bf16), OI_ENULL);
    OI_RETURN_IF(accumulate && !out_f32, OI_EINVAL);
    OI_RETURN_IF(!oi_aligned(A, 16) || !oi_aligned(B, 16), OI_EALIGN);
    // bf16 rows of even pitch are written as pairs (4-byte words), fp32 results as single words
    OI_RETURN_IF(!oi_aligned(out_f32, 4) || !oi_aligned(out_bf16, (ldo & 1) ? 2 : 4), OI_EALIGN);
    const Operand a = {static_cast<const uint16_t*>(A), lda, 0, M, K};
    const Operand b = {static_cast<const uint16_t*>(B), ldb, 0, N, K};
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (a_k_major && b_k_major) return launch_product<true, true>(a, M, b, N, K, out_f32, out_bf16, ldo, accumulate, s);
    if (a_k_major) return launch_product<true, false>(a, M, b, N, K, out_f32, out_bf16, ldo, accumulate, s);
    if (b_k_major) return launch_product<false, true>(a, M, b, N, K, out_f32, out_bf16, ldo, accumulate, s);
    return launch_product<false, false>(a, M, b, N, K, out_f32, out_bf16, ldo, accumulate, s);
}
