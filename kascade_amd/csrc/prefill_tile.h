// Pieces of the prefill attention kernels (prefill.hip): tile geometry, the
// LDS chunk permutation, direct-to-LDS loads and the workgroup -> unit mapping.
#pragma once
#include "budgets.h"
#include "prefill.h"

namespace kascade {
namespace {

// Tile geometry of the attention kernels per head dimension, whatever products they use.  A tile is 16 KB of K (and of
// V) whatever D: 64 keys at D = 128, 128 keys at D = 64, so a wavefront always stages a tile with four 1 KB loads per
// tensor, each product takes as many matrix instructions per tile and 32 queries (16 of 32x32x16, 32 of 16x16x32),
// and the score registers a narrower head frees hold the extra keys.
template <int D> struct AttnTile {
    static constexpr int kKT = 64 * 128 / D;     // keys per tile
    static constexpr int kChunks = D / 8;        // 16-byte chunks of a row
    static constexpr int kRowsPerLoad = 64 / kChunks;   // rows one wavefront-wide 16-byte load covers
    static constexpr int kTileElems = kKT * D;   // 16 KB of K (and of V) whatever D
};

// Chunk permutation of a tile row in LDS (see the head of the file).  What it must give:
// lane (dq, col) reading chunk 4 ks + dq of row col (A operand of S^T), and the 16 lanes of each quarter dq reading
// rows 4 dq .. 4 dq + 3 x 2 consecutive chunks in 8-byte halves (transposing read of V),
// each touch all 64 banks once.  Rows are 256 bytes (D = 128: the row does not move the bank)
// or 128 bytes (D = 64: the row parity picks the bank half, three more row bits permute).  The hardware serves a
// 16-byte read in groups that mix lanes 0-3 and 12-15 of one quarter with lanes 4-11 of the next, whose chunks
// differ in bit 0: hence -(row / 4), not row / 4, in the low bits.
template <int D> __device__ __forceinline__ int swz16(int row);
template <> __device__ __forceinline__ int swz16<128>(int row) { return ((row & 3) << 2) | (-(row >> 2) & 3); }
template <> __device__ __forceinline__ int swz16<64>(int row) { return (((row >> 1) & 1) << 2) | (-(row >> 2) & 3); }

// The same for operands of 32 rows (lane (lg, li) reads chunk 2 ks + lg of row li; V in quarters of 4 rows x 4 chunks)
template <int D> __device__ __forceinline__ int swz(int row);
template <> __device__ __forceinline__ int swz<128>(int row) { return ((row & 3) << 2) | ((row >> 2) & 3); }
template <> __device__ __forceinline__ int swz<64>(int row) { return (((row >> 1) & 1) << 2) | ((row >> 2) & 3); }

// Exponentials of 16x16x32 products in the places they have after 32x32x16 ones.  A result of 16 columns has a column
// in four lanes, of 32 columns in two; v_permlane16_swap of two results of 16 columns each gives lane (lg, li) rows
// 0 .. 3 of quarter 2 lg (first) and 2 lg + 1 (second) of column li.  With operand row r taken from row pair_row(r) of
// the 16 that is rows 4 lg + (0..3) and 8 + 4 lg + (0..3), as a 32x32x16 product has them.
__device__ __forceinline__ int pair_row(int r) { return (r & ~12) | ((r & 4) << 1) | ((r & 8) >> 1); }
__device__ __forceinline__ void swap_pairs(float x, float y, float& first, float& second) {
    const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, y), false, false);
    first = __builtin_bit_cast(float, (uint32_t)r[0]);
    second = __builtin_bit_cast(float, (uint32_t)r[1]);
}
// swz16 for operands whose rows are taken in that order
template <int D> __device__ __forceinline__ int swz_pairs(int row) { return swz16<D>(pair_row(row)); }

// One wavefront-wide load of 16 bytes per lane from global memory into LDS: lane i's bytes
// land at lds_base + OFF + 16 i (lds_base wavefront-uniform).  Counted by vmcnt like any load; the
// compiler does not know that it writes LDS, so whoever reads the bytes waits for vmcnt and
// passes a barrier first (the tile loop does both once per tile).
// No vector ALU instruction belongs in here: the compiler puts no wait states between the matrix instructions and a
// register that inline assembly writes, nor between the restore of a spilled scalar register and its use in there.
// Addresses are formed by the callers, in C++.  OFF is added to lds_base on the way into m0, which takes no scalar register
// per call (sparse units spill theirs: 16384 tokens 266 -> 262 us, 4096 30.8 -> 30.4).
template <int OFF = 0> __device__ __forceinline__ void load_to_lds_16(const void* gptr, uint32_t lds_base) {
    asm volatile("s_add_u32 m0, %1, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
                 :: "v"(gptr), "s"(lds_base), "i"(OFF) : "m0", "scc");
}
template <typename P> __device__ __forceinline__ uint32_t lds_address(P* ptr) {
    return (uint32_t)(size_t)(__attribute__((address_space(3))) void*)ptr;
}

// Workgroup -> (query block, KV head, sequence).  Workgroups go to the eight XCDs round-robin in
// launch order and each XCD has an L2 of its own.  When the number of (sequence, KV head) pairs
// is a multiple of eight, consecutive workgroups take eight different pairs: all units of a pair, which read the same
// K/V rows, run on one XCD.  The launch is (8 pairs, blocks, pairs / 8) then, in that order of dispatch, and
// the pair's sequence is a product with a reciprocal from the host: with a one-dimensional launch every workgroup
// began with two divisions, a hundred dependent instructions in front of its first load.
struct UnitGrid {
    dim3 grid;
    unsigned recip;   // ceil(2^32 / G), G > 1
    int pairs_fill_xcds, all_resident;
};
inline bool unit_grid(int B, int G, long long nblocks, int per_cu, UnitGrid& u) {
    const long long pairs = (long long)B * G;
    // exact quotients below 2^32 / G; grid dimensions behind the first are 16 bits
    u.pairs_fill_xcds = pairs % 8 == 0 && nblocks <= 65535 && pairs / 8 <= 65535 && pairs * G < (1ll << 32);
    u.recip = G > 1 ? (unsigned)(0xffffffffu / (unsigned)G + 1u) : 0u;
    u.all_resident = nblocks * pairs <= (long long)per_cu * 256;
    if (u.pairs_fill_xcds) {
        u.grid = dim3(8, (unsigned)nblocks, (unsigned)(pairs / 8));
        return nblocks * pairs <= 0x7fffffffLL;
    }
    u.grid = dim3((unsigned)nblocks, G, B);
    return nblocks <= 0x7fffffffLL;
}
// Blocks go out long ones first.  Where all workgroups are resident at once (`per_cu` on each of 256
// compute units) nothing evens out their lengths later, and every second round of 32 workgroups of an
// XCD -- one per compute unit -- is taken in reverse, so that a compute unit's workgroups add up to about
// the same work: 32/8 heads, 2048 tokens dense 52 -> 48.5 us, log-sum pass 4096 tokens 97 -> 83.  With more
// workgroups than that the plain order is the better one (dense, 4096 tokens: 142 against 149 us).
__device__ __forceinline__ void unit_of_workgroup(const PrefillParams& p, int G, int nblocks, int& blk, int& g, int& b) {
    if (p.pairs_fill_xcds) {
        const int pair = blockIdx.z * 8 + blockIdx.x;
        blk = blockIdx.y;
        constexpr int kXcdCus = 32;
        if ((blk & kXcdCus) && p.all_resident) {
            const int base = blk & ~(kXcdCus - 1);
            blk = base + min(kXcdCus, nblocks - base) - 1 - (blk - base);
        }
        b = G > 1 ? (int)__umulhi((unsigned)pair, p.pair_recip) : pair;
        g = pair - b * G;
    } else {
        blk = blockIdx.x;
        g = blockIdx.y;
        b = blockIdx.z;
    }
}

// Where sequence b's rows of a chunked call stand: first global position and number of rows.
__device__ __forceinline__ void chunk_of_sequence(const PrefillParams& p, int b, int& q_start, int& rows) {
    q_start = p.q_start;
    rows = p.Lq;
    if (p.q_start_rows) {   // scalar loads: as vector loads they would make every position and address that follows per lane
        typedef const __attribute__((address_space(4))) int* ConstantPtr;
        b = __builtin_amdgcn_readfirstlane(b);
        q_start = max(0, min(((ConstantPtr)p.q_start_rows)[b], p.q_start)) & ~(kTile - 1);
        if (p.q_len_rows) rows = max(0, min(((ConstantPtr)p.q_len_rows)[b], p.Lq));
    }
}

}  // namespace
}  // namespace kascade
