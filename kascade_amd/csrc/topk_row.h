// Selection of a row by one workgroup that holds it in registers (topk.hip, and the prompt pooling kernel of prefill.hip).
#pragma once
#include "common.h"

namespace kascade {
namespace {

// Optional second output: every selected position translated to its row of a paged cache
// (block_table[sequence][pos / page] * page + pos % page), sequence = row / rows_per_seq.  What the
// gather kernels of the reuse layers read, produced here so that no separate launch is needed.
struct RowsOut {
    int* rows;               // [rows, k] or null
    const int* block_table;  // [sequences, max_pages]
    int max_pages;
    int page_shift;
    int rows_per_seq;
};

__device__ __forceinline__ int to_cache_row(const RowsOut& ro, long long row, int pos) {
    const int* bt = ro.block_table + (long long)((uint32_t)row / (uint32_t)ro.rows_per_seq) * ro.max_pages;   // rows fit an int (host)
    pos = max(0, min(pos, (ro.max_pages << ro.page_shift) - 1));
    return (bt[pos >> ro.page_shift] << ro.page_shift) + (pos & ((1 << ro.page_shift) - 1));
}

__device__ __forceinline__ uint32_t order_key(uint16_t bits) {
    // monotone map fp16 -> u16: negatives below positives, -inf lowest finite order
    return (bits & 0x8000u) ? (uint32_t)(uint16_t)~bits : (uint32_t)(bits | 0x8000u);
}

// Inclusive prefix sum over the 64 lanes of a wavefront in six DPP additions: four shifts within
// the rows of 16 lanes, then the last lane of row 0 / 2 added to row 1 / 3 and lane 31 to the
// upper half.
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v) {
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xF, 0xF, false);   // row_shr:1
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xF, 0xF, false);   // row_shr:2
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xF, 0xF, false);   // row_shr:4
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xF, 0xF, false);   // row_shr:8
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xA, 0xF, false);   // row_bcast:15 -> rows 1, 3
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xC, 0xF, false);   // row_bcast:31 -> rows 2, 3
    return v;
}

// Packed 16-bit operations on the two halves of a word.  Not in inline assembly, which a kernel with matrix instructions
// must not do vector arithmetic in; the constants are hidden, because the compiler turns min(sat(a - b), 1) and
// min(a, 1) into two compares, two selects and a byte permute.
typedef unsigned short ushort2_t __attribute__((ext_vector_type(2)));
typedef short short2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pk_hidden(uint32_t x) {
    asm("" : "+s"(x));
    return x;
}
__device__ __forceinline__ uint32_t pk_sub_sat_u16(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_sub_sat(__builtin_bit_cast(ushort2_t, a), __builtin_bit_cast(ushort2_t, b)));
}
__device__ __forceinline__ uint32_t pk_min_u16(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(ushort2_t, a), __builtin_bit_cast(ushort2_t, b)));
}
__device__ __forceinline__ uint32_t pk_max_u16(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(ushort2_t, a), __builtin_bit_cast(ushort2_t, b)));
}
// arithmetic shift right by 15 of both halves: 0xFFFF where a half is negative as int16, else 0
__device__ __forceinline__ uint32_t pk_sign_mask_i16(uint32_t a) {
    const uint32_t by = pk_hidden(0x000F000Fu);
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(short2_t, a) >> __builtin_bit_cast(short2_t, by));
}
__device__ __forceinline__ uint32_t pk_add_u16(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(ushort2_t, a) + __builtin_bit_cast(ushort2_t, b));
}

// ---- selection with the row in registers ----
// A workgroup of THREADS threads holds one row and runs the passes on registers.  Its wavefronts own
// contiguous parts of the row, `nch` chunks of 512 slots each: lane l of a wavefront holds slots
// [512 c + 8 l, +8) of chunk c of its part as packed 16-bit order keys, 0 where there is no entry.
//
// What bounds it is instruction issue on the one compute unit the row runs on -- every entry costs
// about ten instructions, every wavefront about three hundred on top whatever it holds -- so rows get the
// fewest wavefronts that hold them, the work per entry is kept to a few instructions on packed halves,
// nothing has a second copy for partial chunks, and the position order (wavefront, chunk, lane, entry)
// needs one scan over the wavefronts instead of one over all (chunk, wavefront) pairs:
//  * Real entries carry keys >= 1 (the two lowest negative NaN patterns share key 1) and absent
//    slots key 0, so the threshold key T is >= 1 and no count needs a validity test.
//  * The coarse histogram (key >> 5) is kept in four copies selected by the lane number, which
//    spreads the same-address conflicts of the LDS atomics (pooled softmax scores crowd into a few
//    exponent bins).  The bin of +0 and the 31 smallest subnormals, where pooled probabilities
//    underflow to by the thousand, is not counted at all: its count is the row length minus the
//    sum of the others.  NONNEG: no entry is below +0 (pooled probabilities), half the bins.
//  * The fine histogram knows of +0 only where its bin is the threshold's.  min(sat(key - (T-1)), 2) over packed
//    halves, two bits an entry, gives the counts above / equal to T and, kept, the masks of the compaction.
//  * The selected positions are staged in LDS in their final order, so that the list leaves as
//    full-width stores.
// Causal prompt tiles (8 heads x L/32 rows, ragged), against one size of workgroup with a scan over all
// (chunk, wavefront) pairs: L = 4096 18.6 -> 9.4 us, 8192 34.6 -> 20.5, 16384 73.6 -> 48.1, 32768 179 -> 142,
// 65536 907 -> 546 us; 2048 full rows of 65536: 175 -> 130 us = 2.1 TB/s, of 131072 341 us (145 and 369 while 16 chunks
// spilled nine registers where the keys are formed).
// One row on one compute unit (decode anchors, pooling included, 16384 tokens of 4 heads): 13.4 -> 12.3 us with the log-sums'
// parts requested before the length is known, the histograms cleared under the row's loads, counters addressed by the key's
// bits in place, and the codes kept.
// Sum of the entries of s_wave before `wave`, and of all of them (one per wavefront, in LDS).
template <int THREADS>
__device__ __forceinline__ void scan_waves(const uint32_t* s_wave, int wave, uint32_t& before, uint32_t& all) {
    constexpr int kW = THREADS / 64;
    const int lane = threadIdx.x & 63;
    const uint32_t inc = wave_incl_scan(lane < kW ? s_wave[lane] : 0u);
    all = (uint32_t)__builtin_amdgcn_readlane((int)inc, 63);
    before = wave > 0 ? (uint32_t)__builtin_amdgcn_readlane((int)inc, wave - 1) : 0u;
}

// A workgroup's histograms.  Cleared by the caller a barrier before select_row, under the loads of the row.
template <int THREADS, bool NONNEG>
struct SelectLds {
    static constexpr int kCopies = 4;
    static constexpr int kNB = NONNEG ? 1024 : 2048;                 // coarse bins
    uint32_t hist[kNB * kCopies];
    uint32_t hist2[32];
    __device__ __forceinline__ void clear() {
        for (int i = threadIdx.x * 4; i < kNB * kCopies; i += THREADS * 4) *reinterpret_cast<uint4_t*>(&hist[i]) = uint4_t{0, 0, 0, 0};
        if (threadIdx.x < 32) hist2[threadIdx.x] = 0;
    }
};

template <int THREADS, int MAXC, bool NONNEG>
__device__ __forceinline__ void select_row(SelectLds<THREADS, NONNEG>& lds, const uint4_t (&data)[MAXC], int nch, int lead,
                                           int row_len, int n, int k, int fill, int* __restrict__ out, long long row,
                                           const RowsOut& ro) {
    constexpr int kW = THREADS / 64;
    constexpr int kCopies = SelectLds<THREADS, NONNEG>::kCopies;
    constexpr int kNB = SelectLds<THREADS, NONNEG>::kNB;             // coarse bins ...
    constexpr uint32_t kBin0 = NONNEG ? 1024 : 0;                    // ... from this one on
    constexpr int kStage = kNB * kCopies;                            // positions staged in the histogram's LDS
    const uint32_t kOne = pk_hidden(0x00010001u), kTwo = pk_hidden(0x00020002u);
    constexpr uint32_t kZeroKey = 0x8000u;                           // order key of +0
    constexpr uint32_t kSkipBin = kZeroKey >> 5;                     // coarse bin of +0: counted by subtraction
    constexpr int kBPT = kNB / THREADS > 0 ? kNB / THREADS : 1;      // bins per thread in the scan
    static_assert(kNB % THREADS == 0 || kNB < THREADS, "whole bins per thread");
    uint32_t* s_hist = lds.hist;
    uint32_t* s_hist2 = lds.hist2;
    __shared__ uint32_t s_wave[kW], s_gt[kW], s_eq[kW];
    __shared__ uint32_t s_sel[2];  // b1, cum_above

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int* dst = out + row * (long long)k;
    int* rdst = ro.rows ? ro.rows + row * (long long)k : nullptr;

    // ---- pass 1: coarse histogram ----
    // A bin's copies are 16 bytes: the byte offset of a key's counter is its bin in place, shifted by one, and the copy.
    // (NONNEG: the top bit of every bin is set and left out.)
    static_assert(kCopies == 4, "a bin is 16 bytes");
    constexpr uint32_t kBinBytes = NONNEG ? 0x3FF0u : 0x7FF0u;
    const uint32_t copy = (tid & (kCopies - 1)) * 4;
    auto count1 = [&](uint16_t key, uint32_t bytes) {   // absent entries and the bin of +0 are not counted
        if (NONNEG ? key >= kZeroKey + 32 : (key != 0 && key >> 5 != kSkipBin))
            atomicAdd(reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(s_hist) + bytes), 1u);
    };
    static_for<0, MAXC>([&](auto c_c) {
        constexpr int c = decltype(c_c)::value;
        if (c < nch) {   // uniform
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t w = data[c][j];
                count1((uint16_t)w, ((w >> 1) & kBinBytes) | copy);
                count1((uint16_t)(w >> 16), ((w >> 17) & kBinBytes) | copy);
            }
        }
    });
    __syncthreads();
    {
        // thread t owns kBPT bins, in descending order
        uint32_t cnt[kBPT], mine = 0;
        const int first = kNB - 1 - kBPT * tid;
#pragma unroll
        for (int u = 0; u < kBPT; ++u) {
            cnt[u] = 0;
            if (kNB >= THREADS || tid < kNB) {
                const uint4_t h = *reinterpret_cast<const uint4_t*>(&s_hist[(first - u) * kCopies]);
                cnt[u] = h[0] + h[1] + h[2] + h[3];
            }
            mine += cnt[u];
        }
        const uint32_t inc = wave_incl_scan(mine);
        if (lane == 63) s_wave[wave] = inc;
        __syncthreads();
        uint32_t before, total;
        scan_waves<THREADS>(s_wave, wave, before, total);
        uint32_t above = before + inc - mine;
        const uint32_t skipped = (uint32_t)row_len - total;
        constexpr int kSkipAt = kNB - 1 - (int)(kSkipBin - kBin0);   // place of the uncounted bin in descending order
        if (tid > kSkipAt / kBPT) above += skipped;
#pragma unroll
        for (int u = 0; u < kBPT; ++u) {
            const uint32_t c = cnt[u] + (kBPT * tid + u == kSkipAt ? skipped : 0u);
            if (above < (uint32_t)n && (uint32_t)n <= above + c) {
                s_sel[0] = (uint32_t)(first - u) + kBin0;
                s_sel[1] = above;
            }
            above += c;
        }
    }
    __syncthreads();
    const uint32_t b1 = s_sel[0];
    const uint32_t cum_above = s_sel[1];

    // ---- pass 2: fine histogram inside the threshold bin.  +0 is left out of the atomics (that many on one
    // address would serialise) and counted per wavefront where its bin is the threshold's ----
    {
        const uint32_t bb = (b1 << 5) | (b1 << 21);
        auto fine = [&](auto with_zero) {
            constexpr bool ZERO = decltype(with_zero)::value;
            uint32_t nonzero = 0;   // per half: slots of this thread that do not hold +0 (<= 4 MAXC)
            static_for<0, MAXC>([&](auto c_c) {
                constexpr int c = decltype(c_c)::value;
                if (c < nch) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const uint32_t w = data[c][j];
                        const uint32_t x = (w ^ bb) & 0xFFE0FFE0u;   // a half is 0 iff its key lies in the bin
                        if (ZERO) nonzero = pk_add_u16(nonzero, pk_min_u16(w ^ 0x80008000u, kOne));
                        if ((uint16_t)x == 0 && (!ZERO || (uint16_t)w != kZeroKey)) atomicAdd(&s_hist2[w & 31u], 1u);
                        if (x < 0x10000u && (!ZERO || w >> 16 != kZeroKey)) atomicAdd(&s_hist2[(w >> 16) & 31u], 1u);
                    }
                }
            });
            if (ZERO) {
                uint32_t z = 8u * (uint32_t)nch - (nonzero & 0xFFFFu) - (nonzero >> 16);
#pragma unroll
                for (int o = 32; o >= 1; o >>= 1) z += __shfl_xor(z, o);
                if (lane == 0 && z) atomicAdd(&s_hist2[kZeroKey & 31u], z);
            }
        };
        if (b1 == kSkipBin) fine(std::true_type{}); else fine(std::false_type{});   // uniform
    }
    __syncthreads();
    uint32_t T, r;   // threshold key and the number of entries equal to it to take: every wavefront for itself
    {
        // suffix sums of the 32 fine bins, top bin first; the threshold is the first bin whose
        // running count reaches n
        const uint32_t c = (lane < 32) ? s_hist2[31 - lane] : 0u;
        const uint32_t v = wave_incl_scan(c);
        const uint32_t above = cum_above + v - c;             // entries in finer bins above this one
        const bool hit = lane < 32 && above < (uint32_t)n && (uint32_t)n <= above + c;
        // bin 0 takes what is left when no finer bin reaches n (cannot happen for a consistent histogram)
        const unsigned long long m = __ballot(hit);
        const int first = m ? __ffsll((long long)m) - 1 : 31;
        T = max((b1 << 5) | (uint32_t)(31 - first), 1u);
        r = (uint32_t)n - (uint32_t)__builtin_amdgcn_readlane((int)above, first);
    }
    const uint32_t tm1 = (T - 1u) | ((T - 1u) << 16);   // T >= 1

    // ---- pass 3: ordered compaction ----
    // code of a half: min(sat(key - (T-1)), 2) = 0 below T, 1 equal to T, 2 above T.  Kept for both uses, two bits an
    // entry: word j of a chunk at bits 2 j and 16 + 2 j, an odd chunk 8 bits above the even one before it.
    constexpr uint32_t kAbove = 0xAAAAAAAAu, kEqual = 0x55555555u;
    uint32_t codes[(MAXC + 1) / 2];
    {
        uint32_t gt = 0, eq = 0;
#pragma unroll
        for (int i = 0; i < (MAXC + 1) / 2; ++i) codes[i] = 0;
        static_for<0, MAXC>([&](auto c_c) {
            constexpr int c = decltype(c_c)::value;
            if (c < nch) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    codes[c / 2] |= pk_min_u16(pk_sub_sat_u16(data[c][j], tm1), kTwo) << (8 * (c & 1) + 2 * j);
            }
        });
#pragma unroll
        for (int i = 0; i < (MAXC + 1) / 2; ++i) {
            gt += (uint32_t)__popc(codes[i] & kAbove);
            eq += (uint32_t)__popc(codes[i] & kEqual);
        }
        // above T in the low half, equal to T in the high half (a wavefront holds at most 8192 entries)
        const uint32_t all = wave_incl_scan(gt | (eq << 16));
        if (lane == 63) {
            s_gt[wave] = all & 0xFFFFu;
            s_eq[wave] = all >> 16;
        }
    }
    __syncthreads();
    uint32_t gt_before, eq_before, unused;
    scan_waves<THREADS>(s_gt, wave, gt_before, unused);
    scan_waves<THREADS>(s_eq, wave, eq_before, unused);
    // The selected positions are staged in LDS, kStage per round (one round unless n > kStage).
    int* stage = reinterpret_cast<int*>(s_hist);
    const int base0 = wave * nch * 512 + lane * 8 - lead;      // position of this thread's first entry
#pragma clang loop unroll(disable)
    for (uint32_t lo = 0; lo < (uint32_t)n; lo += kStage) {
        uint32_t carry = 0;   // entries of the wavefront's part before the chunk: above T / equal to T, packed
        static_for<0, MAXC>([&](auto c_c) {
            constexpr int c = decltype(c_c)::value;
            if (c < nch) {
                // bit e: entry e of the chunk is above / equal to T (entries 2 j in the low half, 2 j + 1 in the high one)
                const uint32_t cc = codes[c / 2] >> (8 * (c & 1));
                const uint32_t gt2 = (cc & kAbove) >> 1, eq2 = cc & kEqual;
                const uint32_t above = (gt2 | (gt2 >> 15)) & 0xFFu;
                uint32_t equal = (eq2 | (eq2 >> 15)) & 0xFFu;
                const uint32_t cnt = (uint32_t)__popc(above) | ((uint32_t)__popc(equal) << 16);
                const uint32_t v = wave_incl_scan(cnt);
                if (cnt) {
                    const uint32_t ex = carry + v - cnt;
                    const uint32_t my_eq = eq_before + (ex >> 16);
                    // where the next selected entry goes: after the earlier ones above T and the
                    // earlier ties taken
                    uint32_t pos = gt_before + (ex & 0xFFFFu) + min(my_eq, r) - lo;
                    const uint32_t room = r - min(my_eq, r);             // ties that still fit, the lower positions first
                    equal = room == 0 ? 0u : equal;
#pragma clang loop unroll(disable)
                    while ((uint32_t)__popc(equal) > room) equal &= ~(0x80000000u >> __clz(equal));
#pragma clang loop unroll(disable)
                    for (uint32_t m = above | equal; m != 0; m &= m - 1, ++pos)
                        if (pos < (uint32_t)kStage) stage[pos] = base0 + c * 512 + __ffs(m) - 1;
                }
                carry += (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
            }
        });
        __syncthreads();
        // this round's slots; the last round also fills the slots from n to k
        const int hi = (lo + kStage >= (uint32_t)n) ? k : (int)(lo + kStage);
        // k is a multiple of 4 for every budget the library produces; otherwise element stores
        const bool wide = (k & 3) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0 &&
                          (reinterpret_cast<uintptr_t>(ro.rows) & 15) == 0;
        if (wide) {
#pragma clang loop unroll(disable)
            for (int i = (int)lo + tid * 4; i < hi; i += THREADS * 4) {
                int4_t v, w;
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = (i + e < n) ? stage[i + e - lo] : fill;
                *reinterpret_cast<int4_t*>(dst + i) = v;
                if (rdst) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) w[e] = to_cache_row(ro, row, v[e]);
                    *reinterpret_cast<int4_t*>(rdst + i) = w;
                }
            }
        } else {
#pragma clang loop unroll(disable)
            for (int i = (int)lo + tid; i < hi; i += THREADS) {
                const int v = (i < n) ? stage[i - lo] : fill;
                dst[i] = v;
                if (rdst) rdst[i] = to_cache_row(ro, row, v);
            }
        }
        __syncthreads();   // the stage is free for the next round
    }
}

// A row with nothing to select from: its first n positions, then the fill value.
template <int THREADS>
__device__ __forceinline__ void list_head(int n, int k, int fill, int* __restrict__ out, long long row, const RowsOut& ro) {
    int* dst = out + row * (long long)k;
    int* rdst = ro.rows ? ro.rows + row * (long long)k : nullptr;
#pragma clang loop unroll(disable)
    for (int i = threadIdx.x; i < k; i += THREADS) {
        const int pos = (i < n) ? i : fill;
        dst[i] = pos;
        if (rdst) rdst[i] = to_cache_row(ro, row, pos);
    }
}

}  // namespace
}  // namespace kascade
