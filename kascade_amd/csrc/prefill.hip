// Prefill attention kernels for gfx950 (fp16/bf16 MFMA 32x32x16 and 16x16x32, fp32 softmax).
//
// prefill_attn_kernel -- flash attention over one (query block, KV head, batch)
//   per workgroup; 4 wavefronts, wavefront w owns q-head 4g+w and 32*NQB queries,
//   so the four heads of a KV head share every K/V tile staged in LDS.
//   Three key regimes (REUSE): dense causal, gathered top-k rows through the
//   tile's index list, and the within-tile causal diagonal.
//
//   K/V tiles go from global memory straight into LDS (global_load_lds_dwordx4: no staging
//   registers, no LDS store instructions) into one of two buffers, so a tile costs one
//   barrier: wait for the own loads, barrier, start the next tile's loads into the other
//   buffer, compute.  Rows lie in LDS as they lie in memory; the 16-byte chunk c of row R
//   sits at chunk c ^ swz(R) (swz16 and swz_pairs for 16x16x32 products), chosen by the lane that fetches it (each lane picks the global
//   chunk that belongs at its LDS position), which makes both read patterns below free of
//   bank conflicts without padding.
//
//   The kernel works on S^T = K Q^T so that two lanes (four of 16x16x32 products) own one query column:
//   row max / row sum are in-lane reductions plus one or two exchanges, and
//   the exponentiated scores are already in the B-operand layout of the second
//   product O^T = V^T P^T -- P never leaves registers.  The A operand of that product,
//   V^T, comes out of the row-major V tile through the transposing LDS read
//   ds_read_b64_tr_b16 (two per operand: four keys each).
//
//   What bounds long calls is the chip's power, and per product 16x16x32 takes less of it than 32x32x16 (1.84
//   against 1.59 PFLOP/s on random operands in registers): sparse units use it (32/8 heads: 3001 tokens 23.8 -> 23.1 us,
//   4096 31.6 -> 30.4, 16384 277 -> 262, 32768 982 -> 933; no gain at 2048 tokens, 12.8 both and in bf16 12.6 -> 12.8, nor
//   below), and dense passes with an output at head_dim 128; the others keep 32x32x16 (see there).  Against row addresses formed by a
//   64-bit product per tensor and row and block-table entries requested behind the tile's loads: dense 517 tokens
//   14.6 -> 13.5 us, 2048 49.4 -> 46.9, chunks at position 14336 of 512 queries 326 -> 247 us, of 2048 532 -> 520;
//   log-sums alone 517 10.2 -> 9.6 us, 32768 4.39 -> 4.24 ms, chunks of 512 205 -> 173 us, of 2048 310 -> 301.
//
// prefill_aggregate_kernel -- pooled tile scores: S = Q_tile K^T with the 128
//   (query, head) rows of a tile held as A operands in registers by every
//   wavefront; each wavefront takes 32 keys of a 128-key tile, so pooling over
//   rows is an in-lane sum over accumulator registers.
#include "prefill.h"
#include "prefill_tile.h"
#include "topk_row.h"

#include <algorithm>
#include <type_traits>

// Wave priority around the phases of a tile.  Two wavefronts share a SIMD; which of them the
// scheduler serves first when both have an instruction ready decides how well one's softmax hides
// under the other's matrix instructions.  Modes: 0 none; 1 the wavefront in its softmax goes first;
// 2 the one in its products; 4 the one in its second product only; 5 the one in its first product
// only.  Measured at 32K tokens against mode 0 (same box, two rounds): kernels with a second
// product mode 2 -1.1 % (reuse) / -1.4 % (dense), mode 1 +1.2 %, mode 4 +1 %, mode 5 -0.5 %; the
// K-only log-sum pass mode 1 -2.6 %, mode 2 -0.8 %, mode 5 -0.5 %; the pooling kernel mode 2 -1.9 %,
// mode 1 -1.7 %.
#ifndef KASCADE_PRIO_V
#define KASCADE_PRIO_V 2
#endif
#ifndef KASCADE_PRIO_K
#define KASCADE_PRIO_K 1
#endif
#ifndef KASCADE_PRIO_AGG
#define KASCADE_PRIO_AGG 2
#endif

namespace kascade {

namespace {

constexpr int kThreads = 256;

// phase: 0 = first product begins, 1 = softmax begins, 2 = second product begins (or the tile ends)
template <int MODE> __device__ __forceinline__ void tile_phase(int phase) {
    if (MODE == 1) { if (phase == 1) __builtin_amdgcn_s_setprio(1); else if (phase == 2) __builtin_amdgcn_s_setprio(0); }
    if (MODE == 2) { if (phase == 1) __builtin_amdgcn_s_setprio(0); else if (phase == 2) __builtin_amdgcn_s_setprio(1); }
    if (MODE == 4) { if (phase == 0) __builtin_amdgcn_s_setprio(0); else if (phase == 2) __builtin_amdgcn_s_setprio(1); }
    if (MODE == 5) { if (phase == 0) __builtin_amdgcn_s_setprio(1); else if (phase == 1) __builtin_amdgcn_s_setprio(0); }
}

// Registers that loads are filling are waited for here.  The compiler does not see the waits of the tile loops and would put
// one in front of each use in there, behind the next tile's loads.
template <int N, typename X> __device__ __forceinline__ void arrived(X (&x)[N]) {
#pragma unroll
    for (int i = 0; i < N; ++i) asm volatile("" : "+v"(x[i]));
}

// A wavefront's ROWS output rows, chunk c of row r at c ^ r in LDS, leave as whole rows.  All of them are read before the first
// is stored and a row's address is the first one's and a scalar: one after another, each read, its address by a 64-bit
// product and its store took a unit 1.3 us.  out: row 0; row_elems: elements from a row to the next; rows up to last_row.
template <int D, int ROWS, typename T>
__device__ __forceinline__ void store_rows(T* out, unsigned row_elems, const T* so, int lrow, int lchunk, int last_row) {
    constexpr int kChunks = AttnTile<D>::kChunks, kRPL = AttnTile<D>::kRowsPerLoad, kStores = ROWS / kRPL;
    uint4_t row[kStores];
#pragma unroll
    for (int j = 0; j < kStores; ++j) {
        const int r = j * kRPL + lrow;
        row[j] = *reinterpret_cast<const uint4_t*>(&so[r * D + (lchunk ^ (r & (kChunks - 1))) * 8]);
    }
    T* mine = out + ((unsigned)lrow * (unsigned long long)row_elems + lchunk * 8);
    // the output is not read again by these kernels: keep it out of the caches
    auto store = [&](int j) {
        __builtin_nontemporal_store(row[j], reinterpret_cast<uint4_t*>(mine + (unsigned long long)row_elems * (j * kRPL)));
    };
    if (last_row >= ROWS - 1) {   // uniform
#pragma unroll
        for (int j = 0; j < kStores; ++j) store(j);
    } else {
#pragma unroll
        for (int j = 0; j < kStores; ++j)
            if (j * kRPL + lrow <= last_row) store(j);
    }
}

// Queries are rows [0, Lq) of Q at global positions q_start + row (q_start a multiple of 32);
// keys are positions [0, L) with L = q_start + Lq.  PAGED: K/V are pages [P, page, G, D]
// addressed through the block table, and gathered index rows hold physical row numbers.
//
// Sparse passes (and the dense tiles of their first units): products 16x16x32.
// SPARE: the KV head's last sub-group may have fewer than four query heads (gs no multiple of four).  Its wavefronts
// without a head only stage their rows of every tile, which leaves the matrix unit and the power to the others: 28/4
// heads bf16, two prompts of 3001 tokens, eight layers with pooling over the heads there are 780 -> 737 us.  A variant of its own, because
// the second loop costs the allocation of the first (32/8 heads, 517 tokens 119.2 -> 120.4 us; with log-sums, 32768
// tokens, 945 against 958 us).  Rotating the slots over
// the wavefronts, so that the idle one is not always the same SIMD's, gave nothing.
// EXACT_SUM: the softmax denominators are summed in fp32 from the unrounded exponentials (the
// passes whose log-sum is an output); otherwise units sum them as they enter the second product.
// NQ: blocks of 16 queries a wavefront takes.  With two, wavefront w has head slot w; with one, four wavefronts are two head
// slots x two blocks and a unit's four slots take two workgroups.
template <bool PAGED, int D, typename T, bool SPARE, bool EXACT_SUM, int NQ>
__device__ __forceinline__ void prefill_reuse_body(const PrefillParams& p, T* sK, T* sV, int* s_move = nullptr) {
    typedef typename Elem<T>::x8 x8_t;
    typedef typename Elem<T>::x4 x4_t;
    typedef typename Elem<T>::x2 x2_t;
    typedef AttnTile<D> G_;
    constexpr int kKT = G_::kKT, kChunks = G_::kChunks, kRPL = G_::kRowsPerLoad, kTileElems = G_::kTileElems;
    // products 16x16x32: contraction steps of S^T, 16-row blocks of O^T, 16-key blocks of a tile
    constexpr int kKS = D / 32, kDB = D / 16, kKB = kKT / 16;
    constexpr float kScaleLog2 = ScaleLog2<D>::value;
    constexpr int kSlots = 2 * NQ;       // head slots of a workgroup
    const HeadSlots hs = head_slots(p.gs, kSlots);
    const int kvh = p.G, nheads = p.G * hs.gs;
    const T* Qp = (const T*)p.Q;
    const T* Kp = (const T*)p.K;
    const T* Vp = (const T*)p.V;

    // What the first loads need comes in one trip to memory (the compiler would take one for each branch on the way)
    asm volatile("" :: "s"(p.Q), "s"(p.K), "s"(p.V), "s"(p.head_map), "s"(p.q_start_rows), "s"(p.q_len_rows), "s"(p.q_sb), "s"(p.q_sl),
                 "s"(p.q_sh), "s"(p.k_sb), "s"(p.k_sl), "s"(p.k_sh), "s"(p.Lq), "s"(p.q_start), "s"(p.max_topk), "s"(p.topk_percent),
                 "s"(p.gs), "s"(p.pair_recip), "s"(p.pairs_fill_xcds), "s"(p.all_resident));
    constexpr int QT = 32;
    const int Lq = p.Lq;            // rows of Q and of the outputs per sequence
    const int nqt = (Lq + QT - 1) / QT;
    int blk, g, b;
    unit_of_workgroup(p, p.G * hs.subs, nqt, blk, g, b);   // g: KV head and sub-group
    int q_start, Lqv;               // this sequence's first position and how many of the rows are its own
    chunk_of_sequence(p, b, q_start, Lqv);
    const int L = q_start + Lqv;    // keys of this sequence
    int sub;
    split_sub_group(p, hs.subs, g, sub);   // g: the KV head
    // Whose lists a sparse unit reads: a scalar load, on its way while the first rows' addresses are formed (as a vector
    // load every sparse unit waited for it before it requested anything: 3001 tokens 24.3 -> 23.9 us, head_dim 64
    // at 4096 12.4 -> 12.2)
    typedef const __attribute__((address_space(4))) int* ConstantPtr;
    const int mapped = *(ConstantPtr)(p.head_map + __builtin_amdgcn_readfirstlane(g));
    const int tq = nqt - 1 - blk;   // long (late) query blocks first
    const int tid = threadIdx.x;
    const int wave = tid >> 6;
    const int lane = tid & 63;
    const int col = lane & 15;          // of an operand or result of 16 rows or columns
    const int dq = lane >> 4;
    const int q0l = tq * QT;            // first query row of this block
    if (q0l >= Lqv) return;             // a block past this sequence's rows (uniform over the workgroup)
    const int q0 = q_start + q0l;       // its global position
    const int wave_u = __builtin_amdgcn_readfirstlane(wave);
    const int slot = kSlots * sub + (NQ == 2 ? wave_u : wave_u >> 1);
    const int q_off = NQ == 2 ? 0 : 16 * (wave_u & 1);   // this wavefront's first query of the block's
    const int head = g * hs.gs + min(slot, hs.gs - 1);
    const bool has_head = !SPARE || slot < hs.gs;

    // ---- key regime of this block ----
    const int* idx_row = nullptr;
    // a sequence of a mixed batch keeps the budget it has on its own (the rows are as wide as
    // the longest sequence needs)
    const int width = p.q_start_rows ? min(p.max_topk, topk_width_of(p.topk_percent, L)) : p.max_topk;
    // (a block behind the widest list is sparse whatever its budget, which is worked out under its first loads)
    const bool rolls = p.rolling && L > 128;
    int n = width;
    if (rolls && q0 <= width) n = min(rolling_budget(p.topk_percent, q0), width);
    const bool sparse = q0 > n;
    const bool idx_vec = (p.max_topk & 3) == 0 && (reinterpret_cast<uintptr_t>(p.idx) & 15) == 0;

    // ---- tile staging: wavefront w fills rows [4w R, 4(w+1) R) of a tile with four loads of R rows
    // each (R = 4 at D = 128, 8 at D = 64); lane = (row within the load, chunk position) ----
    const int lrow = lane / kChunks;
    const int lchunk = lane % kChunks;
    // This lane's four rows sit at LDS rows slot0 + j R (j = load) and hold the four consecutive
    // tile positions pos0 + j: one 16-byte load brings their four indices, one block-table entry
    // covers their page, and the rows of a tile in LDS are a permutation of its keys -- which only
    // the masks need to know (both products contract over the same order).
    const int slot0 = wave * 4 * kRPL + lrow;
    const int pos0 = 4 * (wave * kRPL + lrow);
    // tile position of LDS row `slot`
    auto pos_of_slot = [](int slot) { return 4 * ((slot / (4 * kRPL)) * kRPL + slot % kRPL) + (slot / kRPL) % 4; };
    const T* kbase = PAGED ? Kp + (long long)g * D : Kp + (long long)b * p.k_sb + (long long)g * p.k_sh;
    const unsigned long long v_from_k = (unsigned long long)Vp - (unsigned long long)Kp;   // V shares K's layout
    const int* bt_row = PAGED ? p.block_table + (long long)b * p.max_pages : nullptr;
    const int page_mask = (1 << p.page_shift) - 1;
    const int max_row = PAGED ? (p.num_pages << p.page_shift) - 1 : 0;
    const uint32_t lds_k = lds_address(sK) + wave_u * 4096;   // this wavefront's 4 KB of a K buffer
    const uint32_t lds_v = lds_address(sV) + wave_u * 4096;

    // tiles: gathered ones [0, ng) and the diagonal one behind them in a sparse unit, else consecutive ones
    int ng = 0, ntiles = 1;
    // first key of a tile of consecutive keys (the only ones of a sparse unit are the diagonal tile's)
    auto tile_start = [&](int ti) { return sparse ? q0 : ti * kKT; };
    // ids[j]: what the loads of row j of the next tile need, fetched a tile ahead so that the
    // loads never wait on it.  Gathered tiles: the key id (physical row when PAGED).
    // Consecutive keys, PAGED: the block-table entry of the key's page.  Consecutive keys,
    // strided: nothing (addresses follow from the tile index).
    int ids[4];
    int pend_ti = 0;        // tile the ids belong to
    const unsigned row_bytes = 2 * (PAGED ? (unsigned)(kvh * D) : (unsigned)p.k_sl);   // host checks stride < 2^31
    auto fetch_ids = [&](int ti) {
        pend_ti = ti;
        if (sparse && ti < ng) {   // values are bounded at use
            if (idx_vec) {   // list length and n are multiples of four: a group lies inside the list or outside
                const int4_t v = *reinterpret_cast<const int4_t*>(idx_row + min(ti * kKT + pos0, n - 4));
#pragma unroll
                for (int j = 0; j < 4; ++j) ids[j] = v[j];
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) ids[j] = idx_row[min(ti * kKT + pos0 + j, n - 1)];
            }
        } else if (PAGED) {   // four consecutive keys from a multiple of four on: one page
            ids[0] = bt_row[min(tile_start(ti) + pos0, L - 1) >> p.page_shift];
        }
    };
    // K row addresses of the tile whose ids are held; V's are a scalar offset away.  The
    // loads themselves are issued one at a time between the matrix instructions of the first
    // product: a wavefront that issued all eight at once would sit in front of the memory
    // pipeline, which takes 16 cycles per 1 KB load, with nothing running behind it.
    // lane_ptr: the chunk this lane fetches for row j, of cache row 0.
    const char* lane_ptr[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        lane_ptr[j] = (const char*)(kbase + (lchunk ^ swz16<D>(slot0 + j * kRPL)) * 8);
    }
    const char* row_ptr[4];
    auto consecutive_rows = [&](int key0) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int key = min(key0 + pos0 + j, L - 1);
            const int row = PAGED ? (ids[0] << p.page_shift) + (key & page_mask) : key;
            row_ptr[j] = lane_ptr[j] + (unsigned long long)row_bytes * (unsigned)row;
        }
    };
    auto next_rows = [&]() {
        if (sparse && pend_ti < ng) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {   // a corrupt index must not leave the tensor
                const int row = max(0, min(ids[j], PAGED ? max_row : L - 1));
                row_ptr[j] = lane_ptr[j] + (unsigned long long)row_bytes * (unsigned)row;
            }
        } else {
            consecutive_rows(tile_start(pend_ti));
        }
    };
    constexpr int kNumLoads = 8;
    auto issue_load = [&](auto i_c, int buf) {   // i < 4: K row group i; else V row group i - 4
        constexpr int i = decltype(i_c)::value;
        if constexpr (i < 4) load_to_lds_16<i * 1024>(row_ptr[i], lds_k + buf * (kTileElems * 2));
        else load_to_lds_16<(i - 4) * 1024>(row_ptr[i - 4] + v_from_k, lds_v + buf * (kTileElems * 2));
    };
    // LDS read positions (elements, within a tile buffer).  A operand of S^T: row 16 kb + col,
    // chunk 4 ks + dq.  A operand of O^T (two transposing reads h = 0, 1 of four keys each):
    // the 16 lanes of a quarter address rows 32 s + 16 h + 4 dq + (0..3), 16 columns
    // of V from column 16 db on, and receive one column of the four rows each.
    const int kx = dq ^ swz16<D>(col);
    const int krd = col * D;
    const int vrow = 4 * dq + (col >> 2);                // + 32 s + 16 h, which do not enter swz16
    const int vchunk = ((col >> 1) & 1) ^ swz16<D>(vrow);   // ^ 2 db
    const int vrd = vrow * D + 4 * (col & 1);

    // Softmax state.  m[] is the reference the exponentials are taken against, in log2 units of
    // the scaled scores.  It follows the running maximum lazily: a tile moves it only when one of
    // its scores lies more than kRefSlack above it, so an exponential never exceeds 2^kRefSlack
    // (representable in fp16 and bf16, sums and products are kept in fp32) and the rescaling of the
    // accumulators -- 64 products per lane -- runs on the first tiles of a unit and then almost
    // never.  The quotient is the same: numerator and denominator carry the same factor.
    constexpr int kPrio = KASCADE_PRIO_V;
    constexpr float kRefSlack = 8.f;
    // Reuse units sum the exponentials as they enter the second product (rounded to the element
    // type, two per instruction); the passes whose log-sum feeds the selection sum them in fp32.
    constexpr bool kPairSum = !EXACT_SUM;
    float m[NQ];
    float l[NQ];
    float4_t oT[NQ][kDB];      // query block, 16 output columns
    const float4_t zero4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        m[q] = -INFINITY;
        l[q] = 0.f;
#pragma unroll
        for (int db = 0; db < kDB; ++db) oT[q][db] = zero4;
    }

    // Order of the tiles.  A sparse unit takes its diagonal tile first: the keys q0 .. q0+31 need
    // no index list, so their loads leave at once and the first products run while the list of
    // the first gathered tile and then its rows are still on their way -- one dependent trip to
    // memory less before the first product of every unit, and units are short (28 tiles on
    // average under rolling budgets).  Softmax is accumulated online, so the order is free.
    auto tile_at = [&](int s) { return sparse ? (s == 0 ? ng : s - 1) : s; };
    if (PAGED) ids[0] = bt_row[min(tile_start(0) + pos0, L - 1) >> p.page_shift];
    consecutive_rows(tile_start(0));
    static_for<0, kNumLoads>([&](auto i) { issue_load(i, 0); });

    // ---- Q fragments (B operand of S^T): query col (+ 16 q), d chunk 32*ks + 8*dq; requested after
    // the first tile's rows, which the first barrier waits for ----
    x8_t qf[NQ][kKS];
    const int last_q = min(QT, Lqv - q0l) - 1;   // of this block
    const T* q_base = Qp + (long long)b * p.q_sb + (long long)q0l * p.q_sl + (long long)head * p.q_sh;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const T* qp = q_base + (unsigned long long)(unsigned)min(q_off + 16 * q + col, last_q) * (unsigned long long)p.q_sl + dq * 8;
#pragma unroll
        for (int ks = 0; ks < kKS; ++ks) {
            PackT<T> t;
            t.u = ld_global_16(qp + ks * 32);
            qf[q][ks] = t.v8;
        }
    }

    if (sparse) {
        if (rolls && q0 > width) n = min(rolling_budget(p.topk_percent, q0), width);
        ng = (n + kKT - 1) / kKT;
        ntiles = ng + 1;
        const int src = max(0, min(mapped, kvh - 1));   // a map built for another head count must not leave the tensor
        idx_row = p.idx + (((long long)b * kvh + src) * p.T + tq) * p.max_topk;
    } else {
        ntiles = (min(q0 + QT, L) + kKT - 1) / kKT;
    }
    if (ntiles > 1) fetch_ids(tile_at(1));
    if (last_q < QT - 1) {   // uniform: rows past the sequence's end are zeros
#pragma unroll
        for (int q = 0; q < NQ; ++q)
#pragma unroll
            for (int ks = 0; ks < kKS; ++ks)
                if (q_off + 16 * q + col > last_q) qf[q][ks] = x8_t{};
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) arrived<kKS>(qf[q]);

    // Of two wavefronts with a head slot's two blocks of 16 queries: whether either says so.  Every wavefront comes here once a
    // tile behind the first; the tile's own barrier keeps this read from the next tile's write.  Rows on their way into LDS are
    // not waited for.
    auto lds_barrier = [&]() {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    auto either_half = [&](bool mine) -> bool {
        if (lane == 0) s_move[wave_u] = mine;
        lds_barrier();
        return mine || __builtin_amdgcn_readfirstlane(s_move[wave_u ^ 1]) != 0;
    };

    // One tile: registers -> LDS, next tile's loads, both products, softmax.  Three copies of
    // the code, each straight-line: tiles that need no mask (all but one or two of a unit), tiles
    // that do (the causal edge, the end of the sequence, a selection that ends inside a tile), and
    // the diagonal tile of a sparse unit (32 keys: half the products).
    constexpr int kFull = 0, kMasked = 1, kDiag = 2;
    auto run_tile = [&](int sq, auto mode_c) {
        constexpr int MODE = decltype(mode_c)::value;
        constexpr int nkb = (MODE == kDiag) ? 2 : kKB;
        const int ti = tile_at(sq);
        const T* bK = sK + (sq & 1) * kTileElems;
        const T* bV = sV + (sq & 1) * kTileElems;
        // own loads of this tile landed; after the barrier everybody's have, and everybody is done
        // reading the other buffer (the tile before), which the next tile's loads may now fill
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        // The next tile's loads go out between the products below, unconditionally: after the last
        // tile they fetch its rows once more into the idle buffer (1/28 of the traffic on average,
        // from the cache) rather than put a branch between the matrix instructions.
        // The ids of the tile behind that one are requested before those loads: the compiler waits for every
        // load on its way when it writes registers that one of its own loads may still fill, and behind the
        // tile's loads that wait was a whole trip to memory.
        if (sq + 1 < ntiles) next_rows();
        if (sq + 2 < ntiles) fetch_ids(tile_at(sq + 2));
        const int nbuf = (sq + 1) & 1;

        tile_phase<kPrio>(0);
        // ---- S^T = K_tile Q^T.  Step c = 16 keys and 32 elements of the contraction, two key blocks in turn;
        // operands are read from LDS two windows (four steps) ahead of the products that use them, in
        // program order, because LDS reads do not move across the load statements ----
        constexpr int kSteps = nkb * kKS;
        float4_t sT[NQ][nkb];
        auto key_block = [](int c) { return 2 * (c / (2 * kKS)) + (c & 1); };
        auto k_step = [](int c) { return (c % (2 * kKS)) >> 1; };
        auto read_a = [&](int c) {
            return *reinterpret_cast<const x8_t*>(&bK[16 * key_block(c) * D + krd + ((4 * k_step(c)) ^ kx) * 8]);
        };
        constexpr int kAhead = (D == 128) ? 2 : 1;   // windows read ahead (registers are scarcer at D = 64)
        x8_t aw[kAhead + 1][2];
#pragma unroll
        for (int c = 0; c < 2 * kAhead && c < kSteps; ++c) aw[c >> 1][c & 1] = read_a(c);
        static_for<0, kSteps / 2>([&](auto w_c) {
            constexpr int w = decltype(w_c)::value;
            if (2 * (w + kAhead) < kSteps) {
                aw[(w + kAhead) % (kAhead + 1)][0] = read_a(2 * (w + kAhead));
                aw[(w + kAhead) % (kAhead + 1)][1] = read_a(2 * (w + kAhead) + 1);
            }
            __builtin_amdgcn_sched_barrier(0);   // the scheduler would sink the reads to their use
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int kb = key_block(2 * w + i), ks = k_step(2 * w + i);
#pragma unroll
                for (int q = 0; q < NQ; ++q)   // the first product starts from a constant zero
                    sT[q][kb] = Elem<T>::mma_16x16x32(aw[w % (kAhead + 1)][i], qf[q][ks], ks == 0 ? zero4 : sT[q][kb]);
            }
            if constexpr (w < kNumLoads) issue_load(w_c, nbuf);
        });
        static_for<kSteps / 2, kNumLoads>([&](auto i) { issue_load(i, nbuf); });
        // ---- masks: accumulator v of key block kb is LDS row 16 kb + 4 dq + v of the tile ----
        if (MODE != kFull) {
            const bool diag_here = MODE == kDiag || (sparse && ti == ng);
            // not known to be the same in every tile: the compiler would form the masks of all rows in front of the loop and
            // keep them in scalar registers, which the loop of the tiles without masks then spills
            // (28/4 heads, two prompts of 3001 tokens 42.8 -> 41.2 us)
            int list_end = n, last_key = L - 1, first_q = q0 + q_off;
            asm volatile("" : "+s"(list_end), "+s"(last_key), "+s"(first_q));
            if (sparse && !diag_here) {   // a selection that ends inside this tile
#pragma unroll
                for (int kb = 0; kb < nkb; ++kb)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const int pos = ti * kKT + pos_of_slot(16 * kb + 4 * dq + v);
#pragma unroll
                        for (int q = 0; q < NQ; ++q)
                            if (pos >= list_end) sT[q][kb][v] = -INFINITY;
                    }
            } else {                           // the causal edge and the end of the sequence
                const int kstart = diag_here ? q0 : ti * kKT;
#pragma unroll
                for (int kb = 0; kb < nkb; ++kb)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const int key = kstart + pos_of_slot(16 * kb + 4 * dq + v);
#pragma unroll
                        for (int q = 0; q < NQ; ++q)   // first_q + 16 q + col: the query's global position
                            if (key > first_q + 16 * q + col || key > last_key) sT[q][kb][v] = -INFINITY;
                    }
            }
        }
        // ---- online softmax (one query column per four lanes: those of equal col) ----
        tile_phase<kPrio>(1);
        x8_t pf[NQ][nkb / 2];
        auto maximum = [&](int q) {
            float mx = -INFINITY;
#pragma unroll
            for (int kb = 0; kb < nkb; ++kb)
#pragma unroll
                for (int v = 0; v < 4; ++v) mx = fmaxf(mx, sT[q][kb][v]);
            return mx * kScaleLog2;
        };
        float ms[NQ];
        bool above = false;
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            ms[q] = maximum(q);
            above |= ms[q] > m[q] + kRefSlack;
        }
        // The references of a block's 32 queries move together: more rows then have their largest probability as an exact 1
        // (each query's for its own scores alone: 1.5 to 2.5 % further from 64-bit outputs).  In halves the other
        // wavefront's queries count too.  (On a first tile the references are -inf and a wavefront in which nothing lies
        // above them has nothing to move.)
        bool move = __any(above);   // wavefront-uniform
        if (NQ == 1 && sq > 0) move = either_half(move);
        if (move) {
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const float mnew = fmaxf(m[q], max_over_quarters(ms[q]));   // the same in the four lanes of a column
                const float corr = (mnew == -INFINITY) ? 1.f : fast_exp2(m[q] - mnew);
                m[q] = mnew;
                l[q] *= corr;
#pragma unroll
                for (int db = 0; db < kDB; ++db) oT[q][db] *= corr;
            }
        }
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const float mu = (m[q] == -INFINITY) ? 0.f : m[q];
            float sum = 0.f;
            float4_t e[nkb];
#pragma unroll
            for (int kb = 0; kb < nkb; ++kb)
#pragma unroll
                for (int v = 0; v < 4; ++v) e[kb][v] = fast_exp2(__builtin_fmaf(sT[q][kb][v], kScaleLog2, -mu));
#pragma unroll
            for (int s = 0; s < nkb / 2; ++s) {
                x8_t t;
#pragma unroll
                for (int i = 0; i < 8; ++i) t[i] = (T)e[2 * s + (i >> 2)][i & 3];
                pf[q][s] = t;
            }
            if (kPairSum) {
#pragma unroll
                for (int s = 0; s < nkb / 2; ++s)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const x2_t pr = {pf[q][s][2 * i], pf[q][s][2 * i + 1]};
                        sum = Elem<T>::add_pair(pr, sum);
                    }
            } else {
#pragma unroll
                for (int kb = 0; kb < nkb; ++kb)
#pragma unroll
                    for (int v = 0; v < 4; ++v) sum += e[kb][v];
            }
            l[q] += sum;   // per-lane partial sum (own key positions)
        }
        tile_phase<kPrio>(2);
        // ---- O^T += V^T P^T: step s covers the keys of blocks 2 s and 2 s + 1, whose scores lane dq holds: rows
        // 32 s + 16 h + 4 dq + (0..3), h = 0, 1, of the tile.  The operands of a group of steps are read
        // while the group before it is multiplied ----
        constexpr int kPS = nkb / 2;
        auto read_v = [&](int db, int s, int h) {
            const T* vp = bV + (32 * s + 16 * h) * D + vrd + ((2 * db) ^ vchunk) * 8;
            return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4_t*)vp);
        };
        // steps in groups of kGrp (a group = 2 kGrp transposing reads, kGrp products per query block),
        // two column blocks in turn
        constexpr int kGrp = (D == 128) ? 4 : 2;
        constexpr int kGroupsPV = kDB * kPS / kGrp;
        auto out_block = [](int t) { return 2 * (t / (2 * kPS)) + (t & 1); };
        auto p_step = [](int t) { return (t % (2 * kPS)) >> 1; };
        short4_t av[2][kGrp][2];
#pragma unroll
        for (int i = 0; i < kGrp; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h) av[0][i][h] = read_v(out_block(i), p_step(i), h);
#pragma unroll
        for (int gq = 0; gq < kGroupsPV; ++gq) {
            if (gq + 1 < kGroupsPV) {
#pragma unroll
                for (int i = 0; i < kGrp; ++i)
#pragma unroll
                    for (int h = 0; h < 2; ++h)
                        av[(gq + 1) & 1][i][h] = read_v(out_block(kGrp * (gq + 1) + i), p_step(kGrp * (gq + 1) + i), h);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < kGrp; ++i) {
                const int db = out_block(kGrp * gq + i), s = p_step(kGrp * gq + i);
                const short8_t both = __builtin_shufflevector(av[gq & 1][i][0], av[gq & 1][i][1], 0, 1, 2, 3, 4, 5, 6, 7);
                const x8_t a = __builtin_bit_cast(x8_t, both);
#pragma unroll
                for (int q = 0; q < NQ; ++q)
                    oT[q][db] = Elem<T>::mma_16x16x32(a, pf[q][s], oT[q][db]);
            }
        }
    };

    if (SPARE && !has_head) {   // wavefront-uniform: this slot only fills its quarter of every tile
#pragma clang loop unroll(disable)
        for (int s = 0; s < ntiles; ++s) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            if (s + 1 < ntiles) {
                next_rows();
                if (s + 2 < ntiles) fetch_ids(tile_at(s + 2));
                static_for<0, kNumLoads>([&](auto i) { issue_load(i, (s + 1) & 1); });
            }
            if (NQ == 1 && s > 0) lds_barrier();   // the one in either_half
        }
        __syncthreads();   // the one behind the last tile
        return;
    }
    int sq = 0;
    if (sparse) {   // a copy of its own where it halves the tile's products (64-key tiles)
        if (kKT == 64) run_tile(0, std::integral_constant<int, kDiag>{});
        else run_tile(0, std::integral_constant<int, kMasked>{});
        sq = 1;
    }
    // tiles wholly below the unit's first query and inside the sequence / wholly inside the selection
    const int full_end = sparse ? 1 + n / kKT : min((q0 + 1) / kKT, L / kKT);
    for (; sq < full_end; ++sq) run_tile(sq, std::integral_constant<int, kFull>{});
    for (; sq < ntiles; ++sq) run_tile(sq, std::integral_constant<int, kMasked>{});
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no load may land in LDS after the workgroup has left

    // ---- epilogue (rows are local to this call).  A lane holds one query's output spread over its
    // registers; the rows go through the wavefront's share of the (now idle) K buffers so that they
    // leave as whole rows: 16-byte stores, four rows per instruction ----
    __syncthreads();   // everybody is done with the tile buffers
    T* so = sK + wave * (32 * D);
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int ql = q0l + q_off + 16 * q + col;
        const float lt = sum_over_quarters(l[q]);
        if (p.log_sum && dq == 0 && ql < Lqv)
            p.log_sum[((long long)b * Lq + ql) * nheads + head] = fast_log2(lt) + m[q];
        const float inv = 1.f / lt;
        const int row = 16 * q + col;
#pragma unroll
        for (int db = 0; db < kDB; ++db) {   // d = 16 db + 4 dq .. +3: half of chunk 2 db + dq / 2
            const x4_t o = {(T)(oT[q][db][0] * inv), (T)(oT[q][db][1] * inv), (T)(oT[q][db][2] * inv), (T)(oT[q][db][3] * inv)};
            *reinterpret_cast<x4_t*>(&so[row * D + (((2 * db + (dq >> 1)) ^ (row & (kChunks - 1))) * 8) + 4 * (dq & 1)]) = o;
        }
    }
    __builtin_amdgcn_wave_barrier();   // the reads below are other lanes' writes (same wavefront: in order)
    store_rows<D, 16 * NQ>((T*)p.O + ((long long)b * Lq + q0l + q_off) * nheads * D + (long long)head * D, (unsigned)(nheads * D),
                           so, lrow, lchunk, last_q - q_off);
}

// Dense passes, with an output or for log-sums alone.
// A row's exponentials are added up in two lanes, as 32x32x16 products leave them, whatever the products: spread over the
// four lanes of 16x16x32 ones the last bits of the log-sums differ, and they decide between tokens whose pooled scores lie
// within one step at a selection's threshold (single output rows of a 32768-token prompt moved by up to 0.27 of the outputs'
// root mean square).  The products' own bits are the same: four chained 16x16x32 products and eight 32x32x16 ones agreed
// in all of 524288 dot products of 128 elements.
// With an output at head_dim 128 (PAIRS): products 16x16x32, and half an instruction per score (swap_pairs) brings the
// exponentials where they are added up.  Against 32x32x16 products, 32/8 heads: 32768 tokens 8.43 -> 7.75 ms, chunks of 2048
// queries at up to 14336 284 -> 268 us, 2300 tokens 62.6 -> 59.7; 517, 1500 and 4096 the same.  The cycles are 1 % more; the clock, which
// the chip's power sets, goes from 1.65 to 1.81 GHz at 32768 tokens.
// Log-sums alone and pooling have half the products per score and wait for vector instructions: with
// the swaps 32768 tokens 4.30 -> 4.34 ms and 4.71 -> 4.85; head_dim 64 with an output, 16000 tokens of 8/2 heads in bf16, 299 ->
// 362 us, 4096 48.4 -> 51.7.  These keep 32x32x16.
template <int NQB, bool WITH_V, bool PAGED, int D, typename T, bool SPARE>
__device__ __forceinline__ void prefill_dense_body(const PrefillParams& p, T* sK, T* sV) {
    typedef typename Elem<T>::x8 x8_t;
    typedef typename Elem<T>::x4 x4_t;
    // Products 16x16x32 (see above)
    constexpr bool PAIRS = WITH_V && D == 128;
    typedef typename std::conditional<PAIRS, float4_t, float16_t>::type Acc;
    typedef AttnTile<D> G_;
    constexpr int kKT = G_::kKT, kChunks = G_::kChunks, kRPL = G_::kRowsPerLoad, kTileElems = G_::kTileElems;
    // rows and columns of a product; contraction steps of S^T, row blocks of O^T, key blocks of a tile, blocks of queries
    constexpr int kOp = PAIRS ? 16 : 32;
    constexpr int kKS = D * kOp / 512, kDB = D / kOp, kKB = kKT / kOp, kQB = NQB * 32 / kOp;
    constexpr int kAcc = kOp * kOp / 64;   // elements of a result per lane
    constexpr float kScaleLog2 = ScaleLog2<D>::value;
    const HeadSlots hs = head_slots(p.gs);
    const int kvh = p.G, nheads = p.G * hs.gs;
    const T* Qp = (const T*)p.Q;
    const T* Kp = (const T*)p.K;
    const T* Vp = (const T*)p.V;

    // All arguments in one trip to memory: left alone, the compiler loads them in three, each where it is first used
    // (with 16x16x32 products: log-sums alone, 1024 tokens 15.9 -> 15.7 us; dense 2048 45.1 -> 44.5).  Sparse units have
    // more arguments than registers to keep them in: 4096 tokens 31.2 -> 31.8.
    asm volatile("" :: "s"(p.q_start_rows), "s"(p.q_len_rows), "s"(p.q_sb), "s"(p.q_sl), "s"(p.q_sh), "s"(p.k_sb), "s"(p.k_sl),
                 "s"(p.k_sh), "s"(p.Q), "s"(p.K), "s"(p.V), "s"(p.L), "s"(p.gs), "s"(p.pair_recip), "s"(p.pairs_fill_xcds),
                 "s"(p.all_resident));
    constexpr int QT = 32 * NQB;
    const int Lq = p.Lq;            // rows of Q and of the outputs per sequence
    const int nqt = (Lq + QT - 1) / QT;
    int blk, g, b;
    unit_of_workgroup(p, p.G * hs.subs, nqt, blk, g, b);   // g: KV head and sub-group
    int q_start, Lqv;               // this sequence's first position and how many of the rows are its own
    chunk_of_sequence(p, b, q_start, Lqv);
    const int L = q_start + Lqv;    // keys of this sequence
    int sub;
    split_sub_group(p, hs.subs, g, sub);   // g: the KV head
    const int tq = nqt - 1 - blk;   // long (late) query blocks first
    const int tid = threadIdx.x;
    const int wave = tid >> 6;
    const int lane = tid & 63;
    const int li = lane & 31;
    const int lg = lane >> 5;
    const int col = lane & (kOp - 1);   // of an operand or result
    const int dq = lane / kOp;          // which 8 elements of a contraction step, which 4 rows of a result
    const int q0l = tq * QT;            // first query row of this block
    if (q0l >= Lqv) return;             // a block past this sequence's rows (uniform over the workgroup)
    const int q0 = q_start + q0l;       // its global position
    const int wave_u = __builtin_amdgcn_readfirstlane(wave);
    const int head = g * hs.gs + min(4 * sub + wave_u, hs.gs - 1);
    const bool has_head = !SPARE || 4 * sub + wave_u < hs.gs;

    const int ntiles = (min(q0 + QT, L) + kKT - 1) / kKT;

    // ---- tile staging: wavefront w fills rows [4w R, 4(w+1) R) of a tile with four loads of R rows
    // each (R = 4 at D = 128, 8 at D = 64); lane = (row within the load, chunk position) ----
    const int lrow = lane / kChunks;
    const int lchunk = lane % kChunks;
    // This lane's four rows sit at LDS rows slot0 + j R (j = load) and hold the four consecutive
    // tile positions pos0 + j: one 16-byte load brings their four indices, one block-table entry
    // covers their page, and the rows of a tile in LDS are a permutation of its keys -- which only
    // the masks need to know (both products contract over the same order).
    const int slot0 = wave * 4 * kRPL + lrow;
    const int pos0 = 4 * (wave * kRPL + lrow);
    // tile position of LDS row `slot`
    auto pos_of_slot = [](int slot) { return 4 * ((slot / (4 * kRPL)) * kRPL + slot % kRPL) + (slot / kRPL) % 4; };
    const T* kbase = PAGED ? Kp + (long long)g * D : Kp + (long long)b * p.k_sb + (long long)g * p.k_sh;
    const unsigned long long v_from_k = (unsigned long long)Vp - (unsigned long long)Kp;   // V shares K's layout
    const int* bt_row = PAGED ? p.block_table + (long long)b * p.max_pages : nullptr;
    const int page_mask = (1 << p.page_shift) - 1;
    const uint32_t lds_k = lds_address(sK) + wave_u * 4096;   // this wavefront's 4 KB of a K buffer
    const uint32_t lds_v = WITH_V ? lds_address(sV) + wave_u * 4096 : 0;
    const unsigned row_bytes = 2 * (PAGED ? (unsigned)(kvh * D) : (unsigned)p.k_sl);   // host checks stride < 2^31

    // PAGED: block-table entry of this lane's rows of a tile (four consecutive keys from a multiple of four on: one
    // page), fetched a tile ahead so that the loads never wait on it
    int page = 0;
    auto fetch_page = [&](int ti) {
        if (PAGED) page = bt_row[min(ti * kKT + pos0, L - 1) >> p.page_shift];
    };
    // K row addresses of a tile; V's are a scalar offset away.  The
    // loads themselves are issued one at a time between the matrix instructions of the first
    // product: a wavefront that issued all eight at once would sit in front of the memory
    // pipeline, which takes 16 cycles per 1 KB load, with nothing running behind it.
    // lane_ptr: the chunk this lane fetches for row j of a tile, within a page if PAGED: one addition a row and
    // tile, one product a tile.
    // At D = 64 rows j and j + 2 are permuted alike: over the paged cache, where registers are scarcer, two pointers do.
    constexpr int kPtrs = PAGED && D == 64 ? 2 : 4;
    const char* lane_ptr[kPtrs];
#pragma unroll
    for (int j = 0; j < kPtrs; ++j)
        lane_ptr[j] = (const char*)(kbase + (lchunk ^ (PAIRS ? swz_pairs<D>(slot0 + j * kRPL) : swz<D>(slot0 + j * kRPL))) * 8) +
                      (unsigned long long)row_bytes * (unsigned)(PAGED ? (pos0 + j) & page_mask : pos0 + j);
    const char* row_ptr[4];
    auto next_rows = [&](int ti) {
        const int k0 = ti * kKT;
        if (k0 + kKT <= L) {   // uniform
            const unsigned long long off = (unsigned long long)row_bytes *
                                           (unsigned)(PAGED ? (page << p.page_shift) + (k0 & page_mask) : k0);
#pragma unroll
            for (int j = 0; j < 4; ++j) row_ptr[j] = lane_ptr[j % kPtrs] + (off + (unsigned long long)row_bytes * (j - j % kPtrs));
        } else {               // rows past the sequence's end: the last one again
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int key = min(k0 + pos0 + j, L - 1);
                const int pos = pos0 + j % kPtrs;   // the row that lane_ptr holds
                const int row = PAGED ? (page << p.page_shift) + (key & page_mask) - (pos & page_mask) : key - pos;
                row_ptr[j] = lane_ptr[j % kPtrs] + (long long)row_bytes * row;
            }
        }
    };
    constexpr int kNumLoads = WITH_V ? 8 : 4;
    auto issue_load = [&](auto i_c, int buf) {   // i < 4: K row group i; else V row group i - 4
        constexpr int i = decltype(i_c)::value;
        if constexpr (i < 4) load_to_lds_16<i * 1024>(row_ptr[i], lds_k + buf * (kTileElems * 2));
        else load_to_lds_16<(i - 4) * 1024>(row_ptr[i - 4] + v_from_k, lds_v + buf * (kTileElems * 2));
    };
    // LDS read positions (elements, within a tile buffer).  A operand of S^T: row 16 kb + pair_row(col), chunk 4 ks + dq; of
    // 32x32x16 products row 32 kb + col, chunk 2 ks + dq.  A operand of O^T (two transposing reads h = 0, 1 of four
    // keys each): the 16 lanes of a quarter address rows 32 s + 16 h + pair_row(4 dq) + (0..3), 16 columns of V from
    // column 16 db on, and receive one column of the four rows each; of 32x32x16 products rows 16 s + 8 h + 4 lg + (0..3)
    // of a key block, 16 columns from column 32 db + 16 (quarter & 1) on.
    const int a_row = PAIRS ? pair_row(col) : col;
    const int kx = dq ^ (PAIRS ? swz_pairs<D>(a_row) : swz<D>(a_row));
    const int krd = a_row * D;
    const int vcol = lane & 15;
    const int vrow = (PAIRS ? pair_row(4 * dq) : 4 * lg) + (vcol >> 2);
    const int vchunk = PAIRS ? ((vcol >> 1) & 1) ^ swz_pairs<D>(vrow)                  // ^ 2 db
                             : 2 * ((lane >> 4) & 1) + ((vcol >> 1) & 1);               // + 4 db
    const int vrd = vrow * D + 4 * (vcol & 1);

    // Softmax state.  m[] is the reference the exponentials are taken against, in log2 units of
    // the scaled scores.  It follows the running maximum lazily: a tile moves it only when one of
    // its scores lies more than kRefSlack above it, so an exponential never exceeds 2^kRefSlack
    // (representable in fp16 and bf16, sums and products are kept in fp32) and the rescaling of the
    // accumulators -- 64 products per lane -- runs on the first tiles of a unit and then almost
    // never.  The quotient is the same: numerator and denominator carry the same factor.
    constexpr int kPrio = WITH_V ? KASCADE_PRIO_V : KASCADE_PRIO_K;
    constexpr float kRefSlack = 8.f;
    float m[kQB], l[NQB];    // m: of the queries kOp q + col; l: of the queries 32 qb + li
    Acc oT[kQB][kDB];        // query block, kOp output columns
#pragma unroll
    for (int q = 0; q < kQB; ++q) {
        m[q] = -INFINITY;
#pragma unroll
        for (int db = 0; db < kDB; ++db)
#pragma unroll
            for (int v = 0; v < kAcc; ++v) oT[q][db][v] = 0.f;
    }
#pragma unroll
    for (int qb = 0; qb < NQB; ++qb) l[qb] = 0.f;

    fetch_page(0);
    next_rows(0);
    static_for<0, kNumLoads>([&](auto i) { issue_load(i, 0); });
    if (ntiles > 1) fetch_page(1);

    // ---- Q fragments (B operand of S^T): query kOp q + col, d chunk dq of step ks; requested after
    // the first tile's rows, which the first barrier waits for ----
    x8_t qf[kQB][kKS];
    const int last_q = min(QT, Lqv - q0l) - 1;   // of this block
    const T* q_base = Qp + (long long)b * p.q_sb + (long long)q0l * p.q_sl + (long long)head * p.q_sh;
#pragma unroll
    for (int q = 0; q < kQB; ++q) {
        const T* qp = q_base + (unsigned long long)(unsigned)min(kOp * q + col, last_q) * (unsigned long long)p.q_sl + dq * 8;
#pragma unroll
        for (int ks = 0; ks < kKS; ++ks) {
            PackT<T> t;
            t.u = ld_global_16(qp + ks * (512 / kOp));
            qf[q][ks] = t.v8;
        }
    }
    if (last_q < QT - 1) {   // uniform: rows past the sequence's end are zeros
#pragma unroll
        for (int q = 0; q < kQB; ++q)
#pragma unroll
            for (int ks = 0; ks < kKS; ++ks)
                if (kOp * q + col > last_q) qf[q][ks] = x8_t{};
    }
#pragma unroll
    for (int q = 0; q < kQB; ++q) arrived<kKS>(qf[q]);

    // One tile: next tile's loads, both products, softmax.  Two copies of
    // the code, each straight-line: tiles that need no mask (all but one or two of a unit) and tiles
    // that do (the causal edge, the end of the sequence).
    auto run_tile = [&](int sq, auto masked_c) {
        constexpr bool MASKED = decltype(masked_c)::value;
        constexpr int nkb = kKB;
        const T* bK = sK + (sq & 1) * kTileElems;
        const T* bV = sV + (sq & 1) * kTileElems;
        // own loads of this tile landed; after the barrier everybody's have, and everybody is done
        // reading the other buffer (the tile before), which the next tile's loads may now fill
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        // The next tile's loads go out between the products below, unconditionally: after the last
        // tile they fetch its rows once more into the idle buffer (1/28 of the traffic on average,
        // from the cache) rather than put a branch between the matrix instructions.
        // The block-table entry of the tile behind that one is requested before those loads: the compiler waits for
        // every load on its way before it lets one of its own overwrite a register, and behind the
        // tile's loads that wait was a whole trip to memory (chunk of 512 queries at 14336: 324 -> 260 us).
        if (sq + 1 < ntiles) next_rows(sq + 1);
        if (sq + 2 < ntiles) fetch_page(sq + 2);
        const int nbuf = (sq + 1) & 1;

        tile_phase<kPrio>(0);
        // ---- S^T = K_tile Q^T.  Step c = (key block, contraction step), with an output two key blocks in turn; operands are
        // read from LDS two windows (four steps) ahead of the products that use them, in program
        // order, because LDS reads do not move across the load statements ----
        constexpr int kSteps = nkb * kKS;
        Acc sT[kQB][nkb];
        Acc zero;
#pragma unroll
        for (int v = 0; v < kAcc; ++v) zero[v] = 0.f;
        auto key_block = [](int c) { return PAIRS ? 2 * (c / (2 * kKS)) + (c & 1) : c / kKS; };
        auto k_step = [](int c) { return PAIRS ? (c % (2 * kKS)) >> 1 : c % kKS; };
        auto read_a = [&](int c) {
            return *reinterpret_cast<const x8_t*>(&bK[kOp * key_block(c) * D + krd + ((64 / kOp * k_step(c)) ^ kx) * 8]);
        };
        constexpr int kAhead = (D == 128) ? 2 : 1;   // windows read ahead (registers are scarcer at D = 64)
        x8_t aw[kAhead + 1][2];
#pragma unroll
        for (int c = 0; c < 2 * kAhead && c < kSteps; ++c) aw[c >> 1][c & 1] = read_a(c);
        static_for<0, kSteps / 2>([&](auto w_c) {
            constexpr int w = decltype(w_c)::value;
            if (2 * (w + kAhead) < kSteps) {
                aw[(w + kAhead) % (kAhead + 1)][0] = read_a(2 * (w + kAhead));
                aw[(w + kAhead) % (kAhead + 1)][1] = read_a(2 * (w + kAhead) + 1);
            }
            __builtin_amdgcn_sched_barrier(0);   // the scheduler would sink the reads to their use
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int kb = key_block(2 * w + i), ks = k_step(2 * w + i);
#pragma unroll
                for (int q = 0; q < kQB; ++q) {   // the first product starts from a constant zero
                    const Acc c = ks == 0 ? zero : sT[q][kb];
                    if constexpr (PAIRS) sT[q][kb] = Elem<T>::mma_16x16x32(aw[w % (kAhead + 1)][i], qf[q][ks], c);
                    else sT[q][kb] = Elem<T>::mma_32x32x16(aw[w % (kAhead + 1)][i], qf[q][ks], c);
                }
            }
            if constexpr (w < kNumLoads) issue_load(w_c, nbuf);
        });
        static_for<kSteps / 2, kNumLoads>([&](auto i) { issue_load(i, nbuf); });
        // ---- masks: accumulator v of key block kb is LDS row 16 kb + pair_row(4 dq) + v of the tile
        // (32x32x16: 32 kb + 8 (v/4) + 4 dq + v%4) ----
        if (MASKED) {   // the causal edge and the end of the sequence
#pragma unroll
            for (int qb = 0; qb < kQB; ++qb) {
                const int q = q0 + kOp * qb + col;   // global position
#pragma unroll
                for (int kb = 0; kb < nkb; ++kb)
#pragma unroll
                    for (int v = 0; v < kAcc; ++v) {
                        const int row = PAIRS ? pair_row(4 * dq) + v : 8 * (v >> 2) + 4 * dq + (v & 3);
                        const int key = sq * kKT + pos_of_slot(kOp * kb + row);
                        if (key > q || key >= L) sT[qb][kb][v] = -INFINITY;
                    }
            }
        }
        // ---- online softmax (a query's scores lie in the four lanes of equal col; of 32x32x16 products in two) ----
        tile_phase<kPrio>(1);
        if constexpr (PAIRS) {
            x8_t pf[2][nkb / 2];
            float ms[2];
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                float mx = -INFINITY;
#pragma unroll
                for (int kb = 0; kb < nkb; ++kb)
#pragma unroll
                    for (int v = 0; v < 4; ++v) mx = fmaxf(mx, sT[q][kb][v]);
                ms[q] = mx * kScaleLog2;
            }
            if (__any(ms[0] > m[0] + kRefSlack || ms[1] > m[1] + kRefSlack)) {   // wavefront-uniform
                float corr[2];
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const float mnew = fmaxf(m[q], max_over_quarters(ms[q]));   // the same in the four lanes of a column
                    corr[q] = (mnew == -INFINITY) ? 1.f : fast_exp2(m[q] - mnew);
                    m[q] = mnew;
#pragma unroll
                    for (int db = 0; db < kDB; ++db) oT[q][db] *= corr[q];
                }
                l[0] *= lane & 16 ? corr[1] : corr[0];
            }
            const float mu[2] = {m[0] == -INFINITY ? 0.f : m[0], m[1] == -INFINITY ? 0.f : m[1]};
            float sum = 0.f;
            float4_t e[2][nkb];
            // The sums are formed where and as those of the pass for log-sums alone: in two lanes per query, by the same
            // additions (lane & 16 picks a lane's query of the two whose reference it holds).  Behind the conversions: the
            // swap is made in place then, in front of them the compiler copied every exponential first (32768
            // tokens 7.74 ms both, 4096 156 -> 149 us, 517 17.0 -> 15.9).
            auto add = [&](int kb) {
                float4_t first, second;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    float x, y;
                    swap_pairs(e[0][kb][v], e[1][kb][v], x, y);
                    first[v] = x;
                    second[v] = y;
                }
#pragma unroll
                for (int v = 0; v < 4; ++v) sum += first[v];
#pragma unroll
                for (int v = 0; v < 4; ++v) sum += second[v];
            };
#pragma unroll
            for (int st = 0; st < nkb / 2; ++st) {
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    x8_t t;
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const int kb = 2 * st + (i >> 2), v = i & 3;
                        e[q][kb][v] = fast_exp2(__builtin_fmaf(sT[q][kb][v], kScaleLog2, -mu[q]));
                        t[i] = (T)e[q][kb][v];
                    }
                    pf[q][st] = t;
                }
                if (st > 0) {
                    add(2 * st - 2);
                    add(2 * st - 1);
                }
            }
            add(nkb - 2);
            add(nkb - 1);
            l[0] += sum;   // per-lane partial sum (own key positions)
            tile_phase<kPrio>(2);
            // ---- O^T += V^T P^T: step s covers the keys of blocks 2 s and 2 s + 1, whose scores lane dq holds: rows
            // 32 s + 16 h + pair_row(4 dq) + (0..3), h = 0, 1, of the tile.  The operands of a group of steps are read
            // while the group before it is multiplied ----
            constexpr int kPS = nkb / 2;
            auto read_v = [&](int db, int s, int h) {
                const T* vp = bV + (32 * s + 16 * h) * D + vrd + ((2 * db) ^ vchunk) * 8;
                return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4_t*)vp);
            };
            // steps in groups of kGrp (a group = 2 kGrp transposing reads, kGrp products per query block),
            // two column blocks in turn
            constexpr int kGrp = (D == 128) ? 4 : 2;
            constexpr int kGroupsPV = kDB * kPS / kGrp;
            auto out_block = [](int t) { return 2 * (t / (2 * kPS)) + (t & 1); };
            auto p_step = [](int t) { return (t % (2 * kPS)) >> 1; };
            short4_t av[2][kGrp][2];
#pragma unroll
            for (int i = 0; i < kGrp; ++i)
#pragma unroll
                for (int h = 0; h < 2; ++h) av[0][i][h] = read_v(out_block(i), p_step(i), h);
#pragma unroll
            for (int gq = 0; gq < kGroupsPV; ++gq) {
                if (gq + 1 < kGroupsPV) {
#pragma unroll
                    for (int i = 0; i < kGrp; ++i)
#pragma unroll
                        for (int h = 0; h < 2; ++h)
                            av[(gq + 1) & 1][i][h] = read_v(out_block(kGrp * (gq + 1) + i), p_step(kGrp * (gq + 1) + i), h);
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < kGrp; ++i) {
                    const int db = out_block(kGrp * gq + i), s = p_step(kGrp * gq + i);
                    const short8_t both = __builtin_shufflevector(av[gq & 1][i][0], av[gq & 1][i][1], 0, 1, 2, 3, 4, 5, 6, 7);
                    const x8_t a = __builtin_bit_cast(x8_t, both);
#pragma unroll
                    for (int q = 0; q < 2; ++q) oT[q][db] = Elem<T>::mma_16x16x32(a, pf[q][s], oT[q][db]);
                }
            }
        } else {
            x8_t pf[NQB][2 * nkb];
#pragma unroll
            for (int qb = 0; qb < NQB; ++qb) {
                float sum;
                auto exponentials = [&](float mu) {
                    sum = 0.f;
                    float e[nkb][16];
                    // At head_dim 64 a tile's 64 additions stand behind all of its exponentials: mixed with them, as at 128,
                    // their chain holds these up (14/2 heads, 4096 tokens: log-sums alone 48.6 -> 45.6 us, dense 66.7 ->
                    // 60.6; 32/8 heads: 53.2 -> 51.7 and 88.7 -> 84.0; a chunk of 2048 queries at 14336 196 -> 181 and 293
                    // -> 277; slower at 3001 tokens of 32/8 heads, log-sums alone 32.7 -> 33.7, and 8192 of 14/2, dense 188
                    // -> 193).  The order of addition is the same.
                    constexpr bool kSumsBehind = D == 64;
#pragma unroll
                    for (int kb = 0; kb < nkb; ++kb)
#pragma unroll
                        for (int v = 0; v < 16; ++v) {
                            e[kb][v] = fast_exp2(__builtin_fmaf(sT[qb][kb][v], kScaleLog2, -mu));
                            if (!kSumsBehind) sum += e[kb][v];
                        }
                    if (WITH_V) {
#pragma unroll
                        for (int s = 0; s < 2 * nkb; ++s) {
                            x8_t t;
#pragma unroll
                            for (int i = 0; i < 8; ++i) t[i] = (T)e[s >> 1][8 * (s & 1) + i];
                            pf[qb][s] = t;
                        }
                    }
                    if (kSumsBehind) {
                        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                        for (int kb = 0; kb < nkb; ++kb)
#pragma unroll
                            for (int v = 0; v < 16; ++v) sum += e[kb][v];
                    }
                };
                // Log-sums alone: the maximum is only formed on a unit's first tiles, which move the reference often (16 of 64
                // keys, all of 128), and where a lane's sum says that a score may lie kRefSlack above the reference (its
                // exponential alone is 2^kRefSlack then), or is no number (the reference still is -inf); then the
                // exponentials are formed anew.  The rule is the same: the log-sums have the bits of the pass with an output.
                constexpr float kSumLimit = 250.f;
                bool look = WITH_V || D == 64 || sq < 16;   // wavefront-uniform
                if (!look) {
                    exponentials(m[qb]);
                    look = __any(!(sum <= kSumLimit));
                }
                if (look) {
                    float mx = -INFINITY;
#pragma unroll
                    for (int kb = 0; kb < nkb; ++kb)
#pragma unroll
                        for (int v = 0; v < 16; ++v) mx = fmaxf(mx, sT[qb][kb][v]);
                    const float ms = mx * kScaleLog2;
                    if (__any(ms > m[qb] + kRefSlack)) {   // wavefront-uniform
                        const float mnew = fmaxf(m[qb], max_with_other_half(ms));   // the same in both lanes of a column
                        const float corr = (mnew == -INFINITY) ? 1.f : fast_exp2(m[qb] - mnew);
                        m[qb] = mnew;
                        l[qb] *= corr;
                        if (WITH_V) {
#pragma unroll
                            for (int db = 0; db < kDB; ++db)
#pragma unroll
                                for (int v = 0; v < 16; ++v) oT[qb][db][v] *= corr;
                        }
                    }
                    exponentials((m[qb] == -INFINITY) ? 0.f : m[qb]);
                }
                l[qb] += sum;   // per-lane partial sum (own key positions)
            }
            tile_phase<kPrio>(2);
            // ---- O^T += V^T P^T: step s covers the keys of accumulators 8(s&1) .. 8(s&1)+7 of key block
            // s/2, i.e. rows 16 s + 8 h + 4 lg + (0..3), h = 0, 1, of the tile.  The operands of a block
            // of 32 output rows are read while the block before it is multiplied ----
            if (WITH_V) {
                constexpr int kPS = 2 * nkb;
                auto read_v = [&](int db, int s, int h) {
                    const int row = 16 * s + 8 * h;   // + vrow; only its low four bits enter swz
                    const T* vp = bV + row * D + vrd + ((4 * db + vchunk) ^ swz<D>(row + vrow)) * 8;
                    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4_t*)vp);
                };
                // steps in groups of kGrp (a group = 2 kGrp transposing reads, kGrp products per query block)
                constexpr int kGrp = (kKB <= 2) ? 4 : 2;
                constexpr int kGroupsPV = kDB * kPS / kGrp;
                short4_t av[2][kGrp][2];
#pragma unroll
                for (int i = 0; i < kGrp; ++i)
#pragma unroll
                    for (int h = 0; h < 2; ++h) av[0][i][h] = read_v(i / kPS, i % kPS, h);
#pragma unroll
                for (int gq = 0; gq < kGroupsPV; ++gq) {
                    if (gq + 1 < kGroupsPV) {
#pragma unroll
                        for (int i = 0; i < kGrp; ++i)
#pragma unroll
                            for (int h = 0; h < 2; ++h)
                                av[(gq + 1) & 1][i][h] = read_v((kGrp * (gq + 1) + i) / kPS, (kGrp * (gq + 1) + i) % kPS, h);
                    }
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int i = 0; i < kGrp; ++i) {
                        const int db = (kGrp * gq + i) / kPS, s = (kGrp * gq + i) % kPS;
                        const short8_t both = __builtin_shufflevector(av[gq & 1][i][0], av[gq & 1][i][1], 0, 1, 2, 3, 4, 5, 6, 7);
                        const x8_t a = __builtin_bit_cast(x8_t, both);
#pragma unroll
                        for (int qb = 0; qb < NQB; ++qb)
                            oT[qb][db] = Elem<T>::mma_32x32x16(a, pf[qb][s], oT[qb][db]);
                    }
                }
            }
        }
    };

    if (SPARE && !has_head) {   // wavefront-uniform: this slot only fills its quarter of every tile
#pragma clang loop unroll(disable)
        for (int s = 0; s < ntiles; ++s) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            if (s + 1 < ntiles) {
                next_rows(s + 1);
                if (s + 2 < ntiles) fetch_page(s + 2);
                static_for<0, kNumLoads>([&](auto i) { issue_load(i, (s + 1) & 1); });
            }
        }
        if (WITH_V) __syncthreads();   // the one behind the last tile
        return;
    }
    // tiles wholly below the unit's first query and inside the sequence need no mask
    const int full_end = min((q0 + 1) / kKT, L / kKT);
    int sq = 0;
    for (; sq < full_end; ++sq) run_tile(sq, std::false_type{});
    for (; sq < ntiles; ++sq) run_tile(sq, std::true_type{});
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no load may land in LDS after the workgroup has left

    // ---- epilogue (rows are local to this call).  A lane holds one query's output spread over its
    // registers; the rows go through the wavefront's share of the (now idle) K buffers so that they
    // leave as whole rows: 16-byte stores, four rows per instruction ----
    static_assert(!WITH_V || NQB == 1, "the output pass is written for 32 queries per wavefront");
    if (WITH_V) __syncthreads();   // everybody is done with the tile buffers
#pragma unroll
    for (int qb = 0; qb < NQB; ++qb) {
        const int ql = q0l + 32 * qb + li;
        const float lt = sum_with_other_half(l[qb]);
        const float ref = !PAIRS ? m[qb] : lane & 16 ? m[kQB - 1] : m[0];
        if (p.log_sum && lg == 0 && ql < Lqv)
            p.log_sum[((long long)b * Lq + ql) * nheads + head] = fast_log2(lt) + ref;
        T* so = sK + wave * (32 * D);
        auto store = [&]() {
            __builtin_amdgcn_wave_barrier();   // the reads below are other lanes' writes (same wavefront: in order)
            store_rows<D, 32>((T*)p.O + ((long long)b * Lq + q0l) * nheads * D + (long long)head * D, (unsigned)(nheads * D), so, lrow,
                              lchunk, last_q);
        };
        if constexpr (PAIRS) {
            const float inv_li = 1.f / lt;
            float inv[2];   // of the queries 16 q + col
            swap_pairs(inv_li, inv_li, inv[0], inv[1]);
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int row = 16 * q + col;
#pragma unroll
                for (int db = 0; db < kDB; ++db) {   // d = 16 db + 4 dq .. +3: half of chunk 2 db + dq / 2
                    const x4_t o = {(T)(oT[q][db][0] * inv[q]), (T)(oT[q][db][1] * inv[q]), (T)(oT[q][db][2] * inv[q]),
                                    (T)(oT[q][db][3] * inv[q])};
                    *reinterpret_cast<x4_t*>(&so[row * D + (((2 * db + (dq >> 1)) ^ (row & (kChunks - 1))) * 8) + 4 * (dq & 1)]) = o;
                }
            }
            store();
        } else if constexpr (WITH_V) {
            const float inv = 1.f / lt;
#pragma unroll
            for (int db = 0; db < kDB; ++db)
#pragma unroll
                for (int v4 = 0; v4 < 4; ++v4) {   // d = 32 db + 8 v4 + 4 lg .. +3: chunk 4 db + v4 of row li
                    x4_t o = {(T)(oT[qb][db][4 * v4 + 0] * inv), (T)(oT[qb][db][4 * v4 + 1] * inv),
                              (T)(oT[qb][db][4 * v4 + 2] * inv), (T)(oT[qb][db][4 * v4 + 3] * inv)};
                    *reinterpret_cast<x4_t*>(&so[li * D + (((4 * db + v4) ^ (li & (kChunks - 1))) * 8) + 4 * lg]) = o;
                }
            store();
        }
    }
}

// 32 queries per wavefront: register budget capped so that two workgroups share a
// compute unit (64 KB of LDS each: two K and two V tile buffers), four without V (log-sums alone over the paged
// cache at head_dim 64, in 134 registers and three: four chunks of 1024 queries at 4096, 32/8 heads, 122.5 -> 116.5 us).
template <bool REUSE, bool WITH_V, bool PAGED, int D, typename T, bool SPARE, bool EXACT_SUM = false>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(REUSE || WITH_V ? 2 : 4)))
void prefill_attn_kernel_q32(PrefillParams p) {
    __shared__ __attribute__((aligned(1024))) T sK[2 * AttnTile<D>::kTileElems];
    __shared__ __attribute__((aligned(1024))) T sV[WITH_V ? 2 * AttnTile<D>::kTileElems : 8];
    if constexpr (REUSE) prefill_reuse_body<PAGED, D, T, SPARE, EXACT_SUM, 2>(p, sK, sV);
    else prefill_dense_body<1, WITH_V, PAGED, D, T, SPARE>(p, sK, sV);
}

// Sparse units in halves of two head slots, 16 queries per wavefront (see kSplitUnits).
template <bool PAGED, int D, typename T, bool SPARE>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2)))
void prefill_sparse_halves_kernel(PrefillParams p) {
    __shared__ __attribute__((aligned(1024))) T sK[2 * AttnTile<D>::kTileElems];
    __shared__ __attribute__((aligned(1024))) T sV[2 * AttnTile<D>::kTileElems];
    __shared__ int s_move[kThreads / 64];   // either_half
    prefill_reuse_body<PAGED, D, T, SPARE, false, 1>(p, sK, sV, s_move);
}

// 64 queries per wavefront for the K-only log-sum pass, whose state fits 256 registers: two
// workgroups per compute unit, and the MFMA results stay in ordinary registers (with the full
// 512-register budget the compiler parks them in accumulation registers and copies each one out
// before the softmax).
template <bool PAGED, int D, typename T, bool SPARE>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2)))
void prefill_attn_kernel_q64(PrefillParams p) {
    __shared__ __attribute__((aligned(1024))) T sK[2 * AttnTile<D>::kTileElems];
    prefill_dense_body<2, false, PAGED, D, T, SPARE>(p, sK, static_cast<T*>(nullptr));
}

// Pooled tile scores: out[b,g,t,key] = sum over the 32 queries of tile t and the 4 q-heads of g
// of exp2(s*scale - log_sum), for keys before the tile's first (global) position.
// NH: query heads of the launch's sub-group.  8 KV heads with 1, 2 and 3 query heads each, as four slots -> as they are: 4096
// tokens 79, 78, 80 -> 32.7, 48.4, 65.0 us, 517 tokens 8.9 -> 5.9, 6.5, 7.5.
// Two workgroups per compute unit (register budget 256): one wavefront's exponentials run
// under the other's matrix instructions.  With 16x16x32 products, row addresses from scalar registers and the last
// head's exponentials across the tile boundary 32768 tokens took 4.1 ms instead of 4.6, but a key's sum was then spread
// over four lanes instead of two, and its last bits decide between tokens whose pooled scores lie within one
// step at a selection's threshold (the products' own bits are the same, see the dense passes).
//
// A wavefront takes 32 keys of every 128-key tile and nobody else reads them.  Their rows go
// from global memory straight into the wavefront's own LDS area (whole rows per load: read as
// B operands directly, a 16-byte piece of 32 different rows per instruction, the same bytes kept
// the data-return path of the memory pipeline busy 96 % of the kernel) and come back as B
// operands (lane = key, 8 elements at d = 16 ks + 8 lg) from the chunk-permuted rows.  Two buffers
// per wavefront, no barrier in the tile loop: the loads of the next tile are issued one per
// contraction step and waited for at the top of that tile.
// ACC: adds to the scores of the KV head's earlier sub-groups, which are requested with the tile's products ahead of them.
// A uniform branch instead of the template: 40/8 heads, 517 tokens 12.9 -> 14.3 us, 28/4 heads, two prompts of 3001 tokens
// 83.6 -> 87.3 (both launches each).
// WAVES: wavefronts of the workgroup, a tile is 32 keys for each.
// MAXC > 0: the workgroup has all keys of its tile, keeps the pooled row in LDS and selects from it (see
// prefill_pool_select_kernel).
template <bool PAGED, int D, typename T, int NH, bool ACC, int WAVES, int MAXC>
__device__ __forceinline__ void prefill_pool_body(const PrefillParams& p, const SelectParams& sel) {
    constexpr int kThreads = WAVES * 64, kAggKT = WAVES * 32;
    constexpr bool SELECT = MAXC > 0;
    typedef typename Elem<T>::x8 x8_t;
    constexpr int kKS = D / 16;
    constexpr int kChunks = D / 8;
    constexpr int kRPL = 64 / kChunks;          // rows per load instruction
    constexpr int kLoads = 32 / kRPL;           // load instructions per wavefront and tile
    constexpr int kWaveElems = 32 * D;          // a wavefront's 32 rows
    constexpr float kScaleLog2 = ScaleLog2<D>::value;
    const HeadSlots hs = head_slots(p.gs);
    const int kvh = p.G, nheads = p.G * hs.gs;
    const T* Qp = (const T*)p.Q;
    const T* Kp = (const T*)p.K;
    typedef SelectLds<kThreads, false> Histograms;   // in the tiles' place
    constexpr size_t kTileBytes = 2 * WAVES * kWaveElems * sizeof(T);
    __shared__ __attribute__((aligned(1024))) char s_tiles[SELECT && sizeof(Histograms) > kTileBytes ? sizeof(Histograms) : kTileBytes];
    T* sK = reinterpret_cast<T*>(s_tiles);
    __shared__ __attribute__((aligned(16))) float s_lse[128];
    __shared__ __attribute__((aligned(16))) uint16_t s_row[SELECT ? kThreads * 8 * MAXC : 8];   // pooled scores as fp16

    // All arguments in one trip to memory, and the log-sums, which the first exponentials need, not waited for before the
    // first rows are requested (with the scores of earlier sub-groups ahead of a tile's products: 517 tokens 8.8 -> 7.9 us,
    // bf16 4096 tokens 81.2 -> 79.6; two prompts of 3001 tokens at 28/4 heads 50.8 -> 48.6 and, adding, 45.4 -> 41.2)
    asm volatile("" :: "s"(p.Q), "s"(p.K), "s"(p.log_sum_in), "s"(p.agg), "s"(p.q_start_rows), "s"(p.q_len_rows), "s"(p.q_sb),
                 "s"(p.q_sl), "s"(p.q_sh), "s"(p.k_sb), "s"(p.k_sl), "s"(p.k_sh), "s"(p.L), "s"(p.gs), "s"(p.part_tiles),
                 "s"(p.vsub), "s"(p.fill_invalid), "s"(p.pair_recip), "s"(p.pairs_fill_xcds), "s"(p.all_resident));
    const int Ls = p.L;                  // width of a row of pooled scores
    const int Lq = p.Lq;
    int blk, g, b;
    unit_of_workgroup(p, p.G, p.T * p.key_parts, blk, g, b);
    const int part = blk / p.T;          // part 0 of every tile first, long tiles first within a part
    blk -= part * p.T;
    int q_start, Lqv;                    // this sequence's first position and how many of the rows are its own
    chunk_of_sequence(p, b, q_start, Lqv);
    const int L = q_start + Lqv;         // keys of this sequence
    const int t = p.T - 1 - blk;
    const int tid = threadIdx.x;
    const int wave = tid >> 6;
    const int lane = tid & 63;
    const int li = lane & 31;
    const int lg = lane >> 5;
    const int tl = t * kTile;            // first query row of the tile
    const int ts = q_start + tl;         // its global position
    half_t* out = p.agg + (((long long)b * kvh + g) * p.T + t) * Ls;
    const half_t neg_inf = (half_t)(-INFINITY);

    const int ntiles = tl < Lqv ? (ts + kAggKT - 1) / kAggKT : 0;   // a tile past the sequence's rows pools nothing
    const int ti0 = part * p.part_tiles, ti1 = min(ntiles, ti0 + p.part_tiles);   // this workgroup's key tiles
    if (ti0 < ti1) {
        const int head0 = g * hs.gs + 4 * p.vsub;
        // wavefronts 0 and 1: the log-sum of a query row and head slot (the others ask for slots of theirs again)
        const int lse_q = tl + (tid & 31), lse_slot = (tid >> 5) & 3;
        const float lse_in = p.log_sum_in[((long long)b * Lq + min(lse_q, Lqv - 1)) * nheads +
                                          min(head0 + lse_slot, g * hs.gs + hs.gs - 1)];

        // ---- staging: load j of a tile covers rows j kRPL + lrow of the wavefront's 32.  Its slices of tiles
        // ti0 .. ti0 + n - 1 hold keys before the query tile (all inside the sequence), in whole slices; for a tile behind
        // those it stages the last one again.  A row address is one addition, a pointer per lane that never
        // changes plus an offset in scalar registers (formed per lane, addresses were one vector instruction in four).
        // kLanePages: rows over the paged cache at D = 64, whose loads take eight rows and so up to two pages, are formed
        // per lane all the same (14/2 heads, 512 tokens 15.1 -> 14.2 us, 2048 queries at 14336 128.5 -> 127.6; 32/8
        // heads: 512 queries at 2048 12.5 -> 12.1) ----
        constexpr bool kLanePages = PAGED && D == 64;
        const int wave_u = __builtin_amdgcn_readfirstlane(wave);
        const int n = min(ti1 - ti0, (ts / 32 - (WAVES * ti0 + wave_u) + WAVES - 1) / WAVES);
        auto key_of_tile = [&](int ti) { return n > 0 ? min(ti, ti0 + n - 1) * kAggKT + 32 * wave_u : 0; };
        const int lrow = lane / kChunks;
        const int lchunk = lane % kChunks;
        constexpr int kPatterns = kLoads / 2;       // chunk permutations: loads j and j + kPatterns have the same
        const unsigned row_stride = PAGED ? (unsigned)(kvh * D) : (unsigned)p.k_sl;
        const T* kbase = PAGED ? Kp + (long long)g * D : Kp + (long long)b * p.k_sb + (long long)g * p.k_sh;
        const char* lane_ptr[kPatterns];
#pragma unroll
        for (int j = 0; j < kPatterns; ++j)
            lane_ptr[j] = (const char*)(kbase + (kLanePages ? 0ll : (long long)((unsigned long long)(unsigned)lrow * row_stride)) +
                                        (lchunk ^ swz<D>(j * kRPL + lrow)) * 8);
        const int* bt_row = PAGED ? p.block_table + (long long)b * p.max_pages : nullptr;
        const int page_mask = (1 << p.page_shift) - 1;
        constexpr int kBufElems = WAVES * kWaveElems;
        const uint32_t lds_w = lds_address(sK) + wave_u * (kWaveElems * 2);   // + buf * kBufElems * 2
        const T* my_k = sK + wave * kWaveElems;
        // Block-table entries of 64 pages, one per lane (pages are at least four tokens, 64 of them two tiles),
        // and of the 64 behind them; with kLanePages the entries of the slice's 32 keys and of the next slice's
        int pages = 0, pages_next = 0, page_group = 0;
        auto fetch_pages = [&](int group) { return bt_row[min(64 * group + lane, p.max_pages - 1)]; };
        auto fetch_slice = [&](int ti) { return bt_row[(key_of_tile(ti) + li) >> p.page_shift]; };
        if (kLanePages) {
            pages_next = fetch_slice(ti0);
        } else if (PAGED) {
            page_group = (key_of_tile(ti0) >> p.page_shift) >> 6;
            pages = fetch_pages(page_group);
            pages_next = fetch_pages(page_group + 1);
        }
        unsigned long long row_off = 0;   // strided: offset of the next load's first row
        const unsigned long long row_step = (unsigned long long)row_stride * (2 * kRPL);
        int key0 = 0;                     // first key of the tile whose loads are being issued
        auto offset_of_key = [&](int key) {   // uniform
            int row = key;
            if (PAGED) {
                const int page = __builtin_amdgcn_readlane(pages, (key >> p.page_shift) & 63);
                row = (page << p.page_shift) + (key & page_mask);
            }
            unsigned long long off = (unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane(row) * row_stride * 2;
            asm("" : "+s"(off));   // stays in scalar registers: the compiler would multiply once per lane
            return off;
        };
        auto enter_tile = [&](int ti) {   // before the loads of a tile, tiles in order
            key0 = key_of_tile(ti);
            if (kLanePages) {
                pages = pages_next;
                pages_next = fetch_slice(ti + 1);
            } else if (PAGED) {
                const int group = (key0 >> p.page_shift) >> 6;
                if (group != page_group) {   // uniform
                    page_group = group;
                    pages = pages_next;
                    pages_next = fetch_pages(group + 1);
                }
            } else {
                row_off = offset_of_key(key0);
            }
        };
        auto issue_load = [&](int j, int buf) {   // loads of a tile in order
            const uint32_t lds = lds_w + buf * (kBufElems * 2) + j * 1024;
            unsigned long long off = row_off;
            if (PAGED) {
                const int key = key0 + j * kRPL;
                if (kLanePages) {
                    const int page = __builtin_amdgcn_ds_bpermute((j * kRPL + lrow) << 2, pages);
                    const unsigned row = (unsigned)((page << p.page_shift) + ((key + lrow) & page_mask));
                    load_to_lds_16(lane_ptr[j % kPatterns] + (unsigned long long)row * row_stride * 2, lds);
                    return;
                }
                off = offset_of_key(key);
            } else {
                row_off += row_step;
            }
            load_to_lds_16(lane_ptr[j % kPatterns] + off, lds);
        };
        // The tile's Q rows, head slot `wave` of the sub-group by this wavefront: whole rows into the
        // other buffer, chunks permuted like the keys' (fragments read from memory directly, every
        // wavefront all four heads, 16 bytes of 32 rows per instruction, held every workgroup up at its start:
        // 32/8 heads, 512 tokens 13.1 -> 10.4 us, 1024 18.9 -> 16.2, 2048 35.5 -> 28.9, 4096 87 -> 84).
        constexpr int kQLoads = kLoads * 4 / WAVES;   // a slot's rows by one wavefront, or half of them by each of two
        const int q_slot = wave_u & 3, q_first = (wave_u >> 2) * kQLoads;
#pragma unroll
        for (int j = 0; j < kQLoads; ++j) {
            const int row = (q_first + j) * kRPL + lrow;
            const T* qp = Qp + (long long)b * p.q_sb + (long long)min(tl + row, Lqv - 1) * p.q_sl +
                          (long long)min(head0 + q_slot, g * hs.gs + hs.gs - 1) * p.q_sh;
            load_to_lds_16(qp + (lchunk ^ swz<D>(row)) * 8, lds_address(sK) + ((ti0 + 1) & 1) * (kBufElems * 2) +
                                                            q_slot * (kWaveElems * 2) + (q_first + j) * 1024);
        }
        enter_tile(ti0);
#pragma unroll
        for (int j = 0; j < kLoads; ++j) issue_load(j, ti0 & 1);
        const int kx = lg ^ swz<D>(li);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // own rows have landed
        // a query row past the chunk, or a slot past the KV head's last query head, adds exp2(-inf) = 0
        if (tid < 128) s_lse[tid] = lse_q < Lqv && 4 * p.vsub + lse_slot < hs.gs ? lse_in : INFINITY;
        __syncthreads();                                   // everybody's, and s_lse
        // A operands: row block rb = head slot rb, row li = query tl + li
        x8_t qa[NH][kKS];
        const T* sQ = sK + ((ti0 + 1) & 1) * kBufElems;
#pragma unroll
        for (int rb = 0; rb < NH; ++rb)
#pragma unroll
            for (int ks = 0; ks < kKS; ++ks) {
                PackT<T> x;
                x.v8 = *reinterpret_cast<const x8_t*>(&sQ[rb * kWaveElems + li * D + ((2 * ks) ^ kx) * 8]);
                if (tl + li >= Lqv) x.u = uint4_t{0, 0, 0, 0};
                qa[rb][ks] = x.v8;
            }
        __syncthreads();   // the other buffer takes the next tile's keys from here on

        for (int ti = ti0; ti < ti1; ++ti) {
            // this tile's rows have landed (and the next tile's block-table entries arrived)
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            const T* bK = my_k + (ti & 1) * kBufElems;
            const int tn = min(ti + 1, ti1 - 1);   // after the last tile: its rows once more, unused
            const int nbuf = (ti + 1) & 1;
            const int key = ti * kAggKT + 32 * wave + li;
            half_t earlier = (half_t)0.f;
            if (ACC) earlier = out[min(key, Ls - 1)];
            enter_tile(tn);

            // Head by head, the exponentials of one head's scores between the matrix instructions of the
            // next head's: a wavefront's vector and matrix work overlap within itself, which counts where
            // few wavefronts share a SIMD (512 tokens 10.1 -> 9.1 us, 1024 12.0 -> 10.7; 32768 4.56 -> 4.44
            // ms, where the clock follows the power limit).  Two heads' scores are live instead of four,
            // which makes room for the tile's eight key operands.
            float16_t acc[2];
            float16_t zero16;   // the first product of a head starts from a constant zero
#pragma unroll
            for (int v = 0; v < 16; ++v) zero16[v] = 0.f;
            x8_t kb[kKS];
#pragma unroll
            for (int ks = 0; ks < kKS; ++ks) kb[ks] = *reinterpret_cast<const x8_t*>(&bK[li * D + ((2 * ks) ^ kx) * 8]);
            float4_t ls[4];   // log-sums of the rows of the head whose exponentials are next
            float sum = 0.f;
            // accumulator v of head rb is query row 8(v/4) + 4lg + v%4, column = key li
            auto exponentials = [&](const float16_t& s, int v0, int v1) {
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    if (v >= v0 && v < v1) sum += fast_exp2(s[v] * kScaleLog2 - ls[v >> 2][v & 3]);
            };
#pragma unroll
            for (int rb = 0; rb < NH; ++rb) {
#pragma unroll
                for (int ks = 0; ks < kKS; ++ks) {
                    acc[rb & 1] = Elem<T>::mma_32x32x16(qa[rb][ks], kb[ks], ks == 0 ? zero16 : acc[rb & 1]);
                    if (rb == 0 && ks < kLoads) issue_load(ks, nbuf);
                    if (rb > 0 && ks > 0) exponentials(acc[(rb - 1) & 1], 16 * (ks - 1) / (kKS - 1), 16 * ks / (kKS - 1));
                    if (ks == kKS - 1) {
#pragma unroll
                        for (int v4 = 0; v4 < 4; ++v4)
                            ls[v4] = *reinterpret_cast<const float4_t*>(&s_lse[rb * 32 + 8 * v4 + 4 * lg]);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
#pragma unroll
            for (int j = kKS; j < kLoads; ++j) issue_load(j, nbuf);
            tile_phase<KASCADE_PRIO_AGG>(1);
            exponentials(acc[(NH - 1) & 1], 0, 16);
            sum = sum_with_other_half(sum);
            tile_phase<KASCADE_PRIO_AGG>(2);
            if (SELECT) {
                if (lg == 0 && key < ts) s_row[key] = __builtin_bit_cast(uint16_t, (half_t)(ACC ? sum + (float)earlier : sum));
            } else if (lg == 0 && key < Ls) {
                if (key < ts)
                    out[key] = (half_t)(ACC ? sum + (float)earlier : sum);
                else if (p.fill_invalid)
                    out[key] = neg_inf;
            }
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no load may land in LDS after the workgroup has left
    }
    if constexpr (SELECT) {
        Histograms& lds = *reinterpret_cast<Histograms*>(s_tiles);
        const long long row = ((long long)b * kvh + g) * p.T + t;
        const int pr = (int)(row % sel.period);
        const int len = min(sel.valid_len[pr], ts);
        const int count = max(0, min(sel.n_sel[pr], sel.k));
        const RowsOut ro{sel.rows.out_rows, sel.rows.block_table, sel.rows.max_pages, sel.rows.page_shift, sel.rows.rows_per_seq};
        if (len <= count || count == 0) {   // uniform
            list_head<kThreads>(count, sel.k, sel.fill, sel.out_idx, row, ro);
            return;
        }
        __syncthreads();   // the row is complete, the tiles are done with
        lds.clear();
        const int nch = (len + kThreads * 8 - 1) / (kThreads * 8);   // <= MAXC (host)
        const int first = wave * nch * 512 + lane * 8;
        const uint32_t one = pk_hidden(0x00010001u);
        uint4_t data[MAXC];
        static_for<0, MAXC>([&](auto c_c) {   // order keys, at least 1; 0 past the row's end
            constexpr int c = decltype(c_c)::value;
            data[c] = uint4_t{0, 0, 0, 0};
            const int j0 = first + c * 512;
            if (c < nch && j0 < len) {
                const uint4_t raw = *reinterpret_cast<const uint4_t*>(&s_row[j0]);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    uint32_t key = pk_max_u16(raw[j] ^ (pk_sign_mask_i16(raw[j]) | 0x80008000u), one);
                    if (j0 + 2 * j + 1 >= len) key = j0 + 2 * j < len ? key & 0xFFFFu : 0u;
                    data[c][j] = key;
                }
            }
        });
        __syncthreads();   // cleared histograms
        select_row<kThreads, MAXC, false>(lds, data, nch, 0, len, count, sel.k, sel.fill, sel.out_idx, row, ro);
    } else if (p.fill_invalid) {
        const int end = part == p.key_parts - 1 ? Ls : min(Ls, (ti0 + p.part_tiles) * kAggKT);
        for (int key = max(ntiles, ti0) * kAggKT + tid; key < end; key += kThreads) out[key] = neg_inf;
    }
}

template <bool PAGED, int D, typename T, int NH, bool ACC>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2)))
void prefill_aggregate_kernel(PrefillParams p) {
    prefill_pool_body<PAGED, D, T, NH, ACC, 4, 0>(p, SelectParams{});
}

// Pooling and selection of a query tile in one workgroup: the pooled row, rounded to fp16 as it would be in memory, goes from the
// products to the selection through LDS (8 KB beside the tiles, whose place the histograms take afterwards), and one
// workgroup's selection runs under the products of the other one on its compute unit.  See prefill_pool_selects.
template <bool PAGED, int D, typename T, int NH, bool ACC, int WAVES, int MAXC>
__global__ __launch_bounds__(WAVES * 64) __attribute__((amdgpu_waves_per_eu(2)))
void prefill_pool_select_kernel(PrefillParams p, SelectParams sel) {
    prefill_pool_body<PAGED, D, T, NH, ACC, WAVES, MAXC>(p, sel);
}

}  // namespace

namespace {

// Sparse units (a query tile and four head slots) up to which they are cut in two, one block of 16 queries to a wavefront:
// where the halves are resident at once, two on each of 256 compute units.  A unit alone on its compute unit is a
// chain of a wavefront's own instructions; half of them, and a barrier a tile for the common references, take, us whole / in
// halves: 32/8 heads, 300 tokens 8.4/6.6, 517 8.6/7.5, 1024 (256 units) 10.3/10.0, 28/4 517 8.7/7.3, 8/2 heads of 64, 2048 8.7/6.7,
// 4096 13.1/12.3.  With more the rows that both halves stage cost more than that: 32/8, 1300 tokens (328 units) 12.4/13.7,
// 2048 14.1/16.9 (without the barrier).
constexpr long long kSplitUnits = 256;

template <int D, typename T>
hipError_t launch_attn_t(PrefillParams p, bool reuse, bool with_v, int nqb, hipStream_t stream) {
    const int qt = 32 * nqb;
    const bool paged = p.block_table != nullptr;
    const int nqt = (p.Lq + qt - 1) / qt;
    const bool split = reuse && !p.log_sum && (long long)nqt * p.G * head_slots(p.gs).subs * p.B <= kSplitUnits;
    const HeadSlots hs = head_slots(p.gs, split ? 2 : 4);
    const int gv = p.G * hs.subs;   // (KV head, sub-group of four or two query heads) pairs
    p.sub_recip = hs.subs > 1 ? 0xffffffffu / (unsigned)hs.subs + 1u : 0u;
    // resident per compute unit: two with V (64 KB of LDS, 256 registers), four with K only (32 KB, 128 registers)
    UnitGrid units;
    if (!unit_grid(p.B, gv, nqt, reuse || with_v || nqb == 2 ? 2 : 4, units)) return hipErrorInvalidConfiguration;
    const dim3 grid = units.grid, block(kThreads);
    p.pair_recip = units.recip;
    p.pairs_fill_xcds = units.pairs_fill_xcds;
    p.all_resident = units.all_resident;
    auto launch = [&](auto paged_c, auto spare_c) -> hipError_t {
        constexpr bool kPaged = decltype(paged_c)::value, kSpare = decltype(spare_c)::value;
        if (nqb == 2) {   // K-only log-sum pass, D = 128 (at 64 the state of 64 queries spills)
            if constexpr (D == 128) hipLaunchKernelGGL((prefill_attn_kernel_q64<kPaged, D, T, kSpare>), grid, block, 0, stream, p);
            else return hipErrorInvalidValue;
        } else if (reuse && p.log_sum) {   // a reuse pass that also reports its log-sums: fp32 sums
            hipLaunchKernelGGL((prefill_attn_kernel_q32<true, true, kPaged, D, T, kSpare, true>), grid, block, 0, stream, p);
        } else if (split) {
            hipLaunchKernelGGL((prefill_sparse_halves_kernel<kPaged, D, T, kSpare>), grid, block, 0, stream, p);
        } else if (reuse) {
            hipLaunchKernelGGL((prefill_attn_kernel_q32<true, true, kPaged, D, T, kSpare>), grid, block, 0, stream, p);
        } else if (with_v) {
            hipLaunchKernelGGL((prefill_attn_kernel_q32<false, true, kPaged, D, T, kSpare>), grid, block, 0, stream, p);
        } else {
            hipLaunchKernelGGL((prefill_attn_kernel_q32<false, false, kPaged, D, T, kSpare>), grid, block, 0, stream, p);
        }
        return hipSuccess;
    };
    const bool spare = hs.gs % (split ? 2 : 4) != 0;
    const hipError_t e = paged ? (spare ? launch(std::true_type{}, std::true_type{}) : launch(std::true_type{}, std::false_type{}))
                               : (spare ? launch(std::false_type{}, std::true_type{}) : launch(std::false_type{}, std::false_type{}));
    if (e != hipSuccess) return e;
    return hipGetLastError();
}

template <int D, typename T>
hipError_t launch_aggregate_t(PrefillParams p, const SelectParams* sel, hipStream_t stream) {
    UnitGrid units;
    if (!unit_grid(p.B, p.G, (long long)p.T * p.key_parts, 2, units)) return hipErrorInvalidConfiguration;
    const dim3 grid = units.grid, block(kThreads);
    p.pair_recip = units.recip;
    p.pairs_fill_xcds = units.pairs_fill_xcds;
    p.all_resident = units.all_resident;
    auto launch_as = [&](auto heads, auto later) {
        constexpr int kHeads = decltype(heads)::value;
        constexpr bool kLater = decltype(later)::value;
        auto select = [&](auto paged, auto waves, auto chunks) {
            constexpr int kWaves = decltype(waves)::value;
            hipLaunchKernelGGL((prefill_pool_select_kernel<decltype(paged)::value, D, T, kHeads, kLater, kWaves, decltype(chunks)::value>),
                               grid, dim3(kWaves * 64), 0, stream, p, *sel);
        };
        if (sel && p.pool_waves == 8)
            p.block_table ? select(std::true_type{}, std::integral_constant<int, 8>{}, std::integral_constant<int, 1>{})
                          : select(std::false_type{}, std::integral_constant<int, 8>{}, std::integral_constant<int, 1>{});
        else if (sel)
            p.block_table ? select(std::true_type{}, std::integral_constant<int, 4>{}, std::integral_constant<int, 2>{})
                          : select(std::false_type{}, std::integral_constant<int, 4>{}, std::integral_constant<int, 2>{});
        else if (p.block_table)
            hipLaunchKernelGGL((prefill_aggregate_kernel<true, D, T, kHeads, kLater>), grid, block, 0, stream, p);
        else
            hipLaunchKernelGGL((prefill_aggregate_kernel<false, D, T, kHeads, kLater>), grid, block, 0, stream, p);
    };
    auto launch = [&](auto heads) { p.vsub > 0 ? launch_as(heads, std::true_type{}) : launch_as(heads, std::false_type{}); };
    switch (head_slots(p.gs).gs - 4 * p.vsub) {   // the sub-group's query heads, at most four of them
    case 1: launch(std::integral_constant<int, 1>{}); break;
    case 2: launch(std::integral_constant<int, 2>{}); break;
    case 3: launch(std::integral_constant<int, 3>{}); break;
    default: launch(std::integral_constant<int, 4>{});
    }
    return hipGetLastError();
}

}  // namespace

// Pooling that selects: units up to which a workgroup has eight wavefronts, one workgroup on each compute unit (pooling and
// selection with four / eight: 32/8 heads, 517 tokens 11.7/11.3 us, 1024 16.5/15.3, 28/4 2048 40.4/36.2; with 328 units 19.8/21.5).
constexpr long long kWidePoolUnits = 256;

// p.head_dim in {64, 128}, p.elem in {kElemF16, kElemBF16}: checked by the callers
hipError_t launch_prefill_attn(const PrefillParams& p, bool reuse, bool with_v, int nqb,
                               hipStream_t stream) {
    if (p.head_dim == 128)
        return p.elem == kElemBF16 ? launch_attn_t<128, bf16_t>(p, reuse, with_v, nqb, stream)
                                   : launch_attn_t<128, half_t>(p, reuse, with_v, nqb, stream);
    return p.elem == kElemBF16 ? launch_attn_t<64, bf16_t>(p, reuse, with_v, nqb, stream)
                               : launch_attn_t<64, half_t>(p, reuse, with_v, nqb, stream);
}

// Pooling that selects saves a launch, its first trip to memory and the pooled scores' way there and back (pooling and
// selection, 32/8 heads: 517 tokens 15.3 -> 11.3 us, 2048 32.7 -> 27.9, 3001 56.1 -> 52.6, 4096 90.3 -> 88.3; three prompts of
// 2048 82.6 -> 76.3), but a tile's keys are not cut into parts then, which small calls need: where workgroups of eight
// wavefronts do not make up for it they keep two launches.  Us with two launches / as the rule would have it:
//   units up to 192, more than 6 tiles of 128 keys: 512 queries at 512 15.8/17.1, at 3584 32.2/38.5, 8/2 heads of 64, 2048 tokens
//   13.8/15.9 (6 tiles: 32/8, 768 tokens 14.0/13.2);  193 to 256: 28/4, 2048 tokens 40.8/36.2, 1024 queries at 3072 47.8/43.7, but
//   at head_dim 64, where products take half the time, 8/2 heads, 4096 tokens 24.6/26.2.
// Up to 512 units all are resident at once, where short and long ones only meet on a compute unit if the (KV head, sequence)
// pairs fill the XCDs (unit_of_workgroup):
//   257 to 448, pairs that do: 32/8, 1100 tokens 19.3/17.9, 1536 24.9/22.1, 1780 31.0/24.8, two prompts of 1600 at 28/4 42.0/40.1;
//   others: two of 1300 at 28/4 34.1/31.3, five of 1300 at 8/2 heads of 64 21.1/18.9 (10 tiles), but 20/5, 2040 tokens 27.5/33.7,
//   two of 2400 at 8/2 heads of 64 21.2/27.1, 28/4, 3001 68.4/69.8;
//   449 to 512, pairs that do: 2048 queries at 2048 74.0/66.3; others: two of 2450 at 12/3 heads of 64 30.0/29.2 (19 tiles), but 8/2
//   heads of 64, two of 3620 35.5/38.8, two of 4000 38.5/44.4, 28/4, 3800 85.9/87.9.
// Beyond, two launches do not cut keys either: two of 2800 at 12/3 heads of 64 (528 units) 39.1/35.5, 3001 tokens 55.8/52.5.
bool prefill_pool_selects(const PrefillParams& p) {
    const int keys = p.q_start + kTile * (p.T - 1), tiles = (keys + 127) / 128;
    const long long pairs = (long long)p.B * p.G, units = pairs * p.T;
    const bool fill_xcds = pairs % 8 == 0;
    if (keys > kPoolSelectKeys) return false;
    if (units > 512) return true;
    if (units > 448) return fill_xcds || tiles <= 20;
    if (units > 256) return tiles <= (fill_xcds ? 16 : 10);
    return tiles <= (units <= 192 ? 6 : p.head_dim == 64 ? 8 : 32);
}

hipError_t launch_prefill_aggregate(const PrefillParams& p0, const SelectParams* select, hipStream_t stream) {
    // one launch per sub-group of four query heads; the launches after the first add to the
    // pooled scores (launches on a stream run in order)
    PrefillParams p = p0;
    const int subs = head_slots(p.gs).subs;
    // A key's pooled score needs no other key, so a query tile's keys can be cut into parts for
    // workgroups of their own.  They are where the tiles' workgroups are all resident at once (two on
    // each of 256 compute units): then the longest is the time, and small calls leave units idle.  Parts
    // for about four workgroups per unit, of at least four key tiles: a workgroup's start (Q through
    // LDS, first rows) costs as much as two or three.  32/8 heads: 1024 tokens 16.2 -> 11.9 us,
    // 2048 28.9 -> 26.0, chunks at position 12288 of 512 queries 159 -> 70, of 1024 168 -> 127, of 2048
    // 250 -> 251; with 752 units (3001 tokens) two parts 48.6 -> 50.2.
    constexpr int kKT = 128;   // keys per tile
    const long long units = (long long)p.B * p.G * p.T;
    const int max_tiles = std::max(1, (p.q_start + kTile * (p.T - 1) + kKT - 1) / kKT);
    const int want = units <= 512 ? (int)((1024 + units - 1) / units) : 1;
    p.part_tiles = std::max((max_tiles + want - 1) / want, std::min(4, max_tiles));
    p.key_parts = (max_tiles + p.part_tiles - 1) / p.part_tiles;
    for (int v = 0; v < subs; ++v) {
        p.vsub = v;
        const SelectParams* sel = v == subs - 1 ? select : nullptr;
        if (sel) {
            p.key_parts = 1;
            p.pool_waves = units <= kWidePoolUnits ? 8 : 4;
            p.part_tiles = max_tiles;
        }
        hipError_t e;
        if (p.head_dim == 128)
            e = p.elem == kElemBF16 ? launch_aggregate_t<128, bf16_t>(p, sel, stream) : launch_aggregate_t<128, half_t>(p, sel, stream);
        else
            e = p.elem == kElemBF16 ? launch_aggregate_t<64, bf16_t>(p, sel, stream) : launch_aggregate_t<64, half_t>(p, sel, stream);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// idx[i] (token position) -> physical row of the paged cache, in place or to another buffer.
__global__ void translate_indices_kernel(const int* __restrict__ idx, int* __restrict__ out,
                                         const int* __restrict__ block_table, long long per_seq,
                                         int max_pages, int page_shift, int L) {
    const int b = blockIdx.y;
    const int* bt = block_table + (long long)b * max_pages;
    const int mask = (1 << page_shift) - 1;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < per_seq;
         i += (long long)gridDim.x * blockDim.x) {
        const int tok = max(0, min(idx[b * per_seq + i], L - 1));
        out[b * per_seq + i] = (bt[tok >> page_shift] << page_shift) + (tok & mask);
    }
}

hipError_t launch_translate_indices(const int* idx, int* out, const int* block_table, int B,
                                    long long per_seq, int max_pages, int page_shift, int L,
                                    hipStream_t stream) {
    if (per_seq <= 0 || B <= 0) return hipSuccess;
    const int blocks = (int)std::min<long long>((per_seq + 255) / 256, 4096);
    hipLaunchKernelGGL(translate_indices_kernel, dim3(blocks, B), dim3(256), 0, stream, idx, out,
                       block_table, per_seq, max_pages, page_shift, L);
    return hipGetLastError();
}

}  // namespace kascade
