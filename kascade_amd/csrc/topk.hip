// Exact per-row top-n selection over fp16 scores (radix select on the 16-bit
// order-preserving key):
//   pass 1  LDS histogram of the high 11 key bits, suffix scan -> threshold bin
//   pass 2  LDS histogram of the low 5 bits inside that bin -> exact threshold
//           key T and the number r of entries equal to T that still fit
//   pass 3  ordered compaction: entries > T and the first r entries == T, written
//           in ascending index order (deterministic, ties to the lower index)
// Rows of up to 131072 entries are held in the registers of one workgroup of 256 to 1024 threads
// (topk_select_reg_kernel; decode anchors pool into those registers, decode_pool_select_kernel).  Longer
// rows run the passes over chunks on several workgroups per row (topk_split_*), given a workspace.  What
// is left -- longer rows without one, tensors that start off a 16-byte boundary -- streams the row three
// times through one workgroup (topk_select_kernel).
#include "topk.h"
#include "topk_row.h"

#include <type_traits>

#include "decode.h"    // score codes
#include "prefill.h"   // launch_translate_indices

namespace kascade {

namespace {

constexpr int kThreads = 1024;
constexpr int kWaves = kThreads / 64;
constexpr int kChunk = kThreads * 8;
constexpr int kComputeUnits = 256;
constexpr int kBins1 = 2048;
}  // namespace
constexpr int kSplitMinLen = 65537;   // longer than a workgroup's registers hold: multi-workgroup path
constexpr int kSplitMaxRows = 4096;   // workspace is 8 KB per row for the coarse histogram
namespace {

// Loads entries [base, base+8) of a row as order keys; entries >= len get key 0xFFFFFFFF
// marker "absent" through the valid mask.
__device__ __forceinline__ int load_keys(const uint16_t* __restrict__ src, bool aligned, int base,
                                         int len, uint32_t keys[8]) {
    int nvalid = min(8, len - base);
    if (aligned && nvalid == 8) {
        uint4_t v = *reinterpret_cast<const uint4_t*>(src + base);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            keys[2 * e] = order_key((uint16_t)(v[e] & 0xFFFFu));
            keys[2 * e + 1] = order_key((uint16_t)(v[e] >> 16));
        }
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) keys[e] = (e < nvalid) ? order_key(src[base + e]) : 0u;
    }
    return nvalid;
}

// Exclusive prefix sum over the 1024 threads of the block; *total receives the block sum.
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t* s_wave, uint32_t* total) {
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const uint32_t inc = wave_incl_scan(v);
    if (lane == 63) s_wave[wave] = inc;
    __syncthreads();
    uint32_t before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        uint32_t t = s_wave[w];
        if (w < wave) before += t;
        all += t;
    }
    __syncthreads();
    *total = all;
    return before + inc - v;
}

__global__ __launch_bounds__(kThreads) void topk_select_kernel(
    const uint16_t* __restrict__ scores, int* __restrict__ out, long long row_stride,
    int uniform_len, const int* __restrict__ valid_len, const int* __restrict__ n_sel, int period,
    int k, int fill, RowsOut ro) {
    __shared__ uint32_t s_hist[kBins1];
    __shared__ uint32_t s_hist2[32];
    __shared__ uint32_t s_wave[kWaves];
    __shared__ uint32_t s_sel[4];  // b1, cum_above, T, r

    const int tid = threadIdx.x;
    const long long row = blockIdx.x;
    const int pr = (int)(row % period);
    const int len = valid_len ? min(valid_len[pr], uniform_len) : uniform_len;
    int n = n_sel ? n_sel[pr] : k;
    n = max(0, min(n, k));
    const uint16_t* src = scores + row * row_stride;
    int* dst = out + row * (long long)k;
    int* rdst = ro.rows ? ro.rows + row * (long long)k : nullptr;
    auto put = [&](int slot, int pos) {
        dst[slot] = pos;
        if (rdst) rdst[slot] = to_cache_row(ro, row, pos);
    };

    if (len <= n || n == 0) {
        for (int i = tid; i < k; i += kThreads) put(i, (i < n) ? i : fill);
        return;
    }
    const bool aligned = ((reinterpret_cast<uintptr_t>(src) & 15) == 0);

    // ---- pass 1: coarse histogram ----
    for (int i = tid; i < kBins1; i += kThreads) s_hist[i] = 0;
    if (tid < 32) s_hist2[tid] = 0;
    __syncthreads();
    for (int base = tid * 8; base < len; base += kChunk) {
        uint32_t keys[8];
        int nv = load_keys(src, aligned, base, len, keys);
#pragma unroll
        for (int e = 0; e < 8; ++e)
            if (e < nv) atomicAdd(&s_hist[keys[e] >> 5], 1u);
    }
    __syncthreads();
    {
        // thread t owns bins 2047-2t and 2046-2t (descending order)
        const int rb0 = kBins1 - 1 - 2 * tid;
        const uint32_t c0 = s_hist[rb0], c1 = s_hist[rb0 - 1];
        uint32_t total;
        const uint32_t above0 = block_excl_scan(c0 + c1, s_wave, &total);
        const uint32_t above1 = above0 + c0;
        const uint32_t un = (uint32_t)n;
        if (above0 < un && un <= above0 + c0) {
            s_sel[0] = rb0;
            s_sel[1] = above0;
        } else if (above1 < un && un <= above1 + c1) {
            s_sel[0] = rb0 - 1;
            s_sel[1] = above1;
        }
    }
    __syncthreads();
    const uint32_t b1 = s_sel[0];
    const uint32_t cum_above = s_sel[1];

    // ---- pass 2: fine histogram inside the threshold bin ----
    for (int base = tid * 8; base < len; base += kChunk) {
        uint32_t keys[8];
        int nv = load_keys(src, aligned, base, len, keys);
#pragma unroll
        for (int e = 0; e < 8; ++e)
            if (e < nv && (keys[e] >> 5) == b1) atomicAdd(&s_hist2[keys[e] & 31u], 1u);
    }
    __syncthreads();
    if (tid == 0) {
        uint32_t above = cum_above;
        int b2 = 31;
        for (; b2 > 0; --b2) {
            uint32_t c = s_hist2[b2];
            if (above + c >= (uint32_t)n) break;
            above += c;
        }
        s_sel[2] = (b1 << 5) | (uint32_t)b2;
        s_sel[3] = (uint32_t)n - above;  // entries equal to T to take
    }
    __syncthreads();
    const uint32_t T = s_sel[2];
    const uint32_t r = s_sel[3];

    // ---- pass 3: ordered compaction ----
    uint32_t gt_base = 0, eq_base = 0;
    for (int cbase = 0; cbase < len; cbase += kChunk) {
        const int base = cbase + tid * 8;
        uint32_t keys[8];
        int nv = (base < len) ? load_keys(src, aligned, base, len, keys) : 0;
        uint32_t gt = 0, eq = 0;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if (e < nv) {
                gt += (keys[e] > T);
                eq += (keys[e] == T);
            }
        }
        uint32_t total;
        const uint32_t ex = block_excl_scan(gt | (eq << 16), s_wave, &total);
        uint32_t my_gt = gt_base + (ex & 0xFFFFu);
        uint32_t my_eq = eq_base + (ex >> 16);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if (e < nv) {
                if (keys[e] > T) {
                    put(my_gt + min(my_eq, r), base + e);
                    ++my_gt;
                } else if (keys[e] == T) {
                    if (my_eq < r) put(my_gt + my_eq, base + e);
                    ++my_eq;
                }
            }
        }
        gt_base += total & 0xFFFFu;
        eq_base += total >> 16;
    }
    for (int i = n + tid; i < k; i += kThreads) put(i, fill);
}


// The tensor must start 16-byte aligned (its rows need not) and a row, with the up to 7 slots
// between the boundary before it and its start, must fit THREADS * 8 * MAXC slots.
template <int THREADS, int MAXC>
__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(4)))
void topk_select_reg_kernel(
    const uint16_t* __restrict__ scores, int* __restrict__ out, long long row_stride,
    int uniform_len, const int* __restrict__ valid_len, const int* __restrict__ n_sel, int period,
    int k, int fill, RowsOut ro) {
    const uint32_t kOne = pk_hidden(0x00010001u);
    const long long row = blockIdx.x;
    const int pr = (int)(blockIdx.x % (uint32_t)period);
    const int len = valid_len ? min(valid_len[pr], uniform_len) : uniform_len;
    int n = n_sel ? n_sel[pr] : k;
    n = max(0, min(n, k));
    if (len <= n || n == 0) {
        list_head<THREADS>(n, k, fill, out, row, ro);
        return;
    }
    // A row that does not start on a 16-byte boundary (a row stride that is no multiple of 8) is
    // read from the boundary before it: `lead` slots in front of the row count as absent, like
    // the slots past its end, and every position below is taken in these shifted coordinates
    // (the tensor itself starts on a boundary, so the slots in front belong to the row before).
    const uint16_t* row_src = scores + row * row_stride;
    const int lead = (int)((reinterpret_cast<uintptr_t>(row_src) & 15) >> 1);
    const uint16_t* src = row_src - lead;
    const int slots = len + lead;   // the row in shifted coordinates: [lead, slots)
    const int nch = (slots + THREADS * 8 - 1) / (THREADS * 8);   // <= MAXC (host)
    const int first = (threadIdx.x >> 6) * nch * 512 + (threadIdx.x & 63) * 8;   // slot of this thread's chunk 0

    // Every thread loads 16 bytes per chunk without a branch around the load, so that the loads
    // are in flight together: where the chunk's share is not wholly inside the row the address is
    // pulled back inside it and the data replaced below.
    uint4_t data[MAXC];
    const int last_full = max(slots - 8, 0) & ~7;
    static_for<0, MAXC>([&](auto c_c) {
        constexpr int c = decltype(c_c)::value;
        data[c] = uint4_t{0, 0, 0, 0};
        if (c < nch && slots >= 8)   // uniform
            data[c] = *reinterpret_cast<const uint4_t*>(src + min(first + c * 512, last_full));
    });
    __shared__ __attribute__((aligned(16))) SelectLds<THREADS, false> s_sel_lds;
    s_sel_lds.clear();
    // the pieces at the row's two ends, one thread each, entry by entry (0: no entry)
    const int tail = slots & ~7;    // first slot of the partial piece at the end
    auto piece = [&](int s0) {
        unsigned long long w[2] = {0, 0};
#pragma clang loop unroll(disable)
        for (int e = 0; e < 8; ++e) {
            const int s = s0 + e;
            const unsigned long long key = (s >= lead && s < slots) ? max(order_key(src[s]), 1u) : 0u;
            if (e < 4) w[0] |= key << (16 * e); else w[1] |= key << (16 * (e - 4));
        }
        return uint4_t{(uint32_t)w[0], (uint32_t)(w[0] >> 32), (uint32_t)w[1], (uint32_t)(w[1] >> 32)};
    };
    const bool at_front = first == 0 && (lead > 0 || tail == 0);
    const int d_tail = tail - first;   // chunk d_tail / 512 of this thread is the partial one, if it is a whole chunk away
    const bool at_tail = tail < slots && d_tail >= 0 && (d_tail & 511) == 0 && d_tail < nch * 512 && !(at_front && tail == 0);
    uint4_t end_w[2] = {};
    if (at_front) end_w[0] = piece(0);
    if (at_tail) end_w[1] = piece(tail);
    static_for<0, MAXC>([&](auto c_c) {
        constexpr int c = decltype(c_c)::value;
        if (c < nch) {
            const int s0 = first + c * 512;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                // order_key on both halves at once: negative values flip every bit, others the sign
                // bit; then at least 1
                const uint32_t raw = data[c][j];
                uint32_t key = pk_max_u16(raw ^ (pk_sign_mask_i16(raw) | 0x80008000u), kOne);
                key = s0 < tail ? key : (at_tail && s0 == tail) ? end_w[1][j] : 0u;
                if (c == 0) key = at_front ? end_w[0][j] : key;
                asm volatile("" : "+v"(key));   // chosen here: sunk below the later chunks' branches, both sides of the choices would stay live
                data[c][j] = key;
            }
        }
    });
    __syncthreads();   // cleared histograms
    select_row<THREADS, MAXC, false>(s_sel_lds, data, nch, lead, len, n, k, fill, out, row, ro);
}

// Decode anchors: pooling and selection of a (sequence, KV head) row in one workgroup.  What the
// scores pass left -- per query head a row of 16-bit score codes with one fp32 reference per 64 tokens
// (decode.h), and the log-sums of its splits -- becomes the row of pooled probabilities
// sum_h exp2(score - lse_h), rounded to fp16 as decode_aggregate_kernel rounds it, and goes straight
// into the selection's registers: no pooled row in memory, one launch instead of two (merge of the
// log-sums included).  Masked tokens need no test of their own (one per code costs a quarter of the
// pooling, 1.1 us at 16384 tokens of 4 heads, 3.3 of 8) unless a log-sum leaves the range the codes are
// made for: a row with nothing but masked tokens, or scores so large that their sum came out as nothing.
// See kScoreNone in decode.h.  Bound by the latency of one workgroup: its exponentials (8 per head and
// lane and chunk) and the selection's scans; kascade_pool_select_row has the line up to which the saved
// launch pays for the few compute units it uses, with both sides measured.
template <int THREADS, int MAXC>
__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(THREADS > 512 ? 4 : THREADS > 256 ? 2 : 1, 4)))
void decode_pool_select_kernel(DecodePoolParams p, int k, int fill, int* __restrict__ out, RowsOut ro) {
    constexpr int kMaxGroup = 16;
    __shared__ float s_lse[kMaxGroup];
    __shared__ __attribute__((aligned(16))) SelectLds<THREADS, true> s_sel_lds;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int row = blockIdx.x, b = row / p.groups;
    // The first parts of the log-sums are requested together with the length, the first scores before those parts have
    // arrived: one trip to memory less each, and the histograms are cleared meanwhile.
    float first_part = -INFINITY;
    if (p.glse && wave < p.group_size && lane < p.num_split)
        first_part = p.glse[((long long)row * p.group_size + wave) * p.num_split + lane];
    const int raw = p.seqlens ? p.seqlens[b] : p.uniform_len;
    const float* base = p.scores + (long long)row * p.group_size * p.scores_stride;   // heads of a KV head are adjacent
    const int len = max(0, min(raw, p.len_cap));           // tokens whose scores were written
    int row_len = min(raw, p.uniform_len), n = k;
    if (p.topk_percent > 0.f) {
        const long long fl = (long long)floor((double)p.topk_percent * (double)raw / 100.0);
        n = (int)min((long long)k, (fl + 127) / 128 * 128);
    } else {
        row_len = p.uniform_len;                           // every row the same: positions past a sequence pool to 0
    }
    n = max(0, n);
    // the heads' log-sums: merged from the splits' parts by a wavefront per head, or ready
    auto merge_log_sums = [&]() {
        for (int h = wave; h < p.group_size; h += THREADS / 64) {
            const long long head = (long long)row * p.group_size + h;
            if (p.glse) {
                const float* gl = p.glse + head * p.num_split;
                const float g0 = h == wave ? first_part : lane < p.num_split ? gl[lane] : -INFINITY;
                float mx = g0;
                for (int s = lane + 64; s < p.num_split; s += 64) mx = fmaxf(mx, gl[s]);
                mx = wave_max(mx);
                const float mref = (mx == -INFINITY) ? 0.f : mx;
                float sum = fast_exp2(g0 - mref);
                for (int s = lane + 64; s < p.num_split; s += 64) sum += fast_exp2(gl[s] - mref);
                sum = wave_sum(sum);
                const float v = (sum > 0.f) ? fast_log2(sum) + mref : -INFINITY;
                if (lane == 0) {
                    s_lse[h] = v;
                    p.row_sums[head] = v;
                }
            } else if (lane == 0) {
                s_lse[h] = p.row_sums[head];
            }
        }
    };
    if (row_len <= n || n == 0) {
        if (p.glse) merge_log_sums();
        list_head<THREADS>(n, k, fill, out, row, ro);
        return;
    }
    // Scores four heads at a time (a batch), two batches ahead on their way.
    const int nch = (row_len + THREADS * 8 - 1) / (THREADS * 8);   // <= MAXC (host)
    const int first = wave * nch * 512 + lane * 8;
    const int last_piece = max(0, len - 1) & ~7;
    struct Batch {
        uint4_t q[4];
        float ref[4];
    };
    const int nb = (p.group_size + 3) / 4;                 // batches per chunk
    auto load_batch = [&](int i, Batch& bt) {              // batch i: heads 4 (i % nb) .. +3 of chunk i / nb
        const int c = min(i / nb, nch - 1), h0 = 4 * (i - i / nb * nb);
        const int jc = min(first + c * 512, last_piece);   // past the tokens: entries that exist, dropped below
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const float* hr = base + (long long)min(h0 + u, p.group_size - 1) * p.scores_stride;
            bt.q[u] = *reinterpret_cast<const uint4_t*>(reinterpret_cast<const uint16_t*>(hr) + jc);
            bt.ref[u] = hr[p.scores_stride / 2 + (jc >> 6)];
        }
    };
    // packed order keys of a piece: no entry is negative, so the key is the value with the top bit set
    auto keys_of = [&](const float (&sum)[8], int j0) {
        uint4_t d;
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
            const half2_t x = {(half_t)sum[e], (half_t)sum[e + 1]};
            d[e >> 1] = __builtin_bit_cast(uint32_t, x) | 0x80008000u;
        }
        if (j0 + 8 > len) {   // the piece at the tokens' end and those behind it: probability 0, or no entry
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int sh = 16 * (e & 1);
                const uint32_t key = j0 + e < len ? (d[e >> 1] >> sh) & 0xFFFFu : j0 + e < row_len ? 0x8000u : 0u;
                d[e >> 1] = (d[e >> 1] & (0xFFFF0000u >> sh)) | (key << sh);
            }
        }
        return d;
    };
    uint4_t data[MAXC];
    Batch cur, n1, n2;
    load_batch(0, n1);
    load_batch(1, n2);
    s_sel_lds.clear();
    merge_log_sums();
    __syncthreads();   // s_lse, cleared histograms
    static_for<0, MAXC>([&](auto c_c) {
        constexpr int c = decltype(c_c)::value;
        data[c] = uint4_t{0, 0, 0, 0};
        const int j0 = first + c * 512;
        if (c < nch && wave * nch * 512 + c * 512 < row_len) {     // uniform over the wavefront
            float sum[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) sum[e] = 0.f;
#pragma clang loop unroll(disable)
            for (int hb = 0; hb < nb; ++hb) {
                cur = n1;
                n1 = n2;
                load_batch(c * nb + hb + 2, n2);
                __builtin_amdgcn_sched_barrier(0);
                const int h0 = 4 * hb;
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    // a slot past the last head adds exp2(-inf) = 0
                    const float ref = h0 + u < p.group_size ? cur.ref[u] - s_lse[h0 + u] : -INFINITY;
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const uint32_t q = (e & 1) ? cur.q[u][e >> 1] >> 16 : cur.q[u][e >> 1] & 0xFFFFu;
                        sum[e] += fast_exp2(__builtin_fmaf((float)q, -1.f / kScoreSteps, ref));
                    }
                }
            }
            data[c] = keys_of(sum, j0);
        }
    });
    // A log-sum outside the range the codes are made for: the same sums again, every code tested for the mark.
    // (Up to kSane a reference lies less than one step above its log-sum, whatever their rounding.)
    constexpr float kSane = 1048576.f;
    const bool odd = lane < p.group_size && !(fabsf(s_lse[min(lane, kMaxGroup - 1)]) < kSane);
    if (__ballot(odd) != 0) {   // the same in every wavefront
        static_for<0, MAXC>([&](auto c_c) {
            constexpr int c = decltype(c_c)::value;
            const int j0 = first + c * 512, jc = min(j0, last_piece);
            if (c < nch) {
                float sum[8] = {};
#pragma clang loop unroll(disable)
                for (int h = 0; h < p.group_size; ++h) {
                    const float* hr = base + (long long)h * p.scores_stride;
                    const uint4_t codes = *reinterpret_cast<const uint4_t*>(reinterpret_cast<const uint16_t*>(hr) + jc);
                    const float ref = hr[p.scores_stride / 2 + (jc >> 6)] - s_lse[h];
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const uint32_t q = (e & 1) ? codes[e >> 1] >> 16 : codes[e >> 1] & 0xFFFFu;
                        const float pr = fast_exp2(__builtin_fmaf((float)q, -1.f / kScoreSteps, ref));
                        sum[e] += (q == kScoreNone) ? 0.f : pr;
                    }
                }
                data[c] = keys_of(sum, j0);
            }
        });
    }
    select_row<THREADS, MAXC, true>(s_sel_lds, data, nch, 0, row_len, n, k, fill, out, row, ro);
}

// --------------------------------------------------------------------------
// Long rows: the same radix select spread over several workgroups per row.
// Every workgroup owns one chunk of kSplitChunk entries of one row and holds it in registers
// (kSplitU 16-byte loads per thread, all in flight at once); per-row state lives in a
// caller-provided workspace:
//   hist1  [rows][2048]           coarse histogram (atomically merged)
//   arrive [rows][2]              workgroups of the row that have finished pass 1 / pass 2
//   sel    [rows][8]              {mode, b1, cum_above, T, r, n, len}
//   cinfo  [rows][chunks][34]     per chunk: fine histogram of bin b1 (32) and the
//                                 number of entries in bins above b1
//   coff   [rows][chunks][2]      per chunk: selected-greater / equal counts before it
// Launch sequence: zero -> hist1 -> [scan1] -> hist2 -> [scan2] -> write.  With few workgroups
// (a handful of very long rows: decode) the scan over a row's merged histogram is done by the
// row's last workgroup to finish its pass (FUSED: an arrival counter per row), which saves the
// two small launches; what one workgroup leaves for another of the same launch goes through
// device-coherent atomics, stores and loads.  With thousands of rows (prefill) the counter's
// round trip at the end of every workgroup costs more than the launches, so the scans stay
// kernels of their own.
// Bound by dependent trips to memory and the counters' turns in LDS, not by bytes.  32 rows of 131072 to 524288 entries:
// coarse pass 26.2 -> 19.9 us with the row's loads in front of its length and behind no branch and a bin's copies side by
// side, fine pass 21.8 -> 18.2 with the same loads and four copies.  Its scan with a lane per bin, instead of every bin's
// sum over 64 lanes, spills nothing (12 bytes of scratch before): the whole selection 53.7 -> 51.5 us.
// --------------------------------------------------------------------------
constexpr int kSplitU = 4;
constexpr int kSplitChunk = kSplitU * kChunk;   // 32768 entries per workgroup
constexpr int kSelWords = 8;
constexpr int kInfoWords = 34;
constexpr int kHistCopies = 4;
constexpr long long kSplitFusedMax = 2048;   // workgroups up to which the scans are fused into the passes

struct SplitWs {
    uint32_t* hist1;
    uint32_t* arrive;
    uint32_t* sel;
    uint32_t* cinfo;
    uint32_t* coff;
};

__device__ __forceinline__ uint32_t load_device_u32(const uint32_t* p) {
    return __hip_atomic_load(const_cast<uint32_t*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void store_device_u32(uint32_t* p, uint32_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void row_params(const int* valid_len, const int* n_sel, int period,
                                           int uniform_len, int k, long long row, int& len, int& n) {
    const int pr = (int)(row % period);
    len = valid_len ? min(valid_len[pr], uniform_len) : uniform_len;
    n = n_sel ? n_sel[pr] : k;
    n = max(0, min(n, k));
}

// The chunk [c0, c1) of a row as order keys: thread t holds entries c0 + u*8192 + 8t .. +8 for
// u = 0..kSplitU-1 (every load instruction covers consecutive 16-byte pieces).  Where no piece crosses the chunk's end the
// loads stand behind no branch (pieces past the end take the last one again): under a branch each waited for the one before.
__device__ __forceinline__ void load_chunk(const uint16_t* __restrict__ src, bool aligned, int c0, int c1,
                                           uint32_t (&keys)[kSplitU][8], int (&nv)[kSplitU]) {
    const int first = c0 + (int)threadIdx.x * 8;
    if (aligned && c1 >= 8 && (c1 & 7) == 0) {   // uniform (a chunk behind the row's end has c1 < c0: nothing is taken)
        uint4_t v[kSplitU];
#pragma unroll
        for (int u = 0; u < kSplitU; ++u) {
            v[u] = ld_global_16(src + min(first + u * kChunk, c1 - 8));
            nv[u] = first + u * kChunk < c1 ? 8 : 0;
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < kSplitU; ++u)
#pragma unroll
            for (int e = 0; e < 8; ++e) keys[u][e] = order_key((uint16_t)(v[u][e >> 1] >> (16 * (e & 1))));
        return;
    }
#pragma unroll
    for (int u = 0; u < kSplitU; ++u) {
        const int base = first + u * kChunk;
        nv[u] = 0;
        if (base < c1) nv[u] = load_keys(src, aligned, base, c1, keys[u]);
    }
}

// True in every thread of the row's last workgroup to get here (all of the row's `expected`
// workgroups call it once per pass).  The caller's device-coherent stores and atomics are
// waited for before the workgroup counts itself in.
__device__ __forceinline__ bool last_of_row(uint32_t* counter, int expected, int* s_flag) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t arrived = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *s_flag = (arrived == (uint32_t)(expected - 1));
    }
    __syncthreads();
    return *s_flag != 0;
}

__global__ __launch_bounds__(256) void topk_zero_kernel(uint32_t* p, long long n) {
    long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = 0;
}

// The bin that holds the n-th largest entry of a row whose coarse histogram is complete (all
// 1024 threads of a workgroup).
__device__ __forceinline__ void split_scan1(const uint32_t* gh, uint32_t* sel, int n, int len, uint32_t* s_wave) {
    const int tid = threadIdx.x;
    const int rb0 = kBins1 - 1 - 2 * tid;   // this thread's bins, in descending order
    const uint32_t h0 = load_device_u32(gh + rb0), h1 = load_device_u32(gh + rb0 - 1);
    uint32_t total;
    const uint32_t above0 = block_excl_scan(h0 + h1, s_wave, &total);
    const uint32_t above1 = above0 + h0;
    const uint32_t un = (uint32_t)n;
    if (above0 < un && un <= above0 + h0) {
        sel[1] = rb0; sel[2] = above0;
    } else if (above1 < un && un <= above1 + h1) {
        sel[1] = rb0 - 1; sel[2] = above1;
    }
    if (tid == 0) { sel[0] = 1; sel[5] = (uint32_t)n; sel[6] = (uint32_t)len; }
}

template <bool FUSED>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(8))) void topk_split_hist1_kernel(
    const uint16_t* __restrict__ scores, long long row_stride, int uniform_len,
    const int* __restrict__ valid_len, const int* __restrict__ n_sel, int period, int k, SplitWs ws) {
    // a bin's copies lie side by side: in one bank each, lanes that count in the same bin took turns whatever their copy
    __shared__ __attribute__((aligned(16))) uint32_t s_hist[kBins1][kHistCopies];
    __shared__ uint32_t s_wave[kWaves];
    __shared__ int s_flag;
    static_assert(kHistCopies == 4, "a bin is 16 bytes");
    const int tid = threadIdx.x;
    const long long row = blockIdx.y;
    const int c0 = blockIdx.x * kSplitChunk;
    if (c0 >= uniform_len) return;
    const uint16_t* src = scores + row * row_stride;
    const bool aligned = ((reinterpret_cast<uintptr_t>(src) & 15) == 0);
    uint32_t* sel = ws.sel + row * kSelWords;
    int len, n, c_end = min(uniform_len, c0 + kSplitChunk);
    // Few workgroups (FUSED): the chunk is requested for the row's full width before its length has arrived, cut down
    // below.  Thousands of rows are bound by their bytes: only what a row holds, in whole pieces (tiles of a 196608-token
    // prompt, the first 512: 124 -> 107 us a selection, 2048 over its whole length 597 -> 540).
    if (!FUSED) {
        row_params(valid_len, n_sel, period, uniform_len, k, row, len, n);
        if (len <= n || n == 0 || c0 >= len) return;   // nothing to select: the write pass lists the row's head
        c_end = min(c_end, (len + 7) & ~7);
    }
    uint32_t keys[kSplitU][8];
    int nv[kSplitU];
    load_chunk(src, aligned, c0, c_end, keys, nv);
    if (FUSED) {
        row_params(valid_len, n_sel, period, uniform_len, k, row, len, n);
        if (len <= n || n == 0) {
            if (blockIdx.x == 0 && tid == 0) { sel[0] = 0; sel[5] = (uint32_t)n; sel[6] = (uint32_t)len; }
            return;
        }
        if (c0 >= len) return;
    }
    const int c1 = min(len, c0 + kSplitChunk);
#pragma unroll
    for (int u = 0; u < kSplitU; ++u) nv[u] = max(0, min(nv[u], len - (c0 + u * kChunk + tid * 8)));
    for (int i = tid; i < kBins1; i += kThreads) *reinterpret_cast<uint4_t*>(s_hist[i]) = uint4_t{0, 0, 0, 0};
    __syncthreads();
    // +0 (pooled probabilities underflow to it by the thousand) is not counted: its number is
    // the chunk's length minus the sum of the others.  The other entries go to one of four
    // copies of the histogram, chosen by the lane, which spreads the crowded bins.
    uint32_t* mine = &s_hist[0][tid & (kHistCopies - 1)];
    uint32_t counted = 0;
#pragma unroll
    for (int u = 0; u < kSplitU; ++u)
#pragma unroll
        for (int e = 0; e < 8; ++e)
            if (e < nv[u] && keys[u][e] != 0x8000u) {
                atomicAdd(&mine[(keys[u][e] >> 5) * kHistCopies], 1u);
                ++counted;
            }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) counted += __shfl_xor(counted, o);
    if ((tid & 63) == 0) s_wave[tid >> 6] = counted;
    __syncthreads();
    uint32_t* gh = ws.hist1 + row * kBins1;
    for (int i = tid; i < kBins1; i += kThreads) {
        const uint4_t h = *reinterpret_cast<const uint4_t*>(s_hist[i]);
        uint32_t c = h[0] + h[1] + h[2] + h[3];
        if (i == (int)(0x8000u >> 5)) {
            uint32_t all = 0;
#pragma unroll
            for (int w = 0; w < kWaves; ++w) all += s_wave[w];
            c += (uint32_t)(c1 - c0) - all;
        }
        if (c) atomicAdd(&gh[i], c);
    }
    if (!FUSED) return;
    const int nchunks = (len + kSplitChunk - 1) / kSplitChunk;
    if (!last_of_row(ws.arrive + 2 * row, nchunks, &s_flag)) return;
    split_scan1(gh, sel, n, len, s_wave);
}

__global__ __launch_bounds__(kThreads) void topk_split_scan1_kernel(
    int uniform_len, const int* __restrict__ valid_len, const int* __restrict__ n_sel, int period,
    int k, SplitWs ws) {
    __shared__ uint32_t s_wave[kWaves];
    const long long row = blockIdx.x;
    int len, n;
    row_params(valid_len, n_sel, period, uniform_len, k, row, len, n);
    uint32_t* sel = ws.sel + row * kSelWords;
    if (len <= n || n == 0) {
        if (threadIdx.x == 0) { sel[0] = 0; sel[5] = (uint32_t)n; sel[6] = (uint32_t)len; }
        return;
    }
    split_scan1(ws.hist1 + row * kBins1, sel, n, len, s_wave);
}

// From the chunks' fine histograms of a row: the threshold key T, the number r of entries equal
// to T that still fit, and every chunk's offsets into the output.  One wavefront: lane l sums fine bin
// 31 - l % 32 over every other chunk, then lane c takes chunk c (64 chunks per round).
__device__ __forceinline__ void split_scan2(uint32_t* sel, const uint32_t* rinfo, uint32_t* off, int nchunks) {
    const int lane = threadIdx.x & 63;
    const uint32_t n = sel[5], b1 = sel[1];
    const uint32_t* bin = rinfo + (31 - (lane & 31));
    uint32_t h = 0;
    for (int c0 = lane >> 5; c0 < nchunks; c0 += 16) {   // eight loads on their way (past the last chunk: that one again)
        uint32_t v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = load_device_u32(bin + min(c0 + 2 * u, nchunks - 1) * kInfoWords);
#pragma unroll
        for (int u = 0; u < 8; ++u) h += c0 + 2 * u < nchunks ? v[u] : 0u;
    }
    h += (uint32_t)__shfl_xor((int)h, 32);
    // the fine bin of the n-th largest entry, from the top (bin 0 takes whatever is left)
    const uint32_t incl = wave_incl_scan(lane < 32 ? h : 0u);
    const uint32_t base = sel[2];
    const int first = __ffsll((unsigned long long)__ballot(lane == 31 || (lane < 31 && base + incl >= n))) - 1;
    const int b2 = 31 - first;
    const uint32_t r = n - (base + (uint32_t)__builtin_amdgcn_readlane((int)(incl - h), first));
    if (lane == 0) { sel[3] = (b1 << 5) | (uint32_t)b2; sel[4] = r; }
    // per-chunk counts of entries above T and equal to T, and their exclusive prefixes
    uint32_t gt_run = 0, eq_run = 0;
    for (int cb = 0; cb < nchunks; cb += 64) {
        const int c = cb + lane;
        uint32_t gt = 0, eq = 0;
        if (c < nchunks) {
            gt = load_device_u32(rinfo + c * kInfoWords + 32);
#pragma unroll
            for (int j = 0; j < 32; ++j) {
                const uint32_t v = load_device_u32(rinfo + c * kInfoWords + j);
                gt += (j > b2) ? v : 0u;
                eq += (j == b2) ? v : 0u;
            }
        }
        const uint32_t gi = wave_incl_scan(gt), ei = wave_incl_scan(eq);
        if (c < nchunks) { off[2 * c] = gt_run + gi - gt; off[2 * c + 1] = eq_run + ei - eq; }
        gt_run += __shfl(gi, 63);
        eq_run += __shfl(ei, 63);
    }
}

// Pass 2 of a chunk: the fine histogram of the threshold bin and the count of entries above it.
// The chunk's loads are issued for the row's full width before the row's state (its length,
// the threshold bin) has arrived, and cut down to the length afterwards.
template <bool FUSED>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(8))) void topk_split_hist2_kernel(
    const uint16_t* __restrict__ scores, long long row_stride, int uniform_len, int max_chunks, SplitWs ws) {
    __shared__ __attribute__((aligned(16))) uint32_t s_hist2[32][kHistCopies];
    __shared__ uint32_t s_gt1;
    __shared__ int s_flag;
    const int tid = threadIdx.x, lane = tid & 63;
    const long long row = blockIdx.y;
    uint32_t* sel = ws.sel + row * kSelWords;
    const int c0 = blockIdx.x * kSplitChunk;
    if (c0 >= uniform_len) return;
    const uint16_t* src = scores + row * row_stride;
    const bool aligned = ((reinterpret_cast<uintptr_t>(src) & 15) == 0);
    uint32_t keys[kSplitU][8];
    int nv[kSplitU];
    load_chunk(src, aligned, c0, min(uniform_len, c0 + kSplitChunk), keys, nv);
    const int len = (int)sel[6];
    if (sel[0] == 0 || c0 >= len) return;
    const uint32_t b1 = sel[1];
#pragma unroll
    for (int u = 0; u < kSplitU; ++u) nv[u] = max(0, min(nv[u], len - (c0 + u * kChunk + tid * 8)));
    if (tid < 32) *reinterpret_cast<uint4_t*>(s_hist2[tid]) = uint4_t{0, 0, 0, 0};
    if (tid == 32) s_gt1 = 0;
    __syncthreads();
    uint32_t* mine = &s_hist2[0][tid & (kHistCopies - 1)];
    uint32_t gt1 = 0, zeros = 0;
    const bool zero_bin = b1 == (0x8000u >> 5);   // uniform: the threshold lies among +0 and the smallest subnormals
#pragma unroll
    for (int u = 0; u < kSplitU; ++u)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const bool in = e < nv[u];
            const uint32_t hb = keys[u][e] >> 5;
            if (zero_bin) {   // that many atomics on one address would serialise: a ballot per wavefront
                const bool zero = in && keys[u][e] == 0x8000u;
                zeros += (uint32_t)__popcll(__ballot(zero));
                if (in && !zero && hb == b1) atomicAdd(&mine[(keys[u][e] & 31u) * kHistCopies], 1u);
            } else if (in && hb == b1) {
                atomicAdd(&mine[(keys[u][e] & 31u) * kHistCopies], 1u);
            }
            gt1 += (in && hb > b1);
        }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) gt1 += __shfl_xor(gt1, o);
    if (lane == 0 && gt1) atomicAdd(&s_gt1, gt1);
    if (lane == 0 && zeros) atomicAdd(&s_hist2[0][0], zeros);   // +0 is entry 0 of its bin
    __syncthreads();
    uint32_t* info = ws.cinfo + (row * max_chunks + blockIdx.x) * kInfoWords;
    if (tid < 32) {
        const uint4_t h = *reinterpret_cast<const uint4_t*>(s_hist2[tid]);
        store_device_u32(info + tid, h[0] + h[1] + h[2] + h[3]);
    }
    if (tid == 32) store_device_u32(info + 32, s_gt1);
    if (!FUSED) return;
    const int nchunks = (len + kSplitChunk - 1) / kSplitChunk;
    if (!last_of_row(ws.arrive + 2 * row + 1, nchunks, &s_flag)) return;
    if (tid >= 64) return;
    split_scan2(sel, ws.cinfo + row * max_chunks * kInfoWords, ws.coff + row * max_chunks * 2, nchunks);
}

__global__ __launch_bounds__(64) void topk_split_scan2_kernel(int max_chunks, SplitWs ws) {
    const long long row = blockIdx.x;
    uint32_t* sel = ws.sel + row * kSelWords;
    if (sel[0] == 0) return;
    const int nchunks = ((int)sel[6] + kSplitChunk - 1) / kSplitChunk;
    split_scan2(sel, ws.cinfo + row * max_chunks * kInfoWords, ws.coff + row * max_chunks * 2, nchunks);
}

__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(8))) void topk_split_write_kernel(
    const uint16_t* __restrict__ scores, int* __restrict__ out, long long row_stride, int uniform_len,
    int k, int fill, int max_chunks, SplitWs ws, RowsOut ro) {
    static_assert(kSplitU * kWaves == 64, "one wavefront scans the (load, wavefront) totals");
    __shared__ uint32_t s_tot[kSplitU * kWaves];
    __shared__ uint32_t s_pre[kSplitU * kWaves];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const long long row = blockIdx.y;
    const uint32_t* sel = ws.sel + row * kSelWords;
    const int c0 = blockIdx.x * kSplitChunk;
    const uint16_t* src = scores + row * row_stride;
    const bool aligned = ((reinterpret_cast<uintptr_t>(src) & 15) == 0);
    // the chunk's loads go out before the row's state has arrived (cut down to its length below)
    uint32_t keys[kSplitU][8];
    int nv[kSplitU];
    load_chunk(src, aligned, c0, min(uniform_len, c0 + kSplitChunk), keys, nv);
    const int len = (int)sel[6];
    const int n = (int)sel[5];
    int* dst = out + row * (long long)k;
    int* rdst = ro.rows ? ro.rows + row * (long long)k : nullptr;
    auto put = [&](int slot, int pos) {
        dst[slot] = pos;
        if (rdst) rdst[slot] = to_cache_row(ro, row, pos);
    };
    if (blockIdx.x == 0) {
        if (sel[0] == 0) {
            for (int i = tid; i < k; i += kThreads) put(i, (i < n) ? i : fill);
            return;
        }
        for (int i = n + tid; i < k; i += kThreads) put(i, fill);
    }
    if (sel[0] == 0 || c0 >= len) return;
    const uint32_t T = sel[3];
    const uint32_t r = sel[4];
    const uint32_t* off = ws.coff + (row * max_chunks + blockIdx.x) * 2;
    const uint32_t gt_base = off[0], eq_base = off[1];
#pragma unroll
    for (int u = 0; u < kSplitU; ++u) nv[u] = max(0, min(nv[u], len - (c0 + u * kChunk + tid * 8)));
    // counts above / equal to T per (load, thread), packed; position order is (load, thread, entry)
    uint32_t cnt[kSplitU], inc[kSplitU];
#pragma unroll
    for (int u = 0; u < kSplitU; ++u) {
        uint32_t gt = 0, eq = 0;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if (e < nv[u]) {
                gt += (keys[u][e] > T);
                eq += (keys[u][e] == T);
            }
        }
        cnt[u] = gt | (eq << 16);
        inc[u] = wave_incl_scan(cnt[u]);
        if (lane == 63) s_tot[u * kWaves + wave] = inc[u];
    }
    __syncthreads();
    if (wave == 0) {
        const uint32_t t = s_tot[lane];
        s_pre[lane] = wave_incl_scan(t) - t;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kSplitU; ++u) {
        const uint32_t ex = s_pre[u * kWaves + wave] + inc[u] - cnt[u];
        uint32_t my_gt = gt_base + (ex & 0xFFFFu);
        uint32_t my_eq = eq_base + (ex >> 16);
        const int base = c0 + u * kChunk + tid * 8;
        // stores straight from the threads: staging the chunk's list in LDS for full-width stores
        // was measured slower (its two extra barriers cost more than the narrow stores)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if (e < nv[u]) {
                if (keys[u][e] > T) {
                    put(my_gt + min(my_eq, r), base + e);
                    ++my_gt;
                } else if (keys[u][e] == T) {
                    if (my_eq < r) put(my_gt + my_eq, base + e);
                    ++my_eq;
                }
            }
        }
    }
}

SplitWs carve_ws(void* workspace, int rows, int max_chunks) {
    SplitWs ws;
    uint32_t* p = reinterpret_cast<uint32_t*>(workspace);
    ws.hist1 = p;  p += (size_t)rows * kBins1;
    ws.arrive = p; p += (size_t)rows * 2;       // right behind hist1: one launch zeroes both
    ws.sel = p;    p += (size_t)rows * kSelWords;
    ws.cinfo = p;  p += (size_t)rows * max_chunks * kInfoWords;
    ws.coff = p;
    return ws;
}


// ---------------------------------------------------------------- rows ordered by score
// Reorders the first n entries of every row's position list by descending score, equal scores by
// ascending position: the order of torch.topk(...).indices.  A radix sort on the 16-bit order key
// in two stable passes (low byte, then high byte), one workgroup per row.  The keys are gathered
// once (the only dependent loads), then keys and positions move together between two buffers: in
// LDS for lists of up to kSortLdsEntries entries, in the caller's workspace for longer ones.  A
// wavefront owns a contiguous share of the list and walks it 64 entries at a time, the next
// step's entries already in flight; the lanes that hold the same digit find each other with
// eight ballots, so every entry's place follows from counters per (wavefront, digit) in LDS: no
// atomics, nothing depends on timing, and the input order (ascending position) survives among
// equal scores.
constexpr int kSortLdsEntries = 4096;

// lanes of the wavefront that are valid and hold the same 8-bit digit as this lane
__device__ __forceinline__ uint64_t digit_peers(uint32_t d, bool valid) {
    uint64_t peers = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        const bool bit = (d >> b) & 1u;
        const uint64_t set = __ballot(bit);
        peers &= bit ? set : ~set;
    }
    return valid ? peers : 0ull;
}

template <int WAVES, int LDS_N>
__global__ __launch_bounds__(WAVES * 64) void topk_sort_rows_kernel(
    const uint16_t* __restrict__ scores, int* __restrict__ idx, int* __restrict__ ws_pos,
    uint16_t* __restrict__ ws_keys, long long row_stride, int uniform_len,
    const int* __restrict__ valid_len, int period, int k) {
    constexpr int kT = WAVES * 64;
    static_assert(kT >= 256, "one thread per digit in the offset step");
    __shared__ uint32_t s_cnt[WAVES][256];
    __shared__ uint32_t s_wsum[4];
    __shared__ int s_pos[LDS_N > 0 ? 2 * LDS_N : 1];
    __shared__ uint16_t s_key[LDS_N > 0 ? 2 * LDS_N : 2];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const long long row = blockIdx.x;
    const int len = valid_len ? min(valid_len[(int)(row % period)], uniform_len) : uniform_len;
    const int n = max(0, min(k, len));   // entries beyond n name positions past the row's end: they stay
    if (n <= 1) return;
    const uint16_t* src = scores + row * row_stride;
    int* first = idx + row * (long long)k;
    int *pos_a, *pos_b;
    uint16_t *key_a, *key_b;
    if constexpr (LDS_N > 0) {
        pos_a = s_pos; pos_b = s_pos + LDS_N; key_a = s_key; key_b = s_key + LDS_N;
    } else {
        pos_a = first; pos_b = ws_pos + row * (long long)k;
        key_a = ws_keys + row * 2ll * k; key_b = key_a + k;
    }
    for (int i = tid; i < n; i += kT) {
        const int pos = first[i];
        if constexpr (LDS_N > 0) pos_a[i] = pos;
        key_a[i] = (uint16_t)order_key(src[pos]);
    }
    __syncthreads();

    const int seg = (n + kT - 1) / kT * 64;
    const int s0 = min(n, wave * seg), s1 = min(n, s0 + seg);
    const uint64_t below = (1ull << lane) - 1ull;
    volatile uint32_t* mine = s_cnt[wave];

    for (int pass = 0; pass < 2; ++pass) {
        const int* from_pos = pass ? pos_b : pos_a;
        const uint16_t* from_key = pass ? key_b : key_a;
        int* to_pos = pass ? first : pos_b;
        const int shift = 8 * pass;
        for (int i = tid; i < WAVES * 256; i += kT) (&s_cnt[0][0])[i] = 0;
        __syncthreads();
        // how many entries of each digit this wavefront's share holds
        {
            bool valid = s0 + lane < s1;
            uint32_t key = valid ? from_key[s0 + lane] : 0u;
            for (int base = s0; base < s1; base += 64) {
                const bool nvalid = base + 64 + lane < s1;
                const uint32_t nkey = nvalid ? from_key[base + 64 + lane] : 0u;
                const uint32_t d = (key >> shift) & 255u;
                const uint64_t peers = digit_peers(d, valid);
                if (valid && (peers & below) == 0) mine[d] += (uint32_t)__popcll(peers);
                valid = nvalid; key = nkey;
            }
        }
        __syncthreads();
        // thread t < 256 owns digit 255 - t: the entries with a larger digit come first, then the
        // earlier shares' entries of the same digit
        {
            const int d = 255 - (tid & 255);
            uint32_t c[WAVES], total = 0;
            if (tid < 256) {
#pragma unroll
                for (int w = 0; w < WAVES; ++w) { c[w] = s_cnt[w][d]; total += c[w]; }
            }
            const uint32_t inc = wave_incl_scan(total);
            if (tid < 256 && lane == 63) s_wsum[wave] = inc;
            __syncthreads();
            if (tid < 256) {
                uint32_t start = inc - total;
#pragma unroll
                for (int w = 0; w < 4; ++w) if (w < wave) start += s_wsum[w];
#pragma unroll
                for (int w = 0; w < WAVES; ++w) { s_cnt[w][d] = start; start += c[w]; }
            }
        }
        __syncthreads();
        // place: the counter of a digit is read by all its lanes, then advanced by the first of them
        {
            bool valid = s0 + lane < s1;
            int pos = valid ? from_pos[s0 + lane] : 0;
            uint32_t key = valid ? from_key[s0 + lane] : 0u;
            for (int base = s0; base < s1; base += 64) {
                const bool nvalid = base + 64 + lane < s1;
                const int npos = nvalid ? from_pos[base + 64 + lane] : 0;
                const uint32_t nkey = nvalid ? from_key[base + 64 + lane] : 0u;
                const uint32_t d = (key >> shift) & 255u;
                const uint64_t peers = digit_peers(d, valid);
                const uint32_t rank = (uint32_t)__popcll(peers & below);
                const uint32_t at = valid ? mine[d] : 0u;
                if (valid && rank == 0) mine[d] = at + (uint32_t)__popcll(peers);
                if (valid) {
                    to_pos[at + rank] = pos;
                    if (pass == 0) key_b[at + rank] = (uint16_t)key;
                }
                valid = nvalid; pos = npos; key = nkey;
            }
        }
        __syncthreads();   // the second pass reads what other wavefronts placed
    }
}

}  // namespace

int topk_max_register_row() { return 16 * kChunk; }

long long topk_split_workspace_bytes(int rows, long long row_len) {
    if (row_len < kSplitMinLen || rows > kSplitMaxRows) return 0;
    const long long chunks = (row_len + kSplitChunk - 1) / kSplitChunk;
    return 4ll * rows * (kBins1 + 2 + kSelWords + chunks * (kInfoWords + 2));
}

namespace {
RowsOut rows_out(const TopkRows* tr) {
    RowsOut ro{};
    if (tr && tr->out_rows) {
        ro.rows = tr->out_rows; ro.block_table = tr->block_table; ro.max_pages = tr->max_pages;
        ro.page_shift = tr->page_shift; ro.rows_per_seq = tr->rows_per_seq;
    }
    return ro;
}
}  // namespace

hipError_t launch_topk_split(const half_t* scores, int* out_idx, int rows, long long row_stride,
                             int max_len, int uniform_len, const int* valid_len, const int* n_sel,
                             int period, int k, int fill, void* workspace, const TopkRows* tr,
                             hipStream_t stream) {
    if (rows == 0) return hipSuccess;
    // The chunk workgroups write their selections to scattered slots, where a block-table lookup
    // per element would sit in the middle of the compaction (+40 us on four rows of 131072 to
    // 524288 entries); the long-row path translates in a launch of its own at the end instead.
    const RowsOut ro{};
    const int max_chunks = (max_len + kSplitChunk - 1) / kSplitChunk;
    SplitWs ws = carve_ws(workspace, rows, max_chunks);
    const uint16_t* src = reinterpret_cast<const uint16_t*>(scores);
    const long long nz = (long long)rows * (kBins1 + 2);   // histograms and arrival counters
    hipLaunchKernelGGL(topk_zero_kernel, dim3((unsigned)((nz + 255) / 256)), dim3(256), 0, stream,
                       ws.hist1, nz);
    dim3 grid(max_chunks, rows);
    // few workgroups: the scans ride on the histogram passes; many: launches of their own
    const bool fused = (long long)rows * max_chunks <= kSplitFusedMax;
    if (fused) {
        hipLaunchKernelGGL(topk_split_hist1_kernel<true>, grid, dim3(kThreads), 0, stream, src, row_stride,
                           uniform_len, valid_len, n_sel, period, k, ws);
        hipLaunchKernelGGL(topk_split_hist2_kernel<true>, grid, dim3(kThreads), 0, stream, src, row_stride,
                           uniform_len, max_chunks, ws);
    } else {
        hipLaunchKernelGGL(topk_split_hist1_kernel<false>, grid, dim3(kThreads), 0, stream, src, row_stride,
                           uniform_len, valid_len, n_sel, period, k, ws);
        hipLaunchKernelGGL(topk_split_scan1_kernel, dim3(rows), dim3(kThreads), 0, stream, uniform_len,
                           valid_len, n_sel, period, k, ws);
        hipLaunchKernelGGL(topk_split_hist2_kernel<false>, grid, dim3(kThreads), 0, stream, src, row_stride,
                           uniform_len, max_chunks, ws);
        hipLaunchKernelGGL(topk_split_scan2_kernel, dim3(rows), dim3(64), 0, stream, max_chunks, ws);
    }
    hipLaunchKernelGGL(topk_split_write_kernel, grid, dim3(kThreads), 0, stream, src, out_idx,
                       row_stride, uniform_len, k, fill, max_chunks, ws, ro);
    if (tr && tr->out_rows)
        return launch_translate_indices(out_idx, tr->out_rows, tr->block_table, rows / tr->rows_per_seq,
                                        (long long)tr->rows_per_seq * k, tr->max_pages, tr->page_shift,
                                        tr->max_pages << tr->page_shift, stream);
    return hipGetLastError();
}

hipError_t launch_topk(const half_t* scores, int* out_idx, int rows, long long row_stride,
                       int uniform_len, const int* valid_len, const int* n_sel, int period, int k,
                       int fill, const TopkRows* tr, hipStream_t stream) {
    if (rows == 0) return hipSuccess;
    const RowsOut ro = rows_out(tr);
    const uint16_t* src = reinterpret_cast<const uint16_t*>(scores);
    // rows of a tensor that starts 16-byte aligned and that fit the register file of a workgroup
    // are selected from registers (rows that start off a boundary bring up to 7 slots in front);
    // anything else streams the row three times
    const bool aligned_rows = (reinterpret_cast<uintptr_t>(scores) & 15) == 0;
    const int slots = uniform_len + (row_stride % 8 != 0 ? 7 : 0);
    auto go = [&](auto threads, auto chunks) {
        constexpr int kT = decltype(threads)::value;
        hipLaunchKernelGGL((topk_select_reg_kernel<kT, decltype(chunks)::value>), dim3(rows), dim3(kT), 0, stream, src,
                           out_idx, row_stride, uniform_len, valid_len, n_sel, period, k, fill, ro);
    };
    // The fewest chunks per wavefront in workgroups of up to 512 threads; long rows take 1024 threads
    // while all their workgroups are resident at once (two per compute unit at four chunks, one at
    // eight), where a row's latency is the time (64 rows: 32768 entries 13.7 -> 11.5 us, 65536
    // 24 -> 19): with more rows the scans over more wavefronts cost throughput (2048 rows: 61 -> 65 us
    // and 141 -> 172).
    const bool few32k = rows <= 2 * kComputeUnits, few64k = rows <= kComputeUnits;
    std::integral_constant<int, 256> t256{};
    std::integral_constant<int, 512> t512{};
    std::integral_constant<int, 1024> t1024{};
    std::integral_constant<int, 1> c1{};
    std::integral_constant<int, 2> c2{};
    std::integral_constant<int, 4> c4{};
    std::integral_constant<int, 8> c8{};
    std::integral_constant<int, 16> c16{};
    if (aligned_rows && slots <= 2048) go(t256, c1);
    else if (aligned_rows && slots <= 4096) go(t512, c1);
    else if (aligned_rows && slots <= 8192) go(t512, c2);
    else if (aligned_rows && slots <= 16384) go(t512, c4);
    else if (aligned_rows && slots <= 32768) few32k ? go(t1024, c4) : go(t512, c8);
    else if (aligned_rows && slots <= 65536) few64k ? go(t1024, c8) : go(t512, c16);
    else if (aligned_rows && slots <= 131072) go(t1024, c16);
    else
        hipLaunchKernelGGL(topk_select_kernel, dim3(rows), dim3(kThreads), 0, stream, src, out_idx,
                           row_stride, uniform_len, valid_len, n_sel, period, k, fill, ro);
    return hipGetLastError();
}

hipError_t launch_decode_pool_select(const DecodePoolParams& p, int rows, int k, int fill, int* out_idx, const TopkRows* tr,
                                     hipStream_t stream) {
    if (rows == 0) return hipSuccess;
    const RowsOut ro = rows_out(tr);
    auto go = [&](auto threads, auto chunks) {
        constexpr int kT = decltype(threads)::value;
        hipLaunchKernelGGL((decode_pool_select_kernel<kT, decltype(chunks)::value>), dim3(rows), dim3(kT), 0, stream, p, k,
                           fill, out_idx, ro);
    };
    std::integral_constant<int, 256> t256{};
    std::integral_constant<int, 512> t512{};
    std::integral_constant<int, 1024> t1024{};
    std::integral_constant<int, 1> c1{};
    std::integral_constant<int, 2> c2{};
    std::integral_constant<int, 4> c4{};
    const int len = p.uniform_len;
    if (len > kPoolSelectRow) return hipErrorInvalidValue;
    if (len <= 2048) go(t256, c1);
    else if (len <= 4096) go(t256, c2);
    else if (len <= 8192) go(t512, c2);
    else if (len <= 16384) go(t512, c4);
    else go(t1024, c4);
    return hipGetLastError();
}

long long topk_sort_workspace_bytes(int rows, int k) {
    return k <= kSortLdsEntries ? 0 : 8ll * rows * k;   // positions (4 bytes) and two key buffers (2 + 2)
}

hipError_t launch_topk_sort_rows(const half_t* scores, int* idx, void* workspace, int rows,
                                 long long row_stride, int uniform_len, const int* valid_len,
                                 int period, int k, hipStream_t stream) {
    if (rows == 0) return hipSuccess;
    const uint16_t* src = reinterpret_cast<const uint16_t*>(scores);
    if (k <= kSortLdsEntries) {
        hipLaunchKernelGGL((topk_sort_rows_kernel<4, kSortLdsEntries>), dim3(rows), dim3(256), 0, stream, src, idx,
                           (int*)nullptr, (uint16_t*)nullptr, row_stride, uniform_len, valid_len, period, k);
    } else {
        int* ws_pos = static_cast<int*>(workspace);
        uint16_t* ws_keys = reinterpret_cast<uint16_t*>(ws_pos + (long long)rows * k);
        hipLaunchKernelGGL((topk_sort_rows_kernel<16, 0>), dim3(rows), dim3(1024), 0, stream, src, idx, ws_pos,
                           ws_keys, row_stride, uniform_len, valid_len, period, k);
    }
    return hipGetLastError();
}

}  // namespace kascade
