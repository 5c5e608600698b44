// Host-visible launcher of the top-k selection kernel (topk.hip).
#pragma once
#include "common.h"

namespace kascade {

// Optional second output of a selection: the selected positions as rows of a paged cache.
struct TopkRows {
    int* out_rows;            // [rows, k], or null: no second output
    const int* block_table;   // [sequences, max_pages]
    int max_pages;
    int page_shift;
    int rows_per_seq;         // consecutive score rows that belong to one sequence
};

hipError_t launch_topk(const half_t* scores, int* out_idx, int rows, long long row_stride,
                       int uniform_len, const int* valid_len, const int* n_sel, int period, int k,
                       int fill, const TopkRows* tr, hipStream_t stream);

// Pooling and selection of decode anchors in one launch, one workgroup per (sequence, KV head) row
// of up to kPoolSelectRow tokens, what its registers hold (kascade_pool_select_row: where it pays).
constexpr int kPoolSelectRow = 32768;
struct DecodePoolParams {
    const float* scores;      // [rows, group_size, scores_stride]: score codes and references (decode.h)
    const float* glse;        // [rows, group_size, num_split] log-sums of the splits, or null: row_sums holds them merged
    float* row_sums;          // [rows, group_size]: written when glse is given
    const int* seqlens;       // [sequences] or null (uniform_len tokens each)
    int num_split, groups, group_size, scores_stride;
    int uniform_len;          // longest row
    int len_cap;              // bound the scores pass put on every length
    float topk_percent;       // > 0: a row selects 128*ceil(floor(percent*len/100)/128) of its len tokens; else k of uniform_len
};
hipError_t launch_decode_pool_select(const DecodePoolParams& p, int rows, int k, int fill, int* out_idx,
                                     const TopkRows* tr, hipStream_t stream);

// Multi-workgroup variant for long rows.  Returns 0 bytes when the single-workgroup kernel
// is the right choice (short rows, or too many rows for the 8 KB/row workspace).
long long topk_split_workspace_bytes(int rows, long long row_len);
// longest row (entries) the one-workgroup selection keeps in registers (the tensor must start 16-byte
// aligned; rows that start off a boundary count 7 slots more)
int topk_max_register_row();
hipError_t launch_topk_split(const half_t* scores, int* out_idx, int rows, long long row_stride,
                             int max_len, int uniform_len, const int* valid_len, const int* n_sel,
                             int period, int k, int fill, void* workspace, const TopkRows* tr,
                             hipStream_t stream);

// Reorders the first min(k, valid length) entries of every row of idx [rows, k] by descending score
// (equal scores: ascending position); workspace: topk_sort_workspace_bytes(rows, k) bytes (0 for
// short lists, which are sorted in LDS).
long long topk_sort_workspace_bytes(int rows, int k);
hipError_t launch_topk_sort_rows(const half_t* scores, int* idx, void* workspace, int rows,
                                 long long row_stride, int uniform_len, const int* valid_len,
                                 int period, int k, hipStream_t stream);

}  // namespace kascade
