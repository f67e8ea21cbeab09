// Products over several activation rows (gemm.hip): split the rows once,
// multiply them by one or more weight matrices.
#pragma once
#include "rina_common.hpp"

// split rows in matrix-core fragment order, inside a caller's buffer
struct RowsX {
    const void* xp;
    const float* xs;
    const void* xg;
    int rows, K;
};

// quant types and row lengths the products take (M >= 2 rows)
bool rows_gemm_ok(int qt, int K);
size_t rows_split_bytes(int qt, int rows, int K);
// x [.., K] -> fragments in buf (rows_split_bytes, 256-byte aligned), with the
// norm prologue; src != NULL: packed row r is x row src[r], a zero row where
// src[r] < 0 (src holds whole 16-row tiles); used != NULL: only the first
// *used 16-row tiles
int rows_split(int qt, const float* x, const int* src, const int* used, int rows, int K, int pro, const float* nw,
               float eps, void* buf, RowsX* out, hipStream_t st);

// Rows grouped by weight matrix (experts), planned on the device: plan[0] row
// tiles in use, plan[1] 16-row tiles in use, then three ints per row tile: its
// group (whose weights start group * stride bytes into the segment), its first
// 16-row tile, its row limit.  A tile may run past its limit into the next
// group's rows: those outputs are not stored.
struct RowsPlan {
    const int* plan;
    int64_t stride;
    int rt;                // rows per tile: 16 << rt
    int tiles_max, tiles_est;   // most row tiles in use, an estimate
};
// up to 3 segments of one quant type (grouped: 1)
int rows_gemm(const rina_linear_seg* segs, int nseg, int qt, const RowsX& x, int epi, const RowsPlan* pl, hipStream_t st);

// Q4 weights in one launch (gemm_bf3.hip): M >= 16 rows at 16-byte alignment,
// where that is the faster of the two; up to 3 segments, no prologue
bool rows_bf3_ok(const rina_linear_seg* segs, int nseg, int qt, const float* x, int M, int K, int epi);
int rows_bf3(const rina_linear_seg* segs, int nseg, int qt, const float* x, int M, int K, int epi, hipStream_t st);

// fp32 weights: rows and weights 16-byte aligned, K % 4 == 0; M >= 2, up to 3 segments
bool rows_f32_ok(const rina_linear_seg* segs, int nseg, const float* x, int K);
int rows_f32(const rina_linear_seg* segs, int nseg, const float* x, int M, int K, int epi, hipStream_t st);
