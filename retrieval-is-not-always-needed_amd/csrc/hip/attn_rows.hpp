// Causal attention of several query rows (prompts, turns that continue a
// cache): attn_rows.hip.
#pragma once
#include "rina_common.hpp"

enum RowsSrc {
    ROWS_GQA = 0,      // keys below pos0 from a GQA cache (fp32 or packed), the others from the current rows
    ROWS_DQ = 1,       // RINA-MLA: every key from the cache, the row's own position from its fp32 rows
    ROWS_MLA = 2,      // latent attention's expanded rows: K = [K_nope | RoPE(k_pe)], V
};

struct RowsAttnArgs {
    const float *q, *k, *v;             // rows [T, H, dq] (DQ: dq_rows_width wide); current K, V rows (MLA: K_nope, V)
    const uint8_t *ck, *cv;             // caches (DQ q2k_q1v: key content, values); MLA: the latent records (ck)
    const float* ckr;                   // DQ q2k_q1v: key RoPE part
    const float *rkc, *rks;             // GQA pre-RoPE caches: tables that rotate cached keys
    float* out;                         // [T, H, dv]
    int mode, pre_rope, T, H, Hkv, start_pos, max_seq;
    int da, db;                         // DQ: key content / RoPE widths; MLA: record offset of k_pe, record width
    const int* d_pos;
    float scale;
    // filled by attn_rows
    int kf, vf, ks_n, vec;
    float *pm, *pl, *po;                // partials of the ks_n key splits
};

// width of the DQ rows (zeros past da + db)
static inline int dq_rows_width(int dq) { return dq <= 64 ? 64 : dq <= 80 ? 80 : dq <= 96 ? 96 : 128; }

// Launches the attention (RINA_ERR_SHAPE, before any launch: a shape or cache
// alignment it does not take; rows need 4-byte alignment only).  dq, dv: ROWS_GQA 64, 64; ROWS_DQ da + db <= 128, 64;
// ROWS_MLA 192, 128.
int attn_rows(RowsSrc src, RowsAttnArgs a, int dq, int dv, hipStream_t st);

// Dim i of a RINA-MLA row [xa | HF-RoPE(xb)] at position pos (tables
// [max_seq][db/2], NULL: no rotation), the rotation in the reference's
// fused-multiply form.  Every load is issued unconditionally (clamped
// indices) so the caller's load counters stay exact.
__device__ __forceinline__ float dq_dim(const float* xa, const float* xb, const float* tc, const float* ts, int da,
                                        int db, int pos, int i) {
    const int hb = db / 2;
    const int j = i - da, pi = j < 0 ? 0 : (j >> 1 < hb ? j >> 1 : hb - 1);
    const float va = gld(xa + (i < da ? i : da - 1));
    const float* xbb = db > 0 ? xb : xa;
    const float x0 = gld(xbb + (db > 0 ? 2 * pi : 0)), x1 = gld(xbb + (db > 0 ? 2 * pi + 1 : 0));
    const bool rot = tc != nullptr && db > 0;
    const float c = gld((rot ? tc : xbb) + (rot ? (int64_t)pos * hb + pi : 0));
    const float sn = gld((rot ? ts : xbb) + (rot ? (int64_t)pos * hb + pi : 0));
    const float cc = rot ? c : 1.0f, ss = rot ? sn : 0.0f;
    const float vb = (j & 1) ? fmaf(x0, ss, x1 * cc) : fmaf(x0, cc, -(x1 * ss));
    return i < da ? va : vb;
}
