// Causal attention of several query rows on the matrix cores
// (v_mfma_f32_16x16x4f32: fp32 products, fp32 sums): prompts from position 0,
// rows that continue a GQA cache in any format, the RINA-MLA prompt over its
// fp32 or packed cache, the latent attention's expanded prompt rows.
//
// A workgroup takes NSET sets of 4 waves.  The four waves of a set share the
// keys and values of one KV head: HPW query heads of it times 4 / HPW tiles of
// 16 query rows (HPW 4, 2, 1 as the head ratio allows).  Set k takes the key
// blocks k, k + NSET, .. (KB keys each) of the workgroup's key range, staged
// once per set in LDS as fp32 (packed records are decoded on the way), the
// next block's bytes loaded while the current one is multiplied; the sets'
// online softmaxes merge through LDS at the end.
// Per block a wave forms S^T = K Q^T (KB / 16 tiles of 16 keys x 16 rows; step
// i multiplies the dims DQ / 4 g + i of the four lane groups g = l / 16: a
// permutation the dot product does not see), so a lane holds KB / 4 scores of
// one query row (l % 16), the row maximum and sum take two cross-lane steps,
// and those scores are directly the B operand of O^T += V^T P^T (dim
// ND (l % 16) + dt of tile dt).  Scores carry log2 e: weights are exp2 values.
// A row's result holds no value past its position, also where that value is
// inf or NaN (a weight of zero times it would not be zero): a block that ends
// past a wave's first row and holds such values is added key by key, over the
// keys that each row sees.
// Where the row tiles leave the chip idle (few rows over a long cache), the
// key range is split over ks_n workgroups whose (m, l, O) partials
// rows_combine_kernel merges.
//
// Bound by the fp32 matrix cores (154 TFLOP/s in a large product).  Before,
// rows that continue a cache took one wave per (row, head), one position per
// step: 512 rows after 1536 cached positions, q8, 32 / 8 heads 5.87 ms.
#include "attn_rows.hpp"
#include "kv_formats.hpp"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

template <typename T>
__device__ __forceinline__ T gld_a2(const uint8_t* p) {   // a load at 2-byte alignment
    typedef T __attribute__((aligned(2))) U;
    return *(const __attribute__((address_space(1))) U*)p;
}

// four floats at 4-byte alignment (one load all the same)
__device__ __forceinline__ f32x4 gld_f4(const float* p) {
    typedef f32x4 __attribute__((aligned(4))) U;
    return *(const __attribute__((address_space(1))) U*)p;
}

// 16 values (half h of a 32-value block) of a packed cache: code bytes and fp16 scale as loaded
struct Half {
    u32x4 c;
    uint32_t s;
};
__device__ __forceinline__ void half_load(int fmt, const uint8_t* b, int h, Half& r) {
    r.s = gld((const uint16_t*)b);
    if (fmt == RINA_KVF_Q8_0) {
        r.c = gld_a2<u32x4>(b + 2 + 16 * h);
    } else if (fmt == RINA_KVF_Q4_0) {
        const u32x2 t = gld_a2<u32x2>(b + 2 + 8 * h);
        r.c.x = t.x; r.c.y = t.y;
    } else if (fmt == RINA_KVF_Q2_1) {
        r.c.x = gld_a2<uint32_t>(b + 2 + 4 * h);
    } else {
        r.c.x = gld((const uint16_t*)(b + 2 + 2 * h));
    }
}
__device__ __forceinline__ void half_values(int fmt, const Half& r, float (&v)[16]) {
    const float s = f16_to_f32((uint16_t)r.s);
    const uint32_t c[4] = {r.c.x, r.c.y, r.c.z, r.c.w};
    if (fmt == RINA_KVF_Q8_0) {
#pragma unroll
        for (int i = 0; i < 16; i++) v[i] = (float)(int8_t)(c[i >> 2] >> (8 * (i & 3))) * s;
    } else if (fmt == RINA_KVF_Q4_0) {
#pragma unroll
        for (int i = 0; i < 16; i++) v[i] = (float)((int)((c[i >> 3] >> (4 * (i & 7))) & 0xF) - 7) * s;
    } else if (fmt == RINA_KVF_Q2_1) {
#pragma unroll
        for (int i = 0; i < 16; i++) v[i] = (float)((int)((c[0] >> (2 * i)) & 3) - 1) * s;
    } else {
#pragma unroll
        for (int i = 0; i < 16; i++) v[i] = ((c[0] >> i) & 1u) ? s : -s;
    }
}

// 0, or NaN if one of the values is inf or NaN
template <int N>
__device__ __forceinline__ float zero_or_nan(const float (&v)[N]) {
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < N; i++) t = fmaf(v[i], 0.f, t);
    return t;
}

// DQ: query / key width held (a multiple of 16; dims past a.da + a.db are
// zero), DV: value width, KB: keys per block.  PK: the cache is packed.
// NSET sets of 4 waves.
template <int SRC, bool PK, int DQ, int DV, int KB, int NSET>
__global__ __launch_bounds__(256 * NSET) void attn_rows_kernel(RowsAttnArgs a, int hpw) {
    constexpr int LDK = DQ + 4, LDV = DV + 4, KT = KB / 16, ND = DV / 16, Q4 = DQ / 16, NC = DQ > 64 ? (DQ > 128 ? 4 : 3) : 2;
    constexpr int TPK = 256 / KB, NK = DQ / TPK / 4, NV = DV / TPK / 4;   // threads per key, float4 each
    __shared__ __align__(16) float s_k[NSET][KB][LDK];
    __shared__ __align__(16) float s_v[NSET][KB][LDV];
    __shared__ int s_bad[NSET];                                  // 1 + the last block whose values are not all finite
    const int tid = threadIdx.x, lane = tid & 63;
    const int set = __builtin_amdgcn_readfirstlane(tid >> 8);
    const int ts = tid & 255;
    const int w = __builtin_amdgcn_readfirstlane((tid >> 6) & 3);
    const int rw = 16 * (4 / hpw);                               // query rows of the workgroup
    const int ntile = (a.T + rw - 1) / rw;
    const int t0 = (ntile - 1 - (int)blockIdx.y) * rw;           // longest row tiles first
    const int h = hpw * (int)blockIdx.x + w % hpw;
    const int kvh = hpw * (int)blockIdx.x / (a.H / a.Hkv);
    const int pos0 = read_pos(a.start_pos, a.d_pos);
    if (pos0 < 0 || pos0 >= a.max_seq) return;                   // capacity guard (device positions)
    const int tmax = min(t0 + rw, a.T) - 1;
    const int fr = lane & 15, g = lane >> 4;
    const int row = t0 + 16 * (w / hpw) + fr, rowc = min(row, a.T - 1);
    // keys 0 .. nkey - 1; row t sees those below lim (DQ: its own position comes from its rows)
    const int nkey = min(pos0 + tmax + (SRC == ROWS_DQ ? 0 : 1), a.max_seq);
    const int lim = pos0 + row + (SRC == ROWS_DQ ? 0 : 1);
    const int nblk = (nkey + KB - 1) / KB, per = (nblk + a.ks_n - 1) / a.ks_n;
    const int b0 = (int)blockIdx.z * per, b1 = min(b0 + per, nblk);
    const float qsc = a.scale * 1.44269504088896341f;
    float qv[DQ / 4];                                            // row fr, dims DQ / 4 g ..
    float m = -INFINITY, l = 0.f;
    f32x4 o[ND];                                                 // tile dt: dims ND (4 g + e) + dt
#pragma unroll
    for (int dt = 0; dt < ND; dt++) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    {
        // (RINA-MLA rows are DQ wide here, zero past their own width)
        const float* qp = a.q + ((int64_t)rowc * a.H + h) * DQ + DQ / 4 * g;
#pragma unroll
        for (int i = 0; i < Q4; i++) {
            const f32x4 v = gld_f4(qp + 4 * i);
            qv[4 * i] = v.x * qsc; qv[4 * i + 1] = v.y * qsc; qv[4 * i + 2] = v.z * qsc; qv[4 * i + 3] = v.w * qsc;
        }
    }
    if (SRC == ROWS_DQ && set == 0 && blockIdx.z == 0) {
        // the row's own position: its fp32 key and value
        const f32x4* kp = (const f32x4*)(a.k + ((int64_t)rowc * a.Hkv + kvh) * DQ + DQ / 4 * g);
        float own = 0.f;
#pragma unroll
        for (int i = 0; i < Q4; i++) {
            const f32x4 v = gld(kp + i);
#pragma unroll
            for (int c = 0; c < 4; c++) own = fmaf(qv[4 * i + c], v[c], own);
        }
        own += __shfl_xor(own, 16);
        own += __shfl_xor(own, 32);
        const float* vp = a.v + ((int64_t)rowc * a.Hkv + kvh) * DV + ND * 4 * g;
        m = own;
        l = 1.f;
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
            for (int dt = 0; dt < ND; dt++) o[dt][e] = gld(vp + ND * e + dt);
    }
    // staging: thread ts of a set moves 4 NK key dims and 4 NV value dims of
    // key j0 + ts / TPK (clamped to the last key: such keys are masked)
    const int sk = ts / TPK, sq = ts % TPK;
    f32x4 kr[NK], vr[NV];
    Half kh, vh;
    int jl = 0;                                                  // the key that is loaded
    auto load_blk = [&](int blk) {
        const int j = min(blk * KB + sk, nkey - 1);
        jl = j;
        if constexpr (SRC == ROWS_GQA) {
            const bool cached = j < pos0;
            if (PK && cached) {
                // 16 dims: half sq & 1 of the head's block sq >> 1
                const int64_t b = ((int64_t)j * a.Hkv + kvh) * 2 + (sq >> 1);
                half_load(a.kf, a.ck + b * kvq::block_bytes(a.kf), sq & 1, kh);
                half_load(a.vf, a.cv + b * kvq::block_bytes(a.vf), sq & 1, vh);
            } else {
                const int64_t off = ((int64_t)(cached ? j : j - pos0) * a.Hkv + kvh) * 64 + 16 * sq;
                const float* kp = (cached ? (const float*)a.ck : a.k) + off;
                const float* vp = (cached ? (const float*)a.cv : a.v) + off;
#pragma unroll
                for (int i = 0; i < 4; i++) { kr[i] = gld_f4(kp + 4 * i); vr[i] = gld_f4(vp + 4 * i); }
            }
        } else if constexpr (SRC == ROWS_DQ) {
            const int64_t r = (int64_t)j * a.Hkv + kvh;
            const int dq = a.da + a.db;
            if (PK) {
                // content dims 16 sq .. (da == 64) from the record, RoPE dims past 64 spread over the four threads
                half_load(RINA_KVF_Q2_1, a.ck + r * 20 + 10 * (sq >> 1), sq & 1, kh);
                half_load(RINA_KVF_Q1_0, a.cv + r * 12 + 6 * (sq >> 1), sq & 1, vh);
                constexpr int NR = (DQ - 64) / 4;                // RoPE dims per thread
#pragma unroll
                for (int i = 0; i < NR; i++) {
                    const int d = NR * sq + i;
                    kr[i / 4][i % 4] = d < a.db ? gld(a.ckr + r * a.db + d) : 0.f;
                }
            } else {
                const float* kp = (const float*)a.ck + r * dq;
                const float* vp = (const float*)a.cv + r * DV + 16 * sq;
                if (a.vec) {                                     // 16-byte aligned rows
#pragma unroll
                    for (int i = 0; i < NK; i++) {
                        const int d = 4 * NK * sq + 4 * i;
                        kr[i] = gld((const f32x4*)(kp + (d < dq ? d : 0)));
                        if (d >= dq) kr[i] = f32x4{0.f, 0.f, 0.f, 0.f};
                    }
#pragma unroll
                    for (int i = 0; i < NV; i++) vr[i] = gld((const f32x4*)vp + i);
                } else {
#pragma unroll
                    for (int i = 0; i < 4 * NK; i++) {
                        const int d = 4 * NK * sq + i;
                        kr[i / 4][i % 4] = d < dq ? gld(kp + d) : 0.f;
                    }
#pragma unroll
                    for (int i = 0; i < 16; i++) vr[i / 4][i % 4] = gld(vp + i);
                }
            }
        } else {
            // [K_nope (128) | k_pe (64)]: thread sq of 8 holds 24 dims, V 16
            const float* kn = a.k + ((int64_t)j * a.H + kvh) * 128;
            const float* kp = (const float*)a.ck + (int64_t)j * a.db + a.da - 128;
#pragma unroll
            for (int i = 0; i < NK; i++) {
                const int d = 4 * NK * sq + 4 * i;
                kr[i] = gld_f4((d < 128 ? kn : kp) + d);
            }
            const float* vp = a.v + ((int64_t)j * a.H + kvh) * 128 + 16 * sq;
#pragma unroll
            for (int i = 0; i < NV; i++) vr[i] = gld_f4(vp + 4 * i);
        }
    };
    // (check: returns NaN if one of the thread's values is not finite)
    auto store_blk = [&](bool check) -> float {
        float* kd = s_k[set][sk];
        float* vd = s_v[set][sk];
        if (SRC == ROWS_GQA && jl < pos0) {
            float kv[16], vv[16];
            if (PK) {
                half_values(a.kf, kh, kv);
                half_values(a.vf, vh, vv);
            } else {
#pragma unroll
                for (int i = 0; i < 16; i++) { kv[i] = kr[i / 4][i % 4]; vv[i] = vr[i / 4][i % 4]; }
            }
            if (a.pre_rope && a.rkc) {
                // raw cached keys: dims d and d + 32 are a pair (gqa_layer.cu:236-238);
                // this thread's partner dims are thread sq ^ 2's
                const float* ct = a.rkc + (int64_t)jl * 32 + 16 * (sq & 1);
                const float* st = a.rks + (int64_t)jl * 32 + 16 * (sq & 1);
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const float y = dpp_f<0x4E>(kv[i]);          // quad_perm [2,3,0,1]
                    const float c = gld(ct + i), s = gld(st + i);
                    kv[i] = sq < 2 ? kv[i] * c - y * s : y * s + kv[i] * c;
                }
            }
#pragma unroll
            for (int i = 0; i < 4; i++) {
                *(f32x4*)&kd[16 * sq + 4 * i] = f32x4{kv[4 * i], kv[4 * i + 1], kv[4 * i + 2], kv[4 * i + 3]};
                *(f32x4*)&vd[16 * sq + 4 * i] = f32x4{vv[4 * i], vv[4 * i + 1], vv[4 * i + 2], vv[4 * i + 3]};
            }
            return check ? zero_or_nan(vv) : 0.f;
        } else if (SRC == ROWS_DQ && PK) {
            float kv[16], vv[16];
            half_values(RINA_KVF_Q2_1, kh, kv);
            half_values(RINA_KVF_Q1_0, vh, vv);
            constexpr int NR = (DQ - 64) / 4;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                *(f32x4*)&kd[16 * sq + 4 * i] = f32x4{kv[4 * i], kv[4 * i + 1], kv[4 * i + 2], kv[4 * i + 3]};
                *(f32x4*)&vd[16 * sq + 4 * i] = f32x4{vv[4 * i], vv[4 * i + 1], vv[4 * i + 2], vv[4 * i + 3]};
            }
#pragma unroll
            for (int i = 0; i < NR / 4; i++) *(f32x4*)&kd[64 + NR * sq + 4 * i] = kr[i];
            return check ? zero_or_nan(vv) : 0.f;
        } else {
#pragma unroll
            for (int i = 0; i < NK; i++) *(f32x4*)&kd[4 * NK * sq + 4 * i] = kr[i];
#pragma unroll
            for (int i = 0; i < NV; i++) *(f32x4*)&vd[4 * NV * sq + 4 * i] = vr[i];
            float vv[4 * NV];
#pragma unroll
            for (int i = 0; i < 4 * NV; i++) vv[i] = vr[i / 4][i % 4];
            return check ? zero_or_nan(vv) : 0.f;
        }
    };
    // the first keys that the workgroup's and this wave's first row do not see
    constexpr int OWN = SRC == ROWS_DQ ? 0 : 1;
    const int lim_wg = pos0 + t0 + OWN, lim_wave = lim_wg + 16 * (w / hpw);
    if (ts == 0) s_bad[set] = 0;
    const int nit = b1 > b0 ? (b1 - b0 + NSET - 1) / NSET : 0;
    if (nit > 0) load_blk(min(b0 + set, b1 - 1));
    for (int it = 0; it < nit; it++) {
        const int blk = b0 + NSET * it + set;                    // past b1: nothing (same for the set)
        __syncthreads();                                         // the previous block's operands are read
        if (store_blk((blk + 1) * KB > lim_wg && blk < b1) != 0.f) s_bad[set] = blk + 1;
        __syncthreads();
        load_blk(min(blk + NSET, b1 - 1));                       // unconditional: clamped past the end
        if (blk >= b1) continue;
        const int j0 = blk * KB;
        // NC partial sums per score (of every NC-th group of 16 dims): one
        // chain over 192 dims had 1.3 times the error of the sum it replaced
        f32x4 sp[NC][KT], s[KT];
#pragma unroll
        for (int c = 0; c < NC; c++)
#pragma unroll
            for (int kt = 0; kt < KT; kt++) sp[c][kt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q4 = 0; q4 < Q4; q4++) {
            f32x4 kv[KT];
#pragma unroll
            for (int kt = 0; kt < KT; kt++) kv[kt] = *(const f32x4*)&s_k[set][16 * kt + fr][DQ / 4 * g + 4 * q4];
#pragma unroll
            for (int c = 0; c < 4; c++)
#pragma unroll
                for (int kt = 0; kt < KT; kt++)
                    sp[q4 % NC][kt] = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[kt][c], qv[4 * q4 + c], sp[q4 % NC][kt], 0, 0, 0);
        }
#pragma unroll
        for (int kt = 0; kt < KT; kt++) {
            s[kt] = sp[0][kt];
#pragma unroll
            for (int c = 1; c < NC; c++) s[kt] += sp[c][kt];
        }
        float mx = -INFINITY;
#pragma unroll
        for (int kt = 0; kt < KT; kt++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                if (j0 + 16 * kt + 4 * g + e >= lim) s[kt][e] = -INFINITY;
                mx = fmaxf(mx, s[kt][e]);
            }
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        const float mn = fmaxf(m, mx);
        const float mr = mn == -INFINITY ? 0.f : mn;             // no key of this block range is visible to the row yet
        const float al = __builtin_amdgcn_exp2f(m - mr);
        float ps = 0.f;
#pragma unroll
        for (int kt = 0; kt < KT; kt++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                s[kt][e] = __builtin_amdgcn_exp2f(s[kt][e] - mr);
                ps += s[kt][e];
            }
        ps += __shfl_xor(ps, 16);
        ps += __shfl_xor(ps, 32);
        l = fmaf(l, al, ps);
        m = mn;
        // the block's own sum first, then added to the running one: two short
        // chains instead of one over all keys (1900 keys: error 2.9e-7 -> below)
        f32x4 ob[ND];
#pragma unroll
        for (int dt = 0; dt < ND; dt++) ob[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (j0 + KB > lim_wave && s_bad[set] == blk + 1) {
            // lane group k4 holds the weights of keys 16 kt + 4 k4 + e
#pragma unroll
            for (int kt = 0; kt < KT; kt++)
#pragma unroll
                for (int e = 0; e < 4; e++)
#pragma unroll 1
                    for (int k4 = 0; k4 < 4; k4++) {
                        const int key = 16 * kt + 4 * k4 + e;
                        const float p = __shfl(s[kt][e], fr + 16 * k4);
                        if (j0 + key >= lim) continue;
#pragma unroll
                        for (int i = 0; i < 4 * ND; i++)
                            ob[i % ND][i / ND] = fmaf(p, s_v[set][key][4 * ND * g + i], ob[i % ND][i / ND]);
                    }
        } else
#pragma unroll
        for (int kt = 0; kt < KT; kt++)
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int d4 = 0; d4 < ND / 4; d4++) {
                    const f32x4 vv = *(const f32x4*)&s_v[set][16 * kt + 4 * g + e][ND * fr + 4 * d4];
#pragma unroll
                    for (int dt = 0; dt < 4; dt++)
                        ob[4 * d4 + dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(vv[dt], s[kt][e], ob[4 * d4 + dt], 0, 0, 0);
                }
#pragma unroll
        for (int dt = 0; dt < ND; dt++)
#pragma unroll
            for (int e = 0; e < 4; e++) o[dt][e] = fmaf(o[dt][e], al, ob[dt][e]);
    }
    // merge the sets through LDS (sets 1 .. leave theirs, set 0 combines)
    __syncthreads();
    float* xm = &s_k[0][0][0];                                   // [NSET - 1][2][256], then O
    f32x4* xo = (f32x4*)(xm + (NSET - 1) * 512);                 // [NSET - 1][ND][256]
    static_assert(NSET == 1 || (NSET - 1) * (512 + ND * 1024) <= NSET * KB * LDK, "exchange fits the key buffer");
    if (set > 0) {
        xm[(set - 1) * 512 + ts] = m;
        xm[(set - 1) * 512 + 256 + ts] = l;
#pragma unroll
        for (int dt = 0; dt < ND; dt++) xo[((set - 1) * ND + dt) * 256 + ts] = o[dt];
    }
    __syncthreads();
    if (set > 0 || row >= a.T || pos0 + row >= a.max_seq) return;
    float mm = m;
#pragma unroll
    for (int k = 1; k < NSET; k++) mm = fmaxf(mm, xm[(k - 1) * 512 + ts]);
    const float mr = mm == -INFINITY ? 0.f : mm;
    const float a0 = __builtin_amdgcn_exp2f(m - mr);
    float lt = l * a0;
    f32x4 ot[ND];
#pragma unroll
    for (int dt = 0; dt < ND; dt++) ot[dt] = o[dt] * a0;
#pragma unroll
    for (int k = 1; k < NSET; k++) {
        const float a1 = __builtin_amdgcn_exp2f(xm[(k - 1) * 512 + ts] - mr);
        lt = fmaf(xm[(k - 1) * 512 + 256 + ts], a1, lt);
#pragma unroll
        for (int dt = 0; dt < ND; dt++) {
            const f32x4 o1 = xo[((k - 1) * ND + dt) * 256 + ts];
#pragma unroll
            for (int e = 0; e < 4; e++) ot[dt][e] = fmaf(o1[e], a1, ot[dt][e]);
        }
    }
    float* op = a.out + ((int64_t)row * a.H + h) * DV;
    if (a.ks_n > 1) {
        const int64_t p = ((int64_t)blockIdx.z * a.T + row) * a.H + h;
        op = a.po + p * DV;
        if (g == 0) {
            gst(a.pm + p, mm);
            gst(a.pl + p, lt);
        }
    }
#pragma unroll
    for (int e = 0; e < 4; e++)
#pragma unroll
        for (int d4 = 0; d4 < ND / 4; d4++) {
            f32x4 v{ot[4 * d4][e], ot[4 * d4 + 1][e], ot[4 * d4 + 2][e], ot[4 * d4 + 3][e]};
            if (a.ks_n == 1) v = f32x4{v.x / lt, v.y / lt, v.z / lt, v.w / lt};
            float* od = op + ND * (4 * g + e) + 4 * d4;
            if (((uintptr_t)op & 15) == 0) {
                gst((f32x4*)od, v);
            } else {
#pragma unroll
                for (int i = 0; i < 4; i++) gst(od + i, v[i]);
            }
        }
}

// one wave per (row, head): the ks_n partials merged and normalized
template <int DV>
__global__ __launch_bounds__(256) void rows_combine_kernel(RowsAttnArgs a) {
    const int lane = threadIdx.x & 63;
    const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6), n = (int64_t)a.T * a.H;
    if (r >= n) return;
    const int pos0 = read_pos(a.start_pos, a.d_pos);
    if (pos0 < 0 || pos0 + (int)(r / a.H) >= a.max_seq) return;  // rows that were not computed
    float mm = -INFINITY;
    for (int z = 0; z < a.ks_n; z++) mm = fmaxf(mm, gld(a.pm + z * n + r));
    float lt = 0.f, o[DV / 64];
#pragma unroll
    for (int i = 0; i < DV / 64; i++) o[i] = 0.f;
    for (int z = 0; z < a.ks_n; z++) {
        const float w = __builtin_amdgcn_exp2f(gld(a.pm + z * n + r) - mm);   // mm is finite: every row sees a key
        lt = fmaf(gld(a.pl + z * n + r), w, lt);
#pragma unroll
        for (int i = 0; i < DV / 64; i++) o[i] = fmaf(gld(a.po + (z * n + r) * DV + 64 * i + lane), w, o[i]);
    }
#pragma unroll
    for (int i = 0; i < DV / 64; i++) gst(a.out + r * DV + 64 * i + lane, o[i] / lt);
}

// Key splits of a launch: the count with the least estimated time.  wg
// workgroups, one per CU at a time (their registers), the longest first; nblk
// key blocks for the last row tile, avg for the one in the middle (causal); tb
// us per block and set.  A round takes as long as its longest workgroup where
// all are alike and as their average where they differ; a split adds the second
// launch (3 us) and its partials (part bytes each, written and read at 4 TB/s).
// us before (two workgroups per CU, two blocks per set at least) / after, 32 / 8
// heads, q8: 2 rows after 400 27.8 / 15.7, 64 rows after 1536 25.9 / 23.1, 128
// rows after 1536 45.2 / 31.7, 512 rows from 0 29.0 / 25.9, after 1536 99.7 /
// 95.9; 300 rows after 1536 70 either way (three splits).
int key_splits(int wg, int nblk, double avg, int nset, double tb, double part) {
    const double tf = 3.5, cus = rina_num_cus();
    int best = 1;
    double least = 1e30;
    for (int ks = 1; ks <= 16 && (ks == 1 || ks * nset < nblk + nset); ks++) {
        const double r = wg * (double)ks / cus, up = ceil(r);
        const double longest = tb * (((nblk + ks - 1) / ks + nset - 1) / nset) + tf;
        const double mean = fmin(longest, tb * fmax(1.0, avg / (ks * nset) + 0.25) + tf);
        const double t = fmax(longest, mean * (r + (up - r) * mean / longest)) + (ks > 1 ? 3.0 + 2.0 * ks * part / 4e6 : 0.0);
        if (t < least) { least = t; best = ks; }
    }
    return best;
}

template <int SRC, bool PK, int DQ, int DV, int KB, int NSET>
int launch(RowsAttnArgs a, hipStream_t st) {
    const int rep = a.H / a.Hkv, hpw = rep % 4 == 0 ? 4 : rep % 2 == 0 ? 2 : 1;
    const int rw = 16 * (4 / hpw), ntile = (a.T + rw - 1) / rw, groups = a.H / hpw;
    const int max_pos = a.d_pos ? a.max_seq : a.start_pos + a.T;
    const int nblk = (max_pos + KB - 1) / KB;
    const double avg = a.d_pos ? nblk : (a.start_pos + 0.5 * (a.T + rw)) / KB;
    const int ks = key_splits(groups * ntile, nblk, avg, NSET, 5.6 * KB * (DQ + DV) / (64 * 128.0),
                              (double)a.T * a.H * (DV + 2) * sizeof(float));
    a.ks_n = ks;
    const size_t n = ks > 1 ? (size_t)ks * a.T * a.H : 0;
    RinaScratch scratch;
    if (n) {
        float* p = (float*)scratch.get(n * (DV + 2) * sizeof(float), st, kScratchOut);
        if (!p) return RINA_ERR_HIP;
        a.po = p;
        a.pm = a.po + n * DV;
        a.pl = a.pm + n;
    }
    hipLaunchKernelGGL((attn_rows_kernel<SRC, PK, DQ, DV, KB, NSET>), dim3(groups, ntile, ks), dim3(256 * NSET), 0, st, a, hpw);
    if (hipGetLastError() != hipSuccess) return RINA_ERR_HIP;
    if (ks > 1) {
        hipLaunchKernelGGL(rows_combine_kernel<DV>, dim3((a.T * a.H + 3) / 4), dim3(256), 0, st, a);
        if (hipGetLastError() != hipSuccess) return RINA_ERR_HIP;
    }
    return RINA_OK;
}

template <bool PK>
int launch_dq(const RowsAttnArgs& a, int dq, hipStream_t st) {
    const int w = dq_rows_width(dq);
    if (w == 64) return launch<ROWS_DQ, PK, 64, 64, 64, 2>(a, st);
    if (w == 80) return launch<ROWS_DQ, PK, 80, 64, 64, 2>(a, st);
    if (w == 96) return launch<ROWS_DQ, PK, 96, 64, 64, 2>(a, st);
    return launch<ROWS_DQ, PK, 128, 64, 64, 2>(a, st);
}

}  // namespace

int attn_rows(RowsSrc src, RowsAttnArgs a, int dq, int dv, hipStream_t st) {
    auto al = [](const void* p, int n) { return (uintptr_t)p % n == 0; };
    if (src == ROWS_GQA) {
        if (dq != 64 || dv != 64) return RINA_ERR_SHAPE;
        const bool cache = a.d_pos || a.start_pos > 0, packed = a.mode != RINA_KV_FP32;
        if (cache && (!al(a.ck, packed ? 2 : 4) || !al(a.cv, packed ? 2 : 4))) return RINA_ERR_SHAPE;
        if (packed) kvq::mode_formats_host(a.mode, a.kf, a.vf);
        return packed && cache ? launch<ROWS_GQA, true, 64, 64, 64, 2>(a, st) : launch<ROWS_GQA, false, 64, 64, 64, 2>(a, st);
    }
    if (src == ROWS_DQ) {
        if (dq > 128 || dv != 64) return RINA_ERR_SHAPE;
        a.vec = dq % 4 == 0 && al(a.ck, 16) && al(a.cv, 16);
        return a.mode == RINA_KV_FP32 ? launch_dq<false>(a, dq, st) : launch_dq<true>(a, dq, st);
    }
    if (dq != 192 || dv != 128) return RINA_ERR_SHAPE;
    return launch<ROWS_MLA, false, 192, 128, 32, 2>(a, st);
}
