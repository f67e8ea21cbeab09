// Matrix products over several activation rows (prompts, short turns, the
// rows of an expert) with quantized weights: out[M, N] = x[M, K] . W[N, K]^T
// for Q4_0, Q4_0F and Q2_K, M >= 2, on the bf16 matrix cores
// (v_mfma_f32_16x16x32_bf16, v_mfma_f32_32x32x16_bf16) with fp32 sums.
//
// Two launches.  x_split_kernel (with the RMSNorm / LayerNorm prologue, or a
// row gather, fused in) writes every row once as three bf16 parts in
// matrix-core fragment order; rows16_kernel / rows32_kernel multiply.
//
// Precision.  A row is scaled by a power of two so that its largest magnitude
// lies in [2^13, 2^14), then split into three bf16 parts, 8 bits each: exact
// for all 24 bits of every value down to 2^-123 of the row's largest.
// Products with the small weight integers are exact in the matrix core's
// fp32, sums are fp32; the row scale comes out again in the epilogue, exactly.
// (Two f16 parts, a third less to load and multiply, lose the last bit of one
// value in four and more below 2^-16 of the row's largest: 512 x 2048 x 8192
// gate/up 82 us against 115, error against 64 bits 8.7e-8 against 7.0e-8 at K
// 512, where the exact split it would have to match has 8.4e-8.)
// inf and NaN stay in the first part: rows that hold them give what fp32
// products give.  (Q2_K rows that hold infinities are added up in a path of
// their own at the end, as their minima are a second product.)
// Error against 64-bit products, Q4_0F, 512 rows: 1.0e-7 at K 2048, 1.8e-7 at
// 8192 (1.56e-7 and 3.05e-7 in one serial K loop): the K dimension is summed
// in up to eight independent slices.
//
// Weights.  Q4: q - 7 is exact in bf16, one fp32 fma per output and 32-value
// block applies the block scale.  Q2_K: sc * q <= 45 is exact in bf16; d is
// applied per 128-value page (per 32-value slice where rows do not start at
// pages); the minima are a second, 16 times shorter contraction
// -(dmin m) . X16 over the sums X16 of each 16 values of x: bf16 parts, two
// of dmin m (exact: 15 bits) and three of X16 (exact).
//
// Structure.  A wave owns 16 MI rows x 16 columns, or 32 R rows x 32 C columns
// (per matrix), over its share of K and reads its operands straight into
// registers: A fragments as contiguous loads, weights as whole blocks (16-row
// tiles: a lane loads one Q4 block, v_permlane16/32_swap transposes the four
// blocks of a 128-value step across the wave's four lane rows; 32-row tiles:
// through LDS of the wave's own).  No barrier in the K loop, so the waves of a
// workgroup (NW across columns, KW along K, interleaved by 128 values) never
// wait for each other; the KW partial tiles meet in LDS once at the end.
// What bounds the 32-row tiles: 512 x 2048 x 8192 gate/up (114 us) without its
// A loads in the K loop 94 us, without the block scales 107, without the
// unpacking 114; matrix cores busy 47 % of its cycles.
#include <type_traits>
#include "rina_common.hpp"
#include "rows_gemm.hpp"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

enum { FMT_Q4_0 = 0, FMT_Q4_0F = 1, FMT_Q2_K = 2, FMT_Q2_S = 3 };   // Q2_S: Q2_K rows that start inside a page

// 16- and 8-byte loads at 4-byte alignment (weight blocks)
__device__ __forceinline__ u32x4 gld4(const uint8_t* p) {
    typedef u32x4 __attribute__((aligned(4))) T;
    return *(const __attribute__((address_space(1))) T*)p;
}
__device__ __forceinline__ u32x2 gld2(const uint8_t* p) {
    typedef u32x2 __attribute__((aligned(4))) T;
    return *(const __attribute__((address_space(1))) T*)p;
}

// the upper halves of two fp32 values as one dword
__device__ __forceinline__ uint32_t hi16_pair(uint32_t lo, uint32_t hi) { return __builtin_amdgcn_perm(hi, lo, 0x07060302u); }

constexpr int kParts = 3;              // bf16 parts of an activation
constexpr int kStep = 64 * kParts;     // 16-byte units of a 16-row tile's 32-value step

// LDS of one wave: its lanes' accesses before are done before those after (no
// wait: a wave's LDS accesses run in order)
__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}
// words of a buffer that is written and read at several widths
typedef uint16_t __attribute__((may_alias)) u16_any;
typedef uint32_t __attribute__((may_alias)) u32_any;

__device__ __forceinline__ float silu_mul(float g, float u) { return g / (1.0f + expf(-g)) * u; }

// ---------------------------------------------------------------------------
// activation rows -> f16 fragments
// ---------------------------------------------------------------------------
// Layout: 16-row tile mt, 32-value step ks, part p (the largest first), 64
// lanes of 16 bytes; lane (r, f) holds row 16 mt + r, values 32 ks + 8 f .. + 7.
// Q2_K also gets the sums of 16 values as three bf16 parts: 16-row tile, window
// of 32 sums, part, lane (r, f) = sums 8 f .. + 7 of row r.  K is padded with
// zeros to whole 128-value steps (and windows), rows to whole tiles.
struct SplitXArgs {
    const float* x;
    const float* nw;
    const int* src;        // row gather: packed row r is x row src[r] (< 0: zero row)
    uint4* xp;
    float* xs;             // [rows] 2^-e of the row scale 2^e (Q2_K: -2^-e if the row holds inf and no NaN)
    uint16_t* xg;          // Q2_K: group-sum fragments
    const int* used;       // grouped rows: 16-row tiles in use (NULL: all)
    int M, K, nks, ngw;
    int pro;
    float eps;
};

// A workgroup takes 4 rows, 256 threads each: the four rows' 16-byte stores of
// one fragment make 64 contiguous bytes, and every load of a row is in flight
// at once.  NU: 8-value units per thread held in registers between the
// statistics and the split (rows of up to 2048 NU values); 0: longer rows, the
// units read again.  One wave per row (16 rows per workgroup, the units in a
// loop) took 12.4 us at 512 x 2048 and 35 us at 512 x 8192.
constexpr int kSplitRows = 4;

template <bool Q2, int NU>
__global__ __launch_bounds__(256 * kSplitRows) void x_split_kernel(SplitXArgs a) {
    __shared__ float s_red[4][kSplitRows][4];
    const int r = threadIdx.x >> 8, tid = threadIdx.x & 255, wave = tid >> 6, lane = tid & 63;
    const int row = blockIdx.x * kSplitRows + r, mt = row >> 4;
    if (a.used && mt >= __builtin_amdgcn_readfirstlane(gld(a.used))) return;   // the whole workgroup: 4 rows of one tile
    int srow = row < a.M ? row : -1;
    if (a.src) srow = __builtin_amdgcn_readfirstlane(gld(a.src + row));
    const int nu = a.K >> 3, nup = a.nks * 4;      // 8-value units, padded
    const float* xr = a.x + (int64_t)(srow < 0 ? 0 : srow) * a.K;
    const f32x4 z4{0.f, 0.f, 0.f, 0.f};
    // 8 values at p: element loads where they are not 16-byte aligned
    auto load8 = [&](const float* p, f32x4& lo, f32x4& hi) {
        if (((uintptr_t)p & 15) == 0) {
            lo = gld((const f32x4*)p);
            hi = gld((const f32x4*)(p + 4));
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                lo[i] = gld(p + i);
                hi[i] = gld(p + 4 + i);
            }
        }
    };
    f32x4 v[NU ? NU : 1][2];
    if (NU > 0) {
#pragma unroll
        for (int i = 0; i < NU; i++) {
            v[i][0] = v[i][1] = z4;
            if (srow >= 0 && tid + 256 * i < nu) load8(xr + 8 * (tid + 256 * i), v[i][0], v[i][1]);
        }
    }
    auto each = [&](auto&& f) {                     // f(unit, low half, high half) over the row
        if (NU > 0) {
#pragma unroll
            for (int i = 0; i < (NU ? NU : 1); i++)
                if (tid + 256 * i < nup) f(tid + 256 * i, v[i][0], v[i][1]);
        } else {
            for (int u = tid; u < nup; u += 256) {
                f32x4 p = z4, q = z4;
                if (srow >= 0 && u < nu) load8(xr + 8 * u, p, q);
                f(u, p, q);
            }
        }
    };
    // a row's sum / maximum over its four waves, each in its own slot
    auto row_sum = [&](float x, int k) {
        x = wave_sum(x);
        if (lane == 0) s_red[k][r][wave] = x;
        __syncthreads();
        return (s_red[k][r][0] + s_red[k][r][1]) + (s_red[k][r][2] + s_red[k][r][3]);
    };
    // the norm of rina_hip_rms_norm / rina_hip_layer_norm, applied to a unit
    float mean = 0.f, inv = 1.f;
    if (a.pro == RINA_PRO_LAYERNORM) {
        float s = 0.f;
        each([&](int, const f32x4& p, const f32x4& q) {
#pragma unroll
            for (int i = 0; i < 4; i++) s += p[i] + q[i];
        });
        mean = row_sum(s, 0) / (float)a.K;
    }
    if (a.pro != RINA_PRO_NONE) {
        float ss = 0.f;
        each([&](int u, const f32x4& p, const f32x4& q) {
            if (u >= nu) return;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                ss = fmaf(p[i] - mean, p[i] - mean, ss);
                ss = fmaf(q[i] - mean, q[i] - mean, ss);
            }
        });
        inv = 1.0f / sqrtf(row_sum(ss, 1) / (float)a.K + a.eps);
    }
    auto normed = [&](int u, f32x4& p, f32x4& q) {
        if (a.pro == RINA_PRO_NONE) return;
        f32x4 g, h;
        load8(a.nw + 8 * (u < nu ? u : 0), g, h);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            p[i] = u < nu ? (p[i] - mean) * inv * g[i] : 0.f;
            q[i] = u < nu ? (q[i] - mean) * inv * h[i] : 0.f;
        }
    };
    if (NU > 0) {
#pragma unroll
        for (int i = 0; i < NU; i++) normed(tid + 256 * i, v[i][0], v[i][1]);
    }
    float mx = 0.f, bad = 0.f;                      // largest finite magnitude; 1: inf, 2: NaN
    each([&](int u, const f32x4& p0, const f32x4& q0) {
        f32x4 p = p0, q = q0;
        if (NU == 0) normed(u, p, q);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            mx = fmaxf(mx, fabsf(p[i]) < INFINITY ? fabsf(p[i]) : 0.f);
            mx = fmaxf(mx, fabsf(q[i]) < INFINITY ? fabsf(q[i]) : 0.f);
            if (Q2) {
                bad = fmaxf(bad, fabsf(p[i]) < INFINITY ? 0.f : p[i] == p[i] ? 1.f : 2.f);
                bad = fmaxf(bad, fabsf(q[i]) < INFINITY ? 0.f : q[i] == q[i] ? 1.f : 2.f);
            }
        }
    });
    mx = wave_max(mx);
    if (Q2) bad = wave_max(bad);
    if (lane == 0) {
        s_red[2][r][wave] = mx;
        if (Q2) s_red[3][r][wave] = bad;
    }
    __syncthreads();
    mx = fmaxf(fmaxf(s_red[2][r][0], s_red[2][r][1]), fmaxf(s_red[2][r][2], s_red[2][r][3]));
    if (Q2) bad = fmaxf(fmaxf(s_red[3][r][0], s_red[3][r][1]), fmaxf(s_red[3][r][2], s_red[3][r][3]));
    // 2^e with mx 2^e in [2^13, 2^14); rows of zeros keep 2^0
    const int ex = (int)((__float_as_uint(mx) >> 23) & 0xFF) - 127;
    const int e = mx > 0.f ? min(max(13 - ex, -126), 126) : 0;
    const float sc = __uint_as_float((uint32_t)(e + 127) << 23);
    if (tid == 0) gst(a.xs + row, __uint_as_float((uint32_t)(127 - e) << 23 | (bad == 1.f ? 0x80000000u : 0u)));
    uint4* xp = a.xp + (int64_t)mt * a.nks * kStep + (row & 15);
    each([&](int u, const f32x4& p0, const f32x4& q0) {
        f32x4 p = p0, q = q0;
        if (NU == 0) normed(u, p, q);
        float w[8];
#pragma unroll
        for (int i = 0; i < 4; i++) { w[i] = p[i] * sc; w[4 + i] = q[i] * sc; }
        uint4* d = xp + (int64_t)(u >> 2) * kStep + (u & 3) * 16;
        float r[8];
#pragma unroll
        for (int i = 0; i < 8; i++) r[i] = w[i];
#pragma unroll
        for (int k = 0; k < kParts; k++) {
            uint32_t b[8];
#pragma unroll
            for (int i = 0; i < 8; i++) {
                b[i] = __float_as_uint(r[i]);
                const bool fin = fabsf(r[i]) < INFINITY;
                if (!(r[i] == r[i])) b[i] = 0x7FC00000u;            // (the low half of a NaN may be all it has)
                r[i] = fin ? r[i] - __uint_as_float(b[i] & 0xFFFF0000u) : 0.f;
            }
            gst((u32x4*)(d + 64 * k), u32x4{hi16_pair(b[0], b[1]), hi16_pair(b[2], b[3]), hi16_pair(b[4], b[5]), hi16_pair(b[6], b[7])});
        }
        if (Q2) {
            // sums of 16 values: threads 2 i, 2 i + 1 hold the two units
            float s = ((w[0] + w[1]) + (w[2] + w[3])) + ((w[4] + w[5]) + (w[6] + w[7]));
            s += dpp_f<0xB1>(s);
            if (!(u & 1)) {
                const int g = u >> 1;
                const uint32_t b0 = __float_as_uint(s) & 0xFFFF0000u;
                const float s1 = s - __uint_as_float(b0);
                const uint32_t b1 = __float_as_uint(s1) & 0xFFFF0000u;
                const float s2 = s1 - __uint_as_float(b1);
                uint16_t* o = a.xg + (((int64_t)mt * a.ngw + (g >> 5)) * 3 * 64 + ((g >> 3) & 3) * 16 + (row & 15)) * 8 + (g & 7);
                gst(o, (uint16_t)(b0 >> 16));
                gst(o + 64 * 8, (uint16_t)(b1 >> 16));
                gst(o + 2 * 64 * 8, (uint16_t)(__float_as_uint(s2) >> 16));
            }
        }
    });
    if (Q2) {
        // zero the sums past the padded row (whole windows are read)
        for (int g = nup / 2 + tid; g < 32 * a.ngw; g += 256) {
            uint16_t* o = a.xg + (((int64_t)mt * a.ngw + (g >> 5)) * 3 * 64 + ((g >> 3) & 3) * 16 + (row & 15)) * 8 + (g & 7);
#pragma unroll
            for (int p = 0; p < 3; p++) gst(o + p * 64 * 8, (uint16_t)0);
        }
    }
}

// ---------------------------------------------------------------------------
// the product
// ---------------------------------------------------------------------------
struct RowsArgs {
    const uint4* xp;
    const float* xs;
    const uint4* xg;
    const uint8_t* w[3];
    const uint8_t* w2;
    float* y[3];
    int N[3];
    int t0[3];             // first column tile of each segment
    int nseg;
    int M, K, nks, ngw, epi;
    int mt, nt;            // row tiles of 16 MI, column tiles of 16 NJ NW
    int xb, mpp, npp;      // XCD split: weight parts, row / column tiles per part
    int NW, KW;
    // grouped rows (experts): plan[0] row tiles in use, plan[1] 16-row tiles in
    // use, then per row tile its group, first 16-row tile and row limit
    const int* plan;
    int64_t stride;
};

// x[j] of lane row g -> x[g] of lane row j (lane rows: 16 lanes each)
__device__ __forceinline__ void transpose4(uint32_t (&x)[4]) {
    const auto a = __builtin_amdgcn_permlane16_swap(x[0], x[1], false, false);
    const auto b = __builtin_amdgcn_permlane16_swap(x[2], x[3], false, false);
    const auto c = __builtin_amdgcn_permlane32_swap(a[0], b[0], false, false);
    const auto d = __builtin_amdgcn_permlane32_swap(a[1], b[1], false, false);
    x[0] = c[0]; x[2] = c[1]; x[1] = d[0]; x[3] = d[1];
}

// o[g] in every lane = v of lane row g (same lane % 16)
__device__ __forceinline__ void spread4(uint32_t v, uint32_t (&o)[4]) {
    const auto a = __builtin_amdgcn_permlane16_swap(v, v, false, false);      // [0 0 2 2], [1 1 3 3]
    const auto b = __builtin_amdgcn_permlane32_swap(a[0], a[0], false, false);
    const auto c = __builtin_amdgcn_permlane32_swap(a[1], a[1], false, false);
    o[0] = b[0]; o[2] = b[1]; o[1] = c[0]; o[3] = c[1];
}

// One column tile's weights for a 128-value step, as loaded
template <int FMT>
struct WRaw;
template <>
struct WRaw<FMT_Q4_0F> { u32x4 n; uint32_t s; };
template <>
struct WRaw<FMT_Q4_0> { u32x4 n; uint32_t s; };
template <>
struct WRaw<FMT_Q2_K> { u32x2 q, s; uint32_t d; };
template <>
struct WRaw<FMT_Q2_S> { u32x2 q[4]; uint32_t s[4], d[4]; };

// Column n, 128-value step ss, lane row f.  Steps past the row's blocks read
// its last block; x is zero there.  Columns past N read column 0.
template <int FMT>
__device__ __forceinline__ void w_load(const uint8_t* w, int n, int K, int ss, int f, WRaw<FMT>& r) {
    if constexpr (FMT == FMT_Q4_0F) {
        const int nb = K >> 5;
        const uint8_t* p = w + ((int64_t)n * nb + min(4 * ss + f, nb - 1)) * 20;
        r.s = gld((const uint32_t*)p);
        r.n = gld4(p + 4);
    } else if constexpr (FMT == FMT_Q4_0) {
        // 18-byte blocks: an odd block's 16 nibble bytes are 4-byte aligned
        // behind its scale, an even block's first 16 bytes are; the other
        // two bytes are the scale or the last four nibbles
        const int nb = K >> 5;
        const int64_t u = (int64_t)n * nb + min(4 * ss + f, nb - 1);
        const uint8_t* p = w + u * 18;
        const int odd = (int)(u & 1);
        r.n = gld4(p + 2 * odd);
        r.s = (uint32_t)gld((const uint16_t*)(p + (odd ? 0 : 16))) | ((uint32_t)odd << 31);
    } else if constexpr (FMT == FMT_Q2_K) {
        const int64_t pg = (int64_t)n * (K >> 7) + ss;
        const uint8_t* b = w + (pg >> 1) * 84;
        const int o = (int)(pg & 1);
        r.s = gld2(b + 8 * o);
        r.q = gld2(b + 16 + 32 * o + 8 * f);
        r.d = gld((const uint16_t*)(b + 80));
    } else {
        const int nb = K >> 5;
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const int64_t sl = (int64_t)n * nb + min(4 * ss + s, nb - 1);   // 32-value slice in flat order
            const uint8_t* b = w + (sl >> 3) * 84;
            const int j = (int)(sl & 7);
            r.q[s] = gld2(b + 16 + 32 * (j >> 2) + 8 * f);
            r.s[s] = (uint32_t)gld(b + 2 * j + (f >> 1)) | ((uint32_t)(2 * (j & 3)) << 8);
            r.d[s] = gld((const uint16_t*)(b + 80));
        }
    }
}

// the eight nibbles of a dword -> q - 7 as bf16, in order (small integers: exact)
__device__ __forceinline__ u32x4 q4_unpack(uint32_t x) {
    const uint32_t lo = and_opaque(x, 0x0F0F0F0Fu), hi = and_opaque(x >> 4, 0x0F0F0F0Fu);
    u32x4 r;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const float f0 = (float)((lo >> (8 * j)) & 0xFF) - 7.0f, f1 = (float)((hi >> (8 * j)) & 0xFF) - 7.0f;
        r[j] = hi16_pair(__float_as_uint(f0), __float_as_uint(f1));
    }
    return r;
}
// sc * q as bf16 (at most 45: exact) for the 2-bit fields at bit 2 st of eight
// bytes, in order; by: the scale byte
__device__ __forceinline__ u32x4 q2_unpack(u32x2 b, uint32_t by, int st) {
    const float sc = (float)(by & 15u);
    u32x4 r;
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const uint32_t q = and_opaque((h ? b.y : b.x) >> (2 * st), 0x03030303u);
        float f[4];
#pragma unroll
        for (int j = 0; j < 4; j++) f[j] = sc * (float)((q >> (8 * j)) & 0xFF);
        r[2 * h] = hi16_pair(__float_as_uint(f[0]), __float_as_uint(f[1]));
        r[2 * h + 1] = hi16_pair(__float_as_uint(f[2]), __float_as_uint(f[3]));
    }
    return r;
}

// nibble dwords and fp32 scale of a Q4 block from the five dwords at its
// (4-byte aligned down) start; odd: a Q4_0 block that starts two bytes in
template <int FMT>
__device__ __forceinline__ void q4_dwords(const uint32_t (&d)[5], bool odd, uint32_t (&n)[4], uint32_t& s) {
    if constexpr (FMT == FMT_Q4_0F) {
        s = d[0];
#pragma unroll
        for (int i = 0; i < 4; i++) n[i] = d[1 + i];
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++) n[i] = odd ? d[1 + i] : __builtin_amdgcn_alignbyte(d[1 + i], d[i], 2);
        s = __float_as_uint(f16_to_f32((odd ? d[0] >> 16 : d[0]) & 0xFFFFu));
    }
}

// nibble dwords and fp32 scale of one loaded Q4 block
template <int FMT>
__device__ __forceinline__ void q4_block(const WRaw<FMT>& r, uint32_t (&n)[4], uint32_t& s) {
    if constexpr (FMT == FMT_Q4_0F) {
        s = r.s;
        n[0] = r.n.x; n[1] = r.n.y; n[2] = r.n.z; n[3] = r.n.w;
    } else {
        const bool odd = (int)r.s < 0;
        const uint32_t x = r.s & 0xFFFFu;
        const uint32_t e0 = __builtin_amdgcn_alignbyte(r.n.y, r.n.x, 2), e1 = __builtin_amdgcn_alignbyte(r.n.z, r.n.y, 2);
        const uint32_t e2 = __builtin_amdgcn_alignbyte(r.n.w, r.n.z, 2), e3 = __builtin_amdgcn_alignbyte(x, r.n.w, 2);
        n[0] = odd ? r.n.x : e0; n[1] = odd ? r.n.y : e1; n[2] = odd ? r.n.z : e2; n[3] = odd ? r.n.w : e3;
        s = __float_as_uint(f16_to_f32(odd ? x : r.n.x & 0xFFFFu));
    }
}

// Weights of a 128-value step ready to use: the four steps' B fragments are
// formed one at a time by step()
template <int FMT>
struct WStep {
    uint32_t n[4];       // Q4: this lane's nibble dword of each 32-value block
    float sc[4];         // Q4 / Q2_S: the column's scale per block; Q2_K: sc[0]
    u32x2 q[FMT == FMT_Q2_S ? 4 : 1];
    uint32_t s[4];
    __device__ __forceinline__ void take(const WRaw<FMT>& r, int f) {
        if constexpr (FMT == FMT_Q4_0F || FMT == FMT_Q4_0) {
            uint32_t s1, s4[4];
            q4_block<FMT>(r, n, s1);
            transpose4(n);
            spread4(s1, s4);
#pragma unroll
            for (int i = 0; i < 4; i++) sc[i] = __uint_as_float(s4[i]);
        } else if constexpr (FMT == FMT_Q2_K) {
            q[0] = r.q;
            // scale byte of group 2 g + half: byte 2 g + (f >> 1) of the page's eight
            const uint32_t sh = 8 * (f >> 1);
            s[0] = r.s.x >> sh; s[1] = r.s.x >> (sh + 16); s[2] = r.s.y >> sh; s[3] = r.s.y >> (sh + 16);
            sc[0] = f16_to_f32(r.d);
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                q[i] = r.q[i];
                s[i] = r.s[i];
                sc[i] = f16_to_f32(r.d[i]);
            }
        }
    }
    __device__ __forceinline__ bf16x8 frag(int st) const {
        if constexpr (FMT == FMT_Q4_0F || FMT == FMT_Q4_0) return __builtin_bit_cast(bf16x8, q4_unpack(n[st]));
        else if constexpr (FMT == FMT_Q2_K) return __builtin_bit_cast(bf16x8, q2_unpack(q[0], s[st], st));
        else return __builtin_bit_cast(bf16x8, q2_unpack(u32x2{q[st].x >> (s[st] >> 8), q[st].y >> (s[st] >> 8)}, s[st], 0));
    }
};

// -(dmin m) of the eight 16-value groups g0 .. g0 + 7 of column n as two bf16 parts
template <int FMT>
__device__ __forceinline__ void min_frag(const uint8_t* w, int n, int K, int g0, bf16x8& hi, bf16x8& lo) {
    const int ng = K >> 4;
    uint32_t ph[4], pl[4];
    u32x2 pb{0, 0};
    float pd = 0.f;
    if constexpr (FMT == FMT_Q2_K) {                // a page of the row: eight groups of one block
        const int64_t pg = (int64_t)n * (K >> 7) + min(g0 >> 3, (K >> 7) - 1);
        const uint8_t* b = w + (pg >> 1) * 84;
        pb = gld2(b + 8 * (pg & 1));
        pd = -f16_to_f32(gld((const uint16_t*)(b + 82)));
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {                   // a 32-value slice: two groups of one block
        uint32_t by;
        float d;
        if constexpr (FMT == FMT_Q2_K) {
            by = ((i & 2) ? pb.y : pb.x) >> (16 * (i & 1));
            d = pd;
        } else {
            const int64_t sl = (int64_t)n * (K >> 5) + (min(g0 + 2 * i, ng - 2) >> 1);
            const uint8_t* b = w + (sl >> 3) * 84;
            by = gld((const uint16_t*)(b + 2 * (sl & 7)));
            d = -f16_to_f32(gld((const uint16_t*)(b + 82)));
        }
        const float v0 = d * (float)((by >> 4) & 15u), v1 = d * (float)((by >> 12) & 15u);
        const uint32_t h0 = __float_as_uint(v0) & 0xFFFF0000u, h1 = __float_as_uint(v1) & 0xFFFF0000u;
        ph[i] = (h0 >> 16) | h1;
        pl[i] = (__float_as_uint(v0 - __uint_as_float(h0)) >> 16) | (__float_as_uint(v1 - __uint_as_float(h1)) & 0xFFFF0000u);
    }
    hi = __builtin_bit_cast(bf16x8, u32x4{ph[0], ph[1], ph[2], ph[3]});
    lo = __builtin_bit_cast(bf16x8, u32x4{pl[0], pl[1], pl[2], pl[3]});
}

// This workgroup's tile.  Workgroups go to the 8 XCDs round-robin in linear
// order: id % 8 owns row part (id % 8) / xb and column part (id % 8) % xb.
struct Tile {
    const uint8_t* w;
    const uint8_t* w2;
    float* y;
    int N, bx;             // bx: column tile inside the segment
    int r16, mend;         // first 16-row tile, row limit
    __device__ __forceinline__ bool find(const RowsArgs& a, int n16) {   // n16: 16-row tiles per row tile
        const int xcd = blockIdx.x & 7, kb = blockIdx.x >> 3;
        const int mm = kb / a.npp, nn = kb - mm * a.npp;
        int mpp = a.mpp, mt = a.mt;
        if (a.plan) {                               // row tiles in use: known on the device only
            mt = min(mt, __builtin_amdgcn_readfirstlane(gld(a.plan)));
            mpp = (mt + 8 / a.xb - 1) / (8 / a.xb);
        }
        const int by = (xcd / a.xb) * mpp + mm;
        bx = (xcd % a.xb) * a.npp + nn;
        if (mm >= mpp || by >= mt || bx >= a.nt) return false;
        const int sg = (a.nseg > 1 && bx >= a.t0[1]) + (a.nseg > 2 && bx >= a.t0[2]);
        w = sg == 0 ? a.w[0] : sg == 1 ? a.w[1] : a.w[2];
        w2 = a.w2;
        y = sg == 0 ? a.y[0] : sg == 1 ? a.y[1] : a.y[2];
        N = sg == 0 ? a.N[0] : sg == 1 ? a.N[1] : a.N[2];
        bx -= sg == 0 ? a.t0[0] : sg == 1 ? a.t0[1] : a.t0[2];
        r16 = by * n16;
        mend = a.M;
        if (a.plan) {
            const int* p = a.plan + 2 + 3 * by;
            const int64_t g = __builtin_amdgcn_readfirstlane(gld(p));
            r16 = __builtin_amdgcn_readfirstlane(gld(p + 1));
            mend = __builtin_amdgcn_readfirstlane(gld(p + 2));
            w += g * a.stride;
            w2 += g * a.stride;
        }
        return true;
    }
};

template <int NMAT>
__device__ __forceinline__ void finish(const RowsArgs& a, const Tile& t, int r, int c, float v, float u) {
    if (r >= t.mend || c >= t.N) return;
    float* o = t.y + (int64_t)r * t.N + c;
    if (NMAT == 2) gst(o, silu_mul(v, u));
    else if (a.epi == RINA_EPI_ADD) gst(o, gld(o) + v);
    else gst(o, v);
}

// Q2_K rows of a tile that hold infinities (xs < 0): the sums over those
// values alone (the others are finite) with the weights dequantized, as fp32
// products give them: the infinity of the weight's sign, NaN for a weight of
// zero or where both signs meet.  Column c per lane, COLS lanes of columns, the
// 64 / COLS lane rows g along K.
template <int NMAT, int COLS>
__device__ void inf_rows(const RowsArgs& a, const Tile& t, int r0, int rows, int c, int g) {
    const int n = c < t.N ? c : 0;
    auto weight = [&](const uint8_t* w, int k) {
        const int64_t e = (int64_t)n * a.K + k;
        const uint8_t* b = w + (e >> 8) * 84;
        const int i = (int)(e & 255);
        const int sc = gld(b + (i >> 4)), q = (gld(b + 16 + 32 * (i >> 7) + (i & 31)) >> (2 * ((i & 127) >> 5))) & 3;
        return fmaf(f16_to_f32(gld((const uint16_t*)(b + 80))) * (float)(sc & 15), (float)q,
                    -(f16_to_f32(gld((const uint16_t*)(b + 82))) * (float)(sc >> 4)));
    };
#pragma unroll 1
    for (int r = r0; r < min(r0 + rows, t.mend); r++) {
        if (!(gld(a.xs + r) < 0.f)) continue;
        float v = 0.f, u = 0.f;
        const u32x4* xp = (const u32x4*)a.xp + (int64_t)(r >> 4) * a.nks * kStep + (r & 15);
#pragma unroll 1
        for (int un = g; un < a.K >> 3; un += 64 / COLS) {
            const u32x4 x = gld(xp + (int64_t)(un >> 2) * kStep + (un & 3) * 16);
#pragma unroll 1
            for (int i = 0; i < 8; i++) {
                const uint32_t d = i < 2 ? x.x : i < 4 ? x.y : i < 6 ? x.z : x.w, h = (i & 1) ? d >> 16 : d & 0xFFFFu;
                if ((h & 0x7FFFu) != 0x7F80u) continue;
                const float xi = __uint_as_float(h << 16);
                v = fmaf(xi, weight(t.w, 8 * un + i), v);
                if (NMAT == 2) u = fmaf(xi, weight(t.w2, 8 * un + i), u);
            }
        }
#pragma unroll
        for (int m = COLS; m < 64; m *= 2) {
            v += __shfl_xor(v, m);
            u += __shfl_xor(u, m);
        }
        if (g == 0) finish<NMAT>(a, t, r, c, v, u);
    }
}

// Weights as loaded for 32-column tiles (two lane rows of 32 columns): a lane holds
// blocks 4 ss + f and 4 ss + 2 + f of its column, or its half of a page
template <int FMT>
struct WRaw32;
template <>
struct WRaw32<FMT_Q2_K> { u32x2 q[2], s; uint32_t d; };
template <>
struct WRaw32<FMT_Q2_S> { u32x2 q[4][2]; uint32_t s[4], d[4]; };

template <int FMT>
__device__ __forceinline__ void w_load32(const uint8_t* w, int n, int K, int ss, int f, WRaw32<FMT>& r) {
    if constexpr (FMT == FMT_Q2_K) {
        const int64_t pg = (int64_t)n * (K >> 7) + ss;
        const uint8_t* b = w + (pg >> 1) * 84;
        const int o = (int)(pg & 1);
        r.s = gld2(b + 8 * o);
        r.q[0] = gld2(b + 16 + 32 * o + 8 * f);
        r.q[1] = gld2(b + 32 + 32 * o + 8 * f);
        r.d = gld((const uint16_t*)(b + 80));
    } else {
        const int nb = K >> 5;
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const int64_t sl = (int64_t)n * nb + min(4 * ss + s, nb - 1);   // 32-value slice in flat order
            const uint8_t* b = w + (sl >> 3) * 84;
            const int j = (int)(sl & 7);
            r.q[s][0] = gld2(b + 16 + 32 * (j >> 2) + 8 * f);
            r.q[s][1] = gld2(b + 32 + 32 * (j >> 2) + 8 * f);
            r.s[s] = (uint32_t)gld((const uint16_t*)(b + 2 * j)) | ((uint32_t)(2 * (j & 3)) << 16);
            r.d[s] = gld((const uint16_t*)(b + 80));
        }
    }
}

template <int FMT>
struct WStep32 {
    uint32_t n[4][2];    // Q4: this lane's nibble dwords (halves 0, 1) of each 32-value block
    float sc[4];
    u32x2 q[FMT == FMT_Q2_S ? 4 : 1][2];
    uint32_t s[4];
    // Q4: blocks 2 b + f of the column, five dwords each (d[b])
    __device__ __forceinline__ void take_q4(const uint32_t (&d)[2][5], bool odd) {
#pragma unroll
        for (int b = 0; b < 2; b++) {               // lane row 0 holds block 2 b, lane row 1 block 2 b + 1
            uint32_t x[4], s1;
            q4_dwords<FMT>(d[b], odd, x, s1);
            // [own d0, d1 of the lower row | d0, d1 of the upper row]: lane row f gets dword f (and 2 + f)
            const auto lo = __builtin_amdgcn_permlane32_swap(x[0], x[1], false, false);
            const auto hi = __builtin_amdgcn_permlane32_swap(x[2], x[3], false, false);
            const auto sp = __builtin_amdgcn_permlane32_swap(s1, s1, false, false);
            n[2 * b][0] = lo[0]; n[2 * b + 1][0] = lo[1];
            n[2 * b][1] = hi[0]; n[2 * b + 1][1] = hi[1];
            sc[2 * b] = __uint_as_float(sp[0]);
            sc[2 * b + 1] = __uint_as_float(sp[1]);
        }
    }
    template <typename Raw>
    __device__ __forceinline__ void take(const Raw& r) {
        if constexpr (FMT == FMT_Q2_K) {
            q[0][0] = r.q[0]; q[0][1] = r.q[1];
            s[0] = r.s.x; s[1] = r.s.x >> 16; s[2] = r.s.y; s[3] = r.s.y >> 16;
            sc[0] = f16_to_f32(r.d);
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                q[i][0] = r.q[i][0]; q[i][1] = r.q[i][1];
                s[i] = r.s[i];
                sc[i] = f16_to_f32(r.d[i]);
            }
        }
    }
    // weights of 16-value half h of 32-value step st
    __device__ __forceinline__ bf16x8 frag(int st, int h) const {
        if constexpr (FMT == FMT_Q4_0F || FMT == FMT_Q4_0) return __builtin_bit_cast(bf16x8, q4_unpack(n[st][h]));
        else if constexpr (FMT == FMT_Q2_K) return __builtin_bit_cast(bf16x8, q2_unpack(q[0][h], s[st] >> (8 * h), st));
        else {
            const uint32_t sh = s[st] >> 16;
            return __builtin_bit_cast(bf16x8, q2_unpack(u32x2{q[st][h].x >> sh, q[st][h].y >> sh}, s[st] >> (8 * h), 0));
        }
    }
};

// 128-value steps whose weights a wave loads together, one batch ahead: with
// few rows the launch is the weight stream, and a wave that asks for one step
// at a time waits a memory round trip per step (8 x 2048 x 8192: 23.6 us with
// one step ahead).  Bounded by the registers.
template <int FMT, int NMAT, int MI>
struct Batch16 { static constexpr int BT = FMT == FMT_Q2_S ? 1 : NMAT * MI >= 4 ? 2 : 4; };

// ---- 16- and 32-row tiles: v_mfma_f32_16x16x32_bf16 ----
// MI 16-row tiles (all the rows of a group), 16 columns (per matrix) per wave.
template <int FMT, int NMAT, int MI>
__global__ __launch_bounds__(512, 2) void rows16_kernel(RowsArgs a) {
    extern __shared__ __align__(16) float s_part[];
    constexpr int BT = Batch16<FMT, NMAT, MI>::BT;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int fr = lane & 15, f = lane >> 4;
    Tile t;
    if (!t.find(a, MI)) return;
    const int wn = wave % a.NW, wk = wave / a.NW;
    const int c0 = (t.bx * a.NW + wn) * 16 + fr, N = t.N;
    const int K = a.K, nss = a.nks >> 2, col = c0 < N ? c0 : 0;
    const int mtiles = (a.M + 15) >> 4;
    const bf16x8* ap[MI];
#pragma unroll
    for (int i = 0; i < MI; i++) ap[i] = (const bf16x8*)a.xp + (int64_t)min(t.r16 + i, mtiles - 1) * a.nks * kStep + lane;
    f32x4 acc[NMAT][MI];
#pragma unroll
    for (int m = 0; m < NMAT; m++)
#pragma unroll
        for (int i = 0; i < MI; i++) acc[m][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    WRaw<FMT> raw[BT][NMAT];
    bf16x8 af[MI][2 * kParts];                      // 64 values: half a step
    // batch b: steps BT b .. + BT - 1 (past the end: the last step again, not multiplied)
    auto load_w = [&](int b) {
#pragma unroll
        for (int s = 0; s < BT; s++)
#pragma unroll
            for (int m = 0; m < NMAT; m++) w_load<FMT>(m ? t.w2 : t.w, col, K, min(BT * b + s, nss - 1), f, raw[s][m]);
    };
    auto load_a = [&](int ss, int half) {
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int c = 0; c < 2 * kParts; c++) af[i][c] = gld(ap[i] + (int64_t)(4 * min(ss, nss - 1) + 2 * half) * kStep + 64 * c);
    };
    constexpr bool PAGE = FMT == FMT_Q2_K;          // one scale per 128-value step
    const int nb = (nss + BT - 1) / BT;
    if (wk < nb) {
        load_w(wk);
        load_a(BT * wk, 0);
    }
    for (int b = wk; b < nb; b += a.KW) {
        WStep<FMT> ws[BT][NMAT];
#pragma unroll
        for (int s = 0; s < BT; s++)
#pragma unroll
            for (int m = 0; m < NMAT; m++) ws[s][m].take(raw[s][m], f);
        const int bn = b + a.KW < nb ? b + a.KW : b;   // the last batch loads itself again
#pragma unroll
        for (int s = 0; s < BT; s++) {
            // (a page's sum: the largest parts and the others apart, or every
            // small product rounds the whole sum)
            f32x4 d[NMAT][MI], ds[NMAT][MI];
#pragma unroll
            for (int half = 0; half < 2; half++) {
                bf16x8 at[MI][2 * kParts];
#pragma unroll
                for (int i = 0; i < MI; i++)
#pragma unroll
                    for (int c = 0; c < 2 * kParts; c++) at[i][c] = af[i][c];
                load_a(half == 0 ? BT * b + s : s + 1 < BT ? BT * b + s + 1 : BT * bn, half ^ 1);
                if (s == 0 && half == 0) load_w(bn);
                __builtin_amdgcn_sched_barrier(0);  // issued before these products
                if (BT > 1 && BT * b + s >= nss) continue;
#pragma unroll
                for (int m = 0; m < NMAT; m++) {
#pragma unroll
                    for (int st = 2 * half; st < 2 * half + 2; st++) {
                        const bf16x8 w = ws[s][m].frag(st);
                        // smallest parts first
#pragma unroll
                        for (int p = kParts - 1; p >= 0; p--)
#pragma unroll
                            for (int i = 0; i < MI; i++) {
                                f32x4& t = PAGE && p > 0 ? ds[m][i] : d[m][i];
                                if (PAGE ? st == 0 && p != 1 : p == kParts - 1) t = f32x4{0.f, 0.f, 0.f, 0.f};
                                t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(at[i][kParts * (st & 1) + p], w, t, 0, 0, 0);
                            }
                        if (!PAGE || st == 3) {
#pragma unroll
                            for (int i = 0; i < MI; i++)
#pragma unroll
                                for (int e = 0; e < 4; e++) {
                                    const float v = PAGE ? d[m][i][e] + ds[m][i][e] : d[m][i][e];
                                    acc[m][i][e] = fmaf(ws[s][m].sc[PAGE ? 0 : st], v, acc[m][i][e]);
                                }
                        }
                    }
                }
            }
        }
    }
    if constexpr (FMT == FMT_Q2_K || FMT == FMT_Q2_S) {
        for (int gw = wk; gw < a.ngw; gw += a.KW) {
            bf16x8 xg[MI][3];
#pragma unroll
            for (int i = 0; i < MI; i++) {
                const bf16x8* gp = (const bf16x8*)a.xg + ((int64_t)min(t.r16 + i, mtiles - 1) * a.ngw + gw) * 192 + lane;
#pragma unroll
                for (int p = 0; p < 3; p++) xg[i][p] = gld(gp + 64 * p);
            }
#pragma unroll
            for (int m = 0; m < NMAT; m++) {
                bf16x8 hi, lo;
                min_frag<FMT>(m ? t.w2 : t.w, col, K, 32 * gw + 8 * f, hi, lo);
#pragma unroll
                for (int i = 0; i < MI; i++) {
                    f32x4 d = acc[m][i];
                    d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xg[i][2], hi, d, 0, 0, 0);
                    d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xg[i][1], lo, d, 0, 0, 0);
                    d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xg[i][1], hi, d, 0, 0, 0);
                    d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xg[i][0], lo, d, 0, 0, 0);
                    acc[m][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xg[i][0], hi, d, 0, 0, 0);
                }
            }
        }
    }
    // the KW partial tiles, halved per round: waves h .. 2 h - 1 leave theirs
    // in LDS, waves 0 .. h - 1 add
    f32x4* sp = (f32x4*)s_part;
    for (int h = a.KW >> 1; h >= 1; h >>= 1) {
        f32x4* d = sp + (int64_t)((wk >= h ? wk - h : wk) * a.NW + wn) * NMAT * MI * 64 + lane;
        if (wk >= h && wk < 2 * h) {
#pragma unroll
            for (int m = 0; m < NMAT; m++)
#pragma unroll
                for (int i = 0; i < MI; i++) d[(m * MI + i) * 64] = acc[m][i];
        }
        __syncthreads();
        if (wk < h) {
#pragma unroll
            for (int m = 0; m < NMAT; m++)
#pragma unroll
                for (int i = 0; i < MI; i++) acc[m][i] += d[(m * MI + i) * 64];
        }
        __syncthreads();
    }
    if (wk > 0) return;
    constexpr bool Q2 = FMT == FMT_Q2_K || FMT == FMT_Q2_S;
    bool inf = false;                               // rows of inf_rows
#pragma unroll
    for (int i = 0; i < MI; i++) {
        const int r0 = (t.r16 + i) * 16 + 4 * f;
        if (r0 >= t.mend) continue;
        const f32x4 sc = gld((const f32x4*)(a.xs + r0));
#pragma unroll
        for (int e = 0; e < 4; e++) {
            if (Q2 && sc[e] < 0.f) inf |= r0 + e < t.mend;
            else finish<NMAT>(a, t, r0 + e, c0, acc[0][i][e] * sc[e], acc[NMAT - 1][i][e] * sc[e]);
        }
    }
    if (Q2 && __any(inf)) inf_rows<NMAT, 16>(a, t, t.r16 * 16, 16 * MI, c0, f);
}

// ---- 64-row tiles: v_mfma_f32_32x32x16_bf16 ----
// A wave owns 32 R rows x 32 C columns (per matrix) of its K slice.  Q4 weights
// pass through a buffer of the wave's own in LDS: the 80 (72) bytes of a
// column's 128-value step are loaded as five 16-byte chunks by neighbouring
// lanes and read back block by block (no barrier: only this wave uses it).
// Loaded block by block straight into the lanes that use them, every 20-byte
// block costs two address slots of the load unit, and the weights alone took
// 39 of the 85 us of a 512 x 2048 x 8192 gate/up launch.
template <int FMT, int NMAT, int R, int C>
__global__ __launch_bounds__(512, 2) void rows32_kernel(RowsArgs a) {
    extern __shared__ __align__(16) float s_part[];
    constexpr bool Q4 = FMT == FMT_Q4_0F || FMT == FMT_Q4_0;
    constexpr int NCOL = 32 * NMAT * C, NCH = (5 * NCOL + 63) / 64;   // column rows, 16-byte chunks per lane
    __shared__ __align__(16) u32x4 s_w[Q4 ? 8 : 1][Q4 ? 64 * NCH : 1];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int fr = lane & 31, f = lane >> 5;
    Tile t;
    if (!t.find(a, 2 * R)) return;
    const int wn = wave % a.NW, wk = wave / a.NW;
    const int n0 = (t.bx * a.NW + wn) * 32 * C, N = t.N;
    const int K = a.K, nss = a.nks >> 2, mtiles = (a.M + 15) >> 4;
    int col[C];
#pragma unroll
    for (int j = 0; j < C; j++) col[j] = n0 + 32 * j + fr < N ? n0 + 32 * j + fr : 0;
    f32x16 acc[NMAT][R][C];
#pragma unroll
    for (int m = 0; m < NMAT; m++)
#pragma unroll
        for (int i = 0; i < R; i++)
#pragma unroll
            for (int j = 0; j < C; j++)
#pragma unroll
                for (int e = 0; e < 16; e++) acc[m][i][j][e] = 0.f;
    typename std::conditional<Q4, char, WRaw32<Q4 ? FMT_Q2_K : FMT>>::type raw[NMAT][C];
    // Q4: chunk i of this lane is bytes 16 c .. of column row q / 5, q = 64 i + lane, c = q % 5
    constexpr int BB = FMT == FMT_Q4_0F ? 20 : 18;
    const int nb = K >> 5;
    u32x4 ch[Q4 ? NCH : 1];
    // the tile's matrices from their first column (4-byte aligned down), the
    // chunk's offset there at step 0 and the last one that stays inside the
    // matrix (a tile's columns are far below 2 GB)
    const int64_t tile0 = ((int64_t)n0 * nb * BB) & ~(int64_t)3;
    int co[Q4 ? NCH : 1];
    const int clast = Q4 ? (int)min((int64_t)N * nb * BB - 16 - tile0, (int64_t)0x7FFFFFFF) : 0;
    const uint8_t* const wt[2] = {t.w + tile0, NMAT == 2 ? t.w2 + tile0 : nullptr};
    auto chunk_m = [&](int i) { return NMAT == 2 && min(64 * i + lane, 5 * NCOL - 1) >= 5 * 32 * C; };
    if constexpr (Q4) {
#pragma unroll
        for (int i = 0; i < NCH; i++) {
            const int q = min(64 * i + lane, 5 * NCOL - 1), cr = q / 5, c = q - 5 * cr;
            const int n = min(n0 + cr % (32 * C), N - 1);
            co[i] = (int)((((int64_t)n * nb * BB) & ~(int64_t)3) - tile0) + 16 * c;
        }
    }
    auto load_w = [&](int ss) {
        if constexpr (Q4) {
#pragma unroll
            for (int i = 0; i < NCH; i++) ch[i] = gld4((chunk_m(i) ? wt[1] : wt[0]) + min(co[i] + ss * (4 * BB), clast));
        } else {
#pragma unroll
            for (int m = 0; m < NMAT; m++)
#pragma unroll
                for (int j = 0; j < C; j++) w_load32<FMT>(m ? t.w2 : t.w, col[j], K, ss, f, raw[m][j]);
        }
    };
    // fragment of 32-row tile i, 16-value half h, part p of a 32-value step:
    // 16-row tile 2 i + (row / 16), lane row 2 h + f of its 64-unit chunk
    const int lu = (fr & 15) + 16 * f;
    constexpr bool PAGE = FMT == FMT_Q2_K;          // one scale per 128-value step
    f32x16 pd[PAGE ? NMAT : 1][PAGE ? R : 1][PAGE ? C : 1];
    // the products of step st (32 values) of a 128-value step for column tile j
    // of matrix m: rows x[half][row tile][part]
    auto mul = [&](const WStep32<FMT>& w, const bf16x8 (&x)[2][R][kParts], int st, int m, int j) {
        f32x16 d[R];
        const bf16x8 b[2] = {w.frag(st, 0), w.frag(st, 1)};
        // smallest parts first, of all 32 values: the sum is rounded at its full size twice
#pragma unroll
        for (int p = kParts - 1; p >= 0; p--)
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int i = 0; i < R; i++) {
                    f32x16 c;
                    if (h == 0 && p == kParts - 1) {
                        if (PAGE && st > 0) c = pd[PAGE ? m : 0][PAGE ? i : 0][PAGE ? j : 0];
                        else {
#pragma unroll
                            for (int e = 0; e < 16; e++) c[e] = 0.f;
                        }
                    } else {
                        c = d[i];
                    }
                    d[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[h][i][p], b[h], c, 0, 0, 0);
                }
#pragma unroll
        for (int i = 0; i < R; i++) {
            if constexpr (PAGE) pd[m][i][j] = d[i];
            if (!PAGE || st == 3) {
                const float sc = w.sc[PAGE ? 0 : st];
#pragma unroll
                for (int e = 0; e < 16; e++) acc[m][i][j][e] = fmaf(sc, d[i][e], acc[m][i][j][e]);
            }
            // consumed here: left alone, the compiler defers the scale
            // products of a whole step and spills
            if constexpr (PAGE) asm volatile("" : "+v"(pd[m][i][j]));
            else asm volatile("" : "+v"(acc[m][i][j]));
        }
    };
    bool edge = false;                              // a chunk of this wave ends past the matrix in the last step
    if constexpr (Q4) {
#pragma unroll
        for (int i = 0; i < NCH; i++) edge |= co[i] + (nss - 1) * (4 * BB) > clast;
        edge = __any(edge);
    }
    auto take = [&](WStep32<FMT> (&ws)[NMAT][C], int ss) {
        if constexpr (Q4) {
            u32x4* wb = s_w[wave];
            if (!edge || ss < nss - 1) {
#pragma unroll
                for (int i = 0; i < NCH; i++) wb[64 * i + lane] = ch[i];
            } else {
                // chunks that were pulled back into the matrix go where their bytes
                // belong (over the chunk before, with the same bytes; a step has
                // one block at least, so never before the row's first)
#pragma unroll
                for (int i = 0; i < NCH; i++) {
                    const int back = co[i] + ss * (4 * BB) - clast;
                    u16_any* d = (u16_any*)(wb + 64 * i + lane) - (back > 0 ? back / 2 : 0);   // (18-byte blocks: an even count)
                    const uint32_t v[4] = {ch[i].x, ch[i].y, ch[i].z, ch[i].w};
#pragma unroll
                    for (int k = 0; k < 4; k++) { d[2 * k] = (uint16_t)v[k]; d[2 * k + 1] = (uint16_t)(v[k] >> 16); }
                }
            }
            wave_fence();
#pragma unroll
            for (int m = 0; m < NMAT; m++)
#pragma unroll
                for (int j = 0; j < C; j++) {
                    // a row that starts two bytes past a dword (Q4_0, odd n nb): its blocks shift by two
                    const u32_any* r = (const u32_any*)wb + 20 * (32 * (m * C + j) + fr);
                    const int lead = FMT == FMT_Q4_0 ? 2 * ((col[j] & nb) & 1) : 0;
                    uint32_t d[2][5];
                    const bool odd = FMT == FMT_Q4_0 && ((lead + BB * f) & 2);
#pragma unroll
                    for (int b = 0; b < 2; b++)
#pragma unroll
                        for (int i = 0; i < 5; i++) d[b][i] = r[min((lead + BB * (2 * b + f)) / 4 + i, 19)];
                    ws[m][j].take_q4(d, odd);
                    if (4 * ss + 4 > nb) {          // blocks past the row: x is zero there, their bytes may be anything
#pragma unroll
                        for (int b = 0; b < 4; b++)
                            if (4 * ss + b >= nb) ws[m][j].sc[b] = 0.f;
                    }
                }
            wave_fence();
        } else {
#pragma unroll
            for (int m = 0; m < NMAT; m++)
#pragma unroll
                for (int j = 0; j < C; j++) ws[m][j].take(raw[m][j]);
        }
    };
    {
        const bf16x8* ap[R];
#pragma unroll
        for (int i = 0; i < R; i++) ap[i] = (const bf16x8*)a.xp + (int64_t)min(t.r16 + 2 * i + (fr >> 4), mtiles - 1) * a.nks * kStep + lu;
        bf16x8 af[2][2][R][kParts];                 // two 32-value steps, by halves
        auto load_a = [&](bf16x8 (&x)[2][R][kParts], int ks) {
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int i = 0; i < R; i++)
#pragma unroll
                    for (int p = 0; p < kParts; p++) x[h][i][p] = gld(ap[i] + (int64_t)ks * kStep + 64 * p + 32 * h);
        };
        if (wk < nss) {
            load_w(wk);
            load_a(af[0], 4 * wk);
        }
        for (int ss = wk; ss < nss; ss += a.KW) {
            const int sn = ss + a.KW < nss ? ss + a.KW : ss;   // the last step loads itself again
            WStep32<FMT> ws[NMAT][C];
            take(ws, ss);
#pragma unroll
            for (int st = 0; st < 4; st++) {
                load_a(af[(st & 1) ^ 1], st < 3 ? 4 * ss + st + 1 : 4 * sn);
                if (st == 0) load_w(sn);
                __builtin_amdgcn_sched_barrier(0);  // issued before this step's products
#pragma unroll
                for (int m = 0; m < NMAT; m++)
#pragma unroll
                    for (int j = 0; j < C; j++) mul(ws[m][j], af[st & 1], st, m, j);
            }
        }
    }
    if constexpr (FMT == FMT_Q2_K || FMT == FMT_Q2_S) {
        for (int g2 = wk; g2 < 2 * a.ngw; g2 += a.KW) {   // 16 groups: half a window
            bf16x8 xg[R][3];
#pragma unroll
            for (int i = 0; i < R; i++) {
                const bf16x8* gp = (const bf16x8*)a.xg + ((int64_t)min(t.r16 + 2 * i + (fr >> 4), mtiles - 1) * a.ngw + (g2 >> 1)) * 192 +
                                   lu + 32 * (g2 & 1);
#pragma unroll
                for (int p = 0; p < 3; p++) xg[i][p] = gld(gp + 64 * p);
            }
#pragma unroll
            for (int m = 0; m < NMAT; m++)
#pragma unroll
                for (int j = 0; j < C; j++) {
                    bf16x8 hi, lo;
                    min_frag<FMT>(m ? t.w2 : t.w, col[j], K, 16 * g2 + 8 * f, hi, lo);
#pragma unroll
                    for (int i = 0; i < R; i++) {
                        f32x16 d = acc[m][i][j];
                        d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xg[i][2], hi, d, 0, 0, 0);
                        d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xg[i][1], lo, d, 0, 0, 0);
                        d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xg[i][1], hi, d, 0, 0, 0);
                        d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xg[i][0], lo, d, 0, 0, 0);
                        acc[m][i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xg[i][0], hi, d, 0, 0, 0);
                    }
                }
        }
    }
    {
        // the KW partial tiles, halved per round (as rows16_kernel)
        f32x4* sp = (f32x4*)s_part;
        constexpr int NR = NMAT * R * C * 4;
        for (int h = a.KW >> 1; h >= 1; h >>= 1) {
            f32x4* d = sp + (int64_t)((wk >= h ? wk - h : wk) * a.NW + wn) * NR * 64 + lane;
            if (wk >= h && wk < 2 * h) {
#pragma unroll
                for (int m = 0; m < NMAT; m++)
#pragma unroll
                    for (int i = 0; i < R; i++)
#pragma unroll
                        for (int j = 0; j < C; j++)
#pragma unroll
                            for (int q = 0; q < 4; q++)
                                d[(((m * R + i) * C + j) * 4 + q) * 64] = f32x4{acc[m][i][j][4 * q], acc[m][i][j][4 * q + 1], acc[m][i][j][4 * q + 2], acc[m][i][j][4 * q + 3]};
            }
            __syncthreads();
            if (wk < h) {
#pragma unroll
                for (int m = 0; m < NMAT; m++)
#pragma unroll
                    for (int i = 0; i < R; i++)
#pragma unroll
                        for (int j = 0; j < C; j++)
#pragma unroll
                            for (int q = 0; q < 4; q++) {
                                const f32x4 v = d[(((m * R + i) * C + j) * 4 + q) * 64];
#pragma unroll
                                for (int e = 0; e < 4; e++) acc[m][i][j][4 * q + e] += v[e];
                            }
            }
            __syncthreads();
        }
        if (wk > 0) return;
    }
    constexpr bool Q2 = FMT == FMT_Q2_K || FMT == FMT_Q2_S;
    bool inf = false;                               // rows of inf_rows
    // result element e of lane l: row 8 (e / 4) + 4 f + e % 4, column l % 32
#pragma unroll
    for (int i = 0; i < R; i++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int r0 = t.r16 * 16 + 32 * i + 8 * q + 4 * f;
            if (r0 >= t.mend) continue;
            const f32x4 sc = gld((const f32x4*)(a.xs + r0));
#pragma unroll
            for (int j = 0; j < C; j++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    if (Q2 && sc[e] < 0.f) inf |= r0 + e < t.mend;
                    else finish<NMAT>(a, t, r0 + e, n0 + 32 * j + fr, acc[0][i][j][4 * q + e] * sc[e], acc[NMAT - 1][i][j][4 * q + e] * sc[e]);
                }
        }
    if (Q2 && __any(inf)) {
#pragma unroll 1
        for (int j = 0; j < C; j++) inf_rows<NMAT, 32>(a, t, t.r16 * 16, 32 * R, n0 + 32 * j + fr, f);
    }
}

template <int FMT, int NMAT, int MI>
int launch16(const RowsArgs& a, hipStream_t st) {
    const size_t lds = a.KW > 1 ? (size_t)(a.KW / 2) * a.NW * NMAT * MI * 1024 : 0;
    hipLaunchKernelGGL((rows16_kernel<FMT, NMAT, MI>), dim3(8 * a.mpp * a.npp), dim3(64 * a.NW * a.KW), lds, st, a);
    return hipGetLastError() == hipSuccess ? RINA_OK : RINA_ERR_HIP;
}

template <int FMT, int NMAT, int R, int C>
int launch32(const RowsArgs& a, hipStream_t st) {
    const size_t lds = a.KW > 1 ? (size_t)(a.KW / 2) * a.NW * NMAT * R * C * 4096 : 0;
    hipLaunchKernelGGL((rows32_kernel<FMT, NMAT, R, C>), dim3(8 * a.mpp * a.npp), dim3(64 * a.NW * a.KW), lds, st, a);
    return hipGetLastError() == hipSuccess ? RINA_OK : RINA_ERR_HIP;
}

// rt: 0 / 1: one or two 16-row tiles (rows16_kernel), 2: 64 rows (rows32_kernel)
template <int FMT>
int launch_fmt(const RowsArgs& a, int nmat, int rt, int ct, hipStream_t st) {
    if (nmat == 2) return rt == 0 ? launch16<FMT, 2, 1>(a, st) : rt == 1 ? launch16<FMT, 2, 2>(a, st) : launch32<FMT, 2, 2, 1>(a, st);
    if (rt < 2) return rt == 0 ? launch16<FMT, 1, 1>(a, st) : launch16<FMT, 1, 2>(a, st);
    return ct == 1 ? launch32<FMT, 1, 2, 1>(a, st) : launch32<FMT, 1, 2, 2>(a, st);
}

// ---- fp32 weights: v_mfma_f32_16x16x4f32 tiles ----
// A wave owns MI 16-row tiles x NJ 16-column tiles (per matrix) of its K
// slice (32-value chunks, interleaved over the KW waves); rows and weights
// come straight from memory, a lane holding 8 consecutive values of its row
// and column per chunk (any order of K does, as long as both agree).  Sums are
// kept per 256 values and added up: the error of one 2048-long chain, as a
// serial product has it, halves.  NT: the weights are read once (one row
// tile), streamed past the caches.
// LM head 128256 x 2048: bound by the weight stream up to 32 rows (1.05 GB),
// beyond by the fp32 matrix cores.
template <int NMAT, int MI, int NJ, bool NT>
__global__ __launch_bounds__(512, 2) void rows_f32_kernel(RowsArgs a) {
    extern __shared__ __align__(16) float s_part[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int fr = lane & 15, g = lane >> 4;
    Tile t;
    if (!t.find(a, MI)) return;
    const int wn = wave % a.NW, wk = wave / a.NW;
    const int n0 = (t.bx * a.NW + wn) * 16 * NJ, N = t.N, K = a.K, nch = (K + 31) >> 5;
    const float* xr[MI];
    const float* wr[NMAT][NJ];
#pragma unroll
    for (int i = 0; i < MI; i++) xr[i] = (const float*)a.xp + (int64_t)min((t.r16 + i) * 16 + fr, a.M - 1) * K;
#pragma unroll
    for (int m = 0; m < NMAT; m++)
#pragma unroll
        for (int j = 0; j < NJ; j++) wr[m][j] = (const float*)(m ? t.w2 : t.w) + (int64_t)min(n0 + 16 * j + fr, N - 1) * K;
    f32x4 tot[NMAT][MI][NJ], acc[NMAT][MI][NJ];
    const f32x4 z4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int m = 0; m < NMAT; m++)
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int j = 0; j < NJ; j++) tot[m][i][j] = acc[m][i][j] = z4;
    struct Chunk {
        f32x4 x[MI][2], w[NMAT][NJ][2];
    };
    // chunk c: values 32 c + 8 g .. + 7 (K % 4 == 0; past K: zeros)
    auto load = [&](int c, Chunk& r) {
        const int k = 32 * c + 8 * g;
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const bool on = k + 4 * u < K;
            const int kk = on ? k + 4 * u : 0;
#pragma unroll
            for (int i = 0; i < MI; i++) {
                r.x[i][u] = gld((const f32x4*)(xr[i] + kk));
                if (!on) r.x[i][u] = z4;
            }
#pragma unroll
            for (int m = 0; m < NMAT; m++)
#pragma unroll
                for (int j = 0; j < NJ; j++) {
                    r.w[m][j][u] = NT ? gld_nt((const f32x4*)(wr[m][j] + kk)) : gld((const f32x4*)(wr[m][j] + kk));
                    if (!on) r.w[m][j][u] = z4;
                }
        }
    };
    auto mul = [&](const Chunk& r) {
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int m = 0; m < NMAT; m++)
#pragma unroll
                    for (int j = 0; j < NJ; j++)
#pragma unroll
                        for (int i = 0; i < MI; i++)
                            acc[m][i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(r.x[i][u][e], r.w[m][j][u][e], acc[m][i][j], 0, 0, 0);
    };
    auto flush = [&]() {
#pragma unroll
        for (int m = 0; m < NMAT; m++)
#pragma unroll
            for (int i = 0; i < MI; i++)
#pragma unroll
                for (int j = 0; j < NJ; j++) {
                    tot[m][i][j] += acc[m][i][j];
                    acc[m][i][j] = z4;
                }
    };
    // two chunks in flight ahead of the one that is multiplied
    Chunk c0, c1;
    const int last = wk < nch ? wk + (nch - 1 - wk) / a.KW * a.KW : 0;   // past the end: the last chunk again, not multiplied
    load(min(wk, last), c0);
    load(min(wk + a.KW, last), c1);
    int n = 0;
    for (int c = wk; c < nch; c += 2 * a.KW) {
        mul(c0);
        load(min(c + 2 * a.KW, last), c0);
        __builtin_amdgcn_sched_barrier(0);
        if (c + a.KW < nch) mul(c1);
        load(min(c + 3 * a.KW, last), c1);
        __builtin_amdgcn_sched_barrier(0);
        n += 2;
        if ((n & 7) == 0) flush();
    }
    flush();
    f32x4* sp = (f32x4*)s_part;
    constexpr int NR = NMAT * MI * NJ;
    for (int h = a.KW >> 1; h >= 1; h >>= 1) {
        f32x4* d = sp + (int64_t)((wk >= h ? wk - h : wk) * a.NW + wn) * NR * 64 + lane;
        if (wk >= h && wk < 2 * h) {
#pragma unroll
            for (int m = 0; m < NMAT; m++)
#pragma unroll
                for (int i = 0; i < MI; i++)
#pragma unroll
                    for (int j = 0; j < NJ; j++) d[((m * MI + i) * NJ + j) * 64] = tot[m][i][j];
        }
        __syncthreads();
        if (wk < h) {
#pragma unroll
            for (int m = 0; m < NMAT; m++)
#pragma unroll
                for (int i = 0; i < MI; i++)
#pragma unroll
                    for (int j = 0; j < NJ; j++) tot[m][i][j] += d[((m * MI + i) * NJ + j) * 64];
        }
        __syncthreads();
    }
    if (wk > 0) return;
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int e = 0; e < 4; e++)
                finish<NMAT>(a, t, (t.r16 + i) * 16 + 4 * g + e, n0 + 16 * j + fr, tot[0][i][j][e], tot[NMAT - 1][i][j][e]);
}

template <int NMAT, int MI, int NJ>
int launch_f32(const RowsArgs& a, hipStream_t st) {
    const size_t lds = a.KW > 1 ? (size_t)(a.KW / 2) * a.NW * NMAT * MI * NJ * 1024 : 0;
    const dim3 grid(8 * a.mpp * a.npp), blk(64 * a.NW * a.KW);
    if (a.mt == 1) hipLaunchKernelGGL((rows_f32_kernel<NMAT, MI, NJ, true>), grid, blk, lds, st, a);
    else hipLaunchKernelGGL((rows_f32_kernel<NMAT, MI, NJ, false>), grid, blk, lds, st, a);
    return hipGetLastError() == hipSuccess ? RINA_OK : RINA_ERR_HIP;
}

// segments, tile counts and the XCD split of a launch: row tiles of tr rows,
// column tiles of bn, weight bytes per value; grouped: most row tiles in use
// (0: rows not grouped)
void plan_tiles(RowsArgs& a, const rina_linear_seg* segs, int nseg, int nmat, int tr, int bn, double wb, int grouped) {
    int t = 0;
    for (int s = 0; s < 3; s++) {
        const int ss = s < nseg ? s : 0;
        a.w[s] = (const uint8_t*)segs[ss].weight;
        a.y[s] = segs[ss].out;
        a.N[s] = segs[ss].N;
        a.t0[s] = s < nseg ? t : 1 << 30;
        if (s < nseg) t += (segs[s].N + bn - 1) / bn;
    }
    a.nseg = nseg;
    a.w2 = nmat == 2 ? (const uint8_t*)segs[0].weight2 : nullptr;
    a.mt = grouped ? grouped : (a.M + tr - 1) / tr;
    a.nt = t;
    // the split with the fewest bytes fetched by the 8 L2s: xb x + (8 / xb) W
    // (grouped rows: every group's weights on one XCD)
    const double xbytes = 4.0 * a.M * a.K, wbytes = (double)nmat * bn * t * a.K * wb;
    int best = 1;
    if (!grouped)
        for (int xb = 2; xb <= 8; xb *= 2)
            if (xb * xbytes + (8 / xb) * wbytes < best * xbytes + (8 / best) * wbytes) best = xb;
    a.xb = best;
    a.mpp = (a.mt + 8 / best - 1) / (8 / best);
    a.npp = (t + best - 1) / best;
}

size_t up256(size_t n) { return (n + 255) & ~(size_t)255; }

}  // namespace

bool rows_gemm_ok(int qt, int K) {
    return (qt == RINA_QT_Q4_0 || qt == RINA_QT_Q4_0F || qt == RINA_QT_GGML_Q2_K) && K % 32 == 0;
}

size_t rows_split_bytes(int qt, int rows, int K) {
    const size_t mt = (rows + 15) / 16, nks = (size_t)(K + 127) / 128 * 4, ngw = (K + 511) / 512;
    return up256(mt * nks * 16 * kStep) + up256(mt * 64) + (qt == RINA_QT_GGML_Q2_K ? mt * ngw * 3072 : 0);
}

int rows_split(int qt, const float* x, const int* src, const int* used, int rows, int K, int pro, const float* nw, float eps, void* buf,
               RowsX* out, hipStream_t st) {
    const int mt = (rows + 15) / 16;
    SplitXArgs a{};
    a.x = x; a.nw = nw; a.src = src; a.used = used; a.M = rows; a.K = K; a.pro = pro; a.eps = eps;
    a.nks = (K + 127) / 128 * 4;
    a.ngw = (K + 511) / 512;
    a.xp = (uint4*)buf;
    a.xs = (float*)((char*)buf + up256((size_t)mt * a.nks * 16 * kStep));
    a.xg = (uint16_t*)((char*)a.xs + up256((size_t)mt * 64));
    const dim3 grid(mt * 16 / kSplitRows), blk(256 * kSplitRows);
    const int nu = (K + 2047) / 2048;
#define X_SPLIT(Q) \
    do { if (nu <= 1) hipLaunchKernelGGL((x_split_kernel<Q, 1>), grid, blk, 0, st, a); \
         else if (nu <= 2) hipLaunchKernelGGL((x_split_kernel<Q, 2>), grid, blk, 0, st, a); \
         else if (nu <= 4) hipLaunchKernelGGL((x_split_kernel<Q, 4>), grid, blk, 0, st, a); \
         else if (nu <= 6) hipLaunchKernelGGL((x_split_kernel<Q, 6>), grid, blk, 0, st, a); \
         else hipLaunchKernelGGL((x_split_kernel<Q, 0>), grid, blk, 0, st, a); } while (0)
    if (qt == RINA_QT_GGML_Q2_K) X_SPLIT(true);
    else X_SPLIT(false);
#undef X_SPLIT
    out->xp = a.xp;
    out->xs = a.xs;
    out->xg = a.xg;
    out->rows = rows;
    out->K = K;
    return hipGetLastError() == hipSuccess ? RINA_OK : RINA_ERR_HIP;
}

int rows_gemm(const rina_linear_seg* segs, int nseg, int qt, const RowsX& x, int epi, const RowsPlan* pl, hipStream_t st) {
    const bool two = epi == RINA_EPI_SWIGLU;
    const int nmat = two ? 2 : 1;
    RowsArgs a{};
    a.xp = (const uint4*)x.xp; a.xs = x.xs; a.xg = (const uint4*)x.xg;
    a.M = x.rows; a.K = x.K; a.epi = epi;
    a.nks = (x.K + 127) / 128 * 4;
    a.ngw = (x.K + 511) / 512;
    a.plan = pl ? pl->plan : nullptr;
    a.stride = pl ? pl->stride : 0;
    const int nss = a.nks / 4;
    // row tiles of 16, 32 or 64 rows (rt 0, 1, 2); columns per wave: 16, or 32 ct
    // at 64 rows.  More than 32 rows take the 64-row tiles where these give every
    // SIMD a wave with K split as far as it goes (us 64-row / 32-row, Q4_0F): N
    // 2048, K 8192: 64 rows (512 waves) 58.0 / 38.8, 96 rows (1024) 58.7 / 59.2,
    // 160 rows 62 / 70; N 512, K 1024: 256 rows (256 waves) 15.9 / 11.7; N 8192 x 2,
    // K 2048: 33 rows (2048 waves) 29.3 / 30.4, 256 rows 70.7 / 88.9.
    const int64_t simds = 4LL * rina_num_cus();
    int64_t w64 = 0;
    for (int s = 0; s < nseg; s++) w64 += (segs[s].N + 31) / 32;
    w64 *= (x.rows + 63) / 64;
    for (int kw = 1; kw < 8 && nss >= 2 * kw; kw *= 2) w64 *= 2;
    const int rt = pl ? pl->rt : x.rows <= 16 ? 0 : x.rows <= 32 || w64 < simds ? 1 : 2;
    const int tr = 16 << rt, tc = rt < 2 ? 16 : 32;
    const int64_t mts = pl ? pl->tiles_est : (x.rows + tr - 1) / tr;
    auto tiles = [&](int ct) {
        int64_t t = 0;
        for (int s = 0; s < nseg; s++) t += (segs[s].N + tc * ct - 1) / (tc * ct);
        return t * mts;
    };
    // 64 columns per wave only where that leaves every SIMD a wave without
    // splitting K
    const int nj = nmat == 1 && rt == 2 && tiles(2) >= simds ? 2 : 1;
    // K slices until there are two waves per SIMD: each slice is also a shorter
    // chain of sums
    int kw = 1;
    while (kw < 8 && tiles(nj) * kw < 2 * simds && nss >= 2 * kw) kw *= 2;
    a.KW = kw;
    a.NW = kw >= 4 ? 1 : 4 / kw;
    const int BN = tc * nj * a.NW;
    plan_tiles(a, segs, nseg, nmat, tr, BN, qt == RINA_QT_Q4_0F ? 0.625 : qt == RINA_QT_GGML_Q2_K ? 84.0 / 256 : 0.5625, pl ? pl->tiles_max : 0);
    if (qt == RINA_QT_Q4_0) return launch_fmt<FMT_Q4_0>(a, nmat, rt, nj, st);
    if (qt == RINA_QT_Q4_0F) return launch_fmt<FMT_Q4_0F>(a, nmat, rt, nj, st);
    return x.K % 128 == 0 ? launch_fmt<FMT_Q2_K>(a, nmat, rt, nj, st) : launch_fmt<FMT_Q2_S>(a, nmat, rt, nj, st);
}

bool rows_f32_ok(const rina_linear_seg* segs, int nseg, const float* x, int K) {
    bool ok = K % 4 == 0 && (uintptr_t)x % 16 == 0;
    for (int s = 0; s < nseg; s++) ok = ok && (uintptr_t)segs[s].weight % 16 == 0 && (uintptr_t)segs[s].weight2 % 16 == 0;
    return ok;
}

int rows_f32(const rina_linear_seg* segs, int nseg, const float* x, int M, int K, int epi, hipStream_t st) {
    const int nmat = epi == RINA_EPI_SWIGLU ? 2 : 1;
    RowsArgs a{};
    a.xp = (const uint4*)x;
    a.M = M; a.K = K; a.epi = epi;
    // (row tiles, column tiles) per wave: 4 x 2, 2 x 4 or 1 x 4 by the row
    // count, smaller where that leaves SIMDs idle with K split over 8
    const int64_t simds = 4LL * rina_num_cus();
    int mi = M > 32 ? 4 : M > 16 ? 2 : 1, nj = (mi == 4 ? 2 : 4) / nmat;
    auto tiles = [&]() {
        int64_t t = 0;
        for (int s = 0; s < nseg; s++) t += (segs[s].N + 16 * nj - 1) / (16 * nj);
        return t * ((M + 16 * mi - 1) / (16 * mi));
    };
    if (tiles() * 8 < simds) { nj = 1; if (mi == 4) mi = 2; }
    if (mi == 2 && tiles() * 8 < simds) mi = 1;
    int kw = 1;
    while (kw < 8 && tiles() * kw < 2 * simds && K >= 256 * kw) kw *= 2;
    a.KW = kw;
    a.NW = kw >= 4 ? 1 : 4 / kw;
    plan_tiles(a, segs, nseg, nmat, 16 * mi, 16 * nj * a.NW, 4.0, 0);
    if (nmat == 2) {
        if (mi == 4) return launch_f32<2, 4, 1>(a, st);
        if (mi == 2) return nj == 1 ? launch_f32<2, 2, 1>(a, st) : launch_f32<2, 2, 2>(a, st);
        return nj == 1 ? launch_f32<2, 1, 1>(a, st) : launch_f32<2, 1, 2>(a, st);
    }
    if (mi == 4) return launch_f32<1, 4, 2>(a, st);
    if (mi == 2) return nj == 1 ? launch_f32<1, 2, 1>(a, st) : launch_f32<1, 2, 4>(a, st);
    return nj == 1 ? launch_f32<1, 1, 1>(a, st) : launch_f32<1, 1, 4>(a, st);
}
