// Products over 16 rows or more with Q4 weights in one launch, for short K:
// out[M, N] = x[M, K] . W[N, K]^T on the bf16 matrix cores
// (v_mfma_f32_16x16x32_bf16), the rows split on the way through LDS.
//
// Every x value is split exactly into three bf16 parts, x = h + m + l (8
// significant bits each: the two remainders are exact in fp32), and a weight
// value q - 7 is a small integer, exact in bf16, so the matrix cores form the
// exact products of the fp32 x with the integer weights and sum them in fp32.
// Per 32-value block and 16 x 16 tile three products (l, m, h into one
// accumulator), then one fp32 fma with the block scale of the tile column.
// Tiles are BM x 32 WN with 2 WN waves (two down the rows, WN across, each wave
// 16 MI rows x 32 columns), so one split of an x tile serves 32 WN columns.  LDS
// rows of (32 KB + 8) bf16 keep the 16-byte fragment reads of 16 rows on
// distinct banks.  Fragment layout (16x16x32): lane l holds A[l % 16][8 (l / 16)
// .. + 7], B[8 (l / 16) .. + 7][l % 16] and D[4 (l / 16) + e][l % 16].
//
// Splitting the rows once in a launch of their own (gemm.hip) costs that launch
// and its round trip, which a short K does not win back, and every wave there
// loads its row fragments itself: see rows_bf3_ok for where the line lies.
#include "rina_common.hpp"
#include "rows_gemm.hpp"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float silu_mul(float g, float u) { return g / (1.0f + expf(-g)) * u; }

// the high halves of two fp32 bit patterns as one dword of two bf16 (a's in
// the low half)
__device__ __forceinline__ uint32_t hi16_pair(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }

// x0, x1 split into three bf16 parts each, x = h + m + l: h is x cut to its
// top 8 significant bits, m the remainder cut the same way, l the rest; packed
// as two-value dwords.  Exact for |x| >= 2^-103 and for 0, where both remainders
// are normal fp32 values.  INF: infinities stay themselves with nothing left
// (inf - inf is NaN).
template <bool INF>
__device__ __forceinline__ void split3_pair(float x0, float x1, uint32_t& ph, uint32_t& pm, uint32_t& pl) {
    const uint32_t u0 = __float_as_uint(x0), u1 = __float_as_uint(x1);
    ph = hi16_pair(u0, u1);
    float r0 = x0 - __uint_as_float(u0 & 0xFFFF0000u), r1 = x1 - __uint_as_float(u1 & 0xFFFF0000u);
    if (INF) {
        r0 = fabsf(x0) == INFINITY ? 0.f : r0;
        r1 = fabsf(x1) == INFINITY ? 0.f : r1;
    }
    const uint32_t v0 = __float_as_uint(r0), v1 = __float_as_uint(r1);
    pm = hi16_pair(v0, v1);
    const float s0 = r0 - __uint_as_float(v0 & 0xFFFF0000u), s1 = r1 - __uint_as_float(v1 & 0xFFFF0000u);
    pl = hi16_pair(__float_as_uint(s0), __float_as_uint(s1));
}

// Up to 3 weight segments sharing x (q / k / v) in one launch: column tiles
// t0[s] .. of segment s, in order.
// XCD-aware tile order: workgroups go to the 8 XCDs round-robin in linear
// order, so workgroup id serves XCD id % 8.  The x rows are split into 8 / xb
// parts and the weight columns into xb parts; XCD x takes row tiles of part
// x / xb and column tiles of part x % xb (the host picks the split with the
// fewest bytes fetched by the eight L2s).
struct Bf3Args {
    const float* x;
    const uint8_t* w[3];
    const uint8_t* w2;
    float* y[3];
    int N[3];
    int t0[3];
    int nseg, M, K, epi;
    int mt, nt;                  // row tiles, column tiles
    int xb;                      // weight parts
    int mpp, npp;                // row tiles, column tiles per part
};

template <bool Q4F, int NMAT, int BM, int WN>
__global__ __launch_bounds__(128 * WN) void gemm_bf3_kernel(Bf3Args ma) {
    constexpr int BB = Q4F ? 20 : 18;
    constexpr int MI = BM / 32;                    // MFMA tiles per wave along M
    // 32-value blocks per LDS stage: four cut the barriers of the one-matrix
    // launches (two at 64 rows, whose LDS would otherwise hold one
    // workgroup per CU); the paired SwiGLU tile keeps one (its registers
    // would cut occupancy to 3 waves per SIMD)
    constexpr int KB = NMAT == 2 ? 1 : BM == 64 ? 2 : 4;
    constexpr int LD = 32 * KB + 8;
    // WN waves across the tile's columns (32 each) and two down its rows
    constexpr int BN = 32 * WN, NT = 128 * WN;
    __shared__ __align__(16) uint16_t xs[3][BM][LD];
    __shared__ __align__(16) uint16_t ws[NMAT][BN][LD];
    __shared__ float wsc_s[NMAT][KB][BN];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int xcd = blockIdx.x & 7, k = blockIdx.x >> 3;
    const int mm = k / ma.npp, nn = k - mm * ma.npp;
    const int by = (xcd / ma.xb) * ma.mpp + mm, bx = (xcd % ma.xb) * ma.npp + nn;
    if (mm >= ma.mpp || by >= ma.mt || bx >= ma.nt) return;   // padding of the split
    // this workgroup's segment (wave-uniform selects, no indexed argument reads)
    const int sg = (ma.nseg > 1 && bx >= ma.t0[1]) + (ma.nseg > 2 && bx >= ma.t0[2]);
    struct {
        const uint8_t *w, *w2;
        const float* x;
        float* y;
        int M, N, K, epi;
    } a;
    a.w2 = ma.w2; a.x = ma.x; a.M = ma.M; a.K = ma.K; a.epi = ma.epi;
    a.w = sg == 0 ? ma.w[0] : sg == 1 ? ma.w[1] : ma.w[2];
    a.y = sg == 0 ? ma.y[0] : sg == 1 ? ma.y[1] : ma.y[2];
    a.N = sg == 0 ? ma.N[0] : sg == 1 ? ma.N[1] : ma.N[2];
    const int tb = sg == 0 ? ma.t0[0] : sg == 1 ? ma.t0[1] : ma.t0[2];
    const int m0 = by * BM, n0 = (bx - tb) * BN;
    const int nb = a.K / 32, nst = (nb + KB - 1) / KB;
    // x staging: every thread splits XV values of one row per block (XT
    // threads per row), so the split work is spread over all the waves;
    // weight staging: thread tid takes values 8 sq .. 8 sq + 7 of column sr
    constexpr int XV = BM * 32 / NT, XT = 32 / XV;
    const int xsr = tid / XT, xsq = tid % XT;
    const int sr = tid >> 2, sq = tid & 3;
    const bool xok = m0 + xsr < a.M, wok = n0 + sr < a.N;
    const float* xrow = a.x + (int64_t)(xok ? m0 + xsr : 0) * a.K + XV * xsq;
    const int64_t wrow = (int64_t)(wok ? n0 + sr : 0) * nb * BB;
    // register sets holding one stage's loads each; with two, a stage's loads
    // are issued two stages before they are stored to LDS
    struct Stage {
        float xr[KB][XV];
        uint32_t wsc[KB][NMAT], wnb[KB][NMAT];
    };
    Stage r0, r1;
    // stage st: blocks KB st .. KB st + KB - 1 (past nb: block nb - 1 again,
    // stored as zeros)
    auto load_stage = [&](Stage& r, int st) {
#pragma unroll
        for (int kb = 0; kb < KB; kb++) {
            const int b = min(KB * st + kb, nb - 1);
            if constexpr (XV >= 4) {
                const f32x4* xp = (const f32x4*)(xrow + 32 * b);
#pragma unroll
                for (int v = 0; v < XV / 4; v++) {
                    const f32x4 t = gld(xp + v);
                    r.xr[kb][4 * v] = t.x; r.xr[kb][4 * v + 1] = t.y; r.xr[kb][4 * v + 2] = t.z; r.xr[kb][4 * v + 3] = t.w;
                }
            } else {
                const f32x2 t = gld((const f32x2*)(xrow + 32 * b));
                r.xr[kb][0] = t.x; r.xr[kb][1] = t.y;
            }
#pragma unroll
            for (int m = 0; m < NMAT; m++) {
                const uint8_t* bp = (m ? a.w2 : a.w) + wrow + (int64_t)b * BB;
                if constexpr (Q4F) {
                    r.wsc[kb][m] = gld((const uint32_t*)bp);
                    r.wnb[kb][m] = gld((const uint32_t*)(bp + 4 + 4 * sq));
                } else {
                    r.wsc[kb][m] = gld((const uint16_t*)bp);
                    r.wnb[kb][m] = (uint32_t)gld((const uint16_t*)(bp + 2 + 4 * sq)) |
                                 ((uint32_t)gld((const uint16_t*)(bp + 4 + 4 * sq)) << 16);
                }
            }
        }
    };
    // value 8 sq + t of a block is nibble t of wnb (byte t / 2, low nibble for even t)
    auto store_stage = [&](const Stage& r, int st) {
#pragma unroll
        for (int kb = 0; kb < KB; kb++) {
            const bool bok = KB * st + kb < nb;
            {
                float xv[XV];
#pragma unroll
                for (int v = 0; v < XV; v++) xv[v] = r.xr[kb][v];
                const bool on = xok && bok;
                uint32_t ph[XV / 2], pm[XV / 2], pl[XV / 2];
                float mx = 0.f;
#pragma unroll
                for (int t = 0; t < XV; t += 2) mx = fmaxf(mx, fmaxf(fabsf(xv[t]), fabsf(xv[t + 1])));
                if (__builtin_expect(!__any(mx == INFINITY), 1)) {
#pragma unroll
                    for (int t = 0; t < XV; t += 2)
                        split3_pair<false>(on ? xv[t] : 0.f, on ? xv[t + 1] : 0.f, ph[t >> 1], pm[t >> 1], pl[t >> 1]);
                } else {
#pragma unroll
                    for (int t = 0; t < XV; t += 2)
                        split3_pair<true>(on ? xv[t] : 0.f, on ? xv[t + 1] : 0.f, ph[t >> 1], pm[t >> 1], pl[t >> 1]);
                }
                uint16_t* d0 = &xs[0][xsr][32 * kb + XV * xsq];
                uint16_t* d1 = &xs[1][xsr][32 * kb + XV * xsq];
                uint16_t* d2 = &xs[2][xsr][32 * kb + XV * xsq];
                if constexpr (XV == 8) {
                    *(u32x4*)d0 = u32x4{ph[0], ph[1], ph[2], ph[3]};
                    *(u32x4*)d1 = u32x4{pm[0], pm[1], pm[2], pm[3]};
                    *(u32x4*)d2 = u32x4{pl[0], pl[1], pl[2], pl[3]};
                } else if constexpr (XV == 2) {
                    *(uint32_t*)d0 = ph[0];
                    *(uint32_t*)d1 = pm[0];
                    *(uint32_t*)d2 = pl[0];
                } else {
                    *(u32x2*)d0 = u32x2{ph[0], ph[1]};
                    *(u32x2*)d1 = u32x2{pm[0], pm[1]};
                    *(u32x2*)d2 = u32x2{pl[0], pl[1]};
                }
            }
#pragma unroll
            for (int m = 0; m < NMAT; m++) {
                // q - 7 as bf16, a small integer (exact): nibble t of wnb is
                // byte t / 2 of lo (even t) or hi (odd t)
                const uint32_t lo = and_opaque(r.wnb[kb][m], 0x0F0F0F0Fu), hi = and_opaque(r.wnb[kb][m] >> 4, 0x0F0F0F0Fu);
                uint32_t pw[4];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float f0 = (float)((lo >> (8 * j)) & 0xFF) - 7.0f, f1 = (float)((hi >> (8 * j)) & 0xFF) - 7.0f;
                    pw[j] = wok && bok ? hi16_pair(__float_as_uint(f0), __float_as_uint(f1)) : 0u;
                }
                *(u32x4*)&ws[m][sr][32 * kb + 8 * sq] = u32x4{pw[0], pw[1], pw[2], pw[3]};
                if (sq == 0) {
                    const float sc = Q4F ? __uint_as_float(r.wsc[kb][m]) : f16_to_f32((uint16_t)r.wsc[kb][m]);
                    wsc_s[m][kb][sr] = wok && bok ? sc : 0.f;
                }
            }
        }
    };
    const int wm = (wave / WN) * 16 * MI, wn = (wave % WN) * 32;
    const int fr = lane & 15, fk = lane >> 4;
    f32x4 acc[NMAT][MI][2];
#pragma unroll
    for (int m = 0; m < NMAT; m++)
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int j = 0; j < 2; j++) acc[m][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto compute_stage = [&]() {
#pragma unroll
        for (int kb = 0; kb < KB; kb++) {
            bf16x8 af[3][MI];
#pragma unroll
            for (int p = 0; p < 3; p++)
#pragma unroll
                for (int i = 0; i < MI; i++) af[p][i] = *(const bf16x8*)&xs[p][wm + 16 * i + fr][32 * kb + 8 * fk];
#pragma unroll
            for (int m = 0; m < NMAT; m++)
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const bf16x8 bf = *(const bf16x8*)&ws[m][wn + 16 * j + fr][32 * kb + 8 * fk];
                    const float sc = wsc_s[m][kb][wn + 16 * j + fr];
#pragma unroll
                    for (int i = 0; i < MI; i++) {
                        f32x4 d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[2][i], bf, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                        d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[1][i], bf, d, 0, 0, 0);
                        d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[0][i], bf, d, 0, 0, 0);
#pragma unroll
                        for (int e = 0; e < 4; e++) acc[m][i][j][e] = fmaf(sc, d[e], acc[m][i][j][e]);
                    }
                }
        }
    };
    load_stage(r0, 0);
    if constexpr (NMAT == 1) {
        // stages in pairs, unconditionally: with nst odd the last pair's
        // second stage lies past nb, is stored as zeros and adds sc 0 times d 0
        load_stage(r1, 1);
        for (int st = 0; st < nst; st += 2) {
            __syncthreads();                       // the previous stage's fragments are read
            store_stage(r0, st);
            __syncthreads();
            load_stage(r0, st + 2);
            compute_stage();
            __syncthreads();
            store_stage(r1, st + 1);
            __syncthreads();
            load_stage(r1, st + 3);
            compute_stage();
        }
    } else {
        // the paired SwiGLU tile keeps one register set (a second would cut
        // occupancy from 5 to 3 waves per SIMD, which costs it more)
        for (int st = 0; st < nst; st++) {
            __syncthreads();
            store_stage(r0, st);
            __syncthreads();
            load_stage(r0, st + 1);                // past the end: block nb - 1, not stored
            compute_stage();
        }
    }
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int row = m0 + wm + 16 * i + 4 * fk + e, col = n0 + wn + 16 * j + fr;
                if (row >= a.M || col >= a.N) continue;
                float* y = a.y + (int64_t)row * a.N + col;
                const float v0 = acc[0][i][j][e];
                if (NMAT == 2) *y = silu_mul(v0, acc[NMAT - 1][i][j][e]);
                else if (a.epi == RINA_EPI_ADD) *y = *y + v0;
                else *y = v0;
            }
}


template <bool Q4F, int NMAT>
void launch(const Bf3Args& a, bool half, bool wide, hipStream_t st) {
    const dim3 g(8 * a.mpp * a.npp);
    if (half && wide) hipLaunchKernelGGL((gemm_bf3_kernel<Q4F, NMAT, 32, 4>), g, dim3(512), 0, st, a);
    else if (half) hipLaunchKernelGGL((gemm_bf3_kernel<Q4F, NMAT, 32, 2>), g, dim3(256), 0, st, a);
    else if (wide) hipLaunchKernelGGL((gemm_bf3_kernel<Q4F, NMAT, 64, 4>), g, dim3(512), 0, st, a);
    else hipLaunchKernelGGL((gemm_bf3_kernel<Q4F, NMAT, 64, 2>), g, dim3(256), 0, st, a);
}

}  // namespace

// The line to gemm.hip (Q4_0F, us here / there).  One matrix: K 96 x 400 5.9 /
// 11, K 288 x 1000 9.1 / 9.8 (40 rows), 9.6 / 12.5 (512), K 512 x 2048 9.5 / 10.0
// (40), 10.8 / 14.9 (512), K 1024 x 512 16.6 / 11.3 (40).  Gate and up: K 512 x 2 x
// 1024 15.2 / 10.2 (40), 15.7 / 18.4 (512), x 8192 15.4 / 15.8 (40), 34.6 / 42.3
// (512); K 768 x 2 x 8192 24.7 / 24.9 (100), 48.5 / 56.1 (512); K 1024 x 2 x 8192 33.5
// / 28.4 (100), 57.4 / 58.7 (330), 62.7 / 68.6 (512); K
// 2048 x 2 x 8192 110 / 96 (330).  One K loop here, whose one chain of sums is less
// exact than the K slices there as K grows (error against 64 bits at K 1024 1.14e-7
// / 0.82e-7, at 512 0.85e-7 / 0.7 to 0.85e-7), so K 1024 and more go there.
bool rows_bf3_ok(const rina_linear_seg* segs, int nseg, int qt, const float* x, int M, int K, int epi) {
    if (M < 16 || (qt != RINA_QT_Q4_0 && qt != RINA_QT_Q4_0F) || K % 32 || (uintptr_t)x % 16) return false;
    const bool two = epi == RINA_EPI_SWIGLU;
    double n = 0;
    for (int s = 0; s < nseg; s++) n += segs[s].N;
    return K <= (two ? 320 : 512) || (two && K < 1024 && 2 * n * M >= 2.4 * K * (double)K);
}

int rows_bf3(const rina_linear_seg* segs, int nseg, int qt, const float* x, int M, int K, int epi, hipStream_t st) {
    Bf3Args a{};
    const bool two = epi == RINA_EPI_SWIGLU;
    a.x = x; a.w2 = two ? (const uint8_t*)segs[0].weight2 : nullptr;
    a.nseg = nseg; a.M = M; a.K = K; a.epi = epi;
    // 128-column tiles of eight waves (the x tile's split and staging then
    // serve twice the columns) when those tiles fill the CUs in whole rounds,
    // else 64-column tiles of four waves (q/k/v at M 512: 384 wide tiles would
    // leave half the CUs a second one)
    auto count = [&](int bn) {
        int t = 0;
        for (int s = 0; s < nseg; s++) t += (segs[s].N + bn - 1) / bn;
        return t;
    };
    const bool half = (int64_t)count(64) * ((M + 63) / 64) < 2LL * rina_num_cus();   // 32-row tiles: more workgroups in flight
    const int64_t mtiles = half ? (M + 31) / 32 : (M + 63) / 64;
    const bool wide = mtiles * count(128) % rina_num_cus() == 0;
    const int BN = wide ? 128 : 64;
    int tiles = 0;
    for (int s = 0; s < 3; s++) {
        const int ss = s < nseg ? s : 0;
        a.w[s] = (const uint8_t*)segs[ss].weight;
        a.y[s] = segs[ss].out;
        a.N[s] = segs[ss].N;
        a.t0[s] = s < nseg ? tiles : 1 << 30;
        if (s < nseg) tiles += (segs[s].N + BN - 1) / BN;
    }
    a.mt = (int)mtiles;
    a.nt = tiles;
    // bytes the 8 L2s fetch for a split of x into 8 / xb parts and the
    // weights into xb parts: xb * (x bytes) + (8 / xb) * (weight bytes)
    const double xbytes = 4.0 * M * K;
    const double wbytes = (two ? 2.0 : 1.0) * BN * (double)tiles * K * (qt == RINA_QT_Q4_0F ? 20.0 / 32 : 18.0 / 32);
    int best = 1;
    for (int xb = 2; xb <= 8; xb *= 2)
        if (xb * xbytes + (8 / xb) * wbytes < best * xbytes + (8 / best) * wbytes) best = xb;
    a.xb = best;
    a.mpp = (a.mt + 8 / best - 1) / (8 / best);
    a.npp = (tiles + best - 1) / best;
    if (qt == RINA_QT_Q4_0F) {
        if (two) launch<true, 2>(a, half, wide, st);
        else launch<true, 1>(a, half, wide, st);
    } else {
        if (two) launch<false, 2>(a, half, wide, st);
        else launch<false, 1>(a, half, wide, st);
    }
    return hipGetLastError() == hipSuccess ? RINA_OK : RINA_ERR_HIP;
}
