// Batched causal attention in f32 with its scores and probabilities written
// out: the six products and two softmax passes of the device tape
// (gpu_step/tape.rs:196-212, 349-372, 475-491; rows.rs:101-123, 295-357) in
// three launches.
//
// Per (window, head) problem z, Q, K, V the head-h column blocks of the fused
// [B T, 3 D] buffer, scale = hd^-1/2:
//   k_attn_rows<.., false>  S = Q K^T, P = softmax(scale S, causal), O = P V
//   k_attn_rows<.., true>   dP = dO V^T, dS = scale P (dP - rowsum(dP P)), dQ = dS K
//   k_attn_cols             dV = P^T dO, dK = dS^T Q
// Everything the separate products write is written: S, P, dP, dS in full
// (masked columns included), ctx and the three blocks of dqkv.  f32 throughout
// (v_mfma_f32_16x16x4_f32), the softmax arithmetic of k_softmax_fwd / _bwd.
//
// One workgroup (4 waves) owns 32 rows of S (or 32 columns, k_attn_cols) and
// streams the other operand in tiles of 64 (32) rows through LDS, the next tile
// in registers meanwhile.  The 32 x T block of S stays in LDS from the first
// product through the softmax into the second, which is what the separate
// launches pay for: each wrote and read T x T per problem, and their 200 x 80 x
// 200 products are three k-stages long, so that a launch was mostly first
// loads and stores.  In the first product the waves split the tile's columns,
// in the others the contraction (16 or 8 of the tile's rows each; the four
// partial results are added in wave order), so that any head width keeps them
// evenly busy.
//
// 96 problems of 200 x 80, us: 39 + 37 + 30 (forward, backward rows, columns)
// against 6 products of 21 to 24 and softmax passes of 12.5 and 10.5.  The
// matrix cores are busy a third of k_attn_rows' time; the rest is the softmax's
// arithmetic (about 2,500 VALU instructions a wave) and the chain of steps of a
// single round of workgroups (2.6 per CU, three fit).  Two tiles in flight
// instead of one: rows the same, columns 39 (registers); S, P and ds written
// between the products instead of inside their loops: 71 -> 43 (a load behind a
// store has to wait for it).
//
// LDS pitches of 4 floats over a multiple of 16 put the 16 rows of a 16-byte
// fragment read into 16 distinct bank groups, and the four k-lines of a 4-byte
// one 16 banks apart.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "lanes.h"

#pragma clang fp contract(off)

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

constexpr int THREADS = 256;
constexpr int RB = 32;       // rows (columns) of S per workgroup
constexpr int KT = 64;       // rows of a streamed tile
constexpr int T_MAX = 512;   // longest sequence (the S block in LDS)
constexpr int HD_MAX = 128;  // widest head

struct AttnArgs {
    const float *qkv, *dctx;
    float *s, *p, *dp, *ds, *ctx, *dqkv;
    int32_t h, t, hd, blocks;  // blocks of RB rows per problem
    float scale;
};

// The workgroup's problem and block: each XCD (workgroup ids go round robin
// over 8) gets a contiguous run, so the blocks of a problem share its L2.
__device__ __forceinline__ void place(int blocks, int64_t &z, int &blk) {
    int64_t lin = blockIdx.x;
    const int64_t total = gridDim.x;
    if (total % 8 == 0) lin = (lin % 8) * (total / 8) + lin / 8;
    z = lin / blocks;
    blk = (int)(lin % blocks);
}

// A ROWS x W tile of a matrix (rows row0 .., columns col0 ..) from global memory
// to registers and on to LDS rows of PITCH floats; rows past nrows and columns
// past ncols are zero.  VEC: ncols and col0 are multiples of 4 (16-byte loads
// of 4-byte alignment, kept inside the row).
template <int ROWS, int W, int PITCH, bool VEC>
struct Tile {
    static constexpr int UNITS = ROWS * W / 4, PER = (UNITS + THREADS - 1) / THREADS;
    f32x4 r[PER];

    // The last units of a tile that is not whole threads are loaded twice.
    static __device__ __forceinline__ int unit(int i, int tid) {
        const int u = tid + THREADS * i;
        return UNITS % THREADS == 0 ? u : min(u, UNITS - 1);
    }

    __device__ __forceinline__ void load(const float *__restrict__ base, int64_t ld, int row0, int nrows, int col0,
                                         int ncols, int tid) {
#pragma unroll
        for (int i = 0; i < PER; i++) {
            const int u = unit(i, tid), row = row0 + u / (W / 4), c = col0 + 4 * (u % (W / 4));
            const float *src = base + (int64_t)min(row, nrows - 1) * ld;
            f32x4 v;
            if constexpr (VEC) {
                v = *reinterpret_cast<const f32x4u *>(src + min(c, ncols - 4));
                if (row >= nrows || c >= ncols) v = f32x4{0.f, 0.f, 0.f, 0.f};
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    v[e] = src[min(c + e, ncols - 1)];
                    if (row >= nrows || c + e >= ncols) v[e] = 0.f;
                }
            }
            r[i] = v;
        }
    }

    __device__ __forceinline__ void store(float *lds, int tid) const {
#pragma unroll
        for (int i = 0; i < PER; i++) {
            const int u = unit(i, tid);
            *reinterpret_cast<f32x4 *>(lds + (u / (W / 4)) * PITCH + 4 * (u % (W / 4))) = r[i];
        }
    }
};

// Maximum and sum over the 16 lanes of a row group.
__device__ __forceinline__ float group_max(float v, int lane) {
    v = fmaxf(v, st::xor_lane(v, 1, lane));
    v = fmaxf(v, st::xor_lane(v, 2, lane));
    v = fmaxf(v, st::xor_lane(v, 4, lane));
    return fmaxf(v, st::xor_lane(v, 8, lane));
}

__device__ __forceinline__ float group_sum(float v, int lane) {
    v += st::xor_lane(v, 1, lane);
    v += st::xor_lane(v, 2, lane);
    v += st::xor_lane(v, 4, lane);
    return v + st::xor_lane(v, 8, lane);
}

// HDP: head width, up to HDP (the rest of a tile's columns is zero).  LDS (of
// rows_lds bytes): the S block, then the tile.
__host__ __device__ constexpr int s_pitch(int t) { return (t + 15) / 16 * 16 + 4; }

template <int HDP>
size_t rows_lds(int t) {
    const size_t block = (size_t)RB * s_pitch(t) + (size_t)KT * (HDP + 4);
    return sizeof(float) * std::max<size_t>(block, (size_t)3 * RB * HDP);  // or the waves' partial outputs
}

template <int HDP, bool VEC, bool BWD>
__global__ __launch_bounds__(THREADS) void k_attn_rows(AttnArgs g) {
    constexpr int P = HDP + 4, NB = HDP / 16;
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, c16 = lane & 15, q4 = lane >> 4;
    int64_t z;
    int blk;
    place(g.blocks, z, blk);
    const int t = g.t, hd = g.hd, row0 = blk * RB, PS = s_pitch(t);
    float *S = lds, *tile = lds + RB * PS;
    const int64_t D = (int64_t)g.h * hd, win = (z / g.h) * t, col = (z % g.h) * hd;
    const float *head = g.qkv + win * 3 * D + col;
    const float *x = BWD ? g.dctx + win * D + col : head;
    const int64_t ldx = BWD ? D : 3 * D;
    const float *y1 = head + (BWD ? 2 : 1) * D, *y2 = head + (BWD ? 1 : 2) * D;
    const int nkt = (t + KT - 1) / KT;

    // The block's own rows go through LDS into every wave's fragments.
    Tile<KT, HDP, P, VEC> kt;
    f32x4 xa[2][NB];
    {
        Tile<RB, HDP, P, VEC> xt;
        xt.load(x, ldx, row0, t, 0, hd, tid);
        kt.load(y1, 3 * D, 0, t, 0, hd, tid);
        xt.store(tile, tid);
    }
    __syncthreads();
#pragma unroll
    for (int kc = 0; kc < NB; kc++)
#pragma unroll
        for (int i = 0; i < 2; i++)
            xa[i][kc] = *reinterpret_cast<const f32x4 *>(tile + (16 * i + c16) * P + 16 * kc + 4 * q4);
    __syncthreads();

    // First product: wave w computes columns 16 w .. of each tile, into LDS only
    // (stores to memory between the loads would have to be waited for with them).
    for (int n = 0; n < nkt; n++) {
        kt.store(tile, tid);
        __syncthreads();
        // The next tile, or the second product's first one.
        const bool more = n + 1 < nkt;
        kt.load(more ? y1 : y2, 3 * D, more ? (n + 1) * KT : 0, t, 0, hd, tid);
        asm volatile("" ::: "memory");  // keeps the loads above the multiplication
        if (n * KT + 16 * w < t) {      // uniform over the wave
            f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
            for (int kc = 0; kc < NB; kc++) {
                const f32x4 b = *reinterpret_cast<const f32x4 *>(tile + (16 * w + c16) * P + 16 * kc + 4 * q4);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(xa[0][kc][e], b[e], acc[0], 0, 0, 0);
                    acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(xa[1][kc][e], b[e], acc[1], 0, 0, 0);
                }
            }
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int r = 0; r < 4; r++) S[(16 * i + 4 * q4 + r) * PS + n * KT + 16 * w + c16] = acc[i][r];
        }
        __syncthreads();
    }

    // The block's rows of S (dP) to memory, and its softmax (or that one's
    // backward): 16 lanes per row, four rows of a wave at a time.  Columns past
    // the row's last visible one (past t, backward) become zero.
    const int tcols = PS - 4;
#pragma unroll
    for (int half = 0; half < 2; half++) {
        const int row = 8 * w + 4 * half + q4, grow = row0 + row;
        float *Sr = S + row * PS;
        const bool live = grow < t;
        const int64_t go = (z * t + min(grow, t - 1)) * (int64_t)t;
        // Eight of a lane's columns at a time, their reads in flight together.
        constexpr int G = 8;
        if constexpr (!BWD) {
            const int limit = min(grow, t - 1) + 1;
            float m = -__builtin_inff();
            for (int j0 = c16; j0 < t; j0 += 16 * G) {
                float v[G];
#pragma unroll
                for (int u = 0; u < G; u++) v[u] = Sr[min(j0 + 16 * u, t - 1)];
#pragma unroll
                for (int u = 0; u < G; u++) {
                    const int j = j0 + 16 * u;
                    if (live && j < t) g.s[go + j] = v[u];
                    if (j < limit) m = fmaxf(m, g.scale * v[u]);
                }
            }
            m = group_max(m, lane);
            float sum = 0.f;
            for (int j0 = c16; j0 < limit; j0 += 16 * G) {
                float v[G];
#pragma unroll
                for (int u = 0; u < G; u++) v[u] = expf(g.scale * Sr[min(j0 + 16 * u, limit - 1)] - m);
#pragma unroll
                for (int u = 0; u < G; u++) {
                    const int j = j0 + 16 * u;
                    if (j < limit) {
                        Sr[j] = v[u];
                        sum += v[u];
                    }
                }
            }
            // e / sum from one reciprocal per row and one correction per quotient, by
            // Markstein's method (IBM J. Res. Dev. 34(1), 1990): the quotient's remainder
            // is exact in an FMA, which makes the result the correctly rounded one (1 <=
            // sum <= t and 0 <= e <= 1, or NaN) unless quotient or remainder underflow:
            // an e below about 1e-30 may give a neighbour of it (1.4e-45 away among the
            // subnormal numbers).
            sum = group_sum(sum, lane);
            const float inv = 1.0f / sum;
            for (int j0 = c16; j0 < tcols; j0 += 16 * G) {
                float v[G];
#pragma unroll
                for (int u = 0; u < G; u++) {
                    const float e = Sr[min(j0 + 16 * u, limit - 1)], q = e * inv;
                    v[u] = __builtin_fmaf(__builtin_fmaf(-q, sum, e), inv, q);
                }
#pragma unroll
                for (int u = 0; u < G; u++) {
                    const int j = j0 + 16 * u;
                    if (j >= limit) v[u] = 0.f;
                    if (j < tcols) Sr[j] = v[u];
                    if (live && j < t) g.p[go + j] = v[u];
                }
            }
        } else {
            float d = 0.f;
            for (int j0 = c16; j0 < t; j0 += 16 * G) {
                float v[G], y[G];
#pragma unroll
                for (int u = 0; u < G; u++) {
                    const int j = min(j0 + 16 * u, t - 1);
                    y[u] = g.p[go + j];
                    v[u] = Sr[j];
                }
#pragma unroll
                for (int u = 0; u < G; u++)
                    if (j0 + 16 * u < t) d += v[u] * y[u];
            }
            d = group_sum(d, lane);
            for (int j0 = c16; j0 < tcols; j0 += 16 * G) {
                float v[G], y[G];
#pragma unroll
                for (int u = 0; u < G; u++) {
                    const int j = min(j0 + 16 * u, t - 1);
                    y[u] = g.p[go + j];
                    v[u] = Sr[j];
                }
#pragma unroll
                for (int u = 0; u < G; u++) {
                    const int j = j0 + 16 * u;
                    if (live && j < t) g.dp[go + j] = v[u];
                    const float x = j < t ? g.scale * y[u] * (v[u] - d) : 0.f;
                    if (j < tcols) Sr[j] = x;
                    if (live && j < t) g.ds[go + j] = x;
                }
            }
        }
    }

    // Second product: wave w contracts rows 16 w .. of each tile.
    f32x4 acc[2][NB];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < NB; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int n = 0; n < nkt; n++) {
        kt.store(tile, tid);
        __syncthreads();
        kt.load(y2, 3 * D, min(n + 1, nkt - 1) * KT, t, 0, hd, tid);
        asm volatile("" ::: "memory");
        if (n * KT + 16 * w < t) {  // uniform over the wave
            const float *Sa = S + c16 * PS + n * KT + 16 * w + 4 * q4;
            const f32x4 a0 = *reinterpret_cast<const f32x4 *>(Sa), a1 = *reinterpret_cast<const f32x4 *>(Sa + 16 * PS);
            const float *tb = tile + (16 * w + 4 * q4) * P + c16;
#pragma unroll
            for (int j = 0; j < NB; j++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float b = tb[e * P + 16 * j];
                    acc[0][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a0[e], b, acc[0][j], 0, 0, 0);
                    acc[1][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1[e], b, acc[1][j], 0, 0, 0);
                }
        }
        __syncthreads();
    }
    // The waves' partial outputs, added in wave order.
    float *out = BWD ? g.dqkv + win * 3 * D + col : g.ctx + win * D + col;
    const int64_t ldo = BWD ? 3 * D : D;
    if (w > 0) {
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < NB; j++)
                *reinterpret_cast<f32x4 *>(lds + (((w - 1) * 2 + i) * NB + j) * 256 + 4 * lane) = acc[i][j];
    }
    __syncthreads();
    if (w > 0) return;
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < NB; j++) {
            f32x4 v = acc[i][j];
#pragma unroll
            for (int o = 0; o < 3; o++) v += *reinterpret_cast<const f32x4 *>(lds + ((o * 2 + i) * NB + j) * 256 + 4 * lane);
            const int cc = 16 * j + c16;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int row = row0 + 16 * i + 4 * q4 + r;
                if (cc < hd && row < t) out[(int64_t)row * ldo + cc] = v[r];
            }
        }
}

// dV and dK of 32 keys: wave w contracts query rows 8 w .. of each tile of 32.
// VT: t is a multiple of 4.
template <int HDP, bool VEC, bool VT>
__global__ __launch_bounds__(THREADS) void k_attn_cols(AttnArgs g) {
    constexpr int QT = 32, P = HDP + 4, PK = RB + 4, NB = HDP / 16;
    constexpr int TILE = QT * P, KTILE = QT * PK;
    constexpr int USED = 2 * TILE + 2 * KTILE, RED = 3 * RB * HDP;  // tiles; the waves' partial results
    __shared__ __attribute__((aligned(16))) float lds[USED > RED ? USED : RED];
    float *tO = lds, *tQ = lds + TILE, *tP = tQ + TILE, *tS = tP + KTILE;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, c16 = lane & 15, q4 = lane >> 4;
    int64_t z;
    int blk;
    place(g.blocks, z, blk);
    const int t = g.t, hd = g.hd, key0 = blk * RB;
    const int64_t D = (int64_t)g.h * hd, win = (z / g.h) * t, col = (z % g.h) * hd;
    const float *q = g.qkv + win * 3 * D + col, *dO = g.dctx + win * D + col;
    const float *pp = g.p + z * t * t, *ss = g.ds + z * t * t;
    const int nqt = (t + QT - 1) / QT;

    Tile<QT, HDP, P, VEC> o, qt;
    Tile<QT, RB, PK, VT> pt, st;
    auto load = [&](int n) {
        o.load(dO, D, n * QT, t, 0, hd, tid);
        qt.load(q, 3 * D, n * QT, t, 0, hd, tid);
        pt.load(pp, t, n * QT, t, key0, t, tid);
        st.load(ss, t, n * QT, t, key0, t, tid);
    };
    f32x4 dv[2][NB], dk[2][NB];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < NB; j++) {
            dv[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
            dk[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    load(0);
    for (int n = 0; n < nqt; n++) {
        o.store(tO, tid);
        qt.store(tQ, tid);
        pt.store(tP, tid);
        st.store(tS, tid);
        __syncthreads();
        load(min(n + 1, nqt - 1));
        asm volatile("" ::: "memory");
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const int k = 8 * w + 4 * e + q4;
            const float p0 = tP[k * PK + c16], p1 = tP[k * PK + 16 + c16];
            const float s0 = tS[k * PK + c16], s1 = tS[k * PK + 16 + c16];
#pragma unroll
            for (int j = 0; j < NB; j++) {
                const float bo = tO[k * P + 16 * j + c16], bq = tQ[k * P + 16 * j + c16];
                dv[0][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(p0, bo, dv[0][j], 0, 0, 0);
                dv[1][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(p1, bo, dv[1][j], 0, 0, 0);
                dk[0][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(s0, bq, dk[0][j], 0, 0, 0);
                dk[1][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(s1, bq, dk[1][j], 0, 0, 0);
            }
        }
        __syncthreads();
    }
    // The waves' partial results, added in wave order: dV by wave 0, dK by wave 1
    // (each from the other three, in two rounds over the same memory).
#pragma unroll
    for (int which = 0; which < 2; which++) {
        if (w != which) {
            const int slot = w - (w > which);
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < NB; j++)
                    *reinterpret_cast<f32x4 *>(lds + ((slot * 2 + i) * NB + j) * 256 + 4 * lane) =
                        which ? dk[i][j] : dv[i][j];
        }
        __syncthreads();
        if (w == which) {
            float *out = g.dqkv + win * 3 * D + col + (which ? 1 : 2) * D;
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < NB; j++) {
                    auto part = [&](int slot) {
                        return *reinterpret_cast<const f32x4 *>(lds + ((slot * 2 + i) * NB + j) * 256 + 4 * lane);
                    };
                    const f32x4 own = which ? dk[i][j] : dv[i][j];
                    const f32x4 v = which ? ((part(0) + own) + part(1)) + part(2) : ((own + part(0)) + part(1)) + part(2);
                    const int cc = 16 * j + c16;
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const int key = key0 + 16 * i + 4 * q4 + r;
                        if (cc < hd && key < t) out[(int64_t)key * 3 * D + cc] = v[r];
                    }
                }
        }
        __syncthreads();
    }
}

// Launches f<width class>(): the narrowest of the compiled head widths that
// holds hd.  A width is padded to its class, at the class's cost and more (96
// problems of T = 200, forward rows and both backward launches, us: 80 wide in
// its own class 106, 96 wide in that of 128 243, 128 wide 185), so there is one
// for each of the widths in use, 32, 64 and 80; 128 takes the rest, where the
// separate launches are mostly faster (a caller of the C interface chooses).
template <class F>
st_status by_width(int64_t hd, F f) {
    if (hd % 4)
        return hd <= 64 ? f(std::integral_constant<int, 64>(), std::false_type())
                        : f(std::integral_constant<int, 128>(), std::false_type());
    if (hd <= 32) return f(std::integral_constant<int, 32>(), std::true_type());
    if (hd <= 64) return f(std::integral_constant<int, 64>(), std::true_type());
    if (hd <= 80) return f(std::integral_constant<int, 80>(), std::true_type());
    return f(std::integral_constant<int, 128>(), std::true_type());
}

template <bool BWD>
st_status launch_rows(const AttnArgs &g, int64_t wgs, hipStream_t stream) {
    return by_width(g.hd, [&](auto width, auto vec) {
        constexpr int HDP = decltype(width)::value;
        auto *k = &k_attn_rows<HDP, decltype(vec)::value, BWD>;
        const size_t lds = rows_lds<HDP>(g.t);
        if (lds > 64 * 1024)
            ST_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(k),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        hipLaunchKernelGGL(k, dim3((unsigned)wgs), dim3(THREADS), lds, stream, g);
        ST_LAUNCH_CHECK();
        return ST_OK;
    });
}

st_status launch_cols(const AttnArgs &g, int64_t wgs, hipStream_t stream) {
    return by_width(g.hd, [&](auto width, auto vec) {
        constexpr int HDP = decltype(width)::value;
        constexpr bool V = decltype(vec)::value;
        auto *k = g.t % 4 ? &k_attn_cols<HDP, V, false> : &k_attn_cols<HDP, V, true>;
        hipLaunchKernelGGL(k, dim3((unsigned)wgs), dim3(THREADS), 0, stream, g);
        ST_LAUNCH_CHECK();
        return ST_OK;
    });
}

st_status check(const char *what, int64_t b, int64_t h, int64_t t, int64_t hd) {
    if (b < 0 || h < 1 || !st_attention_fits(t, hd))
        return st::fail(ST_ERR_INVALID, "%s: needs b >= 0, h >= 1, t in 1..=%d and hd in 1..=%d", what, T_MAX, HD_MAX);
    if (b * h > (int64_t)(INT32_MAX / THREADS) / ((t + RB - 1) / RB))
        return st::fail(ST_ERR_INVALID, "%s: too many problems for one launch", what);
    return ST_OK;
}

}  // namespace

extern "C" int32_t st_attention_fits(int64_t t, int64_t hd) { return t >= 1 && t <= T_MAX && hd >= 1 && hd <= HD_MAX; }

extern "C" st_status st_attention_fwd(const float *qkv, float *s, float *p, float *ctx, int64_t b, int64_t h,
                                      int64_t t, int64_t hd, float scale, st_stream stream) {
    st::clear_error();
    if (!qkv || !s || !p || !ctx) return st::fail(ST_ERR_INVALID, "attention_fwd: NULL buffer");
    const st_status c = check("attention_fwd", b, h, t, hd);
    if (c != ST_OK || b == 0) return c;
    if (!st::device_ok()) return ST_ERR_NO_DEVICE;
    const int32_t blocks = (int32_t)((t + RB - 1) / RB);
    const AttnArgs g{qkv, nullptr, s, p, nullptr, nullptr, ctx, nullptr, (int32_t)h, (int32_t)t, (int32_t)hd, blocks, scale};
    return launch_rows<false>(g, b * h * blocks, st::stream_of(stream));
}

extern "C" st_status st_attention_bwd(const float *qkv, const float *dctx, const float *p, float *dp, float *ds,
                                      float *dqkv, int64_t b, int64_t h, int64_t t, int64_t hd, float scale,
                                      st_stream stream) {
    st::clear_error();
    if (!qkv || !dctx || !p || !dp || !ds || !dqkv) return st::fail(ST_ERR_INVALID, "attention_bwd: NULL buffer");
    const st_status c = check("attention_bwd", b, h, t, hd);
    if (c != ST_OK || b == 0) return c;
    if (!st::device_ok()) return ST_ERR_NO_DEVICE;
    const int32_t blocks = (int32_t)((t + RB - 1) / RB);
    const AttnArgs g{qkv, dctx, nullptr, const_cast<float *>(p), dp, ds, nullptr, dqkv, (int32_t)h, (int32_t)t,
                     (int32_t)hd, blocks, scale};
    const hipStream_t st = st::stream_of(stream);
    const st_status r = launch_rows<true>(g, b * h * blocks, st);
    return r != ST_OK ? r : launch_cols(g, b * h * blocks, st);
}
