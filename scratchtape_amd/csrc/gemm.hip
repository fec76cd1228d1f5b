// GEMM for the three tape forms (C = A·B, dA = dC·Bᵀ, dB = Aᵀ·dC) on gfx950
// matrix cores, f32 and f16-in/f32-accumulate, batched, with head-view
// addressing, the reference's epilogue and deterministic split-k.
//
// Reference semantics: gpu_step/matmul.rs:26-299 (MatRef, Epilogue, matmul,
// matmul_f32, matmul_with, split-k and its ordered sum) and src/tensor.rs:241
// (NdArray::matmul).
//
// Design (gfx950 / CDNA4):
//  - One workgroup of 256 threads = 4 wave64s in a 2x2 grid computes a BM x BN
//    output tile; each wave owns (BM/2) x (BN/2) as 16x16 MFMA blocks.
//  - f16 route: v_mfma_f32_16x16x32_f16; f32 operands are read from HBM with
//    128-bit loads and rounded to f16 (round to nearest even) on the way into
//    LDS.  f32 route: v_mfma_f32_16x16x4_f32 on f32 LDS tiles.
//  - LDS holds an operand [row][k] (rows padded by 16 bytes, so the 128-bit
//    fragment reads of 8 lanes hit distinct banks) or, for an f32 operand whose
//    rows are contiguous in memory (A transposed, B not), [k][row] as loaded.
//    The f16 route turns the latter's 4x4 blocks in registers.  k-stages of 64
//    (f16) / 32 (f32); two LDS buffers and two register sets, so stage s+2 is
//    in flight from global memory while stage s feeds the MFMAs and stage s+1
//    is written to LDS; one barrier per stage and no branch around the loads.
//  - Bound: f32 by the matrix cores (busy 70 % of the CUs' time at 3001 x 2000
//    x 1003) once there are workgroups to overlap, by the LDS round and barrier
//    of a k-stage with one workgroup per CU.  The form before loaded every
//    element of a ragged or misaligned shape by itself, guarded, and waited for
//    each load where it was issued.  Single calls, us before and now:
//    3000 x 250 x 1001 forward 45 -> 26, dW 55 -> 31, dX 50 -> 22; 3001 x 2000 x
//    1003 273 -> 116, 239 -> 138, 273 -> 121 (104 TFLOP/s); 96 products of
//    200 x 80 x 200 52 -> 22; f16 8192 x 1056 x 1056 237 -> 71.
//  - Workgroups are remapped so that each of the 8 XCDs works on a contiguous
//    run of tiles, which share operand panels in that XCD's L2.
//  - Fragment k-order: each lane reads its k-run as one 128-bit LDS read and
//    feeds it to the MFMA; A and B use the same k mapping, so the dot product
//    is over the right pairs whatever order the hardware sums them in.
//  - Split-k (shapes with too few output tiles, e.g. the weight gradients with
//    k = 4096): slices write [m, n] partials to the scratch arena, then one
//    launch sums them in slice order (deterministic), as the reference's
//    k_split_sum (matmul.rs:259-299).
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

#include "common.h"
#include "dma_tile.h"
#include "gemm_dma.h"

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int THREADS = 256;

struct Operand {
    const float *p;  // buffer + element offset
    int64_t stride, group, inner, ld;
};

struct GemmArgs {
    Operand a, b;
    float *out;  // buffer + element offset (or the split-k partials)
    int64_t o_stride, o_group, o_inner, ldo;
    const float *bias;  // + bias_off
    int64_t bias_stride;
    const float *mask;  // + mask_off
    const float *res;   // + residual_off
    float *cs;          // column-sum destination (out buffer + col_sum_off, or partials)
    int64_t cs_stride;
    int32_t cs_direct, has_cs;
    int32_t m, n, k;
    int32_t splits, slice_k;
    int32_t relu, accumulate;
};

__device__ __forceinline__ int64_t mat_base(const Operand &o, int64_t z) {
    return (z / o.group) * o.stride + (z % o.group) * o.inner;
}

template <bool F16>
__device__ __forceinline__ void store4(void *dst, float x0, float x1, float x2, float x3) {
    if constexpr (F16) {
        half4 h = {(_Float16)x0, (_Float16)x1, (_Float16)x2, (_Float16)x3};
        *reinterpret_cast<half4 *>(dst) = h;
    } else {
        f32x4 v = {x0, x1, x2, x3};
        *reinterpret_cast<f32x4 *>(dst) = v;
    }
}

// How a tile's operands are read (Stager), for any shape and alignment:
//  - WHOLE (the matrix is at least one tile in both dimensions): a last tile
//    that would cross the edge is moved back to end there and stores only the
//    rows and columns that are its own, so every load is a 16-byte load (4-byte
//    alignment is enough) with no guard;
//  - otherwise (fewer than 32 rows or columns): element by element, the rows
//    past the matrix repeating its last one.  They feed output rows and columns
//    that are not stored.
// The partial k-stage comes first and is loaded element by element.
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

// Stages one operand's ROWS x BK tile (logical rows = m for A, n for B; k
// across) from global memory into registers, then into LDS.
// KCONTIG: element (r, kk) at base[r*ld + kk]; else at base[kk*ld + r].
template <int ROWS, int BK, bool KCONTIG, bool WHOLE, bool F16>
struct Stager {
    // LDS tile: [row][k] with rows LDS_K apart, or (KROWS) [k][row] with lines
    // LDS_R apart, written as loaded.
    static constexpr bool KROWS = !KCONTIG && !F16;
    static constexpr int LDS_K = BK + (F16 ? 8 : 4);
    static constexpr int LDS_R = ROWS + 4;
    static constexpr int SIZE = KROWS ? BK * LDS_R : ROWS * LDS_K;
    // KCONTIG: 4-wide vectors along k.  Else 4x4 blocks (4 k x 4 rows).
    static constexpr int UNITS = KCONTIG ? ROWS * BK / 4 : ROWS * BK / 16;
    static constexpr int PER = (UNITS + THREADS - 1) / THREADS;
    static constexpr int VEC = KCONTIG ? 1 : 4;  // float4 per unit
    static constexpr int SLOTS = BK / 4;          // column-sum partials per row
    f32x4 r[PER][VEC];
    float cs[PER][KCONTIG ? 1 : 4];

    __device__ __forceinline__ void zero_cs() {
#pragma unroll
        for (int i = 0; i < PER; i++)
#pragma unroll
            for (int x = 0; x < (KCONTIG ? 1 : 4); x++) cs[i][x] = 0.f;
    }

    // Four rows from `row` of one k-line, or (KCONTIG) four k of one row.
    static __device__ __forceinline__ f32x4 rows4(const float *line, int row, int row_lim) {
        if constexpr (WHOLE) return *reinterpret_cast<const f32x4u *>(line + row);
        return f32x4{line[min(row, row_lim - 1)], line[min(row + 1, row_lim - 1)], line[min(row + 2, row_lim - 1)],
                     line[min(row + 3, row_lim - 1)]};
    }

    // Loads the tile of the first k-stage: nk <= BK of k from k0, zeros behind
    // them.
    __device__ __forceinline__ void load_first(const float *__restrict__ base, int64_t ld, int row0, int row_lim,
                                               int k0, int nk, int tid) {
#pragma unroll
        for (int i = 0; i < PER; i++) {
            const int u = tid + THREADS * i;
            if (UNITS % THREADS != 0 && u >= UNITS) break;
            if constexpr (KCONTIG) {
                const int rr = u / (BK / 4), kq = (u % (BK / 4)) * 4;
                const float *row = base + (int64_t)(WHOLE ? row0 + rr : min(row0 + rr, row_lim - 1)) * ld + k0;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float v = row[min(kq + e, nk - 1)];
                    r[i][0][e] = kq + e < nk ? v : 0.f;
                }
            } else {
                const int rq = (u % (ROWS / 4)) * 4, kq = (u / (ROWS / 4)) * 4;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const f32x4 v = rows4(base + (int64_t)(k0 + min(kq + e, nk - 1)) * ld, row0 + rq, row_lim);
                    r[i][e] = kq + e < nk ? v : f32x4{0.f, 0.f, 0.f, 0.f};
                }
            }
        }
    }

    // Loads the tile of a whole k-stage, without a branch.
    __device__ __forceinline__ void load(const float *__restrict__ base, int64_t ld, int row0, int row_lim, int k0,
                                         int tid) {
#pragma unroll
        for (int i = 0; i < PER; i++) {
            const int u = tid + THREADS * i;
            if (UNITS % THREADS != 0 && u >= UNITS) break;
            if constexpr (KCONTIG) {
                const int rr = u / (BK / 4), kq = (u % (BK / 4)) * 4;
                const float *row = base + (int64_t)(WHOLE ? row0 + rr : min(row0 + rr, row_lim - 1)) * ld + kq;
                r[i][0] = *reinterpret_cast<const f32x4u *>(row + k0);
            } else {
                const int rq = (u % (ROWS / 4)) * 4, kq = (u / (ROWS / 4)) * 4;
#pragma unroll
                for (int e = 0; e < 4; e++)
                    r[i][e] = rows4(base + (int64_t)(kq + e) * ld + (int64_t)k0 * ld, row0 + rq, row_lim);
            }
        }
    }

    // Adds the tile's values to the column sums (`on`: uniform, without a branch).
    __device__ __forceinline__ void add_cs(bool on) {
#pragma unroll
        for (int i = 0; i < PER; i++) {
            if constexpr (KCONTIG) {
                const float t = cs[i][0] + (((r[i][0][0] + r[i][0][1]) + r[i][0][2]) + r[i][0][3]);
                cs[i][0] = on ? t : cs[i][0];
            } else {
#pragma unroll
                for (int x = 0; x < 4; x++) {
                    const float t = cs[i][x] + (((r[i][0][x] + r[i][1][x]) + r[i][2][x]) + r[i][3][x]);
                    cs[i][x] = on ? t : cs[i][x];
                }
            }
        }
    }

    template <typename T>
    __device__ __forceinline__ void store(T *lds, int tid) const {
#pragma unroll
        for (int i = 0; i < PER; i++) {
            const int u = tid + THREADS * i;
            if (UNITS % THREADS != 0 && u >= UNITS) break;
            if constexpr (KCONTIG) {
                const int rr = u / (BK / 4), kq = (u % (BK / 4)) * 4;
                store4<F16>(lds + rr * LDS_K + kq, r[i][0][0], r[i][0][1], r[i][0][2], r[i][0][3]);
            } else {
                const int rq = (u % (ROWS / 4)) * 4, kq = (u / (ROWS / 4)) * 4;
#pragma unroll
                for (int x = 0; x < 4; x++) {
                    if constexpr (KROWS)
                        *reinterpret_cast<f32x4 *>(lds + (kq + x) * LDS_R + rq) = r[i][x];
                    else
                        store4<F16>(lds + (rq + x) * LDS_K + kq, r[i][0][x], r[i][1][x], r[i][2][x], r[i][3][x]);
                }
            }
        }
    }

    __device__ __forceinline__ void merge_cs(const Stager &o) {
#pragma unroll
        for (int i = 0; i < PER; i++)
#pragma unroll
            for (int x = 0; x < (KCONTIG ? 1 : 4); x++) cs[i][x] += o.cs[i][x];
    }

    // Writes this thread's column-sum partials to red[col * SLOTS + slot].
    __device__ __forceinline__ void put_cs(float *red, int tid) const {
#pragma unroll
        for (int i = 0; i < PER; i++) {
            const int u = tid + THREADS * i;
            if (UNITS % THREADS != 0 && u >= UNITS) break;
            if constexpr (KCONTIG) {
                red[(u / (BK / 4)) * SLOTS + u % (BK / 4)] = cs[i][0];
            } else {
                const int rq = (u % (ROWS / 4)) * 4, slot = u / (ROWS / 4);
#pragma unroll
                for (int x = 0; x < 4; x++) red[(rq + x) * SLOTS + slot] = cs[i][x];
            }
        }
    }
};

template <int BM, int BN, int BK, bool TA, bool TB, bool F16, bool WHOLE>
__global__ __launch_bounds__(THREADS) void k_gemm(GemmArgs g) {
    using T = typename std::conditional<F16, _Float16, float>::type;
    using SA = Stager<BM, BK, !TA, WHOLE, F16>;
    using SB = Stager<BN, BK, TB, WHOLE, F16>;
    constexpr int LDS_K = SA::LDS_K;
    constexpr int WM = BM / 2, WN = BN / 2;
    constexpr int FM = WM / 16, FN = WN / 16;
    static_assert(BK % (F16 ? 32 : 16) == 0, "k stage");
    __shared__ __attribute__((aligned(16))) T As[2][SA::SIZE];
    __shared__ __attribute__((aligned(16))) T Bs[2][SB::SIZE];

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    // Workgroups are dealt to the 8 XCDs round-robin by linear id; remap so
    // each XCD gets a contiguous run of tiles (columns fastest), which share A
    // rows (and k-slices) in that XCD's L2.
    const int64_t gxy = (int64_t)gridDim.x * gridDim.y, total = gxy * gridDim.z;
    int64_t lin = blockIdx.x + (int64_t)gridDim.x * (blockIdx.y + (int64_t)gridDim.y * blockIdx.z);
    if (total % 8 == 0) lin = (lin % 8) * (total / 8) + lin / 8;
    const int nbx = (g.n + BN - 1) / BN;
    const int64_t z = lin / gxy;
    const int tile = (int)(lin % gxy);
    const int bx = tile % nbx, by = tile / nbx;
    if (by * BM >= g.m) return;  // a grid of several rows may be larger than the tiles
    const int64_t zb = z / g.splits;
    const int slice = (int)(z % g.splits);
    // The tile's own rows and columns begin at row_own, col_own; the last tile
    // of a row or column of tiles may be moved back to row0, col0.
    const int row_own = by * BM, col_own = bx * BN;
    const int row0 = WHOLE ? min(row_own, g.m - BM) : row_own, col0 = WHOLE ? min(col_own, g.n - BN) : col_own;
    const int kbeg = slice * g.slice_k;
    const int kend = min(g.k, kbeg + g.slice_k);
    const int nst = kend > kbeg ? (kend - kbeg + BK - 1) / BK : 0;

    const float *abase = g.a.p + mat_base(g.a, zb);
    const float *bbase = g.b.p + mat_base(g.b, zb);
    const bool do_cs = g.has_cs && by == 0;

    // Two register sets: stage st+2 is fetched into the set stage st came
    // from while stage st is multiplied out of LDS, so two stages of global
    // loads are in flight behind every barrier.
    SA sa[2];
    SB sb[2];
    sb[0].zero_cs();
    sb[1].zero_cs();
    // f32 sums of the smaller tiles run in NA chains (every NA-th group of k),
    // added at the end.  plan_tiles splits small products less than a slice per
    // CU would, and longer sums err more: a step's products at 284 tokens x 320
    // wide, against 64 bits, 2.3e-7 in the earlier splits, 3.2e-7 in one chain
    // each, 1.7e-7 now, in the same time (260, 150 and 152 us for the 15).
    constexpr int NA = F16 || FM * FN > 4 ? 1 : FM * FN > 1 ? 2 : 4;
    f32x4 acc[FM][FN], more[NA > 1 ? NA - 1 : 1][FM][FN];
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++) {
            acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < NA - 1; c++) more[c][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        }

    // The partial k-stage comes first (k1 of k), so that every later one is
    // whole.
    const int k1 = nst > 0 ? kend - kbeg - (nst - 1) * BK : 0;
    const int kfull = kbeg + k1 - BK;  // stage st >= 1 begins at kfull + st BK
    auto load = [&](int p, int st) {
        const int k0 = kfull + st * BK;
        sa[p].load(abase, g.a.ld, row0, g.m, k0, tid);
        sb[p].load(bbase, g.b.ld, col0, g.n, k0, tid);
    };
    auto stage = [&](int p, bool live) {
        sb[p].add_cs(live);
        sa[p].store(As[p], tid);
        sb[p].store(Bs[p], tid);
    };
    if (nst > 0) {
        sa[0].load_first(abase, g.a.ld, row0, g.m, kbeg, k1, tid);
        sb[0].load_first(bbase, g.b.ld, col0, g.n, kbeg, k1, tid);
        if (nst > 1) load(1, 1);
        stage(0, true);
    }
    __syncthreads();

    auto multiply = [&](int p) {
        const T *as = As[p] + (wm * WM + (lane & 15)) * (SA::KROWS ? 1 : LDS_K);
        const T *bs = Bs[p] + (wn * WN + (lane & 15)) * (SB::KROWS ? 1 : LDS_K);
        if constexpr (F16) {
#pragma unroll
            for (int ks = 0; ks < BK / 32; ks++) {
                half8 af[FM], bf[FN];
                const int ko = ks * 32 + 8 * (lane >> 4);
#pragma unroll
                for (int i = 0; i < FM; i++) af[i] = *reinterpret_cast<const half8 *>(as + i * 16 * LDS_K + ko);
#pragma unroll
                for (int j = 0; j < FN; j++) bf[j] = *reinterpret_cast<const half8 *>(bs + j * 16 * LDS_K + ko);
#pragma unroll
                for (int i = 0; i < FM; i++)
#pragma unroll
                    for (int j = 0; j < FN; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[i], bf[j], acc[i][j], 0, 0, 0);
            }
        } else {
#pragma unroll
            for (int kc = 0; kc < BK / 16; kc++) {
                f32x4 af[FM], bf[FN];
                const int ko = kc * 16 + 4 * (lane >> 4);
                // Four k of a row at once, or ([k][row] tiles) one k of each line: the lane groups' lines are
                // 4 LDS_R = 16 banks apart, so the 64 lanes of a read hit 64 banks.
#pragma unroll
                for (int i = 0; i < FM; i++) {
                    if constexpr (SA::KROWS)
                        for (int e = 0; e < 4; e++) af[i][e] = as[(ko + e) * SA::LDS_R + i * 16];
                    else
                        af[i] = *reinterpret_cast<const f32x4 *>(as + i * 16 * LDS_K + ko);
                }
#pragma unroll
                for (int j = 0; j < FN; j++) {
                    if constexpr (SB::KROWS)
                        for (int e = 0; e < 4; e++) bf[j][e] = bs[(ko + e) * SB::LDS_R + j * 16];
                    else
                        bf[j] = *reinterpret_cast<const f32x4 *>(bs + j * 16 * LDS_K + ko);
                }
#pragma unroll
                for (int s = 0; s < 4; s++)
#pragma unroll
                    for (int i = 0; i < FM; i++)
#pragma unroll
                        for (int j = 0; j < FN; j++) {
                            constexpr int PER_KC = NA == 4 ? 2 : 1;
                            const int c = (kc * PER_KC + s % PER_KC) % NA;
                            f32x4 &sum = c == 0 ? acc[i][j] : more[c > 0 ? c - 1 : 0][i][j];
                            sum = __builtin_amdgcn_mfma_f32_16x16x4f32(af[i][s], bf[j][s], sum, 0, 0, 0);
                        }
            }
        }
    };
    // Stages st and st + 1 per trip, stage st in LDS and st + 1 in flight at
    // its head.  No branch inside: the loads past the last stage repeat it, so
    // that the compiler can count the loads in flight (behind a condition it
    // waits for all of them, a memory round trip per stage), and the asm keeps
    // them above the multiplication.
    for (int st = 0; st + 1 < nst; st += 2) {
        load(0, min(st + 2, nst - 1));
        asm volatile("" ::: "memory");
        multiply(0);
        stage(1, true);
        __syncthreads();
        load(1, min(st + 3, nst - 1));
        asm volatile("" ::: "memory");
        multiply(1);
        stage(0, st + 2 < nst);
        __syncthreads();
    }
    if (nst & 1) multiply(0);
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++) {
            if constexpr (NA == 2) acc[i][j] += more[0][i][j];
            if constexpr (NA == 4) acc[i][j] = (acc[i][j] + more[0][i][j]) + (more[1][i][j] + more[NA - 2][i][j]);
        }
    __syncthreads();

    // Column sums of this slice of B (tile row 0 only), reduced in slot order.
    if (do_cs) {
        float *red = reinterpret_cast<float *>(As[0]);  // BN * SLOTS floats fit in As
        static_assert(BN * SB::SLOTS * 4 <= SA::SIZE * (int)sizeof(T), "column-sum buffer");
        sb[0].merge_cs(sb[1]);
        sb[0].put_cs(red, tid);
        __syncthreads();
        if (tid < BN && col0 + tid >= col_own && col0 + tid < g.n) {
            float tot = 0.f;
#pragma unroll
            for (int s = 0; s < SB::SLOTS; s++) tot += red[tid * SB::SLOTS + s];
            float *dst = g.cs + (g.cs_direct ? zb : z) * g.cs_stride + col0 + tid;
            if (g.cs_direct)
                *dst += tot;
            else
                *dst = tot;
        }
    }

    // Epilogue: lane holds rows 4*(lane/16)+r, column lane%16 of each block.
    // A row of blocks' mask, residual and output values are loaded together
    // (one memory round trip, not one per element); elements past the matrix
    // read its last row or column.
    const int64_t o0 = (z / g.o_group) * g.o_stride + (z % g.o_group) * g.o_inner;
    float bv[FN];
#pragma unroll
    for (int j = 0; j < FN; j++)
        bv[j] = g.bias ? g.bias[zb * g.bias_stride + min(col0 + wn * WN + j * 16 + (lane & 15), g.n - 1)] : 0.f;
#pragma unroll
    for (int i = 0; i < FM; i++) {
        float mk[FN][4], rs[FN][4], pv[FN][4];
        int64_t idx[4];
#pragma unroll
        for (int r = 0; r < 4; r++)
            idx[r] = o0 + (int64_t)min(row0 + wm * WM + i * 16 + 4 * (lane >> 4) + r, g.m - 1) * g.ldo;
        auto gather = [&](const float *src, float (&v)[FN][4]) {
#pragma unroll
            for (int j = 0; j < FN; j++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    v[j][r] = src[idx[r] + min(col0 + wn * WN + j * 16 + (lane & 15), g.n - 1)];
        };
        if (g.mask) gather(g.mask, mk);
        if (g.res) gather(g.res, rs);
        if (g.accumulate) gather(g.out, pv);
#pragma unroll
        for (int j = 0; j < FN; j++) {
            const int col = col0 + wn * WN + j * 16 + (lane & 15);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                float v = acc[i][j][r];
                if (g.bias) v += bv[j];
                if (g.relu && v < 0.f) v = 0.f;
                if (g.mask && mk[j][r] <= 0.f) v = 0.f;
                if (g.res) v += rs[j][r];
                if (g.accumulate) v += pv[j][r];
                const int row = row0 + wm * WM + i * 16 + 4 * (lane >> 4) + r;
                if (WHOLE ? col >= col_own && row >= row_own : col < g.n && row < g.m) g.out[idx[r] + col] = v;
            }
        }
    }
}

// out[b] (+)= sum over s (ascending) of partial[b*splits + s]; then the
// column-sum partials into their destination (always +=).
__global__ __launch_bounds__(256) void k_split_sum(const float *__restrict__ partial, float *out,
                                                   int64_t len, int32_t splits, int64_t o_stride,
                                                   int64_t batch, int32_t accumulate, const float *cs_part,
                                                   float *cs_dst, int64_t cs_stride, int64_t n) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e < batch * len) {
        const int64_t b = e / len, i = e % len;
        float v = dma::sum_slices(partial + b * splits * len + i, len, splits, 0.f);
        float *o = out + b * o_stride + i;
        if (accumulate) v += *o;
        *o = v;
    } else if (cs_part) {
        const int64_t c = e - batch * len;
        if (c < batch * n) {
            const int64_t b = c / n, j = c % n;
            const float v = dma::sum_slices(cs_part + b * splits * n + j, n, splits, 0.f);
            cs_dst[b * cs_stride + j] += v;
        }
    }
}

using KernelFn = void (*)(GemmArgs);

template <int BM, int BN, int BK, bool F16, bool WHOLE>
KernelFn pick_trans(bool ta, bool tb) {
    if (!ta && !tb) return &k_gemm<BM, BN, BK, false, false, F16, WHOLE>;
    if (!ta && tb) return &k_gemm<BM, BN, BK, false, true, F16, WHOLE>;
    if (ta && !tb) return &k_gemm<BM, BN, BK, true, false, F16, WHOLE>;
    return &k_gemm<BM, BN, BK, true, true, F16, WHOLE>;
}

struct TileCfg {
    int bm, bn;
    int64_t splits, slice_k;
};

// The tiles that plan_tiles picks.  (f16: m % 64 == 0 and n % 32 == 0, so every
// tile is whole.)
KernelFn pick_kernel(const TileCfg &tc, bool f16, bool ta, bool tb, bool whole) {
    if (f16) {
        if (tc.bm == 128) return pick_trans<128, 64, 64, true, true>(ta, tb);
        if (tc.bm == 64) return pick_trans<64, 64, 64, true, true>(ta, tb);
        return pick_trans<32, 32, 64, true, true>(ta, tb);
    }
    if (tc.bm == 128) return pick_trans<128, 128, 32, false, true>(ta, tb);
    if (tc.bm == 64) return pick_trans<64, 64, 32, false, true>(ta, tb);
    return whole ? pick_trans<32, 32, 32, false, true>(ta, tb) : pick_trans<32, 32, 32, false, false>(ta, tb);
}

int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

st_status check_ref(const st_matref *r, const char *what) {
    if (!r) return st::fail(ST_ERR_INVALID, "%s is NULL", what);
    if (!r->p) return st::fail(ST_ERR_INVALID, "%s.p is NULL", what);
    if (r->off < 0 || r->stride < 0 || r->ld < 0 || r->group < 0 || r->inner < 0)
        return st::fail(ST_ERR_INVALID, "%s has a negative offset, stride, ld, group or inner", what);
    return ST_OK;
}

// The reference's argument checks for one call (its assert!s).
st_status check_call(const st_matref *a, const st_matref *b, const st_matref *out, int64_t batch, int64_t m,
                     int64_t k, int64_t n) {
    st_status s;
    if ((s = check_ref(a, "a")) || (s = check_ref(b, "b")) || (s = check_ref(out, "out"))) return s;
    if (out->trans) return st::fail(ST_ERR_INVALID, "out is stored row-major");
    if (batch < 0 || m < 0 || k < 0 || n < 0) return st::fail(ST_ERR_INVALID, "negative batch or shape");
    if (m > INT32_MAX / 2 || n > INT32_MAX / 2 || k > INT32_MAX / 2)
        return st::fail(ST_ERR_INVALID, "matrix dimension too large");
    return ST_OK;
}

// The reference's f16 eligibility (matmul.rs:108-112, 524-534): k % 32, m % 64
// and n % 64 (or n % 32 for its 64x32 tile), and not column sums of a
// transposed b.
bool f16_route(bool use_f16, const st_epilogue &epi, const st_matref *b, int64_t m, int64_t k, int64_t n) {
    return use_f16 && !(epi.has_col_sum && b->trans) && k > 0 && k % 32 == 0 && m % 64 == 0 && n % 32 == 0;
}

// One call as the LDS-DMA kernels take it: element offsets folded into the
// pointers, group 0 read as 1, packed leading dimensions made explicit.
st::DmaGemm make_dma(const st_matref *a, const st_matref *b, const st_matref *out, int64_t batch, int64_t m,
                     int64_t k, int64_t n, const st_epilogue &epi, bool f16) {
    st::DmaGemm d;
    std::memset(&d, 0, sizeof d);
    d.a = a->p + a->off;
    d.a_stride = a->stride;
    d.a_group = a->group > 0 ? a->group : 1;
    d.a_inner = a->inner;
    d.lda = a->ld ? a->ld : (a->trans ? m : k);
    d.ta = a->trans != 0;
    d.b = b->p + b->off;
    d.b_stride = b->stride;
    d.b_group = b->group > 0 ? b->group : 1;
    d.b_inner = b->inner;
    d.ldb = b->ld ? b->ld : (b->trans ? k : n);
    d.tb = b->trans != 0;
    d.out = out->p + out->off;
    d.o_stride = out->stride;
    d.o_group = out->group > 0 ? out->group : 1;
    d.o_inner = out->inner;
    d.ldo = out->ld ? out->ld : n;
    d.bias = epi.bias ? epi.bias + epi.bias_off : nullptr;
    d.bias_stride = epi.bias_stride;
    d.mask = epi.mask ? epi.mask + epi.mask_off : nullptr;
    d.res = epi.residual ? epi.residual + epi.residual_off : nullptr;
    d.cs = out->p + epi.col_sum_off;
    d.cs_stride = epi.col_sum_stride;
    d.has_cs = epi.has_col_sum;
    d.relu = epi.relu;
    d.accumulate = epi.accumulate;
    d.f16 = f16;
    d.batch = batch;
    d.m = m;
    d.k = k;
    d.n = n;
    return d;
}

// Output tile and split-k of the any-shape kernel, by an estimate of the time.
// A workgroup alone on its CU takes `alone` us per k-stage (its matrix-core time
// plus the LDS round and barrier that nothing hides); W workgroups per CU
// overlap and take W `shared` per stage; `lead` stages stand for each
// workgroup's first loads and its stores.  The constants are fitted to f32
// products from 64 x 80 x 64 (20 workgroups of 32 x 32: 5.0 us, 64 x 64: 8.2) to
// 3001 x 1003 x 2000 (32 x 32: 150 us, 64 x 64: 120, 128 x 128: 152) and agree with
// them to about 15 %; the f16 ones, where a stage is bound by its loads and
// conversions, to f16 shapes.  (f32 tiles of 128 x 64 at 1.28 us a stage and f16
// ones of 128 x 128 at 1.3 are never better than twice as many of half the size.)
// Split-k as the reference allows it (matmul.rs:117-123): no epilogue but +=,
// packed out; each slice at least 4 k-stages, the partials summed by a launch of
// its own.
TileCfg plan_tiles(bool f16, bool ta, bool tb, const st_epilogue &epi, const st_matref *out, int64_t batch, int64_t m, int64_t k,
                   int64_t n) {
    struct Cand {
        int bm, bn;
        double alone, shared, lead;  // us per stage (32 deep in f32, 64 in f16)
    };
    // 32 x 32 tiles of operands whose rows are contiguous load with a quarter of the threads.
    const double narrow = ta && !tb ? 1.45 : ta || !tb ? 1.1 : 1.0;
    const Cand cands32[] = {{128, 128, 2.46, 2.05, 3.0}, {64, 64, 0.80, 0.59, 3.0}, {32, 32, 0.36, 0.19 * narrow, 1.5}};
    const Cand cands16[] = {{128, 64, 0.76, 0.53, 8.0}, {64, 64, 0.56, 0.33, 8.0}, {32, 32, 0.29, 0.145, 8.0}};
    const int BK = f16 ? 64 : 32;
    const bool epi_free = !epi.bias && !epi.relu && !epi.mask && !epi.residual;
    const bool packed_out = (out->ld == 0 || out->ld == n) && out->group <= 1;
    const int64_t cus = 256;
    // Only products whose 64 x 64 tiles leave CUs idle are split, into slices
    // that give every CU one or, for small outputs, more (8 MB of partials).
    const int64_t tiles64 = batch * cdiv(m, 64) * cdiv(n, 64);
    int64_t most = 1;
    if (epi_free && packed_out && tiles64 < cus) {
        const int64_t part = (int64_t)sizeof(float) * batch * (m * n + (epi.has_col_sum ? n : 0));
        most = std::max<int64_t>(1, std::min<int64_t>(std::max(cdiv(cus, tiles64), (8 << 20) / part), k / (4 * BK)));
    }
    const int64_t S = std::max<int64_t>(1, cdiv(k, BK));  // k-stages
    TileCfg best = {32, 32, 1, S * BK};
    double best_t = -1;
    for (const Cand &c : f16 ? cands16 : cands32) {
        if (c.bm > 32 && (m < c.bm || n < c.bn)) continue;  // (see WHOLE)
        const int64_t tiles = batch * cdiv(m, c.bm) * cdiv(n, c.bn);
        const double alone = c.alone, shared = c.shared, lead = c.lead;
        auto time = [&](int64_t sp, int64_t stages) {
            double t = ((double)stages + lead) * std::max(alone, (double)cdiv(tiles * sp, cus) * shared);
            if (sp > 1) t += 3.0 + 8.0 * (double)(sp * batch * m * n) / 4e6;
            return t;
        };
        int64_t c_sp = 1, c_stages = S;
        double c_t = time(1, S);
        // The best slice count without trying them all (k / 128 of them for a dot product): by rounds w of
        // workgroups over the CUs.  No count in round w takes less than `shared` times all its stages and leads
        // spread over the CUs, which grows with w; within a round more slices are shorter, and fewer save only
        // partials, so the walk down from the most of them soon ends.
        for (int64_t w = cdiv(2 * tiles, cus); most > 1; w++) {
            if (shared * ((double)(S * tiles) / (double)cus + lead * (double)w) + 3.0 > c_t) break;
            const int64_t lo = std::max<int64_t>(2, cus * (w - 1) / tiles + 1), hi = std::min(most, cus * w / tiles);
            if (lo > most) break;
            for (int64_t sp = hi; sp >= lo; sp--) {
                const int64_t stages = cdiv(S, sp);
                sp = cdiv(S, stages);  // the fewest slices of that length
                if (sp < lo || ((double)stages + lead) * std::max(alone, (double)w * shared) + 3.0 > c_t) break;
                const double t = time(sp, stages);
                if (t < c_t || (t == c_t && sp < c_sp)) {
                    c_t = t;
                    c_sp = sp;
                    c_stages = stages;
                }
            }
        }
        if (best_t < 0 || c_t < best_t) {
            best_t = c_t;
            best = {c.bm, c.bn, c_sp, c_stages * BK};
        }
    }
    return best;
}

// The limits of the any-shape kernel: its grid's, 31-bit tile numbers, and
// the rows that it has always taken.
constexpr int64_t ANY_SHAPE_ROWS = 65535 * 128;

st_status check_any_shape(const TileCfg &tc, int64_t batch, int64_t m, int64_t n) {
    if (batch * tc.splits > 65535)
        return st::fail(ST_ERR_INVALID, "batch %lld too large for one launch", (long long)batch);
    if (m > ANY_SHAPE_ROWS)
        return st::fail(ST_ERR_INVALID, "m = %lld: the any-shape kernel takes at most %lld rows", (long long)m,
                        (long long)ANY_SHAPE_ROWS);
    if (cdiv(n, tc.bn) * cdiv(m, tc.bm) > INT32_MAX)
        return st::fail(ST_ERR_INVALID, "m = %lld x n = %lld: too many tiles for one launch", (long long)m,
                        (long long)n);
    return ST_OK;
}

// What gemm_impl launches for a call that it accepts and that has work to do.
enum { PLAN_ANY_SHAPE = 0, PLAN_DMA = 1, PLAN_GROUP = 2 };

struct CallPlan {
    int kernel;
    TileCfg tc;  // any-shape kernel
    size_t scratch;
};

CallPlan plan_call(const st_matref *a, const st_matref *b, const st_matref *out, int64_t batch, int64_t m, int64_t k,
                   int64_t n, const st_epilogue &epi, bool use_f16) {
    const bool f16 = f16_route(use_f16, epi, b, m, k, n);
    const st::DmaGemm d = make_dma(a, b, out, batch, m, k, n, epi, f16);
    if (st::group_of_one(d)) return {PLAN_GROUP, {}, st::gemm_group_scratch(&d, 1, f16, true)};
    if (st::gemm_dma_takes(d)) return {PLAN_DMA, {}, st::gemm_dma_scratch(d)};
    const TileCfg tc = plan_tiles(f16, a->trans, b->trans, epi, out, batch, m, k, n);
    if (tc.splits <= 1) return {PLAN_ANY_SHAPE, tc, 0};
    return {PLAN_ANY_SHAPE, tc, sizeof(float) * (size_t)(batch * tc.splits * (m * n + (epi.has_col_sum ? n : 0)))};
}

// Bytes of split-k scratch gemm_impl would request for these arguments (0
// when it would request none or refuse them).
size_t gemm_impl_scratch(const st_matref *a, const st_matref *b, const st_matref *out, int64_t batch, int64_t m,
                         int64_t k, int64_t n, const st_epilogue &epi, bool use_f16) {
    if (!a || !b || !out || !a->p || !b->p || !out->p || out->trans || batch <= 0 || m <= 0 || n <= 0 || k <= 0)
        return 0;
    return plan_call(a, b, out, batch, m, k, n, epi, use_f16).scratch;
}

st_status gemm_impl(const st_matref *a, const st_matref *b, const st_matref *out, int64_t batch, int64_t m,
                    int64_t k, int64_t n, const st_epilogue *epi_in, bool use_f16, hipStream_t stream) {
    st::clear_error();
    st_status s;
    if ((s = check_call(a, b, out, batch, m, k, n))) return s;
    st_epilogue epi;
    std::memset(&epi, 0, sizeof epi);
    if (epi_in) epi = *epi_in;
    if (batch == 0 || m == 0 || n == 0) return ST_OK;
    if (!st::device_ok()) return ST_ERR_NO_DEVICE;

    const bool f16 = f16_route(use_f16, epi, b, m, k, n);
    const int64_t ag = a->group > 0 ? a->group : 1, bg = b->group > 0 ? b->group : 1;
    const int64_t og = out->group > 0 ? out->group : 1;
    const int64_t lda = a->ld ? a->ld : (a->trans ? m : k);
    const int64_t ldb = b->ld ? b->ld : (b->trans ? k : n);
    const int64_t ldo = out->ld ? out->ld : n;

    // Tile-divisible, 16-byte aligned problems run on the LDS-DMA kernel, the
    // larger ones on the grouped kernel.
    {
        const st::DmaGemm d = make_dma(a, b, out, batch, m, k, n, epi, f16);
        if (st::group_of_one(d)) return st::gemm_group(&d, 1, f16, true, stream);
        st_status ds = ST_OK;
        if (st::gemm_dma(d, stream, &ds)) return ds;
    }

    const TileCfg tc = plan_tiles(f16, a->trans, b->trans, epi, out, batch, m, k, n);
    const int64_t splits = tc.splits, slice_k = tc.slice_k;
    if ((s = check_any_shape(tc, batch, m, n))) return s;

    GemmArgs g;
    std::memset(&g, 0, sizeof g);
    g.a = {a->p + a->off, a->stride, ag, a->inner, lda};
    g.b = {b->p + b->off, b->stride, bg, b->inner, ldb};
    g.m = (int32_t)m;
    g.n = (int32_t)n;
    g.k = (int32_t)k;
    g.splits = (int32_t)splits;
    g.slice_k = (int32_t)slice_k;

    float *partial = nullptr;
    if (splits > 1) {
        const size_t base = (size_t)(batch * splits * m * n);
        const size_t extra = epi.has_col_sum ? (size_t)(batch * splits * n) : 0;
        partial = static_cast<float *>(st::scratch(st::SCRATCH_SPLITK, (base + extra) * sizeof(float), stream));
        if (!partial) return st::scratch_status();
        g.out = partial;
        g.o_stride = m * n;
        g.o_group = 1;
        g.o_inner = 0;
        g.ldo = n;
        g.has_cs = epi.has_col_sum;
        g.cs = partial + base;
        g.cs_stride = n;
        g.cs_direct = 0;
    } else {
        g.out = out->p + out->off;
        g.o_stride = out->stride;
        g.o_group = og;
        g.o_inner = out->inner;
        g.ldo = ldo;
        g.bias = epi.bias ? epi.bias + epi.bias_off : nullptr;
        g.bias_stride = epi.bias_stride;
        g.mask = epi.mask ? epi.mask + epi.mask_off : nullptr;
        g.res = epi.residual ? epi.residual + epi.residual_off : nullptr;
        g.relu = epi.relu;
        g.accumulate = epi.accumulate;
        g.has_cs = epi.has_col_sum;
        g.cs = out->p + epi.col_sum_off;
        g.cs_stride = epi.col_sum_stride;
        g.cs_direct = 1;
    }

    const bool whole = m >= tc.bm && n >= tc.bn;
    const KernelFn fn = pick_kernel(tc, f16, a->trans, b->trans, whole);
    // Rows of 2^23 workgroups (a grid has fewer than 2^32 threads along x).
    const int64_t tiles = cdiv(n, tc.bn) * cdiv(m, tc.bm), gx = std::min<int64_t>(tiles, 1 << 23);
    dim3 grid((unsigned)gx, (unsigned)cdiv(tiles, gx), (unsigned)(batch * splits));
    hipLaunchKernelGGL(fn, grid, dim3(THREADS), 0, stream, g);
    ST_LAUNCH_CHECK();

    if (splits > 1) {
        const int64_t len = m * n;
        const int64_t total = batch * (len + (epi.has_col_sum ? n : 0));
        hipLaunchKernelGGL(k_split_sum, dim3((unsigned)cdiv(total, 256)), dim3(256), 0, stream, partial,
                           out->p + out->off, len, (int32_t)splits, out->stride, batch, (int32_t)epi.accumulate,
                           epi.has_col_sum ? partial + batch * splits * len : nullptr, out->p + epi.col_sum_off,
                           epi.col_sum_stride, n);
        ST_LAUNCH_CHECK();
    }
    return ST_OK;
}

}  // namespace

extern "C" int32_t st_f16_enabled(void) {
    static const int32_t on = [] {
        const char *v = std::getenv("TRAIN_F16");
        return (v && std::strcmp(v, "0") == 0) ? 0 : 1;
    }();
    return on;
}

extern "C" st_status st_matmul(const st_matref *a, const st_matref *b, const st_matref *out, int64_t batch,
                               int64_t m, int64_t k, int64_t n, const st_epilogue *epi, st_stream stream) {
    return gemm_impl(a, b, out, batch, m, k, n, epi, st_f16_enabled() != 0, st::stream_of(stream));
}

extern "C" st_status st_matmul_f32(const st_matref *a, const st_matref *b, const st_matref *out, int64_t batch,
                                   int64_t m, int64_t k, int64_t n, const st_epilogue *epi, st_stream stream) {
    return gemm_impl(a, b, out, batch, m, k, n, epi, false, st::stream_of(stream));
}

extern "C" st_status st_matmul_with(const st_matref *a, const st_matref *b, const st_matref *out,
                                    int64_t batch, int64_t m, int64_t k, int64_t n, const st_epilogue *epi,
                                    int32_t use_f16, st_stream stream) {
    return gemm_impl(a, b, out, batch, m, k, n, epi, use_f16 != 0, st::stream_of(stream));
}

extern "C" st_status st_matmul_plan(const st_matref *a, const st_matref *b, const st_matref *out, int64_t batch,
                                    int64_t m, int64_t k, int64_t n, const st_epilogue *epi_in, int32_t use_f16,
                                    int64_t *plan) {
    st::clear_error();
    if (!plan) return st::fail(ST_ERR_INVALID, "plan is NULL");
    const st_status s = check_call(a, b, out, batch, m, k, n);
    if (s) return s;
    st_epilogue epi;
    std::memset(&epi, 0, sizeof epi);
    if (epi_in) epi = *epi_in;
    std::memset(plan, 0, 5 * sizeof *plan);
    if (batch == 0 || m == 0 || n == 0) return ST_OK;
    const CallPlan c = plan_call(a, b, out, batch, m, k, n, epi, use_f16 != 0);
    plan[0] = c.kernel;
    if (c.kernel == PLAN_ANY_SHAPE) {
        const st_status r = check_any_shape(c.tc, batch, m, n);
        if (r) return r;
        plan[1] = c.tc.bm;
        plan[2] = c.tc.bn;
        plan[3] = c.tc.splits;
    }
    plan[4] = (int64_t)c.scratch;
    return ST_OK;
}

extern "C" st_status st_matmul_grouped(const st_gemm *gemms, int64_t count, st_stream stream) {
    st::clear_error();
    if (count < 0 || (count > 0 && !gemms)) return st::fail(ST_ERR_INVALID, "grouped GEMM: bad count or NULL array");
    for (int64_t i = 0; i < count; i++) {
        const st_gemm &g = gemms[i];
        const st_status s = check_call(&g.a, &g.b, &g.out, g.batch, g.m, g.k, g.n);
        if (s) {
            const std::string msg = st_last_error();
            return st::fail(s, "GEMM %lld of the group: %s", (long long)i, msg.c_str());
        }
    }
    if (count == 0) return ST_OK;
    if (!st::device_ok()) return ST_ERR_NO_DEVICE;
    const hipStream_t s = st::stream_of(stream);
    std::vector<st::DmaGemm> elig[2];  // by route (f32, f16)
    std::vector<int64_t> rest;
    for (int64_t i = 0; i < count; i++) {
        const st_gemm &g = gemms[i];
        if (g.batch == 0 || g.m == 0 || g.n == 0) continue;
        const bool f16 = f16_route(g.use_f16 != 0, g.epi, &g.b, g.m, g.k, g.n);
        const st::DmaGemm d = make_dma(&g.a, &g.b, &g.out, g.batch, g.m, g.k, g.n, g.epi, f16);
        if (st::group_eligible(d))
            elig[f16 ? 1 : 0].push_back(d);
        else
            rest.push_back(i);
    }
    // 256-row tiles only when the route's GEMMs give every CU at least one of
    // them; a small group (a single Linear backward) keeps 128-row tiles.
    std::vector<st::DmaGemm> grp[4];  // route + 2 * (256-row tiles)
    for (int f = 0; f < 2; f++) {
        int64_t tall_tiles = 0;
        for (const st::DmaGemm &d : elig[f])
            if (st::group_tall(d)) tall_tiles += d.batch * (d.m / 256) * (d.n / 128);
        const bool use_tall = tall_tiles >= 256;
        for (const st::DmaGemm &d : elig[f]) grp[f + 2 * (use_tall && st::group_tall(d))].push_back(d);
    }
    // All or nothing: the launches below share the split-k scratch one after
    // another, so the largest need among them is requested before the first
    // launch.  A refusal (a fixed scratch too small, an arena that cannot grow
    // under graph capture or out of memory) then leaves every output as it
    // was; every later request fits what is already there.
    size_t need = 0;
    for (int f = 0; f < 4; f++)
        for (size_t c = 0; c < grp[f].size(); c += st::GROUP_MAX) {
            const int cnt = (int)std::min<size_t>(st::GROUP_MAX, grp[f].size() - c);
            need = std::max(need, st::gemm_group_scratch(grp[f].data() + c, cnt, (f & 1) != 0, (f & 2) != 0));
        }
    for (const int64_t i : rest) {
        const st_gemm &g = gemms[i];
        need = std::max(need, gemm_impl_scratch(&g.a, &g.b, &g.out, g.batch, g.m, g.k, g.n, g.epi, g.use_f16 != 0));
    }
    if (need && !st::scratch(st::SCRATCH_SPLITK, need, s)) return st::scratch_status();
    for (int f = 0; f < 4; f++)
        for (size_t c = 0; c < grp[f].size(); c += st::GROUP_MAX) {
            const int cnt = (int)std::min<size_t>(st::GROUP_MAX, grp[f].size() - c);
            const st_status r = st::gemm_group(grp[f].data() + c, cnt, (f & 1) != 0, (f & 2) != 0, s);
            if (r) return r;
        }
    for (const int64_t i : rest) {
        const st_gemm &g = gemms[i];
        const st_status r = gemm_impl(&g.a, &g.b, &g.out, g.batch, g.m, g.k, g.n, &g.epi, g.use_f16 != 0, s);
        if (r) return r;
    }
    return ST_OK;
}

extern "C" st_status st_ndarray_matmul(const float *a, const float *b, float *out, int64_t m, int64_t k,
                                       int64_t n) {
    st::clear_error();
    if (!a || !b || !out) return st::fail(ST_ERR_INVALID, "NULL host buffer");
    if (m < 0 || k < 0 || n < 0) return st::fail(ST_ERR_INVALID, "negative shape");
    if (m == 0 || n == 0) return ST_OK;
    if (!st::device_ok()) return ST_ERR_NO_DEVICE;
    hipStream_t s;
    ST_HIP_CHECK(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    // Split-k partials in buffers of this call's own (freed when it returns):
    // concurrent calls never share the library's arena.
    st::ScratchScope private_scratch;
    float *da = nullptr, *db = nullptr, *dc = nullptr;
    st_status rc = ST_OK;
    const size_t ba = sizeof(float) * (size_t)(m * k), bb = sizeof(float) * (size_t)(k * n),
                 bc = sizeof(float) * (size_t)(m * n);
    auto cleanup = [&] {
        (void)hipStreamSynchronize(s);
        if (da) (void)hipFree(da);
        if (db) (void)hipFree(db);
        if (dc) (void)hipFree(dc);
        (void)hipStreamDestroy(s);
    };
    if (hipMalloc(&da, ba ? ba : 4) != hipSuccess || hipMalloc(&db, bb ? bb : 4) != hipSuccess ||
        hipMalloc(&dc, bc) != hipSuccess) {
        (void)hipGetLastError();
        cleanup();
        return st::fail(ST_ERR_OOM, "device allocation for NdArray::matmul failed");
    }
    if ((ba && hipMemcpyAsync(da, a, ba, hipMemcpyHostToDevice, s) != hipSuccess) ||
        (bb && hipMemcpyAsync(db, b, bb, hipMemcpyHostToDevice, s) != hipSuccess)) {
        cleanup();
        return st::fail(ST_ERR_HIP, "host to device copy failed");
    }
    st_matref ra{da, 0, 0, 0, 0, 0, 1, 0}, rb{db, 0, 0, 0, 0, 0, 1, 0}, rc_{dc, 0, 0, 0, 0, 0, 1, 0};
    if (k == 0) {
        if (hipMemsetAsync(dc, 0, bc, s) != hipSuccess) rc = st::fail(ST_ERR_HIP, "hipMemsetAsync failed");
    } else {
        rc = gemm_impl(&ra, &rb, &rc_, 1, m, k, n, nullptr, false, s);
    }
    if (rc == ST_OK && hipMemcpyAsync(out, dc, bc, hipMemcpyDeviceToHost, s) != hipSuccess)
        rc = st::fail(ST_ERR_HIP, "device to host copy failed");
    if (rc == ST_OK && hipStreamSynchronize(s) != hipSuccess) rc = st::fail(ST_ERR_HIP, "stream synchronize failed");
    cleanup();
    return rc;
}
