// K5: f32 / f64 GEMM on the matrix cores, for the general matmuls of the
// path: the `eval` matmul node (executor.zig:199-326, matmul.zig) with the
// fused bias + activation epilogue of FusedMatmulEpilogueKernel
// (fusion/codegen.zig:78-147), and the ONNX MatMul / Gemm operators
// (onnx/executor.zig:1489-1990, 4561-4634).
//
//   Y[b] = ops( alpha * opA(A[b]) opB(B[b]) ) + beta * C
//
// Products are exact and summed in the operand precision by
// v_mfma_f32_16x16x4_f32 / v_mfma_f64_16x16x4_f64 (157 / 79 TFLOP/s dense
// on MI355X), so the result is the reference's f32 (f64) matmul up to the
// order of the k sum.
//
// Design:
//   - Output tiles of 128 x 128, 64 x 128, 64 x 64 or 32 x 32 per 256-thread
//     block (choose_tile): the large ones reuse each operand most, the small
//     ones leave fewer CUs idle.  Four waves split the tile, or (32 x 32 in
//     f32) the k steps of a stage, their sums meeting in LDS at the end.
//   - k runs in stages of 16 to 128, the deeper the smaller the tile, so that
//     a stage holds about as many matrix instructions (2 048 cycles a wave;
//     32 x 32: 1 024) as a load takes to arrive.  Operands are loaded into
//     registers with bounds checks (zero outside the matrix, 16-byte vector
//     loads where the rows allow) while the stage before computes, then
//     written to a double-buffered LDS tile.
//   - The LDS tile keeps the stored operand's contiguous axis: [row][k] for a
//     k-contiguous operand, [k][row] for a row-contiguous one, so both are
//     written as they were loaded, 16 bytes at a time.  A lane's MFMA operand
//     for k step s of a 16-wide group is k = 4 (lane / 16) + s, the same for
//     both operands: one 16-byte (f32) or 32-byte (f64) read of a [row][k]
//     tile, four element reads of a [k][row] tile.  The pitches spread a
//     wave's reads over all banks.
//   - The MFMA takes B's columns as its A operand, so each lane holds four
//     output columns of one row (consecutive ones in f32: 16-byte stores of
//     Y rows).
//   - Fused ops run on the sums before they are stored: the lane's sums pass
//     through the operand tiles' LDS into a rolled loop, so the code of the
//     ops exists once and the sums can stay in registers during the products.
#include "common.h"
#include "ew_program.h"  // unary_op<T>: the op semantics of the elementwise engine

#include <cmath>
#include <cstring>

namespace {

using tzh_ew::unary_op;

constexpr int kThreads = 256;
constexpr int kMaxEpiOps = 4;

typedef double f64x4_t __attribute__((ext_vector_type(4)));

template <typename T>
struct Vec4 {
    using type = f32x4_t;
};
template <>
struct Vec4<double> {
    using type = f64x4_t;
};

// One tile shape: BM x BN outputs, k stages of BK, KW waves over each
// stage's k (the other 4 / KW split the tile 2 x 2).
template <typename T, int BM_, int BN_, int BK_, int KW_>
struct Tile {
    static constexpr int BM = BM_, BN = BN_, BK = BK_, KW = KW_;
    static constexpr int WM = KW == 1 ? 2 : 1, WN = KW == 1 ? 2 : 1;
    static constexpr int MT = BM / WM / 16, NT = BN / WN / 16;  // 16 x 16 MFMA tiles of a wave
    static_assert(WM * WN * KW == 4 && BK % (16 * KW) == 0, "four waves, whole 16-wide k groups each");
    static_assert(MT >= 1 && NT >= 1, "whole MFMA tiles");
    static_assert(KW == 1 || MT * NT == KW, "split k: each wave finishes one MFMA tile");
};
// LDS pitches in elements: a [row][k] tile's rows start on sixteen different
// bank groups (BK + 4 f32, BK + 2 f64); a [k][row] tile's four k rows of a
// read on different ones (rows + 4).
template <typename T>
constexpr int pitch_k(int bk) {
    return bk + (sizeof(T) == 4 ? 4 : 2);
}
constexpr int pitch_r(int rows) { return rows + 4; }
template <typename T>
constexpr int operand_elems(int rows, int bk, bool kc) {
    return kc ? rows * pitch_k<T>(bk) : bk * pitch_r(rows);
}

template <typename T>
struct GemmArgs {
    int64_t m, n, k;
    int64_t lda, ldb, ldy;  // row pitches (elements) of the stored A, B and of Y
    int64_t tiles_m, tiles_n;
    int32_t nb;             // batch dimensions of the output
    int32_t vec_a, vec_b;   // 1: every 4-element run of a stored row starts 16-byte aligned
    int32_t vec_y;
    int64_t batch_shape[TZH_MAX_RANK];
    int64_t a_bstride[TZH_MAX_RANK], b_bstride[TZH_MAX_RANK];  // 0 where broadcast
    int64_t y_bstride;
    T alpha, beta;
    const T *c;             // beta * c[i * c_rs + j * c_cs], or null
    int64_t c_rs, c_cs;
    const T *bias;          // [n], added where ops[] holds TZH_OP_ADD
    int32_t n_ops;
    int32_t ops[kMaxEpiOps];
};

// Four consecutive elements of one stored row starting at p; element j is
// used only when j < valid (0..4).  `vec`: the run is 16-byte aligned.
template <typename T>
__device__ __forceinline__ void load4(const T *p, int valid, bool vec, T (&v)[4]) {
    if (vec && valid == 4) {
        if constexpr (sizeof(T) == 4) {
            const f32x4_t x = *(const f32x4_t *)p;
            v[0] = x[0], v[1] = x[1], v[2] = x[2], v[3] = x[3];
        } else {
            typedef double f64x2_t __attribute__((ext_vector_type(2)));
            const f64x2_t x = *(const f64x2_t *)p, y = *(const f64x2_t *)(p + 2);
            v[0] = x[0], v[1] = x[1], v[2] = y[0], v[3] = y[1];
        }
    } else {
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = j < valid ? p[j] : (T)0;
    }
}

// One operand tile (ROWS rows of m or n, BK k) per stage, in 4-element
// chunks.  KC: the stored operand is k-contiguous (rows of k); else
// row-contiguous (rows of m or n, one per k).
template <typename T, int ROWS, int BK, bool KC>
struct TileLoader {
    static constexpr int kChunks = ROWS * BK / 4 / kThreads;
    static constexpr int kPerRow = (KC ? BK : ROWS) / 4;  // chunks of one stored row
    static_assert(kChunks * 4 * kThreads == ROWS * BK, "whole chunks per thread");
    T v[kChunks][4];
    __device__ __forceinline__ void load(const T *X, int64_t ld, int64_t r0, int64_t R, int64_t k0, int64_t K,
                                         bool vec, int tid) {
#pragma unroll
        for (int c = 0; c < kChunks; c++) {
            const int q = tid + c * kThreads;
            // the chunk's stored row, its limit, and the same along the row
            const int64_t row = (KC ? r0 : k0) + q / kPerRow, col = (KC ? k0 : r0) + (q % kPerRow) * 4;
            const int64_t rows = KC ? R : K, cols = KC ? K : R;
            const int valid = row < rows ? (int)(cols - col < 4 ? (cols - col > 0 ? cols - col : 0) : 4) : 0;
            load4<T>(X + (valid > 0 ? row * ld + col : 0), valid, vec, v[c]);
        }
    }
    __device__ __forceinline__ void store(T *tile, int tid) const {
        constexpr int P = KC ? pitch_k<T>(BK) : pitch_r(ROWS);
#pragma unroll
        for (int c = 0; c < kChunks; c++) {
            const int q = tid + c * kThreads;
            T *d = tile + (q / kPerRow) * P + (q % kPerRow) * 4;
            if constexpr (sizeof(T) == 4) {
                *(f32x4_t *)d = f32x4_t{(float)v[c][0], (float)v[c][1], (float)v[c][2], (float)v[c][3]};
            } else {
#pragma unroll
                for (int j = 0; j < 4; j++) d[j] = v[c][j];
            }
        }
    }
};

// The four k steps (k = kk + s) of one lane's row of an operand tile.
template <typename T, int ROWS, int BK, bool KC>
__device__ __forceinline__ typename Vec4<T>::type fragment(const T *tile, int row, int kk) {
    if constexpr (KC) {
        return *(const typename Vec4<T>::type *)&tile[row * pitch_k<T>(BK) + kk];
    } else {
        constexpr int P = pitch_r(ROWS);
        const T *t = tile + kk * P + row;
        return typename Vec4<T>::type{t[0], t[P], t[2 * P], t[3 * P]};
    }
}

template <typename T>
__device__ __forceinline__ typename Vec4<T>::type mfma16(T a, T b, typename Vec4<T>::type c) {
    if constexpr (sizeof(T) == 4)
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// TA: A is stored [k][m] (else [m][k]); TB: B is stored [n][k] (else [k][n]).
template <typename T, bool TA, bool TB, typename TL>
__global__ void __launch_bounds__(kThreads) gemm_mfma_kernel(const T *__restrict__ A, const T *__restrict__ B,
                                                             T *__restrict__ Y, const GemmArgs<T> g) {
    using V4 = typename Vec4<T>::type;
    constexpr int BM = TL::BM, BN = TL::BN, BK = TL::BK, KW = TL::KW, MT = TL::MT, NT = TL::NT;
    constexpr int AE = operand_elems<T>(BM, BK, !TA), BE = operand_elems<T>(BN, BK, TB);
    __shared__ __attribute__((aligned(16))) T lds[2 * (AE + BE)];
    auto as = [&](int buf) __attribute__((always_inline)) { return lds + buf * AE; };
    auto bs = [&](int buf) __attribute__((always_inline)) { return lds + 2 * AE + buf * BE; };
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int wm = KW == 1 ? w & 1 : 0, wn = KW == 1 ? w >> 1 : 0, wk = KW == 1 ? 0 : w;

    const int64_t tiles = g.tiles_m * g.tiles_n;
    const int64_t bi = (int64_t)blockIdx.x / tiles, t = (int64_t)blockIdx.x % tiles;
    const int64_t m0 = t / g.tiles_n * BM, n0 = t % g.tiles_n * BN;
    int64_t ao = 0, bo = 0, rem = bi;
    for (int d = g.nb - 1; d >= 0; d--) {
        const int64_t i = rem % g.batch_shape[d];
        rem /= g.batch_shape[d];
        ao += i * g.a_bstride[d];
        bo += i * g.b_bstride[d];
    }
    const T *Ab = A + ao, *Bb = B + bo;
    T *Yb = Y + bi * g.y_bstride;

    TileLoader<T, BM, BK, !TA> la;  // A rows are m
    TileLoader<T, BN, BK, TB> lb;   // B rows are n
    V4 acc[NT][MT];
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
        for (int i = 0; i < MT; i++) acc[j][i] = V4{};

    const int64_t S = (g.k + BK - 1) / BK;
    if (S > 0) {
        la.load(Ab, g.lda, m0, g.m, 0, g.k, g.vec_a, tid);
        lb.load(Bb, g.ldb, n0, g.n, 0, g.k, g.vec_b, tid);
        la.store(as(0), tid);
        lb.store(bs(0), tid);
    }
    __syncthreads();
    const int r16 = lane & 15, k4 = 4 * (lane >> 4);
    constexpr int GW = BK / 16 / KW;  // 16-wide k groups of a wave per stage
    for (int64_t s = 0; s < S; s++) {
        const int buf = (int)(s & 1);
        if (s + 1 < S) {
            la.load(Ab, g.lda, m0, g.m, (s + 1) * BK, g.k, g.vec_a, tid);
            lb.load(Bb, g.ldb, n0, g.n, (s + 1) * BK, g.k, g.vec_b, tid);
        }
#pragma unroll
        for (int gk = 0; gk < GW; gk++) {
            const int kk = 16 * (wk * GW + gk) + k4;
            V4 af[MT], bf[NT];
#pragma unroll
            for (int i = 0; i < MT; i++)
                af[i] = fragment<T, BM, BK, !TA>(as(buf), wm * (BM / TL::WM) + i * 16 + r16, kk);
#pragma unroll
            for (int j = 0; j < NT; j++)
                bf[j] = fragment<T, BN, BK, TB>(bs(buf), wn * (BN / TL::WN) + j * 16 + r16, kk);
#pragma unroll
            for (int q = 0; q < 4; q++)
#pragma unroll
                for (int j = 0; j < NT; j++)
#pragma unroll
                    for (int i = 0; i < MT; i++) acc[j][i] = mfma16<T>(bf[j][q], af[i][q], acc[j][i]);
        }
        if (s + 1 < S) {
            la.store(as(buf ^ 1), tid);
            lb.store(bs(buf ^ 1), tid);
        }
        __syncthreads();
    }

    // Lane l holds, for row m = .. + l%16 of MFMA tile (j, i), accumulator
    // element e of column .. + col(e): v_mfma_f32_16x16x4_f32 gives lane l
    // rows 4 (l/16) + e of its D tile (four consecutive columns here),
    // v_mfma_f64_16x16x4_f64 rows l/16 + 4 e (measured on MI355X).
    const int cq = lane >> 4;
    auto col = [&](int e) __attribute__((always_inline)) { return sizeof(T) == 4 ? 4 * cq + e : cq + 4 * e; };
    // row and first column of MFMA tile (j, i) of this wave's part
    const int64_t mw = m0 + wm * (BM / TL::WM) + r16, nw = n0 + wn * (BN / TL::WN);
    auto put = [&](int64_t m, int64_t nb, const V4 &v) __attribute__((always_inline)) {
        if (m >= g.m) return;
        T *row = Yb + m * g.ldy + nb;
        if (sizeof(T) == 4 && g.vec_y && nb + col(3) < g.n) {
            *(f32x4_t *)(row + col(0)) = f32x4_t{(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (nb + col(e) < g.n) row[col(e)] = v[e];
        }
    };
    auto linear = [&](const V4 &a, int64_t m, int64_t nb) __attribute__((always_inline)) {
        V4 v;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            v[e] = g.alpha * a[e];
            if (g.c && m < g.m && nb + col(e) < g.n) v[e] += g.beta * g.c[m * g.c_rs + (nb + col(e)) * g.c_cs];
        }
        return v;
    };
    // the fused ops (bias adds and unary ops, in order), then beta * C
    auto finish = [&](const V4 &a, int64_t m, int64_t nb) __attribute__((always_inline)) {
        V4 v;
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = g.alpha * a[e];
        for (int o = 0; o < g.n_ops; o++) {
            if (g.ops[o] == TZH_OP_ADD) {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (nb + col(e) < g.n) v[e] += g.bias[nb + col(e)];
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) v[e] = unary_op<T>(g.ops[o], v[e]);
            }
        }
        if (g.c && m < g.m)
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (nb + col(e) < g.n) v[e] += g.beta * g.c[m * g.c_rs + (nb + col(e)) * g.c_cs];
        return v;
    };
    V4 *const slots = (V4 *)lds;  // [tile][thread]; every wave is past the last stage
    if constexpr (KW > 1) {
        // each wave adds up one MFMA tile from the KW waves' sums
        static_assert(KW * MT * NT * 64 * 4 <= 2 * (AE + BE), "the sums fit the operand tiles");
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int i = 0; i < MT; i++) slots[(w * MT * NT + j * MT + i) * 64 + lane] = acc[j][i];
        __syncthreads();
        V4 v = slots[w * 64 + lane];
#pragma unroll
        for (int k = 1; k < KW; k++) v += slots[(k * MT * NT + w) * 64 + lane];
        const int64_t m = m0 + (w % MT) * 16 + r16, nb = n0 + (w / MT) * 16;
        put(m, nb, g.n_ops ? finish(v, m, nb) : linear(v, m, nb));
    } else if (g.n_ops == 0) {
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < NT; j++)
                put(mw + i * 16, nw + j * 16, linear(acc[j][i], mw + i * 16, nw + j * 16));
    } else {
        // through LDS (each lane reads back what it wrote) into a rolled loop
        constexpr int kFit = 2 * (AE + BE) / (kThreads * 4) < 8 ? 4 : 8;
        constexpr int G = MT * NT < kFit ? MT * NT : kFit, JG = G / MT;  // tiles at a time, their j's
        static_assert(G % MT == 0 && NT % JG == 0 && G * kThreads * 4 <= 2 * (AE + BE), "groups of whole j's that fit");
#pragma unroll
        for (int j0 = 0; j0 < NT; j0 += JG) {
#pragma unroll
            for (int j = 0; j < JG; j++)
#pragma unroll
                for (int i = 0; i < MT; i++) slots[(j * MT + i) * kThreads + tid] = acc[j0 + j][i];
#pragma unroll 1
            for (int q = 0; q < G; q++) {
                const int64_t m = mw + (q % MT) * 16, nb = nw + (j0 + q / MT) * 16;
                put(m, nb, finish(slots[q * kThreads + tid], m, nb));
            }
        }
    }
}

// y[i] = a[i] * s (the scalar-operand MatMul of onnx/executor.zig:1545-1577);
// a == null: y[i] = 0 (the empty sums of k == 0)
template <typename T>
__global__ void scale_kernel(const T *__restrict__ a, T s, T *__restrict__ y, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = a ? a[i] * s : (T)0;
}

bool al16(const void *p) { return ((uintptr_t)p & 15) == 0; }

// Tile shapes, and the one a problem runs on: the least time by the number
// of tiles the busiest CU gets, each at its area over the share of the
// 128 x 128 tile's rate it reaches (in eighths; what the smaller reuse
// and the shorter stages cost).  Measured in f32, us, against 128 x 128
// tiles with k stages of 16 at every size (and fused ops re-reading Y):
//   4096 x 384 x 1536: 77 -> 55 (64 x 128), with bias and GELU 137 -> 63;
//   2048 x 2048 x 2048: 229 -> 187 (128 x 128);
//   1000 x 1001 x 1003 with bias: 182 -> 70 (64 x 64);
//   19 x 1125 x 247 with bias: 162 -> 25; 128 x 384 x 1152 with bias and
//   GELU: 89 -> 9; 1 x 2048 x 2048: 251 -> 30 (32 x 32).
// f64 likewise: 4096 x 384 x 1536 152 -> 105, 300 x 2000 x 300 366 -> 51.
struct TileShape {
    int bm, bn, rate8;
};
constexpr TileShape kTileShapes[] = {{128, 128, 8}, {64, 128, 8}, {64, 64, 7}, {32, 32, 4}};

int choose_tile(int num_cus, int64_t m, int64_t n, int64_t batches) {
    int best = 0;
    double best_cost = 0;
    for (int i = 0; i < 4; i++) {
        const TileShape &t = kTileShapes[i];
        const double tiles = (double)((m + t.bm - 1) / t.bm) * (double)((n + t.bn - 1) / t.bn) * (double)batches;
        const double cost = std::ceil(tiles / num_cus) * t.bm * t.bn / t.rate8;
        if (i > 0 && tiles * kThreads > 4294967295.0) break;  // past what HIP launches
        if (i == 0 || cost < best_cost) best = i, best_cost = cost;
    }
    return best;
}

template <typename T, typename TL>
void launch_tile(hipStream_t st, bool a_trans, bool b_trans, const T *A, const T *B, T *Y, const GemmArgs<T> &g,
                 unsigned blocks) {
    const dim3 grid(blocks);
    if (a_trans && b_trans)
        hipLaunchKernelGGL((gemm_mfma_kernel<T, true, true, TL>), grid, dim3(kThreads), 0, st, A, B, Y, g);
    else if (a_trans)
        hipLaunchKernelGGL((gemm_mfma_kernel<T, true, false, TL>), grid, dim3(kThreads), 0, st, A, B, Y, g);
    else if (b_trans)
        hipLaunchKernelGGL((gemm_mfma_kernel<T, false, true, TL>), grid, dim3(kThreads), 0, st, A, B, Y, g);
    else
        hipLaunchKernelGGL((gemm_mfma_kernel<T, false, false, TL>), grid, dim3(kThreads), 0, st, A, B, Y, g);
}

}  // namespace

// The launch behind every entry point below and the eval planner's matmul
// node: a_trans / b_trans say how A and B are stored (see gemm_mfma_kernel).
// d describes the batch and the epilogue; pointers are device pointers.
int tzh_gemm_fp_launch(hipStream_t st, int num_cus, int32_t dtype, bool a_trans, bool b_trans, const void *a,
                       const void *b, void *y, const tzh_gemm_desc &d) {
    if (dtype != TZH_F32 && dtype != TZH_F64) return tzh_fail(TZH_ERR_UNSUPPORTED_DTYPE, "GEMM dtype must be F32 or F64");
    if (d.m < 0 || d.n < 0 || d.k < 0) return tzh_fail(TZH_ERR_INVALID_ARGS, "negative GEMM dimension");
    if (d.nb < 0 || d.nb > TZH_MAX_RANK) return tzh_fail(TZH_ERR_INVALID_ARGS, "batch rank %d out of range", d.nb);
    if (d.n_ops < 0 || d.n_ops > kMaxEpiOps) return tzh_fail(TZH_ERR_INVALID_ARGS, "%d epilogue ops (at most %d)", d.n_ops, kMaxEpiOps);
    int64_t batches = 1;
    for (int i = 0; i < d.nb; i++) {
        if (d.batch_shape[i] < 0) return tzh_fail(TZH_ERR_INVALID_ARGS, "negative batch dimension");
        batches *= d.batch_shape[i];
    }
    if (d.m == 0 || d.n == 0 || batches == 0) return TZH_OK;
    for (int o = 0; o < d.n_ops; o++) {
        const int op = d.ops[o];
        if (op == TZH_OP_ADD && !d.bias) return tzh_fail(TZH_ERR_INVALID_ARGS, "bias add without a bias");
        if (op != TZH_OP_ADD && !tzh_ew::unary_ok(op))
            return tzh_fail(TZH_ERR_UNSUPPORTED_OP, "epilogue op %d is not a unary op or a bias add", op);
    }
    const int ts = choose_tile(num_cus, d.m, d.n, batches);
    const int64_t tm = (d.m + kTileShapes[ts].bm - 1) / kTileShapes[ts].bm;
    const int64_t tn = (d.n + kTileShapes[ts].bn - 1) / kTileShapes[ts].bn;
    if (batches > ((int64_t)1 << 31) / (tm * tn)) return tzh_fail(TZH_ERR_TOO_LARGE, "GEMM grid too large");
    const int64_t vec_e = dtype == TZH_F32 ? 4 : 2;  // elements per 16 bytes
    auto vec_ok = [&](const void *p, int64_t ld, const int64_t *bstride) {
        if (!al16(p) || ld % vec_e) return 0;
        for (int i = 0; i < d.nb; i++)
            if (bstride[i] % vec_e) return 0;
        return 1;
    };
    if (!y || (d.k > 0 && (!a || !b))) return tzh_fail(TZH_ERR_INVALID_ARGS, "null GEMM operand");  // k == 0 reads neither
    auto fill = [&](auto tag) -> int {
        using T = decltype(tag);
        GemmArgs<T> g{};
        g.m = d.m, g.n = d.n, g.k = d.k, g.lda = d.lda, g.ldb = d.ldb, g.ldy = d.ldy;
        g.tiles_m = tm, g.tiles_n = tn, g.nb = d.nb;
        g.vec_a = vec_ok(a, d.lda, d.a_bstride);
        g.vec_b = vec_ok(b, d.ldb, d.b_bstride);
        g.vec_y = al16(y) && d.ldy % vec_e == 0 && (d.nb == 0 || d.y_bstride % vec_e == 0);
        for (int i = 0; i < d.nb; i++) {
            g.batch_shape[i] = d.batch_shape[i];
            g.a_bstride[i] = d.a_bstride[i];
            g.b_bstride[i] = d.b_bstride[i];
        }
        g.y_bstride = d.y_bstride;
        g.alpha = (T)d.alpha, g.beta = (T)d.beta;
        g.c = (const T *)d.c, g.c_rs = d.c_rs, g.c_cs = d.c_cs;
        g.bias = (const T *)d.bias;
        g.n_ops = d.n_ops;
        for (int o = 0; o < d.n_ops; o++) g.ops[o] = d.ops[o];
        const unsigned blocks = (unsigned)(batches * tm * tn);
        const T *A = (const T *)a, *B = (const T *)b;
        T *Y = (T *)y;
        constexpr int E = sizeof(T) == 4 ? 2 : 1;  // k stages half as deep in f64
        switch (ts) {
        case 0: launch_tile<T, Tile<T, 128, 128, 16, 1>>(st, a_trans, b_trans, A, B, Y, g, blocks); break;
        case 1: launch_tile<T, Tile<T, 64, 128, 16 * E, 1>>(st, a_trans, b_trans, A, B, Y, g, blocks); break;
        case 2: launch_tile<T, Tile<T, 64, 64, 32 * E, 1>>(st, a_trans, b_trans, A, B, Y, g, blocks); break;
        default:
            // short k: one stage of 32 or 64 and a quarter or half of the LDS,
            // so eight or four blocks a CU in place of two (f32, us, 128 x 128
            // tiles / stages of 128 / of 32: 100000 x 8 x 8 16 / 30 / 9, 2000
            // products of 40 x 8 x 20 23 / 38 / 11)
            if (d.k <= 32) {
                launch_tile<T, Tile<T, 32, 32, 32, 1>>(st, a_trans, b_trans, A, B, Y, g, blocks);
                break;
            }
            // split k in f32 only: f64 keeps the one order of its sums
            if constexpr (sizeof(T) == 4) {
                if (d.split_k) {
                    if (d.k <= 64) launch_tile<T, Tile<T, 32, 32, 64, 4>>(st, a_trans, b_trans, A, B, Y, g, blocks);
                    else launch_tile<T, Tile<T, 32, 32, 64 * E, 4>>(st, a_trans, b_trans, A, B, Y, g, blocks);
                    break;
                }
            }
            launch_tile<T, Tile<T, 32, 32, 64 * E, 1>>(st, a_trans, b_trans, A, B, Y, g, blocks);
            break;
        }
        TZH_LAUNCHED("gemm_mfma_kernel");
        return TZH_OK;
    };
    return dtype == TZH_F32 ? fill(0.0f) : fill(0.0);
}

// ONNX Gemm (onnx/executor.zig:4561-4634): Y[m,n] = alpha * op(A) op(B) +
// beta * C, C broadcast from [c_rows, c_cols] (rows 1 or m, columns 1 or n;
// NULL: no C); lda / ldb are the stored row pitches (the reference's
// a.shape[1] / b.shape[1]); Y is contiguous [m, n].
extern "C" int tzh_gemm_f32(tzh_ctx *ctx, int32_t trans_a, int32_t trans_b, int64_t m, int64_t n, int64_t k,
                            float alpha, const float *a, int64_t lda, const float *b, int64_t ldb, float beta,
                            const float *c, int64_t c_rows, int64_t c_cols, float *y) {
    tzh_clear_error();
    TZH_TRY(tzh_ctx_enter(ctx));
    if (m < 0 || n < 0 || k < 0) return tzh_fail(TZH_ERR_INVALID_ARGS, "negative Gemm dimension");
    if (m == 0 || n == 0) return TZH_OK;
    if (k > 0 && (lda < (trans_a ? m : k) || ldb < (trans_b ? k : n)))
        return tzh_fail(TZH_ERR_INVALID_ARGS, "row pitch smaller than the stored row");
    if (c && !((c_rows == 1 || c_rows == m) && (c_cols == 1 || c_cols == n)))
        return tzh_fail(TZH_ERR_SHAPE, "C of shape [%lld, %lld] does not broadcast to [%lld, %lld]",
                        (long long)c_rows, (long long)c_cols, (long long)m, (long long)n);
    tzh_gemm_desc d{};
    d.m = m, d.n = n, d.k = k, d.lda = lda, d.ldb = ldb, d.ldy = n;
    d.alpha = alpha, d.beta = beta;
    d.c = c, d.c_rs = c && c_rows > 1 ? c_cols : 0, d.c_cs = c && c_cols > 1 ? 1 : 0;
    return tzh_gemm_fp_launch(ctx->stream, ctx->num_cus, TZH_F32, trans_a != 0, trans_b != 0, a, b, y, d);
}

// ONNX MatMul (onnx/executor.zig:1489-1990): NumPy matmul of A (a_ndim >= 1)
// and B, batch dimensions broadcast, a 1-D A a row and a 1-D B a column
// whose unit dimension the result drops; B of shape [] or [1] scales A
// elementwise (executor.zig:1545-1577); any zero dimension gives an empty
// (or, with k == 0, zero) result.  Writes the result shape to y_shape /
// *y_ndim (host, room for 8), and the result to y unless y is NULL.
extern "C" int tzh_matmul_nd(tzh_ctx *ctx, int32_t dtype, const void *a, const int64_t *a_shape, int32_t a_ndim,
                             const void *b, const int64_t *b_shape, int32_t b_ndim, void *y, int64_t *y_shape,
                             int32_t *y_ndim) {
    tzh_clear_error();
    TZH_TRY(tzh_ctx_enter(ctx));
    if (dtype != TZH_F32 && dtype != TZH_F64) return tzh_fail(TZH_ERR_UNSUPPORTED_DTYPE, "MatMul dtype must be F32 or F64");
    if (!y_shape || !y_ndim || a_ndim < 0 || b_ndim < 0 || a_ndim > TZH_MAX_RANK || b_ndim > TZH_MAX_RANK ||
        (a_ndim && !a_shape) || (b_ndim && !b_shape))
        return tzh_fail(TZH_ERR_INVALID_ARGS, "bad MatMul shape arguments");
    int64_t an = 1;
    for (int i = 0; i < a_ndim; i++) {
        if (a_shape[i] < 0) return tzh_fail(TZH_ERR_INVALID_ARGS, "negative dimension");
        an *= a_shape[i];
    }
    for (int i = 0; i < b_ndim; i++)
        if (b_shape[i] < 0) return tzh_fail(TZH_ERR_INVALID_ARGS, "negative dimension");
    const size_t es = dtype == TZH_F32 ? 4 : 8;  // element bytes
    // scalar B: elementwise scale of A (its result keeps A's shape)
    if (b_ndim == 0 || (b_ndim == 1 && b_shape[0] == 1)) {
        *y_ndim = a_ndim;
        for (int i = 0; i < a_ndim; i++) y_shape[i] = a_shape[i];
        if (!y || an == 0) return TZH_OK;
        if (!a || !b) return tzh_fail(TZH_ERR_INVALID_ARGS, "null MatMul operand");
        double s = 0;
        TZH_HIP(hipMemcpyAsync(&s, b, es, hipMemcpyDeviceToHost, ctx->stream));
        TZH_HIP(hipStreamSynchronize(ctx->stream));
        const dim3 grid((unsigned)((an + 255) / 256));
        if (dtype == TZH_F32) {
            float sf;
            std::memcpy(&sf, &s, 4);
            hipLaunchKernelGGL(scale_kernel<float>, grid, dim3(256), 0, ctx->stream, (const float *)a, sf, (float *)y, an);
        } else {
            hipLaunchKernelGGL(scale_kernel<double>, grid, dim3(256), 0, ctx->stream, (const double *)a, s, (double *)y, an);
        }
        TZH_LAUNCHED("scale_kernel");
        return TZH_OK;
    }
    if (a_ndim < 1) return tzh_fail(TZH_ERR_SHAPE, "MatMul of a scalar A");
    const int64_t m = a_ndim == 1 ? 1 : a_shape[a_ndim - 2], k = a_shape[a_ndim - 1];
    const int64_t k2 = b_ndim == 1 ? b_shape[0] : b_shape[b_ndim - 2], nn = b_ndim == 1 ? 1 : b_shape[b_ndim - 1];
    if (k != k2) return tzh_fail(TZH_ERR_SHAPE, "MatMul inner dimensions differ (%lld vs %lld)", (long long)k, (long long)k2);
    tzh_gemm_desc d{};
    const int lb = a_ndim > 2 ? a_ndim - 2 : 0, rb = b_ndim > 2 ? b_ndim - 2 : 0;
    d.nb = lb > rb ? lb : rb;
    int64_t as = m * k, bs = k * nn;
    for (int i = d.nb - 1; i >= 0; i--) {
        const int li = i - (d.nb - lb), ri = i - (d.nb - rb);
        const int64_t ld = li >= 0 ? a_shape[li] : 1, rd = ri >= 0 ? b_shape[ri] : 1;
        if (ld != rd && ld != 1 && rd != 1) return tzh_fail(TZH_ERR_SHAPE, "MatMul batch dimensions do not broadcast");
        d.batch_shape[i] = ld > rd ? ld : rd;
        d.a_bstride[i] = ld == 1 ? 0 : as;
        d.b_bstride[i] = rd == 1 ? 0 : bs;
        if (li >= 0) as *= ld;
        if (ri >= 0) bs *= rd;
    }
    int w = 0;
    int64_t batches = 1;
    for (int i = 0; i < d.nb; i++) {
        y_shape[w++] = d.batch_shape[i];
        batches *= d.batch_shape[i];
    }
    if (a_ndim > 1) y_shape[w++] = m;
    if (b_ndim > 1) y_shape[w++] = nn;
    *y_ndim = w;
    if (!y) return TZH_OK;
    const int64_t yn = batches * m * nn;
    if (yn == 0) return TZH_OK;
    if (k == 0) {  // empty sums (A and B hold no elements)
        const dim3 grid((unsigned)((yn + 255) / 256));
        if (dtype == TZH_F32)
            hipLaunchKernelGGL(scale_kernel<float>, grid, dim3(256), 0, ctx->stream, (const float *)nullptr, 0.0f,
                               (float *)y, yn);
        else
            hipLaunchKernelGGL(scale_kernel<double>, grid, dim3(256), 0, ctx->stream, (const double *)nullptr, 0.0,
                               (double *)y, yn);
        TZH_LAUNCHED("scale_kernel");
        return TZH_OK;
    }
    if (!a || !b) return tzh_fail(TZH_ERR_INVALID_ARGS, "null MatMul operand");
    d.m = m, d.n = nn, d.k = k, d.lda = k, d.ldb = nn, d.ldy = nn, d.y_bstride = m * nn;
    d.alpha = 1.0, d.beta = 0.0;
    return tzh_gemm_fp_launch(ctx->stream, ctx->num_cus, dtype, false, false, a, b, y, d);
}
