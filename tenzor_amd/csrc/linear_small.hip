// The int8-weight linear for few rows:
//
//   C[t, n] = epi( (sum_k X[t,k] * q[n,k]) * f32(scale[n]) + bias[n] )
//
// the sums and arithmetic of gemm_pipe.hip (matmul_w8a32.zig:14-57: f32
// activations as exact f16 halves hi + lo, codes exact in f16, f32 sums;
// f16 activations as they are), for problems whose 128 x 384 tiles would
// leave most of the chip idle and walk k as one long chain of stages.
//
// Bound by latency, so the design shortens the chain:
//   - Blocks of 16 or 32 rows by 64 outputs (four waves, 16 outputs each) or
//     16 rows by 16 outputs (the four waves share k): enough blocks for the
//     chip at any size this kernel is used for.
//   - A block holds its rows' k range (chunks of 512, 1024 where the waves
//     share k) in LDS, split
//     into f16 halves once.  Every load of a chunk - the wave's codes
//     straight into registers, the rows - is issued before the first wait;
//     nothing is staged in rounds.
//   - The codes are read where they are: row-major int8 [n, k] of any k (no
//     rewriting pass, no scratch), or the models' tiled format.
//   - Optional prologue: the rows are the pre-normalisation rows of the
//     LayerNorm before this linear (arctic.zig:716-746, 779-809), normalised
//     on the way into LDS; the first column of blocks stores them.  A
//     layer's LayerNorms then need no launch of their own.
//   - Row scaling (SCALED: f32 rows of any magnitude): no value is held in
//     fewer bits than by gemm_pipe.hip, whose stages of 64 columns (32 in the
//     LayerNorm linears) each take the exponent that puts the row's largest
//     magnitude so far in [2^14, 2^15).  Here a chunk takes one exponent, and
//     the low halves are held 2^11 times as large (the codes they multiply
//     2^-11 times, exactly), which keeps every bit unless the row grows by
//     more than 2^11 from the chunk's first stage on.  Such rows go in several
//     passes over the products: the first stage, zeros in place of the rest,
//     then the rest likewise.  One exponent a chunk with plain low halves lost
//     them for small values before large ones (2e-4 of the result) and is
//     0 to 1.3 us a call faster; an exponent a stage, the sums rescaled
//     between the products, took 60 us at 1000 x 1536 x 1536, this 34.
#include <type_traits>

#include "pipe.h"

namespace {

enum { SE_BIAS = 0, SE_GELU = 1, SE_RES = 2 };  // SE_RES: + residual, stored f32 (a LayerNorm's input)

struct SmallArgs {
    const void *x;   // [m, k]
    const void *w;   // codes: int8 [n, k] row-major, or W8T
    const uint16_t *scale;
    const float *bias;  // or null
    void *c;            // [m, ldc]
    const void *res;    // SE_RES: [m, n]
    const float *gamma, *beta;  // LayerNorm prologue (k == 384)
    float *xout;                // its rows [m, 384]
    float eps;
    int m, k, n, ldc;
};

#ifdef TZH_EMULATION
inline int frexp_exp(float x) {
    int e = 0;
    if (std::isfinite(x)) std::frexp(x, &e);
    return e;
}
inline float ldexp_f(float x, int e) { return std::ldexp(x, e); }
inline int here(int x) { return x; }
#else
__device__ __forceinline__ int frexp_exp(float x) { return __builtin_amdgcn_frexp_expf(x); }
__device__ __forceinline__ float ldexp_f(float x, int e) { return __builtin_amdgcn_ldexpf(x, e); }
// x, and what is computed from it, formed anew at each use in a loop instead
// of held in registers across it
__device__ __forceinline__ int here(int x) {
    asm volatile("" : "+v"(x));
    return x;
}
#endif

constexpr int kEUnset = 200;  // row exponent before any value: above every 15 - frexp_exp

// BM rows by 16 NF WN outputs per block (NF fragments of 16 a wave), 4 / WN
// waves over each chunk's k.
template <typename TX, typename TC, typename TR, int EPI, bool WT, bool SCALED, bool LNP, int BM, int WN, int NF>
__global__ void __launch_bounds__(256, !SCALED ? 1 : BM == 16 && WN == 4 ? 3 : 2) linear_small_kernel(const SmallArgs a) {
    constexpr bool SPLIT = sizeof(TX) == 4;
    constexpr int WK = 4 / WN, KC = WK == 1 ? 512 : 1024, P = KC + 8, MF = BM / 16;
    constexpr int TPR = 256 / BM;             // threads per row
    constexpr int NP = KC / (8 * TPR);        // 8-value pieces per thread per chunk
    constexpr int CS = KC / 64 / WK;          // 64-code groups of a wave per chunk
    static_assert(WK == 1 || (MF == 1 && NF == 1), "shared k: one fragment to add up");
    constexpr int GC = EPI == SE_RES ? 32 : 64, GP = 8 * TPR / GC;  // SCALED: columns of a stage, stages of a piece
    __shared__ __attribute__((aligned(16))) _Float16 xs[(SPLIT ? 2 : 1) * BM * P];
    // SCALED, by row (in LDS for the registers they would hold over the
    // products): the exponents of this pass and the one before in turns, the
    // first stage of the chunk that is not done, whether any is left
    __shared__ int erow[2][SCALED ? BM : 1], pos_row[SCALED ? BM : 1], left_row[SCALED ? BM : 1];
    __shared__ __attribute__((aligned(16))) f32x4_t part[WK > 1 ? 256 : 1];
    _Float16 *const xhi = xs, *const xlo = xs + (SPLIT ? BM * P : 0);

    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int wn = WK == 1 ? w : 0, wk = WK == 1 ? 0 : w;
    const int t0 = (int)blockIdx.y * BM, n0 = (int)blockIdx.x * (16 * NF * WN);
    const int r16 = lane & 15, g = lane >> 4;
    // this thread's row of X (clamped) and this lane's weight rows (past n:
    // the last)
    const int xr = tid / TPR, sub = tid % TPR;
    const int trow = t0 + xr < a.m ? t0 + xr : a.m - 1;
    auto nrow = [&](int h) __attribute__((always_inline)) {
        const int nr = n0 + 16 * (NF * wn + h) + ((SCALED ? here(lane) : lane) & 15);
        return nr < a.n ? nr : a.n - 1;
    };

    typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
    // whether loads past the end of a row of this block may leave the matrix
    const bool last_rows = !WT && ((int64_t)(n0 + 16 * NF * WN < a.n ? n0 + 16 * NF * WN - 1 : a.n - 1) * a.k +
                                   (a.k + 63) / 64 * 64) > (int64_t)a.n * a.k;
    // codes k .. k + 15, k = k64 + 16 g, of the lane's weight row, as they are
    // stored.  Codes at or past a.k multiply zeros; the loads stay inside the
    // matrix.  The branch is the block's, so that the loads of a chunk are
    // issued without a wait between them.
    auto load_codes = [&](int nrow, int k64) __attribute__((always_inline)) {
        const int k = k64 + 16 * g;
        if constexpr (WT) {
            const size_t o = (((size_t)(nrow / 384) * (a.k / 64) + k / 64) * 384 + nrow % 384) * 64 + k % 64;
            return *(const u32x4_t *)((const uint8_t *)a.w + o);
        } else {
            const uint8_t *const src = (const uint8_t *)a.w + (size_t)nrow * a.k + k;
            u32x4_t v;
            if (!last_rows || k64 + 64 <= a.k) {
                __builtin_memcpy(&v, src, 16);
            } else {
                uint8_t b[16];
#pragma unroll
                for (int i = 0; i < 16; i++) b[i] = k + i < a.k ? src[i] : (uint8_t)0;
                __builtin_memcpy(&v, b, 16);
            }
            return v;
        }
    };

    // A model's linears keep four partial sums, by the 64-code group modulo
    // four, added in order at the end: the same sums whether one wave holds
    // all four or four waves one each, so among forwards on this kernel (up
    // to tzh_small_layer_rows tokens) a sequence's embedding does not depend
    // on the tile, that is on the rest of its batch.
    constexpr int NQ = WT ? 4 / WK : 1;
    f32x4_t acc[NQ][MF][NF];
#pragma unroll
    for (int p = 0; p < NQ; p++)
#pragma unroll
        for (int f = 0; f < MF; f++)
#pragma unroll
            for (int h = 0; h < NF; h++) acc[p][f][h] = f32x4_t{};
    if (SCALED && sub == 0) {
        erow[1][xr] = kEUnset;
        pos_row[xr] = 0;
    }
    wave_lds_order();  // (a row's threads are of one wave)
    int turn = 0;

    // The epilogue's operands, loaded with the first chunk: lane (token r16,
    // g) of fragments (f, h) holds outputs 4 g + e of 16.  Columns past n
    // repeat the last one's (never stored).
    float sc[NF][4], bs[NF][4];
    TR rv[MF][NF][EPI == SE_RES ? 4 : 1];
    auto load_epi = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int h = 0; h < NF; h++) {
            const int n = n0 + 16 * (NF * wn + h) + 4 * g;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int ne = n + e < a.n ? n + e : a.n - 1;
                sc[h][e] = f16_bits_to_f32(a.scale[ne]);
                bs[h][e] = a.bias ? a.bias[ne] : 0.0f;
                if constexpr (EPI == SE_RES)
#pragma unroll
                    for (int f = 0; f < MF; f++) {
                        const int t = t0 + 16 * f + r16 < a.m ? t0 + 16 * f + r16 : a.m - 1;
                        rv[f][h][e] = ((const TR *)a.res)[(size_t)t * a.n + ne];
                    }
            }
        }
    };
    // 64-code groups of the chunk at c0; this wave's are wk, wk + WK, ...
    auto groups_of = [&](int c0) __attribute__((always_inline)) {
        return ((a.k - c0 < KC ? a.k - c0 : KC) + 63) / 64;
    };
    struct Codes {
        u32x4_t v[CS][NF];
    } wc, wnext;
    TX xv[NP][8];
    auto load_chunk = [&](int c0, Codes &wd) __attribute__((always_inline)) {
        const int groups = groups_of(c0);
#pragma unroll
        for (int s = 0; s < CS; s++)
            if (WK * s + wk < groups)
#pragma unroll
                for (int h = 0; h < NF; h++) wd.v[s][h] = load_codes(nrow(h), c0 + 64 * (WK * s + wk));
        const int tl = SCALED ? here(tid) : tid;
        const int tr = t0 + tl / TPR < a.m ? t0 + tl / TPR : a.m - 1;  // (rows past m repeat the last)
        const TX *const row = (const TX *)a.x + (size_t)tr * a.k;
#pragma unroll
        for (int i = 0; i < NP; i++)
            if (8 * TPR * i < 64 * groups) {
                const int j = c0 + 8 * (tl % TPR + TPR * i);
                if (WT || c0 + 8 * TPR * (i + 1) <= a.k) {  // (a model's k: whole pieces)
                    __builtin_memcpy(xv[i], row + j, 8 * sizeof(TX));  // (16-byte loads; element alignment is enough)
                } else {  // the row's last piece: what lies past it is cleared where it is used
#pragma unroll
                    for (int e = 0; e < 8; e++) xv[i][e] = row[j + e < a.k ? j + e : a.k - 1];
                }
            }
    };
    bool begin = true;
    if constexpr (SPLIT) load_chunk(0, wc);
    // (with two fragments a wave they would cost the second block of a CU,
    // with a residual beside the row exponents at 16 x 64 the third)
    constexpr bool EPI_FIRST = NF == 1 && !(SCALED && EPI == SE_RES && BM == 16 && WN == 4);
    if constexpr (EPI_FIRST) load_epi();
    for (int c0 = 0, next; c0 < a.k; c0 = next) {
        next = c0 + KC;
        if constexpr (!SPLIT) load_chunk(c0, wc);
        const int groups = groups_of(c0);
#pragma unroll
        for (int i = 0; i < NP; i++)
            if (!WT && 8 * TPR * i < 64 * groups && c0 + 8 * TPR * (i + 1) > a.k)
#pragma unroll
                for (int e = 0; e < 8; e++)
                    if (c0 + 8 * (sub + TPR * i) + e >= a.k) xv[i][e] = (TX)0;
        if constexpr (LNP) {  // one chunk of 384 columns
            // gamma and beta, loaded before the statistics where registers allow
            constexpr bool EARLY = BM == 16;
            f32x4_t gg[384 / (8 * TPR)][2], bb[384 / (8 * TPR)][2];
            auto load_ln = [&](int i) __attribute__((always_inline)) {
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    gg[i][h] = *(const f32x4_t *)(a.gamma + 8 * (sub + TPR * i) + 4 * h);
                    bb[i][h] = *(const f32x4_t *)(a.beta + 8 * (sub + TPR * i) + 4 * h);
                }
            };
            if constexpr (EARLY)
#pragma unroll
                for (int i = 0; i < 384 / (8 * TPR); i++) load_ln(i);
            // sums by sixteenths of the row (16 threads, or 8 holding two
            // each), then over them in one order for both
            constexpr int HV = 16 / TPR;
            auto row_sum = [&](auto &&term) __attribute__((always_inline)) {
                float s[HV] = {};
#pragma unroll
                for (int i = 0; i < 384 / (8 * TPR); i++)
#pragma unroll
                    for (int e = 0; e < 8; e++) s[i % HV] += term((float)xv[i][e]);
                float v = HV == 2 ? s[0] + s[HV - 1] : s[0];
                if constexpr (HV == 1) v += __shfl_xor(v, 8, 64);
#pragma unroll
                for (int o = 4; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
                return v;
            };
            const float mean = row_sum([](float x) { return x; }) / 384.0f;
            const float sq = row_sum([&](float x) { return (x - mean) * (x - mean); });
            const float inv_std = 1.0f / sqrtf(sq / 384.0f + a.eps);
#pragma unroll
            for (int i = 0; i < 384 / (8 * TPR); i++) {
                const int j = 8 * (sub + TPR * i);
                if constexpr (!EARLY) load_ln(i);
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    f32x4_t y;
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        y[e] = (((float)xv[i][4 * h + e] - mean) * inv_std) * gg[i][h][e] + bb[i][h][e];
                        xv[i][4 * h + e] = (TX)y[e];
                    }
                    if (blockIdx.x == 0 && t0 + xr < a.m) *(f32x4_t *)(a.xout + (size_t)trow * 384 + j + 4 * h) = y;
                }
            }
        }
        const int tv = SCALED ? here(tid) : tid, xr = tv / TPR, sub = tv % TPR;
        int ex = 0, take = KC / GC;  // this pass's exponent and stages of the row
        int mine = 0, left = 0;      // the stage of this lane's part of piece 0, from the first that is not done
        if constexpr (SCALED) {
            const int pos = pos_row[xr];
            mine = 8 * sub / GC - pos;
            float at = 0.0f, rest = 0.0f;  // largest magnitudes of stage pos, and from it on
#pragma unroll
            for (int i = 0; i < NP; i++)
                if (8 * TPR * i < 64 * groups) {
                    float mx = 0.0f;
#pragma unroll
                    for (int e = 0; e < 8; e++) mx = fmaxf(mx, fabsf((float)xv[i][e]));
                    const int st = mine + i * GP;  // of this lane's part, from pos
                    at = st == 0 ? mx : at;
                    rest = st >= 0 ? fmaxf(rest, mx) : rest;
                }
            auto over_row = [&](float mx) __attribute__((always_inline)) {
                mx = fmaxf(mx, dpp_f32<0xB1>(mx));   // lane ^ 1
                mx = fmaxf(mx, dpp_f32<0x4E>(mx));   // lane ^ 2
                mx = fmaxf(mx, dpp_f32<0x141>(mx));  // the other quad of the eight
                if constexpr (TPR == 16) mx = fmaxf(mx, dpp_f32<0x140>(mx));  // the other eight of the sixteen
                return mx;
            };
            at = over_row(at);
            rest = over_row(rest);
            // the exponent that puts mx in [2^14, 2^15); zero, inf and NaN have none
            auto want = [&](float mx) __attribute__((always_inline)) {
                return mx > 0.0f && mx < INFINITY ? 15 - frexp_exp(mx) : kEUnset;
            };
            int e_first = min(erow[turn ^ 1][xr], want(at));
            const int e_all = min(e_first, want(rest));
            ex = e_first;
            if (__any(e_first == kEUnset && e_all < kEUnset)) {
                // rows that start with a stage of zeros: none of theirs asks
                // for more than the smallest of the lanes' eights
                float least = -INFINITY;
#pragma unroll
                for (int i = 0; i < NP; i++)
                    if (8 * TPR * i < 64 * groups) {
                        float mx = 0.0f;
#pragma unroll
                        for (int e = 0; e < 8; e++) mx = fmaxf(mx, fabsf((float)xv[i][e]));
                        if (mx > 0.0f) least = fmaxf(least, -mx);
                    }
                e_first = min(e_first, want(-over_row(least)));
            }
            const bool whole = e_all == kEUnset || (e_first < kEUnset && e_all >= e_first - 11);
            ex = whole ? e_all : ex;
            take = whole ? KC / GC : 1;
            left = pos + take < 64 * groups / GC;
            wave_lds_order();
            if (sub == 0) pos_row[xr] = pos + take;
        }
        if (!begin) __syncthreads();  // the last products' reads are done
        begin = false;
#pragma unroll
        for (int i = 0; i < NP; i++)
            if (8 * TPR * i < 64 * groups) {
                const int o = xr * P + 8 * (sub + TPR * i);
                if constexpr (SPLIT) {
                    f32x4_t lo4, hi4;
                    const int es = (unsigned)(mine + i * GP) < (unsigned)take ? ex : -1000;  // (others: zeros)
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        lo4[e] = SCALED ? ldexp_f((float)xv[i][e], es) : (float)xv[i][e];
                        hi4[e] = SCALED ? ldexp_f((float)xv[i][4 + e], es) : (float)xv[i][4 + e];
                    }
                    half8_t h, l;
                    if constexpr (SCALED) {
                        f32x4_t lou, hiu;
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            lou[e] = 2048.0f * lo4[e];
                            hiu[e] = 2048.0f * hi4[e];
                        }
                        split_f32x8_by<true>(lo4, hi4, lou, hiu, h, l);
                    } else {
                        split_f32x8(lo4, hi4, h, l);
                    }
                    *(half8_t *)(xhi + o) = h;
                    *(half8_t *)(xlo + o) = l;
                } else {
                    half8_t h;
                    __builtin_memcpy(&h, xv[i], 16);
                    *(half8_t *)(xhi + o) = h;
                }
            }
        if constexpr (SCALED)
            if (sub == 0) erow[turn][xr] = ex, left_row[xr] = left;
        __syncthreads();
        if constexpr (SCALED) {
            if (__any(left_row[lane % BM])) next = c0;  // the same chunk again
            else if (sub == 0) pos_row[xr] = 0;
        }
        // f32: the next chunk's loads fly during this one's products (5 % at
        // k = 1536; with f16 rows, at four blocks a CU, 5 % slower)
        if constexpr (SPLIT)
            if (next < a.k) load_chunk(next, wnext);
        if constexpr (SCALED) {  // the sums so far, to this pass's exponents
#pragma unroll
            for (int f = 0; f < MF; f++) {
                const int d = erow[turn][16 * f + r16] - erow[turn ^ 1][16 * f + r16];
#pragma unroll
                for (int h = 0; h < NF; h++)
#pragma unroll
                    for (int q = 0; q < 4; q++)
#pragma unroll
                        for (int p = 0; p < NQ; p++) acc[p][f][h][q] = ldexp_f(acc[p][f][h][q], d);
            }
            turn ^= 1;
        }
#pragma unroll
        for (int s = 0; s < CS; s++)
            if (WK * s + wk < groups) {
                constexpr int kChunkGroups = KC / 64;
                static_assert(kChunkGroups % 4 == 0, "a chunk's groups start a new round of partial sums");
                const int kk = 64 * (WK * s + wk) + 16 * g, p = s % NQ;
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    half8_t wf[NF];
#pragma unroll
                    for (int h = 0; h < NF; h++) {
                        constexpr uint32_t bias = WT ? 0 : 0x80808080u;  // u = q + 128
                        wf[h] = codes_to_f16(wc.v[s][h][2 * j] ^ bias, wc.v[s][h][2 * j + 1] ^ bias);
                    }
                    auto products = [&](const _Float16 *x, int f, const half8_t (&w)[NF]) __attribute__((always_inline)) {
                        const half8_t xf = *(const half8_t *)(x + (16 * f + r16) * P + kk + 8 * j);
#pragma unroll
                        for (int h = 0; h < NF; h++)
                            acc[p][f][h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[h], xf, acc[p][f][h], 0, 0, 0);
                    };
                    if constexpr (SCALED) {  // the low halves' codes 2^-11 times, exactly
                        constexpr _Float16 down = (_Float16)0.00048828125f;
#pragma unroll
                        for (int f = 0; f < MF; f++) products(xhi, f, wf);
#pragma unroll
                        for (int h = 0; h < NF; h++) wf[h] *= down;
#pragma unroll
                        for (int f = 0; f < MF; f++) products(xlo, f, wf);
                    } else {
#pragma unroll
                        for (int f = 0; f < MF; f++) {
                            products(xhi, f, wf);
                            if constexpr (SPLIT) products(xlo, f, wf);
                        }
                    }
                }
            }
        if constexpr (SPLIT) wc = wnext;
    }

    if constexpr (!EPI_FIRST) load_epi();
    if constexpr (WK > 1) {
        part[tid] = acc[0][0][0];
        __syncthreads();
        if (w > 0) return;
#pragma unroll
        for (int k = 1; k < WK; k++) acc[0][0][0] += part[64 * k + lane];
    } else {
#pragma unroll
        for (int p = 1; p < NQ; p++)
#pragma unroll
            for (int f = 0; f < MF; f++)
#pragma unroll
                for (int h = 0; h < NF; h++) acc[0][f][h] += acc[p][f][h];
    }
#pragma unroll
    for (int h = 0; h < NF; h++) {
        const int n = n0 + 16 * (NF * wn + h) + 4 * g;
        if (n >= a.n) continue;
#pragma unroll
        for (int f = 0; f < MF; f++) {
            const int t = t0 + 16 * f + r16;
            if (t >= a.m) continue;
            TC o[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                float v = (SCALED ? ldexp_f(acc[0][f][h][e], -erow[turn ^ 1][16 * f + r16]) : acc[0][f][h][e]) * sc[h][e] +
                          bs[h][e];
                if constexpr (EPI == SE_GELU) v = gelu_fast(v);
                if constexpr (EPI == SE_RES) v = (float)rv[f][h][e] + v;
                o[e] = (TC)v;
            }
            TC *const dst = (TC *)a.c + (size_t)t * a.ldc + n;
            if (n + 4 <= a.n) {
                __builtin_memcpy(dst, o, 4 * sizeof(TC));
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (n + e < a.n) dst[e] = o[e];
            }
        }
    }
}

template <typename TX, typename TC, typename TR, int EPI, bool WT, bool SCALED, bool LNP>
int launch_small(hipStream_t st, int num_cus, const SmallArgs &a) {
    // The largest tile that fills the chip: more outputs or rows a block
    // share its rows' staging, its LDS reads and its code reads; 16 x 16
    // tiles with shared k where even 16 x 64 would leave half the CUs idle
    const int bn = (a.n + 63) / 64;
    const int64_t rows16 = (a.m + 15) / 16, rows32 = (a.m + 31) / 32;
    if (rows16 > 65535) return tzh_fail(TZH_ERR_TOO_LARGE, "internal: %d rows in the small linear", a.m);
    // (a model's linears, with four partial sums, would fall to one block a
    // CU with two fragments a wave)
    constexpr int NFM = WT ? 1 : 2;
    if (NFM == 2 && rows32 * ((a.n + 127) / 128) >= num_cus) {
        hipLaunchKernelGGL((linear_small_kernel<TX, TC, TR, EPI, WT, SCALED, LNP, 32, 4, NFM>),
                           dim3((unsigned)((a.n + 127) / 128), (unsigned)rows32), dim3(256), 0, st, a);
    } else if (rows32 * bn >= num_cus) {
        hipLaunchKernelGGL((linear_small_kernel<TX, TC, TR, EPI, WT, SCALED, LNP, 32, 4, 1>),
                           dim3((unsigned)bn, (unsigned)rows32), dim3(256), 0, st, a);
    } else if (rows16 * bn >= num_cus / 2) {
        hipLaunchKernelGGL((linear_small_kernel<TX, TC, TR, EPI, WT, SCALED, LNP, 16, 4, 1>),
                           dim3((unsigned)bn, (unsigned)rows16), dim3(256), 0, st, a);
    } else {
        hipLaunchKernelGGL((linear_small_kernel<TX, TC, TR, EPI, WT, SCALED, LNP, 16, 1, 1>),
                           dim3((unsigned)((a.n + 15) / 16), (unsigned)rows16), dim3(256), 0, st, a);
    }
    TZH_LAUNCHED("linear_small_kernel");
    return TZH_OK;
}

}  // namespace

// Whether linear_small_kernel is the faster one for m rows: both times in us
// as measured on an MI355X of 256 CUs.  This kernel pays by the product (m n k
// in billions, over the CUs there are), nearly twice as much for f32 rows that
// are not whole 16-byte pieces; the pipelined one walks ceil(k / 64) serial
// stages once per 1536 columns whatever m is, up to one round of tiles (beyond
// it this one has long lost), after passes over the rows and codes where k is
// ragged.  Measured, small / pipelined: f32 128 x 384 x 1152 5.2 / 27, 2048 x
// 384 x 1536 GELU 20.8 / 30.4, 4096 x 384 x 1536 35 / 33, LayerNorm k = 1536
// with 1000 rows 23 / 74, 6000 71 / 74, k = 384 with 4096 rows 21.8 / 27.6,
// 6000 31.5 / 28.2; 197 x 1000 x 1537 11.5 / 119, 2048 x 2049 x 777 87 / 123,
// 4096 x 2049 x 777 169 / 131; f16 128 x 384 x 1152 4.0 / 14.9, 2048 x 384 x
// 1536 11.7 / 18.5, 4096 rows 22 / 19.6, LayerNorm k = 1536 with 1024 rows
// 17 / 21, 2048 rows 27 / 22, k = 384 with 3000 rows 18.4 / 15.3.
bool tzh_linear_small_wins(int num_cus, int64_t m, int64_t k, int64_t n, bool f32, bool ln) {
    if (m > (int64_t)num_cus * 64) return false;
    const double work = (double)m * (double)k * (double)n * 1e-9 * 256.0 / num_cus;
    const double stages = (double)((k + 63) / 64), launches = (double)((n + 1535) / 1536);
    const double pipe32 = launches * (6.0 + 3.0 * stages);
    if (f32 && ln) return 8.0 + 14.0 * work < pipe32 && 12.0 + 18.0 * work < 10.5 + 2.75 * stages;
    if (f32) return 4.0 + 14.0 * work < pipe32 && (k % 4 == 0 || 4.0 + 26.0 * work < pipe32 + 15.0);
    if (!ln) return 3.5 + 7.5 * work < launches * (8.0 + 1.3 * stages);
    return 8.5 + 18.0 * work < (k > 384 ? 20.0 : 8.0 + 1.3 * stages);
}

// C = epi(X q^T s + b) for caller-owned codes q [n, k] (row-major int8, any
// k >= 1), f32 (row-scaled) or f16 activations and output of the same type.
// TZH_EPI_BIAS_RES_LN: pre_ln (f32 [m, n]) receives the rows before the
// LayerNorm, residual added, and c is not written.
int tzh_linear_small_launch(hipStream_t st, int num_cus, const void *x, int32_t x_dtype, const int8_t *q,
                            const uint16_t *scale, const float *bias, void *c, int32_t c_dtype, int64_t m, int64_t k,
                            int64_t n, int32_t epilogue, const void *res, float *pre_ln) {
    SmallArgs a{};
    a.x = x, a.w = q, a.scale = scale, a.bias = bias, a.res = res;
    a.m = (int)m, a.k = (int)k, a.n = (int)n, a.ldc = (int)n;
    a.c = epilogue == TZH_EPI_BIAS_RES_LN ? (void *)pre_ln : c;
    const bool x32 = x_dtype == TZH_F32, c32 = c_dtype == TZH_F32;
    auto typed = [&](auto tx, auto tc) -> int {
        using TX = decltype(tx);
        using TC = decltype(tc);
        constexpr bool S = sizeof(TX) == 4;
        switch (epilogue) {
        case TZH_EPI_BIAS: return launch_small<TX, TC, TC, SE_BIAS, false, S, false>(st, num_cus, a);
        case TZH_EPI_BIAS_GELU: return launch_small<TX, TC, TC, SE_GELU, false, S, false>(st, num_cus, a);
        default: return launch_small<TX, float, TC, SE_RES, false, S, false>(st, num_cus, a);
        }
    };
    if (x32) return c32 ? typed(0.0f, 0.0f) : typed(0.0f, (_Float16)0);
    return c32 ? typed((_Float16)0, 0.0f) : typed((_Float16)0, (_Float16)0);
}

// Rows up to which a model layer's linears run one by one on this file's
// kernel (five launches a layer, each of enough blocks for the chip) rather
// than on the fused kernels, whose 64-token panels walk all of a layer's
// weight stages in series (about 55 us a layer from 1 to 1000 rows).  The
// line moves with the CUs those rows can spread over.  Measured on 256 CUs,
// fused -> here: the forward of one sequence of 16 293 -> 144 us, of 128
// 346 -> 172, of 512 493 -> 298; 5 x 128 367 -> 277; the feed-forward block
// of 128 rows 23 -> 16, 640 31.5 -> 25.7.  Past the lines: 7 x 128 367 ->
// 332, 8 x 128 369 -> 375; the block of 700 rows 27 -> 32.
int64_t tzh_small_layer_rows(int num_cus) { return (int64_t)num_cus * 7 / 2; }
int64_t tzh_small_ffn_rows(int num_cus) { return (int64_t)num_cus * 5 / 2; }

// A model linear over f32 rows inside the split's range (not row-scaled):
// C = epi(X W^T s + b) with W8T codes, n a multiple of 384 and k of 128, all
// pointers 16-byte aligned.  epilogue: TZH_EPI_BIAS, TZH_EPI_BIAS_GELU, or
// TZH_EPI_BIAS_RES_LN for the rows before the LayerNorm (res added).  gamma
// non-null (k == 384): x holds rows before a LayerNorm, normalised on the
// way in and stored to xout (which may not overlap x).
int tzh_linear_small_model_launch(hipStream_t st, int num_cus, const float *x, const float *gamma, const float *beta,
                                  float eps, float *xout, const void *w, const uint16_t *scale, const float *bias,
                                  float *c, int64_t m, int64_t k, int64_t n, int32_t epilogue, const float *res) {
    if (m <= 0 || m > ((int64_t)1 << 20) || k % 128 || n % 384 || (gamma && (k != 384 || !beta || !xout)))
        return tzh_fail(TZH_ERR_INVALID_ARGS, "internal: bad small linear");
    SmallArgs a{};
    a.x = x, a.w = w, a.scale = scale, a.bias = bias, a.c = c, a.res = res;
    a.gamma = gamma, a.beta = beta, a.xout = xout, a.eps = eps;
    a.m = (int)m, a.k = (int)k, a.n = (int)n, a.ldc = (int)n;
    if (epilogue == TZH_EPI_BIAS_RES_LN)
        return launch_small<float, float, float, SE_RES, true, false, false>(st, num_cus, a);
    if (epilogue == TZH_EPI_BIAS_GELU)
        return gamma ? launch_small<float, float, float, SE_GELU, true, false, true>(st, num_cus, a)
                     : launch_small<float, float, float, SE_GELU, true, false, false>(st, num_cus, a);
    return gamma ? launch_small<float, float, float, SE_BIAS, true, false, true>(st, num_cus, a)
                 : launch_small<float, float, float, SE_BIAS, true, false, false>(st, num_cus, a);
}
