// Products of float weights (F32 / F16 / BF16 rows in the natural layout) with several columns on
// the f32 matrix units (gfx950, wave64): every weight widened exactly to f32, x in f32, products
// and sums in f32.
//
// The same product as matvec_float.hip (reference src/core/ref/ops.cpp:891-984, load_float :78-93);
// only the summation order differs. Two kernels:
//
//   k_mvq  3..8 columns of F16 / BF16: 16 rows x 4 or 8 columns per work-group (v_mfma_f32_4x4x1)
//   k_mmf  more columns: 16 x 16, 32 x 32 or 64 x 32 tiles per work-group (v_mfma_f32_16x16x4)
//
// Both read their operands straight from memory into the MFMA's lanes; the waves of a work-group
// take disjoint steps of K and meet once, in LDS, to add their sums in a fixed tree.
//
// Summation: no chain is longer than 8 products before it is added to a longer sum, and pairs of the
// waves' sums are added in 64 bits and rounded once, so the error against 64-bit products is below that
// of the vector kernel, which it must not exceed (activations with one channel in 64 eight times
// larger; F16 4096x4096 at 8 columns 9.2e-8 against 1.06e-7, 12288x2056 at 300 8.5e-8 against 9.3e-8,
// F32 128x2048 at 512 8.8e-8 against 9.2e-8, 512x512 at 1024 7.9e-8 against 8.2e-8, 512x8192 at 2048
// 1.10e-7 against 1.27e-7; with the waves' sums added in f32 it was up to 6% above it at K of 500 to
// 2100; k_mvq at K of 130 to 250, whose steps fill one wave and part of a second, within 0.4% of it;
// k_mmf at K of 8, where nothing follows the tree of 8 products, 5.1e-8 against 4.5e-8).
#include "kernels.h"
#include "weight_float.h"

#include <algorithm>
#include <cstdio>
#include <cstring>

namespace sgk {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

struct MmfArgs {
    MatArgs a;      // mats[0]; a.nb is the row stride in bytes
    int nmat;
    int64_t mt[4];  // matrix j owns row tiles mt[j] .. mt[j + 1]
    const uint8_t * wm[3];
    int64_t Mm[3];
    float * ym[3];
    int64_t ys1m[3];
};

// what a work-group multiplies: the matrix and slice of its blockIdx
struct Part {
    const uint8_t * w;
    const float * x;
    float * y;
    int64_t ys1, M, tile;
    __device__ explicit Part(const MmfArgs & A) {
        const MatArgs & a = A.a;
        tile = blockIdx.x;
        w = a.w, x = a.x, y = a.y, ys1 = a.y_s1, M = a.M;
        if (A.nmat > 1) {
            const int j = tile >= A.mt[1] ? (tile >= A.mt[2] ? 2 : 1) : 0;
            w = A.wm[j], y = A.ym[j], ys1 = A.ys1m[j], M = A.Mm[j], tile -= A.mt[j];
        } else if (gridDim.y > 1) { // (one slice: no 64-bit divisions ahead of the first load)
            const int64_t i2 = blockIdx.y % a.ne12, i3 = blockIdx.y / a.ne12;
            w += (uint64_t) (i2 / a.r2) * a.w_s2 + (uint64_t) (i3 / a.r3) * a.w_s3;
            x += i2 * a.x_s2 + i3 * a.x_s3;
            y += i2 * a.y_s2 + i3 * a.y_s3;
        }
    }
};

__device__ __forceinline__ float4 load4(const float * p, bool aligned) {
    return aligned ? *reinterpret_cast<const float4 *>(p) : make_float4(p[0], p[1], p[2], p[3]);
}

// sum of p[0 .. W) in a fixed tree
template <int W, typename T>
__device__ __forceinline__ T tree(T (&p)[W]) {
#pragma unroll
    for (int h = 1; h < W; h *= 2)
#pragma unroll
        for (int k = 0; k + h < W; k += 2 * h) p[k] += p[k + h];
    return p[0];
}

// the sum of the W waves' values at(wave): pairs in 32 bits, those in 64, rounded once (all in 64 bits
// the error is 5% lower, but F16 8192x128 at 4 columns, 64 slices took 94.4 us against 93.8, and 93.0 all in 32)
template <int W, typename F>
__device__ __forceinline__ float sum_waves(F at) {
    double p[W / 2];
#pragma unroll
    for (int k = 0; k < W / 2; ++k) p[k] = at(2 * k) + at(2 * k + 1);
    return (float) tree<W / 2>(p);
}

// reduce-scatter of V values over the 16 lanes that share lane % 4 (lanes 4 b + j): afterwards lane
// (b, j) holds, in v[0 .. V / 16), the sums over b of the values returned index .. index + V / 16 of
// column j. A recursion over templates: a loop that halves its count is not unrolled by the
// compiler, and the array then lives in LDS.
template <int V, int B = 32>
__device__ __forceinline__ int scatter16(float (&v)[V], int lane) {
    const bool hi = (lane & B) != 0;
    float h[V / 2];
#pragma unroll
    for (int i = 0; i < V / 2; ++i) {
        const float send = hi ? v[i] : v[i + V / 2];
        const float keep = hi ? v[i + V / 2] : v[i];
        h[i] = keep + __shfl_xor(send, B);
    }
    int idx = hi ? V / 2 : 0;
    if constexpr (B > 4) idx += scatter16<V / 2, B / 2>(h, lane);
#pragma unroll
    for (int i = 0; i < V / 2; ++i) v[i] = h[i];
    return idx;
}

// 16 rows x 4 C columns, 8 waves. v_mfma_f32_4x4x1 multiplies 16 independent 4 x 4 blocks: block b
// takes the b-th part of a step, so lane (b, j) loads 16 consecutive bytes of row j, 16 lanes read
// 256 consecutive bytes of a row, and at most 3 columns of the MFMA are padding. One step in flight
// per wave with 4 waves per SIMD beat two steps in flight with 3 (more registers): F16 12288x4096 at
// 8 columns 27 against 35 us, 4096x4096 11.8 against 13.0.
//
// What bounds it: the weight stream up to 4 columns (F16 12288x4096 21 us, 4.8 TB/s), at 8 about
// equally the stream, the matrix units and x from the L2 (without its x loads 24.8, without its
// MFMAs 25.8 of 27 us). The vector kernel took 62.8 us at 4 columns and 73 at 8 with its sums in
// LDS, 27.6 and 36 with them in registers.
//
// TAIL: K is not a whole number of steps; XV: x columns 16-byte aligned (vector loads)
template <int WT, int C, bool XV, bool TAIL>
__global__ __launch_bounds__(512) void k_mvq(MmfArgs A) {
    constexpr int R = 4, W = 8;
    constexpr int E = 8;       // elements per lane and step
    constexpr int KS = 16 * E; // elements of K per step
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int j = lane & 3, b = lane >> 2;
    const Part P(A);
    const int64_t m0 = P.tile * (4 * R), n0 = (int64_t) blockIdx.z * (4 * C);
    const int K = (int) A.a.K; // (K N < 2^31)
    const int64_t N = A.a.N;
    const uint8_t * row[R];
#pragma unroll
    for (int r = 0; r < R; ++r) row[r] = P.w + (uint64_t) min<int64_t>(m0 + 4 * r + j, P.M - 1) * (uint64_t) A.a.nb + 2 * E * b;
    const float * col[C];
#pragma unroll
    for (int c = 0; c < C; ++c) col[c] = P.x + min<int64_t>(n0 + 4 * c + j, N - 1) * A.a.x_s1 + E * b;
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    f32x4 acc[R][C];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < C; ++c) acc[r][c] = zero;
    for (int k0 = wave * KS; k0 < K; k0 += W * KS) {
        // (a lane past K reads its row's last whole group, zeroed below)
        const int k = TAIL ? min(k0, K - E - E * b) : k0;
        const bool ok = !TAIL || k0 + E * b < K;
        float xv[C][E];
        uint4 wl[R];
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
            for (int h = 0; h < E; h += 4) {
                const float4 t = load4(col[c] + k + h, XV);
                xv[c][h] = t.x, xv[c][h + 1] = t.y, xv[c][h + 2] = t.z, xv[c][h + 3] = t.w;
            }
#pragma unroll
        for (int r = 0; r < R; ++r) wl[r] = ld16_nt(row[r] + (int64_t) k * 2);
        if (TAIL) {
#pragma unroll
            for (int c = 0; c < C; ++c)
#pragma unroll
                for (int e = 0; e < E; ++e) xv[c][e] = ok ? xv[c][e] : 0.0f;
        }
#pragma unroll
        for (int r = 0; r < R; r += 2) {
            float wf[2][E];
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                widen16<WT>(wl[r + q], wf[q]);
                if (TAIL) {
#pragma unroll
                    for (int e = 0; e < E; ++e) wf[q][e] = ok ? wf[q][e] : 0.0f;
                }
            }
            f32x4 p[2][C];
#pragma unroll
            for (int e = 0; e < E; ++e)
#pragma unroll
                for (int q = 0; q < 2; ++q)
#pragma unroll
                    for (int c = 0; c < C; ++c) p[q][c] = __builtin_amdgcn_mfma_f32_4x4x1f32(xv[c][e], wf[q][e], e == 0 ? zero : p[q][c], 0, 0, 0);
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int c = 0; c < C; ++c) acc[r + q][c] += p[q][c];
        }
    }
    // lane (b, j) of quad (r, c): row 4 r + j of columns 4 c .. 4 c + 3, block b's share
    constexpr int V = R * C * 4;
    float v[V];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) v[(r * C + c) * 4 + e] = acc[r][c][e];
    const int idx = scatter16<V>(v, lane);
    __shared__ float red[W][4 * V];
#pragma unroll
    for (int i = 0; i < V / 16; ++i) red[wave][(idx + i) * 4 + j] = v[i];
    __syncthreads();
    if (threadIdx.x < 4 * V) {
        const int t = threadIdx.x;
        const float sum = sum_waves<W>([&](int k) { return red[k][t]; });
        const int c = (t >> 4) % C, r = (t >> 4) / C;
        const int64_t m = m0 + 4 * r + (t & 3), n = n0 + 4 * c + ((t >> 2) & 3);
        if (m < P.M && n < N) P.y[n * P.ys1 + m] = sum;
    }
}

// 16 R rows x 16 C columns, W waves; lane (i, q) of a 16 x 16 fragment loads row i's (column i's)
// part q of a 32-element step, one unit (a 128-byte line of every row) ahead of the MFMAs. A step's
// 8 MFMAs (4 products each) are added in a tree; runs of 4 steps are added in order.
//
// What bounds it: the operands' bytes through each CU's L1 (about 40 GB/s of misses per CU), so a
// shape takes the largest tile that still occupies the CUs. Measured, against the vector kernel in
// launches of 8 columns: F32 128x2048 at 512 columns 9.5 us (16 x 16 tiles) against 965; 500x4096 at
// 512 32 us (32 x 32; 58.7 in 16 x 16); 4096x4096 at 512 230 us = 75 TFLOP/s of 157 (64 x 32) against
// 2519; F16 2500x520 at 500 40 us (32 x 32) against 169 for the vector kernel in one launch. Chains of
// 2 MFMAs added in a tree of 4 are faster on large tiles (192 and 30 us) but their error was larger
// than the vector kernel's at short K (256x1024 9.5e-8 against 8.7e-8, with the waves' sums added in
// f32).
constexpr int kRun = 4; // steps per run of the two-level sum

template <int WT, int R, int C, int W, bool XV>
__global__ __launch_bounds__(64 * W) void k_mmf(MmfArgs A) {
    constexpr int esz = WT == F32 ? 4 : 2;
    constexpr int S = WT == F32 ? 1 : 2; // 32-element steps per unit
    constexpr int KU = 32 * S;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int i = lane & 15, q = lane >> 4;
    const Part P(A);
    const int64_t m0 = P.tile * (16 * R), n0 = (int64_t) blockIdx.z * (16 * C);
    const int K = (int) A.a.K;
    const int64_t N = A.a.N;
    const uint8_t * row[R];
#pragma unroll
    for (int r = 0; r < R; ++r) row[r] = P.w + (uint64_t) min<int64_t>(m0 + 16 * r + i, P.M - 1) * (uint64_t) A.a.nb;
    const float * col[C];
#pragma unroll
    for (int c = 0; c < C; ++c) col[c] = P.x + min<int64_t>(n0 + 16 * c + i, N - 1) * A.a.x_s1;

    // the lane's elements of a step: two groups of 4, each 16 bytes of F32, or 16 bytes of F16 / BF16
    // together, so that the four parts of a row read one run of 64 bytes per load. (The parts in
    // descending order: an MFMA adds its 4 products one after the other, so the first is rounded four
    // times and the last once. Random data do not care; with large activations in a step's first part
    // this order has the smaller error, F16 64x64 6.3e-8 against 7.0e-8. F32 keeps the ascending order,
    // 128x2048 at 512 columns 9.6 us against 9.8, but for short K, where the sums that follow do not
    // make up for it: 1270x16 at 471 columns 5.3e-8 in the vector kernel, 5.7e-8 ascending, 5.2e-8
    // descending; 115x120 at 449 7.25e-8 and 7.33e-8 ascending.)
    const int g = WT == F32 && K >= 256 ? q : 3 - q, o0 = WT == F32 ? 4 * g : 8 * g, o1 = WT == F32 ? 16 + 4 * g : 8 * g + 4;
    struct Raw {
        uint4 w[R][S][WT == F32 ? 2 : 1];
        float4 x[C][S][2];
    };
    const auto load = [&](Raw & d, int k0) {
#pragma unroll
        for (int s = 0; s < S; ++s) {
            // (K is a multiple of 8: a group past it reads the last whole one and is zeroed below)
            const int k = k0 + 32 * s;
            const int ka = min(k + o0, WT == F32 ? K - 4 : K - 8), kb = WT == F32 ? min(k + o1, K - 4) : ka + 4;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                d.w[r][s][0] = *reinterpret_cast<const uint4 *>(row[r] + (int64_t) ka * esz);
                if constexpr (WT == F32) d.w[r][s][1] = *reinterpret_cast<const uint4 *>(row[r] + (int64_t) kb * esz);
            }
#pragma unroll
            for (int c = 0; c < C; ++c) {
                d.x[c][s][0] = load4(col[c] + ka, XV);
                d.x[c][s][1] = load4(col[c] + kb, XV);
            }
        }
    };
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    f32x4 run[R][C], tot[R][C];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < C; ++c) run[r][c] = tot[r][c] = zero;
    int n = 0;
    const auto mul = [&](const Raw & d, int k0) {
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const bool va = k0 + 32 * s + o0 < K, vb = k0 + 32 * s + o1 < K;
            float xv[C][8];
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const float4 f = d.x[c][s][0], g = d.x[c][s][1];
                const float v[8] = {f.x, f.y, f.z, f.w, g.x, g.y, g.z, g.w};
#pragma unroll
                for (int e = 0; e < 8; ++e) xv[c][e] = (e < 4 ? va : vb) ? v[e] : 0.0f;
            }
#pragma unroll
            for (int r = 0; r < R; ++r) {
                float wf[8];
                widen16<WT>(d.w[r][s][0], wf);
                if constexpr (WT == F32) widen16<WT>(d.w[r][s][1], wf + 4);
#pragma unroll
                for (int e = 0; e < 8; ++e) wf[e] = (e < 4 ? va : vb) ? wf[e] : 0.0f;
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    f32x4 p[8];
#pragma unroll
                    for (int e = 0; e < 8; ++e) p[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[c][e], wf[e], zero, 0, 0, 0);
                    run[r][c] += tree<8>(p);
                }
            }
        }
        n += S;
        if (n == kRun) {
            n = 0;
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int c = 0; c < C; ++c) tot[r][c] += run[r][c], run[r][c] = zero;
        }
    };
    constexpr int KW = W * KU;
    int k = wave * KU;
    if (k < K) {
        Raw d0, d1;
        load(d0, k);
        for (; k + 2 * KW < K; k += 2 * KW) {
            load(d1, k + KW);
            mul(d0, k);
            load(d0, k + 2 * KW);
            mul(d1, k + KW);
        }
        if (k + KW < K) {
            load(d1, k + KW);
            mul(d0, k);
            mul(d1, k + KW);
        } else {
            mul(d0, k);
        }
    }

    // lane (i, q) of fragment (r, c) holds row 16 r + i of columns 16 c + 4 q .. + 3
    constexpr int V = R * C * 4;
    __shared__ float red[W][V][64];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) red[wave][(r * C + c) * 4 + e][lane] = tot[r][c][e] + run[r][c][e];
    __syncthreads();
    for (int v = wave; v < V; v += W) {
        // (as sum_waves, one after the other; 4 waves' sums all in 64 bits. K of two units has no more than
        // two waves' sums: without the branch 500x64 at 100 columns, 64 slices 59.3 us against 56.1, 2500x72
        // at 300 columns 14.0 against 13.3; not for F32, whose 512x512 at 1024 columns took 13.5 us with
        // such a branch against 13.1)
        constexpr int PW = W > 4 ? 2 : 1;
        const auto part = [&](int h) { return PW == 2 ? red[h][v][lane] + red[h + 1][v][lane] : red[h][v][lane]; };
        double s = part(0);
        if (WT == F32 || K > PW * KU) {
#pragma unroll
            for (int h = PW; h < W; h += PW) s += part(h);
        }
        const float sum = (float) s;
        const int r = v / (4 * C), c = v / 4 % C, e = v % 4;
        const int64_t m = m0 + 16 * r + i, t = n0 + 16 * c + 4 * q + e;
        if (m < P.M && t < N) P.y[t * P.ys1 + m] = sum;
    }
}

// the kernel of a launch: rows and columns of a work-group's tile, its waves
struct Form {
    int rows, cols, waves;
};

// Up to 8 columns: 8 per work-group, or 4 (its rows' weights read twice) where the rows alone would
// not fill the CUs: BF16 2048x4096 at 5 columns 8.5 us in 4-column tiles against 9.4, 1024x4096 8.3
// against 9.3, but 4096x4096 14.6 against 10.3. More columns: the largest tile whose work-groups are
// at least the CUs (figures at k_mmf; 2500x520 at 64 columns, 158 32 x 32 tiles, 7.4 us against 6.7
// in 16 x 16), 64 x 32 for F32 only (F16 / BF16 raw data leave it one wave per SIMD).
Form form_of(const MatArgs & a, int64_t rows, int cu_count) {
    const auto groups = [&](int r, int c) { return (rows + r - 1) / r * ((a.N + c - 1) / c) * (a.ne12 * a.ne13); };
    if (a.N <= 4) return {16, 4, 8};
    if (a.N <= 8) return groups(16, 8) >= cu_count ? Form{16, 8, 8} : Form{16, 4, 8};
    if (a.dtype == F32 && groups(64, 32) >= cu_count) return {64, 32, 4};
    if (4 * groups(32, 32) >= 3 * (int64_t) cu_count) return {32, 32, 8};
    return {16, 16, 8};
}

template <int WT, bool XV, bool TAIL>
void * mvq_kernel(const Form & f) {
    return f.cols == 8 ? (void *) k_mvq<WT, 2, XV, TAIL> : (void *) k_mvq<WT, 1, XV, TAIL>;
}

template <int WT, bool XV>
void * kernel_for(const Form & f, bool tail) {
    if constexpr (WT == F32) {
        if (f.rows == 64) return (void *) k_mmf<WT, 4, 2, 4, XV>;
    } else {
        if (f.cols <= 8) return tail ? mvq_kernel<WT, XV, true>(f) : mvq_kernel<WT, XV, false>(f);
    }
    return f.rows == 32 ? (void *) k_mmf<WT, 2, 2, 8, XV> : (void *) k_mmf<WT, 1, 1, 8, XV>;
}

} // namespace

bool matmul_f32_wins(const MatArgs * mats, int nmat, int cu_count) {
    const MatArgs & a = mats[0];
    int64_t rows = 0, tiles = 0;
    for (int j = 0; j < nmat; ++j) {
        rows += mats[j].M * a.ne12 * a.ne13;
        tiles += (mats[j].M + 7) / 8 * a.ne12 * a.ne13;
    }
    // F16 / BF16 at 3..8 columns: from 16-row tiles on three quarters of the CUs, at 5..8 columns
    // (two 4-column tiles per 16 rows) on a quarter: F16 4096x4096 at 4 / 8 columns 9.2 / 11.8 us against
    // 11.9 / 15.3 in the vector kernel, 2048x4096 8.4 / 8.5 against 8.1 / 9.9, 1024x4096 8.4 / 8.3
    // against 7.6 / 9.4; at 2 columns the vector kernel is as fast (12288x4096 19.2 against 20.2).
    // F32, 4 elements per 16-byte load, gains nothing (4096x4096 at 8 columns 19.3 against 20.0).
    if (a.N <= 8) return a.dtype != F32 && a.N >= 3 && rows * (a.N <= 4 ? 1 : 3) >= 12 * (int64_t) cu_count;
    // more: where the vector kernel's 8 x 8 tiles are more than the CUs: F32 128x2048 at 128 columns
    // (256 tiles) 9.4 us against 8.1 there, 300x1024 at 20 (114) 5.8 against 6.0 and at 64 (304) 6.0
    // against 7.7, F16 2500x520 at 9 (626) 4.1 against 9.8
    return tiles * ((a.N + 7) / 8) > cu_count;
}

hipError_t launch_matmul_f32(const MatArgs * mats, int nmat, int cu_count, hipStream_t stream, const char ** kernel_name, uint64_t * grid_size) {
    const MatArgs & a = mats[0];
    if (nmat < 1 || nmat > 3 || !is_float_weight(a.dtype) || a.N < 1 || (a.N <= 8 && a.dtype == F32) || a.K < 8 || a.K % 8 != 0) return hipErrorInvalidValue;
    MmfArgs A;
    std::memset(&A, 0, sizeof(A));
    A.a = a;
    A.nmat = nmat;
    int64_t rows = 0;
    for (int j = 0; j < nmat; ++j) {
        if (mats[j].dtype != a.dtype || mats[j].K != a.K || mats[j].nb != a.nb || mats[j].N != a.N || (nmat > 1 && mats[j].ne12 * mats[j].ne13 != 1)) return hipErrorInvalidValue;
        rows += mats[j].M;
    }
    const int64_t slices = a.ne12 * a.ne13;
    const Form f = form_of(a, rows, cu_count);
    for (int j = 0; j < 3; ++j) {
        const bool has = j < nmat;
        A.wm[j] = has ? mats[j].w : nullptr;
        A.Mm[j] = has ? mats[j].M : 0;
        A.ys1m[j] = has ? mats[j].y_s1 : 0;
        A.mt[j + 1] = A.mt[j] + (has ? (mats[j].M + f.rows - 1) / f.rows : 0);
    }
    if (A.mt[nmat] > 0x7fffffff || slices > 65535) return hipErrorInvalidValue;
    const bool xv = (reinterpret_cast<uintptr_t>(a.x) & 15) == 0 && a.x_s1 % 4 == 0 && a.x_s2 % 4 == 0 && a.x_s3 % 4 == 0;
    const bool tail = a.K % 128 != 0;
    void * fn = a.dtype == F32 ? (xv ? kernel_for<F32, true>(f, tail) : kernel_for<F32, false>(f, tail))
              : a.dtype == F16 ? (xv ? kernel_for<F16, true>(f, tail) : kernel_for<F16, false>(f, tail))
                               : (xv ? kernel_for<BF16, true>(f, tail) : kernel_for<BF16, false>(f, tail));
    if (kernel_name) *kernel_name = a.dtype == F32 ? "matmul_f32" : a.dtype == F16 ? "matmul_f32_f16" : "matmul_f32_bf16";
    std::snprintf(last_form().form, sizeof(last_form().form), "float mfma tile=%dx%d w=%d", f.rows, f.cols, f.waves);
    last_form().grid = (uint64_t) A.mt[nmat] * (uint64_t) slices * (uint64_t) ((a.N + f.cols - 1) / f.cols);
    if (grid_size) *grid_size = last_form().grid;
    // column tiles on blockIdx.z, at most 65535 per launch
    const int64_t per = 65535 * (int64_t) f.cols;
    for (int64_t c0 = 0; c0 < a.N; c0 += per) {
        A.a.N = std::min(per, a.N - c0);
        A.a.x = a.x + c0 * a.x_s1;
        A.a.y = a.y + c0 * a.y_s1;
        for (int j = 0; j < nmat; ++j) A.ym[j] = mats[j].y + c0 * mats[j].y_s1;
        const dim3 grid((unsigned) A.mt[nmat], (unsigned) slices, (unsigned) ((A.a.N + f.cols - 1) / f.cols));
        void * args[] = {&A};
        const hipError_t e = hipLaunchKernel(fn, grid, dim3(64 * f.waves), args, 0, stream);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

} // namespace sgk
