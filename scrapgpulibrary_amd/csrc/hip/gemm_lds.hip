// Prefill GEMM over 16-bit weights (F16 / BF16 rows in the natural layout, gfx950, wave64): both
// operands through LDS, moved there by LDS-direct loads several stages ahead.
//
// The same product as the other prefill kernels (matmul.hip; reference ops_matmul.cpp:67-204): x as
// f16 rows scaled by a power of two (bf16 for BF16 weights) from the pre-pass, f16 / bf16 MFMA with
// f32 accumulate, the rows' factors undone in the epilogue.
//
// Why: with its weights loaded straight into the MFMA's lanes (32 rows x 32 bytes per load) such a
// GEMM was bound by its cache-line requests; here every load moves 8 whole 128-byte lines, and the
// next stages' loads stay in flight across the stage barriers. Measured (op time with the pre-pass):
// BF16 12288x4096 at 512 tokens 100.3 -> 63.3 us (one 192-row tile per CU), at 2048 268 -> 229;
// 4096x12288 at 512 122 -> 82; 4096x4096 at 512 54.6 -> 34.4; 20000x8192 at 1500 997 -> 529; F16
// 12288x4096 at 128 56 -> 46. What bounds it now: the operands' bytes into each CU, about 50 GB/s per
// CU with all of them at it (2.6 MB per 192 x 128 tile of K = 4096: 53 us without the MFMAs, 40 us
// without the loads; contiguous instead of row-wise addresses, and 3 stages in LDS instead of 4,
// change nothing).
#include "kernels.h"

#include <hip/hip_fp16.h>

#include <algorithm>
#include <cstdio>
#include <cstring>
#include <type_traits>

namespace sgk {
namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

template <int DT>
__device__ __forceinline__ f32x16 mma(const f16x8 & a, const f16x8 & b, const f32x16 & c) {
    if constexpr (DT == BF16) return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

constexpr int SKE = 64;            // elements of K per stage
constexpr int kRowBytes = 2 * SKE; // one row (or token) of a stage: 8 chunks of 16 bytes

// A work-group: RW row waves x 2 token waves x KG K groups (2: the groups take the first and the
// second half of every stage and add their sums at the end). A wave owns 32 RT rows x 64 tokens.
// NBUF stages in LDS.
template <int DT, int RT, int RW, int KG, int NBUF>
__global__ __launch_bounds__(128 * RW * KG, 1) void k_gemm_l(LdsGemm L) {
    constexpr int W = 2 * RW * KG, KS = 4 / KG; // waves, k-steps of a stage per wave
    constexpr int BM = 32 * RT * RW, BN = 128;
    constexpr int WI = BM / 8 / W, XI = (BN / 8 + W - 1) / W; // LDS-direct loads per wave and stage (8 rows each)
    constexpr bool EVEN = BN / 8 % W == 0;
    static_assert(BM / 8 % W == 0 && (EVEN || NBUF == 2), "the waits count the same loads in every wave");
    constexpr int NI = WI + XI;
    constexpr int kBuf = (BM + BN) * kRowBytes;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kg = KG == 1 ? 0 : wid / (2 * RW), tw = wid % (2 * RW) / RW, rw = wid % RW;
    const int j = lane & 31, h = lane >> 5;

    // tiles in runs per XCD (work-groups go round the 8 XCDs in turn), the token tiles of one row
    // tile next to each other: an XCD's L2 serves its rows' weights to all of them
    const int T = L.tiles_m * L.tiles_n;
    const int split = blockIdx.x / T, id = blockIdx.x - split * T;
    const int per = T / 8, rem = T % 8, xcd = id % 8;
    const int lin = xcd * per + min(xcd, rem) + id / 8;
    const int tm = lin / L.tiles_n, tn = lin - tm * L.tiles_n;
    const int mj = tm >= L.mt[1] ? (tm >= L.mt[2] ? 2 : 1) : 0;
    const uint8_t * w = L.wm[mj];
    float * y = L.ym[mj];
    const uint16_t * xb = L.xb;
    const float * xs = L.xs;
    int64_t ys1 = L.ys1m[mj];
    if (gridDim.y > 1) {
        const int64_t sl = blockIdx.y, i2 = sl % L.ne12, i3 = sl / L.ne12;
        w += (uint64_t) (i2 / L.r2) * L.w_s2 + (uint64_t) (i3 / L.r3) * L.w_s3;
        y += i2 * L.y_s2 + i3 * L.y_s3;
        xb += (uint64_t) sl * L.N * L.K;
        xs += (uint64_t) sl * L.N;
    }
    const int M = L.Mm[mj], N = L.N, K = L.K;
    const int m0 = (tm - L.mt[mj]) * BM, n0 = tn * BN;
    const int stages = K / SKE;
    const int s0 = (int) ((int64_t) stages * split / L.split), s1 = (int) ((int64_t) stages * (split + 1) / L.split);

    // Loads: instruction i of a wave moves 8 rows of 128 bytes into 1 KiB of LDS. Row r's chunk c
    // sits at chunk position c ^ (r / 2 % 8), so the 16 rows that one cycle of a 16-byte LDS read
    // serves (one chunk of each) lie in 16 different groups of banks; the lanes of a row read one
    // whole line of memory either way. Rows past M and tokens past N read the last one (their
    // products are never stored).
    uint32_t off[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int ins = wid + W * (i < WI ? i : i - WI);
        const int r = 8 * ins + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
        off[i] = (i < WI ? (uint32_t) min(m0 + r, M - 1) * (uint32_t) L.nb : (uint32_t) min(n0 + r, N - 1) * (uint32_t) (2 * K)) + 16 * c;
    }
    const auto fetch = [&](int s, int buf) __attribute__((always_inline)) {
        const uint32_t k = (uint32_t) min(s, s1 - 1) * kRowBytes; // (past the last stage: its data again, unused)
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const uint8_t * p = (i < WI ? w : reinterpret_cast<const uint8_t *>(xb)) + k;
            const int ins = wid + W * (i < WI ? i : i - WI);
            if (!EVEN && i >= WI && ins >= BN / 8) continue;
            uint8_t * d = lds + buf * kBuf + (i < WI ? 0 : BM * kRowBytes) + ins * 1024;
            __builtin_amdgcn_global_load_lds(reinterpret_cast<const void *>(p + off[i]), (__attribute__((address_space(3))) void *) d, 16, 0, 0);
        }
    };
    // the lane's chunk of its K group's k-step t in a row whose first row is a multiple of 32
    uint32_t lo[KS];
#pragma unroll
    for (int t = 0; t < KS; ++t) lo[t] = j * kRowBytes + 16 * ((4 * kg + 2 * t + h) ^ ((j >> 1) & 7));
    f16x8 fw[2][RT], fx[2][2];
    const auto read = [&](int buf, auto tt) __attribute__((always_inline)) {
        constexpr int t = decltype(tt)::value;
        const uint8_t * b = lds + buf * kBuf + lo[t];
#pragma unroll
        for (int q = 0; q < 2; ++q) fx[t & 1][q] = *reinterpret_cast<const f16x8 *>(b + (BM + 64 * tw + 32 * q) * kRowBytes);
#pragma unroll
        for (int r = 0; r < RT; ++r) fw[t & 1][r] = *reinterpret_cast<const f16x8 *>(b + (32 * RT * rw + 32 * r) * kRowBytes);
    };
    f32x16 acc[RT][2];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[r][q][v] = 0.0f;
    const auto mul = [&](auto tt) __attribute__((always_inline)) {
        constexpr int t = decltype(tt)::value;
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int q = 0; q < 2; ++q) acc[r][q] = mma<DT>(fx[t & 1][q], fw[t & 1][r], acc[r][q]);
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;

    // The waits: loads complete in order, NI per stage. Stage s + 1 has landed when all but the
    // NBUF - 2 newest stages have; the barrier makes that true of every wave's share, and says that
    // every wave has its last fragments of stage s in registers (lgkmcnt(0)), so that its buffer may
    // be refilled. The MFMAs on both sides of the barrier work from registers.
#define SG_WAIT(n) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(n) : "memory")
#pragma unroll
    for (int b = 0; b < NBUF; ++b) fetch(s0 + b, b);
    SG_WAIT(EVEN ? (NBUF - 1) * NI : 0);
    read(0, I0{});
    const auto step = [&](int b, auto tt) __attribute__((always_inline)) {
        constexpr int t = decltype(tt)::value;
        read(b, std::integral_constant<int, t + 1>{});
        __builtin_amdgcn_sched_barrier(0);
        mul(tt);
    };
    const auto stage = [&](int s, auto bt) __attribute__((always_inline)) {
        constexpr int b = decltype(bt)::value;
        step(b, I0{});
        if constexpr (KS == 4) {
            step(b, I1{});
            step(b, std::integral_constant<int, 2>{});
        }
        SG_WAIT((NBUF - 2) * NI);
        fetch(s + NBUF, b);
        read((b + 1) % NBUF, I0{});
        __builtin_amdgcn_sched_barrier(0);
        mul(std::integral_constant<int, KS - 1>{});
    };
    int s = s0;
    for (; s + NBUF <= s1; s += NBUF) {
        stage(s, std::integral_constant<int, 0>{});
        stage(s + 1, std::integral_constant<int, 1>{});
        if constexpr (NBUF == 4) {
            stage(s + 2, std::integral_constant<int, 2>{});
            stage(s + 3, std::integral_constant<int, 3>{});
        }
    }
    if (s < s1) stage(s, std::integral_constant<int, 0>{});
    if constexpr (NBUF == 4) {
        if (s + 1 < s1) stage(s + 1, std::integral_constant<int, 1>{});
        if (s + 2 < s1) stage(s + 2, std::integral_constant<int, 2>{});
    }
    SG_WAIT(0); // (no load in flight writes LDS any more)

    float * o = y;
    int64_t os = ys1;
    if (L.split > 1) {
        const int64_t Mt = L.mo[L.nmat];
        o = L.part + ((uint64_t) split * gridDim.y + blockIdx.y) * N * Mt + L.mo[mj];
        os = Mt;
    }
    // lane (j, h), register v of a fragment: token 8 (v / 4) + 4 h + v % 4, row j
    const auto store = [&](auto qt, const float * other) __attribute__((always_inline)) {
        constexpr int Q = decltype(qt)::value;
        const int nb = n0 + 64 * tw + 32 * Q + 4 * h;
        float u[16];
#pragma unroll
        for (int v = 0; v < 16; ++v) u[v] = xs[min(nb + 8 * (v >> 2) + (v & 3), N - 1)];
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const int m = m0 + 32 * RT * rw + 32 * r + j;
            float c[16];
#pragma unroll
            for (int v = 0; v < 16; ++v) c[v] = (KG == 1 ? acc[r][Q][v] : acc[r][Q][v] + other[(r * 16 + v) * 64]) * u[v];
            if (m >= M) continue;
            if (nb - 4 * h + 32 <= N) {
#pragma unroll
                for (int v = 0; v < 16; ++v) __builtin_nontemporal_store(c[v], o + (nb + 8 * (v >> 2) + (v & 3)) * os + m);
            } else {
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    if (nb + 8 * (v >> 2) + (v & 3) < N) __builtin_nontemporal_store(c[v], o + (nb + 8 * (v >> 2) + (v & 3)) * os + m);
            }
        }
    };
    if constexpr (KG == 1) {
        store(I0{}, nullptr);
        store(I1{}, nullptr);
        return;
    }
    // the K groups exchange half of their sums: group g finishes token fragment g of each row
    // fragment (a + b = b + a: no order to keep)
    float * red = reinterpret_cast<float *>(lds);
    const auto finish = [&](auto gt) __attribute__((always_inline)) {
        constexpr int G = decltype(gt)::value;
        const int peer = wid + (G == 0 ? 2 * RW : -2 * RW);
        float * mine = red + (size_t) (wid * RT * 16) * 64 + lane;
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int v = 0; v < 16; ++v) mine[(r * 16 + v) * 64] = acc[r][1 - G][v];
        __syncthreads();
        store(gt, red + (size_t) (peer * RT * 16) * 64 + lane);
    };
    if (kg == 0) finish(I0{});
    else finish(I1{});
#undef SG_WAIT
}

} // namespace

hipError_t launch_gemm_lds(const LdsGemm & L, int dtype, int rows, int slices, hipStream_t stream) {
    if ((dtype != F16 && dtype != BF16) || (rows != 128 && rows != 192 && rows != 384) || L.K % SKE != 0 || L.K / SKE < L.split) return hipErrorInvalidValue;
    void * fn = nullptr;
    if (dtype == F16) fn = rows == 384 ? (void *) k_gemm_l<F16, 2, 6, 1, 2> : rows == 192 ? (void *) k_gemm_l<F16, 3, 2, 2, 4> : (void *) k_gemm_l<F16, 2, 2, 2, 4>;
    else fn = rows == 384 ? (void *) k_gemm_l<BF16, 2, 6, 1, 2> : rows == 192 ? (void *) k_gemm_l<BF16, 3, 2, 2, 4> : (void *) k_gemm_l<BF16, 2, 2, 2, 4>;
    const size_t lds = (size_t) (rows == 384 ? 2 : 4) * (rows + 128) * kRowBytes;
    const hipError_t e = allow_lds(fn, lds);
    if (e != hipSuccess) return e;
    LdsGemm A = L;
    void * args[] = {&A};
    return hipLaunchKernel(fn, dim3((unsigned) (L.tiles_m * L.tiles_n * L.split), (unsigned) slices), dim3(rows == 384 ? 768 : 512), args, lds, stream);
}

} // namespace sgk
