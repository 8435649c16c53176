// Pipelined FP64 complex GEMM: C = alpha op(A) op(B) + beta C, or one split-K partial of it.
//
// Bound by the FP64 matrix cores.  A 64 x 64 tile a workgroup, k steps of 8 through three LDS
// stages that global memory fills directly (global_load_lds, 16 bytes a lane), so a step's
// loads are issued two steps before its products and cost no registers, no LDS stores and no
// masks; one barrier a step.  48 KB of LDS and at most 168 registers leave three workgroups a
// CU.  The 4 waves are stacked along m, each 16 x (16 TN): the last n-tile of a workgroup
// runs TN = 1..4 as its columns need, so n is padded to 16 and not to 64 (97 columns: 112
// instead of 128).  Each complex product is three real ones (P1 = re re, P2 = im im,
// P3 = (re + im)(re + im)), conjugation only changes signs in the sums.
//
// Measured on one MI355X against staging through registers with a prefetch of one step (the
// loads then had half a step to arrive and both waves of a SIMD waited for them; matrix cores
// 67 % busy), us a product: CN 1024 x 256 x 228487 6542 -> 5376 (89 TFLOP/s of 8 m n k; the
// three-product loop alone, from LDS, reaches 98), CN 512 x 160 x 51627 592 -> 427,
// CN 577 x 97 x 51627 487 -> 397, NN 228487 x 256 x 1024 6607 -> 5333.  Waves 2 x 2 instead of
// stacked: 5997 on the first; four stages (two workgroups a CU): 6159; 128 x 32: 6157;
// 128 x 64 (one workgroup a CU): 7058; 64 x 32: 6070.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

namespace apw {
namespace {

typedef double zacc_t __attribute__((ext_vector_type(4)));

constexpr int ZP_BM = 64, ZP_BN = 64, ZP_BK = 8, ZP_NT = 256, ZP_ST = 3, ZP_OCC = 3;

// slot of element (row, k) in a stage: row-fastest operands as [k][row]; k-fastest ones as
// [row][k] with k xor-ed by the row pair, so that 16 rows at one k fall on all banks
template <bool KF>
__device__ __forceinline__ int zp_slot(int row, int k) {
    static_assert(ZP_BM == ZP_BN, "one row count for both operands");
    return KF ? row * ZP_BK + (k ^ ((row >> 1) & 7)) : k * ZP_BM + row;
}

// The k loop of one tile, TN sub-tiles of 16 columns wide.  s0, s1, s2: one shared variable a
// stage, so that the compiler sees that a read of one does not wait for the loads in flight
// into the others.
template <int TA, int TB, int TN>
__device__ __forceinline__ void zp_tile(int M, int N, const double2* __restrict__ A, int lda,
                                        const double2* __restrict__ B, int ldb, int m0, int n0, int kbeg, int kend,
                                        double2* s0, double2* s1, double2* s2, zacc_t (&p1)[TN], zacc_t (&p2)[TN],
                                        zacc_t (&p3)[TN]) {
    constexpr int BK = ZP_BK, NT = ZP_NT, SA = ZP_BM * BK;
    constexpr bool AK = TA != 0, BKF = TB == 0;   // k-fastest operands
    constexpr int NA = SA / NT, NB = BKF ? (TN + 1) / 2 : ZP_BN * BK / NT, NL = NA + NB;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nsteps = (kend - kbeg + BK - 1) / BK;
    auto stage = [&](auto sc) -> double2* {
        constexpr int s = decltype(sc)::value % ZP_ST;
        if constexpr (s == 0) return s0;
        else if constexpr (s == 1) return s1;
        else return s2;
    };
    auto any_stage = [&](int s) -> double2* { return s == 0 ? s0 : s == 1 ? s1 : s2; };

    // Row and k of each element this lane loads.  Rows past M or N read the last row (their
    // products are never stored); k past the end reads the last k and is zeroed in LDS.
    int arow[NA], ak[NA], brow[NB], bk[NB];
#pragma unroll
    for (int i = 0; i < NA; ++i) {
        const int e = tid + NT * i, r = AK ? e / BK : e % ZP_BM;
        arow[i] = min(m0 + r, M - 1);
        ak[i] = AK ? (e % BK) ^ ((r >> 1) & 7) : e / ZP_BM;
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        const int e = tid + NT * i, r = BKF ? e / BK : e % ZP_BN;
        brow[i] = min(n0 + r, N - 1);
        bk[i] = BKF ? (e % BK) ^ ((r >> 1) & 7) : e / ZP_BN;
    }
    auto fill = [&](const double2* src, double2* dst) {   // 64 lanes x 16 bytes to dst[0 .. 63]
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                         (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
    };
    auto load = [&](int step, double2* dst) {
        const int k0 = kbeg + step * BK;
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const int gk = min(k0 + ak[i], kend - 1);
            fill(A + (AK ? (size_t)arow[i] * lda + gk : (size_t)gk * lda + arow[i]), dst + NT * i + 64 * wave);
        }
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int gk = min(k0 + bk[i], kend - 1);
            fill(B + (BKF ? (size_t)brow[i] * ldb + gk : (size_t)gk * ldb + brow[i]), dst + SA + NT * i + 64 * wave);
        }
    };
    auto compute = [&](const double2* s) {
#pragma unroll
        for (int ks = 0; ks < BK / 4; ++ks) {
            const int kk = ks * 4 + (lane >> 4);
            const double2 y = s[zp_slot<AK>(wave * 16 + (lane & 15), kk)];
            const double ys = TA == 2 ? y.x - y.y : y.x + y.y;
#pragma unroll
            for (int t = 0; t < TN; ++t) {
                const double2 x = s[SA + zp_slot<BKF>(t * 16 + (lane & 15), kk)];
                const double xs = TB == 2 ? x.x - x.y : x.x + x.y;
                p1[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.x, y.x, p1[t], 0, 0, 0);
                p2[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.y, y.y, p2[t], 0, 0, 0);
                p3[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(xs, ys, p3[t], 0, 0, 0);
            }
        }
    };
    // One step: wait for this wave's share of the stage (the next step's loads stay in flight),
    // meet the other waves -- every share has landed, and every wave has read the stage that
    // the new loads overwrite --, issue the loads of step + 2, multiply.
    auto one = [&](int step, auto sc) {
        constexpr int s = decltype(sc)::value, left = NL * (ZP_ST - 2);
        static_assert(left < 16, "vmcnt field");
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(left | (7 << 4));   // vmcnt(left) lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        load(step + ZP_ST - 1, stage(std::integral_constant<int, s + ZP_ST - 1>{}));
        compute(stage(sc));
    };

    if (nsteps > 0) load(0, s0);
    if (nsteps > 1) load(1, s1);
    int step = 0;
    for (; step + 2 * ZP_ST - 2 < nsteps; step += ZP_ST) {
        one(step, std::integral_constant<int, 0>{});
        one(step + 1, std::integral_constant<int, 1>{});
        one(step + 2, std::integral_constant<int, 2>{});
    }
    // the last steps (at most 4), each waiting for every load in flight
    for (; step < nsteps; ++step) {
        double2* const cur = any_stage(step % ZP_ST);
        __syncthreads();
        if (step + ZP_ST - 1 < nsteps) load(step + ZP_ST - 1, any_stage((step + ZP_ST - 1) % ZP_ST));
        const int valid = kend - (kbeg + step * BK);
        if (valid < BK) {   // the last step of a ragged k: zeros past the end
            for (int e = tid; e < ZP_BM * (BK - valid); e += NT) {
                const int row = e % ZP_BM, k = valid + e / ZP_BM;
                cur[zp_slot<AK>(row, k)] = double2{0.0, 0.0};
                cur[SA + zp_slot<BKF>(row, k)] = double2{0.0, 0.0};
            }
            __syncthreads();
        }
        compute(cur);
    }
}

// op codes: 0 = N, 1 = T, 2 = C.  A and B 16-byte aligned.  map 0: grid (m-tiles, n-tiles,
// splits); map 1 (no split, 1-D grid padded to a multiple of 8 m-tiles): workgroup L runs on
// XCD L % 8, so each XCD takes whole m-tiles and walks their n-tiles back to back, and the
// rows of A that they share stay in its L2.
template <int TA, int TB>
__global__ __launch_bounds__(ZP_NT, ZP_OCC) void zgemm_pipe(int M, int N, int K, int kchunk, int map,
                                                            const double2* __restrict__ A, int lda,
                                                            const double2* __restrict__ B, int ldb,
                                                            double2* __restrict__ C, int ldc, double ar, double ai,
                                                            double br, double bi, double2* __restrict__ part) {
    __shared__ __align__(16) double2 s0[(ZP_BM + ZP_BN) * ZP_BK], s1[(ZP_BM + ZP_BN) * ZP_BK],
        s2[(ZP_BM + ZP_BN) * ZP_BK];
    int bm = blockIdx.x, bn = blockIdx.y, sp = blockIdx.z;
    if (map == 1) {
        const int L = blockIdx.x, ntn = (N + ZP_BN - 1) / ZP_BN;
        bm = (L % 8) + 8 * (L / (8 * ntn));
        bn = (L / 8) % ntn;
        if (bm >= (M + ZP_BM - 1) / ZP_BM) return;
    }
    const int m0 = bm * ZP_BM, n0 = bn * ZP_BN;
    const int kbeg = sp * kchunk, kend = min(K, kbeg + kchunk);
    const int lane = threadIdx.x & 63, gm = m0 + (int)(threadIdx.x >> 6) * 16 + (lane & 15);

    auto run = [&](auto tnc) {
        constexpr int TN = decltype(tnc)::value;
        zacc_t p1[TN], p2[TN], p3[TN];
#pragma unroll
        for (int t = 0; t < TN; ++t) p1[t] = p2[t] = p3[t] = zacc_t{0, 0, 0, 0};
        zp_tile<TA, TB, TN>(M, N, A, lda, B, ldb, m0, n0, kbeg, kend, s0, s1, s2, p1, p2, p3);
        if (gm >= M) return;
        // lane holds D[n = lane / 16 + 4 r][m = lane % 16] of each sub-tile
#pragma unroll
        for (int t = 0; t < TN; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int gn = n0 + t * 16 + (lane >> 4) + 4 * r;
                if (gn >= N) continue;
                const double q1 = p1[t][r], q2 = (TA == 2) != (TB == 2) ? -p2[t][r] : p2[t][r];
                const double xr = q1 - q2, xi = p3[t][r] - (q1 + q2);
                if (part) {
                    part[(size_t)sp * M * N + gm + (size_t)gn * M] = double2{xr, xi};
                    continue;
                }
                double cr = ar * xr - ai * xi, ci = ar * xi + ai * xr;
                double2* cp = C + gm + (size_t)gn * ldc;
                if (br != 0.0 || bi != 0.0) {
                    const double2 c = *cp;
                    cr += br * c.x - bi * c.y;
                    ci += br * c.y + bi * c.x;
                }
                *cp = double2{cr, ci};
            }
    };
    switch (min(4, (N - n0 + 15) / 16)) {
        case 1: run(std::integral_constant<int, 1>{}); break;
        case 2: run(std::integral_constant<int, 2>{}); break;
        case 3: run(std::integral_constant<int, 3>{}); break;
        default: run(std::integral_constant<int, 4>{}); break;
    }
}

}  // namespace
}  // namespace apw
