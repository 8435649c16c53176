// Pipelined complex GEMM, c128 and c64: C = alpha op(A) op(B) + beta C, or one split-K partial.
//
// Bound by the matrix cores.  A 64 x 64 tile a workgroup, k steps of 8 (c64: 16) through three
// LDS stages that global memory fills directly (global_load_lds, 16 bytes a lane, at any
// alignment), so a step's loads are issued two steps before its products and cost no
// registers, no LDS stores and no masks; one barrier a step.  48 KB of LDS and at most 168
// registers leave three workgroups a CU.  The 4 waves are stacked along m, each 16 x (16 TN): the
// last n-tile of a workgroup runs TN = 1..4 as its columns need, so n is padded to 16 and not to
// 64 (97 columns: 112 instead of 128).  Each complex product is three real ones (P1 = re re,
// P2 = im im, P3 = (re + im)(re + im); re = P1 - P2, im = P3 - P1 - P2): the error stays normwise,
// a few ulps of |a||b| per term; conjugation only changes signs in the sums.
//
// Measured on one MI355X against staging through registers with a prefetch of one step (the
// loads then had half a step to arrive and both waves of a SIMD waited for them; matrix cores
// 67 % busy), us of device time a product with its split-K reduction, after a warm-up (the first
// ten passes run at lower clocks and take up to 20 % longer): c128 CN 1024 x 256 x 228487 6570 ->
// 5480 (87 TFLOP/s of 8 m n k; the three-product loop alone, from LDS, reaches 98), CN 512 x 160 x
// 51627 579 -> 413, CN 577 x 97 x 51627 498 -> 369, NN 228487 x 256 x 1024 6617 -> 5328; c64 CN 512 x
// 160 x 51627 323 -> 209, NN 51627 x 160 x 512 279 -> 216 (157 TFLOP/s).  The first of these in a
// program of its own, where this form took 5376: waves 2 x 2 instead of stacked 5997; four stages
// (two workgroups a CU) 6159; 128 x 32 6157; 128 x 64 (one workgroup a CU) 7058; 64 x 32 6070.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

namespace apw {
namespace {

template <class R>
struct ZpType;
template <>
struct ZpType<double> {
    using c_t = double2;
    typedef double acc_t __attribute__((ext_vector_type(4)));
    static constexpr int BK = 8;   // k of a step: 128 bytes of a k-fastest row
    __device__ static __forceinline__ acc_t mma(double a, double b, acc_t c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    // row of D in accumulator register r of a lane (column = lane % 16)
    __device__ static __forceinline__ int drow(int lane, int r) { return (lane >> 4) + 4 * r; }
};
template <>
struct ZpType<float> {
    using c_t = float2;
    typedef float acc_t __attribute__((ext_vector_type(4)));
    static constexpr int BK = 16;
    __device__ static __forceinline__ acc_t mma(float a, float b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    __device__ static __forceinline__ int drow(int lane, int r) { return 4 * (lane >> 4) + r; }
};

constexpr int ZP_BM = 64, ZP_BN = 64, ZP_NT = 256, ZP_ST = 3, ZP_OCC = 3;
static_assert(ZP_BM == ZP_BN, "one row count for both operands");
template <class R>
constexpr int zp_stage() { return (ZP_BM + ZP_BN) * ZpType<R>::BK; }   // elements

// Where element (row, k) of an operand lies in its half of a stage, and which element a
// 16-byte piece begins with (c64: two elements along the fastest index).  Row-fastest operands
// lie as [k][row], k-fastest ones as [row][k]; the xors put the lanes that read together (16
// rows at one k, for c64 at two) on all banks.
template <class R, bool KF>
__device__ __forceinline__ int zp_slot(int row, int k) {
    constexpr int BK = ZpType<R>::BK;
    if constexpr (sizeof(R) == 8) return KF ? row * BK + (k ^ ((row >> 1) & 7)) : k * ZP_BM + row;
    else return KF ? row * BK + (k ^ (((row >> 1) & 7) << 1)) : k * ZP_BM + (row ^ ((k & 1) << 4));
}
template <class R, bool KF>
__device__ __forceinline__ void zp_piece(int e, int& row, int& k) {
    if constexpr (KF) {
        row = e / 8;
        k = ((e % 8) ^ ((row >> 1) & 7)) * (16 / (2 * (int)sizeof(R)));
    } else if constexpr (sizeof(R) == 8) {
        row = e % ZP_BM;
        k = e / ZP_BM;
    } else {
        k = e / (ZP_BM / 2);
        row = (2 * (e % (ZP_BM / 2))) ^ ((k & 1) << 4);
    }
}

// The k loop of one tile, TN sub-tiles of 16 columns wide.  s0, s1, s2: one shared variable a
// stage, so that the compiler sees that a read of one does not wait for the loads in flight
// into the others.
template <class R, int TA, int TB, int TN>
__device__ __forceinline__ void zp_tile(int M, int N, const typename ZpType<R>::c_t* __restrict__ A, int lda,
                                        const typename ZpType<R>::c_t* __restrict__ B, int ldb, int m0, int n0,
                                        int kbeg, int kend, typename ZpType<R>::c_t* s0, typename ZpType<R>::c_t* s1,
                                        typename ZpType<R>::c_t* s2, typename ZpType<R>::acc_t (&p1)[TN],
                                        typename ZpType<R>::acc_t (&p2)[TN], typename ZpType<R>::acc_t (&p3)[TN]) {
    using Z = ZpType<R>;
    using C = typename Z::c_t;
    constexpr int BK = Z::BK, NT = ZP_NT, SA = ZP_BM * BK, PC = 16 / (int)sizeof(C);   // elements of a piece
    constexpr bool AK = TA != 0, BKF = TB == 0;   // k-fastest operands
    // c64: a piece may begin at the last row or k and end past it, where the next column still
    // is in the array except in the last k; so the last step comes element by element, through
    // registers that are loaded at the start
    constexpr bool TAIL = PC > 1;
    constexpr int NA = SA / PC / NT, NB = BKF ? (TN + 1) / 2 : NA, NL = NA + NB;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nsteps = (kend - kbeg + BK - 1) / BK, direct = TAIL ? nsteps - 1 : nsteps;
    auto stage = [&](auto sc) -> C* {
        constexpr int s = decltype(sc)::value % ZP_ST;
        if constexpr (s == 0) return s0;
        else if constexpr (s == 1) return s1;
        else return s2;
    };
    auto any_stage = [&](int s) -> C* { return s == 0 ? s0 : s == 1 ? s1 : s2; };

    // Row and k of each piece this lane loads.  Rows past M or N read the last row (their
    // products are never stored); c128: k past the end reads the last k and is zeroed in LDS.
    int arow[NA], ak[NA], brow[NB], bk[NB];
#pragma unroll
    for (int i = 0; i < NA; ++i) {
        zp_piece<R, AK>(tid + NT * i, arow[i], ak[i]);
        arow[i] = min(m0 + arow[i], M - 1);
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        zp_piece<R, BKF>(tid + NT * i, brow[i], bk[i]);
        brow[i] = min(n0 + brow[i], N - 1);
    }
    auto fill = [&](const C* src, C* dst) {   // 64 lanes x 16 bytes to dst
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                         (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
    };
    auto load = [&](int step, C* dst) {
        const int k0 = kbeg + step * BK;
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const int gk = TAIL ? k0 + ak[i] : min(k0 + ak[i], kend - 1);
            fill(A + (AK ? (size_t)arow[i] * lda + gk : (size_t)gk * lda + arow[i]), dst + PC * (NT * i + 64 * wave));
        }
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int gk = TAIL ? k0 + bk[i] : min(k0 + bk[i], kend - 1);
            fill(B + (BKF ? (size_t)brow[i] * ldb + gk : (size_t)gk * ldb + brow[i]),
                 dst + SA + PC * (NT * i + 64 * wave));
        }
    };
    // the last step's elements (TAIL): element e is row e % 64, k e / 64 (k-fastest: the other
    // way round), stored as zero past the end of k
    constexpr int NT_EL = TAIL ? SA / NT : 0;
    C ta[TAIL ? NT_EL : 1], tb[TAIL ? NT_EL : 1];
    auto tail_at = [&](int i, bool kf, int& row, int& k) {
        const int e = tid + NT * i;
        row = kf ? e / BK : e % ZP_BM;
        k = kf ? e % BK : e / ZP_BM;
    };
    if constexpr (TAIL) {
        const int k0 = kbeg + (nsteps - 1) * BK;
#pragma unroll
        for (int i = 0; i < NT_EL; ++i) {
            int row, k;
            tail_at(i, AK, row, k);
            const int r = min(m0 + row, M - 1), gk = min(k0 + k, kend - 1);
            ta[i] = A[AK ? (size_t)r * lda + gk : (size_t)gk * lda + r];
            tail_at(i, BKF, row, k);
            const int rb = min(n0 + row, N - 1), gb = min(k0 + k, kend - 1);
            tb[i] = B[BKF ? (size_t)rb * ldb + gb : (size_t)gb * ldb + rb];
        }
    }
    auto put = [&](int step, C* dst) {
        if (step < direct) {
            load(step, dst);
            return;
        }
        if constexpr (TAIL) {
            if (step != direct) return;
#pragma unroll
            for (int i = 0; i < NT_EL; ++i) {
                int row, k;
                tail_at(i, AK, row, k);
                dst[zp_slot<R, AK>(row, k)] = kbeg + direct * BK + k < kend ? ta[i] : C{0, 0};
                tail_at(i, BKF, row, k);
                dst[SA + zp_slot<R, BKF>(row, k)] = kbeg + direct * BK + k < kend ? tb[i] : C{0, 0};
            }
        }
    };
    auto compute = [&](const C* s) {
#pragma unroll
        for (int ks = 0; ks < BK / 4; ++ks) {
            const int kk = ks * 4 + (lane >> 4);
            const C y = s[zp_slot<R, AK>(wave * 16 + (lane & 15), kk)];
            const R ys = TA == 2 ? y.x - y.y : y.x + y.y;
#pragma unroll
            for (int t = 0; t < TN; ++t) {
                const C x = s[SA + zp_slot<R, BKF>(t * 16 + (lane & 15), kk)];
                const R xs = TB == 2 ? x.x - x.y : x.x + x.y;
                p1[t] = Z::mma(x.x, y.x, p1[t]);
                p2[t] = Z::mma(x.y, y.y, p2[t]);
                p3[t] = Z::mma(xs, ys, p3[t]);
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

    put(0, s0);
    put(1, s1);
    int step = 0;
    for (; step + 2 * ZP_ST - 2 < direct; step += ZP_ST) {
        one(step, std::integral_constant<int, 0>{});
        one(step + 1, std::integral_constant<int, 1>{});
        one(step + 2, std::integral_constant<int, 2>{});
    }
    // the last steps (at most 5), each waiting for every load in flight
    for (; step < nsteps; ++step) {
        C* const cur = any_stage(step % ZP_ST);
        // the barrier alone does not wait for fills in flight: the compiler's own waits cover what
        // this wave reads, not what it has filled for the others
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(7 << 4);   // vmcnt(0) lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        put(step + ZP_ST - 1, any_stage((step + ZP_ST - 1) % ZP_ST));
        if constexpr (!TAIL) {
            const int valid = kend - (kbeg + step * BK);
            if (valid < BK) {   // the last step of a ragged k: zeros past the end
                for (int e = tid; e < ZP_BM * (BK - valid); e += NT) {
                    const int row = e % ZP_BM, k = valid + e / ZP_BM;
                    cur[zp_slot<R, AK>(row, k)] = C{0, 0};
                    cur[SA + zp_slot<R, BKF>(row, k)] = C{0, 0};
                }
                __syncthreads();
            }
        }
        compute(cur);
    }
}

// op codes: 0 = N, 1 = T, 2 = C.  map 0: grid (m-tiles, n-tiles,
// splits); map 1 (1-D grid in x padded to a multiple of 8 m-tiles): workgroup L runs on
// XCD L % 8, so each XCD takes whole m-tiles and walks their n-tiles back to back, and the
// rows of A that they share stay in its L2; a last, narrower n-tile comes after all of those, so
// that the launch ends on short workgroups (a call of 51627 x 160 x 512: 453 -> 437 us, 228487 x 200 x
// 1024 5.31 -> 4.74 ms, against the narrow ones in turn with the others).  map 2 (k split for one or two full rounds of
// workgroups, 1-D grid of 8 (zp_share(wide) + zp_share(narrow))): each XCD takes an eighth of the
// splits, all full-width tiles before those of the last, narrower n-tile, so that the workgroups that meet
// on a CU (one every num_cu / 8 of an XCD) are a like mix of both on every CU; with m-major order
// some CUs got the wide ones only.
__host__ __device__ inline int zp_share(int tiles) { return (tiles + 7) / 8; }
template <class R, int TA, int TB>
__global__ __launch_bounds__(ZP_NT, ZP_OCC) void zgemm_pipe(int M, int N, int K, int kchunk, int map,
                                                            const typename ZpType<R>::c_t* __restrict__ A, int lda,
                                                            const typename ZpType<R>::c_t* __restrict__ B, int ldb,
                                                            typename ZpType<R>::c_t* __restrict__ C, int ldc,
                                                            double ar, double ai, double br, double bi,
                                                            typename ZpType<R>::c_t* __restrict__ part) {
    using Z = ZpType<R>;
    using c_t = typename Z::c_t;
    __shared__ __align__(16) c_t s0[zp_stage<R>()], s1[zp_stage<R>()], s2[zp_stage<R>()];
    int bm = blockIdx.x, bn = blockIdx.y, sp = blockIdx.z;
    if (map == 1) {
        const int L = blockIdx.x, nw = N / ZP_BN, full = (M + 8 * ZP_BM - 1) / (8 * ZP_BM) * 8 * nw;
        if (L < full) {
            bm = (L % 8) + 8 * (L / (8 * nw));
            bn = (L / 8) % nw;
        } else {
            bm = L - full;
            bn = nw;
        }
        if (bm >= (M + ZP_BM - 1) / ZP_BM) return;
    }
    if (map == 2) {
        const int tmt = (M + ZP_BM - 1) / ZP_BM, nw = N / ZP_BN, splits = (K + kchunk - 1) / kchunk;
        const int wide = splits * tmt * nw, narrow = N % ZP_BN ? splits * tmt : 0;
        const int x = blockIdx.x % 8, j = blockIdx.x / 8;
        int g;
        if (j < zp_share(wide)) {
            g = x * zp_share(wide) + j;
            if (g >= wide) return;
            bn = g % nw;
            g /= nw;
        } else {
            g = x * zp_share(narrow) + j - zp_share(wide);
            if (g >= narrow) return;
            bn = nw;
        }
        bm = g % tmt;
        sp = g / tmt;
    }
    const int m0 = bm * ZP_BM, n0 = bn * ZP_BN;
    const int kbeg = sp * kchunk, kend = min(K, kbeg + kchunk);
    const int lane = threadIdx.x & 63, gm = m0 + (int)(threadIdx.x >> 6) * 16 + (lane & 15);

    auto run = [&](auto tnc) {
        constexpr int TN = decltype(tnc)::value;
        typename Z::acc_t p1[TN], p2[TN], p3[TN];
#pragma unroll
        for (int t = 0; t < TN; ++t) p1[t] = p2[t] = p3[t] = typename Z::acc_t{0, 0, 0, 0};
        zp_tile<R, TA, TB, TN>(M, N, A, lda, B, ldb, m0, n0, kbeg, kend, s0, s1, s2, p1, p2, p3);
        if (gm >= M) return;
#pragma unroll
        for (int t = 0; t < TN; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int gn = n0 + t * 16 + Z::drow(lane, r);
                if (gn >= N) continue;
                const double q1 = p1[t][r], q2 = (TA == 2) != (TB == 2) ? -p2[t][r] : p2[t][r];
                const double xr = q1 - q2, xi = (double)p3[t][r] - (q1 + q2);
                c_t v;
                if (part) {
                    v.x = (R)xr;
                    v.y = (R)xi;
                    part[(size_t)sp * M * N + gm + (size_t)gn * M] = v;
                    continue;
                }
                double cr = ar * xr - ai * xi, ci = ar * xi + ai * xr;
                c_t* cp = C + gm + (size_t)gn * ldc;
                if (br != 0.0 || bi != 0.0) {
                    const c_t c = *cp;
                    cr += br * (double)c.x - bi * (double)c.y;
                    ci += br * (double)c.y + bi * (double)c.x;
                }
                v.x = (R)cr;
                v.y = (R)ci;
                *cp = v;
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
