// qt_gemm.hip -- batched complex128 GEMM on the gfx950 FP64 matrix cores.
//
// One workgroup computes a tile of C = alpha*op(A)op(B) + beta*D for one batch
// member: 32x32 or 64x64 with 4 waves, 128x64 with 4 or 8.  K is staged through
// LDS in double-buffered chunks.  Each wave owns 16x16 MFMA tiles; a complex product is
// four v_mfma_f64_16x16x4 (re*re, -im*im into Re; re*im, im*re into Im), or,
// in the three-multiplication form (G3, QT_PREC_FP64_3M), three:
//     P1 = Ar Br,  P2 = Ai Bi,  P3 = (Ar + Ai)(Br + Bi)  (sums rounded to FP64),
//     Re = P1 - P2,  Im = (P3 - P1) - P2  (in the epilogue),
// 3/4 of the matrix-core work, with the imaginary part's rounding error
// bounded by |Ar + Ai||Br + Bi| + |Ar||Br| + |Ai||Bi| instead of
// |Ar||Bi| + |Ai||Br| (Higham, Accuracy and Stability of Numerical
// Algorithms, 2nd ed., sec. 23.2.4).
//
// Operand order: the MFMA is fed (B-fragment, A-fragment), so that the
// 16x16 result lands transposed in the lanes.  v_mfma_f64_16x16x4f64 leaves
// element (r, c) of its product in lane c + 16*(r%4), register r/4 (measured
// on gfx950); with the swapped operands lane l, register q holds
// C[row = l%16][col = 4*q + l/16], so the 16 lanes of a quarter wave write
// 16 consecutive rows of one column (256 B, coalesced for column-major C).
//
// Work mapping: the 1-D grid is ordered so that all tiles of one batch
// member are dispatched to the same XCD (workgroups are dealt round-robin
// over the 8 XCDs), keeping that member's operands in one L2.
#include <cstdio>
#include <cstdlib>
#include <map>
#include <mutex>
#include <string>
#include <tuple>

#include "qt_internal.h"

namespace qt {

namespace {

constexpr int BM = 64;
constexpr int NXCD = 8;

typedef double double4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ double2 cconj(double2 v) { return make_double2(v.x, -v.y); }

// Wider variant: 128x64 block tile, K staged 8 at a time (2 x 24 KB LDS),
// each wave a 64x32 sub-tile (4x2 MFMA tiles): twice the MFMAs per LDS read
// of the 64x64 kernel and fewer global loads per flop.
constexpr int WBM = 128, WBN = 64, WBK = 8;

template <int OPA, int OPB, bool G3>
__global__ __launch_bounds__(256, 2) void zgemm_mfma_wide_kernel(ZGemmArgs a, int tiles_m, int tiles) {
    const int L = blockIdx.x;
    const int lane8 = L % NXCD;
    const int rest = L / NXCD;
    const int tile = rest % tiles;
    const int b = lane8 + NXCD * (rest / tiles);
    if (b >= a.batch) return;
    if (a.active && !a.active[b]) return;

    const int kz = a.kidx ? a.kidx[b >> a.kshift] : 0;
    const double2* __restrict__ Ap = a.A.p + b * a.A.sb + kz * a.A.sk;
    const double2* __restrict__ Bp = a.B.p + b * a.B.sb + kz * a.B.sk;
    const int64_t lda = a.A.ld, ldb = a.B.ld;
    const int M = a.M, N = a.N, K = a.K;
    const int m0 = (tile % tiles_m) * WBM;
    const int n0 = (tile / tiles_m) * WBN;

    // Every load pattern below has consecutive lanes either along the LDS row
    // (contiguous stores) or along k (8 lanes = the 8 rows of a stage).  The
    // rows are padded to 137 and 73 complex (row stride = 144 mod 256 bytes),
    // so 8 lanes writing 8 different rows hit 8 distinct 16-byte bank groups.
    __shared__ double2 As[2][WBK][WBM + 9];
    __shared__ double2 Bs[2][WBK][WBN + 9];

    const int tid = threadIdx.x;
    double2 ra[4], rb[2];

    auto loadA = [&](int k0) {
        if (OPA == OP_N) {
            // element e = tid + 256 q: rows contiguous across lanes
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int e = tid + 256 * q, kk = e >> 7, ii = e & 127;
                const int gi = m0 + ii, gk = k0 + kk;
                ra[q] = (gi < M && gk < K) ? Ap[gi + gk * lda] : make_double2(0.0, 0.0);
            }
        } else {
            // 8 lanes cover the 8 k of one row of op(A) (128 B contiguous)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int kk = tid & 7, ii = (tid >> 3) + 32 * q;
                const int gi = m0 + ii, gk = k0 + kk;
                ra[q] = (gi < M && gk < K) ? Ap[gk + gi * lda] : make_double2(0.0, 0.0);
            }
        }
    };
    auto storeA = [&](int buf) {
        if (OPA == OP_N) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int e = tid + 256 * q;
                As[buf][e >> 7][e & 127] = ra[q];
            }
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q)
                As[buf][tid & 7][(tid >> 3) + 32 * q] = OPA == OP_C ? cconj(ra[q]) : ra[q];
        }
    };
    auto loadB = [&](int k0) {
        if (OPB == OP_N) {
            // 8 lanes cover the 8 k of one column (128 B contiguous)
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int kk = tid & 7, jj = (tid >> 3) + 32 * q;
                const int gj = n0 + jj, gk = k0 + kk;
                rb[q] = (gj < N && gk < K) ? Bp[gk + gj * ldb] : make_double2(0.0, 0.0);
            }
        } else {
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int jj = tid & 63, kk = (tid >> 6) + 4 * q;
                const int gj = n0 + jj, gk = k0 + kk;
                rb[q] = (gj < N && gk < K) ? Bp[gj + gk * ldb] : make_double2(0.0, 0.0);
            }
        }
    };
    auto storeB = [&](int buf) {
        if (OPB == OP_N) {
#pragma unroll
            for (int q = 0; q < 2; ++q) Bs[buf][tid & 7][(tid >> 3) + 32 * q] = rb[q];
        } else {
#pragma unroll
            for (int q = 0; q < 2; ++q)
                Bs[buf][(tid >> 6) + 4 * q][tid & 63] = OPB == OP_C ? cconj(rb[q]) : rb[q];
        }
    };

    const int wave = tid >> 6, lane = tid & 63;
    const int wm = wave & 1, wn = wave >> 1;
    const int li = lane & 15, lk = lane >> 4;

    // G3: accR = P1, accI = P2, acc3 = P3
    double4_t accR[4][2], accI[4][2], acc3[G3 ? 4 : 1][G3 ? 2 : 1];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            accR[i][j] = double4_t{0.0, 0.0, 0.0, 0.0};
            accI[i][j] = double4_t{0.0, 0.0, 0.0, 0.0};
            if constexpr (G3) acc3[i][j] = double4_t{0.0, 0.0, 0.0, 0.0};
        }

    const int nk = (K + WBK - 1) / WBK;
    loadA(0);
    loadB(0);
    storeA(0);
    storeB(0);
    __syncthreads();

    for (int kt = 0; kt < nk; ++kt) {
        const int buf = kt & 1;
        if (kt + 1 < nk) {
            loadA((kt + 1) * WBK);
            loadB((kt + 1) * WBK);
        }
#pragma unroll
        for (int kq = 0; kq < WBK / 4; ++kq) {
            const int k = kq * 4 + lk;
            if constexpr (G3) {
                // one A fragment at a time keeps the registers within two
                // workgroups per CU
                double2 bv[2];
                double bs[2];
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    bv[j] = Bs[buf][k][wn * 32 + j * 16 + li];
                    bs[j] = bv[j].x + bv[j].y;
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const double2 av = As[buf][k][wm * 64 + i * 16 + li];
                    const double as = av.x + av.y;
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        accR[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(bv[j].x, av.x, accR[i][j], 0, 0, 0);
                        accI[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(bv[j].y, av.y, accI[i][j], 0, 0, 0);
                        acc3[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(bs[j], as, acc3[i][j], 0, 0, 0);
                    }
                }
            } else {
                double2 av[4], bv[2];
#pragma unroll
                for (int i = 0; i < 4; ++i) av[i] = As[buf][k][wm * 64 + i * 16 + li];
#pragma unroll
                for (int j = 0; j < 2; ++j) bv[j] = Bs[buf][k][wn * 32 + j * 16 + li];
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        accR[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(bv[j].x, av[i].x, accR[i][j], 0, 0, 0);
                        accI[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(bv[j].y, av[i].x, accI[i][j], 0, 0, 0);
                    }
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        accR[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(-bv[j].y, av[i].y, accR[i][j], 0, 0, 0);
                        accI[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(bv[j].x, av[i].y, accI[i][j], 0, 0, 0);
                    }
            }
        }
        if (kt + 1 < nk) {
            storeA(buf ^ 1);
            storeB(buf ^ 1);
        }
        __syncthreads();
    }

    double2* __restrict__ Cp = a.C + b * a.sbc + kz * a.skc;
    const double2* __restrict__ Dp = a.D.p ? a.D.p + b * a.D.sb + kz * a.D.sk : nullptr;
    const double alpha = a.alpha, beta = a.beta;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int gi = m0 + wm * 64 + i * 16 + li;
        if (gi >= M) continue;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int gj = n0 + wn * 32 + j * 16 + 4 * q + lk;
                if (gj >= N || (gj >= a.skip_lo && gj < a.skip_hi)) continue;
                double cr = accR[i][j][q], ci = accI[i][j][q];
                if constexpr (G3) {
                    const double p1 = accR[i][j][q], p2 = accI[i][j][q];
                    cr = p1 - p2;
                    ci = (acc3[i][j][q] - p1) - p2;
                }
                double re = alpha * cr, im = alpha * ci;
                if (Dp) {
                    const double2 d = Dp[gi + gj * a.D.ld];
                    re += beta * d.x;
                    im += beta * d.y;
                }
                Cp[gi + gj * a.ldc] = make_double2(re, im);
            }
        }
    }
}

// 128x64 tiles with 8 waves of 32x32 (2x2 MFMA tiles each): the 128x64
// kernel's LDS staging and global loads, the 64x64 tile's per-wave register
// tile, so the accumulators of the three-multiplication form fit beside
// more waves per CU.  Every output element sees the MFMAs of the other two
// kernels in the same order.
template <int OPA, int OPB, bool G3>
__global__ __launch_bounds__(512, G3 ? 1 : 2) void zgemm_mfma_w8_kernel(ZGemmArgs a, int tiles_m, int tiles) {
    const int L = blockIdx.x;
    const int lane8 = L % NXCD;
    const int rest = L / NXCD;
    const int tile = rest % tiles;
    const int b = lane8 + NXCD * (rest / tiles);
    if (b >= a.batch) return;
    if (a.active && !a.active[b]) return;

    const int kz = a.kidx ? a.kidx[b >> a.kshift] : 0;
    const double2* __restrict__ Ap = a.A.p + b * a.A.sb + kz * a.A.sk;
    const double2* __restrict__ Bp = a.B.p + b * a.B.sb + kz * a.B.sk;
    const int64_t lda = a.A.ld, ldb = a.B.ld;
    const int M = a.M, N = a.N, K = a.K;
    const int m0 = (tile % tiles_m) * WBM;
    const int n0 = (tile / tiles_m) * WBN;

    __shared__ double2 As[2][WBK][WBM + 9];
    __shared__ double2 Bs[2][WBK][WBN + 9];

    const int tid = threadIdx.x;
    double2 ra[2], rb;

    auto loadA = [&](int k0) {
        if (OPA == OP_N) {
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int e = tid + 512 * q, kk = e >> 7, ii = e & 127;
                const int gi = m0 + ii, gk = k0 + kk;
                ra[q] = (gi < M && gk < K) ? Ap[gi + gk * lda] : make_double2(0.0, 0.0);
            }
        } else {
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int kk = tid & 7, ii = (tid >> 3) + 64 * q;
                const int gi = m0 + ii, gk = k0 + kk;
                ra[q] = (gi < M && gk < K) ? Ap[gk + gi * lda] : make_double2(0.0, 0.0);
            }
        }
    };
    auto storeA = [&](int buf) {
        if (OPA == OP_N) {
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int e = tid + 512 * q;
                As[buf][e >> 7][e & 127] = ra[q];
            }
        } else {
#pragma unroll
            for (int q = 0; q < 2; ++q)
                As[buf][tid & 7][(tid >> 3) + 64 * q] = OPA == OP_C ? cconj(ra[q]) : ra[q];
        }
    };
    auto loadB = [&](int k0) {
        if (OPB == OP_N) {
            const int kk = tid & 7, jj = tid >> 3;
            const int gj = n0 + jj, gk = k0 + kk;
            rb = (gj < N && gk < K) ? Bp[gk + gj * ldb] : make_double2(0.0, 0.0);
        } else {
            const int jj = tid & 63, kk = tid >> 6;
            const int gj = n0 + jj, gk = k0 + kk;
            rb = (gj < N && gk < K) ? Bp[gj + gk * ldb] : make_double2(0.0, 0.0);
        }
    };
    auto storeB = [&](int buf) {
        if (OPB == OP_N)
            Bs[buf][tid & 7][tid >> 3] = rb;
        else
            Bs[buf][tid >> 6][tid & 63] = OPB == OP_C ? cconj(rb) : rb;
    };

    const int wave = tid >> 6, lane = tid & 63;
    const int wm = wave & 3, wn = wave >> 2;
    const int li = lane & 15, lk = lane >> 4;

    double4_t accR[2][2], accI[2][2], acc3[G3 ? 2 : 1][G3 ? 2 : 1];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            accR[i][j] = double4_t{0.0, 0.0, 0.0, 0.0};
            accI[i][j] = double4_t{0.0, 0.0, 0.0, 0.0};
            if constexpr (G3) acc3[i][j] = double4_t{0.0, 0.0, 0.0, 0.0};
        }

    const int nk = (K + WBK - 1) / WBK;
    loadA(0);
    loadB(0);
    storeA(0);
    storeB(0);
    __syncthreads();

    for (int kt = 0; kt < nk; ++kt) {
        const int buf = kt & 1;
        if (kt + 1 < nk) {
            loadA((kt + 1) * WBK);
            loadB((kt + 1) * WBK);
        }
#pragma unroll
        for (int kq = 0; kq < WBK / 4; ++kq) {
            const int k = kq * 4 + lk;
            double2 av[2], bv[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) av[i] = As[buf][k][wm * 32 + i * 16 + li];
#pragma unroll
            for (int j = 0; j < 2; ++j) bv[j] = Bs[buf][k][wn * 32 + j * 16 + li];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    if constexpr (G3) {
                        accR[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(bv[j].x, av[i].x, accR[i][j], 0, 0, 0);
                        accI[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(bv[j].y, av[i].y, accI[i][j], 0, 0, 0);
                        acc3[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(bv[j].x + bv[j].y, av[i].x + av[i].y,
                                                                         acc3[i][j], 0, 0, 0);
                    } else {
                        accR[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(bv[j].x, av[i].x, accR[i][j], 0, 0, 0);
                        accR[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(-bv[j].y, av[i].y, accR[i][j], 0, 0, 0);
                        accI[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(bv[j].y, av[i].x, accI[i][j], 0, 0, 0);
                        accI[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(bv[j].x, av[i].y, accI[i][j], 0, 0, 0);
                    }
                }
        }
        if (kt + 1 < nk) {
            storeA(buf ^ 1);
            storeB(buf ^ 1);
        }
        __syncthreads();
    }

    double2* __restrict__ Cp = a.C + b * a.sbc + kz * a.skc;
    const double2* __restrict__ Dp = a.D.p ? a.D.p + b * a.D.sb + kz * a.D.sk : nullptr;
    const double alpha = a.alpha, beta = a.beta;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int gi = m0 + wm * 32 + i * 16 + li;
        if (gi >= M) continue;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int gj = n0 + wn * 32 + j * 16 + 4 * q + lk;
                if (gj >= N || (gj >= a.skip_lo && gj < a.skip_hi)) continue;
                double cr = accR[i][j][q], ci = accI[i][j][q];
                if constexpr (G3) {
                    const double p1 = accR[i][j][q], p2 = accI[i][j][q];
                    cr = p1 - p2;
                    ci = (acc3[i][j][q] - p1) - p2;
                }
                double re = alpha * cr, im = alpha * ci;
                if (Dp) {
                    const double2 d = Dp[gi + gj * a.D.ld];
                    re += beta * d.x;
                    im += beta * d.y;
                }
                Cp[gi + gj * a.ldc] = make_double2(re, im);
            }
        }
    }
}

// 32x32 and 64x64 tiles: WGM x WGN waves of TM x TN MFMA tiles, K staged KB at a
// time in two LDS buffers with rows padded by one element (lanes along k then
// write distinct banks).  Every output element sees the MFMAs of the other
// kernels in the same order.
//
// 64x64 staged 8 deep: 33 KB of LDS and 125 registers, so four workgroups a CU
// where a 16-deep stage took two; 16 members of 695^3 0.785 -> 0.715 ms, 48 of
// 250^3 0.127 -> 0.115.  32x32 for blocks of a few hundred orbitals and less,
// where 64-row tiles leave the chip short of workgroups (64^3 x 256 members is one
// a CU, 192^3 x 60 is 540 for 512 places) or compute padding (160 = 2.5 x 64):
// 100 of 160^3 0.098 -> 0.068 ms, 60 of 192^3 0.095 -> 0.072, 16 of 128^3
// 0.027 -> 0.013, 256 of 96^3 0.057 (128x64) -> 0.041, 16 of 591x195x591 0.299
// (128x64) -> 0.191, one of 32^3 10.6 -> 6.5 us.  Half the operand reuse makes it
// L2 bound, the slower one, once both sides are above 384.  Staged 16 deep it
// is 1-5% faster where K is below a hundred (fewer barriers), 8 deep (17 KB, up
// to eight workgroups a CU) 3-5% above.
template <int OPA, int OPB, bool G3, int TM, int TN, int WGM, int WGN, int KB>
__global__ __launch_bounds__(WGM * WGN * 64)
    __attribute__((amdgpu_waves_per_eu(G3 ? (TM * TN == 4 ? 2 : 4) : 4))) void zgemm_mfma_small_kernel(ZGemmArgs a,
                                                                                                      int tiles_m,
                                                                                                      int tiles) {
    constexpr int SM = TM * WGM * 16, SN = TN * WGN * 16, NT = WGM * WGN * 64;
    constexpr int QA = SM * KB / NT, QB = SN * KB / NT;
    static_assert(SM * KB % NT == 0 && SN * KB % NT == 0, "whole loads");
    const int L = blockIdx.x;
    const int lane8 = L % NXCD;
    const int rest = L / NXCD;
    const int tile = rest % tiles;
    const int b = lane8 + NXCD * (rest / tiles);
    if (b >= a.batch) return;
    if (a.active && !a.active[b]) return;

    const int kz = a.kidx ? a.kidx[b >> a.kshift] : 0;
    const double2* __restrict__ Ap = a.A.p + b * a.A.sb + kz * a.A.sk;
    const double2* __restrict__ Bp = a.B.p + b * a.B.sb + kz * a.B.sk;
    const int64_t lda = a.A.ld, ldb = a.B.ld;
    const int M = a.M, N = a.N, K = a.K;
    const int m0 = (tile % tiles_m) * SM;
    const int n0 = (tile / tiles_m) * SN;

    __shared__ double2 As[2][KB][SM + 1];
    __shared__ double2 Bs[2][KB][SN + 1];

    const int tid = threadIdx.x;
    double2 ra[QA], rb[QB];
    // element e = tid + NT q of a stage: along the memory's contiguous axis
    auto loadA = [&](int k0) {
#pragma unroll
        for (int q = 0; q < QA; ++q) {
            const int e = tid + NT * q;
            const int ii = OPA == OP_N ? e % SM : e / KB, kk = OPA == OP_N ? e / SM : e % KB;
            const int gi = m0 + ii, gk = k0 + kk;
            ra[q] = (gi < M && gk < K) ? (OPA == OP_N ? Ap[gi + gk * lda] : Ap[gk + gi * lda])
                                       : make_double2(0.0, 0.0);
        }
    };
    auto loadB = [&](int k0) {
#pragma unroll
        for (int q = 0; q < QB; ++q) {
            const int e = tid + NT * q;
            const int jj = OPB == OP_N ? e / KB : e % SN, kk = OPB == OP_N ? e % KB : e / SN;
            const int gj = n0 + jj, gk = k0 + kk;
            rb[q] = (gj < N && gk < K) ? (OPB == OP_N ? Bp[gk + gj * ldb] : Bp[gj + gk * ldb])
                                       : make_double2(0.0, 0.0);
        }
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int q = 0; q < QA; ++q) {
            const int e = tid + NT * q;
            const int ii = OPA == OP_N ? e % SM : e / KB, kk = OPA == OP_N ? e / SM : e % KB;
            As[buf][kk][ii] = OPA == OP_C ? cconj(ra[q]) : ra[q];
        }
#pragma unroll
        for (int q = 0; q < QB; ++q) {
            const int e = tid + NT * q;
            const int jj = OPB == OP_N ? e / KB : e % SN, kk = OPB == OP_N ? e % KB : e / SN;
            Bs[buf][kk][jj] = OPB == OP_C ? cconj(rb[q]) : rb[q];
        }
    };

    const int wave = tid >> 6, lane = tid & 63;
    const int wm = wave % WGM, wn = wave / WGM;
    const int li = lane & 15, lk = lane >> 4;

    double4_t accR[TM][TN], accI[TM][TN], acc3[G3 ? TM : 1][G3 ? TN : 1];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            accR[i][j] = double4_t{0.0, 0.0, 0.0, 0.0};
            accI[i][j] = double4_t{0.0, 0.0, 0.0, 0.0};
            if constexpr (G3) acc3[i][j] = double4_t{0.0, 0.0, 0.0, 0.0};
        }

    const int nk = (K + KB - 1) / KB;
    loadA(0);
    loadB(0);
    store(0);
    __syncthreads();
    for (int kt = 0; kt < nk; ++kt) {
        const int buf = kt & 1;
        if (kt + 1 < nk) {
            loadA((kt + 1) * KB);
            loadB((kt + 1) * KB);
        }
#pragma unroll
        for (int kq = 0; kq < KB / 4; ++kq) {
            const int k = kq * 4 + lk;
            double2 av[TM], bv[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i) av[i] = As[buf][k][(wm * TM + i) * 16 + li];
#pragma unroll
            for (int j = 0; j < TN; ++j) bv[j] = Bs[buf][k][(wn * TN + j) * 16 + li];
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    accR[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(bv[j].x, av[i].x, accR[i][j], 0, 0, 0);
                    if constexpr (G3) {
                        accI[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(bv[j].y, av[i].y, accI[i][j], 0, 0, 0);
                        acc3[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(bv[j].x + bv[j].y, av[i].x + av[i].y,
                                                                         acc3[i][j], 0, 0, 0);
                    } else {
                        accI[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(bv[j].y, av[i].x, accI[i][j], 0, 0, 0);
                        accR[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(-bv[j].y, av[i].y, accR[i][j], 0, 0, 0);
                        accI[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(bv[j].x, av[i].y, accI[i][j], 0, 0, 0);
                    }
                }
        }
        if (kt + 1 < nk) store(buf ^ 1);
        __syncthreads();
    }

    double2* __restrict__ Cp = a.C + b * a.sbc + kz * a.skc;
    const double2* __restrict__ Dp = a.D.p ? a.D.p + b * a.D.sb + kz * a.D.sk : nullptr;
    const double alpha = a.alpha, beta = a.beta;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int gi = m0 + (wm * TM + i) * 16 + li;
        if (gi >= M) continue;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int gj = n0 + (wn * TN + j) * 16 + 4 * q + lk;
                if (gj >= N || (gj >= a.skip_lo && gj < a.skip_hi)) continue;
                double cr = accR[i][j][q], ci = accI[i][j][q];
                if constexpr (G3) {
                    const double p1 = accR[i][j][q], p2 = accI[i][j][q];
                    cr = p1 - p2;
                    ci = (acc3[i][j][q] - p1) - p2;
                }
                double re = alpha * cr, im = alpha * ci;
                if (Dp) {
                    const double2 d = Dp[gi + gj * a.D.ld];
                    re += beta * d.x;
                    im += beta * d.y;
                }
                Cp[gi + gj * a.ldc] = make_double2(re, im);
            }
        }
    }
}

template <int OPA, int OPB, bool G3, int TM, int TN, int WGM, int WGN, int KB>
void launch_small(hipStream_t s, const ZGemmArgs& a) {
    constexpr int SM = TM * WGM * 16, SN = TN * WGN * 16;
    const int tiles_m = (a.M + SM - 1) / SM;
    const int tiles = tiles_m * ((a.N + SN - 1) / SN);
    const int64_t blocks = (int64_t)tiles * ((a.batch + NXCD - 1) / NXCD * NXCD);
    if (blocks > 0x7fffffff) throw hip_error("zgemm: grid too large", 1);
    hipLaunchKernelGGL((zgemm_mfma_small_kernel<OPA, OPB, G3, TM, TN, WGM, WGN, KB>), dim3((unsigned)blocks),
                       dim3(WGM * WGN * 64), 0, s, a, tiles_m, tiles);
    QT_HIP(hipGetLastError());
}

template <int OPA, int OPB, bool G3>
void launch_w8(hipStream_t s, const ZGemmArgs& a) {
    const int tiles_m = (a.M + WBM - 1) / WBM;
    const int tiles_n = (a.N + WBN - 1) / WBN;
    const int tiles = tiles_m * tiles_n;
    const int batch_pad = (a.batch + NXCD - 1) / NXCD * NXCD;
    const int64_t blocks = (int64_t)tiles * batch_pad;
    if (blocks > 0x7fffffff) throw hip_error("zgemm: grid too large", 1);
    hipLaunchKernelGGL((zgemm_mfma_w8_kernel<OPA, OPB, G3>), dim3((unsigned)blocks), dim3(512), 0, s, a, tiles_m,
                       tiles);
    QT_HIP(hipGetLastError());
}

template <int OPA, int OPB, bool G3>
void launch_wide(hipStream_t s, const ZGemmArgs& a) {
    const int tiles_m = (a.M + WBM - 1) / WBM;
    const int tiles_n = (a.N + WBN - 1) / WBN;
    const int tiles = tiles_m * tiles_n;
    const int batch_pad = (a.batch + NXCD - 1) / NXCD * NXCD;
    const int64_t blocks = (int64_t)tiles * batch_pad;
    if (blocks > 0x7fffffff) throw hip_error("zgemm: grid too large", 1);
    hipLaunchKernelGGL((zgemm_mfma_wide_kernel<OPA, OPB, G3>), dim3((unsigned)blocks), dim3(256), 0, s, a,
                       tiles_m, tiles);
    QT_HIP(hipGetLastError());
}

// Tile choice.  QT_GEMM_TILE=64x64, 128x64, 128x64w8, 32x32 or 32x32k8 fixes the
// kernel; otherwise the autotuner below picks per shape (QT_GEMM_TUNE=0: the
// row-waste rule of use_wide alone).  All kernels accumulate every
// output element in the same order (k ascending in groups of 4, the same
// MFMAs per group and component, the same epilogue), so the choice never
// changes a result.
enum { TILE_AUTO = 0, TILE_NARROW = 1, TILE_WIDE = 2, TILE_W8 = 3, TILE_32X32 = 4, TILE_32K8 = 5, NTILE = 5 };
const char* tile_name(int t) {
    static const char* const n[] = {"auto", "64x64", "128x64", "128x64w8", "32x32", "32x32k8"};
    return n[t];
}
int tile_forced() {
    static const int v = [] {
        const char* e = getenv("QT_GEMM_TILE");
        for (int t = 1; e && t <= NTILE; ++t)
            if (std::string(e) == tile_name(t)) return t;
        return (int)TILE_AUTO;
    }();
    return v;
}
bool tune_enabled() {
    static const bool v = [] {
        const char* e = getenv("QT_GEMM_TUNE");
        return !(e && std::string(e) == "0");
    }();
    return v;
}
bool tune_log() {
    static const bool v = getenv("QT_GEMM_TUNE_LOG") != nullptr;
    return v;
}

// 128-row tiles unless they leave more rows idle than 64-row tiles do
// (M = 192, 320, 448, ...: the half-empty last tile costs more than the
// 64x64 kernel's lower peak)
bool use_wide(int M) {
    const int waste_wide = (M + WBM - 1) / WBM * WBM - M;
    const int waste_narrow = (M + BM - 1) / BM * BM - M;
    return M >= WBM && waste_wide <= waste_narrow;
}

// Autotuner: the first product of each shape (op pair, M, N, K, batch) runs
// the kernels in question twice into a scratch output (the operands and the addend are
// only read; at most 512 MiB of scratch, fewer members where the full batch
// needs more) after the work already queued on the stream, and the faster
// kernel is kept for the shape for the life of the process.  Where the
// scratch cannot be allocated the row-waste rule decides; it knows 64- and
// 128-row tiles only, so that 32x32 ones run where they were timed.
struct TuneState {
    std::mutex mu;
    std::map<std::tuple<int, int, int, int, int>, int> tile;
};
TuneState& tune_state() {
    static TuneState t;
    return t;
}

template <int OPA, int OPB, bool G3>
void launch_tile(hipStream_t s, const ZGemmArgs& a, int tile) {
    if (tile == TILE_32X32)
        launch_small<OPA, OPB, G3, 1, 1, 2, 2, 16>(s, a);
    else if (tile == TILE_32K8)
        launch_small<OPA, OPB, G3, 1, 1, 2, 2, 8>(s, a);
    else if (tile == TILE_W8)
        launch_w8<OPA, OPB, G3>(s, a);
    else if (tile == TILE_WIDE)
        launch_wide<OPA, OPB, G3>(s, a);
    else
        launch_small<OPA, OPB, G3, 2, 2, 2, 2, 8>(s, a);
}

// the kernels worth timing for an M x N output: 32x32 tiles where one side is up
// to 384 (above, 64-row tiles fill the chip and need half the operand traffic),
// 128-row ones where more than half of such a tile is used
bool in_question(int tile, int M, int N) {
    switch (tile) {
        case TILE_WIDE: case TILE_W8: return M > 64;
        case TILE_32X32: case TILE_32K8: return std::min(M, N) <= 384;
        default: return true;
    }
}

template <int OPA, int OPB, bool G3>
int tuned_tile(hipStream_t s, const ZGemmArgs& a) {
    const auto key = std::make_tuple((OPA * 3 + OPB) * 2 + (G3 ? 1 : 0), a.M, a.N, a.K, a.batch);
    TuneState& ts = tune_state();
    {
        std::lock_guard<std::mutex> lk(ts.mu);
        auto it = ts.tile.find(key);
        if (it != ts.tile.end()) return it->second;
    }
    const size_t per = sizeof(double2) * (size_t)a.M * (size_t)a.N;
    const size_t cap = (size_t)512 << 20;
    const int members = (int)std::max<size_t>(1, std::min<size_t>((size_t)a.batch, cap / std::max<size_t>(per, 1)));
    ZGemmArgs t = a;
    t.batch = members;
    t.ldc = a.M;
    t.sbc = (int64_t)a.M * a.N;
    t.skc = 0;
    t.skip_lo = t.skip_hi = 0;
    void* scratch = nullptr;
    hipEvent_t ev[3];
    float ms[NTILE + 1];
    for (float& m : ms) m = 1e30f;
    if (hipMalloc(&scratch, per * (size_t)members) != hipSuccess) {
        (void)hipGetLastError();  // no room for the scratch output: the row-waste rule, kept
        const int tile = use_wide(a.M) ? TILE_WIDE : TILE_NARROW;
        std::lock_guard<std::mutex> lk(ts.mu);
        ts.tile[key] = tile;
        return tile;
    }
    for (auto& e : ev) QT_HIP(hipEventCreate(&e));
    t.C = (double2*)scratch;
    for (int rep = 0; rep < 2; ++rep)
        for (int v = 1; v <= NTILE; ++v) {
            if (!in_question(v, a.M, a.N)) continue;
            QT_HIP(hipEventRecord(ev[0], s));
            launch_tile<OPA, OPB, G3>(s, t, v);
            QT_HIP(hipEventRecord(ev[1], s));
            QT_HIP(hipEventSynchronize(ev[1]));
            float m = 0.0f;
            QT_HIP(hipEventElapsedTime(&m, ev[0], ev[1]));
            ms[v] = std::min(ms[v], m);
        }
    for (auto& e : ev) QT_HIP(hipEventDestroy(e));
    QT_HIP(hipFree(scratch));
    int tile = TILE_NARROW;
    for (int v = 1; v <= NTILE; ++v)
        if (ms[v] < ms[tile]) tile = v;
    if (tune_log()) {
        fprintf(stderr, "qt gemm tune: ops %d%s M %d N %d K %d batch %d (%d timed):", OPA * 3 + OPB, G3 ? " (3m)" : "",
                a.M, a.N, a.K, a.batch, members);
        for (int v = 1; v <= NTILE; ++v)
            if (ms[v] < 1e30f) fprintf(stderr, " %s %.4f ms", tile_name(v), ms[v]);
        fprintf(stderr, " -> %s\n", tile_name(tile));
    }
    std::lock_guard<std::mutex> lk(ts.mu);
    ts.tile[key] = tile;
    return tile;
}

template <int OPA, int OPB, bool G3>
void launch_g(hipStream_t s, const ZGemmArgs& a) {
    const int forced = tile_forced();
    int tile;
    if (forced != TILE_AUTO)
        tile = forced;
    else if (tune_enabled())
        tile = tuned_tile<OPA, OPB, G3>(s, a);
    else
        tile = use_wide(a.M) ? TILE_WIDE : TILE_NARROW;
    launch_tile<OPA, OPB, G3>(s, a, tile);
}

template <int OPA, int OPB>
void launch(hipStream_t s, const ZGemmArgs& a) {
    if (a.prec == 3)
        launch_g<OPA, OPB, true>(s, a);
    else
        launch_g<OPA, OPB, false>(s, a);
}

}  // namespace

void zgemm(hipStream_t s, int opa, int opb, const ZGemmArgs& a, Timer* t) {
    if (a.M <= 0 || a.N <= 0 || a.batch <= 0) return;
    if (t && t->enabled) t->begin(s, 0);
    const int key = opa * 3 + opb;
    if ((a.prec == 6 || a.prec == 7) && zgemm_i8_fits(a)) {
        zgemm_i8(s, opa, opb, a, a.prec);
        if (t && t->enabled)
            t->end(s, 0, 8.0 * a.M * a.N * (double)a.K * (a.flop_batch >= 0 ? a.flop_batch : a.batch));
        return;
    }
    switch (key) {
        case 0: launch<OP_N, OP_N>(s, a); break;
        case 2: launch<OP_N, OP_C>(s, a); break;
        case 6: launch<OP_C, OP_N>(s, a); break;
        case 8: launch<OP_C, OP_C>(s, a); break;
        case 1: launch<OP_N, OP_T>(s, a); break;
        case 3: launch<OP_T, OP_N>(s, a); break;
        default: throw hip_error("zgemm: unsupported op pair", 6);
    }
    if (t && t->enabled)
        t->end(s, 0, 8.0 * a.M * a.N * (double)a.K * (a.flop_batch >= 0 ? a.flop_batch : a.batch));
}

}  // namespace qt
