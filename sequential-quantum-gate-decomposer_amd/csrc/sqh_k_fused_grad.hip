// sqh_k_fused_grad.hip -- batched cost and gradient of the circuit as fused dense
// 4-qubit blocks on the matrix cores, every column resident on the chip.
//
// Forward: as the fused cost kernel (sqh_k_fused_cost.hip), X_b = F_b X_{b-1} from the
// target, and the trace entries.  Backward, with Y the trace selector propagated
// through the blocks (Y_{b-1} = F_b^T Y_b, so Tr = sum Y_b * X_b for every b), per block
// from the last:
//   X_{b-1} = F_b^dagger X_b                                   (MFMA, F unitary)
//   M_b[i][k] += sum over the wavefront's (outer group, column) of Y_b[(i,o)] X_{b-1}[(k,o)]
//                                                              (MFMA on transposed tiles)
//   Y_{b-1} = F_b^T Y_b                                        (MFMA)
// so that dTr/dtheta = sum_ik (dF_b/dtheta)_ik M_b[i][k] for a parameter of block b.
// A wavefront sums its M_b over its column groups in registers and its own partial slot, so
// no wavefront waits for another; k_fused_block_corr then sums the partials and runs the
// block's gates backwards, producing each gate's 2x2 correlations in the layout of the
// register-tile adjoint kernel, from which k_finish forms the gradient.
//
// Layouts follow sqh_k_fused_cost.hip: row j of a column under block b is
// base_b[o] + off_b[i]; 16x16x4 MFMA operands A[l % 16][l / 16], B[l / 16][l % 16]; the
// B operand of step s holds rows 4 s + lane / 16, the D layout rows row(r, lane / 16).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "sqh_device.h"
#include "sqh_fused_chain.h"
#include "sqh_kernels.h"

namespace sqh {

namespace {

// Entry (r, c) of a 16 x 16 tile in LDS, columns rotated by the row (XOR) so that both a
// row-wise and a column-wise sweep of 16 lanes touch 16 different bank groups.
__device__ __forceinline__ int fg_tile(int r, int c) { return r * 16 + (c ^ r); }

// Y = A X (CONJ: with A's conjugate) on all tiles.
template <typename R, int T, bool CONJ>
__device__ __forceinline__ void fg_mma(const FcA<R>& A, const R (&xr)[T][4], const R (&xi)[T][4],
                                       typename FcMfma<R>::V (&yr)[T], typename FcMfma<R>::V (&yi)[T]) {
    typedef FcMfma<R> MF;
    if constexpr (!CONJ) {
        fc_mma<R, T, T>(A, xr, xi, yr, yi);
    } else {
#pragma unroll
        for (int t = 0; t < T; ++t) yr[t] = yi[t] = typename MF::V{0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < 4; ++s) {
#pragma unroll
            for (int t = 0; t < T; ++t) {
                yr[t] = MF::op(A.re[s], xr[t][s], yr[t]);
                yi[t] = MF::op(A.re[s], xi[t][s], yi[t]);
            }
#pragma unroll
            for (int t = 0; t < T; ++t) {
                yr[t] = MF::op(A.im[s], xi[t][s], yr[t]);
                yi[t] = MF::op_neg(A.im[s], xr[t][s], yi[t]);
            }
        }
    }
}

// What a wavefront of the gradient kernels works on: element e and the column groups
// first .. last - 1 of it, whose correlations it sums in partial slot `slot`.
struct FgTask {
    int e, slot, first, last;
    bool live;
};
__device__ __forceinline__ FgTask fg_task(const FusedGradArgs& a, int wv) {
    // XCD-ordered workgroups (the grid is a multiple of 8); with a live count (the
    // optimiser's rounds) the plain order, so the live elements spread over the XCDs
    int B = a.B;
    long long lwg = blockIdx.x;
    if (a.count) B = min(*a.count, a.B);
    else lwg = (long long)(blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    const long long task = lwg * (blockDim.x >> 6) + wv;
    FgTask t;
    t.e = (int)(task / a.wgs);
    t.slot = (int)(task % a.wgs);
    t.first = t.slot * a.per;
    t.last = min(t.first + a.per, a.groups);
    t.live = t.e < B;
    return t;
}

// X = the target's columns c0 + w in a block's full layout (tab), zero past column m.
template <typename R, int N, int T>
__device__ __forceinline__ void fg_load_target(const cpx<R>* __restrict__ U, const int* tab, int c0, int m, int lane,
                                               R (&xr)[T][4], R (&xi)[T][4]) {
    constexpr int O = (1 << N) >> 4;
    const unsigned row0 = (unsigned)tab[LT_ROW + lane] * (unsigned)m;
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const int col = c0 + (O > 16 ? t / (O / 16 ? O / 16 : 1) : (16 * t + (lane & 15)) / O);
        const unsigned at = row0 + (unsigned)tab[LT_RT + t] * (unsigned)m + (unsigned)(col < m ? col : 0);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const cpx<R> v = U[at + (unsigned)tab[LT_RS + s] * (unsigned)m];
            xr[t][s] = col < m ? v.re : (R)0;
            xi[t][s] = col < m ? v.im : (R)0;
        }
    }
}

// M += Y X^T over the wavefront's vector columns (Y and X: item i of tile t is row 4 i +
// lane / 16 of its vector columns), tile by tile through the region as two transposed
// tiles, added to the wavefront's own partial of the block at M: [256] real, then [256]
// imaginary parts.  The partial stays in the caches between the column groups, and no
// wavefront waits for another: summing four wavefronts' correlations in LDS behind two
// barriers per block kept them in step, all in their exchanges while the matrix cores idled.
template <typename R, int T, typename Y>
__device__ __forceinline__ void fg_correlate(R* lds, const Y& yr, const Y& yi, const R (&xr)[T][4],
                                             const R (&xi)[T][4], double* __restrict__ M, bool first, int lane) {
    typedef FcMfma<R> MF;
    const int nl = lane & 15, g = lane >> 4;
    constexpr bool D64 = sizeof(R) == 8;
    typename MF::V mr, mi;
    double pr[4], pi[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int idx = MF::row(r, g) * 16 + nl;
        pr[r] = first ? 0.0 : M[idx];
        pi[r] = first ? 0.0 : M[256 + idx];
        mr[r] = D64 ? (R)pr[r] : (R)0;
        mi[r] = D64 ? (R)pi[r] : (R)0;
    }
#pragma unroll
    for (int t = 0; t < T; ++t) {
        R* yb = lds + (T >= 4 && (t & 1) ? 1024 : 0);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int at = fg_tile(4 * s + g, nl);
            yb[at] = yr[t][s];
            yb[256 + at] = yi[t][s];
            yb[512 + at] = xr[t][s];
            yb[768 + at] = xi[t][s];
        }
        fc_wave_fence();
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int at = fg_tile(nl, 4 * s + g);
            const R yvr = yb[at], yvi = yb[256 + at], xvr = yb[512 + at], xvi = yb[768 + at];
            mr = MF::op(yvr, xvr, mr);
            mi = MF::op(yvr, xvi, mi);
            mr = MF::op_neg(yvi, xvi, mr);
            mi = MF::op(yvi, xvr, mi);
        }
        fc_wave_fence();
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int idx = MF::row(r, g) * 16 + nl;
        M[idx] = D64 ? (double)mr[r] : pr[r] + (double)mr[r];
        M[256 + idx] = D64 ? (double)mi[r] : pi[r] + (double)mi[r];
    }
}

}  // namespace

template <typename R, int N, int T>
__global__ __launch_bounds__(512, 2) void k_fused_grad(FusedGradArgs a, const int* __restrict__ tabs) {
    typedef FcMfma<R> MF;
    typedef FcRegion<R, N, T> Reg;
    constexpr int O = Reg::O, W = Reg::W;
    static_assert(W >= 1, "a wavefront holds whole columns");
    extern __shared__ __align__(16) unsigned char fg_smem[];
    int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const FgTask task = fg_task(a, wv);
    if (!task.live) return;
    const int e = task.e, m = a.m;
    const Reg lds{reinterpret_cast<R*>(fg_smem) + wv * 512 * T};
    const cpx<R>* U = static_cast<const cpx<R>*>(a.U);
    if (a.count) U += (long long)a.run_target[a.elem_run[e]] * a.tgt_stride;
    const cpx<R>* Fe = static_cast<const cpx<R>*>(a.F) + (long long)e * a.nb * 256;
    double* const part = a.mpart + ((long long)e * a.wgs + task.slot) * a.nb * 512;
    for (int cg = task.first; cg < task.last; ++cg) {
        const int c0 = cg * W;
        const int nl = lane & 15, g = lane >> 4;
        R xr[T][4], xi[T][4], yr[T][4], yi[T][4];
        FcA<R> A;
        typename MF::V dr[T], di[T];
        fg_load_target<R, N, T>(U, tabs, c0, m, lane, xr, xi);
        // forward; after the last block X stays in its own grouping
        for (int b = 0; b < a.nb; ++b) {
            const int* tab = tabs + b * kLaneTab;
            A.load_n(Fe + (long long)b * 256, nl, g);
            fg_mma<R, T, false>(A, xr, xi, dr, di);
            if (b + 1 < a.nb) {
                int at[4];
                Reg::full_at(at, tab, tab[LT_LANE + lane]);
                lds.template store_full<T>(at, tab, dr, di);
                const int* tn = tab + kLaneTab;
                Reg::full_at(at, tn, tn[LT_LANE + lane]);
                lds.load_full(at, tn, xr, xi);
            }
        }
        // trace entries from X and the selector Y (1 at row c + trace_off of column c)
        {
            const int* tab = tabs + (a.nb - 1) * kLaneTab;
#pragma unroll
            for (int t = 0; t < T; ++t) {
                const int col = c0 + (16 * t + nl) / O;
                const int row = tab[LT_ROW + lane] | tab[LT_RT + t];
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    xr[t][s] = dr[t][s];
                    xi[t][s] = di[t][s];
                    const bool hit = col < m && (row | tab[LT_RS + s]) == col + a.trace_off;
                    if (hit) {
                        double* d = a.diag + 2 * ((long long)e * m + col);
                        d[0] = (double)xr[t][s];
                        d[1] = (double)xi[t][s];
                    }
                    yr[t][s] = hit ? (R)1 : (R)0;
                    yi[t][s] = (R)0;
                }
            }
        }
        // backward: X_{b-1} = F^dagger X_b, M_b += Y_b X_{b-1}^T, Y_{b-1} = F^T Y_b
        for (int b = a.nb - 1; b >= 0; --b) {
            const int* tab = tabs + b * kLaneTab;
            A.load_t(Fe + (long long)b * 256, nl, g);
            fg_mma<R, T, true>(A, xr, xi, dr, di);
#pragma unroll
            for (int t = 0; t < T; ++t)
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    xr[t][s] = dr[t][s];
                    xi[t][s] = di[t][s];
                }
            fg_correlate<R, T>(lds.p, yr, yi, xr, xi, part + b * 512, cg == task.first, lane);
            if (b == 0) break;
            fg_mma<R, T, false>(A, yr, yi, dr, di);
            const int* tn = tab - kLaneTab;
            int at[4], an[4];
            Reg::full_at(at, tab, tab[LT_LANE + lane]);
            Reg::full_at(an, tn, tn[LT_LANE + lane]);
            lds.template store_full<T>(at, tab, dr, di);
            lds.load_full(an, tn, yr, yi);
#pragma unroll
            for (int t = 0; t < T; ++t)
#pragma unroll
                for (int s = 0; s < 4; ++s) lds.put(Reg::full(at, tab, t, s), xr[t][s], xi[t][s]);
            fc_wave_fence();
            lds.load_full(an, tn, xr, xi);
        }
    }
}

// Cost + gradient with the adjoint vectors from the transposed chain (sqh_fused_chain.h).
// In the notation above, the adjoint after block b is Z_{b+1} = F_{b+1}^T ... F_{nb-1}^T
// e_rho (Z_nb = e_rho): exactly the chain's vectors, which touch only the rows inside the
// support of the blocks seen so far.  Phase 1 runs the chain down to Z_1 (block 0's
// operand), then Z_0 = F_0^T Z_1 gives the trace entries (dotted with the target's
// columns).  Phase 2 sweeps up: X_{-1} = the target's columns,
//   M_b += Z_{b+1} X_{b-1}^T,   X_b = F_b X_{b-1},   Z_{b+2} = conj(F_{b+1}) Z_{b+1}
// (F unitary: (F^T)^-1 = conj(F)), Z_nb set to the selector itself.  Block products:
// the chain's, then 3 nb - 3 (the 8-qubit 40-layer ansatz: 4 + 15 = 19 against the
// backward sweep's 23).  The correlations M_b and their partials are those of
// k_fused_grad.  Needs nb >= 2 and block 0's support to cover every qubit (the chain
// then ends in the forward layout).
template <typename R, int N, int T>
__global__ __launch_bounds__(512, 2) void k_fused_grad_chain(FusedGradArgs a, const int* __restrict__ tabs,
                                                             const int* __restrict__ tmaps) {
    typedef FcMfma<R> MF;
    typedef FcRegion<R, N, T> Reg;
    constexpr int O = Reg::O, W = Reg::W;
    static_assert(W >= 1, "a wavefront holds whole columns");
    extern __shared__ __align__(16) unsigned char fg_smem[];
    int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const FgTask task = fg_task(a, wv);
    if (!task.live) return;
    const int e = task.e, m = a.m;
    const Reg lds{reinterpret_cast<R*>(fg_smem) + wv * 512 * T};
    const cpx<R>* U = static_cast<const cpx<R>*>(a.U);
    if (a.count) U += (long long)a.run_target[a.elem_run[e]] * a.tgt_stride;
    const cpx<R>* Fe = static_cast<const cpx<R>*>(a.F) + (long long)e * a.nb * 256;
    double* const part = a.mpart + ((long long)e * a.wgs + task.slot) * a.nb * 512;
    for (int cg = task.first; cg < task.last; ++cg) {
        const int c0 = cg * W;
        const bool first = cg == task.first;
        asm volatile("" : "+v"(lane));  // no lane's addresses kept in registers from group to group
        const int nl = lane & 15, g = lane >> 4;
        // phase 1: Z_1 in block 0's grouping, X = the target's columns there, and the trace
        // entries from Z_0 = F_0^T Z_1
        R zr[T][4], zi[T][4], xr[T][4], xi[T][4];
        typename MF::V er[T], ei[T];
        FcA<R> A;
        fused_chain_to_block0<R, N, T, false>(tabs, tmaps, a.nb, lds, Fe, c0, m, a.trace_off, lane, zr, zi, A);
        fg_mma<R, T, false>(A, zr, zi, er, ei);
        {
            constexpr int C = O > 16 ? W : T;  // sums: per column, or per tile of whole columns
            double sr[C], si[C];
#pragma unroll
            for (int c = 0; c < C; ++c) sr[c] = si[c] = 0;
            const unsigned row0 = (unsigned)tabs[LT_ROW + lane] * (unsigned)m;
#pragma unroll
            for (int t = 0; t < T; ++t) {
                const int c = O > 16 ? t / (O / 16 ? O / 16 : 1) : t;
                const int col = c0 + (16 * t + nl) / O;
                const unsigned at = row0 + (unsigned)tabs[LT_RT + t] * (unsigned)m + (unsigned)(col < m ? col : 0);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const cpx<R> u = U[at + (unsigned)tabs[LT_RS + r] * (unsigned)m];
                    sr[c] += (double)er[t][r] * (double)u.re - (double)ei[t][r] * (double)u.im;
                    si[c] += (double)er[t][r] * (double)u.im + (double)ei[t][r] * (double)u.re;
                }
            }
            fc_column_sums<N, T>(sr, si, a.diag + 2 * ((long long)e * m + c0), c0, m, lane);
        }
        fg_load_target<R, N, T>(U, tabs, c0, m, lane, xr, xi);
        fg_correlate<R, T>(lds.p, zr, zi, xr, xi, part, first, lane);
        // phase 2, one step up: X_b into block b + 1's grouping, Z_{b+2} (block b + 1's
        // grouping, as a result) from Z_{b+1} -- block 0's operand for the first step, the
        // last step's result after it -- then M_{b+1}.  The first step runs on its own, so
        // that its operand is not live through the loop.
        auto step = [&](int b, auto first_step) __attribute__((always_inline)) {
            constexpr bool ZB = decltype(first_step)::value;
            const int* tab = tabs + b * kLaneTab;
            const int* tn = tab + kLaneTab;
            int at[4], an[4];
            Reg::full_at(at, tab, tab[LT_LANE + lane]);
            Reg::full_at(an, tn, tn[LT_LANE + lane]);
            {
                FcA<R> An;
                An.load_n(Fe + (long long)b * 256, nl, g);
                typename MF::V dr[T], di[T];
                fg_mma<R, T, false>(An, xr, xi, dr, di);
                lds.template store_full<T>(at, tab, dr, di);
                lds.load_full(an, tn, xr, xi);
            }
            if (b + 2 < a.nb) {
                if constexpr (ZB) {
#pragma unroll
                    for (int t = 0; t < T; ++t)
#pragma unroll
                        for (int s = 0; s < 4; ++s) lds.put(Reg::full(at, tab, t, s), zr[t][s], zi[t][s]);
                    fc_wave_fence();
                } else {
                    lds.template store_full<T>(at, tab, er, ei);
                }
                R vr[T][4], vi[T][4];
                lds.load_full(an, tn, vr, vi);
                FcA<R> An;
                An.load_n(Fe + (long long)(b + 1) * 256, nl, g);
                fg_mma<R, T, true>(An, vr, vi, er, ei);
            } else {
                // Z_nb: the selector, row rho = c + trace_off of column c
#pragma unroll
                for (int t = 0; t < T; ++t) {
                    const int col = c0 + (16 * t + nl) / O;
                    const int row = tn[LT_ROW + lane] | tn[LT_RT + t];
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        er[t][r] = (col < m && (row | tn[LT_RS + r]) == col + a.trace_off) ? (R)1 : (R)0;
                        ei[t][r] = (R)0;
                    }
                }
            }
            fg_correlate<R, T>(lds.p, er, ei, xr, xi, part + (b + 1) * 512, first, lane);
        };
        step(0, std::true_type{});
        for (int b = 1; b + 1 < a.nb; ++b) step(b, std::false_type{});
    }
}

size_t fused_grad_lds_bytes(bool f32, int nb, int T, int waves) {
    (void)nb;
    return (f32 ? 8 : 16) * (size_t)(256 * T) * waves;  // a region per wavefront
}

template <typename R>
static hipError_t launch_fg(int N, const FusedGradArgs& a, int T, int grid, int threads, size_t shm, hipStream_t s) {
#define SQH_FG_CASE(n, t)                                                                                    \
    if (N == n && T == t) {                                                                                  \
        if (a.tmaps)                                                                                         \
            hipLaunchKernelGGL((k_fused_grad_chain<R, n, t>), dim3(grid), dim3(threads), shm, s, a, a.tabs, a.tmaps); \
        else                                                                                                 \
            hipLaunchKernelGGL((k_fused_grad<R, n, t>), dim3(grid), dim3(threads), shm, s, a, a.tabs);       \
        return hipGetLastError();                                                                            \
    }
    SQH_FG_CASE(4, 4)
    SQH_FG_CASE(5, 4)
    SQH_FG_CASE(6, 4)
    SQH_FG_CASE(7, 4)
    SQH_FG_CASE(8, 4)
    SQH_FG_CASE(9, 4)
    SQH_FG_CASE(10, 4)
    SQH_FG_CASE(4, 2)
    SQH_FG_CASE(5, 2)
    SQH_FG_CASE(6, 2)
    SQH_FG_CASE(7, 2)
    SQH_FG_CASE(8, 2)
    SQH_FG_CASE(9, 2)
#undef SQH_FG_CASE
    return hipErrorInvalidValue;
}

// Column groups (one per wavefront) of an element: 16 T vector columns per wavefront,
// 2^N / 16 of them per matrix column.
static int fg_groups(int N, int m, int T) {
    const int W = 16 * T / ((1 << N) >> 4);
    return W < 1 ? 0 : (m + W - 1) / W;
}

bool fused_grad_shape_valid(bool f32, int N, int m, int nb, int T, int waves) {
    if (N < 4 || N > kFusedCostMaxQubits || (T != 2 && T != 4) || m <= 0 || nb <= 0) return false;
    if (waves != 1 && waves != 2 && waves != 4 && waves != 8) return false;
    const int groups = fg_groups(N, m, T);
    return groups > 0 && groups % waves == 0 && fused_grad_lds_bytes(f32, nb, T, waves) <= device_max_lds();
}

// Column groups a wavefront takes one after another, adding to one partial: as many as
// leave two wavefronts per SIMD (2048), the most that are resident with four tiles.  Fewer
// partials are then written and summed; a small batch keeps a group per wavefront.
int fused_grad_per(int N, int m, int T, int B) {
    const long long total = (long long)fg_groups(N, m, T) * B;
    return (int)std::max<long long>(1, std::min<long long>(total / 2048, fg_groups(N, m, T)));
}

int fused_grad_wgs(int N, int m, int T, int B) {
    const int per = fused_grad_per(N, m, T, B);
    return (fg_groups(N, m, T) + per - 1) / per;
}

hipError_t launch_fused_grad(bool f32, int N, FusedGradArgs a, int T, int waves, hipStream_t s) {
    if (a.B <= 0 || !fused_grad_shape_valid(f32, N, a.m, a.nb, T, waves)) return hipErrorInvalidValue;
    a.groups = fg_groups(N, a.m, T);
    a.per = fused_grad_per(N, a.m, T, a.B);
    if (a.wgs != fused_grad_wgs(N, a.m, T, a.B)) return hipErrorInvalidValue;  // the partials' layout the caller sized
    const long long wgs_total = ((long long)a.B * a.wgs + waves - 1) / waves;
    const int grid = (int)((wgs_total + 7) / 8 * 8);
    const size_t shm = fused_grad_lds_bytes(f32, a.nb, T, waves);
    return f32 ? launch_fg<float>(N, a, T, grid, 64 * waves, shm, s)
               : launch_fg<double>(N, a, T, grid, 64 * waves, shm, s);
}

}  // namespace sqh
