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
// A wavefront sums its M_b over its task's column groups (a node of FusedGradSplit's tree) in
// registers and memory of its own, so no wavefront waits for another; k_fused_block_corr then sums the partials and runs the
// block's gates backwards, producing each gate's 2x2 correlations in the layout of the
// register-tile adjoint kernel, from which k_finish forms the gradient.
//
// Layouts follow sqh_k_fused_cost.hip: row j of a column under block b is
// base_b[o] + off_b[i]; 16x16x4 MFMA operands A[l % 16][l / 16], B[l / 16][l % 16]; the
// B operand of step s holds rows 4 s + lane / 16, the D layout rows row(r, lane / 16).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "sqh_device.h"
#include "sqh_fused_chain.h"
#include "sqh_kernels.h"

namespace sqh {

namespace {

// Entry (r, c) of a 16 x 16 tile in LDS, columns rotated by the row (XOR) so that both a
// row-wise and a column-wise sweep of 16 lanes touch 16 different bank groups.
__device__ __forceinline__ int fg_tile(int r, int c) { return r * 16 + (c ^ r); }

// The regions are padded on 4 and 5 qubits, where a tile's 16 vector columns are of 8 and 16
// columns (4096 gradients on 5 qubits: 255 us against 275); on 6 and 7 the addresses cost as
// much as the conflicts.
constexpr bool fg_padded(int N) { return N < 6; }

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

// What a wavefront of the gradient kernels works on: n column groups of element e, a node of
// the summation tree (FusedGradSplit), whose correlations go to part; sums pending at level
// l > 0 of the tree wait in pend + (l - 1) nb 512, at level 0 in part.
//
// The same node of all full chunks goes to wavefronts side by side, which read neighbouring
// columns.  A column has 16 bytes of a cache line in each row; with chunks of consecutive
// columns the lines were gone from the L2 before a task came to the next of them (calls of 23
// vectors on 10 qubits in 3 blocks: 513 us, 803 so; 365 and 680 in complex64).
struct FgTask {
    int e, first, stride, chunk, n;
    bool live;
    double *part, *pend;
    template <int T>
    __device__ int group(int turn) const {  // its turn-th; with two tiles in the pairs that four would take
        const int p = first + turn;
        return T == 4 ? p * stride + chunk : ((p >> 1) * stride + chunk) * 2 + (p & 1);
    }
};
template <int T, int W>
__device__ __forceinline__ FgTask fg_task(const FusedGradArgs& a, int wv) {
    FusedGradSplit sp = a.split;
    // The workgroups of either part of the split ordered for the XCDs, each XCD a contiguous
    // range; with a live count (the optimiser's rounds) the plain order, so the live elements
    // spread over the XCDs.  No workgroup without work stands before one with work: those
    // between the parts of a split padded to multiples of 8 left the second part's
    // wavefronts two to a SIMD (10 qubits, 3 vectors of 977 columns: 337 us instead of 311).
    unsigned wg = blockIdx.x, wgs = a.wg0;
    const bool rest = !a.count && wg >= wgs;
    if (a.count) {
        fused_grad_split_live(sp, min(*a.count, a.B), T);
    } else {
        if (rest) {
            wg -= wgs;
            wgs = gridDim.x - wgs;
        }
        wg = (wg & 7) * (wgs >> 3) + min(wg & 7, wgs & 7) + (wg >> 3);
    }
    const int per0 = fused_grad_tasks(sp.groups, sp.l0), l = rest ? sp.l1 : sp.l0;
    const int per = fused_grad_tasks(sp.groups, l), n = rest ? a.B - sp.n0 : sp.n0;
    const long long id = (long long)wg * (blockDim.x >> 6) + wv;
    FgTask t;
    t.live = id < (long long)n * per;
    const int k = (int)(id / per), c = (int)(id % per);
    t.e = (rest ? sp.n0 : 0) + k;
    constexpr int levels = fused_grad_levels(T);
    const int full = a.m / (W << levels), nodes = 1 << (levels - l);  // full chunks; a chunk's nodes
    int node = c;  // the task's place in the tree's order
    if (c < full * nodes) {
        t.chunk = c % full;
        t.stride = full;
        t.first = c / full << l;
        t.n = 1 << l;
        node = t.chunk * nodes + c / full;
    } else {
        t.chunk = 0;
        t.stride = 1;
        t.first = c << l;
        t.n = min(1 << l, sp.groups - t.first);
    }
    const long long before = rest ? (long long)sp.n0 * per0 : 0, at = (long long)k * per + node;
    const long long size = (long long)a.nb * 512;
    t.part = a.mpart + (before + at) * size;
    t.pend = a.pend + (before * max(sp.l0 - 1, 0) + at * max(l - 1, 0)) * size;
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

// M_b of a column group, Y X^T over the wavefront's vector columns (Y and X: item i of tile
// t is row 4 i + lane / 16 of its vector columns), tile by tile through the region as two
// transposed tiles, added to the task's sums of block b: [256] real, then [256] imaginary
// parts.  No wavefront waits for another: summing four wavefronts' correlations in LDS behind
// two barriers per block kept them in step, all in their exchanges while the matrix cores
// idled.  idx: the group's number in the task; the sums pending are those of idx's set bits.
template <typename R, int T, typename Y>
__device__ __forceinline__ void fg_correlate(R* lds, const Y& yr, const Y& yi, const R (&xr)[T][4],
                                             const R (&xi)[T][4], const FgTask& task, int nb, int b, int idx,
                                             int lane) {
    typedef FcMfma<R> MF;
    const int nl = lane & 15, g = lane >> 4;
    const bool last = idx + 1 == task.n;
    const unsigned carry = idx & ~(idx + 1);  // the levels whose second half this group completes
    unsigned set = last ? idx : carry;
    auto at_level = [&](int l) { return (l ? task.pend + (long long)(l - 1) * nb * 512 : task.part) + b * 512; };
    double pr[4] = {0, 0, 0, 0}, pi[4] = {0, 0, 0, 0};  // the first of them, on its way while the tiles run
    auto load = [&]() {
        const double* M = at_level(__builtin_ctz(set));
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int at = MF::row(r, g) * 16 + nl;
            pr[r] = M[at];
            pi[r] = M[256 + at];
        }
    };
    if (set) load();
    double vr[4], vi[4];
#pragma unroll
    for (int h = 0; h < T / 2; ++h) {
        typename MF::V mr = {0, 0, 0, 0}, mi = {0, 0, 0, 0};
#pragma unroll
        for (int t = 2 * h; t < 2 * h + 2; ++t) {
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
            vr[r] = h ? vr[r] + (double)mr[r] : (double)mr[r];
            vi[r] = h ? vi[r] + (double)mi[r] : (double)mi[r];
        }
    }
    while (set) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            vr[r] = pr[r] + vr[r];
            vi[r] = pi[r] + vi[r];
        }
        set &= set - 1;
        if (set) load();
    }
    double* M = at_level(last ? 0 : __builtin_popcount(carry));
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int at = MF::row(r, g) * 16 + nl;
        M[at] = vr[r];
        M[256 + at] = vi[r];
    }
}

}  // namespace

template <typename R, int N, int T>
__global__ __launch_bounds__(512, 2) void k_fused_grad(FusedGradArgs a, const int* __restrict__ tabs) {
    typedef FcMfma<R> MF;
    typedef FcRegion<R, N, T, fg_padded(N)> Reg;
    constexpr int O = Reg::O, W = Reg::W;
    static_assert(W >= 1, "a wavefront holds whole columns");
    extern __shared__ __align__(16) unsigned char fg_smem[];
    int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const FgTask task = fg_task<T, W>(a, wv);
    if (!task.live) return;
    const int e = task.e, m = a.m;
    const Reg lds{reinterpret_cast<R*>(fg_smem) + wv * 2 * Reg::PL};
    const cpx<R>* U = static_cast<const cpx<R>*>(a.U);
    if (a.count) U += (long long)a.run_target[a.elem_run[e]] * a.tgt_stride;
    const cpx<R>* Fe = static_cast<const cpx<R>*>(a.F) + (long long)e * a.nb * 256;
    for (int turn = 0; turn < task.n; ++turn) {
        const int c0 = task.template group<T>(turn) * W;
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
                Reg::full_at(at, tab, tab[LT_LANE + lane], lane);
                lds.template store_full<T>(at, tab, dr, di);
                const int* tn = tab + kLaneTab;
                Reg::full_at(at, tn, tn[LT_LANE + lane], lane);
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
        A.load_t(Fe + (long long)(a.nb - 1) * 256, nl, g);
        for (int b = a.nb - 1; b >= 0; --b) {
            const int* tab = tabs + b * kLaneTab;
            fg_mma<R, T, true>(A, xr, xi, dr, di);
#pragma unroll
            for (int t = 0; t < T; ++t)
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    xr[t][s] = dr[t][s];
                    xi[t][s] = di[t][s];
                }
            fg_correlate<R, T>(lds.p, yr, yi, xr, xi, task, a.nb, b, turn, lane);
            if (b == 0) break;
            fg_mma<R, T, false>(A, yr, yi, dr, di);
            A.load_t(Fe + (long long)(b - 1) * 256, nl, g);
            const int* tn = tab - kLaneTab;
            int at[4], an[4];
            Reg::full_at(at, tab, tab[LT_LANE + lane], lane);
            Reg::full_at(an, tn, tn[LT_LANE + lane], lane);
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
    typedef FcRegion<R, N, T, fg_padded(N)> Reg;
    constexpr int O = Reg::O, W = Reg::W;
    static_assert(W >= 1, "a wavefront holds whole columns");
    extern __shared__ __align__(16) unsigned char fg_smem[];
    int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const FgTask task = fg_task<T, W>(a, wv);
    if (!task.live) return;
    const int e = task.e, m = a.m;
    const Reg lds{reinterpret_cast<R*>(fg_smem) + wv * 2 * Reg::PL};
    const cpx<R>* U = static_cast<const cpx<R>*>(a.U);
    if (a.count) U += (long long)a.run_target[a.elem_run[e]] * a.tgt_stride;
    const cpx<R>* Fe = static_cast<const cpx<R>*>(a.F) + (long long)e * a.nb * 256;
    for (int turn = 0; turn < task.n; ++turn) {
        const int c0 = task.template group<T>(turn) * W;
        asm volatile("" : "+v"(lane));  // no lane's addresses kept in registers from group to group
        const int nl = lane & 15, g = lane >> 4;
        // phase 1: Z_1 in block 0's grouping, X = the target's columns there, and the trace
        // entries from Z_0 = F_0^T Z_1
        R zr[T][4], zi[T][4], xr[T][4], xi[T][4];
        typename MF::V er[T], ei[T];
        FcA<R> A;
        fused_chain_to_block0<R, N, T, false, Reg>(tabs, tmaps, a.nb, lds, Fe, c0, m, a.trace_off, lane, zr, zi, A);
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
        // The block that X, then Z pass next, on its way before the branches of the sums; with
        // two tiles it would cost a wavefront per SIMD.
        constexpr bool AHEAD = T == 4;
        FcA<R> An;
        if constexpr (AHEAD) An.load_n(Fe, nl, g);
        fg_correlate<R, T>(lds.p, zr, zi, xr, xi, task, a.nb, 0, turn, lane);
        // phase 2, one step up: X_b into block b + 1's grouping, Z_{b+2} (block b + 1's
        // grouping, as a result) from Z_{b+1} -- block 0's operand for the first step, the
        // last step's result after it -- then M_{b+1}.  The first step runs on its own, so
        // that its operand is not live through the loop.
        auto step = [&](int b, auto first_step) __attribute__((always_inline)) {
            constexpr bool ZB = decltype(first_step)::value;
            const int* tab = tabs + b * kLaneTab;
            const int* tn = tab + kLaneTab;
            int at[4], an[4];
            Reg::full_at(at, tab, tab[LT_LANE + lane], lane);
            Reg::full_at(an, tn, tn[LT_LANE + lane], lane);
            {
                typename MF::V dr[T], di[T];
                if constexpr (!AHEAD) An.load_n(Fe + (long long)b * 256, nl, g);
                fg_mma<R, T, false>(An, xr, xi, dr, di);
                if constexpr (AHEAD) An.load_n(Fe + (long long)(b + 1) * 256, nl, g);
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
                if constexpr (!AHEAD) An.load_n(Fe + (long long)(b + 1) * 256, nl, g);
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
            fg_correlate<R, T>(lds.p, er, ei, xr, xi, task, a.nb, b + 1, turn, lane);
        };
        step(0, std::true_type{});
        for (int b = 1; b + 1 < a.nb; ++b) step(b, std::false_type{});
    }
}

size_t fused_grad_lds_bytes(bool f32, int N, int T, int waves) {
    return (size_t)waves * 2 * fc_plane(N, T, fg_padded(N)) * (f32 ? 4 : 8);  // a region per wavefront
}

// The kernel of a shape, or null.
template <typename R>
static const void* fg_kernel(int N, int T, bool chain) {
#define SQH_FG_CASE(n, t)                                                    \
    if (N == n && T == t)                                                    \
        return chain ? reinterpret_cast<const void*>(&k_fused_grad_chain<R, n, t>) \
                     : reinterpret_cast<const void*>(&k_fused_grad<R, n, t>);
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
    return nullptr;
}
static const void* fg_kernel(bool f32, int N, int T, bool chain) {
    return f32 ? fg_kernel<float>(N, T, chain) : fg_kernel<double>(N, T, chain);
}

// Column groups (one per wavefront) of an element: 16 T vector columns per wavefront,
// 2^N / 16 of them per matrix column.
int fused_grad_groups(int N, int m, int T) {
    const int W = 16 * T / ((1 << N) >> 4);
    return W < 1 ? 0 : (m + W - 1) / W;
}

bool fused_grad_shape_valid(bool f32, int N, int m, int nb, int T, int waves) {
    if (N < 4 || N > kFusedCostMaxQubits || (T != 2 && T != 4) || m <= 0 || nb <= 0) return false;
    if (waves != 1 && waves != 2 && waves != 4 && waves != 8) return false;
    return fused_grad_groups(N, m, T) > 0 && fused_grad_lds_bytes(f32, N, T, waves) <= device_max_lds();
}

// Wavefronts of the kernel that are resident together on the current device.
static int fg_resident(const void* kernel, size_t shm, int waves) {
    int dev = 0, cus = 0, wgs = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&wgs, kernel, 64 * waves, shm) != hipSuccess || wgs < 1) {
        (void)hipGetLastError();
        return 2048;
    }
    return cus * wgs * waves;
}

// The card runs a launch in rounds of its resident wavefronts, and a last round that is not
// full costs as much as a full one.  So the bulk of the elements runs in the largest tasks
// (few partials) that fill whole rounds, and the rest in smaller ones.  Unit of the estimate:
// a column group on a full card (83 us at 8 qubits in complex128); a round with fewer
// wavefronts per SIMD is shorter by less than their share, and a partial costs its way to
// memory and back.  Gradients of 384, 512, 520, 640 and 1000 vectors (8 qubits, 264 angles,
// complex128): 1.06, 1.40, 1.44, 1.85 and 2.75 ms; in equal tasks of total / 2048 groups,
// rounded down, 1.56, 1.41, 2.08, 2.56 and 3.94; a wavefront per group, four summed in LDS,
// 1.32, 1.72, 1.78, 2.13 and 3.30.
constexpr double kFgPartialCost = 1e-4;
FusedGradSplit fused_grad_split(bool f32, int N, int m, int nb, int T, int waves, bool chain, int B, bool live,
                                size_t* partials, size_t* pending) {
    FusedGradSplit s;
    s.groups = fused_grad_groups(N, m, T);
    s.resident = 2048;
    s.n0 = B;
    const long long total = (long long)B * s.groups;
    const int levels = fused_grad_levels(T);
    if (live || total > 1024)
        s.resident = fg_resident(fg_kernel(f32, N, T, chain), fused_grad_lds_bytes(f32, N, T, waves), waves);
    const long long R = s.resident;
    if (live) {
        FusedGradSplit most = s;
        fused_grad_split_live(most, B, T);
        // most tasks of any count up to B (fused_grad_split_live)
        *partials = (size_t)std::min(total, std::max(4 * R + B, (long long)B * fused_grad_tasks(s.groups, levels)));
        *pending = *partials * std::max(most.l0 - 1, 0);
        return s;
    }
    auto tasks = [&](long long n, int l) { return n * fused_grad_tasks(s.groups, l); };
    if (total > R) {
        const double w = std::max(1.0, R / 1024.0);  // wavefronts per SIMD
        auto cost = [&](long long n, int l) {
            const long long t = tasks(n, l), rounds = t / R, over = t % R;
            const double part = over ? 0.3 + 0.7 * std::ceil(over * w / R) / w : 0.0;
            return (rounds + part) * (1 << l) + kFgPartialCost * t;
        };
        double best = -1.0;
        for (int l = 0; l <= levels; ++l) {
            if (l > 0 && (1 << (l - 1)) >= s.groups) break;
            const long long full = tasks(B, l) / R * R / fused_grad_tasks(s.groups, l);  // elements in whole rounds
            for (long long n : {full, (long long)B}) {
                for (int k = 0; k <= (n < B ? l : 0); ++k) {
                    const double c = (n ? cost(n, l) : 0.0) + (n < B ? cost(B - n, k) : 0.0);
                    if (best < 0.0 || c < best) {
                        best = c;
                        s.n0 = (int)n;
                        s.l0 = l;
                        s.l1 = k;
                    }
                }
            }
        }
    }
    *partials = (size_t)(tasks(s.n0, s.l0) + tasks(B - s.n0, s.l1));
    *pending = (size_t)(tasks(s.n0, s.l0) * std::max(s.l0 - 1, 0) + tasks(B - s.n0, s.l1) * std::max(s.l1 - 1, 0));
    return s;
}

hipError_t launch_fused_grad(bool f32, int N, FusedGradArgs a, int T, int waves, hipStream_t s) {
    if (a.B <= 0 || !fused_grad_shape_valid(f32, N, a.m, a.nb, T, waves)) return hipErrorInvalidValue;
    const void* kernel = fg_kernel(f32, N, T, a.tmaps != nullptr);
    if (!kernel || a.split.groups != fused_grad_groups(N, a.m, T) || a.split.resident <= 0) return hipErrorInvalidValue;
    auto wgs = [&](long long tasks) { return (int)((tasks + waves - 1) / waves); };
    int grid;
    if (a.count) {
        grid = wgs((long long)a.live_tasks);
    } else {
        a.wg0 = wgs((long long)a.split.n0 * fused_grad_tasks(a.split.groups, a.split.l0));
        grid = a.wg0 + wgs((long long)(a.B - a.split.n0) * fused_grad_tasks(a.split.groups, a.split.l1));
    }
    const int* tabs = a.tabs;
    const int* tmaps = a.tmaps;
    void* args[] = {&a, &tabs, &tmaps};  // k_fused_grad takes the first two
    return hipLaunchKernel(kernel, dim3(grid), dim3(64 * waves), args, fused_grad_lds_bytes(f32, N, T, waves), s);
}

}  // namespace sqh
