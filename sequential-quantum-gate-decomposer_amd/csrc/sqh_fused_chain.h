// sqh_fused_chain.h -- the fused 4-qubit blocks on the matrix cores: MFMA helpers, the
// exchange of a wavefront's columns between the blocks' groupings, and the transposed chain
// from unit vectors (k_fused_trace, k_fused_grad_chain).
//
// What bounds these kernels: FP64 MFMA and the vector ALU do not overlap on gfx950.  With
// four wavefronts per SIMD, a v_mfma_f64_16x16x4f64 takes 65 cycles alone (77 TFLOP/s on the
// card) and 2.5 to 3 more for every 32-bit VALU instruction, 6 for an FP64 FMA and 13 for
// every 16-byte LDS access that accompanies it
// (profiles/f64_mfma_beside_vector_and_lds.md).  So the code around the MFMAs is what can be saved: addresses come
// from lane tables built by the host, one XOR with a uniform value each (LT_*,
// sqh_kernels.h); real and imaginary parts are separate LDS planes, so a result register
// pair is stored without packing; the negated imaginary part is the MFMA's own operand
// modifier; and the kernels declare at least two wavefronts per SIMD, below which the
// compiler keeps accumulators in the AGPR half of the file and copies them.
//
// Trace entry c is (V U)[rho, c] with rho = c + trace_off and V = F_{nb-1} ... F_0: row
// rho of V dotted with column c of U.  Row rho of V is column rho of
// V^T = F_0^T F_1^T ... F_{nb-1}^T, built from the unit vector e_rho: F_{nb-1}^T e_rho is
// row rho of F_{nb-1} on the rows that agree with rho outside the block's qubits
// (loaded, no arithmetic), and each later block only touches the rows that agree with
// rho outside the union S_b of the qubits seen so far (the support): 2^(|S_b| - 4) of a
// column's 2^N / 16 outer groups.
//
// Layout: a wavefront owns W = 16 T / O columns (O = 2^N / 16); block b's vector column
// n holds column w = n >> lg_b, support group k = n & (2^lg_b - 1), rows
// kb_b[k] | (rho_w & nS_b) | off_b[i] (kTraceMapStride ints per block: off[16], kb[64],
// lg, nS).  Only the first ceil(W 2^lg_b / 16) tiles carry work.  The wavefront's LDS
// region starts at zero and rows outside a support are never stored, so they read as
// zero (the supports only grow).  Once the support covers every qubit the blocks use the
// forward pass's layout (vector column 16 t + nl = column (16 t + nl) / O, outer group
// (16 t + nl) % O), with no row arithmetic.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "sqh_device.h"
#include "sqh_kernels.h"

namespace sqh {

typedef double fc_f64x4 __attribute__((ext_vector_type(4)));
typedef float fc_f32x4 __attribute__((ext_vector_type(4)));

// 16x16x4 MFMA: lane l supplies A[l % 16][l / 16] and B[l / 16][l % 16].  Item r of lane l's
// result is D[4 r + l / 16][l % 16] in double precision and D[4 (l / 16) + r][l % 16] in
// single; a_row(nl) is the row of the block matrix that lane nl supplies to A so that item
// r is row 4 r + l / 16 in both.  op_neg: C - A B.
template <typename R>
struct FcMfma;
template <>
struct FcMfma<double> {
    typedef fc_f64x4 V;
    static __device__ __forceinline__ V op(double a, double b, V c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ V op_neg(double a, double b, V c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 1);  // neg:[1,0,0]
    }
    static __device__ __forceinline__ int a_row(int nl) { return nl; }
    static __device__ __forceinline__ int row(int r, int g) { return 4 * r + g; }
};
template <>
struct FcMfma<float> {
    typedef fc_f32x4 V;
    static __device__ __forceinline__ V op(float a, float b, V c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ V op_neg(float a, float b, V c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(-a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int a_row(int nl) { return ((nl & 3) << 2) | (nl >> 2); }
    static __device__ __forceinline__ int row(int r, int g) { return 4 * g + r; }
};

// LDS position of row j of a column: the row's low nibble XOR its higher bits folded
// down, so the 16 lanes of a lane group that differ in the outer index land in
// distinct 16-element slots for most qubit sets.
template <int N>
__device__ __forceinline__ int fc_slot(int j) {
    if constexpr (N <= 4) {
        return j;
    } else {
        int h = j >> 4;
        if constexpr (N > 8) h ^= h >> 4;
        return j ^ (h & 15);
    }
}

// Wave-scope ordering of the LDS exchange: the stores of a remap are issued before its
// loads (LDS serves one wavefront's requests in order; this keeps the compiler from
// moving the loads up).
__device__ __forceinline__ void fc_wave_fence() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); }

// local index of row j in a block (bit q <-> the block's q-th smallest qubit), from the
// row offsets of local indices 1, 2, 4 and 8
__device__ __forceinline__ int ft_local(const int* mp, int j) {
    return ((j & mp[1]) ? 1 : 0) | ((j & mp[2]) ? 2 : 0) | ((j & mp[4]) ? 4 : 0) | ((j & mp[8]) ? 8 : 0);
}

// A operand of one block: A[4 s + g] of the lane's row, real and imaginary parts.
template <typename R>
struct FcA {
    R re[4], im[4];
    // F^T (the chain) of the block matrix at F
    __device__ __forceinline__ void load_t(const cpx<R>* F, int nl, int g) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const cpx<R> f = F[(4 * s + g) * 16 + FcMfma<R>::a_row(nl)];
            re[s] = f.re;
            im[s] = f.im;
        }
    }
    // F (the forward pass)
    __device__ __forceinline__ void load_n(const cpx<R>* F, int nl, int g) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const cpx<R> f = F[FcMfma<R>::a_row(nl) * 16 + 4 * s + g];
            re[s] = f.re;
            im[s] = f.im;
        }
    }
};

// Y = A X on tiles T0 .. T0 + TS - 1, complex.
template <typename R, int T, int TS, int T0 = 0>
__device__ __forceinline__ void fc_mma(const FcA<R>& A, const R (&xr)[T][4], const R (&xi)[T][4],
                                       typename FcMfma<R>::V (&yr)[TS], typename FcMfma<R>::V (&yi)[TS]) {
    typedef FcMfma<R> MF;
#pragma unroll
    for (int t = 0; t < TS; ++t) yr[t] = yi[t] = typename MF::V{0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
#pragma unroll
        for (int t = 0; t < TS; ++t) {
            yr[t] = MF::op(A.re[s], xr[T0 + t][s], yr[t]);
            yi[t] = MF::op(A.re[s], xi[T0 + t][s], yi[t]);
        }
#pragma unroll
        for (int t = 0; t < TS; ++t) {
            yr[t] = MF::op_neg(A.im[s], xi[T0 + t][s], yr[t]);
            yi[t] = MF::op(A.im[s], xr[T0 + t][s], yi[t]);
        }
    }
}

// Entries between the columns of a region beyond 2^N where the lanes of an access are in
// several columns (which else all start in the same bank): W columns then start 16 / W banks
// apart, four wavefronts' regions 16.
__host__ __device__ constexpr int fc_pad(int N, int T) {
    const int W = 16 * T / ((1 << N) >> 4);
    return W < 1 || W > 16 ? 1 : 16 / W;
}
// Entries of a region's plane (padded).
__host__ __device__ constexpr int fc_plane(int N, int T, bool padded) {
    return 256 * T + (padded ? 16 * T / ((1 << N) >> 4) * fc_pad(N, T) + 8 : 0);
}

// A wavefront's region of W 2^N entries: real parts, then imaginary parts.
template <typename R, int N, int T, bool PADDED = false>
struct FcRegion {
    static constexpr int D = 1 << N, O = D >> 4, W = 16 * T / O, PL = fc_plane(N, T, PADDED);
    static constexpr int PAD = PADDED ? fc_pad(N, T) : 0, CS = D + PAD;  // column stride
    R* p;
    __device__ __forceinline__ void put(int i, R re, R im) const {
        p[i] = re;
        p[i + PL] = im;
    }
    __device__ __forceinline__ void get(int i, R& re, R& im) const {
        re = p[i];
        im = p[i + PL];
    }
    // Slot of row 4 s + g of tile t's vector column in the full layout of a block: lane
    // entry at[s] (LT_LANE ^ LT_S), tile part constant up to 16 outer groups.
    static __device__ __forceinline__ int full(const int (&at)[4], const int* tab, int t, int s) {
        if constexpr (O <= 16) return at[s] + t * (16 / O) * CS;
        return (at[s] ^ tab[LT_T + t]) + t / (O > 16 ? O / 16 : 1) * PAD;
    }
    static __device__ __forceinline__ void full_at(int (&at)[4], const int* tab, int lane_entry, int lane) {
#pragma unroll
        for (int s = 0; s < 4; ++s) at[s] = (lane_entry ^ tab[LT_S + s]) + (PADDED && O < 16 ? (lane & 15) / O * PAD : 0);
    }
    __device__ __forceinline__ void load_full(const int (&at)[4], const int* tab, R (&xr)[T][4], R (&xi)[T][4]) const {
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int s = 0; s < 4; ++s) get(full(at, tab, t, s), xr[t][s], xi[t][s]);
        fc_wave_fence();
    }
    template <int TS, int T0 = 0>
    __device__ __forceinline__ void store_full(const int (&at)[4], const int* tab, const typename FcMfma<R>::V (&yr)[TS],
                                               const typename FcMfma<R>::V (&yi)[TS]) const {
#pragma unroll
        for (int t = 0; t < TS; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) put(full(at, tab, T0 + t, r), yr[t][r], yi[t][r]);
        fc_wave_fence();
    }
};

// Sums of a wavefront's full-layout products over the lanes of each column: sr / si hold a
// partial per column (more than 16 outer groups) or per tile of whole columns; column
// c0 + c's pair of doubles goes to dg + 2 c.
template <int N, int T, int C>
__device__ __forceinline__ void fc_column_sums(const double (&sr)[C], const double (&si)[C], double* dg, int c0, int m,
                                               int lane) {
    constexpr int O = (1 << N) >> 4;
    const int nl = lane & 15, g = lane >> 4;
#pragma unroll
    for (int c = 0; c < C; ++c) {
        // lanes below 32 go on with the real part, the others with the imaginary one
        double s = lane_halves(sr[c], si[c], false);
        s = lane_halves(s, s, true);
        if constexpr (O >= 16) {
            s = row_sum(s);
            if ((lane == 0 || lane == 32) && c0 + c < m) dg[2 * c + (lane >> 5)] = s;
        } else {
#pragma unroll
            for (int d = 1; d < O; d <<= 1) s += __shfl_xor(s, d, 64);
            const int w = (16 * c + nl) / O;
            if ((nl & (O - 1)) == 0 && (g & 1) == 0 && c0 + w < m) dg[2 * w + (g >> 1)] = s;
        }
    }
}

// The chain F_{nb-1}^T, ..., F_1^T on e_rho for the wavefront's W columns c0 + w
// (rho = c0 + w + trace_off; columns past m take row trace_off).  On return xr / xi hold
// block 0's B operand in the chain's grouping of block 0 and A block 0's operand F_0^T.
// With PF, block b - 1's matrix is loaded while block b runs.
template <typename R, int N, int T, bool PF, typename Reg>
__device__ __forceinline__ void fused_chain_to_block0(const int* __restrict__ tabs, const int* __restrict__ tmaps,
                                                      int nb, Reg lds, const cpx<R>* __restrict__ Fe,
                                                      int c0, int m, int trace_off, int lane, R (&xr)[T][4],
                                                      R (&xi)[T][4], FcA<R>& A) {
    typedef FcMfma<R> MF;
    constexpr int D = Reg::D, W = Reg::W;
    const int nl = lane & 15, g = lane >> 4;
    auto rho_of = [&](int w) { return (c0 + w < m ? c0 + w : 0) + trace_off; };
    // The region starts at zero (rows outside a block's support are never stored and read
    // as zero; the supports only grow), then holds F_{nb-1}^T e_rho per column: row
    // loc(rho) of F_{nb-1} on the rows that agree with rho outside its qubits.
    {
        typedef int zero4 __attribute__((ext_vector_type(4)));
        zero4* z = reinterpret_cast<zero4*>(lds.p);
        constexpr int n = 2 * Reg::PL * (int)sizeof(R) / 16;
#pragma unroll
        for (int i = 0; i < (n + 63) / 64; ++i)
            if (64 * i + 63 < n || 64 * i + lane < n) z[64 * i + lane] = zero4{0, 0, 0, 0};
    }
    // the support layout's entry of each tile of block b; vector columns past the
    // wavefront's columns read column 0 (their products are never stored)
    auto support_at = [&](const int* tab, int entry, int ts, int (&at)[T], int (&pad)[T]) {
        const int lg = tab[LT_LG], nS = tab[LT_NS];
#pragma unroll
        for (int t = 0; t < T; ++t) {
            if (t < ts) {
                const int w = (16 * t + nl) >> lg, wc = w < W ? w : 0;
                at[t] = entry ^ tab[LT_ST + t] ^ fc_slot<N>(rho_of(wc) & nS) ^ (wc * D);
                pad[t] = wc * Reg::PAD;
            }
        }
    };
    auto load_support = [&](const int* tab, const int (&at)[T], const int (&pad)[T], int ts) {
#pragma unroll
        for (int t = 0; t < T; ++t)
            if (t < ts) {
#pragma unroll
                for (int s = 0; s < 4; ++s) lds.get((at[t] ^ tab[LT_S + s]) + pad[t], xr[t][s], xi[t][s]);
            }
        fc_wave_fence();
    };
    auto tiles = [&](const int* tab) { return ((W << tab[LT_LG]) + 15) >> 4; };
    int b = nb - 2;
    const int* tab = tabs + b * kLaneTab;
    int entry = tab[LT_SLANE + lane];
    A.load_t(Fe + (long long)b * 256, nl, g);
    {
        const int* mq = tmaps + (nb - 1) * kTraceMapStride;
        const int* tq = tabs + (nb - 1) * kLaneTab;
        const cpx<R>* Fq = Fe + (long long)(nb - 1) * 256;
        fc_wave_fence();
#pragma unroll
        for (int p = lane; p < 16 * W; p += 64) {
            const int w = p >> 4, i = p & 15;
            const int rho = rho_of(w);
            const cpx<R> f = Fq[ft_local(mq, rho) * 16 + i];
            lds.put((tq[LT_S + (i >> 2)] ^ tq[LT_SLANE + 16 * (i & 3)] ^ fc_slot<N>(rho & mq[81])) + w * Reg::CS, f.re, f.im);
        }
        fc_wave_fence();
    }
    // Each block reads its operand where the loop begins, so that no operand is carried
    // around it (the compiler copies registers that are).
    FcA<R> An;
    // The supports only grow along the chain: first the blocks whose support fills fewer
    // than T tiles (1, or 2 of 4), then the dense ones.
    int ts = tiles(tab);
    for (; b > 0 && ts < T; --b) {
        const int* tn = tab - kLaneTab;
        int at[T], pad[T];
        support_at(tab, entry, ts, at, pad);
        if constexpr (PF) An.load_t(Fe + (long long)(b - 1) * 256, nl, g);
        entry = tn[LT_SLANE + lane];
        auto run = [&](auto tiles_run) __attribute__((always_inline)) {
            constexpr int TS = decltype(tiles_run)::value;
            typename MF::V yr[TS], yi[TS];
            R vr[TS][4], vi[TS][4];
#pragma unroll
            for (int t = 0; t < TS; ++t)
#pragma unroll
                for (int s = 0; s < 4; ++s) lds.get((at[t] ^ tab[LT_S + s]) + pad[t], vr[t][s], vi[t][s]);
            fc_wave_fence();
            fc_mma<R, TS, TS>(A, vr, vi, yr, yi);
#pragma unroll
            for (int t = 0; t < TS; ++t) {
                if ((16 * t + nl) >> tab[LT_LG] < W) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) lds.put((at[t] ^ tab[LT_S + r]) + pad[t], yr[t][r], yi[t][r]);
                }
            }
            fc_wave_fence();
        };
        if (T >= 4 && ts >= 2) run(std::integral_constant<int, (T >= 4 ? 2 : 1)>{});
        else run(std::integral_constant<int, 1>{});
        tab = tn;
        ts = tiles(tab);
        if constexpr (PF) A = An;
        else A.load_t(Fe + (long long)(b - 1) * 256, nl, g);
    }
    if (ts < T) {  // block 0, its support short of the register
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int s = 0; s < 4; ++s) xr[t][s] = xi[t][s] = 0;
        int at[T], pad[T];
        support_at(tab, entry, ts, at, pad);
        load_support(tab, at, pad, ts);
        return;
    }
    // Blocks of full support (no row outside it): vector column 16 t + nl is column
    // (16 t + nl) / O, outer group (16 t + nl) % O, as in the forward pass.
    entry = tab[LT_LANE + lane];
    int af[4];
    for (; b > 0; --b) {
        const int* tn = tab - kLaneTab;
        if constexpr (PF) An.load_t(Fe + (long long)(b - 1) * 256, nl, g);
        Reg::full_at(af, tab, entry, lane);
        entry = tn[LT_LANE + lane];
        typename MF::V yr[T], yi[T];
        R vr[T][4], vi[T][4];
        lds.load_full(af, tab, vr, vi);
        fc_mma<R, T, T>(A, vr, vi, yr, yi);
        lds.template store_full<T>(af, tab, yr, yi);
        tab = tn;
        if constexpr (PF) A = An;
        else A.load_t(Fe + (long long)(b - 1) * 256, nl, g);
    }
    Reg::full_at(af, tab, entry, lane);
    lds.load_full(af, tab, xr, xi);
}

}  // namespace sqh
