// sqh_k_fused_cost.hip -- batched cost of the circuit run as fused dense 4-qubit blocks
// on the matrix cores, with every column of the target resident on the chip from its
// first load to its trace entry.
//
// The circuit is the product of nb dense 16 x 16 blocks on sorted 4-qubit sets (the
// fusion plan; per batch element the block matrices F_b are built from its parameters,
// k_fuse_blocks).  A wavefront owns 64 "vector columns": W = 64 / O columns of the target,
// each split into O = 2^N / 16 outer groups of the 16 rows its block touches.  Per
// block it computes Y = F_b X for its 64 vector columns as four 16 x 16 output tiles,
// 16 MFMAs each (four real products, K = 16 in four steps):
// v_mfma_f64_16x16x4f64 for complex128, v_mfma_f32_16x16x4f32 (FP32 accumulation) for
// complex64.  Between blocks the tiles go through the wavefront's own LDS region in
// natural row order and come back in the next block's grouping.  Of the last block the
// cost needs only row c + trace_off of each column c: a 16-term dot product with that
// row of F_nb per column replaces the block product.  The target
// is read once per wavefront (it is shared by the batch and stays in L2); nothing
// else touches HBM but the block matrices and the per-column trace entries.  The columns
// come in (and, in the store pass, go out) through the regions of all the workgroup's
// wavefronts, so it is the workgroup that owns them in that pass.
//
// Row j of a column under block b: j = base_b[o] + off_b[i] for local index i (bit q of
// i <-> the q-th smallest qubit of the block, as apply_large_kernel_to_input,
// apply_large_kernel_to_input.cpp:82-102) and outer index o (the other qubits in
// ascending order); both tables come from the host per block.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "sqh_device.h"
#include "sqh_fused_chain.h"
#include "sqh_kernels.h"

namespace sqh {

// One workgroup's launch shape (FusedCostCfg): T 16-column tiles per wavefront (2 or
// 4: 32 or 64 vector columns), H exchange groups per block (the tiles go through LDS in
// H independent groups, so the exchange of one overlaps the MFMAs of the next; a group
// must hold whole columns), PF: block b + 1's matrix loaded while block b runs (more
// registers, fewer waves), waves per workgroup at run time.  Every shape performs the
// same operations on every column in the same order: results are bit-identical.
//
// Workgroups are ordered for the XCDs: hardware workgroup i runs on XCD i mod 8, and the
// logical order gives each XCD a contiguous range of (element, column group) work, so
// an element's block matrices and the target stay in one XCD's L2.
//
// The columns come in and go out through the LDS regions with a workgroup's threads along
// the rows of the matrix (W columns per wavefront, 128 contiguous bytes a row for four
// wavefronts at 8 qubits): in the operand layout each lane of a load takes another row, and
// the addresses, a cache line per lane, took as long as the blocks.  For that pass the columns
// are padded apart (fc_pad): unpadded, all of them start in the same bank, and at 5 qubits
// the stores into LDS took half the launch (5 qubits, 2 blocks, 4096 matrices of 32 columns
// in complex128: 64 us, 35 so; 20000 in complex64: 210 and 88).
template <typename R, int N, int T, int H, bool PF>
__global__ __launch_bounds__(256, 2) void k_fused_cost(FusedCostArgs a, const int* __restrict__ tabs) {
    typedef FcMfma<R> MF;
    typedef FcRegion<R, N, T, true> Reg;
    constexpr int O = Reg::O, W = Reg::W;
    constexpr int TH = T / H;  // tiles per exchange group
    static_assert(W >= 1 && (16 * TH) % O == 0, "an exchange group holds whole columns");
    extern __shared__ __align__(16) unsigned char fc_smem[];
    R* const region = reinterpret_cast<R*>(fc_smem);
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nw = blockDim.x >> 6;
    const long long per_xcd = gridDim.x >> 3;  // the grid is a multiple of 8
    const long long lwg = (long long)(blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    const long long total = (long long)a.B * a.groups;
    const int m = a.m;
    // the thread's column in the passes over rows: column cq of element eq, in wavefront
    // q / W's region; it takes rows tid / (W nw) + k 64 / W
    const int q = threadIdx.x & (W * nw - 1), v = q / W, wq = q % W;
    const long long first = lwg * nw;  // the workgroup's first (element, column group)
    const int e0 = (int)(first / a.groups), g0 = (int)(first % a.groups);
    const int eq = e0 + (g0 + v) / a.groups, cq = (g0 + v) % a.groups * W + wq;
    const bool okq = first + v < total && cq < m;
    const Reg ldsq{region + v * 2 * Reg::PL};
    const int row_q = threadIdx.x / (W * nw);
    {
        const long long src = a.in_index ? (long long)a.in_index[okq ? eq : 0]
                              : a.dinfo ? (long long)a.dinfo[4 * (okq ? eq : 0)] : (long long)eq;
        const cpx<R>* p = static_cast<const cpx<R>*>(a.U) + src * a.in_bstride + (long long)row_q * a.in_stride + cq;
        const long long step = (long long)(64 / W) * a.in_stride;
        cpx<R> u[4 * T];
#pragma unroll
        for (int k = 0; k < 4 * T; ++k) u[k] = okq ? p[k * step] : mk<R>(0, 0);
#pragma unroll
        for (int k = 0; k < 4 * T; ++k) ldsq.put(fc_slot<N>(row_q + k * (64 / W)) + wq * Reg::CS, u[k].re, u[k].im);
    }
    __syncthreads();
    const long long wave = first + wv;
    const int e = e0 + (g0 + wv) / a.groups;
    const int c0 = (g0 + wv) % a.groups * W;
    const Reg lds{region + wv * 2 * Reg::PL};
    const int nl = lane & 15, g = lane >> 4;
    if (wave < total) {
        const cpx<R>* F = static_cast<const cpx<R>*>(a.F);
        const cpx<R>* Fe = F + (long long)e * a.F_bstride;
        // Blocks lo .. hi - 1: all of them; up to the element's own number (the prefixes of
        // the derivatives); or from the differentiated one, which is the element's own, on.
        // The cost pass stops before the last block: of it only row c + trace_off of each
        // column c is needed (below).
        int lo = 0, hi = a.out ? a.nb : a.nb - 1;
        const cpx<R>* F0 = Fe;
        if (a.prefix) hi = e;
        if (a.dinfo) {
            lo = __builtin_amdgcn_readfirstlane(a.dinfo[4 * e]);
            F0 = F + (long long)(a.nb + e) * 256;
        }
        // A operand of the running block (with PF, the next block's is loaded meanwhile)
        FcA<R> A, An;
        const int* tab = tabs + lo * kLaneTab;
        int entry = tab[LT_LANE + lane];
        if (lo < hi) A.load_n(a.dinfo ? F0 : Fe + (long long)lo * 256, nl, g);
        for (int b = lo; b < hi; ++b) {
            int at[4];
            Reg::full_at(at, tab, entry, lane);
            if (PF && b + 1 < hi) An.load_n(Fe + (long long)(b + 1) * 256, nl, g);
            if (b + 1 < a.nb) entry = tab[kLaneTab + LT_LANE + lane];
            // each exchange group reads and stores its own columns only
#pragma unroll
            for (int h = 0; h < H; ++h) {
                R vr[TH][4], vi[TH][4];
                typename MF::V yr[TH], yi[TH];
#pragma unroll
                for (int u = 0; u < TH; ++u)
#pragma unroll
                    for (int s = 0; s < 4; ++s) lds.get(Reg::full(at, tab, h * TH + u, s), vr[u][s], vi[u][s]);
                fc_wave_fence();
                fc_mma<R, TH, TH>(A, vr, vi, yr, yi);
                if (h == 0) lds.template store_full<TH, 0>(at, tab, yr, yi);
                else lds.template store_full<TH, (H > 1 ? TH : 0)>(at, tab, yr, yi);
            }
            tab += kLaneTab;
            if constexpr (PF) A = An;
            else if (b + 1 < hi) A.load_n(Fe + (long long)(b + 1) * 256, nl, g);
        }
    }
    if (a.out) {
        // apply_to: the columns back to HBM (a workgroup writes only the columns it read,
        // after it has read them all, so the pass may run in place)
        __syncthreads();
        if (okq) {
            cpx<R>* p = static_cast<cpx<R>*>(a.out) + (long long)eq * a.out_bstride + (long long)row_q * a.out_stride + cq;
            const long long step = (long long)(64 / W) * a.out_stride;
#pragma unroll
            for (int k = 0; k < 4 * T; ++k) {
                cpx<R> y;
                ldsq.get(fc_slot<N>(row_q + k * (64 / W)) + wq * Reg::CS, y.re, y.im);
                p[k * step] = y;
            }
        }
        return;
    }
    if (wave >= total) return;
    // cost pass, last block: one 16-term dot product with row c + trace_off of F per
    // column c.  X is in the block's grouping; the vector column whose outer group holds
    // the row contributes, its 4 lane groups summing their 4 entries each.
    {
        const int* tab = tabs + (a.nb - 1) * kLaneTab;
        R xr[T][4], xi[T][4];
        int at[4];
        Reg::full_at(at, tab, tab[LT_LANE + lane], lane);
        lds.load_full(at, tab, xr, xi);
        const int* mp = a.maps + (a.nb - 1) * kFusedMapStride;
        const int mask = mp[15];  // the block's four row bits (off of local index 15)
        const cpx<R>* Fl = static_cast<const cpx<R>*>(a.F) + (long long)e * a.F_bstride + (long long)(a.nb - 1) * 256;
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const int col = c0 + (16 * t + nl) / O;
            const int jt = col + a.trace_off;
            const bool hit = col < m && (jt & ~mask) == ((tab[LT_ROW + lane] & ~mask) | tab[LT_RT + t]);
            // local index of row jt: its bits at the block's qubits
            const int is = ft_local(mp, jt);
            R sr = 0, si = 0;
            if (hit) {
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const cpx<R> f = Fl[is * 16 + 4 * s + g];
                    sr += f.re * xr[t][s] - f.im * xi[t][s];
                    si += f.re * xi[t][s] + f.im * xr[t][s];
                }
            }
            // the four lane groups of the vector column (lanes nl + 16 g)
            sr += __shfl_xor(sr, 16, 64);
            si += __shfl_xor(si, 16, 64);
            sr += __shfl_xor(sr, 32, 64);
            si += __shfl_xor(si, 32, 64);
            if (hit && g == 0) {
                double* d = a.diag + 2 * ((long long)e * m + col);
                d[0] = (double)sr;
                d[1] = (double)si;
            }
        }
    }
}

// ---------------------------------------------------------------------------------
// The cost pass as a transposed chain from unit vectors.
//
// Trace entry c is (V U)[rho, c] with rho = c + trace_off and V = F_{nb-1} ... F_0: row
// rho of V dotted with column c of U.  Row rho of V is column rho of
// V^T = F_0^T F_1^T ... F_{nb-1}^T, which this kernel builds from the unit vector
// e_rho: F_{nb-1}^T e_rho is row rho of F_{nb-1} on the rows that agree with rho
// outside the block's qubits (loaded, no arithmetic), and each later block only touches
// the rows that agree with rho outside the union S_b of the qubits seen so far (the
// support): 2^(|S_b| - 4) of a column's 2^N / 16 outer groups.  The 8-qubit 40-layer
// ansatz's chain has supports of 4, 7, 7, 8, 8, 8 qubits: 4 block products of work,
// where the forward pass over U's columns needs 5; the 10-qubit 60-layer ansatz's 9
// blocks need 6.25 instead of 8.  The last block's output is multiplied elementwise
// with column c of U and summed.
//
// Layout as k_fused_cost: a wavefront owns W = 16 T / O columns; block b's vector
// column n holds column w = n >> lg_b, support group k = n & (2^lg_b - 1), rows
// kb_b[k] | (rho_w & nS_b) | off_b[i] (kTraceMapStride ints per block: off[16],
// kb[64], lg, nS).  Only the first ceil(W 2^lg_b / 16) tiles carry work.  Rows outside
// the support are never stored: the region starts at zero, and since the supports only
// grow they read as zero until a block reaches them.  Every launch shape performs the same operations per column in the
// same order: results are bit-identical across shapes.

// The chain's regions are padded below 8 qubits, where a tile's 16 vector columns are of
// several columns (5 blocks on 5 qubits, 4096 vectors: 45 us in complex128, 27 in complex64;
// unpadded 61 and 33).
constexpr bool ft_padded(int N) { return N < 8; }

template <typename R, int N, int T, bool PF>
__global__ __launch_bounds__(256, 2) void k_fused_trace(FusedCostArgs a, const int* __restrict__ tabs,
                                                        const int* __restrict__ tmaps) {
    typedef FcMfma<R> MF;
    typedef FcRegion<R, N, T, ft_padded(N)> Reg;
    constexpr int O = Reg::O, W = Reg::W;
    static_assert(W >= 1, "a wavefront holds whole columns");
    extern __shared__ __align__(16) unsigned char fc_smem[];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long long per_xcd = gridDim.x >> 3;  // the grid is a multiple of 8
    const long long lwg = (long long)(blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    const long long wave = lwg * (blockDim.x >> 6) + wv;
    if (wave >= (long long)a.B * a.groups) return;
    const int e = (int)(wave / a.groups);
    const int c0 = (int)(wave % a.groups) * W;
    const Reg lds{reinterpret_cast<R*>(fc_smem) + wv * 2 * Reg::PL};
    const int nl = lane & 15, g = lane >> 4;
    const int m = a.m;
    const cpx<R>* Fe = static_cast<const cpx<R>*>(a.F) + (long long)e * a.F_bstride;
    R xr[T][4], xi[T][4];
    FcA<R> A;
    fused_chain_to_block0<R, N, T, PF, Reg>(tabs, tmaps, a.nb, lds, Fe, c0, m, a.trace_off, lane, xr, xi, A);
    // block 0, then row rho of V times column c of U: per lane its rows of the column,
    // then the lanes of the column
    typename MF::V yr[T], yi[T];
    fc_mma<R, T, T>(A, xr, xi, yr, yi);  // (a support short of the register leaves zeros in the last tiles)
    const cpx<R>* U =
        static_cast<const cpx<R>*>(a.U) + (a.in_index ? (long long)a.in_index[e] : (long long)e) * a.in_bstride;
    const unsigned ist = (unsigned)a.in_stride;
    const int lg0 = tabs[LT_LG];
    double* dg = a.diag + 2 * ((long long)e * m + c0);
    if (lg0 == N - 4) {
        // vector column 16 t + nl is column (16 t + nl) / O; its rows' offsets in U fit 32
        // bits (at most 1024 x 1024 entries)
        constexpr int C = O > 16 ? W : T;  // sums: per column, or per tile of whole columns
        double sr[C], si[C];
#pragma unroll
        for (int c = 0; c < C; ++c) sr[c] = si[c] = 0;
        const unsigned row0 = (unsigned)tabs[LT_ROW + lane] * ist;
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const int c = O > 16 ? t / (O / 16 ? O / 16 : 1) : t;
            const int col = c0 + (O > 16 ? c : (16 * t + nl) / O);
            const unsigned at = row0 + (unsigned)tabs[LT_RT + t] * ist + (unsigned)(col < m ? col : 0);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const cpx<R> u = U[at + (unsigned)tabs[LT_RS + r] * ist];
                sr[c] += (double)yr[t][r] * (double)u.re - (double)yi[t][r] * (double)u.im;
                si[c] += (double)yr[t][r] * (double)u.im + (double)yi[t][r] * (double)u.re;
            }
        }
        fc_column_sums<N, T>(sr, si, dg, c0, m, lane);
        return;
    }
    // blocks that leave qubits out: the support layout of block 0, rows outside the support
    // those of rho
    const int* mp = tmaps;
    const int nS = mp[81], ng = 1 << lg0, seg = ng < 16 ? ng : 16;
    const int ts = ((W << lg0) + 15) >> 4;
    double sr = 0, si = 0;
#pragma unroll
    for (int t = 0; t < T; ++t) {
        if (t < ts) {
            const int n = 16 * t + nl, w = n >> lg0, col = c0 + w;
            if (w < W && col < m) {
                const int base = mp[16 + (n & (ng - 1))] | ((col + a.trace_off) & nS);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const cpx<R> u = U[(unsigned)(base + mp[4 * r + g]) * ist + (unsigned)col];
                    sr += (double)yr[t][r] * (double)u.re - (double)yi[t][r] * (double)u.im;
                    si += (double)yr[t][r] * (double)u.im + (double)yi[t][r] * (double)u.re;
                }
            }
            if (lg0 < 4 || (((t + 1) << 4) & (ng - 1)) == 0) {
                sr += __shfl_xor(sr, 16, 64);
                si += __shfl_xor(si, 16, 64);
                sr += __shfl_xor(sr, 32, 64);
                si += __shfl_xor(si, 32, 64);
#pragma unroll
                for (int d = 1; d < 16; d <<= 1) {
                    if (d < seg) {
                        sr += __shfl_xor(sr, d, 64);
                        si += __shfl_xor(si, d, 64);
                    }
                }
                if (g == 0 && (nl & (seg - 1)) == 0 && w < W && col < m) {
                    dg[2 * w] = sr;
                    dg[2 * w + 1] = si;
                }
                sr = 0;
                si = 0;
            }
        }
    }
}

bool fused_trace_cfg_valid(int N, bool f32, int nb, FusedCostCfg cfg) {
    if (N < 4 || N > kFusedCostMaxQubits || nb < 2) return false;
    if ((cfg.tiles != 2 && cfg.tiles != 4) || cfg.groups != 1) return false;
    if (cfg.waves != 1 && cfg.waves != 2 && cfg.waves != 4) return false;
    if (16 * cfg.tiles < ((1 << N) >> 4)) return false;
    return fused_trace_lds_bytes(f32, N, cfg) <= device_max_lds();
}

size_t fused_trace_lds_bytes(bool f32, int N, FusedCostCfg cfg) {
    return (size_t)cfg.waves * 2 * fc_plane(N, cfg.tiles, ft_padded(N)) * (f32 ? 4 : 8);
}

template <typename R, int N>
static void launch_ft_n(const FusedCostArgs& a, FusedCostCfg cfg, int grid, size_t shm, hipStream_t s) {
    const int threads = 64 * cfg.waves;
    if constexpr (16 * 4 >= ((1 << N) >> 4)) {
        if (cfg.tiles == 4 && cfg.prefetch)
            hipLaunchKernelGGL((k_fused_trace<R, N, 4, true>), dim3(grid), dim3(threads), shm, s, a, a.tabs, a.maps);
        else if (cfg.tiles == 4)
            hipLaunchKernelGGL((k_fused_trace<R, N, 4, false>), dim3(grid), dim3(threads), shm, s, a, a.tabs, a.maps);
    }
    if constexpr (16 * 2 >= ((1 << N) >> 4)) {
        if (cfg.tiles == 2 && cfg.prefetch)
            hipLaunchKernelGGL((k_fused_trace<R, N, 2, true>), dim3(grid), dim3(threads), shm, s, a, a.tabs, a.maps);
        else if (cfg.tiles == 2)
            hipLaunchKernelGGL((k_fused_trace<R, N, 2, false>), dim3(grid), dim3(threads), shm, s, a, a.tabs, a.maps);
    }
}

template <typename R>
static hipError_t launch_ft(int N, const FusedCostArgs& a, FusedCostCfg cfg, int grid, size_t shm, hipStream_t s) {
    switch (N) {
    case 4: launch_ft_n<R, 4>(a, cfg, grid, shm, s); break;
    case 5: launch_ft_n<R, 5>(a, cfg, grid, shm, s); break;
    case 6: launch_ft_n<R, 6>(a, cfg, grid, shm, s); break;
    case 7: launch_ft_n<R, 7>(a, cfg, grid, shm, s); break;
    case 8: launch_ft_n<R, 8>(a, cfg, grid, shm, s); break;
    case 9: launch_ft_n<R, 9>(a, cfg, grid, shm, s); break;
    case 10: launch_ft_n<R, 10>(a, cfg, grid, shm, s); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_fused_trace(bool f32, int N, FusedCostArgs a, FusedCostCfg cfg, hipStream_t s) {
    if (a.nb < 2 || a.m <= 0 || a.B <= 0 || a.out || !fused_trace_cfg_valid(N, f32, a.nb, cfg))
        return hipErrorInvalidValue;
    if (a.in_stride < a.m || a.trace_off < 0 || a.trace_off + a.m > (1 << N)) return hipErrorInvalidValue;
    const int W = 16 * cfg.tiles / ((1 << N) >> 4);
    a.groups = (a.m + W - 1) / W;
    const long long waves = (long long)a.B * a.groups;
    const long long wgs = (waves + cfg.waves - 1) / cfg.waves;
    const int grid = (int)((wgs + 7) / 8 * 8);
    const size_t shm = fused_trace_lds_bytes(f32, N, cfg);
    return f32 ? launch_ft<float>(N, a, cfg, grid, shm, s) : launch_ft<double>(N, a, cfg, grid, shm, s);
}

bool fused_cost_cfg_valid(int N, bool f32, int nb, FusedCostCfg cfg) {
    if (N < 4 || N > kFusedCostMaxQubits) return false;
    const int O = (1 << N) >> 4;
    if (!((cfg.tiles == 4 && cfg.groups == 1) || (cfg.tiles == 4 && cfg.groups == 2 && cfg.prefetch) ||
          (cfg.tiles == 2 && cfg.groups == 1)))
        return false;
    if (cfg.waves != 1 && cfg.waves != 2 && cfg.waves != 4) return false;
    if (16 * cfg.tiles < O || (16 * cfg.tiles / cfg.groups) % O != 0) return false;
    return fused_cost_lds_bytes(f32, N, cfg) <= device_max_lds();
}

size_t fused_cost_lds_bytes(bool f32, int N, FusedCostCfg cfg) {
    return (size_t)cfg.waves * 2 * fc_plane(N, cfg.tiles, true) * (f32 ? 4 : 8);
}

template <typename R, int N, int T, int H, bool PF>
static void launch_fc_shape(const FusedCostArgs& a, int grid, int threads, size_t shm, hipStream_t s) {
    if constexpr (16 * T >= ((1 << N) >> 4) && (16 * T / H) % ((1 << N) >> 4) == 0)
        hipLaunchKernelGGL((k_fused_cost<R, N, T, H, PF>), dim3(grid), dim3(threads), shm, s, a, a.tabs);
}

template <typename R, int N>
static void launch_fc_n(const FusedCostArgs& a, FusedCostCfg cfg, int grid, size_t shm, hipStream_t s) {
    const int threads = 64 * cfg.waves;
    if (cfg.tiles == 4 && cfg.groups == 2) launch_fc_shape<R, N, 4, 2, true>(a, grid, threads, shm, s);
    else if (cfg.tiles == 4 && cfg.prefetch) launch_fc_shape<R, N, 4, 1, true>(a, grid, threads, shm, s);
    else if (cfg.tiles == 4) launch_fc_shape<R, N, 4, 1, false>(a, grid, threads, shm, s);
    else if (cfg.prefetch) launch_fc_shape<R, N, 2, 1, true>(a, grid, threads, shm, s);
    else launch_fc_shape<R, N, 2, 1, false>(a, grid, threads, shm, s);
}

template <typename R>
static hipError_t launch_fc(int N, const FusedCostArgs& a, FusedCostCfg cfg, int grid, size_t shm, hipStream_t s) {
    switch (N) {
    case 4: launch_fc_n<R, 4>(a, cfg, grid, shm, s); break;
    case 5: launch_fc_n<R, 5>(a, cfg, grid, shm, s); break;
    case 6: launch_fc_n<R, 6>(a, cfg, grid, shm, s); break;
    case 7: launch_fc_n<R, 7>(a, cfg, grid, shm, s); break;
    case 8: launch_fc_n<R, 8>(a, cfg, grid, shm, s); break;
    case 9: launch_fc_n<R, 9>(a, cfg, grid, shm, s); break;
    case 10: launch_fc_n<R, 10>(a, cfg, grid, shm, s); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_fused_cost(bool f32, int N, FusedCostArgs a, FusedCostCfg cfg, hipStream_t s) {
    if (a.nb <= 0 || a.m <= 0 || a.B <= 0 || !fused_cost_cfg_valid(N, f32, a.nb, cfg)) return hipErrorInvalidValue;
    if (a.in_stride < a.m || (a.out && a.out_stride < a.m)) return hipErrorInvalidValue;
    const int W = 16 * cfg.tiles / ((1 << N) >> 4);
    a.groups = (a.m + W - 1) / W;
    const long long waves = (long long)a.B * a.groups;
    const long long wgs = (waves + cfg.waves - 1) / cfg.waves;
    const int grid = (int)((wgs + 7) / 8 * 8);
    const size_t shm = fused_cost_lds_bytes(f32, N, cfg);
    return f32 ? launch_fc<float>(N, a, cfg, grid, shm, s) : launch_fc<double>(N, a, cfg, grid, shm, s);
}

}  // namespace sqh
