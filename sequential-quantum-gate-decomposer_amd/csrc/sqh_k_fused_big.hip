// sqh_k_fused_big.hip -- apply_to above the tile limit (11 to 13 qubits, 14 in complex64):
// the circuit as fused dense 4-qubit blocks on the matrix cores with whole columns resident
// in a workgroup's LDS, one read and one write of the matrices for all blocks.
//
// A column of 2^N complex entries is 32 to 128 KiB, beyond a wavefront's region, so the
// wavefronts of a workgroup share C columns: per block each takes its tiles of 16 groups of
// 16 rows, reads them, multiplies and writes them back to the same rows; one barrier
// separates the blocks.  Two workgroups of four wavefronts fit a CU where a column is at
// most 64 KiB, so that one's exchange and barrier are covered by the other's MFMAs, and one
// of eight where it is 128 KiB.  What bounds it is the FP64 (FP32) MFMA rate: at 12 qubits
// a matrix is 8 blocks x 128 flop per 32 bytes moved.  Streamed a block at a time
// (k_block_mfma4, one pass over HBM or the Infinity Cache each) 24 matrices of 48 columns
// took 182 us.
//
// Slots are linear over XOR in the row's bits, as in the kernels below 11 qubits
// (sqh_fused_chain.h): an address is the lane's entry XOR a uniform part of the step XOR a
// uniform part of the tile (BT_*, sqh_kernels.h).
#include <hip/hip_runtime.h>

#include "sqh_device.h"
#include "sqh_fused_chain.h"
#include "sqh_kernels.h"

namespace sqh {

namespace {

__host__ __device__ constexpr int big_slot(int j) { return j ^ (((j >> 4) ^ (j >> 8) ^ (j >> 12)) & 15); }

template <typename R, int N>
struct Big {
    static constexpr int D = 1 << N;
    static constexpr int kColBytes = D * 2 * (int)sizeof(R);
    static constexpr int C = kColBytes >= 65536 ? 1 : 65536 / kColBytes;  // columns per workgroup
    static constexpr int NW = kColBytes > 65536 ? 8 : 4;                  // wavefronts
    static constexpr int TW = (C << (N - 8)) / NW;                        // tiles per wavefront
    static constexpr int PL = C * D;                                      // entries per plane
    static_assert(TW % 4 == 0, "four tiles at a time");
};

}  // namespace

template <typename R, int N>
__global__ __launch_bounds__((64 * Big<R, N>::NW), 2) void k_fused_big(FusedCostArgs a, const int* __restrict__ tabs) {
    typedef FcMfma<R> MF;
    typedef Big<R, N> G;
    constexpr int D = G::D, C = G::C, PL = G::PL, threads = 64 * G::NW;
    extern __shared__ __align__(16) unsigned char fb_smem[];
    R* const s = reinterpret_cast<R*>(fb_smem);
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const long long lwg = (long long)(blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    const int e = (int)(lwg / a.groups);
    if (e >= a.B) return;  // the whole workgroup
    const int q = tid & (C - 1), row_q = tid / C, col = (int)(lwg % a.groups) * C + q;
    const bool ok = col < a.m;
    constexpr int RP = threads / C;  // rows per pass
    {
        const cpx<R>* p = static_cast<const cpx<R>*>(a.U) + (long long)e * a.in_bstride + (long long)row_q * a.in_stride + col;
        const long long step = (long long)RP * a.in_stride;
        // sixteen rows in flight per thread
        for (int k0 = 0; k0 < D / RP; k0 += 16) {
            cpx<R> u[16];
#pragma unroll
            for (int k = 0; k < 16; ++k) u[k] = ok ? p[(k0 + k) * step] : mk<R>(0, 0);
#pragma unroll
            for (int k = 0; k < 16; ++k) {
                const int at = big_slot(row_q + (k0 + k) * RP) + q * D;
                s[at] = u[k].re;
                s[at + PL] = u[k].im;
            }
        }
    }
    const int nl = lane & 15, g = lane >> 4;
    const cpx<R>* Fe = static_cast<const cpx<R>*>(a.F) + (long long)e * a.F_bstride;
    FcA<R> A;
    A.load_n(Fe, nl, g);
    const int* tab = tabs;
    int entry = tab[BT_LANE + lane];
    for (int b = 0; b < a.nb; ++b) {
        int at[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) at[r] = entry ^ tab[BT_S + r];
        __syncthreads();  // the columns, or the previous block's rows, are written
#pragma unroll
        for (int c = 0; c < G::TW / 4; ++c) {
            R xr[4][4], xi[4][4];
            typename MF::V yr[4], yi[4];
            int base[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int tile = wv * G::TW + 4 * c + t;
                base[t] = tab[BT_T + (tile & ((1 << (N - 8)) - 1))] ^ ((tile >> (N - 8)) * D);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    xr[t][r] = s[at[r] ^ base[t]];
                    xi[t][r] = s[(at[r] ^ base[t]) + PL];
                }
            }
            fc_wave_fence();
            fc_mma<R, 4, 4>(A, xr, xi, yr, yi);
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    s[at[r] ^ base[t]] = yr[t][r];
                    s[(at[r] ^ base[t]) + PL] = yi[t][r];
                }
            fc_wave_fence();
        }
        tab += kBigTab;
        if (b + 1 < a.nb) {
            A.load_n(Fe + (long long)(b + 1) * 256, nl, g);
            entry = tab[BT_LANE + lane];
        }
    }
    __syncthreads();
    if (ok) {
        cpx<R>* p = static_cast<cpx<R>*>(a.out) + (long long)e * a.out_bstride + (long long)row_q * a.out_stride + col;
        const long long step = (long long)RP * a.out_stride;
#pragma unroll 8
        for (int k = 0; k < D / RP; ++k) {
            const int at = big_slot(row_q + k * RP) + q * D;
            p[k * step] = mk<R>(s[at], s[at + PL]);
        }
    }
}

int fused_big_slot(int row) { return big_slot(row); }

bool fused_big_fits(bool f32, int N) {
    return N > kFusedCostMaxQubits && N <= (f32 ? 14 : 13) && ((size_t)(f32 ? 8 : 16) << N) <= device_max_lds() &&
           device_max_lds() >= 65536;
}

template <typename R, int N>
static hipError_t launch_big(FusedCostArgs a, hipStream_t s) {
    typedef Big<R, N> G;
    a.groups = (a.m + G::C - 1) / G::C;
    const long long wgs = ((long long)a.B * a.groups + 7) / 8 * 8;
    hipLaunchKernelGGL((k_fused_big<R, N>), dim3((unsigned)wgs), dim3(64 * G::NW), (size_t)G::C * G::kColBytes, s, a,
                       a.tabs);
    return hipGetLastError();
}

hipError_t launch_fused_big(bool f32, int N, const FusedCostArgs& a, hipStream_t s) {
    if (!fused_big_fits(f32, N) || a.nb <= 0 || a.m <= 0 || a.B <= 0 || !a.out || a.in_stride < a.m ||
        a.out_stride < a.m)
        return hipErrorInvalidValue;
    switch (N) {
    case 11: return f32 ? launch_big<float, 11>(a, s) : launch_big<double, 11>(a, s);
    case 12: return f32 ? launch_big<float, 12>(a, s) : launch_big<double, 12>(a, s);
    case 13: return f32 ? launch_big<float, 13>(a, s) : launch_big<double, 13>(a, s);
    default: return launch_big<float, 14>(a, s);
    }
}

}  // namespace sqh
