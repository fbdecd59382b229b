// sqh_k_block_gates.hip -- the gates inside the fused 4-qubit blocks: the blocks' 16 x 16
// matrices (k_fuse_blocks) and, for the gradient, each gate's 2 x 2 correlations from its
// block's 16 x 16 correlation (k_fused_block_corr).
//
// Both walk a block's gates on 16-row vectors, one wavefront per (block, element), with
// the 16 columns' 256 entries as 4 rows per lane: lane = column + 16 z holds the quad of
// rows that differ in the two qubits (a, b) a run of gates acts on, z numbering the other
// two qubits.  Gates on a and b, CNOTs between them included, work on the lane's own four
// values; when the pair changes, the rows go through LDS once.  The host orders a block's
// gates into runs per pair (quad_ops): a run of a CNOT layer is the CNOT and two U3.
//
// What bounds these kernels is latency (a block has some twenty dependent gates), so the
// code that a gate runs is kept short enough to stay in the instruction cache: the same
// few operations for every pair, where a walk with every target and control of a 16-row
// register column unrolled took 27 us a block build and 74 us a correlation walk with the
// partials' sum (8 qubits, one element; 30 and 100 for 512).  Now 13 and 28 (16 and 36),
// with the kernel table's launch gone: gradient of one 8-qubit vector 209 -> 95 us.
// Both compute in FP64 in either precision: a complex64 block matrix is then rounded once,
// not after each of its gates.
#include <hip/hip_runtime.h>

#include "sqh_device.h"
#include "sqh_kernels.h"
#include "sqh_quads.h"

namespace sqh {

namespace {

// The 2 x 2 kernels of a chunk's gates for one element into tab[gate][4], a gate per lane:
// computed from the element's parameters, or taken from the element's kernel table.
// Gate dslot gets its derivative with respect to its parameter dparam.
template <typename R>
__device__ __forceinline__ void quad_stage(uint32_t w, bool live, const cpx<R>* kern, const double* params,
                                           const Slot* slots, int lane, cpx<double>* tab, int dslot = -1,
                                           int dparam = 0) {
    const int slot = (int)(w >> kQuadSlotShift) - 1;
    if (live && slot >= 0) {
        if (params) {
            const Slot sl = slots[slot];
            cpx<double> k4[4];
            if (slot == dslot) dev_deriv_kernel(sl.type, params + sl.param_start, dparam, k4);
            else dev_gate_kernel(sl.type, params + sl.param_start, k4);
#pragma unroll
            for (int k = 0; k < 4; ++k) tab[4 * lane + k] = k4[k];
        } else {
#pragma unroll
            for (int k = 0; k < 4; ++k) tab[4 * lane + k] = widen(kern[4 * slot + k]);
        }
    }
}

}  // namespace

constexpr int kQuadWaves = 4;  // elements per workgroup of the block build

// A wavefront per (block, element); DERIV: per block of the one parameter vector, then per
// parameter with its gate differentiated (launch_fuse_deriv_blocks; B is nb + P then).
template <typename R, bool DERIV>
__global__ __launch_bounds__(64 * kQuadWaves) void k_fuse_blocks(const uint32_t* __restrict__ ops,
                                                                 const int* __restrict__ first, int nb,
                                                                 const cpx<R>* __restrict__ kern,
                                                                 long long kern_bstride,
                                                                 const double* __restrict__ params, int pstride,
                                                                 const Slot* __restrict__ slots, int B,
                                                                 cpx<R>* __restrict__ out,
                                                                 const int* __restrict__ count,
                                                                 const int* __restrict__ dinfo) {
    __shared__ cpx<double> state[kQuadWaves][256];
    __shared__ cpx<double> table[kQuadWaves][64 * 4];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int e = (DERIV ? blockIdx.x : blockIdx.x / nb) * kQuadWaves + wave;
    if (count) B = min(*count, B);  // live elements (the optimiser's rounds)
    if (e >= B) return;             // the whole wavefront; the waves share nothing
    int blk = DERIV ? e : blockIdx.x % nb, dslot = -1, dparam = 0;
    bool zero = false;  // the differentiated gate is controlled: its control-0 rows become zero
    if (DERIV && e >= nb) {
        const int* d = dinfo + 4 * (e - nb);
        blk = __builtin_amdgcn_readfirstlane(d[0]);
        dslot = __builtin_amdgcn_readfirstlane(d[1]);
        dparam = d[2];
        zero = d[3] != 0;
    }
    const int col = lane & 15, z = lane >> 4;
    cpx<double>* s = state[wave];
    cpx<double>* tab = table[wave];
    const int p0 = first[blk], p1 = first[blk + 1];
    uint32_t pair = 4;  // qubits 0 and 1
    QuadRows q = quad_rows(pair, z);
    cpx<double> v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = mk(quad_row(q, k) == col ? 1.0 : 0.0, 0.0);
    for (int p = p0; p < p1; p += 64) {
        const int cnt = min(64, p1 - p);
        const uint32_t w = lane < cnt ? ops[p + lane] : 0;
        quad_fence();  // the previous chunk's table is read
        quad_stage<R>(w, lane < cnt, kern + e * kern_bstride, params ? params + (long long)e * pstride : nullptr, slots,
                      lane, tab, dslot, dparam);
        quad_fence();
        for (int i = 0; i < cnt; ++i) {
            const uint32_t op = __builtin_amdgcn_readlane(w, i);
            const uint32_t pr = (op >> kQuadPairShift) & 15;
            cpx<double> k[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) k[t] = tab[4 * i + t];
            if (pr != pair) {
                quad_store(v, q, col, s);
                quad_fence();
                pair = pr;
                q = quad_rows(pair, z);
                quad_load(v, q, col, s);
                quad_fence();
            }
            switch (op & 15) {
            case QK_UA:
                quad_pair(v[0], v[1], k);
                quad_pair(v[2], v[3], k);
                break;
            case QK_UB:
                quad_pair(v[0], v[2], k);
                quad_pair(v[1], v[3], k);
                break;
            case QK_XA: quad_swap(v[2], v[3]); break;
            case QK_XB: quad_swap(v[1], v[3]); break;
            case QK_Z: v[3] = mk(-v[3].re, -v[3].im); break;
            case QK_CUA:
                quad_pair(v[2], v[3], k);
                if (zero && (int)(op >> kQuadSlotShift) - 1 == dslot) v[0] = v[1] = mk(0.0, 0.0);
                break;
            default:  // QK_CUB
                quad_pair(v[1], v[3], k);
                if (zero && (int)(op >> kQuadSlotShift) - 1 == dslot) v[0] = v[2] = mk(0.0, 0.0);
                break;
            }
        }
    }
    cpx<R>* o = out + (DERIV ? (long long)e : (long long)e * nb + blk) * 256;  // [row][col]
#pragma unroll
    for (int k = 0; k < 4; ++k) o[quad_row(q, k) * 16 + col] = cvt<R>(v[k]);
}

// Entries M, M + step, ... of C partials (the first `left` of them, the others count as
// zero), each entry's added as a binary tree.
template <int C, int E>
__device__ __forceinline__ void partial_nodes(const double* __restrict__ M, unsigned stride, int left, int step,
                                              double (&v)[E]) {
    double t[E][C];
#pragma unroll
    for (int k = 0; k < C; ++k)
#pragma unroll
        for (int i = 0; i < E; ++i) {
            const double x = M[(k < left ? k : 0) * stride + i * step];
            t[i][k] = k < left ? x : 0.0;
        }
#pragma unroll
    for (int w = 1; w < C; w *= 2)
#pragma unroll
        for (int k = 0; k < C; k += 2 * w)
#pragma unroll
            for (int i = 0; i < E; ++i) t[i][k] += t[i][k + w];
#pragma unroll
    for (int i = 0; i < E; ++i) v[i] = t[i][0];
}

// Sums over an element's n partials, 1 << up of them per chunk: FusedGradSplit's tree from
// the partials' level on, then its chunks in order.
template <int E>
__device__ __forceinline__ void partial_sum(const double* __restrict__ M, unsigned stride, int n, int up, int step,
                                            double (&out)[E]) {
    constexpr int C = 16;  // partials at a time; 64 of one entry leave a CU one workgroup
#pragma unroll
    for (int i = 0; i < E; ++i) out[i] = 0.0;
    for (int c = 0; c < n; c += 1 << up) {
        const int left = min(1 << up, n - c);
        const double* P = M + (long long)c * stride;
        double v[E];
        if (left <= 4) {
            partial_nodes<4>(P, stride, left, step, v);
        } else if (left <= 16) {
            partial_nodes<16>(P, stride, left, step, v);
        } else {
            double s[128 / C][E];
#pragma unroll
            for (int j = 0; j < 128 / C; ++j) {
                if (C * j < left) {
                    partial_nodes<C>(P + C * j * stride, stride, left - C * j, step, s[j]);
                } else {
#pragma unroll
                    for (int i = 0; i < E; ++i) s[j][i] = 0.0;
                }
            }
#pragma unroll
            for (int w = 1; w < 128 / C; w *= 2)
#pragma unroll
                for (int j = 0; j < 128 / C; j += 2 * w)
#pragma unroll
                    for (int i = 0; i < E; ++i) s[j][i] += s[j + w][i];
#pragma unroll
            for (int i = 0; i < E; ++i) v[i] = s[0][i];
        }
#pragma unroll
        for (int i = 0; i < E; ++i) out[i] += v[i];
    }
}

// Sums the partials of the block's correlation M_b (SPLIT: a workgroup per (block,
// element), an entry per thread, then only the first wavefront goes on; else a wavefront per
// (block, element), four elements per workgroup), starts from x = the
// columns of F_b and y = the columns of M_b and walks the gates backwards: x <- G^dagger x,
// the pair correlations of y and x summed over the wavefront, y <- G^T y.  Two workgroups per
// CU with SPLIT (564 workgroups on 5 qubits: 25.2 us against 26.6 with one), three else.
// corr[e][slot][8] is the register-tile adjoint's layout.
template <typename R, bool SPLIT>
__global__ __launch_bounds__(SPLIT ? 512 : 256, SPLIT ? 4 : 3) void k_fused_block_corr(const uint32_t* __restrict__ ops,
                                                          const int* __restrict__ first, int nb,
                                                          const cpx<R>* __restrict__ kern, long long kern_bstride,
                                                          const double* __restrict__ params, int pstride,
                                                          const Slot* __restrict__ slots, const cpx<R>* __restrict__ F,
                                                          const double* __restrict__ mpart, FusedGradSplit sp, int T,
                                                          int B, double* __restrict__ corr, int ns,
                                                          const int* __restrict__ count) {
    constexpr int E = SPLIT ? 1 : 4;  // elements per workgroup
    // M_b (256 real, then 256 imaginary parts) waits where x and y change pairs once it is
    // read: 48 KiB a workgroup, three per CU (two with a buffer of its own; 512 elements of
    // 6 blocks: 36 us against 46)
    __shared__ cpx<double> states[E][512], tables[E][64 * 4];
    double* const sums = reinterpret_cast<double*>(states[SPLIT ? 0 : threadIdx.x >> 6]);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int blk = blockIdx.x % nb, e = (blockIdx.x / nb) * E + (SPLIT ? 0 : wave);
    if (count) {
        B = min(*count, B);
        fused_grad_split_live(sp, B, T);
    }
    if (e >= B) return;  // the whole workgroup, or a wavefront that shares nothing
    {
        const int l = e < sp.n0 ? sp.l0 : sp.l1, n = fused_grad_tasks(sp.groups, l);
        const long long before = (long long)min(e, sp.n0) * fused_grad_tasks(sp.groups, sp.l0) +
                                 (long long)max(e - sp.n0, 0) * n;
        const double* M = mpart + (before * nb + blk) * 512;
        const unsigned stride = (unsigned)nb * 512;  // 128 partials within 32 bits
        const int up = fused_grad_levels(T) - l;
        if constexpr (SPLIT) {
            double v[1];
            partial_sum(M + threadIdx.x, stride, n, up, 0, v);
            sums[threadIdx.x] = v[0];
            __syncthreads();
            if (wave != 0) return;
        } else {
            double* s = sums + lane;
            M += lane;
            if (n <= 4 && n <= 1 << up) {
                double v[8];
                if (n == 1) partial_nodes<1>(M, stride, 1, 64, v);
                else partial_nodes<4>(M, stride, n, 64, v);
#pragma unroll
                for (int i = 0; i < 8; ++i) s[64 * i] = v[i];
            } else {
#pragma unroll 1
                for (int i = 0; i < 8; i += 2) {
                    double v[2];
                    partial_sum(M + 64 * i, stride, n, up, 64, v);
                    s[64 * i] = v[0];
                    s[64 * i + 64] = v[1];
                }
            }
            quad_fence();
        }
    }
    const int col = lane & 15, z = lane >> 4;
    cpx<double>* sx = states[SPLIT ? 0 : wave];
    cpx<double>* sy = sx + 256;
    cpx<double>* tab = tables[SPLIT ? 0 : wave];
    const cpx<R>* Fb = F + ((long long)e * nb + blk) * 256;
    const int p0 = first[blk], p1 = first[blk + 1];
    uint32_t pair = 4;
    QuadRows q = quad_rows(pair, z);
    cpx<double> x[4], y[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int at = quad_row(q, k) * 16 + col;
        x[k] = widen(Fb[at]);
        y[k] = mk(sums[at], sums[256 + at]);
    }
    for (int pe = p1; pe > p0; pe -= 64) {
        const int p = max(p0, pe - 64), cnt = pe - p;
        const uint32_t w = lane < cnt ? ops[p + lane] : 0;
        quad_fence();
        quad_stage<R>(w, lane < cnt, kern + e * kern_bstride, params ? params + (long long)e * pstride : nullptr, slots,
                      lane, tab);
        quad_fence();
        for (int i = cnt - 1; i >= 0; --i) {
            const uint32_t op = __builtin_amdgcn_readlane(w, i);
            const uint32_t pr = (op >> kQuadPairShift) & 15;
            cpx<double> k[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) k[t] = tab[4 * i + t];
            if (pr != pair) {
                quad_store(x, q, col, sx);
                quad_store(y, q, col, sy);
                quad_fence();
                pair = pr;
                q = quad_rows(pair, z);
                quad_load(x, q, col, sx);
                quad_load(y, q, col, sy);
                quad_fence();
            }
            const cpx<double> kd[4] = {mk(k[0].re, -k[0].im), mk(k[2].re, -k[2].im), mk(k[1].re, -k[1].im),
                                  mk(k[3].re, -k[3].im)};
            const cpx<double> kt[4] = {k[0], k[2], k[1], k[3]};
            cpx<double> acc[4] = {mk(0.0, 0.0), mk(0.0, 0.0), mk(0.0, 0.0), mk(0.0, 0.0)};
            // CNOT and CZ are their own adjoint and transpose
            switch (op & 15) {
            case QK_UA:
                quad_back(x[0], x[1], y[0], y[1], kd, kt, acc);
                quad_back(x[2], x[3], y[2], y[3], kd, kt, acc);
                break;
            case QK_UB:
                quad_back(x[0], x[2], y[0], y[2], kd, kt, acc);
                quad_back(x[1], x[3], y[1], y[3], kd, kt, acc);
                break;
            case QK_CUA: quad_back(x[2], x[3], y[2], y[3], kd, kt, acc); break;
            case QK_CUB: quad_back(x[1], x[3], y[1], y[3], kd, kt, acc); break;
            case QK_XA:
                quad_swap(x[2], x[3]);
                quad_swap(y[2], y[3]);
                continue;
            case QK_XB:
                quad_swap(x[1], x[3]);
                quad_swap(y[1], y[3]);
                continue;
            default:  // QK_Z
                x[3] = mk(-x[3].re, -x[3].im);
                y[3] = mk(-y[3].re, -y[3].im);
                continue;
            }
            double r[8], lo, hi;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                r[2 * t] = acc[t].re;
                r[2 * t + 1] = acc[t].im;
            }
            wave_sum8(r, lo, hi);
            if (col == 0) {
                double* d = corr + ((long long)e * ns + (int)(op >> kQuadSlotShift) - 1) * 8;
                const int at = ((z & 1) << 1) | (z >> 1);  // values 0, 2, 1, 3 for z = 0 .. 3
                d[at] = lo;
                d[4 + at] = hi;
            }
        }
    }
}

hipError_t launch_fuse_blocks(bool f32, const uint32_t* ops, const int* first, int nb, const GateKernels& g, int B,
                              void* out, hipStream_t s, const int* count) {
    if ((long long)B * nb == 0) return hipSuccess;
    const unsigned grid = (unsigned)(nb * (long long)((B + kQuadWaves - 1) / kQuadWaves));
    if (f32)
        hipLaunchKernelGGL((k_fuse_blocks<float, false>), dim3(grid), dim3(64 * kQuadWaves), 0, s, ops, first, nb,
                           (const cpx<float>*)g.kern, g.kern_bstride, g.params, g.pstride, g.slots, B, (cpx<float>*)out,
                           count, nullptr);
    else
        hipLaunchKernelGGL((k_fuse_blocks<double, false>), dim3(grid), dim3(64 * kQuadWaves), 0, s, ops, first, nb,
                           (const cpx<double>*)g.kern, g.kern_bstride, g.params, g.pstride, g.slots, B,
                           (cpx<double>*)out, count, nullptr);
    return hipGetLastError();
}

hipError_t launch_fuse_deriv_blocks(const uint32_t* ops, const int* first, int nb, const double* params,
                                    const Slot* slots, const int* dinfo, int P, void* out, hipStream_t s) {
    const int n = nb + P;
    hipLaunchKernelGGL((k_fuse_blocks<double, true>), dim3((n + kQuadWaves - 1) / kQuadWaves), dim3(64 * kQuadWaves), 0,
                       s, ops, first, nb, (const cpx<double>*)nullptr, 0LL, params, 0, slots, n, (cpx<double>*)out,
                       (const int*)nullptr, dinfo);
    return hipGetLastError();
}

hipError_t launch_fused_block_corr(bool f32, const uint32_t* ops, const int* first, int nb, const GateKernels& g,
                                   const void* F, const double* mpart, const FusedGradSplit& sp, int T, int B,
                                   double* corr, int ns, hipStream_t s, const int* count) {
    if ((long long)B * nb == 0) return hipSuccess;
    // With a wavefront per SIMD's worth of (block, element) pairs each sums its own
    // partials; below that, as with one vector, the sum is the longer part and is split.
    const bool split = (long long)B * nb < 1024;
    const unsigned grid = (unsigned)(nb * (long long)(split ? B : (B + 3) / 4));
#define SQH_CORR(R, SP)                                                                                       \
    hipLaunchKernelGGL((k_fused_block_corr<R, SP>), dim3(grid), dim3(SP ? 512 : 256), 0, s, ops, first, nb,    \
                       (const cpx<R>*)g.kern, g.kern_bstride, g.params, g.pstride, g.slots, (const cpx<R>*)F,  \
                       mpart, sp, T, B, corr, ns, count)
    if (f32 && split) SQH_CORR(float, true);
    else if (f32) SQH_CORR(float, false);
    else if (split) SQH_CORR(double, true);
    else SQH_CORR(double, false);
#undef SQH_CORR
    return hipGetLastError();
}

}  // namespace sqh
