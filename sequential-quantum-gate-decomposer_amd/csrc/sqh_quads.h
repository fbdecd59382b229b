// sqh_quads.h -- 16-row vectors held four rows to a lane, and the gates on them (the block
// kernels' walks and the persistent solver's evaluations on 3 and 4 qubits).
//
// A wavefront holds 16 columns of 16 rows: lane = column + 16 z has the quad of rows that
// differ in two qubits (a, b), z numbering the other two.  Gates on a and b work on the
// lane's own four values; a change of the pair takes the rows through LDS once.  The host
// orders the gates into runs per pair (quad_ops).
#pragma once
#include "sqh_device.h"

namespace sqh {

template <typename R>
__device__ __forceinline__ cpx<double> widen(cpx<R> a) {
    return mk((double)a.re, (double)a.im);
}

__device__ __forceinline__ void quad_fence() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); }

// Rows of the lane's quad for the pair in an op word: row0 | (k & 1 ? u : 0) | (k & 2 ? v : 0).
struct QuadRows {
    int row0, u, v;
};
__device__ __forceinline__ QuadRows quad_rows(uint32_t pair, int z) {
    const int qa = pair & 3, qb = pair >> 2;
    const int rest = 15 ^ (1 << qa) ^ (1 << qb);
    const int c = __builtin_ctz(rest), d = 31 - __builtin_clz(rest);
    return {((z & 1) << c) | ((z >> 1) << d), 1 << qa, 1 << qb};
}
__device__ __forceinline__ int quad_row(const QuadRows& q, int k) {
    return q.row0 | ((k & 1) ? q.u : 0) | ((k & 2) ? q.v : 0);
}

template <typename R>
__device__ __forceinline__ void quad_store(const cpx<R> (&v)[4], const QuadRows& q, int col, cpx<R>* s) {
#pragma unroll
    for (int k = 0; k < 4; ++k) s[quad_row(q, k) * 16 + col] = v[k];
}
template <typename R>
__device__ __forceinline__ void quad_load(cpx<R> (&v)[4], const QuadRows& q, int col, const cpx<R>* s) {
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = s[quad_row(q, k) * 16 + col];
}

template <typename R>
__device__ __forceinline__ void quad_pair(cpx<R>& x0, cpx<R>& x1, const cpx<R> (&k)[4]) {
    const cpx<R> a = mac2(k[0], x0, k[1], x1), b = mac2(k[2], x0, k[3], x1);
    x0 = a;
    x1 = b;
}

template <typename R>
__device__ __forceinline__ void quad_swap(cpx<R>& a, cpx<R>& b) {
    const cpx<R> t = a;
    a = b;
    b = t;
}

// A gate backwards on a pair of rows: x <- G^dagger x, acc += y x^T, y <- G^T y.
template <typename R>
__device__ __forceinline__ void quad_back(cpx<R>& x0, cpx<R>& x1, cpx<R>& y0, cpx<R>& y1, const cpx<R> (&kd)[4],
                                          const cpx<R> (&kt)[4], cpx<R> (&acc)[4]) {
    quad_pair(x0, x1, kd);
    cacc(acc[0], y0, x0);
    cacc(acc[1], y0, x1);
    cacc(acc[2], y1, x0);
    cacc(acc[3], y1, x1);
    quad_pair(y0, y1, kt);
}

// Sums of eight values over the wavefront: on return lanes 0, 16, 32, 48 hold the sums of
// values {0, 2, 1, 3} in lo and of values {4, 6, 5, 7} in hi.  The first two steps halve
// the values held per lane while they add across lane halves and rows
// (lane_halves), so eight sums take 42 instructions where a butterfly for each takes 144.
__device__ __forceinline__ void wave_sum8(const double (&r)[8], double& lo, double& hi) {
    double s[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) s[i] = lane_halves(r[2 * i], r[2 * i + 1], false);
    lo = row_sum(lane_halves(s[0], s[1], true));
    hi = row_sum(lane_halves(s[2], s[3], true));
}

}  // namespace sqh
