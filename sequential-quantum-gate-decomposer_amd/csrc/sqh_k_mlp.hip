// sqh_k_mlp.hip -- kernels of the warm-start network: a multilayer perceptron with
// BF16 weights/activations and FP32 accumulation on the gfx950 matrix cores
// (v_mfma_f32_16x16x32_bf16), GELU hidden layers, mean-squared-error loss and Adam.
//
// Every product is C[M][N] = sum_k A[m][k] B[n][k] with both operands K-contiguous:
// the layer outputs H and gradients dZ are written in both orders by the epilogue that
// produces them, and Adam keeps the transposed BF16 weights beside the plain ones, so
//   forward          H[l+1] = gelu(H[l] W^T + b):  A = H[l]  (rows = samples), B = W
//   data gradient    dZ[l-1] = (dZ[l] W) gelu'(Z): A = dZ[l],                  B = W^T
//   weight gradient  dW = dZ^T H:                  A = dZ[l]^T,                B = H[l]^T
// M, N and K are multiples of 64 (the host pads every dimension with zeros).
#include <hip/hip_runtime.h>

#include <cmath>

#include "sqh_mlp.h"

namespace sqh {

typedef __bf16 bf16;
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

enum MlpEpi : int {
    EPI_HIDDEN = 0,    // z = acc + bias -> Z, H = bf16(gelu(z)) -> H, H^T
    EPI_HIDDEN_ONLY,   // the same, H alone (no backward pass follows)
    EPI_OUTPUT,        // y = acc + bias -> the caller's B x out array
    EPI_MSE,           // y = acc + bias, dY = 2 (y - t) / (B out) -> dZ, dZ^T, FP32 dZ, loss
    EPI_BWD_DATA,      // dz = acc gelu'(Z) -> dZ, dZ^T, FP32 dZ
};

__device__ __forceinline__ float gelu(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }

__device__ __forceinline__ float gelu_grad(float z) {
    const float cdf = 0.5f * (1.0f + erff(z * 0.70710678118654752f));
    const float pdf = 0.39894228040143268f * expf(-0.5f * z * z);
    return cdf + z * pdf;
}

// The product of one TM x TN tile by a workgroup of 4 wavefronts, left in LDS.  Each
// wavefront computes a quarter of the tile over the whole K, every element as one FP32 sum
// in ascending K: a sum's bits depend neither on the tile size nor on the workgroup.  (K split
// over the wavefronts loads half as much and takes 8 us less of a training step of 112, but
// its sums round differently, and Adam's first steps carry that to 5e-4 of the weights.)
// Operands come straight from global memory into the MFMA operand registers (mlp_frag
// order): no LDS and no barrier in the loop, D steps of loads in flight per wavefront.  What
// bounds it is the operands' way from the L2: a CU takes 64 bytes a cycle, 3.4 us for K = 1024
// at 64 x 64.  1024 x 1024 x 1024 with its epilogue takes 11.3 us, 6.8 of them launch, first
// loads and the epilogue; the operands handed round through LDS, 12.4.
// A lane's result item r of tile (i, j) is C[16 i + 4 (lane / 16) + r][16 j + lane % 16] of
// its quarter.
constexpr int kPitch = 4;  // floats of padding per tile row

template <int TM, int TN, int D>
__device__ __forceinline__ void mlp_product(const bf16* __restrict__ A, const bf16* __restrict__ B, int K, int m0,
                                            int n0, float* __restrict__ tile) {
    constexpr int I = TM / 32, J = TN / 32;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nl = lane & 15, g = lane >> 4;
    const int wm = (wave >> 1) * (TM / 2), wn = (wave & 1) * (TN / 2);
    const int S = K >> 5;  // 32-wide K steps
    const bf16* pa = A + (size_t)((m0 + wm) >> 4) * S * 512 + lane * 8;
    const bf16* pb = B + (size_t)((n0 + wn) >> 4) * S * 512 + lane * 8;
    f32x4 acc[I][J];
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
        for (int j = 0; j < J; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    bf16x8 a[D][I], b[D][J];
    auto load = [&](int d, int s) {
#pragma unroll
        for (int i = 0; i < I; ++i) a[d][i] = *reinterpret_cast<const bf16x8*>(pa + ((size_t)i * S + s) * 512);
#pragma unroll
        for (int j = 0; j < J; ++j) b[d][j] = *reinterpret_cast<const bf16x8*>(pb + ((size_t)j * S + s) * 512);
    };
#pragma unroll
    for (int d = 0; d < D; ++d)
        if (d < S) load(d, d);
    for (int s = 0; s < S; s += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            if (s + d < S) {
#pragma unroll
                for (int i = 0; i < I; ++i)
#pragma unroll
                    for (int j = 0; j < J; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[d][i], b[d][j], acc[i][j], 0, 0, 0);
                if (s + d + D < S) load(d, s + d + D);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
        for (int j = 0; j < J; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                tile[(wm + 16 * i + 4 * g + r) * (TN + kPitch) + wn + 16 * j + nl] = acc[i][j][r];
    __syncthreads();
}

// Threads of the epilogue and the 4 x 4 block of the tile each holds: rows 4 rg .. + 3,
// columns 4 cg .. + 3.
template <int TM, int TN>
__device__ __forceinline__ bool mlp_block(const float* __restrict__ tile, int& rg, int& cg, f32x4 (&v)[4]) {
    if (threadIdx.x >= TM * TN / 16) return false;
    rg = threadIdx.x / (TN / 4);
    cg = threadIdx.x % (TN / 4);
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = *reinterpret_cast<const f32x4*>(tile + (4 * rg + r) * (TN + kPitch) + 4 * cg);
    return true;
}

// A 4 x 4 block as BF16 into X (rows x cols) and, when XT is given, into its transpose.
__device__ __forceinline__ void mlp_store_bf16(const f32x4 (&v)[4], int row, int col, bf16* X, int cols, bf16* XT,
                                               int rows) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const bf16x4 h = {(bf16)v[r][0], (bf16)v[r][1], (bf16)v[r][2], (bf16)v[r][3]};
        *reinterpret_cast<bf16x4*>(&X[mlp_frag(row + r, col, cols)]) = h;
    }
    if (XT) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const bf16x4 h = {(bf16)v[0][c], (bf16)v[1][c], (bf16)v[2][c], (bf16)v[3][c]};
            *reinterpret_cast<bf16x4*>(&XT[mlp_frag(col + c, row, rows)]) = h;
        }
    }
}

template <int TM, int TN, int EPI>
__global__ __launch_bounds__(256, 2) void k_mlp_layer(MlpLayerArgs a) {
    __shared__ __align__(16) float tile[TM * (TN + kPitch)];
    const int m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
    mlp_product<TM, TN, (TM < 64 ? 16 : 12)>((const bf16*)a.A, (const bf16*)a.B, a.K, m0, n0, tile);
    int rg = 0, cg = 0;
    f32x4 v[4];
    const bool active = mlp_block<TM, TN>(tile, rg, cg, v);
    const int row = m0 + 4 * rg, col = n0 + 4 * cg;
    if constexpr (EPI == EPI_HIDDEN || EPI == EPI_HIDDEN_ONLY) {
        if (active) {
            const f32x4 bias = *reinterpret_cast<const f32x4*>(&a.bias[col]);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                v[r] += bias;
                if constexpr (EPI == EPI_HIDDEN)
                    *reinterpret_cast<f32x4*>(&a.Z[(size_t)(row + r) * a.N + col]) = v[r];
#pragma unroll
                for (int c = 0; c < 4; ++c) v[r][c] = gelu(v[r][c]);
            }
            mlp_store_bf16(v, row, col, (bf16*)a.X, a.N, EPI == EPI_HIDDEN ? (bf16*)a.XT : nullptr,
                           a.M);
        }
    } else if constexpr (EPI == EPI_OUTPUT) {
        if (active) {
            const f32x4 bias = *reinterpret_cast<const f32x4*>(&a.bias[col]);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                v[r] += bias;
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    if (row + r < a.batch && col + c < a.out) a.y[(size_t)(row + r) * a.out + col + c] = v[r][c];
            }
        }
    } else if constexpr (EPI == EPI_MSE) {
        double l = 0.0;
        if (active) {
            const f32x4 bias = *reinterpret_cast<const f32x4*>(&a.bias[col]);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                v[r] += bias;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    float gr = 0.f;
                    if (row + r < a.batch && col + c < a.out) {
                        const float d = v[r][c] - a.t[(size_t)(row + r) * a.out + col + c];
                        l += (double)d * d;
                        gr = 2.0f * d / ((float)a.batch * (float)a.out);
                    }
                    v[r][c] = gr;
                }
                *reinterpret_cast<f32x4*>(&a.Z[(size_t)(row + r) * a.N + col]) = v[r];
            }
            mlp_store_bf16(v, row, col, (bf16*)a.X, a.N, (bf16*)a.XT, a.M);
        }
        __shared__ double sh[4];
        for (int o = 32; o > 0; o >>= 1) l += __shfl_xor(l, o, 64);
        if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = l;
        __syncthreads();
        if (threadIdx.x == 0) a.loss[blockIdx.y * gridDim.x + blockIdx.x] = sh[0] + sh[1] + sh[2] + sh[3];
    } else {
        if (active) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const f32x4 z = *reinterpret_cast<const f32x4*>(&a.Z[(size_t)(row + r) * a.N + col]);
#pragma unroll
                for (int c = 0; c < 4; ++c) v[r][c] *= gelu_grad(z[c]);
                *reinterpret_cast<f32x4*>(&a.Z[(size_t)(row + r) * a.N + col]) = v[r];
            }
            mlp_store_bf16(v, row, col, (bf16*)a.X, a.N, (bf16*)a.XT, a.M);
        }
    }
}

// Adam on an FP32 master weight.  The roundings are spelled out: left to the compiler, which
// of a moment's two products is rounded changes with the code around it.
__device__ __forceinline__ float mlp_adam(float w, float g, float& m, float& v, const MlpAdam& p) {
    m = fmaf(1.0f - p.b1, g, p.b1 * m);
    v = fmaf((1.0f - p.b2) * g, g, p.b2 * v);
    return w - p.lr * (m / p.c1) / (sqrtf(v / p.c2) + p.eps);
}

// Weight and bias gradients of up to kMlpGroup layers in one launch, each either applied
// by Adam where it is formed (the gradient never travels through memory) or stored.  The
// weights' and moments' 28 bytes a parameter bound it: 33 us for 2.8 M parameters at a batch
// of 1024, where the products, the column sums and the updates of the four layers, a launch
// each, took 148.  The bias workgroups come first: they wait for memory while the tiles run.
// Workgroups, per layer: 16 bias entries each, then the weight tiles.
template <int TM, int TN, bool ADAM>
__global__ __launch_bounds__(256, 3) void k_mlp_weights(MlpWeightsArgs a) {
    __shared__ __align__(16) float tile[TM * (TN + kPitch)];
    int t = blockIdx.x, l = 0;
    while (l + 1 < a.layers && t >= a.first[l + 1]) ++l;
    const MlpWeights& w = a.w[l];
    t -= a.first[l];
    const int nbias = w.out / 16;
    if (t < nbias) {
        // 16 bias entries: 64 row slices, each summing every 64th row of dZ, then the slices in
        // order (the sum is the same on every run and for every tile size)
        constexpr int kSlices = 64;
        const int c4 = threadIdx.x & 3, q = threadIdx.x >> 2;
        const float* z = w.dZ + t * 16 + 4 * c4;
        f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 16
        for (int r = q; r < a.rows; r += kSlices) s += *reinterpret_cast<const f32x4*>(z + (size_t)r * w.out);
#pragma unroll
        for (int i = 0; i < 4; ++i) tile[q * 17 + 4 * c4 + i] = s[i];
        __syncthreads();
        if (threadIdx.x < 16) {
            const int c = threadIdx.x, n = t * 16 + c;
            float g = 0.f;
#pragma unroll 8
            for (int k = 0; k < kSlices; ++k) g += tile[k * 17 + c];
            if constexpr (ADAM) w.b[n] = mlp_adam(w.b[n], g, w.mb[n], w.vb[n], a.adam);
            else w.gb[n] = g;
        }
        return;
    }
    t -= nbias;
    const int tn = w.in / TN;
    const int m0 = t / tn * TM, n0 = t % tn * TN;
    // the thread's block of the tile (mlp_block); its weights and moments are on their way
    // while the product runs
    const int row = m0 + 4 * (threadIdx.x / (TN / 4)), col = n0 + 4 * (threadIdx.x % (TN / 4));
    const bool mine = threadIdx.x < TM * TN / 16;
    f32x4 x[4], mo[4], se[4];
    if constexpr (ADAM) {
        if (mine) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const size_t o = (size_t)(row + r) * w.in + col;
                x[r] = *reinterpret_cast<f32x4*>(&w.W[o]);
                mo[r] = *reinterpret_cast<f32x4*>(&w.mW[o]);
                se[r] = *reinterpret_cast<f32x4*>(&w.vW[o]);
            }
        }
    }
    mlp_product<TM, TN, (TM < 64 ? 8 : 4)>((const bf16*)w.dZT, (const bf16*)w.HT, a.batch, m0, n0, tile);
    int rg = 0, cg = 0;
    f32x4 v[4];
    if (!mlp_block<TM, TN>(tile, rg, cg, v)) return;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const size_t o = (size_t)(row + r) * w.in + col;
        if constexpr (ADAM) {
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                float mc = mo[r][c], sc = se[r][c];
                x[r][c] = mlp_adam(x[r][c], v[r][c], mc, sc, a.adam);
                mo[r][c] = mc;
                se[r][c] = sc;
            }
            *reinterpret_cast<f32x4*>(&w.W[o]) = x[r];
            *reinterpret_cast<f32x4*>(&w.mW[o]) = mo[r];
            *reinterpret_cast<f32x4*>(&w.vW[o]) = se[r];
            v[r] = x[r];
        } else {
            *reinterpret_cast<f32x4*>(&w.gW[o]) = v[r];
        }
    }
    if constexpr (ADAM) mlp_store_bf16(v, row, col, (bf16*)w.Wb, w.in, (bf16*)w.WbT, w.out);
}

// An FP32 array (rows x cols real entries, row stride ldx) as zero-padded BF16 in both
// orders: X[row][col] (Rp x Cp) and, when given, XT[col][row]; P (when given) receives it
// padded in FP32.  64 x 64 per workgroup: the network's input batch, the caller's output
// gradient and the weights.
__global__ __launch_bounds__(256) void k_mlp_convert(const float* __restrict__ x, int rows, int cols, int ldx,
                                                     bf16* __restrict__ X, bf16* __restrict__ XT, int Rp, int Cp,
                                                     float* __restrict__ P) {
    __shared__ __align__(16) float tile[64 * 65];
    const int r0 = blockIdx.y * 64, c0 = blockIdx.x * 64;
    for (int i = threadIdx.x; i < 64 * 64; i += 256) {
        const int r = i >> 6, c = i & 63;
        tile[r * 65 + c] =
            (r0 + r < rows && c0 + c < cols) ? x[(size_t)(r0 + r) * ldx + c0 + c] : 0.0f;
    }
    __syncthreads();
    const int rg = threadIdx.x >> 4, cg = threadIdx.x & 15;
    f32x4 v[4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int c = 0; c < 4; ++c) v[r][c] = tile[(4 * rg + r) * 65 + 4 * cg + c];
    mlp_store_bf16(v, r0 + 4 * rg, c0 + 4 * cg, X, Cp, XT, Rp);
    if (P) {
#pragma unroll
        for (int r = 0; r < 4; ++r) *reinterpret_cast<f32x4*>(&P[(size_t)(r0 + 4 * rg + r) * Cp + c0 + 4 * cg]) = v[r];
    }
}

// One layer's parameters between the padded device layout (W [np][kp], b [np]) and the
// caller's flat one (W [no][ni], then b [no]).  The copy to or from the host is then one
// contiguous transfer: copied row by row (hipMemcpy2D, a transfer per weight row) the
// 2.8 M parameters of the 512-3x1024-168 network took 23 ms, packed they take 0.7 ms.
__global__ __launch_bounds__(256) void k_pack_layer(float* __restrict__ W, float* __restrict__ b, int no, int ni,
                                                    int kp, float* __restrict__ flat, bool to_flat) {
    const long long nw = (long long)no * ni;
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nw + no) return;
    float* p = i < nw ? &W[(i / ni) * kp + i % ni] : &b[i - nw];
    if (to_flat) flat[i] = *p;
    else *p = flat[i];
}

// Host launchers ------------------------------------------------------------------

// 64 x 64 tiles load half the operand bytes per flop of 32 x 32 ones (11.3 against 14.3 us
// for a 1024 x 1024 x 1024 product); below 256 of them, one per CU, the smaller tiles put
// four times the CUs to work (1024 x 192 x 1024: 8.6 against 10.4 us).
static bool small_tiles(long long tiles64) { return tiles64 < 256; }

int mlp_tile_rows(int M, int N) { return small_tiles((long long)(M / 64) * (N / 64)) ? 32 : 64; }

static bool bad_dims(int M, int N, int K) { return M % 64 || N % 64 || K % 64 || M <= 0 || N <= 0 || K <= 0; }

template <int EPI>
static hipError_t layer(const MlpLayerArgs& a, hipStream_t s) {
    if (bad_dims(a.M, a.N, a.K)) return hipErrorInvalidValue;
    if (mlp_tile_rows(a.M, a.N) == 32)
        hipLaunchKernelGGL((k_mlp_layer<32, 32, EPI>), dim3(a.N / 32, a.M / 32), dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL((k_mlp_layer<64, 64, EPI>), dim3(a.N / 64, a.M / 64), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t mlp_hidden(const MlpLayerArgs& a, bool train, hipStream_t s) {
    return train ? layer<EPI_HIDDEN>(a, s) : layer<EPI_HIDDEN_ONLY>(a, s);
}
hipError_t mlp_output(const MlpLayerArgs& a, hipStream_t s) { return layer<EPI_OUTPUT>(a, s); }
hipError_t mlp_output_mse(const MlpLayerArgs& a, hipStream_t s) { return layer<EPI_MSE>(a, s); }
hipError_t mlp_backward_data(const MlpLayerArgs& a, hipStream_t s) { return layer<EPI_BWD_DATA>(a, s); }

hipError_t mlp_weights(MlpWeightsArgs a, bool adam, hipStream_t s) {
    if (a.layers < 1 || a.layers > kMlpGroup) return hipErrorInvalidValue;
    long long tiles64 = 0;
    for (int l = 0; l < a.layers; ++l) {
        if (bad_dims(a.w[l].out, a.w[l].in, a.batch)) return hipErrorInvalidValue;
        tiles64 += (long long)(a.w[l].out / 64) * (a.w[l].in / 64);
    }
    const int T = small_tiles(tiles64) ? 32 : 64;
    int first = 0;
    for (int l = 0; l < a.layers; ++l) {
        a.first[l] = first;
        first += (a.w[l].out / T) * (a.w[l].in / T) + a.w[l].out / 16;
    }
    if (T == 32 && adam) hipLaunchKernelGGL((k_mlp_weights<32, 32, true>), dim3(first), dim3(256), 0, s, a);
    else if (T == 32) hipLaunchKernelGGL((k_mlp_weights<32, 32, false>), dim3(first), dim3(256), 0, s, a);
    else if (adam) hipLaunchKernelGGL((k_mlp_weights<64, 64, true>), dim3(first), dim3(256), 0, s, a);
    else hipLaunchKernelGGL((k_mlp_weights<64, 64, false>), dim3(first), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t mlp_convert(const float* x, int rows, int cols, int ldx, void* X, void* XT, int Rp, int Cp, float* P,
                       hipStream_t s) {
    if (Rp % 64 || Cp % 64 || Rp <= 0 || Cp <= 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_mlp_convert, dim3(Cp / 64, Rp / 64), dim3(256), 0, s, x, rows, cols, ldx, (bf16*)X, (bf16*)XT,
                       Rp, Cp, P);
    return hipGetLastError();
}

hipError_t mlp_pack_layer(float* W, float* b, int no, int ni, int kp, float* flat, bool to_flat, hipStream_t s) {
    const long long n = (long long)no * ni + no;
    hipLaunchKernelGGL(k_pack_layer, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, W, b, no, ni, kp, flat,
                       to_flat);
    return hipGetLastError();
}

}  // namespace sqh
