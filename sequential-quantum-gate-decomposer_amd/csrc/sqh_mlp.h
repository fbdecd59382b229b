// sqh_mlp.h -- arguments and launchers of the warm-start network's kernels
// (sqh_k_mlp.hip), shared with the host side (sqh_mlp.cpp).
#pragma once
#include <hip/hip_runtime.h>

namespace sqh {

// The BF16 arrays (activations, gradients, weights and their transposes) are stored in
// the order the MFMA operands are read: tiles of 16 rows x 32 k values, 1 KiB each, in
// which lane l of a wavefront finds its 8 values (row l % 16, k = 8 (l / 16) ...) at
// 16 l.  An operand load is then 1 KiB contiguous; from row-major arrays the 16 lanes of
// a load phase touched 16 rows, 16 bytes of a cache line each, and a 1024 x 1024 x 1024
// product spent 7 us on its loads instead of 2.
__host__ __device__ inline size_t mlp_frag(int row, int k, int K) {
    return ((size_t)(row >> 4) * (K >> 5) + (k >> 5)) * 512 + ((row & 15) + 16 * ((k & 31) >> 3)) * 8 + (k & 7);
}

// One product C[M][N] = sum_k A[m][k] B[n][k] (BF16, mlp_frag order) with its epilogue.
struct MlpLayerArgs {
    const void* A = nullptr;
    const void* B = nullptr;
    int M = 0, N = 0, K = 0;      // padded; M is the padded batch
    const float* bias = nullptr;  // [N] (forward)
    // FP32 [M][N]: the pre-activations, written forward; the data gradient reads them and
    // leaves dZ in their place (the output layer: dZ), from which the bias gradient is summed
    float* Z = nullptr;
    void* X = nullptr;            // BF16 result [M][N] (H or dZ)
    void* XT = nullptr;           // ... and transposed [N][M]
    float* y = nullptr;           // the caller's output [batch][out]
    const float* t = nullptr;     // the caller's training targets [batch][out]
    int batch = 0, out = 0;       // real rows and columns of y / t
    double* loss = nullptr;       // loss partials, one per workgroup
};

struct MlpAdam {
    float lr, b1, b2, eps, c1, c2;
};

// One layer's weight update: W [out][in], bias [out]; dZT [out][batch], HT [in][batch].
struct MlpWeights {
    const void* dZT;
    const void* HT;
    float *W, *mW, *vW, *gW;
    void *Wb, *WbT;
    float *b, *mb, *vb, *gb;
    const float* dZ;  // FP32 [batch][out]
    int in, out;      // padded
};

constexpr int kMlpGroup = 8;  // layers per launch

struct MlpWeightsArgs {
    MlpWeights w[kMlpGroup];
    int first[kMlpGroup];  // first workgroup of each layer
    int layers;
    int batch;  // padded
    int rows;   // real rows of the batch
    MlpAdam adam;
};

// Rows of the tiles a layer product over M x N runs with.
int mlp_tile_rows(int M, int N);
hipError_t mlp_hidden(const MlpLayerArgs& a, bool train, hipStream_t s);
hipError_t mlp_output(const MlpLayerArgs& a, hipStream_t s);
hipError_t mlp_output_mse(const MlpLayerArgs& a, hipStream_t s);
hipError_t mlp_backward_data(const MlpLayerArgs& a, hipStream_t s);
// The layers' gradients applied by Adam, or (adam = false) stored in gW / gb.
hipError_t mlp_weights(MlpWeightsArgs a, bool adam, hipStream_t s);
hipError_t mlp_convert(const float* x, int rows, int cols, int ldx, void* X, void* XT, int Rp, int Cp, float* P,
                       hipStream_t s);
hipError_t mlp_pack_layer(float* W, float* b, int no, int ni, int kp, float* flat, bool to_flat, hipStream_t s);

}  // namespace sqh
