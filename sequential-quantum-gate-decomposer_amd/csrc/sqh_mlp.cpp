// sqh_mlp.cpp -- the warm-start network (no counterpart in the reference, whose
// nn module only generates data: squander/src-cpp/nn/include/NN.h:58-146).
//
// A multilayer perceptron in -> hidden (GELU) x n_hidden -> out, BF16 weights and
// activations with FP32 accumulation and FP32 master weights, trained with Adam on
// mean-squared error.  Every dimension is padded to the GEMM tile (64); padded
// weights, biases and gradients stay exactly zero.
#include <cmath>
#include <cstring>
#include <random>
#include <vector>

#include "sqh_context.h"
#include "sqh_mlp.h"

using namespace sqh;

namespace {
inline int pad64(int v) { return (v + 63) / 64 * 64; }
}  // namespace

struct sqh_mlp {
    sqh_ctx* ctx = nullptr;
    int L = 0;                       // weight layers
    std::vector<int> dim, dpad;      // real and padded widths, L + 1 entries
    // FP32 master weights, their BF16 copies in both orders, Adam's moments, gradients
    // (kept only by sqh_mlp_gradients)
    std::vector<DevBuf> W, Wb, WbT, b, mW, vW, mb, vb, gW, gb;
    // per layer for a batch: input activations and their transposes, pre-activations (then
    // output gradients) in FP32, output gradients and their transposes
    std::vector<DevBuf> H, HT, Z, dZ, dZT;
    DevBuf loss;                     // loss partials
    DevBuf flat;                     // the parameters in the caller's flat layout
    int loss_parts = 0;              // loss partials the last forward pass wrote
    int step = 0;

    ~sqh_mlp() {
        for (auto* v : {&W, &Wb, &WbT, &b, &mW, &vW, &mb, &vb, &gW, &gb, &H, &HT, &Z, &dZ, &dZT})
            for (auto& x : *v) x.release();
        loss.release();
        flat.release();
    }
    hipStream_t st() const { return ctx->stream; }
};

namespace {

// Activation buffers for a padded batch of Bp (train: those of the backward pass too).
int ensure_batch(sqh_mlp* m, int Bp, bool train) {
    sqh_ctx* c = m->ctx;
    for (int l = 0; l < m->L; ++l) {
        const size_t in = m->dpad[l], outd = m->dpad[l + 1], out = (size_t)Bp * outd;
        HIPTRY(c, m->H[l].ensure((size_t)Bp * in * 2));
        if (!train) continue;
        HIPTRY(c, m->HT[l].ensure(in * Bp * 2));
        HIPTRY(c, m->Z[l].ensure(out * 4));
        HIPTRY(c, m->dZ[l].ensure((size_t)Bp * outd * 2));
        HIPTRY(c, m->dZT[l].ensure(outd * Bp * 2));
    }
    if (train) HIPTRY(c, m->loss.ensure((size_t)Bp * m->dpad[m->L] / 1024 * sizeof(double)));
    return SQH_OK;
}

// Layer l's product over the padded batch, forward (A = its input, B = W).
MlpLayerArgs layer_args(sqh_mlp* m, int l, int Bp) {
    MlpLayerArgs a;
    a.A = m->H[l].p;
    a.B = m->Wb[l].p;
    a.M = Bp;
    a.N = m->dpad[l + 1];
    a.K = m->dpad[l];
    a.bias = m->b[l].as<float>();
    return a;
}

// The input and the hidden layers (train: with what the backward pass reads).
int forward_hidden(sqh_mlp* m, const float* d_x, int B, int Bp, bool train) {
    sqh_ctx* c = m->ctx;
    HIPTRY(c, mlp_convert(d_x, B, m->dim[0], m->dim[0], m->H[0].p, train ? m->HT[0].p : nullptr, Bp, m->dpad[0],
                          nullptr, m->st()));
    for (int l = 0; l + 1 < m->L; ++l) {
        MlpLayerArgs a = layer_args(m, l, Bp);
        a.X = m->H[l + 1].p;
        if (train) {
            a.XT = m->HT[l + 1].p;
            a.Z = m->Z[l].as<float>();
        }
        HIPTRY(c, mlp_hidden(a, train, m->st()));
    }
    return SQH_OK;
}

// The hidden layers' output gradients from the last layer's in dZ[L-1].
int backward_data(sqh_mlp* m, int Bp) {
    sqh_ctx* c = m->ctx;
    for (int l = m->L - 1; l > 0; --l) {
        MlpLayerArgs a;
        a.A = m->dZ[l].p;
        a.B = m->WbT[l].p;
        a.M = Bp;
        a.N = m->dpad[l];
        a.K = m->dpad[l + 1];
        a.Z = m->Z[l - 1].as<float>();
        a.X = m->dZ[l - 1].p;
        a.XT = m->dZT[l - 1].p;
        HIPTRY(c, mlp_backward_data(a, m->st()));
    }
    return SQH_OK;
}

// Weight and bias gradients of every layer: applied by one Adam step of rate lr, or
// (adam = false) stored in gW / gb.  After backward_data, which reads the old weights.
int weights(sqh_mlp* m, int B, int Bp, bool adam, float lr) {
    sqh_ctx* c = m->ctx;
    if (adam) m->step++;
    const float b1 = 0.9f, b2 = 0.999f;
    MlpWeightsArgs g;
    g.batch = Bp;
    g.rows = B;
    g.adam = {lr, b1, b2, 1e-8f, 1.0f - powf(b1, (float)m->step), 1.0f - powf(b2, (float)m->step)};
    for (int l0 = 0; l0 < m->L; l0 += kMlpGroup) {
        g.layers = std::min(kMlpGroup, m->L - l0);
        for (int k = 0; k < g.layers; ++k) {
            const int l = l0 + k;
            if (!adam) {
                HIPTRY(c, m->gW[l].ensure((size_t)m->dpad[l + 1] * m->dpad[l] * 4));
                HIPTRY(c, m->gb[l].ensure((size_t)m->dpad[l + 1] * 4));
            }
            g.w[k] = {m->dZT[l].p,          m->HT[l].p,          m->W[l].as<float>(),  m->mW[l].as<float>(),
                      m->vW[l].as<float>(), m->gW[l].as<float>(), m->Wb[l].p,           m->WbT[l].p,
                      m->b[l].as<float>(),  m->mb[l].as<float>(), m->vb[l].as<float>(), m->gb[l].as<float>(),
                      m->Z[l].as<float>(),  m->dpad[l],           m->dpad[l + 1]};
        }
        HIPTRY(c, mlp_weights(g, adam, m->st()));
    }
    return SQH_OK;
}

// Forward pass of a training step on the MSE loss and the output gradients of every
// layer.
int forward_backward(sqh_mlp* m, const float* d_x, const float* d_t, int B, int Bp) {
    sqh_ctx* c = m->ctx;
    const int L = m->L;
    int rc = forward_hidden(m, d_x, B, Bp, true);
    if (rc) return rc;
    MlpLayerArgs a = layer_args(m, L - 1, Bp);
    a.t = d_t;
    a.batch = B;
    a.out = m->dim[L];
    a.X = m->dZ[L - 1].p;
    a.XT = m->dZT[L - 1].p;
    a.Z = m->Z[L - 1].as<float>();
    a.loss = m->loss.as<double>();
    const int T = mlp_tile_rows(a.M, a.N);
    m->loss_parts = (Bp / T) * (a.N / T);
    HIPTRY(c, mlp_output_mse(a, m->st()));
    return backward_data(m, Bp);
}

// The batch loss of the last forward_backward (synchronises).
int read_loss(sqh_mlp* m, int B, double* loss) {
    sqh_ctx* c = m->ctx;
    std::vector<double> part(m->loss_parts);
    HIPTRY(c, hipMemcpyAsync(part.data(), m->loss.p, part.size() * sizeof(double), hipMemcpyDeviceToHost, m->st()));
    HIPTRY(c, hipStreamSynchronize(m->st()));
    double s = 0.0;
    for (double v : part) s += v;
    *loss = s / ((double)B * m->dim[m->L]);
    return SQH_OK;
}

// The BF16 copies of layer l's master weights, in both orders.
hipError_t convert_weights(sqh_mlp* m, int l) {
    return mlp_convert(m->W[l].as<float>(), m->dpad[l + 1], m->dpad[l], m->dpad[l], m->Wb[l].p, m->WbT[l].p,
                       m->dpad[l + 1], m->dpad[l], nullptr, m->st());
}

// He-style initialisation on the real block; the padding stays zero.
__attribute__((noinline)) void he_init(std::mt19937_64& gen, std::normal_distribution<float>& nd, int no, int ni,
                                       int kp, float* w) {
    const float sd = std::sqrt(2.0f / (float)ni);
    for (int o = 0; o < no; ++o)
        for (int i = 0; i < ni; ++i) w[(size_t)o * kp + i] = sd * nd(gen);
}

// Host flat layout of parameters: per layer W (real out x real in, row-major), then b.
template <typename F>
int for_each_layer(sqh_mlp* m, F&& f) {
    long long off = 0;
    for (int l = 0; l < m->L; ++l) {
        int rc = f(l, off);
        if (rc) return rc;
        off += (long long)m->dim[l + 1] * m->dim[l] + m->dim[l + 1];
    }
    return SQH_OK;
}

int copy_params(sqh_mlp* m, float* host, bool to_host, bool grads) {
    sqh_ctx* c = m->ctx;
    const size_t bytes = (size_t)sqh_mlp_param_count(m) * sizeof(float);
    HIPTRY(c, m->flat.ensure(bytes));
    if (!to_host) HIPTRY(c, hipMemcpyAsync(m->flat.p, host, bytes, hipMemcpyHostToDevice, m->st()));
    int rc = for_each_layer(m, [&](int l, long long off) -> int {
        const int no = m->dim[l + 1], ni = m->dim[l], kp = m->dpad[l];
        DevBuf& Wd = grads ? m->gW[l] : m->W[l];
        DevBuf& bd = grads ? m->gb[l] : m->b[l];
        HIPTRY(c, mlp_pack_layer(Wd.as<float>(), bd.as<float>(), no, ni, kp, m->flat.as<float>() + off, to_host,
                                 m->st()));
        if (!to_host)
            HIPTRY(c, convert_weights(m, l));
        return SQH_OK;
    });
    if (rc) return rc;
    if (to_host) HIPTRY(c, hipMemcpyAsync(host, m->flat.p, bytes, hipMemcpyDeviceToHost, m->st()));
    HIPTRY(c, hipStreamSynchronize(m->st()));
    return SQH_OK;
}

}  // namespace

extern "C" {

int sqh_mlp_create(sqh_ctx* c, int in_dim, int hidden, int n_hidden, int out_dim, unsigned long long seed,
                   sqh_mlp** out) {
    if (!c || !out) return SQH_ERR_ARG;
    std::lock_guard<std::mutex> lk(c->mu);
    *out = nullptr;
    if (in_dim <= 0 || hidden <= 0 || n_hidden < 0 || out_dim <= 0) return fail(c, SQH_ERR_ARG, "bad network shape");
    HIPTRY(c, hipSetDevice(c->device));
    sqh_mlp* m = new (std::nothrow) sqh_mlp();
    if (!m) return SQH_ERR_NOMEM;
    m->ctx = c;
    m->dim.push_back(in_dim);
    for (int i = 0; i < n_hidden; ++i) m->dim.push_back(hidden);
    m->dim.push_back(out_dim);
    m->L = (int)m->dim.size() - 1;
    for (int d : m->dim) m->dpad.push_back(pad64(d));
    for (auto* v : {&m->W, &m->Wb, &m->WbT, &m->b, &m->mW, &m->vW, &m->mb, &m->vb, &m->gW, &m->gb, &m->H, &m->HT,
                    &m->Z, &m->dZ, &m->dZT})
        v->resize(m->L);
    std::mt19937_64 gen(seed);
    std::normal_distribution<float> nd(0.0f, 1.0f);
    for (int l = 0; l < m->L; ++l) {
        const int np = m->dpad[l + 1], kp = m->dpad[l];
        const size_t nw = (size_t)np * kp;
        bool ok = m->W[l].ensure(nw * 4) == hipSuccess && m->Wb[l].ensure((size_t)np * kp * 2) == hipSuccess &&
                  m->WbT[l].ensure((size_t)kp * np * 2) == hipSuccess &&
                  m->mW[l].ensure(nw * 4) == hipSuccess && m->vW[l].ensure(nw * 4) == hipSuccess &&
                  m->b[l].ensure(np * 4) == hipSuccess && m->mb[l].ensure(np * 4) == hipSuccess &&
                  m->vb[l].ensure(np * 4) == hipSuccess;
        if (!ok) {
            delete m;
            return fail(c, SQH_ERR_NOMEM, "network allocation failed");
        }
        std::vector<float> w(nw, 0.0f);
        he_init(gen, nd, m->dim[l + 1], m->dim[l], kp, w.data());
        hipError_t e = hipMemcpy(m->W[l].p, w.data(), nw * 4, hipMemcpyHostToDevice);
        for (DevBuf* z : {&m->mW[l], &m->vW[l]})
            if (e == hipSuccess) e = hipMemset(z->p, 0, nw * 4);
        for (DevBuf* z : {&m->b[l], &m->mb[l], &m->vb[l]})
            if (e == hipSuccess) e = hipMemset(z->p, 0, (size_t)np * 4);
        if (e == hipSuccess) e = convert_weights(m, l);
        if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
        if (e != hipSuccess) {
            delete m;
            return fail(c, SQH_ERR_DEVICE, "network initialisation: %s", hipGetErrorString(e));
        }
    }
    *out = m;
    return SQH_OK;
}

void sqh_mlp_destroy(sqh_mlp* m) {
    if (!m) return;
    (void)hipStreamSynchronize(m->ctx->stream);
    delete m;
}

long long sqh_mlp_param_count(const sqh_mlp* m) {
    if (!m) return SQH_ERR_ARG;
    long long n = 0;
    for (int l = 0; l < m->L; ++l) n += (long long)m->dim[l + 1] * m->dim[l] + m->dim[l + 1];
    return n;
}

int sqh_mlp_get_params(sqh_mlp* m, float* out) {
    if (!m || !out) return SQH_ERR_ARG;
    std::lock_guard<std::mutex> lk(m->ctx->mu);
    HIPTRY(m->ctx, hipSetDevice(m->ctx->device));
    HIPTRY(m->ctx, hipStreamSynchronize(m->st()));
    return copy_params(m, out, true, false);
}

int sqh_mlp_set_params(sqh_mlp* m, const float* in) {
    if (!m || !in) return SQH_ERR_ARG;
    std::lock_guard<std::mutex> lk(m->ctx->mu);
    HIPTRY(m->ctx, hipSetDevice(m->ctx->device));
    HIPTRY(m->ctx, hipStreamSynchronize(m->st()));
    return copy_params(m, const_cast<float*>(in), false, false);
}

int sqh_mlp_forward_dev(sqh_mlp* m, const float* d_x, int B, float* d_y) {
    if (!m || !d_x || !d_y || B <= 0) return SQH_ERR_ARG;
    sqh_ctx* c = m->ctx;
    std::lock_guard<std::mutex> lk(c->mu);
    HIPTRY(c, hipSetDevice(c->device));
    const int Bp = pad64(B);
    int rc = ensure_batch(m, Bp, false);
    if (rc) return rc;
    if ((rc = forward_hidden(m, d_x, B, Bp, false))) return rc;
    MlpLayerArgs a = layer_args(m, m->L - 1, Bp);
    a.y = d_y;
    a.batch = B;
    a.out = m->dim[m->L];
    HIPTRY(c, mlp_output(a, m->st()));
    return SQH_OK;
}

int sqh_mlp_train_step_dev(sqh_mlp* m, const float* d_x, const float* d_t, int B, float lr, double* loss) {
    if (!m || !d_x || !d_t || B <= 0) return SQH_ERR_ARG;
    sqh_ctx* c = m->ctx;
    std::lock_guard<std::mutex> lk(c->mu);
    HIPTRY(c, hipSetDevice(c->device));
    const int Bp = pad64(B);
    int rc = ensure_batch(m, Bp, true);
    if (rc) return rc;
    if ((rc = forward_backward(m, d_x, d_t, B, Bp))) return rc;
    if ((rc = weights(m, B, Bp, true, lr))) return rc;
    return loss ? read_loss(m, B, loss) : SQH_OK;
}

int sqh_mlp_backward_step_dev(sqh_mlp* m, const float* d_x, const float* d_dy, int B, float lr) {
    if (!m || !d_x || !d_dy || B <= 0) return SQH_ERR_ARG;
    sqh_ctx* c = m->ctx;
    std::lock_guard<std::mutex> lk(c->mu);
    HIPTRY(c, hipSetDevice(c->device));
    const int Bp = pad64(B), L = m->L;
    int rc = ensure_batch(m, Bp, true);
    if (rc) return rc;
    // the output itself is not needed: its gradient is the caller's
    if ((rc = forward_hidden(m, d_x, B, Bp, true))) return rc;
    HIPTRY(c, mlp_convert(d_dy, B, m->dim[L], m->dim[L], m->dZ[L - 1].p, m->dZT[L - 1].p, Bp, m->dpad[L],
                          m->Z[L - 1].as<float>(), m->st()));
    if ((rc = backward_data(m, Bp))) return rc;
    return weights(m, B, Bp, true, lr);
}

int sqh_mlp_gradients(sqh_mlp* m, const float* x, const float* t, int B, float* grads, double* loss) {
    if (!m || !x || !t || !grads || B <= 0) return SQH_ERR_ARG;
    sqh_ctx* c = m->ctx;
    std::lock_guard<std::mutex> lk(c->mu);
    HIPTRY(c, hipSetDevice(c->device));
    const int Bp = pad64(B);
    int rc = ensure_batch(m, Bp, true);
    if (rc) return rc;
    DevBuf dx, dt;
    HIPTRY(c, dx.ensure((size_t)B * m->dim[0] * 4));
    HIPTRY(c, dt.ensure((size_t)B * m->dim[m->L] * 4));
    HIPTRY(c, hipMemcpyAsync(dx.p, x, (size_t)B * m->dim[0] * 4, hipMemcpyHostToDevice, m->st()));
    HIPTRY(c, hipMemcpyAsync(dt.p, t, (size_t)B * m->dim[m->L] * 4, hipMemcpyHostToDevice, m->st()));
    rc = forward_backward(m, dx.as<float>(), dt.as<float>(), B, Bp);
    if (!rc) rc = weights(m, B, Bp, false, 0.0f);
    if (!rc && loss) rc = read_loss(m, B, loss);
    if (!rc) rc = copy_params(m, grads, true, true);
    (void)hipStreamSynchronize(m->st());
    dx.release();
    dt.release();
    return rc;
}

}  // extern "C"
