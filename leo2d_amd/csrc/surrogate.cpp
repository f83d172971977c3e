// surrogate.cpp -- C-ABI of the learned local-moment surrogate (include/leo2d.h).
//
// A multilayer perceptron maps the Fourier features of a local stacking
// configuration (interlayer shift, symmetric strain, twist) to the local
// Chebyshev moments of the four sublattices of a bilayer.  Training and
// inference run on the GPU through the BF16 MFMA kernels of mlp.hip; the host
// here only sequences launches, shuffles the training set and initialises the
// weights.  There is no counterpart in the reference: the moments it learns
// come from this library's KPM recursion (leo2d_batch_kpm with target starts).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <numeric>
#include <random>
#include <string>
#include <vector>

#include "devbuf.h"
#include "mlp.h"

using leo2d::check;
using leo2d::dalloc;
using leo2d::DevBuf;
using leo2d::HipError;

struct leo2d_mlp {
    leo2d::DevPool pool;   // first member: the buffers below go back to it
    int device = 0;
    hipStream_t stream = nullptr;
    std::string err;
    std::vector<int> dims;                 // in, hidden x layers, out
    std::vector<int64_t> woff, boff;       // offsets of W_l and b_l in the flat parameter vector
    int64_t nparams = 0;
    DevBuf P32, G, Mom, Var;               // master weights, gradient, Adam moments
    DevBuf P16, PT16, descs;               // bf16 copies of every W and W^T, their layout (mlp.h)
    std::vector<leo2d::LayerDesc> layer;
    int param_blocks = 0;
    int64_t adam_step = 0;
    // batch workspace
    int cap = 0;
    int64_t ldt = 0;                       // leading dimension of the transposed batch operands
    DevBuf X16, XT16, Y, T, lossparts, rowloss, xin;
    std::vector<DevBuf> Z, H, HT;          // per hidden layer: pre-activation FP32, activation bf16 and its transpose
    DevBuf dZ[2], dZT[2];                  // gradients of two neighbouring layers' inputs, bf16, and their transposes

    int layers() const { return (int)dims.size() - 1; }
    int in() const { return dims.front(); }
    int out() const { return dims.back(); }
    ~leo2d_mlp()
    {
        if (stream) (void)hipStreamDestroy(stream);
    }
};

namespace {

struct ArgError : std::runtime_error {
    explicit ArgError(const std::string& m) : std::runtime_error(m) {}
};

template <typename F>
int guarded(leo2d_mlp* m, F&& f)
{
    leo2d::DevPool::Use use(m ? &m->pool : nullptr);
    try {
        if (m) check(hipSetDevice(m->device), "hipSetDevice");
        return f();
    } catch (const HipError& e) {
        if (m) m->err = e.what();
        return e.code;
    } catch (const ArgError& e) {
        if (m) m->err = e.what();
        return LEO2D_ERR_ARG;
    } catch (const std::bad_alloc&) {
        if (m) m->err = "host allocation failed";
        return LEO2D_ERR_ALLOC;
    } catch (const std::exception& e) {
        if (m) m->err = e.what();
        return LEO2D_ERR_ARG;
    }
}

const uint16_t* bf(const DevBuf& b, int64_t off = 0) { return static_cast<const uint16_t*>(b.p) + off; }
uint16_t* bfw(DevBuf& b, int64_t off = 0) { return static_cast<uint16_t*>(b.p) + off; }
float* f32(DevBuf& b, int64_t off = 0) { return static_cast<float*>(b.p) + off; }

void to_device_f32(DevBuf& b, const std::vector<float>& v, hipStream_t s)
{
    dalloc(b, sizeof(float) * v.size(), "adam corrections");
    check(hipMemcpyAsync(b.p, v.data(), sizeof(float) * v.size(), hipMemcpyHostToDevice, s), "adam corrections");
}

// Buffers for batches of up to `rows` rows.  bf16 operands have k contiguous on both
// sides of a product (mlp.h): activations and gradients in both orders, leading
// dimensions padded to 8.
void ensure_capacity(leo2d_mlp* m, int rows)
{
    if (rows <= m->cap) return;
    leo2d::DevPool::Use own(&m->pool);   // the network's buffers, whichever network's call this is
    m->cap = 0;   // until every buffer is there
    const int cap = std::max(rows, 256);
    const int64_t ldt = leo2d::pad8(cap);
    const int64_t widest = leo2d::pad8(*std::max_element(m->dims.begin() + 1, m->dims.end()));
    auto b16 = [&](DevBuf& b, int64_t elems, const char* what) { dalloc(b, sizeof(uint16_t) * (size_t)elems, what); };
    b16(m->X16, cap * leo2d::pad8(m->in()), "mlp inputs");
    b16(m->XT16, ldt * m->in(), "mlp inputs");
    dalloc(m->xin, sizeof(float) * (size_t)cap * m->in(), "mlp inputs");
    dalloc(m->Y, sizeof(float) * (size_t)cap * m->out(), "mlp outputs");
    dalloc(m->T, sizeof(float) * (size_t)cap * m->out(), "mlp targets");
    for (int q = 0; q < 2; ++q) {
        b16(m->dZ[q], cap * widest, "mlp gradient");
        b16(m->dZT[q], ldt * widest, "mlp gradient");
    }
    dalloc(m->lossparts, sizeof(double) * (size_t)cap * ((m->out() + 15) / 16), "mlp loss");
    dalloc(m->rowloss, sizeof(double) * (size_t)cap, "mlp loss");
    m->Z.clear();
    m->H.clear();
    m->HT.clear();
    m->Z.resize(m->layers() - 1);
    m->H.resize(m->layers() - 1);
    m->HT.resize(m->layers() - 1);
    for (int l = 0; l + 1 < m->layers(); ++l) {
        dalloc(m->Z[l], sizeof(float) * (size_t)cap * m->dims[l + 1], "mlp pre-activations");
        b16(m->H[l], cap * leo2d::pad8(m->dims[l + 1]), "mlp activations");
        b16(m->HT[l], ldt * m->dims[l + 1], "mlp activations");
    }
    m->cap = cap;
    m->ldt = ldt;
}

const leo2d::SumArgs kNoSums{nullptr, 0, 0, 0, nullptr};
const leo2d::LossArgs kNoLoss{nullptr, 0, 0, nullptr};

// the product of layer l's inputs with W^T, up to its epilogue
leo2d::GemmArgs layer_product(leo2d_mlp* m, int l, const uint16_t* hin, int rows)
{
    leo2d::GemmArgs g{};
    g.A = hin;
    g.lda = leo2d::pad8(m->dims[l]);
    g.B = bf(m->P16, m->layer[(size_t)l].w16);
    g.ldb = m->layer[(size_t)l].ldw;
    g.M = rows;
    g.N = m->dims[l + 1];
    g.K = m->dims[l];
    g.bias = f32(m->P32, m->boff[l]);
    g.ldc = m->dims[l + 1];
    return g;
}

// The hidden layers on X16 (by default the network's own); train: with what the
// backward pass needs.  Returns the last hidden activations.
const uint16_t* hidden_layers(leo2d_mlp* m, int rows, const uint16_t* X16, bool train)
{
    const uint16_t* hin = X16 ? X16 : bf(m->X16);
    for (int l = 0; l + 1 < m->layers(); ++l) {
        leo2d::GemmArgs g = layer_product(m, l, hin, rows);
        g.epi = leo2d::EPI_BIAS_GELU;
        g.C16 = bfw(m->H[l]);
        g.ld16 = leo2d::pad8(g.N);
        if (train) {
            g.Z = f32(m->Z[l]);
            g.C16T = bfw(m->HT[l]);
            g.ld16t = m->ldt;
        }
        check(leo2d::launch_gemm_bf16(g, nullptr, kNoSums, kNoLoss, m->stream), "mlp forward");
        hin = bf(m->H[l]);
    }
    return hin;
}

// Y[rows][out] = MLP(X16[rows][in]) ; Y and X16 may point outside the workspace
void forward(leo2d_mlp* m, int rows, float* Y, const uint16_t* X16 = nullptr)
{
    const uint16_t* hin = hidden_layers(m, rows, X16, false);
    leo2d::GemmArgs g = layer_product(m, m->layers() - 1, hin, rows);
    g.epi = leo2d::EPI_BIAS_F32;
    g.C32 = Y;
    check(leo2d::launch_gemm_bf16(g, nullptr, kNoSums, kNoLoss, m->stream), "mlp forward");
}

// gradient of the mean squared error over rows x out into m->G, from X16, XT16 and
// T; row losses in row_loss (m->rowloss when null)
void gradients(leo2d_mlp* m, int rows, double* row_loss = nullptr)
{
    hipStream_t s = m->stream;
    const int L = m->layers();
    const uint16_t* hin = hidden_layers(m, rows, nullptr, true);
    leo2d::GemmArgs o = layer_product(m, L - 1, hin, rows);
    o.epi = leo2d::EPI_MSE;
    o.T = f32(m->T);
    o.scale = 2.0f / ((float)rows * (float)m->out());
    o.C16 = bfw(m->dZ[0]);
    o.ld16 = leo2d::pad8(o.N);
    o.C16T = bfw(m->dZT[0]);
    o.ld16t = m->ldt;
    o.loss = static_cast<double*>(m->lossparts.p);
    check(leo2d::launch_gemm_bf16(o, nullptr, kNoSums, kNoLoss, s), "mlp loss");
    leo2d::LossArgs loss{o.loss, rows, (m->out() + 15) / 16, row_loss ? row_loss : static_cast<double*>(m->rowloss.p)};
    int cur = 0;
    for (int l = L - 1; l >= 0; --l) {
        const int din = m->dims[l], dout = m->dims[l + 1];
        // dW_l[o][i] = sum_b dZ[b][o] Hin[b][i], db_l[o] = sum_b dZ[b][o]
        leo2d::GemmArgs gw{};
        gw.epi = leo2d::EPI_STORE_F32;
        gw.A = bf(m->dZT[cur]);
        gw.lda = m->ldt;
        gw.B = l == 0 ? bf(m->XT16) : bf(m->HT[l - 1]);
        gw.ldb = m->ldt;
        gw.M = dout;
        gw.N = din;
        gw.K = rows;
        gw.C32 = f32(m->G, m->woff[l]);
        gw.ldc = din;
        const leo2d::SumArgs db{gw.A, gw.lda, dout, rows, f32(m->G, m->boff[l])};
        // dZ_{l-1} = (dZ_l W_l) * gelu'(Z_{l-1})
        leo2d::GemmArgs gx{};
        if (l > 0) {
            gx.epi = leo2d::EPI_GELU_BWD;
            gx.A = bf(m->dZ[cur]);
            gx.lda = leo2d::pad8(dout);
            gx.B = bf(m->PT16, m->layer[(size_t)l].wt16);
            gx.ldb = m->layer[(size_t)l].ldwt;
            gx.M = rows;
            gx.N = din;
            gx.K = dout;
            gx.Z = f32(m->Z[l - 1]);
            gx.ldc = din;
            gx.C16 = bfw(m->dZ[1 - cur]);
            gx.ld16 = leo2d::pad8(din);
            gx.C16T = bfw(m->dZT[1 - cur]);
            gx.ld16t = m->ldt;
        }
        check(leo2d::launch_gemm_bf16(gw, l > 0 ? &gx : nullptr, db, l == L - 1 ? loss : kNoLoss, s), "mlp gradient");
        cur = 1 - cur;
    }
}

leo2d::ParamArgs param_args(leo2d_mlp* m)
{
    leo2d::ParamArgs a{};
    a.layers = static_cast<const leo2d::LayerDesc*>(m->descs.p);
    a.nlayers = m->layers();
    a.blocks = m->param_blocks;
    a.p = f32(m->P32);
    a.p16 = bfw(m->P16);
    a.pt16 = bfw(m->PT16);
    return a;
}

// one Adam step on the gradient in m->G
leo2d::ParamArgs adam_args(leo2d_mlp* m, const leo2d_mlp_train_params* p)
{
    leo2d::ParamArgs a = param_args(m);
    a.grad = f32(m->G);
    a.m = f32(m->Mom);
    a.v = f32(m->Var);
    a.lr = p->lr;
    a.b1 = p->beta1;
    a.b2 = p->beta2;
    a.eps = p->eps;
    return a;
}

// one mini-batch: rows idx[0 .. rows) of the training set, gradient and row losses
void batch_gradients(leo2d_mlp* m, const float* X, const float* T, const int64_t* idx, int rows, double* row_loss, int* ctr)
{
    check(leo2d::launch_gather(X, m->in(), T, m->out(), idx, rows, bfw(m->X16), leo2d::pad8(m->in()), bfw(m->XT16), m->ldt,
                               f32(m->T), ctr, m->stream),
          "batch gather");
    gradients(m, rows, row_loss);
}

void upload_inputs(leo2d_mlp* m, const float* x, int rows, bool train = false)
{
    check(hipMemcpyAsync(m->xin.p, x, sizeof(float) * (size_t)rows * m->in(), hipMemcpyHostToDevice, m->stream),
          "mlp inputs");
    check(leo2d::launch_cast_rows(f32(m->xin), m->in(), rows, bfw(m->X16), leo2d::pad8(m->in()),
                                  train ? bfw(m->XT16) : nullptr, m->ldt, m->stream),
          "mlp inputs");
}

// Fourier features of one configuration (b1, b2, exx, eyy, exy, theta in degrees):
//   cos, sin 2 pi (p b1 + q b2) over 16 reciprocal vectors (p, q)          32
//   strain / 0.003                                                           3
//   strain x (cos, sin) of the first three harmonics                        18
//   t = (theta - 1.9)/1.1, t^2, 1/theta                                      3
//   t x (cos, sin) of the first three harmonics                              6
//   1, t (exx + eyy)/0.003                                                   2
const int kHarm[16][2] = {{1, 0}, {0, 1}, {1, 1}, {1, -1}, {2, 0}, {0, 2}, {2, 1}, {1, 2},
                          {2, -1}, {1, -2}, {2, 2}, {2, -2}, {3, 0}, {0, 3}, {3, 1}, {1, 3}};

void features_one(const double* c, float* f)
{
    const double two_pi = 6.283185307179586;
    double cs[16], sn[16];
    for (int h = 0; h < 16; ++h) {
        const double ph = two_pi * (kHarm[h][0] * c[0] + kHarm[h][1] * c[1]);
        cs[h] = std::cos(ph);
        sn[h] = std::sin(ph);
    }
    int k = 0;
    for (int h = 0; h < 16; ++h) {
        f[k++] = (float)cs[h];
        f[k++] = (float)sn[h];
    }
    const double e[3] = {c[2] / 0.003, c[3] / 0.003, c[4] / 0.003};
    for (int a = 0; a < 3; ++a) f[k++] = (float)e[a];
    for (int a = 0; a < 3; ++a)
        for (int h = 0; h < 3; ++h) {
            f[k++] = (float)(e[a] * cs[h]);
            f[k++] = (float)(e[a] * sn[h]);
        }
    const double t = (c[5] - 1.9) / 1.1;
    f[k++] = (float)t;
    f[k++] = (float)(t * t);
    f[k++] = (float)(1.0 / c[5]);
    for (int h = 0; h < 3; ++h) {
        f[k++] = (float)(t * cs[h]);
        f[k++] = (float)(t * sn[h]);
    }
    f[k++] = 1.0f;
    f[k++] = (float)(t * (e[0] + e[1]));
}

}  // namespace

extern "C" {

int leo2d_mlp_features(const double* cfg, int64_t n, float* feat)
{
    if (!cfg || !feat || n < 0) return LEO2D_ERR_ARG;
    for (int64_t i = 0; i < n; ++i) {
        if (!(cfg[6 * i + 5] > 0.0)) return LEO2D_ERR_ARG;   // twist in degrees, positive
        features_one(cfg + 6 * i, feat + (size_t)LEO2D_MLP_FEATURES * i);
    }
    return LEO2D_OK;
}

int leo2d_mlp_create(int32_t device, const leo2d_mlp_desc* d, leo2d_mlp** out)
{
    if (!d || !out || d->in <= 0 || d->hidden <= 0 || d->layers < 1 || d->out <= 0) return LEO2D_ERR_ARG;
    *out = nullptr;
    auto* m = new leo2d_mlp;
    m->device = device;
    const int rc = guarded(m, [&]() {
        check(hipStreamCreate(&m->stream), "hipStreamCreate");
        m->dims.push_back(d->in);
        for (int l = 0; l < d->layers; ++l) m->dims.push_back(d->hidden);
        m->dims.push_back(d->out);
        int64_t off = 0, off16 = 0, offt16 = 0;
        for (int l = 0; l < m->layers(); ++l) {
            const int din = m->dims[l], dout = m->dims[l + 1];
            leo2d::LayerDesc d{};
            d.din = din;
            d.dout = dout;
            d.ldw = leo2d::pad8(din);
            d.ldwt = leo2d::pad8(dout);
            d.woff = off;
            m->woff.push_back(off);
            off += (int64_t)dout * din;
            d.boff = off;
            m->boff.push_back(off);
            off += dout;
            d.w16 = off16;
            off16 += dout * d.ldw;
            d.wt16 = offt16;
            offt16 += din * d.ldwt;
            d.tile0 = m->param_blocks;
            m->param_blocks += leo2d::param_tiles(din, dout);
            m->layer.push_back(d);
        }
        m->nparams = off;
        // Glorot-uniform weights, zero biases
        std::vector<float> p((size_t)off, 0.0f);
        std::mt19937_64 rng(d->seed);
        for (int l = 0; l < m->layers(); ++l) {
            const double a = std::sqrt(6.0 / (m->dims[l] + m->dims[l + 1]));
            std::uniform_real_distribution<double> U(-a, a);
            for (int64_t q = 0; q < (int64_t)m->dims[l + 1] * m->dims[l]; ++q) p[m->woff[l] + q] = (float)U(rng);
        }
        dalloc(m->P32, sizeof(float) * off, "mlp weights");
        dalloc(m->P16, sizeof(uint16_t) * off16, "mlp weights");
        dalloc(m->PT16, sizeof(uint16_t) * offt16, "mlp weights");
        dalloc(m->descs, sizeof(leo2d::LayerDesc) * m->layer.size(), "mlp layers");
        check(hipMemcpyAsync(m->descs.p, m->layer.data(), sizeof(leo2d::LayerDesc) * m->layer.size(), hipMemcpyHostToDevice,
                             m->stream),
              "mlp layers");
        dalloc(m->G, sizeof(float) * off, "mlp gradient");
        dalloc(m->Mom, sizeof(float) * off, "mlp optimiser");
        dalloc(m->Var, sizeof(float) * off, "mlp optimiser");
        check(hipMemcpyAsync(m->P32.p, p.data(), sizeof(float) * off, hipMemcpyHostToDevice, m->stream), "mlp init");
        check(leo2d::launch_params(param_args(m), m->stream), "mlp init");
        check(hipMemsetAsync(m->Mom.p, 0, sizeof(float) * off, m->stream), "mlp init");
        check(hipMemsetAsync(m->Var.p, 0, sizeof(float) * off, m->stream), "mlp init");
        check(hipStreamSynchronize(m->stream), "mlp init");
        return LEO2D_OK;
    });
    if (rc != LEO2D_OK) {
        delete m;
        return rc;
    }
    *out = m;
    return LEO2D_OK;
}

void leo2d_mlp_destroy(leo2d_mlp* m)
{
    if (!m) return;
    (void)hipSetDevice(m->device);
    if (m->stream) (void)hipStreamSynchronize(m->stream);
    delete m;
}

const char* leo2d_mlp_last_error(const leo2d_mlp* m) { return m ? m->err.c_str() : "null network"; }

int64_t leo2d_mlp_num_params(const leo2d_mlp* m) { return m ? m->nparams : 0; }

int leo2d_mlp_get_params(leo2d_mlp* m, float* p)
{
    if (!m || !p) return LEO2D_ERR_ARG;
    return guarded(m, [&]() {
        check(hipMemcpy(p, m->P32.p, sizeof(float) * m->nparams, hipMemcpyDeviceToHost), "mlp params");
        return LEO2D_OK;
    });
}

int leo2d_mlp_set_params(leo2d_mlp* m, const float* p)
{
    if (!m || !p) return LEO2D_ERR_ARG;
    return guarded(m, [&]() {
        check(hipMemcpyAsync(m->P32.p, p, sizeof(float) * m->nparams, hipMemcpyHostToDevice, m->stream), "mlp params");
        check(leo2d::launch_params(param_args(m), m->stream), "mlp params");
        check(hipMemsetAsync(m->Mom.p, 0, sizeof(float) * m->nparams, m->stream), "mlp params");
        check(hipMemsetAsync(m->Var.p, 0, sizeof(float) * m->nparams, m->stream), "mlp params");
        m->adam_step = 0;
        check(hipStreamSynchronize(m->stream), "mlp params");
        return LEO2D_OK;
    });
}

int leo2d_mlp_forward(leo2d_mlp* m, const float* x, int64_t n, float* y)
{
    if (!m || !x || !y || n < 0) return LEO2D_ERR_ARG;
    return guarded(m, [&]() {
        const int chunk = 4096;
        ensure_capacity(m, (int)std::min<int64_t>(n, chunk));
        for (int64_t r0 = 0; r0 < n; r0 += chunk) {
            const int rows = (int)std::min<int64_t>(chunk, n - r0);
            upload_inputs(m, x + (size_t)r0 * m->in(), rows);
            forward(m, rows, f32(m->Y));
            check(hipMemcpyAsync(y + (size_t)r0 * m->out(), m->Y.p, sizeof(float) * (size_t)rows * m->out(),
                                 hipMemcpyDeviceToHost, m->stream),
                  "mlp outputs");
            check(hipStreamSynchronize(m->stream), "mlp forward");
        }
        return LEO2D_OK;
    });
}

int leo2d_mlp_gradients(leo2d_mlp* m, const float* x, const float* t, int32_t n, double* loss, float* grad)
{
    if (!m || !x || !t || n <= 0) return LEO2D_ERR_ARG;
    return guarded(m, [&]() {
        ensure_capacity(m, n);
        upload_inputs(m, x, n, true);
        check(hipMemcpyAsync(m->T.p, t, sizeof(float) * (size_t)n * m->out(), hipMemcpyHostToDevice, m->stream),
              "mlp targets");
        gradients(m, n);
        std::vector<double> rl(n);
        check(hipMemcpyAsync(rl.data(), m->rowloss.p, sizeof(double) * n, hipMemcpyDeviceToHost, m->stream), "loss");
        if (grad)
            check(hipMemcpyAsync(grad, m->G.p, sizeof(float) * m->nparams, hipMemcpyDeviceToHost, m->stream),
                  "mlp gradient");
        check(hipStreamSynchronize(m->stream), "mlp gradients");
        if (loss) *loss = std::accumulate(rl.begin(), rl.end(), 0.0) / ((double)n * m->out());
        return LEO2D_OK;
    });
}

int leo2d_mlp_train(leo2d_mlp* m, const float* x, const float* t, int64_t n, const leo2d_mlp_train_params* p,
                    double* epoch_loss)
{
    if (!m || !x || !t || !p || n <= 0 || p->epochs < 0 || p->batch <= 0) return LEO2D_ERR_ARG;
    return guarded(m, [&]() {
        hipStream_t s = m->stream;
        const int B = (int)std::min<int64_t>(p->batch, n);
        ensure_capacity(m, B);
        DevBuf X, T, idx, losses;
        dalloc(X, sizeof(float) * (size_t)n * m->in(), "training inputs");
        dalloc(T, sizeof(float) * (size_t)n * m->out(), "training targets");
        dalloc(idx, sizeof(int64_t) * (size_t)n, "training order");
        dalloc(losses, sizeof(double) * (size_t)n, "training losses");
        check(hipMemcpyAsync(X.p, x, sizeof(float) * (size_t)n * m->in(), hipMemcpyHostToDevice, s), "training inputs");
        check(hipMemcpyAsync(T.p, t, sizeof(float) * (size_t)n * m->out(), hipMemcpyHostToDevice, s), "training targets");
        std::vector<int64_t> order((size_t)n);
        std::iota(order.begin(), order.end(), (int64_t)0);
        std::mt19937_64 rng(p->seed);
        std::vector<double> rl((size_t)n);
        for (int e = 0; e < p->epochs; ++e) {
            std::shuffle(order.begin(), order.end(), rng);
            check(hipMemcpyAsync(idx.p, order.data(), sizeof(int64_t) * (size_t)n, hipMemcpyHostToDevice, s), "order");
            for (int64_t b0 = 0; b0 < n; b0 += B) {
                const int rows = (int)std::min<int64_t>(B, n - b0);
                batch_gradients(m, static_cast<const float*>(X.p), static_cast<const float*>(T.p),
                                static_cast<const int64_t*>(idx.p) + b0, rows, static_cast<double*>(losses.p) + b0, nullptr);
                ++m->adam_step;
                leo2d::ParamArgs pa = adam_args(m, p);
                leo2d::adam_corrections(p->beta1, p->beta2, (int)m->adam_step, &pa.c1, &pa.c2);
                check(leo2d::launch_params(pa, s), "adam");
            }
            check(hipMemcpyAsync(rl.data(), losses.p, sizeof(double) * (size_t)n, hipMemcpyDeviceToHost, s), "loss");
            check(hipStreamSynchronize(s), "epoch");
            if (epoch_loss) epoch_loss[e] = std::accumulate(rl.begin(), rl.end(), 0.0) / ((double)n * m->out());
        }
        return LEO2D_OK;
    });
}

// Several networks trained together: each epoch of each network is captured once
// as a graph (gather, forward, backward, Adam for every mini-batch, the Adam step
// read from a device counter) and replayed per epoch on the network's own stream,
// so the networks' short launches run side by side and the host issues one launch
// per network and epoch.  Each network's arithmetic, shuffles and updates are
// those of leo2d_mlp_train with its own seed, bit for bit.
int leo2d_mlp_train_ensemble(leo2d_mlp* const* nets, int32_t count, const float* x, const float* t, int64_t n,
                             const leo2d_mlp_train_params* p, const uint64_t* seeds, double* losses)
{
    if (!nets || count < 1 || !x || !t || !p || !seeds || n <= 0 || p->epochs < 0 || p->batch <= 0)
        return LEO2D_ERR_ARG;
    leo2d_mlp* m0 = nets[0];
    return guarded(m0, [&]() {
        for (int k = 0; k < count; ++k) {
            if (!nets[k]) throw ArgError("null network");
            if (nets[k]->dims != m0->dims || nets[k]->device != m0->device)
                throw ArgError("ensemble members differ in shape or device");
        }
        const int B = (int)std::min<int64_t>(p->batch, n);
        const int64_t steps = (n + B - 1) / B;
        const int64_t total = steps * (int64_t)p->epochs;
        if (total + 1 > 0x7fffffffLL) throw ArgError("too many training steps");
        if (p->epochs == 0) return LEO2D_OK;
        leo2d::DevPool::Use none(nullptr);   // buffers several streams use are not pooled
        hipStream_t s0 = m0->stream;
        DevBuf X, T;
        dalloc(X, sizeof(float) * (size_t)n * m0->in(), "training inputs");
        dalloc(T, sizeof(float) * (size_t)n * m0->out(), "training targets");
        check(hipMemcpyAsync(X.p, x, sizeof(float) * (size_t)n * m0->in(), hipMemcpyHostToDevice, s0), "training inputs");
        check(hipMemcpyAsync(T.p, t, sizeof(float) * (size_t)n * m0->out(), hipMemcpyHostToDevice, s0),
              "training targets");
        check(hipStreamSynchronize(s0), "training data");
        struct Member {
            DevBuf idx, loss, corr, ctr;
            std::vector<int64_t> order;
            std::vector<double> rl;
            std::mt19937_64 rng;
            hipGraphExec_t exec = nullptr;
        };
        std::vector<Member> mem((size_t)count);
        auto release = [&]() {
            for (auto& q : mem)
                if (q.exec) (void)hipGraphExecDestroy(q.exec);
        };
        try {
            for (int k = 0; k < count; ++k) {
                leo2d_mlp* m = nets[k];
                Member& q = mem[(size_t)k];
                hipStream_t s = m->stream;
                ensure_capacity(m, B);
                dalloc(q.idx, sizeof(int64_t) * (size_t)n, "training order");
                dalloc(q.loss, sizeof(double) * (size_t)n, "training losses");
                dalloc(q.ctr, sizeof(int), "adam step");
                // bias corrections of every step of this call, from the network's own step count
                std::vector<float> corr((size_t)(2 * (total + 1)));
                for (int64_t i = 0; i <= total; ++i)
                    leo2d::adam_corrections(p->beta1, p->beta2, (int)(m->adam_step + 1 + i), &corr[2 * (size_t)i],
                                            &corr[2 * (size_t)i + 1]);
                to_device_f32(q.corr, corr, s);
                const int before = -1;   // the gather of a step advances it
                check(hipMemcpyAsync(q.ctr.p, &before, sizeof(int), hipMemcpyHostToDevice, s), "adam step");
                check(hipStreamSynchronize(s), "training setup");
                q.order.resize((size_t)n);
                std::iota(q.order.begin(), q.order.end(), (int64_t)0);
                q.rng.seed(seeds[k]);
                q.rl.resize((size_t)n);
                // one epoch, captured
                hipGraph_t graph = nullptr;
                check(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal), "epoch capture");
                try {
                    for (int64_t b0 = 0; b0 < n; b0 += B) {
                        const int rows = (int)std::min<int64_t>(B, n - b0);
                        batch_gradients(m, static_cast<const float*>(X.p), static_cast<const float*>(T.p),
                                        static_cast<const int64_t*>(q.idx.p) + b0, rows,
                                        static_cast<double*>(q.loss.p) + b0, static_cast<int*>(q.ctr.p));
                        leo2d::ParamArgs pa = adam_args(m, p);
                        pa.corr = f32(q.corr);
                        pa.ctr = static_cast<const int*>(q.ctr.p);
                        check(leo2d::launch_params(pa, s), "adam");
                    }
                } catch (...) {
                    (void)hipStreamEndCapture(s, &graph);
                    if (graph) (void)hipGraphDestroy(graph);
                    throw;
                }
                check(hipStreamEndCapture(s, &graph), "epoch capture");
                const hipError_t ie = hipGraphInstantiate(&q.exec, graph, nullptr, nullptr, 0);
                (void)hipGraphDestroy(graph);
                if (ie != hipSuccess) {
                    q.exec = nullptr;
                    check(ie, "epoch graph");
                }
            }
            for (int e = 0; e < p->epochs; ++e) {
                // every member's epoch is queued before any loss is copied back: a copy into
                // pageable host memory returns only when its stream has drained
                for (int k = 0; k < count; ++k) {
                    Member& q = mem[(size_t)k];
                    hipStream_t s = nets[k]->stream;
                    std::shuffle(q.order.begin(), q.order.end(), q.rng);
                    check(hipMemcpyAsync(q.idx.p, q.order.data(), sizeof(int64_t) * (size_t)n, hipMemcpyHostToDevice, s),
                          "order");
                    check(hipGraphLaunch(q.exec, s), "epoch launch");
                }
                for (int k = 0; k < count; ++k) {
                    Member& q = mem[(size_t)k];
                    check(hipMemcpyAsync(q.rl.data(), q.loss.p, sizeof(double) * (size_t)n, hipMemcpyDeviceToHost,
                                         nets[k]->stream),
                          "loss");
                }
                for (int k = 0; k < count; ++k) {
                    Member& q = mem[(size_t)k];
                    check(hipStreamSynchronize(nets[k]->stream), "epoch");
                    if (losses)
                        losses[(size_t)k * p->epochs + e] =
                            std::accumulate(q.rl.begin(), q.rl.end(), 0.0) / ((double)n * nets[k]->out());
                }
            }
        } catch (...) {
            release();
            throw;
        }
        release();
        for (int k = 0; k < count; ++k) nets[k]->adam_step += total;
        return LEO2D_OK;
    });
}

int leo2d_mlp_ensemble(leo2d_mlp* const* nets, int32_t count, const float* x, int64_t n, int32_t blocks, float* mean,
                       float* spread)
{
    if (!nets || count < 1 || !x || n < 0 || !spread || blocks < 1) return LEO2D_ERR_ARG;
    leo2d_mlp* m0 = nets[0];
    if (m0->out() % blocks != 0) return LEO2D_ERR_ARG;
    for (int e = 0; e < count; ++e)
        if (!nets[e] || nets[e]->dims != m0->dims || nets[e]->device != m0->device) return LEO2D_ERR_ARG;
    return guarded(m0, [&]() {
        // The inputs go up and are rounded once, on the first network's stream; the networks
        // run side by side on their own streams after it, and the statistics wait for them all:
        // when the first network's stream has drained, and its buffers go back, all have.
        const int chunk = 4096;
        const int out = m0->out();
        hipStream_t s0 = m0->stream;
        DevBuf Ys, dmean, dspread;
        dalloc(Ys, sizeof(float) * (size_t)count * chunk * out, "ensemble outputs");
        if (mean) dalloc(dmean, sizeof(float) * (size_t)chunk * out, "ensemble mean");
        dalloc(dspread, sizeof(float) * (size_t)std::max<int64_t>(n, 1) * blocks, "ensemble spread");
        struct Event {
            hipEvent_t e = nullptr;
            Event() { check(hipEventCreateWithFlags(&e, hipEventDisableTiming), "ensemble event"); }
            Event(const Event&) = delete;
            Event& operator=(const Event&) = delete;
            ~Event() { (void)hipEventDestroy(e); }
        };
        std::vector<Event> done((size_t)count);   // [0]: inputs ready
        for (int e = 0; e < count; ++e) ensure_capacity(nets[e], std::min<int64_t>(n, chunk));
        try {
            for (int64_t r0 = 0; r0 < n; r0 += chunk) {
                const int rows = (int)std::min<int64_t>(chunk, n - r0);
                upload_inputs(m0, x + (size_t)r0 * m0->in(), rows);
                check(hipEventRecord(done[0].e, s0), "ensemble inputs");
                for (int e = 0; e < count; ++e) {
                    leo2d_mlp* m = nets[e];
                    if (m != m0) check(hipStreamWaitEvent(m->stream, done[0].e, 0), "ensemble inputs");
                    forward(m, rows, static_cast<float*>(Ys.p) + (size_t)e * chunk * out, bf(m0->X16));
                    if (m != m0) check(hipEventRecord(done[(size_t)e].e, m->stream), "ensemble forward");
                }
                for (int e = 0; e < count; ++e)
                    if (nets[e] != m0) check(hipStreamWaitEvent(s0, done[(size_t)e].e, 0), "ensemble forward");
                check(leo2d::launch_ensemble_stats(static_cast<const float*>(Ys.p), count, (int64_t)chunk * out, rows, out,
                                                   blocks, f32(dmean), f32(dspread, r0 * blocks), s0),
                      "ensemble stats");
                if (mean)
                    check(hipMemcpyAsync(mean + (size_t)r0 * out, dmean.p, sizeof(float) * (size_t)rows * out,
                                         hipMemcpyDeviceToHost, s0),
                          "ensemble mean");
            }
            if (n) check(hipMemcpyAsync(spread, dspread.p, sizeof(float) * n * blocks, hipMemcpyDeviceToHost, s0), "ensemble spread");
            check(hipStreamSynchronize(s0), "ensemble");
        } catch (...) {
            (void)hipDeviceSynchronize();   // nothing may still run on the buffers freed here
            throw;
        }
        return LEO2D_OK;
    });
}

}  // extern "C"
