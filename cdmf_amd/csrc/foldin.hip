// C ABI of the fold-in extension (include/cdmf_foldin.h): the warm-start MLP
// (training and inference on the device with kernels/mlp_kernels.hip) and
// the fold-in of new rows (kernels/foldin_kernels.hip).
#include "cdmf_foldin.h"
#include "ccd_kernels.h"
#include "host_pipe.h"
#include "layout.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <numeric>
#include <string>
#include <vector>

namespace {

template <class T>
hipError_t dalloc(T** p, size_t count) {
    *p = nullptr;
    return hipMalloc(reinterpret_cast<void**>(p), sizeof(T) * (count ? count : 1));
}

void dfree(void* p) {
    if (p) (void)hipFree(p);
}

// Most device memory that rows on their way through a network leave behind.
constexpr size_t KEEP_BYTES = (size_t)1 << 30;

// Grow-only device buffer.
template <class T>
hipError_t ensure(T** p, size_t* cap, size_t count) {
    if (*p && *cap >= count) return hipSuccess;
    dfree(*p);
    *p = nullptr;
    *cap = 0;
    const hipError_t e = dalloc(p, count);
    if (e == hipSuccess) *cap = count;
    return e;
}

uint64_t splitmix(uint64_t& s) {
    uint64_t z = (s += 0x9e3779b97f4a7c15ull);
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}

double uniform01(uint64_t& s) { return (double)(splitmix(s) >> 11) * (1.0 / 9007199254740992.0); }

}  // namespace

// The runtime's own error is cleared: the next call's launches would find it.
static int obj_err(std::string& err, int code, const std::string& msg) {
    if (code == CCD_ERR_HIP || code == CCD_ERR_ALLOC) (void)hipGetLastError();
    err = msg;
    return code;
}

#define OBJ_TRY(o, expr)                                                                                     \
    do {                                                                                                     \
        hipError_t e_ = (expr);                                                                              \
        if (e_ != hipSuccess)                                                                                \
            return obj_err((o)->err, CCD_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_));        \
    } while (0)

// ------------------------------------------------------------------ MLP ---
struct ccd_mlp {
    int device = 0;
    hipStream_t stream = nullptr;
    ccd::HostPipe pipe;
    std::string err;
    uint32_t in = 0, hid = 0, out = 0;
    uint64_t np = 0;
    size_t oW1 = 0, ob1 = 0, oW2 = 0, ob2 = 0, oW3 = 0, ob3 = 0;
    float* P = nullptr;  // FP32 master parameters
    uint16_t* P16 = nullptr;
    bool p16_valid = false;
    // packed bfloat16 weights of the matrix-core inference path (mlp_mfma.hip)
    uint16_t* pk = nullptr;
    float* pkb = nullptr;
    uint32_t kin = 0, nout = 0;
    bool pk_valid = false;
    float *G = nullptr, *mom = nullptr, *vel = nullptr;
    uint64_t step = 0;
    // affine maps: inputs x_n = (x - in_sub) in_mul; outputs y = (y_n - out_sub) out_mul;
    // training targets t_n = (t - tgt_sub) tgt_mul
    float *in_sub = nullptr, *in_mul = nullptr, *out_sub = nullptr, *out_mul = nullptr, *tgt_sub = nullptr,
          *tgt_mul = nullptr;
    bool has_norm = false;
    // workspace for up to cap rows
    size_t cap = 0;
    float *Xn = nullptr, *Z1 = nullptr, *A1 = nullptr, *Z2 = nullptr, *A2 = nullptr, *Yn = nullptr, *Tn = nullptr,
          *dY = nullptr, *dZ2 = nullptr, *dZ1 = nullptr;
    float *I1 = nullptr, *I2 = nullptr;  // hidden activations of inference
    size_t cap_i1 = 0, cap_i2 = 0;
    double *part = nullptr, *loss = nullptr;
    size_t cap_loss = 0;
    float* gpart = nullptr;  // split-K partials of the weight-gradient products
    uint64_t gpart_cap = 0;
    // training set
    float *X = nullptr, *T = nullptr;
    uint32_t* perm = nullptr;
    size_t cap_x = 0, cap_t = 0, cap_perm = 0;
};

namespace {

int mlp_workspace(ccd_mlp* m, size_t rows) {
    if (rows <= m->cap) return CCD_OK;
    m->cap = 0;
    float** bufs_h[] = {&m->Z1, &m->A1, &m->Z2, &m->A2, &m->dZ2, &m->dZ1};
    for (float** b : bufs_h) {
        dfree(*b);
        OBJ_TRY(m, dalloc(b, rows * m->hid));
    }
    float** bufs_o[] = {&m->Yn, &m->Tn, &m->dY};
    for (float** b : bufs_o) {
        dfree(*b);
        OBJ_TRY(m, dalloc(b, rows * m->out));
    }
    dfree(m->Xn);
    OBJ_TRY(m, dalloc(&m->Xn, rows * m->in));
    m->cap = rows;
    return CCD_OK;
}

const void* wptr(const ccd_mlp* m, bool b16, size_t off) {
    return b16 ? static_cast<const void*>(m->P16 + off) : static_cast<const void*>(m->P + off);
}

// Y = MLP(X) for n rows on stream s, hidden activations to A1 and A2.  infer: X and Y
// raw (the norms are applied on the way in and out); otherwise both
// standardised, and Z1, Z2 are kept for the gradients (n <= cap).
int mlp_layers(ccd_mlp* m, uint32_t n, const float* X, float* A1, float* A2, bool infer, bool b16, float* Y,
               hipStream_t s) {
    const bool norm = infer && m->has_norm;
    ccd::GemmArgs g{};
    g.A = X;
    g.sai = m->in, g.sap = 1, g.sbp = 1, g.sbj = m->in;
    g.M = n, g.N = m->hid, g.K = m->in, g.ldc = m->hid;
    if (norm) g.asub = m->in_sub, g.amul = m->in_mul;
    g.bias = wptr(m, b16, m->ob1), g.C = infer ? nullptr : m->Z1, g.C2 = A1;
    OBJ_TRY(m, ccd::launch_gemm(g, wptr(m, b16, m->oW1), b16, ccd::GEMM_BIAS_GELU, s));
    g.asub = g.amul = nullptr;
    g.A = A1;
    g.sai = m->hid, g.sbj = m->hid, g.K = m->hid;
    g.bias = wptr(m, b16, m->ob2), g.C = infer ? nullptr : m->Z2, g.C2 = A2;
    OBJ_TRY(m, ccd::launch_gemm(g, wptr(m, b16, m->oW2), b16, ccd::GEMM_BIAS_GELU, s));
    g.A = A2;
    g.N = m->out, g.ldc = m->out;
    if (norm) g.csub = m->out_sub, g.cmul = m->out_mul;
    g.bias = wptr(m, b16, m->ob3), g.C = Y, g.C2 = nullptr;
    OBJ_TRY(m, ccd::launch_gemm(g, wptr(m, b16, m->oW3), b16, ccd::GEMM_STORE, s));
    return CCD_OK;
}

// Gradient of mean((Yn - Tn)^2) into G, loss into *loss_dev (after mlp_layers, FP32).
int mlp_backward_ws(ccd_mlp* m, uint32_t n, double* loss_dev, hipStream_t s) {
    OBJ_TRY(m, ccd::launch_mse(m->Yn, m->Tn, (uint64_t)n * m->out, m->dY, m->part, loss_dev, s));
    ccd::GemmArgs g{};
    // gW3 [out][hid] = dY^T A2; the bias gradients are the row sums of the left operands
    g.A = m->dY, g.sai = 1, g.sap = m->out;
    g.sbp = m->hid, g.sbj = 1;
    g.M = m->out, g.N = m->hid, g.K = n, g.ldc = m->hid, g.C = m->G + m->oW3;
    g.part = m->gpart, g.part_cap = m->gpart_cap, g.rowsum = m->G + m->ob3;
    OBJ_TRY(m, ccd::launch_gemm(g, m->A2, false, ccd::GEMM_STORE, s));
    // dZ2 = (dY W3) * gelu'(Z2)
    g = ccd::GemmArgs{};
    g.A = m->dY, g.sai = m->out, g.sap = 1, g.sbp = m->hid, g.sbj = 1;
    g.M = n, g.N = m->hid, g.K = m->out, g.ldc = m->hid, g.C = m->dZ2, g.aux = m->Z2;
    OBJ_TRY(m, ccd::launch_gemm(g, m->P + m->oW3, false, ccd::GEMM_GELU_GRAD, s));
    // gW2 [hid][hid] = dZ2^T A1
    g = ccd::GemmArgs{};
    g.A = m->dZ2, g.sai = 1, g.sap = m->hid, g.sbp = m->hid, g.sbj = 1;
    g.M = m->hid, g.N = m->hid, g.K = n, g.ldc = m->hid, g.C = m->G + m->oW2;
    g.part = m->gpart, g.part_cap = m->gpart_cap, g.rowsum = m->G + m->ob2;
    OBJ_TRY(m, ccd::launch_gemm(g, m->A1, false, ccd::GEMM_STORE, s));
    // dZ1 = (dZ2 W2) * gelu'(Z1)
    g = ccd::GemmArgs{};
    g.A = m->dZ2, g.sai = m->hid, g.sap = 1, g.sbp = m->hid, g.sbj = 1;
    g.M = n, g.N = m->hid, g.K = m->hid, g.ldc = m->hid, g.C = m->dZ1, g.aux = m->Z1;
    OBJ_TRY(m, ccd::launch_gemm(g, m->P + m->oW2, false, ccd::GEMM_GELU_GRAD, s));
    // gW1 [hid][in] = dZ1^T Xn
    g = ccd::GemmArgs{};
    g.A = m->dZ1, g.sai = 1, g.sap = m->hid, g.sbp = m->in, g.sbj = 1;
    g.M = m->hid, g.N = m->in, g.K = n, g.ldc = m->in, g.C = m->G + m->oW1;
    g.part = m->gpart, g.part_cap = m->gpart_cap, g.rowsum = m->G + m->ob1;
    OBJ_TRY(m, ccd::launch_gemm(g, m->Xn, false, ccd::GEMM_STORE, s));
    return CCD_OK;
}

int mlp_sync_bf16(ccd_mlp* m, hipStream_t s) {
    if (m->p16_valid) return CCD_OK;
    OBJ_TRY(m, ccd::launch_to_bf16(m->P, m->P16, m->np, s));
    m->p16_valid = true;
    return CCD_OK;
}

// Packed weights of the matrix-core path (allocated on first use).
int mlp_sync_mfma(ccd_mlp* m, hipStream_t s) {
    if (m->hid != ccd::MLP_MFMA_HIDDEN || ((m->in + 31) & ~31u) > ccd::MLP_MFMA_MAX_KIN ||
        m->out > ccd::MLP_MFMA_HIDDEN)
        return obj_err(m->err, CCD_ERR_UNSUPPORTED, "matrix-core inference needs 256 hidden units, in <= 288, out <= 256");
    if (m->pk_valid) return CCD_OK;
    if (!m->pk) {
        m->kin = (m->in + 31) & ~31u;
        m->nout = (m->out + 15) & ~15u;
        const size_t H = ccd::MLP_MFMA_HIDDEN;
        OBJ_TRY(m, dalloc(&m->pk, H * m->kin + H * H + (size_t)m->nout * H));
        OBJ_TRY(m, dalloc(&m->pkb, 2 * H + m->nout));
    }
    const size_t H = ccd::MLP_MFMA_HIDDEN;
    uint16_t* W1 = m->pk;
    uint16_t* W2 = W1 + H * m->kin;
    uint16_t* W3 = W2 + H * H;
    OBJ_TRY(m, ccd::launch_mlp_pack(m->P, m->in, m->out, m->kin, m->nout, W1, W2, W3, m->pkb, m->pkb + H,
                                    m->pkb + 2 * H, s));
    m->pk_valid = true;
    return CCD_OK;
}

// Y (device, raw) = MLP(X (device, raw)) for any row count.  mode 0: FP32;
// 1: bfloat16 weights, FP32 arithmetic (chunked GEMMs through the
// workspace); 2: the matrix-core path, one launch (bfloat16 weights and
// activations, FP32 accumulation).
int mlp_forward_dev(ccd_mlp* m, uint64_t rows, const float* X, float* Y, int mode, hipStream_t s) {
    if (mode == 2) {
        if (int rc = mlp_sync_mfma(m, s)) return rc;
        if (rows > 0xffffffffull) return obj_err(m->err, CCD_ERR_INVALID, "too many rows");
        const size_t H = ccd::MLP_MFMA_HIDDEN;
        ccd::MlpInferArgs g{};
        g.X = X, g.Y = Y, g.rows = (uint32_t)rows, g.in = m->in, g.out = m->out, g.kin = m->kin, g.nout = m->nout;
        g.W1 = m->pk, g.W2 = m->pk + H * m->kin, g.W3 = m->pk + H * m->kin + H * H;
        g.b1 = m->pkb, g.b2 = m->pkb + H, g.b3 = m->pkb + 2 * H;
        if (m->has_norm) g.in_sub = m->in_sub, g.in_mul = m->in_mul, g.out_sub = m->out_sub, g.out_mul = m->out_mul;
        OBJ_TRY(m, ccd::launch_mlp_infer(g, s));
        return CCD_OK;
    }
    const bool b16 = mode == 1;
    // rows at a time: three waves of 64 x 64 outputs for every SIMD at 256
    // hidden units, at most 2 x 64 MB of activations
    const uint32_t chunk = std::max<uint32_t>(std::min<uint32_t>(65536u, (1u << 24) / m->hid), 4096u);
    const size_t most = (size_t)std::min<uint64_t>(chunk, rows) * m->hid;
    OBJ_TRY(m, ensure(&m->I1, &m->cap_i1, most));
    OBJ_TRY(m, ensure(&m->I2, &m->cap_i2, most));
    if (b16)
        if (int rc = mlp_sync_bf16(m, s)) return rc;
    for (uint64_t r0 = 0; r0 < rows; r0 += chunk) {
        const uint32_t n = (uint32_t)std::min<uint64_t>(chunk, rows - r0);
        if (int rc = mlp_layers(m, n, X + r0 * m->in, m->I1, m->I2, true, b16, Y + r0 * m->out, s)) return rc;
    }
    return CCD_OK;
}

}  // namespace

extern "C" {

int32_t ccd_mlp_create(int32_t device, uint32_t in, uint32_t hidden, uint32_t out, uint64_t seed, ccd_mlp** mo) {
    if (!mo) return CCD_ERR_INVALID;
    *mo = nullptr;
    if (in == 0 || hidden == 0 || out == 0 || in > 4096 || hidden > 4096 || out > 4096) return CCD_ERR_INVALID;
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count <= 0) return CCD_ERR_HIP;
    if (device < 0 || device >= count) return CCD_ERR_INVALID;
    ccd_mlp* m = new (std::nothrow) ccd_mlp();
    if (!m) return CCD_ERR_ALLOC;
    m->device = device;
    m->in = in, m->hid = hidden, m->out = out;
    m->oW1 = 0;
    m->ob1 = m->oW1 + (size_t)hidden * in;
    m->oW2 = m->ob1 + hidden;
    m->ob2 = m->oW2 + (size_t)hidden * hidden;
    m->oW3 = m->ob2 + hidden;
    m->ob3 = m->oW3 + (size_t)out * hidden;
    m->np = m->ob3 + out;
    m->gpart_cap = 16ull * std::max<uint64_t>({(uint64_t)hidden * (hidden + 1), (uint64_t)hidden * (in + 1),
                                                (uint64_t)out * (hidden + 1)});
    // Glorot-uniform weights, zero biases, seeded
    std::vector<float> P(m->np, 0.0f);
    uint64_t st = seed ^ 0x6d6c7021ull;
    auto fill = [&](size_t off, uint32_t fo, uint32_t fi) {
        const double a = std::sqrt(6.0 / (double)(fi + fo));
        for (size_t q = 0; q < (size_t)fo * fi; ++q) P[off + q] = (float)((2.0 * uniform01(st) - 1.0) * a);
    };
    fill(m->oW1, hidden, in);
    fill(m->oW2, hidden, hidden);
    fill(m->oW3, out, hidden);
    bool ok = hipSetDevice(device) == hipSuccess && hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking) == hipSuccess &&
              dalloc(&m->P, m->np) == hipSuccess && dalloc(&m->P16, m->np) == hipSuccess &&
              dalloc(&m->G, m->np) == hipSuccess && dalloc(&m->mom, m->np) == hipSuccess &&
              dalloc(&m->vel, m->np) == hipSuccess && dalloc(&m->in_sub, in) == hipSuccess &&
              dalloc(&m->in_mul, in) == hipSuccess && dalloc(&m->out_sub, out) == hipSuccess &&
              dalloc(&m->out_mul, out) == hipSuccess && dalloc(&m->tgt_sub, out) == hipSuccess &&
              dalloc(&m->tgt_mul, out) == hipSuccess && dalloc(&m->part, ccd::MSE_PARTS) == hipSuccess &&
              dalloc(&m->gpart, m->gpart_cap) == hipSuccess &&
              ccd::copy_sync(m->stream, m->P, P.data(), sizeof(float) * m->np, hipMemcpyHostToDevice) == hipSuccess &&
              ccd::launch_fill(m->mom, 0.0f, m->np, m->stream) == hipSuccess &&
              ccd::launch_fill(m->vel, 0.0f, m->np, m->stream) == hipSuccess &&
              hipStreamSynchronize(m->stream) == hipSuccess;
    if (!ok) {
        ccd_mlp_destroy(m);
        (void)hipGetLastError();
        return CCD_ERR_HIP;
    }
    *mo = m;
    return CCD_OK;
}

int32_t ccd_mlp_destroy(ccd_mlp* m) {
    if (!m) return CCD_OK;
    (void)hipSetDevice(m->device);
    if (m->stream) (void)hipStreamSynchronize(m->stream);
    void* bufs[] = {m->P, m->P16, m->G, m->mom, m->vel, m->in_sub, m->in_mul, m->out_sub, m->out_mul, m->tgt_sub,
                    m->tgt_mul, m->gpart, m->Xn, m->Z1,
                    m->A1, m->Z2, m->A2, m->Yn, m->Tn, m->dY, m->dZ2, m->dZ1, m->I1, m->I2, m->part, m->loss, m->X, m->T, m->perm,
                    m->pk, m->pkb};
    for (void* b : bufs) dfree(b);
    if (m->stream) (void)hipStreamDestroy(m->stream);
    delete m;
    return CCD_OK;
}

const char* ccd_mlp_last_error(ccd_mlp* m) { return m ? m->err.c_str() : "null mlp"; }

uint64_t ccd_mlp_param_count(ccd_mlp* m) { return m ? m->np : 0; }

int32_t ccd_mlp_get_params(ccd_mlp* m, float* P) {
    if (!m || !P) return CCD_ERR_INVALID;
    OBJ_TRY(m, hipSetDevice(m->device));
    OBJ_TRY(m, hipStreamSynchronize(m->stream));
    OBJ_TRY(m, hipMemcpy(P, m->P, sizeof(float) * m->np, hipMemcpyDeviceToHost));
    return CCD_OK;
}

int32_t ccd_mlp_set_params(ccd_mlp* m, const float* P) {
    if (!m || !P) return CCD_ERR_INVALID;
    OBJ_TRY(m, hipSetDevice(m->device));
    OBJ_TRY(m, hipStreamSynchronize(m->stream));
    OBJ_TRY(m, ccd::copy_sync(m->stream, m->P, P, sizeof(float) * m->np, hipMemcpyHostToDevice));
    m->p16_valid = false;
    m->pk_valid = false;
    return CCD_OK;
}

int32_t ccd_mlp_set_norm(ccd_mlp* m, const float* in_mean, const float* in_std, const float* out_mean,
                         const float* out_std) {
    if (!m || !in_mean || !in_std || !out_mean || !out_std) return CCD_ERR_INVALID;
    // x_n = (x - mean) / std;  y = y_n * std + mean = (y_n - (-mean / std)) * std
    std::vector<float> a(m->in), b(m->in), c(m->out), d(m->out), e(m->out), g(m->out);
    for (uint32_t j = 0; j < m->in; ++j) {
        const float sd = std::max(in_std[j], 1e-12f);
        if (!std::isfinite(in_mean[j]) || !std::isfinite(sd)) return obj_err(m->err, CCD_ERR_INVALID, "non-finite norm");
        a[j] = in_mean[j];
        b[j] = 1.0f / sd;
    }
    for (uint32_t j = 0; j < m->out; ++j) {
        const float sd = std::max(out_std[j], 1e-12f);
        if (!std::isfinite(out_mean[j]) || !std::isfinite(sd)) return obj_err(m->err, CCD_ERR_INVALID, "non-finite norm");
        c[j] = -out_mean[j] / sd;
        d[j] = sd;
        e[j] = out_mean[j];
        g[j] = 1.0f / sd;
    }
    OBJ_TRY(m, hipSetDevice(m->device));
    OBJ_TRY(m, hipStreamSynchronize(m->stream));
    OBJ_TRY(m, ccd::copy_sync(m->stream, m->in_sub, a.data(), 4 * m->in, hipMemcpyHostToDevice));
    OBJ_TRY(m, ccd::copy_sync(m->stream, m->in_mul, b.data(), 4 * m->in, hipMemcpyHostToDevice));
    OBJ_TRY(m, ccd::copy_sync(m->stream, m->out_sub, c.data(), 4 * m->out, hipMemcpyHostToDevice));
    OBJ_TRY(m, ccd::copy_sync(m->stream, m->out_mul, d.data(), 4 * m->out, hipMemcpyHostToDevice));
    OBJ_TRY(m, ccd::copy_sync(m->stream, m->tgt_sub, e.data(), 4 * m->out, hipMemcpyHostToDevice));
    OBJ_TRY(m, ccd::copy_sync(m->stream, m->tgt_mul, g.data(), 4 * m->out, hipMemcpyHostToDevice));
    m->has_norm = true;
    return CCD_OK;
}

int32_t ccd_mlp_forward(ccd_mlp* m, uint64_t rows, const float* X, float* Y, int32_t bf16_weights) {
    if (!m || (rows && (!X || !Y))) return CCD_ERR_INVALID;
    if (rows == 0) return CCD_OK;
    OBJ_TRY(m, hipSetDevice(m->device));
    if (bf16_weights < 0 || bf16_weights > 2) return obj_err(m->err, CCD_ERR_INVALID, "bf16_weights must be 0, 1 or 2");
    // the rows pass through the training set's buffers
    OBJ_TRY(m, ensure(&m->X, &m->cap_x, rows * m->in));
    if (ensure(&m->T, &m->cap_t, rows * m->out) != hipSuccess) return obj_err(m->err, CCD_ERR_ALLOC, "output buffer");
    OBJ_TRY(m, m->pipe.in(m->device, m->X, X, 4 * rows * m->in, m->stream));
    if (int rc = mlp_forward_dev(m, rows, m->X, m->T, bf16_weights, m->stream)) {
        (void)hipStreamSynchronize(m->stream);  // the rows may still be on their way out of the caller's array
        return rc;
    }
    OBJ_TRY(m, m->pipe.out(m->device, Y, m->T, 4 * rows * m->out, m->stream));
    // Kept for the next call, where allocating takes longer than a small
    // call's kernels; a large call's copies dwarf it, and its memory goes back.
    if (4 * (m->cap_x + m->cap_t) > KEEP_BYTES) {
        dfree(m->X);
        dfree(m->T);
        m->X = m->T = nullptr;
        m->cap_x = m->cap_t = 0;
    }
    return CCD_OK;
}

int32_t ccd_mlp_loss_grad(ccd_mlp* m, uint64_t rows, const float* Xn, const float* Tn, double* loss, float* grad) {
    if (!m || !Xn || !Tn || !loss || !grad || rows == 0 || rows > (1u << 20)) return CCD_ERR_INVALID;
    OBJ_TRY(m, hipSetDevice(m->device));
    if (int rc = mlp_workspace(m, rows)) return rc;
    if (!m->loss) OBJ_TRY(m, dalloc(&m->loss, 1));
    OBJ_TRY(m, hipMemcpyAsync(m->Xn, Xn, 4 * rows * m->in, hipMemcpyHostToDevice, m->stream));
    OBJ_TRY(m, hipMemcpyAsync(m->Tn, Tn, 4 * rows * m->out, hipMemcpyHostToDevice, m->stream));
    if (int rc = mlp_layers(m, (uint32_t)rows, m->Xn, m->A1, m->A2, false, false, m->Yn, m->stream)) return rc;
    if (int rc = mlp_backward_ws(m, (uint32_t)rows, m->loss, m->stream)) return rc;
    OBJ_TRY(m, hipMemcpyAsync(loss, m->loss, sizeof(double), hipMemcpyDeviceToHost, m->stream));
    OBJ_TRY(m, ccd::copy_sync(m->stream, grad, m->G, 4 * m->np, hipMemcpyDeviceToHost));
    return CCD_OK;
}

int32_t ccd_mlp_train(ccd_mlp* m, uint64_t rows, const float* X, const float* T, uint32_t epochs, uint32_t batch,
                      float lr, uint64_t seed, double* epoch_loss) {
    if (!m || !X || !T || rows == 0 || batch == 0 || batch > 65536 || rows > 0xffffffffull || !(lr > 0.0f))
        return CCD_ERR_INVALID;
    OBJ_TRY(m, hipSetDevice(m->device));
    hipStream_t s = m->stream;
    if (int rc = mlp_workspace(m, batch)) return rc;
    OBJ_TRY(m, ensure(&m->X, &m->cap_x, rows * m->in));
    OBJ_TRY(m, ensure(&m->T, &m->cap_t, rows * m->out));
    OBJ_TRY(m, ensure(&m->perm, &m->cap_perm, rows));
    const uint64_t nb = (rows + batch - 1) / batch;
    OBJ_TRY(m, ensure(&m->loss, &m->cap_loss, nb));
    OBJ_TRY(m, m->pipe.in(m->device, m->X, X, 4 * rows * m->in, m->stream));
    OBJ_TRY(m, m->pipe.in(m->device, m->T, T, 4 * rows * m->out, m->stream));
    std::vector<uint32_t> perm(rows);
    std::vector<double> losses(nb);
    uint64_t st = seed ^ 0x747261696eull;
    const float b1 = 0.9f, b2 = 0.999f;
    double last = NAN;
    for (uint32_t ep = 0; ep < epochs; ++ep) {
        std::iota(perm.begin(), perm.end(), 0u);
        for (uint64_t i = rows - 1; i > 0; --i) std::swap(perm[i], perm[splitmix(st) % (i + 1)]);
        OBJ_TRY(m, hipStreamSynchronize(s));
        OBJ_TRY(m, ccd::copy_sync(m->stream, m->perm, perm.data(), 4 * rows, hipMemcpyHostToDevice));
        for (uint64_t q = 0; q < nb; ++q) {
            const uint32_t n = (uint32_t)std::min<uint64_t>(batch, rows - q * batch);
            const uint32_t* pr = m->perm + q * batch;
            OBJ_TRY(m, ccd::launch_affine_rows(m->X, pr, n, m->in, m->has_norm ? m->in_sub : nullptr, m->in_mul, m->Xn, s));
            OBJ_TRY(m, ccd::launch_affine_rows(m->T, pr, n, m->out, m->has_norm ? m->tgt_sub : nullptr, m->tgt_mul,
                                               m->Tn, s));
            if (int rc = mlp_layers(m, n, m->Xn, m->A1, m->A2, false, false, m->Yn, s)) return rc;
            if (int rc = mlp_backward_ws(m, n, m->loss + q, s)) return rc;
            ++m->step;
            ccd::AdamArgs ad{m->P, m->G, m->mom, m->vel, m->np, lr, b1, b2, 1e-8f,
                             1.0f - std::pow(b1, (float)m->step), 1.0f - std::pow(b2, (float)m->step)};
            OBJ_TRY(m, ccd::launch_adam(ad, s));
        }
        OBJ_TRY(m, hipStreamSynchronize(s));
        OBJ_TRY(m, hipMemcpy(losses.data(), m->loss, sizeof(double) * nb, hipMemcpyDeviceToHost));
        last = 0.0;
        for (double l : losses) last += l;
        last /= (double)nb;
    }
    m->p16_valid = false;
    m->pk_valid = false;
    if (epoch_loss) *epoch_loss = last;
    return CCD_OK;
}

}  // extern "C"

// ------------------------------------------------- allocation-free path ---
// Scratch of ccd_fold_rows_noalloc: one call's staged batch -- row pointer,
// long-row list, indices, values, start factors and result factors -- carved
// from one file-scope device array.  Every GPU the library runs on holds its
// own copy (about 20 MB) until the process ends.  Calls on one GPU share it:
// calls that overlap on one GPU race.  Nothing in it needs to start at zero.
namespace {
constexpr uint64_t NA_MAX_ROWS = 4096;
constexpr uint64_t NA_MAX_NNZ = 1ull << 21;
constexpr size_t na_round(size_t b) { return (b + 255) & ~(size_t)255; }
constexpr size_t NA_OFF_PTR = 0;
constexpr size_t NA_OFF_LONG = NA_OFF_PTR + na_round(4 * (NA_MAX_ROWS + 1));
constexpr size_t NA_OFF_IDX = NA_OFF_LONG + na_round(4 * NA_MAX_ROWS);
constexpr size_t NA_OFF_VAL = NA_OFF_IDX + na_round(4 * NA_MAX_NNZ);
constexpr size_t NA_OFF_W0 = NA_OFF_VAL + na_round(4 * NA_MAX_NNZ);
constexpr size_t NA_OFF_W = NA_OFF_W0 + na_round(4 * NA_MAX_ROWS * ccd::FOLD_KMAX);
constexpr size_t NA_BYTES = NA_OFF_W + na_round(4 * NA_MAX_ROWS * ccd::FOLD_KMAX);
}  // namespace

static __device__ __align__(256) unsigned char scratch[NA_BYTES];

namespace {
// Device address of `scratch` on each device, looked up once per device
// with that device current (the array's host-side name is no device
// address).
std::mutex g_scratch_mu;
std::vector<unsigned char*> g_scratch;

hipError_t scratch_on(int device, unsigned char** out) {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if ((size_t)device >= g_scratch.size()) g_scratch.resize((size_t)device + 1, nullptr);
    if (!g_scratch[device]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        g_scratch[device] = static_cast<unsigned char*>(p);
    }
    *out = g_scratch[device];
    return hipSuccess;
}
}  // namespace

// -------------------------------------------------------------- fold-in ---
struct ccd_fold {
    int device = 0;
    hipStream_t stream = nullptr;
    ccd::HostPipe pipe;
    std::string err;
    uint32_t k = 0;
    int64_t n = 0;
    float lambda = 0.0f;
    float* HT = nullptr;  // [n + 1][fold_ld(k)], ccd::FoldArgs; H and bad lie behind it
    float* H = nullptr;   // the caller's [k][n], transposed into HT
    uint32_t *ptr = nullptr, *idx = nullptr, *long_rows = nullptr;
    uint32_t* bad = nullptr;  // fold_check_device
    uint32_t nlong = 0, nfeat = 0;  // rows longer than FOLD_WAVE, and than FOLD_SHORT
    float *val = nullptr, *W0 = nullptr, *W = nullptr, *F = nullptr;
    size_t cap_ptr = 0, cap_idx = 0, cap_val = 0, cap_w0 = 0, cap_w = 0, cap_f = 0, cap_long = 0;
    hipEvent_t ea = nullptr, eb = nullptr;
    unsigned char* scratch = nullptr;  // this device's scratch (ccd_fold_rows_noalloc)
};

namespace {

// Ratings from which the index check runs on the device: the host's loop takes
// about 0.5 ns a rating (5 ms of a 9.9M-rating batch), the device's about 25 us
// with its wait.
constexpr uint64_t DEVICE_CHECK = 65536;

uint32_t fold_ld(uint32_t k) { return (k + 15) & ~15u; }  // row length of HT

int fold_check(ccd_fold* f, int64_t rows, const uint32_t* ptr, const uint32_t* idx, const float* val) {
    if (rows < 0 || rows > 0x7fffffff || !ptr || (rows && !idx && ptr[rows] > 0) || (rows && !val && ptr[rows] > 0))
        return obj_err(f->err, CCD_ERR_INVALID, "bad rows / null arrays");
    if (ptr[0] != 0) return obj_err(f->err, CCD_ERR_INVALID, "ptr[0] must be 0");
    for (int64_t i = 0; i < rows; ++i)
        if (ptr[i + 1] < ptr[i]) return obj_err(f->err, CCD_ERR_INVALID, "ptr not monotone");
    const uint64_t nnz = ptr[rows];
    if (nnz >= DEVICE_CHECK) return CCD_OK;  // indices: fold_check_device
    for (uint64_t e = 0; e < nnz; ++e)
        if ((int64_t)idx[e] >= f->n) return obj_err(f->err, CCD_ERR_INVALID, "column index out of range");
    return CCD_OK;
}

// The index check of a large batch on the device, before anything reads
// through the indices.  didx: the batch's indices, their copy in the stream.
int fold_check_device(ccd_fold* f, const uint32_t* didx, uint64_t nnz) {
    if (nnz < DEVICE_CHECK) return CCD_OK;
    uint32_t bad = 0;
    OBJ_TRY(f, ccd::launch_fill(reinterpret_cast<float*>(f->bad), 0.0f, 1, f->stream));
    OBJ_TRY(f, ccd::launch_index_check(didx, nnz, (uint32_t)f->n, f->bad, f->stream));
    OBJ_TRY(f, ccd::copy_sync(f->stream, &bad, f->bad, sizeof(bad), hipMemcpyDeviceToHost));
    return bad ? obj_err(f->err, CCD_ERR_INVALID, "column index out of range") : CCD_OK;
}

uint32_t count_long(int64_t rows, const uint32_t* ptr, uint32_t len) {
    uint32_t c = 0;
    for (int64_t i = 0; i < rows; ++i) c += ptr[i + 1] - ptr[i] > len ? 1u : 0u;
    return c;
}

// Rows of more than FOLD_WAVE ratings by falling length class (the binary
// exponent of length - 1; FOLD_WAVE and FOLD_SHORT are class bounds), in row
// order inside a class: the costliest blocks of a launch start first.
void list_long(int64_t rows, const uint32_t* ptr, uint32_t* out) {
    static_assert((ccd::FOLD_WAVE & (ccd::FOLD_WAVE - 1)) == 0 && (ccd::FOLD_SHORT & (ccd::FOLD_SHORT - 1)) == 0,
                  "length classes end at powers of two");
    uint32_t at[33] = {};
    auto cls = [&](int64_t i) { return __builtin_clz(ptr[i + 1] - ptr[i] - 1); };  // longer: smaller
    for (int64_t i = 0; i < rows; ++i)
        if (ptr[i + 1] - ptr[i] > ccd::FOLD_WAVE) ++at[cls(i) + 1];
    for (int q = 1; q < 33; ++q) at[q] += at[q - 1];
    for (int64_t i = 0; i < rows; ++i)
        if (ptr[i + 1] - ptr[i] > ccd::FOLD_WAVE) out[at[cls(i)]++] = (uint32_t)i;
}

int fold_upload(ccd_fold* f, int64_t rows, const uint32_t* ptr, const uint32_t* idx, const float* val,
                ccd::FoldArgs* a) {
    if (int rc = fold_check(f, rows, ptr, idx, val)) return rc;
    const uint64_t nnz = ptr[rows];
    std::vector<uint32_t> lr((size_t)count_long(rows, ptr, ccd::FOLD_WAVE));
    list_long(rows, ptr, lr.data());
    OBJ_TRY(f, hipSetDevice(f->device));
    OBJ_TRY(f, ensure(&f->ptr, &f->cap_ptr, (size_t)rows + 1));
    OBJ_TRY(f, ensure(&f->idx, &f->cap_idx, nnz));
    OBJ_TRY(f, ensure(&f->val, &f->cap_val, nnz));
    OBJ_TRY(f, ensure(&f->long_rows, &f->cap_long, lr.size()));
    OBJ_TRY(f, hipMemcpyAsync(f->ptr, ptr, 4 * ((size_t)rows + 1), hipMemcpyHostToDevice, f->stream));
    // lr goes out of scope here, so its copy is complete on return
    if (!lr.empty()) OBJ_TRY(f, ccd::copy_sync(f->stream, f->long_rows, lr.data(), 4 * lr.size(), hipMemcpyHostToDevice));
    f->nlong = (uint32_t)lr.size();
    f->nfeat = count_long(rows, ptr, ccd::FOLD_SHORT);
    if (nnz) {
        OBJ_TRY(f, f->pipe.in(f->device, f->idx, idx, 4 * nnz, f->stream));
        OBJ_TRY(f, f->pipe.in(f->device, f->val, val, 4 * nnz, f->stream));
        if (int rc = fold_check_device(f, f->idx, nnz)) return rc;
    }
    *a = ccd::FoldArgs{f->ptr, f->idx, f->val, f->HT, (uint32_t)rows, f->k, fold_ld(f->k), (uint32_t)f->n, 0, f->lambda};
    return CCD_OK;
}

}  // namespace

extern "C" {

int32_t ccd_fold_create(int32_t device, uint32_t k, int64_t n, const float* H, float lambda, ccd_fold** fo) {
    if (!fo) return CCD_ERR_INVALID;
    *fo = nullptr;
    if (k == 0 || k > (uint32_t)ccd::FOLD_KMAX || n <= 0 || n > 0x7fffffff || !H || !std::isfinite(lambda) ||
        lambda < 0.0f)
        return CCD_ERR_INVALID;
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count <= 0) return CCD_ERR_HIP;
    if (device < 0 || device >= count) return CCD_ERR_INVALID;
    ccd_fold* f = new (std::nothrow) ccd_fold();
    if (!f) return CCD_ERR_ALLOC;
    f->device = device, f->k = k, f->n = n, f->lambda = lambda;
    const size_t kn = (size_t)k * n, nht = ((size_t)n + 1) * fold_ld(k);
    bool ok = hipSetDevice(device) == hipSuccess && hipStreamCreateWithFlags(&f->stream, hipStreamNonBlocking) == hipSuccess &&
              hipEventCreate(&f->ea) == hipSuccess && hipEventCreate(&f->eb) == hipSuccess &&
              dalloc(&f->HT, nht + kn + 1) == hipSuccess;
    if (ok) {
        f->H = f->HT + nht;
        f->bad = reinterpret_cast<uint32_t*>(f->H + kn);
    }
    ok = ok && ccd::launch_fill(f->HT, 0.0f, nht, f->stream) == hipSuccess &&
         ccd::copy_sync(f->stream, f->H, H, 4 * kn, hipMemcpyHostToDevice) == hipSuccess &&
         ccd::launch_transpose(f->H, f->HT, k, (uint32_t)n, fold_ld(k), f->stream) == hipSuccess &&
         hipStreamSynchronize(f->stream) == hipSuccess && scratch_on(device, &f->scratch) == hipSuccess;
    if (!ok) {
        ccd_fold_destroy(f);
        (void)hipGetLastError();
        return CCD_ERR_HIP;
    }
    *fo = f;
    return CCD_OK;
}

int32_t ccd_fold_destroy(ccd_fold* f) {
    if (!f) return CCD_OK;
    (void)hipSetDevice(f->device);
    if (f->stream) (void)hipStreamSynchronize(f->stream);
    void* bufs[] = {f->HT, f->ptr, f->idx, f->val, f->W0, f->W, f->F, f->long_rows};
    for (void* b : bufs) dfree(b);
    if (f->ea) (void)hipEventDestroy(f->ea);
    if (f->eb) (void)hipEventDestroy(f->eb);
    if (f->stream) (void)hipStreamDestroy(f->stream);
    delete f;
    return CCD_OK;
}

const char* ccd_fold_last_error(ccd_fold* f) { return f ? f->err.c_str() : "null fold"; }

int32_t ccd_fold_features(ccd_fold* f, int64_t rows, const uint32_t* ptr, const uint32_t* idx, const float* val,
                          float* F) {
    if (!f || !F) return CCD_ERR_INVALID;
    ccd::FoldArgs a{};
    if (int rc = fold_upload(f, rows, ptr, idx, val, &a)) return rc;
    const size_t nf = (size_t)rows * (2 * f->k + 2);
    OBJ_TRY(f, ensure(&f->F, &f->cap_f, nf));
    OBJ_TRY(f, ccd::launch_fold_features(a, f->long_rows, f->nfeat, f->F, f->stream));
    OBJ_TRY(f, hipStreamSynchronize(f->stream));
    OBJ_TRY(f, f->pipe.out(f->device, F, f->F, 4 * nf, f->stream));
    return CCD_OK;
}

int32_t ccd_fold_rows(ccd_fold* f, int64_t rows, const uint32_t* ptr, const uint32_t* idx, const float* val,
                      const float* W0, int32_t sweeps, float* W, double* seconds) {
    if (!f || !W || sweeps < 0) return CCD_ERR_INVALID;
    ccd::FoldArgs a{};
    if (int rc = fold_upload(f, rows, ptr, idx, val, &a)) return rc;
    a.sweeps = sweeps;
    const size_t nw = (size_t)rows * f->k;
    OBJ_TRY(f, ensure(&f->W, &f->cap_w, nw));
    if (W0) {
        OBJ_TRY(f, ensure(&f->W0, &f->cap_w0, nw));
        if (nw) OBJ_TRY(f, ccd::copy_sync(f->stream, f->W0, W0, 4 * nw, hipMemcpyHostToDevice));
    }
    OBJ_TRY(f, hipEventRecord(f->ea, f->stream));
    OBJ_TRY(f, ccd::launch_fold_sweeps(a, f->long_rows, f->nlong, W0 ? f->W0 : nullptr, f->W, f->stream));
    OBJ_TRY(f, hipEventRecord(f->eb, f->stream));
    OBJ_TRY(f, hipEventSynchronize(f->eb));
    float ms = 0.0f;
    OBJ_TRY(f, hipEventElapsedTime(&ms, f->ea, f->eb));
    if (seconds) *seconds = ms * 1e-3;
    OBJ_TRY(f, f->pipe.out(f->device, W, f->W, 4 * nw, f->stream));
    return CCD_OK;
}

int32_t ccd_fold_rows_noalloc(ccd_fold* f, int64_t rows, const uint32_t* ptr, const uint32_t* idx, const float* val,
                              const float* W0, int32_t sweeps, float* W, double* seconds) {
    if (!f || !W || sweeps < 0) return CCD_ERR_INVALID;
    if (!f->scratch) return obj_err(f->err, CCD_ERR_STATE, "no scratch on this device");
    if (int rc = fold_check(f, rows, ptr, idx, val)) return rc;
    const uint64_t nnz = ptr[rows];
    if ((uint64_t)rows > NA_MAX_ROWS || nnz > NA_MAX_NNZ)
        return obj_err(f->err, CCD_ERR_INVALID,
                       "ccd_fold_rows_noalloc: at most 4096 rows and 2097152 ratings per call (got " +
                           std::to_string(rows) + " rows, " + std::to_string(nnz) + " ratings)");
    // long rows (one block each), listed in a fixed-size host array
    uint32_t lr[NA_MAX_ROWS];
    const uint32_t nlong = count_long(rows, ptr, ccd::FOLD_WAVE);
    list_long(rows, ptr, lr);
    unsigned char* S = f->scratch;
    uint32_t* dptr = reinterpret_cast<uint32_t*>(S + NA_OFF_PTR);
    uint32_t* dlong = reinterpret_cast<uint32_t*>(S + NA_OFF_LONG);
    uint32_t* didx = reinterpret_cast<uint32_t*>(S + NA_OFF_IDX);
    float* dval = reinterpret_cast<float*>(S + NA_OFF_VAL);
    float* dW0 = reinterpret_cast<float*>(S + NA_OFF_W0);
    float* dW = reinterpret_cast<float*>(S + NA_OFF_W);
    const size_t nw = (size_t)rows * f->k;
    OBJ_TRY(f, hipSetDevice(f->device));
    OBJ_TRY(f, hipMemcpyAsync(dptr, ptr, 4 * ((size_t)rows + 1), hipMemcpyHostToDevice, f->stream));
    if (nlong) OBJ_TRY(f, ccd::copy_sync(f->stream, dlong, lr, 4 * (size_t)nlong, hipMemcpyHostToDevice));
    if (nnz) {
        OBJ_TRY(f, hipMemcpyAsync(didx, idx, 4 * nnz, hipMemcpyHostToDevice, f->stream));
        OBJ_TRY(f, hipMemcpyAsync(dval, val, 4 * nnz, hipMemcpyHostToDevice, f->stream));
        if (int rc = fold_check_device(f, didx, nnz)) return rc;
    }
    if (W0 && nw) OBJ_TRY(f, ccd::copy_sync(f->stream, dW0, W0, 4 * nw, hipMemcpyHostToDevice));
    const ccd::FoldArgs a{dptr, didx, dval, f->HT, (uint32_t)rows, f->k, fold_ld(f->k), (uint32_t)f->n, sweeps,
                          f->lambda};
    OBJ_TRY(f, hipEventRecord(f->ea, f->stream));
    OBJ_TRY(f, ccd::launch_fold_sweeps(a, dlong, nlong, W0 ? dW0 : nullptr, dW, f->stream));
    OBJ_TRY(f, hipEventRecord(f->eb, f->stream));
    OBJ_TRY(f, hipEventSynchronize(f->eb));
    float ms = 0.0f;
    OBJ_TRY(f, hipEventElapsedTime(&ms, f->ea, f->eb));
    if (seconds) *seconds = ms * 1e-3;
    if (nw) OBJ_TRY(f, hipMemcpy(W, dW, 4 * nw, hipMemcpyDeviceToHost));
    return CCD_OK;
}

int32_t ccd_fold_warm(ccd_fold* f, ccd_mlp* m, int64_t rows, const uint32_t* ptr, const uint32_t* idx,
                      const float* val, int32_t sweeps, int32_t bf16_weights, float* W, double* seconds) {
    if (!f || !m || !W || sweeps < 0) return CCD_ERR_INVALID;
    if (m->in != 2 * f->k + 2 || m->out != f->k)
        return obj_err(f->err, CCD_ERR_INVALID, "the MLP must map 2k + 2 features to k outputs");
    if (m->device != f->device) return obj_err(f->err, CCD_ERR_INVALID, "MLP on another device");
    ccd::FoldArgs a{};
    if (int rc = fold_upload(f, rows, ptr, idx, val, &a)) return rc;
    a.sweeps = sweeps;
    const size_t nw = (size_t)rows * f->k, nf = (size_t)rows * (2 * f->k + 2);
    OBJ_TRY(f, ensure(&f->W, &f->cap_w, nw));
    OBJ_TRY(f, ensure(&f->W0, &f->cap_w0, nw));
    OBJ_TRY(f, ensure(&f->F, &f->cap_f, nf));
    OBJ_TRY(f, hipStreamSynchronize(m->stream));
    OBJ_TRY(f, hipEventRecord(f->ea, f->stream));
    OBJ_TRY(f, ccd::launch_fold_features(a, f->long_rows, f->nfeat, f->F, f->stream));
    int rc = CCD_OK;
    if (bf16_weights < 0 || bf16_weights > 2)
        rc = obj_err(f->err, CCD_ERR_INVALID, "bf16_weights must be 0, 1 or 2");
    else if ((rc = mlp_forward_dev(m, (uint64_t)rows, f->F, f->W0, bf16_weights, f->stream)))
        rc = obj_err(f->err, rc, "MLP: " + m->err);
    if (rc) {  // refused: the batch may still be on its way out of the caller's arrays
        (void)hipStreamSynchronize(f->stream);
        return rc;
    }
    OBJ_TRY(f, ccd::launch_fold_sweeps(a, f->long_rows, f->nlong, f->W0, f->W, f->stream));
    OBJ_TRY(f, hipEventRecord(f->eb, f->stream));
    OBJ_TRY(f, hipEventSynchronize(f->eb));
    float ms = 0.0f;
    OBJ_TRY(f, hipEventElapsedTime(&ms, f->ea, f->eb));
    if (seconds) *seconds = ms * 1e-3;
    OBJ_TRY(f, f->pipe.out(f->device, W, f->W, 4 * nw, f->stream));
    return CCD_OK;
}

}  // extern "C"
