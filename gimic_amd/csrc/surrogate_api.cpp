// C-ABI for the learned surrogate (include/gimic_hip.h, gimic_mlp_*): owns the
// FP32 master parameters, their BF16 copies, Adam state and work buffers,
// and sequences the kernels of surrogate.hip for training and inference.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <random>
#include <stdexcept>
#include <string>
#include <vector>

#include "../../include/gimic_hip.h"
#include "surrogate.h"

namespace gimic {
std::string &error_slot();
hipError_t shared_stream(hipStream_t *stream);
}

using namespace gimic;

namespace {

constexpr int kF = kMlpF, kK0 = kMlpK0, kH = kMlpH, kD = kMlpD, kNO = kMlpNO;

struct MlpError : std::runtime_error {
    int code;
    MlpError(int c, const std::string &m) : std::runtime_error(m), code(c) {}
};

void chk(hipError_t e, const char *what) {
    if (e != hipSuccess)
        throw MlpError(e == hipErrorOutOfMemory ? GIMIC_ENOMEM : GIMIC_EDEVICE,
                       std::string(what) + ": " + hipGetErrorString(e));
}

struct Buf {
    void *p = nullptr;
    size_t n = 0;
    ~Buf() {
        if (p) (void)hipFree(p);
    }
    void need(size_t bytes) {
        if (bytes <= n && p) return;
        if (p) (void)hipFree(p);
        p = nullptr;
        n = 0;
        const hipError_t e = hipMalloc(&p, bytes ? bytes : 256);
        if (e != hipSuccess) {
            p = nullptr;
            (void)hipGetLastError();  // else the next launch reports it
        }
        chk(e, "hipMalloc");
        n = bytes;
    }
    template <class T>
    T *as() const { return (T *)p; }
};

// a range of a Buf
struct Part {
    void *p = nullptr;
    template <class T>
    T *as() const { return (T *)p; }
};

}  // namespace

struct gimic_mlp {
    hipStream_t stream = nullptr;     // shared_stream() of its device
    hipStream_t user = nullptr;       // caller's stream, when set
    long long np = 0;                 // parameter count
    long long woff[kD + 1], boff[kD + 1];
    int kin[kD + 1], nout[kD + 1];
    Buf state;  // the parts below in one allocation (each costs about 1 ms)
    Part params, params_b, params_t, grad, adam_m, adam_v, freq, cs, oscale, loss;
    Buf X[kD + 1], dZ[kD], dY, part, bpart;
    long long cap = 0;  // batch capacity of the work buffers
    long long step = 0;
    ~gimic_mlp() {
        if (stream) (void)hipStreamSynchronize(stream);
    }
};

namespace {

std::string &errstr() { return error_slot(); }

hipStream_t work_stream(const gimic_mlp *n) { return n->user ? n->user : n->stream; }

template <class F>
int guard(F &&f) {
    try {
        f();
        errstr().clear();
        return GIMIC_OK;
    } catch (const MlpError &e) {
        errstr() = e.what();
        return e.code;
    } catch (const std::exception &e) {
        errstr() = e.what();
        return GIMIC_EINVAL;
    }
}

void reserve(gimic_mlp *n, long long P) {
    if (P <= n->cap) return;
    n->cap = 0;  // until every buffer is there: one that cannot grow is gone
    const size_t rows = (size_t)(P + 63) / 64 * 64;  // whole tiles
    for (int l = 0; l <= kD; l++) n->X[l].need(rows * n->kin[l] * 2);
    for (int l = 0; l < kD; l++) n->dZ[l].need(rows * kH * 2);
    n->dY.need(rows * kNO * 2);
    n->part.need((size_t)kMlpMaxRanges * kMlpParams * 4);
    n->bpart.need((size_t)mlp_tile_groups(1ll << 30) * kMlpBiasPart * 4);
    n->cap = P;
}

MlpTileArgs tile_args(gimic_mlp *n, long long P, const double *d_r) {
    MlpTileArgs a{};
    a.r = d_r;
    a.npts = P;
    a.freq = n->freq.as<float>();
    a.cs = n->cs.as<float>();
    a.oscale = n->oscale.as<float>();
    a.prm = n->params.as<float>();
    a.W = n->params_b.as<__bf16>();
    a.WT = n->params_t.as<__bf16>();
    return a;
}

// one batch: forward, backward, and the gradient (adam == 0) or an Adam step
void batch(gimic_mlp *n, long long P, const double *d_r, const double *d_target, float eps2,
           MlpAdamArgs o, hipStream_t s) {
    reserve(n, P);
    MlpTileArgs a = tile_args(n, P, d_r);
    a.target = d_target;
    a.eps2 = eps2;
    for (int l = 0; l <= kD; l++) a.X[l] = n->X[l].as<__bf16>();
    for (int l = 0; l < kD; l++) a.dZ[l] = n->dZ[l].as<__bf16>();
    a.dY = n->dY.as<__bf16>();
    a.bpart = n->bpart.as<float>();
    chk(mlp_tiles(a, true, s), "tiles");
    chk(mlp_dw(a, n->part.as<float>(), s), "dW");
    o.part = n->part.as<float>();
    o.bpart = n->bpart.as<float>();
    o.ranges = mlp_ranges(P);
    o.groups = mlp_tile_groups(P);
    o.grad = n->grad.as<float>();
    o.loss = n->loss.as<float>();
    o.prm = n->params.as<float>();
    o.m = n->adam_m.as<float>();
    o.v = n->adam_v.as<float>();
    o.W = n->params_b.as<__bf16>();
    o.WT = n->params_t.as<__bf16>();
    chk(mlp_adam(o, s), "adam");
}

}  // namespace

extern "C" {

int gimic_mlp_create(gimic_mlp **out, double sigma, const double *center_scale,
                     const double *out_scale, uint64_t seed) {
    return guard([&] {
        if (!out || !center_scale || !out_scale) throw MlpError(GIMIC_EINVAL, "null argument");
        auto *n = new gimic_mlp();
        try {
            chk(shared_stream(&n->stream), "shared_stream");
            long long off = 0;
            for (int l = 0; l <= kD; l++) {
                n->kin[l] = l == 0 ? kK0 : kH;
                n->nout[l] = l == kD ? kNO : kH;
                n->woff[l] = off;
                off += (long long)n->kin[l] * n->nout[l];
                n->boff[l] = off;
                off += n->nout[l];
            }
            n->np = off;
            // He-style initialisation, zero biases; frequencies ~ N(0, sigma^2)
            std::mt19937_64 rng(seed);
            std::normal_distribution<float> nd(0.f, 1.f);
            std::vector<float> p((size_t)off, 0.f);
            for (int l = 0; l <= kD; l++) {
                const float sc = std::sqrt((l == kD ? 1.f : 2.f) / (float)n->kin[l]);
                for (long long i = 0; i < (long long)n->kin[l] * n->nout[l]; i++)
                    p[n->woff[l] + i] = sc * nd(rng);
            }
            std::vector<float> fr(3 * kF);
            for (auto &x : fr) x = (float)sigma * nd(rng);
            float cs[4] = {(float)center_scale[0], (float)center_scale[1], (float)center_scale[2],
                           (float)center_scale[3]};
            float os[9];
            for (int i = 0; i < 9; i++) os[i] = (float)out_scale[i];
            hipStream_t s = work_stream(n);
            struct {
                Part *q;
                size_t bytes;
            } parts[] = {{&n->params, (size_t)off * 4}, {&n->params_b, (size_t)off * 2},
                         {&n->params_t, (size_t)kMlpTransposed * 2}, {&n->grad, (size_t)off * 4},
                         {&n->adam_m, (size_t)off * 4}, {&n->adam_v, (size_t)off * 4},
                         {&n->freq, fr.size() * 4}, {&n->cs, 16}, {&n->oscale, 36}, {&n->loss, 4}};
            size_t total = 0;
            for (auto &x : parts) total += (x.bytes + 255) / 256 * 256;
            n->state.need(total);
            total = 0;
            for (auto &x : parts) {
                x.q->p = n->state.as<unsigned char>() + total;
                total += (x.bytes + 255) / 256 * 256;
            }
            chk(hipMemcpyAsync(n->params.p, p.data(), off * 4, hipMemcpyHostToDevice, s), "copy");
            chk(hipMemsetAsync(n->adam_m.p, 0, off * 4, s), "memset");
            chk(hipMemsetAsync(n->adam_v.p, 0, off * 4, s), "memset");
            chk(hipMemcpyAsync(n->freq.p, fr.data(), fr.size() * 4, hipMemcpyHostToDevice, s), "copy");
            chk(hipMemcpyAsync(n->cs.p, cs, 16, hipMemcpyHostToDevice, s), "copy");
            chk(hipMemcpyAsync(n->oscale.p, os, 36, hipMemcpyHostToDevice, s), "copy");
            chk(mlp_cast(n->params.as<float>(), n->params_b.as<__bf16>(), n->params_t.as<__bf16>(), s),
                "cast");
            chk(hipStreamSynchronize(s), "sync");
        } catch (...) {
            delete n;
            throw;
        }
        *out = n;
    });
}

int gimic_mlp_destroy(gimic_mlp *n) {
    return guard([&] { delete n; });
}

int gimic_mlp_set_stream(gimic_mlp *n, void *stream) {
    return guard([&] {
        if (!n) throw MlpError(GIMIC_EINVAL, "null network");
        chk(hipStreamSynchronize(work_stream(n)), "sync");
        n->user = (hipStream_t)stream;
    });
}

int gimic_mlp_info(const gimic_mlp *n, long long *nparams, float *freqs) {
    return guard([&] {
        if (!n) throw MlpError(GIMIC_EINVAL, "null network");
        if (nparams) *nparams = n->np;
        if (freqs) chk(hipMemcpy(freqs, n->freq.p, 3 * kF * 4, hipMemcpyDeviceToHost), "copy");
    });
}

int gimic_mlp_params(gimic_mlp *n, float *host, int set) {
    return guard([&] {
        if (!n || !host) throw MlpError(GIMIC_EINVAL, "null argument");
        hipStream_t s = work_stream(n);
        if (set) {
            chk(hipMemcpyAsync(n->params.p, host, n->np * 4, hipMemcpyHostToDevice, s), "copy");
            chk(mlp_cast(n->params.as<float>(), n->params_b.as<__bf16>(), n->params_t.as<__bf16>(), s),
                "cast");
        } else {
            chk(hipMemcpyAsync(host, n->params.p, n->np * 4, hipMemcpyDeviceToHost, s), "copy");
        }
        chk(hipStreamSynchronize(s), "sync");
    });
}

int gimic_mlp_loss_grad(gimic_mlp *n, long long npts, const double *d_r, const double *d_target,
                        double eps, double *loss, float *host_grad) {
    return guard([&] {
        if (!n || npts <= 0 || !d_r || !d_target) throw MlpError(GIMIC_EINVAL, "bad argument");
        hipStream_t s = work_stream(n);
        batch(n, npts, d_r, d_target, (float)(eps * eps), MlpAdamArgs{}, s);
        float l = 0.f;
        chk(hipMemcpyAsync(&l, n->loss.p, 4, hipMemcpyDeviceToHost, s), "copy");
        if (host_grad)
            chk(hipMemcpyAsync(host_grad, n->grad.p, n->np * 4, hipMemcpyDeviceToHost, s), "copy");
        chk(hipStreamSynchronize(s), "sync");
        if (loss) *loss = l;
    });
}

int gimic_mlp_train_step(gimic_mlp *n, long long npts, const double *d_r, const double *d_target,
                         double eps, double lr, double *loss) {
    return guard([&] {
        if (!n || npts <= 0 || !d_r || !d_target) throw MlpError(GIMIC_EINVAL, "bad argument");
        hipStream_t s = work_stream(n);
        const float b1 = 0.9f, b2 = 0.999f;
        const float t = (float)(n->step + 1);
        MlpAdamArgs o{};
        o.adam = 1;
        o.lr = (float)lr;
        o.b1 = b1;
        o.b2 = b2;
        o.eps = 1e-8f;
        o.bc1 = 1.f - std::pow(b1, t);
        o.bc2 = 1.f - std::pow(b2, t);
        batch(n, npts, d_r, d_target, (float)(eps * eps), o, s);
        n->step++;
        if (loss) {
            float l = 0.f;
            chk(hipMemcpyAsync(&l, n->loss.p, 4, hipMemcpyDeviceToHost, s), "copy");
            chk(hipStreamSynchronize(s), "sync");
            *loss = l;
        }
    });
}

int gimic_mlp_predict(gimic_mlp *n, long long npts, const double *d_r, double *d_J, void *stream) {
    return guard([&] {
        if (!n || npts < 0 || (npts > 0 && (!d_r || !d_J))) throw MlpError(GIMIC_EINVAL, "bad argument");
        hipStream_t s = stream ? (hipStream_t)stream : work_stream(n);
        chk(mlp_infer(d_r, npts, n->freq.as<float>(), n->cs.as<float>(), n->params_b.as<__bf16>(),
                      n->params.as<float>(), n->oscale.as<float>(), d_J, s), "infer");
    });
}

int gimic_mlp_predict_unfused(gimic_mlp *n, long long npts, const double *d_r, double *d_J) {
    return guard([&] {
        if (!n || npts <= 0 || !d_r || !d_J) throw MlpError(GIMIC_EINVAL, "bad argument");
        hipStream_t s = work_stream(n);
        MlpTileArgs a = tile_args(n, npts, d_r);
        a.J = d_J;
        chk(mlp_tiles(a, false, s), "tiles");
        chk(hipStreamSynchronize(s), "sync");
    });
}

}  // extern "C"
