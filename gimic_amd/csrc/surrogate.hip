// Learned coordinate surrogate of the J-tensor field: kernels (gfx950).
//
// Network (per molecule): u = (r - centre) / scale;
//   f = [sin(2 pi B u), cos(2 pi B u), u, 0...]   (2F + 3 features, padded to K0)
//   h1..hD = SiLU(W_l h + b_l)                      (width H)
//   y = W_out hD + b_out                            (16 rows: 9 used + 1 log scale)
//   J_i = out_scale_i * y_i * exp(y_9)              (i < 9)
// The learned log amplitude y_9 lets the network follow a field whose size
// changes by orders of magnitude while y_0..8 stay of order one.
// Training: BF16 operands on MFMA (v_mfma_f32_16x16x32_bf16) with FP32
// accumulation, FP32 master weights and Adam.  With t = J / out_scale,
// n = sqrt(|t|^2 + eps^2) and u = t / n, the loss is the mean over points of
//   sum_i (y_i - u_i)^2 + (y_9 - log n)^2
// (direction and log magnitude fitted separately, so every point weighs the
// same whatever the size of its current; the prediction y e^{y_9} then has
// relative error ~ |y - u| + |y_9 - log n|).
// Inference: one fused kernel, activations in registers, weights in LDS.
//
// Training (mlp_tile_kernel, mlp_dw_kernel, mlp_adam_kernel): three launches a
// step.  The first takes 64-point tiles through the whole network and back:
// activations in LDS, pre-activations in registers, the weights of one stage
// streamed into LDS while the previous stage computes; it leaves the BF16
// activations and dZ in memory.  The second forms the weight gradients from
// them, split over point ranges; the third adds the ranges and applies Adam.
// As one strided GEMM per product with separate element-wise kernels a step of
// 16,384 points took 683 us in 38 launches; this takes 58 (33 of them the first).
// Products keep the k order of 32-wide MFMA steps throughout, so the BF16
// values are those of one FP32 accumulation per output whichever kernel.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "device_common.h"
#include "surrogate.h"

namespace gimic {

namespace {

__device__ __forceinline__ float silu(float z) { return z / (1.f + __expf(-z)); }
// exp of the log amplitude, bounded so that no product overflows FP32
__device__ __forceinline__ float amp(float z) { return __expf(fminf(z, 60.f)); }
__device__ __forceinline__ float dsilu(float z) {
    const float s = 1.f / (1.f + __expf(-z));
    return s * (1.f + z * (1.f - s));
}

}  // namespace

namespace {

// flat parameter layout: W_l[n][k] then b_l[n]
constexpr int kF = kMlpF, kK0 = kMlpK0, kH = kMlpH, kD = kMlpD, kNO = kMlpNO;
constexpr int kin(int l) { return l == 0 ? kK0 : kH; }
constexpr int nout(int l) { return l == kD ? kNO : kH; }
constexpr int woff(int l) { return l == 0 ? 0 : woff(l - 1) + (kin(l - 1) + 1) * nout(l - 1); }
constexpr int boff(int l) { return woff(l) + kin(l) * nout(l); }
static_assert(boff(kD) + kNO == kMlpParams, "parameter count");
// transposed BF16 weights of layers 1 .. D, WT_l[k][n]
constexpr int toff(int l) { return (l - 1) * kH * kH; }
// bias gradients of all layers, then the loss, per workgroup of the tile kernel
constexpr int kBiasN = kD * kH + kNO;

constexpr int kTP = 64;        // points per tile
constexpr int kAS = kK0 + 8;   // row stride of the activations in LDS (16-byte columns spread)
constexpr int kTileThreads = 512;
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef __bf16 v4bf __attribute__((ext_vector_type(4)));

// x as a value of which the compiler knows only that it is below `limit`: what
// is derived from it is computed where it is used (nine stages' addresses,
// kept over the loop over tiles, would be spilled)
__device__ __forceinline__ unsigned fresh(unsigned x, unsigned limit) {
    asm volatile("" : "+v"(x));
    __builtin_assume(x < limit);
    return x;
}

// this thread's share of a ROWS x K weight matrix, from global memory and
// into LDS rows of K + 8 (PAD > K: zero-filled to PAD + 8)
template <int ROWS, int K>
__device__ __forceinline__ void fetch_w(const __bf16 *W, v4u (&st)[5], unsigned thread) {
    const unsigned tid = fresh(thread, kTileThreads);
#pragma unroll
    for (int i = 0; i < (ROWS * K / 8 + kTileThreads - 1) / kTileThreads; i++) {
        const unsigned u = tid + kTileThreads * i;
        if (u < ROWS * K / 8) st[i] = *(const v4u *)((const char *)W + u * 16u);
    }
}
template <int ROWS, int K, int PAD = K>
__device__ __forceinline__ void put_w(__bf16 *lds, const v4u (&st)[5], unsigned thread) {
    const unsigned tid = fresh(thread, kTileThreads);
#pragma unroll
    for (int i = 0; i < (ROWS * K / 8 + kTileThreads - 1) / kTileThreads; i++) {
        const unsigned u = tid + kTileThreads * i;
        if (u < ROWS * K / 8) *(v4u *)(lds + u / (K / 8) * (PAD + 8) + u % (K / 8) * 8) = st[i];
    }
    if (PAD > K)
        for (unsigned u = tid; u < ROWS * (PAD - K) / 8; u += kTileThreads)
            *(v4u *)(lds + u / ((PAD - K) / 8) * (PAD + 8) + K + u % ((PAD - K) / 8) * 8) = v4u{0, 0, 0, 0};
}

// acc[j] = rows n0 + 16 j .. of W (LDS, K wide) times the points of `act`: lane
// (g, c) gets rows n0 + 16 j + 4 g .. + 3 of point c
template <int NB, int K>
__device__ __forceinline__ void stage_mfma(const __bf16 *w, int n0, const __bf16 *act, int g, int lc,
                                           v4f (&acc)[4]) {
    const unsigned c = fresh(lc, 16);
#pragma unroll
    for (int j = 0; j < NB; j++) acc[j] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k0 = 0; k0 < K; k0 += 32) {
        const v8bf b = *(const v8bf *)(act + k0 + 8 * g);
#pragma unroll
        for (int j = 0; j < NB; j++) {
            const v8bf a = *(const v8bf *)(w + (n0 + 16 * j + c) * (K + 8) + k0 + 8 * g);
            acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc[j], 0, 0, 0);
        }
    }
}

// rows of an LDS activation buffer (width K) to global rows of K
template <int K>
__device__ __forceinline__ void store_rows(const __bf16 *act, __bf16 *dst, unsigned thread) {
    const unsigned tid = fresh(thread, kTileThreads);
#pragma unroll
    for (int i = 0; i < (kTP * K / 8 + kTileThreads - 1) / kTileThreads; i++) {
        const unsigned u = tid + kTileThreads * i;
        if (u < kTP * K / 8)
            *(v4u *)((char *)dst + u * 16u) =
                *(const v4u *)(act + u / (K / 8) * kAS + u % (K / 8) * 8);
    }
}

// of values v[0..15] per lane, each summed over the 16 points (lanes c) of its
// lane group, lane c keeps sum c
__device__ __forceinline__ float point_sums(const v4f (&v)[4], int c) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const float t = row16_sum(v[i >> 2][i & 3]);
        s = c == i ? t : s;
    }
    return s;
}

}  // namespace

// One workgroup: tiles blockIdx.x, + gridDim.x, ... of 64 points, forward and
// (TRAIN) backward.  Wavefront w owns points 16 (w & 3) .. + 15 and half w >> 2
// of every layer's rows.  Bound by latency at the usual batch (one tile per
// CU): nine stages of a weight copy (L2), a few MFMAs and a barrier each.
template <bool TRAIN>
__global__ __launch_bounds__(kTileThreads, 1) void mlp_tile_kernel(MlpTileArgs a) {
    __shared__ __align__(16) __bf16 act[2][kTP * kAS];
    __shared__ __align__(16) __bf16 wbuf[2][kH * (kK0 + 8)];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, c = lane & 15;
    const int pl = 16 * (wave & 3) + c, n0 = 64 * (wave >> 2);
    const int ao = pl * kAS;  // this lane's point in the activations
    const int ntiles = (int)((a.npts + kTP - 1) / kTP);
    v4u st[5];
    int wb = 0;  // weight buffer of the current stage
    float db[kD] = {0.f, 0.f, 0.f, 0.f}, dbo = 0.f, loss = 0.f;
    fetch_w<kH, kK0>(a.W + woff(0), st, tid);
    put_w<kH, kK0>(wbuf[0], st, tid);
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const long long p0 = (long long)tile * kTP, p = p0 + pl;
        const bool valid = p < a.npts;  // padding points carry zeros
        // Fourier features: thread (point, part) takes eight frequencies
        {
            const int q = tid >> 3, part = tid & 7;
            const long long pf = p0 + q;
            const float inv = 1.f / a.cs[3];
            float u[3] = {0.f, 0.f, 0.f};
            if (pf < a.npts) {
                u[0] = (float)(a.r[3 * pf] - a.cs[0]) * inv;
                u[1] = (float)(a.r[3 * pf + 1] - a.cs[1]) * inv;
                u[2] = (float)(a.r[3 * pf + 2] - a.cs[2]) * inv;
            }
            __bf16 *x = act[0] + q * kAS;
#pragma unroll 1
            for (int f = 8 * part; f < 8 * part + 8; f++) {
                const float t = 6.283185307179586f *
                                (a.freq[3 * f] * u[0] + a.freq[3 * f + 1] * u[1] + a.freq[3 * f + 2] * u[2]);
                float s, co;
                sincosf(t, &s, &co);
                x[f] = (__bf16)s;
                x[kF + f] = (__bf16)co;
            }
            if (part < (kK0 - 2 * kF) / 8) {
                v8bf z = {};
                if (part == 0) {
                    z[0] = (__bf16)u[0];
                    z[1] = (__bf16)u[1];
                    z[2] = (__bf16)u[2];
                }
                *(v8bf *)(x + 2 * kF + 8 * part) = z;
            }
        }
        __syncthreads();
        v4f z[kD][4], acc[4];
        // hidden layer l: act[from] -> act[from ^ 1], pre-activations kept
        auto hidden = [&](auto lc) {
            constexpr int l = decltype(lc)::value, K = kin(l), from = l & 1;
            if (TRAIN) store_rows<K>(act[from], a.X[l] + p0 * K, tid);
            if constexpr (l + 1 < kD) fetch_w<kH, kH>(a.W + woff(l + 1), st, tid);
            else fetch_w<kNO, kH>(a.W + woff(kD), st, tid);
            stage_mfma<4, K>(wbuf[wb], n0, act[from] + ao, g, c, acc);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const v4f b = *(const v4f *)((const char *)(a.prm + boff(l) + n0 + 16 * j) + (unsigned)g * 16u);
                v4bf h;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    z[l][j][i] = acc[j][i] + b[i];
                    h[i] = valid ? (__bf16)silu(z[l][j][i]) : (__bf16)0.f;
                }
                *(v4bf *)(act[from ^ 1] + ao + n0 + 16 * j + 4 * g) = h;
            }
            if constexpr (l + 1 < kD) put_w<kH, kH>(wbuf[wb ^ 1], st, tid);
            else put_w<kNO, kH>(wbuf[wb ^ 1], st, tid);
            wb ^= 1;
            __syncthreads();
        };
        hidden(std::integral_constant<int, 0>{});
        hidden(std::integral_constant<int, 1>{});
        hidden(std::integral_constant<int, 2>{});
        hidden(std::integral_constant<int, 3>{});
        // output layer, rows 4 g + i: tensor elements 0 .. 8, log amplitude 9
        if (TRAIN) {
            store_rows<kH>(act[0], a.X[kD] + p0 * kH, tid);
            fetch_w<kH, kNO>(a.WT + toff(kD), st, tid);
        } else {
            fetch_w<kH, kK0>(a.W + woff(0), st, tid);
        }
        float y[4];
        {
            v4f o[4];
            stage_mfma<1, kH>(wbuf[wb], 0, act[0] + ao, g, c, o);
            const v4f b = *(const v4f *)((const char *)(a.prm + boff(kD)) + (unsigned)g * 16u);
#pragma unroll
            for (int i = 0; i < 4; i++) y[i] = o[0][i] + b[i];
        }
        if (!TRAIN) {
            const float e = amp(__shfl(y[1], 32 + c));
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int n = 4 * g + i;
                if (wave < 4 && n < 9 && valid) a.J[9 * p + n] = (double)(y[i] * e * a.oscale[n]);
            }
            put_w<kH, kK0>(wbuf[wb ^ 1], st, tid);
            wb ^= 1;
            __syncthreads();
            continue;
        }
        {
            // loss and dY; |t|^2 summed in element order over the lane groups
            float t[4] = {0.f, 0.f, 0.f, 0.f}, tn = a.eps2;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int n = 4 * g + i;
                if (n < 9 && valid) t[i] = (float)a.target[9 * p + n] / a.oscale[n];
            }
#pragma unroll
            for (int q = 0; q < 3; q++) {
                float s = tn;
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (4 * q + i < 9) s += t[i] * t[i];
                tn = __shfl(s, 16 * q + c);
            }
            const float inv = rsqrtf(tn), s = 2.f / (float)a.npts;
            v4f dy = {0.f, 0.f, 0.f, 0.f};
            float part = 0.f;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int n = 4 * g + i;
                float d = y[i] - t[i] * inv;
                if (n == 9) d = y[i] - 0.5f * __logf(tn);
                if (n > 9 || !valid) d = 0.f;
                part += d * d;
                dy[i] = s * d;
            }
            if (wave < 4) loss += part;
            v4f v[4] = {dy, v4f{0.f, 0.f, 0.f, 0.f}, v4f{0.f, 0.f, 0.f, 0.f}, v4f{0.f, 0.f, 0.f, 0.f}};
            const float sums = point_sums(v, c);
            if (wave < 4) dbo += sums;
            v4bf h;
#pragma unroll
            for (int i = 0; i < 4; i++) h[i] = wave < 4 ? (__bf16)dy[i] : (__bf16)0.f;
            // the product below is 32 wide: columns 16 .. 31 are zero
            *(v4bf *)(act[1] + ao + 16 * (wave >> 2) + 4 * g) = h;
        }
        put_w<kH, kNO, 32>(wbuf[wb ^ 1], st, tid);
        wb ^= 1;
        __syncthreads();
        // dZ of layer l from the stage's input in act[from]
        auto back = [&](auto lc) {
            constexpr int l = decltype(lc)::value, from = l & 1, K = l == kD - 1 ? 32 : kH;
            if constexpr (l == kD - 1) store_rows<kNO>(act[from], a.dY + p0 * kNO, tid);
            else store_rows<kH>(act[from], a.dZ[l + 1] + p0 * kH, tid);
            if constexpr (l > 0) fetch_w<kH, kH>(a.WT + toff(l), st, tid);
            else fetch_w<kH, kK0>(a.W + woff(0), st, tid);
            stage_mfma<4, K>(wbuf[wb], n0, act[from] + ao, g, c, acc);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                v4bf h;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float d = valid ? acc[j][i] * dsilu(z[l][j][i]) : 0.f;
                    acc[j][i] = d;
                    h[i] = (__bf16)d;
                }
                *(v4bf *)(act[from ^ 1] + ao + n0 + 16 * j + 4 * g) = h;
            }
            db[l] += point_sums(acc, c);
            if constexpr (l > 0) put_w<kH, kH>(wbuf[wb ^ 1], st, tid);
            else put_w<kH, kK0>(wbuf[wb ^ 1], st, tid);
            wb ^= 1;
            __syncthreads();
        };
        back(std::integral_constant<int, 3>{});
        back(std::integral_constant<int, 2>{});
        back(std::integral_constant<int, 1>{});
        back(std::integral_constant<int, 0>{});
        // (the next tile writes act[0] first, and act[1] after a barrier)
        store_rows<kH>(act[1], a.dZ[0] + p0 * kH, tid);
    }
    if (!TRAIN) return;
    // bias gradients: lane (g, c) holds row n0 + 16 (c >> 2) + 4 g + (c & 3) of
    // each layer, summed over the wavefronts of its half in a fixed order
    __syncthreads();
    float *red = (float *)act[0];  // [8 wavefronts][kD + 2][64]
#pragma unroll
    for (int l = 0; l < kD; l++) red[(wave * (kD + 2) + l) * 64 + lane] = db[l];
    red[(wave * (kD + 2) + kD) * 64 + lane] = dbo;
    red[(wave * (kD + 2) + kD + 1) * 64 + lane] = loss;
    __syncthreads();
    float *out = a.bpart + (size_t)blockIdx.x * (kBiasN + 1);
    for (int n = tid; n < kBiasN + 1; n += kTileThreads) {
        float s = 0.f;
        if (n < kBiasN) {
            const int l = n < kD * kH ? n / kH : kD, m = n < kD * kH ? n % kH : n - kD * kH;
            const int w = m / 64 * 4, i = m % 64;
            const int ln = 16 * (i >> 2 & 3) + 4 * (i >> 4) + (i & 3);
            for (int k = 0; k < 4; k++) s += red[((w + k) * (kD + 2) + l) * 64 + ln];
        } else {
            for (int k = 0; k < 4; k++)
                for (int ln = 0; ln < 64; ln++) s += red[(k * (kD + 2) + kD + 1) * 64 + ln];
            s /= (float)a.npts;
        }
        out[n] = s;
    }
}

// Weight gradients of one point range: dW_l[n][k] = sum_p dZ_l[p][n] X_l[p][k].
// grid (ranges, layers).  64 points at a time, both operands transposed on
// their way into LDS (pairs of points packed into 32-bit writes; the 16-byte
// column of points is swizzled so that writes and reads spread over the
// banks).  The range's sums go to part[range][flat parameter].
template <int K, int N>
__device__ __forceinline__ void dw_range(const __bf16 *dZ, const __bf16 *X, int t0, int t1, float *out,
                                         __bf16 *lds) {
    constexpr int NU = N / 8, KU = K / 8;               // 8-wide column groups
    constexpr int UN = (32 * NU + 255) / 256, UK = (32 * KU + 255) / 256;
    constexpr int IB = N == kNO ? 1 : 2;                // blocks of 16 rows n per wavefront
    constexpr int JB = N == kNO ? K / 64 : K / 16;      // blocks of 16 columns k
    __bf16 *zt = lds, *xt = lds + N * 64;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int g = lane >> 4, c = lane & 15;
    const int i0 = N == kNO ? 0 : 32 * wave, j0 = N == kNO ? wave * (K / 4) : 0;
    // 16-byte column ch of row n is at n * 64 + 8 * (ch ^ ((n ^ n >> 3) & 7))
    auto place = [](int n, int ch) { return n * 64 + 8 * (ch ^ ((n ^ n >> 3) & 7)); };
    v4f acc[IB][JB];
#pragma unroll
    for (int i = 0; i < IB; i++)
#pragma unroll
        for (int j = 0; j < JB; j++) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
    v4u zr[UN][2], xr[UK][2];
    auto fetch = [&](int t) {
        const v4u *z = (const v4u *)(dZ + (size_t)t * 64 * N), *x = (const v4u *)(X + (size_t)t * 64 * K);
#pragma unroll
        for (int i = 0; i < UN; i++) {
            const int u = tid + 256 * i, pp = u / NU, q = u % NU;
            if (u < 32 * NU) {
                zr[i][0] = z[2 * pp * NU + q];
                zr[i][1] = z[(2 * pp + 1) * NU + q];
            }
        }
#pragma unroll
        for (int i = 0; i < UK; i++) {
            const int u = tid + 256 * i, pp = u / KU, q = u % KU;
            if (u < 32 * KU) {
                xr[i][0] = x[2 * pp * KU + q];
                xr[i][1] = x[(2 * pp + 1) * KU + q];
            }
        }
    };
    // columns 8 q .. + 7 of points 2 pp, 2 pp + 1
    auto put = [&](__bf16 *d, const v4u (&v)[2], int pp, int q) {
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const uint32_t a = v[0][e >> 1], b = v[1][e >> 1];
            const uint32_t w = e & 1 ? (a >> 16) | (b & 0xffff0000u) : (a & 0xffffu) | b << 16;
            *(uint32_t *)(d + place(8 * q + e, pp >> 2) + 2 * (pp & 3)) = w;
        }
    };
    fetch(t0);
    for (int t = t0; t < t1; t++) {
        __syncthreads();  // the previous points have been read
#pragma unroll
        for (int i = 0; i < UN; i++) {
            const int u = tid + 256 * i;
            if (u < 32 * NU) put(zt, zr[i], u / NU, u % NU);
        }
#pragma unroll
        for (int i = 0; i < UK; i++) {
            const int u = tid + 256 * i;
            if (u < 32 * KU) put(xt, xr[i], u / KU, u % KU);
        }
        __syncthreads();
        if (t + 1 < t1) fetch(t + 1);
#pragma unroll
        for (int kk = 0; kk < 2; kk++) {
            v8bf za[IB];
#pragma unroll
            for (int i = 0; i < IB; i++)
                za[i] = *(const v8bf *)(zt + place(i0 + 16 * i + c, 4 * kk + g));
#pragma unroll
            for (int j = 0; j < JB; j++) {
                const v8bf xb = *(const v8bf *)(xt + place(j0 + 16 * j + c, 4 * kk + g));
#pragma unroll
                for (int i = 0; i < IB; i++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(za[i], xb, acc[i][j], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < IB; i++)
#pragma unroll
        for (int j = 0; j < JB; j++)
#pragma unroll
            for (int q = 0; q < 4; q++)
                out[(i0 + 16 * i + 4 * g + q) * K + j0 + 16 * j + c] = acc[i][j][q];
}

__global__ __launch_bounds__(256) void mlp_dw_kernel(MlpTileArgs a, int ntiles, float *part) {
    __shared__ __align__(16) __bf16 lds[(kH + kK0) * 64];
    const int l = blockIdx.y, ranges = gridDim.x;
    const int t0 = (int)((long long)blockIdx.x * ntiles / ranges),
              t1 = (int)((long long)(blockIdx.x + 1) * ntiles / ranges);
    float *out = part + (size_t)blockIdx.x * kMlpParams;
    if (l == 0) dw_range<kK0, kH>(a.dZ[0], a.X[0], t0, t1, out + woff(0), lds);
    else if (l < kD) dw_range<kH, kH>(a.dZ[l], a.X[l], t0, t1, out + woff(l), lds);
    else dw_range<kH, kNO>(a.dY, a.X[kD], t0, t1, out + woff(kD), lds);
}

// layer and place of flat parameter i: b < 0 a weight (row n, column k), else
// index b of the bias sums
struct ParamAt {
    int l, n, k, b;
};
__device__ __forceinline__ ParamAt param_at(int i) {
    constexpr int first = (kK0 + 1) * kH, mid = (kH + 1) * kH;
    const int l = i < first ? 0 : min(kD, 1 + (i - first) / mid);
    const int o = l == 0 ? i : i - first - (l - 1) * mid, K = l == 0 ? kK0 : kH;
    const int nw = K * (l == kD ? kNO : kH);
    return o < nw ? ParamAt{l, o / K, o % K, -1} : ParamAt{l, o - nw, 0, l * kH + o - nw};
}

// BF16 copy of a parameter, and of a weight of layers 1 .. D its transposed one
__device__ __forceinline__ void store_bf16(int i, const ParamAt &q, float x, __bf16 *W, __bf16 *WT) {
    W[i] = (__bf16)x;
    if (q.b < 0 && q.l > 0) WT[toff(q.l) + q.k * (q.l == kD ? kNO : kH) + q.n] = (__bf16)x;
}

// The gradient of every parameter from the partial sums (weights: one per
// point range; biases and the loss: one per tile workgroup, 16 lanes each), in
// a fixed order; with `adam` the Adam step on the FP32 master parameters and
// their BF16 copies, else the gradient itself.  Parameters in workgroups of
// 64; the last workgroups take 16 biases each and the loss.
__global__ __launch_bounds__(256) void mlp_adam_kernel(MlpAdamArgs a) {
    constexpr int kWeightGroups = (kMlpParams + 63) / 64;
    __shared__ float red[4][64];
    float gr = 0.f;
    int i = -1;
    if (blockIdx.x < kWeightGroups) {
        // 64 parameters, every fourth range per wavefront
        const int q = threadIdx.x >> 6, ln = threadIdx.x & 63, j = blockIdx.x * 64 + ln;
        const float *src = a.part + min(j, kMlpParams - 1);
#pragma unroll 4
        for (int s = q; s < a.ranges; s += 4) gr += src[(size_t)s * kMlpParams];
        red[q][ln] = gr;
        __syncthreads();
        if (q > 0 || j >= kMlpParams || param_at(j).b >= 0) return;
        i = j;
        gr = ((red[0][ln] + red[1][ln]) + red[2][ln]) + red[3][ln];
    } else {
        const int b = (blockIdx.x - kWeightGroups) * 16 + (threadIdx.x >> 4), q = threadIdx.x & 15;
        if (b > kBiasN) return;
        for (int s = q; s < a.groups; s += 16) gr += a.bpart[(size_t)s * (kBiasN + 1) + b];
        gr = row16_sum(gr);
        if (q != 0) return;
        if (b == kBiasN) {
            a.loss[0] = gr;
            return;
        }
        const int l = b < kD * kH ? b / kH : kD;
        i = (l == 0 ? kK0 * kH : (kK0 + 1) * kH + (l - 1) * (kH + 1) * kH + kH * (l == kD ? kNO : kH)) +
            b - l * kH;
    }
    if (!a.adam) {
        a.grad[i] = gr;
        return;
    }
    const float mi = a.b1 * a.m[i] + (1.f - a.b1) * gr;
    const float vi = a.b2 * a.v[i] + (1.f - a.b2) * gr * gr;
    a.m[i] = mi;
    a.v[i] = vi;
    const float pi = a.prm[i] - a.lr * (mi / a.bc1) / (sqrtf(vi / a.bc2) + a.eps);
    a.prm[i] = pi;
    store_bf16(i, param_at(i), pi, a.W, a.WT);
}

__global__ __launch_bounds__(256) void mlp_cast_kernel(const float *p, __bf16 *W, __bf16 *WT) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < kMlpParams) store_bf16(i, param_at(i), p[i], W, WT);
}

// ---- fused inference ----

namespace {

// weights, biases and frequencies in LDS, weight rows of K + 8
constexpr int kInferW(int l) { return l == 0 ? 0 : kInferW(l - 1) + nout(l - 1) * (kin(l - 1) + 8); }
constexpr int kInferElems = kInferW(kD) + kNO * (kH + 8);
constexpr int kInferThreads = 1024;
constexpr size_t kInferLds = (size_t)kInferElems * 2 + (kBiasN + 4 * kF) * 4;
typedef unsigned short v2us __attribute__((ext_vector_type(2)));

// (bf16)(z / (1 + e^-z)) of four values, bit for bit that of the exact
// division: z times the hardware reciprocal (1 ulp) is within 3 ulp of the
// correctly rounded quotient, so the BF16 values agree unless one of the four
// lies that close to the middle between two BF16 values (or the divisor's
// reciprocal is denormal, z < -80), where the wavefront divides: 3% of the
// time.
__device__ __forceinline__ v4bf silu_bf16(v4f z) {
    float h[4];
    v2us near = {0xffff, 0xffff};
#pragma unroll
    for (int i = 0; i < 4; i++) h[i] = z[i] * __builtin_amdgcn_rcpf(1.f + __expf(-z[i]));
#pragma unroll
    for (int i = 0; i < 4; i += 2) {
        // the halves that rounding drops, 0x7ffd .. 0x8003 -> 0 .. 6
        const uint32_t lo = __builtin_amdgcn_perm(__float_as_uint(h[i + 1]), __float_as_uint(h[i]), 0x05040100u);
        v2us d;
        __builtin_memcpy(&d, &lo, 4);
        d = d - (v2us){0x7ffd, 0x7ffd};
        near = __builtin_elementwise_min(near, d);
    }
    const float low = fminf(fminf(z[0], z[1]), fminf(z[2], z[3]));
    const bool redo = near[0] <= 6 || near[1] <= 6 || !(low >= -80.f);
    if (__builtin_expect(__any(redo), 0)) {
#pragma unroll
        for (int i = 0; i < 4; i++) h[i] = silu(z[i]);
    }
    v4bf r;
#pragma unroll
    for (int i = 0; i < 4; i++) r[i] = (__bf16)h[i];
    return r;
}

}  // namespace

// 16 points per wavefront, all in registers; 16 wavefronts share the weights
// in LDS (152 KB) and step through the points without a barrier.  With the
// weights as the first MFMA operand the lane (g, c) holds rows 4 g .. + 3 of
// every 16-row block of point c; the next layer wants 8 g .. + 7 of every 32,
// two lane-group swaps away.  Bound by VALU: 512 SiLU and 64 sine-cosine pairs
// a point.
__global__ __launch_bounds__(kInferThreads, 1) void mlp_infer_kernel(
    const double *r, long long npts, const float *freq, const float *cs, const __bf16 *W,
    const float *prm, const float *oscale, double *J) {
    extern __shared__ __align__(16) unsigned char infer_lds[];
    __bf16 *w = (__bf16 *)infer_lds;
    float *bias = (float *)(w + kInferElems);  // the layers' biases one after another
    float *fr = bias + kBiasN;                 // [f][4]
    const int tid = threadIdx.x, lane = tid & 63;
    const int g = lane >> 4, c = lane & 15;
    auto stage = [&](auto lc) {
        constexpr int l = decltype(lc)::value, K = kin(l), N = nout(l);
        for (int u = tid; u < N * K / 8; u += kInferThreads)
            *(v4u *)(w + kInferW(l) + u / (K / 8) * (K + 8) + u % (K / 8) * 8) =
                *(const v4u *)(W + woff(l) + u * 8);
        for (int n = tid; n < N; n += kInferThreads) bias[l * kH + n] = prm[boff(l) + n];
    };
    stage(std::integral_constant<int, 0>{});
    stage(std::integral_constant<int, 1>{});
    stage(std::integral_constant<int, 2>{});
    stage(std::integral_constant<int, 3>{});
    stage(std::integral_constant<int, 4>{});
    for (int i = tid; i < 4 * kF; i += kInferThreads) fr[i] = (i & 3) < 3 ? freq[3 * (i >> 2) + (i & 3)] : 0.f;
    __syncthreads();
    const float inv = 1.f / cs[3];
    const long long step = (long long)gridDim.x * (kInferThreads / 64) * 16;
    for (long long p0 = ((long long)blockIdx.x * (kInferThreads / 64) + (tid >> 6)) * 16; p0 < npts;
         p0 += step) {
        const long long p = p0 + c;
        const bool valid = p < npts;
        float u[3] = {0.f, 0.f, 0.f};
        if (valid) {
            u[0] = (float)(r[3 * p] - cs[0]) * inv;
            u[1] = (float)(r[3 * p + 1] - cs[1]) * inv;
            u[2] = (float)(r[3 * p + 2] - cs[2]) * inv;
        }
        // features 32 q + 8 g .. + 7 in x[q]: sines, cosines, the coordinates
        v8bf x[kK0 / 32];
        const float *fq = fr + fresh(32 * g, 4 * kF);
#pragma unroll
        for (int q = 0; q < 2; q++)
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const v4f b = *(const v4f *)(fq + 4 * (32 * q + i));
                const float t = 6.283185307179586f * (b[0] * u[0] + b[1] * u[1] + b[2] * u[2]);
                float s, co;
                sincosf(t, &s, &co);
                x[q][i] = (__bf16)s;
                x[2 + q][i] = (__bf16)co;
            }
        x[4] = v8bf{};
        if (g == 0) {
            x[4][0] = (__bf16)u[0];
            x[4][1] = (__bf16)u[1];
            x[4][2] = (__bf16)u[2];
        }
        auto layer = [&](auto lc) {
            constexpr int l = decltype(lc)::value, K = kin(l);
            // (else the loads of all weights move out of the loop over points)
            const __bf16 *wl = w + fresh(kInferW(l) + c * (K + 8) + 8 * g, kInferElems);
            const float *bl = bias + fresh(l * kH + 4 * g, kBiasN);
            v8bf nx[kH / 32];
#pragma unroll
            for (int q = 0; q < kH / 32; q++) {
                union {
                    v4bf h;
                    uint32_t d[2];
                } b[2];
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int k = 0; k < K / 32; k++)
                        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            *(const v8bf *)(wl + (32 * q + 16 * j) * (K + 8) + 32 * k), x[k], acc, 0, 0, 0);
                    const v4f bb = *(const v4f *)(bl + 32 * q + 16 * j);
                    v4f z;
#pragma unroll
                    for (int i = 0; i < 4; i++) z[i] = acc[i] + bb[i];
                    b[j].h = silu_bf16(z);
                }
                // rows 4 g' of two blocks to rows 8 g of the 32: groups (0, 1,
                // 2, 3) of block A and B become (A0 A1), (A2 A3), (B0 B1), (B2 B3)
                union {
                    v8bf v;
                    uint32_t d[4];
                } o;
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    const auto s = __builtin_amdgcn_permlane32_swap(b[0].d[e], b[1].d[e], false, false);
                    const auto t = __builtin_amdgcn_permlane16_swap(s[0], s[1], false, false);
                    o.d[e] = t[0];
                    o.d[2 + e] = t[1];
                }
                nx[q] = o.v;
            }
#pragma unroll
            for (int q = 0; q < kH / 32; q++) x[q] = nx[q];
        };
        layer(std::integral_constant<int, 0>{});
        layer(std::integral_constant<int, 1>{});
        layer(std::integral_constant<int, 2>{});
        layer(std::integral_constant<int, 3>{});
        v4f acc = {0.f, 0.f, 0.f, 0.f};
        const __bf16 *wo = w + fresh(kInferW(kD) + c * (kH + 8) + 8 * g, kInferElems);
#pragma unroll
        for (int k = 0; k < kH / 32; k++)
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const v8bf *)(wo + 32 * k), x[k], acc, 0, 0, 0);
        const v4f bb = *(const v4f *)(bias + fresh(kD * kH + 4 * g, kBiasN));
        float y[4];
#pragma unroll
        for (int i = 0; i < 4; i++) y[i] = acc[i] + bb[i];
        // row 9, the log amplitude, is element 1 of lane group 2
        const float e = amp(__shfl(y[1], 32 + c));
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int n = 4 * g + i;
            if (n < 9 && valid) J[9 * p + n] = (double)(y[i] * e * oscale[n]);
        }
    }
}

// ---------------------------------------------------------------- launchers

static inline unsigned blocks(long long n, int t) { return (unsigned)((n + t - 1) / t); }

// tiles of 64 points over at most one workgroup per CU; returns the workgroups
int mlp_tile_groups(long long npts) {
    return (int)std::min<long long>((npts + kTP - 1) / kTP, 256);
}

// point ranges of the weight gradients: enough workgroups (five per range) to
// fill the chip at four tiles a range
int mlp_ranges(long long npts) {
    return (int)std::max<long long>(1, std::min<long long>(kMlpMaxRanges, (npts + kTP - 1) / kTP / 4));
}

static bool tiles_ok(const MlpTileArgs &a) { return a.npts > 0 && a.npts <= (1ll << 36); }

hipError_t mlp_tiles(const MlpTileArgs &a, bool train, hipStream_t s) {
    if (!tiles_ok(a)) return hipErrorInvalidValue;
    const dim3 grid(mlp_tile_groups(a.npts));
    if (train) hipLaunchKernelGGL(mlp_tile_kernel<true>, grid, dim3(kTileThreads), 0, s, a);
    else hipLaunchKernelGGL(mlp_tile_kernel<false>, grid, dim3(kTileThreads), 0, s, a);
    return hipGetLastError();
}

hipError_t mlp_dw(const MlpTileArgs &a, float *part, hipStream_t s) {
    if (!tiles_ok(a)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(mlp_dw_kernel, dim3(mlp_ranges(a.npts), kD + 1), dim3(256), 0, s, a,
                       (int)((a.npts + kTP - 1) / kTP), part);
    return hipGetLastError();
}

hipError_t mlp_adam(const MlpAdamArgs &a, hipStream_t s) {
    hipLaunchKernelGGL(mlp_adam_kernel, dim3(blocks(kMlpParams, 64) + blocks(kBiasN + 1, 16)),
                       dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t mlp_cast(const float *p, __bf16 *W, __bf16 *WT, hipStream_t s) {
    hipLaunchKernelGGL(mlp_cast_kernel, dim3(blocks(kMlpParams, 256)), dim3(256), 0, s, p, W, WT);
    return hipGetLastError();
}

hipError_t mlp_infer(const double *r, long long npts, const float *freq, const float *cs,
                     const __bf16 *W, const float *prm, const float *oscale, double *J, hipStream_t s) {
    if (npts <= 0) return hipSuccess;
    hipError_t e = hipFuncSetAttribute((const void *)mlp_infer_kernel,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)kInferLds);
    if (e != hipSuccess) return e;
    // one workgroup per CU at most, 256 points at a time
    const unsigned groups = (unsigned)std::min<long long>((npts + 255) / 256, 256);
    hipLaunchKernelGGL(mlp_infer_kernel, dim3(groups), dim3(kInferThreads), kInferLds, s, r, npts, freq,
                       cs, W, prm, oscale, J);
    return hipGetLastError();
}

}  // namespace gimic
