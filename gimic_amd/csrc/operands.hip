// Right operands of the contraction, built on the device from the density
// family (gfx950).
//
// The densities are uploaded once as the caller gave them; a spin case's
// operand is then one pass over its matrices: gather in the internal function
// order (fun), combine the spin sets, form W_d(mu,nu) = D(mu,nu)
// (R_nu - R_mu)_d, and write the layout a kernel reads.  One thread per
// element (mu, nu) computes all seven matrices, so D and the centres are
// loaded once; the stores of a wavefront are whole 128-byte pieces.  Bound by memory: 32 bytes read and 56 (FP64) or 42
// (split) bytes written per element.  Building them on the host and copying them
// took most of a first evaluation: a whole run on the 60-atom cage (nbf 1800:
// context, densities, one 140 x 140 plane in FP64) went from 214 to 101 ms, the
// first mixed evaluation of a 200-atom open shell (nbf 2620, two spin cases)
// from 1352 to 288 ms, its tuning runs included.
#include "device_common.h"

namespace gimic {

namespace {

// the seven matrix values at internal indices (mu, nu), zero in the padding
__device__ __forceinline__ void operand_values(const OperandArgs &a, int mu, int nu,
                                               double (&v)[kNMat]) {
#pragma unroll
    for (int m = 0; m < kNMat; m++) v[m] = 0.0;
    if (mu >= a.n || nu >= a.n) return;
    const size_t n = (size_t)a.n, om = (size_t)a.fun[mu], on = (size_t)a.fun[nu];
    const size_t i = a.row_major ? om * n + on : om + n * on;
#pragma unroll
    for (int m = 0; m < 4; m++) {
        const double x = a.dens[(size_t)m * n * n + i];
        v[m] = x;
        if (a.second) {
            const double y = a.second[(size_t)m * n * n + i];
            v[m] = a.subtract ? x - y : x + y;
        }
    }
#pragma unroll
    for (int d = 0; d < 3; d++)
        v[4 + d] = v[0] * (a.rf64[(size_t)d * a.ld + nu] - a.rf64[(size_t)d * a.ld + mu]);
}

// FP64: 16 threads per pair block, 16 pair blocks of one K-granule row per
// workgroup; a matrix's 16 elements are 128 contiguous bytes
__global__ __launch_bounds__(256) void operand_f64_kernel(OperandArgs a, double *out) {
    const int t = threadIdx.x & 15, ng = a.ld / 4;
    const int gn = blockIdx.x * 16 + (threadIdx.x >> 4), gk = blockIdx.y;
    if (gn > ng) return;
    // consecutive threads take the elements in their order in the block
    const int k = 2 * (t >> 3) + (t & 1), n = (t >> 1) & 3;
    double v[kNMat];
    // (the zero blocks' indices are at least ld >= n: operand_values gives 0)
    operand_values(a, gk * 4 + k, gn * 4 + n, v);
    double *dst = out + ((size_t)gk * (ng + 1) + gn) * kF64PairElems + t;
#pragma unroll
    for (int m = 0; m < kNMat; m++) dst[m * 16] = v[m];
}

// split: the FP32 value of each element as kBParts BF16 parts (three parts:
// x = h + m + l exactly), one pair block per wavefront (device_common.h); the
// last K-row and N-column of pair blocks are the zero ones
__global__ __launch_bounds__(256) void operand_split_kernel(OperandArgs a, uint16_t *out) {
    const int lane = threadIdx.x & 63, ng = a.ld / 8;
    const int gn = blockIdx.x * 4 + (threadIdx.x >> 6), gk = blockIdx.y;
    if (gn > ng) return;
    const int nn = lane >> 3, kk = lane & 7;
    double v[kNMat];
    operand_values(a, gk * 8 + kk, gn * 8 + nn, v);
    uint16_t *dst = out + ((size_t)gk * (ng + 1) + gn) * kMx2PairElems + lane;
#pragma unroll
    for (int m = 0; m < kNMat; m++) {
        float x = (float)v[m];
#pragma unroll
        for (int p = 0; p < kBParts; p++) {
            const uint16_t h = f32_to_bf16_rn(x);
            dst[(p * kNMat + m) * 64] = h;
            x -= bf16_to_f32(h);
        }
    }
}

}  // namespace

hipError_t launch_operand_f64(const OperandArgs &a, double *out, hipStream_t s) {
    if (a.n < 0 || a.ld < a.n || a.ld % 32 || a.ld / 4 + 1 > 65535) return hipErrorInvalidValue;
    const int ng = a.ld / 4;
    hipLaunchKernelGGL(operand_f64_kernel, dim3(ng / 16 + 1, ng + 1), dim3(256), 0, s, a, out);
    return hipGetLastError();
}

hipError_t launch_operand_split(const OperandArgs &a, __bf16 *out, hipStream_t s) {
    if (a.n < 0 || a.ld < a.n || a.ld % 32 || a.ld / 8 + 1 > 65535) return hipErrorInvalidValue;
    const int ng = a.ld / 8;
    hipLaunchKernelGGL(operand_split_kernel, dim3(ng / 4 + 1, ng + 1), dim3(256), 0, s, a,
                       (uint16_t *)out);
    return hipGetLastError();
}

}  // namespace gimic
