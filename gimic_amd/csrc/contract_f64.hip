// FP64 contraction of basis values with the density family on MFMA, with the
// per-point reductions fused into the epilogue (gfx950).
//
// The reference's contract (jtensor.F90:148-237) does, per point, seven
// length-n GEMVs phi*D, phi*DB_b, db_b*D and 27 dot products.  db_b = S_b phi
// with S = r x R_A (bfeval.f90:168-293), so every GEMV shares the left
// operand phi and a tile of P points is one GEMM
//     Y[P x 7n] = Phi[P x n] * [D | DBx | DBy | DBz | Wx | Wy | Wz]
// followed by reductions over the output column nu against phi_nu,
// grad phi_nu and R_nu (the kNQ partial sums listed in device_common.h).
// The finalize kernel turns the partials into the 3x3 tensor.
//
// With W_d(mu,nu) = D(mu,nu)(R_nu - R_mu)_d in place of R_d D, the GIAO
// reduction needs no difference of large terms, and the diamagnetic term
// is accumulated as sum Y0 phi (r - R_nu) (gauge origin at each function's
// centre), again free of cancellation.
//
// Tiling: one wavefront owns 16 points, a workgroup four of them.  Only what
// screening leaves non-zero over the row tile (tiles.hip; 64 or 128 points, one
// or two workgroups) is visited, in granules of four functions, the K of one
// v_mfma_f64_16x16x4: an N-tile is four of the tile's live granules (16
// functions x 7 matrices), a K-step another four (lane group g owns the g-th).
// The N-tiles of a row tile are split evenly over ranges and, where a launch
// has too few of these for the chip, the K-steps over ksplit ranges too (the
// sums are linear in Y): nsplit pairs of ranges in all.
//
// The matrices are the first MFMA operand and the points the second, so the
// lane (g, c) of an output block holds Y of the four functions of granule g
// at point c.  Each of the 22 sums then lives in one register pair per lane
// over all N-tiles of the workgroup, and lanes are added once at its end (the
// other way round each N-tile ends in a 16-lane reduction of 22 sums for
// every row: 5,000 VALU cycles per N-tile and wavefront instead of 450).
//
// The right operand comes in pair blocks of 4 x 4 elements x 7 matrices
// (operands.hip), 16 of which make a K-step: the workgroup copies them
// through registers into one of three LDS buffers ahead of their use, so a
// block is read once for 64 points.  Two workgroups share a CU (256 registers,
// 43 KB of LDS each) and fill each other's barriers, starts and epilogues: one
// workgroup of 128 points per CU with the same pipeline took 82.0 ms where
// this takes 77.5, two buffers and a barrier that drains the matrix pipe 86.9.
//
// Bound: the matrix pipe.  On the 60-atom cage (857,375 points, 4.1 TFLOP of
// listed work) 68.2 ms, 60 TF/s, 84% of a large FP64 matrix product on the
// same card (71.6 TF/s); the kernel it replaced (points first, 8-function
// groups, operands from global memory into registers) took 136 ms.  With every
// operand load redirected to one cached block it ran within 1% of that.  A
// wavefront takes its columns of compressed rows from the step's number: with
// the place read from the list entry it took 69.2 ms, and 256 planes of the
// 30-atom sheet 2.51 ms against 2.46.
//
// Workgroup order: the ranges of a row tile run back to back on one XCD
// (workgroup i goes to XCD i mod 8), so its basis rows come from that L2; with
// few tiles they go to all XCDs in turn (a.spread).
#include "device_common.h"

namespace gimic {

namespace {

typedef double v2d __attribute__((ext_vector_type(2)));

constexpr int kUnits = kF64PairElems / 2;  // 16-byte units of a pair block
constexpr int kStepUnits = 16 * kUnits;    // of a K-step: 16 pair blocks
// s_waitcnt immediate: lgkmcnt 0, the other counters at their maximum
constexpr int kWaitLds = 0xC07F;

}  // namespace

// one workgroup: 64 points of a row tile of a.tile_rows (64 or 128), a range
// of its N-tiles; 4 wavefronts, two workgroups per CU
template <bool CMP>
__global__ __launch_bounds__(256, 2) void contract_f64_kernel(ContractArgs a) {
    constexpr int kRows = 64;
    // [step mod 3][matrix][k pair][lane][2 k], lanes swizzled (below)
    __shared__ v2d buf[3 * kStepUnits];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, c = lane & 15;
    const int parts = a.tile_rows / kRows;  // workgroups that share a list and a range
    const int part = (a.spread ? blockIdx.x : blockIdx.x >> 3) % parts;
    const int slot = (a.spread ? blockIdx.x : blockIdx.x >> 3) / parts;
    const int ntile = a.rows / a.tile_rows, tiles = a.spread ? ntile : (ntile + 7) / 8;
    const int set = slot / (tiles * a.nsplit), split = slot % a.nsplit;
    const int rt = slot % (tiles * a.nsplit) / a.nsplit;
    const int rank = a.spread ? rt : rt * 8 + (blockIdx.x & 7);
    if (rank >= ntile) return;
    const int2 tile = a.order ? a.order[rank] : make_int2(rank, a.kcount[rank]);
    const int rtile = tile.x, count = tile.y;
    const int *K4 = a.klist + (size_t)rtile * a.nblk * 8;
    const int nks = (count + 3) >> 2;
    // this workgroup's N-tiles e0 .. e1 and, of each, kn K-steps from k0 on
    const int nsn = a.nsplit / a.ksplit, sn = split / a.ksplit, sk = split % a.ksplit;
    const int e0 = (int)((long long)sn * nks / nsn), e1 = (int)((long long)(sn + 1) * nks / nsn);
    const int k0 = (int)((long long)sk * nks / a.ksplit);
    const int kn = (int)((long long)(sk + 1) * nks / a.ksplit) - k0;
    const int *KK = K4 + 4 * k0;

    const int ng = a.lda / 4;  // granules per row; index ng: the zero blocks
    const v2d *B = (const v2d *)(a.b64 + (size_t)set * f64_set_elems(a.lda));
    const size_t rowst = (size_t)(ng + 1) * kUnits;
    const int rin = part * kRows + wave * 16 + c;
    const size_t row = (size_t)rtile * a.tile_rows + rin;
    // the point's values and gradients: dense, or compressed to the tile's granules
    const size_t w = CMP ? (size_t)count * 4 : (size_t)a.lda;
    const size_t base = (size_t)rtile * a.tile_rows * a.lda;
    const double *A = a.a64 + base + rin * w;
    const double *G = a.g64 + (CMP ? 3 * base : base) + rin * w;
    const size_t gplane = CMP ? (size_t)a.tile_rows * w : (size_t)a.gplane;
    const bool valid = row < (size_t)a.npts;
    const double r[3] = {valid ? a.pts[3 * row] : 0.0, valid ? a.pts[3 * row + 1] : 0.0,
                         valid ? a.pts[3 * row + 2] : 0.0};
    // column of the lane's granule of four-granule step s: compressed rows hold
    // the granules in list order, so no list entry is waited for (a padding
    // entry reads some granule of the row against zero blocks)
    auto acol = [&](int s) -> unsigned {
        if (CMP) return 4u * min(4 * s + g, count - 1);
        const int v = K4[4 * s + g];
        return v < 0 ? 0u : (v >> 13) * 4u;
    };

    // Element pair sp of matrix m for lane l is at (2 m + sp) * 64 +
    // (l ^ (l >> 3 & 1) ^ 2 sp): eight consecutive lanes of a read (c fixed in
    // bit 3) and of a write (functions n = c >> 2 and sp of one pair block)
    // then fall into different 16-byte columns.
    // Wavefront w copies the pair blocks of K-granule w, one N-granule i a
    // pass: lane < kUnits takes unit (m, sp, function n), for lane
    // (w, i + 4 n), whose place is put0 ^ i.
    const int unit = min(lane, kUnits - 1), un = unit & 3;
    const int put0 = (unit >> 2) * 64 + ((wave * 16 + 4 * un) ^ un >> 1 ^ (unit >> 1 & 2));
    const int rd0 = lane ^ (lane >> 3 & 1), rd1 = 64 + (rd0 ^ 2);

    double q[kNQ];
#pragma unroll
    for (int i = 0; i < kNQ; i++) q[i] = 0.0;

    if (e0 < e1 && kn > 0) {
        // The K-steps of all N-tiles form one sequence t.  During step t the
        // workgroup computes on buffer t mod 3, stores step t + 2 (loaded
        // during step t - 1) and loads step t + 3; one barrier ends a step.
        // Step t + 1 was complete before step t began, so its first operands
        // are read before the barrier and the matrix pipe does not drain.
        int fe = e0, fk = 0;  // N-tile and K-step of the next load
        // (list entries are read a K-step or an N-tile early and used raw, per
        // lane: a scalar or converted value would be waited for at once)
        unsigned noff[4];
        int4 nxt;
        auto offsets = [&] {
            const int x[4] = {nxt.x, nxt.y, nxt.z, nxt.w};
#pragma unroll
            for (int i = 0; i < 4; i++)
                noff[i] = ((unsigned)(x[i] < 0 ? ng : x[i] >> 13) * kUnits + unit) * 16u;
        };
        nxt = *(const int4 *)(K4 + 4 * fe);
        offsets();
        nxt = *(const int4 *)(K4 + 4 * min(fe + 1, e1 - 1));
        v2d st[4];
        const int wv = tid >> 6;
        int kent = KK[wv];
        auto source = [&] {
            const int x = __builtin_amdgcn_readfirstlane(kent);
            return (const char *)(B + (size_t)(x < 0 ? ng : x >> 13) * rowst);
        };
        auto load = [&](const char *src) {
#pragma unroll
            for (int i = 0; i < 4; i++) st[i] = *(const v2d *)(src + noff[i]);
            if (++fk == kn) {  // on to the next N-tile (past the last: it again)
                fk = 0;
                fe = min(fe + 1, e1 - 1);
                offsets();
                nxt = *(const int4 *)(K4 + 4 * min(fe + 1, e1 - 1));
            }
            kent = KK[4 * fk + wv];  // for the next step's load
        };
        auto put = [&](v2d *b) {
            if (lane < kUnits)
#pragma unroll
                for (int i = 0; i < 4; i++) b[put0 ^ i] = st[i];
        };
        int cur = 0, nx1 = kStepUnits, nx2 = 2 * kStepUnits;  // buffers of steps t, t + 1, t + 2
        load(source());
        put(buf + cur);
        load(source());
        put(buf + nx1);
        load(source());
        v4d an = *(const v4d *)(A + acol(k0));
        unsigned xa = acol(k0 + (kn > 1 ? 1 : 0));  // the next K-step's column
        __syncthreads();
        v2d b0[kNMat];
#pragma unroll
        for (int m = 0; m < kNMat; m++) b0[m] = buf[cur + rd0 + m * 128];

        for (int e = e0; e < e1; e++) {
            // the epilogue's operands: the four functions of this lane's granule
            const int xn = K4[4 * e + g];
            const unsigned xc = acol(e);
            const v4d ph = *(const v4d *)(A + xc);
            const v4d g0 = *(const v4d *)(G + xc), g1 = *(const v4d *)(G + gplane + xc),
                      g2 = *(const v4d *)(G + 2 * gplane + xc);
            v4d acc[kNMat];
#pragma unroll
            for (int m = 0; m < kNMat; m++) acc[m] = v4d{0.0, 0.0, 0.0, 0.0};
            for (int ks = 0; ks < kn; ks++) {
                const v4d av = an;
                v2d b1[kNMat];
#pragma unroll
                for (int m = 0; m < kNMat; m++) b1[m] = buf[cur + rd1 + m * 128];
                an = *(const v4d *)(A + xa);
                xa = acol(k0 + (ks + 2 < kn ? ks + 2 : ks + 2 - kn < kn ? ks + 2 - kn : 0));
#pragma unroll
                for (int m = 0; m < kNMat; m++)
                    acc[m] = __builtin_amdgcn_mfma_f64_16x16x4f64(b0[m].x, av[0], acc[m], 0, 0, 0);
                const char *src = source();
#pragma unroll
                for (int m = 0; m < kNMat; m++)
                    acc[m] = __builtin_amdgcn_mfma_f64_16x16x4f64(b0[m].y, av[1], acc[m], 0, 0, 0);
                put(buf + nx2);
                load(src);
#pragma unroll
                for (int m = 0; m < kNMat; m++) b0[m] = buf[nx1 + rd0 + m * 128];
#pragma unroll
                for (int m = 0; m < kNMat; m++)
                    acc[m] = __builtin_amdgcn_mfma_f64_16x16x4f64(b1[m].x, av[2], acc[m], 0, 0, 0);
#pragma unroll
                for (int m = 0; m < kNMat; m++)
                    acc[m] = __builtin_amdgcn_mfma_f64_16x16x4f64(b1[m].y, av[3], acc[m], 0, 0, 0);
                // every wavefront has stored its part of step t + 2 and read
                // buffer t (a bare barrier: a fence would wait for the loads)
                __builtin_amdgcn_s_waitcnt(kWaitLds);
                __builtin_amdgcn_s_barrier();
                const int done = cur;
                cur = nx1;
                nx1 = nx2;
                nx2 = done;
            }

            // lane (g, c) holds Y_mat of function i of granule g at point c in
            // element i of each block (row g + 4 i of the block: the MFMA
            // layout self-test); a padding granule's products are zero
            const int fn = xn < 0 ? 0 : (xn >> 13) * 4;
            const v4d R0 = *(const v4d *)(a.rf64 + fn), R1 = *(const v4d *)(a.rf64 + a.lda + fn),
                      R2 = *(const v4d *)(a.rf64 + 2 * (size_t)a.lda + fn);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const double t = acc[0][i] * ph[i];
                const double gr[3] = {g0[i], g1[i], g2[i]};
                q[0] += t;
                q[1] += t * (r[0] - R0[i]);
                q[2] += t * (r[1] - R1[i]);
                q[3] += t * (r[2] - R2[i]);
#pragma unroll
                for (int b = 0; b < 3; b++)
#pragma unroll
                    for (int m = 0; m < 3; m++) {
                        q[4 + m + 3 * b] += acc[1 + b][i] * gr[m];
                        q[13 + m + 3 * b] += gr[m] * acc[4 + b][i];
                    }
            }
        }
    }

    // add the four lane groups; group g stores sums g, g + 4, ...
    double *out = a.part + ((size_t)set * a.nsplit + split) * kNQ * (size_t)a.rows + row;
#pragma unroll
    for (int j = 0; j < kNQ; j += 4) {
        double s[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            s[i] = j + i < kNQ ? q[j + i < kNQ ? j + i : 0] : 0.0;
            s[i] += __shfl_xor(s[i], 16);
            s[i] += __shfl_xor(s[i], 32);
        }
        const double v = g == 0 ? s[0] : g == 1 ? s[1] : g == 2 ? s[2] : s[3];
        if (j + g < kNQ) out[(size_t)(j + g) * a.rows] = v;
    }
}

hipError_t launch_contract_f64(const ContractArgs &a, hipStream_t s) {
    if ((a.tile_rows != 64 && a.tile_rows != 128) || a.rows % a.tile_rows || a.lda % 32 ||
        a.ncol_pad != a.lda || a.ksplit < 1 || a.nsplit % a.ksplit)
        return hipErrorInvalidValue;
    ContractArgs b = a;
    const int ntile = a.rows / a.tile_rows;
    b.spread = a.spread && ntile < kSpreadTiles;
    const long long nwg = (b.spread ? ntile : 8LL * ((ntile + 7) / 8)) * a.nsplit * a.nmatset *
                          (a.tile_rows / 64);
    if (nwg > 0x7fffffffLL) return hipErrorInvalidValue;
    if (a.compressed)
        hipLaunchKernelGGL(contract_f64_kernel<true>, dim3((unsigned)nwg), dim3(256), 0, s, b);
    else
        hipLaunchKernelGGL(contract_f64_kernel<false>, dim3((unsigned)nwg), dim3(256), 0, s, b);
    return hipGetLastError();
}

}  // namespace gimic
