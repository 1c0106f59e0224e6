// Spatial point tiles and their screening-driven block lists (gfx950).
//
// Basis functions are zero beyond their contraction's screening radius
// (basis.f90:118-136), so over a compact tile of points most 32-function
// blocks of the basis are exactly zero in both the values phi and the
// gradients.  A zero K-block adds exact zeros to Y = Phi * B, and a zero
// N-block is multiplied by zeros in the epilogue, so a contraction
// workgroup that walks only the blocks that can be non-zero over its tile
// produces the same numbers as the dense product.
//
// Two steps per chunk of points:
//  1. Order the points along a curve through 32^3 cubic cells over their
//     bounding box (the Hilbert curve for the FP64 kernel, whose tiles list 2 to
//     12% fewer pairs than on the Morton curve, the 60-atom cage on 95^3 76.6
//     to 74.2 ms; the mixed kernels keep the latter, as their last digits
//     depend on the tiles; a stable LSD radix sort with two 8-bit digits of the
//     15-bit cell key, so the order - and with it every result bit - is the
//     same on every run); the basis, contraction and finalize kernels work on the
//     sorted rows, and finalize writes each tensor back to its caller index.
//  2. For every row tile of the contraction kernel, list in ascending order
//     the groups of 8 or 4 functions touched by a shell whose centre lies
//     within its screening radius of the tile's bounding box (a conservative
//     test: a group that is zero over the tile may be listed, one that is
//     not is never left out) and, for the FP64 kernel, of one of its points:
//     4 to 33% fewer (N-tile, K-step) pairs (shielding of the 30-atom sheet
//     1.17 to 1.06 ms, 256 planes of it 4.90 to 4.71, the 60-atom cage on 95^3
//     80.1 to 76.6).  The points are tested once per atom, 43 us for 5735 tiles
//     (28 with the box alone; 53 when every shell tested them).  The
//     mixed kernels keep the box alone: which groups share a K-step decides
//     the last digits of their FP32 sums.
#include "device_common.h"

namespace gimic {

namespace {

constexpr int kSortBlock = 1024;  // elements per radix block (4 rounds of 256)
constexpr int kBins = 256;        // 8-bit digits
// atoms whose distances an FP64 list takes into account (4 KiB of LDS); the
// lists of a larger molecule go by the box alone
constexpr int kListAtoms = 512;
constexpr int kCellBits = 5;      // 32 cells per axis: a 15-bit key, two digits
constexpr int kSmallSort = 2048;  // points that one workgroup sorts by itself
constexpr int kSmallBits = 11;    // of their index

__device__ __forceinline__ unsigned spread3(unsigned v) {
    // bits b0..b4 -> positions 0, 3, 6, 9, 12
    unsigned r = 0;
#pragma unroll
    for (int i = 0; i < kCellBits; i++) r |= ((v >> i) & 1u) << (3 * i);
    return r;
}

// min/max of the points, one partial box per workgroup: out[blk][6]
__global__ __launch_bounds__(256) void bbox_partial_kernel(const double *pts, int n, double *out) {
    __shared__ double s[6][256];
    const int t = threadIdx.x;
    double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (long long i = (long long)blockIdx.x * 256 + t; i < n; i += (long long)gridDim.x * 256)
#pragma unroll
        for (int d = 0; d < 3; d++) {
            const double x = pts[3 * i + d];
            lo[d] = fmin(lo[d], x);
            hi[d] = fmax(hi[d], x);
        }
#pragma unroll
    for (int d = 0; d < 3; d++) {
        s[d][t] = lo[d];
        s[3 + d][t] = hi[d];
    }
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (t < w)
#pragma unroll
            for (int d = 0; d < 3; d++) {
                s[d][t] = fmin(s[d][t], s[d][t + w]);
                s[3 + d][t] = fmax(s[3 + d][t], s[3 + d][t + w]);
            }
        __syncthreads();
    }
    if (t < 6) out[blockIdx.x * 6 + t] = s[t][0];
}

// Index of a cell along the Hilbert curve, three bits an octant (J. Skilling,
// "Programming the Hilbert curve", AIP Conf. Proc. 707, 381 (2004))
__device__ __forceinline__ unsigned hilbert3(unsigned x, unsigned y, unsigned z) {
    unsigned v[3] = {x, y, z};
#pragma unroll
    for (unsigned q = 1u << (kCellBits - 1); q > 1; q >>= 1) {
        const unsigned low = q - 1;
#pragma unroll
        for (int i = 0; i < 3; i++) {
            // set: invert the low bits of x; clear: exchange them with x's
            const unsigned t = (v[0] ^ v[i]) & low;
            const bool set = v[i] & q;
            v[0] ^= set ? low : t;
            if (i > 0) v[i] ^= set ? 0u : t;
        }
    }
    v[1] ^= v[0];
    v[2] ^= v[1];
    unsigned t = 0;
#pragma unroll
    for (unsigned q = 1u << (kCellBits - 1); q > 1; q >>= 1)
        if (v[2] & q) t ^= q - 1;
    return spread3(v[0] ^ t) << 2 | spread3(v[1] ^ t) << 1 | spread3(v[2] ^ t);
}

// Key of the cell of a point in the box [lo, hi]: its place on the Morton or
// the Hilbert curve
__device__ __forceinline__ unsigned cell_key(const double *pt, const double (&lo)[3],
                                             const double (&hi)[3], bool hilbert) {
    double h = fmax(fmax(hi[0] - lo[0], hi[1] - lo[1]), hi[2] - lo[2]) / (1 << kCellBits);
    if (!(h > 0.0) || !isfinite(h)) h = 1.0;
    unsigned c[3];
#pragma unroll
    for (int d = 0; d < 3; d++)
        // fmax/fmin map NaN to the first cell
        c[d] = (unsigned)fmin(fmax((pt[d] - lo[d]) / h, 0.0), (double)((1 << kCellBits) - 1));
    return hilbert ? hilbert3(c[0], c[1], c[2])
                   : spread3(c[0]) | spread3(c[1]) << 1 | spread3(c[2]) << 2;
}

// Up to kSmallSort points in one workgroup and launch: box, keys, a bitonic
// sort of (key, index) in LDS (unique keys, so the order is the stable one),
// and the sorted points.  A single point took 14 launches of the general sort,
// half of the time of its tensor.
__global__ __launch_bounds__(1024) void small_sort_kernel(const double *pts, int n, double *spts,
                                                          int *perm, bool hilbert) {
    __shared__ unsigned v[kSmallSort];
    __shared__ double box[16][6];
    const int t = threadIdx.x, nt = blockDim.x, lane = t & 63, wave = t >> 6;
    double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (int i = t; i < n; i += nt)
#pragma unroll
        for (int d = 0; d < 3; d++) {
            lo[d] = fmin(lo[d], pts[3 * i + d]);
            hi[d] = fmax(hi[d], pts[3 * i + d]);
        }
    wave_box(lo, hi);
    if (lane == 0)
#pragma unroll
        for (int d = 0; d < 3; d++) {
            box[wave][d] = lo[d];
            box[wave][3 + d] = hi[d];
        }
    __syncthreads();
    for (int w = 0; w < nt / 64; w++)
#pragma unroll
        for (int d = 0; d < 3; d++) {
            lo[d] = fmin(lo[d], box[w][d]);
            hi[d] = fmax(hi[d], box[w][3 + d]);
        }
    int m = 1;
    while (m < n) m <<= 1;
    for (int i = t; i < m; i += nt)
        v[i] = i < n ? cell_key(pts + 3 * i, lo, hi, hilbert) << kSmallBits | (unsigned)i : ~0u;
    for (int k = 2; k <= m; k <<= 1)
        for (int j = k >> 1; j > 0; j >>= 1) {
            __syncthreads();
            for (int q = t; q < m / 2; q += nt) {
                const int i = (q & ~(j - 1)) << 1 | (q & (j - 1)), o = i | j;
                const unsigned x = v[i], y = v[o];
                if ((x > y) == ((i & k) == 0)) {
                    v[i] = y;
                    v[o] = x;
                }
            }
        }
    __syncthreads();
    for (int j = t; j < n; j += nt) {
        const int i = (int)(v[j] & ((1u << kSmallBits) - 1));
        perm[j] = i;
#pragma unroll
        for (int d = 0; d < 3; d++) spts[3 * j + d] = pts[3 * i + d];
    }
}

// Counts of digit `shift` of 1024 keys, digit-major: hist[d * nb + b].  FIRST:
// the keys come from the points and the partial boxes, and are stored.
template <bool FIRST>
__global__ __launch_bounds__(256) void radix_hist_kernel(const double *pts, const double *bpart,
                                                         int nbpart, unsigned *keys, int n, int shift,
                                                         int *hist, bool hilbert) {
    __shared__ int cnt[kBins];
    __shared__ double box[4][6];
    const int t = threadIdx.x, b = blockIdx.x, nb = gridDim.x;
    double lo[3], hi[3];
    cnt[t] = 0;
    if (FIRST) {
#pragma unroll
        for (int d = 0; d < 3; d++) {
            lo[d] = t < nbpart ? bpart[t * 6 + d] : INFINITY;
            hi[d] = t < nbpart ? bpart[t * 6 + 3 + d] : -INFINITY;
        }
        wave_box(lo, hi);
        if ((t & 63) == 0)
#pragma unroll
            for (int d = 0; d < 3; d++) {
                box[t >> 6][d] = lo[d];
                box[t >> 6][3 + d] = hi[d];
            }
    }
    __syncthreads();
    if (FIRST)
        for (int w = 0; w < 4; w++)
#pragma unroll
            for (int d = 0; d < 3; d++) {
                lo[d] = fmin(lo[d], box[w][d]);
                hi[d] = fmax(hi[d], box[w][3 + d]);
            }
    for (int r = 0; r < kSortBlock / 256; r++) {
        const long long i = (long long)b * kSortBlock + r * 256 + t;
        if (i >= n) break;
        unsigned key;
        if (FIRST) keys[i] = key = cell_key(pts + 3 * i, lo, hi, hilbert);
        else key = keys[i];
        atomicAdd(&cnt[(key >> shift) & (kBins - 1)], 1);
    }
    __syncthreads();
    hist[t * nb + b] = cnt[t];
}

// exclusive scan over the 256 threads of a workgroup; wsum: 4 ints of LDS
__device__ __forceinline__ int scan256(int x, int *wsum, int &total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int inc = x;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int y = __shfl_up(inc, d);
        if (lane >= d) inc += y;
    }
    __syncthreads();  // wsum may still be read from an earlier scan
    if (lane == 63) wsum[wave] = inc;
    __syncthreads();
    int before = 0;
    total = 0;
#pragma unroll
    for (int w = 0; w < 4; w++) {
        if (w < wave) before += wsum[w];
        total += wsum[w];
    }
    return before + inc - x;
}

// workgroup d: exclusive scan of digit d's counts over the radix blocks in
// place, their sum into digits[d]
__global__ __launch_bounds__(256) void radix_scan_kernel(int *hist, int nb, int *digits) {
    __shared__ int wsum[4];
    int *v = hist + (long long)blockIdx.x * nb;
    int carry = 0;
    for (int base = 0; base < nb; base += 256) {
        const int i = base + threadIdx.x, x = i < nb ? v[i] : 0;
        int total;
        const int before = scan256(x, wsum, total);
        if (i < nb) v[i] = carry + before;
        carry += total;
    }
    if (threadIdx.x == 0) digits[blockIdx.x] = carry;
}

// stable scatter by digit: element order within a digit is kept.  LAST: the
// output is the permutation and the points in its order
template <bool LAST>
__global__ __launch_bounds__(256) void radix_scatter_kernel(const unsigned *kin, const int *iin, int n,
                                                            int shift, const int *hist,
                                                            const int *digits, unsigned *kout, int *iout,
                                                            const double *pts, double *spts) {
    __shared__ int wcnt[4][kBins];
    __shared__ int run[kBins];
    __shared__ int wsum[4];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, b = blockIdx.x, nb = gridDim.x;
    int total;
    run[t] = scan256(digits[t], wsum, total) + hist[(long long)t * nb + b];
    const unsigned long long below = (1ull << lane) - 1ull;
    for (int r = 0; r < kSortBlock / 256; r++) {
        const long long i = (long long)b * kSortBlock + r * 256 + t;
        const bool valid = i < n;
        const unsigned key = valid ? kin[i] : 0u;
        const int dig = (int)((key >> shift) & (kBins - 1));
#pragma unroll
        for (int w = 0; w < 4; w++) wcnt[w][t] = 0;
        // lanes of this wavefront with the same digit
        unsigned long long same = __ballot(valid);
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const unsigned long long m = __ballot((dig >> k) & 1);
            same &= (dig >> k) & 1 ? m : ~m;
        }
        const int rank = __popcll(same & below);
        __syncthreads();  // wcnt cleared, run up to date
        if (valid && rank == 0) wcnt[wave][dig] = __popcll(same);
        __syncthreads();
        if (valid) {
            int pos = run[dig] + rank;
            for (int w = 0; w < wave; w++) pos += wcnt[w][dig];
            const int idx = LAST ? iin[i] : (int)i;
            iout[pos] = idx;
            if (LAST) {
#pragma unroll
                for (int d = 0; d < 3; d++) spts[3 * (long long)pos + d] = pts[3 * (long long)idx + d];
            } else {
                kout[pos] = key;
            }
        }
        __syncthreads();  // every thread has read run and wcnt
        run[t] += wcnt[0][t] + wcnt[1][t] + wcnt[2][t] + wcnt[3][t];
    }
}

// One workgroup per row tile: bounding box of its valid rows, the granules (4
// functions) that a shell within reach of it touches, and the ascending list
// of the live groups.  Threads take shells for the liveness test and blocks
// for the list (positions by a prefix sum): one thread walking the blocks
// took 12 us for a single tile, this 5.
constexpr int kMaxBlk = 1024;  // 32-function blocks per row (32768 functions)

__global__ __launch_bounds__(256) void block_list_kernel(TileArgs a) {
    __shared__ double box[4][6];
    __shared__ int wsum[4][3];
    __shared__ unsigned live[kMaxBlk];  // live granules of each block, 8 bits
    __shared__ double pts[3 * kWgRows], near2[kListAtoms];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const long long r0 = (long long)blockIdx.x * a.tile_rows;
    double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (int r = t; r < a.tile_rows; r += 256) {
        const long long p = r0 + r;
        if (p < a.npts)
#pragma unroll
            for (int d = 0; d < 3; d++) {
                const double x = a.spts[3 * p + d];
                if (a.gran == 4) pts[3 * r + d] = x;
                lo[d] = fmin(lo[d], x);
                hi[d] = fmax(hi[d], x);
            }
    }
    for (int b = t; b < a.nblk; b += 256) live[b] = 0u;
    wave_box(lo, hi);
    if (lane == 0)
#pragma unroll
        for (int d = 0; d < 3; d++) {
            box[wave][d] = lo[d];
            box[wave][3 + d] = hi[d];
        }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < 4; w++)
#pragma unroll
        for (int d = 0; d < 3; d++) {
            lo[d] = fmin(lo[d], box[w][d]);
            hi[d] = fmax(hi[d], box[w][3 + d]);
        }
    // FP64 lists: the points after the box, by the squared distance of every
    // atom from the nearest one (`share` lanes an atom)
    const bool points = a.gran == 4 && a.natoms <= kListAtoms;
    if (points) {
        const int np = (int)min((long long)a.tile_rows, max(0LL, a.npts - r0));
        const int share = a.natoms <= 32 ? 8 : a.natoms <= 64 ? 4 : a.natoms <= 128 ? 2 : 1;
        for (int i0 = 0; i0 < a.natoms * share; i0 += 256) {
            const int atom = (i0 + t) / share, q = t % share;
            const double *R = a.coords + 3 * min(atom, a.natoms - 1);
            const double R0 = R[0], R1 = R[1], R2 = R[2];
            double m = INFINITY;
#pragma unroll 4
            for (int p = q; p < np; p += share) {
                const double x = pts[3 * p] - R0, y = pts[3 * p + 1] - R1, z = pts[3 * p + 2] - R2;
                m = fmin(m, x * x + y * y + z * z);
            }
            for (int d = 1; d < share; d <<= 1) m = fmin(m, __shfl_xor(m, d));
            if (q == 0 && atom < a.natoms) near2[atom] = m;
        }
        __syncthreads();
    }
    if (r0 < a.npts)
        for (int k = t; k < a.nshell; k += 256) {
            const DevShell sh = a.shells[k];
            const double reach = shell_reach(sh);
            if (box_distance(lo, hi, a.coords + 3 * sh.atom) <= reach &&
                (!points || near2[sh.atom] <= reach * reach))
                for (int q = sh.fout >> 2; q <= (sh.fout + sh.ncomp_out - 1) >> 2; q++)
                    atomicOr(&live[q >> 3], 1u << (q & 7));
        }
    __syncthreads();
    const int per = 32 / a.gran, shift = a.gran == 8 ? 12 : 13;
    int *list = a.klist + (long long)blockIdx.x * a.nblk * per;
    int base = 0, nb = 0, n8 = 0;
    for (int b0 = 0; b0 < a.nblk; b0 += 256) {
        const int b = b0 + t;
        const unsigned m4 = b < a.nblk ? live[b] : 0u;   // granules of 4
        const unsigned m8 = (m4 | m4 >> 1) & 0x55u;      // groups of 8, every second bit
        const unsigned m = a.gran == 8 ? m8 : m4;
        const int cnt = __popc(m);
        int inc = cnt;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int y = __shfl_up(inc, d);
            if (lane >= d) inc += y;
        }
        int g8 = __popc(m8);
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) g8 += __shfl_xor(g8, d);
        const int blocks = __popcll(__ballot(m4 != 0u));
        if (lane == 63) {
            wsum[wave][0] = inc;
            wsum[wave][1] = g8;
            wsum[wave][2] = blocks;
        }
        __syncthreads();
        int pos = base + inc - cnt;
        for (int w = 0; w < 4; w++) {
            if (w < wave) pos += wsum[w][0];
            base += wsum[w][0];
            n8 += wsum[w][1];
            nb += wsum[w][2];
        }
        for (int q = 0; q < per; q++)
            if (m >> (a.gran == 8 ? 2 * q : q) & 1u) {
                list[pos] = (per * b + q) << shift | pos;
                pos++;
            }
        __syncthreads();
    }
    if (t == 0) {
        a.bcount[blockIdx.x] = nb;
        a.k8count[blockIdx.x] = n8;
        a.kcount[blockIdx.x] = base;
    }
    if (t < (-base & 3)) list[base + t] = -1;  // four per N-tile and K-step
}

}  // namespace

int sort_scratch_ints(int n) {
    const int nb = (n + kSortBlock - 1) / kSortBlock;
    return 3 * n + kBins * nb + kBins;  // keys twice, indices, digit counts
}

hipError_t launch_sort_points(const double *pts, int n, double *spts, int *perm, double *bpart,
                              int *scratch, bool hilbert, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    if (n <= kSmallSort) {
        const int threads = n <= 128 ? 64 : n <= 512 ? 256 : 1024;
        hipLaunchKernelGGL(small_sort_kernel, dim3(1), dim3(threads), 0, s, pts, n, spts, perm,
                           hilbert);
        return hipGetLastError();
    }
    const int nb = (n + kSortBlock - 1) / kSortBlock;
    unsigned *k0 = (unsigned *)scratch, *k1 = k0 + n;
    int *i1 = scratch + 2 * (long long)n, *hist = i1 + n, *digits = hist + (long long)kBins * nb;
    const int npart = n < 256 * 256 ? (n + 255) / 256 : 256;
    hipLaunchKernelGGL(bbox_partial_kernel, dim3(npart), dim3(256), 0, s, pts, n, bpart);
    hipLaunchKernelGGL(radix_hist_kernel<true>, dim3(nb), dim3(256), 0, s, pts, (const double *)bpart,
                       npart, k0, n, 0, hist, hilbert);
    hipLaunchKernelGGL(radix_scan_kernel, dim3(kBins), dim3(256), 0, s, hist, nb, digits);
    hipLaunchKernelGGL(radix_scatter_kernel<false>, dim3(nb), dim3(256), 0, s, (const unsigned *)k0,
                       (const int *)nullptr, n, 0, (const int *)hist, (const int *)digits, k1, i1,
                       (const double *)nullptr, (double *)nullptr);
    hipLaunchKernelGGL(radix_hist_kernel<false>, dim3(nb), dim3(256), 0, s, (const double *)nullptr,
                       (const double *)nullptr, 0, k1, n, 8, hist, hilbert);
    hipLaunchKernelGGL(radix_scan_kernel, dim3(kBins), dim3(256), 0, s, hist, nb, digits);
    hipLaunchKernelGGL(radix_scatter_kernel<true>, dim3(nb), dim3(256), 0, s, (const unsigned *)k1,
                       (const int *)i1, n, 8, (const int *)hist, (const int *)digits,
                       (unsigned *)nullptr, perm, pts, spts);
    return hipGetLastError();
}

// One workgroup: counting sort of the row tiles by list length, longest first.
// In points' order the last workgroups of a launch are as long as any, and CUs
// stand idle behind them, 10 to 20% of the launch: shielding of the 30-atom
// sheet 1.29 ms against 1.18, 256 planes of it in FP64 5.28 against 4.91, the
// open-shell sheet in mixed precision 19.6 against 18.7, the 60-atom cage
// 82.6 against 80.1 (FP64) and 70.6 against 68.1 (mixed).
constexpr int kOrderBins = 1024;
__global__ __launch_bounds__(kOrderBins) void tile_order_kernel(const int *kcount, int ntile,
                                                                int most, int2 *order) {
    __shared__ int hist[kOrderBins], wsum[kOrderBins / 64];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    auto bin = [&](int k) {
        return kOrderBins - 1 - (int)((long long)min(k, most) * (kOrderBins - 1) / most);
    };
    hist[t] = 0;
    __syncthreads();
    for (int i = t; i < ntile; i += kOrderBins) atomicAdd(&hist[bin(kcount[i])], 1);
    __syncthreads();
    const int n = hist[t];
    int sum = n;  // inclusive over the wavefront
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int v = __shfl_up(sum, d);
        if (lane >= d) sum += v;
    }
    if (lane == 63) wsum[w] = sum;
    __syncthreads();
    int before = 0;
    for (int i = 0; i < w; i++) before += wsum[i];
    hist[t] = before + sum - n;
    __syncthreads();
    for (int i = t; i < ntile; i += kOrderBins) {
        const int k = kcount[i];
        order[atomicAdd(&hist[bin(k)], 1)] = make_int2(i, k);
    }
}

hipError_t launch_tile_order(const int *kcount, int ntile, int most, int2 *order, hipStream_t s) {
    if (ntile <= 0 || most <= 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(tile_order_kernel, dim3(1), dim3(kOrderBins), 0, s, kcount, ntile, most,
                       order);
    return hipGetLastError();
}

hipError_t launch_block_lists(const TileArgs &a, hipStream_t s) {
    if (a.gran == 4 && a.tile_rows > kWgRows) return hipErrorInvalidValue;
    if (a.tile_rows <= 0 || a.rows % a.tile_rows || a.nblk <= 0 || a.nblk > kMaxBlk ||
        (a.gran != 8 && a.gran != 4))
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(block_list_kernel, dim3(a.rows / a.tile_rows), dim3(256), 0, s, a);
    return hipGetLastError();
}

}  // namespace gimic
