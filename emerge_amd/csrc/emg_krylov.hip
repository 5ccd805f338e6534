// Complex sparse Krylov solver for the frequency-domain systems on MI355X.
//
// Replaces the per-frequency direct solve of the reference
// (fem/solver.py:405-469: PEC elimination, PARDISO / SuperLU / GMRES+ILU) with
// right-preconditioned restarted GMRES on the GPU:
//   * PEC DOFs are eliminated implicitly: the operator is
//     y = mask.(K (mask.x)) + (1 - mask).x, so x_PEC = 0 exactly and no
//     reduced matrix is ever formed (solver.py:430-435 builds one per call);
//   * the solver's own vectors hold the two modes of an entity side by side and
//     its matrix 2x2 blocks in a real and an imaginary plane, the latter read
//     only where there are losses ("packed solver layout" below);
//   * Gram-Schmidt is classical, as a tiled multi-dot and a fused multi-AXPY
//     + norm, so each Arnoldi step streams the basis twice instead of j
//     times; the multi-dot also brings the basis' Gram matrix up, which takes
//     the place of a second pass (k_gram_correct);
//   * the preconditioner is the inverse of the 2x2 blocks coupling the two
//     modes of each edge / face, with the gradient correction and the GMRES
//     polynomial when set;
//   * precision 32 runs GMRES in complex64 inside FP64 iterative refinement:
//     the residual b - K x is always formed in complex128, and the cycles of
//     one solve share their Krylov spaces (gmres_cycle).

#include <algorithm>
#include <cmath>
#include <complex>
#include <cstring>
#include <limits>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/emerge_amd.h"
#include "emg_common.h"

using emg::cplx;

template <typename R>
struct cx {
    R re, im;
    __device__ __forceinline__ cx() : re(0), im(0) {}
    __device__ __forceinline__ cx(R r, R i) : re(r), im(i) {}
};
template <typename R>
__device__ __forceinline__ cx<R> cmul(cx<R> a, cx<R> b) { return cx<R>(a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re); }
template <typename R>
__device__ __forceinline__ cx<R> cadd(cx<R> a, cx<R> b) { return cx<R>(a.re + b.re, a.im + b.im); }

template <typename R>
__device__ __forceinline__ cx<R> ld(const R *p, int64_t i) {
    if constexpr (sizeof(R) == 8) {
        const double2 v = reinterpret_cast<const double2 *>(p)[i];
        return cx<R>(v.x, v.y);
    } else {
        const float2 v = reinterpret_cast<const float2 *>(p)[i];
        return cx<R>(v.x, v.y);
    }
}
template <typename R>
__device__ __forceinline__ void st(R *p, int64_t i, cx<R> v) {
    if constexpr (sizeof(R) == 8) {
        reinterpret_cast<double2 *>(p)[i] = make_double2(v.re, v.im);
    } else {
        reinterpret_cast<float2 *>(p)[i] = make_float2(v.re, v.im);
    }
}

// Sum over groups of L = 4 .. 64 consecutive lanes, left in every lane: the steps within 16 lanes are
// data-parallel-primitive adds (quad permutes, half-row and row mirrors), a few cycles each where a
// shuffle through LDS takes over a hundred; the pairs added are those of the xor butterfly.
template <int CTRL>
__device__ __forceinline__ float dpp_mov(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ double dpp_mov(double v) {
    return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true),
                            __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true));
}
static constexpr int DPP_XOR1 = 0xB1, DPP_XOR2 = 0x4E, DPP_HALF_MIRROR = 0x141, DPP_MIRROR = 0x140, DPP_ROR8 = 0x128;
template <int L, typename T>
__device__ __forceinline__ T lane_sum(T v) {
    static_assert(L == 4 || L == 8 || L == 16 || L == 32 || L == 64, "lane_sum: group size");
    v += dpp_mov<DPP_XOR1>(v);
    v += dpp_mov<DPP_XOR2>(v);
    if constexpr (L >= 8) v += dpp_mov<DPP_HALF_MIRROR>(v);
    if constexpr (L >= 16) v += dpp_mov<DPP_MIRROR>(v);
    if constexpr (L >= 32) v += __shfl_xor(v, 16, 64);
    if constexpr (L >= 64) v += __shfl_xor(v, 32, 64);
    return v;
}

static constexpr int SUB = 16;  // lanes per CSR row
// (SpMV rows stay in dispatch order: giving each XCD a contiguous share of the
// rows fetched a third fewer bytes but ran 30 % slower.)

// y = mask.(A (mask.x)) + (1-mask).x   (mask == nullptr: plain y = A x).  L lanes share one CSR row.
template <int L>
__global__ void __launch_bounds__(256) k_spmv(int64_t n, const int32_t *__restrict__ rowptr, const int32_t *__restrict__ cols,
                                              const double *__restrict__ vals, const uint8_t *__restrict__ mask,
                                              const double *__restrict__ x, double *__restrict__ y) {
    const int64_t row = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) / L;
    const int lane = threadIdx.x % L;
    if (row >= n) return;
    const bool keep = mask == nullptr || mask[row];
    cx<double> acc;
    if (keep) {
        const int32_t p0 = rowptr[row], p1 = rowptr[row + 1];
        for (int32_t p = p0 + lane; p < p1; p += L) {
            const int32_t c = cols[p];
            if (mask != nullptr && !mask[c]) continue;
            acc = cadd(acc, cmul(ld(vals, p), ld(x, c)));
        }
    }
    acc = cx<double>(lane_sum<L>(acc.re), lane_sum<L>(acc.im));
    if (lane == 0) st(y, row, keep ? acc : ld(x, row));
}

// Lanes per CSR row for the SpMV: EMG_SPMV_LANES (4, 8, 16 or 32) if set, else 16.
static int spmv_lanes() {
    static int lanes = 0;
    if (lanes == 0) {
        const char *e = getenv("EMG_SPMV_LANES");
        const int v = e ? atoi(e) : 16;
        lanes = (v == 4 || v == 8 || v == 16 || v == 32) ? v : 16;
    }
    return lanes;
}

static void launch_spmv(hipStream_t st, int64_t n, const int32_t *rowptr, const int32_t *cols, const double *vals,
                        const uint8_t *mask, const double *x, double *y) {
    const int L = spmv_lanes();
    const unsigned grid = (unsigned)((n * L + 255) / 256);
    switch (L) {
        case 4: k_spmv<4><<<grid, 256, 0, st>>>(n, rowptr, cols, vals, mask, x, y); break;
        case 8: k_spmv<8><<<grid, 256, 0, st>>>(n, rowptr, cols, vals, mask, x, y); break;
        case 32: k_spmv<32><<<grid, 256, 0, st>>>(n, rowptr, cols, vals, mask, x, y); break;
        default: k_spmv<16><<<grid, 256, 0, st>>>(n, rowptr, cols, vals, mask, x, y); break;
    }
}

// SpMV of a matrix on an entity pattern (emg_pattern_csr): DOF = mode * ne +
// entity, and the rows (0, e) and (1, e) hold the same entities e'_j, row
// (m, e) storing its (0, e'_j) entries at r_m + j and its (1, e'_j) entries at
// r_m + deg + j, r_0 = rowptr[e], r_1 = r_0 + half (half = nnz / 2).  One
// group of L lanes computes both rows of entity e: each column index and each
// pair of x gathers serves four matrix entries.  Same masking as k_spmv.
template <int L>
__global__ void __launch_bounds__(256) k_spmv_blk(int64_t ne, int64_t half, const int32_t *__restrict__ rowptr,
                                                  const int32_t *__restrict__ cols, const double *__restrict__ vals,
                                                  const uint8_t *__restrict__ mask, const double *__restrict__ x,
                                                  const double *__restrict__ b, double *__restrict__ y) {
    const int64_t e = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) / L;
    const int lane = threadIdx.x % L;
    if (e >= ne) return;
    const bool k0 = mask == nullptr || mask[e], k1 = mask == nullptr || mask[ne + e];
    cx<double> a0, a1;
    if (k0 || k1) {
        const int32_t r0 = rowptr[e];
        // a row beyond the first half is not an entity pattern: read nothing past nnz
        const int32_t deg = (rowptr[e + 1] <= half && rowptr[e + 1] >= r0) ? (rowptr[e + 1] - r0) >> 1 : 0;
        for (int32_t j = lane; j < deg; j += L) {
            const int32_t c = cols[r0 + j];
            if (c < 0 || c >= ne) continue;   // not an entity pattern: no out-of-range reads
            cx<double> x0 = ld(x, c), x1 = ld(x, ne + c);
            if (mask != nullptr) {
                if (!mask[c]) x0 = cx<double>();
                if (!mask[ne + c]) x1 = cx<double>();
            }
            const int64_t p = r0 + j;
            a0 = cadd(a0, cadd(cmul(ld(vals, p), x0), cmul(ld(vals, p + deg), x1)));
            a1 = cadd(a1, cadd(cmul(ld(vals, half + p), x0), cmul(ld(vals, half + p + deg), x1)));
        }
    }
    a0 = cx<double>(lane_sum<L>(a0.re), lane_sum<L>(a0.im));
    a1 = cx<double>(lane_sum<L>(a1.re), lane_sum<L>(a1.im));
    if (lane == 0) {
        cx<double> v0 = k0 ? a0 : ld(x, e), v1 = k1 ? a1 : ld(x, ne + e);
        if (b != nullptr) {
            const cx<double> b0 = ld(b, e), b1 = ld(b, ne + e);
            v0 = cx<double>(b0.re - v0.re, b0.im - v0.im);
            v1 = cx<double>(b1.re - v1.re, b1.im - v1.im);
        }
        st(y, e, v0);
        st(y, ne + e, v1);
    }
}

// Lanes per entity row of the blocked SpMV when nothing was tuned (the public
// emg_spmv_blocked, or EMG_SPMV_BLK_LANES set): EMG_SPMV_BLK_LANES (4, 8, 16 or
// 32) if set, else 16.  Solvers tune their own (tune_spmv).
static int spmv_blk_lanes() {
    const char *e = getenv("EMG_SPMV_BLK_LANES");
    const int v = e ? atoi(e) : 16;
    return (v == 4 || v == 8 || v == 16 || v == 32) ? v : 16;
}

static void launch_spmv_blk(hipStream_t st, int64_t n, int64_t nnz, const int32_t *rowptr, const int32_t *cols,
                            const double *vals, const uint8_t *mask, const double *x, const double *b, double *y, int L) {
    const int64_t ne = n / 2, half = nnz / 2;
    if (L != 4 && L != 8 && L != 32) L = 16;
    const unsigned grid = (unsigned)((ne * L + 255) / 256);
    if (L == 4) k_spmv_blk<4><<<grid, 256, 0, st>>>(ne, half, rowptr, cols, vals, mask, x, b, y);
    else if (L == 8) k_spmv_blk<8><<<grid, 256, 0, st>>>(ne, half, rowptr, cols, vals, mask, x, b, y);
    else if (L == 32) k_spmv_blk<32><<<grid, 256, 0, st>>>(ne, half, rowptr, cols, vals, mask, x, b, y);
    else k_spmv_blk<16><<<grid, 256, 0, st>>>(ne, half, rowptr, cols, vals, mask, x, b, y);
}

// ---------------------------------------------------------------- BLAS-1
static constexpr int RB = 256;   // reduction block
static constexpr int DT = 8;     // dot products per tile

// Two consecutive complex values: in the solver's own vectors the two modes of an
// entity (DOFs e and ne + e side by side), one 16-byte access in complex64.
template <typename R>
struct cx2 {
    R ar, ai, br, bi;
};
template <typename R>
__device__ __forceinline__ cx2<R> ld2(const R *p, int64_t i) {
    if constexpr (sizeof(R) == 8) {
        const double2 u = reinterpret_cast<const double2 *>(p)[2 * i], v = reinterpret_cast<const double2 *>(p)[2 * i + 1];
        return cx2<R>{u.x, u.y, v.x, v.y};
    } else {
        const float4 u = reinterpret_cast<const float4 *>(p)[i];
        return cx2<R>{u.x, u.y, u.z, u.w};
    }
}
template <typename R>
__device__ __forceinline__ void st2(R *p, int64_t i, cx2<R> v) {
    if constexpr (sizeof(R) == 8) {
        reinterpret_cast<double2 *>(p)[2 * i] = make_double2(v.ar, v.ai);
        reinterpret_cast<double2 *>(p)[2 * i + 1] = make_double2(v.br, v.bi);
    } else {
        reinterpret_cast<float4 *>(p)[i] = make_float4(v.ar, v.ai, v.br, v.bi);
    }
}

__device__ __forceinline__ double block_sum(double v, double *sh) {
    v = lane_sum<64>(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    double t = 0.0;
    for (int q = 0; q < (int)(blockDim.x >> 6); q++) t += sh[q];
    return t;
}

// partial[r][tile][blk][k] = sum over the block's elements of conj(V_{t*DT+k}) . w_r for RHS = 1 or 2
// vectors w_r, two complex values per lane and vector (an odd n leaves its last value to the first
// lane).  A tile past the last vector reads that one again and its sums are not used: a test per vector
// instead keeps the eight loads from being in flight together.  Bound by the bytes of V, which two
// right-hand sides share.
template <typename R, int RHS>
__global__ void __launch_bounds__(RB) k_mdot(int64_t n, int nv, const R *__restrict__ V, int64_t ldv,
                                             const R *__restrict__ w, const R *__restrict__ w2,
                                             double *__restrict__ partial) {
    constexpr int NS = 2 * DT * RHS;   // sums: real parts, imaginary parts, of each right-hand side
    static_assert(NS == 16 || NS == 32, "the wavefront reduction handles 16 or 32 sums");
    __shared__ double sv[NS][RB / 64];
    const int tile = blockIdx.y;
    const int i0 = tile * DT;
    double v[NS];
#pragma unroll
    for (int k = 0; k < NS; k++) v[k] = 0;
    auto add = [&](double *a, const cx2<R> &x, const cx2<R> &y) {
        a[0] += (double)x.ar * y.ar + (double)x.ai * y.ai + (double)x.br * y.br + (double)x.bi * y.bi;
        a[DT] += (double)x.ar * y.ai - (double)x.ai * y.ar + (double)x.br * y.bi - (double)x.bi * y.br;
    };
    // two complex values per lane; of complex128 with two right-hand sides one (DOT1), which leaves registers
    // for 4 waves per SIMD (1,947,698 DOFs, 75 vectors: 706 -> 427 us for 2.3 GB, where 3 waves did not hide the loads)
    constexpr bool DOT1 = sizeof(R) == 8 && RHS == 2;
    if constexpr (DOT1) {
        for (int64_t e = blockIdx.x * (int64_t)RB + threadIdx.x; e < n; e += (int64_t)gridDim.x * RB) {
            const cx<R> wv = ld(w, e), wv2 = ld(w2, e);
            cx<R> x[DT];
#pragma unroll
            for (int k = 0; k < DT; k++) x[k] = ld(V + (int64_t)min(i0 + k, nv - 1) * ldv * 2, e);
#pragma unroll
            for (int k = 0; k < DT; k++) {
                v[k] += x[k].re * wv.re + x[k].im * wv.im;
                v[DT + k] += x[k].re * wv.im - x[k].im * wv.re;
                v[2 * DT + k] += x[k].re * wv2.re + x[k].im * wv2.im;
                v[3 * DT + k] += x[k].re * wv2.im - x[k].im * wv2.re;
            }
        }
    }
    const int64_t n2 = DOT1 ? 0 : n >> 1;
    for (int64_t e = blockIdx.x * (int64_t)RB + threadIdx.x; e < n2; e += (int64_t)gridDim.x * RB) {
        const cx2<R> wv = ld2(w, e);
        cx2<R> wv2{};
        if constexpr (RHS == 2) wv2 = ld2(w2, e);
        cx2<R> x[DT];
#pragma unroll
        for (int k = 0; k < DT; k++) x[k] = ld2(V + (int64_t)min(i0 + k, nv - 1) * ldv * 2, e);
#pragma unroll
        for (int k = 0; k < DT; k++) {
            add(v + k, x[k], wv);
            if constexpr (RHS == 2) add(v + 2 * DT + k, x[k], wv2);
        }
    }
    if (!DOT1 && (n & 1) && blockIdx.x == 0 && threadIdx.x == 0) {
        auto last = [&](const R *a) {
            const cx<R> u = ld(a, n - 1);
            return cx2<R>{u.re, u.im, R(0), R(0)};
        };
        const cx2<R> wv = last(w);
#pragma unroll
        for (int k = 0; k < DT; k++) {
            const cx2<R> x = last(V + (int64_t)min(i0 + k, nv - 1) * ldv * 2);
            add(v + k, x, wv);
            if constexpr (RHS == 2) add(v + 2 * DT + k, x, last(w2));
        }
    }
    // the sums over the wavefront: each step hands half of the values to the partner lane and adds the
    // other half, NS - 1 exchanges and a last add or two instead of the 6 NS shuffles of NS butterflies
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int half = NS / 2, bit = 32; half >= 1; half >>= 1, bit >>= 1) {
#pragma unroll
        for (int k = 0; k < half; k++) {
            const double give = (lane & bit) ? v[k] : v[k + half], keep = (lane & bit) ? v[k + half] : v[k];
            v[k] = keep + (bit == 8 ? dpp_mov<DPP_ROR8>(give) : bit == 2 ? dpp_mov<DPP_XOR2>(give) : __shfl_xor(give, bit, 64));
        }
    }
    // value i is with lanes (64 / NS) i ...: the highest bit of the lane is the highest of i, and so on
    if constexpr (NS == 16) v[0] += dpp_mov<DPP_XOR2>(v[0]);
    v[0] += dpp_mov<DPP_XOR1>(v[0]);
    if (lane % (64 / NS) == 0) sv[lane / (64 / NS)][threadIdx.x >> 6] = v[0];
    __syncthreads();
    if (threadIdx.x < NS) {
        double t = 0;
        for (int q = 0; q < RB / 64; q++) t += sv[threadIdx.x][q];
        const int r = threadIdx.x / (2 * DT), c = (threadIdx.x / DT) & 1, k = threadIdx.x % DT;
        const int64_t o = (((int64_t)r * gridDim.y + tile) * gridDim.x + blockIdx.x) * DT + k;
        partial[2 * o + c] = t;
    }
}

// h[i] = sc_i * sum over blocks of the partials (complex, i < nv); one block per value.
// gridDim.y = 2 (k_mdot<R, 2> with the last basis vector as second right-hand side): the second sums
// are that vector's column of the basis' Gram matrix, of which E (row length ld) keeps the deviation
// from the identity.
__global__ void k_mdot_finish(int nv, int nblk, const double *__restrict__ partial, const double *__restrict__ sc,
                              double *__restrict__ h, double *__restrict__ E, int ld) {
    const int i = blockIdx.x;
    if (i >= nv) return;
    const int tile = i / DT, k = i % DT, ntile = (nv + DT - 1) / DT;
    double r = 0, im = 0;
    for (int b = threadIdx.x; b < nblk; b += blockDim.x) {
        const int64_t o = (((int64_t)blockIdx.y * ntile + tile) * nblk + b) * DT + k;
        r += partial[2 * o];
        im += partial[2 * o + 1];
    }
    r = lane_sum<64>(r);
    im = lane_sum<64>(im);
    __shared__ double s[2][4];
    if ((threadIdx.x & 63) == 0) { s[0][threadIdx.x >> 6] = r; s[1][threadIdx.x >> 6] = im; }
    __syncthreads();
    if (threadIdx.x == 0) {
        r = 0; im = 0;
        for (int q = 0; q < (int)(blockDim.x >> 6); q++) { r += s[0][q]; im += s[1][q]; }
        const double c = sc != nullptr ? sc[i] : 1.0;
        if (blockIdx.y == 0) {
            h[2 * i] = c * r;
            h[2 * i + 1] = c * im;
        } else {
            const int l = nv - 1;
            const double f = i == l ? 0.0 : c * sc[l];   // every scale is its vector's own norm's: the diagonal does not deviate
            E[2 * ((int64_t)i * ld + l)] = f * r;
            E[2 * ((int64_t)i * ld + l) + 1] = f * im;
            E[2 * ((int64_t)l * ld + i)] = f * r;
            E[2 * ((int64_t)l * ld + i) + 1] = -f * im;
        }
    }
}

// The spaces kept from earlier refinement cycles of a solve (see gmres_cycle): cycle c holds the
// basis vectors start[c] .. start[c + 1] - 1, of which K M maps all but the last into the range
// C_c = V Q_c; qp_i holds the coefficients of the one direction of their span outside C_c.
static constexpr int KEEP_MAX = 32;
struct kept_dev {
    int32_t t0;                    // first basis vector of the running cycle
    int32_t ncyc;                  // kept cycles
    int32_t start[KEEP_MAX + 1];
};
// h (LDS, coefficients against all basis vectors) less the components along the kept cycles' outside
// directions: what is left projects on the ranges only.  One wavefront per cycle.
__device__ __forceinline__ void project_kept(double *h, const kept_dev *kept, const double *qp) {
    const int nc = kept->ncyc;
    for (int c = threadIdx.x >> 6; c < nc; c += RB / 64) {
        const int a = kept->start[c], b = kept->start[c + 1];
        double sr = 0.0, si = 0.0;
        for (int i = a + (threadIdx.x & 63); i < b; i += 64) {
            sr += qp[2 * i] * h[2 * i] + qp[2 * i + 1] * h[2 * i + 1];
            si += qp[2 * i] * h[2 * i + 1] - qp[2 * i + 1] * h[2 * i];
        }
        sr = lane_sum<64>(sr);
        si = lane_sum<64>(si);
        for (int i = a + (threadIdx.x & 63); i < b; i += 64) {
            h[2 * i] -= qp[2 * i] * sr - qp[2 * i + 1] * si;
            h[2 * i + 1] -= qp[2 * i] * si + qp[2 * i + 1] * sr;
        }
    }
    __syncthreads();
}

// c = h~ - E h~ with h~ the coefficients h projected (project_kept): the coefficients that take the basis'
// part out of a vector although the basis is orthonormal only to complex64's rounding.  V^H (w - V c)
// is E^2 h~ where plain Gram-Schmidt leaves E h~, so the deviations E of later vectors do not
// grow with the earlier ones, and the second pass over the basis that kept them down is not needed: this
// reads nv^2 numbers.  (A second pass only after 99 % of the squared norm had cancelled, as
// before, let E grow until kept spaces were useless: mixed media, 3,072 tets, degree 1: 706 steps to 1e-9
// with it, 232 with a pass in every step.)  16 rows per block.
__global__ void __launch_bounds__(RB) k_gram_correct(int nv, const double *__restrict__ h, const double *__restrict__ E,
                                                     int lde, const kept_dev *__restrict__ kept,
                                                     const double *__restrict__ qp, double *__restrict__ c) {
    __shared__ double hs[2 * 512];
    for (int i = threadIdx.x; i < 2 * nv; i += RB) hs[i] = h[i];
    __syncthreads();
    project_kept(hs, kept, qp);
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int i = blockIdx.x * 16 + (threadIdx.x >> 6) * 4 + q;
        double r = 0.0, im = 0.0;
        if (i < nv)
            for (int j = lane; j < nv; j += 64) {
                const cx<double> e = ld(E, (int64_t)i * lde + j), x(hs[2 * j], hs[2 * j + 1]);
                r += e.re * x.re - e.im * x.im;
                im += e.re * x.im + e.im * x.re;
            }
        r = lane_sum<64>(r);
        im = lane_sum<64>(im);
        if (lane == 0 && i < nv) {
            c[2 * i] = hs[2 * i] - r;
            c[2 * i + 1] = hs[2 * i + 1] - im;
        }
    }
}

// w -= sum_i h_i (sc_i V_i) ; partial norm^2 of the result per block.  Two complex values per
// lane; the vectors are read four at a time so that four loads are in flight.  S = 4 (maxpy_split:
// problems too small to fill the GPU): four lanes share an element, each takes a quarter of the
// vectors, so the chain of loads is a quarter as long and four times the lanes are busy (7.5 us
// with S = 1 at 19,664 DOFs and 50 vectors).  With kept spaces (kept not NULL) h is first projected
// (project_kept); block 0 leaves the coefficients used in hout (NULL: nowhere).
template <typename R, int S>
__global__ void __launch_bounds__(RB) k_maxpy_norm(int64_t n, int nv, const R *__restrict__ V, int64_t ldv,
                                                   const double *__restrict__ h, const double *__restrict__ sc,
                                                   R *__restrict__ w, double *__restrict__ partial,
                                                   const kept_dev *__restrict__ kept, const double *__restrict__ qp,
                                                   double *__restrict__ hout) {
    __shared__ double hs[2 * 512];
    for (int i = threadIdx.x; i < 2 * nv; i += RB) hs[i] = h[i];
    __syncthreads();
    if (kept != nullptr) project_kept(hs, kept, qp);
    if (hout != nullptr && blockIdx.x == 0)
        for (int i = threadIdx.x; i < 2 * nv; i += RB) hout[i] = hs[i];
    if (sc != nullptr) {
        __syncthreads();
        for (int i = threadIdx.x; i < 2 * nv; i += RB) hs[i] *= sc[i >> 1];
        __syncthreads();
    }
    double nrm = 0;
    const int64_t n2 = n >> 1;
    constexpr int EB = RB / S;                       // elements of a block's pass
    const int part = threadIdx.x / EB, el = threadIdx.x % EB;
    const int per = (nv + S - 1) / S, i0 = part * per, i1 = min(nv, i0 + per);
    __shared__ double red[S > 1 ? (S - 1) * EB * 4 : 1];
    // every lane makes the same number of passes (the barriers below need them all)
    const int64_t passes = (n2 + (int64_t)gridDim.x * EB - 1) / ((int64_t)gridDim.x * EB);
    for (int64_t ps = 0; ps < passes; ps++) {
        const int64_t e = (ps * gridDim.x + blockIdx.x) * EB + el;
        const bool in = e < n2;
        double ar = 0, ai = 0, br = 0, bi = 0;       // sum of this lane's vectors
        if (in) {
            auto add = [&](int i, const cx2<R> &v) {
                const double hr = hs[2 * i], hi = hs[2 * i + 1];
                ar += hr * v.ar - hi * v.ai;
                ai += hr * v.ai + hi * v.ar;
                br += hr * v.br - hi * v.bi;
                bi += hr * v.bi + hi * v.br;
            };
            int i = i0;
            for (; i + 4 <= i1; i += 4) {
                cx2<R> v[4];
#pragma unroll
                for (int q = 0; q < 4; q++) v[q] = ld2(V + (int64_t)(i + q) * ldv * 2, e);
#pragma unroll
                for (int q = 0; q < 4; q++) add(i + q, v[q]);
            }
            for (; i < i1; i++) add(i, ld2(V + (int64_t)i * ldv * 2, e));
        }
        if constexpr (S > 1) {
            if (part > 0) {
                double *r = red + ((part - 1) * 4) * EB + el;
                r[0] = ar; r[EB] = ai; r[2 * EB] = br; r[3 * EB] = bi;
            }
            __syncthreads();
            if (part == 0) {
#pragma unroll
                for (int q = 0; q < S - 1; q++) {
                    const double *r = red + (q * 4) * EB + el;
                    ar += r[0]; ai += r[EB]; br += r[2 * EB]; bi += r[3 * EB];
                }
            }
            __syncthreads();
        }
        if (in && part == 0) {
            const cx2<R> wv = ld2(w, e);
            const cx2<R> o{(R)(wv.ar - ar), (R)(wv.ai - ai), (R)(wv.br - br), (R)(wv.bi - bi)};
            st2(w, e, o);
            nrm += (double)o.ar * o.ar + (double)o.ai * o.ai + (double)o.br * o.br + (double)o.bi * o.bi;
        }
    }
    if ((n & 1) && blockIdx.x == 0 && threadIdx.x == 0) {
        const cx<R> wv = ld(w, n - 1);
        double wr = wv.re, wi = wv.im;
        for (int i = 0; i < nv; i++) {
            const cx<R> v = ld(V + (int64_t)i * ldv * 2, n - 1);
            wr -= hs[2 * i] * v.re - hs[2 * i + 1] * v.im;
            wi -= hs[2 * i] * v.im + hs[2 * i + 1] * v.re;
        }
        st(w, n - 1, cx<R>((R)wr, (R)wi));
        nrm += (double)(R)wr * (double)(R)wr + (double)(R)wi * (double)(R)wi;
    }
    nrm = lane_sum<64>(nrm);
    __shared__ double s[RB / 64];
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = nrm;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0;
        for (int q = 0; q < RB / 64; q++) t += s[q];
        partial[blockIdx.x] = t;
    }
}

// Lanes per element of k_maxpy_norm: four on problems of a few ten thousand DOFs, where one lane
// per element leaves most of the GPU idle (19,664 DOFs: 7.5 us with one, 5.9 with four; 245,000 DOFs:
// 28.8 and 31.5).
static int maxpy_split(int64_t n) { return n < 65536 ? 4 : 1; }
template <typename R>
static void launch_maxpy(hipStream_t st, int nb, int64_t n, int nv, const R *V, const double *h, const double *sc, R *w,
                         double *partial, const kept_dev *kept = nullptr, const double *qp = nullptr,
                         double *hout = nullptr) {
    if (maxpy_split(n) == 4)
        k_maxpy_norm<R, 4><<<nb, RB, 0, st>>>(n, nv, V, n, h, sc, w, partial, kept, qp, hout);
    else
        k_maxpy_norm<R, 1><<<nb, RB, 0, st>>>(n, nv, V, n, h, sc, w, partial, kept, qp, hout);
}

// x += sum_i y_i V_i   (y on device, complex)
template <typename R>
__global__ void __launch_bounds__(RB) k_mcomb(int64_t n, int nv, const R *__restrict__ V, int64_t ldv,
                                              const double *__restrict__ y, R *__restrict__ x, int overwrite) {
    __shared__ double ys[2 * 512];
    for (int i = threadIdx.x; i < 2 * nv; i += RB) ys[i] = y[i];
    __syncthreads();
    for (int64_t e = blockIdx.x * (int64_t)RB + threadIdx.x; e < n; e += (int64_t)gridDim.x * RB) {
        double xr = 0, xi = 0;
        if (!overwrite) {
            const cx<R> xv = ld(x, e);
            xr = xv.re; xi = xv.im;
        }
        for (int i = 0; i < nv; i++) {
            const cx<R> v = ld(V + (int64_t)i * ldv * 2, e);
            xr += ys[2 * i] * v.re - ys[2 * i + 1] * v.im;
            xi += ys[2 * i] * v.im + ys[2 * i + 1] * v.re;
        }
        st(x, e, cx<R>((R)xr, (R)xi));
    }
}

template <typename R>
__global__ void __launch_bounds__(RB) k_norm2(int64_t n, const R *__restrict__ x, double *__restrict__ partial) {
    double s = 0;
    for (int64_t e = blockIdx.x * (int64_t)RB + threadIdx.x; e < n; e += (int64_t)gridDim.x * RB) {
        const cx<R> v = ld(x, e);
        s += (double)v.re * v.re + (double)v.im * v.im;
    }
    s = lane_sum<64>(s);
    __shared__ double sh[RB / 64];
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0;
        for (int q = 0; q < RB / 64; q++) t += sh[q];
        partial[blockIdx.x] = t;
    }
}

// y = alpha * x (alpha real, on device as 1/sqrt(norm2 sum) when from_norm)
template <typename R>
__global__ void __launch_bounds__(RB) k_scale_by_norm(int64_t n, const double *__restrict__ partial, int nblk,
                                                      const R *x, R *y, double *__restrict__ out_norm) {   // x may be y
    __shared__ double inv;
    if (threadIdx.x < 64) {
        double s = 0;
        for (int b = threadIdx.x; b < nblk; b += 64) s += partial[b];
        s = lane_sum<64>(s);
        if (threadIdx.x == 0) {
            const double nv = sqrt(s);
            inv = nv > 0 ? 1.0 / nv : 0.0;
            if (out_norm && blockIdx.x == 0) *out_norm = nv;
        }
    }
    __syncthreads();
    for (int64_t e = blockIdx.x * (int64_t)RB + threadIdx.x; e < n; e += (int64_t)gridDim.x * RB) {
        const cx<R> v = ld(x, e);
        st(y, e, cx<R>((R)(v.re * inv), (R)(v.im * inv)));
    }
}

// 2x2 mode-block Jacobi: z = blk^{-1} r on DOF pairs (e, e + n_ent).
// inv holds per entity the 4 complex entries of the inverse block (row-major).
__global__ void __launch_bounds__(RB) k_bj_apply(int64_t n_ent, const double *__restrict__ inv, const double *__restrict__ r,
                                                 double *__restrict__ z) {
    const int64_t e = blockIdx.x * (int64_t)RB + threadIdx.x;
    if (e >= n_ent) return;
    const cx<double> a = ld(inv, 4 * e), b = ld(inv, 4 * e + 1), c = ld(inv, 4 * e + 2), d = ld(inv, 4 * e + 3);
    const cx<double> r0 = ld(r, e), r1 = ld(r, e + n_ent);
    st(z, e, cadd(cmul(a, r0), cmul(b, r1)));
    st(z, e + n_ent, cadd(cmul(c, r0), cmul(d, r1)));
}

__device__ __forceinline__ int32_t find_col(const int32_t *cols, int32_t p0, int32_t p1, int32_t c) {
    int32_t lo = p0, hi = p1 - 1;
    while (lo < hi) {
        const int32_t mid = (lo + hi) >> 1;
        if (cols[mid] < c) lo = mid + 1; else hi = mid;
    }
    return (lo < p1 && cols[lo] == c) ? lo : -1;
}

// Build the inverse 2x2 blocks from K (complex128); PEC DOFs get identity.
// ---------------------------------------------------------------- gradient correction
static constexpr int G_ROW_MAX = 8;   // entries per row of G (edge rows 3, face rows 6)

// dS[p] += g_ip * sum_j K_ij g_jp over the unmasked entries of row i, for the
// P2 nodes p of row i of G: diag(G^T K G) with one atomic per entry of G.  GD lanes
// per row: bound by the chain of loads (an entry's column, that row of G, its nodes), which
// one lane per row went through 74 times: 600 us at 38,400 tets, 243 with 16; at 3,072 tets 196 and 36.
static constexpr int GD = 16;
__global__ void __launch_bounds__(RB) k_gdiag(int64_t n, const int32_t *__restrict__ rowptr,
                                              const int32_t *__restrict__ cols, const double *__restrict__ K,
                                              const uint8_t *__restrict__ mask, const int32_t *__restrict__ grp,
                                              const int32_t *__restrict__ gcol, const double *__restrict__ gval,
                                              double *__restrict__ dS) {
    const int64_t i = (blockIdx.x * (int64_t)RB + threadIdx.x) / GD;
    const int lane = threadIdx.x % GD;
    if (i >= n || (mask && !mask[i])) return;
    const int32_t q0 = grp[i], ni = min(grp[i + 1] - q0, G_ROW_MAX);
    if (ni == 0) return;
    int32_t pk[G_ROW_MAX];
    double ar[G_ROW_MAX], ai[G_ROW_MAX];
#pragma unroll
    for (int k = 0; k < G_ROW_MAX; k++) { pk[k] = k < ni ? gcol[q0 + k] : -1; ar[k] = 0.0; ai[k] = 0.0; }
    for (int32_t e = rowptr[i] + lane; e < rowptr[i + 1]; e += GD) {
        const int32_t j = cols[e];
        if (mask && !mask[j]) continue;
        const int32_t r0 = grp[j], r1 = grp[j + 1];
        if (r0 == r1) continue;
        const double kr = K[2 * e], ki = K[2 * e + 1];
        for (int32_t q = r0; q < r1; q++) {
            const int32_t pj = gcol[q];
            const double gj = gval[q];
#pragma unroll
            for (int k = 0; k < G_ROW_MAX; k++)
                if (pk[k] == pj) { ar[k] += kr * gj; ai[k] += ki * gj; }
        }
    }
#pragma unroll
    for (int k = 0; k < G_ROW_MAX; k++) {
        if (k >= ni) break;
        ar[k] = lane_sum<GD>(ar[k]);
        ai[k] = lane_sum<GD>(ai[k]);
        if (lane == 0) {
            const double gi = gval[q0 + k];
            atomicAdd(&dS[2 * pk[k]], gi * ar[k]);
            atomicAdd(&dS[2 * pk[k] + 1], gi * ai[k]);
        }
    }
}

__global__ void __launch_bounds__(RB) k_dsinv(int64_t np2, const double *__restrict__ dS, double *__restrict__ inv64,
                                              float *__restrict__ inv32) {
    const int64_t p = blockIdx.x * (int64_t)RB + threadIdx.x;
    if (p >= np2) return;
    const double a = dS[2 * p], b = dS[2 * p + 1], d = a * a + b * b;
    const double r = d > 0.0 ? a / d : 0.0, im = d > 0.0 ? -b / d : 0.0;
    inv64[2 * p] = r;
    inv64[2 * p + 1] = im;
    if (inv32) { inv32[2 * p] = (float)r; inv32[2 * p + 1] = (float)im; }
}

// t[p] = dsinv[p] * sum over row p of G^T of g * r, 8 lanes per row (caller's layout)
static constexpr int GT_STD = 8;
__global__ void __launch_bounds__(256) k_gt_apply(int64_t np2, const int32_t *__restrict__ rp, const int32_t *__restrict__ ci,
                                                  const double *__restrict__ gv, const double *__restrict__ dsinv,
                                                  const double *__restrict__ r, double *__restrict__ t) {
    const int64_t p = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) / GT_STD;
    const int lane = threadIdx.x % GT_STD;
    if (p >= np2) return;
    double ar = 0.0, ai = 0.0;
    for (int32_t e = rp[p] + lane; e < rp[p + 1]; e += GT_STD) {
        const cx<double> v = ld(r, ci[e]);
        ar += gv[e] * v.re;
        ai += gv[e] * v.im;
    }
    ar = lane_sum<GT_STD>(ar);
    ai = lane_sum<GT_STD>(ai);
    if (lane == 0) {
        const cx<double> d = ld(dsinv, p);
        st(t, p, cx<double>(d.re * ar - d.im * ai, d.re * ai + d.im * ar));
    }
}

static void launch_gt(hipStream_t st, int64_t np2, const int32_t *rp, const int32_t *ci, const double *gv,
                      const double *dsinv, const double *r, double *t) {
    k_gt_apply<<<(unsigned)((np2 * GT_STD + 255) / 256), 256, 0, st>>>(np2, rp, ci, gv, dsinv, r, t);
}

// z = BJ(r) + G t, both modes of entity e per thread (caller's layout)
__global__ void __launch_bounds__(RB) k_bj_grad_apply(int64_t n_ent, const double *__restrict__ inv,
                                                      const double *__restrict__ r, const int32_t *__restrict__ grp,
                                                      const int32_t *__restrict__ gcol, const double *__restrict__ gv,
                                                      const double *__restrict__ t, double *__restrict__ z) {
    const int64_t e = blockIdx.x * (int64_t)RB + threadIdx.x;
    if (e >= n_ent) return;
    const cx<double> a = ld(inv, 4 * e), b = ld(inv, 4 * e + 1), c = ld(inv, 4 * e + 2), d = ld(inv, 4 * e + 3);
    const cx<double> r0 = ld(r, e), r1 = ld(r, e + n_ent);
    cx<double> z0 = cadd(cmul(a, r0), cmul(b, r1));
    cx<double> z1 = cadd(cmul(c, r0), cmul(d, r1));
    for (int32_t q = grp[e]; q < grp[e + 1]; q++) {
        const cx<double> tv = ld(t, gcol[q]);
        z0 = cx<double>(z0.re + gv[q] * tv.re, z0.im + gv[q] * tv.im);
    }
    for (int32_t q = grp[e + n_ent]; q < grp[e + n_ent + 1]; q++) {
        const cx<double> tv = ld(t, gcol[q]);
        z1 = cx<double>(z1.re + gv[q] * tv.re, z1.im + gv[q] * tv.im);
    }
    st(z, e, z0);
    st(z, e + n_ent, z1);
}

__global__ void __launch_bounds__(RB) k_bj_setup(int64_t n_ent, const int32_t *__restrict__ rowptr,
                                                 const int32_t *__restrict__ cols, const double *__restrict__ vals,
                                                 const uint8_t *__restrict__ mask, double *__restrict__ inv64,
                                                 float *__restrict__ inv32) {
    const int64_t e = blockIdx.x * (int64_t)RB + threadIdx.x;
    if (e >= n_ent) return;
    const int64_t r0 = e, r1 = e + n_ent;
    const bool m0 = mask == nullptr || mask[r0], m1 = mask == nullptr || mask[r1];
    auto get = [&](int64_t r, int64_t c) -> cx<double> {
        const int32_t p = find_col(cols, rowptr[r], rowptr[r + 1], (int32_t)c);
        return p < 0 ? cx<double>(0, 0) : ld(vals, p);
    };
    cx<double> a = m0 ? get(r0, r0) : cx<double>(1, 0);
    cx<double> d = m1 ? get(r1, r1) : cx<double>(1, 0);
    cx<double> b = (m0 && m1) ? get(r0, r1) : cx<double>(0, 0);
    cx<double> c = (m0 && m1) ? get(r1, r0) : cx<double>(0, 0);
    const cx<double> ad = cmul(a, d), bc = cmul(b, c);
    cx<double> det(ad.re - bc.re, ad.im - bc.im);
    const double dn = det.re * det.re + det.im * det.im;
    cx<double> idet(det.re / dn, -det.im / dn);
    if (!(dn > 0) || !std::isfinite(dn)) {  // singular block: fall back to the diagonal
        idet = cx<double>(1, 0);
        b = c = cx<double>(0, 0);
        const double na = a.re * a.re + a.im * a.im, nd = d.re * d.re + d.im * d.im;
        a = na > 0 ? cx<double>(a.re / na, -a.im / na) : cx<double>(1, 0);
        d = nd > 0 ? cx<double>(d.re / nd, -d.im / nd) : cx<double>(1, 0);
        const cx<double> tmp = a;
        a = d;
        d = tmp;  // undone by the swap below
    }
    const cx<double> ia = cmul(d, idet), ib = cmul(cx<double>(-b.re, -b.im), idet);
    const cx<double> ic = cmul(cx<double>(-c.re, -c.im), idet), id = cmul(a, idet);
    st(inv64, 4 * e, ia); st(inv64, 4 * e + 1, ib); st(inv64, 4 * e + 2, ic); st(inv64, 4 * e + 3, id);
    if (inv32) {
        st(inv32, 4 * e, cx<float>((float)ia.re, (float)ia.im));
        st(inv32, 4 * e + 1, cx<float>((float)ib.re, (float)ib.im));
        st(inv32, 4 * e + 2, cx<float>((float)ic.re, (float)ic.im));
        st(inv32, 4 * e + 3, cx<float>((float)id.re, (float)id.im));
    }
}

// u += z (same element type)
template <typename R>
__global__ void __launch_bounds__(RB) k_add(int64_t n, const R *__restrict__ z, R *__restrict__ u) {
    for (int64_t e = blockIdx.x * (int64_t)RB + threadIdx.x; e < 2 * n; e += (int64_t)gridDim.x * RB) u[e] += z[e];
}

// K = E - s B (complex128 values on the shared pattern)
__global__ void __launch_bounds__(RB) k_affine(int64_t nnz, const double *__restrict__ E, const double *__restrict__ B,
                                               double s, double *__restrict__ K) {
    for (int64_t e = blockIdx.x * (int64_t)RB + threadIdx.x; e < 2 * nnz; e += (int64_t)gridDim.x * RB) K[e] = E[e] - s * B[e];
}
// K[pos[i]] += g * v[i]   (complex; positions may repeat -> atomics)
__global__ void __launch_bounds__(RB) k_scatter_add(int64_t m, const int32_t *__restrict__ pos, const double *__restrict__ v,
                                                    double gre, double gim, double *__restrict__ K) {
    const int64_t i = blockIdx.x * (int64_t)RB + threadIdx.x;
    if (i >= m) return;
    const int32_t p = pos[i];
    if (p < 0) return;
    const double vr = v[2 * i], vi = v[2 * i + 1];
    atomicAdd(&K[2 * (int64_t)p], gre * vr - gim * vi);
    atomicAdd(&K[2 * (int64_t)p + 1], gre * vi + gim * vr);
}
// pos[i] = CSR position of (rows[i], cols[i]) or -1
__global__ void __launch_bounds__(RB) k_csr_find(int64_t m, const int32_t *__restrict__ rowptr,
                                                 const int32_t *__restrict__ cols, const int32_t *__restrict__ qr,
                                                 const int32_t *__restrict__ qc, int32_t *__restrict__ pos) {
    const int64_t i = blockIdx.x * (int64_t)RB + threadIdx.x;
    if (i >= m) return;
    const int32_t r = qr[i];
    pos[i] = find_col(cols, rowptr[r], rowptr[r + 1], qc[i]);
}

// ---------------------------------------------------------------- packed solver layout
// The vectors of the solver's own steps hold the two modes of an entity side by side
// (V[2 e + m] for DOF m * ne + e), and its operators are stored for that:
//  * K as 2x2 blocks over the entity pattern in two planes, the real parts kre[4 p ..] and
//    the imaginary parts kim[4 p ..] of entry p (p = rowptr[e] / 2 + k), the columns acol[p]
//    once per block.  A row whose imaginary parts all vanish (lossless media: every row but
//    those of ports and absorbing boundaries) is flagged and its kim plane is never read, so
//    a complex64 product moves 20 instead of 36 bytes per block.  PEC columns are zeroed.
//  * G in slices of 64 entities, transposed (slot k of the 64 lanes together): one column and
//    both modes' values per slot; G^T in rows of (entity, both modes' values).
static constexpr uint8_t ROW0 = 1, ROW1 = 2, ROW_CPLX = 4;   // flags: row (0, e) free, (1, e) free, kim used

// acol[p] of every block (16 lanes per entity)
__global__ void __launch_bounds__(256) k_pack_cols(int64_t ne, const int32_t *__restrict__ rowptr,
                                                   const int32_t *__restrict__ cols, int32_t *__restrict__ acol) {
    const int64_t e = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) / SUB;
    if (e >= ne) return;
    const int32_t r0 = rowptr[e], deg = (rowptr[e + 1] - r0) >> 1;
    for (int32_t k = threadIdx.x % SUB; k < deg; k += SUB) acol[(r0 >> 1) + k] = cols[r0 + k];
}

// The planes and flags of K (complex128 CSR values) in element type R.
template <typename R>
__global__ void __launch_bounds__(256) k_pack_matrix(int64_t ne, int64_t half, const int32_t *__restrict__ rowptr,
                                                     const int32_t *__restrict__ acol, const double *__restrict__ vals,
                                                     const uint8_t *__restrict__ mask, R *__restrict__ kre,
                                                     R *__restrict__ kim, uint8_t *__restrict__ flag) {
    const int64_t e = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) / SUB;
    const int lane = threadIdx.x % SUB;
    if (e >= ne) return;
    const bool m0 = mask == nullptr || mask[e], m1 = mask == nullptr || mask[ne + e];
    const int32_t r0 = rowptr[e], deg = (rowptr[e + 1] - r0) >> 1, a0 = r0 >> 1;
    int any = 0;
    for (int pass = 0; pass < 2; pass++) {
        for (int32_t k = lane; k < deg; k += SUB) {
            const int32_t c = acol[a0 + k];
            const bool c0 = mask == nullptr || mask[c], c1 = mask == nullptr || mask[ne + c];
            const int64_t p = (int64_t)r0 + k;
            cx<double> v00 = ld(vals, p), v01 = ld(vals, p + deg), v10 = ld(vals, half + p), v11 = ld(vals, half + p + deg);
            if (!(m0 && c0)) v00 = cx<double>();
            if (!(m0 && c1)) v01 = cx<double>();
            if (!(m1 && c0)) v10 = cx<double>();
            if (!(m1 && c1)) v11 = cx<double>();
            const cx2<R> im{(R)v00.im, (R)v01.im, (R)v10.im, (R)v11.im};
            if (pass == 0) {
                st2(kre, a0 + k, cx2<R>{(R)v00.re, (R)v01.re, (R)v10.re, (R)v11.re});
                // != is true of NaN too: such a row keeps its imaginary plane
                any |= (im.ar != R(0)) | (im.ai != R(0)) | (im.br != R(0)) | (im.bi != R(0));
            } else {
                st2(kim, a0 + k, im);
            }
        }
        if (pass == 0) {
#pragma unroll
            for (int off = SUB / 2; off > 0; off >>= 1) any |= __shfl_xor(any, off, SUB);
            if (!any) break;
        }
    }
    if (lane == 0) flag[e] = (uint8_t)((m0 ? ROW0 : 0) | (m1 ? ROW1 : 0) | (any ? ROW_CPLX : 0));
}

// Workgroup b of a grid as work item: XCD b % 8 takes runs of XCD_RUN consecutive items, whose rows
// gather mostly the same parts of x, instead of every eighth (complex64 product on air: 40.1 -> 36.2 us
// at 60 x 30 x 12 hexes, 114.6 -> 113.4 at 80 x 40 x 16; runs of 8 and 128 the same within 2 %, runs of
// 512 slower again, an eighth of the grid per XCD 30 % slower).
static constexpr unsigned XCD_RUN = 32;
__device__ __forceinline__ unsigned xcd_run(unsigned b, unsigned n) {
    const unsigned full = n / (8 * XCD_RUN) * (8 * XCD_RUN);
    if (b >= full) return b;
    const unsigned i = b / 8;
    return i / XCD_RUN * (8 * XCD_RUN) + (b % 8) * XCD_RUN + i % XCD_RUN;
}

// The flags of rows whose values stay in the caller's CSR.
__global__ void __launch_bounds__(256) k_row_flags(int64_t ne, const uint8_t *__restrict__ mask, uint8_t *__restrict__ flag) {
    const int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (e < ne) flag[e] = (uint8_t)((mask == nullptr || mask[e] ? ROW0 : 0) | (mask == nullptr || mask[ne + e] ? ROW1 : 0) | ROW_CPLX);
}

// What follows a product v = K x in the same launch:
//   SP_Y: y = v;   SP_RESID: y = b - v;
//   SP_POLY: p = q - c_i v, y = (i == 0 ? c_0 q : y) + c_{i+1} p (apply_prec_poly; q scaled by *qs)
enum { SP_Y, SP_RESID, SP_POLY };
template <typename R>
struct sp_args {
    const R *b;          // SP_RESID: b; SP_POLY: q (may be p)
    R *y;
    R *p;                // SP_POLY
    const double *c;     // SP_POLY: the polynomial's coefficients
    int i;               // SP_POLY
    const double *qs;    // SP_POLY: scale of q, or NULL
};

// v = K x on the packed matrix: L lanes per entity, every lane loading the columns and blocks of
// up to U entries before it gathers x for them, so that a row of average length (21 blocks) costs
// two round trips to memory instead of two per L entries.  Bound by the bytes of kre, acol and (in
// rows with losses) kim; small problems by the latency of that chain.  STD: x, y, b in the caller's
// layout (mode * ne + e) instead of interleaved (SP_Y and SP_RESID only).
// LOC: a workgroup first gathers x for the distinct columns of its LOC_ROWS rows into LDS (loc_tab: the columns, and
// in acol's place 16-bit places among them).  The gathers of the other form take a line of the L2 each, 21 of them
// per row and no two lanes of a row the same; 64 rows share theirs 3.3 times, and an index is 2 bytes.  Products of
// the posts box, rates by the bytes of the format: complex64 on air at 1,947,698 DOFs 114 -> 90 us (4.7 TB/s; the HBM
// counters show 0.53 GB, 6.1), with losses at 831,972 70 -> 63 (5.3), complex128 on air at 883,652 91 -> 71 (5.1).  (8 lanes per row, which is 512 of them: 92, 61, 79; 32, 96 or 128
// rows: 96, 66, 85; 113, 65, 86; 93, 65, 74; 2, 3 or 6 blocks in flight per lane: 95, 69, 73; 96, 68, 73; 93, 63, 89.)
static constexpr int LOC_ROWS = 64, LOC_L = 4, LOC_MAX = 1024, LOC_CAND = 8192;
static constexpr int LOC_LANES = LOC_ROWS * LOC_L;
// CSR: the caller's columns and complex128 values in place of acol and kre (kim unused), for solvers without a packed
// copy; `half` as in k_spmv_blk.
struct loc_tab {
    const int32_t *ptr, *col;
    const uint16_t *idx;
};
template <typename R, int L, int EP, bool STD, bool LOC, bool CSR = false>
__global__ void __launch_bounds__(LOC ? LOC_LANES : 256) k_spmv_pk(int64_t ne, const int32_t *__restrict__ rowptr,
                                                 const int32_t *__restrict__ acol, const R *__restrict__ kre,
                                                 const R *__restrict__ kim, const uint8_t *__restrict__ flag,
                                                 const R *__restrict__ x, sp_args<R> a, loc_tab loc, int64_t half) {
    static_assert(!CSR || (sizeof(R) == 8 && !STD && !LOC), "the caller's CSR serves complex128 steps");
    constexpr int U = L <= 4 ? 4 : L == 8 ? 3 : L == 16 ? 2 : 1;
    __shared__ __align__(16) R xs[LOC ? 4 * LOC_MAX : 4];
    const int64_t blk = xcd_run(blockIdx.x, gridDim.x);
    const int64_t e = (blk * blockDim.x + threadIdx.x) / L;
    const int lane = threadIdx.x % L;
    if constexpr (LOC) {
        const int32_t b = loc.ptr[blk], nu = loc.ptr[blk + 1] - b;
        for (int i = threadIdx.x; i < nu; i += LOC_LANES) {
            const int32_t c = loc.col[b + i];
            if constexpr (STD) {
                cx<R> u0 = ld(x, c), u1 = ld(x, ne + c);
                if constexpr (sizeof(R) == 8) {
                    const uint8_t cf = flag[c];
                    if (!(cf & ROW0)) u0 = cx<R>();
                    if (!(cf & ROW1)) u1 = cx<R>();
                }
                st2(xs, i, cx2<R>{u0.re, u0.im, u1.re, u1.im});
            } else {
                st2(xs, i, ld2(x, c));
            }
        }
        __syncthreads();
    }
    if (e >= ne) return;
    const uint8_t fl = flag[e];
    const int32_t p0 = rowptr[e] >> 1, p1 = rowptr[e + 1] >> 1;
    // real or imaginary parts of block q
    auto block = [&](const R *plane, int32_t q, int im) {
        if constexpr (CSR) {
            const int64_t i = 2 * ((int64_t)p0 + q) + im, d = 2 * (p1 - p0);
            return cx2<R>{kre[i], kre[i + d], kre[i + 2 * half], kre[i + 2 * half + d]};
        } else {
            return ld2(plane, q);
        }
    };
    cx2<R> own{}, qv{}, yv{};
    // the epilogue's operands, asked for before the row
    if (lane == 0) {
        auto get = [&](const R *v) {
            if constexpr (STD) {
                const cx<R> u0 = ld(v, e), u1 = ld(v, ne + e);
                return cx2<R>{u0.re, u0.im, u1.re, u1.im};
            } else {
                return ld2(v, e);
            }
        };
        if ((fl & (ROW0 | ROW1)) != (ROW0 | ROW1)) own = get(x);
        if constexpr (EP != SP_Y) qv = get(a.b);
        if constexpr (EP == SP_POLY)
            if (a.i > 0) yv = get(a.y);
    }
    // fewer than 16 lanes make longer chains: complex64 sums in FP64 there.  Errors against 64 bits: with 16 lanes 7.3e-8 on
    // air and 7.4e-8 with losses, with 4 or 8 and sums in FP32 7.2e-8 and 7.7e-8, so 5.9e-8 and 6.5e-8, in the same time.
    // The Krylov steps, whose lanes are tuned, keep sums in FP32 (250,000 DOFs: 260 us a step, 266 with FP64): what they
    // round goes into the FP64 residual that the refinement forms anew.
    using S = std::conditional_t<(L < 16) && STD, double, R>;
    S s0r = 0, s0i = 0, s1r = 0, s1i = 0;
    if (fl & (ROW0 | ROW1)) {
        for (int32_t p = p0 + lane; p < p1; p += L * U) {
            int32_t c[U];
            cx2<R> k[U], xv[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int32_t q = p + u * L < p1 ? p + u * L : p;   // past the row's end: its own entry again, not used
                c[u] = LOC ? loc.idx[q] : acol[CSR ? p0 + q : q];
                k[u] = block(kre, q, 0);
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                if constexpr (CSR) {
                    const uint8_t cf = flag[c[u]];   // the caller's values hold the PEC columns too
                    xv[u] = ld2(x, c[u]);
                    if (!(cf & ROW0)) xv[u].ar = xv[u].ai = 0;
                    if (!(cf & ROW1)) xv[u].br = xv[u].bi = 0;
                } else if constexpr (LOC) {
                    xv[u] = ld2(xs, c[u]);
                } else if constexpr (STD) {
                    cx<R> u0 = ld(x, c[u]), u1 = ld(x, ne + c[u]);
                    if constexpr (sizeof(R) == 8) {
                        // a caller's x may hold anything on PEC DOFs (their columns are zero, but 0 * inf is not)
                        const uint8_t cf = flag[c[u]];
                        if (!(cf & ROW0)) u0 = cx<R>();
                        if (!(cf & ROW1)) u1 = cx<R>();
                    }
                    xv[u] = cx2<R>{u0.re, u0.im, u1.re, u1.im};
                } else {
                    xv[u] = ld2(x, c[u]);
                }
            }
            // an entry's products are summed before they join the row's sums, as in the complex product
            cx2<R> v[U];
#pragma unroll
            for (int u = 0; u < U; u++)
                v[u] = cx2<R>{k[u].ar * xv[u].ar + k[u].ai * xv[u].br, k[u].ar * xv[u].ai + k[u].ai * xv[u].bi,
                              k[u].br * xv[u].ar + k[u].bi * xv[u].br, k[u].br * xv[u].ai + k[u].bi * xv[u].bi};
            if (fl & ROW_CPLX) {
#pragma unroll
                for (int u = 0; u < U; u++) k[u] = block(kim, p + u * L < p1 ? p + u * L : p, 1);
#pragma unroll
                for (int u = 0; u < U; u++) {
                    v[u].ar -= k[u].ar * xv[u].ai + k[u].ai * xv[u].bi;
                    v[u].ai += k[u].ar * xv[u].ar + k[u].ai * xv[u].br;
                    v[u].br -= k[u].br * xv[u].ai + k[u].bi * xv[u].bi;
                    v[u].bi += k[u].br * xv[u].ar + k[u].bi * xv[u].br;
                }
            }
            // pairwise, then to the row's sums
#pragma unroll
            for (int u = 0; u < U; u++)
                if (p + u * L >= p1) v[u] = cx2<R>{0, 0, 0, 0};
#pragma unroll
            for (int h = 1; h < U; h *= 2)
#pragma unroll
                for (int u = 0; u + h < U; u += 2 * h) {
                    v[u].ar += v[u + h].ar;
                    v[u].ai += v[u + h].ai;
                    v[u].br += v[u + h].br;
                    v[u].bi += v[u + h].bi;
                }
            s0r += v[0].ar;
            s0i += v[0].ai;
            s1r += v[0].br;
            s1i += v[0].bi;
        }
    }
    s0r = lane_sum<L>(s0r);
    s0i = lane_sum<L>(s0i);
    s1r = lane_sum<L>(s1r);
    s1i = lane_sum<L>(s1i);
    if (lane != 0) return;
    cx2<R> v{(fl & ROW0) ? (R)s0r : own.ar, (fl & ROW0) ? (R)s0i : own.ai, (fl & ROW1) ? (R)s1r : own.br, (fl & ROW1) ? (R)s1i : own.bi};
    if constexpr (EP == SP_RESID) v = cx2<R>{qv.ar - v.ar, qv.ai - v.ai, qv.br - v.br, qv.bi - v.bi};
    if constexpr (EP == SP_POLY) {
        const double *cc = a.c + 2 * a.i;
        const double cr = cc[0], ci = cc[1], nr = cc[2], ni = cc[3];
        const double s = a.qs != nullptr ? a.qs[0] : 1.0;
        const double q0r = s * qv.ar, q0i = s * qv.ai, q1r = s * qv.br, q1i = s * qv.bi;
        double y0r = yv.ar, y0i = yv.ai, y1r = yv.br, y1i = yv.bi;
        if (a.i == 0) {
            y0r = cr * q0r - ci * q0i; y0i = cr * q0i + ci * q0r;
            y1r = cr * q1r - ci * q1i; y1i = cr * q1i + ci * q1r;
        }
        const double p0r = q0r - (cr * v.ar - ci * v.ai), p0i = q0i - (cr * v.ai + ci * v.ar);
        const double p1r = q1r - (cr * v.br - ci * v.bi), p1i = q1i - (cr * v.bi + ci * v.br);
        st2(a.p, e, cx2<R>{(R)p0r, (R)p0i, (R)p1r, (R)p1i});
        st2(a.y, e, cx2<R>{(R)(y0r + nr * p0r - ni * p0i), (R)(y0i + nr * p0i + ni * p0r),
                           (R)(y1r + nr * p1r - ni * p1i), (R)(y1i + nr * p1i + ni * p1r)});
    } else if constexpr (STD) {
        st(a.y, e, cx<R>(v.ar, v.ai));
        st(a.y, ne + e, cx<R>(v.br, v.bi));
    } else {
        st2(a.y, e, v);
    }
}

template <typename R, int EP, bool STD>
static void launch_spmv_pk(hipStream_t st, int L, int64_t ne, const int32_t *rowptr, const int32_t *acol, const R *kre,
                           const R *kim, const uint8_t *flag, const R *x, const sp_args<R> &a, const loc_tab &loc,
                           int64_t half = 0) {
    if constexpr (sizeof(R) == 8 && !STD)
        if (half > 0) {
            k_spmv_pk<R, 16, EP, STD, false, true><<<(unsigned)((ne * 16 + 255) / 256), 256, 0, st>>>(ne, rowptr, acol, kre, kim, flag, x, a, loc, half);
            return;
        }
    if (loc.ptr != nullptr) {
        k_spmv_pk<R, LOC_L, EP, STD, true><<<(unsigned)((ne + LOC_ROWS - 1) / LOC_ROWS), LOC_LANES, 0, st>>>(ne, rowptr, acol, kre, kim, flag, x, a, loc, 0);
        return;
    }
    if (L != 4 && L != 8 && L != 32) L = 16;
    const unsigned grid = (unsigned)((ne * L + 255) / 256);
    if (L == 4) k_spmv_pk<R, 4, EP, STD, false><<<grid, 256, 0, st>>>(ne, rowptr, acol, kre, kim, flag, x, a, loc, 0);
    else if (L == 8) k_spmv_pk<R, 8, EP, STD, false><<<grid, 256, 0, st>>>(ne, rowptr, acol, kre, kim, flag, x, a, loc, 0);
    else if (L == 32) k_spmv_pk<R, 32, EP, STD, false><<<grid, 256, 0, st>>>(ne, rowptr, acol, kre, kim, flag, x, a, loc, 0);
    else k_spmv_pk<R, 16, EP, STD, false><<<grid, 256, 0, st>>>(ne, rowptr, acol, kre, kim, flag, x, a, loc, 0);
}

// The distinct columns of every LOC_ROWS rows, ascending, and every block's 16-bit place among them: counts first
// (idx NULL), then with their prefix the lists and places.  *over where a workgroup's rows hold more than LOC_CAND
// blocks or LOC_MAX distinct columns.
__global__ void __launch_bounds__(512) k_loc_columns(int64_t ne, const int32_t *__restrict__ rowptr,
                                                     const int32_t *__restrict__ acol, const int32_t *__restrict__ ptr,
                                                     int32_t *__restrict__ cnt, int32_t *__restrict__ col,
                                                     uint16_t *__restrict__ idx, int *__restrict__ over) {
    __shared__ int32_t key[LOC_CAND];
    __shared__ int32_t wsum[8];
    const int tid = threadIdx.x;
    const int64_t e0 = blockIdx.x * (int64_t)LOC_ROWS, e1 = min(e0 + LOC_ROWS, ne);
    const int32_t p0 = rowptr[e0] >> 1, n = (rowptr[e1] >> 1) - p0;
    if (n > LOC_CAND) {
        if (tid == 0) { *over = 1; if (cnt) cnt[blockIdx.x] = 0; }
        return;
    }
    int size = 512;
    while (size < n) size <<= 1;
    for (int i = tid; i < size; i += 512) key[i] = i < n ? acol[p0 + i] : INT32_MAX;
    __syncthreads();
    for (int len = 2; len <= size; len <<= 1)
        for (int stride = len >> 1; stride > 0; stride >>= 1) {
            for (int i = tid; i < size; i += 512) {
                const int j = i ^ stride;
                if (j > i) {
                    const bool asc = (i & len) == 0;
                    const int32_t a = key[i], b = key[j];
                    if ((a > b) == asc) { key[i] = b; key[j] = a; }
                }
            }
            __syncthreads();
        }
    // each lane's stretch of the sorted keys: how many are first of their value
    const int per = size / 512, s0 = tid * per;
    int mine = 0;
    for (int i = s0; i < s0 + per; i++) mine += i < n && (i == 0 || key[i] != key[i - 1]);
    int pre = mine;
    for (int off = 1; off < 64; off <<= 1) {
        const int v = __shfl_up(pre, off, 64);
        if ((tid & 63) >= off) pre += v;
    }
    if ((tid & 63) == 63) wsum[tid >> 6] = pre;
    __syncthreads();
    int total = 0, before = pre - mine;
    for (int w = 0; w < 8; w++) {
        if (w < tid >> 6) before += wsum[w];
        total += wsum[w];
    }
    if (total > LOC_MAX && tid == 0) *over = 1;
    if (idx == nullptr) {
        if (tid == 0) cnt[blockIdx.x] = total;
        return;
    }
    const int32_t b = ptr[blockIdx.x];
    for (int i = s0; i < s0 + per; i++)
        if (i < n && (i == 0 || key[i] != key[i - 1])) col[b + before++] = key[i];
    __syncthreads();
    __threadfence_block();
    for (int i = tid; i < n; i += 512) {
        const int32_t c = acol[p0 + i];
        int lo = 0, hi = total - 1;
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (col[b + mid] < c) lo = mid + 1; else hi = mid;
        }
        idx[p0 + i] = (uint16_t)lo;
    }
}

// Entries of entity e's packed G row: the nodes of row e with both modes' values where rows e and
// ne + e list the same nodes in the same order (the entity's nodes less the dropped ones), else the
// entries of both rows one after the other, each with a zero for the other mode.
__device__ __forceinline__ int g_entries(const int32_t *grp, const int32_t *gcol, int64_t ne, int64_t e, bool &same) {
    const int32_t q0 = grp[e], n0 = grp[e + 1] - q0, q1 = grp[ne + e], n1 = grp[ne + e + 1] - q1;
    same = n0 == n1;
    for (int32_t k = 0; same && k < n0; k++) same = gcol[q0 + k] == gcol[q1 + k];
    return same ? n0 : n0 + n1;
}
// width[s]: the longest packed row of the 64 entities of slice s
__global__ void __launch_bounds__(64) k_g_width(int64_t ne, const int32_t *__restrict__ grp,
                                                const int32_t *__restrict__ gcol, int32_t *__restrict__ width) {
    const int64_t e = blockIdx.x * (int64_t)64 + threadIdx.x;
    bool same;
    int w = e < ne ? g_entries(grp, gcol, ne, e, same) : 0;
    for (int off = 32; off > 0; off >>= 1) w = max(w, __shfl_xor(w, off, 64));
    if (threadIdx.x == 0) width[blockIdx.x] = w;
}
// Where the slots of a slice begin: slices before `cut` have w0 slots per entity, the others w1 (edges
// hold 3 nodes and come first, faces 6), so no table is read ahead of the slots.
struct g_shape {
    int64_t cut;
    int w0, w1;
    __host__ __device__ int width(int64_t s) const { return s < cut ? w0 : w1; }
    __host__ __device__ int64_t first(int64_t s) const { return 64 * (s < cut ? s * w0 : cut * w0 + (s - cut) * w1); }
};
template <typename R>
__global__ void __launch_bounds__(64) k_g_fill(int64_t ne, const int32_t *__restrict__ grp,
                                               const int32_t *__restrict__ gcol, const double *__restrict__ gv,
                                               g_shape sh, int32_t *__restrict__ pcol, R *__restrict__ pval) {
    const int64_t e = blockIdx.x * (int64_t)64 + threadIdx.x;
    const int64_t b = sh.first(blockIdx.x) + threadIdx.x;
    const int w = sh.width(blockIdx.x);
    bool same = true;
    const int n = e < ne ? g_entries(grp, gcol, ne, e, same) : 0;
    const int32_t q0 = e < ne ? grp[e] : 0, n0 = e < ne ? grp[e + 1] - q0 : 0, q1 = e < ne ? grp[ne + e] : 0;
    for (int k = 0; k < w; k++) {
        int32_t c = -1;
        double v0 = 0.0, v1 = 0.0;
        if (k < n) {
            if (same) { c = gcol[q0 + k]; v0 = gv[q0 + k]; v1 = gv[q1 + k]; }
            else if (k < n0) { c = gcol[q0 + k]; v0 = gv[q0 + k]; }
            else { c = gcol[q1 + k - n0]; v1 = gv[q1 + k - n0]; }
        }
        pcol[b + 64 * (int64_t)k] = c;
        st(pval, b + 64 * (int64_t)k, cx<R>((R)v0, (R)v1));
    }
}

// Row p of G^T (DOF columns, mode 0 before mode 1 when ascending) as (entity, both modes'
// values): the two runs merged when the row is strictly ascending, else every entry by itself
// with a zero for the other mode.  Returns the number of entries; writes them when ocol is given.
template <typename R>
__device__ int gt_entries(const int32_t *ci, const double *gv, int32_t a, int32_t b, int64_t ne, int32_t *ocol, R *oval) {
    bool asc = true;
    int32_t m = b;
    for (int32_t i = a; i < b; i++) {
        if (i > a && ci[i] <= ci[i - 1]) asc = false;
        if (m == b && ci[i] >= ne) m = i;
    }
    int n = 0;
    auto put = [&](int32_t e, double v0, double v1) {
        if (ocol != nullptr) { ocol[n] = e; st(oval, n, cx<R>((R)v0, (R)v1)); }
        n++;
    };
    if (!asc) {
        for (int32_t i = a; i < b; i++) {
            if (ci[i] < ne) put(ci[i], gv[i], 0.0); else put((int32_t)(ci[i] - ne), 0.0, gv[i]);
        }
        return n;
    }
    int32_t i = a, j = m;
    while (i < m || j < b) {
        const int64_t ei = i < m ? ci[i] : INT64_MAX, ej = j < b ? ci[j] - ne : INT64_MAX;
        if (ei == ej) { put((int32_t)ei, gv[i], gv[j]); i++; j++; }
        else if (ei < ej) { put((int32_t)ei, gv[i], 0.0); i++; }
        else { put((int32_t)ej, 0.0, gv[j]); j++; }
    }
    return n;
}
__global__ void __launch_bounds__(RB) k_gt_count(int64_t np2, int64_t ne, const int32_t *__restrict__ rp,
                                                 const int32_t *__restrict__ ci, int32_t *__restrict__ cnt) {
    const int64_t p = blockIdx.x * (int64_t)RB + threadIdx.x;
    if (p < np2) cnt[p] = gt_entries<float>(ci, nullptr, rp[p], rp[p + 1], ne, nullptr, nullptr);
}
template <typename R>
__global__ void __launch_bounds__(RB) k_gt_fill(int64_t np2, int64_t ne, const int32_t *__restrict__ rp,
                                                const int32_t *__restrict__ ci, const double *__restrict__ gv,
                                                const int32_t *__restrict__ prp, int32_t *__restrict__ pcol,
                                                R *__restrict__ pval) {
    const int64_t p = blockIdx.x * (int64_t)RB + threadIdx.x;
    if (p < np2) gt_entries<R>(ci, gv, rp[p], rp[p + 1], ne, pcol + prp[p], pval + 2 * (int64_t)prp[p]);
}

// t = diag(G^T K G)^{-1} G^T (xs x), GL lanes per row, up to U entries of a lane loaded before
// their gathers (a vertex row of a Kuhn mesh holds 50 entities: two round trips at 8 lanes where
// one entry at a time took seven).  Sums in FP64.
template <typename R, int GL>
__global__ void __launch_bounds__(256) k_gt_pk(int64_t np2, const int32_t *__restrict__ rp, const int32_t *__restrict__ col,
                                               const R *__restrict__ val, const R *__restrict__ dsinv,
                                               const R *__restrict__ x, const double *__restrict__ xs, R *__restrict__ t) {
    constexpr int U = GL == 16 ? 2 : 4;
    const int64_t p = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) / GL;
    const int lane = threadIdx.x % GL;
    if (p >= np2) return;
    const double s = xs != nullptr ? xs[0] : 1.0;
    const cx<R> d = ld(dsinv, p);
    double ar = 0.0, ai = 0.0;
    const int32_t e1 = rp[p + 1];
    for (int32_t e = rp[p] + lane; e < e1; e += GL * U) {
        int32_t c[U];
        cx<R> g[U];
        cx2<R> v[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int32_t q = e + u * GL < e1 ? e + u * GL : e;
            c[u] = col[q];
            g[u] = ld(val, q);
        }
#pragma unroll
        for (int u = 0; u < U; u++) v[u] = ld2(x, c[u]);
#pragma unroll
        for (int u = 0; u < U; u++)
            if (e + u * GL < e1) {
                ar += (double)g[u].re * v[u].ar + (double)g[u].im * v[u].br;
                ai += (double)g[u].re * v[u].ai + (double)g[u].im * v[u].bi;
            }
    }
    ar = lane_sum<GL>(ar);
    ai = lane_sum<GL>(ai);
    if (lane == 0) {
        ar *= s;
        ai *= s;
        st(t, p, cx<R>((R)(d.re * ar - d.im * ai), (R)(d.re * ai + d.im * ar)));
    }
}

template <typename R>
static void launch_gt_pk(hipStream_t st, int L, int64_t np2, const int32_t *rp, const int32_t *col, const R *val,
                         const R *dsinv, const R *x, const double *xs, R *t) {
    if (L != 4 && L != 16) L = 8;
    const unsigned grid = (unsigned)((np2 * L + 255) / 256);
    if (L == 4) k_gt_pk<R, 4><<<grid, 256, 0, st>>>(np2, rp, col, val, dsinv, x, xs, t);
    else if (L == 16) k_gt_pk<R, 16><<<grid, 256, 0, st>>>(np2, rp, col, val, dsinv, x, xs, t);
    else k_gt_pk<R, 8><<<grid, 256, 0, st>>>(np2, rp, col, val, dsinv, x, xs, t);
}

// z = BJ(xs x) + G t (G in slices of 64 entities, gcol NULL: no gradient part; inv NULL: x in place of BJ(xs x)),
// one entity per lane
template <typename R>
__global__ void __launch_bounds__(RB) k_bj_grad_pk(int64_t ne, const R *__restrict__ inv, const R *__restrict__ x,
                                                   const double *__restrict__ xs, g_shape sh,
                                                   const int32_t *__restrict__ gcol, const R *__restrict__ gval,
                                                   const R *__restrict__ t, R *__restrict__ z) {
    const int64_t e = blockIdx.x * (int64_t)RB + threadIdx.x;
    if (e >= ne) return;
    cx2<R> r = ld2(x, e);
    cx<R> z0(r.ar, r.ai), z1(r.br, r.bi);
    if (inv != nullptr) {
        const double s = xs != nullptr ? xs[0] : 1.0;
        const cx2<R> i0 = ld2(inv, 2 * e), i1 = ld2(inv, 2 * e + 1);
        r = cx2<R>{(R)(s * r.ar), (R)(s * r.ai), (R)(s * r.br), (R)(s * r.bi)};
        const cx<R> r0(r.ar, r.ai), r1(r.br, r.bi);
        z0 = cadd(cmul(cx<R>(i0.ar, i0.ai), r0), cmul(cx<R>(i0.br, i0.bi), r1));
        z1 = cadd(cmul(cx<R>(i1.ar, i1.ai), r0), cmul(cx<R>(i1.br, i1.bi), r1));
    }
    if (gcol != nullptr) {
        const int64_t si = e >> 6;
        const int w = sh.width(si);
        const int64_t b = sh.first(si) + (e & 63);
        constexpr int U = 3;   // edges hold 3 nodes, faces 6
        for (int k = 0; k < w; k += U) {
            int32_t c[U];
            cx<R> g[U], tv[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int64_t q = b + 64 * (int64_t)(k + u < w ? k + u : k);
                c[u] = k + u < w ? gcol[q] : -1;
                g[u] = ld(gval, q);
            }
#pragma unroll
            for (int u = 0; u < U; u++) tv[u] = c[u] >= 0 ? ld(t, c[u]) : cx<R>();
#pragma unroll
            for (int u = 0; u < U; u++) {
                z0 = cx<R>(z0.re + g[u].re * tv[u].re, z0.im + g[u].re * tv[u].im);
                z1 = cx<R>(z1.re + g[u].im * tv[u].re, z1.im + g[u].im * tv[u].im);
            }
        }
    }
    st2(z, e, cx2<R>{z0.re, z0.im, z1.re, z1.im});
}

// ---------------------------------------------------------------- one launch per smoother application and product
// With M = L + G D G^T (L the 2x2 block inverses, D the inverted diagonal) and t = D G^T q,
//   K M q = K (L q) + (K G) t   and   G^T (K M q) = (G^T K) (L q) + (G^T K G) t,
// so with the matrices KG = K G, H = G^T K and HG = G^T K G at hand the polynomial's recurrence on q carries
// G^T q along and needs one launch per product where smoother and product take three (G^T, then L and G, then
// K).  KG's rows are the entities', with the P2 nodes of their columns' rows of G; H's and HG's are the nodes',
// with the columns of the entities in their rows of G^T and the nodes of those' KG rows.  KG and H are formed in
// complex128 and kept in complex64 beside K; HG is summed in FP64 from KG as it is kept.

// The distinct values that GEN(row, put) puts, ascending: their number to cnt, or with out the values
// themselves at out[ptr[row]].  A row with more than CAND candidates or UNIQ values sets *over.
static constexpr int FUSE_CAND = 8192, FUSE_UNIQ = 512;
template <typename GEN>
__global__ void __launch_bounds__(256) k_distinct(GEN gen, int32_t *__restrict__ cnt, const int32_t *__restrict__ ptr,
                                                  int32_t *__restrict__ out, int *__restrict__ over) {
    __shared__ int32_t cand[FUSE_CAND];
    __shared__ uint8_t first[FUSE_CAND];
    __shared__ int found, kept;
    const int64_t row = blockIdx.x;
    if (threadIdx.x == 0) { found = 0; kept = 0; }
    __syncthreads();
    gen(row, [&](int32_t v) {
        const int i = atomicAdd(&found, 1);
        if (i < FUSE_CAND) cand[i] = v;
    });
    __syncthreads();
    const int n = min(found, FUSE_CAND);
    for (int i = threadIdx.x; i < n; i += 256) {
        bool f = true;
        for (int j = 0; f && j < i; j++) f = cand[j] != cand[i];
        first[i] = f;
        if (f) atomicAdd(&kept, 1);
    }
    __syncthreads();
    if (threadIdx.x == 0 && (found > FUSE_CAND || kept > FUSE_UNIQ)) *over = 1;
    if (out == nullptr) {
        if (threadIdx.x == 0) cnt[row] = kept;
        return;
    }
    for (int i = threadIdx.x; i < n; i += 256) {
        if (!first[i]) continue;
        int rank = 0;
        for (int j = 0; j < n; j++) rank += first[j] && cand[j] < cand[i];
        out[ptr[row] + rank] = cand[i];
    }
}
struct gen_kg {   // the nodes of the G rows of entity row's columns
    int64_t ne;
    const int32_t *rowptr, *acol, *grp, *gcol;
    template <typename PUT>
    __device__ void operator()(int64_t e, PUT &&put) const {
        const int32_t a0 = rowptr[e] >> 1, deg = (rowptr[e + 1] >> 1) - a0;
        for (int k = threadIdx.x; k < 2 * deg; k += 256) {
            const int64_t d = (k & 1 ? ne : 0) + acol[a0 + (k >> 1)];
            for (int32_t q = grp[d]; q < grp[d + 1]; q++) put(gcol[q]);
        }
    }
};
struct gen_of_nodes {   // what the rows (of rp and col, at rp[i] >> shift) of the entities in node row's row of G^T list
    int64_t ne;
    const int32_t *trp, *tcol, *rp, *col;
    int shift;
    template <typename PUT>
    __device__ void operator()(int64_t p, PUT &&put) const {
        for (int32_t q = trp[p]; q < trp[p + 1]; q++) {
            const int64_t e = tcol[q] % ne;
            for (int32_t k = (rp[e] >> shift) + threadIdx.x; k < rp[e + 1] >> shift; k += 256) put(col[k]);
        }
    }
};

// KG: a wavefront per entity, a node per lane; sums in the order of the row.
__global__ void __launch_bounds__(64) k_kg_values(int64_t ne, int64_t half, const int32_t *__restrict__ rowptr,
                                                  const int32_t *__restrict__ acol, const double *__restrict__ vals,
                                                  const uint8_t *__restrict__ mask, const int32_t *__restrict__ grp,
                                                  const int32_t *__restrict__ gcol, const double *__restrict__ gv,
                                                  const int32_t *__restrict__ kgp, const int32_t *__restrict__ kgc,
                                                  float *__restrict__ kgv) {
    const int64_t e = blockIdx.x;
    const int32_t r0 = rowptr[e], deg = (rowptr[e + 1] - r0) >> 1;
    const bool m0 = mask == nullptr || mask[e], m1 = mask == nullptr || mask[ne + e];
    for (int32_t k0 = kgp[e]; k0 < kgp[e + 1]; k0 += 64) {
        const int32_t k = k0 + (int)threadIdx.x, p = k < kgp[e + 1] ? kgc[k] : -1;
        cx<double> a, b;
        for (int32_t j = 0; j < deg; j++) {
            const int64_t c = acol[(r0 >> 1) + j];
            for (int m = 0; m < 2; m++) {
                const int64_t d = m * ne + c;
                if (mask != nullptr && !mask[d]) continue;
                double g = 0.0;
                for (int32_t q = grp[d]; q < grp[d + 1]; q++)
                    if (gcol[q] == p) g += gv[q];
                const cx<double> u = ld(vals, (int64_t)r0 + j + m * deg), v = ld(vals, half + r0 + j + m * deg);
                a = cx<double>(a.re + g * u.re, a.im + g * u.im);
                b = cx<double>(b.re + g * v.re, b.im + g * v.im);
            }
        }
        // a masked row of K is the identity's: G's own row
        for (int m = 0; m < 2; m++) {
            if (m == 0 ? m0 : m1) continue;
            double g = 0.0;
            for (int32_t q = grp[m * ne + e]; q < grp[m * ne + e + 1]; q++)
                if (gcol[q] == p) g += gv[q];
            (m == 0 ? a : b) = cx<double>(g, 0.0);
        }
        if (p >= 0) st2(kgv, k, cx2<float>{(float)a.re, (float)a.im, (float)b.re, (float)b.im});
    }
}

__device__ __forceinline__ int place_of(const int32_t *list, int n, int32_t v) {
    int lo = 0;
    for (int hi = n - 1; lo < hi;) {
        const int mid = (lo + hi) >> 1;
        if (list[mid] < v) lo = mid + 1; else hi = mid;
    }
    return lo;
}
// H (FROM_KG false: rows of K) or HG (rows of KG): a wavefront per node, one entry of its row of G^T after the
// other, whose distinct columns go to different lanes; sums in LDS in the order of the row.
template <bool FROM_KG>
__global__ void __launch_bounds__(64) k_node_values(int64_t ne, int64_t half, const int32_t *__restrict__ rowptr,
                                                    const int32_t *__restrict__ acol, const double *__restrict__ vals,
                                                    const uint8_t *__restrict__ mask, const int32_t *__restrict__ kgp,
                                                    const int32_t *__restrict__ kgc, const float *__restrict__ kgv,
                                                    const int32_t *__restrict__ trp, const int32_t *__restrict__ tcol,
                                                    const double *__restrict__ tv, const int32_t *__restrict__ ptr,
                                                    const int32_t *__restrict__ col, float *__restrict__ out) {
    __shared__ int32_t list[FUSE_UNIQ];
    __shared__ double acc[FUSE_UNIQ][4];
    const int64_t p = blockIdx.x;
    const int lane = threadIdx.x, n = min(ptr[p + 1] - ptr[p], FUSE_UNIQ);
    for (int i = lane; i < n; i += 64) {
        list[i] = col[ptr[p] + i];
        for (int q = 0; q < 4; q++) acc[i][q] = 0.0;
    }
    __syncthreads();
    for (int32_t q = trp[p]; q < trp[p + 1]; q++) {
        const int64_t d = tcol[q], e = d % ne;
        const int r = d >= ne;
        const double g = tv[q];
        if constexpr (FROM_KG) {
            for (int32_t k = kgp[e] + lane; k < kgp[e + 1]; k += 64) {
                const cx2<float> v = ld2(kgv, k);
                double *a = acc[place_of(list, n, kgc[k])];
                a[0] += g * (r ? v.br : v.ar);
                a[1] += g * (r ? v.bi : v.ai);
            }
        } else if (mask != nullptr && !mask[d]) {
            if (lane == 0) acc[place_of(list, n, (int32_t)e)][2 * r] += g;
        } else {
            const int32_t r0 = rowptr[e], deg = (rowptr[e + 1] - r0) >> 1;
            const int64_t b = (int64_t)r * half + r0;
            for (int32_t j = lane; j < deg; j += 64) {
                const int32_t c = acol[(r0 >> 1) + j];
                const bool c0 = mask == nullptr || mask[c], c1 = mask == nullptr || mask[ne + c];
                const cx<double> u = ld(vals, b + j), v = ld(vals, b + j + deg);
                double *a = acc[place_of(list, n, c)];
                if (c0) { a[0] += g * u.re; a[1] += g * u.im; }
                if (c1) { a[2] += g * v.re; a[3] += g * v.im; }
            }
        }
        __syncthreads();
    }
    for (int i = lane; i < n; i += 64) {
        if constexpr (FROM_KG) st(out, (int64_t)ptr[p] + i, cx<float>((float)acc[i][0], (float)acc[i][1]));
        else st2(out, (int64_t)ptr[p] + i, cx2<float>{(float)acc[i][0], (float)acc[i][1], (float)acc[i][2], (float)acc[i][3]});
    }
}

// The matrices of the fused steps and the vectors they work on.
struct fuse_mat {
    int64_t ne, np2;
    const int32_t *rowptr, *acol;
    const float *kre, *kim;
    const uint8_t *flag;
    const int32_t *kgp, *kgc, *hp, *hc, *hgp, *hgc;
    const float *kgv, *hv, *hgv;
    const float *inv, *dsinv;   // L and D
    double *s, *sy;             // G^T q and G^T y, complex
};

// Start of a step: yl = L (xs x), s = G^T (xs x), t = D s.  One lane per entity, then 16 per node.
__global__ void __launch_bounds__(256) k_fuse_start(fuse_mat f, unsigned eblocks, const int32_t *__restrict__ trp,
                                                    const int32_t *__restrict__ tcol, const float *__restrict__ tval,
                                                    const float *__restrict__ x, const double *__restrict__ xs,
                                                    float *__restrict__ yl, float *__restrict__ t) {
    const double sc = xs != nullptr ? xs[0] : 1.0;
    if (blockIdx.x < eblocks) {
        const int64_t e = blockIdx.x * (int64_t)256 + threadIdx.x;
        if (e >= f.ne) return;
        const cx2<float> i0 = ld2(f.inv, 2 * e), i1 = ld2(f.inv, 2 * e + 1);
        const cx2<float> r = ld2(x, e);
        const cx<float> r0((float)(sc * r.ar), (float)(sc * r.ai)), r1((float)(sc * r.br), (float)(sc * r.bi));
        const cx<float> z0 = cadd(cmul(cx<float>(i0.ar, i0.ai), r0), cmul(cx<float>(i0.br, i0.bi), r1));
        const cx<float> z1 = cadd(cmul(cx<float>(i1.ar, i1.ai), r0), cmul(cx<float>(i1.br, i1.bi), r1));
        st2(yl, e, cx2<float>{z0.re, z0.im, z1.re, z1.im});
        return;
    }
    const int64_t p = ((blockIdx.x - eblocks) * (int64_t)256 + threadIdx.x) / 16;
    const int lane = threadIdx.x % 16;
    if (p >= f.np2) return;
    const cx<float> d = ld(f.dsinv, p);
    double ar = 0.0, ai = 0.0;
    const int32_t q1 = trp[p + 1];
    for (int32_t q = trp[p] + lane; q < q1; q += 32) {
        const bool two = q + 16 < q1;
        const int32_t qb = two ? q + 16 : q;
        const cx<float> ga = ld(tval, q), gb = ld(tval, qb);
        const cx2<float> va = ld2(x, tcol[q]), vb = ld2(x, tcol[qb]);
        ar += (double)ga.re * va.ar + (double)ga.im * va.br;
        ai += (double)ga.re * va.ai + (double)ga.im * va.bi;
        if (two) {
            ar += (double)gb.re * vb.ar + (double)gb.im * vb.br;
            ai += (double)gb.re * vb.ai + (double)gb.im * vb.bi;
        }
    }
    ar = lane_sum<16>(ar) * sc;
    ai = lane_sum<16>(ai) * sc;
    if (lane == 0) {
        st(f.s, p, cx<double>(ar, ai));
        st(t, p, cx<float>((float)(d.re * ar - d.im * ai), (float)(d.re * ai + d.im * ar)));
    }
}

// v = K M q from yl = L q and t = D G^T q, on the rows of K and (END false) of G^T K, and what follows it:
// END false: p = q - c_i v, y = (i == 0 ? c_0 q : y) + c_{i+1} p and the same for s = G^T q and sy = G^T y, then
// yl2 = L p, t2 = D s (last: of y and sy, for the product that ends the step).  END true: y = v.
// L lanes per entity, then LN per node, each lane with all its loads of a trip in flight: an edge's 37 blocks
// and 27 nodes, or a vertex' 220 entities and 65 nodes, take one trip or four.  Bound by the latency of a launch
// and of its chain of loads: 7.7 us at 21,000 DOFs where the three launches it replaces took 3.9 (G^T), 4.0
// (L and G) and 4.1 (K); a step 121 -> 90 us.  (8 or 32 lanes per entity, 16 or 64 per node: 2 - 8 % slower.)
struct fuse_args {
    const float *q, *yl, *t;
    float *y, *p, *yl2, *t2;
    const double *c, *qs;
    int i, last;
};
template <int L, int LN, bool END>
__global__ void __launch_bounds__(256) k_fuse_step(fuse_mat f, unsigned eblocks, fuse_args a) {
    if (blockIdx.x < eblocks) {
        constexpr int UK = 48 / L, UG = UK;   // blocks of K and nodes of a lane whose loads are in flight together
        const int64_t e = (blockIdx.x * (int64_t)256 + threadIdx.x) / L;
        const int lane = threadIdx.x % L;
        if (e >= f.ne) return;
        const uint8_t fl = f.flag[e];
        const int32_t p0 = f.rowptr[e] >> 1, p1 = f.rowptr[e + 1] >> 1, g0 = f.kgp[e], g1 = f.kgp[e + 1];
        const int32_t gs = g0 < g1 ? g0 : 0;   // a slot to read in place of none
        cx2<float> own{}, qv{}, yv{}, i0{}, i1{};
        if (lane == 0) {
            if ((fl & (ROW0 | ROW1)) != (ROW0 | ROW1)) own = ld2(a.yl, e);
            if constexpr (!END) {
                qv = ld2(a.q, e);
                i0 = ld2(f.inv, 2 * e);
                i1 = ld2(f.inv, 2 * e + 1);
                if (a.i > 0) yv = ld2(a.y, e);
            }
        }
        float s0r = 0, s0i = 0, s1r = 0, s1i = 0;
        const int32_t none = fl & (ROW0 | ROW1) ? p1 : p0;   // end of the row's blocks of K
        for (int32_t o = lane; p0 + o < none || g0 + o < g1; o += L * UK) {
            int32_t c[UK], n[UG];
            cx2<float> k[UK], xv[UK], kg[UG], v[UK];
            cx<float> t[UG];
#pragma unroll
            for (int u = 0; u < UK; u++) {
                const int32_t q = p0 + o + u * L < none ? p0 + o + u * L : p0;
                c[u] = f.acol[q];
                k[u] = ld2(f.kre, q);
            }
#pragma unroll
            for (int u = 0; u < UG; u++) {
                const int32_t q = g0 + o + u * L < g1 ? g0 + o + u * L : gs;
                n[u] = f.kgc[q];
                kg[u] = ld2(f.kgv, q);
            }
#pragma unroll
            for (int u = 0; u < UK; u++) xv[u] = ld2(a.yl, c[u]);
#pragma unroll
            for (int u = 0; u < UG; u++) t[u] = ld(a.t, n[u]);
#pragma unroll
            for (int u = 0; u < UK; u++)
                v[u] = cx2<float>{k[u].ar * xv[u].ar + k[u].ai * xv[u].br, k[u].ar * xv[u].ai + k[u].ai * xv[u].bi,
                                  k[u].br * xv[u].ar + k[u].bi * xv[u].br, k[u].br * xv[u].ai + k[u].bi * xv[u].bi};
            if (fl & ROW_CPLX) {
#pragma unroll
                for (int u = 0; u < UK; u++) k[u] = ld2(f.kim, p0 + o + u * L < none ? p0 + o + u * L : p0);
#pragma unroll
                for (int u = 0; u < UK; u++) {
                    v[u].ar -= k[u].ar * xv[u].ai + k[u].ai * xv[u].bi;
                    v[u].ai += k[u].ar * xv[u].ar + k[u].ai * xv[u].br;
                    v[u].br -= k[u].br * xv[u].ai + k[u].bi * xv[u].bi;
                    v[u].bi += k[u].br * xv[u].ar + k[u].bi * xv[u].br;
                }
            }
#pragma unroll
            for (int u = 0; u < UK; u++)
                if (p0 + o + u * L < none) {
                    s0r += v[u].ar;
                    s0i += v[u].ai;
                    s1r += v[u].br;
                    s1i += v[u].bi;
                }
#pragma unroll
            for (int u = 0; u < UG; u++)
                if (g0 + o + u * L < g1) {
                    s0r += kg[u].ar * t[u].re - kg[u].ai * t[u].im;
                    s0i += kg[u].ar * t[u].im + kg[u].ai * t[u].re;
                    s1r += kg[u].br * t[u].re - kg[u].bi * t[u].im;
                    s1i += kg[u].br * t[u].im + kg[u].bi * t[u].re;
                }
        }
        // a masked row of K is the identity's (its entries are zero, its KG row is G's)
        s0r = lane_sum<L>(s0r);
        s0i = lane_sum<L>(s0i);
        s1r = lane_sum<L>(s1r);
        s1i = lane_sum<L>(s1i);
        if (lane != 0) return;
        cx2<float> v{s0r, s0i, s1r, s1i};
        if (!(fl & ROW0)) { v.ar += own.ar; v.ai += own.ai; }
        if (!(fl & ROW1)) { v.br += own.br; v.bi += own.bi; }
        if constexpr (END) {
            st2(a.y, e, v);
        } else {
            const double *cc = a.c + 2 * a.i;
            const double cr = cc[0], ci = cc[1], nr = cc[2], ni = cc[3];
            const double s = a.qs != nullptr ? a.qs[0] : 1.0;
            const double q0r = s * qv.ar, q0i = s * qv.ai, q1r = s * qv.br, q1i = s * qv.bi;
            double y0r = yv.ar, y0i = yv.ai, y1r = yv.br, y1i = yv.bi;
            if (a.i == 0) {
                y0r = cr * q0r - ci * q0i; y0i = cr * q0i + ci * q0r;
                y1r = cr * q1r - ci * q1i; y1i = cr * q1i + ci * q1r;
            }
            const double p0r = q0r - (cr * v.ar - ci * v.ai), p0i = q0i - (cr * v.ai + ci * v.ar);
            const double p1r = q1r - (cr * v.br - ci * v.bi), p1i = q1i - (cr * v.bi + ci * v.br);
            const cx2<float> pn{(float)p0r, (float)p0i, (float)p1r, (float)p1i};
            const cx2<float> yn{(float)(y0r + nr * p0r - ni * p0i), (float)(y0i + nr * p0i + ni * p0r),
                                (float)(y1r + nr * p1r - ni * p1i), (float)(y1i + nr * p1i + ni * p1r)};
            if (!a.last) {
                st2(a.p, e, pn);
                st2(a.y, e, yn);
            }
            const cx2<float> w = a.last ? yn : pn;
            const cx<float> r0(w.ar, w.ai), r1(w.br, w.bi);
            const cx<float> z0 = cadd(cmul(cx<float>(i0.ar, i0.ai), r0), cmul(cx<float>(i0.br, i0.bi), r1));
            const cx<float> z1 = cadd(cmul(cx<float>(i1.ar, i1.ai), r0), cmul(cx<float>(i1.br, i1.bi), r1));
            st2(a.yl2, e, cx2<float>{z0.re, z0.im, z1.re, z1.im});
        }
        return;
    }
    if constexpr (!END) {
        const int64_t p = ((blockIdx.x - eblocks) * (int64_t)256 + threadIdx.x) / LN;
        const int lane = threadIdx.x % LN;
        if (p >= f.np2) return;
        const int32_t h0 = f.hp[p], h1 = f.hp[p + 1], g0 = f.hgp[p], g1 = f.hgp[p + 1];
        const int32_t hs = h0 < h1 ? h0 : 0, gs = g0 < g1 ? g0 : 0;
        cx<float> d;
        cx<double> sv, yv;
        if (lane == 0) {
            d = ld(f.dsinv, p);
            sv = ld(f.s, p);
            if (a.i > 0) yv = ld(f.sy, p);
        }
        double zr = 0.0, zi = 0.0;
        constexpr int UH = 2;
        for (int32_t o = lane; h0 + o < h1 || g0 + o < g1; o += UH * LN) {
            int32_t c[UH], n[UH];
            cx2<float> hv[UH], xv[UH];
            cx<float> gv[UH], tv[UH];
#pragma unroll
            for (int u = 0; u < UH; u++) {
                const int32_t q = h0 + o + u * LN < h1 ? h0 + o + u * LN : hs, r = g0 + o + u * LN < g1 ? g0 + o + u * LN : gs;
                c[u] = f.hc[q];
                hv[u] = ld2(f.hv, q);
                n[u] = f.hgc[r];
                gv[u] = ld(f.hgv, r);
            }
#pragma unroll
            for (int u = 0; u < UH; u++) {
                xv[u] = ld2(a.yl, c[u]);
                tv[u] = ld(a.t, n[u]);
            }
#pragma unroll
            for (int u = 0; u < UH; u++) {
                if (h0 + o + u * LN < h1) {
                    zr += (double)hv[u].ar * xv[u].ar - (double)hv[u].ai * xv[u].ai + (double)hv[u].br * xv[u].br - (double)hv[u].bi * xv[u].bi;
                    zi += (double)hv[u].ar * xv[u].ai + (double)hv[u].ai * xv[u].ar + (double)hv[u].br * xv[u].bi + (double)hv[u].bi * xv[u].br;
                }
                if (g0 + o + u * LN < g1) {
                    zr += (double)gv[u].re * tv[u].re - (double)gv[u].im * tv[u].im;
                    zi += (double)gv[u].re * tv[u].im + (double)gv[u].im * tv[u].re;
                }
            }
        }
        zr = lane_sum<LN>(zr);
        zi = lane_sum<LN>(zi);
        if (lane != 0) return;
        const double *cc = a.c + 2 * a.i;
        const double cr = cc[0], ci = cc[1], nr = cc[2], ni = cc[3];
        if (a.i == 0) yv = cx<double>(cr * sv.re - ci * sv.im, cr * sv.im + ci * sv.re);
        const cx<double> sn(sv.re - (cr * zr - ci * zi), sv.im - (cr * zi + ci * zr));
        const cx<double> yn(yv.re + nr * sn.re - ni * sn.im, yv.im + nr * sn.im + ni * sn.re);
        st(f.s, p, sn);
        st(f.sy, p, yn);
        const cx<double> w = a.last ? yn : sn;
        st(a.t2, p, cx<float>((float)(d.re * w.re - d.im * w.im), (float)(d.re * w.im + d.im * w.re)));
    }
}

// b (interleaved, R) = s a (caller's layout, complex128)
template <typename R>
__global__ void __launch_bounds__(RB) k_pack_vec(int64_t ne, const double *__restrict__ a, double s, R *__restrict__ b) {
    const int64_t e = blockIdx.x * (int64_t)RB + threadIdx.x;
    if (e >= ne) return;
    const cx<double> u = ld(a, e), v = ld(a, ne + e);
    st2(b, e, cx2<R>{(R)(u.re * s), (R)(u.im * s), (R)(v.re * s), (R)(v.im * s)});
}
// x (caller's layout, complex128) = (add ? x : 0) + s d (interleaved, R)
template <typename R>
__global__ void __launch_bounds__(RB) k_unpack_vec(int64_t ne, const R *__restrict__ d, double s, int add,
                                                   double *__restrict__ x) {
    const int64_t e = blockIdx.x * (int64_t)RB + threadIdx.x;
    if (e >= ne) return;
    const cx2<R> v = ld2(d, e);
    cx<double> u0, u1;
    if (add) { u0 = ld(x, e); u1 = ld(x, ne + e); }
    st(x, e, cx<double>(u0.re + s * (double)v.ar, u0.im + s * (double)v.ai));
    st(x, ne + e, cx<double>(u1.re + s * (double)v.br, u1.im + s * (double)v.bi));
}

// ---------------------------------------------------------------- solver object
struct emg_solver {
    int64_t n = 0, nnz = 0, n_ent = 0;
    int restart = 0, precision = 64;
    int cap = 0;                    // Krylov steps the basis storage holds: restart, up to twice that in complex64
    const int32_t *rowptr = nullptr, *cols = nullptr;
    const double *vals = nullptr;   // complex128 K (caller-owned)
    const uint8_t *mask = nullptr;  // caller-owned, may be null
    // K in the packed layout, in the precision of the solver's steps (k_pack_matrix); at precision 64 acol and the
    // planes are NULL where the card has no room for them, and the steps read the caller's CSR
    int32_t *acol = nullptr;        // nnz / 4 column entities
    void *kre = nullptr, *kim = nullptr;   // real and imaginary planes, nnz values each
    uint8_t *row_flag = nullptr;    // n_ent
    int32_t *loc_ptr = nullptr, *loc_col = nullptr;   // distinct columns of every LOC_ROWS rows (k_loc_columns) or NULL
    uint16_t *loc_idx = nullptr;
    double *inv64 = nullptr;
    float *inv32 = nullptr;
    double *V = nullptr;            // cap + 1 basis vectors, element type per precision
    double *w = nullptr, *z = nullptr, *r = nullptr, *d = nullptr;   // d: precision 64 only
    double *partial = nullptr, *h = nullptr;
    int nblk = 0;
    // Arnoldi steps run from captured HIP graphs (chunks of CHUNK_IT steps)
    // with the Hessenberg column, Givens rotations and residual estimate
    // updated on the device; the host reads the estimates once per chunk.
    double *arn = nullptr;        // device Arnoldi state (see arn_off)
    double *pn = nullptr;         // per-block partial norms of the new basis vector
    double *gram = nullptr;       // the basis' Gram matrix less the identity, (cap + 1)^2 complex
    double *flag = nullptr;       // scratch of the pattern check
    double *host = nullptr;       // pinned host memory the kernels write to and small uploads go through (host_off)
    double *host_dev = nullptr;   // the device's address of it
    kept_dev *kept = nullptr;     // spaces kept from the running solve's earlier refinement cycles (in arn)
    hipStream_t cap_stream = nullptr;   // capture stream (graphs are launched on the caller's stream)
    // optional gradient correction of the smoother: G (n x np2), G^T (np2 x n)
    int64_t np2 = 0;
    const int32_t *g_rowptr = nullptr, *g_cols = nullptr, *gt_rowptr = nullptr, *gt_cols = nullptr;
    const double *g_vals = nullptr, *gt_vals = nullptr;   // caller-owned
    // the same in the packed layout, in the precision of the solver's steps
    g_shape g_sh{0, 0, 0};
    int32_t *g_pcol = nullptr, *gt_prp = nullptr, *gt_pcol = nullptr;
    void *g_pval = nullptr, *gt_pval = nullptr;
    double *dS = nullptr, *dsinv64 = nullptr, *tg = nullptr;
    float *dsinv32 = nullptr;
    // the matrices of the fused steps (fuse_pattern), all or none
    bool fused = false;
    int32_t *kg_ptr = nullptr, *kg_col = nullptr, *h_ptr = nullptr, *h_col = nullptr, *hg_ptr = nullptr, *hg_col = nullptr;
    void *kg_val = nullptr, *h_val = nullptr, *hg_val = nullptr;
    double *fuse_s = nullptr;       // G^T q and G^T y, np2 complex each
    float *fuse_t = nullptr;        // two buffers of t, np2 complex each
    // optional learned weights of the smoother (caller-owned complex128):
    // w_e per entity scales its 2x2 block inverse, w_p per P2 node its diagonal
    const double *w_e = nullptr, *w_p = nullptr;
    // optional polynomial acceleration of the smoother (emg_solver_set_poly):
    // M p(K M) with 1 - z p(z) = prod_i (1 - z c_i), c_i = 1/theta_i on the device
    int poly_deg = 1;
    double *poly_c = nullptr;                               // POLY_MAX complex coefficients
    double *pp = nullptr, *py = nullptr, *pu = nullptr;   // work vectors (n complex each)
    // blocked-SpMV lanes per entity, [0] complex128, [1] complex64: 0 until tuned on
    // the first matrix (tune_spmv), with the measured milliseconds per variant
    int lanes[2] = {0, 0};
    float tune_ms[2][4] = {};
    // lanes per row of the smoother's G^T product (k_gt_apply): 0 until tuned with the
    // SpMV (gradient set), then 4, 8 or 16, with the measured milliseconds per launch
    int gt_lanes = 0;
    float gt_ms[3] = {};
    // captured steps by the basis vector they start from, as cycles first reach them; every buffer
    // they name is the solver's own, so only another gradient or degree makes them stale
    std::vector<hipGraphExec_t> exec;
    hipGraphExec_t tail = nullptr;   // the preconditioner at a cycle's end
    int64_t exec_np2 = 0;
    int exec_poly = 0;
};
static constexpr int POLY_MAX = 16;

static void drop_graphs(emg_solver *s) {
    for (hipGraphExec_t e : s->exec)
        if (e != nullptr) (void)hipGraphExecDestroy(e);
    s->exec.clear();
    if (s->tail != nullptr) (void)hipGraphExecDestroy(s->tail);
    s->tail = nullptr;
}

static void drop_fused(emg_solver *s) {
    void *ps[] = {s->kg_ptr, s->kg_col, s->h_ptr, s->h_col, s->hg_ptr, s->hg_col, s->kg_val, s->h_val, s->hg_val,
                  s->fuse_s, s->fuse_t};
    for (void *p : ps) (void)hipFree(p);
    s->kg_ptr = s->kg_col = s->h_ptr = s->h_col = s->hg_ptr = s->hg_col = nullptr;
    s->kg_val = s->h_val = s->hg_val = nullptr;
    s->fuse_s = nullptr;
    s->fuse_t = nullptr;
    s->fused = false;
}

template <typename... T>
static void drop(T *&...p) {   // frees device buffers and forgets them
    ((void)hipFree(p), ...);
    ((p = nullptr), ...);
}
static void drop_gradient(emg_solver *s) {
    drop(s->g_pcol, s->g_pval, s->gt_prp, s->gt_pcol, s->gt_pval, s->dS, s->dsinv64, s->tg, s->dsinv32);
    drop_fused(s);
}
static void drop_local(emg_solver *s) { drop(s->loc_ptr, s->loc_col, s->loc_idx); }
static void drop_buffers(emg_solver *s) {   // what emg_solver_create allocates
    drop(s->acol, s->kre, s->kim, s->row_flag, s->inv64, s->inv32, s->V, s->w, s->z, s->r, s->d, s->partial, s->h, s->arn,
         s->pn, s->gram, s->flag, s->poly_c, s->pp, s->py, s->pu);
    drop_local(s);
}

static void free_solver(emg_solver *s) {
    if (!s) return;
    drop_graphs(s);
    drop_gradient(s);
    drop_buffers(s);
    if (s->host) (void)hipHostFree(s->host);
    if (s->cap_stream) (void)hipStreamDestroy(s->cap_stream);
    delete s;
}

// The smoother in the caller's layout and complex128 (the Arnoldi probe): 2x2 block Jacobi, plus the
// gradient correction when set.
static void apply_prec_std(emg_solver *s, const double *x, double *y, hipStream_t st) {
    if (s->np2 > 0) {
        launch_gt(st, s->np2, s->gt_rowptr, s->gt_cols, s->gt_vals, s->dsinv64, x, s->tg);
        k_bj_grad_apply<<<emg::grid_for(s->n_ent, RB), RB, 0, st>>>(s->n_ent, s->inv64, x, s->g_rowptr, s->g_cols,
                                                                    s->g_vals, s->tg, y);
    } else {
        k_bj_apply<<<emg::grid_for(s->n_ent, RB), RB, 0, st>>>(s->n_ent, s->inv64, x, y);
    }
}

// The smoother in the solver's layout: y = M (xs x), xs a scale on the device or NULL.
template <typename R>
static void apply_prec(emg_solver *s, const R *x, const double *xs, R *y, hipStream_t st) {
    const bool grad = s->np2 > 0;
    const R *inv = sizeof(R) == 8 ? reinterpret_cast<const R *>(s->inv64) : reinterpret_cast<const R *>(s->inv32);
    R *t = reinterpret_cast<R *>(s->tg);
    if (grad) {
        const R *dsi = sizeof(R) == 8 ? reinterpret_cast<const R *>(s->dsinv64) : reinterpret_cast<const R *>(s->dsinv32);
        launch_gt_pk<R>(st, s->gt_lanes, s->np2, s->gt_prp, s->gt_pcol, static_cast<const R *>(s->gt_pval), dsi, x, xs, t);
    }
    k_bj_grad_pk<R><<<emg::grid_for(s->n_ent, RB), RB, 0, st>>>(s->n_ent, inv, x, xs, s->g_sh, grad ? s->g_pcol : nullptr,
                                                                static_cast<const R *>(s->g_pval), t, y);
}

// A product with the packed matrix; L lanes per entity.
template <typename R, int EP, bool STD>
static void spmv_pk(emg_solver *s, int L, const R *x, const sp_args<R> &a, hipStream_t st) {
    if constexpr (sizeof(R) == 8 && !STD)
        if (s->kre == nullptr) {
            launch_spmv_pk<R, EP, STD>(st, L, s->n_ent, s->rowptr, s->cols, s->vals, nullptr, s->row_flag, x, a, loc_tab{}, s->nnz / 2);
            return;
        }
    launch_spmv_pk<R, EP, STD>(st, L, s->n_ent, s->rowptr, s->acol, static_cast<const R *>(s->kre),
                               static_cast<const R *>(s->kim), s->row_flag, x, a, loc_tab{s->loc_ptr, s->loc_col, s->loc_idx});
}

// Lanes per entity for vectors in the caller's layout, whose two gathers per block favour few: 8 / 16
// lanes take 116 / 141 us (complex64, air), 185 / 193 (complex64, lossy), 208 / 237 and 318 / 346
// (complex128) on the posts box at 80 x 40 x 16 hexes, and 8 is within 2 % of the best down to 2,000 tets.
static constexpr int STD_LANES = 8;

// y = K x, or b - K x, in complex128 and the caller's layout: the packed planes where they are
// complex128 (precision 64), else the caller's CSR values.
static void spmv_std(emg_solver *s, const double *x, const double *b, double *y, hipStream_t st) {
    if (s->precision == 64 && s->kre != nullptr) {
        sp_args<double> a{b, y, nullptr, nullptr, 0, nullptr};
        if (b != nullptr) spmv_pk<double, SP_RESID, true>(s, STD_LANES, x, a, st);
        else spmv_pk<double, SP_Y, true>(s, STD_LANES, x, a, st);
    } else {
        launch_spmv_blk(st, s->n, s->nnz, s->rowptr, s->cols, s->vals, s->mask, x, b, y, s->lanes[0]);
    }
}

// The preconditioner: the smoother M, or with a polynomial of degree d > 1,
// M p(K M) x evaluated as  y = c_0 x, q_0 = x;  q_{i+1} = q_i - c_i K M q_i,
// y += c_{i+1} q_{i+1}  (i < d-1);  out = M y.  d - 1 extra SpMVs and d - 1
// extra smoother applications per call; the updates of q and y follow each product in
// its own launch (SP_POLY), which at 19,664 DOFs saves the 2.7 us launch they took
// after every product and at any size the pass over t = K M q.
static void apply_fused(emg_solver *s, const float *vt, const double *xs, float *out, bool product, hipStream_t st);
template <typename R>
static void apply_prec_poly(emg_solver *s, const R *x, const double *xs, R *out, hipStream_t st) {
    if constexpr (sizeof(R) == 4)
        if (s->fused) {
            apply_fused(s, x, xs, out, false, st);
            return;
        }
    if (s->poly_deg <= 1) {
        apply_prec<R>(s, x, xs, out, st);
        return;
    }
    R *pp = reinterpret_cast<R *>(s->pp), *py = reinterpret_cast<R *>(s->py), *pu = reinterpret_cast<R *>(s->pu);
    for (int i = 0; i < s->poly_deg - 1; i++) {
        const R *q = i == 0 ? x : pp;
        const double *qs = i == 0 ? xs : nullptr;
        apply_prec<R>(s, q, qs, pu, st);
        spmv_pk<R, SP_POLY, false>(s, s->lanes[sizeof(R) == 4], pu, sp_args<R>{q, py, pp, s->poly_c, i, qs}, st);
    }
    apply_prec<R>(s, py, nullptr, out, st);
}

// out = K M p(K M) (xs vt) or, with product false, M p(K M) (xs vt) through the fused steps (complex64): a launch
// to start and one per product.
static constexpr int FUSE_L = 16, FUSE_LN = 32;
static void apply_fused(emg_solver *s, const float *vt, const double *xs, float *out, bool product, hipStream_t st) {
    const int64_t ne = s->n_ent, np2 = s->np2;
    fuse_mat f{ne, np2, s->rowptr, s->acol, static_cast<const float *>(s->kre), static_cast<const float *>(s->kim), s->row_flag,
               s->kg_ptr, s->kg_col, s->h_ptr, s->h_col, s->hg_ptr, s->hg_col,
               static_cast<const float *>(s->kg_val), static_cast<const float *>(s->h_val), static_cast<const float *>(s->hg_val),
               s->inv32, s->dsinv32, s->fuse_s, s->fuse_s + 2 * np2};
    float *pp = reinterpret_cast<float *>(s->pp), *py = reinterpret_cast<float *>(s->py);
    float *yl[2] = {reinterpret_cast<float *>(s->pu), reinterpret_cast<float *>(s->pu) + 2 * s->n};
    float *t[2] = {s->fuse_t, s->fuse_t + 2 * np2};
    const unsigned eb = emg::grid_for(ne, 256);
    k_fuse_start<<<eb + emg::grid_for(np2 * 16, 256), 256, 0, st>>>(f, eb, s->gt_prp, s->gt_pcol, static_cast<const float *>(s->gt_pval),
                                                                   vt, xs, yl[0], t[0]);
    const int d = std::max(1, s->poly_deg);
    const unsigned el = emg::grid_for(ne * FUSE_L, 256), nl = emg::grid_for(np2 * FUSE_LN, 256);
    for (int i = 0; i < d - 1; i++) {
        fuse_args a{i == 0 ? vt : pp, yl[i & 1], t[i & 1], py, pp, yl[(i + 1) & 1], t[(i + 1) & 1], s->poly_c, i == 0 ? xs : nullptr,
                    i, i == d - 2};
        k_fuse_step<FUSE_L, FUSE_LN, false><<<el + nl, 256, 0, st>>>(f, el, a);
    }
    const float *ye = yl[(d - 1) & 1], *te = t[(d - 1) & 1];
    if (product) {
        fuse_args a{nullptr, ye, te, out, nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0};
        k_fuse_step<FUSE_L, FUSE_LN, true><<<el, 256, 0, st>>>(f, el, a);
    } else {
        k_bj_grad_pk<float><<<emg::grid_for(ne, RB), RB, 0, st>>>(ne, nullptr, ye, nullptr, s->g_sh, s->g_pcol,
                                                                  static_cast<const float *>(s->g_pval), te, out);
    }
}

// Blocks per tile of the multi-dot: about 2048 blocks in total, so each block
// streams many rows and the per-block reduction is amortised.
static int mdot_blocks(int64_t n, int nv) {
    const int ntile = (nv + DT - 1) / DT;
    const int64_t cap = std::max<int64_t>(64, 2048 / ntile);
    return (int)std::max<int64_t>(1, std::min<int64_t>({(n / 2 + RB - 1) / RB, 1024, cap}));
}

// Offsets (in doubles) into the device Arnoldi state for m steps.
struct arn_off {
    int64_t H, cs, sn, g, fin, res, sc, qp, kept, total;
    explicit arn_off(int m) {
        H = 0;                                  // column t at 2 t (m + 1), rows 0 .. t
        cs = 2 * (int64_t)m * (m + 1);
        sn = cs + 2 * m;
        g = sn + 2 * m;                         // m + 1 complex
        fin = g + 2 * (m + 1);                  // g[t] as step t leaves it, m complex
        res = fin + 2 * m;                      // |g[t+1]| after step t
        sc = res + m;                           // sc[j]: basis vector j is sc[j] V_j
        qp = sc + m + 1;                        // outside directions of the kept cycles, m + 1 complex,
        kept = qp + 2 * (m + 1);                // then the kept_dev that says where they are (one upload)
        total = kept + sizeof(kept_dev) / sizeof(double) + 1;
    }
};
// Offsets (in doubles) into the pinned host memory: what k_arn_report and others tell the host (a
// cycle's end needs no copies), then the staging of small uploads.
struct host_off {
    int64_t H, cs, sn, g, sc, res, h0, norm, y, qp, kept, total;
    explicit host_off(int m) {
        H = 0;                                  // as arn_off
        cs = 2 * (int64_t)m * (m + 1);
        sn = cs + 2 * m;
        g = sn + 2 * m;
        sc = g + 2 * (m + 1);
        res = sc + m + 1;                       // |g[t+1]| after step t
        h0 = res + m;                           // coefficients of a cycle's start vector in the kept spaces
        norm = h0 + 2 * (m + 1);                // squared norms
        y = norm + 2;
        qp = y + 2 * (m + 1);
        kept = qp + 2 * (m + 1);                // right behind qp, as on the device
        total = kept + sizeof(kept_dev) / sizeof(double) + 1;
    }
};
// Arnoldi steps between two looks of the host at the residual estimates.  A look costs about 20 us
// and a cycle of about 40 steps overruns its end by half a chunk on average, so the best length is
// about sqrt(1600 us / step): a step takes 0.1 ms at 20,000 DOFs and over 1 ms at a million.
static int chunk_it(int64_t n) { return n < 400000 ? 4 : 2; }

// Sets *bad when the CSR is not on an entity pattern (the layout k_spmv_blk and
// the smoother rely on): rows (0, e) and (1, e) list the same column entities
// c_j < ne, the (1, c_j) entries of a row follow its (0, c_j) entries, and row
// (1, e) starts half = nnz / 2 entries after row (0, e).
__global__ void __launch_bounds__(256) k_check_entity_pattern(int64_t ne, int64_t nnz,
                                                              const int32_t *__restrict__ rowptr,
                                                              const int32_t *__restrict__ cols, int *bad) {
    const int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (e > ne) return;
    const int64_t half = nnz / 2;
    if (e == ne) {
        if (rowptr[0] != 0 || rowptr[ne] != half || rowptr[2 * ne] != nnz || (nnz & 1)) atomicOr(bad, 1);
        return;
    }
    const int64_t r0 = rowptr[e], r1 = rowptr[e + 1];
    if (r1 < r0 || r1 > half || ((r1 - r0) & 1) || rowptr[ne + e] != r0 + half || rowptr[ne + e + 1] != r1 + half) {
        atomicOr(bad, 1);
        return;
    }
    const int64_t deg = (r1 - r0) / 2;
    for (int64_t j = 0; j < deg; j++) {
        const int32_t c = cols[r0 + j];
        if (c < 0 || c >= ne || cols[r0 + deg + j] != c + ne || cols[half + r0 + j] != c ||
            cols[half + r0 + deg + j] != c + ne) {
            atomicOr(bad, 1);
            return;
        }
    }
}

// Device memory; NO_MEMORY where there is none, for callers that can do with less (the C entries return -2).
static constexpr int NO_MEMORY = -4;
template <typename T>
static int device_alloc(T **p, size_t bytes) {
    const hipError_t e = hipMalloc((void **)p, bytes);
    if (e == hipSuccess) return 0;
    *p = nullptr;
    emg::set_error(std::string("emg_solver: hipMalloc: ") + hipGetErrorString(e));
    if (e != hipErrorOutOfMemory) return -2;
    (void)hipGetLastError();
    return NO_MEMORY;
}

// off[i] = sum of cnt[0 .. i) for i <= n, through the host (once per solver or gradient)
static int prefix_on_host(const int32_t *d_cnt, int64_t n, int32_t **d_off, int64_t *total, hipStream_t st) {
    std::vector<int32_t> c, o;
    if (int rc = emg::host_zeros(c, n)) return rc;
    if (int rc = emg::host_zeros(o, n + 1)) return rc;
    EMG_HIP(hipMemcpyAsync(c.data(), d_cnt, n * sizeof(int32_t), hipMemcpyDeviceToHost, st));
    EMG_HIP(hipStreamSynchronize(st));
    int64_t t = 0;
    for (int64_t i = 0; i < n; i++) {
        t += c[i];
        EMG_CHECK(t < ((int64_t)1 << 31), "emg_solver: too many entries");
        o[i + 1] = (int32_t)t;
    }
    if (int rc = device_alloc(d_off, (n + 1) * sizeof(int32_t))) return rc;
    EMG_HIP(hipMemcpyAsync(*d_off, o.data(), (n + 1) * sizeof(int32_t), hipMemcpyHostToDevice, st));
    EMG_HIP(hipStreamSynchronize(st));
    *total = t;
    return 0;
}

// Where products take k_spmv_pk's LOC form: with fewer rows its workgroups, 64 rows each, leave CUs idle between
// their gathers and their sums.  Complex64 and complex128 products, air then losses: 250,000 DOFs 12.9 -> 12.0,
// 18.7 -> 20.0, 20.4 -> 18.7 and 29.9 -> 31.2 us, 96,000 DOFs 5.4 -> 4.5, 7.1 -> 7.9, 9.6 -> 7.9 and 13.5 -> 13.0; a solve's
// step at 60,000 DOFs 134 -> 140 us, at 250,000 257 -> 255; above it see k_spmv_pk.  EMG_LOCAL_COLUMNS overrides (0: never,
// else wherever the rows fit).
static constexpr int64_t LOC_MIN_N = 400000;
static int fill_local(emg_solver *s, int32_t *cnt, int64_t nb) {
    int *d_over = reinterpret_cast<int *>(s->flag), over = 0;
    int64_t total = 0;
    EMG_HIP(hipMemset(d_over, 0, sizeof(int)));
    k_loc_columns<<<(unsigned)nb, 512>>>(s->n_ent, s->rowptr, s->acol, nullptr, cnt, nullptr, nullptr, d_over);
    EMG_LAUNCH_CHECK();
    EMG_HIP(hipMemcpy(&over, d_over, sizeof(int), hipMemcpyDeviceToHost));
    if (over) return 0;
    if (int rc = prefix_on_host(cnt, nb, &s->loc_ptr, &total, nullptr)) return rc;
    if (int rc = device_alloc(&s->loc_col, std::max<int64_t>(total, 1) * sizeof(int32_t))) return rc;
    if (int rc = device_alloc(&s->loc_idx, s->nnz / 4 * sizeof(uint16_t))) return rc;
    k_loc_columns<<<(unsigned)nb, 512>>>(s->n_ent, s->rowptr, s->acol, s->loc_ptr, nullptr, s->loc_col, s->loc_idx, d_over);
    EMG_LAUNCH_CHECK();
    EMG_HIP(hipStreamSynchronize(nullptr));
    return 0;
}
// The tables of the LOC form, or none where a workgroup's rows exceed it or the memory does not suffice.
static int local_columns(emg_solver *s) {
    const char *env = getenv("EMG_LOCAL_COLUMNS");
    if (s->acol == nullptr || (env != nullptr ? atoi(env) == 0 : s->n < LOC_MIN_N)) return 0;
    const int64_t nb = (s->n_ent + LOC_ROWS - 1) / LOC_ROWS;
    int32_t *cnt = nullptr;
    int rc = device_alloc(&cnt, nb * sizeof(int32_t));
    if (rc == 0) rc = fill_local(s, cnt, nb);
    (void)hipFree(cnt);
    if (rc != 0) drop_local(s);
    return rc == NO_MEMORY ? 0 : rc;
}

// The solver's device buffers for a basis of s->cap + 1 vectors, with or without (precision 64) a packed copy of K.
static int allocate(emg_solver *s, bool packed) {
    const int64_t n = s->n, nnz = s->nnz;
    const bool c64 = s->precision == 32;
    const size_t es = c64 ? 8 : 16;   // bytes per complex element of the basis
    const int ntile = (s->cap + 1 + DT - 1) / DT;
    int rc = 0;
    auto A = [&](auto **p, size_t bytes) { if (rc == 0) rc = device_alloc(p, bytes); };
    A(&s->V, (size_t)(s->cap + 1) * n * es);
    A(&s->w, n * 16); A(&s->z, n * 16); A(&s->r, n * 16);
    if (!c64) A(&s->d, n * 16);
    A(&s->partial, ((size_t)2 * ntile * 1024 * DT * 2 + 1024) * sizeof(double));
    A(&s->gram, (size_t)(s->cap + 1) * (s->cap + 1) * 16);
    A(&s->h, 4 * 2 * 512 * sizeof(double));   // dots | corrected | the part subtracted | y
    A(&s->inv64, s->n_ent * 4 * 16);
    A(&s->arn, arn_off(s->cap).total * sizeof(double));
    A(&s->pn, 1024 * sizeof(double));
    A(&s->flag, 8 * sizeof(double));
    if (c64) A(&s->inv32, s->n_ent * 4 * 8);
    if (packed) {
        A(&s->acol, (size_t)nnz / 4 * sizeof(int32_t));
        A(&s->kre, (size_t)nnz * es / 2);
        A(&s->kim, (size_t)nnz * es / 2);
    }
    A(&s->row_flag, s->n_ent);
    A(&s->poly_c, 2 * POLY_MAX * sizeof(double));
    A(&s->pp, n * 16); A(&s->py, n * 16); A(&s->pu, n * 16);
    if (rc == 0) s->kept = reinterpret_cast<kept_dev *>(s->arn + arn_off(s->cap).kept);
    return rc;
}

// The planes and row flags of the caller's values and mask as they are now.
static void pack_matrix(emg_solver *s, hipStream_t st) {
    const unsigned gp = (unsigned)((s->n_ent * SUB + 255) / 256);
    if (s->kre == nullptr)
        k_row_flags<<<emg::grid_for(s->n_ent, 256), 256, 0, st>>>(s->n_ent, s->mask, s->row_flag);
    else if (s->precision == 32)
        k_pack_matrix<float><<<gp, 256, 0, st>>>(s->n_ent, s->nnz / 2, s->rowptr, s->acol, s->vals, s->mask,
                                                 static_cast<float *>(s->kre), static_cast<float *>(s->kim), s->row_flag);
    else
        k_pack_matrix<double><<<gp, 256, 0, st>>>(s->n_ent, s->nnz / 2, s->rowptr, s->acol, s->vals, s->mask,
                                                  static_cast<double *>(s->kre), static_cast<double *>(s->kim), s->row_flag);
}

// Gives back what a solver of a full card can do without: the tables of the LOC form, and the longer half of a
// complex64 basis or the packed complex128 copy of K.  False where there is nothing of the kind.  Not during a solve.
static bool give_back(emg_solver *s) {
    const bool copy = s->precision == 64 && s->kre != nullptr, any = s->loc_ptr != nullptr || s->cap > s->restart || copy;
    drop_graphs(s);
    drop_local(s);
    if (copy) drop(s->acol, s->kre, s->kim);   // solves and probes set the row flags anew
    if (s->cap > s->restart) {
        s->cap = s->restart;
        s->kept = reinterpret_cast<kept_dev *>(s->arn + arn_off(s->cap).kept);
        drop(s->V);
        if (device_alloc(&s->V, (size_t)(s->cap + 1) * s->n * 8) != 0) return false;
    }
    return any;
}

extern "C" int emg_solver_create(int64_t n, int64_t nnz, const int32_t *d_rowptr, const int32_t *d_cols, int restart,
                                 int precision, emg_solver **out) {
    EMG_CHECK(out && d_rowptr && d_cols, "emg_solver_create: null argument");
    EMG_CHECK(n > 0 && (n % 2) == 0, "emg_solver_create: n must be 2 * n_entities");
    EMG_CHECK(restart >= 2 && restart <= 500, "emg_solver_create: restart must be in [2, 500]");
    EMG_CHECK(precision == 64 || precision == 32, "emg_solver_create: precision must be 64 or 32");
    auto s = new emg_solver();
    s->n = n; s->nnz = nnz; s->n_ent = n / 2; s->restart = restart; s->precision = precision;
    s->rowptr = d_rowptr; s->cols = d_cols;
    s->nblk = (int)std::min<int64_t>((n / 2 * maxpy_split(n) + RB - 1) / RB, 1024);
    // the blocked SpMV and the 2x2 block smoother need an entity pattern: check it once
    auto refuse = [&](const char *what, hipError_t e) {
        emg::set_error(std::string("emg_solver_create: ") + what + hipGetErrorString(e));
        free_solver(s);
        return -2;
    };
    int bad = nnz <= 0 || nnz >= ((int64_t)1 << 31);
    if (!bad) {
        // complex64 refinement cycles keep up to two restart lengths of basis vectors (gmres_cycle), the
        // bytes of the complex128 basis of one; where the card does not hold everything then, one.  Complex128 steps
        // do without the packed copy of K there (883,652 DOFs: 267 -> 392 us per step, 895 -> 1,642 at degree 6).
        s->cap = precision == 32 ? std::min(2 * restart, 500) : restart;
        const char *env = getenv("EMG_PACKED_MATRIX");
        int rc = precision == 64 && env != nullptr && atoi(env) == 0 ? NO_MEMORY : allocate(s, true);
        if (rc == NO_MEMORY) {
            drop_buffers(s);
            s->cap = restart;
            rc = allocate(s, precision == 32);
        }
        if (rc != 0) {
            free_solver(s);
            return -2;
        }
        hipError_t e = hipHostMalloc((void **)&s->host, host_off(s->cap).total * sizeof(double), hipHostMallocDefault);
        if (e == hipSuccess) e = hipHostGetDevicePointer((void **)&s->host_dev, s->host, 0);
        if (e == hipSuccess) e = hipStreamCreateWithFlags(&s->cap_stream, hipStreamNonBlocking);
        if (e != hipSuccess) return refuse("", e);
        int *d_bad = reinterpret_cast<int *>(s->flag);
        e = hipMemset(d_bad, 0, sizeof(int));
        if (e == hipSuccess) {
            k_check_entity_pattern<<<emg::grid_for(s->n_ent + 1, 256), 256>>>(s->n_ent, nnz, d_rowptr, d_cols, d_bad);
            e = hipGetLastError();
        }
        if (e == hipSuccess) e = hipMemcpy(&bad, d_bad, sizeof(int), hipMemcpyDeviceToHost);
        if (e != hipSuccess) return refuse("pattern check: ", e);
    }
    if (bad) {
        emg::set_error("emg_solver_create: the CSR is not on an entity pattern (emg_pattern_csr layout: rows e and "
                       "e + n/2 share their column entities, mode-1 columns after mode-0 ones, row e + n/2 starting "
                       "nnz/2 after row e); pass the full unreduced matrix and the PEC mask");
        free_solver(s);
        return -1;
    }
    if (s->acol != nullptr)
        k_pack_cols<<<(unsigned)((s->n_ent * SUB + 255) / 256), 256>>>(s->n_ent, d_rowptr, d_cols, s->acol);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipStreamSynchronize(nullptr);
    if (e != hipSuccess) return refuse("packing the pattern: ", e);
    if (int rc = local_columns(s)) {
        free_solver(s);
        return rc;
    }
    *out = s;
    return 0;
}

extern "C" void emg_solver_destroy(emg_solver *s) { free_solver(s); }

// inv blocks of entity e *= w_e[e] (complex64 copy too); dsinv[p] *= w_p[p]
__global__ void __launch_bounds__(RB) k_scale_tables(int64_t n_ent, const double *__restrict__ we, double *__restrict__ inv64,
                                                     float *__restrict__ inv32, int64_t np2, const double *__restrict__ wp,
                                                     double *__restrict__ ds64, float *__restrict__ ds32) {
    const int64_t i = blockIdx.x * (int64_t)RB + threadIdx.x;
    if (we != nullptr && i < n_ent) {
        const double wr = we[2 * i], wi = we[2 * i + 1];
        for (int q = 0; q < 4; q++) {
            double *a = inv64 + 2 * (4 * i + q);
            const double ar = a[0], ai = a[1];
            a[0] = wr * ar - wi * ai;
            a[1] = wr * ai + wi * ar;
            if (inv32) { inv32[2 * (4 * i + q)] = (float)a[0]; inv32[2 * (4 * i + q) + 1] = (float)a[1]; }
        }
    }
    if (wp != nullptr && i < np2) {
        const double wr = wp[2 * i], wi = wp[2 * i + 1];
        double *a = ds64 + 2 * i;
        const double ar = a[0], ai = a[1];
        a[0] = wr * ar - wi * ai;
        a[1] = wr * ai + wi * ar;
        if (ds32) { ds32[2 * i] = (float)a[0]; ds32[2 * i + 1] = (float)a[1]; }
    }
}

// Autotuners: each candidate shape runs eight times in a captured graph between HIP events, after one
// untimed replay, on the solver's first matrix and zeroed work vectors, and the fastest is kept for the
// solver's life.  Before each run goes what precedes it in a step (`lead`, whose own time is measured
// and taken off): launched back to back by itself, a small product finds everything in the L2 it ran
// from, or takes as long as it takes to issue, and all candidates look alike (the G^T product at 3,072
// tets takes 5.5 us with 4 lanes and 4.1 us with 16 in the steps, and was chosen now the one way and now
// the other).
static constexpr int TUNE_RUNS = 8;
template <typename LEAD, typename RUN>
static int tune_lanes(emg_solver *s, int n, const int *cand, LEAD &&lead, RUN &&run, float *ms, int *choice,
                      hipStream_t st) {
    hipEvent_t ev[2];
    EMG_HIP(hipEventCreate(&ev[0]));
    if (hipEventCreate(&ev[1]) != hipSuccess) {
        (void)hipEventDestroy(ev[0]);
        emg::set_error("tune_lanes: hipEventCreate failed");
        return -2;
    }
    hipError_t e = hipSuccess;
    float base = 0.f;
    for (int i = -1; i < n && e == hipSuccess; i++) {   // -1: the lead alone
        hipGraph_t graph = nullptr;
        hipGraphExec_t exec = nullptr;
        float t = 0.f;
        e = hipStreamBeginCapture(s->cap_stream, hipStreamCaptureModeThreadLocal);
        if (e != hipSuccess) break;
        for (int r = 0; r < TUNE_RUNS; r++) {
            lead(s->cap_stream);
            if (i >= 0) run(cand[i], s->cap_stream);
        }
        e = hipStreamEndCapture(s->cap_stream, &graph);
        if (e == hipSuccess) e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
        if (graph != nullptr) (void)hipGraphDestroy(graph);
        if (e == hipSuccess) e = hipGraphLaunch(exec, st);
        if (e == hipSuccess) e = hipEventRecord(ev[0], st);
        if (e == hipSuccess) e = hipGraphLaunch(exec, st);
        if (e == hipSuccess) e = hipEventRecord(ev[1], st);
        if (e == hipSuccess) e = hipEventSynchronize(ev[1]);
        if (e == hipSuccess) e = hipEventElapsedTime(&t, ev[0], ev[1]);
        if (exec != nullptr) (void)hipGraphExecDestroy(exec);
        t /= (float)TUNE_RUNS;
        if (i < 0) base = t; else ms[i] = std::max(t - base, 1e-6f);
    }
    (void)hipEventDestroy(ev[0]);
    (void)hipEventDestroy(ev[1]);
    EMG_HIP(e);
    *choice = cand[std::min_element(ms, ms + n) - ms];
    return 0;
}

// Lanes per entity of the solver's products: complex128 (slot 0: the packed matrix for precision 64,
// the caller's CSR for precision 32) and complex64 (slot 1); EMG_SPMV_BLK_LANES overrides.  Fused solvers run
// the products and the G^T product of their choice once the gradient is taken off (emg_solver_set_gradient, np2 = 0).
static const int TUNE_LANES[4] = {4, 8, 16, 32};
// Lanes per row of the smoother's G^T product; EMG_GT_LANES (4, 8 or 16) overrides.
static const int GT_LANES[3] = {4, 8, 16};

template <typename R>
static int tune_steps(emg_solver *s, hipStream_t st) {
    R *z = reinterpret_cast<R *>(s->z), *pu = reinterpret_cast<R *>(s->pu), *pp = reinterpret_cast<R *>(s->pp);
    const int slot = sizeof(R) == 4;
    EMG_HIP(hipMemsetAsync(z, 0, s->n * 2 * sizeof(R), st));
    auto product = [&](int L, hipStream_t rs) {
        spmv_pk<R, SP_Y, false>(s, L, pu, sp_args<R>{nullptr, pp, nullptr, nullptr, 0, nullptr}, rs);
    };
    if (s->kre == nullptr || s->loc_ptr != nullptr) {   // these forms have one shape
        s->lanes[slot] = s->kre == nullptr ? 16 : LOC_L;
    } else if (getenv("EMG_SPMV_BLK_LANES") != nullptr) {
        s->lanes[slot] = spmv_blk_lanes();
    } else {
        auto smooth = [&](hipStream_t rs) { apply_prec<R>(s, z, nullptr, pu, rs); };
        if (int rc = tune_lanes(s, 4, TUNE_LANES, smooth, product, s->tune_ms[slot], &s->lanes[slot], st)) return rc;
    }
    if (s->np2 <= 0) return 0;
    if (const char *env = getenv("EMG_GT_LANES")) {
        const int v = atoi(env);
        s->gt_lanes = (v == 4 || v == 16) ? v : 8;
        return 0;
    }
    EMG_HIP(hipMemsetAsync(pu, 0, s->n * 2 * sizeof(R), st));
    auto before = [&](hipStream_t rs) { product(s->lanes[slot], rs); };
    auto gt = [&](int L, hipStream_t rs) {
        const R *dsi = slot ? reinterpret_cast<const R *>(s->dsinv32) : reinterpret_cast<const R *>(s->dsinv64);
        launch_gt_pk<R>(rs, L, s->np2, s->gt_prp, s->gt_pcol, static_cast<const R *>(s->gt_pval), dsi, pp, nullptr,
                        reinterpret_cast<R *>(s->tg));
    };
    return tune_lanes(s, 3, GT_LANES, before, gt, s->gt_ms, &s->gt_lanes, st);
}

static int tune_spmv(emg_solver *s, hipStream_t st) {
    if (s->precision == 64) {
        if (int rc = tune_steps<double>(s, st)) return rc;
        s->lanes[1] = s->lanes[0];
        return 0;
    }
    if (getenv("EMG_SPMV_BLK_LANES") != nullptr) {
        s->lanes[0] = spmv_blk_lanes();
    } else {
        EMG_HIP(hipMemsetAsync(s->z, 0, s->n * 16, st));
        EMG_HIP(hipMemsetAsync(s->r, 0, s->n * 16, st));
        auto input = [&](hipStream_t rs) {
            k_pack_vec<double><<<emg::grid_for(s->n_ent, RB), RB, 0, rs>>>(s->n_ent, s->r, 1.0, s->z);
        };
        auto csr = [&](int L, hipStream_t rs) {
            launch_spmv_blk(rs, s->n, s->nnz, s->rowptr, s->cols, s->vals, s->mask, s->z, nullptr, s->pp, L);
        };
        if (int rc = tune_lanes(s, 4, TUNE_LANES, input, csr, s->tune_ms[0], &s->lanes[0], st)) return rc;
    }
    return tune_steps<float>(s, st);
}

extern "C" int emg_solver_smoother_tuning(emg_solver *s, int *h_lanes, float *h_ms) {
    EMG_CHECK(s && h_lanes && h_ms, "emg_solver_smoother_tuning: null argument");
    *h_lanes = s->gt_lanes;
    for (int i = 0; i < 3; i++) h_ms[i] = s->gt_ms[i];
    return 0;
}

extern "C" int emg_solver_spmv_tuning(emg_solver *s, int *h_lanes, float *h_ms) {
    EMG_CHECK(s && h_lanes && h_ms, "emg_solver_spmv_tuning: null argument");
    for (int p = 0; p < 2; p++) {
        h_lanes[p] = s->lanes[p];
        for (int i = 0; i < 4; i++) h_ms[4 * p + i] = s->tune_ms[p][i];
    }
    return 0;
}

extern "C" int emg_solver_set_matrix(emg_solver *s, const double *d_vals, const uint8_t *d_mask, void *stream) {
    EMG_CHECK(s && d_vals, "emg_solver_set_matrix: null argument");
    hipStream_t st = (hipStream_t)stream;
    s->vals = d_vals;
    s->mask = d_mask;
    k_bj_setup<<<emg::grid_for(s->n_ent, RB), RB, 0, st>>>(s->n_ent, s->rowptr, s->cols, d_vals, d_mask, s->inv64, s->inv32);
    pack_matrix(s, st);
    if (s->np2 > 0) {
        EMG_HIP(hipMemsetAsync(s->dS, 0, s->np2 * 16, st));
        k_gdiag<<<emg::grid_for(s->n * GD, RB), RB, 0, st>>>(s->n, s->rowptr, s->cols, d_vals, d_mask, s->g_rowptr,
                                                         s->g_cols, s->g_vals, s->dS);
        k_dsinv<<<emg::grid_for(s->np2, RB), RB, 0, st>>>(s->np2, s->dS, s->dsinv64, s->dsinv32);
    }
    if (s->fused) {
        const int64_t ne = s->n_ent, half = s->nnz / 2;
        float *kgv = static_cast<float *>(s->kg_val);
        k_kg_values<<<(unsigned)ne, 64, 0, st>>>(ne, half, s->rowptr, s->acol, d_vals, d_mask, s->g_rowptr, s->g_cols, s->g_vals,
                                                 s->kg_ptr, s->kg_col, kgv);
        k_node_values<false><<<(unsigned)s->np2, 64, 0, st>>>(ne, half, s->rowptr, s->acol, d_vals, d_mask, s->kg_ptr, s->kg_col, kgv,
                                                              s->gt_rowptr, s->gt_cols, s->gt_vals, s->h_ptr, s->h_col,
                                                              static_cast<float *>(s->h_val));
        k_node_values<true><<<(unsigned)s->np2, 64, 0, st>>>(ne, half, s->rowptr, s->acol, d_vals, d_mask, s->kg_ptr, s->kg_col, kgv,
                                                             s->gt_rowptr, s->gt_cols, s->gt_vals, s->hg_ptr, s->hg_col,
                                                             static_cast<float *>(s->hg_val));
    }
    if (s->w_e != nullptr || (s->w_p != nullptr && s->np2 > 0)) {
        const int64_t nmax = std::max<int64_t>(s->n_ent, s->np2);
        k_scale_tables<<<emg::grid_for(nmax, RB), RB, 0, st>>>(s->n_ent, s->w_e, s->inv64, s->inv32, s->np2,
                                                               s->np2 > 0 ? s->w_p : nullptr, s->dsinv64, s->dsinv32);
    }
    EMG_LAUNCH_CHECK();
    if (s->lanes[0] == 0) {
        const int rc = tune_spmv(s, st);
        if (rc) return rc;
    }
    return 0;
}

extern "C" int emg_solver_set_weights(emg_solver *s, const double *d_we, const double *d_wp) {
    EMG_CHECK(s != nullptr, "emg_solver_set_weights: null solver");
    s->w_e = d_we;
    s->w_p = d_wp;
    return 0;
}

// The two parts of the smoother for a vector r (complex128): u = BJ(r) (n) and,
// with the gradient correction set, t = diag(G^T K G)^{-1} G^T r (np2).
extern "C" int emg_solver_smoother_parts(emg_solver *s, const double *d_r, double *d_u, double *d_t, void *stream) {
    EMG_CHECK(s && d_r && d_u, "emg_solver_smoother_parts: null argument");
    hipStream_t st = (hipStream_t)stream;
    k_bj_apply<<<emg::grid_for(s->n_ent, RB), RB, 0, st>>>(s->n_ent, s->inv64, d_r, d_u);
    if (s->np2 > 0 && d_t != nullptr)
        launch_gt(st, s->np2, s->gt_rowptr, s->gt_cols, s->gt_vals, s->dsinv64, d_r, d_t);
    EMG_LAUNCH_CHECK();
    return 0;
}

// Polynomial of the preconditioner: degree d (1 = none) and its coefficients
// c_i = 1/theta_i (complex128, host array of 2 d doubles) in application order.
extern "C" int emg_solver_set_poly(emg_solver *s, int degree, const double *h_coef) {
    EMG_CHECK(s != nullptr, "emg_solver_set_poly: null solver");
    EMG_CHECK(degree >= 1 && degree <= POLY_MAX, "emg_solver_set_poly: degree must be in [1, 16]");
    EMG_CHECK(degree == 1 || h_coef != nullptr, "emg_solver_set_poly: null coefficients");
    if (degree > 1) {
        for (int i = 0; i < 2 * degree; i++)
            EMG_CHECK(std::isfinite(h_coef[i]), "emg_solver_set_poly: non-finite coefficient");
        EMG_HIP(hipMemcpy(s->poly_c, h_coef, 2 * degree * sizeof(double), hipMemcpyHostToDevice));
    }
    s->poly_deg = degree;
    return 0;
}

// d steps of Arnoldi (complex128, two classical Gram-Schmidt passes) on K M
// (M = the smoother without polynomial, K masked) from d_v0; writes the
// (d + 1) x d Hessenberg matrix column-major as complex128 to h_out (host).
// Uses the solver's Krylov basis storage, so it must not run during a solve.
extern "C" int emg_solver_arnoldi_probe(emg_solver *s, int d, const double *d_v0, double *h_out, void *stream) {
    EMG_CHECK(s && d_v0 && h_out, "emg_solver_arnoldi_probe: null argument");
    EMG_CHECK(s->vals != nullptr, "emg_solver_arnoldi_probe: emg_solver_set_matrix was not called");
    EMG_CHECK(s->V != nullptr, "emg_solver_arnoldi_probe: no memory for the basis");
    const int64_t n = s->n;
    const size_t es = s->precision == 64 ? 16 : 8;
    EMG_CHECK(d >= 1 && d <= POLY_MAX && (size_t)(d + 1) * 16 <= (size_t)(s->restart + 1) * es,
              "emg_solver_arnoldi_probe: d out of range for this solver");
    hipStream_t st = (hipStream_t)stream;
    const int nb = s->nblk;
    double *V = s->V;   // d + 1 complex128 vectors
    double *z = s->z;
    // Everything stays on the device until the end (two waits per pass took a third of the probe's time at
    // 20,000 DOFs): norms, then the coefficients of pass 0 and 1 of every column.
    constexpr int PROBE_H = POLY_MAX + 2;   // POLY_MAX + 1 norms
    static_assert(PROBE_H % 2 == 0 && PROBE_H + 4 * POLY_MAX * (POLY_MAX + 1) <= 4 * 2 * 512, "the probe's results fit s->h");
    double *norms = s->h, *coef = s->h + PROBE_H;
    if (s->precision == 64) pack_matrix(s, st);   // the caller's values as they are now, as in a solve
    const int ldc = 2 * (d + 1);
    EMG_HIP(hipMemcpyAsync(V, d_v0, n * 16, hipMemcpyDeviceToDevice, st));
    k_norm2<double><<<nb, RB, 0, st>>>(n, V, s->partial);
    k_scale_by_norm<double><<<nb, RB, 0, st>>>(n, s->partial, nb, V, V, norms);
    for (int j = 0; j < d; j++) {
        double *vj = V + (size_t)j * n * 2, *w = V + (size_t)(j + 1) * n * 2;
        const int nv = j + 1, nbm = mdot_blocks(n, nv);
        const dim3 grid(nbm, (nv + DT - 1) / DT);
        apply_prec_std(s, vj, z, st);
        spmv_std(s, z, nullptr, w, st);
        for (int pass = 0; pass < 2; pass++) {
            double *h = coef + (2 * j + pass) * ldc;
            k_mdot<double, 1><<<grid, RB, 0, st>>>(n, nv, V, n, w, nullptr, s->partial);
            k_mdot_finish<<<nv, 256, 0, st>>>(nv, nbm, s->partial, nullptr, h, nullptr, 0);
            launch_maxpy<double>(st, nb, n, nv, V, h, nullptr, w, s->pn);
        }
        k_scale_by_norm<double><<<nb, RB, 0, st>>>(n, s->pn, nb, w, w, norms + j + 1);
    }
    EMG_LAUNCH_CHECK();
    std::vector<double> got(PROBE_H + (size_t)2 * d * ldc), H(2 * (size_t)(d + 1) * d, 0.0);
    EMG_HIP(hipMemcpyAsync(got.data(), s->h, got.size() * sizeof(double), hipMemcpyDeviceToHost, st));
    EMG_HIP(hipStreamSynchronize(st));
    EMG_CHECK(got[0] > 0 && std::isfinite(got[0]), "emg_solver_arnoldi_probe: zero or non-finite start vector");
    for (int j = 0; j < d; j++) {
        const double *h = got.data() + PROBE_H + (size_t)2 * j * ldc, wn = got[j + 1];
        EMG_CHECK(wn > 0 && std::isfinite(wn), "emg_solver_arnoldi_probe: breakdown");
        for (int i = 0; i < 2 * (j + 1); i++) H[(size_t)2 * j * (d + 1) + i] = h[i] + h[ldc + i];
        H[2 * ((size_t)j * (d + 1) + j + 1)] = wn;
    }
    memcpy(h_out, H.data(), H.size() * sizeof(double));
    return 0;
}

template <typename R>
static int pack_gradient(emg_solver *s, int64_t np2, const int32_t *grp, const int32_t *gcol, const double *gv,
                         const int32_t *tp, const int32_t *tcol, const double *tv, int32_t *cnt, hipStream_t st) {
    const int64_t ne = s->n_ent, ns = (ne + 63) / 64;
    int64_t total = 0;
    k_g_width<<<(unsigned)ns, 64, 0, st>>>(ne, grp, gcol, cnt);
    EMG_LAUNCH_CHECK();
    // the cut between two runs of slices, each as wide as its widest, that leaves the fewest slots
    std::vector<int32_t> wd, after_max;
    if (int rc = emg::host_zeros(wd, ns)) return rc;
    if (int rc = emg::host_zeros(after_max, ns + 1)) return rc;
    EMG_HIP(hipMemcpyAsync(wd.data(), cnt, ns * sizeof(int32_t), hipMemcpyDeviceToHost, st));
    EMG_HIP(hipStreamSynchronize(st));
    for (int64_t i = ns - 1; i >= 0; i--) after_max[i] = std::max(after_max[i + 1], wd[i]);
    int64_t best = INT64_MAX;
    int32_t before_max = 0;
    for (int64_t c = 0; c <= ns; c++) {
        const int64_t size = c * before_max + (ns - c) * after_max[c];
        if (size < best) { best = size; s->g_sh = g_shape{c, before_max, after_max[c]}; }
        if (c < ns) before_max = std::max(before_max, wd[c]);
    }
    const int64_t slots = std::max<int64_t>(s->g_sh.first(ns), 1);
    if (int rc = device_alloc(&s->g_pcol, slots * sizeof(int32_t))) return rc;
    if (int rc = device_alloc(&s->g_pval, slots * 2 * sizeof(R))) return rc;
    k_g_fill<R><<<(unsigned)ns, 64, 0, st>>>(ne, grp, gcol, gv, s->g_sh, s->g_pcol, static_cast<R *>(s->g_pval));
    k_gt_count<<<emg::grid_for(np2, RB), RB, 0, st>>>(np2, ne, tp, tcol, cnt);
    EMG_LAUNCH_CHECK();
    if (int rc = prefix_on_host(cnt, np2, &s->gt_prp, &total, st)) return rc;
    if (int rc = device_alloc(&s->gt_pcol, std::max<int64_t>(total, 1) * sizeof(int32_t))) return rc;
    if (int rc = device_alloc(&s->gt_pval, std::max<int64_t>(total, 1) * 2 * sizeof(R))) return rc;
    k_gt_fill<R><<<emg::grid_for(np2, RB), RB, 0, st>>>(np2, ne, tp, tcol, tv, s->gt_prp, s->gt_pcol,
                                                        static_cast<R *>(s->gt_pval));
    EMG_LAUNCH_CHECK();
    return 0;
}

// The patterns of KG, H and HG and room for their values: *fits false (and nothing kept) where a row is too long
// or the memory does not suffice.
template <typename GEN>
static int fuse_rows(int64_t rows, const GEN &gen, int32_t *cnt, int *d_over, int32_t **ptr, int32_t **col, void **val,
                     size_t bytes, bool *fits, hipStream_t st) {
    EMG_HIP(hipMemsetAsync(d_over, 0, sizeof(int), st));
    k_distinct<<<(unsigned)rows, 256, 0, st>>>(gen, cnt, nullptr, nullptr, d_over);
    EMG_LAUNCH_CHECK();
    int over = 0;
    EMG_HIP(hipMemcpyAsync(&over, d_over, sizeof(int), hipMemcpyDeviceToHost, st));
    int64_t total = 0;
    EMG_HIP(hipStreamSynchronize(st));
    if (over) { *fits = false; return 0; }
    int rc = prefix_on_host(cnt, rows, ptr, &total, st);
    if (rc == 0 && total > 0) rc = device_alloc(col, total * sizeof(int32_t));
    if (rc == 0 && total > 0) rc = device_alloc(val, total * bytes);
    // too many entries, no memory, or none (the steps read slot 0 in place of a missing one)
    if (rc == -1 || rc == NO_MEMORY || (rc == 0 && total == 0)) { *fits = false; return 0; }
    if (rc != 0) return rc;
    k_distinct<<<(unsigned)rows, 256, 0, st>>>(gen, nullptr, *ptr, *col, d_over);
    EMG_LAUNCH_CHECK();
    return 0;
}
static int fuse_pattern(emg_solver *s, int64_t np2, const int32_t *grp, const int32_t *gcol, const int32_t *trp, const int32_t *tcol,
                        int32_t *cnt, hipStream_t st) {
    int *d_over = reinterpret_cast<int *>(s->flag);
    bool fits = true;
    int rc = fuse_rows(s->n_ent, gen_kg{s->n_ent, s->rowptr, s->acol, grp, gcol}, cnt, d_over, &s->kg_ptr, &s->kg_col, &s->kg_val, 16,
                       &fits, st);
    if (rc == 0 && fits)
        rc = fuse_rows(np2, gen_of_nodes{s->n_ent, trp, tcol, s->rowptr, s->acol, 1}, cnt, d_over, &s->h_ptr, &s->h_col, &s->h_val, 16,
                       &fits, st);
    if (rc == 0 && fits)
        rc = fuse_rows(np2, gen_of_nodes{s->n_ent, trp, tcol, s->kg_ptr, s->kg_col, 0}, cnt, d_over, &s->hg_ptr, &s->hg_col, &s->hg_val,
                       8, &fits, st);
    if (rc == 0 && fits) {
        rc = device_alloc(&s->fuse_s, (size_t)np2 * 32);
        if (rc == 0) rc = device_alloc(&s->fuse_t, (size_t)np2 * 16);
        if (rc == NO_MEMORY) { rc = 0; fits = false; }
    }
    if (rc == 0 && fits) s->fused = true;
    if (rc != 0 || !fits) {
        (void)hipStreamSynchronize(st);
        drop_fused(s);
    }
    return rc;
}

// Where the fused steps are used.  KG, H and HG hold about as many bytes as K, so steps are faster while a launch
// costs more than its bytes: posts box at 20,000 / 34,000 / 58,424 / 71,896 / 94,092 DOFs, air, degree 6: 124 -> 90, 123 -> 99,
// 133 -> 122, 140 -> 140, 153 -> 165 us; lossy 124 -> 90, 130 -> 100, 142 -> 130, 152 -> 146, 168 -> 173.  The line lies
// below where they cross, because the patterns are set up once (create and first matrix) and the values formed for every
// matrix: a frequency point (matrix and one solve) takes 10.3 -> 9.4 ms at 49,414 DOFs on air for 3.0 ms of set-up,
// and 10.7 -> 10.4 at 58,424 for 4.9, which 17 points would earn; 12.4 -> 13.0 at 71,896.
// Complex64 only: complex128 steps are mostly above it.  EMG_FUSED_STEPS overrides (0: never, else wherever the rows fit).
static constexpr int64_t FUSE_MAX_N = 50000;
static bool fuse_wanted(const emg_solver *s) {
    if (s->precision != 32) return false;
    if (const char *env = getenv("EMG_FUSED_STEPS")) return atoi(env) != 0;
    return s->n <= FUSE_MAX_N;
}

extern "C" int emg_solver_set_gradient(emg_solver *s, int64_t np2, const int32_t *d_g_rowptr, const int32_t *d_g_cols,
                                       const double *d_g_vals, const int32_t *d_gt_rowptr, const int32_t *d_gt_cols,
                                       const double *d_gt_vals, void *stream) {
    EMG_CHECK(s != nullptr && np2 >= 0, "emg_solver_set_gradient: bad argument");
    hipStream_t st = (hipStream_t)stream;
    if (np2 == 0) {
        s->np2 = 0;
        s->fused = false;
        return 0;
    }
    EMG_CHECK(d_g_rowptr && d_g_cols && d_g_vals && d_gt_rowptr && d_gt_cols && d_gt_vals,
              "emg_solver_set_gradient: null argument");
    int32_t nnz_g = 0, nnz_gt = 0;
    EMG_HIP(hipMemcpyAsync(&nnz_g, d_g_rowptr + s->n, sizeof(int32_t), hipMemcpyDeviceToHost, st));
    EMG_HIP(hipMemcpyAsync(&nnz_gt, d_gt_rowptr + np2, sizeof(int32_t), hipMemcpyDeviceToHost, st));
    EMG_HIP(hipStreamSynchronize(st));
    EMG_CHECK(nnz_g == nnz_gt && nnz_g > 0, "emg_solver_set_gradient: G and G^T entry counts differ");
    EMG_CHECK(nnz_g <= G_ROW_MAX * s->n, "emg_solver_set_gradient: more than 8 entries per row of G");
    // captured step graphs hold the old gradient buffers: drop them before the buffers go
    EMG_HIP(hipStreamSynchronize(st));
    drop_graphs(s);
    auto make = [&]() {
        drop_gradient(s);
        s->np2 = 0;
        const bool fuse = fuse_wanted(s);
        int32_t *cnt = nullptr;
        int rc = device_alloc(&s->dS, (size_t)np2 * 16);
        if (rc == 0) rc = device_alloc(&s->dsinv64, (size_t)np2 * 16);
        if (rc == 0) rc = device_alloc(&s->dsinv32, (size_t)np2 * 8);
        if (rc == 0) rc = device_alloc(&s->tg, (size_t)np2 * 16);
        if (rc == 0) rc = device_alloc(&cnt, std::max<int64_t>(np2, fuse ? s->n_ent : s->n_ent / 64 + 1) * sizeof(int32_t));
        if (rc == 0)
            rc = s->precision == 32 ? pack_gradient<float>(s, np2, d_g_rowptr, d_g_cols, d_g_vals, d_gt_rowptr, d_gt_cols,
                                                           d_gt_vals, cnt, st)
                                    : pack_gradient<double>(s, np2, d_g_rowptr, d_g_cols, d_g_vals, d_gt_rowptr, d_gt_cols,
                                                            d_gt_vals, cnt, st);
        if (rc == 0 && fuse) rc = fuse_pattern(s, np2, d_g_rowptr, d_g_cols, d_gt_rowptr, d_gt_cols, cnt, st);
        const hipError_t e = hipStreamSynchronize(st);   // cnt is read by kernels in flight
        (void)hipFree(cnt);
        if (rc) return rc;
        EMG_HIP(e);
        return 0;
    };
    int rc = make();
    if (rc == NO_MEMORY && give_back(s)) rc = make();
    if (rc != 0) return rc == NO_MEMORY ? -2 : rc;
    s->g_rowptr = d_g_rowptr; s->g_cols = d_g_cols; s->g_vals = d_g_vals;
    s->gt_rowptr = d_gt_rowptr; s->gt_cols = d_gt_cols; s->gt_vals = d_gt_vals;
    s->np2 = np2;
    return 0;
}

// ---------------------------------------------------------------- device Arnoldi bookkeeping
// A cycle whose first basis vector is V_t0 = w: g[t0] = ||w|| from its nb partial sums, and the scale 1 / ||w||.
// Like every basis vector it is kept as it is with that scale beside it: normalised in complex64 its norm would be
// off by the rounding, which the Gram matrix' diagonal (0 deviation) does not hold, and where the next vector
// is all but cancelled (K M near the identity) that much of w stays in it: the bases of later cycles
// were no longer orthogonal and one of them ran to the end of the restart without a gain.
template <typename R>
__global__ void __launch_bounds__(RB) k_arn_start(int64_t n, int t0, int nb, const double *__restrict__ pn,
                                                  const R *__restrict__ w, R *__restrict__ vt, double *__restrict__ arn,
                                                  arn_off o) {
    for (int64_t e = blockIdx.x * (int64_t)RB + threadIdx.x; e < n; e += (int64_t)gridDim.x * RB) st(vt, e, ld(w, e));
    if (blockIdx.x != 0) return;
    __shared__ double sh[RB / 64];
    double a = 0.0;
    for (int i = threadIdx.x; i < nb; i += RB) a += pn[i];
    a = block_sum(a, sh);
    if (threadIdx.x == 0) {
        const double beta = sqrt(a);
        arn[o.g + 2 * t0] = beta;
        arn[o.g + 2 * t0 + 1] = 0.0;
        arn[o.sc + t0] = beta > 0.0 ? 1.0 / beta : 0.0;
    }
}

// out = sum of nb partial sums (one block)
__global__ void __launch_bounds__(RB) k_sum_partials(int nb, const double *__restrict__ p, double *__restrict__ out) {
    __shared__ double sh[RB / 64];
    double a = 0.0;
    for (int i = threadIdx.x; i < nb; i += RB) a += p[i];
    a = block_sum(a, sh);
    if (threadIdx.x == 0) *out = a;
}

// x -> a x + b, complex: the maps whose composition carries a column through the rotations
struct affine {
    cx<double> a, b;
};
__device__ __forceinline__ affine after(const affine &l, const affine &e) {   // l after e
    return affine{cmul(l.a, e.a), cadd(cmul(l.a, e.b), l.b)};
}
__device__ __forceinline__ affine shfl_up(const affine &v, int off) {
    return affine{cx<double>(__shfl_up(v.a.re, off, 64), __shfl_up(v.a.im, off, 64)),
                  cx<double>(__shfl_up(v.b.re, off, 64), __shfl_up(v.b.im, off, 64))};
}

// Step t of the cycle that began at basis vector t0: the column h with ||new vector||; rows below t0 (the kept spaces) are stored as they are, the rows of
// the cycle after the previous rotations; then the new rotation, the update of g, the residual
// estimate |g[t+1]| and the new vector's scale 1 / norm.
// The rotations carry x_{i+1} = -s_i x_i + c_i y_{i+1} down the column: a chain of maps x -> a x + b,
// composed by a scan over the block, two per lane (all |s_i| <= 1: the compositions stay bounded).
// One lane walking the chain took 70 ns a rotation, 4.8 us a step on average at 31 steps per cycle.
__global__ void __launch_bounds__(RB) k_arn_givens(int t, int m, int nb, const double *__restrict__ pn,
                                                   const double *__restrict__ h, const kept_dev *__restrict__ kept,
                                                   double *__restrict__ arn, arn_off o) {
    __shared__ double sh[RB / 64];
    __shared__ double tot[RB / 64][4];
    static_assert(2 * RB >= 512, "two rotations per lane cover the longest restart");
    const int t0 = kept->t0, j = t - t0;   // j rotations
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    double *Hc = arn + o.H + 2 * (int64_t)t * (m + 1);
    double *cs = arn + o.cs + 2 * t0, *sn = arn + o.sn + 2 * t0, *g = arn + o.g;
    auto col = [&](int i) { return ld(h, i); };   // row i of the column, of all basis vectors
    double a = 0.0;
    for (int i = threadIdx.x; i < nb; i += RB) a += pn[i];
    for (int i = threadIdx.x; i < t0; i += RB) {
        const cx<double> v = col(i);
        Hc[2 * i] = v.re;
        Hc[2 * i + 1] = v.im;
    }
    cx<double> c[2], s[2], y[2];
    affine f[2];
#pragma unroll
    for (int q = 0; q < 2; q++) {
        const int i = 2 * threadIdx.x + q;
        f[q] = affine{cx<double>(1.0, 0.0), cx<double>()};
        if (i < j) {
            c[q] = cx<double>(cs[2 * i], cs[2 * i + 1]);
            s[q] = cx<double>(sn[2 * i], sn[2 * i + 1]);
            y[q] = col(t0 + i + 1);
            f[q] = affine{cx<double>(-s[q].re, -s[q].im), cmul(c[q], y[q])};
        }
    }
    const cx<double> x0 = col(t0), g0(g[2 * t], g[2 * t + 1]);
    affine v = after(f[1], f[0]);
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const affine u = shfl_up(v, off);
        if (lane >= off) v = after(v, u);
    }
    if (lane == 63) { tot[wave][0] = v.a.re; tot[wave][1] = v.a.im; tot[wave][2] = v.b.re; tot[wave][3] = v.b.im; }
    affine before = shfl_up(v, 1);
    if (lane == 0) before = affine{cx<double>(1.0, 0.0), cx<double>()};
    a = block_sum(a, sh);          // contains __syncthreads: tot is visible after it
    cx<double> x = x0, last = x0;
    for (int w = 0; w < RB / 64; w++) {
        last = cadd(cmul(cx<double>(tot[w][0], tot[w][1]), last), cx<double>(tot[w][2], tot[w][3]));
        if (w + 1 == wave) x = last;
    }
    x = cadd(cmul(before.a, x), before.b);
#pragma unroll
    for (int q = 0; q < 2; q++) {
        const int i = 2 * threadIdx.x + q;
        if (i < j) {   // conj(c) x + conj(s) y
            Hc[2 * (t0 + i)] = c[q].re * x.re + c[q].im * x.im + s[q].re * y[q].re + s[q].im * y[q].im;
            Hc[2 * (t0 + i) + 1] = c[q].re * x.im - c[q].im * x.re + s[q].re * y[q].im - s[q].im * y[q].re;
            x = cadd(cmul(f[q].a, x), f[q].b);
        }
    }
    if (threadIdx.x != 0) return;
    const double hn = sqrt(a), xr = last.re, xi = last.im;
    // new rotation from (x, hn)
    const double den = sqrt(xr * xr + xi * xi + hn * hn);
    double cr = 1.0, ci = 0.0, sr = 0.0;
    if (den > 0.0) { cr = xr / den; ci = xi / den; sr = hn / den; }
    Hc[2 * t] = cr * xr + ci * xi + sr * hn;          // conj(c) x + conj(s) hn
    Hc[2 * t + 1] = cr * xi - ci * xr;
    cs[2 * j] = cr;
    cs[2 * j + 1] = ci;
    sn[2 * j] = sr;
    sn[2 * j + 1] = 0.0;
    const double er = -sr * g0.re, ei = -sr * g0.im;
    g[2 * t + 2] = er;
    g[2 * t + 3] = ei;
    double *fin = arn + o.fin + 2 * t;   // g[t] after its rotation
    fin[0] = cr * g0.re + ci * g0.im;
    fin[1] = cr * g0.im - ci * g0.re;
    arn[o.sc + t + 1] = hn > 0.0 ? 1.0 / hn : 0.0;
    arn[o.res + t] = sqrt(er * er + ei * ei);
}

// What the host wants to know of steps t .. t + gridDim.x - 1, one block each, into pinned memory.
// One launch per look: written by each step, the stores across PCIe held up every one by 2.5 us.
__global__ void __launch_bounds__(RB) k_arn_report(int t, int m, const double *__restrict__ arn, arn_off o,
                                                   double *__restrict__ hst, host_off ho) {
    t += blockIdx.x;
    const int64_t c = 2 * (int64_t)t * (m + 1);
    for (int i = threadIdx.x; i < 2 * (t + 1); i += RB) hst[ho.H + c + i] = arn[o.H + c + i];
    if (threadIdx.x < 2) {
        const int i = 2 * t + threadIdx.x;
        hst[ho.cs + i] = arn[o.cs + i];
        hst[ho.sn + i] = arn[o.sn + i];
        hst[ho.g + i] = arn[o.fin + i];
    }
    if (threadIdx.x == 2) hst[ho.sc + t + 1] = arn[o.sc + t + 1];
    if (threadIdx.x == 4) hst[ho.sc + t] = arn[o.sc + t];   // a cycle's first vector has a scale of its own
    if (threadIdx.x == 3) hst[ho.res + t] = arn[o.res + t];
}

// Takes the parts along the nv basis vectors (of kept cycles: along their ranges) out of w, after
// bringing the last vector's Gram column up: coefficients in h, partial squared norms of what is left.
template <typename R>
static void orthogonalise(emg_solver *s, int nv, R *w, double *norms, double *h, hipStream_t st) {
    const int64_t n = s->n;
    const arn_off o(s->cap);
    const double *sc = s->arn + o.sc, *qp = s->arn + o.qp;
    const R *V = reinterpret_cast<const R *>(s->V);
    const int nbm = mdot_blocks(n, nv), ldg = s->cap + 1;
    double *dots = s->h, *c = s->h + 2 * 512;
    k_mdot<R, 2><<<dim3(nbm, (nv + DT - 1) / DT), RB, 0, st>>>(n, nv, V, n, w, V + (size_t)(nv - 1) * n * 2, s->partial);
    k_mdot_finish<<<dim3(nv, 2), 256, 0, st>>>(nv, nbm, s->partial, sc, dots, s->gram, ldg);
    k_gram_correct<<<(nv + 15) / 16, RB, 0, st>>>(nv, dots, s->gram, ldg, s->kept, qp, c);
    launch_maxpy<R>(st, s->nblk, n, nv, V, c, sc, w, norms, s->kept, qp, h);
}

// One Arnoldi step t: v_{t+1} = K M^{-1} v_t, classical Gram-Schmidt with the basis' Gram matrix
// (k_gram_correct) and the Hessenberg/Givens update.  Basis vector i is kept as it came out of the
// projection, with its scale sc[i] = 1 / norm beside it: every reader multiplies by it, and the
// pass over the new vector that normalised it is gone.  Only kernel launches, so it can be
// captured: 23 of them at degree 6 with the gradient correction, 12 with the fused steps (33 before, at
// 19,664 DOFs 174 us of kernels that take 2.5 us and more each whatever their size).
template <typename R>
static void enqueue_step(emg_solver *s, int t, hipStream_t st) {
    const int64_t n = s->n;
    const int m = s->cap, nb = s->nblk, nv = t + 1;
    R *V = reinterpret_cast<R *>(s->V);
    R *z = reinterpret_cast<R *>(s->z);
    R *vt = V + (size_t)t * n * 2, *vn = V + (size_t)(t + 1) * n * 2;
    const arn_off o(m);
    bool done = false;
    if constexpr (sizeof(R) == 4)
        if (s->fused) {
            apply_fused(s, vt, s->arn + o.sc + t, vn, true, st);
            done = true;
        }
    if (!done) {
        apply_prec_poly<R>(s, vt, s->arn + o.sc + t, z, st);
        spmv_pk<R, SP_Y, false>(s, s->lanes[sizeof(R) == 4], z, sp_args<R>{nullptr, vn, nullptr, nullptr, 0, nullptr}, st);
    }
    double *h = s->h + 4 * 512;
    orthogonalise<R>(s, nv, vn, s->pn, h, st);
    k_arn_givens<<<1, RB, 0, st>>>(t, m, nb, s->pn, h, s->kept, s->arn, o);
}

// Captures what `fill` enqueues as one graph.
template <typename FN>
static int capture(emg_solver *s, FN &&fill, hipGraphExec_t *out) {
    *out = nullptr;
    EMG_HIP(hipStreamBeginCapture(s->cap_stream, hipStreamCaptureModeThreadLocal));
    fill(s->cap_stream);
    hipGraph_t graph = nullptr;
    EMG_HIP(hipStreamEndCapture(s->cap_stream, &graph));
    const hipError_t e = hipGraphInstantiate(out, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    if (e != hipSuccess) *out = nullptr;
    EMG_HIP(e);
    return 0;
}

// Step t as a graph, captured when a cycle first gets to it (few get to the end of the basis), or
// with t = -1 the preconditioner that closes a cycle: z = M p(K M) w.
template <typename R>
static int step_graph(emg_solver *s, int t, hipGraphExec_t *out) {
    if (s->exec_np2 != s->np2 || s->exec_poly != s->poly_deg) drop_graphs(s);
    s->exec_np2 = s->np2;
    s->exec_poly = s->poly_deg;
    s->exec.resize(s->cap, nullptr);
    hipGraphExec_t &g = t >= 0 ? s->exec[t] : s->tail;
    if (g == nullptr) {
        const int rc = capture(s, [&](hipStream_t cs) {
            if (t >= 0) enqueue_step<R>(s, t, cs);
            else apply_prec_poly<R>(s, reinterpret_cast<const R *>(s->w), nullptr, reinterpret_cast<R *>(s->z), cs);
        }, &g);
        if (rc) return rc;
    }
    *out = g;
    return 0;
}

// The cycles of one solve that share the basis storage, as the host sees them: basis vectors
// t0 .. t0 + k with k columns each, the upper triangular factor over all of them and the rotations.
struct kept_host {
    using C = std::complex<double>;
    int m;
    struct cyc { int t0, k; };
    std::vector<cyc> cycles;
    std::vector<C> R, cs, sn, g;      // R: column t at t * (m + 1)
    std::vector<double> sc;
    explicit kept_host(int m_) : m(m_), R((size_t)m_ * (m_ + 1)), cs(m_), sn(m_), g(m_ + 1), sc(m_ + 1) {}
    int used() const { return cycles.empty() ? 0 : cycles.back().t0 + cycles.back().k + 1; }
    C &r(int i, int t) { return R[(size_t)t * (m + 1) + i]; }
    // rows t0 .. t0 + k of a column through the rotations of cycle c
    void rotate(const cyc &c, C *col) const {
        C x = col[c.t0];
        for (int i = c.t0; i < c.t0 + c.k; i++) {
            const C y = col[i + 1];
            col[i] = std::conj(cs[i]) * x + std::conj(sn[i]) * y;
            x = -sn[i] * x + cs[i] * y;
        }
        col[c.t0 + c.k] = x;
    }
};

// Residual reduction at which a complex64 cycle ends.  With the spaces kept a new cycle costs little
// (an FP64 residual and three passes over the basis), and the sooner the residual is formed anew the
// less complex64 rounding the estimates carry: 200 / 241 / 263 steps to 3e-13 at 1e-1 / 3e-2 / 1e-2 on
// the posts box at 40 x 20 x 8 hexes.
static constexpr double CYCLE_CUT = 1e-1;
static constexpr int CYCLE_ROOM = 12;       // basis vectors worth starting another kept cycle for
// Where the caller limits the refinements, each is to reach as far as it can be worth: to 1e-2, with room for a whole
// restart length.
static constexpr double LIMITED_CUT = 1e-2;

// What the device knows of the kept cycles: their spans, and where the next cycle begins.  (The
// staging is not written again before the stream has been waited for.)
static int upload_kept(emg_solver *s, const kept_host &kh, hipStream_t st) {
    kept_dev *kd = reinterpret_cast<kept_dev *>(s->host + host_off(s->cap).kept);
    kd->t0 = kh.used();
    kd->ncyc = (int32_t)kh.cycles.size();
    for (size_t c = 0; c < kh.cycles.size(); c++) kd->start[c] = kh.cycles[c].t0;
    kd->start[kh.cycles.size()] = kd->t0;
    // with the outside direction of the last cycle, which lies before it (gmres_cycle)
    const host_off ho(s->cap);
    const int64_t from = kh.cycles.empty() ? ho.kept - ho.qp : 2 * kh.cycles.back().t0;
    EMG_HIP(hipMemcpyAsync(s->arn + arn_off(s->cap).qp + from, s->host + ho.qp + from,
                           (ho.total - ho.qp - from) * sizeof(double), hipMemcpyHostToDevice, st));
    return 0;
}

// One cycle of GMRES on K u = w (right preconditioned), beginning at the free end of the basis:
// until the residual estimate relative to `unit` is at most tol, at most maxiter steps, or the basis is
// full.  On entry s->w holds w; on return s->z holds u.  iters: steps done; rel: the last estimate
// relative to `unit`.
//
// With cycles kept in kh (the refinement cycles of one mixed-precision solve) the operator is
// projected off their ranges, as GCRO does: the cycle minimises over the kept spaces and its own
// together, so in exact arithmetic the cycles continue ONE unrestarted GMRES although each starts
// from a residual that was formed anew in FP64.  A cycle that forgets the others pays their first steps
// again: the posts box at 40 x 20 x 8 hexes took 425 steps in 7 cycles to 3e-13, where complex128
// GMRES, which never restarts on the way, takes 155.  The ranges are not stored: C_c = V Q_c is applied
// through the basis vectors and the rotations of cycle c (project_kept), and what the projections
// take away enters the triangular factor of the least-squares problem.  When the basis is nearly full
// everything is forgotten (the caller clears kh).
template <typename R>
static int gmres_cycle(emg_solver *s, double unit, double tol, int maxiter, kept_host &kh, int *iters, double *rel,
                       hipStream_t st) {
    using C = std::complex<double>;
    const int64_t n = s->n;
    const int m = s->cap, nb = s->nblk, t0 = kh.used();
    const arn_off o(m);
    const host_off ho(m);
    R *V = reinterpret_cast<R *>(s->V), *w = reinterpret_cast<R *>(s->w), *vt = V + (size_t)t0 * n * 2;
    *iters = 0;
    if (t0 > 0) {
        // the kept ranges' part of w is solved by them: coefficients to the host, w projected
        orthogonalise<R>(s, t0, w, s->pn, s->host_dev + ho.h0, st);
    } else {
        k_norm2<R><<<nb, RB, 0, st>>>(n, w, s->pn);
    }
    k_arn_start<R><<<nb, RB, 0, st>>>(n, t0, nb, s->pn, w, vt, s->arn, o);
    EMG_LAUNCH_CHECK();
    const int len = chunk_it(n), most = std::min({m - t0, s->restart, maxiter});
    int k = 0;
    for (bool done = false; !done && k < most;) {
        const int k1 = std::min(k + len, most);
        for (int q = k; q < k1; q++) {
            hipGraphExec_t graph = nullptr;
            if (int rc = step_graph<R>(s, t0 + q, &graph)) return rc;
            EMG_HIP(hipGraphLaunch(graph, st));
        }
        k_arn_report<<<k1 - k, RB, 0, st>>>(t0 + k, m, s->arn, o, s->host_dev, ho);
        EMG_HIP(hipStreamSynchronize(st));
        for (; k < k1; k++) {   // steps of the chunk past the one that reaches tol serve too
            const double e = s->host[ho.res + t0 + k] / unit;
            if (!std::isfinite(e)) { done = true; break; }
            *rel = e;
            if (e <= tol) done = true;
        }
    }
    *iters = k;
    if (k == 0) { *rel = std::numeric_limits<double>::quiet_NaN(); return 0; }
    // the new columns of the triangular factor, then y = R^{-1} g over all kept columns
    auto from_host = [&](int64_t off, int64_t i) { return C(s->host[off + 2 * i], s->host[off + 2 * i + 1]); };
    std::vector<C> g(m + 1), y(m + 1);
    for (int i = 0; i < t0; i++) g[i] = from_host(ho.h0, i);
    for (int t = t0; t < t0 + k; t++) {
        kh.cs[t] = from_host(ho.cs, t);
        kh.sn[t] = from_host(ho.sn, t);
        g[t] = from_host(ho.g, t);
        for (int i = 0; i <= t; i++) kh.r(i, t) = from_host(ho.H + 2 * (int64_t)t * (m + 1), i);
        for (const auto &c : kh.cycles) kh.rotate(c, &kh.r(0, t));
    }
    for (int t = t0; t <= t0 + k; t++) kh.sc[t] = s->host[ho.sc + t];
    for (const auto &c : kh.cycles) kh.rotate(c, g.data());
    kh.cycles.push_back({t0, k});
    for (int c = (int)kh.cycles.size() - 1; c >= 0; c--) {
        const auto &cy = kh.cycles[c];
        for (int i = cy.t0 + cy.k - 1; i >= cy.t0; i--) {
            const C *r = &kh.r(0, i);
            // a zero pivot is a breakdown: the columns past it add nothing
            const C yi = r[i] == C(0.0) ? C(0.0) : g[i] / r[i];
            y[i] = yi;
            for (int q = 0; q < i; q++)   // the rows of the cycles' last vectors are not read again
                g[q] -= C(r[q].real() * yi.real() - r[q].imag() * yi.imag(), r[q].real() * yi.imag() + r[q].imag() * yi.real());
        }
    }
    const int nv = t0 + k;
    C *ys = reinterpret_cast<C *>(s->host + ho.y), *qs = reinterpret_cast<C *>(s->host + ho.qp + 2 * t0);
    for (int i = 0; i < nv; i++) ys[i] = y[i] * kh.sc[i];   // a cycle's last vector has no column: y = 0
    double *yd = s->h + 6 * 512;
    EMG_HIP(hipMemcpyAsync(yd, ys, nv * sizeof(C), hipMemcpyHostToDevice, st));
    k_mcomb<R><<<nb, RB, 0, st>>>(n, nv, V, n, yd, w, 1);
    EMG_LAUNCH_CHECK();
    hipGraphExec_t graph = nullptr;
    if (int rc = step_graph<R>(s, -1, &graph)) return rc;
    EMG_HIP(hipGraphLaunch(graph, st));
    // the direction of the cycle's span outside its range, Q e_{k+1}, back through the rotations; it
    // stays in the staging for the next upload_kept
    for (int i = 0; i < k; i++) qs[i] = 0.0;
    qs[k] = 1.0;
    for (int i = k - 1; i >= 0; i--) {
        const C a = qs[i], b = qs[i + 1], cc = kh.cs[t0 + i], ss = kh.sn[t0 + i];
        qs[i] = cc * a - std::conj(ss) * b;
        qs[i + 1] = ss * a + std::conj(cc) * b;
    }
    return 0;
}

// sqrt of the sum of |v|^2 (waits for the stream)
static int norm_to_host(emg_solver *s, const double *v, int slot, double *out, hipStream_t st) {
    const host_off ho(s->cap);
    k_norm2<double><<<s->nblk, RB, 0, st>>>(s->n, v, s->partial);
    k_sum_partials<<<1, RB, 0, st>>>(s->nblk, s->partial, s->host_dev + ho.norm + slot);
    EMG_HIP(hipStreamSynchronize(st));
    *out = std::sqrt(s->host[ho.norm + slot]);
    return 0;
}

// ---- restarted GMRES solve of K u = rhs in complex128: u holds the initial guess and the solution;
// *iters the steps done.
static int gmres_full(emg_solver *s, const double *rhs, double *u, double tol, int maxiter, int *iters, hipStream_t st) {
    const int64_t n = s->n;
    *iters = 0;
    double bnorm = 0, beta = 0;
    if (int rc = norm_to_host(s, rhs, 0, &bnorm, st)) return rc;
    if (bnorm == 0) {
        EMG_HIP(hipMemsetAsync(u, 0, n * 2 * sizeof(double), st));
        return 0;
    }
    kept_host kh(s->cap);
    while (true) {
        spmv_pk<double, SP_RESID, false>(s, s->lanes[0], u, sp_args<double>{rhs, s->w, nullptr, nullptr, 0, nullptr}, st);
        if (int rc = norm_to_host(s, s->w, 0, &beta, st)) return rc;
        if (beta / bnorm <= tol || *iters >= maxiter || !(beta > 0) || !std::isfinite(beta)) return 0;
        kh.cycles.clear();
        if (int rc = upload_kept(s, kh, st)) return rc;
        int it = 0;
        double rel = 0;
        if (int rc = gmres_cycle<double>(s, bnorm, tol, maxiter - *iters, kh, &it, &rel, st)) return rc;
        *iters += it;
        if (it > 0) k_add<double><<<s->nblk, RB, 0, st>>>(n, s->z, u);
        EMG_HIP(hipStreamSynchronize(st));   // the upload staging is written again
        if (it == 0 || !std::isfinite(rel)) return 0;
    }
}

extern "C" int emg_solver_solve(emg_solver *s, const double *d_b, double *d_x, double tol, int maxiter, int max_refine,
                                emg_solve_info *info, void *stream) {
    EMG_CHECK(s && d_b && d_x && info, "emg_solver_solve: null argument");
    EMG_CHECK(s->vals != nullptr, "emg_solver_solve: emg_solver_set_matrix was not called");
    EMG_CHECK(s->V != nullptr, "emg_solver_solve: no memory for the basis");
    hipStream_t st = (hipStream_t)stream;
    memset(info, 0, sizeof(*info));
    double bn = -1.0;   // ||b||, formed with the first residual
    auto true_resid = [&](double *out_rel) -> int {
        // r = b - K x in complex128 (masked)
        double rn = 0;
        if (bn < 0)
            if (int rc = norm_to_host(s, d_b, 0, &bn, st)) return rc;
        spmv_std(s, d_x, d_b, s->r, st);
        if (int rc = norm_to_host(s, s->r, 1, &rn, st)) return rc;
        *out_rel = bn > 0 ? rn / bn : 0.0;
        return 0;
    };
    double rel;
    if (s->precision == 64) {
        int it;
        // K and the residual are the caller's values as they are now, the preconditioner the last
        // emg_solver_set_matrix's (1 - 2 products' time)
        pack_matrix(s, st);
        k_pack_vec<double><<<emg::grid_for(s->n_ent, RB), RB, 0, st>>>(s->n_ent, d_b, 1.0, s->r);
        k_pack_vec<double><<<emg::grid_for(s->n_ent, RB), RB, 0, st>>>(s->n_ent, d_x, 1.0, s->d);
        int rc = gmres_full(s, s->r, s->d, tol, maxiter, &it, st);
        if (rc) return rc;
        k_unpack_vec<double><<<emg::grid_for(s->n_ent, RB), RB, 0, st>>>(s->n_ent, s->d, 1.0, 0, d_x);
        info->iterations = it;
        info->refinements = 0;
        rc = true_resid(&rel);
        if (rc) return rc;
        info->residual = rel;
    } else {
        // Mixed-precision GMRES: every cycle runs in complex64 on K d = r / |r|, then x += d and
        // r = b - K x are formed in FP64.
        int rc = true_resid(&rel);
        if (rc) return rc;
        int total = 0, ref = 0;
        const bool limited = max_refine > 0;
        const int limit = limited ? max_refine : (1 << 30), room = limited ? s->restart : CYCLE_ROOM;
        int stall = 0;
        kept_host kh(s->cap);
        while (rel > tol && ref < limit && total < maxiter) {
            // here, not behind a cycle: nothing of a solve is in flight when it returns
            rc = upload_kept(s, kh, st);
            if (rc) return rc;
            const double rs = 1.0 / (rel * bn);
            k_pack_vec<float><<<emg::grid_for(s->n_ent, RB), RB, 0, st>>>(s->n_ent, s->r, rs, reinterpret_cast<float *>(s->w));
            // A cycle stops once complex64 GMRES has reduced its residual by CYCLE_CUT (or
            // reached what tol needs), so that complex64 never has to resolve more than that.
            const double inner_tol = std::max(0.5 * tol / rel, limited ? LIMITED_CUT : CYCLE_CUT);
            int it = 0;
            double est = 0;
            rc = gmres_cycle<float>(s, 1.0, inner_tol, maxiter - total, kh, &it, &est, st);
            if (rc) return rc;
            if (it == 0 && kh.cycles.empty()) break;
            total += it;
            ref++;
            if (it > 0)
                k_unpack_vec<float><<<emg::grid_for(s->n_ent, RB), RB, 0, st>>>(
                    s->n_ent, reinterpret_cast<const float *>(s->z), 1.0 / rs, 1, d_x);
            const double prev = rel;
            rc = true_resid(&rel);
            if (rc) return rc;
            if (it > 0 && !(rel <= 2.0 * prev)) {
                // the kept spaces no longer fit the operator in complex64: take the step back and forget
                k_unpack_vec<float><<<emg::grid_for(s->n_ent, RB), RB, 0, st>>>(
                    s->n_ent, reinterpret_cast<const float *>(s->z), -1.0 / rs, 1, d_x);
                rc = true_resid(&rel);
                if (rc) return rc;
                if (kh.cycles.size() == 1) break;   // nothing was kept: complex64 cannot do better here
                it = 0;
            }
            stall = (rel > 0.999 * prev) ? stall + 1 : 0;
            if (stall >= 3) break;   // no progress in complex64: stop (caller sees converged = 0)
            // A full basis, or two cycles without progress, end the memory of the cycles before.  One
            // such cycle does not: rounding of a large correction can undo its gain, which the next
            // cycles of the same space make up in a few steps (posts box at 2.2 GHz: 244 steps to 1e-9,
            // 500 when it forgot there).
            if (it == 0 || s->cap - kh.used() < room || (int)kh.cycles.size() == KEEP_MAX || stall >= 2) kh.cycles.clear();
        }
        info->iterations = total;
        info->refinements = ref;
        info->residual = rel;
    }
    info->converged = info->residual <= tol ? 1 : 0;
    EMG_LAUNCH_CHECK();
    return 0;
}

extern "C" int emg_affine_combine(int64_t nnz, const double *d_E, const double *d_B, double s, double *d_K, void *stream) {
    EMG_CHECK(d_E && d_B && d_K, "emg_affine_combine: null argument");
    k_affine<<<2048, RB, 0, (hipStream_t)stream>>>(nnz, d_E, d_B, s, d_K);
    EMG_LAUNCH_CHECK();
    return 0;
}

extern "C" int emg_csr_find(int64_t m, const int32_t *d_rowptr, const int32_t *d_cols, const int32_t *d_qr,
                            const int32_t *d_qc, int32_t *d_pos, void *stream) {
    EMG_CHECK(d_rowptr && d_cols && d_qr && d_qc && d_pos, "emg_csr_find: null argument");
    if (m == 0) return 0;
    k_csr_find<<<emg::grid_for(m, RB), RB, 0, (hipStream_t)stream>>>(m, d_rowptr, d_cols, d_qr, d_qc, d_pos);
    EMG_LAUNCH_CHECK();
    return 0;
}

extern "C" int emg_scatter_add(int64_t m, const int32_t *d_pos, const double *d_v, double gre, double gim, double *d_K,
                               void *stream) {
    EMG_CHECK(d_pos && d_v && d_K, "emg_scatter_add: null argument");
    if (m == 0) return 0;
    k_scatter_add<<<emg::grid_for(m, RB), RB, 0, (hipStream_t)stream>>>(m, d_pos, d_v, gre, gim, d_K);
    EMG_LAUNCH_CHECK();
    return 0;
}

// ------------------------------------------------------------------ vector primitives
// complex128 building blocks for the eigen driver (Arnoldi with CGS2).
extern "C" int emg_spmv(int64_t n, const int32_t *d_rowptr, const int32_t *d_cols, const double *d_vals,
                        const uint8_t *d_mask, const double *d_x, double *d_y, void *stream) {
    EMG_CHECK(d_rowptr && d_cols && d_vals && d_x && d_y, "emg_spmv: null argument");
    launch_spmv((hipStream_t)stream, n, d_rowptr, d_cols, d_vals, d_mask, d_x, d_y);
    EMG_LAUNCH_CHECK();
    return 0;
}

extern "C" int emg_spmv_blocked(int64_t n, int64_t nnz, const int32_t *d_rowptr, const int32_t *d_cols,
                                const double *d_vals, const uint8_t *d_mask, const double *d_x, double *d_y,
                                void *stream) {
    EMG_CHECK(d_rowptr && d_cols && d_vals && d_x && d_y, "emg_spmv_blocked: null argument");
    EMG_CHECK(n > 0 && n % 2 == 0 && nnz % 2 == 0, "emg_spmv_blocked: n and nnz must be even");
    launch_spmv_blk((hipStream_t)stream, n, nnz, d_rowptr, d_cols, d_vals, d_mask, d_x, nullptr, d_y,
                            spmv_blk_lanes());
    EMG_LAUNCH_CHECK();
    return 0;
}

// y = mask.(K (mask.x)) with the matrix of the last emg_solver_set_matrix, complex128 (precision 64) or the
// complex64 copy (precision 32, x and y complex64), PEC columns folded into that copy; x and y in the caller's
// layout (k_spmv_pk's STD form, STD_LANES lanes per entity).
extern "C" int emg_solver_apply(emg_solver *s, int precision, const void *d_x, void *d_y, void *stream) {
    EMG_CHECK(s != nullptr && d_x && d_y, "emg_solver_apply: null argument");
    EMG_CHECK(s->vals != nullptr, "emg_solver_apply: no matrix set");
    hipStream_t st = (hipStream_t)stream;
    if (precision == 64) {
        spmv_std(s, static_cast<const double *>(d_x), nullptr, static_cast<double *>(d_y), st);
    } else {
        EMG_CHECK(precision == 32 && s->precision == 32, "emg_solver_apply: precision 32 needs a precision-32 solver");
        spmv_pk<float, SP_Y, true>(s, STD_LANES, static_cast<const float *>(d_x),
                                   sp_args<float>{nullptr, static_cast<float *>(d_y), nullptr, nullptr, 0, nullptr}, st);
    }
    EMG_LAUNCH_CHECK();
    return 0;
}

static int nblk_for(int64_t n) {
    return (int)std::max<int64_t>(1, std::min<int64_t>((n / 2 * maxpy_split(n) + RB - 1) / RB, 1024));
}

// d_h[i] = sum_k conj(V_i[k]) w[k], i < nv; V holds nv vectors of n entries back to back.
// d_work: at least ceil(nv/8) * 1024 * 16 + 16 doubles.
extern "C" int emg_mdotc(int64_t n, int nv, const double *d_V, const double *d_w, double *d_h, double *d_work,
                         void *stream) {
    EMG_CHECK(d_V && d_w && d_h && d_work && nv > 0 && nv <= 512, "emg_mdotc: bad argument");
    hipStream_t st = (hipStream_t)stream;
    const int nbm = mdot_blocks(n, nv);
    k_mdot<double, 1><<<dim3(nbm, (nv + DT - 1) / DT), RB, 0, st>>>(n, nv, d_V, n, d_w, nullptr, d_work);
    k_mdot_finish<<<nv, 256, 0, st>>>(nv, nbm, d_work, nullptr, d_h, nullptr, 0);
    EMG_LAUNCH_CHECK();
    return 0;
}

// w -= sum_i h_i V_i ; *d_norm (on device) = ||w|| after the update.
extern "C" int emg_maxpy(int64_t n, int nv, const double *d_V, const double *d_h, double *d_w, double *d_norm,
                         double *d_work, void *stream) {
    EMG_CHECK(d_V && d_h && d_w && d_norm && d_work && nv >= 0 && nv <= 512, "emg_maxpy: bad argument");
    hipStream_t st = (hipStream_t)stream;
    const int nb = nblk_for(n);
    launch_maxpy<double>(st, nb, n, nv, d_V, d_h, nullptr, d_w, d_work);
    k_scale_by_norm<double><<<1, RB, 0, st>>>(0, d_work, nb, d_w, d_w, d_norm);   // n = 0: norm only
    EMG_LAUNCH_CHECK();
    return 0;
}

// y (+)= A x for a real CSR matrix A (float64 values) and complex128 x, y.
__global__ void __launch_bounds__(256) k_csr_real(int64_t nrows, const int32_t *__restrict__ rp, const int32_t *__restrict__ ci,
                                                  const double *__restrict__ av, const double *__restrict__ x,
                                                  double *__restrict__ y, int accumulate) {
    const int64_t r = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) / SUB;
    const int lane = threadIdx.x % SUB;
    if (r >= nrows) return;
    double ar = 0.0, ai = 0.0;
    for (int32_t e = rp[r] + lane; e < rp[r + 1]; e += SUB) {
        ar += av[e] * x[2 * ci[e]];
        ai += av[e] * x[2 * ci[e] + 1];
    }
    ar = lane_sum<SUB>(ar);
    ai = lane_sum<SUB>(ai);
    if (lane == 0) {
        if (accumulate) { y[2 * r] += ar; y[2 * r + 1] += ai; }
        else { y[2 * r] = ar; y[2 * r + 1] = ai; }
    }
}

extern "C" int emg_csr_real_apply(int64_t nrows, const int32_t *d_rowptr, const int32_t *d_cols, const double *d_vals,
                                  const double *d_x, double *d_y, int accumulate, void *stream) {
    EMG_CHECK(nrows >= 0 && d_rowptr && d_cols && d_vals && d_x && d_y, "emg_csr_real_apply: null argument");
    if (nrows == 0) return 0;
    k_csr_real<<<(unsigned)((nrows * SUB + 255) / 256), 256, 0, (hipStream_t)stream>>>(nrows, d_rowptr, d_cols, d_vals,
                                                                                     d_x, d_y, accumulate);
    EMG_LAUNCH_CHECK();
    return 0;
}

// x = sum_i y_i V_i  (y complex on device)
extern "C" int emg_mcomb(int64_t n, int nv, const double *d_V, const double *d_y, double *d_x, void *stream) {
    EMG_CHECK(d_V && d_y && d_x && nv > 0 && nv <= 512, "emg_mcomb: bad argument");
    k_mcomb<double><<<nblk_for(n), RB, 0, (hipStream_t)stream>>>(n, nv, d_V, n, d_y, d_x, 1);
    EMG_LAUNCH_CHECK();
    return 0;
}
