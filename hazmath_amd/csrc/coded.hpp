// Kernels over a matrix's entry codes: a byte an entry instead of the 10 (FP64)
// or 6 (FP32) of a value and a 16-bit column offset, so the vectors are what
// such a kernel moves.  One skeleton, a row a lane; what a row does with its
// entries is the operation's (begin, entry, end).
#pragma once
#include "hz_common.h"
#include "hz_internal.h"

namespace hz {

constexpr int kCodedBlock = 256, kCodedSlices = kCodedBlock / kWave;

// A slice a wavefront, its codes in `words` words a row (the same for every
// slice, so their address needs no load), the table in LDS; addresses are
// 32-bit byte offsets from the vector's start.  What is left of a row's cost is
// the chain codes, table, gathers.  2,048,383 rows, before (columns and values,
// stored zeros left out) and with codes: FP64 7-entry rows product 30 -> 18.5 us,
// residual 31 -> 17, last sweep 38 -> 21; 15-entry rows FP32 Chebyshev step 39
// -> 16, FP64 product 63 -> 25; 438,976 rows of 15: 15.5 -> 7.4-10.  With the
// slices' places loaded first the Chebyshev step took 20 us, with 64-bit
// addresses as well 24; several slices in turn by a workgroup gained nothing.
// Entries are added in stored order and the partial of a workgroup is that of
// its 256 rows, as in the kernels that read columns and values: results and dots
// are bit-identical to theirs.
template <int U, class T, class Op>
__global__ __launch_bounds__(kCodedBlock) void k_coded(int n, int nslices, int words, const code8 *__restrict__ code,
                                                       const CodeEntry<T> *__restrict__ table, Op op,
                                                       double *__restrict__ partials) {
    static_assert(U % 4 == 0, "words");
    __shared__ CodeEntry<T> tab[kCodes];
    __shared__ double sh[kCodedBlock / kWave];
    const int blk = xcd_block_id();
    const CodedLane l = coded_lane(blk * kCodedSlices + threadIdx.x / kWave, threadIdx.x % kWave, n, nslices, words,
                                   sizeof(T));
    const int r = l.row;
    const auto load = [&](int k, unsigned int (&w)[U / 4]) {
#pragma unroll
        for (int u = 0; u < U / 4; ++u) w[u] = coded_word(l, code, k + u, words);
    };
    unsigned int w[U / 4];
    load(0, w);
    if (l.in) op.begin(r);
    for (int i = threadIdx.x; i < kCodes; i += kCodedBlock) tab[i] = table[i];
    __syncthreads();
    for (int k = 0; k < words; k += U / 4) {
        if (k > 0) load(k, w);
        T vv[U], xx[U];
        unsigned int at[U];
        bool pad[U], diag[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const unsigned int h = coded_entry(w[u / 4], u % 4);
            const CodeEntry<T> e = tab[h];
            pad[u] = h == (unsigned int)kCodePad;
            diag[u] = e.off == 0;
            at[u] = l.base + (unsigned int)e.off;   // padding reads the row's own entry
            vv[u] = e.val;
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            xx[u] = *reinterpret_cast<const T *>(reinterpret_cast<const char *>(op.x) + at[u]);
#pragma unroll
        for (int u = 0; u < U; ++u) op.entry(pad[u], diag[u], vv[u], xx[u]);
    }
    const double prod = l.in ? op.end(r) : 0.0;
    if constexpr (Op::kDot) {
        const double bs = block_sum<kCodedBlock>(prod, sh);
        if (threadIdx.x == 0) partials[blk] = bs;
    }
}

template <class T, class Op>
void launch_coded(const DevSELL &S, const Op &op, double *partials = nullptr) {
    const int grid = div_up(S.nslices, kCodedSlices);
    const auto *code = reinterpret_cast<const code8 *>(S.code);
    const auto *tab = static_cast<const CodeEntry<T> *>(std::is_same_v<T, float> ? S.ctabf : S.ctab);
    if (S.cwords <= 2)
        k_coded<8, T, Op><<<grid, kCodedBlock, 0, stream()>>>(S.n, S.nslices, S.cwords, code, tab, op, partials);
    else
        k_coded<16, T, Op><<<grid, kCodedBlock, 0, stream()>>>(S.n, S.nslices, S.cwords, code, tab, op, partials);
    HZ_LAUNCH_CHECK();
}

// bytes of the matrix a coded kernel cannot do without: a code an entry (padding
// ends a row, so no row pointers or lengths are read)
inline double coded_bytes(const DevSELL &S) { return (double)S.nnz; }

// w = b - A x
template <class T>
struct CodedResidual {
    static constexpr bool kDot = false;
    const T *__restrict__ b, *__restrict__ x;
    T *__restrict__ w;
    T bi = 0, acc = 0;
    __device__ void begin(int r) { bi = b[r]; }
    __device__ void entry(bool pad, bool, T v, T xv) { acc = pad ? acc : acc + v * xv; }
    __device__ double end(int r) {
        w[r] = bi - acc;
        return 0.0;
    }
};

// one Jacobi (weight wgt) or L1DIAG sweep, as k_sweep (FP64) and k_sweep_m
// (FP32) without a prolongation; FP32 with kOut: the result to out64 and the
// dot with r64
template <class T, int kSmoother, bool kWithDot>
struct CodedSweep {
    static constexpr bool kDot = kWithDot;
    const T *__restrict__ b, *__restrict__ x;
    T *__restrict__ xout;
    double *__restrict__ out64;
    const double *__restrict__ r64;
    T wgt;
    T t = 0, d = 0, xi = 0, bi = 0;
    __device__ void begin(int r) {
        t = bi = b[r];
        xi = x[r];
    }
    __device__ void entry(bool pad, bool diag, T v, T xv) {
        if (kSmoother == HZ_SMOOTHER_L1DIAG) {
            t = pad ? t : t - v * xv;
            d = d + (v < 0 ? -v : v);
        } else {
            d = diag && !pad ? v : d;
            t = diag ? t : t - v * xv;   // padding has offset 0 too
        }
    }
    __device__ double end(int r) {
        T xn = xi;
        if ((d < 0 ? -d : d) > (T)(std::is_same_v<T, float> ? 1e-20f : kSmallReal)) {
            if (kSmoother == HZ_SMOOTHER_L1DIAG) xn = xi + t / d;
            else xn = ((T)1 - wgt) * xi + wgt * t / d;
        }
        if constexpr (std::is_same_v<T, double>) {
            xout[r] = xn;
            return kDot ? xn * bi : 0.0;
        } else if constexpr (kDot) {
            const double z = (double)xn;
            out64[r] = z;
            return z * r64[r];
        } else {
            xout[r] = xn;
            return 0.0;
        }
    }
};

// one Chebyshev step, as k_cheb_step (FP64) and k_cheb_step_m (FP32; kWithDot:
// the cycle's last, to out64 with the dot with r64)
template <class T, bool kWithDot>
struct CodedCheb {
    static constexpr bool kDot = kWithDot;
    const T *__restrict__ diag, *__restrict__ b, *__restrict__ x;
    T *__restrict__ xout, *__restrict__ d;
    double *__restrict__ out64;
    const double *__restrict__ r64;
    T c1, c2;
    T t = 0, di = 0, dv = 0, xi = 0;
    __device__ void begin(int r) {
        t = b[r];
        di = diag[r];
        dv = c1 == (T)0 ? (T)0 : c1 * d[r];
        xi = x[r];
    }
    __device__ void entry(bool pad, bool, T v, T xv) { t = pad ? t : t - v * xv; }
    __device__ double end(int r) {
        const T dn = dv + (di != (T)0 ? c2 * t / di : (T)0);
        d[r] = dn;
        const T xn = xi + dn;
        if constexpr (kDot) {
            const double z = (double)xn;
            out64[r] = z;
            return z * r64[r];
        } else {
            xout[r] = xn;
            return 0.0;
        }
    }
};

// y = A x with the partials of (y, x)
struct CodedProduct {
    static constexpr bool kDot = true;
    const double *__restrict__ x;
    double *__restrict__ y;
    double xi = 0, acc = 0;
    __device__ void begin(int r) { xi = x[r]; }
    __device__ void entry(bool pad, bool, double v, double xv) { acc = pad ? acc : acc + v * xv; }
    __device__ double end(int r) {
        y[r] = acc;
        return acc * xi;
    }
};

}  // namespace hz
