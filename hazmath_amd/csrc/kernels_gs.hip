// kernels_gs.hip -- Gauss-Seidel-type smoothers (smoother_dcsr_gs / _sgs /
// _sor, src/solver/smoother.c:109-307, dispatched like dcsr_presmoothing /
// dcsr_postsmoothing, src/solver/mgcycle.c:76-223) as multicolour sweeps.
//
// The rows are coloured so that no two rows of one colour are coupled in
// either direction (Jones-Plassmann on the pattern of A + A^T: a row takes the
// smallest colour its coloured neighbours leave free once its hash priority
// beats every uncoloured neighbour's).  A forward sweep visits the colours in
// increasing order, a backward sweep in decreasing order, and the rows of one
// colour update in parallel.  That is Gauss-Seidel in the colour-major row
// order, bit for bit (the rows of a colour read no value written in the same
// colour), not in the natural order the reference sweeps in: results follow
// the reference's by convergence behaviour, not bit for bit.
//
// Layout: the rows are listed colour by colour (ascending inside one), each
// colour padded to slices of 64 positions; a slice stores its rows'
// off-diagonal entries column-major as positions (entry k of lane t at
// 64 (W slice + k) + t, CSR order inside the row, W the longest row, padding a
// zero entry on the lane's own position) and the diagonal a_ii separately, so
// that nothing has to be loaded to find a slice's data.  Where the padding to W
// costs more than that (large levels, or rows of very different lengths) every
// slice has the width of its own longest row, and its place is loaded: with one
// width a row of 30,000 entries among 1,000,000 would ask for 360 GB.  Stored
// zeros are left out.  A wave handles one slice; one launch per colour, or on
// levels whose x fits LDS one workgroup for the whole smoothing call.
//
// What bounds a sweep on all but the largest levels is the chain of a colour
// visit: a launch or a barrier, the entries' loads, the gathers, the division
// (SGS visits 21 colours a call, twice a level and cycle).  Entries go in
// rounds of 8 or 16 masked loads (rows of 6 entries took six dependent pairs of
// loads when only whole rounds of eight were batched), and the one-workgroup
// form loads a wave's next two slices ahead.  Measured on the 64^3 Poisson
// hierarchy (SGS, 11 colours): a colour's launch 7.5 -> 3.5-4.0 us, the
// one-workgroup call on 7,811 / 3,902 / 1,950 rows 165 / 90 / 65 -> 62 / 40 / 29
// us, PCG 42.5 -> 25.8 ms; the preparation (rows sorted and placed on the GPU, no
// transpose where the pattern is symmetric) 9 -> 5 ms over eight levels.
#include <algorithm>
#include <type_traits>
#include <vector>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include "hz_internal.h"

namespace hz {

namespace {

constexpr int kBlock = 256;
static_assert(kSlice == 64, "one wave per slice");
constexpr int kGsMaxPass = 8;               // passes per single-workgroup launch
// Levels of up to this many positions keep x in LDS (144 of the CU's 160 KiB)
// and run as one workgroup.  At the upper end, 15,627 rows of 10 entries, 21
// colour visits take 105 us (the random LDS gathers of eight waves bound it)
// against 21 launches of 4.1 us and a permutation of 5; with one pass and
// shorter rows (10,000 rows of 5, 10 visits) 24 us against 46.
constexpr int kGsLdsPos = 18432;
constexpr int kGsMaxPhase = 1024;           // colour visits per single-workgroup launch
constexpr int kSlicesPerBlock = kBlock / kSlice;
constexpr int kHistBins = 256;

int grid_rows(long n) { return (int)std::max(1L, std::min<long>((n + kBlock - 1) / kBlock, 16384)); }

__device__ __forceinline__ unsigned jp_priority(int i) {
    unsigned h = (unsigned)i * 2654435761u;
    h ^= h >> 16;
    h *= 0x85EBCA6Bu;
    h ^= h >> 13;
    return h;
}

// Neighbour j of row i beats i: higher priority, ties by index.
__device__ __forceinline__ bool beats(int j, unsigned pj, int i, unsigned pi) {
    return pj > pi || (pj == pi && j > i);
}

// Whether some uncoloured neighbour in one list beats row i, a round of eight
// columns' loads at a time.
__device__ __forceinline__ bool jp_beaten(int i, unsigned pi, const int *__restrict__ p, const int *__restrict__ q,
                                          const int *__restrict__ color) {
    const int k1 = p[i + 1];
    for (int k = p[i]; k < k1; k += 8) {
        int j[8], c[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) j[u] = k + u < k1 ? q[k + u] : i;
#pragma unroll
        for (int u = 0; u < 8; ++u) c[u] = color[j[u]];
        bool lost = false;
#pragma unroll
        for (int u = 0; u < 8; ++u) lost = lost || (j[u] != i && c[u] < 0 && beats(j[u], jp_priority(j[u]), i, pi));
        if (lost) return true;
    }
    return false;
}

__device__ __forceinline__ unsigned long long jp_used(int i, int base, const int *__restrict__ p,
                                                      const int *__restrict__ q, const int *__restrict__ color) {
    unsigned long long used = 0ull;
    const int k1 = p[i + 1];
    for (int k = p[i]; k < k1; k += 8) {
        int j[8], c[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) j[u] = k + u < k1 ? q[k + u] : i;
#pragma unroll
        for (int u = 0; u < 8; ++u) c[u] = j[u] != i ? color[j[u]] - base : -1;
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (c[u] >= 0 && c[u] < 64) used |= 1ull << c[u];
    }
    return used;
}

// One Jones-Plassmann round over the pattern of A (ia/ja) and of A^T
// (ta/tj; null when the pattern is symmetric).  color_in[i] = -1 while row i is
// uncoloured.
__global__ void k_jp_round(int n, const int *__restrict__ ia, const int *__restrict__ ja,
                           const int *__restrict__ ta, const int *__restrict__ tj, const int *__restrict__ color_in,
                           int *__restrict__ color_out, int *__restrict__ left) {
    int local = 0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        int c = color_in[i];
        if (c < 0) {
            const unsigned pi = jp_priority(i);
            if (jp_beaten(i, pi, ia, ja, color_in) || (ta && jp_beaten(i, pi, ta, tj, color_in))) {
                ++local;
            } else {
                // smallest colour free among the coloured neighbours, 64 at a time
                for (int base = 0;; base += 64) {
                    unsigned long long used = jp_used(i, base, ia, ja, color_in);
                    if (ta) used |= jp_used(i, base, ta, tj, color_in);
                    if (~used) {
                        c = base + __ffsll((long long)~used) - 1;
                        break;
                    }
                }
            }
        }
        color_out[i] = c;
    }
    if (left) {
#pragma unroll
        for (int off = kWave / 2; off > 0; off >>= 1) local += __shfl_xor(local, off, kWave);
        if (threadIdx.x % kWave == 0 && local) atomicAdd(left, local);
    }
}

// *bad is set when some entry (i, j) has no (j, i).  16 lanes a row: a lane a
// row spent row length x row length dependent steps on a long one (a row of
// 30,000 entries: 15 ms).
constexpr int kSymmetricLanes = 16;
__global__ void k_gs_symmetric(int n, const int *__restrict__ ia, const int *__restrict__ ja, int *__restrict__ bad) {
    const int lane = threadIdx.x % kSymmetricLanes;
    const int step = gridDim.x * blockDim.x / kSymmetricLanes;
    for (int i = (blockIdx.x * blockDim.x + threadIdx.x) / kSymmetricLanes; i < n; i += step) {
        const int k1 = ia[i + 1];
        for (int k = ia[i] + lane; k < k1; k += kSymmetricLanes) {
            const int j = ja[k];
            if (j == i) continue;
            bool found = false;
            const int q1 = ia[j + 1];
            for (int q = ia[j]; q < q1 && !found; q += 8) {
                int c[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) c[u] = q + u < q1 ? ja[q + u] : -1;
#pragma unroll
                for (int u = 0; u < 8; ++u) found = found || c[u] == i;
            }
            if (!found) {
                *bad = 1;
                return;
            }
        }
    }
}

// rows per colour and info[0] = the largest colour; keys and idx for the sort
__global__ __launch_bounds__(kBlock) void k_color_hist(int n, const int *__restrict__ color, int *__restrict__ cnt,
                                                       int *__restrict__ info, unsigned int *__restrict__ keys,
                                                       int *__restrict__ idx) {
    __shared__ int h[kHistBins];
    for (int t = threadIdx.x; t < kHistBins; t += kBlock) h[t] = 0;
    __syncthreads();
    int most = 0;
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        const int c = color[i];
        keys[i] = (unsigned int)c;
        idx[i] = i;
        most = max(most, c);
        if (c < kHistBins) atomicAdd(&h[c], 1);
        else atomicAdd(&cnt[c], 1);
    }
    __syncthreads();
    for (int t = threadIdx.x; t < kHistBins; t += kBlock)
        if (h[t]) atomicAdd(&cnt[t], h[t]);
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) most = max(most, __shfl_xor(most, off, kWave));
    if (threadIdx.x % kWave == 0) atomicMax(info, most);
}

// One wave per slice: the rows at its positions, their positions, and the
// widest row's off-diagonal entries that a sweep reads (stored zeros are left
// out; the colouring sees the whole pattern).  cptr: first sorted row of each
// colour, sl0: first slice.  width: nslices + 1, the last 0.
__global__ __launch_bounds__(kBlock) void k_gs_place(int nslices, int nc, const int *__restrict__ cptr,
                                                     const int *__restrict__ sl0, const int *__restrict__ sorted,
                                                     const int *__restrict__ ia, const int *__restrict__ ja,
                                                     const double *__restrict__ a, int *__restrict__ rows,
                                                     int *__restrict__ pos_of, int *__restrict__ width,
                                                     int *__restrict__ info) {
    const int s = blockIdx.x * kSlicesPerBlock + threadIdx.x / kSlice;
    const int lane = threadIdx.x % kSlice;
    if (s >= nslices) return;
    int lo = 0, hi = nc - 1;   // the last colour whose first slice is not after s
    while (lo < hi) {
        const int mid = (lo + hi + 1) / 2;
        if (sl0[mid] <= s) lo = mid;
        else hi = mid - 1;
    }
    const int q = cptr[lo] + (s - sl0[lo]) * kSlice + lane;
    const int i = q < cptr[lo + 1] ? sorted[q] : -1;
    rows[s * kSlice + lane] = i;
    int w = 0;
    if (i >= 0) {
        pos_of[i] = s * kSlice + lane;
        for (int k = ia[i]; k < ia[i + 1]; ++k) w += ja[k] != i && a[k] != 0.0;
    }
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) w = max(w, __shfl_xor(w, off, kWave));
    if (lane == 0) {
        width[s] = w;
        if (s == 0) width[nslices] = 0;
        if (w > info[1]) atomicMax(info + 1, w);
    }
}

// Slice fill: one thread per position.  Columns are stored as positions
// (pos_of[j]): the sweeps work on vectors in that order, where the rows a
// colour's slice reads lie close together, as they do in the natural order.
__global__ void k_gs_fill(int nslices, int W, const int *__restrict__ place, const int *__restrict__ rows,
                          const int *__restrict__ pos_of,
                          const int *__restrict__ ia, const int *__restrict__ ja, const double *__restrict__ a,
                          int *__restrict__ col, double *__restrict__ val, double *__restrict__ diag) {
    const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= (long)nslices * kSlice) return;
    const int s = (int)(p / kSlice);
    const long long base = (place ? (long long)place[s] : (long long)s * W) * kSlice + p % kSlice;
    const int wd = place ? place[s + 1] - place[s] : W;
    const int i = rows[p];
    int k2 = 0;
    double d = 0.0;
    if (i >= 0)
        for (int k = ia[i]; k < ia[i + 1]; ++k) {
            const int j = ja[k];
            if (j == i) {
                d = a[k];
            } else if (a[k] != 0.0) {
                col[base + (long long)k2 * kSlice] = pos_of[j];
                val[base + (long long)k2 * kSlice] = a[k];
                ++k2;
            }
        }
    diag[p] = d;   // 0.0 at an empty position, whose value then stays
    for (; k2 < wd; ++k2) {
        col[base + (long long)k2 * kSlice] = (int)p;
        val[base + (long long)k2 * kSlice] = 0.0;
    }
}

// xp[p] = x[rows[p]] (0 where x is zero: x null), bp[p] = b[rows[p]]
__global__ void k_perm_in(int npos, const int *__restrict__ rows, const double *__restrict__ x,
                          const double *__restrict__ b, double *__restrict__ xp, double *__restrict__ bp) {
    for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < npos; p += gridDim.x * blockDim.x) {
        const int i = rows[p];
        xp[p] = x && i >= 0 ? x[i] : 0.0;
        bp[p] = i >= 0 ? b[i] : 0.0;
    }
}

// The update of one row from t = b_i - sum_{j != i} a_ij x_j (CSR order):
//   mode 0 (GS)  x_i = t * (1 / a_ii)          (smoother.c:140-146)
//   mode 1 (SGS) x_i = t / a_ii                (smoother.c:222-227)
//   mode 2 (SOR) x_i = w (t / a_ii) + (1 - w) x_i  (smoother.c:283-289)
// rows with |a_ii| <= SMALLREAL keep their value.
__device__ __forceinline__ double gs_update(int mode, double t, double d, double xo, double w) {
    if (!(fabs(d) > kSmallReal)) return xo;
    if (mode == 0) return t * (1.0 / d);
    if (mode == 1) return t / d;
    return w * (t / d) + (1 - w) * xo;
}

// A slice's first U entries in a lane's registers (zero past its width).
template <int U>
struct GsEntries {
    int c[U];
    double v[U];
};
template <bool kNt, int U>
__device__ __forceinline__ void gs_load(GsEntries<U> &e, const int *__restrict__ cp, const double *__restrict__ vp,
                                        int k, int width, int self) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const bool ok = k + u < width;
        const int *c = cp + (long long)(k + u) * kSlice;
        const double *v = vp + (long long)(k + u) * kSlice;
        e.c[u] = ok ? (kNt ? ld_nt(c) : *c) : self;
        e.v[u] = ok ? (kNt ? ld_nt(v) : *v) : 0.0;
    }
}
// t - sum of products, subtracted in entry order
template <int U, class XT>
__device__ __forceinline__ double gs_subtract(double t, const GsEntries<U> &e, const XT *x) {
    double xv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) xv[u] = x[e.c[u]];
#pragma unroll
    for (int u = 0; u < U; ++u) t -= e.v[u] * xv[u];
    return t;
}

// One colour (slices s0 .. s0 + ns - 1); a wave per slice.  xout (optional):
// the new values in the rows' own order as well (the colour's last visit).
// kNt: the entries stream past the caches (levels whose matrix does not stay
// there from one colour visit to the next).  kPlaces: the slices' own widths.
template <int kMode, int U, bool kNt, bool kPlaces>
__global__ void __launch_bounds__(kBlock) k_gs_color(int s0, int ns, int W, const int *__restrict__ place,
                                                     const int *__restrict__ rows, const int *__restrict__ col,
                                                     const double *__restrict__ val, const double *__restrict__ diag,
                                                     const double *__restrict__ bp, double *__restrict__ xp, double w,
                                                     double *__restrict__ xout) {
    const int sl = blockIdx.x * kSlicesPerBlock + threadIdx.x / kSlice;
    const int lane = threadIdx.x % kSlice;
    if (sl >= ns) return;
    const int s = s0 + sl, p = s * kSlice + lane;
    const int q0 = kPlaces ? place[s] : s;
    const int wd = kPlaces ? place[s + 1] - q0 : W;
    const int *cp = col + (kPlaces ? (long long)q0 : (long long)s * W) * kSlice + lane;
    const double *vp = val + (kPlaces ? (long long)q0 : (long long)s * W) * kSlice + lane;
    const double bi = bp[p], d = diag[p], xo = xp[p];
    const int row = xout ? rows[p] : -1;
    double t = bi;
    for (int k = 0; k < wd; k += U) {
        GsEntries<U> e;
        gs_load<kNt>(e, cp, vp, k, wd, p);
        t = gs_subtract(t, e, xp);
    }
    const double xn = gs_update(kMode, t, d, xo, w);
    xp[p] = xn;
    if (row >= 0) xout[row] = xn;
}

// Whole smoothing call of a small level in one workgroup, x held in LDS: the
// passes in turn, the colours of a pass in turn, a barrier after each colour.
// Same arithmetic as k_gs_color.  The slices a wave visits are known ahead, so
// the entries of its next kGsAhead slices are on their way while one is
// computed, and the barrier waits for LDS only, not for those loads.
constexpr int kGsAhead = 2;
struct GsProgram {
    int npass;
    int forward[kGsMaxPass], mode[kGsMaxPass], skip[kGsMaxPass];
    double w[kGsMaxPass];
};

__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// kMixed: the passes differ in mode or weight (looked up per colour visit).
// kPlaces: the slices' own widths (their places are kept in LDS).  x and xout
// may be one vector: it is read into LDS before anything is written.
template <int U, int kThreads, bool kMixed, bool kPlaces>
__global__ void __launch_bounds__(kThreads) k_gs_lds(int npos, int ncolors, int W, const int *__restrict__ place,
                                                     int steps, const int *__restrict__ sl0, const int *__restrict__ rows,
                                                     const int *__restrict__ col, const double *__restrict__ val,
                                                     const double *__restrict__ diag, double *__restrict__ bp,
                                                     const double *__restrict__ b, const double *x, double *xout,
                                                     GsProgram prog) {
    extern __shared__ double xs[];
    __shared__ int ph_s0[kGsMaxPhase], ph_s1[kGsMaxPhase];
    __shared__ unsigned char ph_pass[kMixed ? kGsMaxPhase : 1];
    __shared__ int s_place[kPlaces ? kGsLdsPos / kSlice + 1 : 1];
    int nph = 0;
    for (int ps = 0; ps < prog.npass; ++ps) {
        const int count = ncolors - prog.skip[ps];
        for (int q = threadIdx.x; q < count; q += kThreads) {
            const int c = prog.forward[ps] ? q + prog.skip[ps] : ncolors - 1 - prog.skip[ps] - q;
            ph_s0[nph + q] = sl0[c];
            ph_s1[nph + q] = sl0[c + 1];
            if (kMixed) ph_pass[nph + q] = (unsigned char)ps;
        }
        nph += count;
    }
    if (kPlaces)
        for (int s = threadIdx.x; s <= npos / kSlice; s += kThreads) s_place[s] = place[s];
    for (int p = threadIdx.x; p < npos; p += kThreads) {
        const int i = rows[p];
        xs[p] = x && i >= 0 ? x[i] : 0.0;
        bp[p] = i >= 0 ? b[i] : 0.0;
    }
    __syncthreads();
    constexpr int kWaves = kThreads / kSlice;
    const int wave = threadIdx.x / kSlice, lane = threadIdx.x % kSlice;
    struct Slice {
        bool on;
        int p, pass;
        double bi, d;
        GsEntries<U> e;
    };
    const int total = nph * steps;   // a colour takes `steps` slices a wave at most
    const int mode0 = prog.mode[0];
    const double w0 = prog.w[0];
    const auto first = [&](int s) {   // of a lane's entries in slice s
        return (kPlaces ? (long long)s_place[s] : (long long)s * W) * kSlice + lane;
    };
    const auto width = [&](int s) { return kPlaces ? s_place[s + 1] - s_place[s] : W; };
    // the visit that is loaded next: colour visit ph, its step j
    int ph = 0, j = 0;
    auto load = [&](Slice &S) {
        const bool more = ph < nph;
        const int s = __builtin_amdgcn_readfirstlane(more ? ph_s0[ph] + wave + kWaves * j : 0);
        const int s1 = __builtin_amdgcn_readfirstlane(more ? ph_s1[ph] : 0);
        S.on = s < s1;
        if (kMixed) S.pass = more ? ph_pass[ph] : 0;
        if (++j == steps) {
            j = 0;
            ++ph;
        }
        if (!S.on) return;
        S.p = s * kSlice + lane;
        S.bi = bp[S.p];
        S.d = diag[S.p];
        const long long base = first(s);
        gs_load<false>(S.e, col + base, val + base, 0, width(s), S.p);
    };
    int done = 0;   // steps of the current visit
    auto compute = [&](Slice &S) {
        if (S.on) {
            double t = gs_subtract(S.bi, S.e, xs);
            const long long base = first(S.p / kSlice);
            const int wd = width(S.p / kSlice);
            for (int k = U; k < wd; k += U) {
                GsEntries<U> e;
                gs_load<false>(e, col + base, val + base, k, wd, S.p);
                t = gs_subtract(t, e, xs);
            }
            const int mode = kMixed ? prog.mode[S.pass] : mode0;
            const double w = kMixed ? prog.w[S.pass] : w0;
            xs[S.p] = gs_update(mode, t, S.d, xs[S.p], w);
        }
        if (++done == steps) {   // the same in every wave
            done = 0;
            lds_barrier();
        }
    };
    Slice S[kGsAhead];
#pragma unroll
    for (int q = 0; q < kGsAhead; ++q) load(S[q]);
    for (int idx = 0; idx < total; idx += kGsAhead)
#pragma unroll
        for (int q = 0; q < kGsAhead; ++q)
            if (idx + q < total) {   // the same in every wave
                compute(S[q]);
                load(S[q]);
            }
    __syncthreads();
    for (int p = threadIdx.x; p < npos; p += kThreads) {
        const int i = rows[p];
        if (i >= 0) xout[i] = xs[p];
    }
}

}  // namespace

bool is_gs_family(int smoother) {
    return smoother == HZ_SMOOTHER_GS || smoother == HZ_SMOOTHER_SGS || smoother == HZ_SMOOTHER_SOR ||
           smoother == HZ_SMOOTHER_SSOR || smoother == HZ_SMOOTHER_GSOR || smoother == HZ_SMOOTHER_SGSOR;
}

void gs_prepare(const DevCSR &A, GsLevel &G) {
    G = GsLevel();
    const int n = A.n;
    if (n == 0) return;
    hipStream_t st = stream();
    // colouring on the pattern of A + A^T: A's own where that is symmetric
    int *c0 = arena().alloc_n<int>((size_t)n + 1);
    int *c1 = arena().alloc_n<int>((size_t)n + 1);
    int *left = arena().alloc_n<int>(1);
    int h = 0;
    HZ_CHECK(hipMemsetAsync(left, 0, sizeof(int), st));
    k_gs_symmetric<<<grid_rows((long)n * kSymmetricLanes), kBlock, 0, st>>>(n, A.ia, A.ja, left);
    HZ_LAUNCH_CHECK();
    HZ_CHECK(memcpy_sync(&h, left, sizeof(int), hipMemcpyDeviceToHost));
    DevCSR AT;
    if (h) csr_transpose_gpu(A, AT);
    HZ_CHECK(hipMemsetAsync(c0, 0xff, sizeof(int) * n, st));
    // Rounds after the last one change nothing, so the count of uncoloured
    // rows is read back only every kCheck rounds.  Every round colours at
    // least the uncoloured row of highest priority: n rounds always suffice.
    constexpr int kCheck = 8;
    for (int round = 0; round <= n; round += kCheck) {
        HZ_CHECK(hipMemsetAsync(left, 0, sizeof(int), st));
        for (int r = 0; r < kCheck; ++r) {
            k_jp_round<<<grid_rows(n), kBlock, 0, st>>>(n, A.ia, A.ja, AT.ia, AT.ja, c0, c1,
                                                        r == kCheck - 1 ? left : nullptr);
            HZ_LAUNCH_CHECK();
            std::swap(c0, c1);
        }
        int hl = 0;
        HZ_CHECK(memcpy_sync(&hl, left, sizeof(int), hipMemcpyDeviceToHost));
        if (hl == 0) break;
    }
    // rows by colour: a stable sort keeps them ascending inside a colour
    int *info = arena().alloc_n<int>((size_t)n + 3);   // largest colour, widest row, then rows per colour
    int *cnt = info + 2;
    unsigned int *keys = arena().alloc_n<unsigned int>((size_t)n), *keys_out = arena().alloc_n<unsigned int>((size_t)n);
    int *idx = arena().alloc_n<int>((size_t)n), *sorted = arena().alloc_n<int>((size_t)n);
    HZ_CHECK(hipMemsetAsync(info, 0, sizeof(int) * ((size_t)n + 3), st));
    k_color_hist<<<std::min(256, div_up(n, kBlock)), kBlock, 0, st>>>(n, c0, cnt, info, keys, idx);
    HZ_LAUNCH_CHECK();
    const int first = std::min(n + 3, 258);
    std::vector<int> hi(first);
    HZ_CHECK(memcpy_sync(hi.data(), info, sizeof(int) * first, hipMemcpyDeviceToHost));
    const int nc = hi[0] + 1;
    if (nc + 2 > first) {
        hi.resize((size_t)nc + 2);
        HZ_CHECK(memcpy_sync(hi.data(), info, sizeof(int) * hi.size(), hipMemcpyDeviceToHost));
    }
    int bits = 1;
    while ((1u << bits) < (unsigned)nc && bits < 32) ++bits;
    size_t tmp_bytes = 0;
    HZ_CHECK(rocprim::radix_sort_pairs(nullptr, tmp_bytes, keys, keys_out, idx, sorted, (size_t)n, 0, bits, st));
    void *tmp = arena().alloc(tmp_bytes);
    HZ_CHECK(rocprim::radix_sort_pairs(tmp, tmp_bytes, keys, keys_out, idx, sorted, (size_t)n, 0, bits, st));
    G.n = n;
    G.ncolors = nc;
    G.cptr.assign(nc + 1, 0);
    G.sl0.assign(nc + 1, 0);
    G.most_slices = 0;
    for (int c = 0; c < nc; ++c) {
        const int ns = div_up(hi[2 + c], kSlice);
        G.cptr[c + 1] = G.cptr[c] + hi[2 + c];
        G.sl0[c + 1] = G.sl0[c] + ns;
        G.most_slices = std::max(G.most_slices, ns);
    }
    const int ns = G.sl0[nc];
    G.nslices = ns;
    G.npos = ns * kSlice;
    G.order = sorted;
    std::vector<int> tables(G.cptr);
    tables.insert(tables.end(), G.sl0.begin(), G.sl0.end());
    int *dtab = arena().alloc_n<int>(tables.size());
    HZ_CHECK(hipMemcpyAsync(dtab, tables.data(), sizeof(int) * tables.size(), hipMemcpyHostToDevice, st));
    G.dsl0 = dtab + nc + 1;
    G.rows = arena().alloc_n<int>((size_t)G.npos);
    // widths of the slices (and 0), then their places in units of kSlice entries
    int *width = arena().alloc_n<int>((size_t)ns + 1), *place = arena().alloc_n<int>((size_t)ns + 1);
    int *pos_of = c1;   // scratch: the colouring buffers are free now
    k_gs_place<<<div_up(ns, kSlicesPerBlock), kBlock, 0, st>>>(ns, nc, dtab, G.dsl0, sorted, A.ia, A.ja, A.val, G.rows,
                                                                pos_of, width, info);
    HZ_LAUNCH_CHECK();
    HZ_CHECK(memcpy_sync(&G.W, info + 1, sizeof(int), hipMemcpyDeviceToHost));
    // one width for all where it pads little, and on levels whose sweeps are
    // chains of loads while it adds no round of loads (16 entries); else the
    // slices' own (dense coarse levels of 4,052 and 1,067 rows, 909 to 1,353 the
    // longest: a call 8.4 ms at up to twice the entries)
    bool one_width = n <= 65536 && G.W <= 16;
    int total = 0;   // of kSlice entries
    if (!one_width) {
        HZ_CHECK(rocprim::exclusive_scan(nullptr, tmp_bytes, width, place, 0, (size_t)ns + 1, rocprim::plus<int>(), st));
        tmp = arena().alloc(tmp_bytes);
        HZ_CHECK(rocprim::exclusive_scan(tmp, tmp_bytes, width, place, 0, (size_t)ns + 1, rocprim::plus<int>(), st));
        HZ_CHECK(memcpy_sync(&total, place + ns, sizeof(int), hipMemcpyDeviceToHost));   // at most the matrix's entries
        one_width = (long long)ns * G.W <= 1.25 * total;
    }
    G.place = one_width ? nullptr : place;
    G.stream = n > 65536;
    const size_t room = (one_width ? (size_t)ns * G.W : (size_t)total) * kSlice + 1;
    if (trace_enabled())
        std::fprintf(stderr, "[hz]   Gauss-Seidel n=%d: %d colours, %d slices, longest row %d, %s\n", n, nc, ns, G.W,
                     one_width ? "one width" : "widths by slice");
    G.diag = arena().alloc_n<double>((size_t)G.npos);
    G.col = arena().alloc_n<int>(room);
    G.val = arena().alloc_n<double>(room);
    G.xp = arena().alloc_n<double>((size_t)G.npos);
    G.bp = arena().alloc_n<double>((size_t)G.npos);
    k_gs_fill<<<div_up(G.npos, kBlock), kBlock, 0, st>>>(ns, G.W, G.place, G.rows, pos_of, A.ia, A.ja, A.val, G.col, G.val,
                                                         G.diag);
    HZ_LAUNCH_CHECK();
    G.in_lds = G.npos <= kGsLdsPos;   // one workgroup where x and the rest fit LDS
}

namespace {

struct Pass {
    bool forward;
    int mode;      // as in gs_update
    double w;
    bool skip;     // skip the first colour visited (the backward half of SGS starts at n-2, smoother.c:236)
};

// dcsr_presmoothing (mgcycle.c:76-137, rows 0..n-1 step 1) and
// dcsr_postsmoothing (mgcycle.c:162-223, step -1) as a list of passes;
// smoother_dcsr_gs / _sor with L sweeps are L passes in one direction.
std::vector<Pass> gs_program(int smoother, bool post, int L, double relax) {
    std::vector<Pass> prog;
    auto call = [&](bool fwd, int mode, double w) {
        for (int s = 0; s < L; ++s) prog.push_back({fwd, mode, w, false});
    };
    constexpr bool F = true, B = false;
    switch (smoother) {
        case HZ_SMOOTHER_GS: call(post ? B : F, 0, 1.0); break;
        case HZ_SMOOTHER_SGS:   // smoother_dcsr_sgs: L times forward, backward
            for (int s = 0; s < L; ++s) {
                prog.push_back({F, 1, 1.0, false});
                prog.push_back({B, 1, 1.0, true});
            }
            break;
        case HZ_SMOOTHER_SOR: call(post ? B : F, 2, relax); break;
        case HZ_SMOOTHER_SSOR:
            call(F, 2, relax);
            call(B, 2, relax);
            break;
        case HZ_SMOOTHER_GSOR:
            if (!post) {
                call(F, 0, 1.0);
                call(B, 2, relax);
            } else {
                call(F, 2, relax);
                call(B, 0, 1.0);
            }
            break;
        case HZ_SMOOTHER_SGSOR:
            if (!post) {
                call(F, 0, 1.0);
                call(B, 0, 1.0);
                call(F, 2, relax);
                call(B, 2, relax);
            } else {
                call(F, 2, relax);
                call(B, 2, relax);
                call(F, 0, 1.0);
                call(B, 0, 1.0);
            }
            break;
        default: break;
    }
    return prog;
}

void color_launch(const GsLevel &G, int c, int mode, double w, double *xout) {
    const int s0 = G.sl0[c], ns = G.sl0[c + 1] - G.sl0[c];
    if (ns == 0) return;
    const int grid = div_up(ns, kSlicesPerBlock);
    auto launch = [&](auto m, auto u, auto nt, auto places) {
        k_gs_color<decltype(m)::value, decltype(u)::value, decltype(nt)::value, decltype(places)::value>
            <<<grid, kBlock, 0, stream()>>>(s0, ns, G.W, G.place, G.rows, G.col, G.val, G.diag, G.bp, G.xp, w, xout);
    };
    auto go = [&](auto m, auto u) {
        if (G.stream && G.place) launch(m, u, std::true_type{}, std::true_type{});
        else if (G.stream) launch(m, u, std::true_type{}, std::false_type{});
        else if (G.place) launch(m, u, std::false_type{}, std::true_type{});
        else launch(m, u, std::false_type{}, std::false_type{});
    };
    auto by_mode = [&](auto u) {
        if (mode == 0) go(std::integral_constant<int, 0>{}, u);
        else if (mode == 1) go(std::integral_constant<int, 1>{}, u);
        else go(std::integral_constant<int, 2>{}, u);
    };
    if (G.W <= 8) by_mode(std::integral_constant<int, 8>{});
    else by_mode(std::integral_constant<int, 16>{});
}

// The one-workgroup form: 16 waves with eight entries in flight for short
// rows, 8 waves with sixteen for longer ones (registers).
template <int U, int kThreads, bool kMixed, bool kPlaces>
void lds_launch_form(const GsLevel &G, const double *b, const double *x, double *xout, const GsProgram &gp) {
    static const bool ready = [] {
        HZ_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_gs_lds<U, kThreads, kMixed, kPlaces>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, kGsLdsPos * (int)sizeof(double)));
        return true;
    }();
    (void)ready;
    const int steps = std::max(1, div_up(G.most_slices, kThreads / kSlice));
    k_gs_lds<U, kThreads, kMixed, kPlaces><<<1, kThreads, sizeof(double) * G.npos, stream()>>>(
        G.npos, G.ncolors, G.W, G.place, steps, G.dsl0, G.rows, G.col, G.val, G.diag, G.bp, b, x, xout, gp);
    HZ_LAUNCH_CHECK();
}

template <int U, int kThreads, bool kMixed>
void lds_launch(const GsLevel &G, const double *b, const double *x, double *xout, const GsProgram &gp) {
    if constexpr (U > 8)   // levels of short rows have one width
        if (G.place) return lds_launch_form<U, kThreads, kMixed, true>(G, b, x, xout, gp);
    lds_launch_form<U, kThreads, kMixed, false>(G, b, x, xout, gp);
}

}  // namespace

void gs_smooth(const GsLevel &G, int smoother, bool post, int nsweeps, double relax, const double *b, double *x,
               bool x_zero) {
    const std::vector<Pass> prog = gs_program(smoother, post, nsweeps, relax);
    if (G.n == 0) return;
    if (prog.empty()) {
        if (x_zero) fill(x, 0.0, G.n);
        return;
    }
    hipStream_t st = stream();
    if (G.in_lds && G.ncolors <= kGsMaxPhase) {
        const size_t per = std::max<size_t>(1, std::min<size_t>(kGsMaxPass, kGsMaxPhase / G.ncolors));
        for (size_t p0 = 0; p0 < prog.size(); p0 += per) {
            GsProgram gp{};
            gp.npass = (int)std::min<size_t>(per, prog.size() - p0);
            for (int k = 0; k < gp.npass; ++k) {
                const Pass &P = prog[p0 + k];
                gp.forward[k] = P.forward;
                gp.mode[k] = P.mode;
                gp.skip[k] = (P.skip && G.ncolors > 0) ? 1 : 0;
                gp.w[k] = P.w;
            }
            const double *xin = x_zero && p0 == 0 ? nullptr : x;
            bool mixed = false;
            for (int k = 1; k < gp.npass; ++k) mixed = mixed || gp.mode[k] != gp.mode[0] || gp.w[k] != gp.w[0];
            if (mixed) {
                if (G.W <= 8) lds_launch<8, 1024, true>(G, b, xin, x, gp);
                else lds_launch<16, 512, true>(G, b, xin, x, gp);
            } else {
                if (G.W <= 8) lds_launch<8, 1024, false>(G, b, xin, x, gp);
                else lds_launch<16, 512, false>(G, b, xin, x, gp);
            }
        }
        return;
    }
    k_perm_in<<<grid_rows(G.npos), kBlock, 0, st>>>(G.npos, G.rows, x_zero ? nullptr : x, b, G.xp, G.bp);
    HZ_LAUNCH_CHECK();
    // a colour's last visit writes its rows of x as well
    std::vector<int> last(G.ncolors, -1);
    for (int k = 0; k < (int)prog.size(); ++k)
        for (int q = prog[k].skip ? 1 : 0; q < G.ncolors; ++q) last[prog[k].forward ? q : G.ncolors - 1 - q] = k;
    for (int k = 0; k < (int)prog.size(); ++k) {
        const Pass &P = prog[k];
        for (int q = P.skip ? 1 : 0; q < G.ncolors; ++q) {
            const int c = P.forward ? q : G.ncolors - 1 - q;
            color_launch(G, c, P.mode, P.w, last[c] == k ? x : nullptr);
        }
    }
    HZ_LAUNCH_CHECK();
}

}  // namespace hz
