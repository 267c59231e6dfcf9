// kernels_fused.hip -- the small levels' two cycle kernels on a layout of
// their own: residual + restriction (+ the coarse level's first sweep) going
// down, prolongation + first post-smoothing sweep going up.
//
// What bounds them: a level of up to a few 100,000 rows moves a few MB, so its
// launches (two a level and cycle, 16 to 20 a cycle) are chains of dependent
// loads, each 0.7-1 us through the last-level cache, and not bandwidth.
// Walking R's lists over the CSR rows took five loads in a row (row pointer,
// member, its row pointer, column, x) and the sweep four (slice pointer,
// column, aggregate of the column, coarse x).  Here the rows lie in the order
// in which the restriction adds them: a workgroup owns C consecutive coarse
// rows, its positions (their member rows, members ascending) are cut into K
// slices of 64, lane t of a slice holds one row, entry k of it at t + 64 k of
// the slice's piece, and every slice's piece has room for the level's longest
// row, so that its place is computed and not loaded.  Where that padding costs
// more than the load (fused_prepare) the pieces are as wide as their own longest
// row instead: one row of 60 entries in a level of 287,496 rows of 15 would
// otherwise take four times the level's memory, twice.
// Down is then (row, column, value) -> x -> LDS -> store, the row sums formed
// in the same order as over CSR.  It keeps the rows' residuals w, and up uses
// them: after the correction the residual is w - alpha (A P) xc, so the sweep
// needs the entries of A P (a row's entries merged by the aggregate of their
// column: 11 of 15, 6 of 7), one gather an entry and no second look at x:
// (aggregate, value) -> xc -> store.
// Measured (rocprofv3, FP64, 128^3 Poisson hierarchy): down 7.4 -> 5.0 us on
// the levels of 2,000 to 64,000 rows, 26 -> 10.7 us on 256,047 rows; up
// 7.0 -> 4.7 us and 10.8 -> 8.8 us.  One FP64 cycle at 80^3 (coefficient
// jumps) 275 -> 166 us, PCG of the 94-iteration 76^3 anisotropic solve
// 21.2 -> 16.4 ms.
#include <algorithm>
#include <vector>

#include <rocprim/device/device_scan.hpp>

#include "amg.hpp"

namespace hz {

namespace {

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / kWave;
constexpr int kTargetPos = 240;     // mean positions per workgroup: four slices, with room for uneven aggregates
constexpr int kMaxSlices = 32;      // per workgroup: aggregates of up to 8 times the mean size

// info[0]: the most positions of a workgroup, info[1]: the longest row,
// info[2]: positions in all (info[3] and info[4]: k_fused_fill's amax and dup)
__global__ __launch_bounds__(kBlock) void k_fused_info(int n, int nc, int C, const int *__restrict__ rptr,
                                                       const int *__restrict__ len, int *__restrict__ info) {
    int pos = 0, l = 0;
    const int nb = (nc + C - 1) / C;
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        l = max(l, len[i]);
        if (i < nb) pos = max(pos, rptr[min(nc, (i + 1) * C)] - rptr[i * C]);
    }
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) {
        pos = max(pos, __shfl_xor(pos, off, kWave));
        l = max(l, __shfl_xor(l, off, kWave));
    }
    if (threadIdx.x % kWave == 0) {
        if (pos > 0) atomicMax(info, pos);
        if (l > info[1]) atomicMax(info + 1, l);   // most waves find the maximum there already
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) info[2] = rptr[nc];
}

template <class MT>
__device__ __forceinline__ MT narrow_value(double v) {
    if constexpr (std::is_same_v<MT, unsigned short>) return f2bf((float)v);
    else return (MT)v;
}

// Width of every slice (and 0 after the last): its longest row.
__global__ __launch_bounds__(kBlock) void k_fused_width(int slices, int nc, int C, int K, const int *__restrict__ rptr,
                                                        const int *__restrict__ rmem, const int *__restrict__ len,
                                                        int *__restrict__ width) {
    const int s = blockIdx.x * kWaves + threadIdx.x / kWave, lane = threadIdx.x % kWave;
    if (s >= slices) return;
    const int blk = s / K, c0 = blk * C, c1 = min(nc, c0 + C);
    const int q = rptr[c0] + (s - blk * K) * kWave + lane;
    int w = q < rptr[c1] ? len[rmem[q]] : 0;
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) w = max(w, __shfl_xor(w, off, kWave));
    if (lane == 0) {
        width[s] = w;
        if (s == 0) width[slices] = 0;
    }
}

// First entry of slice s: places in units of kWave entries, or wmax apart.
__device__ __forceinline__ long long slice_base(const int *place, int s, int wmax) {
    return (place ? (long long)place[s] : (long long)s * wmax) * kWave;
}

// One wave per slice (and workgroup): its rows' entries from the SELL copy, and
// the same merged by the aggregate of their column, in order of its first
// entry, each sum in stored order (the merge runs in LDS).  amax: the longest
// merged row; *dup: set when a row stores its diagonal more than once.
constexpr int kMergeMax = 64;
template <class MT>
__global__ __launch_bounds__(kWave) void k_fused_fill(int nc, int C, int K, int wmax, const int *__restrict__ place,
                                                      const int *__restrict__ rptr, const int *__restrict__ rmem,
                                                      const int *__restrict__ agg, const int *__restrict__ len,
                                                      const long long *__restrict__ sptr,
                                                      const int *__restrict__ scol, const double *__restrict__ sval,
                                                      int *__restrict__ prow, int *__restrict__ pagg,
                                                      int *__restrict__ awidth, int *__restrict__ col, MT *__restrict__ val,
                                                      int *__restrict__ acol, MT *__restrict__ aval,
                                                      int *__restrict__ amax, int *__restrict__ dup) {
    extern __shared__ double s_merge[];   // wmax x 64 sums, then wmax x 64 aggregates
    double *m_val = s_merge;
    int *m_agg = reinterpret_cast<int *>(s_merge + (size_t)wmax * kWave);
    const int s = blockIdx.x, lane = threadIdx.x;
    const int blk = s / K, c0 = blk * C, c1 = min(nc, c0 + C);
    const int q = rptr[c0] + (s - blk * K) * kWave + lane;
    const int row = q < rptr[c1] ? rmem[q] : -1;
    prow[s * kWave + lane] = row;
    pagg[s * kWave + lane] = row >= 0 ? agg[row] : -1;
    const int l = row >= 0 ? len[row] : 0;
    const long long src = row >= 0 ? sptr[row / kSlice] + row % kSlice : 0;
    const long long dst = slice_base(place, s, wmax) + lane;
    const int w = place ? place[s + 1] - place[s] : wmax;
    int m = 0, ndiag = 0;   // merged entries, stored diagonals
    for (int k = 0; k < w; ++k) {
        const bool ok = k < l;
        const int c = ok ? scol[src + (long long)k * kSlice] : -1;
        const double a = ok ? sval[src + (long long)k * kSlice] : 0.0;
        col[dst + (long long)k * kWave] = c;
        val[dst + (long long)k * kWave] = narrow_value<MT>(a);
        if (ok) {
            ndiag += c == row;
            const int g = agg[c];
            int j = 0;
            while (j < m && m_agg[j * kWave + lane] != g) ++j;
            if (j == m) {
                m_agg[j * kWave + lane] = g;
                m_val[j * kWave + lane] = a;
                ++m;
            } else {
                m_val[j * kWave + lane] += a;
            }
        }
    }
    int wa = m;
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) wa = max(wa, __shfl_xor(wa, off, kWave));
    for (int k = 0; k < (place ? wa : wmax); ++k) {
        acol[dst + (long long)k * kWave] = k < m ? m_agg[k * kWave + lane] : -1;
        aval[dst + (long long)k * kWave] = narrow_value<MT>(k < m ? m_val[k * kWave + lane] : 0.0);
    }
    if (lane == 0) {
        awidth[s] = wa;
        if (wa > *amax) atomicMax(amax, wa);   // most waves find the maximum there already
    }
    if (ndiag > 1) *dup = 1;
}

__device__ __forceinline__ double wide(double v) { return v; }
__device__ __forceinline__ float wide(float v) { return v; }
__device__ __forceinline__ float wide(unsigned short v) { return __uint_as_float(((unsigned int)v) << 16); }

constexpr float kSmallRealF = 1e-20f;
// a sweep from zero at one row (FP64: the signs of zeros as k_smooth_from_zero forms them)
__device__ __forceinline__ double first_sweep(int smoother, double w, double b, double d) {
    if (!(fabs(d) > kSmallReal)) return 0.0;
    return smoother == HZ_SMOOTHER_L1DIAG ? 0.0 + b / d : (1 - w) * 0.0 + w * b / d;
}
__device__ __forceinline__ float first_sweep(int smoother, float w, float b, float d) {
    if (!(fabsf(d) > kSmallRealF)) return 0.0f;
    return smoother == HZ_SMOOTHER_L1DIAG ? b / d : w * b / d;
}

// Entries k .. k+U-1 of a position (index -1 and value 0 for padding and past wd).
template <int U, class VT, class MT>
__device__ __forceinline__ void ld_entries(const int *__restrict__ idx, const MT *__restrict__ val, long long base,
                                           int k, int wd, int (&cc)[U], VT (&vv)[U]) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const bool ok = k + u < wd;
        cc[u] = ok ? idx[base + (k + u) * kWave] : -1;
        vv[u] = ok ? wide(val[base + (k + u) * kWave]) : VT(0);
    }
}

// wpos = b - A x by position, bc = R (b - A x) and optionally xc = the coarse
// level's first sweep from zero.
template <class VT, class MT, int U, bool kPlaces>
__global__ __launch_bounds__(kBlock) void k_fused_down(int nc, int C, int K, int wmax, const int *__restrict__ place,
                                                       const int *__restrict__ rptr, const int *__restrict__ prow,
                                                       const int *__restrict__ col, const MT *__restrict__ val,
                                                       const VT *__restrict__ b, const VT *__restrict__ x,
                                                       VT *__restrict__ wpos, VT *__restrict__ bc, int smoother, VT wgt,
                                                       const VT *__restrict__ dc, VT *__restrict__ xc) {
    extern __shared__ double s_raw[];
    VT *s_w = reinterpret_cast<VT *>(s_raw);   // one residual a position
    const int blk = xcd_block_id();
    const int wv = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    // the second half's loads, issued ahead of the rows' chain
    const int c = blk * C + threadIdx.x;
    const bool own = (int)threadIdx.x < C && c < nc;
    const int p0 = rptr[blk * C];
    const int q0 = own ? rptr[c] : 0, q1 = own ? rptr[c + 1] : 0;
    const VT di = own && xc ? dc[c] : VT(0);
    for (int sl = wv; sl < K; sl += kWaves) {
        const int s = blk * K + sl;
        const int row = prow[s * kWave + lane];
        const int wd = kPlaces ? place[s + 1] - place[s] : wmax;
        const long long base = slice_base(kPlaces ? place : nullptr, s, wmax) + lane;
        const VT bi = row >= 0 ? b[row] : VT(0);
        VT t = 0;
        for (int k = 0; k < wd; k += U) {
            int cc[U];
            VT vv[U], xx[U];
            ld_entries<U>(col, val, base, k, wd, cc, vv);
#pragma unroll
            for (int u = 0; u < U; ++u) xx[u] = cc[u] >= 0 ? x[cc[u]] : VT(0);
#pragma unroll
            for (int u = 0; u < U; ++u) t = t + vv[u] * xx[u];   // padding adds 0 * 0
        }
        const VT w = bi - t;
        s_w[sl * kWave + lane] = w;
        wpos[s * kWave + lane] = w;
    }
    __syncthreads();
    if (!own) return;
    VT s = 0;
    for (int q = q0 - p0; q < q1 - p0; ++q) s = s + s_w[q];
    bc[c] = s;
    if (xc) xc[c] = first_sweep(smoother, wgt, s, di);
}

// xout = sweep(x'), x' = x + alpha P xc, whose residual is wpos - alpha (A P) xc:
//   Jacobi  x' + w r / d,  L1DIAG  x' + r / d  (rows with |d| <= SMALLREAL keep x').
// kOut 1: also partials of sum xout b; kOut 2: the result in FP64 to out64
// instead, with partials of sum out64 r64.
template <class VT, class MT, int kOut, int U, bool kPlaces>
__global__ __launch_bounds__(kBlock) void k_fused_up(int K, int wmax, int wd0, const int *__restrict__ place,
                                                     const int *__restrict__ awidth,
                                                     const int *__restrict__ prow, const int *__restrict__ pagg,
                                                     const int *__restrict__ acol, const MT *__restrict__ aval,
                                                     VT wgt, const VT *__restrict__ dsm, const VT *__restrict__ xc,
                                                     double alpha, const double *__restrict__ alpha_dev,
                                                     const VT *__restrict__ wpos, const VT *__restrict__ b,
                                                     const VT *__restrict__ x, VT *__restrict__ xout,
                                                     double *__restrict__ out64, const double *__restrict__ r64,
                                                     double *__restrict__ partials) {
    __shared__ double sh[kWaves];
    const int blk = xcd_block_id();
    const int wv = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const VT al = alpha_dev ? (VT)*alpha_dev : (VT)alpha;
    double prod = 0.0;
    for (int sl = wv; sl < K; sl += kWaves) {
        const int s = blk * K + sl;
        const int row = prow[s * kWave + lane], g = pagg[s * kWave + lane];
        const VT w = wpos[s * kWave + lane];
        const int wd = kPlaces ? awidth[s] : wd0;
        const long long base = slice_base(kPlaces ? place : nullptr, s, wmax) + lane;
        VT x0 = 0, xg0 = 0, d = 0, bi = 0;
        double ri = 0.0;
        VT t = 0;
        for (int k = 0; k < wd; k += U) {
            int cc[U];
            VT vv[U], xg[U];
            ld_entries<U>(acol, aval, base, k, wd, cc, vv);
            if (k == 0 && row >= 0) {   // beside the first round's gathers
                x0 = x[row];
                xg0 = xc[g];
                d = dsm[row];
                if (kOut == 1) bi = b[row];
                if (kOut == 2) ri = r64[row];
            }
#pragma unroll
            for (int u = 0; u < U; ++u) xg[u] = cc[u] >= 0 ? xc[cc[u]] : VT(0);
#pragma unroll
            for (int u = 0; u < U; ++u) t = t + vv[u] * xg[u];   // padding adds 0 * 0
        }
        if (row >= 0) {
            const VT xi = x0 + al * xg0;
            const VT r = w - al * t;
            const VT small = sizeof(VT) == 8 ? VT(kSmallReal) : VT(kSmallRealF);
            const VT xn = (d < 0 ? -d : d) > small ? xi + wgt * r / d : xi;
            if (kOut == 2) {
                const double z = (double)xn;
                out64[row] = z;
                prod += z * ri;
            } else {
                xout[row] = xn;
                if (kOut == 1) prod += (double)xn * (double)bi;
            }
        }
    }
    if (kOut) {
        const double bs = block_sum<kBlock>(prod, sh);
        if (threadIdx.x == 0) partials[blk] = bs;
    }
}

// Entries a round, and whether the slices have places: the longest row's, up
// to 32 where the whole row is one round of loads on the levels with a common
// width (latency-bound: a second round doubles the chain), up to 16 where the
// widths differ.
template <class F>
void by_width(int longest, bool places, F &&launch) {
    const auto go = [&](auto u) {
        if (places) launch(u, std::true_type{});
        else launch(u, std::false_type{});
    };
    if (longest <= 8) go(std::integral_constant<int, 8>{});
    else if (longest <= 16 || places) go(std::integral_constant<int, 16>{});
    else launch(std::integral_constant<int, 32>{}, std::false_type{});
}

template <class F>
void by_kind(int kind, F &&launch) {
    if (kind == 0) launch(double{});
    else if (kind == kLowF32) launch(float{});
    else launch((unsigned short)0);
}

}  // namespace

void fused_prepare(std::vector<Level *> &levels, const std::vector<int> &kinds, int smoother) {
    constexpr int kInfo = 5;
    const int nl = (int)levels.size();
    if (nl == 0) return;
    hipStream_t st = stream();
    int *info = arena().alloc_n<int>((size_t)nl * kInfo);
    HZ_CHECK(hipMemsetAsync(info, 0, sizeof(int) * nl * kInfo, st));
    for (int i = 0; i < nl; ++i) {
        Level &L = *levels[i];
        FusedLevel &F = L.F;
        F = FusedLevel();
        // coarse rows of a workgroup: the thread that adds a row's members is one of kBlock
        F.C = std::min<long>(kBlock, std::max<long>(1, (long)kTargetPos * L.nagg / L.A.n));
        F.nblk = div_up(L.nagg, F.C);
        k_fused_info<<<std::min(1024, div_up(std::max(L.A.n, F.nblk), kBlock)), kBlock, 0, st>>>(
            L.A.n, L.nagg, F.C, L.rptr, L.S.len, info + kInfo * i);
        HZ_LAUNCH_CHECK();
    }
    std::vector<int> h((size_t)nl * kInfo);
    HZ_CHECK(memcpy_sync(h.data(), info, sizeof(int) * nl * kInfo, hipMemcpyDeviceToHost));
    std::vector<int> total(nl, 0);   // of kWave entries
    bool placed = false;
    for (int i = 0; i < nl; ++i) {
        Level &L = *levels[i];
        FusedLevel &F = L.F;
        F.K = div_up(std::max(1, h[kInfo * i]), kWave);
        F.wmax = std::max(1, h[kInfo * i + 1]);
        F.kind = kinds[i];
        const long long slices = (long long)F.nblk * F.K, room = slices * kWave * F.wmax;
        // rows outside every aggregate, aggregates far from the mean size, or
        // rows too long for the merge or far longer than the others: the
        // list-walking kernels
        if (h[kInfo * i + 2] != L.A.n || F.K > kMaxSlices || F.wmax > kMergeMax || room > 8 * L.S.nent + (1 << 20))
            continue;
        F.slices = (int)slices;
        // a common width where the padding costs little, or on the latency-bound
        // levels while it is not many times the entries (measured: 1.1 to 3.7
        // times); else the slices' own widths
        if (L.A.n <= 65536 ? room > 4 * L.S.nent + (1 << 16) : room > L.S.nent + L.S.nent / 4) {
            int *width = arena().alloc_n<int>((size_t)slices + 1);
            F.place = arena().alloc_n<int>((size_t)slices + 1);
            k_fused_width<<<div_up(slices, kWaves), kBlock, 0, st>>>(F.slices, L.nagg, F.C, F.K, L.rptr, L.rmem, L.S.len,
                                                                     width);
            HZ_LAUNCH_CHECK();
            size_t tmp_bytes = 0;
            HZ_CHECK(rocprim::exclusive_scan(nullptr, tmp_bytes, width, F.place, 0, (size_t)slices + 1,
                                             rocprim::plus<int>(), st));
            void *tmp = arena().alloc(tmp_bytes);
            HZ_CHECK(rocprim::exclusive_scan(tmp, tmp_bytes, width, F.place, 0, (size_t)slices + 1,
                                             rocprim::plus<int>(), st));
            placed = true;
            HZ_CHECK(hipMemcpyAsync(&total[i], F.place + slices, sizeof(int), hipMemcpyDeviceToHost, st));
        } else {
            total[i] = (int)(slices * F.wmax);   // at most 8 S.nent + 2^20 entries of kWave
        }
        F.on = true;
    }
    if (placed) HZ_CHECK(hipStreamSynchronize(st));
    for (int i = 0; i < nl; ++i) {
        Level &L = *levels[i];
        FusedLevel &F = L.F;
        if (!F.on) continue;
        const int slices = F.slices;
        const size_t room = (size_t)total[i] * kWave;
        F.prow = arena().alloc_n<int>((size_t)slices * kWave);
        F.pagg = arena().alloc_n<int>((size_t)slices * kWave);
        F.awidth = arena().alloc_n<int>((size_t)slices);
        F.col = arena().alloc_n<int>(room);
        F.acol = arena().alloc_n<int>(room);
        F.wpos = arena().alloc((size_t)slices * kWave * (F.kind == 0 ? sizeof(double) : sizeof(float)));
        by_kind(F.kind, [&](auto m) {
            using MT = decltype(m);
            MT *v = arena().alloc_n<MT>(room), *av = arena().alloc_n<MT>(room);
            F.val = v;
            F.aval = av;
            k_fused_fill<MT><<<slices, kWave, (size_t)F.wmax * kWave * (sizeof(double) + sizeof(int)), st>>>(
                L.nagg, F.C, F.K, F.wmax, F.place, L.rptr, L.rmem, L.agg, L.S.len, L.S.sptr, L.S.col, L.S.val, F.prow,
                F.pagg, F.awidth, F.col, v, F.acol, av, info + kInfo * i + 3, info + kInfo * i + 4);
        });
        HZ_LAUNCH_CHECK();
    }
    HZ_CHECK(memcpy_sync(h.data(), info, sizeof(int) * nl * kInfo, hipMemcpyDeviceToHost));
    for (int i = 0; i < nl; ++i) {
        levels[i]->F.amax = std::max(1, h[kInfo * i + 3]);
        // Jacobi divides by the last stored diagonal entry and leaves every
        // one out of its sum: not a residual when a row stores several
        if (smoother == HZ_SMOOTHER_JACOBI && h[kInfo * i + 4]) levels[i]->F.on = false;
    }
}

template <class VT>
static void fused_down_impl(const Level &L, const VT *b, const VT *x, VT *bc, int smoother, double w, const VT *dc,
                            VT *xc) {
    const FusedLevel &F = L.F;
    const int vb = F.kind == 0 ? 8 : (F.kind == kLowF32 ? 4 : 2);
    count_bytes((vb + 4.0) * L.S.nnz + (4.0 + 3.0 * sizeof(VT)) * L.A.n + 4.0 * (L.nagg + 1) +
                (xc ? 3.0 : 1.0) * sizeof(VT) * L.nagg);
    by_width(F.wmax, F.place != nullptr, [&](auto u, auto places) {
        constexpr int U = decltype(u)::value;
        constexpr bool kPlaces = decltype(places)::value;
        auto go = [&](auto m) {
            using MT = decltype(m);
            k_fused_down<VT, MT, U, kPlaces><<<F.nblk, kBlock, sizeof(VT) * F.K * kWave, stream()>>>(
                L.nagg, F.C, F.K, F.wmax, F.place, L.rptr, F.prow, F.col, static_cast<const MT *>(F.val), b, x,
                static_cast<VT *>(F.wpos), bc, smoother, (VT)w, dc, xc);
        };
        if constexpr (sizeof(VT) == 8) go(double{});
        else if (F.kind == kLowF32) go(float{});
        else go((unsigned short)0);
    });
    HZ_LAUNCH_CHECK();
}

template <class VT>
static void fused_up_impl(const Level &L, int smoother, double w, const VT *dsm, const VT *xc, double alpha,
                          const double *alpha_dev, const VT *b, const VT *x, VT *xout, double *out64,
                          const double *r64, double *dot_out, const ReduceWs &ws) {
    const FusedLevel &F = L.F;
    const int vb = F.kind == 0 ? 8 : (F.kind == kLowF32 ? 4 : 2);
    // (the merged entries are counted as the row's own)
    count_bytes((vb + 4.0) * L.S.nnz + (8.0 + 4.0 * sizeof(VT)) * L.A.n + (out64 ? 16.0 * L.A.n : 0.0));
    double *part = dot_out || out64 ? ws.dots(F.nblk) : nullptr;
    const VT wgt = smoother == HZ_SMOOTHER_L1DIAG ? VT(1) : (VT)w;
    by_width(F.amax, F.place != nullptr, [&](auto u, auto places) {
        constexpr int U = decltype(u)::value;
        constexpr bool kPlaces = decltype(places)::value;
        auto launch = [&](auto m, auto out) {
            using MT = decltype(m);
            k_fused_up<VT, MT, decltype(out)::value, U, kPlaces><<<F.nblk, kBlock, 0, stream()>>>(
                F.K, F.wmax, F.amax, F.place, F.awidth, F.prow, F.pagg, F.acol, static_cast<const MT *>(F.aval), wgt, dsm,
                xc, alpha, alpha_dev, static_cast<const VT *>(F.wpos), b, x, xout, out64, r64, part);
        };
        if constexpr (sizeof(VT) == 8) {
            if (dot_out) launch(double{}, std::integral_constant<int, 1>{});
            else launch(double{}, std::integral_constant<int, 0>{});
        } else {
            auto by_out = [&](auto m) {
                if (out64) launch(m, std::integral_constant<int, 2>{});
                else launch(m, std::integral_constant<int, 0>{});
            };
            if (F.kind == kLowF32) by_out(float{});
            else by_out((unsigned short)0);
        }
    });
    HZ_LAUNCH_CHECK();
    if (dot_out) finish_dot(ws, F.nblk, dot_out);
}

void fused_down(const Level &L, const double *b, const double *x, double *bc, int smoother, double w, const double *dc,
                double *xc) {
    fused_down_impl<double>(L, b, x, bc, smoother, w, dc, xc);
}
void fused_down(const Level &L, const float *b, const float *x, float *bc, int smoother, double w, const float *dc,
                float *xc) {
    fused_down_impl<float>(L, b, x, bc, smoother, w, dc, xc);
}
void fused_up(const Level &L, int smoother, double w, const double *xc, double alpha, const double *alpha_dev,
              const double *b, const double *x, double *xout, double *dot_out, const ReduceWs &ws) {
    fused_up_impl<double>(L, smoother, w, L.dsm, xc, alpha, alpha_dev, b, x, xout, nullptr, nullptr, dot_out, ws);
}
void fused_up(const Level &L, int smoother, double w, const float *xc, const float *b, const float *x, float *xout,
              double *out64, const double *r64, double *dot_out, const ReduceWs &ws) {
    fused_up_impl<float>(L, smoother, w, L.dsmf, xc, 1.0, nullptr, b, x, xout, out64, r64, dot_out, ws);
}

}  // namespace hz
