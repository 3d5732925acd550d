// qp_solver_kernels.h -- the three launches of the periodic 2D solve.
// Sources (what the row-forward pass reads) and sinks (what the row-inverse
// pass does with each real output) are small functors so the fused slice
// step can assemble sources and finalise fields inside the transform launches.
//
// Batches: blockIdx.y = wake * nspec + which.  `which` selects spec0 / spec1
// (two independent solves of one wake, e.g. B_y and B_z), `wake` offsets the
// spectra by sstride and the control block by one Ctl; sources and sinks get
// (wake, which) and offset their own grids.
#pragma once

#include <algorithm>

#include "qp_fft_lds.h"

namespace qp {

// skip_mode: 0 never, 1 skip when stop_acc (and latch stop_now), 2 skip when stop_now.
// ctl: the control block of this block's wake (or null).  The flag is loaded at kernel
// start, next to the data loads, and acted on when they arrive, so that a launch does
// not begin with a round trip to memory of its own.  (Loads are safe whatever it says.)
__device__ __forceinline__ int solver_skip_flag(const Ctl *ctl, int skip_mode) {
    if (!ctl || skip_mode == 0) return 0;
    return skip_mode == 1 ? ctl->stop_acc : ctl->stop_now;
}
__device__ __forceinline__ bool solver_skip_act(const Ctl *ctl, int skip_mode, int flag) {
    if (flag != 0 && skip_mode == 1) ctl_latch(const_cast<Ctl *>(ctl));
    return flag != 0;
}
// A caller without a control block (a solve by itself, envelope steps) passes NoCtl: its
// launches hold nothing of the flag, and their loads need not be kept ahead of it.  A plain
// 1024^2 solve 26.15 -> 25.81 us, with the inverse rows' staged spectrum combined as it is
// read from LDS (93 -> 86 VGPRs).
struct NoCtl {};
__device__ __forceinline__ int solver_skip_flag(NoCtl, int) { return 0; }
__device__ __forceinline__ bool solver_skip_act(NoCtl, int, int) { return false; }
__device__ __forceinline__ const Ctl *ctl_of(const Ctl *c, int wk) { return c ? c + wk : c; }
__device__ __forceinline__ NoCtl ctl_of(NoCtl c, int) { return c; }

// Keeps the computation of x ahead of what follows (the compiler would move
// loads used only behind a branch below it).
__device__ __forceinline__ void keep_here(double &x) { asm volatile("" : "+v"(x)); }
template <int E>
__device__ __forceinline__ void keep_here(double2 (&v)[E]) {
#pragma unroll
    for (int r = 0; r < E; ++r) {
        keep_here(v[r].x);
        keep_here(v[r].y);
    }
}
// The same where a skip flag is acted on next.
template <int E>
__device__ __forceinline__ void keep_for_skip(const Ctl *, double2 (&v)[E]) {
    keep_here(v);
}
template <int E>
__device__ __forceinline__ void keep_for_skip(NoCtl, double2 (&)[E]) {}

// Sum over the wavefront, the same value in every lane: DPP moves inside each
// 16-lane row (lane ^ 1, lane ^ 2, half-row mirror, row mirror), then the four
// rows by readlane.  Every lane of the wavefront must call it.
template <int CTRL>
__device__ __forceinline__ double dpp_row_d(double x) {
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_mov_dpp((int)(b & 0xffffffffLL), CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xF, 0xF, false);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}
__device__ __forceinline__ double readlane_d(double x, int lane) {
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffLL), lane);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}
__device__ __forceinline__ double wave_sum(double x) {
    x += dpp_row_d<0xB1>(x);   // quad_perm(1, 0, 3, 2)
    x += dpp_row_d<0x4E>(x);   // quad_perm(2, 3, 0, 1)
    x += dpp_row_d<0x141>(x);  // row_half_mirror
    x += dpp_row_d<0x140>(x);  // row_mirror
    return (readlane_d(x, 0) + readlane_d(x, 16)) + (readlane_d(x, 32) + readlane_d(x, 48));
}

// A source hands out elements k0, k0 + dk, ... of row j (row), all loads before
// the arithmetic, and is told when they have been read (done).  TAIL: elements past
// the row's end are asked for as well (row: any value; done: leaves them alone).
template <bool TAIL>
__device__ __forceinline__ int row_k(int k, int n2) {
    return TAIL ? min(k, n2 - 1) : k;
}
struct SrcPlain {
    const double *a;
    int n2;
    template <int E, bool TAIL = false>
    __device__ void row(int, int, int j, int k0, int dk, double (&x)[E]) const {
#pragma unroll
        for (int r = 0; r < E; ++r) x[r] = a[(size_t)j * n2 + row_k<TAIL>(k0 + dk * r, n2)];
    }
    template <int E, bool TAIL = false>
    __device__ void done(int, int, int, int, int) const {}
};

// Real output v of the unnormalised c2r; the reference divides by n1 then n2
// (src/System_3d.cpp:361).
//
// A sink is prepared (prep: loads of its own are issued) ahead of the transform
// and begun (begin) after it, before it takes the outputs.
struct SinkScaled {
    double *dst;
    int n1, n2;
    __device__ void prep(int) {}
    __device__ void begin(int) {}
    __device__ void operator()(int, int, int j, int k, double v) const { dst[(size_t)j * n2 + k] = v / n1 / n2; }
};

// Raw unnormalised c2r output (Fourier2d::backward_transform semantics).
struct SinkRaw {
    double *dst;
    int n2;
    __device__ void prep(int) {}
    __device__ void begin(int) {}
    __device__ void operator()(int, int, int j, int k, double v) const { dst[(size_t)j * n2 + k] = v; }
};

// ------------------------------------------------ generic kernels (any side up to 1024)
// Spectrum element (row j, frequency l) at j * sj + l * sl: column-major (sj = 1,
// sl = n1) for the solves, so that column transforms read and write contiguous
// memory, row-major (sj = nh, sl = 1) for Fourier2d.  ONE: blocks of one wavefront.
constexpr int kGenThreads = 256;
__device__ __forceinline__ double2 swap_parts(double2 v) { return make_double2(v.y, v.x); }

// Rows forward: two real rows (2p, 2p+1) packed as z = x_a + i x_b, complex
// FFT along n2, then X_a[k] = (Z[k] + conj Z[-k])/2, X_b[k] = (Z[k] - conj Z[-k])/(2i).
// One row pair per block.
template <class Src, bool ONE>
__global__ __launch_bounds__(kGenThreads) void k_rows_fwd(Src src, double2 *spec0, double2 *spec1, int n1, int n2,
                                                          int nh, FftAxisDev ax, const Ctl *ctl, int skip_mode,
                                                          int nspec, size_t sstride, int sj, int sl) {
    constexpr int E = 4;  // n2 <= E threads
    const int which = blockIdx.y % nspec, wk = blockIdx.y / nspec;
    if (ctl) ctl += wk;
    const int skip = solver_skip_flag(ctl, skip_mode);
    double2 *spec = (which == 0 ? spec0 : spec1) + wk * sstride;
    extern __shared__ double2 lds[];
    double2 *a = lds, *b = lds + n2, *twl = lds + 2 * n2;
    const int ra = 2 * blockIdx.x, rb = ra + 1, T = blockDim.x, k0 = threadIdx.x;
    LdsTw tw;
    tw.load(ax);
    double xa[E], xb[E];
    src.template row<E, true>(wk, which, ra, k0, T, xa);
    if (rb < n1) {
        src.template row<E, true>(wk, which, rb, k0, T, xb);
    } else {
#pragma unroll
        for (int r = 0; r < E; ++r) xb[r] = 0.0;
    }
#pragma unroll
    for (int r = 0; r < E; ++r)
        if (k0 + r * T < n2) a[k0 + r * T] = make_double2(xa[r], xb[r]);
    if (solver_skip_act(ctl, skip_mode, skip)) return;
    tw.store(twl, n2);
    lds_sync<ONE>();
    src.template done<E, true>(wk, which, ra, k0, T);
    if (rb < n1) src.template done<E, true>(wk, which, rb, k0, T);
    const double2 *z = lds_fft<ONE>(a, b, ax, twl);
#pragma unroll
    for (int r = 0; r < E; ++r) {
        const int k = k0 + r * T;
        if (k >= nh) break;
        const double2 Z = z[k];
        const double2 Zm = z[k == 0 ? 0 : n2 - k];
        const double cr = Zm.x, ci = -Zm.y;
        double2 *o = spec + (ra * sj + k * sl);
        o[0] = make_double2(0.5 * (Z.x + cr), 0.5 * (Z.y + ci));
        if (rb < n1) o[sj] = make_double2(0.5 * (Z.y - ci), -0.5 * (Z.x - cr));
    }
}

// Columns: kColsSolve forward along n1, drop (0,0), divide by the eigenvalue
// -D + lam1[m] + lam2[l], inverse; kColsForward / kColsInverse one way only
// (Fourier2d).  One column per block.  With bpart != nullptr (psi solves) also the
// border-mean partial sums, as in wcols_body.
enum { kColsForward = 0, kColsInverse = 1, kColsSolve = 2 };
template <bool ONE>
__global__ __launch_bounds__(kGenThreads) void k_cols(double2 *spec0, double2 *spec1, int n1, int n2, FftAxisDev ax,
                                                      const double *lam1, const double *lam2, double D, double *bpart,
                                                      const Ctl *ctl, int skip_mode, int mode, int nspec,
                                                      size_t sstride, size_t bstride, int sj, int sl) {
    constexpr int E = 4;  // n1 <= E threads
    const int which = blockIdx.y % nspec, wk = blockIdx.y / nspec;
    if (ctl) ctl += wk;
    const int skip = solver_skip_flag(ctl, skip_mode);
    extern __shared__ double2 lds[];
    double2 *a = lds, *b = lds + n1, *twl = lds + 2 * n1;
    const int l = blockIdx.x, T = blockDim.x, j0 = threadIdx.x;
    double2 *spec = (which == 0 ? spec0 : spec1) + (wk * sstride + l * sl);
    LdsTw tw;
    tw.load(ax);
    double2 v[E];
    double lm[E];
#pragma unroll
    for (int r = 0; r < E; ++r) {
        const int j = min(j0 + r * T, n1 - 1);
        v[r] = spec[j * sj];
        lm[r] = mode == kColsSolve ? lam1[j] : 0.0;
    }
    const double l2 = mode == kColsSolve ? lam2[l] : 0.0;
#pragma unroll
    for (int r = 0; r < E; ++r)
        if (j0 + r * T < n1) a[j0 + r * T] = mode == kColsInverse ? swap_parts(v[r]) : v[r];
    if (solver_skip_act(ctl, skip_mode, skip)) return;
    tw.store(twl, n1);
    lds_sync<ONE>();
    double2 *o = a, *t = b;
    double s1 = 0.0, s2 = 0.0;
    // one copy of the transform's code for both directions: a launch starts with a cold
    // instruction cache, and what it fetches once it need not fetch again
#pragma unroll 1
    for (int pass = 0;; ++pass) {
        double2 *in = o;
        o = lds_fft<ONE>(in, t, ax, twl);
        t = o == in ? t : in;
        if (pass == 1 || mode != kColsSolve) break;
#pragma unroll
        for (int r = 0; r < E; ++r) {
            const int m = j0 + r * T;
            if (m < n1) {
                // v / mult with one division for both parts, each quotient corrected by
                // its remainder
                const double2 x = o[m];
                const double mult = -D + lm[r] + l2, inv = 1.0 / mult;
                double2 q = make_double2(x.x * inv, x.y * inv);
                q.x = fma(fma(-q.x, mult, x.x), inv, q.x);
                q.y = fma(fma(-q.y, mult, x.y), inv, q.y);
                if (m == 0 && l == 0) q = make_double2(0.0, 0.0);
                if (m == 0) s1 = q.x;
                s2 += q.x;
                o[m] = swap_parts(q);
            }
        }
        lds_sync<ONE>();
    }
#pragma unroll
    for (int r = 0; r < E; ++r) {
        const int j = j0 + r * T;
        if (j < n1) spec[j * sj] = mode == kColsForward ? o[j] : swap_parts(o[j]);
    }
    if (bpart) {
        bpart += wk * bstride;
        const double wl = (l == 0 || 2 * l == n2) ? 1.0 : 2.0;
        double g00 = wave_sum(s2);
        if constexpr (!ONE) {
            __shared__ double part[kGenThreads / 64];
            if ((j0 & 63) == 0) part[j0 >> 6] = g00;
            __syncthreads();
            g00 = 0.0;
            for (int i = 0; i < T >> 6; ++i) g00 += part[i];
        }
        if (j0 == 0) {  // (thread 0 holds element 0)
            bpart[2 * l] = wl * (double)n1 * s1;
            bpart[2 * l + 1] = wl * g00;
            if (l == 0) bpart[2 * gridDim.x] = g00;
        }
    }
}

// Rows inverse (c2r): Z[k] = X[k] + i Y[k] with the Hermitian extension
// X[-k] = conj X[k]; imaginary parts of the k = 0 and k = n2/2 terms ignored
// (FFTW c2r semantics).  Re z -> row 2p, Im z -> row 2p+1.
template <class Sink, bool ONE>
__global__ __launch_bounds__(kGenThreads) void k_rows_inv(const double2 *spec0, const double2 *spec1, Sink sink, int n1,
                                                          int n2, int nh, FftAxisDev ax, const Ctl *ctl, int skip_mode,
                                                          int nspec, size_t sstride, int sj, int sl) {
    constexpr int E = 4, EH = 3;  // n2 <= E threads, nh = n2/2 + 1 <= EH threads
    const int which = blockIdx.y % nspec, wk = blockIdx.y / nspec;
    if (ctl) ctl += wk;
    const int skip = solver_skip_flag(ctl, skip_mode);
    const double2 *spec = (which == 0 ? spec0 : spec1) + wk * sstride;
    extern __shared__ double2 lds[];
    double2 *a = lds, *b = lds + n2, *twl = lds + 2 * n2;
    const int ra = 2 * blockIdx.x, rb = ra + 1, T = blockDim.x, k0 = threadIdx.x;
    LdsTw tw;
    tw.load(ax);
    double2 X[EH], Y[EH];
#pragma unroll
    for (int e = 0; e < EH; ++e) {
        const double2 *p = spec + (ra * sj + min(k0 + e * T, nh - 1) * sl);
        X[e] = p[0];
        Y[e] = p[rb < n1 ? sj : 0];
    }
    sink.prep(wk);
#pragma unroll
    for (int e = 0; e < EH; ++e) {
        const int k = k0 + e * T;
        if (k < nh) {
            if (rb >= n1) Y[e] = make_double2(0.0, 0.0);
            const bool self = k == 0 || 2 * k == n2;
            if (self) X[e].y = Y[e].y = 0.0;
            // parts swapped: forward again for the inverse
            a[k] = make_double2(X[e].y + Y[e].x, X[e].x - Y[e].y);
            if (!self) a[n2 - k] = make_double2(Y[e].x - X[e].y, X[e].x + Y[e].y);
        }
    }
    if (solver_skip_act(ctl, skip_mode, skip)) return;
    tw.store(twl, n2);
    lds_sync<ONE>();
    const double2 *z = lds_fft<ONE>(a, b, ax, twl);
    sink.begin(wk);
#pragma unroll
    for (int r = 0; r < E; ++r) {
        const int k = k0 + r * T;
        if (k < n2) {
            const double2 v = z[k];
            sink(wk, which, ra, k, v.y);
            if (rb < n1) sink(wk, which, rb, k, v.x);
        }
    }
}

// ------------------------------------------------------------ launchers
// One transform per block.  LDS: two data buffers and the twiddle table.
#define QP_GEN_LAUNCH(kern1, kernN, grid, ax, ...)                                                             \
    do {                                                                                                       \
        const int threads = (ax).dev.threads;                                                                  \
        const size_t lds = sizeof(double2) * 3 * (size_t)(ax).dev.n;                                           \
        if (threads == 64) hipLaunchKernelGGL(kern1, grid, dim3(64), lds, s, __VA_ARGS__);                     \
        else hipLaunchKernelGGL(kernN, grid, dim3(threads), lds, s, __VA_ARGS__);                              \
        QP_HIP_CHECK(hipGetLastError());                                                                       \
    } while (0)

// nw wakes of one batch: spectra of wake w at spec0/spec1 + w * n1 * nh, control
// blocks at ctl + w.  fftw: row-major spectrum.
template <class Src>
int glaunch_rows_fwd(const Solver2d &S, const Src &src, double2 *spec0, double2 *spec1, int nspec, hipStream_t s,
                     const Ctl *ctl, int skip_mode, int nw = 1, bool fftw = false) {
    QP_GEN_LAUNCH((k_rows_fwd<Src, true>), (k_rows_fwd<Src, false>), dim3((S.n1 + 1) / 2, nspec * nw), S.ax2, src, spec0,
                  spec1, S.n1, S.n2, S.nh, S.ax2.dev, ctl, skip_mode, nspec, (size_t)S.n1 * S.nh, fftw ? S.nh : 1,
                  fftw ? 1 : S.n1);
    return QP_OK;
}
inline int glaunch_cols(const Solver2d &S, int mode, double D, int nspec, double *bpart, hipStream_t s, const Ctl *ctl,
                        int skip_mode, int nw = 1, size_t bstride = 0, bool fftw = false) {
    QP_GEN_LAUNCH(k_cols<true>, k_cols<false>, dim3(S.nh, nspec * nw), S.ax1, S.spec[0], S.spec[1], S.n1, S.n2,
                  S.ax1.dev, (const double *)S.d_lam1, (const double *)S.d_lam2, D, bpart, ctl, skip_mode, mode, nspec,
                  (size_t)S.n1 * S.nh, bstride, fftw ? S.nh : 1, fftw ? 1 : S.n1);
    return QP_OK;
}
template <class Sink>
int glaunch_rows_inv(const Solver2d &S, const double2 *spec0, const double2 *spec1, const Sink &sink, int nspec,
                     hipStream_t s, const Ctl *ctl, int skip_mode, int nw = 1, bool fftw = false) {
    QP_GEN_LAUNCH((k_rows_inv<Sink, true>), (k_rows_inv<Sink, false>), dim3((S.n1 + 1) / 2, nspec * nw), S.ax2, spec0,
                  spec1, sink, S.n1, S.n2, S.nh, S.ax2.dev, ctl, skip_mode, nspec, (size_t)S.n1 * S.nh,
                  fftw ? S.nh : 1, fftw ? 1 : S.n1);
    return QP_OK;
}

}  // namespace qp
