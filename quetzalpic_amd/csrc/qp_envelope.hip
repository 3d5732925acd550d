// qp_envelope.hip -- laser-envelope advance (no counterpart in the reference).
//
// Equation (x toward the front, slice i at x = i dx, tau the time of the
// moving window, a the complex envelope of the vector potential
// Re[a exp(i k0 (x - t))]):
//     lap_perp a + 2 d_tau (d_x + i k0) a = chi a.
// One step tau -> tau + dt, slices swept from the front (i = nx - 1) down to
// 0 like the wake, with d_i = a+_i - a_i (Crank-Nicolson in tau, d_x as the
// difference toward the front, d_{nx} = 0):
//     (2/dx)(d_{i+1} - d_i) + 2 i k0 d_i = (dt/2)(chi_i - lap_perp)(a+_i + a_i).
// With lap_perp the periodic 5-point Laplacian (eigenvalues lambda =
// (2cos(2 pi j/ny)-2)/dy^2 + (2cos(2 pi k/nz)-2)/dz^2) and c_i the midrange
// (min + max)/2 of chi_i, each transverse mode of slice i reads
//     d_i = M_i(lambda) * [ -(2/dx) d_{i+1} + dt chi_i a_i - dt lap_perp a_i
//                           + (dt/2)(chi_i - c_i) d_i ],
//     M_i = 1 / (alpha + (lambda - c_i) dt/2),  alpha = -2/dx + 2 i k0.
// (chi_i - c_i) d_i couples the modes and is iterated: the first transform
// takes it as 0, each of m further transforms the previous d_i.  For chi >= 0
// the iteration contracts by at most (max - min)/(max + min + 8/(dx dt)) < 1
// for any dt, and a uniform chi is exact in one transform.  The bracket is
// assembled in real space in the row pass (the stencil gives lap_perp a_i
// exactly as the spectrum would), its real and imaginary parts take two real
// transforms, the column pass applies the complex multiplier (mixing the two
// spectra), and the last row pass stores d_i (and, after the last transform
// of the slice, adds it to a_i).  |alpha + (lambda - c_i) dt/2| > 2/dx for
// every mode, so the sweep over the slices is stable for any dt.
//
// Several steps run as one pipeline: step s may take slice i as soon as step s - 1 has
// left it and step s has left slice i + 1, so at time t the steps s = 0 .. ns - 1 work
// on the slices nx - 1 - (t - s), each in its own spectra and increments, in one set of
// launches.  ns steps then take nx + ns - 1 turns of 3 (m + 1) launches instead of
// ns nx: a lone transform of a 256^2 grid is a chain of latency-bound launches (64-129
// blocks).  Twelve steps of 256^2 x 100 slices: 35 -> 7.5 ms of launches.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>

#include "qp_envelope.h"
#include "qp_wave_solver.h"

namespace qp {

namespace {

constexpr int kET = 256;

inline int eblk(size_t n) { return (int)std::min<size_t>((n + kET - 1) / kET, 65535 * 4); }

// a = a0 exp(-4 ((x-x0)^2/xs^2 + (y-y0)^2/ys^2 + (z-z0)^2/zs^2)), real, so
// <a^2> = |a|^2/2 is the Gaussian <a^2> of the wake's laser with the same
// arguments (0.5 a0^2 exp(-8 (...)), src/Config_reader.cpp:114-128).
__global__ void k_env_gauss(double *a, double *asq, size_t vol, size_t nn, int nz, double dx, double dy, double dz,
                            double a0, double ixs2, double iys2, double izs2, double x0, double y0, double z0) {
    for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < vol; t += (size_t)gridDim.x * blockDim.x) {
        const size_t i = t / nn, r = t - i * nn;
        const int j = (int)(r / nz), k = (int)(r - (size_t)j * nz);
        const double x = i * dx - x0, y = j * dy - y0, z = k * dz - z0;
        const double v = a0 * exp(-4.0 * (x * x * ixs2 + y * y * iys2 + z * z * izs2));
        a[t] = v;
        a[vol + t] = 0.0;
        asq[t] = 0.5 * v * v;
    }
}

// Real and imaginary parts side by side, for the copy to the host.
__global__ void k_env_join(const double *re, const double *im, double2 *out, size_t n) {
    const size_t t = (size_t)blockIdx.x * kET + threadIdx.x;
    if (t < n) out[t] = make_double2(re[t], im[t]);
}

__global__ void k_env_asq(const double *a, double *asq, size_t vol) {
    for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < vol; t += (size_t)gridDim.x * blockDim.x) {
        const double re = a[t], im = a[vol + t];
        asq[t] = 0.5 * (re * re + im * im);
    }
}

// Midrange (min + max)/2 of chi for every slice: one block per slice.
__global__ __launch_bounds__(kET) void k_env_cmid(const double *chi3, double *cm, size_t nn) {
    const double *c = chi3 + (size_t)blockIdx.x * nn;
    double lo = c[0], hi = c[0];
    for (size_t t = threadIdx.x; t < nn; t += kET) {
        lo = fmin(lo, c[t]);
        hi = fmax(hi, c[t]);
    }
    for (int off = 32; off > 0; off >>= 1) {
        lo = fmin(lo, __shfl_xor(lo, off));
        hi = fmax(hi, __shfl_xor(hi, off));
    }
    __shared__ double plo[kET / 64], phi[kET / 64];
    if ((threadIdx.x & 63) == 0) {
        plo[threadIdx.x >> 6] = lo;
        phi[threadIdx.x >> 6] = hi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 1; i < kET / 64; ++i) {
            lo = fmin(lo, plo[i]);
            hi = fmax(hi, phi[i]);
        }
        lo = fmin(lo, plo[0]);
        hi = fmax(hi, phi[0]);
        cm[blockIdx.x] = 0.5 * (lo + hi);
    }
}

// Row-pass source of slice e: part `which` (0 re, 1 im) of
// -(2/dx) d_{e+1} + dt (chi a - lap_perp a) + (dt/2)(chi - c_e) d_e.
struct SrcEnv {
    const double *a;      // real parts of all slices (imaginary parts at + vol)
    const double *chi;    // chi of all slices
    const double *inc;    // per step: 2 slots x (re, im) x nn increments
    const double *cmid;   // c of all slices
    size_t vol, nn;
    int nx, n1, n2, use_dcur;
    double idy2, idz2, dt, c2dx;
    int e0, s0;  // the launch's member wk is step s0 + wk at slice e0 + wk
    template <int E, bool TAIL = false>
    __device__ void row(int wk, int which, int j, int k0, int dk, double (&v)[E]) const {
        const int e = e0 + wk;
        const double *ac = a + (size_t)which * vol + (size_t)e * nn;
        const double *r0 = ac + (size_t)j * n2;
        const double *rm = ac + (size_t)(j == 0 ? n1 - 1 : j - 1) * n2, *rp = ac + (size_t)(j + 1 == n1 ? 0 : j + 1) * n2;
        const double *xr = chi + (size_t)e * nn + (size_t)j * n2;
        const double *is = inc + (size_t)(s0 + wk) * 4 * nn + (size_t)which * nn + (size_t)j * n2;
        const double *ip = is + (size_t)((e + 1) & 1) * 2 * nn, *ic = is + (size_t)(e & 1) * 2 * nn;
        double c[E], cp[E], cm[E], kp[E], km[E], x[E], dp[E], dc[E], mid = 0.0;
#pragma unroll
        for (int r = 0; r < E; ++r) {
            const int k = row_k<TAIL>(k0 + dk * r, n2);
            c[r] = r0[k];
            cp[r] = rp[k];
            cm[r] = rm[k];
            kp[r] = r0[k + 1 == n2 ? 0 : k + 1];
            km[r] = r0[k == 0 ? n2 - 1 : k - 1];
            x[r] = xr[k];
            dp[r] = dc[r] = 0.0;
        }
        if (e != nx - 1) {
#pragma unroll
            for (int r = 0; r < E; ++r) dp[r] = ip[row_k<TAIL>(k0 + dk * r, n2)];
        }
        if (use_dcur) {
            mid = cmid[e];
#pragma unroll
            for (int r = 0; r < E; ++r) dc[r] = ic[row_k<TAIL>(k0 + dk * r, n2)];
        }
#pragma unroll
        for (int r = 0; r < E; ++r) {
            const double lap = (cp[r] - 2.0 * c[r] + cm[r]) * idy2 + (kp[r] - 2.0 * c[r] + km[r]) * idz2;
            double u = dt * (x[r] * c[r] - lap);
            u -= c2dx * dp[r];                                  // 0 ahead of the first slice
            if (use_dcur) u += 0.5 * dt * (x[r] - mid) * dc[r];
            v[r] = u;
        }
    }
    template <int E, bool TAIL = false>
    __device__ void done(int, int, int, int, int) const {}
};

// Last row pass: d_e (unnormalised c2r output / (n1 n2)) to the increment
// buffer, and onto a_e after the last transform of the slice.
struct SinkEnv {
    double *a;     // all slices (imaginary parts at + vol); null: store d_e only
    double *inc;
    size_t vol, nn;
    int n1, n2, e0, s0;
    __device__ void prep(int) {}
    __device__ void begin(int) {}
    __device__ void operator()(int wk, int which, int j, int k, double v) const {
        const int e = e0 + wk;
        const size_t t = (size_t)j * n2 + k;
        const double d = v / n1 / n2;
        inc[(size_t)(s0 + wk) * 4 * nn + (size_t)(e & 1) * 2 * nn + (size_t)which * nn + t] = d;
        if (a) a[(size_t)which * vol + (size_t)e * nn + t] += d;
    }
};

// M = 1/(alpha + lam dt/2) (lam = lambda - c_i) applied to the spectra X (of
// the real parts) and Y (of the imaginary parts): X' = Re M X - Im M Y,
// Y' = Im M X + Re M Y.
__device__ __forceinline__ void env_mix(double2 &X, double2 &Y, double lam, double ar, double ai, double hdt) {
    const double qr = ar + hdt * lam, qi = ai;
    const double den = qr * qr + qi * qi;
    const double mr = qr / den, mi = -qi / den;
    const double2 x = X, y = Y;
    X = make_double2(mr * x.x - mi * y.x, mr * x.y - mi * y.y);
    Y = make_double2(mi * x.x + mr * y.x, mi * x.y + mr * y.y);
}

// Column pass on the register-resident FFTs: one block holds column l of
// both spectra (column-major spec[l * n1 + j]), forward, mix, inverse.
template <int N1, int E, int TB>
__global__ __launch_bounds__(TB) void kw_cols_env(double2 *spec0, double2 *spec1, int nh, const double2 *tw1,
                                                  const double *lam1, const double *lam2, double ar, double ai,
                                                  double hdt, const double *cmid) {
    const int wk = blockIdx.y;  // step of the pipeline
    cmid += wk;
    spec0 += (size_t)wk * N1 * nh;
    spec1 += (size_t)wk * N1 * nh;
    using W = WfShape<N1, E, TB>;
    __shared__ double2 sb0[W::LDS], sb1[W::LDS], twl[WfTw<N1, E, TB>::NL];
    const int tid = threadIdx.x;
    const int tt = tid / W::L, j = tid % W::L;
    WfTw<N1, E, TB> tw;
    tw.init(tw1, twl, j);
    const int l = blockIdx.x * W::T + tt;
    const bool valid = l < nh;
    double2 x[E], y[E];
    double lm[E];
    const double2 *c0 = spec0 + (size_t)l * N1, *c1 = spec1 + (size_t)l * N1;
#pragma unroll
    for (int r = 0; r < E; ++r) {
        x[r] = valid ? c0[j + W::L * r] : make_double2(0.0, 0.0);
        y[r] = valid ? c1[j + W::L * r] : make_double2(0.0, 0.0);
        lm[r] = lam1[j + W::L * r];
    }
    const double l2 = (valid ? lam2[l] : 0.0) - *cmid;
    double2 *b0 = sb0 + tt * W::PADN, *b1 = sb1 + tt * W::PADN;
    wave_fft<N1, E, -1>(x, b0, b1, tw, j);
    wave_fft<N1, E, -1>(y, b0, b1, tw, j);
#pragma unroll
    for (int m = 0; m < E; ++m) env_mix(x[m], y[m], lm[m] + l2, ar, ai, hdt);
    wave_fft<N1, E, +1>(x, b0, b1, tw, j);
    wave_fft<N1, E, +1>(y, b0, b1, tw, j);
    if (!valid) return;
    double2 *o0 = spec0 + (size_t)l * N1, *o1 = spec1 + (size_t)l * N1;
#pragma unroll
    for (int m = 0; m < E; ++m) {
        o0[j + W::L * m] = x[m];
        o1[j + W::L * m] = y[m];
    }
}

// The same on the LDS transforms: one block per column l, both spectra.
template <bool ONE>
__global__ __launch_bounds__(kGenThreads) void kg_cols_env(double2 *spec0, double2 *spec1, int n1, FftAxisDev ax,
                                                           const double *lam1, const double *lam2, double ar, double ai,
                                                           double hdt, const double *cmid) {
    extern __shared__ double2 lds[];
    constexpr int E = 4;  // n1 <= E threads
    const int l = blockIdx.x, T = blockDim.x, wk = blockIdx.y;
    cmid += wk;
    spec0 += (size_t)wk * n1 * gridDim.x;
    spec1 += (size_t)wk * n1 * gridDim.x;
    double2 *a = lds, *b = lds + 2 * n1, *twl = lds + 4 * n1;
    LdsTw tw;
    tw.load(ax);
    double2 *c0 = spec0 + (size_t)l * n1, *c1 = spec1 + (size_t)l * n1;
    double2 x[E], y[E];
    double lm[E];
#pragma unroll
    for (int r = 0; r < E; ++r) {
        const int t = min((int)threadIdx.x + r * T, n1 - 1);
        x[r] = c0[t];
        y[r] = c1[t];
        lm[r] = lam1[t];
    }
    const double l2 = lam2[l] - *cmid;
#pragma unroll
    for (int r = 0; r < E; ++r) {
        const int t = threadIdx.x + r * T;
        if (t < n1) {
            a[t] = x[r];
            a[n1 + t] = y[r];
        }
    }
    tw.store(twl, n1);
    lds_sync<ONE>();
    double2 *z = lds_fft<ONE, 2>(a, b, ax, twl);
#pragma unroll
    for (int r = 0; r < E; ++r) {
        const int t = threadIdx.x + r * T;
        if (t < n1) {
            double2 X = z[t], Y = z[n1 + t];
            env_mix(X, Y, lm[r] + l2, ar, ai, hdt);
            z[t] = swap_parts(X);  // forward again for the inverse
            z[n1 + t] = swap_parts(Y);
        }
    }
    lds_sync<ONE>();
    const double2 *o = lds_fft<ONE, 2>(z, z == a ? b : a, ax, twl);
#pragma unroll
    for (int r = 0; r < E; ++r) {
        const int t = threadIdx.x + r * T;
        if (t < n1) {
            c0[t] = swap_parts(o[t]);
            c1[t] = swap_parts(o[n1 + t]);
        }
    }
}

#define ELAUNCH(kern, grid, block, lds, ...)                                  \
    do {                                                                      \
        hipLaunchKernelGGL(kern, grid, dim3(block), lds, s, __VA_ARGS__);     \
        QP_HIP_CHECK(hipGetLastError());                                      \
    } while (0)

void drop_graphs(Envelope *e) {
    for (int n = 0; n <= kEnvPipeMax; ++n) {
        if (e->gexec[n]) (void)hipGraphExecDestroy(e->gexec[n]);
        e->gexec[n] = nullptr;
        e->g_seen[n] = false;
    }
}

// One transform per block, as the wake solves' column pass: 256^2 x 1000 slices
// 36.50 -> 35.3 ms per envelope step, 512^2 x 2000 slices 120.5 -> 114.0 ms.
int wlaunch_cols_env(const Solver2d &S, double2 *spec0, double2 *spec1, double ar, double ai, double hdt,
                     const double *cmid, int ns, hipStream_t s) {
    wf_dispatch(S.n1, [&](auto NC) {
        constexpr int N = decltype(NC)::value, E = WfCfg<N>::E, TB = WfCfg<N>::TBC;
        const dim3 grid(wcols_blocks_t(S.nh, WfShape<N, E, TB>::T), ns);
        hipLaunchKernelGGL((kw_cols_env<N, E, TB>), grid, dim3(TB), 0, s, spec0, spec1, S.nh,
                           (const double2 *)S.ax1.dev.tw, (const double *)S.d_lam1, (const double *)S.d_lam2, ar,
                           ai, hdt, cmid);
    });
    QP_HIP_CHECK(hipGetLastError());
    return QP_OK;
}

// One transform of the steps s0 .. s0 + ns - 1 at the slices e0 .. e0 + ns - 1: each d
// from the bracket with the previous iterate (use_dcur) or without it, onto a when `last`.
int env_transform(Envelope *e, int e0, int s0, int ns, double dt, bool use_dcur, bool last, hipStream_t s) {
    const Solver2d &S = e->S;
    const size_t nn = e->nn(), vol = e->vol();
    const double ar = -2.0 / e->dx, ai = 2.0 * e->k0, hdt = 0.5 * dt;
    double *inc = e->pipe_inc ? e->pipe_inc : e->inc;
    double2 *sp0 = e->pipe_spec ? e->pipe_spec : S.spec[0];
    double2 *sp1 = e->pipe_spec ? e->pipe_spec + (size_t)e->pipe * S.n1 * S.nh : S.spec[1];
    SrcEnv src{e->a, e->chi3, inc, e->cmid, vol, nn, e->nx, S.n1, S.n2, use_dcur ? 1 : 0,
               1.0 / (e->dy * e->dy), 1.0 / (e->dz * e->dz), dt, 2.0 / e->dx, e0, s0};
    SinkEnv snk{last ? e->a : nullptr, inc, vol, nn, S.n1, S.n2, e0, s0};
    const double *cmid = e->cmid + e0;
    const Ctl *none = nullptr;
    if (S.wave) {
        QP_TRY(wlaunch_rows_fwd(S, src, sp0, sp1, 2, s, NoCtl{}, 0, ns));
        QP_TRY(wlaunch_cols_env(S, sp0, sp1, ar, ai, hdt, cmid, ns, s));
        return wlaunch_rows_inv(S, (const double2 *)sp0, (const double2 *)sp1, snk, 2, s, NoCtl{}, 0, ns);
    }
    QP_TRY(glaunch_rows_fwd(S, src, sp0, sp1, 2, s, none, 0, ns));
    const int threads = S.ax1.dev.threads;
    const size_t lds = sizeof(double2) * 5 * (size_t)S.n1;
    if (threads == 64)
        ELAUNCH(kg_cols_env<true>, dim3(S.nh, ns), threads, lds, sp0, sp1, S.n1, S.ax1.dev, (const double *)S.d_lam1,
                (const double *)S.d_lam2, ar, ai, hdt, cmid);
    else
        ELAUNCH(kg_cols_env<false>, dim3(S.nh, ns), threads, lds, sp0, sp1, S.n1, S.ax1.dev, (const double *)S.d_lam1,
                (const double *)S.d_lam2, ar, ai, hdt, cmid);
    return glaunch_rows_inv(S, (const double2 *)sp0, (const double2 *)sp1, snk, 2, s, none, 0, ns);
}

// Steps in flight at once: enough to fill the chip (2^20 nodes), at most kEnvPipeMax; 256^2 takes
// 16, 512^2 four, 1024^2 (whose launches fill it alone) one.
int pipe_depth(const Envelope *e) {
    return (int)std::max<size_t>(1, std::min<size_t>(kEnvPipeMax, ((size_t)1 << 20) / e->nn()));
}

// Spectra and increments of `depth` steps in flight (kept: 2^20 nodes take 50 MB).  Where
// the device has no room for them, of half as many, down to one step, which needs neither;
// depth: what the envelope can run.
int ensure_pipe(Envelope *e, int &depth) {
    if (depth <= std::max(1, e->pipe)) return QP_OK;
    QP_HIP_CHECK(hipStreamSynchronize(e->stream()));
    drop_graphs(e);
    for (;; depth /= 2) {
        if (e->pipe_inc) (void)hipFree(e->pipe_inc);
        if (e->pipe_spec) (void)hipFree(e->pipe_spec);
        e->pipe_inc = nullptr;
        e->pipe_spec = nullptr;
        e->pipe = 0;
        if (depth <= 1) return QP_OK;
        if (hipMalloc(&e->pipe_inc, sizeof(double) * 4 * e->nn() * depth) == hipSuccess &&
            hipMalloc(&e->pipe_spec, sizeof(double2) * 2 * (size_t)e->S.n1 * e->S.nh * depth) == hipSuccess)
            break;
        (void)hipGetLastError();
    }
    e->pipe = depth;
    return QP_OK;
}

// ns steps of the whole envelope as one pipeline (every slice, then <a^2>); m corrections
// of the (chi - c) d term per slice.  c_i are set before the first step.
int env_sweep(Envelope *e, double dt, int m, int ns, hipStream_t s) {
    const size_t vol = e->vol();
    const int nx = e->nx;
    for (int t = 0; t < nx + ns - 1; ++t) {
        const int s0 = std::max(0, t - nx + 1), s1 = std::min(ns - 1, t);
        for (int it = 0; it <= m; ++it)
            QP_TRY(env_transform(e, nx - 1 - t + s0, s0, s1 - s0 + 1, dt, it > 0, it == m, s));
    }
    ELAUNCH(k_env_asq, dim3(eblk(vol)), kET, 0, (const double *)e->a, e->asq3, vol);
    return QP_OK;
}

// The same, when use_graph, as a captured graph of this (dt, m, ns, stream): launched
// directly the first time (a capture costs more than the launches it replaces once),
// captured the second, replayed after.  Graphs of several ns stay side by side, for callers
// who vary the steps of a call, whose steps split unevenly or who step the envelope in a
// wake's passes too (one, then twelve steps of 128^2 x 60 slices: 8.3-12.7 ms with one graph
// captured anew each time, 5.7 so); beyond kEnvGraphs of them the launches are direct.
constexpr int kEnvGraphs = 4;
int env_run(Envelope *e, double dt, int m, int ns, int use_graph, hipStream_t s) {
    if (!use_graph) return env_sweep(e, dt, m, ns, s);
    if (e->g_dtau != dt || e->g_iter != m || e->g_stream != s) {
        drop_graphs(e);
        e->g_dtau = dt;
        e->g_iter = m;
        e->g_stream = s;
    }
    hipGraphExec_t &gexec = e->gexec[ns];
    if (!gexec) {
        int held = 0;
        for (hipGraphExec_t g : e->gexec) held += g != nullptr;
        if (!e->g_seen[ns] || held >= kEnvGraphs) {
            e->g_seen[ns] = true;
            return env_sweep(e, dt, m, ns, s);
        }
        hipGraph_t gr;
        QP_HIP_CHECK(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
        const int st = env_sweep(e, dt, m, ns, s);
        const hipError_t ce = hipStreamEndCapture(s, &gr);
        if (st < 0) {
            if (ce == hipSuccess) (void)hipGraphDestroy(gr);
            return st;
        }
        if (ce != hipSuccess) {
            set_error(std::string("hipStreamEndCapture: ") + hipGetErrorString(ce));
            return QP_ERR_HIP;
        }
        const hipError_t ie = hipGraphInstantiate(&gexec, gr, nullptr, nullptr, 0);
        (void)hipGraphDestroy(gr);
        if (ie != hipSuccess) {
            gexec = nullptr;
            set_error(std::string("hipGraphInstantiate: ") + hipGetErrorString(ie));
            return QP_ERR_HIP;
        }
    }
    QP_HIP_CHECK(hipGraphLaunch(gexec, s));
    return QP_OK;
}

}  // namespace

// ------------------------------------------------------- wake-side step
// One step of the whole envelope after a wake pass, enqueued on s: midranges
// of chi, then the sweep, replayed from the captured graph of this (dt, m)
// when use_graph, else launched directly.
int envelope_step(Envelope *e, double dt, int m, int use_graph, hipStream_t s) {
    ELAUNCH(k_env_cmid, dim3(e->nx), kET, 0, (const double *)e->chi3, e->cmid, e->nn());
    return env_run(e, dt, m, 1, use_graph, s);
}

}  // namespace qp

using namespace qp;

#define EARG_CHECK(cond, msg)        \
    do {                             \
        if (!(cond)) {               \
            set_error(msg);          \
            return QP_ERR_ARG;       \
        }                            \
    } while (0)

extern "C" {

int qp_envelope_create(qp_ctx ctx, int nx, int ny, int nz, double dx, double dy, double dz, double k0,
                       qp_envelope *out) {
    EARG_CHECK(ctx && out, "qp_envelope_create: null argument");
    EARG_CHECK(nx >= 1 && ny >= 2 && nz >= 2 && ny <= kMaxN && nz <= kMaxN,
               "qp_envelope_create: need nx >= 1 and 2 <= ny, nz <= 1024");
    EARG_CHECK(dx > 0 && dy > 0 && dz > 0 && k0 > 0, "qp_envelope_create: steps and k0 must be positive");
    *out = nullptr;
    qp_envelope h = new qp_envelope_s();
    Envelope *e = &h->e;
    e->ctx = ctx;
    e->nx = nx;
    e->ny = ny;
    e->nz = nz;
    e->dx = dx;
    e->dy = dy;
    e->dz = dz;
    e->k0 = k0;
    auto fail = [&](int st) {
        qp_envelope_destroy(h);
        return st;
    };
    if (hipSetDevice(ctx->device) != hipSuccess) return fail(QP_ERR_HIP);
    int st = e->S.init(ny, nz, dy, dz, 1);
    if (st != QP_OK) return fail(st);
    const size_t nn = e->nn(), vol = e->vol();
    if (hipMalloc(&e->a, sizeof(double) * 2 * vol) != hipSuccess ||
        hipMalloc(&e->inc, sizeof(double) * 4 * nn) != hipSuccess ||
        hipMalloc(&e->chi3, sizeof(double) * vol) != hipSuccess ||
        hipMalloc(&e->asq3, sizeof(double) * vol) != hipSuccess ||
        hipMalloc(&e->cmid, sizeof(double) * nx) != hipSuccess) {
        set_error("qp_envelope_create: device allocation failed");
        return fail(QP_ERR_ALLOC);
    }
    hipStream_t s = e->stream();
    const void *bufs[] = {e->a, e->chi3, e->asq3};
    const size_t sizes[] = {2 * vol, vol, vol};
    for (int b = 0; b < 3; ++b)
        if (hipMemsetAsync(const_cast<void *>(bufs[b]), 0, sizeof(double) * sizes[b], s) != hipSuccess)
            return fail(QP_ERR_HIP);
    if (hipStreamSynchronize(s) != hipSuccess) return fail(QP_ERR_HIP);
    *out = h;
    return QP_OK;
}

int qp_envelope_destroy(qp_envelope h) {
    if (!h) return QP_OK;
    Envelope *e = &h->e;
    if (e->attached) {
        set_error("qp_envelope_destroy: a wake still reads this envelope (detach or destroy it first)");
        return QP_ERR_STATE;
    }
    if (e->ctx) (void)hipStreamSynchronize(e->stream());
    drop_graphs(e);
    e->S.destroy();
    for (double *p : {e->a, e->inc, e->chi3, e->asq3, e->cmid, e->pipe_inc})
        if (p) (void)hipFree(p);
    if (e->pipe_spec) (void)hipFree(e->pipe_spec);
    if (e->join) (void)hipFree(e->join);
    delete h;
    return QP_OK;
}

int qp_envelope_set(qp_envelope h, const double *re, const double *im) {
    EARG_CHECK(h && re, "qp_envelope_set: null argument");
    Envelope *e = &h->e;
    hipStream_t s = e->stream();
    const size_t vol = e->vol();
    QP_HIP_CHECK(hipMemcpy(e->a, re, sizeof(double) * vol, hipMemcpyHostToDevice));
    if (im) {
        QP_HIP_CHECK(hipMemcpy(e->a + vol, im, sizeof(double) * vol, hipMemcpyHostToDevice));
    } else {
        QP_HIP_CHECK(hipMemsetAsync(e->a + vol, 0, sizeof(double) * vol, s));
    }
    hipLaunchKernelGGL(k_env_asq, dim3(eblk(vol)), dim3(kET), 0, s, (const double *)e->a, e->asq3, vol);
    QP_HIP_CHECK(hipGetLastError());
    QP_HIP_CHECK(hipStreamSynchronize(s));
    return QP_OK;
}

int qp_envelope_set_gaussian(qp_envelope h, double a0, double xsigma, double ysigma, double zsigma, double x0,
                             double y0, double z0) {
    EARG_CHECK(h, "null envelope");
    EARG_CHECK(xsigma > 0 && ysigma > 0 && zsigma > 0, "qp_envelope_set_gaussian: widths must be positive");
    Envelope *e = &h->e;
    hipStream_t s = e->stream();
    const size_t vol = e->vol();
    hipLaunchKernelGGL(k_env_gauss, dim3(eblk(vol)), dim3(kET), 0, s, e->a, e->asq3, vol, e->nn(), e->nz, e->dx,
                       e->dy, e->dz, a0, 1.0 / (xsigma * xsigma), 1.0 / (ysigma * ysigma), 1.0 / (zsigma * zsigma),
                       x0, y0, z0);
    QP_HIP_CHECK(hipGetLastError());
    QP_HIP_CHECK(hipStreamSynchronize(s));
    return QP_OK;
}

int qp_envelope_get(qp_envelope h, double *re, double *im) {
    EARG_CHECK(h, "null envelope");
    Envelope *e = &h->e;
    QP_HIP_CHECK(hipStreamSynchronize(e->stream()));
    const size_t vol = e->vol();
    if (re) QP_HIP_CHECK(hipMemcpy(re, e->a, sizeof(double) * vol, hipMemcpyDeviceToHost));
    if (im) QP_HIP_CHECK(hipMemcpy(im, e->a + vol, sizeof(double) * vol, hipMemcpyDeviceToHost));
    return QP_OK;
}

// Through at most 32 MB of device memory at a time (one copy to pageable memory runs at
// 18 GB/s, a chunk's launch is lost in it).  105 MB: 25.3 ms as two parts that the caller
// joined (three passes over fresh host memory), 9.8 ms so, 3.9 of them page faults.
int qp_envelope_get_complex(qp_envelope h, double *a) {
    EARG_CHECK(h && a, "qp_envelope_get_complex: null argument");
    Envelope *e = &h->e;
    hipStream_t s = e->stream();
    const size_t vol = e->vol();
    QP_HIP_CHECK(hipSetDevice(e->ctx->device));
    std::lock_guard<std::mutex> lock(e->join_lock);
    if (!e->join) {
        size_t n = std::min(vol, (size_t)1 << 21);
        while (hipMalloc(&e->join, sizeof(double2) * n) != hipSuccess) {
            (void)hipGetLastError();
            e->join = nullptr;
            if (n <= 4096) {
                set_error("qp_envelope_get_complex: device allocation failed");
                return QP_ERR_ALLOC;
            }
            n /= 2;
        }
        e->njoin = n;
    }
    for (size_t o = 0; o < vol; o += e->njoin) {
        const size_t n = std::min(e->njoin, vol - o);
        hipLaunchKernelGGL(k_env_join, dim3(eblk(n)), dim3(kET), 0, s, (const double *)e->a + o,
                           (const double *)e->a + vol + o, e->join, n);
        QP_HIP_CHECK(hipGetLastError());
        QP_HIP_CHECK(hipMemcpyAsync(a + 2 * o, e->join, sizeof(double2) * n, hipMemcpyDeviceToHost, s));
    }
    QP_HIP_CHECK(hipStreamSynchronize(s));
    return QP_OK;
}

int qp_envelope_set_chi(qp_envelope h, const double *chi) {
    EARG_CHECK(h, "null envelope");
    Envelope *e = &h->e;
    const size_t vol = e->vol();
    if (chi) {
        QP_HIP_CHECK(hipMemcpy(e->chi3, chi, sizeof(double) * vol, hipMemcpyHostToDevice));
    } else {
        QP_HIP_CHECK(hipMemsetAsync(e->chi3, 0, sizeof(double) * vol, e->stream()));
        QP_HIP_CHECK(hipStreamSynchronize(e->stream()));
    }
    return QP_OK;
}

int qp_envelope_get_chi(qp_envelope h, double *chi) {
    EARG_CHECK(h && chi, "qp_envelope_get_chi: null argument");
    Envelope *e = &h->e;
    QP_HIP_CHECK(hipStreamSynchronize(e->stream()));
    QP_HIP_CHECK(hipMemcpy(chi, e->chi3, sizeof(double) * e->vol(), hipMemcpyDeviceToHost));
    return QP_OK;
}

int qp_envelope_get_a_sqr(qp_envelope h, double *a_sqr) {
    EARG_CHECK(h && a_sqr, "qp_envelope_get_a_sqr: null argument");
    Envelope *e = &h->e;
    QP_HIP_CHECK(hipStreamSynchronize(e->stream()));
    QP_HIP_CHECK(hipMemcpy(a_sqr, e->asq3, sizeof(double) * e->vol(), hipMemcpyDeviceToHost));
    return QP_OK;
}

int qp_envelope_advance(qp_envelope h, double dtau, int steps, int chi_iterations, int use_graph, double *ms) {
    EARG_CHECK(h, "null envelope");
    EARG_CHECK(dtau > 0 && std::isfinite(dtau), "qp_envelope_advance: dtau must be positive");
    EARG_CHECK(steps >= 0, "qp_envelope_advance: steps must be >= 0");
    EARG_CHECK(chi_iterations >= 0 && chi_iterations <= 16, "qp_envelope_advance: chi_iterations in [0, 16]");
    Envelope *e = &h->e;
    hipStream_t s = e->stream();
    QP_HIP_CHECK(hipSetDevice(e->ctx->device));  // (it may allocate)
    struct Events {
        hipEvent_t a = nullptr, b = nullptr;
        ~Events() {
            if (a) (void)hipEventDestroy(a);
            if (b) (void)hipEventDestroy(b);
        }
    } ev;
    if (ms) {
        QP_HIP_CHECK(hipEventCreate(&ev.a));
        QP_HIP_CHECK(hipEventCreate(&ev.b));
        QP_HIP_CHECK(hipEventRecord(ev.a, s));
    }
    if (steps > 0) ELAUNCH(k_env_cmid, dim3(e->nx), kET, 0, (const double *)e->chi3, e->cmid, e->nn());
    // pipelines of nearly equal depth
    auto split = [steps](int depth) { return steps > 0 ? (steps + depth - 1) / depth : 0; };
    int groups = split(pipe_depth(e)), depth = groups ? (steps + groups - 1) / groups : 1;
    QP_TRY(ensure_pipe(e, depth));
    groups = split(depth);
    for (int g = 0, left = steps; g < groups; ++g) {
        const int ns = (left + groups - g - 1) / (groups - g);
        QP_TRY(env_run(e, dtau, chi_iterations, ns, use_graph, s));
        left -= ns;
    }
    if (ms) {
        QP_HIP_CHECK(hipEventRecord(ev.b, s));
        QP_HIP_CHECK(hipEventSynchronize(ev.b));
        float f = 0.f;
        QP_HIP_CHECK(hipEventElapsedTime(&f, ev.a, ev.b));
        *ms = f;
    }
    QP_HIP_CHECK(hipStreamSynchronize(s));
    return QP_OK;
}

}  // extern "C"
