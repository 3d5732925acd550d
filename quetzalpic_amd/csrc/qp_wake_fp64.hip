// qp_wake_fp64.hip -- the plain FP64 slice loop on the device.
//
// The loops of System_3d::solve_wakefield (src/System_3d.cpp:238-627) that need
// nothing from one another share a launch; FP64 structure-of-arrays particles,
// global FP64 atomics for the CIC deposits, the three-launch periodic solve.
// Arithmetic follows the reference's operation order (this file is built with
// -ffp-contract=off) so the result agrees with the FP64 oracle at rounding level.
// It is the baseline the fused mixed path is measured against.
//
// A slice is a chain of dependent launches of a few microseconds each, so what it
// costs is their number: 10 per iteration (one per loop: 23), 10 beside the
// iterations.  200^2 x 60 slices with inline output, K = 5: 57.1 -> 29.4 ms.
#include <cstring>

#include "qp_solver_small.h"
#include "qp_wake.h"
#include "qp_wave_solver.h"

namespace qp {

constexpr int kT = 256;
static inline int nblk(size_t n) { return (int)((n + kT - 1) / kT); }

#define SKIP_OR_LATCH(ctl)        \
    if (ctl_skip(ctl)) {          \
        ctl_latch(ctl);           \
        return;                   \
    }

// ------------------------------------------------------------- grid kernels
// fourier.in = jx_bunch(i) - rho_bunch(i) - rho_ion (src/System_3d.cpp:343-347).
__device__ __forceinline__ double static_src(const double *jxb, const double *rhob, const double *rho_ion, size_t t) {
    return (jxb ? jxb[t] : 0.0) - (rhob ? rhob[t] : 0.0) - rho_ion[t];
}

__global__ void k_copy(double *dst, const double *src, size_t n, Ctl *ctl) {
    SKIP_OR_LATCH(ctl);
    size_t t = (size_t)blockIdx.x * kT + threadIdx.x;
    if (t < n) dst[t] = src[t];
}

// Start of a slice: psi_prev = psi (:342), the transverse currents of the slice before
// (:612-613), the static part of the psi source.
__global__ void k_slice_begin(double *psi_prev, const double *psi, double *jy, const double *jyn, double *jz,
                              const double *jzn, double *src, const double *jxb, const double *rhob,
                              const double *rho_ion, size_t n, Ctl *ctl) {
    SKIP_OR_LATCH(ctl);
    size_t t = (size_t)blockIdx.x * kT + threadIdx.x;
    if (t < n) {
        psi_prev[t] = psi[t];
        jy[t] = jyn[t];
        jz[t] = jzn[t];
        src[t] = static_src(jxb, rhob, rho_ion, t);
    }
}

// rho = rho_bunch(i), jx = jx_bunch(i), susceptibility(i) = 0 (src/System_3d.cpp:381-388,
// 511-518); in an iteration also jy* = jz* = 0 (:473-478) and the static part of the
// psi_middle source.
__global__ void k_init(double *rho, double *jx, double *chi, double *jyn, double *jzn, double *src, const double *jxb,
                       const double *rhob, const double *rho_ion, size_t n, int iteration, Ctl *ctl) {
    SKIP_OR_LATCH(ctl);
    size_t t = (size_t)blockIdx.x * kT + threadIdx.x;
    if (t < n) {
        rho[t] = rhob ? rhob[t] : 0.0;
        jx[t] = jxb ? jxb[t] : 0.0;
        chi[t] = 0.0;
        if (iteration) {
            jyn[t] = 0.0;
            jzn[t] = 0.0;
            src[t] = static_src(jxb, rhob, rho_ion, t);
        }
    }
}

// normalize_potential's border mean (src/System_3d.cpp:30-40), summed in the reference's
// order by one thread of every block from an LDS copy of the border, then psi minus the
// mean and increase_minimum (:41-46, 830-841) from the solve's output `raw` (which no
// block writes) to psi.  Loaded one by one by the summing thread the border took 46 us
// at 200^2, with a second launch for the subtraction.
constexpr int kNormPer = 4;  // nodes per thread: fewer blocks that repeat the sum
__global__ __launch_bounds__(kT) void k_norm_clamp(double *psi, const double *raw, int n1, int n2, double thr, Ctl *ctl) {
    __shared__ double border[2 * kMaxN];
    __shared__ double mean;
    SKIP_OR_LATCH(ctl);
    const size_t n = (size_t)n1 * n2;
    const size_t t0 = (size_t)blockIdx.x * (kT * kNormPer) + threadIdx.x;
    double v[kNormPer];
#pragma unroll
    for (int r = 0; r < kNormPer; ++r) v[r] = raw[min(t0 + r * kT, n - 1)];
    const int m = n1 + n2 - 1;
    for (int i = threadIdx.x; i < m; i += kT) border[i] = i < n1 ? raw[(size_t)n2 * i] : raw[i - n1 + 1];
    __syncthreads();
    if (threadIdx.x == 0) {
        double b = 0.0;
#pragma unroll 16
        for (int i = 0; i < m; ++i) b += border[i];
        mean = b / (n1 + n2 - 1);
    }
    __syncthreads();
    const double b = mean;
#pragma unroll
    for (int r = 0; r < kNormPer; ++r) {
        if (t0 + r * kT >= n) break;
        double x = v[r] - b;
        if (x < thr) x = thr;
        psi[t0 + r * kT] = x;
    }
}

// Sources of the B_y (which = 0, src/System_3d.cpp:530-536) and B_z (which = 1,
// :555-564) Helmholtz solves, with d/dxi of the transverse currents (:489-495).  The
// last row of B_z takes bz(i, 0, k), as the reference writes it at :563.
struct SrcB64 {
    const double *by, *bz, *jx, *jy, *jz, *jyn, *jzn;
    int n1, n2;
    double D, dx, dy, dz;
    template <int E, bool TAIL = false>
    __device__ void row(int, int which, int j, int k0, int dk, double (&x)[E]) const {
        const size_t rj = (size_t)j * n2;
        const bool last = j == n1 - 1;
        double b[E], jc[E], jn[E], ja[E], jb[E];
#pragma unroll
        for (int r = 0; r < E; ++r) {
            const int k = row_k<TAIL>(k0 + dk * r, n2);
            const size_t t = rj + k;
            jc[r] = jx[t];
            if (which == 0) {
                b[r] = by[t];
                jn[r] = jx[rj + (k < n2 - 1 ? k + 1 : 0)];
                ja[r] = jz[t];
                jb[r] = jzn[t];
            } else {
                b[r] = bz[last ? (size_t)k : t];
                jn[r] = jx[last ? (size_t)k : t + n2];
                ja[r] = jy[t];
                jb[r] = jyn[t];
            }
        }
#pragma unroll
        for (int r = 0; r < E; ++r) {
            const double dj = (ja[r] - jb[r]) / dx;
            x[r] = which == 0 ? -D * b[r] - (jn[r] - jc[r]) / dz + dj : -D * b[r] + (jn[r] - jc[r]) / dy - dj;
        }
    }
    template <int E, bool TAIL = false>
    __device__ void done(int, int, int, int, int) const {}
};

// B store with the stop rule (src/System_3d.cpp:541-552, 569-580).
struct SinkB64 {
    double *by, *bz;
    int n1, n2;
    double thr;
    Ctl *ctl;
    int slice;
    __device__ void prep(int) {}
    __device__ void begin(int) {}
    __device__ void operator()(int, int which, int j, int k, double v) const {
        const double b = v / n1 / n2;
        (which == 0 ? by : bz)[(size_t)j * n2 + k] = b;
        if (fabs(b) > thr || isnan(b)) {
            ctl->stop_acc = 1;
            ctl->stop_slice = slice;
        }
    }
};

// output_step's fields (src/System_3d.cpp:633-661).
__global__ void k_output(double *ex, double *ey, double *ez, const double *psi, const double *psi_prev,
                         const double *by, const double *bz, int n1, int n2, double dx, double dy, double dz,
                         int with_ex, Ctl *ctl, int final_step, int *prog, int slice) {
    if (!final_step) {
        const bool stopped = ctl_skip(ctl);
        if (blockIdx.x == 0 && threadIdx.x == 0) note_progress(prog, 0, stopped ? kStopped : slice);
        SKIP_OR_LATCH(ctl);
    } else if (ctl->stop_acc) {
        by = nullptr;  // after a stop, by(0)/bz(0) are still the pass's zeros
        bz = nullptr;
    }
    size_t t = (size_t)blockIdx.x * kT + threadIdx.x;
    if (t >= (size_t)n1 * n2) return;
    const int j = (int)(t / n2), k = (int)(t % n2);
    if (with_ex) ex[t] = (psi[t] - psi_prev[t]) / dx;
    const size_t tj = j < n1 - 1 ? t + n2 : (size_t)k;
    const size_t tk = k < n2 - 1 ? t + 1 : (size_t)n2 * j;
    ey[t] = -(psi[tj] - psi[t]) / dy + (bz ? bz[t] : 0.0);
    ez[t] = -(psi[tk] - psi[t]) / dz - (by ? by[t] : 0.0);
}

// Gaussian <a^2> plane of slice i on the nodes (src/System_3d.cpp:805-816).
__global__ void k_laser_slice(double *asq, LaserGauss L, int i, double dx, double dy, double dz, int n1, int n2) {
    size_t t = (size_t)blockIdx.x * kT + threadIdx.x;
    if (t >= (size_t)n1 * n2) return;
    const int j = (int)(t / n2), k = (int)(t % n2);
    const double x = i * dx, y = j * dy, z = k * dz;
    asq[t] = L.amp * exp(-(x - L.x0) * (x - L.x0) / L.wx / L.wx - (y - L.y0) * (y - L.y0) / L.wy / L.wy -
                         (z - L.z0) * (z - L.z0) / L.wz / L.wz);
}

// --------------------------------------------------------- particle kernels
struct G2 {
    int n1, n2;
    double d1, d2, ly, lz, dx;
};

// deposit(y,z,value,array2d&) with origin (o1,o2), src/array_utils.cpp:85-118.
__device__ __forceinline__ void dep_o(double y, double z, double v, double *a, const G2 &g, double o1, double o2) {
    int j1, j2, k1, k2;
    double yf, zf;
    cic_floor(y, g.d1, o1, g.n1, j1, j2, yf);
    cic_floor(z, g.d2, o2, g.n2, k1, k2, zf);
    scatter4_global(a, g.n2, j1, j2, k1, k2, yf, zf, v);
}

// rho_ion = S(y,z)(-n) (src/System_3d.cpp:318-323).
__global__ void k_dep_ion(const double *y, const double *z, const double *n, double *rho_ion, size_t np, G2 g) {
    size_t p = (size_t)blockIdx.x * kT + threadIdx.x;
    if (p < np) dep_o(y[p], z[p], -n[p], rho_ion, g, 0.0, 0.0);
}

// psi source deposit with the truncating raw-pointer CIC (src/array_utils.cpp:120-142).
__device__ __forceinline__ void dep_raw(double y, double z, double v, double *src, const G2 &g) {
    int j1, j2, k1, k2;
    double yf, zf;
    cic_trunc(y, g.d1, g.n1, j1, j2, yf);
    cic_trunc(z, g.d2, g.n2, k1, k2, zf);
    scatter4_global(src, g.n2, j1, j2, k1, k2, yf, zf, v);
}
__global__ void k_dep_raw(const double *y, const double *z, const double *n, double *src, size_t np, G2 g,
                          Ctl *ctl) {
    SKIP_OR_LATCH(ctl);
    size_t p = (size_t)blockIdx.x * kT + threadIdx.x;
    if (p < np) dep_raw(y[p], z[p], -n[p], src, g);
}

// gamma and px of S4 (src/System_3d.cpp:368-378) and, with the half-step momentum, of P6 (:498-508).
__device__ __forceinline__ double gamma_of64(double p2, double a, double ps) {
    return 0.5 * (1 + p2 + a + (1 + ps) * (1 + ps)) / (1 + ps);
}
__device__ __forceinline__ double px_of64(double p2, double a, double ps) {
    return 0.5 * (1 + p2 + a - (1 + ps) * (1 + ps)) / (1 + ps);
}
// The reference sums 1 + py py + pz pz + a in that order for S4.
__device__ __forceinline__ double gamma_s4(double py, double pz, double a, double ps) {
    return 0.5 * (1 + py * py + pz * pz + a + (1 + ps) * (1 + ps)) / (1 + ps);
}

// jx, rho, susceptibility deposits (src/System_3d.cpp:390-397, 520-527).
__device__ __forceinline__ void dep_rho_jx_chi(double y, double z, double n, double gm, double px, double *jx,
                                               double *rho, double *chi, const G2 &g) {
    const double vx = px / gm;
    int j1, j2, k1, k2;
    double yf, zf;
    cic_floor(y, g.d1, 0.0, g.n1, j1, j2, yf);
    cic_floor(z, g.d2, 0.0, g.n2, k1, k2, zf);
    scatter4_global(jx, g.n2, j1, j2, k1, k2, yf, zf, n * vx / (1 - vx));
    scatter4_global(rho, g.n2, j1, j2, k1, k2, yf, zf, n / (1 - vx));
    scatter4_global(chi, g.n2, j1, j2, k1, k2, yf, zf, -n / (1 - vx) / gm);
}

// S4 and S5 (:368-397), for the slices without iterations: with K > 0 the iterations
// deposit rho, jx and chi anew before anyone reads them, and compute S4's gamma.
__global__ void k_s_phase(PartFP64 P, const double *asq, const double *psi, double *jx, double *rho, double *chi,
                          size_t np, G2 g, Ctl *ctl) {
    SKIP_OR_LATCH(ctl);
    size_t p = (size_t)blockIdx.x * kT + threadIdx.x;
    if (p >= np) return;
    const double y = P.y[p], z = P.z[p];
    const double a = gather_o(y, z, asq, g.n1, g.n2, g.d1, g.d2, 0.0, 0.0);
    const double ps = gather_o(y, z, psi, g.n1, g.n2, g.d1, g.d2, 0.0, 0.0);
    const double py = P.py[p], pz = P.pz[p];
    const double px = 0.5 * (1 + py * py + pz * pz + a - (1 + ps) * (1 + ps)) / (1 + ps);
    dep_rho_jx_chi(y, z, P.n[p], gamma_s4(py, pz, a, ps), px, jx, rho, chi, g);
}

// Momentum predictor (src/System_3d.cpp:416-433), with S4's gamma in the first iteration;
// half-step coordinates (:436-443) and their psi source deposit (:453-457).
__global__ void k_predict(PartFP64 P, const double *asq, const double *psi, const double *by, const double *bz,
                          double *src, size_t np, G2 g, int first, Ctl *ctl) {
    SKIP_OR_LATCH(ctl);
    size_t p = (size_t)blockIdx.x * kT + threadIdx.x;
    if (p >= np) return;
    const double y = P.y[p], z = P.z[p], py = P.py[p], pz = P.pz[p], n = P.n[p];
    const double ps = gather_o(y, z, psi, g.n1, g.n2, g.d1, g.d2, 0.0, 0.0);
    const double gm = first ? gamma_s4(py, pz, gather_o(y, z, asq, g.n1, g.n2, g.d1, g.d2, 0.0, 0.0), ps) : P.gamma[p];
    const double day = gather_yder(y, z, asq, g.n1, g.n2, g.d1, g.d2);
    const double daz = gather_zder(y, z, asq, g.n1, g.n2, g.d1, g.d2);
    const double dpy = gather_yder(y, z, psi, g.n1, g.n2, g.d1, g.d2);
    const double dpz = gather_zder(y, z, psi, g.n1, g.n2, g.d1, g.d2);
    const double byp = gather_o(y, z, by, g.n1, g.n2, g.d1, g.d2, 0.0, 0.5 * g.d2);
    const double bzp = gather_o(y, z, bz, g.n1, g.n2, g.d1, g.d2, 0.5 * g.d1, 0.0);
    const double dx = g.dx;
    double pyn = py - dx * 0.5 * day / (1 + ps);
    pyn += dx * gm * dpy / (1 + ps);
    pyn -= dx * bzp;
    double pzn = pz - dx * 0.5 * daz / (1 + ps);
    pzn += dx * gm * dpz / (1 + ps);
    pzn += dx * byp;
    P.pyn[p] = pyn;
    P.pzn[p] = pzn;
    double ym = y + 0.5 * dx * pyn / (1 + ps);
    double zm = z + 0.5 * dx * pzn / (1 + ps);
    wrap_coords(ym, zm, g.ly, g.lz);
    P.ym[p] = ym;
    P.zm[p] = zm;
    dep_raw(ym, zm, -n, src, g);
}

// Transverse current at the half-step positions (src/System_3d.cpp:480-486), gamma and px
// with the half-step momentum (:498-508), jx, rho and susceptibility deposits (:520-527).
__global__ void k_currents(PartFP64 P, const double *asq, const double *psi, const double *psim, double *jyn,
                           double *jzn, double *jx, double *rho, double *chi, size_t np, G2 g, Ctl *ctl) {
    SKIP_OR_LATCH(ctl);
    size_t p = (size_t)blockIdx.x * kT + threadIdx.x;
    if (p >= np) return;
    const double y = P.y[p], z = P.z[p], ym = P.ym[p], zm = P.zm[p], n = P.n[p];
    const double py = P.py[p], pz = P.pz[p], pyn = P.pyn[p], pzn = P.pzn[p];
    const double a = gather_o(y, z, asq, g.n1, g.n2, g.d1, g.d2, 0.0, 0.0);
    const double ps = gather_o(y, z, psi, g.n1, g.n2, g.d1, g.d2, 0.0, 0.0);
    const double psm = gather_o(ym, zm, psim, g.n1, g.n2, g.d1, g.d2, 0.0, 0.0);
    dep_o(ym, zm, n * pyn / (1 + psm), jyn, g, 0.5 * g.d1, 0.0);
    dep_o(ym, zm, n * pzn / (1 + psm), jzn, g, 0.0, 0.5 * g.d2);
    const double p2 = 0.25 * (py + pyn) * (py + pyn) + 0.25 * (pz + pzn) * (pz + pzn);
    const double gm = gamma_of64(p2, a, ps);
    P.gamma[p] = gm;
    dep_rho_jx_chi(y, z, n, gm, px_of64(p2, a, ps), jx, rho, chi, g);
}

// p = p* (src/System_3d.cpp:593-598), then the coordinate advance with psi_middle at the
// old position (:601-608).
__global__ void k_advance(PartFP64 P, const double *psim, size_t np, G2 g, Ctl *ctl) {
    SKIP_OR_LATCH(ctl);
    size_t p = (size_t)blockIdx.x * kT + threadIdx.x;
    if (p >= np) return;
    double y = P.y[p], z = P.z[p];
    const double py = P.pyn[p], pz = P.pzn[p];
    P.py[p] = py;
    P.pz[p] = pz;
    const double ps = gather_o(y, z, psim, g.n1, g.n2, g.d1, g.d2, 0.0, 0.0);
    y += g.dx * py / (1 + ps);
    z += g.dx * pz / (1 + ps);
    wrap_coords(y, z, g.ly, g.lz);
    P.y[p] = y;
    P.z[p] = z;
}

// ------------------------------------------------------------------ driver
#define LAUNCH(kern, blocks, ...)                                              \
    do {                                                                       \
        hipLaunchKernelGGL(kern, dim3(blocks), dim3(kT), 0, s, __VA_ARGS__);   \
        QP_HIP_CHECK(hipGetLastError());                                       \
    } while (0)

int wake_upload_fp64(Wake *w) {
    const size_t np = w->np();
    hipStream_t s = w->stream();
    PartFP64 &P = w->pf;
    if (w->cap < np || !P.y) {
        double **arrs[] = {&P.y, &P.z, &P.py, &P.pz, &P.n, &P.gamma, &P.ym, &P.zm, &P.pyn, &P.pzn,
                           &w->init64[0], &w->init64[1], &w->init64[2], &w->init64[3], &w->init64[4]};
        for (double **a : arrs) {
            if (*a) (void)hipFree(*a);
            QP_HIP_CHECK(hipMalloc(a, sizeof(double) * (np ? np : 1)));
        }
        w->cap = np;
        w->particles_dirty = true;
    }
    const size_t b = sizeof(double) * np;
    if (w->particles_dirty) {
        const WakeMember &m0 = w->mem[0];
        const std::vector<double> *src[5] = {&m0.h_y, &m0.h_z, &m0.h_py, &m0.h_pz, &m0.h_w};
        for (int i = 0; i < 5; ++i)
            QP_HIP_CHECK(hipMemcpy(w->init64[i], src[i]->data(), b, hipMemcpyHostToDevice));
        w->particles_dirty = false;
    }
    double *dst[5] = {P.y, P.z, P.py, P.pz, P.n};
    for (int i = 0; i < 5; ++i) QP_HIP_CHECK(hipMemcpyAsync(dst[i], w->init64[i], b, hipMemcpyDeviceToDevice, s));
    // init_wake_particles: py_next = pz_next = 0, gamma = 0 (src/System_3d.cpp:740-742)
    QP_HIP_CHECK(hipMemsetAsync(P.pyn, 0, b, s));
    QP_HIP_CHECK(hipMemsetAsync(P.pzn, 0, b, s));
    QP_HIP_CHECK(hipMemsetAsync(P.gamma, 0, b, s));
    QP_HIP_CHECK(hipMemsetAsync(P.ym, 0, b, s));
    QP_HIP_CHECK(hipMemsetAsync(P.zm, 0, b, s));
    return QP_OK;
}

int wake_download_fp64(Wake *w, double *y, double *z, double *py, double *pz) {
    const size_t b = sizeof(double) * w->np();
    QP_HIP_CHECK(hipStreamSynchronize(w->stream()));
    if (y) QP_HIP_CHECK(hipMemcpy(y, w->pf.y, b, hipMemcpyDeviceToHost));
    if (z) QP_HIP_CHECK(hipMemcpy(z, w->pf.z, b, hipMemcpyDeviceToHost));
    if (py) QP_HIP_CHECK(hipMemcpy(py, w->pf.py, b, hipMemcpyDeviceToHost));
    if (pz) QP_HIP_CHECK(hipMemcpy(pz, w->pf.pz, b, hipMemcpyDeviceToHost));
    return QP_OK;
}

// psi (or psi_middle) from the assembled source, which the solve overwrites.
static int solve_psi(Wake *w, double *psi) {
    const Solver2d &S = w->S;
    hipStream_t s = w->stream();
    const SrcPlain src{w->src, S.n2};
    const SinkScaled snk{w->src, S.n1, S.n2};
    const Ctl *ctl = w->ctl;
    const double2 *s0 = S.spec[0];
    prof_begin(w, "solve");
    if (small_solve(S)) {
        QP_TRY(slaunch(S, src, snk, 0.0, 1, s, ctl, 1));
    } else if (S.wave) {
        QP_TRY(wlaunch_rows_fwd(S, src, S.spec[0], S.spec[0], 1, s, ctl, 1));
        QP_TRY(solve_cols(S, 0.0, 1, s, ctl, 1));
        QP_TRY(wlaunch_rows_inv(S, s0, s0, snk, 1, s, ctl, 1));
    } else {
        QP_TRY(glaunch_rows_fwd(S, src, S.spec[0], S.spec[0], 1, s, ctl, 1));
        QP_TRY(solve_cols(S, 0.0, 1, s, ctl, 1));
        QP_TRY(glaunch_rows_inv(S, s0, s0, snk, 1, s, ctl, 1));
    }
    prof_end(w, "solve");
    const int per = kT * kNormPer;
    LAUNCH(k_norm_clamp, (int)((w->nn() + per - 1) / per), psi, w->src, S.n1, S.n2, w->p.psi_threshold - 1, w->ctl);
    return QP_OK;
}

// B_y and B_z in one set of launches (their sources do not depend on one another; both
// finish when one trips the stop rule, :582-584).
static int solve_b(Wake *w, int slice) {
    const Solver2d &S = w->S;
    const qp_wake_params &p = w->p;
    hipStream_t s = w->stream();
    const Ctl *ctl = w->ctl;
    const SrcB64 src{w->by, w->bz, w->jx, w->jy, w->jz, w->jyn, w->jzn, S.n1, S.n2, p.D, p.dx, p.dy, p.dz};
    const SinkB64 snk{w->by, w->bz, S.n1, S.n2, p.b_threshold, w->ctl, slice};
    const double2 *s0 = S.spec[0], *s1 = S.spec[1];
    prof_begin(w, "solve");
    if (small_solve(S)) {
        QP_TRY(slaunch(S, src, snk, p.D, 2, s, ctl, 2));
    } else if (S.wave) {
        QP_TRY(wlaunch_rows_fwd(S, src, S.spec[0], S.spec[1], 2, s, ctl, 2));
        QP_TRY(solve_cols(S, p.D, 2, s, ctl, 2));
        QP_TRY(wlaunch_rows_inv(S, s0, s1, snk, 2, s, ctl, 2));
    } else {
        QP_TRY(glaunch_rows_fwd(S, src, S.spec[0], S.spec[1], 2, s, ctl, 2));
        QP_TRY(solve_cols(S, p.D, 2, s, ctl, 2));
        QP_TRY(glaunch_rows_inv(S, s0, s1, snk, 2, s, ctl, 2));
    }
    prof_end(w, "solve");
    return QP_OK;
}

int wake_run_fp64(Wake *w, qp_slice_cb cb, void *user, int *stop_slice) {
    const qp_wake_params &p = w->p;
    hipStream_t s = w->stream();
    const size_t nn = w->nn(), np = w->np();
    const int n1 = p.ny, n2 = p.nz;
    const G2 g{n1, n2, p.dy, p.dz, p.ly, p.lz, p.dx};
    const int gb = nblk(nn), pb = nblk(np);
    Ctl *ctl = w->ctl;

    // Upload first: it allocates the particle arrays on the first pass.
    QP_TRY(wake_upload_fp64(w));
    const PartFP64 P = w->pf;
    if (np && !(P.y && P.z && P.py && P.pz && P.n && P.gamma && P.ym && P.zm && P.pyn && P.pzn)) {
        set_error("wake_run_fp64: particle arrays not allocated");
        return QP_ERR_STATE;
    }
    QP_HIP_CHECK(hipMemsetAsync(ctl, 0, sizeof(Ctl), s));
    // zero psi, by, bz, rho_ion, jy, jz (src/System_3d.cpp:265-316)
    double *zero_list[] = {w->psi, w->psi_prev, w->by, w->bz, w->rho_ion, w->jy, w->jz, w->jyn, w->jzn,
                           w->psim, w->rho, w->jx, w->chi, w->ex, w->ey, w->ez};
    for (double *a : zero_list) QP_HIP_CHECK(hipMemsetAsync(a, 0, sizeof(double) * nn, s));
    QP_HIP_CHECK(hipEventRecord(w->ev0, s));
    if (np) LAUNCH(k_dep_ion, pb, P.y, P.z, P.n, w->rho_ion, np, g);
    if (w->bunch) QP_TRY(bunch_clear_fields(w->bunch, s));

    int delivered_stop = 0;
    auto planes = [w] {
        return OutPlanes{{w->psi, w->rho, w->jx, w->jy, w->jz, w->ex, w->ey, w->ez, w->by, w->bz, w->chi, nullptr}};
    };
    const int i_end = (p.slice_limit > 0 && p.slice_limit < p.nx) ? p.nx - p.slice_limit : 0;
    watch_reset(w);
    for (int i = p.nx - 1; i >= i_end; --i) {
        if (!cb) {
            int running = 1;
            QP_TRY(watch_stops(&w, 1, i, s, running));
            if (!running) break;
        }
        const double *asq;
        QP_TRY(wake_asq_slice(w, i, &asq));
        if (w->bunch) QP_TRY(bunch_slice_sources(w->bunch, ctl, -1, i, s));
        const double *rb = wake_rho_b(w, i), *jb = wake_jx_b(w, i);
        // S1-S3
        LAUNCH(k_slice_begin, gb, w->psi_prev, w->psi, w->jy, w->jyn, w->jz, w->jzn, w->src, jb, rb, w->rho_ion, nn, ctl);
        prof_begin(w, "push");
        if (np) LAUNCH(k_dep_raw, pb, P.y, P.z, P.n, w->src, np, g, ctl);
        prof_end(w, "push");
        QP_TRY(solve_psi(w, w->psi));
        // S4-S5
        if (i == 0 || p.K == 0) {
            LAUNCH(k_init, gb, w->rho, w->jx, w->chi, w->jyn, w->jzn, w->src, jb, rb, w->rho_ion, nn, 0, ctl);
            prof_begin(w, "push");
            if (np) LAUNCH(k_s_phase, pb, P, asq, w->psi, w->jx, w->rho, w->chi, np, g, ctl);
            prof_end(w, "push");
        }
        // S6: by(i) = by(i+1) is the carried buffer
        if (i == 0) {
            if (w->env) LAUNCH(k_copy, gb, w->chi_store(i), (const double *)w->chi, nn, ctl);
            break;
        }
        for (int it = 0; it < p.K; ++it) {
            LAUNCH(k_init, gb, w->rho, w->jx, w->chi, w->jyn, w->jzn, w->src, jb, rb, w->rho_ion, nn, 1, ctl);
            prof_begin(w, "push");
            if (np) LAUNCH(k_predict, pb, P, asq, w->psi, w->by, w->bz, w->src, np, g, it == 0 ? 1 : 0, ctl);
            prof_end(w, "push");
            QP_TRY(solve_psi(w, w->psim));
            prof_begin(w, "push");
            if (np)
                LAUNCH(k_currents, pb, P, asq, w->psi, w->psim, w->jyn, w->jzn, w->jx, w->rho, w->chi, np, g, ctl);
            prof_end(w, "push");
            QP_TRY(solve_b(w, i));
        }
        if (w->env) LAUNCH(k_copy, gb, w->chi_store(i), (const double *)w->chi, nn, ctl);
        prof_begin(w, "push");
        if (np) LAUNCH(k_advance, pb, P, w->psim, np, g, ctl);
        prof_end(w, "push");
        LAUNCH(k_output, gb, w->ex, w->ey, w->ez, w->psi, w->psi_prev, w->by, w->bz, n1, n2, p.dx, p.dy, p.dz,
               i < p.nx - 1 ? 1 : 0, ctl, 0, w->h_prog, i);
        if (w->bunch) QP_TRY(bunch_slice_gather(w->bunch, w->ex, w->ey, w->ez, w->by, w->bz, ctl, -1, i, s));
        if (cb) {
            Ctl hc;
            QP_TRY(stage_slice(w, planes(), ctl, &hc));
            if (hc.stop_acc) {
                QP_TRY(call_slice(w, cb, user, hc.stop_slice, QP_SLICE_STOPPED, false));
                delivered_stop = 1;
                break;
            }
            QP_TRY(call_slice(w, cb, user, i, QP_SLICE_NORMAL, false));
        }
    }
    if (i_end == 0) {
        // output_step(0) after the loop (src/System_3d.cpp:622)
        LAUNCH(k_output, gb, w->ex, w->ey, w->ez, w->psi, w->psi_prev, w->by, w->bz, n1, n2, p.dx, p.dy, p.dz,
               p.nx > 1 ? 1 : 0, ctl, 1, w->h_prog, 0);
        // bunch bucket 0: slice 0's fields are final only after output_step(0)
        if (w->bunch) QP_TRY(bunch_slice_gather(w->bunch, w->ex, w->ey, w->ez, w->by, w->bz, ctl, -1, 0, s));
        // the envelope step after the pass (the plain path keeps the launches in order)
        if (w->env_step()) QP_TRY(envelope_step(w->env, w->env_dtau, w->env_chi_it, w->p.use_graph, s));
    }
    QP_HIP_CHECK(hipEventRecord(w->ev1, s));
    QP_HIP_CHECK(hipStreamSynchronize(s));
    float ms = 0.f;
    QP_HIP_CHECK(hipEventElapsedTime(&ms, w->ev0, w->ev1));
    w->last_ms = ms;
    Ctl hc;
    QP_HIP_CHECK(hipMemcpy(&hc, ctl, sizeof(Ctl), hipMemcpyDeviceToHost));
    if (hc.stop_acc && cb && !delivered_stop)
        QP_TRY(deliver_slice(w, cb, user, hc.stop_slice, QP_SLICE_STOPPED, planes()));
    if (cb && i_end == 0) {
        OutPlanes o = planes();
        if (hc.stop_acc) o.p[8] = o.p[9] = o.p[10] = w->zero2;
        QP_TRY(deliver_slice(w, cb, user, 0, QP_SLICE_FINAL, o));
    }
    if (stop_slice) *stop_slice = hc.stop_acc ? hc.stop_slice : -1;
    return hc.stop_acc ? QP_STOPPED : QP_OK;
}

}  // namespace qp

namespace qp {

int wake_asq_slice(Wake *w, int i, const double **asq) {
    const qp_wake_params &p = w->p;
    if (w->asq3()) {
        *asq = w->asq3() + (size_t)i * w->nn();
        return QP_OK;
    }
    if (w->mem[0].laser_set) {
        hipStream_t s = w->stream();
        LAUNCH(k_laser_slice, nblk(w->nn()), w->asq2, w->mem[0].laser, i, p.dx, p.dy, p.dz, p.ny, p.nz);
        *asq = w->asq2;
        return QP_OK;
    }
    *asq = w->zero2;  // no [laser] block: a_sqr stays zero (src/System_parameters.h:22)
    return QP_OK;
}

}  // namespace qp
