// qp_fft.hip -- periodic 2D solve on the device, FP64.
//
// Replaces Fourier2d (src/Fourier2d.h:4-19) and
// System_3d::solve_poisson_equation (src/System_3d.cpp:686-706):
//   r2c over n1 x n2 -> (0,0) := 0 -> divide by the 5-point eigenvalue
//   -D + (2cos(2 pi j/n1) - 2)/d1^2 + (2cos(2 pi k/n2) - 2)/d2^2 -> c2r.
// Three launches: rows forward (two real rows packed per complex transform),
// columns forward + divide + inverse (one block owns whole columns), rows
// inverse (Hermitian rows packed two per complex transform).  Power-of-two
// grids from 16 to 1024 per side use the register-resident kernels of
// qp_wave_solver.h; other sizes, and Fourier2d's transforms (FFTW's r2c
// layout), use the generic LDS kernels of qp_solver_kernels.h.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <utility>
#include <vector>

#include "qp_solver_small.h"
#include "qp_wave_solver.h"

namespace qp {

int FftAxis::plan(int n) {
    if (n < 1 || n > kMaxN) {
        set_error("transform length " + std::to_string(n) + " outside [1, " + std::to_string(kMaxN) + "]");
        return QP_ERR_ARG;
    }
    dev.n = n;
    dev.nstages = 0;
    int m = n;
    auto push = [&](int r) -> bool {
        if (dev.nstages >= kMaxStages) return false;
        dev.st[dev.nstages++].R = r;
        return true;
    };
    // odd radices first (their first-stage writes spread over the LDS banks)
    for (int f : {5, 7, 3})
        while (m % f == 0) { if (!push(f)) return QP_ERR_ARG; m /= f; }
    while (m % 8 == 0) { if (!push(8)) return QP_ERR_ARG; m /= 8; }
    while (m % 4 == 0) { if (!push(4)) return QP_ERR_ARG; m /= 4; }
    if (m % 2 == 0) { if (!push(2)) return QP_ERR_ARG; m /= 2; }
    for (int f = 11; m > 1; f += 2) {
        while (m % f == 0) { if (!push(f)) return QP_ERR_ARG; m /= f; }
        if ((long)f * f > m && m > 1) { if (!push(m)) return QP_ERR_ARG; m = 1; }
    }
    // A thread for four elements; for one where a prime above 7 makes every output a sum
    // over that many terms (a 127^2 solve 80.6 us with 256 threads and 64-bit modulos, 47.7
    // us so; with a thread for four a 191 x 140 FP64 pass grew from 59.8 to 73.1 ms).
    dev.threads = 64 * ((n + 255) / 256);
    for (int s = 0; s < dev.nstages; ++s)
        if (dev.st[s].R > 8) dev.threads = std::min(256, 64 * ((n + 63) / 64));
    auto factor = [](int d) { return (1u << 22) / (unsigned)d + 1u; };
    int Ns = 1;
    for (int s = 0; s < dev.nstages; ++s) {
        FftAxisDev::Stage &t = dev.st[s];
        t.nR = n / t.R;
        t.fns = factor(Ns);
        Ns *= t.R;
        t.tws = n / Ns;
    }
    dev.tw = nullptr;
    return QP_OK;
}

int FftAxis::init(int n) {
    QP_TRY(plan(n));
    std::vector<double2> tw(n);
    const long double two_pi = 6.283185307179586476925286766559005768L;
    for (int t = 0; t < n; ++t) {
        long double a = two_pi * (long double)t / (long double)n;
        tw[t] = make_double2((double)cosl(a), (double)(-sinl(a)));
    }
    QP_HIP_CHECK(hipMalloc(&d_tw, sizeof(double2) * n));
    QP_HIP_CHECK(hipMemcpy(d_tw, tw.data(), sizeof(double2) * n, hipMemcpyHostToDevice));
    dev.tw = d_tw;
    return QP_OK;
}

void FftAxis::destroy() {
    if (d_tw) (void)hipFree(d_tw);
    d_tw = nullptr;
}

int Solver2d::set_steps(double d1_, double d2_) {
    d1 = d1_;
    d2 = d2_;
    // Same expression as the reference (src/System_3d.cpp:699), split per axis.
    std::vector<double> l1(n1), l2(nh);
    for (int j = 0; j < n1; ++j) l1[j] = (2 * cos(2 * M_PI * j / n1) - 2) / d1 / d1;
    for (int k = 0; k < nh; ++k) l2[k] = (2 * cos(2 * M_PI * k / n2) - 2) / d2 / d2;
    QP_HIP_CHECK(hipMemcpy(d_lam1, l1.data(), sizeof(double) * n1, hipMemcpyHostToDevice));
    QP_HIP_CHECK(hipMemcpy(d_lam2, l2.data(), sizeof(double) * nh, hipMemcpyHostToDevice));
    return QP_OK;
}

int Solver2d::init(int n1_, int n2_, double d1_, double d2_, int nbatch_) {
    nbatch = nbatch_ < 1 ? 1 : nbatch_;
    n1 = n1_;
    n2 = n2_;
    nh = n2 / 2 + 1;
    QP_TRY(ax1.init(n1));
    QP_TRY(ax2.init(n2));
    QP_HIP_CHECK(hipMalloc(&d_lam1, sizeof(double) * n1));
    QP_HIP_CHECK(hipMalloc(&d_lam2, sizeof(double) * nh));
    QP_TRY(set_steps(d1_, d2_));
    for (int i = 0; i < 2; ++i) QP_HIP_CHECK(hipMalloc(&spec[i], sizeof(double2) * (size_t)n1 * nh * nbatch));
    pick_kernels();
    return QP_OK;
}

// Kernel family of an n1 x n2 solver (no device work).
void Solver2d::pick_kernels() {
    // QP_FFT=generic keeps the generic kernels for every size (A/B comparisons).
    const char *sel = getenv("QP_FFT");
    wave = (wf_supported(n1) && wf_supported(n2) && !(sel && strcmp(sel, "generic") == 0)) ? 1 : 0;
}

void Solver2d::destroy() {
    ax1.destroy();
    ax2.destroy();
    if (d_lam1) (void)hipFree(d_lam1);
    if (d_lam2) (void)hipFree(d_lam2);
    for (int i = 0; i < 2; ++i)
        if (spec[i]) (void)hipFree(spec[i]);
    d_lam1 = d_lam2 = nullptr;
    spec[0] = spec[1] = nullptr;
}

// ------------------------------------------------------------ launches
int solve_cols(const Solver2d &S, double D, int nspec, hipStream_t s, const Ctl *ctl, int skip_mode) {
    if (S.wave) return wlaunch_cols(S, D, nspec, nullptr, s, ctl, skip_mode);
    return glaunch_cols(S, kColsSolve, D, nspec, nullptr, s, ctl, skip_mode);
}

int fourier_forward(const Solver2d &S, const double *src, double2 *spec, hipStream_t s) {
    QP_TRY(glaunch_rows_fwd(S, SrcPlain{src, S.n2}, spec, spec, 1, s, (const Ctl *)nullptr, 0, 1, true));
    return glaunch_cols(S, kColsForward, 0.0, 1, nullptr, s, nullptr, 0, 1, 0, true);
}

int fourier_backward(const Solver2d &S, double2 *spec, double *dst, hipStream_t s) {
    QP_TRY(glaunch_cols(S, kColsInverse, 0.0, 1, nullptr, s, nullptr, 0, 1, 0, true));
    return glaunch_rows_inv(S, (const double2 *)spec, (const double2 *)spec, SinkRaw{dst, S.n2}, 1, s,
                            (const Ctl *)nullptr, 0, 1, true);
}

int solve_plain(const Solver2d &S, double D, const double *src, double *dst, hipStream_t s) {
    const SrcPlain f{src, S.n2};
    const SinkRaw o{dst, S.n2};
    const Ctl *none = nullptr;
    const double2 *spec = S.spec[0];
    if (small_solve(S)) return slaunch(S, f, o, D, 1, s, none, 0);
    if (S.wave) {
        QP_TRY(wlaunch_rows_fwd(S, f, S.spec[0], S.spec[0], 1, s, NoCtl{}, 0));
        QP_TRY(wlaunch_cols(S, D, 1, nullptr, s, NoCtl{}, 0));
        return wlaunch_rows_inv(S, spec, spec, o, 1, s, NoCtl{}, 0);
    }
    QP_TRY(glaunch_rows_fwd(S, f, S.spec[0], S.spec[0], 1, s, none, 0));
    QP_TRY(solve_cols(S, D, 1, s, none, 0));
    return glaunch_rows_inv(S, spec, spec, o, 1, s, none, 0);
}

}  // namespace qp
