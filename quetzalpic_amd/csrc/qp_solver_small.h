// qp_solver_small.h -- the periodic 2D solve of a small grid in one launch.
//
// A small solve is three dependent launches of 3.1-3.6 us each, none with work for more
// than a few CUs: what they take is the launches themselves, the way of the spectrum
// through memory between them, and one transform's latency each.  Here one block makes
// the whole solve with the half spectrum in LDS: rows forward, columns (forward, divide,
// inverse), rows inverse, on the transforms of qp_wave_fft.h.  A transform lies inside one
// wavefront, so the block meets twice only, at the transposes.  Same sources and sinks,
// same member convention (blockIdx.y = wake * nspec + which).
// The transforms give the three launches' bits; psi's border mean sums the same terms in
// another order (wavefront by wavefront), so psi agrees to rounding.
// One CU's LDS bandwidth, its loads and FP64 rate bound it now (64^2: 9 us in a slice, its
// sources coming from other CUs' deposits), so it ends at sides of 64.  Eight elements to a
// lane instead of four (half the exchanges, half the wavefronts) took as long.
// A chain of plain solves: 32^2 8.6 -> 4.3 us, 48^2 10.5 -> 7.4, 64^2 9.6-10.4 -> 7.4.  A 200-slice
// wake of 48^2 48.0 -> 37.4 ms, of 64^2 42.5 -> 39.0 (FP64 61.7 -> 57.9); batches of 24 wakes of
// 48^2 15.3 -> 13.2 ms, of 64^2 16.7 -> 16.2, of two wakes of 64^2 9.6 -> 10.0 (12.1 before the
// three launches were shortened).  Sides of 16 keep the three launches: not measured.
#pragma once

#include <type_traits>

#include "qp_wave_solver.h"

namespace qp {

// Sinks that need the border-mean sums (SinkPsiFinal) take them from the block.
template <class Sink, class = void>
struct sink_takes_sums : std::false_type {};
template <class Sink>
struct sink_takes_sums<Sink, std::void_t<decltype(&Sink::set_sums)>> : std::true_type {};

template <int N1, int N2>
struct SmallCfg {
    static constexpr int E1 = WfCfg<N1>::E, E2 = WfCfg<N2>::E, L1 = N1 / E1, L2 = N2 / E2;
    static constexpr int NP = N1 / 2, NH = N2 / 2 + 1;  // row pairs, columns (N1 is even)
    static_assert(64 % L1 == 0 && 64 % L2 == 0, "a transform lies inside one wavefront");
    static constexpr int T = NP * L2 > NH * L1 ? NP * L2 : NH * L1;
    static constexpr int TB = (T + 63) / 64 * 64;
    static_assert(TB <= 1024, "one transform per group of lanes");
    static constexpr int P1 = WfShape<N1, E1, 64>::PADN, P2 = WfShape<N2, E2, 64>::PADN;
    static constexpr int BUF = NP * P2 > NH * P1 ? NP * P2 : NH * P1;  // exchange buffer of all groups
    static constexpr int COL = N1 + 1;                                 // column stride of the spectrum
};

template <int N1, int N2, class Src, class Sink>
__global__ __launch_bounds__((SmallCfg<N1, N2>::TB)) void k_solve_small(Src src, Sink sink, const double2 *tw1g,
                                                                      const double2 *tw2g, const double *lam1,
                                                                      const double *lam2, double D, const Ctl *ctl,
                                                                      int skip_mode, int nspec) {
    using C = SmallCfg<N1, N2>;
    constexpr int E1 = C::E1, E2 = C::E2, L1 = C::L1, L2 = C::L2, COL = C::COL, NW = C::TB / 64;
    __shared__ double2 sb0[C::BUF], sb1[C::BUF], spec[C::NH * COL];
    __shared__ double part[3][NW];
    const int which = blockIdx.y % nspec, wk = blockIdx.y / nspec, tid = threadIdx.x;
    if (ctl) ctl += wk;
    const int skip = solver_skip_flag(ctl, skip_mode);
    const int t = tid / L2, j2 = tid % L2, l = tid / L1, j1 = tid % L1;
    const bool row = t < C::NP, col = l < C::NH;
    const int ra = 2 * t, rb = ra + 1;
    WfTw<N2, E2, 64> tw2;
    tw2.init(tw2g, nullptr, j2);
    double2 v[E2];
    {
        double xa[E2], xb[E2];
#pragma unroll
        for (int r = 0; r < E2; ++r) xa[r] = xb[r] = 0.0;
        if (row) {
            src.template row<E2>(wk, which, ra, j2, L2, xa);
            src.template row<E2>(wk, which, rb, j2, L2, xb);
        }
#pragma unroll
        for (int r = 0; r < E2; ++r) v[r] = make_double2(xa[r], xb[r]);
    }
    // the column pass's factors and twiddles with the first loads
    WfTw<N1, E1, 64> tw1;
    tw1.init(tw1g, nullptr, j1);
    double lm[E1];
#pragma unroll
    for (int r = 0; r < E1; ++r) lm[r] = lam1[j1 + L1 * r];
    const double l2 = col ? lam2[l] : 0.0;
    keep_here(v);
    if (solver_skip_act(ctl, skip_mode, skip)) return;
    if (row) {
        src.template done<E2>(wk, which, ra, j2, L2);
        src.template done<E2>(wk, which, rb, j2, L2);
    }
    const int bt = row ? t : 0, bl = col ? l : 0;
    double2 *b0 = sb0 + bt * C::P2, *b1 = sb1 + bt * C::P2;
    if (row) {
        // z = x_a + i x_b: X_a[k] = (Z[k] + conj Z[-k])/2, X_b[k] = (Z[k] - conj Z[-k])/(2i)
        wave_fft<N2, E2, -1>(v, b0, b1, tw2, j2);
        wf_sync<L2>();
#pragma unroll
        for (int m = 0; m < E2; ++m) b0[wf_pad(j2 + L2 * m)] = v[m];
        wf_sync<L2>();
#pragma unroll
        for (int i = 0; i <= E2 / 2; ++i) {
            const int k = j2 + L2 * i;
            if (k <= N2 / 2) {
                const double2 Z = b0[wf_pad(k)], Zm = b0[wf_pad(k == 0 ? 0 : N2 - k)];
                spec[k * COL + ra] = make_double2(0.5 * (Z.x + Zm.x), 0.5 * (Z.y - Zm.y));
                spec[k * COL + rb] = make_double2(0.5 * (Z.y + Zm.y), -0.5 * (Z.x - Zm.x));
            }
        }
    }
    __syncthreads();
    // columns, in place (as wcols_body, which also derives the border-mean sums)
    double s1 = 0.0, s2 = 0.0, g00 = 0.0;
    if (col) {
        double2 u[E1], *c = spec + bl * COL;
        double2 *c0 = sb0 + bl * C::P1, *c1 = sb1 + bl * C::P1;
#pragma unroll
        for (int r = 0; r < E1; ++r) u[r] = c[j1 + L1 * r];
        wave_fft<N1, E1, -1>(u, c0, c1, tw1, j1);
        double g = 0.0;
#pragma unroll
        for (int m = 0; m < E1; ++m) {
            const double inv = 1.0 / (-D + lm[m] + l2);
            u[m].x *= inv;
            u[m].y *= inv;
            if (l == 0 && j1 == 0 && m == 0) u[m] = make_double2(0.0, 0.0);
            g += u[m].x;
        }
        const double wl = (l == 0 || 2 * l == N2) ? 1.0 : 2.0;
        s1 = j1 == 0 ? wl * (double)N1 * u[0].x : 0.0;
        s2 = wl * g;
        g00 = l == 0 ? g : 0.0;
        wave_fft<N1, E1, +1>(u, c0, c1, tw1, j1);
#pragma unroll
        for (int m = 0; m < E1; ++m) c[j1 + L1 * m] = u[m];
    }
    if constexpr (sink_takes_sums<Sink>::value) {
        s1 = wave_sum(s1);
        s2 = wave_sum(s2);
        g00 = wave_sum(g00);
        if ((tid & 63) == 0) {
            part[0][tid >> 6] = s1;
            part[1][tid >> 6] = s2;
            part[2][tid >> 6] = g00;
        }
    }
    __syncthreads();
    if constexpr (sink_takes_sums<Sink>::value) {
        s1 = s2 = g00 = 0.0;
#pragma unroll
        for (int i = 0; i < NW; ++i) {
            s1 += part[0][i];
            s2 += part[1][i];
            g00 += part[2][i];
        }
        sink.set_sums(s1, s2, g00);
    } else {
        sink.begin(wk);
    }
    if (!row) return;
    // rows inverse (as wrows_inv_body)
#pragma unroll
    for (int r = 0; r < E2; ++r) {
        const int k = j2 + L2 * r;
        const bool cj = k > N2 / 2;
        const int kk = cj ? N2 - k : k;
        double2 X = spec[kk * COL + ra], Y = spec[kk * COL + rb];
        if (cj) {
            X.y = -X.y;
            Y.y = -Y.y;
        }
        if (kk == 0 || 2 * kk == N2) X.y = Y.y = 0.0;
        v[r] = make_double2(X.x - Y.y, X.y + Y.x);
    }
    wave_fft<N2, E2, +1>(v, b0, b1, tw2, j2);
#pragma unroll
    for (int m = 0; m < E2; ++m) {
        const int k = j2 + L2 * m;
        sink(wk, which, ra, k, v[m].x);
        sink(wk, which, rb, k, v[m].y);
    }
}

// Sides served by the one launch.
constexpr bool small_side(int n) { return n == 32 || n == 48 || n == 64; }
inline bool small_solve(const Solver2d &S) { return S.wave && small_side(S.n1) && small_side(S.n2); }

template <class Src, class Sink>
int slaunch(const Solver2d &S, const Src &src, const Sink &sink, double D, int nspec, hipStream_t s, const Ctl *ctl,
            int skip_mode, int nw = 1) {
    auto go = [&](auto N1C, auto N2C) {
        constexpr int N1 = decltype(N1C)::value, N2 = decltype(N2C)::value;
        hipLaunchKernelGGL((k_solve_small<N1, N2, Src, Sink>), dim3(1, nspec * nw), dim3(SmallCfg<N1, N2>::TB), 0, s,
                           src, sink, (const double2 *)S.ax1.dev.tw, (const double2 *)S.ax2.dev.tw,
                           (const double *)S.d_lam1, (const double *)S.d_lam2, D, ctl, skip_mode, nspec);
    };
    auto side = [](int n, auto &&f) {
        if (n == 32) f(std::integral_constant<int, 32>{});
        else if (n == 48) f(std::integral_constant<int, 48>{});
        else f(std::integral_constant<int, 64>{});
    };
    side(S.n1, [&](auto N1C) { side(S.n2, [&](auto N2C) { go(N1C, N2C); }); });
    QP_HIP_CHECK(hipGetLastError());
    return QP_OK;
}

}  // namespace qp
