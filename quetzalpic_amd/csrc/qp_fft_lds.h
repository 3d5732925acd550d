// qp_fft_lds.h -- one complex FFT of any length up to 1024 held in LDS (device code).
//
// Stockham autosort, mixed radix, natural order in and out.  Stage with radix
// R after sub-transforms of size Ns:
//   for j in [0, n/R), k = j mod Ns:
//     v_r = in[j + r n/R] * w^{k r (n/(Ns R))}         (w = e^{-2 pi i / n})
//     out[(j/Ns) Ns R + k + q Ns] = sum_r v_r w_R^{r q}
// Radices 2 to 5, 7 and 8 use register butterflies (dft<R> of qp_wave_fft.h); a
// larger prime evaluates each output as sum_r in[j + r n/R] * w^{r (k + q Ns) n/(Ns R)}.
// Only the forward transform is coded: the inverse of z is the forward of z with
// its parts swapped, swapped back, which costs nothing where the values are
// written and read.
//
// What bounds these launches is the instruction stream of a wavefront that has its
// SIMD to itself (few blocks, four elements of one transform to a lane).  So odd radices
// stay at 5 and 7 and go first (with padded addresses, 32-bit multiplies and an eight
// ahead of the fives a row pass at 200 took 7.4 us), index divisions are a 24-bit
// multiply and a shift with factors from the host, element addresses have no padding
// (consecutive lanes read consecutive elements; only the first stage's writes can meet
// in a bank), a block of one wavefront orders its stages without barriers, loads go out
// four to a lane, and the column pass runs both directions through one copy of the code.
// Solve launches at 200^2: rows 9.5 -> 5.7-6.7 us, columns 12.0 -> 7.5 us (before: one
// kernel for any radix, the fives as direct sums with a 64-bit modulo per term).
#pragma once

#include "qp_wave_fft.h"

namespace qp {

// Quotient x / d for x < 1024 and the factor f = 2^22 / d + 1 (d <= 1024): the error
// x (f d - 2^22) / (2^22 d) < 1024 d / (2^22 d) stays below 1/d.
__device__ __forceinline__ int quot(int x, unsigned f) {
    return (int)((unsigned)__umul24((unsigned)x, f) >> 22);  // (the product can pass 2^31)
}
__device__ __forceinline__ int mul24(int a, int b) { return (int)__umul24((unsigned)a, (unsigned)b); }

// The axis twiddle table on its way to LDS: every lane loads its entries (element
// threadIdx + r T, r < 4; a block has a thread for four elements) before it loads
// data, and writes them before the sync that precedes lds_fft.  In a plain copy loop
// each turn waited for its own load.
struct LdsTw {
    double2 w[4];
    __device__ __forceinline__ void load(const FftAxisDev &ax) {
#pragma unroll
        for (int r = 0; r < 4; ++r) w[r] = ax.tw[min((int)threadIdx.x + r * (int)blockDim.x, ax.n - 1)];
    }
    __device__ __forceinline__ void store(double2 *tw_lds, int n) const {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int t = threadIdx.x + r * blockDim.x;
            if (t < n) tw_lds[t] = w[r];
        }
    }
};

// Orders LDS accesses of a block of one wavefront (ONE) or several.
template <bool ONE>
__device__ __forceinline__ void lds_sync() {
    wf_sync<ONE ? 64 : 128>();
}

// One stage of NT transforms stored n apart.
template <int R, int NT>
__device__ __forceinline__ void lds_stage(const double2 *a, double2 *b, int n, int nR, int Ns, int tws, unsigned fns,
                                          const double2 *twl) {
    for (int j = threadIdx.x; j < nR; j += blockDim.x) {
        const int k = j - mul24(quot(j, fns), Ns);
        const int t = mul24(k, tws), o = mul24(j, R) - mul24(k, R - 1);  // (j/Ns) Ns R + k
        double2 u[NT][R];
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            const double2 *in = a + i * n + j;
#pragma unroll
            for (int r = 0; r < R; ++r) u[i][r] = in[r * nR];
        }
        if (k != 0) {
            double2 w[R];
#pragma unroll
            for (int r = 1; r < R; ++r) w[r] = twl[r * t];
#pragma unroll
            for (int i = 0; i < NT; ++i)
#pragma unroll
                for (int r = 1; r < R; ++r) u[i][r] = cmul(u[i][r], w[r]);
        }
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            dft<R, -1>(u[i]);
            double2 *out = b + i * n + o;
#pragma unroll
            for (int q = 0; q < R; ++q) out[q * Ns] = u[i][q];
        }
    }
}

// Forward transform of NT sequences of length ax.n, n apart in `a`; `b` is scratch of
// the same size; `twl` is the LDS copy of the twiddles.  All threads of the block call
// it, after a sync; a sync ends it.  Returns the buffer holding the result (a or b).
template <bool ONE, int NT = 1>
__device__ inline double2 *lds_fft(double2 *a, double2 *b, const FftAxisDev &ax, const double2 *twl) {
    const int n = ax.n;
    int Ns = 1;
    FftAxisDev::Stage st = ax.st[0];
    for (int s = 0; s < ax.nstages; ++s) {
        const FftAxisDev::Stage next = ax.st[s + 1];
        const int R = st.R, nR = st.nR, tws = st.tws;
        const unsigned fns = st.fns;
        switch (R) {
            case 2: lds_stage<2, NT>(a, b, n, nR, Ns, tws, fns, twl); break;
            case 3: lds_stage<3, NT>(a, b, n, nR, Ns, tws, fns, twl); break;
            case 4: lds_stage<4, NT>(a, b, n, nR, Ns, tws, fns, twl); break;
            case 5: lds_stage<5, NT>(a, b, n, nR, Ns, tws, fns, twl); break;
            case 8: lds_stage<8, NT>(a, b, n, nR, Ns, tws, fns, twl); break;
            case 7: lds_stage<7, NT>(a, b, n, nR, Ns, tws, fns, twl); break;
            default: {
                // one output per thread and turn: idx = q nR + j
                const unsigned fnb = (1u << 22) / (unsigned)nR + 1u;
                for (int idx = threadIdx.x; idx < n; idx += blockDim.x) {
                    const int q = quot(idx, fnb), j = idx - mul24(q, nR);
                    const int jn = quot(j, fns), k = j - mul24(jn, Ns);
                    const int kNs = k + mul24(q, Ns), kq = mul24(kNs, tws);  // < n
#pragma unroll
                    for (int i = 0; i < NT; ++i) {
                        const double2 *in = a + i * n + j;
                        double2 acc = *in;
                        int ti = 0;
                        for (int r = 1; r < R; ++r) {
                            ti += kq;
                            if (ti >= n) ti -= n;
                            in += nR;
                            acc = cadd(acc, cmul(*in, twl[ti]));
                        }
                        b[i * n + mul24(mul24(jn, Ns), R) + kNs] = acc;
                    }
                }
            }
        }
        lds_sync<ONE>();
        double2 *tmp = a;
        a = b;
        b = tmp;
        Ns *= R;
        st = next;
    }
    return a;
}

}  // namespace qp
