// qp_output.hip -- what a pass hands to the host while it runs: per-slice output, where the
// planes of a view leave the device in one launch (output_step, src/System_3d.cpp:629-666,
// writes them slice by slice), and the number of members that have not stopped.
#include <climits>
#include <string>
#include <thread>

#include "qp_wake.h"

namespace qp {

namespace {

constexpr int kPackT = 256;

// blockIdx.y: the plane, kOutPlanes for the control blocks.  Bound by the link when dst
// is pinned host memory and by launch latency when it is device memory: what it saves is
// the twelve or thirteen copy commands of a slice, each with its own start and end.  A
// 64^2 x 200-slice pass with streamed output 49.0 -> 42.5 ms, a 200^2 x 120-slice one
// 52.5 -> 48.7 ms, a 200^2 x 60-slice FP64 pass with inline output 68.8 -> 62.3 ms.
__global__ __launch_bounds__(kPackT) void k_pack(OutPlanes o, size_t plane, const double *ctl, size_t ctl_words,
                                                 double *dst) {
    const int f = blockIdx.y;
    const double *src = f < kOutPlanes ? o.p[f] : ctl;
    const size_t n = f < kOutPlanes ? plane : ctl_words;
    if (!src && f >= kOutPlanes - 1) return;  // no bx, no control blocks
    double *d = dst + (size_t)f * plane;
    for (size_t t = (size_t)blockIdx.x * kPackT + threadIdx.x; t < n; t += (size_t)gridDim.x * kPackT)
        d[t] = src ? src[t] : 0.0;
}

}  // namespace

void watch_reset(Wake *w) {
    for (int m = 0; m < w->nw; ++m) w->h_prog[m] = INT_MAX;
}

int watch_stops(Wake *const *b, int nb, int i, hipStream_t s, int &running) {
    int first = INT_MAX;  // the slice that the device has reached
    auto read = [&] {
        running = 0;
        for (int k = 0; k < nb; ++k)
            for (int m = 0; m < b[k]->nw; ++m) {
                const int p = __atomic_load_n(b[k]->h_prog + m, __ATOMIC_RELAXED);
                if (p == kStopped) continue;
                ++running;
                first = p < first ? p : first;
            }
    };
    read();
    // slice i + 1 set a mark: wait for the one before it, i + 1 + kWatchSlices
    const int mark = i + 1 + kWatchSlices;
    if ((i + 1) % kWatchSlices != 0 || mark >= b[0]->p.nx) return QP_OK;
    for (unsigned turn = 1; running && first > mark; ++turn) {
        if (turn % 65536 == 0) {  // the wait ends with the stream, whatever ended it
            const hipError_t e = hipStreamQuery(s);
            if (e != hipErrorNotReady) {
                read();
                QP_HIP_CHECK(e);
                return QP_OK;
            }
        }
        std::this_thread::yield();
        read();
    }
    return QP_OK;
}

int pack_planes(const OutPlanes &o, size_t plane, const Ctl *ctl, int nctl, double *dst, hipStream_t s) {
    const size_t blocks = (plane + kPackT - 1) / kPackT;
    hipLaunchKernelGGL(k_pack, dim3((unsigned)(blocks < 4096 ? blocks : 4096), kOutPlanes + 1), dim3(kPackT), 0, s, o,
                       plane, reinterpret_cast<const double *>(ctl), kCtlWords * (size_t)nctl, dst);
    QP_HIP_CHECK(hipGetLastError());
    return QP_OK;
}

int stage_slice(Wake *w, const OutPlanes &o, const Ctl *ctl, Ctl *host_ctl) {
    hipStream_t s = w->stream();
    // the kernel writes the pinned buffer itself: one launch, no copy command per plane
    QP_TRY(pack_planes(o, w->nn(), ctl, ctl ? 1 : 0, w->h_out, s));
    QP_HIP_CHECK(hipStreamSynchronize(s));
    if (ctl && host_ctl) *host_ctl = *reinterpret_cast<const Ctl *>(w->h_out + kOutPlanes * w->nn());
    return QP_OK;
}

int call_slice(Wake *w, qp_slice_cb cb, void *user, int slice, int kind, bool with_bx) {
    const size_t nn = w->nn();
    const double *h = w->h_out;
    qp_slice_view v;
    v.slice = slice;
    v.kind = kind;
    v.psi = h;
    v.rho = h + nn;
    v.jx = h + 2 * nn;
    v.jy = h + 3 * nn;
    v.jz = h + 4 * nn;
    v.ex = h + 5 * nn;
    v.ey = h + 6 * nn;
    v.ez = h + 7 * nn;
    v.by = h + 8 * nn;
    v.bz = h + 9 * nn;
    v.chi = h + 10 * nn;
    v.bx = with_bx ? h + 11 * nn : nullptr;
    const int r = cb(&v, user);
    if (r != 0) {
        set_error("slice callback returned " + std::to_string(r));
        return QP_ERR_STATE;
    }
    return QP_OK;
}

int deliver_slice(Wake *w, qp_slice_cb cb, void *user, int slice, int kind, const OutPlanes &o) {
    QP_TRY(stage_slice(w, o, nullptr, nullptr));
    return call_slice(w, cb, user, slice, kind, o.p[kOutPlanes - 1] != nullptr);
}

}  // namespace qp
