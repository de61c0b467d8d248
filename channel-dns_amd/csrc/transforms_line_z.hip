// z stages with the line FFTs of runtime factors (linefft.hpp).
#include "linefft.hpp"

namespace cdns {

// ------------------------------------------------------------------ z stages --
// Backward: a block owns KT consecutive kx lines of one (field, l); its output goes through the LDS
// tile [iz][kx] so that HBM sees rows of KT values.
template <typename R, bool BIG>
__global__ void __launch_bounds__(512) k_zbwd_line(ZArgs a, LinePlan p) {
    extern __shared__ unsigned char smem_raw[];
    cpx<R> *tw = reinterpret_cast<cpx<R> *>(smem_raw), *buf = tw + p.n;
    const int N = p.n, NZS = a.NZS, KT = a.KT;
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63, g = lane / p.gs, t = lane - g * p.gs;
    const int line = wv * p.ng + g;
    const int nb = (a.nkx + KT - 1) / KT, L = xcd_block((int)gridDim.x);
    const int lf = L / nb, kx0 = (L - lf * nb) * KT, f = lf / a.NL, l = lf - f * a.NL;
    const int nl = min(KT, a.nkx - kx0);
    const bool on = g < p.ng && line < nl;
    const cpx<R> *Y = reinterpret_cast<const cpx<R> *>(a.in) + (size_t)f * a.in_fs + (size_t)l * a.QP +
                      (size_t)(on ? kx0 + line : 0) * a.nzk;
    load_line_roots<R>(tw, a.tw, N);
    __syncthreads();
    cpx<R> *T = buf + line * p.lb;
    // slot s holds kz = s (s <= NZS) or s - N (s >= N - NZS); at an overlap the slot N - NZS takes
    // kz = -NZS (transforms.cpp:717-726)
    auto slot = [&](int s) {
        const bool low = s <= NZS && s != N - NZS, high = s >= N - NZS;
        const cpx<R> v = Y[low ? s + NZS : (high ? s - N + NZS : 0)];
        return cpx<R>{low || high ? v.x : R(0), low || high ? v.y : R(0)};
    };
    pass_a<R, +1, BIG>(p, t, on, tw, T, slot, NoSync{});
    lsync();
    const int pitch = KT | 1;
    pass_b<R, +1, BIG>(p, t, on, T, [&](int iz, cpx<R> v) { buf[iz * pitch + line] = v; }, Bsync{});
    __syncthreads();
    cpx<R> *Z = reinterpret_cast<cpx<R> *>(a.out) + (size_t)f * a.out_fs + (size_t)l * N * a.nkx + kx0;
    for (int e = threadIdx.x; e < N * nl; e += blockDim.x) {
        const int iz = e / nl, li = e - iz * nl;
        Z[(size_t)iz * a.nkx + li] = buf[iz * pitch + li];
    }
}

// Forward: lines of the line-major layout, one wavefront per block; keeps the retained kz, x 1/NZ2.
template <typename R, bool BIG>
__global__ void __launch_bounds__(64) k_zfwd_line(ZArgs a, LinePlan p) {
    extern __shared__ unsigned char smem_raw[];
    const cpx<R> *tw = reinterpret_cast<const cpx<R> *>(a.tw); // cache-resident, as in the tuned kernel
    const int N = p.n, NZS = a.NZS;
    const int lane = threadIdx.x, g = lane / p.gs, t = lane - g * p.gs;
    const int L = xcd_block((int)gridDim.x);
    const int kxg = L % a.nkxg, lf = L / a.nkxg, l = lf % a.NL, f = lf / a.NL;
    const int kx = kxg * p.ng + g;
    const bool on = g < p.ng && kx < a.nkx;
    const cpx<R> *Z = reinterpret_cast<const cpx<R> *>(a.in) + (size_t)f * a.in_fs +
                      ((size_t)l * a.nkx + (on ? kx : 0)) * N;
    cpx<R> *T = reinterpret_cast<cpx<R> *>(smem_raw) + g * p.lb;
    pass_a<R, -1, BIG>(p, t, on, tw, T, [&](int n) { return Z[n]; }, NoSync{});
    lsync();
    const R inv = R(1.0 / N);
    cpx<R> *Y = reinterpret_cast<cpx<R> *>(a.out) + (size_t)f * a.out_fs + (size_t)l * a.QP + (size_t)(on ? kx : 0) * a.nzk;
    pass_b<R, -1, BIG>(
        p, t, on, T,
        [&](int s, cpx<R> v) {
            const cpx<R> o = {inv * v.x, inv * v.y};
            if (s <= NZS) Y[s + NZS] = o;
            if (s >= N - NZS) Y[s - N + NZS] = o;
        },
        NoSync{});
}

// ------------------------------------------------------------------ launch --
namespace {

template <typename R, bool BIG> void go_zbwd_line(ZArgs a, const LinePlan &p, int nf, hipStream_t st) {
    // up to 16 lines per block, the same number in every block, with at most 8 wavefronts
    // and two blocks in a CU's LDS
    auto waves = [&](int kt) { return (kt + p.ng - 1) / p.ng; };
    auto lds = [&](int kt) {
        return ((size_t)std::max(waves(kt) * p.ng * p.lb, p.n * (kt | 1)) + p.n) * sizeof(cpx<R>);
    };
    int cap = std::min(16, 8 * p.ng);
    while (cap > 1 && lds(cap) > 80 * 1024) --cap;
    const int nb = (a.nkx + cap - 1) / cap;
    a.KT = (a.nkx + nb - 1) / nb;
    allow_lds(k_zbwd_line<R, BIG>, lds(a.KT));
    hipLaunchKernelGGL((k_zbwd_line<R, BIG>), dim3((a.nkx + a.KT - 1) / a.KT * a.NL * nf), dim3(64 * waves(a.KT)),
                       lds(a.KT), st, a, p);
}
template <typename R, bool BIG> void go_zfwd_line(ZArgs a, const LinePlan &p, int nf, hipStream_t st) {
    a.nkxg = (a.nkx + p.ng - 1) / p.ng;
    hipLaunchKernelGGL((k_zfwd_line<R, BIG>), dim3(a.nkxg * a.NL * nf), dim3(64),
                       (size_t)p.ng * p.lb * sizeof(cpx<R>), st, a, p);
}

} // namespace
bool launch_zbwd_line(const ZArgs &a, int nf, bool fp32, hipStream_t st) {
    LinePlan p;
    if (a.coarse || !line_plan(a.plan.n, p)) return false;
    line_dispatch(p, fp32, [&](auto r, auto big) { go_zbwd_line<decltype(r), decltype(big)::value>(a, p, nf, st); });
    return true;
}
bool launch_zfwd_line(const ZArgs &a, int nf, bool fp32, hipStream_t st) {
    LinePlan p;
    if (a.coarse || !line_plan(a.plan.n, p)) return false;
    line_dispatch(p, fp32, [&](auto r, auto big) { go_zfwd_line<decltype(r), decltype(big)::value>(a, p, nf, st); });
    return true;
}

} // namespace cdns
