// x stages of single physical fields with the line FFTs of runtime factors (linefft.hpp).
#include "linefft.hpp"

namespace cdns {

// ------------------------------------------- single-field x stages (physical) --
// A block carries P consecutive (l, iz) points, two of them per complex line a + i b, of one field
// (blockIdx.y).  The physical rows are whole runs in HBM: they pass through the line buffers so that a
// wavefront moves one row at a time; the forward stage's retained kx go out as rows of P points.
template <typename R, bool BIG>
__global__ void __launch_bounds__(512) k_xbwd_phys_line(XArgs a, LinePlan p) {
    extern __shared__ unsigned char smem_raw[];
    cpx<R> *tw = reinterpret_cast<cpx<R> *>(smem_raw), *buf = tw + p.n;
    const int N = p.n, K = a.nkx - 1, P = a.P, np = a.NL * a.NZ2, p0 = blockIdx.x * P;
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63, g = lane / p.gs, t = lane - g * p.gs;
    const int line = wv * p.ng + g, pa = p0 + 2 * line, pb = pa + 1;
    const bool on = g < p.ng && 2 * line < P && pa < np;
    const cpx<R> *Z = reinterpret_cast<const cpx<R> *>(a.in) + (size_t)blockIdx.y * a.in_fs;
    const cpx<R> *A = Z + (size_t)(on ? pa : 0) * a.nkx, *B = Z + (size_t)(on && pb < np ? pb : 0) * a.nkx;
    load_line_roots<R>(tw, a.tw, N);
    __syncthreads();
    cpx<R> *T = buf + line * p.lb;
    auto slot = [&](int k) {
        const cpx<R> v = pack_pair(A, B, k, N, K, on, on && pb < np);
        // coarse grid, NXS = N/2: the Nyquist coefficient doubled (transforms.cpp:576-578)
        const R w = a.coarse && 2 * k == N ? R(2) : R(1);
        return cpx<R>{w * v.x, w * v.y};
    };
    pass_a<R, +1, BIG>(p, t, on, tw, T, slot, NoSync{});
    lsync();
    pass_b<R, +1, BIG>(p, t, on, T, [&](int n, cpx<R> v) { T[n] = v; }, Lsync{});
    __syncthreads();
    double *phys = a.phys + (size_t)blockIdx.y * a.phys_fs;
    for (int j = wv; j < P && p0 + j < np; j += blockDim.x >> 6) {
        const int l = (p0 + j) / a.NZ2, iz = p0 + j - l * a.NZ2;
        double *row = phys + ((size_t)iz * a.NL + l) * N;
        const R *src = reinterpret_cast<const R *>(buf + (j >> 1) * p.lb) + (j & 1);
        for (int n = lane; n < N; n += 64) row[n] = double(src[2 * n]);
    }
}

// U: rows in flight per wavefront (a block's 16 rows over its wavefronts)
template <typename R, bool BIG, int U>
__global__ void __launch_bounds__(512) k_xfwd_phys_line(XArgs a, LinePlan p) {
    extern __shared__ unsigned char smem_raw[];
    cpx<R> *tw = reinterpret_cast<cpx<R> *>(smem_raw), *buf = tw + p.n;
    const int N = p.n, P = a.P, np = a.NL * a.NZ2, p0 = blockIdx.x * P;
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63, g = lane / p.gs, t = lane - g * p.gs;
    const int line = wv * p.ng + g;
    const bool on = g < p.ng && 2 * line < P && p0 + 2 * line < np;
    load_line_roots<R>(tw, a.tw, N);
    // rows wv, wv + W, ... of the block on wavefront wv, U loads in flight
    const int W = blockDim.x >> 6, w0 = __builtin_amdgcn_readfirstlane(wv);
    for (int j0 = w0; j0 < P; j0 += U * W) {
        const double *row[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int pt = min(p0 + min(j0 + u * W, P - 1), np - 1), l = pt / a.NZ2, iz = pt - l * a.NZ2;
            row[u] = a.phys + ((size_t)iz * a.NL + l) * N;
        }
        for (int n = lane; n < N; n += 64) {
            double v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) v[u] = row[u][n];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int j = j0 + u * W;
                if (j < P) reinterpret_cast<R *>(buf + (j >> 1) * p.lb + n)[j & 1] = p0 + j < np ? R(v[u]) : R(0);
            }
        }
    }
    __syncthreads();
    cpx<R> *T = buf + line * p.lb;
    pass_a<R, -1, BIG>(p, t, on, tw, T, [&](int n) { return T[n]; }, Lsync{});
    lsync();
    pass_b<R, -1, BIG>(p, t, on, T, [&](int k, cpx<R> v) { T[k] = v; }, Lsync{});
    __syncthreads();
    const R half = R(0.5) / R(N);
    const int wj = threadIdx.x % P, pw = p0 + wj;
    if (pw >= np) return;
    const int wl = pw / a.NZ2;
    cpx<R> *ZN = reinterpret_cast<cpx<R> *>(a.out) + ((size_t)wl * a.nkx) * a.NZ2 + (pw - wl * a.NZ2);
    const cpx<R> *F = buf + (wj >> 1) * p.lb;
    for (int k = threadIdx.x / P; k < a.nkx; k += blockDim.x / P) {
        const cpx<R> f = F[k], m = F[k == 0 ? 0 : N - k];
        // coarse grid, NXS = N/2: the Nyquist coefficient halved (transforms.cpp:496-497)
        const R hk = a.coarse && 2 * k == N ? R(0.5) * half : half;
        ZN[(size_t)k * a.NZ2] = (wj & 1) ? cpx<R>{hk * (f.y + m.y), hk * (m.x - f.x)}
                                         : cpx<R>{hk * (f.x + m.x), hk * (f.y - m.y)};
    }
}

// ------------------------------------------------------------------ launch --
namespace {

// 16 points (256-byte output rows of the forward stage in FP64) on at least the wavefronts that their eight lines
// need.  Short lines need one or two, which then move all 16 rows by themselves: a grid that is resident as a
// whole with four wavefronts a block (or two) takes four (two).  us per launch (about 5 of them the events'), as
// needed / four, backward and forward: 10-point lines of 38 blocks FP64 8.5 / 6.4, 8.7 / 6.4; 42 points, 160 blocks
// 9.2 / 7.0, 9.2 / 6.9; 96 points, 294 blocks FP32 9.3 / 8.2, 9.0 / 8.1; 144 points, 657 blocks FP64 13.4 / 11.9,
// 13.0 / 12.2; 196 points, 1213 blocks FP32 15.8 / 14.4, 16.6 / 15.4.  Beyond that (FP64 backward: 768 blocks) the
// smaller blocks pack better: 196 points, 1213 blocks FP64 19.2 / 21.8, 19.1 / 21.1; 30 points, 3015 blocks
// 14.3 / 18.5, 14.6 / 17.2.
constexpr int kXPhysWaves = 4;
size_t xphys_lds(const LinePlan &p, size_t esz) { return ((size_t)kXPhysPoints / 2 * p.lb + p.n) * esz; }
int xphys_waves(const LinePlan &p) { return (kXPhysPoints / 2 + p.ng - 1) / p.ng; }
// resident blocks of `waves` wavefronts; the wavefronts that the registers of a kernel leave a CU are asked for once
template <auto Kernel> int xphys_resident(int waves, size_t lds) {
    static const int slots = [] {
        int n = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, Kernel, 64, 0) == hipSuccess) return n;
        (void)hipGetLastError();
        return 0;
    }();
    constexpr size_t kCuLds = 160 * 1024;
    return device_cus() * std::min(slots / waves, (int)(kCuLds / lds));
}
// Wide: the kernel for four wavefronts a block, Narrow: for fewer
template <auto Narrow, auto Wide> void go_xphys_line(size_t esz, XArgs a, const LinePlan &p, int nf, hipStream_t st) {
    a.P = kXPhysPoints;
    const int blocks = (a.NL * a.NZ2 + a.P - 1) / a.P;
    const size_t lds = xphys_lds(p, esz);
    int waves = xphys_waves(p);
    for (int w = kXPhysWaves; w > waves; w /= 2)
        if (blocks * nf <= (w < kXPhysWaves ? xphys_resident<Narrow>(w, lds) : xphys_resident<Wide>(w, lds))) waves = w;
    const auto kernel = waves < kXPhysWaves ? Narrow : Wide;
    allow_lds(kernel, lds);
    hipLaunchKernelGGL(kernel, dim3(blocks, nf), dim3(64 * waves), lds, st, a, p);
}
} // namespace

int xphys_line_resident(int n, bool fp32, bool backward, bool wide) {
    LinePlan p;
    if (!line_plan(n, p)) return 0;
    int blocks = 0;
    line_dispatch(p, fp32, [&](auto r, auto big) {
        using R = decltype(r);
        constexpr bool B = decltype(big)::value;
        const int waves = wide ? std::max(kXPhysWaves, xphys_waves(p)) : xphys_waves(p);
        const size_t lds = xphys_lds(p, sizeof(cpx<R>));
        if (backward) blocks = xphys_resident<&k_xbwd_phys_line<R, B>>(waves, lds);
        else if (waves < kXPhysWaves) blocks = xphys_resident<&k_xfwd_phys_line<R, B, 8>>(waves, lds);
        else blocks = xphys_resident<&k_xfwd_phys_line<R, B, 4>>(waves, lds);
    });
    return blocks;
}

bool launch_xbwd_phys_line(const XArgs &a, int nf, bool fp32, hipStream_t st) {
    LinePlan p;
    if (!line_plan(a.plan.n, p)) return false;
    line_dispatch(p, fp32, [&](auto r, auto big) {
        using R = decltype(r);
        constexpr bool B = decltype(big)::value;
        go_xphys_line<&k_xbwd_phys_line<R, B>, &k_xbwd_phys_line<R, B>>(sizeof(cpx<R>), a, p, nf, st);
    });
    return true;
}
bool launch_xfwd_phys_line(const XArgs &a, bool fp32, hipStream_t st) {
    LinePlan p;
    if (!line_plan(a.plan.n, p)) return false;
    line_dispatch(p, fp32, [&](auto r, auto big) {
        using R = decltype(r);
        constexpr bool B = decltype(big)::value;
        go_xphys_line<&k_xfwd_phys_line<R, B, 8>, &k_xfwd_phys_line<R, B, 4>>(sizeof(cpx<R>), a, p, 1, st);
    });
    return true;
}

} // namespace cdns
