// Line FFTs of runtime factors: the x and z stages for every length N = N1 x N2 with factors of the
// list below.  transforms_rf.hip instantiates the two-pass register FFT for a few tuned lengths; here
// one kernel per stage serves all of them: the factors are kernel arguments, each pass switches
// (uniformly over the grid) to the register DFT of its factor, and no value stays in registers
// between passes, so the allocation is that of the largest DFT and not of a whole line.
//
//   pass A: lane t < N1 of a line's group loads x[t + N1 j], j < N2; DFT of length N2; times w^(t k);
//           to the line's LDS buffer T[t][k]
//   pass B: lane t < N2 reads T[i][t], i < N1; DFT of length N1 -> X[t + N2 k]
//
// A group has exactly max(N1, N2) lanes, so a wavefront carries 64 / max(N1, N2) lines.  What bounds
// the stages is LDS and HBM traffic with few waves resident, not arithmetic: a line crosses LDS twice
// per transform, where the Stockham kernels of transforms.hip cross it twice per radix (8 to 12 times
// at these lengths) with a workgroup barrier and integer divisions at each.  Measured against them
// (z backward 6 fields, x product, z forward 3 fields; us per launch):
//   product grid 150 x 136 x 126  FP64 95.8, 180, 44.9 -> 36.7, 64.7, 21.8   FP32 51.4, 108, 27.4 -> 24.2, 38.6, 14.2
//   product grid 216 x 161 x 240  FP64 319, 573, 113 -> 112, 234, 52         FP32 128, 306, 59 -> 63, 123, 27
// The lengths of transforms_rf.hip stay there: its lane-pair kernels keep a point's three physical
// lines in registers (196 x 193 x 196, FP64: x product 112 us there, 151 us here).
#include "internal.hpp"
#include "regfft.hpp"

#include <algorithm>

namespace cdns {

#define CDNS_LINE_RADICES(X) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(12) X(14) X(15) X(16)
#define CDNS_LINE_RADICES_BIG(X) X(18) X(20) X(21) X(24) X(25) X(27)

// Factors of a length and the lane and LDS layout that follow from them.
struct LinePlan {
    int n, n1, n2;
    int gs, ng; // lanes per line, lines per wavefront
    int pa;     // row pitch of the pass-A output (odd: the rows of a group start on distinct banks)
    int lb;     // entries of one line's buffer (odd, for the same reason between lines)
};

namespace {

constexpr bool is_line_radix(int r) {
#define X(A) if (r == A) return true;
    CDNS_LINE_RADICES(X) CDNS_LINE_RADICES_BIG(X)
#undef X
    return false;
}
constexpr int kSmallRadix = 16;

// The factor pair with the smaller larger factor; false when there is none.
bool line_plan(int n, LinePlan &p) {
    int best = 0;
    for (int r = 2; r * r <= n; ++r)
        if (n % r == 0 && is_line_radix(r) && is_line_radix(n / r)) best = r;
    if (!best) return false;
    p.n = n;
    p.n1 = best;
    p.n2 = n / best;
    p.gs = p.n2;
    p.ng = 64 / p.gs;
    p.pa = p.n2 | 1;
    p.lb = std::max(p.n1 * p.pa, n) | 1;
    return true;
}

struct NoSync {
    __device__ inline void operator()() const {}
};

// f(integral constant r) for the radix r; BIG: the radices above 16 too
template <bool BIG, typename F> __device__ __attribute__((always_inline)) inline void with_radix(int r, F &&f) {
    switch (r) {
#define X(A) case A: f(ic<A>{}); break;
        CDNS_LINE_RADICES(X)
#undef X
    default:
        if constexpr (BIG) {
            switch (r) {
#define X(A) case A: f(ic<A>{}); break;
                CDNS_LINE_RADICES_BIG(X)
#undef X
            default: break;
            }
        }
    }
}

// load(n) gives x[n] of this lane's line; mid() runs, on every lane, after the last load and before
// the first store to T
template <typename R, int S, bool BIG, typename Load, typename Mid>
__device__ __attribute__((always_inline)) inline void pass_a(const LinePlan &p, int t, bool on, const cpx<R> *tw, cpx<R> *T, Load load,
                                                             Mid mid) {
    with_radix<BIG>(p.n2, [&](auto rad) {
        constexpr int N2 = decltype(rad)::value;
        cpx<R> x[N2];
        if (on && t < p.n1) {
            sfor<0, N2>([&](auto j) { x[j] = load(t + p.n1 * decltype(j)::value); });
            RDft<R, N2, S>::run(x);
            sfor<1, N2>([&](auto k) {
                cpx<R> w = tw[t * decltype(k)::value];
                if (S > 0) w.y = -w.y;
                x[k] = cpx<R>{x[k].x * w.x - x[k].y * w.y, x[k].x * w.y + x[k].y * w.x};
            });
        }
        mid();
        if (on && t < p.n1) sfor<0, N2>([&](auto k) { T[t * p.pa + decltype(k)::value] = x[k]; });
    });
}
// store(k, X[k]); mid() as above, between the reads of T and the stores
template <typename R, int S, bool BIG, typename Store, typename Mid>
__device__ __attribute__((always_inline)) inline void pass_b(const LinePlan &p, int t, bool on, const cpx<R> *T, Store store, Mid mid) {
    with_radix<BIG>(p.n1, [&](auto rad) {
        constexpr int N1 = decltype(rad)::value;
        cpx<R> x[N1];
        if (on && t < p.n2) {
            sfor<0, N1>([&](auto i) { x[i] = T[decltype(i)::value * p.pa + t]; });
            RDft<R, N1, S>::run(x);
        }
        mid();
        if (on && t < p.n2) sfor<0, N1>([&](auto k) { store(t + p.n2 * decltype(k)::value, x[k]); });
    });
}

struct Lsync {
    __device__ inline void operator()() const { lsync(); }
};
struct Bsync {
    __device__ inline void operator()() const { __syncthreads(); }
};

// Slot k of the full-length array whose inverse DFT is a + i b for the real lines with half spectra
// at A and B, kx <= K (c2r: the imaginary parts of DC and Nyquist are ignored).  Branch-free: both
// loads are issued for every lane at a clamped index and the value is selected afterwards.
template <typename R>
__device__ inline cpx<R> pack_pair(const cpx<R> *A, const cpx<R> *B, int k, int N, int K, bool usea, bool useb) {
    const bool mirror = k > K, zero = mirror && N - k > K;
    int src = mirror ? N - k : k;
    src = src > K ? K : src;
    cpx<R> av = A[src], bv = B[src];
    const bool real_end = src == 0 || 2 * src == N;
    const R ay = real_end ? R(0) : (mirror ? -av.y : av.y), by = real_end ? R(0) : (mirror ? -bv.y : bv.y);
    const R ax = usea && !zero ? av.x : R(0), bx = useb && !zero ? bv.x : R(0);
    return {ax - (useb && !zero ? by : R(0)), (usea && !zero ? ay : R(0)) + bx};
}

template <typename R> __device__ inline void load_line_roots(cpx<R> *tw, const void *src, int n) {
    const cpx<R> *s = reinterpret_cast<const cpx<R> *>(src);
    for (int i = threadIdx.x; i < n; i += blockDim.x) tw[i] = s[i];
}

} // namespace

// ------------------------------------------------------- x stage + product --
// A block carries P consecutive (l, iz) points: 3 P c2r lines (u,v), (w,wx), (wy,wz), one lane group
// each; the products are formed where the forward transforms load their input (P lines Nx + i Ny and
// P/2 lines Nz of two points); the retained kx go out as rows of P points of the line-major layout.
template <typename R, bool BIG>
__global__ void __launch_bounds__(512) k_xprod_line(XArgs a, LinePlan p) {
    extern __shared__ unsigned char smem_raw[];
    cpx<R> *tw = reinterpret_cast<cpx<R> *>(smem_raw), *buf = tw + p.n;
    const int N = p.n, K = a.nkx - 1, P = a.P, lb = p.lb;
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63, g = lane / p.gs, t = lane - g * p.gs;
    const int np = a.NL * a.NZ2, p0 = blockIdx.x * P;
    const int line = wv * p.ng + g; // backward: line i of point j at 3 j + i
    const bool lane_on = g < p.ng;
    const int j = line / 3, i = line - 3 * j;
    const bool on = lane_on && j < P;
    const bool valid = on && p0 + j < np;
    {
        const void *fa = i == 0 ? a.fin[0] : (i == 1 ? a.fin[2] : a.fin[4]);
        const void *fb = i == 0 ? a.fin[1] : (i == 1 ? a.fin[3] : a.fin[5]);
        const size_t row = (size_t)(valid ? p0 + j : 0) * a.nkx;
        const cpx<R> *A = reinterpret_cast<const cpx<R> *>(fa) + row, *B = reinterpret_cast<const cpx<R> *>(fb) + row;
        load_line_roots<R>(tw, a.tw, N);
        __syncthreads();
        cpx<R> *T = buf + line * lb;
        pass_a<R, +1, BIG>(p, t, on, tw, T, [&](int k) { return pack_pair(A, B, k, N, K, valid, valid); }, NoSync{});
        lsync();
        pass_b<R, +1, BIG>(p, t, on, T, [&](int n, cpx<R> v) { T[n] = v; }, Lsync{});
    }
    __syncthreads();
    // forward line f < P: Nx + i Ny of point f, in the buffer of its first line; f = P + h: Nz of the
    // points 2h and 2h + 1, in the second buffer of point 2h
    const bool fon = lane_on && line < P + P / 2;
    const int h2 = 2 * (line - P);
    cpx<R> *T = buf + (line < P ? 3 * line : 3 * h2 + 1) * lb;
    const cpx<R> *C = buf + 3 * (line < P ? line : h2) * lb;
    auto product = [&](int n) {
        const cpx<R> c0 = C[n], c1 = C[lb + n], c2 = C[2 * lb + n];
        const R u = c0.x, v = c0.y, w = c1.x, ox = c1.y, oy = c2.x, oz = c2.y;
        if (line < P) return cpx<R>{v * oz - w * oy, w * ox - u * oz};
        const cpx<R> d0 = C[3 * lb + n], d2 = C[5 * lb + n];
        return cpx<R>{u * oy - v * ox, d0.x * d2.x - d0.y * C[4 * lb + n].y};
    };
    pass_a<R, -1, BIG>(p, t, fon, tw, T, product, Bsync{});
    lsync();
    pass_b<R, -1, BIG>(p, t, fon, T, [&](int k, cpx<R> v) { T[k] = v; }, Lsync{});
    __syncthreads();
    const R half = R(0.5) / R(N);
    const int wj = threadIdx.x % P, pw = p0 + wj;
    if (pw >= np) return;
    const int wl = pw / a.NZ2;
    const size_t base = ((size_t)wl * a.nkx) * a.NZ2 + (pw - wl * a.NZ2);
    cpx<R> *o0 = reinterpret_cast<cpx<R> *>(a.fout[0]) + base, *o1 = reinterpret_cast<cpx<R> *>(a.fout[1]) + base,
           *o2 = reinterpret_cast<cpx<R> *>(a.fout[2]) + base;
    const cpx<R> *F = buf + 3 * wj * lb, *Z = buf + (3 * (wj & ~1) + 1) * lb;
    for (int k = threadIdx.x / P; k < a.nkx; k += blockDim.x / P) {
        const int m = k == 0 ? 0 : N - k;
        const cpx<R> f = F[k], fm = F[m], z = Z[k], zm = Z[m];
        const size_t o = (size_t)k * a.NZ2;
        o0[o] = {half * (f.x + fm.x), half * (f.y - fm.y)};
        o1[o] = {half * (f.y + fm.y), half * (fm.x - f.x)};
        if (wj & 1) o2[o] = {half * (z.y + zm.y), half * (zm.x - z.x)};
        else o2[o] = {half * (z.x + zm.x), half * (z.y - zm.y)};
    }
}

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
    const int kx0 = blockIdx.x * KT, l = blockIdx.y, f = blockIdx.z;
    const int nl = min(KT, a.nkx - kx0);
    const bool on = g < p.ng && line < nl;
    const cpx<R> *Y = reinterpret_cast<const cpx<R> *>(a.in) + (size_t)f * a.in_fs + (size_t)l * a.NQ +
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
    cpx<R> *Y = reinterpret_cast<cpx<R> *>(a.out) + (size_t)f * a.out_fs + (size_t)l * a.NQ + (size_t)(on ? kx : 0) * a.nzk;
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

// Dynamic LDS above 64 KB has to be allowed for each kernel and device; the attribute call is cheap
// and idempotent.
template <typename K> void allow_lds(K kernel, size_t bytes) {
    if (bytes > 64 * 1024)
        CDNS_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int)bytes));
}

template <typename R, bool BIG> void go_xprod_line(XArgs a, const LinePlan &p, hipStream_t st) {
    // Four points per block: 12 lines on 2 to 6 wavefronts.  More points write longer output rows but
    // wait longer at the three block barriers, and the LDS then holds fewer blocks (150 x 126 lines of
    // a 136-plane grid, FP64: 2, 4, 8 points 75.7, 64.7, 92.3 us; FP32 46.1, 38.6, 43.5).
    const int P = 4, waves = (3 * P + p.ng - 1) / p.ng;
    const size_t lds = ((size_t)3 * P * p.lb + p.n) * sizeof(cpx<R>);
    a.P = P;
    allow_lds(k_xprod_line<R, BIG>, lds);
    hipLaunchKernelGGL((k_xprod_line<R, BIG>), dim3((a.NL * a.NZ2 + P - 1) / P), dim3(64 * waves), lds, st, a, p);
}
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
    hipLaunchKernelGGL((k_zbwd_line<R, BIG>), dim3((a.nkx + a.KT - 1) / a.KT, a.NL, nf), dim3(64 * waves(a.KT)),
                       lds(a.KT), st, a, p);
}
template <typename R, bool BIG> void go_zfwd_line(ZArgs a, const LinePlan &p, int nf, hipStream_t st) {
    a.nkxg = (a.nkx + p.ng - 1) / p.ng;
    hipLaunchKernelGGL((k_zfwd_line<R, BIG>), dim3(a.nkxg * a.NL * nf), dim3(64),
                       (size_t)p.ng * p.lb * sizeof(cpx<R>), st, a, p);
}

// f(type tag, BIG tag) for the precision and the factors of a plan
template <typename F> void line_dispatch(const LinePlan &p, bool fp32, F &&f) {
    const bool big = p.n2 > kSmallRadix;
    if (fp32) {
        if (big) f(float{}, std::true_type{});
        else f(float{}, std::false_type{});
    } else {
        if (big) f(double{}, std::true_type{});
        else f(double{}, std::false_type{});
    }
}

} // namespace

bool launch_xprod_line(const XArgs &a, bool fp32, hipStream_t st) {
    LinePlan p;
    if (!line_plan(a.plan.n, p)) return false;
    line_dispatch(p, fp32, [&](auto r, auto big) { go_xprod_line<decltype(r), decltype(big)::value>(a, p, st); });
    return true;
}
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
