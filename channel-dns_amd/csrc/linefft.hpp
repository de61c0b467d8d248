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
#pragma once

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

// Dynamic LDS above 64 KB has to be allowed for each kernel and device; the attribute call is cheap
// and idempotent.
template <typename K> void allow_lds(K kernel, size_t bytes) {
    if (bytes > 64 * 1024)
        CDNS_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int)bytes));
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

} // namespace cdns
