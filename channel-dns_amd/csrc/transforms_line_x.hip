// x stages with the line FFTs of runtime factors (linefft.hpp).
#include "linefft.hpp"

namespace cdns {

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
    const int np = a.NL * a.NZ2, p0 = xcd_block((int)gridDim.x) * P;
    const int line = wv * p.ng + g; // backward: line i of point j at 3 j + i
    const bool lane_on = g < p.ng;
    const int j = line / 3, i = line - 3 * j;
    const bool on = lane_on && j < P;
    const bool valid = on && p0 + j < np;
    {
        const void *fa = i == 0 ? a.fin[blockIdx.y][0] : (i == 1 ? a.fin[blockIdx.y][2] : a.fin[blockIdx.y][4]);
        const void *fb = i == 0 ? a.fin[blockIdx.y][1] : (i == 1 ? a.fin[blockIdx.y][3] : a.fin[blockIdx.y][5]);
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
    cpx<R> *o0 = reinterpret_cast<cpx<R> *>(a.fout[blockIdx.y][0]) + base, *o1 = reinterpret_cast<cpx<R> *>(a.fout[blockIdx.y][1]) + base,
           *o2 = reinterpret_cast<cpx<R> *>(a.fout[blockIdx.y][2]) + base;
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

// ------------------------------------------------------------------ launch --
namespace {

template <typename R, bool BIG> void go_xprod_line(XArgs a, const LinePlan &p, hipStream_t st) {
    // Four points per block: 12 lines on 2 to 6 wavefronts.  More points write longer output rows but
    // wait longer at the three block barriers, and the LDS then holds fewer blocks (150 x 126 lines of
    // a 136-plane grid, FP64: 2, 4, 8 points 75.7, 64.7, 92.3 us; FP32 46.1, 38.6, 43.5).
    const int P = 4, waves = (3 * P + p.ng - 1) / p.ng;
    const size_t lds = ((size_t)3 * P * p.lb + p.n) * sizeof(cpx<R>);
    a.P = P;
    allow_lds(k_xprod_line<R, BIG>, lds);
    hipLaunchKernelGGL((k_xprod_line<R, BIG>), dim3((a.NL * a.NZ2 + P - 1) / P, a.nprod), dim3(64 * waves), lds, st, a, p);
}
} // namespace

bool launch_xprod_line(const XArgs &a, bool fp32, hipStream_t st) {
    LinePlan p;
    if (!line_plan(a.plan.n, p)) return false;
    line_dispatch(p, fp32, [&](auto r, auto big) { go_xprod_line<decltype(r), decltype(big)::value>(a, p, st); });
    return true;
}

} // namespace cdns
