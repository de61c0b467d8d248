// Spectral-space kernels: curl with the curl part of the pressure wall condition, and
// conversions between the reference's interleaved layout and the backend's column planes.
#include "internal.hpp"
#include "wave.hpp"

namespace cdns {

// vector_ops::enqueue_curl (src/solver/vector_ops.cpp:112-151) plus the curl terms of
// TimeStepper::enqueue_pressure_boundary (src/solver/timestepper.cpp:26-43):
//   wx = D w - i kz v,  wy = i kz u - i kx w,  wz = i kx v - D u,
//   bcw(wall 0) = sum_j t_j,  bcw(wall 1) = sum_j (-1)^(j+1) t_j,  t_j = (i kx/Re) wz_j - (i kz/Re) wx_j.
// One wavefront per (kx,kz) column.
template <int CH>
__global__ void __launch_bounds__(256) k_curl(CurlArgs a) {
    const int lane = lane_id();
    const int q = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (q >= a.NQ) return;
    const int kxi = q / a.nzk, kzi = q - kxi * a.nzk;
    const double kx = a.WAVX[kxi], kz = a.WAVZ[kzi];
    const size_t off = (size_t)q * a.JS;
    zd u[2][CH], v[2][CH], w[2][CH], du[2][CH], dw[2][CH];
    load_col<CH>(a.u[0] + off, lane, a.ny, u);
    load_col<CH>(a.u[1] + off, lane, a.ny, v);
    load_col<CH>(a.u[2] + off, lane, a.ny, w);
    cheb_dy<CH>(u, du, lane, a.ny);
    cheb_dy<CH>(w, dw, lane, a.ny);
    zd ox[2][CH], oy[2][CH], oz[2][CH];
    zd s0 = {0.0, 0.0}, s1 = {0.0, 0.0};
    const zd cxre = {0.0 / a.Re, kx / a.Re}, czre = {0.0, kz / a.Re};
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            ox[p][c] = dw[p][c] - ikmul(kz, v[p][c]);
            oy[p][c] = ikmul(kz, u[p][c]) - ikmul(kx, w[p][c]);
            oz[p][c] = ikmul(kx, v[p][c]) - du[p][c];
            const int j = jof<CH>(lane, c, p);
            if (j <= a.ny) {
                const zd t = cmul(cxre, oz[p][c]) - cmul(czre, ox[p][c]);
                s0 = s0 + t;
                s1 = (p == 0) ? s1 - t : s1 + t;
            }
        }
    store_col<CH>(a.w[0] + off, lane, a.ny, ox);
    store_col<CH>(a.w[1] + off, lane, a.ny, oy);
    store_col<CH>(a.w[2] + off, lane, a.ny, oz);
    if (a.bcw) {
        s0 = wave_sum(s0);
        s1 = wave_sum(s1);
        if (lane == 0) {
            a.bcw[(size_t)q * 2 + 0] = s0;
            a.bcw[(size_t)q * 2 + 1] = s1;
        }
    }
}

void launch_curl(const CurlArgs &a, int E, hipStream_t st) {
    dim3 grid((a.NQ + 3) / 4), block(256);
    if (E == 2) hipLaunchKernelGGL((k_curl<1>), grid, block, 0, st, a);
    else if (E == 4) hipLaunchKernelGGL((k_curl<2>), grid, block, 0, st, a);
    else throw std::runtime_error("unsupported column length");
}

template <int CH>
__global__ void __launch_bounds__(256) k_wall_sum(const zd *nly, const zd *bcw, zd *pbc, int ny, int JS, int NQ) {
    const int lane = lane_id();
    const int q = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (q >= NQ) return;
    zd n[2][CH];
    load_col<CH>(nly + (size_t)q * JS, lane, ny, n);
    zd s0 = {0.0, 0.0}, s1 = {0.0, 0.0};
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            s0 = s0 + n[p][c];
            s1 = p == 0 ? s1 - n[p][c] : s1 + n[p][c];
        }
    s0 = wave_sum(s0);
    s1 = wave_sum(s1);
    if (lane == 0) {
        pbc[(size_t)q * 2 + 0] = bcw[(size_t)q * 2 + 0] + s0;
        pbc[(size_t)q * 2 + 1] = bcw[(size_t)q * 2 + 1] + s1;
    }
}
void launch_wall_sum(const zd *nly, const zd *bcw, zd *pbc, int ny, int JS, int NQ, int E, hipStream_t st) {
    dim3 grid((NQ + 3) / 4), block(256);
    if (E == 2) hipLaunchKernelGGL((k_wall_sum<1>), grid, block, 0, st, nly, bcw, pbc, ny, JS, NQ);
    else hipLaunchKernelGGL((k_wall_sum<2>), grid, block, 0, st, nly, bcw, pbc, ny, JS, NQ);
}

// Reference layout (izi, row, kx, c) <-> plane c, column q = kx*nzk + izi, row.  For one izi this is a
// transpose of (row, kx) per component: a block carries a tile of kLayRows rows x TK kx through LDS, so
// that the reference side moves runs of TK*NC values (768 bytes for vectors) and the plane side runs of
// kLayRows values (512 bytes).  HBM-bound; without the tile one side moved single 16-byte values at a
// stride of a row (Re_tau=180: velocity to planes 45.8 -> 23.9 us with it, velocity and pressure back
// 64 -> 33 us; 102 MB and 136 MB).
constexpr int kLayRows = 32;
template <int NC> constexpr int kLayKx = NC == 1 ? 32 : 16;
template <int NC> struct LayTile {
    static constexpr int TK = kLayKx<NC>, W = TK * NC, PITCH = kLayRows + 1, N = kLayRows * W;
    // entry of component c, tile column k, tile row r
    __device__ static inline int at(int c, int k, int r) { return (c * TK + k) * PITCH + r; }
};

// rows beyond nrow (the planes' padding) are written as zeros
template <int NC> __global__ void __launch_bounds__(256) k_ref_to_planes(LayoutArgs a) {
    using T = LayTile<NC>;
    __shared__ zd tile[NC * T::TK * T::PITCH];
    const int kx0 = blockIdx.x * T::TK, r0 = blockIdx.y * kLayRows, izi = blockIdx.z;
    const zd *ref = a.ref_in + (size_t)izi * a.nrow * a.nkx * a.stride;
#pragma unroll
    for (int e = threadIdx.x; e < T::N; e += 256) {
        const int r = e / T::W, w = e - r * T::W, k = w / NC, c = w - k * NC;
        const bool in = r0 + r < a.nrow && kx0 + k < a.nkx;
        const zd v = ref[in ? ((size_t)(r0 + r) * a.nkx + kx0 + k) * a.stride + c : 0];
        tile[T::at(c, k, r)] = in ? v : zd{0.0, 0.0};
    }
    __syncthreads();
#pragma unroll
    for (int e = threadIdx.x; e < T::N; e += 256) {
        const int w = e / kLayRows, r = e - w * kLayRows, c = w / T::TK, k = w - c * T::TK;
        if (r0 + r < a.JS && kx0 + k < a.nkx)
            a.plane_out[c][((size_t)(kx0 + k) * a.nzk + izi) * a.JS + r0 + r] = tile[T::at(c, k, r)];
    }
}
template <int NC> __global__ void __launch_bounds__(256) k_planes_to_ref(LayoutArgs a) {
    using T = LayTile<NC>;
    __shared__ zd tile[NC * T::TK * T::PITCH];
    const int kx0 = blockIdx.x * T::TK, r0 = blockIdx.y * kLayRows, izi = blockIdx.z;
#pragma unroll
    for (int e = threadIdx.x; e < T::N; e += 256) {
        const int w = e / kLayRows, r = e - w * kLayRows, c = w / T::TK, k = w - c * T::TK;
        const bool in = r0 + r < a.nrow && kx0 + k < a.nkx;
        tile[T::at(c, k, r)] = a.plane_in[c][in ? ((size_t)(kx0 + k) * a.nzk + izi) * a.JS + r0 + r : 0];
    }
    __syncthreads();
    zd *ref = a.ref_out + (size_t)izi * a.nrow * a.nkx * a.stride;
#pragma unroll
    for (int e = threadIdx.x; e < T::N; e += 256) {
        const int r = e / T::W, w = e - r * T::W, k = w / NC, c = w - k * NC;
        if (r0 + r < a.nrow && kx0 + k < a.nkx)
            ref[((size_t)(r0 + r) * a.nkx + kx0 + k) * a.stride + c] = tile[T::at(c, k, r)];
    }
}
__global__ void k_real_planes_to_ref(const double *plane, double *ref, int nrow, int nkx, int nzk, int JS) {
    const size_t total = (size_t)nzk * nrow * nkx;
    for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < total; e += (size_t)gridDim.x * blockDim.x) {
        const int kx = (int)(e % nkx);
        const size_t r = e / nkx;
        const int row = (int)(r % nrow), izi = (int)(r / nrow);
        ref[e] = plane[((size_t)kx * nzk + izi) * JS + row];
    }
}

static dim3 grid_for(size_t n) {
    size_t b = (n + 255) / 256;
    if (b > 65535 * 4) b = 65535 * 4;
    return dim3((unsigned)(b ? b : 1));
}

// n complex entries between an FP64 plane and a single-precision plane (the mixed step's N)
__global__ void k_widen(const cpx<float> *src, zd *dst, size_t n) {
    for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x)
        dst[e] = {double(src[e].x), double(src[e].y)};
}
__global__ void k_narrow(const zd *src, cpx<float> *dst, size_t n) {
    for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x)
        dst[e] = {float(src[e].x), float(src[e].y)};
}
// One launch for the ten planes of an adjoint checkpoint: as ten device copies each waits for the one
// before (64 x 65 x 64, 20 MB: 49 us of copy kernels, in one launch 10 us).
__global__ void __launch_bounds__(256) k_copy_planes(CopyArgs a) {
    const zd *src = a.src[blockIdx.y];
    zd *dst = a.dst[blockIdx.y];
    const size_t n = a.n[blockIdx.y];
    for (size_t e = blockIdx.x * (size_t)256 + threadIdx.x; e < n; e += (size_t)gridDim.x * 256) dst[e] = src[e];
}
void launch_copy_planes(const CopyArgs &a, hipStream_t st) {
    size_t most = 0;
    for (int i = 0; i < a.count; ++i) most = a.n[i] > most ? a.n[i] : most;
    const unsigned blocks = (unsigned)((most + 1023) / 1024); // four values a thread
    hipLaunchKernelGGL(k_copy_planes, dim3(blocks ? blocks : 1, a.count), dim3(256), 0, st, a);
}
void launch_widen(const void *src, zd *dst, size_t n, hipStream_t st) {
    hipLaunchKernelGGL(k_widen, grid_for(n), dim3(256), 0, st, reinterpret_cast<const cpx<float> *>(src), dst, n);
}
void launch_narrow(const zd *src, void *dst, size_t n, hipStream_t st) {
    hipLaunchKernelGGL(k_narrow, grid_for(n), dim3(256), 0, st, src, reinterpret_cast<cpx<float> *>(dst), n);
}
template <int NC> static dim3 layout_grid(const LayoutArgs &a, int rows) {
    return dim3((a.nkx + kLayKx<NC> - 1) / kLayKx<NC>, (rows + kLayRows - 1) / kLayRows, a.nzk);
}
void launch_ref_to_planes(const LayoutArgs &a, hipStream_t st) {
    if (a.ncomp == 1) hipLaunchKernelGGL(k_ref_to_planes<1>, layout_grid<1>(a, a.JS), dim3(256), 0, st, a);
    else if (a.ncomp == 3) hipLaunchKernelGGL(k_ref_to_planes<3>, layout_grid<3>(a, a.JS), dim3(256), 0, st, a);
    else throw std::runtime_error("unsupported number of components");
}
void launch_planes_to_ref(const LayoutArgs &a, hipStream_t st) {
    if (a.ncomp == 1) hipLaunchKernelGGL(k_planes_to_ref<1>, layout_grid<1>(a, a.nrow), dim3(256), 0, st, a);
    else if (a.ncomp == 3) hipLaunchKernelGGL(k_planes_to_ref<3>, layout_grid<3>(a, a.nrow), dim3(256), 0, st, a);
    else throw std::runtime_error("unsupported number of components");
}
void launch_real_planes_to_ref(const double *plane, double *ref, int nrow, int nkx, int nzk, int JS, hipStream_t st) {
    hipLaunchKernelGGL(k_real_planes_to_ref, grid_for((size_t)nzk * nrow * nkx), dim3(256), 0, st, plane, ref, nrow,
                       nkx, nzk, JS);
}

} // namespace cdns
