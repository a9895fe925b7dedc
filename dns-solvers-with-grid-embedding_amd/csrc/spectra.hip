// spectra.hip -- 1-D energy spectra of the velocity planes (dnsg_spectra).
//
// The reference computes them offline from the velocity files (e-spectra/src/
// 1d-spectra-mgrd.c:119-230): per wall-normal plane a 2-D real-to-complex DFT over
// (x streamwise, y spanwise) of u, v, w, scaled by 1/(N0 N1), the mean mode
// removed, then
//   E_x(i) = sum_j fac_j 1/2 |c(i, j)|^2   (streamwise wavenumber index i, all N0)
//   E_y(j) = sum_i fac_j 1/2 |c(i, j)|^2   (spanwise index j = 0 .. N1/2)
// with fac_j = 1 for j = 0 and 2 otherwise (the folded half of the spectrum).
// Here the velocity planes are formed on the device from the lattice (the
// vel_print.c formula), transformed with hipFFT in one batched plan, and folded by a wave
// per E_x value and a workgroup per 64 E_y values.
#include <hipfft/hipfft.h>

#include <new>

#include "internal.hpp"
#include "lattice.hpp"

namespace dnsg {

namespace {

// Velocity planes vel[3][nzg][nx][ny] (y fastest: the DFT's last, halved dimension) of every
// layer of a grid's velocity file, its wall layer kwall (-1: none) from the wall-layer copy
// [nx][ny][19].  A workgroup takes a tile of TS x TS columns of one layer: the lattice is
// read along x and the planes written along y, through LDS (written along x, the stores
// were a line each: 0.45 ms for the Re_tau=180 FP32 grids, now 0.1; the wall layer used to
// be formed on the host).
constexpr int TS = 32, TB = 256;
template <class S>
__global__ __launch_bounds__(TB) void k_vel_planes(const S *__restrict__ lat, const double *__restrict__ wall, int nx,
                                                   int ny, int zlo, int kwall, int nzg, double *__restrict__ vel) {
    __shared__ double t[3][TS][TS + 1];  // [component][y][x]
    const int nxc = (nx + TS - 1) / TS, nyc = (ny + TS - 1) / TS;
    const int x0 = (int)(blockIdx.x % nxc) * TS, y0 = (int)(blockIdx.x / nxc % nyc) * TS, k = (int)(blockIdx.x / (nxc * nyc));
    const int c = threadIdx.x % TS, r0 = threadIdx.x / TS;
    for (int r = r0; r < TS; r += TB / TS) {
        const int x = x0 + c, y = y0 + r;
        if (x >= nx || y >= ny) continue;
        double ux = 0., uy = 0., uz = 0., dens = 0.;
        unroll<0, Q>([&](auto qc) {  // vel_print.c:86-104, in its order
            constexpr int q = decltype(qc)::value;
            double f;
            if (k == kwall) {
                f = wall[((size_t)x * ny + y) * Q + q];
            } else {
                f = (double)load_s(lat + lat_at(q, (size_t)(k - zlo) * ny + y, x, nx));
                if constexpr (sizeof(S) != 8) f += WQ[q];
            }
            ux += (double)EX[q] * f;
            uy += (double)EY[q] * f;
            uz += (double)EZ[q] * f;
            dens += f;
        });
        if (dens > 0.) { ux /= dens; uy /= dens; uz /= dens; }
        else { ux = 0.; uy = 0.; uz = 0.; }
        t[0][r][c] = ux;
        t[1][r][c] = uy;
        t[2][r][c] = uz;
    }
    __syncthreads();
    for (int r = r0; r < TS; r += TB / TS) {  // row r: x = x0 + r, lanes along y
        const int x = x0 + r, y = y0 + c;
        if (x >= nx || y >= ny) continue;
#pragma unroll
        for (int m = 0; m < 3; m++) vel[(((size_t)m * nzg + k) * nx + x) * ny + y] = t[m][c][r];
    }
}

// E_x(c, i, k) of the DFT coefficients cf[3 nzg][N0][N1h]: one wave per (c, k, i), its lanes
// along j; then E_y(c, j, k): one thread per value, lanes along j, over i in order
__device__ __forceinline__ double fold_term(const double2 c, double s, int i, int j) {
    if (i == 0 && j == 0) return 0.;  // the mean removed (1d-spectra-mgrd.c:195-200)
    const double re = c.x * s, im = c.y * s;
    const double fac = j == 0 ? 1. : 2.;
    return fac * 0.5 * (re * re + im * im);
}
__global__ __launch_bounds__(TB) void k_fold_x(const double2 *__restrict__ cf, int N0, int N1, int nzg, double *__restrict__ ex) {
    const int N1h = N1 / 2 + 1, lane = threadIdx.x & 63;
    const long t = (long)blockIdx.x * (TB / 64) + (threadIdx.x >> 6);  // (c k, i)
    if (t >= 3L * nzg * N0) return;
    const int i = (int)(t % N0), k = (int)((t / N0) % nzg), c = (int)(t / ((long)N0 * nzg));
    const double s = 2. * (1. / ((double)(2. * N0 * N1)));  // 1d-spectra-mgrd.c:183
    const double2 *p = cf + (size_t)t * N1h;
    double e = 0.;
    for (int j = lane; j < N1h; j += 64) e += fold_term(p[j], s, i, j);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) e += __shfl_down(e, o, 64);
    if (lane == 0) ex[((size_t)c * N0 + i) * nzg + k] = e;
}
// a workgroup: 64 wavenumbers j of one (c, k), its waves sharing the N0 rows
__global__ __launch_bounds__(TB) void k_fold_y(const double2 *__restrict__ cf, int N0, int N1, int nzg, double *__restrict__ ey) {
    __shared__ double l[TB / 64][64];
    const int N1h = N1 / 2 + 1, njc = (N1h + 63) / 64, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int j = (int)(blockIdx.x % njc) * 64 + lane, ck = (int)(blockIdx.x / njc), k = ck % nzg, c = ck / nzg;
    const double s = 2. * (1. / ((double)(2. * N0 * N1)));
    const double2 *p = cf + (size_t)ck * N0 * N1h;
    double e = 0.;
    if (j < N1h)
        for (int i = w; i < N0; i += TB / 64) e += fold_term(p[(size_t)i * N1h + j], s, i, j);
    l[w][lane] = e;
    __syncthreads();
    if (w == 0 && j < N1h) {
        double a = l[0][lane];
        for (int v = 1; v < TB / 64; v++) a += l[v][lane];
        ey[((size_t)c * N1h + j) * nzg + k] = a;
    }
}

// A plan's preparation takes 8 ms of host time, its transforms of the Re_tau=180 grids
// under 1 ms, so a handle keeps the plans of its coarse grid and of its bands (equal in
// size) from their first use; the work area, as large as the data, lives for the call.
struct FftPlan {
    hipfftHandle plan;
    size_t work;
};

FftPlan *fft_plan(void **slot, int N0, int N1, int batch) {
    if (*slot) return static_cast<FftPlan *>(*slot);
    FftPlan *f = new (std::nothrow) FftPlan{};
    if (!f) return nullptr;
    if (hipfftCreate(&f->plan) != HIPFFT_SUCCESS) {
        delete f;
        return nullptr;
    }
    int dims[2] = {N0, N1};
    if (hipfftSetAutoAllocation(f->plan, 0) != HIPFFT_SUCCESS ||
        hipfftMakePlanMany(f->plan, 2, dims, nullptr, 1, 0, nullptr, 1, 0, HIPFFT_D2Z, batch, &f->work) != HIPFFT_SUCCESS) {
        (void)hipfftDestroy(f->plan);
        delete f;
        return nullptr;
    }
    *slot = f;
    return f;
}

}  // namespace

void spectra_release(dnsg_ctx *h) {
    for (void *&p : h->fft) {
        if (!p) continue;
        (void)hipfftDestroy(static_cast<FftPlan *>(p)->plan);
        delete static_cast<FftPlan *>(p);
        p = nullptr;
    }
}

}  // namespace dnsg

using namespace dnsg;

#define SPCHK(h, expr)                                                                      \
    do {                                                                                    \
        hipError_t e_ = (expr);                                                             \
        if (e_ != hipSuccess) {                                                             \
            (h)->err = std::string(#expr) + ": " + hipGetErrorString(e_);                   \
            rc = e_ == hipErrorOutOfMemory ? DNSG_ERR_OOM : DNSG_ERR_HIP;                   \
            goto done;                                                                      \
        }                                                                                   \
    } while (0)

extern "C" int dnsg_spectra(dnsg_t *h, int grid, double *ex, double *ey) {
    if (!h || !h->stream || grid < 0 || grid > 2 || !ex || !ey) return DNSG_ERR_ARG;
    if (!h->have_state) {
        h->err = "no state: call dnsg_init_state or dnsg_upload_state first";
        return DNSG_ERR_STATE;
    }
    const Grid &g = grid == 0 ? h->coarse : (grid == 1 ? h->lower : h->upper);
    const int N0 = g.nx, N1 = g.ny, N1h = N1 / 2 + 1;
    const int nzg = grid == 0 ? h->d.zdc : h->d.zdf;  // planes in the velocity file
    const int k0 = grid == 1 ? 1 : 0;                 // lower band: the wall is plane 0
    const size_t plane = (size_t)N0 * N1;
    int rc = grid == 0 ? DNSG_OK : ensure_fwall(h);  // the coarse grid has no wall layer
    if (rc) return rc;
    double *vel = nullptr, *dex = nullptr, *dey = nullptr;
    double2 *cf = nullptr;
    void *work = nullptr;
    FftPlan *plan = nullptr;
    SPCHK(h, scratch_get(&vel, 3 * (size_t)nzg * plane * sizeof(double)));
    SPCHK(h, scratch_get(&cf, 3 * (size_t)nzg * N0 * N1h * sizeof(double2)));
    SPCHK(h, scratch_get(&dex, 3 * (size_t)N0 * nzg * sizeof(double)));
    SPCHK(h, scratch_get(&dey, 3 * (size_t)N1h * nzg * sizeof(double)));
    {
        const int kwall = grid == 0 ? -1 : (grid == 1 ? 0 : nzg - 1);
        const double *wall = grid == 2 ? h->fwall + plane * Q : h->fwall;  // not read where kwall < 0
        const dim3 grd((unsigned)(((N0 + TS - 1) / TS) * ((N1 + TS - 1) / TS) * nzg)), blk(TB);
        if (h->p.precision == DNSG_PREC_FP64)
            hipLaunchKernelGGL(k_vel_planes<double>, grd, blk, 0, h->stream, (const double *)g.c(), wall, N0, N1, k0, kwall, nzg, vel);
        else if (h->p.precision == DNSG_PREC_FP32)
            hipLaunchKernelGGL(k_vel_planes<float>, grd, blk, 0, h->stream, (const float *)g.c(), wall, N0, N1, k0, kwall, nzg, vel);
        else
            hipLaunchKernelGGL(k_vel_planes<__half>, grd, blk, 0, h->stream, (const __half *)g.c(), wall, N0, N1, k0, kwall, nzg, vel);
        SPCHK(h, hipGetLastError());
    }
    {
        plan = fft_plan(&h->fft[grid == 0 ? 0 : 1], N0, N1, 3 * nzg);
        if (!plan) {  // its tables found no memory
            scratch_trim();
            plan = fft_plan(&h->fft[grid == 0 ? 0 : 1], N0, N1, 3 * nzg);
        }
        if (!plan) {
            h->err = "hipfftMakePlanMany failed";
            rc = DNSG_ERR_HIP;
            goto done;
        }
        if (plan->work) SPCHK(h, scratch_get(&work, plan->work));
        if (hipfftSetStream(plan->plan, h->stream) != HIPFFT_SUCCESS ||
            (work && hipfftSetWorkArea(plan->plan, work) != HIPFFT_SUCCESS) ||
            hipfftExecD2Z(plan->plan, vel, reinterpret_cast<hipfftDoubleComplex *>(cf)) != HIPFFT_SUCCESS) {
            h->err = "hipfftExecD2Z failed";
            rc = DNSG_ERR_HIP;
            goto done;
        }
    }
    {
        hipLaunchKernelGGL(k_fold_x, dim3((unsigned)((3L * nzg * N0 + TB / 64 - 1) / (TB / 64))), dim3(TB), 0, h->stream,
                           (const double2 *)cf, N0, N1, nzg, dex);
        hipLaunchKernelGGL(k_fold_y, dim3((unsigned)(3 * nzg * ((N1h + 63) / 64))), dim3(TB), 0, h->stream,
                           (const double2 *)cf, N0, N1, nzg, dey);
        SPCHK(h, hipGetLastError());
    }
    SPCHK(h, hipMemcpyAsync(ex, dex, 3 * (size_t)N0 * nzg * sizeof(double), hipMemcpyDeviceToHost, h->stream));
    SPCHK(h, hipMemcpyAsync(ey, dey, 3 * (size_t)N1h * nzg * sizeof(double), hipMemcpyDeviceToHost, h->stream));
    SPCHK(h, hipStreamSynchronize(h->stream));
done:
    (void)scratch_put(h->stream, {work, vel, cf, dex, dey});
    return rc;
}
