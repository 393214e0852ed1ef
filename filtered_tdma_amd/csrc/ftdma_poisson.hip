// Channel pressure Poisson solve on one GPU: the reference's
// PressureSolver::solve (apps/channel_cpu/PressureSolver.cpp:493-533) with
// its pencil transposes gone. The field stays in HBM as [z][y][x]; one
// batched 2-D real-to-complex FFT of every z plane (hipFFT) leaves the
// spectra as [z][ky][kx] complex, which is already the row-major
// [n_row = nz x n_sys = ny * (nx/2+1)] layout of the complex tridiagonal
// solve (mode s = kx + (nx/2+1) * ky, the reference's system order), so
// the wall-normal solve runs on it in place (ftd_solve_complex), and the
// inverse FFT and the projection follow.
//
//   divergence   compute_rhs_ (:193-212)
//   FFT x, y     plan_fwd_x_, plan_fwd_y_ (:110-135) as one 2-D D2Z
//   z solve      solve_tdma_z_ (:400-464): a, c from the z metrics, the
//                modified wavenumbers of :72-78, the (0, 0) mode pinned. With
//                one caller partition k_mode_solve forms the coefficients as
//                it solves (a, c of a row are the same for every mode), and the
//                spectra's lines start on 128-byte boundaries
//   inverse FFT  plan_bwd_y_, plan_bwd_x_ as one 2-D Z2D, scale 1/(nx ny)
//   projection   project_ (:470-490) with dp's ghosts (Neumann in z,
//                periodic in x and y, :512-526) read by index
#include <hip/hip_runtime.h>
#include <hipfft/hipfft.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <string>
#include <vector>

#include "../../include/ftdma.h"
#include "ftdma_device.h"
#include "ftdma_fft.h"
#include "ftdma_kernels.h"
#include "ftdma_xcd.h"

struct ftd_poisson {
    int nx = 0, ny = 0, nz = 0, nxh = 0, nm = 0;
    int pitch = 0;  // modes from one line of the spectra to the next (0: no k_mode_solve)
    hipStream_t stream = nullptr;  // the caller's
    // plans of lines of nxh modes back to back (ftd_solve_complex's layout) and
    // of lines of `pitch` modes where that is another layout
    ftd::FftPair fft[2];
    double* A = nullptr;    // [nz][nm] coefficients, built once
    double* B = nullptr;
    double* C = nullptr;
    double* rhs = nullptr;  // [nz][ny][nx]: divergence, then dp (unscaled)
    double* coef = nullptr; // k_mode_solve: a, c, -(a + c) per row, kx2, ky2
    double* hat = nullptr;  // [nz][ny][nxh or pitch] complex, interleaved (re, im)
    double* met = nullptr;  // dx, dmx [nx+2]; dy, dmy [ny+2]; dz, dmz [nz+2]
    ftd_handle* solver = nullptr;
    double scale = 1.0;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    int profiling = 0;  // time each step (waits for it)
    double last_ms = 0.0;
};

namespace {

thread_local std::string g_perr;

ftd_status perr(ftd_status s, const std::string& m) {
    g_perr = m;
    return s;
}

#define PH(call)                                                                              \
    do {                                                                                      \
        hipError_t e_ = (call);                                                               \
        if (e_ != hipSuccess) return perr(FTD_ERR_HIP, std::string(#call ": ") + hipGetErrorString(e_)); \
    } while (0)
#define PF(call)                                                                              \
    do {                                                                                      \
        hipfftResult r_ = (call);                                                             \
        if (r_ != HIPFFT_SUCCESS) return perr(FTD_ERR_HIP, std::string(#call ": hipFFT error ") + std::to_string((int)r_)); \
    } while (0)

// One axis of Grid::build_axis (Grid.cpp:47-95) on the whole domain:
// dx[i] = face spacing, dmx[i] = centre spacing, i = 0..n+1, mirrored
// ghosts at walls, wrapped ones when periodic.
void axis_metrics(int n, int uniform, double gamma, double L, bool periodic, double* dx,
                  double* dmx) {
    std::vector<double> xf(n + 1), xc(n + 2);
    if (uniform == 1 || std::fabs(gamma) < 1.0e-14) {
        for (int i = 0; i <= n; ++i) xf[i] = L * static_cast<double>(i) / static_cast<double>(n);
    } else {
        const double th = std::tanh(gamma);
        for (int i = 0; i <= n; ++i) {
            const double zeta = static_cast<double>(i) / static_cast<double>(n);
            xf[i] = 0.5 * L * (1.0 - std::tanh(gamma * (1.0 - 2.0 * zeta)) / th);
        }
    }
    for (int i = 1; i <= n; ++i) xc[i] = 0.5 * (xf[i - 1] + xf[i]);
    if (periodic) {
        xc[0] = xc[n] - L;
        xc[n + 1] = xc[1] + L;
    } else {
        xc[0] = xf[0] - (xc[1] - xf[0]);
        xc[n + 1] = xf[n] + (xf[n] - xc[n]);
    }
    for (int i = 1; i <= n; ++i) dx[i] = xf[i] - xf[i - 1];
    dx[0] = periodic ? dx[n] : dx[1];
    dx[n + 1] = periodic ? dx[1] : dx[n];
    for (int i = 1; i <= n + 1; ++i) dmx[i] = xc[i] - xc[i - 1];
    dmx[0] = periodic ? dmx[n] : dmx[1];
}

struct Dims3 {
    int nx, ny, nz;
};

__device__ inline size_t fidx(const Dims3& g, int i, int j, int k) {
    return (size_t)i + (size_t)(g.nx + 2) * ((size_t)j + (size_t)(g.ny + 2) * (size_t)k);
}

// (1/dt) div u* of every interior cell into rhs [z][y][x]
__global__ void k_divergence(const double* __restrict__ U, const double* __restrict__ V,
                             const double* __restrict__ W, double* __restrict__ rhs, Dims3 g,
                             const double* __restrict__ dx, const double* __restrict__ dy,
                             const double* __restrict__ dz, double inv_dt) {
    // one wave per 64 cells of a line; lines in (x, y, z) order dealt to the
    // XCDs in contiguous runs, so V's row j + 1 is the next line's own row,
    // read on the same XCD
    const int nbx = (g.nx + 63) / 64;
    const int T = ftd::xcd_tile(blockIdx.x, gridDim.x);
    const int i = (T % nbx) * 64 + threadIdx.x + 1;
    const int j = (T / nbx) % g.ny + 1, k = T / (nbx * g.ny) + 1;
    if (i > g.nx) return;
    const size_t c = fidx(g, i, j, k);
    const double d = (U[c + 1] - U[c]) / dx[i] + (V[c + (g.nx + 2)] - V[c]) / dy[j] +
                     (W[c + (size_t)(g.nx + 2) * (g.ny + 2)] - W[c]) / dz[k];
    rhs[((size_t)(k - 1) * g.ny + (j - 1)) * g.nx + (i - 1)] = d * inv_dt;
}

// the (0, 0) mode's wall row: A = C = 0, B = 1 (built in), right-hand side 0
__global__ void k_pin_zero_mode(double* hat) {
    if (threadIdx.x < 2) hat[threadIdx.x] = 0.0;
}

// P += dp; u -= dt grad dp on the faces (project_), dp = 0 + raw * scale as
// the reference's accumulation into a zeroed field gives it
__global__ void k_project(double* __restrict__ U, double* __restrict__ V, double* __restrict__ W,
                          double* __restrict__ P, const double* __restrict__ raw, Dims3 g,
                          double scale, double dt, const double* __restrict__ dmx,
                          const double* __restrict__ dmy, const double* __restrict__ dmz) {
    // tile order as in k_divergence: dp's row j - 1 was the previous line's
    const int nbx = (g.nx + 63) / 64;
    const int T = ftd::xcd_tile(blockIdx.x, gridDim.x);
    const int i = (T % nbx) * 64 + threadIdx.x + 1;
    const int j = (T / nbx) % g.ny + 1, k = T / (nbx * g.ny) + 1;
    if (i > g.nx) return;
    auto dp = [&](int ii, int jj, int kk) {
        return 0.0 + raw[((size_t)(kk - 1) * g.ny + (jj - 1)) * g.nx + (ii - 1)] * scale;
    };
    const double p = dp(i, j, k);
    const double pw = dp(i > 1 ? i - 1 : g.nx, j, k);  // periodic ghost in x
    const double ps = dp(i, j > 1 ? j - 1 : g.ny, k);  // periodic ghost in y
    const double pb = dp(i, j, k > 1 ? k - 1 : 1);     // Neumann ghost at the lower wall
    const size_t c = fidx(g, i, j, k);
    P[c] += p;
    U[c] -= dt * (p - pw) / dmx[i];
    V[c] -= dt * (p - ps) / dmy[j];
    W[c] -= dt * (p - pb) / dmz[k];
}

__global__ void k_unpack_dp(const double* __restrict__ raw, double* __restrict__ dp, int n,
                            double scale) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) dp[t] = 0.0 + raw[t] * scale;
}

// ---------------------------------------------------------------------------
// The wall-normal solves of every mode, coefficients formed in the kernel:
// row k of mode (i, j) is a_k, b = -(a_k + c_k) - (kx2_i + ky2_j), c_k, the
// (0, 0) mode's wall row pinned (a = c = 0, b = 1, right-hand side 0): the values
// of the arrays that ftd_solve_complex reads, by the same expressions.
//
// PaScaL over ceil(nz / 16) partitions of up to 16 rows, one lane per (mode,
// partition): a', c' once for both parts of the right-hand side, which come in
// and go out 16 bytes per lane. A mode costs 32 B per row where the solve on
// arrays reads A, B, C as well (56), and half the divisions: 34816 modes of 256
// rows (286 MB) in 58 us, 4.9 TB/s, where that solve took 125 and the pin's
// launch 5 more.
//
// Bound by the loads in flight: all rows of a lane are requested at once, and
// three waves per SIMD pay for 80 B of spills (67 us with two and none).
// Workgroups of 256 lanes, three to a CU, so that one solves its 2Q-row system
// while the others load: 86 us with 512, 64 with 128; partitions of 8 rows 85,
// of 32 (one wave per SIMD) 80.
// ---------------------------------------------------------------------------
constexpr int kModeRows = 16;
constexpr int kModeThreads = 256;
typedef double mode_dbl2 __attribute__((ext_vector_type(2)));

// the modes' shape: Q partitions, S modes per workgroup (0: nz is outside what
// the kernel holds, up to 512 rows, and the solve on arrays takes them; below 17
// rows one partition is left)
void mode_shape(int nz, int& Q, int& S) {
    Q = (nz + kModeRows - 1) / kModeRows;
    S = 0;
    if (Q < 2 || Q > 32 || nz / Q < 3) return;
    S = 64;
    while (S * Q > kModeThreads) S >>= 1;
}

size_t mode_lds(int nz, int Q, int S) {
    return sizeof(double) * ((size_t)8 * Q * S + 3 * (size_t)nz);
}

__global__ __launch_bounds__(kModeThreads, 3) void k_mode_solve(double* __restrict__ hat, int nxh,
                                                             int pitch, int ny, int nz, int Q,
                                                             int lgS,
                                                             const double* __restrict__ coef) {
    constexpr int M = kModeRows;
    extern __shared__ double lds[];
    const int S = 1 << lgS;
    const int t = threadIdx.x;
    const int sl = t & (S - 1);
    const int q = t >> lgS;
    const int n = ny * pitch;
    const int s_raw = ftd::xcd_tile(blockIdx.x, gridDim.x) * S + sl;
    const int s = s_raw < n ? s_raw : n - 1;
    const int jy = s / pitch, ix = s - jy * pitch;
    const bool live = s_raw < n && ix < nxh;
    int r0, cnt;
    ftd::part_of(nz, Q, q, r0, cnt);
    // a, c, -(a + c) of every row to LDS
    double* const ta = lds + 8 * Q * S;
    for (int k = t; k < 3 * nz; k += S * Q) ta[k] = coef[k];
    const double* const tc = ta + nz;
    const double* const tb = tc + nz;
    // (modes in the padding have no wavenumber: the last one's)
    const double lam = coef[3 * nz + (ix < nxh ? ix : nxh - 1)] + coef[3 * nz + nxh + jy];
    const bool pin = s == 0 && q == 0;

    mode_dbl2* const z = (mode_dbl2*)hat + (size_t)r0 * n + s;
    mode_dbl2 d[M];
#pragma unroll
    for (int j = 0; j < M; ++j) d[j] = z[(size_t)(j < cnt ? j : cnt - 1) * n];
    __syncthreads();
    double a[M], c[M];
    double aN = 0.0, cN = 0.0;
    mode_dbl2 dN = {0.0, 0.0};
#pragma unroll
    for (int j = 0; j < M; ++j) {
        if (j < cnt) {
            double aj = ta[r0 + j], cj = tc[r0 + j], bj = tb[r0 + j] - lam;
            if (j == 0) {
                aj = pin ? 0.0 : aj;
                cj = pin ? 0.0 : cj;
                bj = pin ? 1.0 : bj;
                d[0].x = pin ? 0.0 : d[0].x;
                d[0].y = pin ? 0.0 : d[0].y;
            }
            if (j < 2) {
                a[j] = aj / bj;
                c[j] = cj / bj;
                d[j].x = d[j].x / bj;
                d[j].y = d[j].y / bj;
            } else {
                const double inv = 1.0 / (bj - aj * c[j - 1]);
                d[j].x = inv * (d[j].x - aj * d[j - 1].x);
                d[j].y = inv * (d[j].y - aj * d[j - 1].y);
                c[j] = inv * cj;
                a[j] = -inv * aj * a[j - 1];
            }
            if (j == cnt - 1) {
                aN = a[j];
                cN = c[j];
                dN = d[j];
            }
        }
    }
#pragma unroll
    for (int j = M - 3; j >= 1; --j) {
        if (j <= cnt - 3) {
            const double cj = c[j];
            d[j].x = d[j].x - cj * d[j + 1].x;
            d[j].y = d[j].y - cj * d[j + 1].y;
            a[j] = a[j] - cj * a[j + 1];
            c[j] = -cj * c[j + 1];
        }
    }
    const double r = 1.0 / (1.0 - a[1] * c[0]);
    const int NR = 2 * Q;
    double* const rA = lds;
    double* const rC = rA + NR * S;
    double* const rX = rC + NR * S;
    double* const rY = rX + NR * S;
    const int o0 = 2 * q * S + sl, oN = o0 + S;
    rA[o0] = r * a[0];
    rC[o0] = -r * c[0] * c[1];
    rX[o0] = r * (d[0].x - c[0] * d[1].x);
    rY[o0] = r * (d[0].y - c[0] * d[1].y);
    rA[oN] = aN;
    rC[oN] = cN;
    rX[oN] = dN.x;
    rY[oN] = dN.y;
    __syncthreads();
    if (q == 0) {
        // Thomas on the 2Q rows (b == 1) of both parts, 4 rows read at a time
        double cp = rC[sl], xp = rX[sl], yp = rY[sl];
        int k = 1;
        for (; k + 4 <= NR; k += 4) {
            double ak[4], ck[4], xk[4], yk[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int o = (k + u) * S + sl;
                ak[u] = rA[o];
                ck[u] = rC[o];
                xk[u] = rX[o];
                yk[u] = rY[o];
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int o = (k + u) * S + sl;
                const double inv = 1.0 / (1.0 - ak[u] * cp);
                xp = inv * (xk[u] - ak[u] * xp);
                yp = inv * (yk[u] - ak[u] * yp);
                cp = inv * ck[u];
                rX[o] = xp;
                rY[o] = yp;
                rC[o] = cp;
            }
        }
        for (; k < NR; ++k) {
            const int o = k * S + sl;
            const double ak = rA[o];
            const double inv = 1.0 / (1.0 - ak * cp);
            xp = inv * (rX[o] - ak * xp);
            yp = inv * (rY[o] - ak * yp);
            cp = inv * rC[o];
            rX[o] = xp;
            rY[o] = yp;
            rC[o] = cp;
        }
        for (k = NR - 2; k >= 0; --k) {
            const int o = k * S + sl;
            const double ck = rC[o];
            xp = rX[o] - ck * xp;
            yp = rY[o] - ck * yp;
            rX[o] = xp;
            rY[o] = yp;
        }
    }
    __syncthreads();
    const double x0 = rX[o0], y0 = rY[o0], xN = rX[oN], yN = rY[oN];
    if (live) {
#pragma unroll
        for (int j = 0; j < M; ++j) {
            if (j < cnt) {
                mode_dbl2 x;
                x.x = j == 0 ? x0 : j == cnt - 1 ? xN : d[j].x - (a[j] * x0 + c[j] * xN);
                x.y = j == 0 ? y0 : j == cnt - 1 ? yN : d[j].y - (a[j] * y0 + c[j] * yN);
                z[(size_t)j * n] = x;
            }
        }
    }
}

// the FFT plans of layout k: lines of nxh modes (0) or of p->pitch (1). A pair
// takes about 13 ms to make: create makes the one that the step uses,
// ftd_poisson_solver the other, since a solver has to be asked for to be tuned
ftd_status fft_plans(ftd_poisson* p, int k) {
    const char* failed =
        ftd::fft_make(p->fft[k], p->nx, p->ny, p->nz, k ? p->pitch : p->nxh, p->stream);
    return failed ? perr(FTD_ERR_HIP, failed) : FTD_OK;
}

ftd_status poisson_spectral(ftd_poisson* p) {
    // the solver as it was made solves in k_mode_solve; one that the caller
    // tuned or moved to another stream solves by itself
    if (p->pitch && ftd::handle_is_plain(p->solver, p->stream)) {
        int Q, S;
        mode_shape(p->nz, Q, S);
        const int k = p->pitch != p->nxh;
        PF(hipfftExecD2Z(p->fft[k].fwd, p->rhs, reinterpret_cast<hipfftDoubleComplex*>(p->hat)));
        int lgS = 0;
        while ((1 << lgS) < S) ++lgS;
        const int n = p->ny * p->pitch;
        char path[96];
        std::snprintf(path, sizeof path, "pascal_modes M=%d T=%d S=%d Q=%d", kModeRows,
                      kModeThreads, S, Q);
        ftd::handle_note_path(p->solver, path);
        PH(ftd::handle_time_begin(p->solver));
        hipLaunchKernelGGL(k_mode_solve, dim3((n + S - 1) / S), dim3(S * Q), mode_lds(p->nz, Q, S),
                           p->stream, p->hat, p->nxh, p->pitch, p->ny, p->nz, Q, lgS, p->coef);
        PH(hipGetLastError());
        PH(ftd::handle_time_end(p->solver));
        PF(hipfftExecZ2D(p->fft[k].bwd, reinterpret_cast<hipfftDoubleComplex*>(p->hat), p->rhs));
        return FTD_OK;
    }
    ftd_status s = fft_plans(p, 0);
    if (s != FTD_OK) return s;
    PF(hipfftExecD2Z(p->fft[0].fwd, p->rhs, reinterpret_cast<hipfftDoubleComplex*>(p->hat)));
    hipLaunchKernelGGL(k_pin_zero_mode, dim3(1), dim3(64), 0, p->stream, p->hat);
    PH(hipGetLastError());
    s = ftd_solve_complex(p->solver, p->A, p->B, p->C, p->hat);
    if (s != FTD_OK) return perr(s, std::string("z solve: ") + ftd_last_error_string());
    PF(hipfftExecZ2D(p->fft[0].bwd, reinterpret_cast<hipfftDoubleComplex*>(p->hat), p->rhs));
    return FTD_OK;
}

}  // namespace

extern "C" {

ftd_status ftd_poisson_create(ftd_poisson** out, int nx, int ny, int nz, double Lx, double Ly,
                              double Lz, double gamma_z, int kind, int partitions,
                              double eps_constant, void* stream) {
    if (!out) return perr(FTD_ERR_INVALID, "null output pointer");
    *out = nullptr;
    if (nx < 2 || ny < 1 || nz < 3 || (nx & 1))
        return perr(FTD_ERR_INVALID, "need even nx >= 2, ny >= 1, nz >= 3");
    if (!(Lx > 0.0) || !(Ly > 0.0) || !(Lz > 0.0)) return perr(FTD_ERR_INVALID, "lengths must be > 0");
    const size_t cells = (size_t)nx * ny * nz;
    if (cells >= ((size_t)1 << 31)) return perr(FTD_ERR_INVALID, "grid too large");
    ftd_poisson* p = new ftd_poisson();
    p->nx = nx;
    p->ny = ny;
    p->nz = nz;
    p->nxh = nx / 2 + 1;
    p->nm = p->nxh * ny;
    p->scale = 1.0 / (static_cast<double>(nx) * ny);
    auto bail = [&](ftd_status s) {
        ftd_poisson_destroy(p);
        return s;
    };
    // NULL is the null stream, as for ftd_create: ordered with the caller's
    // work there (torch's default stream among it)
    hipError_t e = hipSuccess;
    p->stream = (hipStream_t)stream;
    // metrics: x and y uniform periodic, z tanh-stretched walls
    std::vector<double> met(2 * (nx + 2) + 2 * (ny + 2) + 2 * (nz + 2));
    double* dx = met.data();
    double* dmx = dx + (nx + 2);
    double* dy = dmx + (nx + 2);
    double* dmy = dy + (ny + 2);
    double* dz = dmy + (ny + 2);
    double* dmz = dz + (nz + 2);
    axis_metrics(nx, 1, 0.0, Lx, true, dx, dmx);
    axis_metrics(ny, 1, 0.0, Ly, true, dy, dmy);
    axis_metrics(nz, 0, gamma_z, Lz, false, dz, dmz);
    // coefficients (solve_tdma_z_), modified wavenumbers (:72-78)
    const int nxh = p->nxh, nm = p->nm;
    std::vector<double> kx2(nxh), ky2(ny);
    const double hx = Lx / nx, hy = Ly / ny;
    for (int i = 0; i < nxh; ++i) kx2[i] = 2.0 * (1.0 - std::cos(2.0 * M_PI * i / nx)) / (hx * hx);
    for (int j = 0; j < ny; ++j) {
        const int jj = (j <= ny / 2) ? j : j - ny;
        ky2[j] = 2.0 * (1.0 - std::cos(2.0 * M_PI * jj / ny)) / (hy * hy);
    }
    std::vector<double> hA((size_t)nz * nm), hB((size_t)nz * nm), hC((size_t)nz * nm);
    for (int k = 0; k < nz; ++k) {
        const double a = k == 0 ? 0.0 : 1.0 / (dz[k + 1] * dmz[k + 1]);
        const double c = k == nz - 1 ? 0.0 : 1.0 / (dz[k + 1] * dmz[k + 2]);
        for (int j = 0; j < ny; ++j)
            for (int i = 0; i < nxh; ++i) {
                const size_t idx = (size_t)k * nm + i + (size_t)nxh * j;
                hA[idx] = a;
                hC[idx] = c;
                hB[idx] = -(a + c) - (kx2[i] + ky2[j]);
            }
    }
    hA[0] = 0.0;
    hB[0] = 1.0;
    hC[0] = 0.0;
    // one caller partition: every kind solves exactly, over partitions of the
    // engine's choice. Lines of the spectra padded to whole 128-byte lines (the
    // FFTs of 256^3 in 96 + 94 us where lines of 129 modes took 134 + 137),
    // unless the padding would be more than a fifth of them
    int mq, ms;
    mode_shape(nz, mq, ms);
    const int padded = (nxh + 7) / 8 * 8;
    if (partitions == 1 && ms) p->pitch = 5 * padded <= 6 * nxh ? padded : nxh;
    std::vector<double> coef(3 * (size_t)nz + nxh + ny);
    for (int k = 0; k < nz; ++k) {
        const double a = k == 0 ? 0.0 : 1.0 / (dz[k + 1] * dmz[k + 1]);
        const double c = k == nz - 1 ? 0.0 : 1.0 / (dz[k + 1] * dmz[k + 2]);
        coef[k] = a;
        coef[nz + k] = c;
        coef[2 * (size_t)nz + k] = -(a + c);
    }
    for (int i = 0; i < nxh; ++i) coef[3 * (size_t)nz + i] = kx2[i];
    for (int j = 0; j < ny; ++j) coef[3 * (size_t)nz + nxh + j] = ky2[j];
    const size_t hb = 2 * sizeof(double) * (size_t)nz * ny * std::max(nxh, p->pitch);
    const size_t cb = sizeof(double) * (size_t)nz * nm;
    if (e == hipSuccess) e = hipMalloc(&p->A, cb);
    if (e == hipSuccess) e = hipMalloc(&p->B, cb);
    if (e == hipSuccess) e = hipMalloc(&p->C, cb);
    if (e == hipSuccess) e = hipMalloc(&p->rhs, sizeof(double) * cells);
    if (e == hipSuccess) e = hipMalloc(&p->hat, hb);
    if (e == hipSuccess) e = hipMemset(p->hat, 0, hb);  // (the padding is read)
    if (e == hipSuccess) e = hipMalloc(&p->coef, sizeof(double) * coef.size());
    if (e == hipSuccess)
        e = hipMemcpy(p->coef, coef.data(), sizeof(double) * coef.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMalloc(&p->met, sizeof(double) * met.size());
    if (e == hipSuccess) e = hipMemcpy(p->A, hA.data(), cb, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(p->B, hB.data(), cb, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(p->C, hC.data(), cb, hipMemcpyHostToDevice);
    if (e == hipSuccess)
        e = hipMemcpy(p->met, met.data(), sizeof(double) * met.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipEventCreate(&p->e0);
    if (e == hipSuccess) e = hipEventCreate(&p->e1);
    if (e != hipSuccess)
        return bail(perr(FTD_ERR_HIP, std::string("ftd_poisson_create: ") + hipGetErrorString(e)));
    ftd_status s = fft_plans(p, p->pitch > nxh);
    if (s != FTD_OK) return bail(s);
    s = ftd_create(&p->solver, kind, nm, nz, partitions, eps_constant, p->stream);
    if (s != FTD_OK) return bail(perr(s, std::string("z solver: ") + ftd_last_error_string()));
    *out = p;
    return FTD_OK;
}

ftd_status ftd_poisson_destroy(ftd_poisson* p) {
    if (!p) return FTD_OK;
    for (ftd::FftPair& f : p->fft) ftd::fft_free(f);
    if (p->solver) ftd_destroy(p->solver);
    for (double* b : {p->A, p->B, p->C, p->rhs, p->hat, p->met, p->coef})
        if (b) hipFree(b);
    if (p->e0) hipEventDestroy(p->e0);
    if (p->e1) hipEventDestroy(p->e1);
    delete p;
    return FTD_OK;
}

ftd_handle* ftd_poisson_solver(ftd_poisson* p) {
    if (!p) return nullptr;
    (void)fft_plans(p, 0);  // (if they cannot be made, the step that needs them says so)
    return p->solver;
}

const char* ftd_poisson_last_path(const ftd_poisson* p) {
    return p ? ftd_last_path(p->solver) : "none";
}

ftd_status ftd_poisson_solve(ftd_poisson* p, double* U, double* V, double* W, double* P, double dt) {
    if (!p) return perr(FTD_ERR_INVALID, "null handle");
    if (!U || !V || !W || !P) return perr(FTD_ERR_INVALID, "null field pointer");
    if (!(dt > 0.0)) return perr(FTD_ERR_INVALID, "dt must be > 0");
    const Dims3 g{p->nx, p->ny, p->nz};
    const double* dx = p->met;
    const double* dmx = dx + (p->nx + 2);
    const double* dy = dmx + (p->nx + 2);
    const double* dmy = dy + (p->ny + 2);
    const double* dz = dmy + (p->ny + 2);
    const double* dmz = dz + (p->nz + 2);
    const dim3 block(64), grid(((p->nx + 63) / 64) * p->ny * p->nz);
    if (p->profiling) PH(hipEventRecord(p->e0, p->stream));
    hipLaunchKernelGGL(k_divergence, grid, block, 0, p->stream, U, V, W, p->rhs, g, dx, dy, dz,
                       1.0 / dt);
    PH(hipGetLastError());
    ftd_status s = poisson_spectral(p);
    if (s != FTD_OK) return s;
    hipLaunchKernelGGL(k_project, grid, block, 0, p->stream, U, V, W, P, p->rhs, g, p->scale, dt,
                       dmx, dmy, dmz);
    PH(hipGetLastError());
    if (p->profiling) {
        PH(hipEventRecord(p->e1, p->stream));
        PH(hipEventSynchronize(p->e1));
        float ms = 0.0f;
        PH(hipEventElapsedTime(&ms, p->e0, p->e1));
        p->last_ms = ms;
    }
    return FTD_OK;
}

ftd_status ftd_poisson_set_profiling(ftd_poisson* p, int enable) {
    if (!p) return perr(FTD_ERR_INVALID, "null handle");
    p->profiling = enable != 0;
    return FTD_OK;
}

ftd_status ftd_poisson_solve_rhs(ftd_poisson* p, const double* rhs, double* dp) {
    if (!p) return perr(FTD_ERR_INVALID, "null handle");
    if (!rhs || !dp) return perr(FTD_ERR_INVALID, "null array pointer");
    const size_t cells = (size_t)p->nx * p->ny * p->nz;
    PH(hipMemcpyAsync(p->rhs, rhs, sizeof(double) * cells, hipMemcpyDeviceToDevice, p->stream));
    ftd_status s = poisson_spectral(p);
    if (s != FTD_OK) return s;
    hipLaunchKernelGGL(k_unpack_dp, dim3((unsigned)((cells + 255) / 256)), dim3(256), 0, p->stream,
                       p->rhs, dp, (int)cells, p->scale);
    PH(hipGetLastError());
    PH(hipStreamSynchronize(p->stream));
    return FTD_OK;
}

double ftd_poisson_last_ms(const ftd_poisson* p) { return p ? p->last_ms : 0.0; }

const char* ftd_poisson_last_error_string(void) { return g_perr.c_str(); }

}  // extern "C"
