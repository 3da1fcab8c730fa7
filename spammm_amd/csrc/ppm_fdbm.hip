// ppm_fdbm.hip — FDBM force-field producer: FFT Pauli overlap, FFT Poisson / electrostatic
// convolution, London dispersion, energy composition and the central-difference force grid.
//
// Follows the reference's GPU FDBM stage 3 (spammm/SPM/AFM.py:3304-3566 _FDBMGpyFFT,
// :4204-4253 stage3_fdbm_fields_fast; kernels/AFM.cl:1151-1303 gradient_central_diff and the
// fdbm_* kernels, :1066-1113 evalDispersion_toImg with getLondon :804-814):
//   overlap(R) = dV * IFFT( FFT(rho) . conj(FFT(tip_tot)) )              (tip rolled to index 0)
//   E_pauli    = A * max(overlap, 1e-30)^beta
//   E_es       = dV * IFFT( FFT(rho_diff) . FFT(flip(tip_del)) . 4 pi C / k^2 ),  k = 0 -> 0
//   E_vdw      = - sum_a C6eff_a / (|r - r_a|^2 + RA^2)^3
//   F          = -(E[i+1] - E[i-1]) / (2 step) per axis, periodic; grid = (F, E)
// Scalar fields are (nx,ny,nz) C-order (z fastest), the reference's host layout; the force
// grid is written in the (nz,ny,nx,4) x-fastest layout the relaxation kernels read.
//
// FFTs are real-to-complex / complex-to-real hipFFT plans (FP32, as the reference's
// complex64), cached per shape and device; the half spectrum (nx, ny, nz/2+1) is combined in
// one pointwise kernel (k^2 from the index, no k-grid in memory).  Everything else but the dispersion
// is memory-bound elementwise / stencil work.
#include "ppm_common.hpp"
#include "ppm_rn.hpp"

#include <hipfft/hipfft.h>

#include <mutex>
#include <type_traits>
#include <vector>

namespace ppm {
namespace {

__device__ __forceinline__ int freq(int i, int n) { return i <= (n - 1) / 2 ? i : i - n; }

// a[i] <- a[i] op b[i] (x k-factor) x scale, over the half spectrum (nx, ny, nzh).
__global__ __launch_bounds__(256) void k_spectrum(float2* __restrict__ a, const float2* __restrict__ b, int mode,
                                                  int nx, int ny, int nz, int nzh, float kx0, float ky0, float kz0,
                                                  float scale) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    const long long n = (long long)nx * ny * nzh;
    if (i >= n) return;
    const int iz = (int)(i % nzh);
    const int iy = (int)((i / nzh) % ny);
    const int ix = (int)(i / ((long long)nzh * ny));
    float2 v = a[i];
    if (mode == PPM_FFT_CORRELATE || mode == PPM_FFT_CONVOLVE || mode == PPM_FFT_POISSON_CONVOLVE) {
        const float2 w = b[i];
        const float wy = mode == PPM_FFT_CORRELATE ? -w.y : w.y;
        v = make_float2(v.x * w.x - v.y * wy, v.x * wy + v.y * w.x);
    }
    if (mode == PPM_FFT_POISSON || mode == PPM_FFT_POISSON_CONVOLVE) {
        const float kx = kx0 * (float)freq(ix, nx), ky = ky0 * (float)freq(iy, ny), kz = kz0 * (float)iz;
        const float k2 = kx * kx + ky * ky + kz * kz;
        const float s = i == 0 ? 0.f : 1.0f / k2;   // k = 0 (neutralising background) -> 0
        v.x *= s;
        v.y *= s;
    }
    a[i] = make_float2(v.x * scale, v.y * scale);
}

__global__ __launch_bounds__(256) void k_pauli_scale(float* __restrict__ f, long long n, float A, float beta,
                                                     float clip) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float o = fmaxf(f[i], clip);
    f[i] = A * powf(o, beta);
}

// dst[i] = padded[(i + r) mod n]; padded = zeros except the source block at (ox, oy, oz).
__global__ __launch_bounds__(256) void k_pad_roll(const float* __restrict__ src, int sx, int sy, int sz,
                                                  float* __restrict__ dst, int nx, int ny, int nz, int ox, int oy,
                                                  int oz, int rx, int ry, int rz) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= (long long)nx * ny * nz) return;
    const int iz = (int)(i % nz), iy = (int)((i / nz) % ny), ix = (int)(i / ((long long)nz * ny));
    const int jx = ((ix + rx) % nx + nx) % nx, jy = ((iy + ry) % ny + ny) % ny, jz = ((iz + rz) % nz + nz) % nz;
    const int lx = jx - ox, ly = jy - oy, lz = jz - oz;
    float v = 0.f;
    if (lx >= 0 && lx < sx && ly >= 0 && ly < sy && lz >= 0 && lz < sz) v = src[((size_t)lx * sy + ly) * sz + lz];
    dst[i] = v;
}

// dst[ix,iy,iz] = src[nx-1-ix, ny-1-iy, nz-1-iz]
__global__ __launch_bounds__(256) void k_flip3(const float* __restrict__ src, float* __restrict__ dst, int nx, int ny,
                                               int nz) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    const long long n = (long long)nx * ny * nz;
    if (i >= n) return;
    dst[i] = src[n - 1 - i];
}

// out[ix,iy,iz] (+)= - sum_a C6eff_a / (|p - r_a|^2 + RA^2)^3,  p = origin + step*(ix,iy,iz).
// VALU bound.  A thread takes V voxels along x, which share dy^2 + dz^2 + RA^2 and the atom's LDS read; the
// reciprocals are rcp_rn (the correctly rounded one in 3 instructions instead of 11), and a thread that met a
// denominator outside 2^+-100 sums its voxels again with the IEEE quotient.  200 x 160 x 128 voxels, 38 atoms:
// 83 -> 46 us.
template <int V>
__global__ __launch_bounds__(256) void k_dispersion(const float4* __restrict__ atoms, int na, float ox, float oy,
                                                    float oz, float step, int nx, int ny, int nz, float ra2,
                                                    int accumulate, float* __restrict__ out) {
    __shared__ float4 sa[256];
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    const long long n = (long long)((nx + V - 1) / V) * ny * nz;
    const long long ic = i < n ? i : n - 1;
    const int iz = (int)(ic % nz), iy = (int)((ic / nz) % ny), ix = (int)(ic / ((long long)nz * ny)) * V;
    const float py = oy + step * (float)iy, pz = oz + step * (float)iz;
    float px[V], e[V];
#pragma unroll
    for (int k = 0; k < V; ++k) px[k] = ox + step * (float)(ix + k);
    unsigned lo = ~0u, hi = 0u;
    auto sum = [&](auto mid) {
#pragma unroll
        for (int k = 0; k < V; ++k) e[k] = 0.f;
        for (int t0 = 0; t0 < na; t0 += 256) {
            __syncthreads();
            if (t0 + (int)threadIdx.x < na) sa[threadIdx.x] = atoms[t0 + threadIdx.x];
            __syncthreads();
            const int cnt = min(256, na - t0);
            for (int j = 0; j < cnt; ++j) {
                const float4 a = sa[j];
                const float dy = py - a.y, dz = pz - a.z, s = fmaf(dy, dy, fmaf(dz, dz, ra2));
#pragma unroll
                for (int k = 0; k < V; ++k) {
                    const float dx = px[k] - a.x, r2 = fmaf(dx, dx, s);
                    float ir2;
                    if constexpr (decltype(mid)::value) {
                        ir2 = rcp_rn(r2);
                        lo = min(lo, __float_as_uint(r2));
                        hi = max(hi, __float_as_uint(r2));
                    } else {
                        ir2 = 1.0f / r2;
                    }
                    e[k] = fmaf(-a.w, ir2 * ir2 * ir2, e[k]);
                }
            }
        }
    };
    sum(std::true_type{});
    if (__syncthreads_or(na > 0 && (lo < 0x0d800000u || hi > 0x71800000u))) sum(std::false_type{});   // 2^-100, 2^100
    if (i >= n) return;
#pragma unroll
    for (int k = 0; k < V; ++k)
        if (ix + k < nx) {
            const size_t o = ((size_t)(ix + k) * ny + iy) * nz + iz;
            out[o] = accumulate ? out[o] + e[k] : e[k];
        }
}

// F = -(E[+1] - E[-1]) / (2 step) per axis with periodic neighbours, E = e1 + e2 + e3 (any may be
// NULL); written as float4 (Fx,Fy,Fz,E) in the (nz,ny,nx,4) layout.
// Bound by its loads and stores.  The fields are z fastest and the grid x fastest: a workgroup takes a tile of 16 x 16
// (x, z) of one y in field order, keeps E of the tile and its four edges in LDS (10 loads a voxel instead of 21), and
// turns its result there, so that stores are runs of 256 bytes along x instead of 16 bytes at a plane's stride.
// Workgroups go to the XCDs in turn, so each XCD is given a contiguous share of the tiles (z, then x, then y) and
// finds its neighbours in y in its own L2.  80^3 | 200 x 160 x 128 voxels: 13.4 | 60 -> 7.8 | 40 us (without the
// XCDs' shares and E in LDS 9.6 | 61; tiles of 32 x 32 with their halo in LDS, several y at once: 20..26 | 46..65).
constexpr int kT = 16, kXcds = 8;

__global__ __launch_bounds__(kT * kT) void k_compose_gradient(const float* __restrict__ e1, const float* __restrict__ e2,
                                                              const float* __restrict__ e3, int nx, int ny, int nz,
                                                              float step, float4* __restrict__ grid) {
    __shared__ float S[kT + 2][kT + 3];
    __shared__ float4 tile[kT][kT + 1];
    const int bz = (nz + kT - 1) / kT, bx = (nx + kT - 1) / kT;
    const long long share = gridDim.x / kXcds, b = (long long)(blockIdx.x % kXcds) * share + blockIdx.x / kXcds;
    if (b >= (long long)bz * bx * ny) return;
    const int z0 = (int)(b % bz) * kT, x0 = (int)(b / bz % bx) * kT, iy = (int)(b / ((long long)bz * bx));
    auto E = [&](int x, int y, int z) {
        const size_t k = ((size_t)x * ny + y) * nz + z;
        float s = 0.f;
        if (e1) s += e1[k];
        if (e2) s += e2[k];
        if (e3) s += e3[k];
        return s;
    };
    const int tz = threadIdx.x % kT, tx = threadIdx.x / kT;
    const int ix = min(x0 + tx, nx - 1), iz = min(z0 + tz, nz - 1);         // clamped: stored nowhere
    const float e = E(ix, iy, iz);
    S[tx + 1][tz + 1] = e;
    int sx = -1, sz = 0;
    float edge = 0.f;
    if (threadIdx.x < 4 * kT) {             // the edges: x below, x above, z below, z above the tile
        const int side = threadIdx.x / kT, j = threadIdx.x % kT;
        const int xe = min(x0 + kT, nx), ze = min(z0 + kT, nz);
        const int x = side == 0 ? (x0 == 0 ? nx - 1 : x0 - 1) : side == 1 ? (xe == nx ? 0 : xe) : min(x0 + j, nx - 1);
        const int z = side == 2 ? (z0 == 0 ? nz - 1 : z0 - 1) : side == 3 ? (ze == nz ? 0 : ze) : min(z0 + j, nz - 1);
        sx = side == 0 ? 0 : side == 1 ? xe - x0 + 1 : j + 1;
        sz = side == 2 ? 0 : side == 3 ? ze - z0 + 1 : j + 1;
        edge = E(x, iy, z);
    }
    __syncthreads();
    if (sx >= 0) S[sx][sz] = edge;          // after the tile: the upper edges may lie within it
    const float up = E(ix, iy == ny - 1 ? 0 : iy + 1, iz), down = E(ix, iy == 0 ? ny - 1 : iy - 1, iz);
    __syncthreads();
    const float h2 = 2.0f * step;
    const float fx = -(S[tx + 2][tz + 1] - S[tx][tz + 1]) / h2;
    const float fy = -(up - down) / h2;
    const float fz = -(S[tx + 1][tz + 2] - S[tx + 1][tz]) / h2;
    tile[tx][tz] = make_float4(fx, fy, fz, e);
    __syncthreads();
    const int ox = threadIdx.x % kT, oz = threadIdx.x / kT;
    if (x0 + ox < nx && z0 + oz < nz) grid[((size_t)(z0 + oz) * ny + iy) * nx + x0 + ox] = tile[ox][oz];
}

// hipFFT plans per (device, shape), created on first use and kept until ppm_fdbm_release_plans.
// A plan's stream is state of the plan, so one caller's hipfftSetStream and its hipfftExec* calls
// run under g_plan_mu as a unit (calls on other streams wait for the enqueue, not for the GPU).
struct Plans {
    int dev, nx, ny, nz;
    hipfftHandle r2c, c2r;
};
std::mutex g_plan_mu;
std::vector<Plans> g_plans;

// The caller holds g_plan_mu.
int get_plans(int nx, int ny, int nz, hipStream_t stream, hipfftHandle* r2c, hipfftHandle* c2r) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) { set_error("fdbm: hipGetDevice failed"); return PPM_ERR_HIP; }
    for (const Plans& p : g_plans)
        if (p.dev == dev && p.nx == nx && p.ny == ny && p.nz == nz) {
            *r2c = p.r2c;
            *c2r = p.c2r;
            return hipfftSetStream(*r2c, stream) == HIPFFT_SUCCESS && hipfftSetStream(*c2r, stream) == HIPFFT_SUCCESS
                       ? PPM_OK : (set_error("fdbm: hipfftSetStream failed"), PPM_ERR_HIP);
        }
    Plans p{dev, nx, ny, nz, 0, 0};
    if (hipfftPlan3d(&p.r2c, nx, ny, nz, HIPFFT_R2C) != HIPFFT_SUCCESS) {
        set_error("fdbm: hipfftPlan3d R2C (%d,%d,%d) failed", nx, ny, nz);
        return PPM_ERR_HIP;
    }
    if (hipfftPlan3d(&p.c2r, nx, ny, nz, HIPFFT_C2R) != HIPFFT_SUCCESS) {
        hipfftDestroy(p.r2c);
        set_error("fdbm: hipfftPlan3d C2R (%d,%d,%d) failed", nx, ny, nz);
        return PPM_ERR_HIP;
    }
    g_plans.push_back(p);
    *r2c = p.r2c;
    *c2r = p.c2r;
    if (hipfftSetStream(*r2c, stream) != HIPFFT_SUCCESS || hipfftSetStream(*c2r, stream) != HIPFFT_SUCCESS) {
        set_error("fdbm: hipfftSetStream failed");
        return PPM_ERR_HIP;
    }
    return PPM_OK;
}

inline unsigned blocks_for(long long n) { return (unsigned)((n + 255) / 256); }

}  // namespace

size_t fdbm_spectrum_bytes(int nx, int ny, int nz) { return (size_t)nx * ny * (nz / 2 + 1) * sizeof(float2); }

int release_fft_plans() {
    std::lock_guard<std::mutex> lock(g_plan_mu);
    int cur = 0;
    const bool have_cur = hipGetDevice(&cur) == hipSuccess;
    int rc = PPM_OK;
    for (const Plans& p : g_plans) {
        if (hipSetDevice(p.dev) != hipSuccess) { rc = PPM_ERR_HIP; continue; }
        if (hipfftDestroy(p.r2c) != HIPFFT_SUCCESS || hipfftDestroy(p.c2r) != HIPFFT_SUCCESS) rc = PPM_ERR_HIP;
    }
    g_plans.clear();
    if (have_cur) (void)hipSetDevice(cur);
    if (rc) set_error("fdbm: destroying a cached hipFFT plan failed");
    return rc;
}

int launch_fft_combine(int mode, int nx, int ny, int nz, float step, const float* a, const float* b, float scale,
                       float* out, void* workspace, hipStream_t stream) {
    std::lock_guard<std::mutex> lock(g_plan_mu);
    hipfftHandle r2c, c2r;
    if (int r = get_plans(nx, ny, nz, stream, &r2c, &c2r)) return r;
    const size_t half = fdbm_spectrum_bytes(nx, ny, nz);
    float2* A = reinterpret_cast<float2*>(workspace);
    float2* B = reinterpret_cast<float2*>(reinterpret_cast<char*>(workspace) + half);
    if (hipfftExecR2C(r2c, const_cast<float*>(a), reinterpret_cast<hipfftComplex*>(A)) != HIPFFT_SUCCESS) {
        set_error("fdbm: forward FFT failed");
        return PPM_ERR_HIP;
    }
    if (mode != PPM_FFT_POISSON) {
        if (hipfftExecR2C(r2c, const_cast<float*>(b), reinterpret_cast<hipfftComplex*>(B)) != HIPFFT_SUCCESS) {
            set_error("fdbm: forward FFT failed");
            return PPM_ERR_HIP;
        }
    }
    const int nzh = nz / 2 + 1;
    const double two_pi = 6.283185307179586;
    const long long nh = (long long)nx * ny * nzh;
    // the inverse transform is unnormalised: fold 1/(nx ny nz) into the spectrum scale
    const float sc = (float)((double)scale / ((double)nx * ny * nz));
    hipLaunchKernelGGL(k_spectrum, dim3(blocks_for(nh)), dim3(256), 0, stream, A, B, mode, nx, ny, nz, nzh,
                       (float)(two_pi / (nx * (double)step)), (float)(two_pi / (ny * (double)step)),
                       (float)(two_pi / (nz * (double)step)), sc);
    if (int r = check_launch("fdbm_spectrum")) return r;
    if (hipfftExecC2R(c2r, reinterpret_cast<hipfftComplex*>(A), out) != HIPFFT_SUCCESS) {
        set_error("fdbm: inverse FFT failed");
        return PPM_ERR_HIP;
    }
    return PPM_OK;
}

int launch_pauli_scale(float* field, long long n, float A, float beta, float clip, hipStream_t stream) {
    hipLaunchKernelGGL(k_pauli_scale, dim3(blocks_for(n)), dim3(256), 0, stream, field, n, A, beta, clip);
    return check_launch("fdbm_pauli_scale");
}

int launch_pad_roll(const float* src, const int s[3], float* dst, const int n[3], const int o[3], const int r[3],
                    hipStream_t stream) {
    hipLaunchKernelGGL(k_pad_roll, dim3(blocks_for((long long)n[0] * n[1] * n[2])), dim3(256), 0, stream, src, s[0],
                       s[1], s[2], dst, n[0], n[1], n[2], o[0], o[1], o[2], r[0], r[1], r[2]);
    return check_launch("fdbm_pad_roll");
}

int launch_flip3(const float* src, float* dst, const int n[3], hipStream_t stream) {
    hipLaunchKernelGGL(k_flip3, dim3(blocks_for((long long)n[0] * n[1] * n[2])), dim3(256), 0, stream, src, dst, n[0],
                       n[1], n[2]);
    return check_launch("fdbm_flip3");
}

int launch_dispersion(const float* atoms, int na, const float origin[3], float step, const int n[3], float ra2,
                      int accumulate, float* out, hipStream_t stream) {
    // four voxels a thread where that leaves 2 waves for every SIMD (80^3, 38 atoms: 9.3 us
    // with four, 10.6 with one; 64 x 60 x 64: 7.3 and 6.8)
    auto launch = [&](auto kernel, int V) {
        const long long threads = (long long)((n[0] + V - 1) / V) * n[1] * n[2];
        hipLaunchKernelGGL(kernel, dim3(blocks_for(threads)), dim3(256), 0, stream, reinterpret_cast<const float4*>(atoms),
                           na, origin[0], origin[1], origin[2], step, n[0], n[1], n[2], ra2, accumulate, out);
    };
    if ((long long)n[0] * n[1] * n[2] >= 4LL * 2 * 1024 * 64) launch(k_dispersion<4>, 4);
    else launch(k_dispersion<1>, 1);
    return check_launch("fdbm_dispersion");
}

int launch_compose_gradient(const float* e1, const float* e2, const float* e3, const int n[3], float step,
                            float* grid, hipStream_t stream) {
    const long long tiles = (long long)((n[2] + kT - 1) / kT) * ((n[0] + kT - 1) / kT) * n[1];
    hipLaunchKernelGGL(k_compose_gradient, dim3((unsigned)((tiles + kXcds - 1) / kXcds * kXcds)), dim3(kT * kT), 0, stream,
                       e1, e2, e3, n[0], n[1], n[2], step, reinterpret_cast<float4*>(grid));
    return check_launch("fdbm_compose_gradient");
}

}  // namespace ppm
