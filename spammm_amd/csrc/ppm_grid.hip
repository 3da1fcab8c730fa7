// ppm_grid.hip — force-field grid projection for gfx950 (stage a).
//
// Computes, for every voxel of a (nx,ny,nz) grid, the probe's sample force and
// energy (Fx,Fy,Fz,E) from all atoms and their periodic x,y images:
//   LJ     getLJ         kernels/AFM.cl:738-745
//   Morse  getMorse      kernels/AFM.cl:747-757
//   charge getCoulombAFM kernels/AFM.cl:730-736, one term per tip charge site
//          (Qs[k], z offset QZs[k]); COULOMB_CONST applied as in kernels/AFM.cl:961
//   cap    |E|>100 => all four channels scaled by 100/|E|   kernels/AFM.cl:984-985
//   images atom shifted by ix*lvA + iy*lvB, ix,iy in [-npbc,npbc] (kernels/gridFF.cl:960-996)
//
// Two forms, chosen by far_level from the grid alone.  Grids of more than a few sites and blocks
// take the interpolated one (ppm_grid_far.hpp): the flake's 300x300x240 voxels x 1800 sites 13.06 -> 0.73 ms,
// a 9216-site slab on 320x320x96 at 0.05 A 32.9 -> 1.04 ms.  The rest is the direct sum (FP32 VALU-bound):
//   * one workgroup = 256 columns (ia,ib) x V consecutive z voxels per thread (V = 16 or 8
//     for LJ, chosen per launch shape; 8 for Morse, 4 for a tilted dC, 1 for launches of few
//     workgroups); voxels of one thread
//     share dx, dy and dx^2+dy^2 for every site;
//   * the atom x image "sites" are expanded once per 256-site tile into LDS by the
//     workgroup (one site per thread), then read as broadcasts by every lane;
//   * the tip charge at z offset 0 shares r^2 with the pair law (one rsqrt for both);
//     charge sites with a nonzero offset are evaluated separately;
//   * stores are float4 per voxel, consecutive lanes -> consecutive x (1 KiB per wave).
#include <algorithm>

#include "ppm_grid_core.hpp"
#include "ppm_grid_far.hpp"

namespace ppm {
namespace {

using namespace gc;
using gf::expected_near;
using gf::far_level;
using gf::near2;

// Planes [klo, kend) of the grid (klo = 0, kend = nz: the whole grid), stored from plane klo on:
// a z window has the voxel values of the same planes of the whole grid, bit for bit.
template <int MODEL, bool HASQ0, int V, bool DCZ, typename ACC = float>
__global__ __launch_bounds__(256) void k_grid_project(const float4* __restrict__ atoms,
                                                      const float* __restrict__ cpar, GridArgs a,
                                                      float4* __restrict__ out, const float4* base, int klo,
                                                      int kend) {
    __shared__ Site sites[kTile + 1];
    grid_tile<MODEL, HASQ0, V, DCZ, kOffDynamic, ACC>(atoms, cpar, a, sites, blockIdx.x * 256 + threadIdx.x,
                                                      klo + blockIdx.y * V, kend, out, klo, base);
}

// The interpolated form: workgroup (blockIdx.x, blockIdx.y) takes the (x,y) and z block (two levels: of
// 32 voxels a side, one level: 16) of the planes [klo, kend); blocks are aligned to plane 0.
template <int MODEL, bool HASQ0, bool OFFS, bool TWO, bool BASE>
__global__ __launch_bounds__(256, TWO ? 2 : 3) void k_grid_far(
    const float4* __restrict__ atoms, const float* __restrict__ cpar, GridArgs a, float4* __restrict__ out,
    const float4* base, int klo, int kend, int split) {
    __shared__ gf::Shared s;
    constexpr int B = TWO ? 2 * gf::kB : gf::kB;
    const int nbx = (a.nx + B - 1) / B;
    const int by = (int)blockIdx.x / nbx, bx = (int)blockIdx.x - by * nbx;
    gf::far_blocks<MODEL, HASQ0, OFFS ? kOffDynamic : kOffNone, TWO, BASE>(
        s, atoms, cpar, a, bx * B, by * B, (klo / B + (int)blockIdx.y) * B, (int)blockIdx.z * (TWO ? 8 : 1) / split,
        ((int)blockIdx.z + 1) * (TWO ? 8 : 1) / split, klo, kend, out, base);
}

// ── grid -> atom adjoint ─────────────────────────────────────────────────────────────
//
// Given the cotangent g = dL/dG of every voxel (float4, same layout as the grid), accumulates
// per atom j:  dL/d(x,y,z)_j, dL/dq_j and dL/d(p0,p1)_j with (p0,p1) = (c6,c12) for LJ and
// (R0,E0) for Morse, summed over voxels and periodic images.  For one pair with
// d = v - a, s = |d|^2 + R2SAFE, F = fr(s) d, E = E(s) (dE/ds = -fr/2):
//   dL/da = -[ fr gF + (2 (gF.d) dfr/ds - gE fr) d ]
// and the parameter derivatives follow from the pair law.  Capped voxels (|E| = 100 after
// the rescale) are differentiated through the rescale: g_raw = s g - s (g.fe_raw)/E_raw e_w,
// s = 100/|E_raw|, with fe_raw recomputed for the workgroup.
// Only octets (a column x V consecutive planes) with a nonzero cotangent are evaluated: the
// probes touch a small part of the grid, and within the z blocks they reach whole columns stay
// untouched (pixel and grid spacings differ), so the octets are first listed in octet order
// (k_adj_mark, k_adj_offsets, k_adj_list) and k_grid_adjoint takes 256 listed octets and one of
// up to gridDim.z shares of the atoms per workgroup (when few octets are listed, the shares keep
// ~4096 workgroups in flight, so the last ones do not run alone on the chip; every share re-reads
// its octets' cotangent, so large lists are not split).  Each workgroup
// writes one FP64 partial sum per atom of its share (the V voxels of one site image summed in
// FP32, the rest in FP64), reduced over workgroups by k_reduce_partials in FP64.
// The list order is fixed, so the result does not depend on scheduling.

// Octet o = (z block zb, padded column col) = zb * (gridDim.x * 256) + col, the workgroup layout
// of the grid projection: flag[o] = any voxel of the octet has a nonzero cotangent, count[b] =
// flags set in workgroup b.
template <int V>
__global__ __launch_bounds__(256) void k_adj_mark(GridArgs a, const float4* __restrict__ gcot,
                                                  unsigned char* __restrict__ flag, int* __restrict__ count) {
    const int bid = blockIdx.y * gridDim.x + blockIdx.x;
    const int col = blockIdx.x * 256 + threadIdx.x;
    const int ic0 = blockIdx.y * V;
    bool any = false;
    if (col < a.ncol) {
#pragma unroll
        for (int k = 0; k < V; ++k) {
            if (ic0 + k < a.nz) {
                const float4 g = gcot[(size_t)(ic0 + k) * a.ncol + col];
                any |= (g.x != 0.f) | (g.y != 0.f) | (g.z != 0.f) | (g.w != 0.f);
            }
        }
    }
    flag[(size_t)bid * 256 + threadIdx.x] = any ? 1 : 0;
    const int n = __syncthreads_count(any);
    if (threadIdx.x == 0) count[bid] = n;
}

// Exclusive offsets of the per-workgroup counts (one workgroup, each thread a contiguous run of
// counts) and their total.
__global__ __launch_bounds__(1024) void k_adj_offsets(const int* __restrict__ count, int nb, int* __restrict__ off,
                                                      int* __restrict__ total) {
    __shared__ int s[1024];
    const int per = (nb + 1023) / 1024;
    const int b0 = min(nb, (int)threadIdx.x * per), b1 = min(nb, b0 + per);
    int sum = 0;
    for (int b = b0; b < b1; ++b) sum += count[b];
    s[threadIdx.x] = sum;
    __syncthreads();
    for (int d = 1; d < 1024; d <<= 1) {
        const int v = (int)threadIdx.x >= d ? s[threadIdx.x - d] : 0;
        __syncthreads();
        s[threadIdx.x] += v;
        __syncthreads();
    }
    int run = s[threadIdx.x] - sum;
    for (int b = b0; b < b1; ++b) {
        off[b] = run;
        run += count[b];
    }
    if (threadIdx.x == 1023) *total = s[1023];
}

// list[off[b] + rank] = octet id of every flagged octet, in octet order.
__global__ __launch_bounds__(256) void k_adj_list(const unsigned char* __restrict__ flag, const int* __restrict__ off,
                                                  int* __restrict__ list) {
    __shared__ int wc[4];
    const int bid = blockIdx.y * gridDim.x + blockIdx.x;
    const int o = bid * 256 + (int)threadIdx.x;
    const bool f = flag[o] != 0;
    const unsigned long long m = __ballot(f);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int below = __popcll(m & ((1ull << lane) - 1ull));
    if (lane == 0) wc[w] = __popcll(m);
    __syncthreads();
    int base = off[bid];
    for (int i = 0; i < w; ++i) base += wc[i];
    if (f) list[base + below] = o;
}
template <int MODEL>
__device__ __forceinline__ void pair_fe_raw(float dx, float dy, float dz, float dxy2, float q, float p0, float p1,
                                            float K, const GridArgs& a, float4& fe) {
    const float r2 = fmaf(dz, dz, dxy2);
    const float ir = rsq(r2), ir2 = ir * ir;
    float fr, e;
    if (MODEL == PPM_MODEL_LJ) {
        const float ir6 = ir2 * ir2 * ir2;
        e = fmaf(p1, ir6, -p0) * ir6;
        fr = fmaf(12.f * p1, ir6, -6.f * p0) * ir6 * ir2;
    } else {
        const float r = r2 * ir;
        const float ex = __expf(K * (r - p0));
        e = p1 * ex * (ex - 2.f);
        fr = -2.f * K * p1 * ex * (ex - 1.f) * ir;
    }
    const float ec = q * a.q0 * ir;
    fr = fmaf(ec, ir2, fr);
    e += ec;
    fe.x = fmaf(fr, dx, fe.x); fe.y = fmaf(fr, dy, fe.y); fe.z = fmaf(fr, dz, fe.z); fe.w += e;
    for (int o = 0; o < a.noff; ++o) {
        const float dzo = dz + a.zoff[o];
        const float iro = rsq(fmaf(dzo, dzo, dxy2));
        const float eo = q * a.qoff[o] * iro;
        const float fro = eo * iro * iro;
        fe.x = fmaf(fro, dx, fe.x); fe.y = fmaf(fro, dy, fe.y); fe.z = fmaf(fro, dzo, fe.z); fe.w += eo;
    }
}

// Contributions of one pair to the 6 per-atom accumulators: t[0..2] += d(g.(F,E))/d(voxel - atom)
// (the caller subtracts them: the atom moves opposite to the voxel offset), t[3] += d/dq,
// t[4], t[5] += d/d(c6, c12) (LJ) or d/d(R0, E0) (Morse), only when PAR (the caller wants the
// pair-parameter gradient; without it they stay zero).  OFFS: the tip has charge sites at
// nonzero z offsets.
// FINE (k_adj_far, whose 512 nodes for 4096 voxels average roundings less): the reciprocal roots take a Newton step, and
// t[3] is left to *tq, in FP64.
template <int MODEL, bool OFFS, bool PAR, bool FINE = false>
__device__ __forceinline__ void pair_adjoint(float dx, float dy, float dz, float dxy2, float q, float p0, float p1,
                                             float K, const GridArgs& a, float4 g, float t[6], double* tq = nullptr) {
#pragma clang fp contract(fast)
    auto root = [](float x) {
        const float y = rsq(x);
        return FINE ? fmaf(0.5f * y, fmaf(-x * y, y, 1.0f), y) : y;
    };
    const float s = fmaf(dz, dz, dxy2);
    const float ir = root(s), ir2 = ir * ir;
    const float gd = fmaf(g.z, dz, fmaf(g.y, dy, g.x * dx));
    const float gdi = gd * ir2;
    float fr, dfr;
    if (MODEL == PPM_MODEL_LJ) {
        const float ir6 = ir2 * ir2 * ir2, ir8 = ir6 * ir2;
        const float t12 = p1 * ir6;
        fr = fmaf(12.f, t12, -6.f * p0) * ir8;
        dfr = fmaf(-84.f, t12, 24.f * p0) * (ir8 * ir2);
        if (PAR) {
            t[4] = fmaf(-ir6, fmaf(6.f, gdi, g.w), t[4]);             // d/dc6
            t[5] = fmaf(ir6 * ir6, fmaf(12.f, gdi, g.w), t[5]);       // d/dc12
        }
    } else {
        const float r = s * ir;
        const float ex = __expf(K * (r - p0));
        const float A = p1 * ex;
        fr = -2.f * K * A * (ex - 1.f) * ir;
        // d fr / d r, then / (2 r) for d/ds
        const float dfr_dr = -2.f * K * A * (K * (2.f * ex - 1.f) * ir - (ex - 1.f) * ir2);
        dfr = dfr_dr * 0.5f * ir;
        const float dE_dR0 = -2.f * K * A * (ex - 1.f);
        const float dfr_dR0 = 2.f * K * K * A * (2.f * ex - 1.f) * ir;
        if (PAR) {
            t[4] += gd * dfr_dR0 + g.w * dE_dR0;                                   // d/dR0
            t[5] += gd * (-2.f * K * ex * (ex - 1.f) * ir) + g.w * ex * (ex - 2.f); // d/dE0
        }
    }
    if (a.q0 != 0.f) {
        const float ec = q * a.q0 * ir;          // Coulomb at z offset 0 shares d with the pair law
        const float frc = ec * ir2;
        fr += frc;
        dfr = fmaf(-1.5f * frc, ir2, dfr);
        if (FINE) *tq = fma((double)a.q0 * (double)ir, (double)(gdi + g.w), *tq);
        else t[3] = fmaf(a.q0 * ir, gdi + g.w, t[3]);
    }
    const float coef = fmaf(2.f * gd, dfr, -g.w * fr);
    t[0] = fmaf(fr, g.x, fmaf(coef, dx, t[0]));
    t[1] = fmaf(fr, g.y, fmaf(coef, dy, t[1]));
    t[2] = fmaf(fr, g.z, fmaf(coef, dz, t[2]));
    if (OFFS) {
        for (int o = 0; o < a.noff; ++o) {
            const float dzo = dz + a.zoff[o];
            const float so = fmaf(dzo, dzo, dxy2);
            const float iro = root(so), iro2 = iro * iro;
            const float gdo = fmaf(g.z, dzo, fmaf(g.y, dy, g.x * dx));
            const float eo = q * a.qoff[o] * iro;
            const float fro = eo * iro2;
            const float co = 2.f * gdo * (-1.5f * fro * iro2) - g.w * fro;
            t[0] = fmaf(fro, g.x, fmaf(co, dx, t[0]));
            t[1] = fmaf(fro, g.y, fmaf(co, dy, t[1]));
            t[2] = fmaf(fro, g.z, fmaf(co, dzo, t[2]));
            if (FINE) {
                const double x = dx, y = dy, z = (double)dz + (double)a.zoff[o];       // these charges nearly cancel
                const double r2 = fma(z, z, fma(x, x, fma(y, y, (double)kR2SAFE)));
                double i = iro;
                i = fma(0.5 * i, fma(-r2 * i, i, 1.0), i);
                const double h = fma((double)g.z, z, fma((double)g.y, y, (double)g.x * x));
                *tq = fma((double)a.qoff[o] * i, fma(h, i * i, (double)g.w), *tq);
            } else {
                t[3] = fmaf(a.qoff[o] * iro, fmaf(gdo, iro2, g.w), t[3]);
            }
        }
    }
}

template <int MODEL, int V, bool DCZ, bool OFFS, bool PAR>
__global__ __launch_bounds__(256) void k_grid_adjoint(const float4* __restrict__ atoms, const float* __restrict__ cpar,
                                                      GridArgs a, const float4* __restrict__ grid,
                                                      const float4* __restrict__ gcot, const float4* __restrict__ base,
                                                      const int* __restrict__ list, const int* __restrict__ total,
                                                      double* __restrict__ partials, int* __restrict__ active) {
#pragma clang fp contract(fast)
    __shared__ double red[4][6];
    const int bid = blockIdx.y * gridDim.x + blockIdx.x;
    const int n_list = *total;
    if (bid * 256 >= n_list) {           // the same for every thread of the workgroup
        if (threadIdx.x == 0 && blockIdx.z == 0) active[bid] = 0;
        return;
    }
    if (threadIdx.x == 0 && blockIdx.z == 0) active[bid] = 1;
    // atoms [j_begin, j_end): share blockIdx.z of n_share, n_share = the number of shares (at most
    // gridDim.z) that brings the listed workgroups to ~4096 (16 per CU)
    const int n_wg = (n_list + 255) / 256;
    const int n_share = min((int)gridDim.z, max(1, (4096 + n_wg - 1) / n_wg));
    if ((int)blockIdx.z >= n_share) return;
    const int per = (a.na + n_share - 1) / n_share;
    const int j_begin = min(a.na, (int)blockIdx.z * per), j_end = min(a.na, j_begin + per);
    const int e = bid * 256 + (int)threadIdx.x;
    const bool colok = e < n_list;
    const int oct = list[colok ? e : n_list - 1];
    const int ncolp = (int)gridDim.x * 256;
    const int zb = oct / ncolp;
    const int col = oct - zb * ncolp;     // < a.ncol: only octets holding voxels are listed
    const int ia = col % a.nx, ib = col / a.nx;
    const int ic0 = zb * V;
    float4 g[V];
#pragma unroll
    for (int k = 0; k < V; ++k) {
        const bool ok = colok && ic0 + k < a.nz;
        g[k] = ok ? gcot[(size_t)(ic0 + k) * a.ncol + col] : make_float4(0.f, 0.f, 0.f, 0.f);
    }

    float px[DCZ ? 1 : V], py[DCZ ? 1 : V], pz[V];
#pragma unroll
    for (int k = 0; k < V; ++k) {
        const float fic = (float)(ic0 + k), fia = (float)ia, fib = (float)ib;
        pz[k] = a.p0[2] + a.dA[2] * fia + a.dB[2] * fib + a.dC[2] * fic;
        if (!DCZ || k == 0) {
            px[k] = a.p0[0] + a.dA[0] * fia + a.dB[0] * fib + a.dC[0] * fic;
            py[k] = a.p0[1] + a.dA[1] * fia + a.dB[1] * fib + a.dC[1] * fic;
        }
    }
    const int cs = MODEL == PPM_MODEL_LJ ? 2 : 4;

    // voxels clipped by the |E|>100 rescale: recompute the raw sum, chain through the rescale
    bool capped = false;
    if (a.cap) {
#pragma unroll
        for (int k = 0; k < V; ++k) {
            const bool nzk = (g[k].x != 0.f) | (g[k].y != 0.f) | (g[k].z != 0.f) | (g[k].w != 0.f);
            if (nzk && colok && ic0 + k < a.nz) {
                if (fabsf(grid[(size_t)(ic0 + k) * a.ncol + col].w) >= 99.999f) capped = true;
            }
        }
    }
    if (__syncthreads_or(capped)) {
        float4 fe[V];
#pragma unroll
        for (int k = 0; k < V; ++k) fe[k] = make_float4(0.f, 0.f, 0.f, 0.f);
        for (int j = 0; j < a.na; ++j) {
            const float4 at = atoms[j];
            const float p0 = cpar[j * cs], p1 = cpar[j * cs + 1], K = MODEL == PPM_MODEL_LJ ? 0.f : cpar[j * cs + 2];
            for (int iy = -a.npbc_b; iy <= a.npbc_b; ++iy)
                for (int ix = -a.npbc_a; ix <= a.npbc_a; ++ix) {
                    const float sx = at.x + ix * a.lvA[0] + iy * a.lvB[0];
                    const float sy = at.y + ix * a.lvA[1] + iy * a.lvB[1];
                    const float sz = at.z + ix * a.lvA[2] + iy * a.lvB[2];
#pragma unroll
                    for (int k = 0; k < V; ++k) {
                        const int kk = DCZ ? 0 : k;
                        const float dx = px[kk] - sx, dy = py[kk] - sy;
                        pair_fe_raw<MODEL>(dx, dy, pz[k] - sz, fmaf(dx, dx, fmaf(dy, dy, kR2SAFE)), at.w, p0, p1, K,
                                           a, fe[k]);
                    }
                }
        }
        if (base) {            // the raw sum includes the base grid's atoms
#pragma unroll
            for (int k = 0; k < V; ++k) {
                if (colok && ic0 + k < a.nz) {
                    const float4 b = base[(size_t)(ic0 + k) * a.ncol + col];
                    fe[k].x += b.x; fe[k].y += b.y; fe[k].z += b.z; fe[k].w += b.w;
                }
            }
        }
#pragma unroll
        for (int k = 0; k < V; ++k) {
            if (fabsf(fe[k].w) > 100.f) {
                const float sc = 100.f / fabsf(fe[k].w);
                const float gdf = g[k].x * fe[k].x + g[k].y * fe[k].y + g[k].z * fe[k].z + g[k].w * fe[k].w;
                g[k].x *= sc; g[k].y *= sc; g[k].z *= sc;
                g[k].w = sc * g[k].w - sc * gdf / fe[k].w;
            }
        }
    }

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    constexpr int NC = PAR ? 6 : 4;      // accumulated columns: xyz, q (+ the pair parameters)
    for (int j = j_begin; j < j_end; ++j) {
        const float4 at = atoms[j];
        const float p0 = cpar[j * cs], p1 = cpar[j * cs + 1], K = MODEL == PPM_MODEL_LJ ? 0.f : cpar[j * cs + 2];
        // The V voxels of one image are summed in FP32, everything above in FP64: the grid
        // cotangent alternates in sign along z (it is a Δf adjoint), so contractions with the
        // long-range charge field cancel by ~1e3 and an FP32 sum over the workgroup would lose
        // ~1e-3 of the charge gradient.
        double acc[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        for (int iy = -a.npbc_b; iy <= a.npbc_b; ++iy)
            for (int ix = -a.npbc_a; ix <= a.npbc_a; ++ix) {
                const float sx = at.x + ix * a.lvA[0] + iy * a.lvB[0];
                const float sy = at.y + ix * a.lvA[1] + iy * a.lvB[1];
                const float sz = at.z + ix * a.lvA[2] + iy * a.lvB[2];
                float t[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int k = 0; k < V; ++k) {
                    const int kk = DCZ ? 0 : k;
                    const float dx = px[kk] - sx, dy = py[kk] - sy;
                    pair_adjoint<MODEL, OFFS, PAR>(dx, dy, pz[k] - sz, fmaf(dx, dx, fmaf(dy, dy, kR2SAFE)), at.w,
                                                   p0, p1, K, a, g[k], t);
                }
#pragma unroll
                for (int c = 0; c < 3; ++c) acc[c] -= (double)t[c];
#pragma unroll
                for (int c = 3; c < NC; ++c) acc[c] += (double)t[c];
            }
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            double v = acc[c];
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
            if (lane == 0) red[wave][c] = v;
        }
        __syncthreads();
        if (threadIdx.x < 6)
            partials[((size_t)bid * a.na + j) * 6 + threadIdx.x] =
                (int)threadIdx.x < NC
                    ? red[0][threadIdx.x] + red[1][threadIdx.x] + red[2][threadIdx.x] + red[3][threadIdx.x]
                    : 0.0;
        __syncthreads();
    }
}

// The interpolated form (ppm_grid_far.hpp), transposed: for the sites far from a block of 16^3 voxels the block's
// cotangents are gathered at its 8^3 Chebyshev nodes, G_n = sum_v w_n(v) g_v, and the pair terms are taken with G_n at
// the nodes; the near sites take theirs at the voxels.  The direct form is bound by the VALU (37 instructions per
// site and voxel); this one evaluates 512 far and 4096 near points per site and block.  The gather is in FP64, so
// the cancellation of an alternating cotangent happens there and FP32 rounds what is left.
// A thread holds a site and walks the points, whose cotangents the workgroup reads alike (LDS for nodes, scalar loads for
// voxels): no sums across lanes, which cost the direct form 48 exchanges per atom.
// Structure gradients of 200 atoms on 300 x 300 x 240 voxels, 45 planes touched: 6.5 -> 2.3 ms in all.
// Errors against FP64, rms over 60 atoms, of the direct form's (0.05 and 0.1 A; cotangents random, of one sign, smooth): xyz
// 0.86 to 1.10, parameters 0.80 to 1.17, q 0.06 to 1.06.  The pair terms' own roundings make them up, so the direct
// form's positions (one FMA an axis) and, for q, whose near and far parts cancel, FINE in both parts.
constexpr int kFarRows = 2048;      // workgroups (x shares) and rows of partials
constexpr int kNearList = 512;
// Near sites: closer than kAdjRatio half-widths of a block (10 in the projection: the terms are one derivative steeper
// than the field), and farther out by the projection's rule (gf::is_near) for the derivatives r^-8 and r^-14 or of
// exponentials against the charges'.
constexpr float kAdjRatio = 12.5f;
constexpr float kAdjErr6 = 50.3f, kAdjErr12 = 1590.f;       // C(p + 7, 8) / 2^7 of p = 8 and 14

// PAR (LJ): the c12 column stands alone, and its r^-14 terms may be off by 4 kTol (13.3 half-widths).  The transposed sum
// is a cotangent's product with the interpolation error, which alternates within a block.
template <int MODEL, bool PAR>
__device__ __forceinline__ bool adj_near(const float4& at, const gf::Centre& c, const gf::NearRule& n, float p0, float p1,
                                         float K) {
    gc::Site S{};
    S.x = at.x; S.y = at.y; S.z = at.z;
    if (gf::closer(S, c, kAdjRatio * kAdjRatio * n.h2, n.zlo, n.zhi)) return true;
    const float dx = at.x - c.x, dy = at.y - c.y, dz = at.z - c.z, dxy2 = dx * dx + dy * dy, d2 = dxy2 + dz * dz;
    const float fq = fmaxf(fabsf(dz - n.zlo), fabsf(dz - n.zhi)), iq = rsq(dxy2 + fq * fq), ir = rsq(d2);
    const float tc = 2.0f * fabsf(at.w) * n.q * (iq * iq * iq);
    if constexpr (MODEL == PPM_MODEL_LJ) {
        const float i2 = ir * ir, i6 = i2 * i2 * i2, e2 = n.h2 * i2, e4 = e2 * e2, e8 = e4 * e4;
        if (PAR && !(e8 * kAdjErr12 <= 4.0f * gf::kTol)) return true;
        const float t6 = fabsf(42.f * p0) * i6, t12 = fabsf(156.f * p1) * i6 * i6;   // times distance squared
        return !(e8 * (kAdjErr6 * t6 + kAdjErr12 * t12) <= gf::kTol * (t6 + t12 + tc * d2));
    } else {
        const float ex = __expf(K * (d2 * ir - p0)), t = fabsf(p1) * (2.0f * fabsf(K) + ir) * (fabsf(K) + ir);
        return !(t * gf::morse_error(ex, K * K * n.h2) <= gf::kTol * tc);
    }
}

// Squared near radius for the costs (an uncharged LJ atom as gf::near2's; Morse with charges: kAdjRatio).
inline double adj_near2(const GridArgs& a, int model, bool params) {
    const double h2 = gf::half2(a, false);
    double q2 = (double)kAdjRatio * kAdjRatio;
    if (model == PPM_MODEL_LJ) {
        if (params) q2 = std::max(q2, 13.3 * 13.3);
        for (int i = 0; i < 40; ++i, q2 *= 1.03) {
            const double i2 = 12.25 / (q2 * h2), t12 = 156.0 / 84.0 * 2.0 * i2 * i2 * i2, w = 1.0 / (q2 * q2 * q2 * q2);
            if (w * (kAdjErr6 + kAdjErr12 * t12) <= gf::kTol * (1.0 + t12)) break;
        }
    }
    return q2 * h2;
}

struct AdjFar {
    int bx, by, bz;                 // blocks per axis
    int rows;
};

// state[b]: 0 untouched, 1 for k_adj_far, which takes it whole, 2 for k_grid_adjoint (it holds a touched voxel at the
// |E| = 100 rescale, whose raw sum is taken there).  One workgroup per block, V = 8.
__global__ __launch_bounds__(256) void k_adj_blocks(GridArgs a, AdjFar f, const float4* __restrict__ grid,
                                                    const float4* __restrict__ gcot, int ncolp,
                                                    const unsigned char* __restrict__ flag, int* __restrict__ state) {
    const int b = blockIdx.x, x = b % f.bx, y = b / f.bx % f.by, z = b / (f.bx * f.by);
    const int ia = x * gf::kB + (threadIdx.x & 15), ib = y * gf::kB + (threadIdx.x >> 4);
    const bool in = ia < a.nx && ib < a.ny;
    const int col = in ? ib * a.nx + ia : 0;
    bool touched = false, capped = false;
    for (int h = 0; h < 2; ++h) {
        const int ic0 = z * gf::kB + h * 8;
        if (!in || ic0 >= a.nz || !flag[(size_t)(ic0 / 8) * ncolp + col]) continue;
        touched = true;
        if (!a.cap) continue;
        for (int k = ic0; k < min(ic0 + 8, a.nz); ++k) {
            const float4 g = gcot[(size_t)k * a.ncol + col];
            const bool nz = (g.x != 0.f) | (g.y != 0.f) | (g.z != 0.f) | (g.w != 0.f);
            if (nz && fabsf(grid[(size_t)k * a.ncol + col].w) >= 99.999f) capped = true;
        }
    }
    const bool any = __syncthreads_or(touched), direct = __syncthreads_or(capped);
    if (threadIdx.x == 0) state[b] = any ? (direct ? 2 : 1) : 0;
}

// Unlists the octets of k_adj_far's blocks (if it has any); count: the octets left per workgroup of the listing kernels.
__global__ __launch_bounds__(256) void k_adj_count(GridArgs a, AdjFar f, const int* __restrict__ state,
                                                   const int* __restrict__ n_blocks, unsigned char* __restrict__ flag,
                                                   int* __restrict__ count) {
    if (*n_blocks == 0) return;
    const int bid = blockIdx.y * gridDim.x + blockIdx.x, col = blockIdx.x * 256 + (int)threadIdx.x;
    const size_t o = (size_t)bid * 256 + threadIdx.x;
    bool left = flag[o] != 0;
    if (left) {                         // so col is a column of the grid
        const int b = ((int)blockIdx.y / 2 * f.by + col / a.nx / gf::kB) * f.bx + col % a.nx / gf::kB;
        if (state[b] == 1) {
            left = false;
            flag[o] = 0;
        }
    }
    const int n = __syncthreads_count(left);
    if (threadIdx.x == 0) count[bid] = n;
}

// list[0, n) = the blocks with state 1, in order; total = n, or 0 if they are fewer than least (they are then left to
// k_grid_adjoint).
__global__ __launch_bounds__(1024) void k_adj_block_list(const int* __restrict__ state, int nblk, int least,
                                                         int* __restrict__ list, int* __restrict__ total) {
    __shared__ int s[1024];
    const int per = (nblk + 1023) / 1024;
    const int b0 = min(nblk, (int)threadIdx.x * per), b1 = min(nblk, b0 + per);
    int sum = 0;
    for (int b = b0; b < b1; ++b) sum += state[b] == 1;
    s[threadIdx.x] = sum;
    __syncthreads();
    for (int d = 1; d < 1024; d <<= 1) {
        const int v = (int)threadIdx.x >= d ? s[threadIdx.x - d] : 0;
        __syncthreads();
        s[threadIdx.x] += v;
        __syncthreads();
    }
    int at = s[threadIdx.x] - sum;
    for (int b = b0; b < b1; ++b)
        if (state[b] == 1) list[at++] = b;
    if (threadIdx.x == 1023) *total = s[1023] < least ? 0 : s[1023];
}

struct NodeWeights {
    double w[gf::kM][gf::kB];
    constexpr NodeWeights() : w() {
        for (int k = 0; k < gf::kM; ++k)
            for (int i = 0; i < gf::kB; ++i) w[k][i] = gf::lagrange(k, (i - 7.5) / 7.5);
    }
};
constexpr NodeWeights kNodeWeights{};
static __constant__ NodeWeights c_node_weights = kNodeWeights;

struct AdjShared {
    union {
        struct {
            double z[gf::kM * 256];            // gathered along z: [node z][column]
            double y[gf::kM * gf::kM * 16];    // and along y: [node z][node y][x]
        } t;
        double res[256][6];                    // the threads' sums
    };
    float4 g[512];                             // node cotangents [node y][node x][node z]
    float4 node[64];                           // node columns (x, y, z of the middle), relative to the centre
    float4 vox[256];                           // voxel columns (x, y, z of plane 0)
    int list[kNearList];                       // near sites
    int cnt[2][4];
};

template <int MODEL, bool OFFS, bool PAR>
__global__ __launch_bounds__(256, 3) void k_adj_far(const float4* __restrict__ atoms, const float* __restrict__ cpar,
                                                    GridArgs a, AdjFar f, const float4* __restrict__ gcot, const int* __restrict__ list,
                                                    const int* __restrict__ total, double* __restrict__ partials,
                                                    int* __restrict__ active) {
#pragma clang fp contract(fast)
    __shared__ AdjShared s;
    constexpr int NC = PAR ? 6 : 4, cs = MODEL == PPM_MODEL_LJ ? 2 : 4;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n_list = *total, row = blockIdx.x;
    const gf::NearRule rule = gf::near_rule<OFFS ? kOffStatic : kOffNone>(a, false);
    if (row >= n_list) {
        if (tid == 0 && blockIdx.y == 0) active[row] = 0;
        return;
    }
    if (tid == 0 && blockIdx.y == 0) active[row] = 1;
    // few blocks: the atoms in shares, so that ~1024 workgroups are in flight
    const int n_share = min((int)gridDim.y, max(1, 1024 / min(n_list, f.rows)));
    if ((int)blockIdx.y >= n_share) return;
    const int per = (a.na + n_share - 1) / n_share;
    const int j_begin = min(a.na, (int)blockIdx.y * per), j_end = min(a.na, j_begin + per);
    const int nimg = a.nimg_a * a.nimg_b, s_begin = j_begin * nimg, s_end = j_end * nimg;
    double* part = partials + (size_t)row * a.na * 6;
    for (int i = j_begin * 6 + tid; i < j_end * 6; i += 256) part[i] = 0.0;

    auto site = [&](int i, float4& at, float& p0, float& p1, float& K) {
        const int j = i / nimg, m = i - j * nimg, iy = m / a.nimg_a - a.npbc_b, ix = m % a.nimg_a - a.npbc_a;
        at = atoms[j];
        at.x = fmaf((float)iy, a.lvB[0], fmaf((float)ix, a.lvA[0], at.x));
        at.y = fmaf((float)iy, a.lvB[1], fmaf((float)ix, a.lvA[1], at.y));
        at.z = fmaf((float)iy, a.lvB[2], fmaf((float)ix, a.lvA[2], at.z));
        p0 = cpar[j * cs];
        p1 = cpar[j * cs + 1];
        K = MODEL == PPM_MODEL_LJ ? 0.f : cpar[j * cs + 2];
    };
    for (int b = row; b < n_list; b += f.rows) {
        const int blk = __builtin_amdgcn_readfirstlane(list[b]);
        const int i0 = blk % f.bx * gf::kB, j0 = blk / f.bx % f.by * gf::kB, k0 = blk / (f.bx * f.by) * gf::kB;
        const gf::Centre c = gf::centre_of(a, i0, j0, k0, 0.5 * (gf::kB - 1));
        // ── node cotangents ──
        const int ia = i0 + (tid & 15), ib = j0 + (tid >> 4);
        const bool in = ia < a.nx && ib < a.ny;
        float4 g[gf::kB];
#pragma unroll
        for (int k = 0; k < gf::kB; ++k)
            g[k] = in && k0 + k < a.nz ? gcot[(size_t)(k0 + k) * a.ncol + (size_t)ib * a.nx + ia]
                                       : make_float4(0.f, 0.f, 0.f, 0.f);
        __syncthreads();                       // the previous block's sums are taken
        s.vox[tid] = make_float4(a.p0[0] + a.dA[0] * (float)ia + a.dB[0] * (float)ib,
                                 a.p0[1] + a.dA[1] * (float)ia + a.dB[1] * (float)ib,
                                 a.p0[2] + a.dA[2] * (float)ia + a.dB[2] * (float)ib, 0.f);
        if (tid < 64) {
            const float u = 7.5f * (float)gf::kNode[tid & 7], v = 7.5f * (float)gf::kNode[tid >> 3];
            s.node[tid] = make_float4(a.dA[0] * u + a.dB[0] * v, a.dA[1] * u + a.dB[1] * v, a.dA[2] * u + a.dB[2] * v, 0.f);
        }
#pragma unroll
        for (int ch = 0; ch < 4; ++ch) {
#pragma unroll 1
            for (int n = 0; n < gf::kM; ++n) {
                double v = 0.0;
#pragma unroll
                for (int k = 0; k < gf::kB; ++k) v = fma(c_node_weights.w[n][k], (double)(&g[k].x)[ch], v);
                s.t.z[n * 256 + tid] = v;
            }
            __syncthreads();
            for (int u = tid; u < gf::kM * gf::kM * 16; u += 256) {         // x = u % 16, node y, node z
                const double* q = s.t.z + (u >> 7) * 256 + (u & 15);
                double v = 0.0;
                for (int k = 0; k < gf::kB; ++k) v = fma(c_node_weights.w[(u >> 4) & 7][k], q[k * 16], v);
                s.t.y[u] = v;
            }
            __syncthreads();
            for (int u = tid; u < 512; u += 256) {                          // node z = u % 8, node x, node y
                const double* q = s.t.y + ((u & 7) * 8 + (u >> 6)) * 16;
                double v = 0.0;
                for (int k = 0; k < gf::kB; ++k) v = fma(c_node_weights.w[(u >> 3) & 7][k], q[k], v);
                (&s.g[u].x)[ch] = (float)v;
            }
            __syncthreads();
        }
        // ── sites: far ones at the nodes; near ones listed and taken at the voxels ──
        auto add_to_row = [&](int j, const double (&v)[6]) {
#pragma unroll
            for (int q = 0; q < NC; ++q) part[(size_t)j * 6 + q] += v[q];
        };
        auto near = [&](int n) {               // the listed sites, 64 at a time, a quarter of the planes to each wave
            for (int n0 = 0; n0 < n; n0 += 64) {
                const int m = min(64, n - n0);
                float4 at;
                float p0, p1, K;
                site(s.list[n0 + min(lane, m - 1)], at, p0, p1, K);
                double acc[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
                for (int col = 0; col < 256; ++col) {
                    const int ja = i0 + (col & 15), jb = j0 + (col >> 4);
                    if (ja >= a.nx || jb >= a.ny) continue;
                    const float4 vx = s.vox[col];
                    const float dx = vx.x - at.x, dy = vx.y - at.y, dxy2 = fmaf(dx, dx, fmaf(dy, dy, kR2SAFE));
                    const float4* gp = gcot + (size_t)jb * a.nx + ja;
                    float t[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const int ic = k0 + wave * 4 + k;
                        const float4 gv = ic < a.nz ? gp[(size_t)ic * a.ncol] : make_float4(0.f, 0.f, 0.f, 0.f);
                        if (gv.x == 0.f && gv.y == 0.f && gv.z == 0.f && gv.w == 0.f) continue;
                        // written out as the direct form's: contraction is off within a lambda
                        pair_adjoint<MODEL, OFFS, PAR, true>(dx, dy, fmaf(a.dC[2], (float)ic, vx.z) - at.z, dxy2, at.w, p0,
                                                             p1, K, a, gv, t, &acc[3]);
                    }
#pragma unroll
                    for (int q = 0; q < 3; ++q) acc[q] -= (double)t[q];
#pragma unroll
                    for (int q = 4; q < NC; ++q) acc[q] += (double)t[q];
                }
                __syncthreads();
#pragma unroll
                for (int q = 0; q < NC; ++q) s.res[tid][q] = acc[q];
                __syncthreads();
                if (tid < m) {                 // the first of an atom's successive sites takes them all
                    const int j = s.list[n0 + tid] / nimg;
                    if (tid == 0 || s.list[n0 + tid - 1] / nimg != j) {
                        double v[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
                        for (int u = tid; u < m && s.list[n0 + u] / nimg == j; ++u)
                            for (int w = 0; w < 4; ++w)
#pragma unroll
                                for (int q = 0; q < NC; ++q) v[q] += s.res[w * 64 + u][q];
                        add_to_row(j, v);
                    }
                }
                __syncthreads();
            }
        };
        int n_near = 0;
        for (int c0 = s_begin; c0 < s_end; c0 += 256) {
            const int i = c0 + tid;
            const bool ok = i < s_end;
            float4 at;
            float p0, p1, K;
            site(ok ? i : s_end - 1, at, p0, p1, K);
            const bool nr = ok && adj_near<MODEL, PAR>(at, c, rule, p0, p1, K);
            int rk, nk, ro, no;
            gf::ranks(nr, ok && !nr, s.cnt, rk, nk, ro, no);
            if (nr) s.list[n_near + rk] = i;
            n_near += nk;
            // the site from the centre: a rounding of it would be the same for all the block's nodes
            const double sx = ((double)at.x - (double)c.x) - (double)c.rx, sy = ((double)at.y - (double)c.y) - (double)c.ry,
                         sz = ((double)at.z - (double)c.z) - (double)c.rz;
            double acc[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
            if (ok && !nr) {
                for (int col = 0; col < 64; ++col) {
                    const float4 nd = s.node[col];
                    const float dx = (float)((double)nd.x - sx), dy = (float)((double)nd.y - sy);
                    const float dz0 = (float)((double)nd.z - sz), dxy2 = fmaf(dx, dx, fmaf(dy, dy, kR2SAFE));
                    float t[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int k = 0; k < gf::kM; ++k)
                        pair_adjoint<MODEL, OFFS, PAR, true>(dx, dy, fmaf(a.dC[2], 7.5f * (float)gf::kNode[k], dz0), dxy2,
                                                             at.w, p0, p1, K, a, s.g[col * 8 + k], t, &acc[3]);
#pragma unroll
                    for (int q = 0; q < 3; ++q) acc[q] -= (double)t[q];
#pragma unroll
                    for (int q = 4; q < NC; ++q) acc[q] += (double)t[q];
                }
            }
#pragma unroll
            for (int q = 0; q < NC; ++q) s.res[tid][q] = acc[q];
            __syncthreads();
            const int ja = c0 / nimg, jn = (min(c0 + 256, s_end) - 1) / nimg - ja + 1;
            if (tid < jn) {
                const int u0 = max(c0, (ja + tid) * nimg), u1 = min(min(c0 + 256, s_end), (ja + tid + 1) * nimg);
                double v[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
                for (int u = u0; u < u1; ++u)
#pragma unroll
                    for (int q = 0; q < NC; ++q) v[q] += s.res[u - c0][q];
                add_to_row(ja + tid, v);
            }
            __syncthreads();
            if (n_near > kNearList - 256 || c0 + 256 >= s_end) {
                near(n_near);
                n_near = 0;
            }
        }
    }
}

// grad[j*6 + c] = sum over active workgroups b of partials[(b*na + j)*6 + c], in FP64.
__global__ __launch_bounds__(256) void k_reduce_partials(const double* __restrict__ partials,
                                                         const int* __restrict__ active, int nblocks, int na,
                                                         double* __restrict__ grad) {
    __shared__ double red[256];
    const int j = blockIdx.x / 6, c = blockIdx.x - (blockIdx.x / 6) * 6;
    double acc = 0.0;
    for (int b = threadIdx.x; b < nblocks; b += 256)
        if (active[b]) acc += partials[((size_t)b * na + j) * 6 + c];
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) grad[j * 6 + c] = red[0];
}

// 16 or 8 voxels per thread for an LJ launch of ncol columns x nzw planes.  Per voxel, 16 is ~8 %
// cheaper once every compute unit holds several workgroups, but its workgroups take twice as long,
// pad z to a multiple of 16, and, one per compute unit (one wave per SIMD), run latency-bound.
// With k = ceil(workgroups / compute units), the busiest unit's share, the launch time of either
// form, measured on MI355X over 128^2..480^2 columns x 16..256 planes, fits (least squares)
//   16 voxels: 61.0 k + 29 (+ 12 when k = 1),   8 voxels: 33.4 k + 18
// in units of 10 us for 1800 sites (200 atoms x 9 images); the ratio of the two forms does not
// depend on the site count (20..600 atoms measured), so the smaller prediction picks the form
// (within 1.4 % of the faster one on every measured shape).  The two forms sum each voxel's pair
// terms in the same order: their grids are bit-identical.
bool lj_16_voxels(int ncol, int nzw) {
    const long long cus = device_cus();
    const long long cb = (ncol + 255) / 256;
    const long long k16 = (cb * ((nzw + 15) / 16) + cus - 1) / cus;
    const long long k8 = (cb * ((nzw + 7) / 8) + cus - 1) / cus;
    return 610 * k16 + 290 + (k16 == 1 ? 120 : 0) <= 334 * k8 + 180;
}

// Workgroups per 2^3 blocks of the two-level form (1, 2, 4 or 8; each repeats the sums at the 32^3
// voxels' nodes and takes its share of the blocks; the bits do not depend on it).  With F = 512 x far
// sites, S the work of the 8 blocks (in pair evaluations) and nb launched 2^3 blocks, the time
// measured over 98..1125 blocks and 180..9216 sites follows nb (s F + S) / 2.9e9 + 0.6 (F + S / s) /
// 3.5e6 ms: the card's rate and one workgroup's serial time.  300x300x62 planes, 1800 sites: s = 1, 2,
// 4, 8 take 597, 459, 522, 714 us; 300x300x240: 722, 916, 1324, 2247.
int far_split(const GridArgs& a, double nb) {
    const double n = a.nsites, near = expected_near(a, near2(a, PPM_MODEL_LJ, false)),
                 mid = expected_near(a, near2(a, PPM_MODEL_LJ, true));
    const double F = 512.0 * (n - mid), S = 8.0 * (512.0 * (mid - near) + 4096.0 * near + 62e3);
    int best = 1;
    double t = 0.0;
    for (int s = 1; s <= 8; s *= 2) {
        const double ts = nb * (s * F + S) / 2.9e9 + 0.6 * (F + S / s) / 3.5e6;
        if (s == 1 || ts < t) { best = s; t = ts; }
    }
    return best;
}

template <int MODEL, bool HASQ0, bool TWO>
int launch_far(const float4* atoms, const float* cpar, const GridArgs& a, float4* out, const float4* base, hipStream_t st,
               int klo, int kend) {
    constexpr int B = TWO ? 2 * gf::kB : gf::kB;
    const unsigned nxy = (unsigned)(((a.nx + B - 1) / B) * ((a.ny + B - 1) / B)), nz = (kend - 1) / B - klo / B + 1;
    const int split = TWO ? far_split(a, (double)nxy * nz) : 1;
    const dim3 grd(nxy, nz, (unsigned)split), blk(256);
#define PPM_FAR(OF, BA) \
    hipLaunchKernelGGL((k_grid_far<MODEL, HASQ0, OF, TWO, BA>), grd, blk, 0, st, atoms, cpar, a, out, base, klo, kend, split)
    if (a.noff) { if (base) PPM_FAR(true, true); else PPM_FAR(true, false); }
    else { if (base) PPM_FAR(false, true); else PPM_FAR(false, false); }
#undef PPM_FAR
    return check_launch("grid_project_far");
}

template <int MODEL, bool HASQ0>
int dispatch(const float4* atoms, const float* cpar, const GridArgs& a, float4* out, const float4* base,
             bool acc64, hipStream_t st, int klo, int nzw) {
    const bool dcz = (a.dC[0] == 0.f && a.dC[1] == 0.f);
    const int kend = klo + nzw;
    dim3 blk(256);
    // FP64 sums of the FP32 terms at every voxel: the direct sum at any size
    const int level = acc64 ? 0 : far_level(a, MODEL);
    if constexpr (MODEL == PPM_MODEL_LJ)
        if (level == 2) return launch_far<MODEL, HASQ0, true>(atoms, cpar, a, out, base, st, klo, kend);
    if (level) return launch_far<MODEL, HASQ0, false>(atoms, cpar, a, out, base, st, klo, kend);
    if (acc64) {          // FP64 sums: 8 voxels per thread (16 would need 128 VGPRs of sums alone)
        const int V = dcz ? 8 : 4;
        dim3 grd((a.ncol + 255) / 256, (nzw + V - 1) / V);
        if (dcz)
            hipLaunchKernelGGL((k_grid_project<MODEL, HASQ0, 8, true, double>), grd, blk, 0, st, atoms, cpar, a, out,
                               base, klo, kend);
        else
            hipLaunchKernelGGL((k_grid_project<MODEL, HASQ0, 4, false, double>), grd, blk, 0, st, atoms, cpar, a,
                               out, base, klo, kend);
        return check_launch("grid_project_acc64");
    }
    if (dcz) {
        // few workgroups of 8 voxels per thread (up to ~4 per compute unit): one voxel per thread, so the
        // sites' serial loop has more waves to hide it (same bits).  8 against 1, microseconds: 48x48x40
        // voxels and 180 sites 57 / 19, 104x104x60 and 540 246 / 165, 170x170x60 and 1800 1430 / 1260;
        // past that 8 wins: 177x177x150 and 180 338 / 341, 160^3 and 180 275 / 295
        if ((long long)((a.ncol + 255) / 256) * ((nzw + 7) / 8) <= 4LL * device_cus()) {
            dim3 grd((a.ncol + 255) / 256, nzw);
            hipLaunchKernelGGL((k_grid_project<MODEL, HASQ0, 1, true>), grd, blk, 0, st, atoms, cpar, a, out, base, klo,
                               kend);
        } else if (MODEL == PPM_MODEL_LJ && nzw >= 16 && lj_16_voxels(a.ncol, nzw)) {   // 16 on Morse: +2 %
            dim3 grd((a.ncol + 255) / 256, (nzw + 15) / 16);
            hipLaunchKernelGGL((k_grid_project<MODEL, HASQ0, 16, true>), grd, blk, 0, st, atoms, cpar, a, out, base,
                               klo, kend);
        } else if (nzw >= 8) {
            dim3 grd((a.ncol + 255) / 256, (nzw + 7) / 8);
            hipLaunchKernelGGL((k_grid_project<MODEL, HASQ0, 8, true>), grd, blk, 0, st, atoms, cpar, a, out, base,
                               klo, kend);
        } else {
            dim3 grd((a.ncol + 255) / 256, (nzw + 3) / 4);
            hipLaunchKernelGGL((k_grid_project<MODEL, HASQ0, 4, true>), grd, blk, 0, st, atoms, cpar, a, out, base,
                               klo, kend);
        }
    } else {
        dim3 grd((a.ncol + 255) / 256, (nzw + 3) / 4);
        hipLaunchKernelGGL((k_grid_project<MODEL, HASQ0, 4, false>), grd, blk, 0, st, atoms, cpar, a, out, base, klo,
                           kend);
    }
    return check_launch("grid_project");
}

}  // namespace

static GridArgs make_args(int na, const PpmGridSpec& g, const float Qs[4], const float QZs[4], int npbc_a,
                          int npbc_b, const float lvA[3], const float lvB[3], int cap) {
    GridArgs a{};
    a.nx = g.nx; a.ny = g.ny; a.nz = g.nz; a.ncol = g.nx * g.ny;
    for (int k = 0; k < 3; ++k) {
        a.p0[k] = g.p0[k]; a.dA[k] = g.dA[k]; a.dB[k] = g.dB[k]; a.dC[k] = g.dC[k];
        a.lvA[k] = lvA ? lvA[k] : 0.f; a.lvB[k] = lvB ? lvB[k] : 0.f;
    }
    a.na = na;
    a.npbc_a = npbc_a; a.npbc_b = npbc_b;
    a.nimg_a = 2 * npbc_a + 1; a.nimg_b = 2 * npbc_b + 1;
    a.nsites = na * a.nimg_a * a.nimg_b;
    a.cap = cap;
    a.q0 = 0.f;
    a.noff = 0;
    for (int k = 0; k < 4; ++k) {
        if (Qs[k] == 0.f) continue;   // a zero-weight site adds exactly zero
        if (QZs[k] == 0.f) {
            a.q0 += Qs[k] * kCOULOMB;
        } else {
            a.qoff[a.noff] = Qs[k] * kCOULOMB;
            a.zoff[a.noff] = QZs[k];
            ++a.noff;
        }
    }
    return a;
}

// workgroup grid of both the projection and its adjoint
static dim3 grid_blocks(const PpmGridSpec& g, int V) {
    return dim3((unsigned)((g.nx * g.ny + 255) / 256), (unsigned)((g.nz + V - 1) / V));
}

static int adjoint_V(const PpmGridSpec& g) { return (g.dC[0] == 0.f && g.dC[1] == 0.f) ? 8 : 4; }

int launch_grid_project(int model, const float* atoms, const float* cpar, int na, const PpmGridSpec& g,
                        const float Qs[4], const float QZs[4], int npbc_a, int npbc_b, const float lvA[3],
                        const float lvB[3], int cap, const float* base, float* grid, bool acc64,
                        hipStream_t stream, int klo, int nzw) {
    const GridArgs a = make_args(na, g, Qs, QZs, npbc_a, npbc_b, lvA, lvB, cap);
    const float4* at = reinterpret_cast<const float4*>(atoms);
    float4* o = reinterpret_cast<float4*>(grid);
    const float4* b = reinterpret_cast<const float4*>(base);
    const bool hasq0 = a.q0 != 0.f;
    if (nzw <= 0) { klo = 0; nzw = g.nz; }
    if (model == PPM_MODEL_LJ)
        return hasq0 ? dispatch<PPM_MODEL_LJ, true>(at, cpar, a, o, b, acc64, stream, klo, nzw)
                     : dispatch<PPM_MODEL_LJ, false>(at, cpar, a, o, b, acc64, stream, klo, nzw);
    return hasq0 ? dispatch<PPM_MODEL_MORSE, true>(at, cpar, a, o, b, acc64, stream, klo, nzw)
                 : dispatch<PPM_MODEL_MORSE, false>(at, cpar, a, o, b, acc64, stream, klo, nzw);
}

// Workspace of the grid adjoint: per-workgroup FP64 partial rows, active flags, octet flags,
// per-workgroup octet counts and offsets, the octet count and the octet list, the blocks' states and list, each 256-B
// aligned.
struct AdjWorkspace {
    double* partials;
    int* active;
    unsigned char* flag;
    int *count, *off, *total, *list;
    int *state, *blocks, *n_blocks;         // of k_adj_far: 16^3 blocks, the list of its own and their number
};

static AdjFar adj_far(const PpmGridSpec& g) {
    AdjFar f;
    f.bx = (g.nx + gf::kB - 1) / gf::kB;
    f.by = (g.ny + gf::kB - 1) / gf::kB;
    f.bz = (g.nz + gf::kB - 1) / gf::kB;
    f.rows = (int)std::min<long long>(kFarRows, (long long)f.bx * f.by * f.bz);
    return f;
}

// The interpolated form's least number of touched blocks, or 0 if it does not pay at any.  Per block it costs, in pair
// evaluations, 512 for every far site in chunks of 256 and 4096 for every near one in groups of 64, and about 40e3 for
// gathering, against 4096 for every site; and it needs enough blocks to fill the card with its longer workgroups.
// Milliseconds direct | interpolated with 45 planes touched: 200 atoms x 9 images on 300 x 300 x 240 voxels 6.5 | 2.0,
// with 9 % of the columns touched (1.1e9 evaluations direct) 0.89 | 0.61; 60 x 9 on 480 x 480 x 149 at 0.05 A 4.4 | 2.1,
// on 150 x 150 x 120 at 0.1 A (8.8e8) 0.55 | 0.60; 200 on 180 x 180 x 120 0.51 | 0.52; 20 x 9 on 160 x 160 x 120
// 0.26 | 0.57 (k_adj_far takes 10 % more since its roots are finer).  The first bound on the whole grid keeps small
// grids clear of the block kernels (30 us).
static int adj_far_least(const GridArgs& a, const AdjFar& f, int model, bool params) {
    if (a.dC[0] != 0.f || a.dC[1] != 0.f) return 0;
    // Morse: the parameters' columns are exponentials alone, and without tip charges every column is (gf::is_near)
    if (model == PPM_MODEL_MORSE && (params || (a.q0 == 0.f && a.noff == 0))) return 0;
    const double n = a.nsites, near = gf::expected_near(a, adj_near2(a, model, params)), direct = 4096.0 * n;
    const double far = 512.0 * 256.0 * std::ceil(n / 256.0) + 4096.0 * 64.0 * std::ceil(near / 64.0) + 40e3;
    if (far > 0.45 * direct || direct * f.bx * f.by * f.bz < 4e9) return 0;
    return std::max(1, (int)std::ceil(1e9 / direct));
}

static size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }

static size_t adjoint_layout(int na, const PpmGridSpec& g, void* base, AdjWorkspace* w) {
    const dim3 b = grid_blocks(g, adjoint_V(g));
    const size_t nb = (size_t)b.x * b.y, noct = nb * 256;
    const AdjFar f = adj_far(g);
    const size_t nblk = (size_t)f.bx * f.by * f.bz, rows = nb + f.rows;
    const size_t sizes[10] = {rows * (size_t)na * 6 * sizeof(double), rows * sizeof(int), noct, nb * sizeof(int),
                              nb * sizeof(int), sizeof(int), noct * sizeof(int), nblk * sizeof(int), nblk * sizeof(int),
                              sizeof(int)};
    size_t off[10], at = 0;
    for (int i = 0; i < 10; ++i) {
        off[i] = at;
        at += align256(sizes[i]);
    }
    if (w) {
        char* p = reinterpret_cast<char*>(base);
        w->partials = reinterpret_cast<double*>(p + off[0]);
        w->active = reinterpret_cast<int*>(p + off[1]);
        w->flag = reinterpret_cast<unsigned char*>(p + off[2]);
        w->count = reinterpret_cast<int*>(p + off[3]);
        w->off = reinterpret_cast<int*>(p + off[4]);
        w->total = reinterpret_cast<int*>(p + off[5]);
        w->list = reinterpret_cast<int*>(p + off[6]);
        w->state = reinterpret_cast<int*>(p + off[7]);
        w->blocks = reinterpret_cast<int*>(p + off[8]);
        w->n_blocks = reinterpret_cast<int*>(p + off[9]);
    }
    return at + 256;
}

size_t grid_adjoint_workspace(int na, const PpmGridSpec& g) { return adjoint_layout(na, g, nullptr, nullptr); }

int launch_grid_adjoint(int model, const float* atoms, const float* cpar, int na, const PpmGridSpec& g,
                        const float Qs[4], const float QZs[4], int npbc_a, int npbc_b, const float lvA[3],
                        const float lvB[3], int cap, const float* grid, const float* grid_cot, const float* base,
                        void* workspace, int params, double* grad, hipStream_t stream) {
    const GridArgs a = make_args(na, g, Qs, QZs, npbc_a, npbc_b, lvA, lvB, cap);
    const int V = adjoint_V(g);
    const dim3 blocks = grid_blocks(g, V);
    const size_t nb = (size_t)blocks.x * blocks.y;
    size_t n_rows = nb;
    // atom shares per listed workgroup: 4 while each share keeps >= 8 atoms
    const dim3 adj_blocks(blocks.x, blocks.y, (unsigned)std::max(1, std::min(4, na / 8)));
    if (nb * 256 > (size_t)INT32_MAX) {
        set_error("grid_adjoint: %zu voxel octets exceed the int range", nb * 256);
        return PPM_ERR_INVALID_ARG;
    }
    AdjWorkspace w;
    adjoint_layout(na, g, workspace, &w);
    double* partials = w.partials;
    int* active = w.active;
    const float4* at = reinterpret_cast<const float4*>(atoms);
    const float4* G = reinterpret_cast<const float4*>(grid);
    const float4* gc = reinterpret_cast<const float4*>(grid_cot);
    const float4* B = reinterpret_cast<const float4*>(base);
    const bool offs = a.noff > 0;
    if (V == 8) hipLaunchKernelGGL(k_adj_mark<8>, blocks, dim3(256), 0, stream, a, gc, w.flag, w.count);
    else hipLaunchKernelGGL(k_adj_mark<4>, blocks, dim3(256), 0, stream, a, gc, w.flag, w.count);
    const AdjFar far = adj_far(g);
    if (const int least = adj_far_least(a, far, model, params)) {
        const int nblk = far.bx * far.by * far.bz;
        hipLaunchKernelGGL(k_adj_blocks, dim3((unsigned)nblk), dim3(256), 0, stream, a, far, G, gc, (int)blocks.x * 256, w.flag,
                           w.state);
        hipLaunchKernelGGL(k_adj_block_list, dim3(1), dim3(1024), 0, stream, w.state, nblk, least, w.blocks,
                           w.n_blocks);
        hipLaunchKernelGGL(k_adj_count, blocks, dim3(256), 0, stream, a, far, w.state, w.n_blocks, w.flag, w.count);
        if (int r = check_launch("grid_adjoint_blocks")) return r;
        const dim3 fb((unsigned)far.rows, (unsigned)std::max(1, std::min(4, na / 8)));
#define PPM_ADJF(M, OF, PA) \
    hipLaunchKernelGGL((k_adj_far<M, OF, PA>), fb, dim3(256), 0, stream, at, cpar, a, far, gc, w.blocks, w.n_blocks, \
                       partials + nb * (size_t)na * 6, active + nb)
#define PPM_ADJF2(M, PA) if (offs) PPM_ADJF(M, true, PA); else PPM_ADJF(M, false, PA)
        if (model == PPM_MODEL_MORSE) { PPM_ADJF2(PPM_MODEL_MORSE, false); }
        else if (params) { PPM_ADJF2(PPM_MODEL_LJ, true); }
        else { PPM_ADJF2(PPM_MODEL_LJ, false); }
#undef PPM_ADJF2
#undef PPM_ADJF
        if (int r = check_launch("grid_adjoint_far")) return r;
        n_rows += (size_t)far.rows;
    }
    hipLaunchKernelGGL(k_adj_offsets, dim3(1), dim3(1024), 0, stream, w.count, (int)nb, w.off, w.total);
    hipLaunchKernelGGL(k_adj_list, blocks, dim3(256), 0, stream, w.flag, w.off, w.list);
    if (int r = check_launch("grid_adjoint_list")) return r;
#define PPM_ADJ1(M, VV, DCZ, OF, PA)                                                                         \
    hipLaunchKernelGGL((k_grid_adjoint<M, VV, DCZ, OF, PA>), adj_blocks, dim3(256), 0, stream, at, cpar, a, G, gc, \
                       B, w.list, w.total, partials, active)
#define PPM_ADJ(M, VV, DCZ, OF)                                                                              \
    do {                                                                                                     \
        if (params) PPM_ADJ1(M, VV, DCZ, OF, true);                                                         \
        else PPM_ADJ1(M, VV, DCZ, OF, false);                                                               \
    } while (0)
    if (model == PPM_MODEL_LJ) {
        if (V == 8) { if (offs) PPM_ADJ(PPM_MODEL_LJ, 8, true, true); else PPM_ADJ(PPM_MODEL_LJ, 8, true, false); }
        else { if (offs) PPM_ADJ(PPM_MODEL_LJ, 4, false, true); else PPM_ADJ(PPM_MODEL_LJ, 4, false, false); }
    } else {
        if (V == 8) { if (offs) PPM_ADJ(PPM_MODEL_MORSE, 8, true, true); else PPM_ADJ(PPM_MODEL_MORSE, 8, true, false); }
        else { if (offs) PPM_ADJ(PPM_MODEL_MORSE, 4, false, true); else PPM_ADJ(PPM_MODEL_MORSE, 4, false, false); }
    }
#undef PPM_ADJ
#undef PPM_ADJ1
    if (int r = check_launch("grid_adjoint")) return r;
    hipLaunchKernelGGL(k_reduce_partials, dim3((unsigned)(na * 6)), dim3(256), 0, stream, partials, active,
                       (int)n_rows, na, grad);
    return check_launch("grid_adjoint_reduce");
}

}  // namespace ppm
