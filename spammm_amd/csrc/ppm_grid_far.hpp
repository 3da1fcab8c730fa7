// ppm_grid_far.hpp — force-field grid projection with interpolated far fields (device code shared
// by the plain and the batched kernels).
//
// The direct sum (ppm_grid_core.hpp) evaluates every atom image at every voxel and is bound by the
// VALU: 1800 sites per voxel on a 300x300x240 grid, while the field of a site a few block sizes
// away is a smooth function over a block of voxels.  Here a block's voxels are split from its sites
// by distance:
//   * near sites are summed directly at the 16^3 voxels of a block;
//   * the other sites are summed at 8^3 Chebyshev nodes of the block (512 points instead of 4096),
//     and the polynomial through the node values is evaluated at the voxels;
//   * with two levels a workgroup takes 2^3 blocks: sites far from all of them are summed at the
//     8^3 nodes of the 32^3 voxels (512 instead of 32768), and that polynomial is evaluated at the
//     nodes of each block.
// No site is left out: every site enters every voxel once, through exactly one of the three sums.
// The interpolation error of a force r^-p at distance d from the centre of a block of half-width h is about
// C(p + 7, 8) / 2^7 (h/d)^8 of it: the steeper the law, the larger (p = 2: 7e-10 at d = 10 h, 7: 2.3e-7, 13: 1e-5).
// A site is near closer than kRatio h, and farther out while that error of its terms is above the FP32 rounding of
// their sum (is_near).
// Blocks are aligned to voxel 0 of the grid, whatever planes are stored, and which sums a site takes
// depends on the block alone, so a z window has the bits of the same planes of the whole grid.
//
// Node positions are taken relative to the block's centre (the centre in FP64), which leaves less
// rounding in dx, dy, dz than absolute FP32 positions.
#pragma once
#pragma clang fp contract(off)
#include "ppm_grid_core.hpp"

namespace ppm {
namespace gf {

using gc::GridArgs;
using gc::Site;

constexpr int kM = 8;              // Chebyshev nodes per axis
constexpr int kB = 16;             // voxels per axis of a block
constexpr int kList = 512;         // sites near a workgroup's blocks that LDS holds at a time
constexpr float kRatio = 10.0f;    // near: closer than kRatio half-widths
constexpr float kTol = 0x1p-22f;   // and while the interpolation error is above this share of a site's terms
// C(p + 7, 8) / 2^7 of the forces r^-7 and r^-13 (measured against FP64 over a block's voxels at 10 to 16 half-widths:
// rms 0.8 to 1.1 of this, largest 1.4 to 3.1)
constexpr float kErr6 = 23.5f, kErr12 = 984.f;
constexpr int kBase = 8;           // planes of a base grid read at a time
constexpr int kMinMid = 6;         // fewer sites than this are cheaper summed at the voxels

// cos((2 i + 1) pi / 16): the nodes on [-1, 1], descending
constexpr double kNode[kM] = {0.98078528040323044913, 0.83146961230254523708, 0.55557023301960222474,
                              0.19509032201612826785, -0.19509032201612826785, -0.55557023301960222474,
                              -0.83146961230254523708, -0.98078528040323044913};

// Weight of node k in the polynomial through the 8 nodes, at u.
constexpr double lagrange(int k, double u) {
    double w = 1.0;
    for (int j = 0; j < kM; ++j)
        if (j != k) w *= (u - kNode[j]) / (kNode[k] - kNode[j]);
    return w;
}

struct Tables {
    float vox[kB][kM];        // block nodes -> the 16 voxels of an axis
    float sub[2][kM][kM];     // nodes of 32 voxels -> the nodes of their lower / upper 16
    constexpr Tables() : vox(), sub() {
        for (int k = 0; k < kM; ++k) {
            for (int i = 0; i < kB; ++i) vox[i][k] = (float)lagrange(k, (i - 7.5) / 7.5);
            for (int h = 0; h < 2; ++h)
                for (int i = 0; i < kM; ++i) sub[h][i][k] = (float)lagrange(k, ((h ? 8.0 : -8.0) + 7.5 * kNode[i]) / 15.5);
        }
    }
};
constexpr Tables kTab{};
static __constant__ Tables c_tab = kTab;

struct Shared {
    float top[4][kM * kM * kM];                // node values of the 32^3 voxels, per channel
    Site list[kList];
    unsigned short mid[kList], near[kList];    // entries of list summed at the nodes / at the voxels
    float a[4][kM * 72];                       // node values of a block; its z-interpolated planes
    union {
        float b[4][kM * 136];
        Site tile[256];
    };
    int cnt[2][4];
};

// Largest squared half edge of a voxel-step cube, in units of half voxels: a skewed or flat block
// counts with its largest edge or diagonal / sqrt(3).
__host__ __device__ inline double step2(const GridArgs& a) {
    double m = 0.0, e[3] = {0.0, 0.0, 0.0};
    for (int s = 0; s < 4; ++s) {
        const double sb = (s & 1) ? -1.0 : 1.0, sc = (s & 2) ? -1.0 : 1.0;
        double d = 0.0;
        for (int q = 0; q < 3; ++q) {
            const double v = (double)a.dA[q] + sb * (double)a.dB[q] + sc * (double)a.dC[q];
            d += v * v;
        }
        if (d / 3.0 > m) m = d / 3.0;
    }
    for (int q = 0; q < 3; ++q) {
        e[0] += (double)a.dA[q] * (double)a.dA[q];
        e[1] += (double)a.dB[q] * (double)a.dB[q];
        e[2] += (double)a.dC[q] * (double)a.dC[q];
    }
    for (int q = 0; q < 3; ++q)
        if (e[q] > m) m = e[q];
    return m;
}

// Squared half-width of a block, and of 2^3 blocks.
__host__ __device__ inline double half2(const GridArgs& a, bool top) {
    const double h = top ? kB - 0.5 : 0.5 * (kB - 1);
    return step2(a) * (h * h);
}

// Squared near radius for the costs: at least kRatio half-widths, and for LJ what is_near gives an uncharged atom with
// its minimum at 3.5 A (10.5 half-widths at 0.1 A, 13 at 0.05 A, 15 at 0.03 A).
__host__ __device__ inline double near2(const GridArgs& a, int model, bool top) {
    const double h2 = half2(a, top);
    double q2 = (double)kRatio * (double)kRatio;
    if (model == PPM_MODEL_LJ)
        for (int i = 0; i < 40; ++i, q2 *= 1.03) {
            const double d2 = q2 * h2, i2 = 12.25 / d2, t12 = 2.0 * i2 * i2 * i2, w = 1.0 / (q2 * q2 * q2 * q2);
            if (w * ((double)kErr6 + (double)kErr12 * t12) <= (double)kTol * (1.0 + t12)) break;
        }
    return q2 * h2;
}

// Expected number of sites within r of a point of the molecule's plane, from the sites' area density
// (over the lattice cell of the images, or over the grid), averaged over heights within r.
__host__ __device__ inline double expected_near(const GridArgs& a, double r2) {
    const double gx = ((double)a.dA[0] * (double)a.dB[1] - (double)a.dA[1] * (double)a.dB[0]) * a.nx * a.ny;
    const double lx = (double)a.lvA[0] * (double)a.lvB[1] - (double)a.lvA[1] * (double)a.lvB[0];
    double area = (a.npbc_a > 0 && a.npbc_b > 0) ? lx : gx;
    if (area < 0.0) area = -area;
    const double n = (double)a.nsites, e = area > 0.0 ? 1.885 * r2 * (double)a.na / area : n;
    return e < n ? e : n;
}

// The form of a whole grid: 0 the direct sum, 1 one level of blocks, 2 two levels (LJ only: 2 I_8(K h)
// of 32 voxels is 300 times that of 16 or more).  It depends on the grid, never on the planes a launch stores, and is
// plain double arithmetic, so host and device agree.
// Costs are in pair evaluations, of which the card does 2.9e9 per ms (5.8e7: the 20 us any launch
// takes): direct N per voxel; one level 512 N_far + 4096 N_near per block and 25e3 for its
// interpolation, but at least one workgroup's own time (8e6 evaluations per ms).  Measured, direct
// against one level: 20 sites on 160^3 38 / 43 us, 60 on 160^3 96 / 77, 180 on 160x160x48 119 / 47, 540
// on 83x83x48 at 0.25 A 98 / 152, at 0.2 A and 104x104x60 245 / 115; hence the 0.85.  A second level
// replaces 7/8 of a block's far evaluations by about 62e3 of interpolation and serial work and has
// an eighth of the workgroups: measured, one level against two: 300x300x240 voxels with 60 sites 165 /
// 253 us, 180 sites 253 / 225, 540 655 / 401, 1800 2114 / 722; 160^3 with 1800 538 / 596; 200x200x40
// with 2304 320 / 357, with 5184 772 / 574.
// A Morse field without tip charges is summed directly (is_near).
__host__ __device__ inline int far_level(const GridArgs& a, int model) {
    if (a.dC[0] != 0.f || a.dC[1] != 0.f) return 0;
    if (model == PPM_MODEL_MORSE && a.q0 == 0.f && a.noff == 0) return 0;
    const double n = (double)a.nsites, vox = (double)a.nx * a.ny * a.nz;
    const double near = expected_near(a, near2(a, model, false));
    const double per = 512.0 * (n - near) + 4096.0 * near;
    auto blocks = [&](int b) { return (double)((a.nx + b - 1) / b) * ((a.ny + b - 1) / b) * ((a.nz + b - 1) / b); };
    double one = blocks(kB) * (per + 25e3);
    if (one < 362.0 * per) one = 362.0 * per;
    if (!(one + 5.8e7 < 0.85 * (vox * n + 5.8e7))) return 0;
    const double nb = blocks(2 * kB), far = (n - expected_near(a, near2(a, model, true))) * nb;
    return model == PPM_MODEL_LJ && far >= (nb >= 150.0 ? 1e5 : 4e5) ? 2 : 1;
}

// A value every lane holds alike, in a scalar register.
__device__ __forceinline__ float uniform(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
}

struct Centre {          // centre of a block: FP32 value and the rest of the FP64 one
    float x, y, z, rx, ry, rz;
};

__device__ __forceinline__ Centre centre_of(const GridArgs& a, int i0, int j0, int k0, double half) {
    Centre c;
    double p[3];
    for (int q = 0; q < 3; ++q)
        p[q] = (double)a.p0[q] + (double)a.dA[q] * (i0 + half) + (double)a.dB[q] * (j0 + half) +
               (double)a.dC[q] * (k0 + half);
    c.x = uniform((float)p[0]); c.y = uniform((float)p[1]); c.z = uniform((float)p[2]);
    c.rx = uniform((float)(p[0] - c.x)); c.ry = uniform((float)(p[1] - c.y)); c.rz = uniform((float)(p[2] - c.z));
    return c;
}

// What decides whether a site is near a block: the squared half-width, the span [zlo, zhi] of 0 and the tip charges'
// z offsets, and the sum of the |charges|.
struct NearRule {
    float h2, zlo, zhi, q;
};

template <int OFF>
__device__ __forceinline__ NearRule near_rule(const GridArgs& a, bool top) {
    NearRule n{uniform((float)half2(a, top)), 0.f, 0.f, fabsf(a.q0)};
#pragma unroll
    for (int o = 0; o < 4; ++o)
        if (OFF != gc::kOffNone && o < a.noff) {
            n.zlo = fminf(n.zlo, a.zoff[o]);
            n.zhi = fmaxf(n.zhi, a.zoff[o]);
            n.q += fabsf(a.qoff[o]);
        }
    return n;
}

// Closer than r to the centre c, with every charge of the tip's sites (the tip charge at z offset zo sees the site at
// S.z - zo; [zlo, zhi] spans 0 and the offsets).  A NaN position is.
__device__ __forceinline__ bool closer(const Site& S, const Centre& c, float r2, float zlo, float zhi) {
    const float dx = S.x - c.x, dy = S.y - c.y;
    const float up = S.z - zlo - c.z, lo = S.z - zhi - c.z;      // the interval the charges span
    const float dz = lo > 0.f ? lo : (up < 0.f ? up : 0.f);
    return !(dx * dx + dy * dy + dz * dz >= r2);
}

// Interpolation error of ex (ex - 2), ex = e^(-K r) up to a factor, at (K h)^2 = u; 1e-8 is what the distance alone gives.
__device__ __forceinline__ float morse_error(float ex, float u) {
    auto bessel = [](float x2) { const float x4 = x2 * x2; return x4 * x4 * gc::ex2(0.04f * x2); };
    return ex * (1e-8f + 3.9e-7f * (bessel(u) + ex * bessel(4.0f * u)));
}

// Near the centre c: closer than kRatio half-widths, or with an interpolation error above kTol of the site's terms.
// Morse: the error of e^(-K r) is 2 I_8(K h) of its value at the centre, at any distance (2 (K h / 2)^8 / 8! and a
// little more; taken twice: FP64 over a block's voxels gives up to 1.7 times it at K h <= 2).  It is weighed against the
// charges' terms alone: a field of exponentials keeps the direct sum, whose error the interpolated one exceeds at every
// K h >= 0.4 (rms 1.2 to 1.8 times at K = -1.8 and 0.03 to 0.1 A, 160 times at 0.2 A), so that atoms or tips without
// charges are near at any distance.
// LJ without charges, rms error against FP64 of the direct sum | with kRatio alone | so, relative, where kRatio alone is
// worst: 0.04 A voxels at 3 A 9.5e-7 | 4.5e-6 | 2.7e-7, 0.03 A at 2 A 1.1e-6 | 2.5e-6 | 6.4e-7.
template <int MODEL>
__device__ __forceinline__ bool is_near(const Site& S, const Centre& c, const NearRule& n) {
    if (closer(S, c, kRatio * kRatio * n.h2, n.zlo, n.zhi)) return true;
    if constexpr (MODEL == PPM_MODEL_LJ) {
        const float dx = S.x - c.x, dy = S.y - c.y, dz = S.z - c.z, dxy2 = dx * dx + dy * dy;
        const float up = dz - n.zlo, lo = dz - n.zhi;
        const float d2 = dxy2 + dz * dz;
        if (d2 >= 256.f * n.h2) return false;                    // kErr12 (h/d)^8 < kTol
        const float ir = gc::rsq(d2), i2 = ir * ir, i6 = i2 * i2 * i2, e2 = n.h2 * i2, e4 = e2 * e2;
        const float fq = fmaxf(fabsf(up), fabsf(lo)), iq = gc::rsq(dxy2 + fq * fq);  // of the farthest charge
        const float t6 = fabsf(S.c2) * i6, t12 = fabsf(S.c3) * i6 * i6;              // forces times distance
        const float tc = fabsf(S.q) * n.q * (d2 * ir) * (iq * iq);
        return !(e4 * e4 * (kErr6 * t6 + kErr12 * t12) <= kTol * (t6 + t12 + tc));
    }
    if constexpr (MODEL == PPM_MODEL_MORSE) {
        const float dx = S.x - c.x, dy = S.y - c.y, dz = S.z - c.z, dxy2 = dx * dx + dy * dy;
        const float up = dz - n.zlo, lo = dz - n.zhi, fq = fmaxf(fabsf(up), fabsf(lo)), iq = gc::rsq(dxy2 + fq * fq);
        const float d2 = dxy2 + dz * dz, ir = gc::rsq(d2), ex = gc::ex2(fmaf(S.c2, d2 * ir, S.c0));
        const float t = fabsf(S.c1) * (fabsf(S.c3) + ir);                           // forces
        const float tc = fabsf(S.q) * n.q * (iq * iq);
        return !(t * morse_error(ex, S.c2 * S.c2 * n.h2 * 0.480453f) <= kTol * tc);
    }
    return false;
}

// One site at N points of a column (same dx, dy; dz[k] = oz[k] - sz): f[k] += (Fx, Fy, Fz, E).
// The pair laws are grid_tile's.
template <int MODEL, bool HASQ0, int OFF, int N>
__device__ __forceinline__ void add_site(const Site& S, const GridArgs& a, float dx, float dy, float sz,
                                         const float (&oz)[N], float (&f)[N][4]) {
    const float dxy2 = fmaf(dx, dx, fmaf(dy, dy, kR2SAFE));
    const float qq0 = S.q * a.q0;
#pragma unroll
    for (int k = 0; k < N; ++k) {
        const float dz = oz[k] - sz;
        const float r2 = fmaf(dz, dz, dxy2);
        const float ir = gc::rsq(r2);
        const float ir2 = ir * ir;
        float fr;
        if (MODEL == PPM_MODEL_LJ) {
            const float ir6 = ir2 * ir2 * ir2;
            const float t6 = fmaf(S.c1, ir6, -S.c0), t7 = fmaf(S.c3, ir6, -S.c2);
            if (HASQ0) {
                const float ec = qq0 * ir;
                f[k][3] = fmaf(t6, ir6, f[k][3] + ec);
                fr = fmaf(t7, ir6, ec) * ir2;
            } else {
                f[k][3] = fmaf(t6, ir6, f[k][3]);
                fr = t7 * ir6 * ir2;
            }
        } else {
            const float r = r2 * ir;
            const float ex = gc::ex2(fmaf(S.c2, r, S.c0));
            const float Ae = S.c1 * ex;
            f[k][3] = fmaf(ex - 2.0f, Ae, f[k][3]);
            fr = S.c3 * (Ae * (ex - 1.0f)) * ir;
            if (HASQ0) {
                const float ec = qq0 * ir;
                fr = fmaf(ec, ir2, fr);
                f[k][3] += ec;
            }
        }
        f[k][0] = fmaf(fr, dx, f[k][0]);
        f[k][1] = fmaf(fr, dy, f[k][1]);
        f[k][2] = fmaf(fr, dz, f[k][2]);
    }
    auto charge = [&](float qf, float zf) {
        const float qo = S.q * qf, zo = zf;
#pragma unroll
        for (int k = 0; k < N; ++k) {
            const float dzo = (oz[k] - sz) + zo;
            const float iro = gc::rsq(fmaf(dzo, dzo, dxy2));
            const float eo = qo * iro;
            const float fro = eo * iro * iro;
            f[k][0] = fmaf(fro, dx, f[k][0]);
            f[k][1] = fmaf(fro, dy, f[k][1]);
            f[k][2] = fmaf(fro, dzo, f[k][2]);
            f[k][3] += eo;
        }
    };
    if (OFF == gc::kOffNone || S.q == 0.f) return;          // the same for the whole wave: S comes from LDS
    if constexpr (OFF == gc::kOffStatic) {
#pragma unroll
        for (int o = 0; o < 4; ++o) {
            if (o >= a.noff) break;
            charge(a.qoff[o], a.zoff[o]);
        }
    } else if constexpr (OFF == gc::kOffDynamic) {
        for (int o = 0; o < a.noff; ++o) charge(a.qoff[o], a.zoff[o]);
    }
}

// Rank of this thread among the workgroup's threads with flag f (in thread order), and their number;
// the other flag list g likewise.  Ends with every thread past a barrier; cnt may be reused after
// the caller's next barrier.
__device__ __forceinline__ void ranks(bool f, bool g, int (&cnt)[2][4], int& rf, int& nf, int& rg, int& ng) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const unsigned long long mf = __ballot(f), mg = __ballot(g), below = (1ull << lane) - 1ull;
    if (lane == 0) { cnt[0][w] = __popcll(mf); cnt[1][w] = __popcll(mg); }
    __syncthreads();
    rf = __popcll(mf & below);
    rg = __popcll(mg & below);
    nf = ng = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (i < w) { rf += cnt[0][i]; rg += cnt[1][i]; }
        nf += cnt[0][i];
        ng += cnt[1][i];
    }
}

// Sum over the 4 waves of the node sums f (lane = column y * 8 + x, k = z) into dst[channel][z * 64 + lane].
__device__ __forceinline__ void reduce_nodes(Shared& s, const float (&f)[kM][4], float (*dst)[kM * kM * kM]) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    float* part = &s.b[0][0];                       // 2 x 2048 floats, and the third part in a
    float* buf[3] = {part, part + 2048, &s.a[0][0]};
    if (w > 0)
#pragma unroll
        for (int k = 0; k < kM; ++k)
#pragma unroll
            for (int c = 0; c < 4; ++c) buf[w - 1][(c * kM + k) * 64 + lane] = f[k][c];
    __syncthreads();
    float v[kM][4];
    if (w == 0)
#pragma unroll
        for (int k = 0; k < kM; ++k)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int i = (c * kM + k) * 64 + lane;
                v[k][c] = (f[k][c] + buf[0][i]) + (buf[1][i] + buf[2][i]);
            }
    if (dst == nullptr) {                           // into a, which buf[2] is part of: one wave, in order
        if (w == 0)
#pragma unroll
            for (int k = 0; k < kM; ++k)
#pragma unroll
                for (int c = 0; c < 4; ++c) s.a[c][k * 64 + lane] = v[k][c];
    } else if (w == 0) {
#pragma unroll
        for (int k = 0; k < kM; ++k)
#pragma unroll
            for (int c = 0; c < 4; ++c) dst[c][k * 64 + lane] = v[k][c];
    }
    __syncthreads();
}

// a += the polynomial of the 32^3 voxels (top) at the nodes of their block (hx, hy, hz).
__device__ __forceinline__ void add_top(Shared& s, int hx, int hy, int hz) {
    const int lane = threadIdx.x & 63, ch = threadIdx.x >> 6;
    float* t0 = &s.b[0][0] + ch * 512;
    float* t1 = &s.b[0][0] + 2048 + ch * 512;
    float v[kM];
#pragma unroll
    for (int k = 0; k < kM; ++k) v[k] = s.top[ch][k * 64 + lane];
#pragma unroll
    for (int j = 0; j < kM; ++j) {                  // z: lane = (y, x)
        float o = 0.f;
#pragma unroll
        for (int k = 0; k < kM; ++k) o = fmaf(c_tab.sub[hz][j][k], v[k], o);
        t0[j * 64 + lane] = o;
    }
    __syncthreads();
    const int hi = lane >> 3, lo = lane & 7;
#pragma unroll
    for (int k = 0; k < kM; ++k) v[k] = t0[hi * 64 + k * 8 + lo];
#pragma unroll
    for (int j = 0; j < kM; ++j) {                  // y: lane = (z, x)
        float o = 0.f;
#pragma unroll
        for (int k = 0; k < kM; ++k) o = fmaf(c_tab.sub[hy][j][k], v[k], o);
        t1[hi * 64 + j * 8 + lo] = o;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kM; ++k) v[k] = t1[lane * 8 + k];
#pragma unroll
    for (int j = 0; j < kM; ++j) {                  // x: lane = (z, y)
        float o = 0.f;
#pragma unroll
        for (int k = 0; k < kM; ++k) o = fmaf(c_tab.sub[hx][j][k], v[k], o);
        s.a[ch][lane * 8 + j] += o;
    }
    __syncthreads();
}

// f = the polynomial through the node values a at this thread's column (x, y) = (tid & 15, tid >> 4)
// of the block's voxels: z in registers, then y and x through LDS, 8 planes at a time.
__device__ __forceinline__ void interpolate(Shared& s, float (&f)[kB][4]) {
    const int lane = threadIdx.x & 63, ch = threadIdx.x >> 6;
    const int x = threadIdx.x & 15, y = threadIdx.x >> 4;
    float wx[kM], v[kM], z[kB];
#pragma unroll
    for (int k = 0; k < kM; ++k) wx[k] = c_tab.vox[x][k];
#pragma unroll
    for (int k = 0; k < kM; ++k) v[k] = s.a[ch][k * 64 + lane];
#pragma unroll
    for (int i = 0; i < kB; ++i) {
        z[i] = 0.f;
#pragma unroll
        for (int k = 0; k < kM; ++k) z[i] = fmaf(kTab.vox[i][k], v[k], z[i]);
    }
    __syncthreads();
    const int hi = lane >> 3, lo = lane & 7;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
        for (int i = 0; i < 8; ++i) s.a[ch][i * 72 + lane] = z[half * 8 + i];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kM; ++k) v[k] = s.a[ch][hi * 72 + k * 8 + lo];
#pragma unroll
        for (int j = 0; j < kB; ++j) {              // y: lane = (z, x)
            float o = 0.f;
#pragma unroll
            for (int k = 0; k < kM; ++k) o = fmaf(kTab.vox[j][k], v[k], o);
            s.b[ch][hi * 136 + j * 8 + lo] = o;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            __builtin_amdgcn_sched_barrier(0);      // keep the reads of later planes out of the registers
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const float4* p = reinterpret_cast<const float4*>(&s.b[c][i * 136 + y * 8]);
                const float4 p0 = p[0], p1 = p[1];
                float o = wx[0] * p0.x;
                o = fmaf(wx[1], p0.y, o); o = fmaf(wx[2], p0.z, o); o = fmaf(wx[3], p0.w, o);
                o = fmaf(wx[4], p1.x, o); o = fmaf(wx[5], p1.y, o); o = fmaf(wx[6], p1.z, o);
                f[half * 8 + i][c] = fmaf(wx[7], p1.w, o);
            }
        }
    }
}

// Sites [0, nsites) that `keep` accepts, from rank `first` on and at most kList of them, into s.list in
// site order; returns how many sites `keep` accepts in all.  far(S) is called once per tile of 256
// sites with the workgroup's other sites in s.tile[0, n).
template <int MODEL, class KEEP, class FAR>
__device__ __forceinline__ int collect(Shared& s, const float4* __restrict__ atoms, const float* __restrict__ cpar,
                                       const GridArgs& a, int first, KEEP keep, FAR far) {
    int total = 0;
    for (int t0 = 0; t0 < a.nsites; t0 += 256) {
        const int i = t0 + (int)threadIdx.x;
        Site S;
        bool ok = i < a.nsites, k = false;
        if (ok) {
            gc::load_site<MODEL>(atoms, cpar, a, i, S);
            k = keep(S);
        }
        int rk, nk, ro, no;
        ranks(ok && k, ok && !k, s.cnt, rk, nk, ro, no);
        const int at = total + rk - first;
        if (ok && k && at >= 0 && at < kList) s.list[at] = S;
        if (ok && !k) s.tile[ro] = S;
        total += nk;
        __syncthreads();
        far(no);
        __syncthreads();
    }
    return total;
}

// The 16^3 blocks of one workgroup of 256 threads: TWO: the 2^3 blocks whose first voxel is (i0, j0, k0),
// otherwise the one block there.  Voxels with klo <= ic < kend are stored at out[(ic - klo) * ncol + col];
// base as for grid_tile.  Every thread of the workgroup must call it.
// BASE: base is added (a form of its own: its loads cost the others 1 to 3 %).
template <int MODEL, bool HASQ0, int OFF, bool TWO, bool BASE = false>
__device__ __forceinline__ void far_blocks(Shared& s, const float4* __restrict__ atoms, const float* __restrict__ cpar,
                                           const GridArgs& a, int i0, int j0, int k0, int sub0, int sub1, int klo,
                                           int kend, float4* __restrict__ out, const float4* base) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const NearRule n0 = near_rule<OFF>(a, false), n1 = near_rule<OFF>(a, true);

    // offsets of this lane's column of nodes from a centre, for half-width `half` (voxels)
    auto node_offsets = [&](const Centre& c, float half, float& ox, float& oy, float (&oz)[kM]) {
        const int nx = lane & 7, ny = lane >> 3;
        float ux = 0.f, uy = 0.f;
#pragma unroll
        for (int k = 0; k < kM; ++k) {
            if (k == nx) ux = (float)kNode[k] * half;
            if (k == ny) uy = (float)kNode[k] * half;
        }
        ox = fmaf(a.dA[0], ux, fmaf(a.dB[0], uy, c.rx));
        oy = fmaf(a.dA[1], ux, fmaf(a.dB[1], uy, c.ry));
        const float o = fmaf(a.dA[2], ux, fmaf(a.dB[2], uy, c.rz));
#pragma unroll
        for (int k = 0; k < kM; ++k) oz[k] = fmaf(a.dC[2], (float)kNode[k] * half, o);
    };

    // sites first, first + 1, ... into the list: of one level every site passes through it (a look for them among all
    // sites in each round made 180,000 Morse sites on 100x100x60 voxels take 291 ms; so 18.6, the direct sum 108)
    auto load_sites = [&](int first) {
        for (int i = threadIdx.x; i < kList && first + i < a.nsites; i += 256)
            gc::load_site<MODEL>(atoms, cpar, a, first + i, s.list[i]);
        __syncthreads();
    };
    bool top = false;
    int total;
    if constexpr (TWO) {
        const Centre c = centre_of(a, i0, j0, k0, kB - 0.5);
        float ox, oy, oz[kM];
        node_offsets(c, kB - 0.5f, ox, oy, oz);
        float f[kM][4];
#pragma unroll
        for (int k = 0; k < kM; ++k) f[k][0] = f[k][1] = f[k][2] = f[k][3] = 0;
        int nfar = 0;
        total = collect<MODEL>(s, atoms, cpar, a, 0, [&](const Site& S) { return is_near<MODEL>(S, c, n1); },
                               [&](int n) {
                                   nfar += n;
                                   if (wave >= n) return;
                                   Site Sn = s.tile[wave];      // read one site ahead of use
                                   for (int j = wave; j < n; j += 4) {
                                       const Site S = Sn;
                                       Sn = s.tile[min(j + 4, n - 1)];
                                       add_site<MODEL, HASQ0, OFF, kM>(S, a, ox - (S.x - c.x), oy - (S.y - c.y),
                                                                       S.z - c.z, oz, f);
                                   }
                               });
        top = nfar > 0;
        if (top) reduce_nodes(s, f, s.top);
    } else {
        total = a.nsites;
        load_sites(0);
    }
    const int rounds = (total + kList - 1) / kList;

#pragma unroll 1
    for (int sub = sub0; sub < sub1; ++sub) {
        const int hx = sub & 1, hy = (sub >> 1) & 1, hz = sub >> 2;
        const int bi = i0 + hx * kB, bj = j0 + hy * kB, bk = k0 + hz * kB;
        if (bi >= a.nx || bj >= a.ny || bk >= kend || bk + kB <= klo) continue;
        const Centre c = centre_of(a, bi, bj, bk, 0.5 * (kB - 1));
        auto load_round = [&](int r) {              // the sites of this round into the list (one round: there)
            if (rounds > 1) {
                __syncthreads();
                if constexpr (TWO) {
                    const Centre ct = centre_of(a, i0, j0, k0, kB - 0.5);
                    collect<MODEL>(s, atoms, cpar, a, r * kList,
                                   [&](const Site& S) { return is_near<MODEL>(S, ct, n1); }, [](int) {});
                } else {
                    load_sites(r * kList);
                }
            }
            return min(kList, total - r * kList);
        };
        // entries of the list that are near this block (s.near) and not (s.mid); their numbers
        auto split = [&](int n, int& nmid, int& nnear) {
            nmid = nnear = 0;
            for (int i = 0; i < n; i += 256) {
                const int e = i + (int)threadIdx.x;
                const bool ok = e < n;
                const bool nr = ok && is_near<MODEL>(s.list[e], c, n0);
                int rn, nn, rm, nm;
                __syncthreads();
                ranks(ok && nr, ok && !nr, s.cnt, rn, nn, rm, nm);
                if (ok && nr) s.near[nnear + rn] = (unsigned short)e;
                if (ok && !nr) s.mid[nmid + rm] = (unsigned short)e;
                nnear += nn;
                nmid += nm;
            }
            __syncthreads();
        };
        int nmid = 0, nnear = 0, mids = 0;
        {
            float ox, oy, oz[kM];
            node_offsets(c, 0.5f * (kB - 1), ox, oy, oz);
            float f[kM][4];
#pragma unroll
            for (int k = 0; k < kM; ++k) f[k][0] = f[k][1] = f[k][2] = f[k][3] = 0;
            for (int r = 0; r < rounds; ++r) {
                const int n = load_round(r);
                split(n, nmid, nnear);
                if (rounds == 1 && !top && nmid < kMinMid) break;
                mids += nmid;
                Site Sn;
                if (wave < nmid) Sn = s.list[s.mid[wave]];
                for (int j = wave; j < nmid; j += 4) {
                    const Site S = Sn;
                    Sn = s.list[s.mid[min(j + 4, nmid - 1)]];
                    add_site<MODEL, HASQ0, OFF, kM>(S, a, ox - (S.x - c.x), oy - (S.y - c.y), S.z - c.z, oz, f);
                }
            }
            if (top || mids > 0) reduce_nodes(s, f, nullptr);
        }
        const int x = threadIdx.x & 15, y = threadIdx.x >> 4;
        float f[kB][4];
        if (top || mids > 0) {
            if (top) add_top(s, hx, hy, hz);
            interpolate(s, f);
        } else {
#pragma unroll
            for (int k = 0; k < kB; ++k) f[k][0] = f[k][1] = f[k][2] = f[k][3] = 0;
        }
        // the voxels' positions as grid_tile has them: a near site's terms are the direct sum's
        const float fia = (float)(bi + x), fib = (float)(bj + y);
        const float px = a.p0[0] + a.dA[0] * fia + a.dB[0] * fib + a.dC[0] * (float)bk;
        const float py = a.p0[1] + a.dA[1] * fia + a.dB[1] * fib + a.dC[1] * (float)bk;
        float pz[kB];
#pragma unroll
        for (int k = 0; k < kB; ++k) pz[k] = a.p0[2] + a.dA[2] * fia + a.dB[2] * fib + a.dC[2] * (float)(bk + k);
        for (int r = 0; r < rounds; ++r) {
            if (rounds > 1) {
                const int n = load_round(r);
                split(n, nmid, nnear);
            }
            auto site = [&](const Site& S) {
                add_site<MODEL, HASQ0, OFF, kB>(S, a, px - S.x, py - S.y, S.z, pz, f);
            };
            auto all = [&](const unsigned short* idx, int n) {
                if (n == 0) return;
                Site Sn = s.list[idx[0]];
                for (int j = 0; j < n; ++j) {
                    const Site S = Sn;
                    Sn = s.list[idx[min(j + 1, n - 1)]];
                    site(S);
                }
            };
            all(s.near, nnear);
            if (rounds == 1 && mids == 0) all(s.mid, nmid);
        }
        if (bi + x < a.nx && bj + y < a.ny) {
            const int col = (bj + y) * a.nx + bi + x;
            // base may be out: the compiler keeps a load behind the stores before it, so eight planes of base are
            // read before the first of them is stored (480x480x149 with a base: 629 -> 522 us,
            // 543 since the near set follows the error bound)
#pragma unroll
            for (int k0 = 0; k0 < kB; k0 += kBase) {
                float4 b[kBase];
                if constexpr (BASE) {
#pragma unroll
                    for (int k = 0; k < kBase; ++k) {
                        const int ic = min(max(bk + k0 + k, klo), kend - 1);
                        b[k] = base[(size_t)(ic - klo) * a.ncol + col];
                    }
                }
#pragma unroll
                for (int k = 0; k < kBase; ++k) {
                    const int ic = bk + k0 + k;
                    if (ic < klo || ic >= kend) continue;
                    float4 v = make_float4(f[k0 + k][0], f[k0 + k][1], f[k0 + k][2], f[k0 + k][3]);
                    if constexpr (BASE) { v.x += b[k].x; v.y += b[k].y; v.z += b[k].z; v.w += b[k].w; }
                    if (a.cap) {
                        const float renorm = 100.0f / fabsf(v.w);
                        if (renorm < 1.0f) { v.x *= renorm; v.y *= renorm; v.z *= renorm; v.w *= renorm; }
                    }
                    out[(size_t)(ic - klo) * a.ncol + col] = v;
                }
            }
        }
        __syncthreads();                            // the next block reuses the lists and buffers
    }
}

}  // namespace gf
}  // namespace ppm
