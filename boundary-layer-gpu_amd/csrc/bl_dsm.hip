// Smagorinsky-type eddy viscosities on the device, the semantics of the
// reference's CPU build:
//   LES = 2  dynamic, z-averaged   sgs_dynamic_Smagorinsky (subgrid.f90:261-414)
//   LES = 3  dynamic, per cell     sgs_dynamic_Smagorinsky_noaverage (:436-583)
//   LES = 1  constant coefficient  sgs_Smagorinsky (:609-662)
// with filter_xzy (:140-187) and compute_Sij (:672-730).
//
// The dynamic models build work arrays, then fix their ghost entries in place
// with apply_Neumann_bc_x (LES = 2, boundary_conditions.f90:326-344) or
// apply_periodic_bc_x (LES = 3, :295-314) and apply_periodic_bc_z (:732-757).
// Here those fixes become index maps applied when an entry is read: an x index
// is clamped into the interior (Neumann) or redirected to its periodic source,
// and a z index on a ghost or duplicated plane is redirected to the plane it
// is copied from.
//   xmap_c periodic (x centres):               0 <- nxg-3, nxg-2 <- 1, nxg-1 <- 2
//   xmap_f periodic (x faces, U):              0 <- nx-2,  nx-1 <- 1
//   zmap_c (cell-centred in z, periodic id 1/2/4): 0 <- nzg-3, nzg-2 <- 1, nzg-1 <- 2
//   z faces (W, id 3):                           0 <- nz-2,  nz-1 <- 1
//
// Passes (0-based indices, every array in the padded field layout):
//   k_dsm_vfilter  test-filtered velocities Uf, Vf, Wf (:329-344)
//   k_dsm_stress   marching in z: cell-centred velocities (interpolation.f90:
//                  24-114 with the fixes of subgrid.f90:282-284), |S| and
//                  |S|*S_ij (:351-357), their test filters and those of the
//                  products, the filtered strain, L_ij, M_ij, then L:M and M:M,
//                  summed over the planes of the block's chunk
//   k_dsm_column   z averages per (x, y) column, nu_t = max(-<L:M>/<M:M>/2*|S|, 0)
//                  and the y ghost rows (:371-412)
//   k_dsm_cellwise LES = 3: the ratio per cell (formed in k_dsm_stress) with the
//                  periodic x and z copies and the y ghost rows (:545-581)
//   k_smag         LES = 1: (Cs Delta_j f_j)^2 |S| on the interior cells
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "../../include/blgpu.h"
#include "bl_internal.hpp"

namespace blgpu {

namespace {

// field-sized work arrays; behind them the chunk sums of L:M and M:M
enum DsmSlot {
    D_S = 0,  // |S| of the unfiltered field (LES = 3: max(-(L:M)/(M:M)/2*|S|, 0)), interior cells
    D_UF,
    D_VF,
    D_WF,
    D_END
};

__device__ __forceinline__ int clampi(int i, int lo, int hi) { return i < lo ? lo : (i > hi ? hi : i); }
__device__ __forceinline__ int zmap_c(const Dims &d, int k) {
    return k == 0 ? d.nzg - 3 : (k == d.nzg - 2 ? 1 : (k == d.nzg - 1 ? 2 : k));
}
// x fix of the cell-centred work arrays (extent nxg) and of the filtered U (extent nx)
template <bool PX>
__device__ __forceinline__ int xmap_c(const Dims &d, int i) {
    if constexpr (PX) return i == 0 ? d.nxg - 3 : (i == d.nxg - 2 ? 1 : (i == d.nxg - 1 ? 2 : i));
    return clampi(i, 1, d.nxg - 2);
}
template <bool PX>
__device__ __forceinline__ int xmap_f(const Dims &d, int i) {
    if constexpr (PX) return i == 0 ? d.nx - 2 : (i == d.nx - 1 ? 1 : i);
    return clampi(i, 1, d.nx - 2);
}

// the x and y metrics that compute_Sij reads at one (i, j), held in registers
// along a march in z (they would be loaded again behind every store)
struct StrainMet {
    double rdx, rdxg0, rdxg1;  // 1/dx(i), 1/dxg(i-1), 1/dxg(i)
    double rdy, rdyg0, rdyg1;
};
__device__ __forceinline__ StrainMet strain_met(const Metrics &m, int i, int j) {
    return {m.rdx[i], m.rdxg[i - 1], m.rdxg[i], m.rdy[j], m.rdyg[j - 1], m.rdyg[j]};
}

// A plane of a field as a wave-uniform global pointer whose origin the compiler
// does not see, and its elements at 32-bit byte offsets (a plane is below
// 4 GB: twenty arrays of the smallest grid's five such planes would not fit the
// card).  The many neighbours of a stencil are then a scalar base and one
// shared register per row; with plain indexing the loop-invariant part of
// every neighbour's 64-bit address was kept in two registers of each lane
// across the march.
template <class T>
using PlanePtr = const T __attribute__((address_space(1))) *;
template <class T>
__device__ __forceinline__ PlanePtr<T> plane_ptr(const T *p) {
    PlanePtr<T> q = (PlanePtr<T>)p;
    asm volatile("" : "+s"(q));
    return q;
}
template <class T>
__device__ __forceinline__ double at(PlanePtr<T> base, unsigned o) {
    return (double)*(PlanePtr<T>)((PlanePtr<char>)base + o * (unsigned)sizeof(T));
}

// compute_Sij at interior cell (i, j, k) with o = i + sx j: diagonal terms at
// the centre, the off-diagonal terms averaged from the four surrounding edges;
// returns |S|.
template <class T>
__device__ __forceinline__ double strain(const Dims &d, const Metrics &m, const StrainMet &sm,
                                         const T *__restrict__ U, const T *__restrict__ V, const T *__restrict__ W,
                                         unsigned o, int k, double s[6]) {
    const unsigned sx = d.sx;
    const double rz0 = m.rdzg[k - 1], rz1 = m.rdzg[k];
    // planes k-1, k, k+1 (of W: k-1 and k)
    const PlanePtr<T> Uc = plane_ptr(U + k * d.sxy), Vc = plane_ptr(V + k * d.sxy), Wc = plane_ptr(W + k * d.sxy);
    const PlanePtr<T> Um = plane_ptr(U + (k - 1) * d.sxy), Up = plane_ptr(U + (k + 1) * d.sxy);
    const PlanePtr<T> Vm = plane_ptr(V + (k - 1) * d.sxy), Vp = plane_ptr(V + (k + 1) * d.sxy);
    const PlanePtr<T> Wm = plane_ptr(W + (k - 1) * d.sxy);
    s[0] = (at<T>(Uc, o) - at<T>(Uc, o - 1)) * sm.rdx;
    s[1] = (at<T>(Vc, o) - at<T>(Vc, o - sx)) * sm.rdy;
    s[2] = (at<T>(Wc, o) - at<T>(Wm, o)) * m.rdz[k];
    // edges (i + a, j + b, k), (i + a, j, k + c), (i, j + b, k + c)
    auto e4 = [&](int a, int b) {
        const unsigned q = o + a + (b ? sx : 0u);
        return 0.5 * ((at<T>(Uc, q - 1) - at<T>(Uc, q - 1 - sx)) * (b ? sm.rdyg1 : sm.rdyg0) +
                      (at<T>(Vc, q - sx) - at<T>(Vc, q - 1 - sx)) * (a ? sm.rdxg1 : sm.rdxg0));
    };
    auto e5 = [&](int a, int c) {
        const unsigned q = o + a;
        const PlanePtr<T> Wq = c ? Wc : Wm;
        return 0.5 * ((at<T>(c ? Up : Uc, q - 1) - at<T>(c ? Uc : Um, q - 1)) * (c ? rz1 : rz0) +
                      (at<T>(Wq, q) - at<T>(Wq, q - 1)) * (a ? sm.rdxg1 : sm.rdxg0));
    };
    auto e6 = [&](int b, int c) {
        const unsigned q = o + (b ? sx : 0u);
        const PlanePtr<T> Wq = c ? Wc : Wm;
        return 0.5 * ((at<T>(c ? Vp : Vc, q - sx) - at<T>(c ? Vc : Vm, q - sx)) * (c ? rz1 : rz0) +
                      (at<T>(Wq, q) - at<T>(Wq, q - sx)) * (b ? sm.rdyg1 : sm.rdyg0));
    };
    s[3] = 0.25 * (e4(0, 0) + e4(1, 0) + e4(0, 1) + e4(1, 1));
    s[4] = 0.25 * (e5(0, 0) + e5(1, 0) + e5(0, 1) + e5(1, 1));
    s[5] = 0.25 * (e6(0, 0) + e6(1, 0) + e6(0, 1) + e6(1, 1));
    double a = 0.0;
#pragma unroll
    for (int c = 0; c < 6; ++c) a = a + (c < 3 ? 2.0 : 4.0) * s[c] * s[c];
    return sqrt(a);
}

// filter_xzy (subgrid.f90:140-187) is separable: its xz weights (4/9, 1/9,
// 1/36; :163-173) are the products of (1/6, 2/3, 1/6) in x and in z, and the
// y part is (1/6, 2/3, 1/6), one-sided (2/3, 1/3) at the ends of a section
// (:179-181).
constexpr double kF0 = 2.0 / 3.0, kF1 = 1.0 / 6.0;

struct YWeights {
    double m, c, p;  // rows j-1, j, j+1
};
__device__ __forceinline__ YWeights yweights(int j, int jlo, int jhi) {
    if (j == jlo) return {0.0, 2.0 / 3.0, 1.0 / 3.0};
    if (j == jhi) return {1.0 / 3.0, 2.0 / 3.0, 0.0};
    return {kF1, kF0, kF1};
}

// the x and y parts of filter_xzy at (ic, j), o = ic + sx j, of a plane of a
// face array with rows 0..jhi
template <class T>
__device__ __forceinline__ double filt_xy(PlanePtr<T> F, unsigned o, unsigned sx, int j, int jhi,
                                          const YWeights &w) {
    // all nine loads before the first use (rows past the section's ends are
    // read from its end row and their terms left out)
    const unsigned lo = j == 0 ? o : o - sx, hi = j == jhi ? o : o + sx;
    double r[3][3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        r[a][0] = at<T>(F, lo + a - 1);
        r[a][1] = at<T>(F, o + a - 1);
        r[a][2] = at<T>(F, hi + a - 1);
    }
    auto col = [&](int a) {
        const double c = w.c * r[a][1];
        const double b = j == 0 ? c : w.m * r[a][0] + c;
        return j == jhi ? b : b + w.p * r[a][2];
    };
    return kF1 * col(0) + kF0 * col(1) + kF1 * col(2);
}

// Uf, Vf, Wf with their x fixes, marching over the z centres of a chunk so that
// each plane is filtered in x and y once and the z part works on registers
// (27 instead of 81 loads per cell).  The ghost and duplicated planes are
// copies of centres 1, 2 and nzg-3, written with them.
template <bool PX, class T>
__global__ __launch_bounds__(256) void k_dsm_vfilter(Dims d, const T *__restrict__ U, const T *__restrict__ V,
                                                     const T *__restrict__ W, double *__restrict__ Uf,
                                                     double *__restrict__ Vf, double *__restrict__ Wf, int chunk) {
    const int i = blockIdx.x * 64 + (threadIdx.x & 63);
    const int j = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (i >= d.nxg || j >= d.nyg) return;
    const int kb = 1 + blockIdx.z * chunk, ke = min(kb + chunk, d.nzg - 2);  // centres 1..nzg-3
    const int iu = xmap_f<PX>(d, min(i, d.nx - 1)), ic = xmap_c<PX>(d, i);
    const int jv = min(j, d.ny - 1);
    const YWeights wu = yweights(j, 0, d.nyg - 1), wv = yweights(jv, 0, d.ny - 1);
    const unsigned sx = d.sx, ou = iu + sx * j, ov = ic + sx * jv, ow = ic + sx * j;
    auto plane = [&](int k, double f[3]) {
        f[0] = filt_xy<T>(plane_ptr(U + k * d.sxy), ou, sx, j, d.nyg - 1, wu);
        f[1] = filt_xy<T>(plane_ptr(V + k * d.sxy), ov, sx, jv, d.ny - 1, wv);
        f[2] = filt_xy<T>(plane_ptr(W + k * d.sxy), ow, sx, j, d.nyg - 1, wu);
    };
    double a[3], b[3], c[3];
    plane(kb - 1, a);
    plane(kb, b);
    for (int k = kb; k < ke; ++k) {
        plane(k + 1, c);
        double f[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) f[q] = kF1 * a[q] + kF0 * b[q] + kF1 * c[q];
        auto put = [&](int kk) {
            const long long p = fidx(d, i, j, kk);
            if (i < d.nx) Uf[p] = f[0];
            if (j < d.ny) Vf[p] = f[1];
            if (kk < d.nz) Wf[p] = f[2];
        };
        put(k);
        if (k == d.nzg - 3) put(0);
        if (k == 1) put(d.nzg - 2);
        if (k == 2) {  // W has no plane nzg-1
            const long long p = fidx(d, i, j, d.nzg - 1);
            if (i < d.nx) Uf[p] = f[0];
            if (j < d.ny) Vf[p] = f[1];
        }
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            a[q] = b[q];
            b[q] = c[q];
        }
    }
}

// L:M and M:M.  A block owns 30 x 6 cells and a chunk of z planes and marches
// in z.  Each of its 256 threads forms, at its cell of the tile with a
// one-cell halo (32 x 8), the centred velocities, |S| and |S| S_ij of a plane
// from the fields and leaves nine values in LDS (three more where a ghost
// index is read unmapped); the threads of the inner cells then filter the
// three velocities, six products and six |S| S_ij in x and y from LDS and in z
// through two running values per quantity in registers.  Nothing but |S| and
// the two sums per column and chunk goes to memory.  The work is FP64
// arithmetic and LDS reads (81 per cell), two blocks per CU by its registers.
// At 257x97x64 in FP32 fields the model's three passes take 0.024 + 0.153 +
// 0.011 ms per stage; the form in which every cell read the 27 neighbours of
// twelve FP64 arrays written by other passes took 0.04 + 0.07 + 0.53 + 0.05.
constexpr int kDsX = 32, kDsY = 8;  // tile with its halo

template <bool PX, class T>
__global__ __launch_bounds__(256) void k_dsm_stress(Dims d, Metrics m, const T *__restrict__ U,
                                                    const T *__restrict__ V, const T *__restrict__ W,
                                                    const double *__restrict__ Uf, const double *__restrict__ Vf,
                                                    const double *__restrict__ Wf, double *__restrict__ S,
                                                    double *__restrict__ part, int chunk) {
    __shared__ double sq[12][kDsX * kDsY];  // 0-2 centred velocities, 3-8 |S| S_ij (mapped), 9-11 velocities unmapped
    const int tid = threadIdx.x, tx = tid % kDsX, ty = tid / kDsX;
    const int nbx = (d.nxg - 2 + kDsX - 3) / (kDsX - 2);
    const int bx = blockIdx.x % nbx, by = blockIdx.x / nbx;
    const int i = min(bx * (kDsX - 2) + tx, d.nxg - 1), j = min(by * (kDsY - 2) + ty, d.nyg - 1);
    const int im = xmap_c<PX>(d, i);
    const bool row = j >= 1 && j <= d.nyg - 2;  // rows 0 and nyg-1 have weight 0 and no value
    const bool own = tx >= 1 && tx <= kDsX - 2 && ty >= 1 && ty <= kDsY - 2 && row && bx * (kDsX - 2) + tx <= d.nxg - 2 &&
                     by * (kDsY - 2) + ty <= d.nyg - 2;
    // whether some cell of the tile has an x ghost index
    const bool xghost = bx == 0 || bx * (kDsX - 2) + kDsX - 1 >= d.nxg - 2;
    const int jc = max(1, min(j, d.nyg - 2));
    const StrainMet sm = strain_met(m, im, jc);  // im = i at the cells whose results are used
    const YWeights w = yweights(jc, 1, d.nyg - 2);
    const int kb = 1 + blockIdx.y * chunk, ke = min(kb + chunk, d.nzg - 2);  // planes 1..nzg-3
    const long long sxy = d.sxy;
    const unsigned sx = d.sx, oi = i + sx * j, om = im + sx * j;
    double last[15], pend[15], lmsum = 0.0, mmsum = 0.0, magp = 0.0;
#pragma unroll
    for (int q = 0; q < 15; ++q) last[q] = pend[q] = 0.0;
    for (int kk = kb - 1; kk <= ke; ++kk) {
        const int km = zmap_c(d, kk);
        const bool ghost = xghost || km != kk;
        double v[12], mag = 0.0;
#pragma unroll
        for (int q = 0; q < 12; ++q) v[q] = 0.0;
        if (row) {
            double s[6];
            const PlanePtr<T> Uk = plane_ptr(U + km * sxy), Vk = plane_ptr(V + km * sxy), Wk = plane_ptr(W + km * sxy);
            const PlanePtr<T> Wb = plane_ptr(W + (km - 1) * sxy);
            v[0] = 0.5 * (at<T>(Uk, om - 1) + at<T>(Uk, om));
            v[1] = 0.5 * (at<T>(Vk, om - sx) + at<T>(Vk, om));
            v[2] = 0.5 * (at<T>(Wb, om) + at<T>(Wk, om));
            mag = strain(d, m, sm, U, V, W, om, km, s);
#pragma unroll
            for (int c = 0; c < 6; ++c) v[3 + c] = mag * s[c];
            if (ghost) {
                const PlanePtr<T> Ug = plane_ptr(U + kk * sxy), Vg = plane_ptr(V + kk * sxy);
                v[9] = 0.5 * (at<T>(Ug, om - 1) + at<T>(Ug, om));
                v[10] = 0.5 * (at<T>(Vg, oi - sx) + at<T>(Vg, oi));
                v[11] = 0.5 * (at<T>(Wb, oi) + at<T>(Wk, oi));
            }
            if (own && !PX) {
                // nu_t reads |S| on planes 1..nzg-2, the duplicated plane's own value among them
                if (kk >= kb && kk < ke)
                    S[kk * sxy + oi] = mag;
                else if (kk == d.nzg - 2)
                    S[kk * sxy + oi] = strain(d, m, sm, U, V, W, oi, kk, s);
            }
        }
        __syncthreads();  // the previous plane is read
#pragma unroll
        for (int q = 0; q < 9; ++q) sq[q][tid] = v[q];
        if (ghost)
#pragma unroll
            for (int q = 9; q < 12; ++q) sq[q][tid] = v[q];
        __syncthreads();
        if (own) {
            auto filt_row = [&](double q0, double q1, double q2) { return w.m * q0 + w.c * q1 + w.p * q2; };
            // the z part: the plane kk - 1 of quantity q is complete with this
            // plane's value f
            auto zstep = [&](int q, double f) {
                const double h = pend[q] + kF1 * f;
                pend[q] = kF1 * last[q] + kF0 * f;
                last[q] = f;
                return h;
            };
            auto filt_lds = [&](const double *Q) {
                double c[3];
#pragma unroll
                for (int a = 0; a < 3; ++a) c[a] = filt_row(Q[tid + a - 1 - kDsX], Q[tid + a - 1], Q[tid + a - 1 + kDsX]);
                return kF1 * c[0] + kF0 * c[1] + kF1 * c[2];
            };
            // one group of quantities at a time: with all 81 LDS reads in
            // flight the kernel took 390 registers
            double L[6], hs[6];
            {
                double f[6];
#pragma unroll
                for (int c = 0; c < 6; ++c) f[c] = 0.0;
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    double x[3], y[3], z[3];
#pragma unroll
                    for (int r = 0; r < 3; ++r) {
                        const int e = tid + a - 1 + (r - 1) * kDsX;
                        x[r] = sq[0][e];
                        y[r] = sq[1][e];
                        z[r] = sq[2][e];
                    }
                    const double wx = a == 1 ? kF0 : kF1;
                    f[0] += wx * filt_row(x[0] * x[0], x[1] * x[1], x[2] * x[2]);
                    f[1] += wx * filt_row(y[0] * y[0], y[1] * y[1], y[2] * y[2]);
                    f[2] += wx * filt_row(z[0] * z[0], z[1] * z[1], z[2] * z[2]);
                    f[3] += wx * filt_row(x[0] * y[0], x[1] * y[1], x[2] * y[2]);
                    f[4] += wx * filt_row(x[0] * z[0], x[1] * z[1], x[2] * z[2]);
                    f[5] += wx * filt_row(y[0] * z[0], y[1] * z[1], y[2] * z[2]);
                    __builtin_amdgcn_sched_barrier(0);
                }
                const int uo = ghost ? 9 : 0;
                double h[3];
#pragma unroll
                for (int c = 0; c < 3; ++c) h[c] = zstep(c, filt_lds(sq[uo + c]));
#pragma unroll
                for (int c = 0; c < 6; ++c) L[c] = zstep(3 + c, f[c]);
                L[0] -= h[0] * h[0];
                L[1] -= h[1] * h[1];
                L[2] -= h[2] * h[2];
                L[3] -= h[0] * h[1];
                L[4] -= h[0] * h[2];
                L[5] -= h[1] * h[2];
            }
#pragma unroll
            for (int c = 0; c < 6; ++c) {
                __builtin_amdgcn_sched_barrier(0);
                hs[c] = zstep(9 + c, filt_lds(sq[3 + c]));
            }
            __builtin_amdgcn_sched_barrier(0);
            if (kk > kb) {  // plane k = kk - 1 has its three planes
                const int k = kk - 1;
                double M[6];
                const double magh = strain(d, m, sm, Uf, Vf, Wf, oi, k, M);
#pragma unroll
                for (int e = 0; e < 6; ++e) M[e] = 4.0 * magh * M[e] - hs[e];
                double lm = M[0] * L[0];
                lm = lm + M[1] * L[1];
                lm = lm + M[2] * L[2];
                lm = lm + 2.0 * M[3] * L[3];
                lm = lm + 2.0 * M[4] * L[4];
                lm = lm + 2.0 * M[5] * L[5];
                const double mm = M[0] * M[0] + M[1] * M[1] + M[2] * M[2] +
                                  2.0 * (M[3] * M[3] + M[4] * M[4] + M[5] * M[5]);
                if constexpr (PX) {
                    S[k * sxy + oi] = fmax(-0.5 * (lm / mm) * magp, 0.0);
                } else {
                    lmsum += lm;
                    mmsum += mm;
                }
            }
            magp = mag;
        }
    }
    if (!PX && own) {
        double *o = part + 2 * (long long)blockIdx.y * sxy + oi;
        o[0] = lmsum;
        o[sxy] = mmsum;
    }
}

// nu_t of planes kColPlanes blockIdx.z .. from |S| and the column's mean
// ratio; every thread adds the column's nch chunk sums in the same order
constexpr int kColPlanes = 8;
template <class T>
__global__ __launch_bounds__(256) void k_dsm_column(Dims d, const double *__restrict__ S,
                                                    const double *__restrict__ part, int nch, int dirichlet,
                                                    T *__restrict__ nu_t) {
    const int i = blockIdx.x * 64 + (threadIdx.x & 63);
    const int j = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (i >= d.nxg || j >= d.nyg) return;
    const int k0 = blockIdx.z * kColPlanes, k1 = min(k0 + kColPlanes, d.nzg);
    const bool ghost_y = (j == 0 || j == d.nyg - 1);
    const int js = j == 0 ? 1 : (j == d.nyg - 1 ? d.nyg - 2 : j);
    const double sgn = (ghost_y && dirichlet == 1) ? -1.0 : 1.0;
    const bool ghost_x = i == 0 || i == d.nxg - 1;
    double avg = 0.0;
    if (!ghost_x) {
        double slm = 0.0, smm = 0.0;
        const double *q = part + i + (long long)d.sx * js;
        for (int c = 0; c < nch; ++c) {
            slm += q[2 * c * d.sxy];
            smm += q[(2 * c + 1) * d.sxy];
        }
        const double nz3 = (double)(d.nzg - 3);
        avg = (slm / nz3) / (smm / nz3);
    }
    for (int k = k0; k < k1; ++k) {
        const bool zero = ghost_x || k == 0 || k == d.nzg - 1;
        nu_t[fidx(d, i, j, k)] = (T)(sgn * (zero ? 0.0 : fmax(-0.5 * avg * S[fidx(d, i, js, k)], 0.0)));
    }
}

// LES = 3: the values of k_dsm_stress with the periodic x and z copies and
// the y ghost rows from rows 1 and nyg-2 (subgrid.f90:571-581)
template <class T>
__global__ __launch_bounds__(256) void k_dsm_cellwise(Dims d, const double *__restrict__ nt, int dirichlet,
                                                      T *__restrict__ nu_t) {
    const int i = blockIdx.x * 64 + (threadIdx.x & 63);
    const int j = blockIdx.y * 4 + (threadIdx.x >> 6);
    const int k = blockIdx.z;
    if (i >= d.nxg || j >= d.nyg) return;
    const bool ghost_y = (j == 0 || j == d.nyg - 1);
    const int js = j == 0 ? 1 : (j == d.nyg - 1 ? d.nyg - 2 : j);
    const double sgn = (ghost_y && dirichlet == 1) ? -1.0 : 1.0;
    nu_t[fidx(d, i, j, k)] = (T)(sgn * nt[fidx(d, xmap_c<true>(d, i), js, zmap_c(d, k))]);
}

// LES = 1: nu_t = coef[j] |S| on the interior cells, coef[j] = (Cs Delta_j
// f_j)^2 from the host; the ghost entries are left as they are
template <class T>
__global__ __launch_bounds__(256) void k_smag(Dims d, Metrics m, const T *__restrict__ U, const T *__restrict__ V,
                                              const T *__restrict__ W, const double *__restrict__ coef,
                                              T *__restrict__ nu_t) {
    const int i = 1 + blockIdx.x * 64 + (threadIdx.x & 63);
    const int j = 1 + blockIdx.y * 4 + (threadIdx.x >> 6);
    const int k = 1 + blockIdx.z;
    if (i > d.nxg - 2 || j > d.nyg - 2) return;
    double s[6];
    const double mag = strain(d, m, strain_met(m, i, j), U, V, W, (unsigned)(i + d.sx * j), k, s);
    nu_t[fidx(d, i, j, k)] = (T)(coef[j] * mag);
}

void check() {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        last_error() = std::string("kernel launch: ") + hipGetErrorString(e);
        throw DeviceError();
    }
}

// z chunk length of a marching pass over nk planes with `tiles` column tiles,
// of which `slots` blocks are resident at a time: the one with the fewest plane
// steps in sequence, rounds of blocks times (chunk + 2), since a chunk also
// forms the plane before and the plane behind it.  At 257x97x64 (144 tiles, 512
// slots) that is 9 planes, two full rounds, against 8 planes in 2.25 rounds.
int dsm_chunk(int nk, int tiles, int slots) {
    int best = nk;
    long long cost = -1;
    for (int chunk = nk; chunk >= 1; --chunk) {
        const long long blocks = (long long)tiles * ((nk + chunk - 1) / chunk);
        const long long c = (blocks + slots - 1) / slots * (chunk + 2);
        if (cost < 0 || c < cost) {
            cost = c;
            best = chunk;
        }
    }
    return best;
}
// resident blocks per compute unit, by their registers
constexpr int kStressPerCU = 2, kVfilterPerCU = 4;
int stress_tiles(const Dims &d) {
    return ((d.nxg - 2 + kDsX - 3) / (kDsX - 2)) * ((d.nyg - 2 + kDsY - 3) / (kDsY - 2));
}

template <bool PX, class T>
void dsm_t(Handle &h, const Fld3<T> &f, T *nu_t) {
    const Dims &d = h.d;
    const long long nf = d.sxy * d.nzg;
    const dim3 block(256);
    const int nk = d.nzg - 3;
    double *S = h.dsm + D_S * nf, *Uf = h.dsm + D_UF * nf, *Vf = h.dsm + D_VF * nf, *Wf = h.dsm + D_WF * nf;
    double *part = h.dsm + D_END * nf;
    const dim3 gcol((d.nxg + 63) / 64, (d.nyg + 3) / 4);
    {
        ProfScope ps(h, KID_DSM_VFILTER);
        const int chunk = dsm_chunk(nk, gcol.x * gcol.y, kVfilterPerCU * h.n_cu);
        hipLaunchKernelGGL((k_dsm_vfilter<PX, T>), dim3(gcol.x, gcol.y, (nk + chunk - 1) / chunk), block, 0, h.stream,
                           d, f.u, f.v, f.w, Uf, Vf, Wf, chunk);
        check();
    }
    const int tiles = stress_tiles(d);
    const int chunk = dsm_chunk(nk, tiles, kStressPerCU * h.n_cu), nch = (nk + chunk - 1) / chunk;
    {
        ProfScope ps(h, KID_DSM_FILTER);
        hipLaunchKernelGGL((k_dsm_stress<PX, T>), dim3(tiles, nch), block, 0, h.stream, d, h.m, f.u, f.v, f.w, Uf, Vf,
                           Wf, S, part, chunk);
        check();
    }
    {
        ProfScope ps(h, KID_DSM_COLUMN);
        if constexpr (PX)
            hipLaunchKernelGGL(k_dsm_cellwise<T>, dim3(gcol.x, gcol.y, d.nzg), block, 0, h.stream, d, S, h.nut_bc,
                               nu_t);
        else
            hipLaunchKernelGGL(k_dsm_column<T>, dim3(gcol.x, gcol.y, (d.nzg + kColPlanes - 1) / kColPlanes), block, 0,
                               h.stream, d, S, part, nch, h.nut_bc, nu_t);
        check();
    }
}

template <class T>
void smag_t(Handle &h, const Fld3<T> &f, T *nu_t) {
    const Dims &d = h.d;
    ProfScope ps(h, KID_DSM_CELLS);
    const dim3 g((d.nxg - 2 + 63) / 64, (d.nyg - 2 + 3) / 4, d.nzg - 2);
    hipLaunchKernelGGL(k_smag<T>, g, dim3(256), 0, h.stream, d, h.m, f.u, f.v, f.w, (const double *)h.smag_c, nu_t);
    check();
}

template <class T>
void eddy_t(Handle &h, const Fld3<T> &f, T *nu_t) {
    if (h.les == 1)
        smag_t(h, f, nu_t);
    else if (h.les == 3)
        dsm_t<true>(h, f, nu_t);
    else
        dsm_t<false>(h, f, nu_t);
}

}  // namespace

size_t dsm_doubles(const Handle &h) {
    const Dims &d = h.d;
    const int nk = d.nzg - 3, chunk = dsm_chunk(nk, stress_tiles(d), kStressPerCU * h.n_cu);
    return (size_t)d.sxy * ((size_t)D_END * d.nzg + 2 * (size_t)((nk + chunk - 1) / chunk));
}

void launch_dsm(Handle &h, const Field3 &f) {
    if (h.precision == BL_PREC_MIXED)
        eddy_t(h, as<float>(f), reinterpret_cast<float *>(h.nu_t));
    else
        eddy_t(h, as<double>(f), h.nu_t);
}

}  // namespace blgpu
