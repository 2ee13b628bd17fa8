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

// A plane as a buffer resource: an element is a scalar base, one register with
// the byte offset of a cell's south-west neighbour (shared by all arrays of one
// element size), a scalar row offset and an immediate column offset.
template <class T>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t plane_rsrc(const Dims &d, const T *p, long long k) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)(p + k * d.sxy), 0, (int)(unsigned)(d.sxy * sizeof(T)), 0x00020000);
}
template <class T>
__device__ __forceinline__ T buf_at(__amdgpu_buffer_rsrc_t r, unsigned sw, unsigned row, int col) {
    if constexpr (sizeof(T) == 4)
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, sw + col * 4, row, 0));
    else
        return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, sw + col * 8, row, 0));
}

// compute_Sij along z at one column of cells: diagonal terms at the centre, the
// off-diagonal terms averaged from the four surrounding edges.  A cell needs U at
// two points of five rows or planes, V likewise and W at five points of two
// planes; what the next plane uses again stays in
// registers (17 loads a plane instead of 30).  All loads of a plane are issued
// together by load(); eval() uses them.
template <class T>
struct StrainMarch {
    T u[2], v[2];          // plane k: U(i-1), U(i); V(j-1), V(j)
    T um[2], vm[2], wm[5];  // plane k-1; W at the cell, i-1, i+1, j-1, j+1
    T us[2], un[2], ve[2], vw[2], up[2], vp[2], w[5];

    __device__ __forceinline__ static void load_u(const Dims &d, const T *U, unsigned sw, int k, T o[2]) {
        const unsigned sxb = (unsigned)(d.sx * sizeof(T));
        const auto r = plane_rsrc(d, U, k);
        o[0] = buf_at<T>(r, sw, sxb, 0);
        o[1] = buf_at<T>(r, sw, sxb, 1);
    }
    __device__ __forceinline__ static void load_v(const Dims &d, const T *V, unsigned sw, int k, T o[2]) {
        const unsigned sxb = (unsigned)(d.sx * sizeof(T));
        const auto r = plane_rsrc(d, V, k);
        o[0] = buf_at<T>(r, sw, 0, 1);
        o[1] = buf_at<T>(r, sw, sxb, 1);
    }
    __device__ __forceinline__ static void load_w(const Dims &d, const T *W, unsigned sw, int k, T o[5]) {
        const unsigned sxb = (unsigned)(d.sx * sizeof(T));
        const auto r = plane_rsrc(d, W, k);
        o[0] = buf_at<T>(r, sw, sxb, 1);
        o[1] = buf_at<T>(r, sw, sxb, 0);
        o[2] = buf_at<T>(r, sw, sxb, 2);
        o[3] = buf_at<T>(r, sw, 0, 1);
        o[4] = buf_at<T>(r, sw, 2 * sxb, 1);
    }
    // what plane k takes from planes k-1 and k, at the start and where k jumps
    __device__ __forceinline__ void begin(const Dims &d, const T *U, const T *V, const T *W, unsigned sw, int k) {
        load_u(d, U, sw, k, u);
        load_v(d, V, sw, k, v);
        load_u(d, U, sw, k - 1, um);
        load_v(d, V, sw, k - 1, vm);
        load_w(d, W, sw, k - 1, wm);
    }
    __device__ __forceinline__ void load(const Dims &d, const T *U, const T *V, const T *W, unsigned sw, int k) {
        const unsigned sxb = (unsigned)(d.sx * sizeof(T));
        const auto ru = plane_rsrc(d, U, k), rv = plane_rsrc(d, V, k);
        us[0] = buf_at<T>(ru, sw, 0, 0);
        us[1] = buf_at<T>(ru, sw, 0, 1);
        un[0] = buf_at<T>(ru, sw, 2 * sxb, 0);
        un[1] = buf_at<T>(ru, sw, 2 * sxb, 1);
        vw[0] = buf_at<T>(rv, sw, 0, 0);
        vw[1] = buf_at<T>(rv, sw, sxb, 0);
        ve[0] = buf_at<T>(rv, sw, 0, 2);
        ve[1] = buf_at<T>(rv, sw, sxb, 2);
        load_w(d, W, sw, k, w);
        load_u(d, U, sw, k + 1, up);
        load_v(d, V, sw, k + 1, vp);
    }
    // S_ij and |S| of plane k, the centred velocities too where asked for
    __device__ __forceinline__ double eval(const Metrics &m, const StrainMet &sm, int k, double s[6],
                                           double *c = nullptr) {
        const double rz0 = m.rdzg[k - 1], rz1 = m.rdzg[k];
        // the four edges around the cell (twice their value): the pair b of one
        // component against the pairs before (a) and behind (e) it along one
        // direction, and the other component's pair along the other, in the
        // reference's order
        auto edges = [](const T a[2], const T b[2], const T e[2], double ra, double re, const T f[2], const T g[2],
                        const T h[2], double rf, double rh) {
            auto dif = [](T p, T q) { return (double)p - (double)q; };
            return ((dif(b[0], a[0]) * ra + dif(g[0], f[0]) * rf) + (dif(b[1], a[1]) * ra + dif(h[0], g[0]) * rh)) +
                   (dif(e[0], b[0]) * re + dif(g[1], f[1]) * rf) + (dif(e[1], b[1]) * re + dif(h[1], g[1]) * rh);
        };
        const T wc[2] = {wm[0], w[0]}, ww[2] = {wm[1], w[1]}, we[2] = {wm[2], w[2]}, ws[2] = {wm[3], w[3]},
                wn[2] = {wm[4], w[4]};
        s[0] = ((double)u[1] - (double)u[0]) * sm.rdx;
        s[1] = ((double)v[1] - (double)v[0]) * sm.rdy;
        s[2] = ((double)w[0] - (double)wm[0]) * m.rdz[k];
        s[3] = 0.125 * edges(us, u, un, sm.rdyg0, sm.rdyg1, vw, v, ve, sm.rdxg0, sm.rdxg1);
        s[4] = 0.125 * edges(um, u, up, rz0, rz1, ww, wc, we, sm.rdxg0, sm.rdxg1);
        s[5] = 0.125 * edges(vm, v, vp, rz0, rz1, ws, wc, wn, sm.rdyg0, sm.rdyg1);
        if (c) {
            c[0] = 0.5 * ((double)u[0] + (double)u[1]);
            c[1] = 0.5 * ((double)v[0] + (double)v[1]);
            c[2] = 0.5 * ((double)wm[0] + (double)w[0]);
        }
        double a = 0.0;
#pragma unroll
        for (int q = 0; q < 6; ++q) a = a + (q < 3 ? 2.0 : 4.0) * s[q] * s[q];
        return sqrt(a);
    }
    __device__ __forceinline__ void next() {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            um[q] = u[q];
            vm[q] = v[q];
            u[q] = up[q];
            v[q] = vp[q];
        }
#pragma unroll
        for (int q = 0; q < 5; ++q) wm[q] = w[q];
    }
};
// byte offset of the south-west neighbour of (i, j), i, j >= 1
template <class T>
__device__ __forceinline__ unsigned sw_offset(const Dims &d, int i, int j) {
    return (unsigned)(i - 1 + (int)d.sx * (j - 1)) * (unsigned)sizeof(T);
}
template <class T>
__device__ __forceinline__ double strain(const Dims &d, const Metrics &m, const StrainMet &sm, const T *U, const T *V,
                                         const T *W, int i, int j, int k, double s[6]) {
    StrainMarch<T> q;
    const unsigned sw = sw_offset<T>(d, i, j);
    q.begin(d, U, V, W, sw, k);
    q.load(d, U, V, W, sw, k);
    return q.eval(m, sm, k, s);
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
__global__ __launch_bounds__(256, vfilter_resident<T>()) void k_dsm_vfilter(
    Dims d, const T *__restrict__ U, const T *__restrict__ V, const T *__restrict__ W, double *__restrict__ Uf,
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
// in z with two kinds of waves.  Four waves form, at each cell of the tile with a
// one-cell halo (32 x 8), the centred velocities, |S| and |S| S_ij of a plane and
// the filtered field's 4 |S^| S^_ij of the plane before and leave them in LDS (three
// more values where a ghost index is read unmapped).  Three waves, one thread
// per cell of the six inner rows, filter the three velocities, six products and
// six |S| S_ij of the other buffer in y from LDS, in x between lanes and in z
// through two running values per quantity in registers, and contract.  Nothing
// but |S| and the two sums per column and chunk goes to memory.  Bound by
// issue: FP64 arithmetic with two blocks (14 waves) per CU; 120 registers in FP32
// fields, in FP64 fields all 128 and 60 bytes a lane spilled.
// At 257x97x64 in FP32 fields the model's three passes take 0.022 + 0.064 +
// 0.010 ms per stage.  With all steps in four waves, filters of 9 LDS reads and
// plain loads, which waited one after the other, the middle one took 0.153;
// the form in which every cell read the 27 neighbours of twelve FP64 arrays
// written by other passes took 0.04 + 0.07 + 0.53 + 0.05.  Tiles of 32 x 16
// measured the same (0.063), loads of the filtered field a plane ahead 0.093
// (registers).
constexpr int kDsX = 32, kDsY = 8;  // tile with its halo

constexpr int kDsOwn = kDsX * (kDsY - 2);  // threads of the second role: its inner rows

// the value of the lane one below (-1) or above (+1), its two halves by DPP
template <int D>
__device__ __forceinline__ double lane_shift(double x) {
    const int2 v = __builtin_bit_cast(int2, x);
    constexpr int ctl = D < 0 ? 0x138 : 0x130;  // wave_shr:1, wave_shl:1
    const int2 r = {__builtin_amdgcn_mov_dpp(v.x, ctl, 0xf, 0xf, true), __builtin_amdgcn_mov_dpp(v.y, ctl, 0xf, 0xf, true)};
    return __builtin_bit_cast(double, r);
}

template <bool PX, class T>
__global__ __launch_bounds__(kDsX *kDsY + kDsOwn, 4) void k_dsm_stress(
    Dims d, Metrics m, const T *__restrict__ U, const T *__restrict__ V, const T *__restrict__ W,
    const double *__restrict__ Uf, const double *__restrict__ Vf, const double *__restrict__ Wf, double *__restrict__ S,
    double *__restrict__ part, int chunk) {
    // per plane: 0-2 centred velocities, 3-8 |S| S_ij (both mapped), 9-11 velocities
    // unmapped where that differs; of the plane before: 12-17 4 |S^| S^_ij, 18 |S|
    __shared__ double sq[2][18 + PX][kDsX * kDsY];
    const int role = __builtin_amdgcn_readfirstlane(threadIdx.x >= kDsX * kDsY);
    const int nbx = (d.nxg - 2 + kDsX - 3) / (kDsX - 2);
    const int bx = blockIdx.x % nbx, by = blockIdx.x / nbx;
    // whether some cell of the tile has an x ghost index
    const bool xghost = bx == 0 || bx * (kDsX - 2) + kDsX - 1 >= d.nxg - 2;
    const int tid = role == 0 ? threadIdx.x : threadIdx.x - (kDsX * kDsY - kDsX), tx = tid % kDsX, ty = tid / kDsX;
    const int i = min(bx * (kDsX - 2) + tx, d.nxg - 1), j = min(by * (kDsY - 2) + ty, d.nyg - 1);
    const bool row = j >= 1 && j <= d.nyg - 2;  // rows 0 and nyg-1 have weight 0 and no value
    const bool own = tx >= 1 && tx <= kDsX - 2 && ty >= 1 && ty <= kDsY - 2 && row && bx * (kDsX - 2) + tx <= d.nxg - 2 &&
                     by * (kDsY - 2) + ty <= d.nyg - 2;
    const int jc = clampi(j, 1, d.nyg - 2);
    const int kb = 1 + blockIdx.y * chunk, ke = min(kb + chunk, d.nzg - 2);  // planes 1..nzg-3
    const long long sxy = d.sxy;
    const unsigned oi = i + (unsigned)d.sx * j;
    // Both roles make the same steps kk and pass the same barrier in each: behind
    // it the second reads the buffer that the first has left, the first fills the
    // other one, which the second has read before it.
    if (role == 0) {
        const int im = xmap_c<PX>(d, i), ic = clampi(i, 1, d.nxg - 2);
        // every lane's cell is inside, so that no load depends on a mask; im = i
        // at the cells whose results are used
        const unsigned swm = sw_offset<T>(d, im, jc), swf = sw_offset<double>(d, ic, jc);
        const unsigned south = (unsigned)(i + (int)d.sx * (jc - 1)) * (unsigned)sizeof(T);  // unmapped, row j-1
        const StrainMet sm = strain_met(m, im, jc);
        StrainMarch<T> a;
        StrainMarch<double> f;
        double mag1 = 0.0;
        a.begin(d, U, V, W, swm, zmap_c(d, kb - 1));
        a.load(d, U, V, W, swm, zmap_c(d, kb - 1));
        f.begin(d, Uf, Vf, Wf, swf, kb);
        for (int kk = kb - 1; kk <= ke; ++kk) {
            double(&o)[18 + PX][kDsX * kDsY] = sq[(kk - kb + 1) & 1];
            const int km = zmap_c(d, kk);
            double s[6], c[3];
            const double mag = a.eval(m, sm, km, s, c);
#pragma unroll
            for (int q = 0; q < 3; ++q) o[q][tid] = row ? c[q] : 0.0;
#pragma unroll
            for (int q = 0; q < 6; ++q) o[3 + q][tid] = row ? mag * s[q] : 0.0;
            if (xghost || km != kk) {  // U at the mapped x index
                const unsigned sxb = (unsigned)(d.sx * sizeof(T));
                const auto rv = plane_rsrc(d, V, kk), rw0 = plane_rsrc(d, W, km - 1), rw1 = plane_rsrc(d, W, km);
                T g[6];
                StrainMarch<T>::load_u(d, U, swm, kk, g);
                g[2] = buf_at<T>(rv, south, 0, 0);
                g[3] = buf_at<T>(rv, south, sxb, 0);
                g[4] = buf_at<T>(rw0, south, sxb, 0);
                g[5] = buf_at<T>(rw1, south, sxb, 0);
#pragma unroll
                for (int q = 0; q < 3; ++q) o[9 + q][tid] = row ? 0.5 * ((double)g[2 * q] + (double)g[2 * q + 1]) : 0.0;
            }
            // nu_t reads |S| on planes 1..nzg-2
            if (own && !PX && kk >= kb && kk < ke) S[kk * sxy + oi] = mag;
            if (kk > kb) f.load(d, Uf, Vf, Wf, swf, kk - 1);
            if (kk > kb) {
                const double magh = f.eval(m, sm, kk - 1, s);
#pragma unroll
                for (int q = 0; q < 6; ++q) o[12 + q][tid] = 4.0 * magh * s[q];
                if constexpr (PX) o[18][tid] = mag1;
                f.next();
            }
            mag1 = mag;
            __builtin_amdgcn_sched_barrier(0);
            a.next();
            if (kk < ke) {
                const int kn = zmap_c(d, kk + 1);
                if (kn != km + 1) a.begin(d, U, V, W, swm, kn);
                a.load(d, U, V, W, swm, kn);
            }
            __syncthreads();
        }
        if (!PX && own && ke == d.nzg - 2) {  // the duplicated plane's own value
            double s[6];
            S[ke * sxy + oi] = strain(d, m, sm, U, V, W, i, j, ke, s);
        }
    } else {
        const YWeights w = yweights(jc, 1, d.nyg - 2);
        double last[15], pend[15], lmsum = 0.0, mmsum = 0.0;
#pragma unroll
        for (int q = 0; q < 15; ++q) last[q] = pend[q] = 0.0;
        for (int kk = kb - 1; kk <= ke; ++kk) {
            const double(&o)[18 + PX][kDsX * kDsY] = sq[(kk - kb + 1) & 1];
            const bool ghost = xghost || zmap_c(d, kk) != kk;
            __syncthreads();
            auto filt_y = [&](double q0, double q1, double q2) { return w.m * q0 + w.c * q1 + w.p * q2; };
            auto filt_lds = [&](const double *Q) { return filt_y(Q[tid - kDsX], Q[tid], Q[tid + kDsX]); };
            // the x part between lanes (a tile row's first and last lane are not
            // its own), then the z part: the plane kk - 1 of quantity q is complete
            // with this plane's value
            auto xzstep = [&](int q, double g) {
                const double f = kF1 * lane_shift<-1>(g) + kF0 * g + kF1 * lane_shift<1>(g);
                const double h = pend[q] + kF1 * f;
                pend[q] = kF1 * last[q] + kF0 * f;
                last[q] = f;
                return h;
            };
            double L[6];
            {
                double x[3], y[3], z[3], h[3];
#pragma unroll
                for (int r = 0; r < 3; ++r) {
                    const int e = tid + (r - 1) * kDsX;
                    x[r] = o[0][e];
                    y[r] = o[1][e];
                    z[r] = o[2][e];
                }
                L[0] = xzstep(3, filt_y(x[0] * x[0], x[1] * x[1], x[2] * x[2]));
                L[1] = xzstep(4, filt_y(y[0] * y[0], y[1] * y[1], y[2] * y[2]));
                L[2] = xzstep(5, filt_y(z[0] * z[0], z[1] * z[1], z[2] * z[2]));
                L[3] = xzstep(6, filt_y(x[0] * y[0], x[1] * y[1], x[2] * y[2]));
                L[4] = xzstep(7, filt_y(x[0] * z[0], x[1] * z[1], x[2] * z[2]));
                L[5] = xzstep(8, filt_y(y[0] * z[0], y[1] * z[1], y[2] * z[2]));
                __builtin_amdgcn_sched_barrier(0);
                const int uo = ghost ? 9 : 0;
#pragma unroll
                for (int c = 0; c < 3; ++c) h[c] = xzstep(c, filt_lds(o[uo + c]));
                L[0] -= h[0] * h[0];
                L[1] -= h[1] * h[1];
                L[2] -= h[2] * h[2];
                L[3] -= h[0] * h[1];
                L[4] -= h[0] * h[2];
                L[5] -= h[1] * h[2];
            }
            double lm = 0.0, mm = 0.0, mo = 0.0;
#pragma unroll
            for (int c = 0; c < 6; ++c) {
                if (c % 2 == 0) __builtin_amdgcn_sched_barrier(0);
                const double M = o[12 + c][tid] - xzstep(9 + c, filt_lds(o[3 + c]));
                lm = lm + (c < 3 ? 1.0 : 2.0) * M * L[c];
                (c < 3 ? mm : mo) += M * M;
            }
            mm += 2.0 * mo;
            if (own && kk > kb) {  // plane k = kk - 1 has its three planes
                if constexpr (PX) {
                    S[(kk - 1) * sxy + oi] = fmax(-0.5 * (lm / mm) * o[18][tid], 0.0);
                } else {
                    lmsum += lm;
                    mmsum += mm;
                }
            }
        }
        if (!PX && own) {
            double *o = part + 2 * (long long)blockIdx.y * sxy + oi;
            o[0] = lmsum;
            o[sxy] = mmsum;
        }
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
    const double mag = strain(d, m, strain_met(m, i, j), U, V, W, i, j, k, s);
    nu_t[fidx(d, i, j, k)] = (T)(coef[j] * mag);
}

void check() {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        last_error() = std::string("kernel launch: ") + hipGetErrorString(e);
        throw DeviceError();
    }
}

int stress_tiles(const Dims &d) {
    return ((d.nxg - 2 + kDsX - 3) / (kDsX - 2)) * ((d.nyg - 2 + kDsY - 3) / (kDsY - 2));
}
int stress_chunk(const Handle &h, int nk) {
    return fewest_plane_steps(nk, stress_tiles(h.d), kStressResident * h.n_cu).planes;
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
        const int chunk = fewest_plane_steps(nk, gcol.x * gcol.y, vfilter_resident<T>() * h.n_cu, 6 * h.n_cu).planes;
        hipLaunchKernelGGL((k_dsm_vfilter<PX, T>), dim3(gcol.x, gcol.y, (nk + chunk - 1) / chunk), block, 0, h.stream,
                           d, f.u, f.v, f.w, Uf, Vf, Wf, chunk);
        check();
    }
    const int tiles = stress_tiles(d);
    const int chunk = stress_chunk(h, nk), nch = (nk + chunk - 1) / chunk;
    {
        ProfScope ps(h, KID_DSM_FILTER);
        hipLaunchKernelGGL((k_dsm_stress<PX, T>), dim3(tiles, nch), dim3(kDsX * kDsY + kDsOwn), 0, h.stream, d, h.m, f.u, f.v, f.w, Uf, Vf,
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
    const int nk = d.nzg - 3, chunk = stress_chunk(h, nk);
    return (size_t)d.sxy * ((size_t)D_END * d.nzg + 2 * (size_t)((nk + chunk - 1) / chunk));
}

void launch_dsm(Handle &h, const Field3 &f) {
    if (h.precision == BL_PREC_MIXED)
        eddy_t(h, as<float>(f), reinterpret_cast<float *>(h.nu_t));
    else
        eddy_t(h, as<double>(f), h.nu_t);
}

}  // namespace blgpu
