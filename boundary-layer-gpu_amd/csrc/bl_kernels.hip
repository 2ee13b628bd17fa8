// HIP kernels for the per-time-step path (gfx950, FP64 mode).
//
// Reference correspondence (0-based indices here, the reference is 1-based):
//   k_rk_march      equations.f90:24-415 fused with time_integration.f90:351-458
//   k_bc_*          boundary_conditions.f90:127-262
//   k_dct_*, k_zdft_*  the DCT-II/DFT stages of solve_poisson_gpu projection.f90:110-202,
//                   and in k_dct_fwd_m the divergence :34-49
//   k_thomas        projection.f90:137-150
//   k_project       projection.f90:355-386 with apply_periodic_z_pressure :293-303,
//                   and the P record of the first sub-step :75-85
//   reductions      projection.f90:391-413, statistics.f90:137-160, monitor.f90:29-52,
//                   time_integration.f90:546-558
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>
#include <vector>

#include "bl_internal.hpp"

namespace blgpu {

namespace {

constexpr int kWave = 64;

template <class T>
__device__ __forceinline__ T sq(T a) {
    return a * a;
}

// Accesses past the caches (NT: non-temporal) for values that a kernel touches
// once, where the arrays in use do not fit the caches anyway, so that they don't
// push out what is read again.
template <bool NT, class T>
__device__ __forceinline__ void put(T *p, T v) {
    if constexpr (NT)
        __builtin_nontemporal_store(v, p);
    else
        *p = v;
}
template <bool NT, class T>
__device__ __forceinline__ T get(const T *p) {
    if constexpr (NT) return __builtin_nontemporal_load(p);
    return *p;
}

// ------------------------------------------------------------------------
// Fused RHS + Runge-Kutta stage update, marching in z.
// MODE 0: new = old + c0*F              (first stage, and RK2 second stage;
//         FP64 RK3 stages 2 and 3 with old = G, below)
// MODE 1: new = old + dt*(c1*F1 + c0*F) (RK3 stages 2 and 3, FP32 fields)
// MODE 2: write F only (operator test)
// FOUT (first stage of RK3): 1 writes F1 = F; 2 writes G = old + g2*F
// instead (g2 = dt a21), so that stages 2 and 3 read one field per component
// instead of two (old and F1): a21 = a31 = 1/4 (initialization.f90:526,528)
// makes Uo + dt a21 F1 and Uo + dt a31 F1 the same field, and nothing
// writes G between stages 2 and 3.  A block owns a
// 64 (x) x 4 RPT (y) column of cells and a chunk of z planes; U and V of
// planes k, k+1 and W of planes k-1, k, k+1 live in an LDS ring with a
// one-cell halo in x and y (the stencil reads U and V of plane k-1 only at
// the cell itself, which each thread carries in registers from the previous
// plane), so every velocity value is read from HBM once per chunk (plus
// halo) instead of once per neighbour.  Loads are x-fastest and 512-byte
// aligned rows.  The x and y metrics of the tile are staged in LDS once:
// read from global memory inside each equation's branch they cost a load
// latency per branch and plane (2.69 -> 2.00 ms of RK stages per FP64 step,
// 1.71 -> 1.47 in FP32, at 814x257x193).  Thread (tx, ty) computes cells
// (i0+tx, j0+RPT ty+r), r < RPT.  FP64: 64 x 8 tiles (RPT = 2, 39.5 KB of
// LDS, 140 VGPRs: 3 blocks per CU; RPT = 1 took 16 % longer, and 4 blocks
// per CU forced by a 128-VGPR bound spilled and took 12 % longer); FP32:
// 64 x 12 tiles (RPT = 3, 27 KB; 64 x 16 tiles held 2 blocks per CU and
// took 3 % longer).  128-wide FP32 tiles (fewer x-halo lines) measured
// slower.
// ------------------------------------------------------------------------
// LES: the viscous terms use nu + nu_t (equations.f90:97-132, 231-270,
// 367-404); nu_t is staged in a fourth LDS ring.
template <int MODE, int FOUT, bool LES, bool NT, class T>
__global__ __launch_bounds__(256) void k_rk_march(
    Dims d, MetricsT<T> m, T nu, T dPdx, T dPdz, int kchunk,
    const T *__restrict__ U, const T *__restrict__ V, const T *__restrict__ W,
    const T *__restrict__ Nt,
    const T *__restrict__ Uo, const T *__restrict__ Vo, const T *__restrict__ Wo,
    const T *__restrict__ F1u, const T *__restrict__ F1v, const T *__restrict__ F1w,
    T *__restrict__ Un, T *__restrict__ Vn, T *__restrict__ Wn, T *__restrict__ Fou,
    T *__restrict__ Fov, T *__restrict__ Fow, T c0, T c1, T dt, T g2) {
    constexpr int RPT = MarchTile<T>::RPT, kTY = MarchTile<T>::TY, kPlane = MarchTile<T>::Plane;
    constexpr int kTX = MarchTile<T>::TX, kHX = MarchTile<T>::HX;
    // the halves of the averages are taken at the metrics, where scaling by a
    // power of two changes no bit of the product; FP32 fields keep the sum of the
    // three convective differences in FP64 and round it once (13 % fewer
    // instructions: 466 -> 453 us per stage at 814x257x193)
    constexpr T kHalf = 0.5, kQuarter = 0.25;
    // U and V: planes k and k+1 (their plane k-1 value at the thread's own
    // cells is carried in registers); W: planes k-1, k, k+1
    __shared__ T sU[2][kPlane], sV[2][kPlane], sW[3][kPlane];
    __shared__ T sN[LES ? 3 : 1][LES ? kPlane : 1];
    // the tile's x metrics (rdx(i), rdx(i+1), rdxg(i), rdxg(i-1)) and y metrics
    // (wy0(j), wy1(j), wy0(j-1), wy1(j-1), rdy(j), rdy(j+1), rdyg(j),
    // rdyg(j-1)): constant along the march, read from LDS with the velocities
    // instead of from global memory inside each equation's branch
    __shared__ T sMx[4][kTX], sMy[8][kTY];
    static_assert(!LES || sizeof(sU) + sizeof(sV) + sizeof(sW) + sizeof(sN) + sizeof(sMx) + sizeof(sMy) ==
                              march_lds<T>(LES), "the residency rule counts this");
    const int tid = threadIdx.x;
    const int tx = tid % kTX, ty = tid / kTX;
    const int nbx = (d.nxg - 1 + kTX - 1) / kTX, nby = (d.nyg - 2 + kTY - 1) / kTY;
    const int ntile = nbx * nby * ((d.nzg - 2 + kchunk - 1) / kchunk);
    const int t = xcd_tile(blockIdx.x, ntile);
    if (t >= ntile) return;
    // the tile's cells are i0 .. i0 + kTX - 1 with i0 a multiple of kTX, so
    // that the per-cell rows start on a 128-byte line (cell 0 is idle)
    const int i0 = (t % nbx) * kTX, j0 = ((t / nbx) % nby) * kTY + 1;
    const int kb = 1 + (t / (nbx * nby)) * kchunk;
    const int ke = min(kb + kchunk, d.nzg - 1);  // exclusive
    const long long sx = d.sx, sxy = d.sxy;
    // halo tile origin (i0-1, j0-1); loads clamped into the allocation (the
    // column i0-1 = -1 of the first tile feeds only the idle cell 0)
    // each thread moves up to kPer halo elements of a plane; they are fetched
    // into registers one iteration ahead and committed to LDS after the sync
    constexpr int kPer = (kPlane + 255) / 256;
    long long off[kPer];
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
        const int e = tid + 256 * q;
        const int ee = e < kPlane ? e : kPlane - 1;
        const int hy = ee / kHX, hx = ee - hy * kHX;
        const int ii = max(0, min(i0 - 1 + hx, d.sx - 1)), jj = min(j0 - 1 + hy, d.nyg - 1);
        off[q] = (long long)jj * sx + ii;
    }
    T ru[kPer], rv[kPer], rw[kPer], rn[LES ? kPer : 1];
    auto fetch = [&](int k) {
        const long long base = (long long)k * sxy;
#pragma unroll
        for (int q = 0; q < kPer; ++q) {
            ru[q] = U[base + off[q]];
            rv[q] = V[base + off[q]];
            rw[q] = W[base + off[q]];
            if constexpr (LES) rn[q] = Nt[base + off[q]];
        }
    };
    auto commit = [&](int plane) {
        const int s2 = plane & 1, s3 = plane % 3;
#pragma unroll
        for (int q = 0; q < kPer; ++q) {
            const int e = tid + 256 * q;
            if (e < kPlane) {
                sU[s2][e] = ru[q];
                sV[s2][e] = rv[q];
                sW[s3][e] = rw[q];
                if constexpr (LES) sN[s3][e] = rn[q];
            }
        }
    };
    if (tid < kTX) {
        const int ii = max(1, i0 + tid);  // entries of cells outside the grid are clamped and never used
        sMx[0][tid] = m.rdx[min(ii, d.nx - 1)];
        sMx[1][tid] = m.rdx[min(ii + 1, d.nx - 1)];
        sMx[2][tid] = m.rdxg[min(ii, d.nxg - 1)];
        sMx[3][tid] = m.rdxg[min(ii - 1, d.nxg - 1)];
    } else if (tid < kTX + kTY) {
        const int jt = tid - kTX, jj = j0 + jt;
        sMy[0][jt] = m.wy0[min(jj, d.ny - 1)];
        sMy[1][jt] = m.wy1[min(jj, d.ny - 1)];
        sMy[2][jt] = m.wy0[min(jj - 1, d.ny - 1)];
        sMy[3][jt] = m.wy1[min(jj - 1, d.ny - 1)];
        sMy[4][jt] = m.rdy[min(jj, d.ny - 1)];
        sMy[5][jt] = m.rdy[min(jj + 1, d.ny - 1)];
        sMy[6][jt] = m.rdyg[min(jj, d.nyg - 1)];
        sMy[7][jt] = m.rdyg[min(jj - 1, d.nyg - 1)];
    }
    fetch(kb - 1);
    commit(kb - 1);
    fetch(kb);
    commit(kb);
    fetch(kb + 1);
    const int i = i0 + tx;
    // U and V of plane kb-1 at the thread's cells, before plane kb+1 takes
    // their slot
    __syncthreads();
    T ubr[RPT], vbr[RPT];
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
        const int e = (RPT * ty + r + 1) * kHX + (tx + 1);
        ubr[r] = sU[(kb - 1) & 1][e];
        vbr[r] = sV[(kb - 1) & 1][e];
    }
    __syncthreads();  // before plane kb+1 overwrites that slot
    // a first stage starts from the field it differentiates: the old values
    // are then the LDS centre values and are not read again
    const bool old_is_cur = MODE == 0 && Uo == U && Vo == V && Wo == W;
    // MODE 0 with a separate old field (G, or the RK2 second stage) and
    // MODE 1: the old values per cell (and MODE 1's F1) are loaded one plane
    // ahead of their use; with the metrics in LDS MODE 1's six values fit
    // the registers at 3 blocks per CU too (FP32 RK stages 1.47 -> 1.39 ms
    // per step at 814x257x193)
    constexpr bool kAheadOld = (MODE == 0 && FOUT == 0) || MODE == 1;
    const bool ahead = kAheadOld && (MODE == 1 || !old_is_cur);
    T nuo[kAheadOld ? RPT : 1][3] = {}, nfo[MODE == 1 ? RPT : 1][3] = {};
    auto fetch_old = [&](int k) {
#pragma unroll
        for (int r = 0; r < (kAheadOld ? RPT : 1); ++r) {
            const long long p = fidx(d, max(1, min(i0 + tx, d.nxg - 2)), min(j0 + RPT * ty + r, d.nyg - 2), k);
            nuo[r][0] = get<NT>(Uo + p);
            nuo[r][1] = get<NT>(Vo + p);
            nuo[r][2] = get<NT>(Wo + p);
            if constexpr (MODE == 1) {
                nfo[r][0] = get<NT>(F1u + p);
                nfo[r][1] = get<NT>(F1v + p);
                nfo[r][2] = get<NT>(F1w + p);
            }
        }
    };
    if (ahead) fetch_old(kb);
    for (int k = kb; k < ke; ++k) {
        // this plane's step-start and first-stage values, issued before the
        // barrier so that their latency overlaps the stencil work
        T uo[RPT][3] = {}, fo[RPT][3] = {};
        if (ahead) {
#pragma unroll
            for (int r = 0; r < (kAheadOld ? RPT : 1); ++r)
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    uo[r][c] = nuo[r][c];
                    if constexpr (MODE == 1) fo[r][c] = nfo[r][c];
                }
        } else if (MODE == 1 || (MODE == 0 && !old_is_cur)) {
#pragma unroll
            for (int r = 0; r < RPT; ++r) {
                const int j = j0 + RPT * ty + r;
                if (i < 1 || i > d.nxg - 2 || j > d.nyg - 2) continue;
                const long long p = fidx(d, i, j, k);
                uo[r][0] = Uo[p];
                uo[r][1] = Vo[p];
                uo[r][2] = Wo[p];
                if constexpr (MODE == 1) {
                    fo[r][0] = F1u[p];
                    fo[r][1] = F1v[p];
                    fo[r][2] = F1w[p];
                }
            }
        }
        commit(k + 1);
        __syncthreads();
        if (k + 2 <= ke) fetch(k + 2);
        if (ahead && k + 1 < ke) fetch_old(k + 1);
        // W (and nu_t): three slots; U, V: two
        const int sm = (k - 1) % 3, sc = k % 3, sp = (k + 1) % 3;
        const int uc = k & 1, up1 = (k + 1) & 1;
        const T rdzk = m.rdz[k], rdzgk = m.rdzg[k], rdzgm = m.rdzg[k - 1];
#pragma unroll
        for (int r = 0; r < RPT; ++r) {
            const int jt = RPT * ty + r;     // row in the tile
            const int j = j0 + jt;
            const int e = (jt + 1) * kHX + (tx + 1);  // LDS index of (i, j)
            // U, V of plane k-1 at this cell, and plane k's for the next plane
            const T ubc = ubr[r], vbc = vbr[r];
            ubr[r] = sU[uc][e];
            vbr[r] = sV[uc][e];
            if (i < 1 || i > d.nxg - 2 || j > d.nyg - 2) continue;
            const T x_rdx = sMx[0][tx], x_rdx1 = sMx[1][tx], x_rdxg = sMx[2][tx], x_rdxgm = sMx[3][tx];
            const T y_w0 = sMy[0][jt], y_w1 = sMy[1][jt], y_w0m = sMy[2][jt], y_w1m = sMy[3][jt];
            const T y_rdy = sMy[4][jt], y_rdy1 = sMy[5][jt], y_rdyg = sMy[6][jt], y_rdygm = sMy[7][jt];
            const long long p = fidx(d, i, j, k);
            // ---- u (equations.f90:47-94, 149-154)
            if (i <= d.nx - 2) {
                T rr = 0.0;
                if (i < d.nx - 2) {
                    const T up = sU[uc][e], ue = sU[uc][e + 1], uw = sU[uc][e - 1];
                    const T un = sU[uc][e + kHX], us = sU[uc][e - kHX];
                    const T ut = sU[up1][e], ub = ubc;
                    double c = -(sq<double>(up + ue) - sq<double>(uw + up)) * (kQuarter * x_rdxg);
                    c = c - ((double)(y_w0 * up + y_w1 * un) * (sV[uc][e] + sV[uc][e + 1]) -
                             (double)(y_w0m * us + y_w1m * up) * (sV[uc][e - kHX] + sV[uc][e + 1 - kHX])) *
                                (kHalf * y_rdy);
                    c = c - ((double)(up + ut) * (sW[sc][e] + sW[sc][e + 1]) -
                             (double)(ub + up) * (sW[sm][e] + sW[sm][e + 1])) *
                                (kQuarter * rdzk);
                    rr = (T)c;
                    if constexpr (!LES) {
                        rr = rr + dPdx +
                             nu * ((x_rdx1 * (ue - up) - x_rdx * (up - uw)) * x_rdxg +
                                   ((un - up) * y_rdyg - (up - us) * y_rdygm) * y_rdy +
                                   (rdzgk * (ut - up) - rdzgm * (up - ub)) * rdzk);
                    } else {
                        const T *N = sN[sc], *Nm = sN[sm], *Np = sN[sp];
                        const T a0 = y_w0m, a1 = y_w1m, b0 = y_w0, b1 = y_w1;
                        const T nx1 = nu + N[e];
                        const T nx2 = nu + N[e + 1];
                        const T ny1 = nu + kHalf * (a0 * N[e - kHX] + a1 * N[e] + a0 * N[e + 1 - kHX] + a1 * N[e + 1]);
                        const T ny2 = nu + kHalf * (b0 * N[e] + b1 * N[e + kHX] + b0 * N[e + 1] + b1 * N[e + 1 + kHX]);
                        const T nz1 = nu + kQuarter * (N[e] + Nm[e] + N[e + 1] + Nm[e + 1]);
                        const T nz2 = nu + kQuarter * (N[e] + Np[e] + N[e + 1] + Np[e + 1]);
                        rr = rr + dPdx +
                             (nx2 * x_rdx1 * (ue - up) - nx1 * x_rdx * (up - uw)) * x_rdxg +
                             (ny2 * ((un - up) * y_rdyg) - ny1 * ((up - us) * y_rdygm)) * y_rdy +
                             (nz2 * rdzgk * (ut - up) - nz1 * rdzgm * (up - ub)) * rdzk;
                    }
                }
                if (MODE == 2) {
                    put<NT>(Fou + p, rr);
                } else {
                    const T base = old_is_cur ? sU[uc][e] : uo[r][0];
                    if (FOUT == 1) put<NT>(Fou + p, rr);
                    if (FOUT == 2) put<NT>(Fou + p, base + g2 * rr);
                    put<NT>(Un + p, (MODE == 0) ? base + c0 * rr : uo[r][0] + dt * (c1 * fo[r][0] + c0 * rr));
                }
            }
            // ---- v (equations.f90:183-230, 287-292)
            if (j <= d.ny - 2) {
                T rr = 0.0;
                if (i < d.nxg - 2) {
                    const T vp = sV[uc][e], ve = sV[uc][e + 1], vw = sV[uc][e - 1];
                    const T vn = sV[uc][e + kHX], vs = sV[uc][e - kHX];
                    const T vt = sV[up1][e], vb = vbc;
                    double c = -(sq<double>(vp + vn) - sq<double>(vs + vp)) * (kQuarter * y_rdyg);
                    c = c - ((double)(y_w0 * sU[uc][e] + y_w1 * sU[uc][e + kHX]) * (vp + ve) -
                             (double)(y_w0 * sU[uc][e - 1] + y_w1 * sU[uc][e - 1 + kHX]) * (vw + vp)) *
                                (kHalf * x_rdx);
                    c = c - ((double)(vp + vt) * (y_w0 * sW[sc][e] + y_w1 * sW[sc][e + kHX]) -
                             (double)(vb + vp) * (y_w0 * sW[sm][e] + y_w1 * sW[sm][e + kHX])) *
                                (kHalf * rdzk);
                    rr = (T)c;
                    if constexpr (!LES) {
                        rr = rr + nu * ((x_rdxg * (ve - vp) - x_rdxgm * (vp - vw)) * x_rdx +
                                        (y_rdy1 * (vn - vp) - y_rdy * (vp - vs)) * y_rdyg +
                                        (rdzgk * (vt - vp) - rdzgm * (vp - vb)) * rdzk);
                    } else {
                        const T *N = sN[sc], *Nm = sN[sm], *Np = sN[sp];
                        const T b0 = y_w0, b1 = y_w1;
                        const T nx1 = nu + kHalf * (b0 * N[e - 1] + b1 * N[e - 1 + kHX] + b0 * N[e] + b1 * N[e + kHX]);
                        const T nx2 = nu + kHalf * (b0 * N[e] + b1 * N[e + kHX] + b0 * N[e + 1] + b1 * N[e + 1 + kHX]);
                        const T ny1 = nu + N[e];
                        const T ny2 = nu + N[e + kHX];
                        const T nz1 = nu + kHalf * (b0 * Nm[e] + b1 * Nm[e + kHX] + b0 * N[e] + b1 * N[e + kHX]);
                        const T nz2 = nu + kHalf * (b0 * N[e] + b1 * N[e + kHX] + b0 * Np[e] + b1 * Np[e + kHX]);
                        rr = rr + x_rdx * (nx2 * x_rdxg * (ve - vp) - nx1 * x_rdxgm * (vp - vw)) +
                             y_rdyg * (ny2 * y_rdy1 * (vn - vp) - ny1 * y_rdy * (vp - vs)) +
                             rdzk * (nz2 * rdzgk * (vt - vp) - nz1 * rdzgm * (vp - vb));
                    }
                }
                if (MODE == 2) {
                    put<NT>(Fov + p, rr);
                } else {
                    const T base = old_is_cur ? sV[uc][e] : uo[r][1];
                    if (FOUT == 1) put<NT>(Fov + p, rr);
                    if (FOUT == 2) put<NT>(Fov + p, base + g2 * rr);
                    put<NT>(Vn + p, (MODE == 0) ? base + c0 * rr : uo[r][1] + dt * (c1 * fo[r][1] + c0 * rr));
                }
            }
            // ---- w (equations.f90:323-366, 408-413)
            if (k <= d.nz - 2) {
                T rr = 0.0;
                if (i < d.nxg - 2) {
                    const T wp = sW[sc][e], we = sW[sc][e + 1], ww = sW[sc][e - 1];
                    const T wn = sW[sc][e + kHX], ws = sW[sc][e - kHX];
                    const T wt = sW[sp][e], wb = sW[sm][e];
                    double c = -(sq<double>(wp + wt) - sq<double>(wb + wp)) * (kQuarter * rdzgk);
                    c = c - ((double)(sU[uc][e] + sU[up1][e]) * (wp + we) -
                             (double)(sU[uc][e - 1] + sU[up1][e - 1]) * (ww + wp)) *
                                (kQuarter * x_rdx);
                    c = c - ((double)(sV[uc][e] + sV[up1][e]) * (y_w0 * wp + y_w1 * wn) -
                             (double)(sV[uc][e - kHX] + sV[up1][e - kHX]) * (y_w0m * ws + y_w1m * wp)) *
                                (kHalf * y_rdy);
                    rr = (T)c;
                    if constexpr (!LES) {
                        rr = rr + dPdz +
                             nu * ((x_rdxg * (we - wp) - x_rdxgm * (wp - ww)) * x_rdx +
                                   ((wn - wp) * y_rdyg - (wp - ws) * y_rdygm) * y_rdy +
                                   (m.rdz[k + 1] * (wt - wp) - rdzk * (wp - wb)) * rdzgk);
                    } else {
                        const T *N = sN[sc], *Np = sN[sp];
                        const T a0 = y_w0m, a1 = y_w1m, b0 = y_w0, b1 = y_w1;
                        const T nx1 = nu + kQuarter * (N[e] + Np[e] + N[e - 1] + Np[e - 1]);
                        const T nx2 = nu + kQuarter * (N[e] + Np[e] + N[e + 1] + Np[e + 1]);
                        const T ny1 = nu + kHalf * (a0 * N[e - kHX] + a1 * N[e] + a0 * Np[e - kHX] + a1 * Np[e]);
                        const T ny2 = nu + kHalf * (b0 * N[e] + b1 * N[e + kHX] + b0 * Np[e] + b1 * Np[e + kHX]);
                        const T nz1 = nu + N[e];
                        const T nz2 = nu + Np[e];
                        rr = rr + dPdz +
                             (nx2 * x_rdxg * (we - wp) - nx1 * x_rdxgm * (wp - ww)) * x_rdx +
                             (ny2 * ((wn - wp) * y_rdyg) - ny1 * ((wp - ws) * y_rdygm)) * y_rdy +
                             (nz2 * m.rdz[k + 1] * (wt - wp) - nz1 * rdzk * (wp - wb)) * rdzgk;
                    }
                }
                if (MODE == 2) {
                    put<NT>(Fow + p, rr);
                } else {
                    const T base = old_is_cur ? sW[sc][e] : uo[r][2];
                    if (FOUT == 1) put<NT>(Fow + p, rr);
                    if (FOUT == 2) put<NT>(Fow + p, base + g2 * rr);
                    put<NT>(Wn + p, (MODE == 0) ? base + c0 * rr : uo[r][2] + dt * (c1 * fo[r][2] + c0 * rr));
                }
            }
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------------------
// Boundary conditions (boundary_conditions.f90:135-260)
// ------------------------------------------------------------------------

// deterministic block sum of 256 values; returns the sum in thread 0
__device__ __forceinline__ double block_sum_256(double v, double *sh) {
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
        if ((int)threadIdx.x < st) sh[threadIdx.x] += sh[threadIdx.x + st];
        __syncthreads();
    }
    return sh[0];
}

// temporal inflow modes Re(q e^{i(beta z - omega t)}) of row j, plane k at
// time t (boundary_conditions.f90:153-170)
__device__ __forceinline__ void inflow_modes(const Dims &d, const Metrics &m, const BCTables &b, int j, int k,
                                             double t, double &ut, double &vt, double &wt) {
    ut = vt = wt = 0.0;
    const double zc = m.zg[k];
    const double zf = (k < d.nz) ? m.z[k] : 0.0;
    for (int n = 0; n < b.n_modes; ++n)
        for (int mm = 0; mm < b.m_modes; ++mm) {
            const double pc = b.zmode[n] * zc - b.tmode[mm] * t;
            const double pf = b.zmode[n] * zf - b.tmode[mm] * t;
            const long long qi = (long long)n + (long long)b.n_modes * mm;
            const long long qu = j + (long long)d.nyg * qi;
            const double cc = cos(pc), sc = sin(pc);
            ut = ut + (b.qu_re[qu] * cc - b.qu_im[qu] * sc);
            if (j < d.ny) {
                const long long qv = j + (long long)d.ny * qi;
                vt = vt + (b.qv_re[qv] * cc - b.qv_im[qv] * sc);
            }
            const double cf = cos(pf), sf = sin(pf);
            wt = wt + (b.qw_re[qu] * cf - b.qw_im[qu] * sf);
        }
}

// inflow_flag 4: uniform [0, 1) value of (step, component, j, k) from a
// counter hash (splitmix64 finaliser) of the stream's seed
__device__ __forceinline__ unsigned long long bc_mix64(unsigned long long z) {
    z += 0x9E3779B97F4A7C15ULL;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
}
__device__ __forceinline__ double inflow_rand(unsigned long long seed, long long step, int comp, int j, int k) {
    const unsigned long long key = (((unsigned long long)step * 4ULL + (unsigned long long)comp) << 40) ^
                                   ((unsigned long long)k << 20) ^ (unsigned long long)j;
    return (double)(bc_mix64(seed ^ bc_mix64(key)) >> 11) * 0x1.0p-53;
}

// the inflow values of row j, plane k (FP64, before storage rounding):
// Blasius + temporal modes at time t (boundary_conditions.f90:183-190), or
// Blasius + the perturbations of step `step` (inflow_flag 4, :423-445)
__device__ __forceinline__ void inflow_values(const Dims &d, const Metrics &m, const BCTables &b, int j, int k,
                                              double t, long long step, double &u, double &v, double &w) {
    if (b.inflow_flag == 4) {
        const double a = b.amp * (1.0 - b.U_inlet[j]);
        u = b.U_inlet[j] + a * (inflow_rand(b.seed, step, 0, j, k) - 0.5);
        w = b.W_inlet[j] + a * (inflow_rand(b.seed, step, 2, j, k) - 0.5);
        v = (j < d.ny) ? b.V_inlet[j] + a * (inflow_rand(b.seed, step, 1, j, k) - 0.5) : 0.0;
        return;
    }
    double ut = 0.0, vt = 0.0, wt = 0.0;
    if (b.n_modes > 0) inflow_modes(d, m, b, j, k, t, ut, vt, wt);
    u = b.U_inlet[j] + ut;
    w = b.W_inlet[j] + wt;
    v = (j < d.ny) ? b.V_inlet[j] + vt : 0.0;
}

// The boundary values depend on the step-start field, the time and the tables,
// not on the stage's interior: one launch computes them for the stages of a
// step (blockIdx.z), with the two parts of the mass flux.  The inflow
// (boundary_conditions.f90:137-190) and the outflow (:193-202) are one thread per
// (j, k), blockIdx.x < nb_in; the wall and top V one thread per (i, k).
struct BcStages {
    double coef[3], t[3];  // rk_t(stage) dt Uc, and the stage's time
};
template <class T>
__global__ __launch_bounds__(256) void k_bc_planes(Dims d, Metrics m, BCTables b, BcPlanes<T> p0, long long stride,
                                                   const T *__restrict__ Uo, const T *__restrict__ Vo,
                                                   const T *__restrict__ Wo, BcStages st, int nb_in,
                                                   double *__restrict__ qpart, double *inc1, double t_old) {
    __shared__ double sh[256];
    const int k = blockIdx.y, z = blockIdx.z;
    const long long o = z * stride;
    double q = 0.0;
    if ((int)blockIdx.x < nb_in) {
        // mass flux through the x boundaries (:246-249):
        // (U(1,j,k) - U(nx-1,j,k))*(y(j)-y(j-1)) for j in [1,nyg-2], k in [1,nzg-3]
        const int j = blockIdx.x * 256 + threadIdx.x;
        if (j < d.nyg) {
            const int nx = d.nx, nxg = d.nxg;
            const double coef = st.coef[z], t = st.t[z];
            double ui, vi, wi;
            const bool lund = b.inflow_flag == 3 || b.inflow_flag == 5;
            if (lund) {
                // the step's rescaled plane (:569-597); flag 5 adds it to the inlet
                // means, with W's planes shifted by 16 (:512-559)
                const bool f5 = b.inflow_flag == 5;
                ui = (f5 ? b.U_inlet[j] : 0.0) + b.lund_u[j + (long long)d.nyg * k];
                wi = 0.0;
                if (k < d.nz) {
                    const int ks = f5 ? (k + 17) % d.nz : k;
                    wi = (f5 ? b.W_inlet[j] : 0.0) + b.lund_w[j + (long long)d.nyg * ks];
                }
                vi = (j < d.ny) ? (f5 ? b.V_inlet[j] : 0.0) + b.lund_v[j + (long long)d.ny * k] : 0.0;
            } else {
                inflow_values(d, m, b, j, k, t, b.istep, ui, vi, wi);
            }
            const double uin = (double)(T)ui;  // the value stored
            const long long pl = j + (long long)d.nyg * k;
            if (inc1 && z == 0) {
                // FP64 increment of the inflow face over the step-start value: that
                // value is taken unrounded when it is the stored boundary value of
                // t_old (the previous step), as it is after any step
                double uo = 0.0, vo, wo;
                if (!lund) inflow_values(d, m, b, j, k, t_old, b.istep - 1, uo, vo, wo);
                const double so = (double)Uo[fidx(d, 0, j, k)];
                // (the previous step's rescaled plane is gone: the stored value)
                inc1[pl] = ui - (!lund && (double)(T)uo == so ? uo : so);
            }
            p0.uin[o + pl] = (T)uin;
            {
                const long long pa = fidx(d, nx - 2, j, k);
                const double o1 = Uo[pa], o0 = Uo[pa - 1];
                const double du = coef * (o1 - o0) / (m.x[nx - 2] - m.x[nx - 3]);
                const double v = (double)(T)(o1 - du);
                p0.uo[o + pl] = (T)v;
                // FP64 increment of the outflow face before the mass-flux shift
                if (inc1 && z == 0) inc1[(long long)d.nyg * d.nzg + pl] = -du;
                if (j >= 1 && j <= d.nyg - 2 && k >= 1 && k <= d.nzg - 3) q = (uin - v) * (m.y[j] - m.y[j - 1]);
            }
            const long long pa = fidx(d, nxg - 2, j, k);
            const double dxo = m.xg[nxg - 2] - m.xg[nxg - 3];
            if (k < d.nz) {
                const double o1 = Wo[pa], o0 = Wo[pa - 1];
                p0.win[o + pl] = (T)wi;
                p0.wo[o + pl] = (T)(o1 - coef * (o1 - o0) / dxo);
            }
            if (j < d.ny) {
                const double o1 = Vo[pa], o0 = Vo[pa - 1];
                p0.vin[o + pl] = (T)vi;
                p0.vo[o + pl] = (T)(o1 - coef * (o1 - o0) / dxo);
            }
        }
    } else {
        // mass flux through the y boundaries (:251-253):
        // (V(i,1,k) - V(i,ny,k))*(x(i)-x(i-1))
        const int i = (blockIdx.x - nb_in) * 256 + threadIdx.x;
        if (i < d.nxg) {
            // V(i, ny) as stored at the top: V_top (top_flag 0), blowing/suction
            // (1, 2: :648-673; columns below i_rescale keep it, because the
            // reference's V_top copy of zero_wz_top, :279, writes V(i, nyg), one row
            // past the top face, which the wall condition then overwrites), or 0
            // (Falkner-Skan, :1001)
            const double vtop = b.top_flag == 0 ? (double)(T)b.V_top[i]
                                                : (b.top_flag == 3 ? 0.0 : (double)(T)b.vtop_bs[i]);
            // V(i, 1) as the wall condition stores it: 0, or with a Robin wall
            // model the pseudo-Robin alpha_y dVo/dy less its wall mean beta_y
            // (apply_pseudo_Robin_bc_y_bottom :1152-1180, id 2)
            double vwall = 0.0;
            if (p0.wld) {
                const long long pw = fidx(d, i, 0, k);
                vwall = (double)(T)(b.wm_ay[i] * ((double)Vo[pw + d.sx] - (double)Vo[pw]) / (m.y[1] - m.y[0]) -
                                    b.wm_beta[0]);
            }
            if (k == 0) p0.vtop[o + i] = (T)vtop;
            if (p0.wld || k == 0) p0.vwall[o + p0.wld * k + i] = (T)vwall;
            if (i >= 1 && i <= d.nxg - 3 && k >= 1 && k <= d.nzg - 3) q = (vwall - vtop) * (m.x[i] - m.x[i - 1]);
        }
    }
    q = block_sum_256(q, sh);
    if (threadIdx.x == 0) {
        // the x parts first, then the y parts
        const long long nq_in = (long long)nb_in * gridDim.y;
        const long long e = (int)blockIdx.x < nb_in
                                ? blockIdx.x + (long long)nb_in * k
                                : nq_in + (blockIdx.x - nb_in) + (long long)(gridDim.x - nb_in) * k;
        qpart[e + (long long)gridDim.x * gridDim.y * z] = q;
    }
}

// global mass conservation (:241-260): the shift of the outflow U of stage
// blockIdx.x from its nq flux partials
__global__ __launch_bounds__(256) void k_bc_shift(Dims d, double length_y, const double *__restrict__ qpart, int nq,
                                                  double *__restrict__ du, double *inc_du) {
    __shared__ double sh[256];
    double acc = 0.0;
    for (int t = threadIdx.x; t < nq; t += 256) acc += qpart[(long long)nq * blockIdx.x + t];
    const double Q = block_sum_256(acc, sh);
    if (threadIdx.x == 0) {
        const double v = Q / length_y / (double)(d.nzg - 3);
        du[blockIdx.x] = v;
        if (inc_du && blockIdx.x == 0) inc_du[0] = v;
    }
}

// Every boundary and ghost entry, in one launch: the reference applies inflow and
// outflow, the periodic planes (:205-217), the top (:220-228, 947-1007), the
// wall (:231-238, 73-108) and the mass-flux shift one after the other; here
// each entry is computed from what those leave of the interior entries and
// the stage's boundary values it derives from, and no entry that another
// thread reads is written.  Three ranges of one thread index: the ghost z
// planes (entries (i, j) of three planes), the wall and top rows of planes
// 1..nzg-3 (entries (i, k)), and the x faces of those planes (entries (j, k)).
// Eight dependent launches per stage (this, and the same before the pressure
// solve, which now takes the boundary values directly) were the larger part of
// the time on small grids: a step of 192x32x8 took 45 launches of 4 to 10 us.
template <class T>
struct BcField {
    Dims d;
    const Metrics &m;
    const BCTables &b;
    const BcPlanes<T> &p;
    const T *U, *V, *W;
    double dyg;
    bool robin;

    __device__ int zc(int k) const { return k == 0 ? d.nzg - 3 : (k == d.nzg - 2 ? 1 : (k == d.nzg - 1 ? 2 : k)); }
    __device__ int zf(int k) const { return k == 0 ? d.nz - 2 : (k == d.nz - 1 ? 1 : k); }
    // interior rows and planes, any i, before the shift
    __device__ T ubase(int i, int j, int k) const {
        const long long pl = j + (long long)d.nyg * k;
        return i == 0 ? p.uin[pl] : (i >= d.nx - 2 ? p.uo[pl] : U[fidx(d, i, j, k)]);
    }
    __device__ T wbase(int i, int j, int k) const {
        const long long pl = j + (long long)d.nyg * k;
        return i == 0 ? p.win[pl] : (i >= d.nxg - 2 ? p.wo[pl] : W[fidx(d, i, j, k)]);
    }
    __device__ T u(int i, int j, int k) const {
        const int kc = zc(k), ib = min(i, d.nx - 2);
        T v;
        if (j == 0) {
            const T x = ubase(ib, 1, kc);
            if (b.iwall == 0) {
                v = -x;  // no-slip
            } else if (!robin) {
                // Neumann (iwall_model 11, 15: apply_Nozero_Neumann_bc_y :359-372)
                v = (T)((double)x - b.wm_ax[ib] * dyg);
            } else {
                // Robin (apply_Robin_bc_y_bottom :1107-1132, id 2)
                const double r = 2.0 * b.wm_ax[ib] / dyg;
                v = (T)((r - 1.0) * (double)x / (r + 1.0));
            }
        } else if (j == d.nyg - 1) {
            if (b.top_flag == 0 || (b.top_flag != 3 && ib < b.i_rescale)) {
                v = (T)b.U_top[ib];
            } else if (b.top_flag == 3) {
                v = (T)b.utop_fs[ib];
            } else {
                // zero spanwise vorticity under blowing/suction (zero_wz_top :264-283)
                const double vp = (double)(T)b.vtop_bs[ib + 1], vm = (double)(T)b.vtop_bs[ib];
                v = (T)(b.dy_dx * (vp - vm) + (double)ubase(ib, j - 1, kc));
            }
        } else {
            v = ubase(ib, j, kc);
        }
        return i >= d.nx - 2 ? (T)((double)v + p.du[0]) : v;
    }
    __device__ T v(int i, int j, int k) const {
        if (j == 0) return p.vwall[p.wld * k + i];
        if (j == d.ny - 1) return p.vtop[i];
        const int kc = zc(k);
        const long long pl = j + (long long)d.nyg * kc;
        return i == 0 ? p.vin[pl] : (i >= d.nxg - 2 ? p.vo[pl] : V[fidx(d, i, j, kc)]);
    }
    __device__ T w(int i, int j, int k) const {
        const int kc = zf(k);
        if (j == 0) {
            const T x = wbase(i, 1, kc);
            if (!robin) return -x;
            const double r = 2.0 * b.wm_az[i] / dyg;
            return (T)((r - 1.0) * (double)x / (r + 1.0));
        }
        if (j == d.nyg - 1) {
            if (b.top_flag == 0 || (b.top_flag != 3 && i < b.i_rescale)) return (T)b.W_top[i];
            return wbase(i, j - 1, kc);
        }
        return wbase(i, j, kc);
    }
};

template <class T>
__global__ __launch_bounds__(256) void k_bc_apply(Dims d, Metrics m, BCTables b, BcPlanes<T> p, T *U, T *V, T *W) {
    const long long nA = 3LL * d.nxg * d.nyg, nB = (long long)d.nxg * (d.nzg - 3), nC = (long long)(d.nyg - 2) * (d.nzg - 3);
    long long e = (long long)blockIdx.x * 256 + threadIdx.x;
    const BcField<T> f{d, m, b, p, U, V, W, m.yg[1] - m.yg[0], p.wld != 0};
    if (e < nA) {
        const int r = (int)(e % (3 * d.nxg)), j = (int)(e / (3 * d.nxg));
        const int q = r / d.nxg, i = r - q * d.nxg;
        const int k = q == 0 ? 0 : d.nzg - 3 + q;  // U, V: planes 0, nzg-2, nzg-1; W: 0 and nz-1 = nzg-2
        const long long o = fidx(d, i, j, k);
        if (i < d.nx) U[o] = f.u(i, j, k);
        if (j < d.ny) V[o] = f.v(i, j, k);
        if (k < d.nz) W[o] = f.w(i, j, k);
        return;
    }
    e -= nA;
    if (e < nB) {
        const int k = 1 + (int)(e / d.nxg), i = (int)(e % d.nxg);
        const long long o = fidx(d, i, 0, k), top = (long long)d.sx * (d.nyg - 1);
        if (i < d.nx) {
            const T lo = f.u(i, 0, k), hi = f.u(i, d.nyg - 1, k);
            U[o] = lo;
            U[o + top] = hi;
        }
        V[o] = f.v(i, 0, k);
        V[o + top - d.sx] = f.v(i, d.ny - 1, k);
        const T lo = f.w(i, 0, k), hi = f.w(i, d.nyg - 1, k);
        W[o] = lo;
        W[o + top] = hi;
        return;
    }
    e -= nB;
    if (e < nC) {
        const int k = 1 + (int)(e / (d.nyg - 2)), j = 1 + (int)(e % (d.nyg - 2));
        const long long o = fidx(d, 0, j, k), pl = j + (long long)d.nyg * k;
        U[o] = p.uin[pl];
        const T u = (T)((double)p.uo[pl] + p.du[0]);
        U[o + d.nx - 2] = u;
        U[o + d.nx - 1] = u;
        if (j < d.ny - 1) {
            V[o] = p.vin[pl];
            const T v = p.vo[pl];
            V[o + d.nxg - 2] = v;
            V[o + d.nxg - 1] = v;
        }
        W[o] = p.win[pl];
        const T w = p.wo[pl];
        W[o + d.nxg - 2] = w;
        W[o + d.nxg - 1] = w;
    }
}

// ------------------------------------------------------------------------
// Projection pieces
// ------------------------------------------------------------------------
// phi with the x-Neumann and z-periodic copies of apply_periodic_z_pressure
__device__ __forceinline__ long long phi_at(const Dims &d, int i, int j, int k) {
    if (i > d.nxg - 3) i = d.nxg - 3;
    if (k == d.nzg - 2) k = 1;
    return fidx(d, i, j, k);
}

// a thread walks kProjZ planes of one (i, j) column, so phi(k+1) of a plane
// is phi(k) of the next; all loads of its planes are issued before the first
// update (0.81 -> 0.71 ms/step in FP32 at 814x257x193).  Tiles cover cells
// 64 bx .. 64 bx + 63 (cell 0 idle), so that a wave's row segment starts on
// a 128-byte line (-5 % FP64, -7 % FP32).  Tiles in XCD-contiguous order in
// FP32 only: at that size it is 3 % faster there and 4 % slower in FP64 than
// plain order.
constexpr int kProjZ = 4;

// With P set (the first sub-step), also P = phi / den on the same cells
// (projection.f90:75-85), and on the ghost cells next to them the same value
// (the copies of apply_periodic_z_pressure and the P ghost faces), without a
// second read of phi.
template <class T>
__global__ __launch_bounds__(256) void k_project(Dims d, MetricsT<T> m, T *U, T *V, T *W, const T *phi, T *P,
                                                 double den) {
    const int nbx = (d.nxg - 1 + kWave - 1) / kWave, nby = (d.nyg - 2 + 3) / 4;
    const int ntile = nbx * nby * ((d.nzg - 2 + kProjZ - 1) / kProjZ);
    const int t = sizeof(T) == 4 ? xcd_tile(blockIdx.x, ntile) : blockIdx.x;
    if (t >= ntile) return;
    const int i = (t % nbx) * kWave + threadIdx.x;
    const int j = ((t / nbx) % nby) * 4 + threadIdx.y + 1;
    const int k0 = (t / (nbx * nby)) * kProjZ + 1;
    if (i < 1 || i > d.nxg - 2 || j > d.nyg - 2) return;
    const int k1 = min(k0 + kProjZ, d.nzg - 1);  // exclusive
    const T rdxg = m.rdxg[i], rdyg = m.rdyg[j];
    // every load of the kProjZ planes first (planes past the last one clamped
    // and not stored), then the updates
    T pz[kProjZ + 1], px[kProjZ], py[kProjZ], u[kProjZ], v[kProjZ], w[kProjZ], rz[kProjZ];
    pz[0] = phi[phi_at(d, i, j, k0)];
#pragma unroll
    for (int r = 0; r < kProjZ; ++r) {
        const int k = min(k0 + r, k1 - 1);
        const long long p = fidx(d, i, j, k);
        pz[r + 1] = phi[phi_at(d, i, j, k + 1)];
        px[r] = phi[phi_at(d, i + 1, j, k)];
        py[r] = phi[phi_at(d, i, j + 1, k)];
        u[r] = U[p];
        v[r] = V[p];
        w[r] = W[p];
        rz[r] = m.rdzg[k];
    }
#pragma unroll
    for (int r = 0; r < kProjZ; ++r) {
        const int k = k0 + r;
        if (k >= k1) break;
        const long long p = fidx(d, i, j, k);
        if (i <= d.nx - 2) U[p] = u[r] - (px[r] - pz[r]) * rdxg;
        if (j <= d.ny - 2) V[p] = v[r] - (py[r] - pz[r]) * rdyg;
        if (k <= d.nz - 2) W[p] = w[r] - (pz[r + 1] - pz[r]) * rz[r];
    }
    if (P) {
        const int gi = i == 1 ? 0 : (i == d.nxg - 2 ? d.nxg - 1 : -1);
        const int gj = j == 1 ? 0 : (j == d.nyg - 2 ? d.nyg - 1 : -1);
#pragma unroll
        for (int r = 0; r < kProjZ; ++r) {
            const int k = k0 + r;
            if (k >= k1) break;
            const int gk = k == 1 ? 0 : (k == d.nzg - 2 ? d.nzg - 1 : -1);
            const T pv = (T)((double)pz[r] / den);
            for (int a = 0; a < 2; ++a) {
                const int ii = a ? gi : i;
                if (ii < 0) continue;
                for (int b = 0; b < 2; ++b) {
                    const int jj = b ? gj : j;
                    if (jj < 0) continue;
                    P[fidx(d, ii, jj, k)] = pv;
                    if (gk >= 0) P[fidx(d, ii, jj, gk)] = pv;
                }
            }
        }
    }
}

// ------------------------------------------------------------------------
// Real DFT along z (M = nzp points, periodic) of many columns, folded by the
// symmetry m <-> M-m so that each (cos, sin) pair of outputs costs M FMAs.
// Spectrum rows: q = 0 (k = 0), q = 2k-1 Re X_k, q = 2k Im X_k with
// X_k = sum_m T[m] e^{-2 pi i k m/M} (the z part of the reference's 2-D FFT,
// projection.f90:123); the inverse is the unnormalised sum over all k.
// Tables (transposed for wave-uniform scalar loads): ctab[m][k] = cos(2 pi k m/M),
// stab[m][k] = sin(2 pi k m/M), m, k < lda rows/cols (zero padded).
// Columns are c = kx + N*j, contiguous; stride between z planes is `plane`.
// ------------------------------------------------------------------------
// A block is 256 columns (four waves of 64) times one group of RW output
// rows, so that its four waves read the same table rows.  Tiles run in
// XCD-contiguous order with the row group fastest: the row groups of one
// column block follow each other on one XCD and share its L2 for the input.
// The next PF inputs of a column are loaded ahead of their use.
__device__ __forceinline__ void zdft_tile(int M, int C, int RW, int &k0, int &c0, bool &live) {
    const int ng = (M / 2 + 1 + RW - 1) / RW, nt = ng * ((C + 255) / 256);
    const int t = xcd_tile(blockIdx.x, nt);
    live = t < nt;
    k0 = (t % ng) * RW;
    c0 = (t / ng) * 256;
}

template <int RW, int PF>
__global__ __launch_bounds__(256) void k_zdft_fwd(int M, int C, long long plane, int lda,
                                                  const double *__restrict__ ctab,
                                                  const double *__restrict__ stab,
                                                  const double *__restrict__ in,
                                                  double *__restrict__ out) {
    int k0, c0;
    bool live;
    zdft_tile(M, C, RW, k0, c0, live);
    const int c = c0 + threadIdx.x;
    if (!live || c >= C) return;
    const int Kc = M / 2 + 1;  // cos rows k = 0..M/2
    const double *src = in + c;
    const double t0 = src[0];
    double ac[RW], as[RW];
#pragma unroll
    for (int r = 0; r < RW; ++r) {
        ac[r] = t0;
        as[r] = 0.0;
    }
    const int hm = M / 2;
    if (hm >= 1) {
        double rp[PF], rm[PF];
#pragma unroll
        for (int u = 0; u < PF; ++u) {
            const int m = min(1 + u, hm);
            rp[u] = src[(long long)m * plane];
            rm[u] = src[(long long)(M - m) * plane];
        }
        for (int m0 = 1; m0 <= hm; m0 += PF) {
#pragma unroll
            for (int u = 0; u < PF; ++u) {
                const int m = m0 + u;
                const double tp = rp[u], tm = rm[u];
                const int mn = min(m + PF, hm);
                rp[u] = src[(long long)mn * plane];
                rm[u] = src[(long long)(M - mn) * plane];
                if (m <= hm) {
                    const double e = (2 * m == M) ? tp : tp + tm;
                    const double o = tp - tm;  // zero for the middle element of even M
                    const double *cr = ctab + (long long)m * lda + k0;
                    const double *sr = stab + (long long)m * lda + k0;
#pragma unroll
                    for (int r = 0; r < RW; ++r) {
                        ac[r] = fma(e, cr[r], ac[r]);
                        as[r] = fma(o, sr[r], as[r]);
                    }
                }
            }
        }
    }
    double *dst = out + c;
#pragma unroll
    for (int r = 0; r < RW; ++r) {
        const int k = k0 + r;
        if (k >= Kc) break;
        dst[(long long)(k == 0 ? 0 : 2 * k - 1) * plane] = ac[r];
        if (k >= 1 && 2 * k <= M - 1) dst[(long long)(2 * k) * plane] = -as[r];
    }
}

// inverse: g[m] = S0 + sum_k c_k (Re_k cos - Im_k sin)(2 pi k m/M), c_k = 2
// (1 for the Nyquist row of even M); outputs m and M-m come from the same
// cos and sin sums.  Row groups cover the outputs m = 0..M/2.
template <int RW, int PF>
__global__ __launch_bounds__(256) void k_zdft_inv(int M, int C, long long plane, int lda,
                                                  const double *__restrict__ ctab,
                                                  const double *__restrict__ stab,
                                                  const double *__restrict__ in,
                                                  double *__restrict__ out) {
    int m0, c0;
    bool live;
    zdft_tile(M, C, RW, m0, c0, live);
    const int c = c0 + threadIdx.x;
    if (!live || c >= C) return;
    const int hm = M / 2;  // outputs m = 0..M/2 (paired with M-m)
    const double *src = in + c;
    const double s0 = src[0];
    double cc[RW], ss[RW];
#pragma unroll
    for (int r = 0; r < RW; ++r) {
        cc[r] = s0;
        ss[r] = 0.0;
    }
    const int Kc = M / 2 + 1;
    if (Kc >= 2) {
        // Re_k = row 2k-1, Im_k = row 2k (absent for the Nyquist row of even M)
        double rr[PF], ri[PF];
#pragma unroll
        for (int u = 0; u < PF; ++u) {
            const int k = min(1 + u, Kc - 1);
            rr[u] = src[(long long)(2 * k - 1) * plane];
            ri[u] = src[(long long)min(2 * k, M - 1) * plane];
        }
        for (int kb = 1; kb < Kc; kb += PF) {
#pragma unroll
            for (int u = 0; u < PF; ++u) {
                const int k = kb + u;
                const double re = rr[u], imr = ri[u];
                const int kn = min(k + PF, Kc - 1);
                rr[u] = src[(long long)(2 * kn - 1) * plane];
                ri[u] = src[(long long)min(2 * kn, M - 1) * plane];
                if (k < Kc) {
                    const bool nyq = (2 * k == M);
                    const double im = nyq ? 0.0 : imr;
                    const double cw = nyq ? re : 2.0 * re;
                    const double sw = 2.0 * im;
                    // tables indexed [k][m] here: ctab is symmetric in (k, m)
                    const double *cr = ctab + (long long)k * lda + m0;
                    const double *sr = stab + (long long)k * lda + m0;
#pragma unroll
                    for (int r = 0; r < RW; ++r) {
                        cc[r] = fma(cw, cr[r], cc[r]);
                        ss[r] = fma(sw, sr[r], ss[r]);
                    }
                }
            }
        }
    }
    double *dst = out + c;
#pragma unroll
    for (int r = 0; r < RW; ++r) {
        const int m = m0 + r;
        if (m > hm) break;
        dst[(long long)m * plane] = cc[r] - ss[r];
        if (m >= 1 && M - m != m) dst[(long long)(M - m) * plane] = cc[r] + ss[r];
    }
}

// ------------------------------------------------------------------------
// DCT-II x2 along x (forward) and its normalised inverse, per line, by
// Makhoul's reordering and a two-factor (N = N1*N2) DFT of the real
// reordered sequence, all in LDS.  Only k1 <= N1/2 is formed; the other half
// follows from Hermitian symmetry.  Forward: X[k] = sum_n 2 f[n]
// cos(pi k (2n+1)/(2N)) (the reference's 2N-point symmetric extension plus
// twiddle, projection.f90:110-134).  Inverse: f[n] = (1/(N M)) (g[0]/2 +
// sum_k g[k] cos(pi k (2n+1)/(2N))) (projection.f90:160-202 with the
// 1/(2 nxp nzp) factor).
//
// Both short DFTs run on the FP64 matrix cores (v_mfma_f64_16x16x4_f64; lane l
// holds A[l%16][l/16], B[l/16][l%16] and D[l/16 + 4r][l%16], r < 4), folded by
// the symmetry of cosine and sine: the sums over n of a length L take the pairs
// x[n] + x[L-n] and x[n] - x[L-n], and the outputs k and L-k come from the same
// two sums, so a product has (L/2)^2 terms instead of L^2.  At 814x257x193
// (28 x 29) that is 64 matrix instructions per two lines where the unfolded
// products took 176.
// Forward, step A (N1 points, real): B[k1][n2] = W_N^{n2 k1} sum_n1 v[N2 n1 + n2]
//   W_N1^{n1 k1}; columns (line, n2), rows k1.
// Forward, step C (N2 points, complex): V[k1 + N1 k2] = sum_n2 B W_N2^{n2 k2};
//   columns (line, k1), rows k2; X[k] = 2 Re(rot_k V), X[N-k] = -2 Im(rot_k V).
// Inverse, step C': the conjugate of C on V[k] = conj(rot_k) (g[k] - i g[N-k])/2;
//   step A': v[N2 n1 + n2] = sum_k1 c_k1 Re(C~ conj(W_N1^{n1 k1})) with the
//   Hermitian weights (1, 2, .., 1) in the table.
// Tables: rot[k] = e^{-i pi k/(2N)}; twA, twC = W_N^{n2 k1} as [k1][n2] and [n2][k1]
// (16 lanes read consecutive entries); t1, t1i, t2: (cos, sin)(2 pi a b/L) for
// row a and column b in lane order per (row tile, k step), b weighted in t1i.
// ------------------------------------------------------------------------
typedef double dbl4 __attribute__((ext_vector_type(4)));
typedef float flt4 __attribute__((ext_vector_type(4)));
constexpr int kLd = 4;  // loads per thread in flight in the line load phases

__device__ __forceinline__ dbl4 mfma64(double a, double b, dbl4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// the matrix instruction of a storage type: the operands' layout is the same,
// the rows of the accumulator are 4 apart in FP64 and consecutive in FP32
template <class T>
struct Mf;
template <>
struct Mf<double> {
    typedef double2 T2;
    typedef dbl4 V4;
    static __device__ __forceinline__ V4 mul(double a, double b, V4 c) { return mfma64(a, b, c); }
    static __device__ __forceinline__ int row(int q, int r) { return q + 4 * r; }
    static __device__ __forceinline__ T2 make(double a, double b) { return make_double2(a, b); }
};
template <>
struct Mf<float> {
    typedef float2 T2;
    typedef flt4 V4;
    static __device__ __forceinline__ V4 mul(float a, float b, V4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int q, int r) { return 4 * q + r; }
    static __device__ __forceinline__ T2 make(float a, float b) { return make_float2(a, b); }
};

template <class T>
struct DctArgs {
    typedef typename Mf<T>::T2 T2;
    int N, N1, N2, K1h;
    int LB;        // lines per block
    int C1, C;     // lines c = c1 + C1*c2
    long long in_base, in_c1, in_c2;
    long long out_base, out_c1, out_c2;
    T scale;       // inverse only: 1/(N*M)
    const T2 *twA, *twC, *rot, *t1, *t1i, *t2;
    double *part;       // forward, not null: FP64 line sums of the rhs, part[c1 part_ld + c2]
    int part_ld;
    const double *add;  // inverse, not null: a constant per c1 added to the line
};

template <class T2>
__device__ __forceinline__ T2 cmul(T2 a, T2 b) {
    return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}
template <class T2>
__device__ __forceinline__ T2 cmulc(T2 a, T2 b) {  // a * conj(b)
    return {a.x * b.x + a.y * b.y, a.y * b.x - a.x * b.y};
}

// the folded length-N2 DFT of the complex rows Bl (one per column): the four
// real sums of row tile rt
template <class T>
struct DctSums {
    typename Mf<T>::V4 cr, ci, sr, si;  // sum E cos, sum O sin (real and imaginary parts)
};
// REAL: the rows' imaginary parts are zero (N1 = 1)
template <bool REAL, class T>
__device__ __forceinline__ DctSums<T> dct_sums(const DctArgs<T> &a, const typename Mf<T>::T2 *Bl, bool cok, int rt,
                                               int q, int lane) {
    typedef typename Mf<T>::T2 T2;
    const int H = a.N2 / 2 + 1, KS = (H + 3) / 4;
    const typename Mf<T>::V4 z = {0, 0, 0, 0};
    DctSums<T> s{z, z, z, z};
    const T2 *t = a.t2 + (long long)rt * KS * 64 + lane;
    // four k steps at a time, their operands read before the first product, from the last to the first: a smooth
    // field's spectrum falls with k, and adding its large end last rounds the
    // large partial sums least often
    for (int k0 = (KS - 1) / 4 * 4; k0 >= 0; k0 -= 4) {
        T2 w[4], x[4], y[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int n = 4 * (k0 + u) + q;
            w[u] = t[min(k0 + u, KS - 1) * 64];
            x[u] = y[u] = Mf<T>::make(0, 0);
            if (cok && n < H) {
                x[u] = Bl[n];
                y[u] = Bl[n == 0 ? 0 : a.N2 - n];
            }
        }
#pragma unroll
        for (int u = 3; u >= 0; --u) {
            const int n = 4 * (k0 + u) + q;
            const bool single = n == 0 || 2 * n == a.N2;  // x = y there
            if (k0 + u >= KS) continue;
            s.cr = Mf<T>::mul(w[u].x, single ? x[u].x : x[u].x + y[u].x, s.cr);
            if (!REAL) s.ci = Mf<T>::mul(w[u].x, single ? x[u].y : x[u].y + y[u].y, s.ci);
            s.sr = Mf<T>::mul(w[u].y, x[u].x - y[u].x, s.sr);
            if (!REAL) s.si = Mf<T>::mul(w[u].y, x[u].y - y[u].y, s.si);
        }
    }
    return s;
}

// SMALL (N1, N2 <= 31): two lines and two waves per block; step A has two
// column tiles per wave, step C one, so every product stays in registers until
// its inputs are read and the lines and the spectra share one LDS area (13.9 KB
// at N = 812: the blocks' load, product and store phases overlap across ten
// blocks per CU).  Otherwise four or eight waves, and LB lines in an area of their
// own, by dct_plan.  At 814x257x193 the forward (inverse) transform takes 0.327
// (0.203) ms, bound by the latency of its loads (HBM time 0.25 (0.125)); the
// unfolded products in four waves took 0.42 (0.30).  511 points (7 x 73): 0.077
// (0.050) ms per 12288 lines, on the vector units alone 0.15 (0.15).  FP32
// (v_mfma_f32_16x16x4_f32, 814x257x193): 0.209 (0.124) ms; unfolded split-BF16x3
// products in four waves 0.25 (0.144).
// A first factor of 2 to 7 points (kDctShort rows k1) has no product in steps A
// and A' but a column per thread on the vector units: of the 16 rows of a tile it
// would use N1/2 + 1, and its many column tiles waited for their loads one after
// the other.  Both directions, products -> vector units: 4 x 127 points, 20352
// lines FP32 279 -> 204 us; 2 x 47, 2296 lines FP64 31 -> 24.  With dct_plan's
// waves and lines FP32 4 x 251 points take 374 us there (955 before) and 2 x 251
// 228 (468); the dense split-BF16 product, with factors to 2^-18 instead of 2^-24,
// takes 502 and 209.  It is ahead for first factors of 1 and 2 with many lines only
// (2 x 53 50 us against 55, 2 x 181 132 against 167), which keep the more exact product.
// DIV: the line is the pseudo-pressure rhs (projection.f90:38-47) evaluated
// on the fly from U, V, W (in = U, in2 = V, in3 = W, lines over cells
// i = 1..N, j = 1..NM, k = 1..M) instead of being read from memory; with
// bc.du set the boundary faces come from the stage's boundary values (DivLine),
// and with inc.inc1 set from the stage's increment (IncLine, FP32 fields).
template <bool DIV, bool SMALL, class T>
__global__ __launch_bounds__(SMALL ? 128 : 512, SMALL ? (sizeof(T) == 4 ? 6 : 5) : 4) void k_dct_fwd_m(DctArgs<T> a, Dims d, Metrics mt, BcPlanes<T> bc, IncSrc inc,
                                                                 const T *__restrict__ in,
                                                                 const T *__restrict__ in2,
                                                                 const T *__restrict__ in3,
                                                                 T *__restrict__ out) {
    extern __shared__ double2 smem16[];
    typedef typename Mf<T>::T2 T2;
    typedef typename Mf<T>::V4 V4;
    T2 *smem2 = reinterpret_cast<T2 *>(smem16);
    const int NW = SMALL ? 2 : blockDim.x >> 6;
    const int N = a.N, N1 = a.N1, N2 = a.N2, K1 = a.K1h + 1, LB = SMALL ? 2 : a.LB, ld = dct_ld(N2);
    T *v = reinterpret_cast<T *>(smem2);
    T2 *Bc = SMALL ? smem2 : smem2 + dct_lines(LB, N) / 2;  // [line][k1][ld]
    const int tid = threadIdx.x, lane = tid & 63, q = lane >> 4, c16 = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int line0 = blockIdx.x * LB;
    // load and reorder: v[n/2] = f[n] (n even), v[N-1-(n-1)/2] = f[n] (n odd);
    // a line per wave, kLd elements per lane loaded before the first is used
    for (int l = wave; l < LB; l += NW) {
        const int c = min(line0 + l, a.C - 1);
        const int c1 = c % a.C1, c2 = c / a.C1;
        T *vl = v + l * N;
        auto put = [&](int n, T x) { vl[(n & 1) ? N - 1 - (n >> 1) : (n >> 1)] = x; };
        if constexpr (DIV) {
            double sum = 0.0;
            auto line = [&](const auto &dl) {
                for (int n0 = lane; n0 < N; n0 += 64 * kLd) {
                    typename std::decay<decltype(dl)>::type::Raw r[kLd];
#pragma unroll
                    for (int u = 0; u < kLd; ++u) r[u] = dl.load(min(n0 + 64 * u, N - 1));
#pragma unroll
                    for (int u = 0; u < kLd; ++u) {
                        const int n = n0 + 64 * u;
                        if (n >= N) continue;
                        const double x = dl.div(r[u], n);
                        if constexpr (sizeof(T) == 4) sum += x;
                        put(n, (T)x);
                    }
                }
            };
            if constexpr (sizeof(T) == 4) {
                if (inc.inc1)
                    line(IncLine(d, mt, inc, bc, c1, c2));
                else
                    line(DivLine<T>(d, mt, bc, in, in2, in3, c1, c2));
                for (int o = 32; o > 0; o >>= 1) sum += __shfl_down(sum, o);
                if (lane == 0 && line0 + l < a.C) a.part[(long long)c1 * a.part_ld + c2] = sum;
            } else {
                line(DivLine<T>(d, mt, bc, in, in2, in3, c1, c2));
            }
        } else {
            const T *src = in + a.in_base + c1 * a.in_c1 + c2 * a.in_c2;
            for (int n0 = lane; n0 < N; n0 += 64 * kLd) {
                T f[kLd];
#pragma unroll
                for (int u = 0; u < kLd; ++u) f[u] = src[min(n0 + 64 * u, N - 1)];
#pragma unroll
                for (int u = 0; u < kLd; ++u)
                    if (n0 + 64 * u < N) put(n0 + 64 * u, f[u]);
            }
        }
    }
    __syncthreads();
    // ---- step A
    const int H1 = K1, KS1 = (H1 + 3) / 4, RT1 = (H1 + 15) / 16, CA = (LB * N2 + 15) / 16;
    auto sums_a = [&](int ct, int rt, V4 &re, V4 &im) {
        const int col = ct * 16 + c16, ln = col / N2, n2 = col - ln * N2;
        const bool cok = col < LB * N2;
        const T *vl = v + ln * N + n2;
        const T2 *t = a.t1 + rt * KS1 * 64 + lane;
        re = im = V4{0, 0, 0, 0};
        for (int k0 = 0; k0 < KS1; k0 += 4) {
            T2 w[4];
            T x[4], y[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int n = 4 * (k0 + u) + q;
                w[u] = t[min(k0 + u, KS1 - 1) * 64];
                x[u] = y[u] = 0;
                if (cok && n < H1) {
                    x[u] = vl[N2 * n];
                    y[u] = vl[n == 0 ? 0 : N2 * (N1 - n)];
                }
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int n = 4 * (k0 + u) + q;
                const bool single = n == 0 || 2 * n == N1;  // x = y there
                if (k0 + u >= KS1) continue;
                re = Mf<T>::mul(w[u].x, single ? x[u] : x[u] + y[u], re);
                im = Mf<T>::mul(w[u].y, x[u] - y[u], im);
            }
        }
    };
    auto put_a = [&](int ct, int rt, const V4 &re, const V4 &im) {
        const int col = ct * 16 + c16, ln = col / N2, n2 = col - ln * N2;
        if (col >= LB * N2) return;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int k1 = 16 * rt + Mf<T>::row(q, r);
            if (k1 < K1) Bc[(ln * K1 + k1) * ld + n2] = cmul(Mf<T>::make(re[r], -im[r]), a.twA[k1 * N2 + n2]);
        }
    };
    if constexpr (SMALL) {
        V4 re[2], im[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) sums_a(2 * wave + h, 0, re[h], im[h]);
        __syncthreads();  // v is read; Bc overwrites it
#pragma unroll
        for (int h = 0; h < 2; ++h) put_a(2 * wave + h, 0, re[h], im[h]);
    } else if (N1 == 1) {  // one point: a copy
        for (int e = tid; e < LB * N; e += blockDim.x) {
            const int ln = e / N, n2 = e - ln * N;
            Bc[ln * ld + n2] = Mf<T>::make(v[e], 0);
        }
    } else if (K1 <= kDctShort) {  // a column per thread on the vector units
        for (int e = tid; e < LB * N2; e += blockDim.x) {
            const int ln = e / N2, n2 = e - ln * N2;
            const T *vl = v + ln * N + n2;
            T xs[kDctShort], xd[kDctShort];
#pragma unroll
            for (int n = 0; n < kDctShort; ++n) {
                xs[n] = xd[n] = 0;
                if (n < K1) {
                    const T x = vl[N2 * n], y = vl[n == 0 ? 0 : N2 * (N1 - n)];
                    xs[n] = n == 0 || 2 * n == N1 ? x : x + y;
                    xd[n] = x - y;
                }
            }
#pragma unroll
            for (int k1 = 0; k1 < kDctShort; ++k1) {
                if (k1 >= K1) continue;
                T re = 0, im = 0;
#pragma unroll
                for (int n = 0; n < kDctShort; ++n) {
                    const T2 w = a.t1[16 * n + k1];
                    re = fma(w.x, xs[n], re);
                    im = fma(w.y, xd[n], im);
                }
                Bc[(ln * K1 + k1) * ld + n2] = cmul(Mf<T>::make(re, -im), a.twA[k1 * N2 + n2]);
            }
        }
    } else {
        for (int e = wave; e < CA * RT1; e += NW) {
            const int ct = e / RT1, rt = e - ct * RT1;
            V4 re, im;
            sums_a(ct, rt, re, im);
            put_a(ct, rt, re, im);
        }
    }
    __syncthreads();
    // ---- step C
    const int H2 = N2 / 2 + 1, RT2 = (H2 + 15) / 16, CC = (LB * K1 + 15) / 16;
    auto put_c = [&](int ct, int rt, const DctSums<T> &s) {
        const int col = ct * 16 + c16, ln = col / K1, k1 = col - ln * K1;
        if (col >= LB * K1) return;
        auto put = [&](int k2, T re, T im) {
            const int k = k1 + N1 * k2;
            const T2 wv = cmul(a.rot[k], Mf<T>::make(re, im));
            v[ln * N + k] = 2 * wv.x;
            // the mirror N - k of k1 = 0 and k1 = N1/2 is one of their own outputs
            if (k1 != 0 && 2 * k1 != N1) v[ln * N + N - k] = -2 * wv.y;
        };
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int k2 = 16 * rt + Mf<T>::row(q, r);
            if (k2 >= H2) continue;
            put(k2, s.cr[r] + s.si[r], s.ci[r] - s.sr[r]);
            if (k2 != 0 && 2 * k2 != N2) put(N2 - k2, s.cr[r] - s.si[r], s.ci[r] + s.sr[r]);
        }
    };
    auto sums_c = [&](int ct, int rt) {
        const int col = ct * 16 + c16, ln = col / K1, k1 = col - ln * K1;
        const T2 *Bl = Bc + (ln * K1 + k1) * ld;
        return N1 == 1 ? dct_sums<true>(a, Bl, col < LB * K1, rt, q, lane)
                       : dct_sums<false>(a, Bl, col < LB * K1, rt, q, lane);
    };
    if constexpr (SMALL) {
        const DctSums<T> s = sums_c(wave, 0);
        __syncthreads();  // Bc is read; v overwrites it
        put_c(wave, 0, s);
    } else {
        for (int e = wave; e < CC * RT2; e += NW) {
            const int ct = e / RT2, rt = e - ct * RT2;
            put_c(ct, rt, sums_c(ct, rt));
        }
    }
    __syncthreads();
    for (int l = wave; l < LB; l += NW) {
        const int c = line0 + l;
        if (c >= a.C) break;
        T *dst = out + a.out_base + (long long)(c % a.C1) * a.out_c1 + (long long)(c / a.C1) * a.out_c2;
        for (int kx = lane; kx < N; kx += 64) dst[kx] = v[l * N + kx];
    }
}

template <bool SMALL, class T>
__global__ __launch_bounds__(SMALL ? 128 : 512, SMALL ? (sizeof(T) == 4 ? 6 : 5) : 4) void k_dct_inv_m(DctArgs<T> a, const T *__restrict__ in,
                                                                 T *__restrict__ out) {
    extern __shared__ double2 smem16[];
    typedef typename Mf<T>::T2 T2;
    typedef typename Mf<T>::V4 V4;
    T2 *smem2 = reinterpret_cast<T2 *>(smem16);
    const int NW = SMALL ? 2 : blockDim.x >> 6;
    const int N = a.N, N1 = a.N1, N2 = a.N2, K1 = a.K1h + 1, LB = SMALL ? 2 : a.LB, ld = dct_ld(N2);
    const float rK1 = 1.0f / (float)K1;
    // SMALL: one area for V, C~ and the output lines in turn; otherwise V (later
    // the lines, which are no longer) and C~ apart
    T2 *Vs = smem2, *Cs = SMALL ? smem2 : smem2 + LB * K1 * ld;
    T *o = reinterpret_cast<T *>(smem2);
    const int tid = threadIdx.x, lane = tid & 63, q = lane >> 4, c16 = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int line0 = blockIdx.x * LB;
    // V[k1 + N1 k2] = conj(rot_k) (g[k] - i g[N-k]) / 2 for k1 <= N1/2: Vs[l][k1][k2],
    // a line per wave, k1 fastest over the lanes (runs of K1 consecutive entries of
    // the line), kLd elements per lane loaded before the first is used
    const int nv = K1 * N2;
    for (int l = wave; l < LB; l += NW) {
        const int c = min(line0 + l, a.C - 1);
        const T *g = in + a.in_base + (long long)(c % a.C1) * a.in_c1 + (long long)(c / a.C1) * a.in_c2;
        for (int i0 = lane; i0 < nv; i0 += 64 * kLd) {
            T gk[kLd], gm[kLd];
            T2 rt[kLd];
#pragma unroll
            for (int u = 0; u < kLd; ++u) {
                const int r = min(i0 + 64 * u, nv - 1), k2 = small_div(r, rK1), k1 = r - k2 * K1;
                const int k = k1 + N1 * k2;
                gk[u] = g[k];
                gm[u] = g[k == 0 ? 0 : N - k];
                rt[u] = a.rot[k];
                if (k == 0) gm[u] = 0;
            }
#pragma unroll
            for (int u = 0; u < kLd; ++u) {
                const int r = i0 + 64 * u, k2 = small_div(r, rK1), k1 = r - k2 * K1;
                if (r < nv)
                    Vs[(l * K1 + k1) * ld + k2] = cmulc(Mf<T>::make((T)0.5 * gk[u], (T)-0.5 * gm[u]), rt[u]);
            }
        }
    }
    __syncthreads();
    // ---- step C': C~[k1][n2] = W_N^{-n2 k1} sum_k2 V W_N2^{-n2 k2}
    const int H2 = N2 / 2 + 1, RT2 = (H2 + 15) / 16, CC = (LB * K1 + 15) / 16;
    auto sums_c = [&](int ct, int rt) {
        const int col = ct * 16 + c16, ln = col / K1, k1 = col - ln * K1;
        return dct_sums<false>(a, Vs + (ln * K1 + k1) * ld, col < LB * K1, rt, q, lane);
    };
    auto put_c = [&](int ct, int rt, const DctSums<T> &s) {
        const int col = ct * 16 + c16, ln = col / K1, k1 = col - ln * K1;
        if (col >= LB * K1) return;
        auto put = [&](int n2, T re, T im) {
            Cs[(ln * K1 + k1) * ld + n2] = cmulc(Mf<T>::make(re, im), a.twC[n2 * K1 + k1]);
        };
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int n2 = 16 * rt + Mf<T>::row(q, r);
            if (n2 >= H2) continue;
            put(n2, s.cr[r] - s.si[r], s.ci[r] + s.sr[r]);
            if (n2 != 0 && 2 * n2 != N2) put(N2 - n2, s.cr[r] + s.si[r], s.ci[r] - s.sr[r]);
        }
    };
    if constexpr (SMALL) {
        const DctSums<T> s = sums_c(wave, 0);
        __syncthreads();  // Vs is read; Cs overwrites it
        put_c(wave, 0, s);
    } else {
        for (int e = wave; e < CC * RT2; e += NW) {
            const int ct = e / RT2, rt = e - ct * RT2;
            put_c(ct, rt, sums_c(ct, rt));
        }
    }
    __syncthreads();
    // ---- step A'
    const int KS1 = (K1 + 3) / 4, RT1 = (K1 + 15) / 16, CA = (LB * N2 + 15) / 16;
    auto sums_a = [&](int ct, int rt, V4 &p, V4 &s) {
        const int col = ct * 16 + c16, ln = col / N2, n2 = col - ln * N2;
        const bool cok = col < LB * N2;
        const T2 *cl = Cs + ln * K1 * ld + n2;
        const T2 *t = a.t1i + rt * KS1 * 64 + lane;
        p = s = V4{0, 0, 0, 0};
        for (int k0 = (KS1 - 1) / 4 * 4; k0 >= 0; k0 -= 4) {  // the large end last, as in dct_sums
            T2 w[4], x[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int k1 = 4 * (k0 + u) + q;
                w[u] = t[min(k0 + u, KS1 - 1) * 64];
                x[u] = Mf<T>::make(0, 0);
                if (cok && k1 < K1) x[u] = cl[k1 * ld];
            }
#pragma unroll
            for (int u = 3; u >= 0; --u) {
                if (k0 + u >= KS1) continue;
                p = Mf<T>::mul(w[u].x, x[u].x, p);
                s = Mf<T>::mul(w[u].y, x[u].y, s);
            }
        }
    };
    auto put_a = [&](int ct, int rt, const V4 &p, const V4 &s) {
        const int col = ct * 16 + c16, ln = col / N2, n2 = col - ln * N2;
        if (col >= LB * N2) return;
        auto put = [&](int n1, T x) {
            const int n = N2 * n1 + n2;
            const int pos = (n < (N + 1) / 2) ? 2 * n : 2 * (N - 1 - n) + 1;
            o[ln * N + pos] = x * a.scale;
        };
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int n1 = 16 * rt + Mf<T>::row(q, r);
            if (n1 >= K1) continue;
            put(n1, p[r] - s[r]);
            if (n1 != 0 && 2 * n1 != N1) put(N1 - n1, p[r] + s[r]);
        }
    };
    if constexpr (SMALL) {
        V4 p[2], s[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) sums_a(2 * wave + h, 0, p[h], s[h]);
        __syncthreads();  // Cs is read; o overwrites it
#pragma unroll
        for (int h = 0; h < 2; ++h) put_a(2 * wave + h, 0, p[h], s[h]);
    } else if (N1 == 1) {
        for (int e = tid; e < LB * N; e += blockDim.x) {
            const int ln = e / N, n = e - ln * N;
            o[ln * N + ((n < (N + 1) / 2) ? 2 * n : 2 * (N - 1 - n) + 1)] = Cs[ln * ld + n].x * a.scale;
        }
    } else if (K1 <= kDctShort) {  // a column per thread, as in k_dct_fwd_m
        for (int e = tid; e < LB * N2; e += blockDim.x) {
            const int ln = e / N2, n2 = e - ln * N2;
            const T2 *cl = Cs + ln * K1 * ld + n2;
            T2 x[kDctShort];
#pragma unroll
            for (int k1 = 0; k1 < kDctShort; ++k1) x[k1] = k1 < K1 ? cl[k1 * ld] : Mf<T>::make(0, 0);
            auto put = [&](int n1, T y) {
                const int n = N2 * n1 + n2;
                o[ln * N + ((n < (N + 1) / 2) ? 2 * n : 2 * (N - 1 - n) + 1)] = y * a.scale;
            };
#pragma unroll
            for (int n1 = 0; n1 < kDctShort; ++n1) {
                if (n1 >= K1) continue;
                T p = 0, s = 0;
#pragma unroll
                for (int k1 = kDctShort - 1; k1 >= 0; --k1) {
                    const T2 w = a.t1i[16 * k1 + n1];
                    p = fma(w.x, x[k1].x, p);
                    s = fma(w.y, x[k1].y, s);
                }
                put(n1, p - s);
                if (n1 != 0 && 2 * n1 != N1) put(N1 - n1, p + s);
            }
        }
    } else {
        for (int e = wave; e < CA * RT1; e += NW) {
            const int ct = e / RT1, rt = e - ct * RT1;
            V4 p, s;
            sums_a(ct, rt, p, s);
            put_a(ct, rt, p, s);
        }
    }
    __syncthreads();
    for (int l = wave; l < LB; l += NW) {
        const int c = line0 + l;
        if (c >= a.C) break;
        T *dst = out + a.out_base + (long long)(c % a.C1) * a.out_c1 + (long long)(c / a.C1) * a.out_c2;
        const T ad = a.add ? (T)a.add[c % a.C1] : (T)0;
        for (int n = lane; n < N; n += 64) dst[n] = a.add ? o[l * N + n] + ad : o[l * N + n];
    }
}

// ------------------------------------------------------------------------
// The folded real z DFT above on the FP64 matrix cores, for M/2 + 1 <= 96
// rows.  Both directions are two real products D = A B over the folded
// index kk = 0..M/2 with A[row][kk] = cos or sin(2 pi row kk / M), the entry
// (row kk) mod M of a single M-point table:
//   forward  B = e[kk], o[kk] (the pairs T[kk] +- T[M-kk]); rows k give
//            Re X_k and -Im X_k;
//   inverse  B = R[k], I[k] (the Hermitian-weighted Re and Im rows); rows m
//            give c[m], s[m], and g[m] = c - s, g[M-m] = c + s.
// The products run in kk order, so the sums are those of the VALU kernels
// bit for bit.  A block holds every A fragment (cos, sin) in LDS in lane
// order (RT x KS x 64 pairs, 144 KB at M = 191; the table zf of
// z_dft_tables) and its waves loop over
// 16-column tiles, each owning every row tile of both products for its
// columns; the raw inputs of the next kZmPF k steps (into the next tile at
// the end of one) are loaded ahead.
// ------------------------------------------------------------------------
constexpr int kZmRT = 6, kZmKS = 24, kZmPF = 4, kZmW = 8;

// RT = (M/2 + 1 + 15) / 16 row tiles
template <bool FWD, int RT>
__global__ __launch_bounds__(64 * kZmW) void k_zdft_mf(int M, int C, long long plane,
                                                       const double2 *__restrict__ zf,
                                                       const double *__restrict__ in,
                                                       double *__restrict__ out) {
    __shared__ double2 sA[RT * kZmKS * 64];
    const int hm = M / 2, Kc = hm + 1, KS = (Kc + 3) / 4;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r16 = lane & 15, q4 = lane >> 4;
    // fragment (t, ks), lane l: A[16 t + l % 16][4 ks + l / 16] as (cos, sin),
    // built on the host in this order (zf)
    for (int e = threadIdx.x; e < RT * KS * 64; e += 64 * kZmW) sA[e] = zf[e];
    __syncthreads();
    // A wave takes tile after tile; the last, partial round goes to the first waves
    // of all blocks instead of all waves of the first ones (812x256x191: the
    // busiest SIMDs do 13 tiles instead of 14; 191 -> 180 and 200 -> 187 us,
    // 511x96x128 46 -> 38 and 44 -> 37).  A first round that is the only one keeps
    // neighbouring tiles in one block.
    const int ntile = (C + 15) / 16, stride = gridDim.x * kZmW;
    auto tile_of = [&](int base) {
        return base == 0 || base + stride <= ntile ? base + (int)blockIdx.x * kZmW + wave
                                                   : base + wave * (int)gridDim.x + (int)blockIdx.x;
    };
    int base = 0, tile = tile_of(0);
    if (tile >= ntile) return;
    // k steps past M/2 multiply zeros
    const int KSr = (KS + kZmPF - 1) / kZmPF * kZmPF;
    // raw inputs of folded index kk = 4 ks + q4 of tile tl (rows clamped to
    // M/2, columns to C - 1); the loads are unconditional and masked only
    // where they are used, so that those issued ahead stay in flight
    auto raw = [&](int tl, int ks, double &a, double &b) {
        const int kk = min(4 * ks + q4, hm);
        const bool single = kk == 0 || 2 * kk == M;
        int ra, rb;
        if (FWD) {
            ra = kk;
            rb = single ? kk : M - kk;
        } else {
            ra = kk == 0 ? 0 : (2 * kk == M ? M - 1 : 2 * kk - 1);
            rb = single ? ra : 2 * kk;
        }
        const double *src = in + min(16 * tl + r16, C - 1);
        a = src[(long long)ra * plane];
        b = src[(long long)rb * plane];
    };
    double pa[kZmPF], pb[kZmPF];
#pragma unroll
    for (int u = 0; u < kZmPF; ++u) raw(tile, u, pa[u], pb[u]);

    for (int next; tile < ntile; tile = next) {
        base += stride;
        next = tile_of(base);
        const int ahead = min(next, ntile - 1);
        dbl4 ac[RT], as[RT];
#pragma unroll
        for (int t = 0; t < RT; ++t) {
            ac[t] = dbl4{0.0, 0.0, 0.0, 0.0};
            as[t] = dbl4{0.0, 0.0, 0.0, 0.0};
        }
        for (int ks0 = 0; ks0 < KSr; ks0 += kZmPF) {
#pragma unroll
            for (int u = 0; u < kZmPF; ++u) {
                const int ks = ks0 + u;
                const int kk = 4 * ks + q4;
                const bool live = kk <= hm, single = kk == 0 || 2 * kk == M;
                const double a = live ? pa[u] : 0.0, b = live && !single ? pb[u] : 0.0;
                // ahead: k step ks + kZmPF of this tile, or of the next one
                const int kn = ks + kZmPF;
                const bool here = kn < KSr;
                raw(here ? tile : ahead, here ? kn : kn - KSr, pa[u], pb[u]);
                double bc, bs;
                if (FWD) {
                    bc = a + b;                  // b = 0 for the single elements
                    bs = single ? 0.0 : a - b;
                } else {
                    bc = single ? a : 2.0 * a;   // R: weight 1 for k = 0 and the Nyquist row
                    bs = 2.0 * b;                // I: b = 0 there
                }
                // A fragments of this step (clamped to the table: steps past
                // M/2 multiply zero operands)
                const double2 *fa = sA + min(ks, KS - 1) * 64 + lane;
#pragma unroll
                for (int t = 0; t < RT; ++t) {
                    const double2 w = fa[t * KS * 64];
                    ac[t] = mfma64(w.x, bc, ac[t]);
                    as[t] = mfma64(w.y, bs, as[t]);
                }
            }
        }
        const int col = 16 * tile + r16;
        if (col < C) {
            double *dst = out + col;
#pragma unroll
            for (int t = 0; t < RT; ++t) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int row = 16 * t + q4 + 4 * r;
                    if (row > hm) continue;
                    const double c = ac[t][r], s = as[t][r];
                    if (FWD) {
                        dst[(long long)(row == 0 ? 0 : 2 * row - 1) * plane] = c;
                        if (row >= 1 && 2 * row <= M - 1) dst[(long long)(2 * row) * plane] = -s;
                    } else {
                        dst[(long long)row * plane] = c - s;
                        if (row >= 1 && M - row != row) dst[(long long)(M - row) * plane] = c + s;
                    }
                }
            }
        }
    }
}

// Thomas sweep with precomputed factors (projection.f90:137-150).  One real
// system (kx, q) per lane: q = 0 is the kz = 0 row, q = 2k-1 / 2k the real /
// imaginary rows of wavenumber k, which share the factors of k.  The sweep is
// unrolled by TJ rows so that the loads of a chunk are issued together.
template <int TJ>
__global__ __launch_bounds__(256) void k_thomas(Dims d, const double *__restrict__ dl,
                                                const double *__restrict__ dp,
                                                const double *__restrict__ du, double *S) {
    const int N = d.N, NM = d.NM;
    int kxb, q;
    thomas_block(blockIdx.x, (N + 255) / 256, d.M, kxb, q);
    const int kx = kxb * 256 + threadIdx.x;
    if (kx >= N) return;
    const long long plane = (long long)N * NM;
    const int kk = (q + 1) / 2;
    double *a = S + q * plane + kx;
    const double *L = dl + kk * plane + kx;
    const double *D = dp + kk * plane + kx;
    // forward elimination with the stored multipliers
    double r = a[0];
    int j = 1;
    for (; j + TJ <= NM; j += TJ) {
        double x[TJ], l[TJ];
#pragma unroll
        for (int t = 0; t < TJ; ++t) {
            x[t] = a[(long long)(j + t) * N];
            l[t] = L[(long long)(j + t - 1) * N];
        }
#pragma unroll
        for (int t = 0; t < TJ; ++t) {
            r = x[t] - l[t] * r;
            x[t] = r;
        }
#pragma unroll
        for (int t = 0; t < TJ; ++t) a[(long long)(j + t) * N] = x[t];
    }
    for (; j < NM; ++j) {
        r = a[(long long)j * N] - L[(long long)(j - 1) * N] * r;
        a[(long long)j * N] = r;
    }
    // back substitution with the stored reciprocal pivots
    r = r * D[(long long)(NM - 1) * N];
    a[(long long)(NM - 1) * N] = r;
    j = NM - 2;
    for (; j - TJ + 1 >= 0; j -= TJ) {
        double x[TJ], p[TJ], u[TJ];
#pragma unroll
        for (int t = 0; t < TJ; ++t) {
            x[t] = a[(long long)(j - t) * N];
            p[t] = D[(long long)(j - t) * N];
            u[t] = du[j - t];
        }
#pragma unroll
        for (int t = 0; t < TJ; ++t) {
            r = (x[t] - u[t] * r) * p[t];
            x[t] = r;
        }
#pragma unroll
        for (int t = 0; t < TJ; ++t) a[(long long)(j - t) * N] = x[t];
    }
    for (; j >= 0; --j) {
        r = (a[(long long)j * N] - du[j] * r) * D[(long long)j * N];
        a[(long long)j * N] = r;
    }
}

// 1/x for the normal, finite pivots of the Thomas sweeps: the hardware
// reciprocal refined by two Newton steps (within an ulp or so of the rounded
// quotient, without the special-case scaling of a full division)
__device__ __forceinline__ double rcp64(double x) {
    double r = __builtin_amdgcn_rcp(x);
    double e = fma(-x, r, 1.0);
    r = fma(r, e, r);
    e = fma(-x, r, 1.0);
    return fma(r, e, r);
}

typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

template <int NMAX>
__device__ void solve00_block(const Solve00 &z, int NM);

// Partitioned Thomas solve held in registers (the systems of
// projection.f90:137-150, factors formed on the fly instead of read from
// tables).  A block is P waves; wave p holds rows [32 p, 32 p + 32) of the 64
// systems (q, kx0 + lane), so S is read and written once.  Per segment:
//   LU sweep (top-down): reciprocal pivots ip (kept), y_last, and the last
//     row's responses to the left and right neighbour values xL, xR;
//   UL sweep (bottom-up, nothing kept): y_first and the first row's responses;
// with x = y + alpha xL + beta xR on the segment ends, the 2P interface
// values follow from a two-term recurrence over the segments (every lane
// runs it for its own system), and the segment is solved again with the
// neighbour values moved to its right-hand side.  Rows past NM stand alone
// (a = c = 0, b = -1: the pivot b + kxx + kzz <= -1).  co = {a[L], b[L], c[L], kxx[N], kzz[Kz]},
// L = 32 P: a[j] couples x(j-1), c[j] couples x(j+1), b[j] + kxx + kzz is
// the diagonal.  The (0,0) system (kx = 0, q = 0, pinned first pivot) is
// skipped (zero00 = 0) or zeroed (zero00 = 1); block 0 solves it (z) while
// the other blocks run.  The other blocks, as many as reside (thomas_resident:
// up to eight waves a CU, four with one segment), loop over the nq * ceil(N/64)
// tiles of 64 systems.
// A tile's time is that of its loads plus that of its arithmetic (the waves of
// a CU go through both together).  The coefficients come from LDS, a row is a
// scalar offset into a buffer and no row is masked: with scalar coefficient
// loads and guarded rows 900 of the 2500 instructions were scalar register
// spills and selects.  At 511x96x128 45 -> 30 us (with more than one block a CU),
// 260x65x228 FP32 39 -> 24, 812x256x191 FP32 117 -> 109, FP64 156 -> 152, on
// 255x96x62 and 127x48x32 FP32 27 -> 13 and 19 -> 10 (with the sums of block 0).
template <class T>
__global__ __launch_bounds__(64 * kThMaxP) void k_thomas_seg(int N, int NM, int P, int nq, int ldj, long long ldq,
                                                             const double *__restrict__ co, int zero00,
                                                             T *__restrict__ S, Solve00 z) {
    __shared__ double xs[6][kThMaxP][64];
    __shared__ double ca[kThSeg * kThMaxP], cb[kThSeg * kThMaxP], cc[kThSeg * kThMaxP];
    static_assert(sizeof(xs) + 8 * sizeof(ca) == kThomasLds, "the residency rule counts this and solve00_block's rows");
    if (blockIdx.x == 0) {  // the (0,0) system, alongside the other blocks
        solve00_block<kThSeg * kThMaxP>(z, NM);
        return;
    }
    const int lane = threadIdx.x & 63;
    const int p = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nkb = (N + 63) / 64, ntiles = nkb * nq, nblk = gridDim.x - 1;
    const int L = P * kThSeg;
    const int r0 = p * kThSeg;
    for (int e = threadIdx.x; e < L; e += blockDim.x) {
        ca[e] = co[e];
        cb[e] = co[L + e];
        cc[e] = co[2 * L + e];
    }
    __syncthreads();
    const unsigned rowb = (unsigned)ldj * (unsigned)sizeof(T);  // a plane is below 4 GB
    // tiles (q, 64 kx) bid, bid + nblk, ... (holding the next tile's rows
    // in registers during a solve spills them)
    for (int tile = blockIdx.x - 1; tile < ntiles; tile += nblk) {
        const int q = tile / nkb;
        const int kx = (tile - q * nkb) * 64 + lane;
        const bool live = kx < N;
        const int kxc = live ? kx : N - 1;
        const double lam = co[3 * L + kxc] + co[3 * L + N + (q + 1) / 2];
        const unsigned vo = (unsigned)kxc * (unsigned)sizeof(T);
        // rows of the segment left below NM; hidden from the compiler, which would
        // keep the comparison with each row across the tiles
        int left = NM - r0;
        asm volatile("" : "+s"(left));
        // the q plane as a buffer: a row is a scalar offset
        const auto rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)(S + q * ldq), 0, (int)((unsigned)NM * rowb), 0x00020000);
        const unsigned row0 = (unsigned)min(r0, NM - 1) * rowb;
        double dv[kThSeg], ip[kThSeg];
        {
            // unconditional loads (rows past NM repeat the last one, their
            // systems are apart), all issued before the first conversion waits
            T raw[kThSeg];
            unsigned ro = row0;
#pragma unroll
            for (int i = 0; i < kThSeg; ++i) {
                if constexpr (sizeof(T) == 4)
                    raw[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, vo, ro, 0));
                else
                    raw[i] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rsrc, vo, ro, 0));
                ro += i + 1 < left ? rowb : 0u;
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < kThSeg; ++i) dv[i] = (double)raw[i];
        }
        // LU (index i) and UL (index kThSeg-1-i) sweeps, interleaved
        double dp = dv[0], s = 1.0;
        ip[0] = rcp64(cb[r0] + lam);
        double iu = rcp64(cb[r0 + kThSeg - 1] + lam), du = dv[kThSeg - 1], t = 1.0;
#pragma unroll
        for (int i = 1; i < kThSeg; ++i) {
            const int j = r0 + i;
            const double m = ca[j] * ip[i - 1];
            ip[i] = rcp64(cb[j] + lam - m * cc[j - 1]);
            dp = dv[i] - m * dp;
            s = -m * s;
            const int iv = kThSeg - 1 - i, jv = r0 + iv;
            const double mu = cc[jv] * iu;
            iu = rcp64(cb[jv] + lam - mu * ca[jv + 1]);
            du = dv[iv] - mu * du;
            t = -mu * t;
            if (i % 4 == 0) __builtin_amdgcn_sched_barrier(0);
        }
        const double aL = ca[r0], cR = cc[r0 + kThSeg - 1];
        xs[0][p][lane] = du * iu;                        // y first
        xs[1][p][lane] = -aL * iu;                       // d x_first / d xL
        xs[2][p][lane] = -cR * t * iu;                   // d x_first / d xR
        xs[3][p][lane] = dp * ip[kThSeg - 1];            // y last
        xs[4][p][lane] = -aL * s * ip[kThSeg - 1];       // d x_last / d xL
        xs[5][p][lane] = -cR * ip[kThSeg - 1];           // d x_last / d xR
        __syncthreads();
        // segment ends: A_p (first row), B_p (last row); B_{p-1} = u + v A_p
        double g[kThMaxP], hh[kThMaxP];
        double u = 0.0, v = 0.0, ul = 0.0, vl = 0.0;  // (ul, vl): B_{p-1} = ul + vl A_p
#pragma unroll
        for (int pp = 0; pp < kThMaxP; ++pp) {
            if (pp < P) {
                if (pp == p) {
                    ul = u;
                    vl = v;
                }
                const double a0 = xs[1][pp][lane], an = xs[4][pp][lane];
                const double den = 1.0 / (1.0 - a0 * v);
                g[pp] = (xs[0][pp][lane] + a0 * u) * den;
                hh[pp] = xs[2][pp][lane] * den;
                const double un = xs[3][pp][lane] + an * (u + v * g[pp]);
                v = an * v * hh[pp] + xs[5][pp][lane];
                u = un;
            }
        }
        __syncthreads();  // xs is read; the next tile writes it
        double Anext = 0.0, xL = 0.0, xR = 0.0;
#pragma unroll
        for (int pp = kThMaxP - 1; pp >= 0; --pp) {
            if (pp < P) {
                const double Ap = g[pp] + hh[pp] * Anext;
                if (pp == p + 1) xR = Ap;
                if (pp == p) xL = ul + vl * Ap;
                Anext = Ap;
            }
        }
        // the segment with its neighbour values on the right-hand side
        dv[0] -= aL * xL;
        dv[kThSeg - 1] -= cR * xR;
#pragma unroll
        for (int i = 1; i < kThSeg; ++i) {
            dv[i] -= ca[r0 + i] * ip[i - 1] * dv[i - 1];
            if (i % 8 == 0) __builtin_amdgcn_sched_barrier(0);
        }
        dv[kThSeg - 1] *= ip[kThSeg - 1];
#pragma unroll
        for (int i = kThSeg - 2; i >= 0; --i) {
            dv[i] = (dv[i] - cc[r0 + i] * dv[i + 1]) * ip[i];
            if (i % 8 == 0) __builtin_amdgcn_sched_barrier(0);
        }
        const bool is00 = q == 0 && kx == 0;
        if (is00 && zero00)
#pragma unroll
            for (int i = 0; i < kThSeg; ++i) dv[i] = 0.0;
        if (live && !(is00 && !zero00)) {
            unsigned ro = row0;
            asm volatile("" : "+s"(left));
            if (left >= kThSeg) left = kThSeg;
#pragma unroll
            for (int i = 0; i < kThSeg; ++i) {
                if (i < left) {
                    if constexpr (sizeof(T) == 4)
                        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, (T)dv[i]), rsrc, vo, ro, 0);
                    else
                        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, (T)dv[i]), rsrc, vo, ro, 0);
                }
                ro += rowb;
            }
        }
    }
}

// The pinned (0,0) system (kx = 0, kz = 0) in place in z.x (row stride
// z.ldx), scaled by z.scale: one lane, in the elimination order of the
// table kernel, from LDS copies of the stored multipliers L00 and reciprocal
// pivots D00.  With z.part set, the right-hand side is first formed as
// r(j) = 2 sum_q part[j][q] (the FP64 plane sums of the mixed path's
// divergence), 16 lanes per row.  The sweeps read one array and write
// another, so that the LDS reads of the unrolled iterations are issued ahead
// of the dependent chain.  Any block size that is a multiple of 64.
template <int NMAX>
__device__ void solve00_block(const Solve00 &z, int NM) {
    __shared__ double r[NMAX], o[NMAX], L[NMAX], D[NMAX], U[NMAX];
    const int tid = threadIdx.x, nt = blockDim.x;
    if (z.part) {
        // 16 lanes a row, 32 rows of a wave at a time: their loads are in flight
        // together (one row after the other waited 0.6 us for each, 20 us for 96
        // rows on three waves, longer than the other blocks take there)
        const int lane = tid & 63, l16 = lane & 15;
        for (int j0 = (tid >> 6) * 32; j0 < NM; j0 += (nt >> 6) * 32) {
            const int j = j0 + (lane >> 4);
            double v[8];
#pragma unroll
            for (int t = 0; t < 8; ++t) v[t] = 0.0;
#pragma unroll 2
            for (int q = l16; q < z.npart; q += 16)
#pragma unroll
                for (int t = 0; t < 8; ++t) v[t] += z.part[(long long)min(j + 4 * t, NM - 1) * z.npart + q];
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                for (int off = 8; off > 0; off >>= 1) v[t] += __shfl_xor(v[t], off);
                if (l16 == 0 && j + 4 * t < NM) r[j + 4 * t] = 2.0 * v[t];
            }
        }
    } else {
        for (int j = tid; j < NM; j += nt) r[j] = z.x[(long long)j * z.ldx];
    }
    for (int j = tid; j < NM; j += nt) {
        L[j] = j > 0 ? z.L00[j - 1] : 0.0;
        D[j] = z.D00[j];
        U[j] = z.du[j];
    }
    __syncthreads();
    if (tid == 0) {
        double v = r[0];
        o[0] = v;
#pragma unroll 8
        for (int j = 1; j < NM; ++j) {
            v = r[j] - L[j] * v;
            o[j] = v;
        }
        v *= D[NM - 1];
        r[NM - 1] = v;
#pragma unroll 8
        for (int j = NM - 2; j >= 0; --j) {
            v = (o[j] - U[j] * v) * D[j];
            r[j] = v;
        }
    }
    __syncthreads();
    for (int j = tid; j < NM; j += nt) z.x[(long long)j * z.ldx] = r[j] * z.scale;
}

__global__ __launch_bounds__(256) void k_solve00(int NM, Solve00 z) { solve00_block<kMax00>(z, NM); }

// ------------------------------------------------------------------------
// Reductions
// ------------------------------------------------------------------------
// block max of non-negative values over 4 waves; the caller stores one
// partial per block and k_reduce_max reduces the partials
__device__ __forceinline__ double block_max_256(double v, double *sh) {
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_down(v, o));
    const int t = threadIdx.x + blockDim.x * threadIdx.y;
    if ((t & 63) == 0) sh[t >> 6] = v;
    __syncthreads();
    return fmax(fmax(sh[0], sh[1]), fmax(sh[2], sh[3]));
}

// max |div u| partials (check_divergence projection.f90:391-413); each field
// has its own row and plane strides (the padded solver layout, or the
// reference's unpadded extents for bl_max_divergence_noalloc)
template <class T>
__global__ __launch_bounds__(256) void k_maxdiv(DivArgs a, const T *U, const T *V, const T *W, double *out) {
    __shared__ double sh[4];
    const int i = blockIdx.x * kWave + threadIdx.x;
    const int j = blockIdx.y * 4 + threadIdx.y + 1;
    double v = 0.0;
    if (i >= 1 && i <= a.nxg - 3 && j <= a.nyg - 2)
        for (int k = 1 + blockIdx.z; k <= a.nzg - 2; k += gridDim.z) {
            const long long pu = i + a.u1 * j + a.u2 * k, pv = i + a.v1 * j + a.v2 * k;
            const long long pw = i + a.w1 * j + a.w2 * k;
            v = fmax(v, fabs(((double)U[pu] - (double)U[pu - 1]) * a.rdx[i] +
                             ((double)V[pv] - (double)V[pv - a.v1]) * a.rdy[j] +
                             ((double)W[pw] - (double)W[pw - a.w2]) * a.rdz[k]));
        }
    v = block_max_256(v, sh);
    const long long bid = blockIdx.x + (long long)gridDim.x * (blockIdx.y + (long long)gridDim.y * blockIdx.z);
    if (threadIdx.x == 0 && threadIdx.y == 0) out[bid] = v;
}

template <class T>
__global__ __launch_bounds__(256) void k_dtconv(Dims d, Metrics m, const T *U, const T *V, const T *W,
                                                double *out) {
    __shared__ double sh[3][4];
    const int i = blockIdx.x * kWave + threadIdx.x;
    const int j = blockIdx.y * 4 + threadIdx.y + 1;
    double a = 0.0, b = 0.0, c = 0.0;
    if (i >= 1 && i <= d.nxg - 2 && j <= d.nyg - 2) {
        const double dxi = m.xg[i + 1] - m.xg[i], dyj = m.yg[j + 1] - m.yg[j];
        const int gz = gridDim.z;
        // four of the thread's planes loaded before the first is used
        for (int k0 = 1 + blockIdx.z; k0 <= d.nzg - 2; k0 += 4 * gz) {
            T u[4], v[4], w[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const long long p = fidx(d, i, j, min(k0 + r * gz, d.nzg - 2));
                u[r] = U[p];
                v[r] = V[p];
                w[r] = W[p];
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int k = k0 + r * gz;
                if (k > d.nzg - 2) break;
                a = fmax(a, dxi / fabs((double)u[r]));
                b = fmax(b, dyj / fabs((double)v[r]));
                c = fmax(c, (m.zg[k + 1] - m.zg[k]) / fabs((double)w[r]));
            }
        }
    }
    a = block_max_256(a, sh[0]);
    b = block_max_256(b, sh[1]);
    c = block_max_256(c, sh[2]);
    const long long bid = blockIdx.x + (long long)gridDim.x * (blockIdx.y + (long long)gridDim.y * blockIdx.z);
    if (threadIdx.x == 0 && threadIdx.y == 0) {
        out[3 * bid + 0] = a;
        out[3 * bid + 1] = b;
        out[3 * bid + 2] = c;
    }
}

// max over n partial values part[c + stride*q] for c < ncomp, one block
__global__ __launch_bounds__(1024) void k_reduce_max(const double *part, long long n, int ncomp,
                                                     double *out) {
    __shared__ double sh[1024];
    for (int c = 0; c < ncomp; ++c) {
        double v = 0.0;
        for (long long q = threadIdx.x; q < n; q += 1024) v = fmax(v, part[c + ncomp * q]);
        sh[threadIdx.x] = v;
        __syncthreads();
        for (int st = 512; st > 0; st >>= 1) {
            if ((int)threadIdx.x < st) sh[threadIdx.x] = fmax(sh[threadIdx.x], sh[threadIdx.x + st]);
            __syncthreads();
        }
        if (threadIdx.x == 0) out[c] = sh[0];
        __syncthreads();
    }
}

// Cf(x) (statistics.f90:137-160).  64 x faces by 16 groups of z planes per
// block, whose seven sums meet in LDS in a fixed order; one thread per face
// walking every plane was a serial chain of 191 loads in four blocks at
// 814x257x193 (0.116 -> 0.022 ms).
constexpr int kWsZ = 16;
template <class T>
__global__ __launch_bounds__(64 * kWsZ) void k_wallstats(Dims d, Metrics m, double nu, const T *U, const T *V,
                                                         const T *nu_t, double *cf) {
    __shared__ double sh[7][kWsZ][64];
    const int tx = threadIdx.x & 63, g = threadIdx.x >> 6, i = blockIdx.x * 64 + tx;
    const double nz2 = (double)(d.nzg - 2);
    // the x neighbour of the last station is column nxg of nu_t_mean, which
    // compute_statistics never fills (statistics.f90:77 runs ii = 1..nx): 0
    const bool last = i >= d.nx - 1;
    double s[7] = {0, 0, 0, 0, 0, 0, 0};  // u1, u2, uv, n1a, n2a, n1b, n2b
    if (i < d.nx)
        for (int k = 1 + g; k <= d.nzg - 2; k += kWsZ) {
            const long long p = fidx(d, i, 0, k);
            const double a = (double)U[p], b = (double)U[p + d.sx];
            s[0] += a;
            s[1] += b;
            s[2] += (m.wy0[0] * a + m.wy1[0] * b) * (0.5 * ((double)V[p] + (double)V[p + 1]));
            s[3] += (double)nu_t[p];
            s[4] += (double)nu_t[p + d.sx];
            if (!last) {
                s[5] += (double)nu_t[p + 1];
                s[6] += (double)nu_t[p + 1 + d.sx];
            }
        }
#pragma unroll
    for (int q = 0; q < 7; ++q) sh[q][g][tx] = s[q];
    __syncthreads();
    if (g != 0 || i >= d.nx) return;
#pragma unroll
    for (int q = 0; q < 7; ++q) {
        s[q] = 0.0;
        for (int r = 0; r < kWsZ; ++r) s[q] += sh[q][r][tx];
    }
    const double dudy = (s[1] / nz2 - s[0] / nz2) / (m.yg[1] - m.yg[0]);
    const double tau = 0.25 * (s[3] / nz2 + s[4] / nz2 + s[5] / nz2 + s[6] / nz2) * dudy;
    cf[i] = 2.0 * (-(s[2] / nz2) + nu * dudy + tau) / 1.0;
}

// sums and maxima of the four monitored interiors (monitor.f90:29-52): eight
// partials per block of kMonJ rows of one plane, then k_monitor_reduce.  Bound
// by the read of the four fields (1.3 GB, 0.25 ms of HBM time at 814x257x193);
// one block per plane left the chip idle and took 1.71 ms, this form 0.23.
constexpr int kMonJ = 8;
template <class T>
__global__ __launch_bounds__(256) void k_monitor(Dims d, const T *__restrict__ U, const T *__restrict__ V,
                                                 const T *__restrict__ W, const T *__restrict__ nu_t,
                                                 double *__restrict__ part) {
    const int k = blockIdx.y + 1;  // plane
    __shared__ double sh[8][4];
    double s[4] = {0, 0, 0, 0}, mx[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
    const int j0 = 1 + blockIdx.x * kMonJ;
    for (int i = threadIdx.x; i <= d.nxg - 2; i += 256) {  // from 0, so that a wave's row starts on a 128-byte line
        T u[kMonJ], v[kMonJ], w[kMonJ], n[kMonJ];
#pragma unroll
        for (int r = 0; r < kMonJ; ++r) {
            const long long p = fidx(d, i, min(j0 + r, d.nyg - 2), k);
            u[r] = U[p];
            v[r] = V[p];
            w[r] = W[p];
            n[r] = nu_t[p];
        }
#pragma unroll
        for (int r = 0; r < kMonJ; ++r) {
            const int j = j0 + r;
            if (i < 1 || j > d.nyg - 2) continue;
            if (i <= d.nx - 2) {
                s[0] += (double)u[r];
                mx[0] = fmax(mx[0], (double)u[r]);
            }
            if (j <= d.ny - 2) {
                s[1] += (double)v[r];
                mx[1] = fmax(mx[1], (double)v[r]);
            }
            if (k <= d.nz - 2) {
                s[2] += (double)w[r];
                mx[2] = fmax(mx[2], (double)w[r]);
            }
            s[3] += (double)n[r];
            mx[3] = fmax(mx[3], (double)n[r]);
        }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q)
        for (int o = 32; o > 0; o >>= 1) {
            s[q] += __shfl_down(s[q], o);
            mx[q] = fmax(mx[q], __shfl_down(mx[q], o));
        }
    if ((threadIdx.x & 63) == 0)
        for (int q = 0; q < 4; ++q) {
            sh[q][threadIdx.x >> 6] = s[q];
            sh[4 + q][threadIdx.x >> 6] = mx[q];
        }
    __syncthreads();
    if (threadIdx.x < 8) {
        const double *v = sh[threadIdx.x];
        const double r = threadIdx.x < 4 ? (v[0] + v[1]) + (v[2] + v[3]) : fmax(fmax(v[0], v[1]), fmax(v[2], v[3]));
        part[8 * ((long long)blockIdx.x + (long long)gridDim.x * blockIdx.y) + threadIdx.x] = r;
    }
}

// block q reduces quantity q (0-3 sums, 4-7 maxima) of the n partials
__global__ __launch_bounds__(256) void k_monitor_reduce(const double *__restrict__ part, long long n,
                                                        double *__restrict__ out) {
    __shared__ double sh[256];
    const int q = blockIdx.x;
    double v = q < 4 ? 0.0 : -INFINITY;
    for (long long t = threadIdx.x; t < n; t += 256) v = q < 4 ? v + part[8 * t + q] : fmax(v, part[8 * t + q]);
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
        if ((int)threadIdx.x < st) {
            const double b = sh[threadIdx.x + st];
            sh[threadIdx.x] = q < 4 ? sh[threadIdx.x] + b : fmax(sh[threadIdx.x], b);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) out[q] = sh[0];
}

// reductions: each thread walks z planes with stride kRedZ, so the partials
// per launch are kRedZ times fewer than the interior blocks; x tiles cover
// cells 64 bx .. 64 bx + 63 (cell 0 idle) so that rows start on a 128-byte line
constexpr int kRedZ = 12;
dim3 reduce_grid(const Dims &d) {
    return dim3((d.nxg - 1 + kWave - 1) / kWave, (d.nyg - 2 + 3) / 4, std::min(d.nzg - 2, kRedZ));
}

void check_launch() {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        last_error() = std::string("kernel launch: ") + hipGetErrorString(e);
        throw DeviceError();
    }
}

constexpr int kZRows = 16, kZPre = 4;

// the matrix-core z DFT with RT row tiles (RT = rt, one instantiation per
// count); persistent blocks, one per compute unit
template <int RT>
void zdft_mf_launch(hipStream_t s, int rt, const ZTables &z, int C, long long plane, bool forward,
                    const double *in, double *out) {
    if constexpr (RT > 1) {
        if (rt < RT) {
            zdft_mf_launch<RT - 1>(s, rt, z, C, plane, forward, in, out);
            return;
        }
    }
    const double2 *zf = reinterpret_cast<const double2 *>(z.zf);
    int dev = 0, ncu = 0;
    BL_HIP(hipGetDevice(&dev));
    BL_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    const int tiles = (C + 15) / 16;
    const dim3 grid((unsigned)std::max(1, std::min(ncu, (tiles + kZmW - 1) / kZmW)));
    if (forward)
        hipLaunchKernelGGL((k_zdft_mf<true, RT>), grid, dim3(64 * kZmW), 0, s, z.M, C, plane, zf, in, out);
    else
        hipLaunchKernelGGL((k_zdft_mf<false, RT>), grid, dim3(64 * kZmW), 0, s, z.M, C, plane, zf, in, out);
    check_launch();
}

// the real z DFT (M points) of C columns with plane stride `plane`
void zdft_raw(hipStream_t s, const ZTables &z, int C, long long plane, bool forward, const double *in,
              double *out) {
    const int M = z.M, lda = z.lda, rows = M / 2 + 1;
    const double *zc = z.zc, *zs = z.zs;
    if (rows <= 16 * kZmRT) {
        if (!z.zf) {
            last_error() = "z transform: matrix-core tables missing";
            throw DeviceError();
        }
        zdft_mf_launch<kZmRT>(s, (rows + 15) / 16, z, C, plane, forward, in, out);
        return;
    }
    const dim3 grid(xcd_blocks((rows + kZRows - 1) / kZRows * ((C + 255) / 256)));
    if (forward)
        hipLaunchKernelGGL((k_zdft_fwd<kZRows, kZPre>), grid, dim3(256), 0, s, M, C, plane, lda, zc, zs, in, out);
    else
        hipLaunchKernelGGL((k_zdft_inv<kZRows, kZPre>), grid, dim3(256), 0, s, M, C, plane, lda, zc, zs, in, out);
    check_launch();
}

void zdft_launch(Handle &h, int kid, bool forward, const double *in, double *out) {
    ProfScope ps(h, kid);
    const Dims &d = h.d;
    const int C = d.N * d.NM;
    ZTables z;
    z.M = d.M;
    z.lda = h.lda_zt;
    z.zc = h.zc;
    z.zs = h.zs;
    z.zf = h.zf;
    zdft_raw(h.stream, z, C, (long long)C, forward, in, out);
}

template <class T>
void dct_launch(Handle &h, int kid, DctArgs<T> a, bool forward, const T *in, T *out, const Fld3<T> *div = nullptr,
                const BcPlanes<T> *bcp = nullptr, const IncSrc *incp = nullptr) {
    typedef typename Mf<T>::T2 T2;
    ProfScope ps(h, kid);
    const Dims &d = h.d;
    const BcPlanes<T> bc = bcp ? *bcp : BcPlanes<T>{};
    const IncSrc inc = incp ? *incp : IncSrc{};
    a.N = d.N;
    a.N1 = h.dct_n1;
    a.N2 = d.N / h.dct_n1;
    a.K1h = h.dct_n1 / 2;
    a.C1 = d.NM;
    a.C = d.NM * d.M;
    const int K1 = a.K1h + 1, ld = dct_ld(a.N2);
    a.rot = reinterpret_cast<const T2 *>(h.dct_tab);
    a.twA = a.rot + a.N;
    a.twC = a.twA + K1 * a.N2;
    a.t1 = a.twC + K1 * a.N2;
    a.t1i = a.t1 + dct_frag(a.N1);
    a.t2 = a.t1i + dct_frag(a.N1);
    const bool small = dct_small(a.N, a.N1);
    const DctPlan plan = dct_plan(a.N, a.N1, sizeof(T), a.C, h.n_cu);
    a.LB = plan.lines;
    const size_t lines = sizeof(T) * dct_lines(a.LB, a.N), spec = sizeof(T2) * (size_t)a.LB * K1 * ld;
    // the inverse past the SMALL shapes: V (an area that also holds the lines) and C~
    const size_t lds = small ? std::max(lines, spec) : (forward ? lines + spec : std::max(lines, spec) + spec);
    if (lds > 163840) {
        last_error() = "x transform length too large for the LDS-resident DCT (N = " + std::to_string(a.N) + ")";
        throw ArgError();
    }
    const dim3 grid((a.C + a.LB - 1) / a.LB), block(64 * plan.waves);
    auto fwd = [&](auto kern) {
        if (div)
            hipLaunchKernelGGL(kern, grid, block, lds, h.stream, a, d, h.m, bc, inc, div->u, div->v, div->w, out);
        else
            hipLaunchKernelGGL(kern, grid, block, lds, h.stream, a, d, h.m, bc, inc, in, nullptr, nullptr, out);
    };
    if (forward) {
        if (div)
            small ? fwd(k_dct_fwd_m<true, true, T>) : fwd(k_dct_fwd_m<true, false, T>);
        else if constexpr (sizeof(T) == 8)
            small ? fwd(k_dct_fwd_m<false, true, T>) : fwd(k_dct_fwd_m<false, false, T>);
    } else if (small) {
        hipLaunchKernelGGL((k_dct_inv_m<true, T>), grid, block, lds, h.stream, a, in, out);
    } else {
        hipLaunchKernelGGL((k_dct_inv_m<false, T>), grid, block, lds, h.stream, a, in, out);
    }
    check_launch();
}

}  // namespace

void launch_zdft(hipStream_t s, const ZTables &z, int C, long long plane, bool forward, const double *in,
                 double *out) {
    zdft_raw(s, z, C, plane, forward, in, out);
}

const char *kernel_name(int id) {
    static const char *names[KID_COUNT] = {
        "rk_stage", "bc_inout", "bc_periodic", "bc_topwall", "bc_massflux", "divergence",
        "xform_x_fwd", "xform_z_fwd", "thomas", "xform_z_inv", "xform_x_inv", "project",
        "reduce", "dsm_cells", "dsm_vfilter", "dsm_filter", "dsm_column", "closure"};
    return (id >= 0 && id < KID_COUNT) ? names[id] : "";
}

// ------------------------------------------------------------------------
// launch wrappers
// ------------------------------------------------------------------------
template <>
const MetricsT<double> &metrics<double>(const Handle &h) {
    return h.m;
}
template <>
const MetricsT<float> &metrics<float>(const Handle &h) {
    return h.mf;
}


// Whether a march accesses what it touches once (the old field and all results)
// past the caches: where its nine arrays (the field, the old one or F1, the
// result) exceed the 256 MB of the last-level cache.  RK stage and the x
// transform behind it, plain -> non-temporal: 814x257x193 FP64 670 -> 646 and
// 345 -> 327 us, FP32 453 -> 452 and 220 -> 209; 513x97x130 FP64 (470 MB) 109 ->
// 95 and 87 -> 84; but 262x66x230 FP32 (150 MB) 47 -> 48 and 39 -> 42.
template <class T>
bool march_streams(const Dims &d) {
    return 9.0 * sizeof(T) * (double)d.sxy * d.nzg > 256.0 * 1024 * 1024;
}

template <int MODE, int FOUT, class T>
void march(Handle &h, const Fld3<T> &cur, const Fld3<T> *old, const Fld3<T> *f1, Fld3<T> *nxt, Fld3<T> *fo,
           double c0, double c1, double dt, double g2 = 0.0) {
    const Dims &d = h.d;
    const int tiles = march_tiles<T>(d.nxg, d.nyg);
    const int chunk = march_chunk(d.nzg - 2, tiles, h.n_cu, march_resident<T>(h.les != 0));
    const dim3 grid(xcd_blocks(tiles * ((d.nzg - 2 + chunk - 1) / chunk))), block(256);
    const T *o[3] = {old ? old->u : nullptr, old ? old->v : nullptr, old ? old->w : nullptr};
    const T *f[3] = {f1 ? f1->u : nullptr, f1 ? f1->v : nullptr, f1 ? f1->w : nullptr};
    T *n[3] = {nxt ? nxt->u : nullptr, nxt ? nxt->v : nullptr, nxt ? nxt->w : nullptr};
    T *r[3] = {fo ? fo->u : nullptr, fo ? fo->v : nullptr, fo ? fo->w : nullptr};
    const MetricsT<T> &m = metrics<T>(h);
    auto launch = [&](auto kernel, const T *nut) {
        hipLaunchKernelGGL(kernel, grid, block, 0, h.stream, d, m, (T)h.nu, (T)h.dPdx, (T)h.dPdz, chunk, cur.u, cur.v,
                           cur.w, nut, o[0], o[1], o[2], f[0], f[1], f[2], n[0], n[1], n[2], r[0], r[1], r[2], (T)c0,
                           (T)c1, (T)dt, (T)g2);
    };
    const T *nut = reinterpret_cast<const T *>(h.nu_t);
    if (h.les != 0 && march_streams<T>(d))
        launch(k_rk_march<MODE, FOUT, true, true, T>, nut);
    else if (h.les != 0)
        launch(k_rk_march<MODE, FOUT, true, false, T>, nut);
    else if (march_streams<T>(d))
        launch(k_rk_march<MODE, FOUT, false, true, T>, nullptr);
    else
        launch(k_rk_march<MODE, FOUT, false, false, T>, nullptr);
    check_launch();
}

template <class T>
void launch_rk_stage(Handle &h, const Fld3<T> &cur, const Fld3<T> &old, Fld3<T> &nxt, int stage, double dt) {
    const bool rk3 = h.scheme == 3;
    Fld3<T> F1 = as<T>(h.F1);
    ProfScope ps(h, KID_RK_STAGE);
    // FP64 RK3 carries G = Uo + dt a21 F1 (= Uo + dt a31 F1) from the first
    // stage in the F1 buffers; FP32 fields carry Uo and F1, since storing G in
    // FP32 would round a velocity-sized value once more per stage
    const bool gform = rk3 && sizeof(T) == 8;
    if (stage == 1) {
        const double c0 = dt * (rk3 ? h.rk_coef[1][1] : h.rk2_coef[1][1]);
        if (gform)
            march<0, 2>(h, cur, &old, (const Fld3<T> *)nullptr, &nxt, &F1, c0, 0.0, dt, dt * h.rk_coef[2][1]);
        else if (rk3 || sizeof(T) == 4)
            // FP32 RK2 keeps F1 too: it is the first stage's pressure source
            march<0, 1>(h, cur, &old, (const Fld3<T> *)nullptr, &nxt, &F1, c0, 0.0, dt);
        else
            march<0, 0>(h, cur, &old, (const Fld3<T> *)nullptr, &nxt, (Fld3<T> *)nullptr, c0, 0.0, dt);
    } else if (!rk3) {
        // RK2 second stage: Uo + dt*(0*F1 + 1*F2) == Uo + dt*F2 exactly
        march<0, 0>(h, cur, &old, (const Fld3<T> *)nullptr, &nxt, (Fld3<T> *)nullptr, dt * h.rk2_coef[2][2],
                    0.0, dt);
    } else if (gform) {
        // RK3 stages 2, 3: new = G + dt a_ss F (a_32 = 0 so F2 is never needed)
        march<0, 0>(h, cur, &F1, (const Fld3<T> *)nullptr, &nxt, (Fld3<T> *)nullptr, dt * h.rk_coef[stage][stage],
                    0.0, dt);
    } else {
        // RK3 stages 2, 3: a_32 = 0 so F2 is never needed
        const double c1 = h.rk_coef[stage][1], c0 = h.rk_coef[stage][stage];
        march<1, 0>(h, cur, &old, &F1, &nxt, (Fld3<T> *)nullptr, c0, c1, dt);
    }
}

template <class T>
void launch_rhs_only(Handle &h, const Fld3<T> &cur, Fld3<T> &rhs) {
    march<2, 0>(h, cur, (const Fld3<T> *)nullptr, (const Fld3<T> *)nullptr, (Fld3<T> *)nullptr, &rhs, 0.0, 0.0,
                0.0);
}

namespace {
// elements of one stage's BcPlanes
long long bc_stride(const Dims &d) {
    return ((6LL * d.nyg + d.nxg) * d.nzg + d.nxg + 31) / 32 * 32;
}
int bc_partials(const Dims &d) { return ((d.nyg + 255) / 256 + (d.nxg + 255) / 256) * d.nzg; }
}  // namespace

size_t bc_doubles(const Dims &d) { return 3 * ((size_t)bc_stride(d) + bc_partials(d)) + 8; }

template <class T>
BcPlanes<T> bc_planes(const Handle &h, int stage) {
    const Dims &d = h.d;
    const long long npl = (long long)d.nyg * d.nzg;
    T *p = reinterpret_cast<T *>(h.bc_mem) + (stage - 1) * bc_stride(d);
    BcPlanes<T> b;
    T **f[6] = {&b.uin, &b.vin, &b.win, &b.uo, &b.vo, &b.wo};
    for (int q = 0; q < 6; ++q) *f[q] = p + q * npl;
    b.vtop = p + 6 * npl;
    b.vwall = b.vtop + d.nxg;
    b.wld = wall_model_robin(h.bc.iwall) ? d.nxg : 0;
    b.du = h.bc_mem + 3 * bc_stride(d) + (stage - 1);
    return b;
}

template <class T>
void launch_bc_planes(Handle &h, const Fld3<T> &old, int first, int nst, double dt, const double *t, double *inc1,
                      double t_old) {
    const Dims &d = h.d;
    BcStages st{};
    for (int s = 0; s < nst; ++s) {
        st.coef[s] = h.rk_t[first + s] * dt * h.bc_uc;
        st.t[s] = t[s];
    }
    const BcPlanes<T> p = bc_planes<T>(h, first);
    const int nb_in = (d.nyg + 255) / 256, nb = nb_in + (d.nxg + 255) / 256, nq = bc_partials(d);
    double *qpart = h.bc_mem + 3 * bc_stride(d) + 8;
    {
        ProfScope ps(h, KID_BC_INOUT);
        hipLaunchKernelGGL(k_bc_planes<T>, dim3(nb, d.nzg, nst), dim3(256), 0, h.stream, d, h.m, h.bc, p, bc_stride(d),
                           old.u, old.v, old.w, st, nb_in, qpart, inc1, t_old);
        check_launch();
    }
    ProfScope ps(h, KID_BC_MASSFLUX);
    hipLaunchKernelGGL(k_bc_shift, dim3(nst), dim3(256), 0, h.stream, d, h.length_y, qpart, nq, p.du,
                       inc1 ? inc1 + 2 * (long long)d.nyg * d.nzg : nullptr);
    check_launch();
}

template <class T>
void launch_bc(Handle &h, Fld3<T> &f, int stage) {
    const Dims &d = h.d;
    ProfScope ps(h, KID_BC_TOPWALL);
    const long long n = 3LL * d.nxg * d.nyg + (long long)d.nxg * (d.nzg - 3) + (long long)(d.nyg - 2) * (d.nzg - 3);
    hipLaunchKernelGGL(k_bc_apply<T>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, h.stream, d, h.m, h.bc,
                       bc_planes<T>(h, stage), f.u, f.v, f.w);
    check_launch();
}

bool bc_called(Handle &h) {
    // U_top is the Falkner-Skan profile from the first call on, and with it
    // the outflow's convective velocity U_top(nx)
    if (!h.fs_uc_pending) return false;
    h.bc_uc = h.fs_uc;
    h.fs_uc_pending = false;
    return true;
}

void launch_poisson(Handle &h, double *phi, const Field3 *div, const BcPlanes<double> *bc) {
    const Dims &d = h.d;
    const int N = d.N, M = d.M, NM = d.NM;
    const long long plane = (long long)N * NM;
    // forward x: lines (j, m) of the padded field -> T1[m][j][kx]
    DctArgs<double> da{};
    da.in_base = fidx(d, 1, 1, 1);
    da.in_c1 = d.sx;
    da.in_c2 = d.sxy;
    da.out_base = 0;
    da.out_c1 = N;
    da.out_c2 = plane;
    da.scale = 1.0;
    dct_launch(h, KID_XFORM_X_FWD, da, true, (const double *)phi, h.T1, div, bc);
    // forward z: columns (kx, j) of T1 -> S[q][j][kx]
    zdft_launch(h, KID_XFORM_Z_FWD, true, h.T1, h.S);
    {
    ProfScope ps(h, KID_THOMAS);
    // the partitioned kernel leaves the (0,0) column of S to its block 0,
    // which solves it in place; the table kernel (no length limit) solves it
    // with the other systems
    if (h.th_p != 0) {
        launch_thomas_seg<double>(h, h.S, N, (long long)plane, solve00_args(h, h.S, N, 1.0, nullptr, 0));
    } else {
        hipLaunchKernelGGL(k_thomas<8>, dim3((N + 255) / 256 * M), dim3(256), 0, h.stream, d, h.lu_dl,
                           h.lu_dp, h.lu_du, h.S);
        check_launch();
    }
    }
    // inverse z: S -> T1
    zdft_launch(h, KID_XFORM_Z_INV, false, h.S, h.T1);
    // inverse x: T1[m][j][kx] -> phi cells (1..N, 1..NM, 1..M)
    da.in_base = 0;
    da.in_c1 = N;
    da.in_c2 = plane;
    da.out_base = fidx(d, 1, 1, 1);
    da.out_c1 = d.sx;
    da.out_c2 = d.sxy;
    da.scale = 1.0 / ((double)N * (double)M);
    dct_launch(h, KID_XFORM_X_INV, da, false, (const double *)h.T1, phi);
}

void launch_xfwd_mixed(Handle &h, const Fld3<float> &f, float *T1, const BcPlanes<float> *bc, const IncSrc *inc) {
    const Dims &d = h.d;
    DctArgs<float> a{};
    a.out_c1 = h.NP;
    a.out_c2 = (long long)h.NP * d.NM;
    a.part = h.p00;
    a.part_ld = d.M;
    dct_launch(h, KID_XFORM_X_FWD, a, true, (const float *)nullptr, T1, &f, bc, inc);
}

void launch_xinv_mixed(Handle &h, const float *T1, const double *add, float *phi) {
    const Dims &d = h.d;
    DctArgs<float> a{};
    a.in_c1 = h.NP;
    a.in_c2 = (long long)h.NP * d.NM;
    a.out_base = fidx(d, 1, 1, 1);
    a.out_c1 = d.sx;
    a.out_c2 = d.sxy;
    a.scale = (float)(1.0 / ((double)d.N * (double)d.M));
    a.add = add;
    dct_launch(h, KID_XFORM_X_INV, a, false, T1, phi);
}

template <class T>
bool launch_thomas_seg(Handle &h, T *S, int ldj, long long ldq, const Solve00 &z) {
    const Dims &d = h.d;
    if (h.th_p == 0) return false;
    // the resident blocks, each looping over its tiles, one of them block 0 for the
    // (0,0) system.  With one block per CU also where a block is 3 waves the solve
    // took 39 us at 260x65x228 (FP32).
    const int ntiles = (d.N + 63) / 64 * d.M;
    const int nblk = std::max(1, std::min(ntiles, std::max(2, h.n_cu) * thomas_resident(h.th_p) - 1));
    hipLaunchKernelGGL(k_thomas_seg<T>, dim3(1 + nblk), dim3(64 * h.th_p), 0, h.stream, d.N, d.NM, h.th_p, d.M,
                       ldj, ldq, (const double *)h.th_co, z.part ? 1 : 0, S, z);
    check_launch();
    return true;
}

Solve00 solve00_args(const Handle &h, double *x, int ldx, double scale, const double *part, int npart) {
    if (h.d.NM > kMax00) {
        last_error() = "internal: the (0,0) system is longer than the solve kernel holds";
        throw ArgError();
    }
    Solve00 z;
    z.L00 = h.lu00;
    z.D00 = h.lu00 + h.d.NM;
    z.du = h.lu_du;
    z.part = part;
    z.npart = npart;
    z.x = x;
    z.ldx = ldx;
    z.scale = scale;
    return z;
}

void launch_solve00(Handle &h, const Solve00 &z) {
    hipLaunchKernelGGL(k_solve00, dim3(1), dim3(256), 0, h.stream, h.d.NM, z);
    check_launch();
}

template <class T>
void launch_project(Handle &h, Fld3<T> &f, const T *phi, T *P, double dt) {
    const Dims &d = h.d;
    ProfScope ps(h, KID_PROJECT);
    const dim3 grid(xcd_blocks((d.nxg - 1 + kWave - 1) / kWave * ((d.nyg - 2 + 3) / 4) *
                               ((d.nzg - 2 + kProjZ - 1) / kProjZ)));
    const double den = dt * h.rk2_coef[1][1];
    hipLaunchKernelGGL(k_project<T>, grid, dim3(kWave, 4), 0, h.stream, d, metrics<T>(h), f.u, f.v, f.w, phi, P,
                       den);
    check_launch();
}

long long maxdiv_partials(int nxg, int nyg, int nzg) {
    Dims d{};
    d.nxg = nxg;
    d.nyg = nyg;
    d.nzg = nzg;
    const dim3 g = reduce_grid(d);
    return (long long)g.x * g.y * g.z;
}

template <class T>
void launch_maxdiv(hipStream_t stream, const DivArgs &a, const T *U, const T *V, const T *W, double *part,
                   double *out) {
    Dims d{};
    d.nxg = a.nxg;
    d.nyg = a.nyg;
    d.nzg = a.nzg;
    const dim3 g = reduce_grid(d);
    const long long nb = (long long)g.x * g.y * g.z;
    hipLaunchKernelGGL(k_maxdiv<T>, g, dim3(kWave, 4), 0, stream, a, U, V, W, part);
    check_launch();
    hipLaunchKernelGGL(k_reduce_max, dim3(1), dim3(1024), 0, stream, part, nb, 1, out);
    check_launch();
}
template void launch_maxdiv<double>(hipStream_t, const DivArgs &, const double *, const double *, const double *,
                                    double *, double *);

template <class T>
double max_divergence(Handle &h, const Fld3<T> &f) {
    const Dims &d = h.d;
    DivArgs a{};
    a.nxg = d.nxg;
    a.nyg = d.nyg;
    a.nzg = d.nzg;
    a.u1 = a.v1 = a.w1 = d.sx;
    a.u2 = a.v2 = a.w2 = d.sxy;
    a.rdx = h.m.rdx;
    a.rdy = h.m.rdy;
    a.rdz = h.m.rdz;
    launch_maxdiv(h.stream, a, f.u, f.v, f.w, h.red, h.scal);
    double v = 0.0;
    BL_HIP(hipMemcpyAsync(&v, h.scal, sizeof(double), hipMemcpyDeviceToHost, h.stream));
    BL_HIP(hipStreamSynchronize(h.stream));
    return v;
}

template <class T>
double dt_convective(Handle &h, const Fld3<T> &f) {
    const Dims &d = h.d;
    ProfScope ps(h, KID_REDUCE);
    const dim3 g = reduce_grid(d);
    const long long nb = (long long)g.x * g.y * g.z;
    hipLaunchKernelGGL(k_dtconv<T>, g, dim3(kWave, 4), 0, h.stream, d, h.m, f.u, f.v, f.w, h.red);
    check_launch();
    hipLaunchKernelGGL(k_reduce_max, dim3(1), dim3(1024), 0, h.stream, h.red, nb, 3, h.scal);
    check_launch();
    double v[3];
    BL_HIP(hipMemcpyAsync(v, h.scal, 3 * sizeof(double), hipMemcpyDeviceToHost, h.stream));
    BL_HIP(hipStreamSynchronize(h.stream));
    const double CFLa = std::fabs(h.cfl);
    const double dcu = CFLa * v[0], dcv = CFLa * v[1], dcw = CFLa * v[2];
    return std::fmin(dcu, std::fmin(dcv, dcw));
}

template <class T>
void wall_stats(Handle &h, const Fld3<T> &f, double *cf_host) {
    const Dims &d = h.d;
    hipLaunchKernelGGL(k_wallstats<T>, dim3((d.nx + 63) / 64), dim3(64 * kWsZ), 0, h.stream, d, h.m, h.nu, f.u, f.v,
                       reinterpret_cast<const T *>(h.nu_t), h.red);
    check_launch();
    BL_HIP(hipMemcpyAsync(cf_host, h.red, sizeof(double) * d.nx, hipMemcpyDeviceToHost, h.stream));
    BL_HIP(hipStreamSynchronize(h.stream));
}

template <class T>
void monitor(Handle &h, const Fld3<T> &f, double *out) {
    const Dims &d = h.d;
    const dim3 g((d.nyg - 2 + kMonJ - 1) / kMonJ, d.nzg - 2);
    hipLaunchKernelGGL(k_monitor<T>, g, dim3(256), 0, h.stream, d, f.u, f.v, f.w, reinterpret_cast<const T *>(h.nu_t),
                       h.red);
    check_launch();
    hipLaunchKernelGGL(k_monitor_reduce, dim3(8), dim3(256), 0, h.stream, h.red, (long long)g.x * g.y, h.scal);
    check_launch();
    BL_HIP(hipMemcpyAsync(out, h.scal, 8 * sizeof(double), hipMemcpyDeviceToHost, h.stream));
    BL_HIP(hipStreamSynchronize(h.stream));
}

long long monitor_partials(const Dims &d) { return 8LL * ((d.nyg - 2 + kMonJ - 1) / kMonJ) * (d.nzg - 2); }

#define BL_INSTANTIATE(T)                                                                                   \
    template void launch_rk_stage<T>(Handle &, const Fld3<T> &, const Fld3<T> &, Fld3<T> &, int, double); \
    template void launch_rhs_only<T>(Handle &, const Fld3<T> &, Fld3<T> &);                                \
    template BcPlanes<T> bc_planes<T>(const Handle &, int);                                                \
    template void launch_bc_planes<T>(Handle &, const Fld3<T> &, int, int, double, const double *, double *, \
                                      double);                                                             \
    template void launch_bc<T>(Handle &, Fld3<T> &, int);                                                  \
    template void launch_project<T>(Handle &, Fld3<T> &, const T *, T *, double);                         \
    template bool launch_thomas_seg<T>(Handle &, T *, int, long long, const Solve00 &);                   \
    template double max_divergence<T>(Handle &, const Fld3<T> &);                                         \
    template double dt_convective<T>(Handle &, const Fld3<T> &);                                          \
    template void wall_stats<T>(Handle &, const Fld3<T> &, double *);                                     \
    template void monitor<T>(Handle &, const Fld3<T> &, double *);
BL_INSTANTIATE(double)
BL_INSTANTIATE(float)
#undef BL_INSTANTIATE

}  // namespace blgpu
